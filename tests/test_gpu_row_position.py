"""A token's FP8 result does not depend on where its row stands in the call:
one activation row repeated over all rows gives one output row, on every
planned kernel family whose K walk starts at different places in different
workgroups. The operands cancel (the second half of K repeats the first with
the weights negated, so every exact sum is zero): what is left is the rounding
of the fp32 sums, which any change of their order changes."""
import numpy as np
import pytest
import torch

from breeze_tts_cpp_amd import qlinear
from tests.test_gpu_gemm import bits_to_f32, dev_f32, dev_u8, gpu_gemm, operands

FP8 = 3
SLICED = [(16, 16), (16, 64), (32, 32), (32, 80), (48, 96), (64, 48), (64, 128), (96, 96)]


def cancelling(N, K, seed):
    """One row of codes [K] and weights [N, K], finite e4m3 codes of every size."""
    rng = np.random.default_rng(seed)
    def codes(shape):
        c = rng.integers(0, 256, shape, dtype=np.uint8)
        return np.where(c & 0x7F == 0x7F, c ^ 1, c).astype(np.uint8)
    a, b = codes(K // 2), codes((N, K // 2))
    return np.concatenate([a, a]), np.concatenate([b, b ^ 0x80], axis=1)


def check(dev, M, N, K, path=None):
    row, w = cancelling(N, K, M + N + K)
    x = dev_u8(np.broadcast_to(row, (M, K)), dev)
    sx, sw = dev_f32(np.full(M, 64.0), dev), dev_f32(np.full(N, 64.0), dev)
    wq = dev_u8(w, dev)
    for weights in (wq, qlinear.pack_weights(wq)):
        y = qlinear.gemm(x, sx, weights, sw, FP8, path=path).float()
        torch.cuda.synchronize()
        assert torch.isfinite(y).all() and (y[0] != 0).any()  # rounding is visible
        moved = (y != y[0]).any(dim=1).nonzero().flatten().tolist()
        assert not moved, f"{len(moved)} of {M} rows differ from row 0: {moved[:8]}"


# K-sliced tiles at 33 to 999 rows; macro tiles whose walk may be turned (one
# round of 128x128, 128x64 and 256x128 tiles; all of K in one window).
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 1024, 6144), (57, 2048, 6144), (187, 2048, 6144),
                                   (431, 2048, 6144), (999, 1024, 4096), (730, 4096, 2048),
                                   (1024, 4096, 2048), (1024, 2048, 6144), (4096, 2048, 6144),
                                   (431, 12288, 2048), (64, 4096, 2048), (2048, 12288, 2048)])
def test_planned(dev, M, N, K):
    print(f"row position {qlinear.plan(M, N, K, FP8)} M={M} N={N} K={K}", flush=True)
    check(dev, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("channels,tokens", SLICED)
def test_sliced_tiles(dev, channels, tokens):
    print(f"row position sliced {channels}x{tokens}", flush=True)
    check(dev, 3 * tokens + 5, 8 * channels, 6144,
          qlinear.Path(qlinear.KIND_SKINNY, tokens, channels, 1, 8, 3))


@pytest.mark.gpu
@pytest.mark.parametrize("channels,tokens", [(128, 64), (128, 128), (256, 128), (256, 256)])
def test_macro_tiles(dev, channels, tokens):
    print(f"row position tile {channels}x{tokens}", flush=True)
    check(dev, 3 * tokens + 5, 6 * channels, 4096,
          qlinear.Path(qlinear.KIND_TILED, tokens, channels, 1, 8))


# Windows with nothing, whole stages, an odd stage and a partial one behind
# them; K too short for a window; five token tiles, the last one ragged.
@pytest.mark.gpu
@pytest.mark.parametrize("K", [512, 1024, 1280, 1424, 2064, 4096, 5264])
def test_turned_sums(dev, orc, K):
    """The turned tiles' outputs against the 256x256 tile's, which sums K in
    ascending order: the two fp32 sums of a row differ by about K * 2^-24 of
    its terms' size, an output by at most one bf16 unit (2^-7 relative of the
    larger of the two, or of the row's scale)."""
    M, N = 4 * 128 + 37, 272
    xq, sx, wq, sw = operands(orc, M, N, K, FP8, seed=K)
    ref = bits_to_f32(gpu_gemm(dev, xq, sx, wq, sw, FP8,
                               path=qlinear.Path(qlinear.KIND_TILED, 256, 256, 1, 8)))
    bound = 2.0 ** -7 * np.maximum(np.abs(ref), 2.0 ** -9 * np.abs(ref).max(axis=1, keepdims=True))
    for channels in (128, 256):
        print(f"turned sums {channels}x128 K={K}", flush=True)
        path = qlinear.Path(qlinear.KIND_TILED, 128, channels, 1, 8)
        y = gpu_gemm(dev, xq, sx, wq, sw, FP8, path=path)
        assert (np.abs(bits_to_f32(y) - ref) <= bound).all()
        packed = qlinear.gemm(dev_u8(xq, dev), dev_f32(sx, dev), qlinear.pack_weights(dev_u8(wq, dev)),
                              dev_f32(sw, dev), FP8, path=path)
        assert np.array_equal(packed.cpu().view(torch.int16).numpy().view(np.uint16), y)
