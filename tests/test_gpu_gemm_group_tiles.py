"""The 64-channel macro tiles of the K-group GEMM (groups of 128): ragged rows,
channels and K, one side per row, finish, packed weights and f16 outputs,
against the oracle; and the planner's rule for them."""
import numpy as np
import pytest
import torch

from breeze_tts_cpp_amd import qlinear, synthetic
from tests.test_gpu_finish import run_finish
from tests.test_gpu_gemm import FP8_REL_L2, bits_to_f32, dev_f32, dev_u8, gpu_gemm, out_bits, rel_l2

I8, FP8, BF16, F16 = 4, 3, 0, 5
TILES = [(64, 32, 4), (64, 64, 8)]


def path(channels, tokens, waves):
    return qlinear.Path(qlinear.KIND_TILED, tokens, channels, 1, waves)


def operands(orc, M, N, K, fmt, ig=128, wg=128):
    quantize = lambda b, g: orc.quantize_rows(b, fmt, group=g) if g else orc.quantize_rows(b, fmt)
    return (*quantize(synthetic.activations(M, K, seed=M + K), ig),
            *quantize(synthetic.weights(N, K, seed=N + K), wg))


# K = 16: one partial group; 1040: a short last group; 2048: whole groups past
# the ring; N not a multiple of 64, M one row, a partial and a whole last tile.
@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [I8, FP8])
@pytest.mark.parametrize("M,N,K,ig,wg", [(1, 16, 16, 128, 128), (100, 112, 1040, 128, 128),
                                         (256, 128, 2048, 128, 128), (131, 208, 2048, 128, 0),
                                         (131, 208, 912, 0, 128)])
def test_group_tiles(dev, orc, fmt, M, N, K, ig, wg):
    xq, sx, wq, sw = operands(orc, M, N, K, fmt, ig, wg)
    x, s, w, t = dev_u8(xq, dev), dev_f32(sx, dev), dev_u8(wq, dev), dev_f32(sw, dev)
    groups = dict(input_group=ig, weight_group=wg)
    for tile in TILES:
        p = path(*tile)
        print(f"group tile {tile} fmt={fmt} M={M} N={N} K={K} groups {ig}/{wg}", flush=True)
        y = out_bits(qlinear.gemm(x, s, w, t, fmt, path=p, **groups))
        if fmt == I8:
            ref, _ = orc.gemm_grouped(xq, sx, wq, sw, fmt, ig, wg,
                                      *qlinear.grouped_partition(p, K))
            assert np.array_equal(y, ref), f"{np.count_nonzero(y != ref)} mismatches"
        else:
            assert rel_l2(bits_to_f32(y), orc.gemm_grouped_ideal(xq, sx, wq, sw, fmt, ig, wg)) <= FP8_REL_L2
        packed = qlinear.gemm(x, s, qlinear.pack_weights(w), t, fmt, path=p, **groups)
        assert np.array_equal(out_bits(packed), y), "packed weights differ"
        # an output that starts 8 bytes past 16-byte alignment
        flat = torch.empty(M * N + 4, dtype=torch.bfloat16, device=dev)
        qlinear.gemm(x, s, w, t, fmt, path=p, out=flat[4:].view(M, N), **groups)
        torch.cuda.synchronize()
        assert np.array_equal(out_bits(flat[4:]).reshape(M, N), y)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [I8, FP8])
@pytest.mark.parametrize("out_dtype,out_type", [(torch.bfloat16, BF16), (torch.float16, F16)])
def test_group_tiles_finish(dev, orc, fmt, out_dtype, out_type):
    M, N, K = 75, 176, 1072
    xq, sx, wq, sw = operands(orc, M, N, K, fmt)
    bias = np.random.default_rng(fmt).standard_normal(N).astype(np.float32) * 0.5
    bias = (bias.astype(np.float16).view(np.uint16) if out_type == F16
            else (bias.view(np.uint32) >> 16).astype(np.uint16))
    for tile in TILES:
        p = path(*tile)
        plain = gpu_gemm(dev, xq, sx, wq, sw, fmt, group=128, path=p, out_dtype=out_dtype)
        for act in (0, 1, 2):
            for packed in (False, True):
                print(f"group tile finish {tile} fmt={fmt} out={out_type} act={act} packed={packed}",
                      flush=True)
                y = run_finish(dev, xq, sx, wq, sw, fmt, bias, act, path=p, out_dtype=out_dtype,
                               group=128, packed=packed)
                assert np.array_equal(y, orc.finish(plain, bias, act, out_type=out_type))


def test_group_tile_plans():
    """The smallest tile whose grid is one round of workgroups."""
    def tile(M, N, K, ig=128, wg=128):
        p = qlinear.plan(M, N, K, I8, ig, wg)
        return (p.channels, p.tokens, p.waves)
    assert tile(187, 2048, 6144) == (64, 32, 4)
    assert tile(187, 4096, 2048) == (64, 64, 8)
    assert tile(431, 4096, 2048, 0, 128) == (128, 64, 8)
    assert tile(260, 6144, 1024) == (128, 64, 8)
    assert tile(640, 4096, 2048) == (128, 128, 8)
    assert tile(431, 12288, 2048) == (256, 128, 8)
    assert tile(1024, 2048, 2048) == (128, 64, 8)


@pytest.mark.gpu
def test_group_tiles_refused(dev, orc):
    """Per-channel scales and smaller groups have no 64-channel tile."""
    xq, sx, wq, sw = operands(orc, 40, 64, 256, I8, 0, 0)
    for group in (0, 32, 64):
        for tile in TILES:
            with pytest.raises(RuntimeError, match="64x32"):
                gpu_gemm(dev, xq, sx, wq, sw, I8, group=group, path=path(*tile))
