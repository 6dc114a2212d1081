"""The K-sliced GEMM (gemm_sliced.hip): every tile on ragged shapes, K slices
that are short or empty, the finish, packed weights, f16 outputs and outputs
of 8-byte alignment, against the oracle and the macro-tile path; and the
planner's rule for it."""
import numpy as np
import pytest
import torch

from breeze_tts_cpp_amd import qlinear
from tests.test_gpu_finish import run_finish
from tests.test_gpu_gemm import (FP8_REL_L2, bits_to_f32, check_i8, dev_f32, dev_u8, gpu_gemm,
                                 operands, out_bits, rel_l2)

I8, FP8, BF16, F16 = 4, 3, 0, 5
TILES = [(16, 16), (16, 32), (16, 48), (16, 64), (32, 16), (32, 32), (32, 48), (32, 64), (32, 80),
         (48, 32), (48, 48), (48, 64), (48, 80), (48, 96), (64, 32), (64, 48), (64, 64),
         (64, 96), (64, 128), (96, 64), (96, 96)]


def path(channels, tokens):
    return qlinear.Path(qlinear.KIND_SKINNY, tokens, channels, 1, 8, 3)


# K = 16: one chunk, all slices but the first empty; 1040: a slice of one
# stage and an empty one; 3088: stages past the ring of all but the 16x16
# tile, the last one partial; 4096: slices of four whole stages; 5264: slices
# of six stages, past every ring, which INT8 tiles of 32 and more channels walk
# from different starts, a slice that ends in a partial stage and an empty one.
@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [I8, FP8])
@pytest.mark.parametrize("M,N,K", [(1, 16, 16), (100, 112, 1040), (197, 208, 3088), (130, 96, 4096),
                                   (130, 96, 5264)])
def test_sliced_tiles(dev, orc, fmt, M, N, K):
    xq, sx, wq, sw = operands(orc, M, N, K, fmt, seed=M + K)
    ideal = None if fmt == I8 else orc.gemm_fp8_ideal(xq, sx, wq, sw)
    for channels, tokens in TILES:
        p = path(channels, tokens)
        print(f"sliced {channels}x{tokens} fmt={fmt} M={M} N={N} K={K}", flush=True)
        y = gpu_gemm(dev, xq, sx, wq, sw, fmt, path=p)
        if fmt == I8:
            check_i8(orc, y, xq, sx, wq, sw)
        else:
            assert rel_l2(bits_to_f32(y), ideal) <= FP8_REL_L2
        w = qlinear.pack_weights(dev_u8(wq, dev))
        packed = qlinear.gemm(dev_u8(xq, dev), dev_f32(sx, dev), w, dev_f32(sw, dev), fmt, path=p)
        assert np.array_equal(out_bits(packed), y), "packed weights differ"
        # an output that starts 8 bytes past 16-byte alignment
        flat = torch.empty(M * N + 4, dtype=torch.bfloat16, device=dev)
        qlinear.gemm(dev_u8(xq, dev), dev_f32(sx, dev), dev_u8(wq, dev), dev_f32(sw, dev), fmt,
                     path=p, out=flat[4:].view(M, N))
        torch.cuda.synchronize()
        assert np.array_equal(out_bits(flat[4:]).reshape(M, N), y)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [I8, FP8])
@pytest.mark.parametrize("out_dtype,out_type", [(torch.bfloat16, BF16), (torch.float16, F16)])
def test_sliced_finish(dev, orc, fmt, out_dtype, out_type):
    M, N, K = 75, 176, 1072
    xq, sx, wq, sw = operands(orc, M, N, K, fmt, seed=7)
    bias = np.random.default_rng(fmt).standard_normal(N).astype(np.float32) * 0.5
    bias = (bias.astype(np.float16).view(np.uint16) if out_type == F16
            else (bias.view(np.uint32) >> 16).astype(np.uint16))
    for channels, tokens in ((16, 32), (32, 48), (64, 64), (96, 96)):
        p = path(channels, tokens)
        plain = gpu_gemm(dev, xq, sx, wq, sw, fmt, path=p, out_dtype=out_dtype)
        for act in (0, 1, 2):
            for packed in (False, True):
                print(f"sliced finish {p} fmt={fmt} out={out_type} act={act} packed={packed}",
                      flush=True)
                y = run_finish(dev, xq, sx, wq, sw, fmt, bias, act, path=p, out_dtype=out_dtype,
                               packed=packed)
                assert np.array_equal(y, orc.finish(plain, bias, act, out_type=out_type))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [I8, FP8])
def test_planned_equals_macro_tile(dev, orc, fmt):
    """Shapes whose plan is K-sliced give the macro tile's output: the same
    bits for INT8; for FP8 sums in another order, which move an fp32 sum by
    about K * 2^-24 of its terms' size and so an output by at most one bf16
    unit (2^-7 relative of the larger of the two, or of the row's scale)."""
    for M, N, K in ((33, 1024, 6144), (65, 1168, 1040), (187, 2048, 6144), (300, 2832, 1536),
                    (999, 1024, 1024)):
        planned = qlinear.plan(M, N, K, fmt)
        assert planned.kind == qlinear.KIND_SKINNY and planned.staged == 3, (M, N, K, planned)
        print(f"planned {planned} fmt={fmt} M={M} N={N} K={K}", flush=True)
        xq, sx, wq, sw = operands(orc, M, N, K, fmt, seed=M)
        y = gpu_gemm(dev, xq, sx, wq, sw, fmt)
        tile = gpu_gemm(dev, xq, sx, wq, sw, fmt, path=qlinear.Path(qlinear.KIND_TILED, 128, 128, 1, 8))
        if fmt == I8:
            assert np.array_equal(y, tile)
        else:
            a, b = bits_to_f32(y), bits_to_f32(tile)
            bound = 2.0 ** -7 * np.maximum(np.abs(b), 2.0 ** -9 * np.abs(b).max(axis=1, keepdims=True))
            assert (np.abs(a - b) <= bound).all()


def test_sliced_plan_rule():
    """One round of workgroups, nothing from 1024 rows or with K groups, and
    decode shapes only above 32 rows with K above 2048."""
    for M, N, K, fmt in ((65, 4096, 2048, I8), (187, 2048, 6144, FP8), (431, 2048, 2048, I8),
                         (698, 2768, 1536, I8)):
        p = qlinear.plan(M, N, K, fmt)
        assert p.staged == 3 and (p.channels, p.tokens) in TILES
        assert -(-N // p.channels) * -(-M // p.tokens) <= 256
    assert qlinear.plan(1024, 1024, 1024, I8).kind == qlinear.KIND_TILED
    assert qlinear.plan(431, 12288, 2048, I8).kind == qlinear.KIND_TILED
    assert qlinear.plan(187, 2048, 2048, I8, 128, 128).kind == qlinear.KIND_TILED
    assert qlinear.plan(64, 4096, 2048, I8).staged == 2
    assert qlinear.plan(64, 12288, 2048, I8).staged == 1
    assert qlinear.plan(32, 2048, 6144, I8).staged == 1
    assert qlinear.plan(33, 2048, 6144, I8).staged == 3


def test_sliced_path_validation():
    L = qlinear.load()
    import ctypes
    fake = 1 << 20

    def call(p, M=64, N=64, K=256, ig=0, wg=0):
        return L.qlin_gemm(ctypes.byref(p.to_c()), fake, fake, fake, fake, fake, M, N, K, I8, BF16,
                           ig, wg, None, 0, None)
    assert call(qlinear.Path(qlinear.KIND_SKINNY, 80, 64, 1, 8, 3)) == -4  # no such tile
    assert call(qlinear.Path(qlinear.KIND_SKINNY, 32, 32, 2, 8, 3)) == -4  # no grid split
    assert call(qlinear.Path(qlinear.KIND_SKINNY, 32, 32, 1, 4, 3)) == -4
    assert call(path(32, 32), ig=128, wg=128) == -4                        # per-channel only
    assert call(path(16, 16), M=1 << 30, N=1 << 30, K=16) == -4            # grid limit
    assert call(qlinear.Path(qlinear.KIND_SKINNY, 32, 32, 1, 8, 4)) == -4


def test_decode_plan_with_room_for_both_operands():
    """33 to 64 rows: K-sliced only where the decode kernel cannot stage the
    activation tile beside its weight slab."""
    assert qlinear.plan(41, 896, 3584, FP8).staged == 2
    assert qlinear.plan(57, 2048, 6144, FP8).staged == 3


def test_short_k_gives_way():
    """Shapes whose K-sliced tile is large for a short K, and which 128x64 macro
    tiles cover in one round, take the macro tile."""
    for M, N, K in ((204, 6912, 1408), (499, 4096, 1024), (900, 2048, 2048), (361, 4576, 1024),
                    (517, 2688, 896), (175, 10848, 384), (192, 8320, 1408), (517, 1856, 384),
                    (191, 5536, 640)):
        p = qlinear.plan(M, N, K, FP8)
        assert (p.kind, p.channels, p.tokens) == (qlinear.KIND_TILED, 128, 64), (M, N, K, p)
    for M, N, K in ((555, 2784, 5120), (900, 2048, 6144), (700, 2048, 2048), (187, 12288, 2048),
                    (191, 5536, 768), (340, 2912, 768), (187, 2048, 128)):
        assert qlinear.plan(M, N, K, FP8).staged == 3, (M, N, K)


def test_sliced_plan_operand_range():
    """A K-sliced tile's rows of an operand stay below 2 GiB (32-bit buffer
    ranges): FP8 shapes with a K past that keep the plans they had, which
    address rows by 64 bits (33-64 rows), and a saved path is refused."""
    for K in (1 << 25, (1 << 27) + 16, 1 << 30):
        for M, N in ((64, 4096), (64, 16), (33, 1024), (187, 2048)):
            p = qlinear.plan(M, N, K, FP8)
            assert p.staged != 3 or max(p.channels, p.tokens) * K < 1 << 31, (M, N, K, p)
    assert qlinear.plan(64, 4096, 1 << 27, FP8).staged == 0
    assert qlinear.plan(64, 4096, 1 << 25, FP8).staged == 3  # 32 x 32 rows, 1 GiB
    L = qlinear.load()
    import ctypes
    fake = 1 << 20
    assert L.qlin_gemm(ctypes.byref(path(32, 32).to_c()), fake, fake, fake, fake, fake, 64, 64,
                       1 << 26, FP8, BF16, 0, 0, None, 0, None) == -4
