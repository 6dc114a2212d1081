// K-sliced quantized GEMM for gfx950: token counts between the decode and the
// prefill regime (65 to about 1000 tokens; from 33 with K above 2048), per-channel
// scales.
//
// Same contract as the other families: y = D((acc * sx) * sw), the optional
// finish, row-major or packed weights.
//
// What bounds these shapes: with 65 to a few hundred tokens the macro tiles of
// the prefill kernel leave most CUs without work (o_proj at M = 187: 48 tiles
// of 128x64), and each CU that has one walks all of K through LDS fragments
// that several waves read again (a 32x32 wave of a 128x64 tile reads 64 KB of
// LDS per 24 KB stage). So the macro tile here is chosen small enough that
// one round of workgroups covers the 256 CUs, and the eight waves of a
// workgroup split K instead of the tile: wave q accumulates the whole BN x BM
// tile over its own K slice (KS = 8) and reads each staged byte from LDS
// once. Larger tiles (64x96 and up), whose operands would not fit the LDS
// eight times, run two slices of four waves (KS = 2, 2 x 2 waves) that share
// a ring per slice. The partial tiles are summed through LDS in ascending
// slice order (exact for INT8). L2 -> LDS runs at 128 B/ns per CU when every
// line hits L2; these tiles reach about 70, the rest is memory-side latency
// of a ring that holds at most 160 KB per CU.
//
// Measured (INT8, weights from HBM, us, prefill tile -> this kernel): M = 187
// qkv 9.9 -> 7.2, o_proj 9.1 -> 5.1, gate_up 17.0 -> 13.0, down 21.7 -> 9.9;
// M = 431 o_proj 8.9 -> 7.1, down 20.7 -> 14.9. FP8 within 3% of INT8. A whole
// decoder layer among its other launches: M = 187 INT8 80 -> 53 us, M = 431
// FP8 84.7 -> 75.5, M = 57 FP8 (down only) 43.0 -> 42.0.
#include "qlin_device.hpp"
#include "qlin_internal.hpp"

#include <algorithm>
#include <type_traits>

// Built per format, without and with the fused finish (see the Makefile); the
// build without QLIN_SLICED_PART holds the dispatcher.
#ifndef QLIN_FIN
#define QLIN_FIN 0
#endif

namespace qlin {
#ifdef QLIN_SLICED_PART
namespace {

constexpr bool kFin = QLIN_FIN;
constexpr int kRing = int(kLdsBytes);

// KS slices of K, WN x WM waves per slice, NF weight and MT token fragments of
// 16 rows per wave, S stages of 128 K bytes per slice's LDS ring. `steps`
// stages per slice; slices past K are short or empty and add zeros. WAUX: the
// weight DMA's cache policy. `turned` (INT8, whose sums are exact in any
// order): each workgroup walks its slices' stages from another start. Rows of
// a power-of-two pitch put one K column of all rows on few L2 channels, and
// every workgroup begins at the same columns. Tiles of 32 and more channels
// gain 5-10% with slices of five or more stages (down at M = 187 10.3 -> 9.5 us,
// 431 x 1536 x 4352 10.4 -> 8.5); 16-channel tiles lose 5-20% (down at M = 57 7.7 ->
// 8.5) and slices of four stages 2-5% (499 x 1024 x 4096 6.5 -> 7.0). FP8 walks K
// in order: a token's fp32 sum must not depend on the tile its row falls in,
// and starts taken from the weight tile alone gain nothing.
template <int Fmt, int KS, int WN, int WM, int NF, int MT, int S, int WAUX>
__global__ __launch_bounds__(64 * KS * WN * WM, 1) void sliced_gemm(
    const uint8_t *__restrict__ x, const float *__restrict__ sx, const uint8_t *__restrict__ w,
    const float *__restrict__ sw, void *__restrict__ y, int M, int N, int K, int tiles_m,
    int tiles_n, int steps, int packed, const uint16_t *__restrict__ bias, int act, int out_f16, int turned) {
    using Mma = TileMma<Fmt>;
    using Acc = typename Mma::Acc;
    constexpr int NWS = WN * WM, W = KS * NWS;
    constexpr int BN = 16 * NF * WN, BM = 16 * MT * WM, BK = 128;
    constexpr int STAGE = (BN + BM) * BK, WI = BN / 8 / NWS, INSTS = WI + BM / 8 / NWS;
    static_assert(BN / 8 % NWS == 0 && BM / 8 % NWS == 0, "whole DMA instructions per wave");
    static_assert(NWS == 1 || (NWS % 2 == 0 && S > 1), "a shared ring refills behind the readers");
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    const int b = xcd_major(blockIdx.x, tiles_m * tiles_n);
    const int n_base = b / tiles_m * BN, m_base = b % tiles_m * BM;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row16 = lane & 15, quad = lane >> 4;

    // Epilogue scales, loaded ahead of everything else.
    constexpr int PITCH = BN + 4;  // 32-bit values per row of a partial tile
    static_assert(KS * BM * PITCH * 4 <= kRing, "the slices' partial tiles fit the LDS");
    // Threads own four channels each and every kRows-th row, so a thread's
    // weight scales are the same for all its rows.
    constexpr int kRows = 64 * W / (BN / 4), kMaxU = (BM + kRows - 1) / kRows;
    const int nl = tid % (BN / 4) * 4, r0 = tid / (BN / 4);
    float pre_x[kMaxU], pre_w[4];
#pragma unroll
    for (int u = 0; u < kMaxU; ++u) pre_x[u] = sx[min(m_base + r0 + u * kRows, M - 1)];
#pragma unroll
    for (int r = 0; r < 4; ++r) pre_w[r] = sw[min(n_base + nl, N - 4) + r];

    const int ks = wave / NWS, ws = wave % NWS, wn = ws % WN, wm = ws / WN;
    const int k_begin = ks * steps * BK;
    const int count = NWS > 1 ? steps : max(0, min(steps, (K - k_begin + BK - 1) / BK));
    const int turn = Fmt == I8 && turned && count > 0 ? b * 3 % count : 0;
    const int tiles_k = (K + 63) / 64;
    const int rows_w = min(BN, N - n_base), rows_x = min(BM, M - m_base);
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(packed ? w + size_t(n_base / 16) * tiles_k * 1024
                                     : w + size_t(n_base) * K),
        0, packed ? rows_w / 16 * tiles_k * 1024 : rows_w * K, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(x + size_t(m_base) * K), 0, rows_x * K, 0x00020000);
    // One DMA instruction fills 8 stage rows of 128 bytes in lane order. Row
    // r of the tile keeps 16-byte chunk c at c ^ ((r >> 1) & 7) (fragment
    // reads on distinct banks): lane l of the instruction at row 8i takes
    // source chunk (l % 8) ^ (4 (i & 1) + l / 16). Chunk 0 is for even i (with
    // a shared ring, for the one parity of all the wave's instructions).
    const int lane_row = lane >> 3;
    const int chunk0 = (lane & 7) ^ (lane_row >> 1) ^ (NWS > 1 ? 4 * (ws & 1) : 0), chunk1 = chunk0 ^ 4;
    const uint32_t voff0 = uint32_t(lane_row) * uint32_t(K) + uint32_t(chunk0 * 16);
    const uint32_t voff1 = uint32_t(lane_row) * uint32_t(K) + uint32_t(chunk1 * 16);
    const uint32_t woff0 = packed ? uint32_t((chunk0 / 4) * 1024 + (chunk0 % 4) * 256 + lane_row * 16) : voff0;
    const uint32_t woff1 = packed ? uint32_t((chunk1 / 4) * 1024 + (chunk1 % 4) * 256 + lane_row * 16) : voff1;
    const uint32_t wrow16 = packed ? uint32_t(tiles_k) * 1024u : uint32_t(K) * 16u;
    const uint32_t wrow8 = packed ? 128u : uint32_t(K) * 8u;
    const uint32_t wk = packed ? 16u : 1u;  // bytes per K byte of a stage step
    uint8_t *ring = lds + ks * S * STAGE;
    // Buffer descriptors cover the tile's valid rows, so rows past the matrix
    // and (through an out-of-range offset) chunks past K arrive as zeros. `aim`
    // sets the offsets of one stage's DMA, `dma` issues its instructions.
    uint8_t *dma_base = ring;
    uint32_t dx0 = 0, dx1 = 0, dw0 = 0, dw1 = 0, dws = 0;
    auto aim = [&](int st, int slot) {
        dma_base = ring + slot * STAGE;
        const uint32_t k0 = uint32_t(k_begin + (st + turn < count ? st + turn : st + turn - count) * BK);
        const bool in0 = int(k0) + chunk0 * 16 < K, in1 = int(k0) + chunk1 * 16 < K;
        dx0 = in0 ? voff0 + k0 : 0x80000000u, dx1 = in1 ? voff1 + k0 : 0x80000000u;
        dw0 = in0 ? woff0 : 0x80000000u, dw1 = in1 ? woff1 : 0x80000000u;
        dws = k0 * wk;
    };
    auto dma = [&](auto i_) {
        constexpr int i = decltype(i_)::value;
        if constexpr (NWS == 1) {
            if constexpr (i < WI)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (lds_ptr_t)(dma_base + i * 1024), 16,
                                                         i & 1 ? dw1 : dw0,
                                                         uint32_t(i / 2) * wrow16 + (i & 1 ? wrow8 : 0u) + dws,
                                                         0, WAUX);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_x, (lds_ptr_t)(dma_base + i * 1024),
                                                         16, i & 1 ? dx1 : dx0,
                                                         uint32_t(i - WI) * 8u * uint32_t(K), 0, 0);
        } else {
            constexpr int j = i < WI ? i : i - WI;
            const uint32_t g = uint32_t(j * NWS + ws);  // 8-row group of the operand
            lds_ptr_t dst = (lds_ptr_t)(dma_base + ((i < WI ? 0 : BN / 8) + j * NWS + ws) * 1024);
            if constexpr (i < WI)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, dst, 16, dw0,
                                                         g / 2 * wrow16 + (ws & 1 ? wrow8 : 0u) + dws, 0, 0);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_x, dst, 16, dx0, g * 8u * uint32_t(K), 0, 0);
        }
    };
    // Wait for a stage with at most `newer` later ones outstanding.
    auto wait_stage = [&](int newer) {
        if (newer >= S - 1) wait_vmcnt<INSTS * (S - 1)>();
        else if (S >= 2 && newer == S - 2) wait_vmcnt<INSTS * (S >= 2 ? S - 2 : 0)>();
        else if (S > 3 && newer == S - 3) wait_vmcnt<INSTS * (S > 3 ? S - 3 : 0)>();
        else wait_vmcnt<0>();
    };
    Acc acc[NF][MT];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[f][t] = Acc{0, 0, 0, 0};

    const int sw7 = (row16 >> 1) & 7;
    const int c0 = (quad ^ sw7) * 16, c1 = ((4 + quad) ^ sw7) * 16;
    auto read = [&](int slot, i32x8 (&a)[NF], i32x8 (&bb)[MT]) {
        const uint8_t *p = ring + slot * STAGE + row16 * BK;
        auto frag = [&](const uint8_t *q) {
            const i32x4 lo = *reinterpret_cast<const i32x4 *>(q + c0);
            const i32x4 hi = *reinterpret_cast<const i32x4 *>(q + c1);
            return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        };
#pragma unroll
        for (int t = 0; t < MT; ++t) bb[t] = frag(p + (BN + (wm * MT + t) * 16) * BK);
#pragma unroll
        for (int f = 0; f < NF; ++f) a[f] = frag(p + (wn * NF + f) * 16 * BK);
    };
    // Stage s's MFMAs, one (weight, token) tile at a time, with the next
    // DMA's instructions spread between them.
    auto mma = [&](auto dma_, const i32x8 (&a)[NF], const i32x8 (&bb)[MT]) {
        constexpr bool kDma = decltype(dma_)::value;
        static_for<0, NF * MT>([&](auto j_) {
            constexpr int j = decltype(j_)::value, f = j / MT, t = j % MT;
            Mma::run(acc[f][t], a[f], bb[t]);
            if constexpr (kDma) {
                static_for<j * INSTS / (NF * MT), (j + 1) * INSTS / (NF * MT)>(dma);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    };
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < count) {
            aim(s, s);
            static_for<0, INSTS>(dma);
        }
    if constexpr (S == 1) {
        // One stage in LDS, one set of fragments in registers (a second set
        // spills): the next stage's DMA runs under this stage's MFMAs, and
        // the other waves' work hides its latency.
        i32x8 fa[NF], fb[MT];
        for (int s = 0; s < count; ++s) {
            wait_vmcnt<0>();
            __builtin_amdgcn_sched_barrier(0);
            read(0, fa, fb);
            wait_lds_reads();
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < count) {
                aim(s + 1, 0);
                mma(std::true_type{}, fa, fb);
            } else {
                mma(std::false_type{}, fa, fb);
            }
        }
    } else {
        int slot = 0;  // of the stage whose fragments are in registers
        // Step s: stage s's fragments have arrived, so its slot is free for
        // stage s + S (a shared ring: once every wave of the slice has them,
        // after the barrier, which also makes stage s + 1 visible). Where the
        // ring is deeper than two or shared, the next fragments are read
        // under this stage's MFMAs; a private two-stage ring reads them after
        // the MFMAs, giving stage s + 1's DMA that time to land.
        auto step = [&](int s, const i32x8 (&a)[NF], const i32x8 (&bb)[MT], i32x8 (&na)[NF],
                        i32x8 (&nb)[MT]) {
            wait_lds_reads();
            __builtin_amdgcn_sched_barrier(0);
            const int next = slot + 1 == S ? 0 : slot + 1;
            if constexpr (S >= 3 || NWS > 1) {
                if (s + 1 < count) wait_stage(min(count - 2 - s, S - 2));
                if constexpr (NWS > 1) __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                read(next, na, nb);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (s + S < count) {
                aim(s + S, slot);
                mma(std::true_type{}, a, bb);
            } else {
                mma(std::false_type{}, a, bb);
            }
            slot = next;
            if constexpr (S == 2 && NWS == 1) {
                if (s + 1 < count) wait_stage(count - 2 - s);
                __builtin_amdgcn_sched_barrier(0);
                read(slot, na, nb);
            }
        };
        i32x8 a0[NF], b0[MT], a1[NF], b1[MT];
        if (count > 0) {
            wait_stage(count - 1);
            if constexpr (NWS > 1) __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            read(0, a0, b0);
            int s = 0;
            for (; s + 1 < count; s += 2) {
                step(s, a0, b0, a1, b1);
                step(s + 1, a1, b1, a0, b0);
            }
            if (s < count) step(s, a0, b0, a1, b1);
        }
    }

    // Sum the slices' partial tiles through LDS (all DMA has landed and been
    // read), ascending slices; then scales, finish and 8-byte stores, consecutive
    // threads on consecutive channels.
    using Red = std::conditional_t<Fmt == I8, int, float>;
    typedef Red Red4 __attribute__((ext_vector_type(4)));
    Red *red = reinterpret_cast<Red *>(lds);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            Red4 v;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = acc[f][t][r];
            *reinterpret_cast<Red4 *>(red + (ks * BM + (wm * MT + t) * 16 + row16) * PITCH + (wn * NF + f) * 16 + quad * 4) = v;
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kMaxU; ++u) {
        const int ml = r0 + u * kRows, m = m_base + ml, n = n_base + nl;
        if (r0 >= kRows || ml >= BM || m >= M || n >= N) continue;
        Red4 sum = {0, 0, 0, 0};
#pragma unroll
        for (int q = 0; q < KS; ++q)
            sum += *reinterpret_cast<const Red4 *>(red + (q * BM + ml) * PITCH + nl);
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float s = float(sum[r]) * pre_x[u];
            v[r] = s * pre_w[r];
        }
        uint2 out;
        if (out_f16) {
            if constexpr (kFin) finish4<f16_t>(v, bias, n, N - 1, act);
            out.x = pack2(v[0], v[1], f16_t{});
            out.y = pack2(v[2], v[3], f16_t{});
        } else {
            if constexpr (kFin) finish4<bf16_t>(v, bias, n, N - 1, act);
            out.x = pack2(v[0], v[1], bf16_t{});
            out.y = pack2(v[2], v[3], bf16_t{});
        }
        *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(y) + size_t(m) * N + n) = out;
    }
}

template <int Fmt, int KS, int WN, int WM, int NF, int MT>
int launch(const GemmArgs &a, hipStream_t stream) {
    constexpr int W = KS * WN * WM, BN = 16 * NF * WN, BM = 16 * MT * WM;
    // As many stages as the LDS holds; more than four measured no faster.
    constexpr int S = std::min(4, kRing / (KS * (BN + BM) * 128));
    constexpr size_t ring = size_t(KS) * S * (BN + BM) * 128;
    constexpr size_t lds = std::max(ring, size_t(KS) * BM * (BN + 4) * 4);
    static_assert(lds <= size_t(kRing), "LDS");
    // 16-channel tiles carry the weight DMA's nt bit, as the decode kernel: they
    // serve decode batches, where one token tile, seldom more, reads the weights
    // (down at M = 57 7.8 -> 7.7 us). Wider tiles' weights are read again by the
    // other token tiles (o_proj at M = 187 5.2 us against 5.5 with the bit).
    constexpr int WAUX = BN == 16 ? 2 : 0;
    const int tiles_n = (a.N + BN - 1) / BN, tiles_m = (a.M + BM - 1) / BM;
    const int steps = ((a.K + 127) / 128 + KS - 1) / KS;
    hipLaunchKernelGGL((sliced_gemm<Fmt, KS, WN, WM, NF, MT, S, WAUX>),
                       dim3(unsigned(tiles_n * tiles_m)), dim3(64 * W), lds, stream, a.x, a.sx, a.w,
                       a.sw, a.y, a.M, a.N, a.K, tiles_m, tiles_n, steps, a.packed, a.bias, a.act,
                       int(a.out_type == F16), int(KS == 8 && BN > 16 && steps >= 5));
    return 0;
}

}  // namespace

// One kernel per tile of kSlicedTiles.
int QLIN_SLICED_PART(const GemmArgs &a, const GemmPath &p, hipStream_t s) {
    constexpr int F = QLIN_SLICED_FMT;
    switch (p.channels * 256 + p.tokens) {
#define QLIN_SLICE8(NF, MT) \
    case 16 * NF * 256 + 16 * MT: return launch<F, 8, 1, 1, NF, MT>(a, s);
#define QLIN_SLICE2(NF, MT) \
    case 32 * NF * 256 + 32 * MT: return launch<F, 2, 2, 2, NF, MT>(a, s);
        QLIN_SLICE8(1, 1) QLIN_SLICE8(1, 2) QLIN_SLICE8(1, 3) QLIN_SLICE8(1, 4) QLIN_SLICE8(2, 1)
        QLIN_SLICE8(2, 2) QLIN_SLICE8(2, 3) QLIN_SLICE8(2, 4) QLIN_SLICE8(2, 5) QLIN_SLICE8(3, 2)
        QLIN_SLICE8(3, 3) QLIN_SLICE8(3, 4) QLIN_SLICE8(3, 5) QLIN_SLICE8(3, 6) QLIN_SLICE8(4, 2)
        QLIN_SLICE8(4, 3) QLIN_SLICE8(4, 4) QLIN_SLICE2(2, 3) QLIN_SLICE2(2, 4) QLIN_SLICE2(3, 2)
        QLIN_SLICE2(3, 3)
#undef QLIN_SLICE8
#undef QLIN_SLICE2
    }
    return -4;
}
#else
int launch_sliced_i8(const GemmArgs &, const GemmPath &, hipStream_t);
int launch_sliced_i8_fin(const GemmArgs &, const GemmPath &, hipStream_t);
int launch_sliced_fp8(const GemmArgs &, const GemmPath &, hipStream_t);
int launch_sliced_fp8_fin(const GemmArgs &, const GemmPath &, hipStream_t);
int launch_sliced(const GemmArgs &a, const GemmPath &p, hipStream_t s) {
    const bool fin = a.bias || a.act;
    if (a.fmt == I8) return fin ? launch_sliced_i8_fin(a, p, s) : launch_sliced_i8(a, p, s);
    return fin ? launch_sliced_fp8_fin(a, p, s) : launch_sliced_fp8(a, p, s);
}
#endif

}  // namespace qlin
