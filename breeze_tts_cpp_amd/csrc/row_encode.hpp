// Row encoders shared by the row quantizer and the fused quantizing producers
// (residual + RMSNorm, gated activation, LayerNorm and pointwise epilogue ->
// quant), with their 8-column load/store helpers: a 256-thread
// workgroup holds a row in registers, lane t owning the 8 columns
// (it * 256 + t) * 8 .. +8 of each 2048-column chunk `it`, and encodes it per
// token, per token after the H128 rotation, or per K group (optionally
// rotated) exactly as the reference quant_device helpers do
// (ops/kernels/quant/quant_device.cuh:63-195).
#pragma once
#include "qlin_device.hpp"

#include <type_traits>

namespace qlin {
namespace {

constexpr int kThreads = 256;
constexpr int kChunk = kThreads * 8;  // columns covered by one pass of the block

// Eight 16-bit values of a row as stored, zeros past its end. The vector form
// loads without a branch (lanes past the end read the row's start and drop
// it), and callers load all operands of a row before they use one: a load
// under a lane's `if`, or after another operand's arithmetic, waits for the
// one before it, a memory latency each (residual RMSNorm of one row of 2048:
// 2.78 -> 2.55 us, of 4096 rows 15.8 -> 13.9; gated, width 6144, 32 rows 3.9 ->
// 3.8, 4096 rows 34.7 -> 33.6).
template <bool Vec>
__device__ __forceinline__ uint4 load_raw8(const uint16_t *row, int column, int cols) {
    if constexpr (Vec) {
        const bool in = column < cols;
        const uint4 raw = *reinterpret_cast<const uint4 *>(row + (in ? column : 0));
        return uint4{in ? raw.x : 0, in ? raw.y : 0, in ? raw.z : 0, in ? raw.w : 0};
    } else {
        uint32_t e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = column + i < cols ? row[column + i] : 0;
        return uint4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16),
                     e[6] | (e[7] << 16)};
    }
}

template <class Tin> __device__ __forceinline__ void widen8(const uint4 &raw, float (&v)[8]) {
    const uint32_t words[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = to_float(uint16_t(words[i] & 0xffffu), Tin{});
        v[2 * i + 1] = to_float(uint16_t(words[i] >> 16), Tin{});
    }
}

template <class Tin, bool Vec>
__device__ __forceinline__ void load8(const uint16_t *row, int column, int cols, float (&v)[8]) {
    widen8<Tin>(load_raw8<Vec>(row, column, cols), v);
}

template <int Fmt, bool Vec>
__device__ __forceinline__ void store8(uint8_t *row, int column, int cols, const float (&v)[8],
                                       float inverse) {
    if constexpr (Vec) {
        auto codes = [&](int i) {
            const float a = v[i] * inverse, b = v[i + 1] * inverse, c = v[i + 2] * inverse,
                        d = v[i + 3] * inverse;
            return Fmt == FP8 ? encode_fp8x4(a, b, c, d) : encode_i8x4(a, b, c, d);
        };
        const uint32_t lo = codes(0), hi = codes(4);
        if (column < cols) *reinterpret_cast<uint2 *>(row + column) = uint2{lo, hi};
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (column + i < cols) row[column + i] = uint8_t(encode<Fmt>(v[i] * inverse));
    }
}

// 16-bit values of 8 columns [column, column+8) stored (rounded to T).
template <class T, bool Vec>
__device__ __forceinline__ void store16x8(uint16_t *row, int column, int cols, const float (&v)[8]) {
    if constexpr (Vec) {
        if (column < cols) {
            uint4 packed;
            packed.x = pack2(v[0], v[1], T{});
            packed.y = pack2(v[2], v[3], T{});
            packed.z = pack2(v[4], v[5], T{});
            packed.w = pack2(v[6], v[7], T{});
            *reinterpret_cast<uint4 *>(row + column) = packed;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (column + i < cols) row[column + i] = from_float(v[i], T{});
    }
}

// Correctly rounded 1/sqrt(a) in fp32: the hardware's fp64 estimate with two
// Newton steps (equal to float(1.0 / sqrt(double(a))), whose fp64 root and
// division take three times the instructions, for every a); zeros, infinity,
// negative values and NaN take the estimate itself.
__device__ __forceinline__ float rsqrt_rn(float a) {
    const double x = a;
    const double estimate = __builtin_amdgcn_rsq(x);
    double y = estimate;
#pragma unroll
    for (int i = 0; i < 2; ++i) y = __builtin_fma(0.5 * y, __builtin_fma(-x * y, y, 1.0), y);
    return float(a > 0.f && a < __builtin_inff() ? y : estimate);
}

// H128 rotation of the 8 columns [column, column+8) held by this lane; the 16
// lanes sharing (lane >> 4) hold one aligned 128-column block. A rotated row
// is bound by these instructions (12288 x 2048, INT8, groups of 128: 18.6 us
// unrotated; rotated 29.5 -> 25.7 with 24-bit hash products, lane exchanges
// folded into their additions and packed codes; two or four rows a thread,
// which share the signs, were no faster).
__device__ __forceinline__ void rotate8(float (&v)[8], int column) {
    uint32_t sign[8];
    rotation_signs(column, sign);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = __uint_as_float(__float_as_uint(v[i]) ^ sign[i]);
#pragma unroll
    for (int span = 1; span < 8; span *= 2) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (!(i & span)) {
                float a = v[i], b = v[i | span];
                v[i] = a + b;
                v[i | span] = a - b;
            }
    }
    const int lane = threadIdx.x & 63;
    // The partner's value plus or minus the lane's own: the product by +-1 is exact.
    auto stage = [&](auto span_) {
        constexpr int span = decltype(span_)::value;
        const float own = (lane & span) ? -1.f : 1.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = lane_xor<span>(v[i]) + own * v[i];
    };
    stage(std::integral_constant<int, 1>{});
    stage(std::integral_constant<int, 2>{});
    stage(std::integral_constant<int, 4>{});
    stage(std::integral_constant<int, 8>{});
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] *= 0.08838834764831845f;
}

// Max over the NT threads of the workgroup.
template <int NT = kThreads> __device__ __forceinline__ float block_max(float v) {
    __shared__ float partial[NT / 64];
    v = group_max<64>(v);
    if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = partial[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) r = fmaxf(r, partial[w]);
    return r;
}

// One lane's 8 columns [column, column+8) of a K-group encoding (group 32,
// 64 or 128, so the group spans group/8 adjacent lanes): the group's amax by
// lane shuffles, its scale written by the group's first lane, the codes.
template <int Fmt, bool Vec>
__device__ __forceinline__ void encode_group8(const float (&v)[8], uint8_t *__restrict__ dst,
                                              float *__restrict__ scales, int row, int rows,
                                              int cols, int column, int group) {
    const int lanes = group / 8;
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
    if (lanes > 1) amax = fmaxf(amax, lane_xor<1>(amax));
    if (lanes > 2) amax = fmaxf(amax, lane_xor<2>(amax));
    if (lanes > 4) amax = fmaxf(amax, lane_xor<4>(amax));
    if (lanes > 8) amax = fmaxf(amax, lane_xor<8>(amax));
    const float step = quant_scale<Fmt>(amax);
    if (column < cols && (column % group) == 0) scales[size_t(column / group) * rows + row] = step;
    store8<Fmt, Vec>(dst, column, cols, v, 1.f / step);
}

// Encode a row held in registers by NT threads (v[it][i] = column
// (it*NT + t)*8 + i; columns past `cols` hold 0): optional H128 rotation
// (`rot`), then per-(row, group) scales ([ceil(cols/group), rows]) for group
// 32, 64 or 128, else (group 0) one per-token scale ([rows]). The reference's
// rotated_quantize / encode_group / token paths (quant_device.cuh:63-88,
// 145-195, row_quantize.cu:24-165). Groups and rotation blocks stay inside one
// wave for any NT (multiples of 64). `group` and `rot` are uniform across the
// workgroup, so their branches never diverge.
template <int Fmt, int Items, bool Vec, int NT = kThreads>
__device__ __forceinline__ void encode_row(float (&v)[Items][8], uint8_t *__restrict__ q,
                                           float *__restrict__ scales, int row, int rows,
                                           int cols, int group, int rot) {
    uint8_t *dst = q + size_t(row) * cols;
    if (rot) {
#pragma unroll
        for (int it = 0; it < Items; ++it) rotate8(v[it], (it * NT + threadIdx.x) * 8);
    }
    if (group) {
#pragma unroll
        for (int it = 0; it < Items; ++it)
            encode_group8<Fmt, Vec>(v[it], dst, scales, row, rows, cols,
                                    (it * NT + threadIdx.x) * 8, group);
    } else {
        float amax = 0.f;
#pragma unroll
        for (int it = 0; it < Items; ++it)
#pragma unroll
            for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[it][i]));
        const float step = quant_scale<Fmt>(block_max<NT>(amax));
        const float inverse = 1.f / step;
        if (threadIdx.x == 0) scales[row] = step;
#pragma unroll
        for (int it = 0; it < Items; ++it)
            store8<Fmt, Vec>(dst, (it * NT + threadIdx.x) * 8, cols, v[it], inverse);
    }
}

}  // namespace
}  // namespace qlin
