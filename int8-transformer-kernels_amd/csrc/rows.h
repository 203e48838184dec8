// rows.h — vectorised per-row int8 quantization (internal header).
//
// The per-token quantizers (quant.hip) and the producer-fused ones
// (producer.hip) all reduce one row to its absmax and then quantize it.  Rows
// are short (a head of 64 or 128 elements, a model row of 1–8K), so one lane
// per element leaves most of a wave's load slots empty.  Here each lane owns
// 16-byte chunks of a row instead: a row of C chunks is spread over L lanes (C
// rounded up to a power of two, at most 64) with ceil(C / L) chunks per lane,
// so a wave holds 64 / L rows, loads are 16 bytes per lane and the row
// reductions are shuffles inside an aligned lane group.  Where C is not L times
// a chunk count that has an instance, the slots past C repeat the row's last
// chunk (PAD): the same loads, maxima and stored bytes again, and no branch.
// Rows that are not whole chunks, or of more than 1024, keep the
// one-element-per-lane kernels.
#pragma once

#include <type_traits>

#include "int8k_common.h"

namespace int8k {

// Elements of a dtype per 16-byte chunk.
template <int DT>
struct Vec {
    static constexpr int W = DT == INT8K_DTYPE_F32 ? 4 : 8;
};

// At most this many chunks per lane (a row of 64 * 16 chunks = 16 KiB).
constexpr int kMaxChunksPerLane = 16;

// How a row of `cols` elements maps onto lanes: cpr chunks on 1 << lg lanes, at
// most nc each.
struct RowShape {
    int lg = 0, nc = 0, cpr = 0;
    bool ok = false;
};

inline RowShape row_shape(int cols, int dtype) {
    RowShape r;
    const int w = dtype == INT8K_DTYPE_F32 ? 4 : 8;
    if (cols <= 0 || cols % w) return r;
    r.cpr = cols / w;
    while (r.lg < 6 && (1 << r.lg) < r.cpr) ++r.lg;
    r.nc = (r.cpr + (1 << r.lg) - 1) >> r.lg;
    r.ok = r.nc <= kMaxChunksPerLane;
    return r;
}

// Calls f(std::integral_constant<int, NC>, PAD as a bool constant) with the
// smallest instance of at least sh.nc chunks per lane; PAD false when the row
// fills every slot.  3, 6 and 12 beside the powers of two keep the repeated
// chunks to a third of the row.
template <typename F>
inline void with_chunks(const RowShape& sh, F&& f) {
    auto go = [&](auto nc, auto pow2) {
        if constexpr (pow2.value) {
            if (sh.cpr == (nc.value << sh.lg)) {
                f(nc, std::false_type{});
                return;
            }
        }
        f(nc, std::true_type{});
    };
    using T = std::true_type;
    using N = std::false_type;
    if (sh.nc <= 1) go(std::integral_constant<int, 1>{}, T{});
    else if (sh.nc <= 2) go(std::integral_constant<int, 2>{}, T{});
    else if (sh.nc <= 3) go(std::integral_constant<int, 3>{}, N{});
    else if (sh.nc <= 4) go(std::integral_constant<int, 4>{}, T{});
    else if (sh.nc <= 6) go(std::integral_constant<int, 6>{}, N{});
    else if (sh.nc <= 8) go(std::integral_constant<int, 8>{}, T{});
    else if (sh.nc <= 12) go(std::integral_constant<int, 12>{}, N{});
    else go(std::integral_constant<int, 16>{}, T{});
}

// Chunk of slot i of the lane whose first chunk is c0, in a row of cpr chunks.
template <bool PAD>
__device__ __forceinline__ uint32_t slot_chunk(int i, int lg, uint32_t c0, uint32_t cpr) {
    const uint32_t c = ((uint32_t)i << lg) + c0;
    return PAD ? min(c, cpr - 1) : c;
}

// Calls f(std::integral_constant<int, DT>) for a dtype code.
template <typename F>
inline void with_dtype(int dtype, F&& f) {
    switch (dtype) {
        case INT8K_DTYPE_F16: f(std::integral_constant<int, INT8K_DTYPE_F16>{}); break;
        case INT8K_DTYPE_BF16: f(std::integral_constant<int, INT8K_DTYPE_BF16>{}); break;
        default: f(std::integral_constant<int, INT8K_DTYPE_F32>{});
    }
}

// Makes the compiler treat a chunk as rewritten, so values unpacked from it
// before this point are not kept live across it (they are cheaper to unpack
// again than to hold in 2 W registers per chunk).
__device__ __forceinline__ void reload_barrier(uint4& w) {
    asm volatile("" : "+v"(w.x), "+v"(w.y), "+v"(w.z), "+v"(w.w));
}

template <int DT>
__device__ __forceinline__ void unpack_chunk(const uint4& w, float (&v)[Vec<DT>::W]) {
    const uint32_t d[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (DT == INT8K_DTYPE_F32) {
            v[i] = __uint_as_float(d[i]);
        } else if constexpr (DT == INT8K_DTYPE_F16) {
            v[2 * i] = __half2float(__ushort_as_half((unsigned short)(d[i] & 0xffffu)));
            v[2 * i + 1] = __half2float(__ushort_as_half((unsigned short)(d[i] >> 16)));
        } else {
            v[2 * i] = __uint_as_float(d[i] << 16);
            v[2 * i + 1] = __uint_as_float(d[i] & 0xffff0000u);
        }
    }
}

// Reduction over the aligned group of 1 << lg lanes that holds one row; every
// lane of the group gets it.  On the VALU: DPP inside a 16-lane row (after the
// xor 1 and xor 2 steps a quad's lanes agree, so the mirrors pair whole quads and
// halves as xor 4 and xor 8 would), then the row and half swaps.
template <typename Op>
__device__ __forceinline__ float row_reduce(float v, int lg, Op op) {
    auto f = [](int x) { return __int_as_float(x); };
    auto i = [](float x) { return __float_as_int(x); };
    if (lg > 0) v = op(v, f(dpp_xor1(i(v))));
    if (lg > 1) v = op(v, f(dpp_xor2(i(v))));
    if (lg > 2) v = op(v, f(dpp_half_mirror(i(v))));
    if (lg > 3) v = op(v, f(dpp_row_mirror(i(v))));
    if (lg > 4) {
        const auto r = __builtin_amdgcn_permlane16_swap(i(v), i(v), false, false);
        v = op(f(r[0]), f(r[1]));
    }
    if (lg > 5) {
        const auto r = __builtin_amdgcn_permlane32_swap(i(v), i(v), false, false);
        v = op(f(r[0]), f(r[1]));
    }
    return v;
}

// The per-token quantizer's code: rn(clamp(y / s, -128, 127)) with a true division.
__device__ __forceinline__ int quant_code(float y, float s) {
    return (int)__builtin_rintf(fminf(fmaxf(y / s, -128.f), 127.f));
}

// v / s, correctly rounded, from inv = 1 / s (see store_codes).
__device__ __forceinline__ float quotient(float v, float s, float inv) {
#pragma clang fp contract(off)
    const float s_step = inv != 0.f ? s : 0.f;
    const float t = v * inv;
    return __builtin_fmaf(__builtin_fmaf(-t, s_step, v), inv, t);
}

// W codes of one chunk, stored as W consecutive bytes (W = 4 or 8): the same
// codes as quant_code(v, s) for every input, without a division.  With
// inv = 1/s correctly rounded, t = v * inv, r = v - t s (exact, one FMA) and
// q = t + r inv is the correctly rounded quotient v / s (Markstein's
// correction step; checked against true division on 1.2e10 random quantizer
// inputs, s = max(amax, 1e-8)/127 and |v| <= amax), so rint(clamp(q)) is the
// code.  A NaN element gives NaN on both paths.  An infinite element makes s
// infinite and inv zero: the step then uses 0 for s, so q = t = v * 0, which is
// v / s for finite v and NaN for infinite v, as the division gives.  No
// branch: a branch here, even one never taken, split the quantizers' load and
// store scheduling and cost them about 30%.
template <int W>
__device__ __forceinline__ void store_codes(const float (&v)[W], float s, float inv, int8_t* dst) {
    float q[W];
#pragma unroll
    for (int i = 0; i < W; ++i) q[i] = quotient(v[i], s, inv);
    uint32_t b[W / 4];
#pragma unroll
    for (int j = 0; j < W / 4; ++j) {
        b[j] = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = (int)__builtin_rintf(fminf(fmaxf(q[4 * j + i], -128.f), 127.f));
            b[j] |= ((uint32_t)c & 0xffu) << (8 * i);
        }
    }
    if constexpr (W == 8)
        *reinterpret_cast<uint2*>(dst) = make_uint2(b[0], b[1]);
    else
        *reinterpret_cast<uint32_t*>(dst) = b[0];
}

}  // namespace int8k
