// producer.hip — quantize-on-emit kernels for the ops that feed the INT8 attention and MLP.
//
// In the reference's transformer block every INT8 kernel input is produced by a
// separate eager quantization after the fp16 producer (bench/bench_block.py:59-63,
// 104-110, 119-121, 138-139): LayerNorm -> fp16 -> per-token quant for the MLP
// input, and QKV projection -> split heads -> .contiguous() -> per-token quant of
// Q, K and V.  These kernels do each of those chains in one pass:
//
//   layernorm_quant_kernel : y = LN(x) [fp32, biased variance, eps inside the
//       rsqrt, optional affine], rounded to the input dtype (what F.layer_norm
//       returns), then the per-token quantizer on that rounded y.  Optionally y
//       itself is written too.
//   quant_heads_kernel     : x [B, S, parts, H, Dh] (the QKV projection output
//       viewed by part and head) -> for each part, int8 [B, H, S, Dh] and fp32
//       scales [B, H, S]: per-token quantization over Dh, the layout the attention
//       kernels read.
//
// The quantizer is the one of quant.hip: s = max(amax, 1e-8) / 127,
// q = rn(clamp(y / s, -128, 127)) with a true division.
#include <algorithm>

#include "int8k_common.h"
#include "rows.h"

namespace int8k {
namespace {

__device__ __forceinline__ float load_any(const void* p, size_t i, int dtype) {
    switch (dtype) {
        case INT8K_DTYPE_F16: return __half2float(reinterpret_cast<const __half*>(p)[i]);
        case INT8K_DTYPE_BF16:
            return __uint_as_float((uint32_t)reinterpret_cast<const uint16_t*>(p)[i] << 16);
        default: return reinterpret_cast<const float*>(p)[i];
    }
}

// Rounds an fp32 value to the storage dtype and back (what a tensor of that
// dtype would hold), and stores it.
__device__ __forceinline__ float round_to(float v, int dtype) {
    switch (dtype) {
        case INT8K_DTYPE_F16: return __half2float(__float2half_rn(v));
        case INT8K_DTYPE_BF16: {
            // round to nearest even on the upper 16 bits (finite inputs)
            const uint32_t u = __float_as_uint(v);
            const uint32_t r = (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u;
            return __uint_as_float(r);
        }
        default: return v;
    }
}

__device__ __forceinline__ void store_any(void* p, size_t i, float v, int dtype) {
    switch (dtype) {
        case INT8K_DTYPE_F16: reinterpret_cast<__half*>(p)[i] = __float2half_rn(v); break;
        case INT8K_DTYPE_BF16:
            reinterpret_cast<uint16_t*>(p)[i] = (uint16_t)(__float_as_uint(v) >> 16);
            break;
        default: reinterpret_cast<float*>(p)[i] = v;
    }
}

__device__ __forceinline__ int8_t quantize(float y, float s) {
    return (int8_t)(int)__builtin_rintf(fminf(fmaxf(y / s, -128.f), 127.f));
}

constexpr int kWaves = 4;
// Row kernels launch at most this many blocks (a launch must hold fewer than 2^32
// work-items) and stride over the remaining rows.
constexpr long long kMaxBlocks = 1LL << 20;
// The vectorised kernels stride over rows from a grid of at most this many
// blocks (about 8 resident blocks per CU of a 256-CU device, 4 rounds).
constexpr long long kVecBlocks = 8192;

// LayerNorm keeps gamma and beta in registers over a wave's rows: a grid of 4
// blocks per CU, so that many rows share one read of them.  Without either the
// rows spread over more blocks (fp32 30000 x 512 16.9 -> 14.8 us, 100000 x 256 36.3 -> 29.0).
constexpr long long kLnBlocks = 1024;
// Elements per lane of the longest row of layernorm_quant_row_kernel (768 columns).  The
// whole range below gains on a block per row, with gamma and beta: 4000 rows fp16, block ->
// wave: 320 columns 11.4 -> 6.1 us, 520 15.0 -> 6.7, 768 16.4 -> 7.3; 7 rows 5.1 -> 3.3 and
// 6.3 -> 3.5.  Rows up to 1280 would too, on an instance of 20 elements (776 18.4 -> 9.6,
// 960 19.5 -> 9.8, 1280 23.5 -> 10.4), which costs the shorter rows a third if they share it
// (768 columns 9.4 us): there is none yet.
constexpr int kRowElems = 12;

template <typename Op>
__device__ __forceinline__ float wave_reduce(float v, Op op) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) v = op(v, __shfl_xor(v, off));
    return v;
}

// One block of 4 waves per row.  Pass 1: mean; pass 2: centred sum of squares;
// pass 3: y and its absmax; pass 4: y again (bit-identical) and its codes.  The
// row is re-read from L2/L1 after the first pass.
__global__ __launch_bounds__(256) void layernorm_quant_kernel(
    const void* __restrict__ x, int dtype, const float* __restrict__ gamma,
    const float* __restrict__ beta, float eps, int8_t* __restrict__ q, float* __restrict__ scales,
    void* __restrict__ y_out, long long rows, int cols) {
    __shared__ float red[kWaves];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    for (long long row = blockIdx.x; row < rows; row += gridDim.x) {  // < 2^32 work-items/launch
    const size_t base = (size_t)row * (size_t)cols;
    auto block_reduce = [&](float v, auto op) {
        v = wave_reduce(v, op);
        if (lane == 0) red[wave] = v;
        __syncthreads();
        float r = red[0];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) r = op(r, red[w]);
        __syncthreads();
        return r;
    };
    auto add = [](float a, float b) { return a + b; };
    auto mx = [](float a, float b) { return fmaxf(a, b); };

    float s = 0.f;
    for (int c = t; c < cols; c += 256) s += load_any(x, base + c, dtype);
    const float mean = block_reduce(s, add) / (float)cols;
    float v = 0.f;
    for (int c = t; c < cols; c += 256) {
        const float d = load_any(x, base + c, dtype) - mean;
        v = fmaf(d, d, v);
    }
    const float rstd = 1.f / sqrtf(block_reduce(v, add) / (float)cols + eps);
    auto ln = [&](int c) {
        float y = (load_any(x, base + c, dtype) - mean) * rstd;
        if (gamma) y *= gamma[c];
        if (beta) y += beta[c];
        return round_to(y, dtype);
    };
    float m = 0.f;
    for (int c = t; c < cols; c += 256) m = fmaxf(m, fabsf(ln(c)));
    const float sc = fmaxf(block_reduce(m, mx), 1e-8f) / 127.f;
    for (int c = t; c < cols; c += 256) {
        const float y = ln(c);
        q[base + c] = quantize(y, sc);
        if (y_out) store_any(y_out, base + c, y, dtype);
    }
    if (t == 0) scales[row] = sc;
    }
}

// One wave per source row (b, s, part, h) of Dh elements (grid-stride).
__global__ __launch_bounds__(256) void quant_heads_kernel(
    const void* __restrict__ x, int dtype, int8_t* __restrict__ q0, float* __restrict__ s0,
    int8_t* __restrict__ q1, float* __restrict__ s1, int8_t* __restrict__ q2,
    float* __restrict__ s2, long long rows, int S, int parts, int H, int Dh) {
    const int lane = threadIdx.x & 63;
    for (long long r = (long long)blockIdx.x * kWaves + (threadIdx.x >> 6); r < rows;
         r += (long long)gridDim.x * kWaves) {
        // r = ((b * S + s) * parts + p) * H + h
        const int h = (int)(r % H);
        const long long r1 = r / H;
        const int p = (int)(r1 % parts);
        const long long bs = r1 / parts;
        const long long b = bs / S, s = bs - b * S;
        const size_t src = (size_t)r * Dh;
        float m = 0.f;
        for (int c = lane; c < Dh; c += 64) m = fmaxf(m, fabsf(load_any(x, src + c, dtype)));
        m = wave_reduce(m, [](float a, float bb) { return fmaxf(a, bb); });
        const float sc = fmaxf(m, 1e-8f) / 127.f;
        int8_t* q = p == 0 ? q0 : (p == 1 ? q1 : q2);
        float* sp = p == 0 ? s0 : (p == 1 ? s1 : s2);
        const size_t drow = ((size_t)b * H + h) * S + s;  // [B, H, S] row of the part
        for (int c = lane; c < Dh; c += 64)
            q[drow * Dh + c] = quantize(load_any(x, src + c, dtype), sc);
        if (lane == 0) sp[drow] = sc;
    }
}

// ------------------------------------------------- vectorised paths (rows.h)

// Storage bits of y (already rounded to the dtype by round_to) for one chunk.
template <int DT>
__device__ __forceinline__ uint4 pack_chunk(const float (&y)[Vec<DT>::W]) {
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (DT == INT8K_DTYPE_F32) {
            d[i] = __float_as_uint(y[i]);
        } else if constexpr (DT == INT8K_DTYPE_F16) {
            d[i] = (uint32_t)__half_as_ushort(__float2half_rn(y[2 * i])) |
                   ((uint32_t)__half_as_ushort(__float2half_rn(y[2 * i + 1])) << 16);
        } else {
            d[i] = (__float_as_uint(y[2 * i]) >> 16) | (__float_as_uint(y[2 * i + 1]) & 0xffff0000u);
        }
    }
    return make_uint4(d[0], d[1], d[2], d[3]);
}

// gamma or beta of the W columns from col0 (a multiple of W): as 16-byte vectors
// where the array is aligned for them, else one by one.
template <int W>
__device__ __forceinline__ void load_affine(const float* p, int col0, bool vec, float (&v)[W]) {
    if (vec) {
#pragma unroll
        for (int j = 0; j < W; j += 4) {
            const float4 f = *reinterpret_cast<const float4*>(p + col0 + j);
            v[j] = f.x, v[j + 1] = f.y, v[j + 2] = f.z, v[j + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int e = 0; e < W; ++e) v[e] = p[col0 + e];
    }
}

// LayerNorm + per-token quantizer with the row in registers: 1 << lg lanes per
// row, NC 16-byte chunks per lane.  One read of x; the passes of the
// one-element-per-lane kernel above become register passes.  PAD: slots past the
// row repeat its last chunk and count for nothing in the sums.  gamma and beta stay in
// registers over a wave's rows where they fit (up to 4 chunks per lane): re-read per
// row they are up to 4x the bytes of x through L2.
// HBM-bound, and latency-bound for few rows.  us with gamma and beta, element by
// element -> as vectors: 16384 x 1024 fp16 66 -> 16.7, 8192 x 5120 fp16 180 -> 63, 4096
// x 8192 bf16 155 -> 66.
template <int DT, int NC, bool PAD>
__global__ __launch_bounds__(256) void layernorm_quant_vec_kernel(
    const void* __restrict__ x, const float* __restrict__ gamma, const float* __restrict__ beta,
    float eps, int8_t* __restrict__ q, float* __restrict__ scales, void* __restrict__ y_out,
    uint32_t rows, int lg, uint32_t cpr, int affine_vec) {
    constexpr int W = Vec<DT>::W;
    constexpr bool kHold = NC <= 4;  // gamma and beta in registers
    const int lane = threadIdx.x & 63;
    const uint32_t rpw = 64u >> lg;
    const uint32_t c0 = lane & ((1u << lg) - 1);
    if (!PAD) cpr = (uint32_t)NC << lg;
    auto real = [&](int i) { return !PAD || ((uint32_t)i << lg) + c0 < cpr; };
    auto col_of = [&](int i) { return (int)(slot_chunk<PAD>(i, lg, c0, cpr) * W); };
    const int cols = (int)cpr * W;
    const float inv_cols = 1.f / (float)cols;
    const uint4* src = reinterpret_cast<const uint4*>(x);
    auto add = [](float a, float b) { return a + b; };
    float eg[kHold ? NC : 1][W], eb[kHold ? NC : 1][W];
    if constexpr (kHold) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            if (gamma) load_affine<W>(gamma, col_of(i), affine_vec, eg[i]);
            if (beta) load_affine<W>(beta, col_of(i), affine_vec, eb[i]);
        }
    }
    const uint32_t nw = gridDim.x * 4;
    for (uint32_t rb = (blockIdx.x * 4 + (threadIdx.x >> 6)) * rpw; rb < rows; rb += nw * rpw) {
        // rows past the end take the last row and store it again (the same bytes
        // its own lane stores): no divergent branch around loads or stores
        const uint32_t r = min(rb + (lane >> lg), rows - 1);
        uint4 w[NC];
#pragma unroll
        for (int i = 0; i < NC; ++i)
            w[i] = src[(size_t)r * cpr + slot_chunk<PAD>(i, lg, c0, cpr)];
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            float v[W];
            unpack_chunk<DT>(w[i], v);
#pragma unroll
            for (int e = 0; e < W; ++e) sum += real(i) ? v[e] : 0.f;
        }
        float mean = row_reduce(sum, lg, add) * inv_cols;
        // rounded here: the compiler fused the product into x - mean of the variance alone in
        // some instances, which left the error of 1 / cols in every deviation
        asm("" : "+v"(mean));
#pragma unroll
        for (int i = 0; i < NC; ++i) reload_barrier(w[i]);
        float var = 0.f;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            float v[W];
            unpack_chunk<DT>(w[i], v);
#pragma unroll
            for (int e = 0; e < W; ++e) {
                const float d = real(i) ? v[e] - mean : 0.f;
                var = fmaf(d, d, var);
            }
        }
        const float rstd = 1.f / sqrtf(row_reduce(var, lg, add) * inv_cols + eps);
#pragma unroll
        for (int i = 0; i < NC; ++i) reload_barrier(w[i]);
        // y, rounded to the dtype, replaces x in the chunk registers (its storage
        // bits: unpacking them gives the rounded values back exactly)
        const float* g = gamma;
        const float* bt = beta;
        asm volatile("" : "+s"(g), "+s"(bt));  // re-read here, not hoisted (!kHold)
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            float y[W];
            unpack_chunk<DT>(w[i], y);
#pragma unroll
            for (int e = 0; e < W; ++e) y[e] = (y[e] - mean) * rstd;
            if (gamma) {
                float p[W];
                if constexpr (!kHold) load_affine<W>(g, col_of(i), affine_vec, p);
#pragma unroll
                for (int e = 0; e < W; ++e) y[e] *= kHold ? eg[kHold ? i : 0][e] : p[e];
            }
            if (beta) {
                float p[W];
                if constexpr (!kHold) load_affine<W>(bt, col_of(i), affine_vec, p);
#pragma unroll
                for (int e = 0; e < W; ++e) y[e] += kHold ? eb[kHold ? i : 0][e] : p[e];
            }
#pragma unroll
            for (int e = 0; e < W; ++e) {
                y[e] = round_to(y[e], DT);
                m = fmaxf(m, fabsf(y[e]));
            }
            w[i] = pack_chunk<DT>(y);
        }
        const float sc = fmaxf(row_reduce(m, lg, [](float a, float b) { return fmaxf(a, b); }),
                               1e-8f) / 127.f;
        const float inv = 1.f / sc;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            float y[W];
            unpack_chunk<DT>(w[i], y);
            const size_t chunk = (size_t)r * cpr + slot_chunk<PAD>(i, lg, c0, cpr);
            store_codes<W>(y, sc, inv, q + chunk * W);
            if (y_out) reinterpret_cast<uint4*>(y_out)[chunk] = w[i];
        }
        if (c0 == 0) scales[r] = sc;
    }
}

// Short rows whose chunks fill neither a power of two of lanes nor whole waves (80, 768
// columns): one wave per row, the row in registers, one element per lane and
// 64 columns (NE of them).  The sums keep the order of layernorm_quant_kernel, whose
// thread t + 64 w is this lane's column group w modulo 4, so both give the same
// bytes: a code on a rounding tie follows the last bit of mean and rstd.  One read of
// x instead of five.  Against a block per row: 100000 x 80 fp16 155 -> 46 us, 4000 x 768
// 16.4 -> 7.3 (bound by the latency of the row's loads and reductions; kRowElems).
template <int DT, int NE>
__global__ __launch_bounds__(256) void layernorm_quant_row_kernel(
    const void* __restrict__ x, const float* __restrict__ gamma, const float* __restrict__ beta,
    float eps, int8_t* __restrict__ q, float* __restrict__ scales, void* __restrict__ y_out,
    long long rows, int cols) {
    const int lane = threadIdx.x & 63;
    auto add = [](float a, float b) { return a + b; };
    // the four waves' sums of a block, each over its 64 lanes, then in wave order
    auto block_sum = [&](const float (&s)[4]) {
        float r = row_reduce(s[0], 6, add);
#pragma unroll
        for (int w = 1; w < 4; ++w) r = r + row_reduce(s[w], 6, add);
        return r;
    };
    for (long long row = (long long)blockIdx.x * kWaves + (threadIdx.x >> 6); row < rows;
         row += (long long)gridDim.x * kWaves) {
        const size_t base = (size_t)row * (size_t)cols;
        float v[NE];
#pragma unroll
        for (int k = 0; k < NE; ++k) v[k] = load_any(x, base + min(lane + 64 * k, cols - 1), DT);
        // gamma and beta in flight beside x: behind the sums each was a round trip to L2 of
        // its own (4.3 us of 4000 x 768 bf16)
        float eg[NE], eb[NE];
#pragma unroll
        for (int k = 0; k < NE; ++k) {
            const int c = min(lane + 64 * k, cols - 1);
            eg[k] = gamma ? gamma[c] : 1.f;
            eb[k] = beta ? beta[c] : 0.f;
        }
        float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < NE; ++k) s[k & 3] += lane + 64 * k < cols ? v[k] : 0.f;
        const float mean = block_sum(s) / (float)cols;
        float t[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < NE; ++k) {
            const float d = lane + 64 * k < cols ? v[k] - mean : 0.f;
            t[k & 3] = fmaf(d, d, t[k & 3]);
        }
        const float rstd = 1.f / sqrtf(block_sum(t) / (float)cols + eps);
        float m = 0.f;
#pragma unroll
        for (int k = 0; k < NE; ++k) {
            float y = (v[k] - mean) * rstd;
            if (gamma) y *= eg[k];
            if (beta) y += eb[k];
            // past the row: the last column's x with the last column's parameters
            v[k] = round_to(y, DT);
            m = fmaxf(m, fabsf(v[k]));
        }
        const float sc =
            fmaxf(row_reduce(m, 6, [](float a, float b) { return fmaxf(a, b); }), 1e-8f) / 127.f;
        const float inv = 1.f / sc;  // one division per row, not per element (0.7 us there)
#pragma unroll
        for (int k = 0; k < NE; ++k) {
            const int c = lane + 64 * k;
            if (c < cols) {
                q[base + c] = (int8_t)(int)__builtin_rintf(
                    fminf(fmaxf(quotient(v[k], sc, inv), -128.f), 127.f));
                if (y_out) store_any(y_out, base + c, v[k], DT);
            }
        }
        if (lane == 0) scales[row] = sc;
    }
}

// Split-heads + per-token quantizer: source row ((b S + s) parts + p) H + h of
// Dh elements, 1 << lg lanes per row, one 16-byte chunk per lane.  Rows are
// walked in destination order k = ((p B + b) H + h) S + s, so the rows of a
// wave are consecutive tokens of one head: its codes and scales go out as one
// contiguous run (not as 64-byte pieces of H different heads), while each row
// is still read as one full source row.  Each wave takes U row groups of its
// grid stride at a time (U loads per lane in flight).  PAD: rows of cpr chunks on
// more lanes (head_dim 80: 10 chunks on 16 lanes), the spare ones repeating the last.
template <int DT, bool PAD, int U>
__global__ __launch_bounds__(256) void quant_heads_vec_kernel(
    const void* __restrict__ x, int8_t* __restrict__ q0, float* __restrict__ s0,
    int8_t* __restrict__ q1, float* __restrict__ s1, int8_t* __restrict__ q2,
    float* __restrict__ s2, uint32_t rows, uint32_t S, uint32_t parts, uint32_t H, int lg,
    uint32_t cpr) {
    constexpr int W = Vec<DT>::W;
    const int lane = threadIdx.x & 63;
    const uint32_t rpw = 64u >> lg;
    if (!PAD) cpr = 1u << lg;
    const uint32_t c0 = slot_chunk<PAD>(0, lg, lane & ((1u << lg) - 1), cpr);
    const int Dh = (int)cpr * W;
    const uint4* src = reinterpret_cast<const uint4*>(x);
    const uint32_t stride = gridDim.x * 4 * rpw;
    const uint32_t part_rows = rows / parts;  // B H S rows per part
    for (uint32_t kb = (blockIdx.x * 4 + (threadIdx.x >> 6)) * rpw; kb < rows; kb += U * stride) {
        uint4 w[U];
        uint32_t drow[U], pp[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // rows past the end take the last row: they load, quantize and store
            // it again, the same bytes its own lane stores.  No divergent branch
            // around the loads or the stores, which keeps them all in flight.
            const uint32_t k = min(kb + u * stride + (lane >> lg), rows - 1);
            pp[u] = k / part_rows;
            drow[u] = k - pp[u] * part_rows;  // (b H + h) S + s
            const uint32_t bh = drow[u] / S, s = drow[u] - bh * S;
            const uint32_t b = bh / H, h = bh - b * H;
            const uint32_t r = ((b * S + s) * parts + pp[u]) * H + h;
            w[u] = src[(size_t)r * cpr + c0];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float v[W];
            unpack_chunk<DT>(w[u], v);
            float m = 0.f;
#pragma unroll
            for (int e = 0; e < W; ++e) m = fmaxf(m, fabsf(v[e]));
            m = row_reduce(m, lg, [](float a, float b) { return fmaxf(a, b); });
            const float sc = fmaxf(m, 1e-8f) / 127.f;
            const float inv = 1.f / sc;
            int8_t* q = pp[u] == 0 ? q0 : (pp[u] == 1 ? q1 : q2);
            float* sp = pp[u] == 0 ? s0 : (pp[u] == 1 ? s1 : s2);
            store_codes<W>(v, sc, inv, q + (size_t)drow[u] * Dh + (size_t)c0 * W);
            if (c0 == 0) sp[drow[u]] = sc;
        }
    }
}

}  // namespace
}  // namespace int8k

using namespace int8k;

extern "C" int int8k_layernorm_quantize_per_token(const void* x, int dtype, const float* gamma,
                                                  const float* beta, float eps, int8_t* q,
                                                  float* scales, void* y_out, long long rows,
                                                  int cols, void* stream) {
    clear_last_error();
    if (!x || !q || !scales || rows < 0 || cols <= 0 || !(eps >= 0.f))
        return INT8K_ERR_INVALID_ARGUMENT;
    if (dtype != INT8K_DTYPE_F16 && dtype != INT8K_DTYPE_BF16 && dtype != INT8K_DTYPE_F32)
        return INT8K_ERR_INVALID_ARGUMENT;
    if (rows == 0) return INT8K_OK;
    hipStream_t st = as_stream(stream);
    const RowShape sh = row_shape(cols, dtype);
    const int w = dtype == INT8K_DTYPE_F32 ? 4 : 8;
    // rows that fill a power of two of lanes, or whole waves
    const bool fills = sh.ok && (sh.nc == 1 ? sh.cpr == 1 << sh.lg : sh.cpr % 64 == 0);
    if (fills && rows < (1LL << 31) && aligned_to(x, 16) && aligned_to(q, w) &&
        (!y_out || aligned_to(y_out, 16))) {
        const long long waves = ceil_div(rows, 64 >> sh.lg);
        const unsigned blocks =
            (unsigned)std::min(ceil_div(waves, 4), gamma || beta ? kLnBlocks : kVecBlocks);
        const int affine_vec =
            (!gamma || aligned_to(gamma, 16)) && (!beta || aligned_to(beta, 16));
        with_dtype(dtype, [&](auto dt) {
            with_chunks(sh, [&](auto ncc, auto pad) {
                layernorm_quant_vec_kernel<decltype(dt)::value, decltype(ncc)::value,
                                           decltype(pad)::value>
                    <<<blocks, 256, 0, st>>>(x, gamma, beta, eps, q, scales, y_out,
                                             (uint32_t)rows, sh.lg, (uint32_t)sh.cpr, affine_vec);
            });
        });
        return check_launch("layernorm_quant_vec_kernel");
    }
    if (cols <= 64 * kRowElems) {
        const unsigned blocks = (unsigned)std::min(ceil_div(rows, kWaves), kMaxBlocks);
        with_dtype(dtype, [&](auto dt) {
            auto launch = [&](auto ne) {
                layernorm_quant_row_kernel<decltype(dt)::value, decltype(ne)::value>
                    <<<blocks, 256, 0, st>>>(x, gamma, beta, eps, q, scales, y_out, rows, cols);
            };
            if (cols <= 256) launch(std::integral_constant<int, 4>{});
            else launch(std::integral_constant<int, kRowElems>{});
        });
        return check_launch("layernorm_quant_row_kernel");
    }
    layernorm_quant_kernel<<<(unsigned)std::min(rows, kMaxBlocks), 256, 0, st>>>(
        x, dtype, gamma, beta, eps, q, scales, y_out, rows, cols);
    return check_launch("layernorm_quant_kernel");
}

extern "C" int int8k_quantize_heads(const void* x, int dtype, int parts, int8_t* q0, float* s0,
                                    int8_t* q1, float* s1, int8_t* q2, float* s2, int B, int S,
                                    int H, int head_dim, void* stream) {
    clear_last_error();
    if (!x || parts < 1 || parts > 3 || B <= 0 || S <= 0 || H <= 0 || head_dim <= 0)
        return INT8K_ERR_INVALID_ARGUMENT;
    if (dtype != INT8K_DTYPE_F16 && dtype != INT8K_DTYPE_BF16 && dtype != INT8K_DTYPE_F32)
        return INT8K_ERR_INVALID_ARGUMENT;
    int8_t* qs[3] = {q0, q1, q2};
    float* ss[3] = {s0, s1, s2};
    for (int p = 0; p < parts; ++p)
        if (!qs[p] || !ss[p]) return INT8K_ERR_INVALID_ARGUMENT;
    const long long rows = (long long)B * S * parts * H;
    hipStream_t st = as_stream(stream);
    const RowShape sh = row_shape(head_dim, dtype);
    const int w = dtype == INT8K_DTYPE_F32 ? 4 : 8;
    bool vec = sh.ok && sh.nc == 1 && rows < (1LL << 31) && aligned_to(x, 16);
    for (int p = 0; p < parts; ++p) vec = vec && aligned_to(qs[p], w);
    if (vec) {
        constexpr int U = 4;
        const long long waves = ceil_div(rows, 64 >> sh.lg);
        const unsigned blocks = (unsigned)std::min(ceil_div(waves, 4 * U), kVecBlocks);
        with_dtype(dtype, [&](auto dt) {
            with_chunks(sh, [&](auto ncc, auto pad) {
                if constexpr (decltype(ncc)::value == 1)
                    quant_heads_vec_kernel<decltype(dt)::value, decltype(pad)::value, U>
                        <<<blocks, 256, 0, st>>>(x, q0, s0, q1, s1, q2, s2, (uint32_t)rows,
                                                 (uint32_t)S, (uint32_t)parts, (uint32_t)H, sh.lg,
                                                 (uint32_t)sh.cpr);
            });
        });
        return check_launch("quant_heads_vec_kernel");
    }
    quant_heads_kernel<<<(unsigned)std::min(ceil_div(rows, kWaves), kMaxBlocks), 256, 0, st>>>(
        x, dtype, q0, s0, q1, s1, q2, s2, rows, S, parts, H, head_dim);
    return check_launch("quant_heads_kernel");
}
