// decode.hip — split-KV flash-decoding over a contiguous INT8 KV cache (gfx950).
//
// Computes, for every (b,h) = bh and a single query token,
//     out[bh,:] = sum_j softmax_j(score_j) * (V[bh,j,:] * sV[bh*S+j])
//     score_j   = (Q[bh,:] . K[bh,j,:]) * sQ[bh] * sK[bh*S+j] / sqrt(D)
// which is the contract of the reference launcher
// int8_decode_attention_forward (kernels/int8_decode_attention.cu:443-547) and
// of its partial/combine pair (kernels/int8_decode_attention.cu:274-426).
//
// Design (CDNA4 first, not a translation of the warp-per-unit CUDA kernel):
//
//  * HBM-bound: one pass over K and V (2*BH*S*D bytes) dominates.  Each wave64
//    lane issues 16-byte global loads; a wave's load instruction covers
//    64 x 16 B = 1 KiB made of whole 128-byte (D=128) or 64-byte (D=64) rows.
//  * Lane layout: LPR = D/16 lanes share a row (lane s of the group holds row
//    bytes [16s, 16s+16)); G = 64/LPR row-groups per wave.  One wave
//    iteration covers R = G*NSLOT rows: group g owns rows g*NSLOT .. +NSLOT-1
//    of the block, one per load slot, so every slot of every lane is an
//    immediate offset from one base address.
//  * Paired rows (D=64, 4 slots, the 8-wave one-launch kernels): a 64-byte
//    row is half a 128-byte line, so groups 2h and 2h+1 take the even and the
//    odd rows of block rows 8h..8h+7 (slot t: row 8h + o + 2t) and every load
//    instruction covers whole lines.  That makes non-temporal K/V loads pay
//    at D=64 too; with half lines per instruction they cost 20-100%.
//  * Scales: lane s of a group loads the scales of slots s % 4 (+ 4), one dword
//    each, and the quad reads them with a DPP broadcast folded into the multiply:
//    a wave's scale load is 256 contiguous bytes with no alignment beyond a
//    dword, so odd row strides cost nothing.
//  * QK: 4 v_dot4_i32_i8 per slot per lane (exact int32), then a DPP sum over
//    the LPR lanes of the group (no LDS).  The group's lanes all hold the score.
//  * Softmax: every row-group keeps its own online-softmax state (m, l) in the
//    log2 domain and its own fp32 accumulator for the 16 dims its lane holds,
//    so the hot loop has no cross-group traffic at all.  The G group states of
//    a wave are merged once, at the end of the wave's KV chunk.
//  * PV: each V byte is converted with one SDWA v_cvt_f32_i32 and folded in
//    with one FMA: acc += (p_j * sV_j) * v_j.
//  * Split-KV: a wave walks one chunk of one (b,h), the up to 8 waves of a block
//    merge on chip, and where one block per (b,h) would leave CUs idle several
//    blocks share it: their partial states (m, l, acc[D]) go to the workspace and
//    a combine kernel merges them with the log-sum-exp rule (plan_groups).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

#include "int8k_common.h"
#include "rows.h"

namespace int8k {
namespace {

constexpr int kWavesPerBlock = 4;
constexpr int kNtKV = 1;      // non-temporal K/V loads (each row is read once)
constexpr int kNtScales = 2;  // non-temporal sK/sV loads
constexpr int kBlockThreads = 64 * kWavesPerBlock;

// NS = load slots: rows per row-group per wave iteration (each slot is one
// 16-byte K load and one 16-byte V load per lane).
template <int D, int NS>
struct DecodeGeom {
    static_assert(D == 64 || D == 128, "decode supports head_dim 64 and 128");
    static_assert(NS == 4 || NS == 8, "slots per iteration: 4 or 8");
    static constexpr int kLanesPerRow = D / 16;
    static constexpr int kGroups = 64 / kLanesPerRow;
    static constexpr int kRowsPerIter = kGroups * NS;
};

// Rows per wave iteration for a head dim (host side).
inline int rows_per_iter(int D, int ns) { return (64 / (D / 16)) * ns; }

// Paired rows (the 8-wave one-launch kernels at D=64 with 4 slots): group
// 2h+o owns rows 8h+o, +2, +4, +6 of a wave iteration's block, so each load
// slot covers whole 128-byte lines; otherwise group g owns rows g*NS .. +NS-1.
constexpr bool paired_rows(int D, int NS, int MAXW) { return D == 64 && NS == 4 && MAXW <= 8; }

// Two register sets (the next iteration's loads in flight) in the 8-wave
// one-launch kernels: at 4 slots, and at D = 128 with 8 slots.
constexpr bool two_sets(int D, int NS, int MAXW) { return MAXW <= 8 && (NS == 4 || D == 128); }

template <bool PAIRED, int NS>
__device__ __forceinline__ int group_row0(int grp) {
    if constexpr (PAIRED) return 8 * (grp >> 1) + (grp & 1);
    else return grp * NS;
}

// Launch-time tuning of the decode kernel.
struct DecodeTuning {
    int slots;         // NS
    int flags;         // kNtKV | kNtScales
    int target_units;  // units (waves) to aim for
    int stagger;       // rotate each unit's starting iteration
    int pair_flags;    // load flags of the paired-row kernels (D=64, 4 slots, <= 8 chunks)
};


// How the chunks of a (b,h) are laid out on blocks: `blocks` blocks of `waves`
// waves, each wave `chunk` rows.  The states of a block's waves merge on chip;
// with more than one block per (b,h) each leaves a partial for
// decode_combine_kernel.
struct GroupPlan {
    int blocks, waves, chunk;
};

// A decode's plan: chunks per (b,h) and their rows, the blocks that run them, and the
// partials per (b,h) that the workspace has room for.  An automatic plan above
// kMaxBlockSplits chunks has its own rows per wave in g; its nsplit is only what
// num_splits reports.
struct SplitPlan {
    int nsplit;
    int chunk;
    bool forced;  // the caller's split count
    GroupPlan g;
    int partials;
};

// Most waves (chunks) per block of the one-launch and grouped kernels' fast instance.
constexpr int kGroupWaves = 8;

// Most chunks per (b,h) that run as one launch (decode_block_kernel: one wave
// per chunk, merged in LDS); larger plans run several blocks and the combine.
constexpr int kMaxBlockSplits = 16;
// The automatic plan never picks 9..16 chunks: those would run the 16-wave
// instance (one register set), and 8 chunks on the 8-wave instance (two
// register sets, paired rows at D=64) measured 2-27% faster at every shape
// tried (B1 H12 D64 1K to B16 H32 D128 8K).  Forced split counts still may.
constexpr int kMaxAutoBlockSplits = 8;
// Work units (a (b,h) of a one-launch plan, a (b,h,chunk) of a split plan) that
// met a page id outside [0, num_pages) among the pages their positions use
// (int8k_decode_paged_bad_page_ids).  Such an id reads the last page instead.
__device__ unsigned int g_paged_bad_ids;

// Largest page-id table the paged one-launch kernel stages in LDS (12288 ids);
// a block whose rows need more runs decode_paged_kernel + the combine.
constexpr long long kPagedLdsTableBytes = 48 << 10;

// Plans of at most kMaxBlockSplits chunks run as one launch (decode_block_kernel);
// INT8K_DECODE_BLOCK=0 makes them leave partials for the combine kernel (read once).
bool use_block_kernel() {
    static const bool on = [] {
        const char* e = std::getenv("INT8K_DECODE_BLOCK");
        return !(e != nullptr && e[0] == '0');
    }();
    return on;
}

inline int env_int(const char* name, int dflt) {
    const char* e = std::getenv(name);
    return e ? std::atoi(e) : dflt;
}

// Defaults measured on MI355X at the BASELINE shapes (B32 H32 D128 8K and
// B8 H32 D64 2K..32K): D=128 — 8 slots, non-temporal K/V loads, ~8192 units
// (two resident rounds at 16 waves/CU); D=64 — 4 slots, non-temporal scale
// loads, ~2048 units (8 chunks per (b,h) at B8 H32: two waves per SIMD);
// its paired-row kernels (plans of up to 8 chunks) load K/V non-temporally
// and the scales as plain loads (ctx 2K-32K: 5-11% faster than the grouped
// rows with non-temporal scales).  Both rotate each unit's starting
// iteration (stagger), which was worth 2-5%.  The INT8K_DECODE_* variables
// override these for tuning sweeps (read once per process).
DecodeTuning tuning_for(int D) {
    static const int e_slots = env_int("INT8K_DECODE_SLOTS", 0);
    static const int e_flags = env_int("INT8K_DECODE_FLAGS", -1);
    static const int e_units = env_int("INT8K_DECODE_TARGET_UNITS", 0);
    static const int e_stagger = env_int("INT8K_DECODE_STAGGER", -1);
    static const int e_pair = env_int("INT8K_DECODE_PAIR_FLAGS", -1);
    DecodeTuning t;
    if (D == 128) t = DecodeTuning{8, kNtKV, 8192, 1, kNtKV};
    else t = DecodeTuning{4, kNtScales, 2048, 1, kNtKV};
    if (e_slots == 4 || e_slots == 8) t.slots = e_slots;
    if (e_flags >= 0) t.flags = e_flags & 3;
    if (e_units > 0) t.target_units = e_units;
    if (e_stagger >= 0) t.stagger = e_stagger;
    if (e_pair >= 0) t.pair_flags = e_pair & 3;
    return t;
}

constexpr int kNumCus = 256;

constexpr long long kChunkAlias = 512 << 10;  // bytes (see plan_groups)

// Most blocks per (b,h) of an automatic plan: 8, or one for each CU.
inline long long most_groups(int BH, long long iters) {
    return std::min(ceil_div(iters, kGroupWaves), std::max(8LL, (long long)kNumCus / BH));
}

// Automatic plans of the 8-wave kernels take the blocks per (b,h) (at most `most`)
// with the smallest cost in wave iterations: a round is one block on each CU,
// a block costs its waves' iterations plus about 2 for its first loads and its
// merge, and the second launch about 4 at D = 64 and 2 at D = 128 (a CU streams
// one block at ~55 GB/s: 1.27 and 2.5 us per iteration).  So short sequences stay
// on one block (B1 H16 D128 1500 rows, B1 H12 D64 2500 rows) and longer ones spread
// (paged B4 H16 D64 4000 rows: 15.7 us on one block, 10.4 on four and a combine; B1 H12
// D64 4096 rows: 13.2 -> 12.3 us on 8 blocks, B1 H8 D128 3000 rows 19.6 -> 12.2, B4 H12
// D128 2500 rows 18.4 -> 12.3).
// Sweeps of 1..32 blocks at 8 to 64 (b,h) put the best time at one full round or
// within 3% of it (B2 H8 D128 60013 rows: 53.2 / 44.1 / 46.0 us at 8 / 16 / 32
// blocks; B1 H32 D64 128K: 103 / 87 / 88 us at 4 / 8 / 16): a partial extra round
// leaves CUs idle, and fewer blocks than CUs read at a CU's ~55 GB/s each.
// Chunks of whole multiples of 512 KB cost an eighth more: their waves read slower than
// those of other lengths, probably in step on the same HBM channels (B8 H32 D128 on one
// block: 6.7 TB/s at 32000 and 33001 rows, 6.2 at 32768, and 6.6 on two blocks: 343 -> 322
// us; B2 H32 131072 rows on 4 and 8 blocks 350 -> 321, B4 H32 65536 on 2 and 4 350 -> 320).
GroupPlan plan_groups(int BH, int S, int D, int slots, long long most) {
    const int R = rows_per_iter(D, slots);
    const long long iters = ceil_div(S, R);
    most = std::max(1LL, std::min(most, most_groups(BH, iters)));
    long long best = -1, per_wave = 0, blocks = 1;
    for (long long nb = 1; nb <= most; ++nb) {
        const long long pw = ceil_div(iters, nb * kGroupWaves);
        const long long bl = ceil_div(iters, pw * kGroupWaves);
        const long long rounds = ceil_div(BH * bl, kNumCus);
        long long cost = 2 * rounds * (pw + 2) + (bl > 1 ? (D == 128 ? 4 : 8) : 0);
        if (pw * R * D % kChunkAlias == 0) cost += cost / 8;
        if (best < 0 || cost < best) best = cost, per_wave = pw, blocks = bl;
    }
    const int waves = (int)std::min<long long>(kGroupWaves, ceil_div(iters, per_wave));
    return GroupPlan{(int)blocks, waves, (int)(per_wave * R)};
}

// A forced plan keeps its chunks, up to kGroupWaves to a block.
inline GroupPlan forced_groups(int nsplit, int chunk) {
    const int blocks = (int)ceil_div(nsplit, kGroupWaves);
    return GroupPlan{blocks, (int)ceil_div(nsplit, blocks), chunk};
}

// Split-count choice: a unit is one wave over one KV chunk of one (b,h);
// aim for tuning.target_units units in total, each chunk a multiple of the
// rows one wave iteration covers.  on_chip: an automatic plan that merges on chip
// wherever it did without the choice of several blocks.
SplitPlan plan_splits(int BH, int S, int D, int nsplit_req, bool on_chip = false) {
    const DecodeTuning tn = tuning_for(D);
    const int R = rows_per_iter(D, tn.slots);
    const long long max_split = ceil_div(S, R);
    long long ns;
    bool several = false;  // blocks per (b,h) from plan_groups
    GroupPlan g{};
    if (nsplit_req > 0) {
        ns = nsplit_req;
    } else {
        ns = ceil_div(tn.target_units, BH);
        // keep at least 4 iterations per unit unless S is short; an under-filled
        // grid (few (b,h)) may still take up to kMaxAutoBlockSplits short chunks,
        // which the one-launch kernel merges on chip
        const long long by_len = std::max<long long>(
            1, std::max(ceil_div(S, 4LL * R), std::min<long long>(kMaxAutoBlockSplits, ceil_div(S, R))));
        ns = std::min(ns, by_len);
        if (ns > kMaxAutoBlockSplits && ns <= kMaxBlockSplits) ns = kMaxAutoBlockSplits;
        // Few (b,h): several blocks each, where that pays for the second launch; reported
        // as 8 chunks per block, and more than kMaxBlockSplits also for two blocks
        if (ns == kMaxAutoBlockSplits && !on_chip && max_split > kMaxBlockSplits) {
            g = plan_groups(BH, S, D, tn.slots, max_split);
            if (g.blocks > 1)
                ns = std::min(max_split, std::max(3LL, (long long)g.blocks) * kGroupWaves);
            several = ns > kMaxBlockSplits;
        }
    }
    ns = std::max<long long>(1, std::min(ns, max_split));
    long long chunk = round_up((size_t)ceil_div(S, ns), (size_t)R);
    if (!several) ns = ceil_div(S, chunk);
    if (ns <= kMaxBlockSplits && use_block_kernel())
        return SplitPlan{(int)ns, (int)chunk, nsplit_req > 0, GroupPlan{1, (int)ns, (int)chunk}, 0};
    if (nsplit_req > 0 || !use_block_kernel())
        return SplitPlan{(int)ns, (int)chunk, nsplit_req > 0, forced_groups((int)ns, (int)chunk), (int)ns};
    if (!several) g = plan_groups(BH, S, D, tn.slots, ns);
    // room for the most blocks, not those picked: it does not shrink with S, so that a
    // workspace sized for the longest sequence serves the shorter ones
    return SplitPlan{(int)ns, (int)chunk, false, g, (int)most_groups(BH, max_split)};
}

struct Int4 {
    int x, y, z, w;
};

__device__ __forceinline__ Int4 load16(const int8_t* p) {
    const int4 v = *reinterpret_cast<const int4*>(p);
    return Int4{v.x, v.y, v.z, v.w};
}

template <bool NT>
__device__ __forceinline__ float load_f32(const float* p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

// Four scales of consecutive rows as one 16-byte load, which needs only the
// alignment of a float.
template <bool NT>
__device__ __forceinline__ void load_scales4(const float* p, float* s) {
    typedef float v4f __attribute__((ext_vector_type(4), aligned(4)));
    v4f v;
    if constexpr (NT) v = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(p));
    else v = *reinterpret_cast<const v4f*>(p);
    s[0] = v.x, s[1] = v.y, s[2] = v.z, s[3] = v.w;
}

template <bool NT>
__device__ __forceinline__ Int4 load_kv16(const int8_t* p) {
    if constexpr (NT) {
        typedef int v4i __attribute__((ext_vector_type(4)));
        const v4i v = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(p));
        return Int4{v.x, v.y, v.z, v.w};
    } else {
        return load16(p);
    }
}

__device__ __forceinline__ void fma_bytes(float* acc, int word, float w) {
    acc[0] = fmaf(w, sbyte_to_f32<0>(word), acc[0]);
    acc[1] = fmaf(w, sbyte_to_f32<1>(word), acc[1]);
    acc[2] = fmaf(w, sbyte_to_f32<2>(word), acc[2]);
    acc[3] = fmaf(w, sbyte_to_f32<3>(word), acc[3]);
}

template <int D>
__device__ __forceinline__ int group_sum(int v) {
    if constexpr (D == 128) return group8_sum(v);
    else return group4_sum(v);
}

// Lane t's value of each 4-lane quad, in every lane of the quad (DPP
// quad_perm [t,t,t,t]); t is a compile-time constant after unrolling.
__device__ __forceinline__ float quad_bcast(float x, int t) {
    const int v = __float_as_int(x);
    switch (t) {
        case 0: return __int_as_float(__builtin_amdgcn_mov_dpp(v, 0x00, 0xF, 0xF, false));
        case 1: return __int_as_float(__builtin_amdgcn_mov_dpp(v, 0x55, 0xF, 0xF, false));
        case 2: return __int_as_float(__builtin_amdgcn_mov_dpp(v, 0xAA, 0xF, 0xF, false));
        default: return __int_as_float(__builtin_amdgcn_mov_dpp(v, 0xFF, 0xF, 0xF, false));
    }
}

// QK^T, online softmax and PV for one wave iteration whose NSLOT rows per
// group are loaded (kv, vv, sk, sv).  MASKED: rows outside [jlo, j1) get score -inf
// and weight 0 (their loads point at some valid row), and sk[t] / sv[t] are slot t's
// scales, as they are unmasked without QUAD.  QUAD: lane s of a quad holds those of
// slots s, s + 4 in sk[0], sk[1] and the quad reads them with quad_bcast.  RS: rows
// between slots (2 for paired rows, the only ones with a jlo).
template <int D, int NS, bool MASKED, int RS = 1, bool QUAD = true>
__device__ __forceinline__ void decode_math(const Int4 (&kv)[NS], const Int4 (&vv)[NS],
                                            const float (&sk)[NS], const float (&sv)[NS],
                                            int row0, int j1, const Int4& q, float qscale,
                                            float& m, float& l, float* acc, int jlo = 0) {
    constexpr bool QB = !MASKED && QUAD;
    // QK^T: exact int32 dot per row, summed over the LPR lanes of the group.
    float sc[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        int d = __builtin_amdgcn_sdot4(q.x, kv[t].x, 0, false);
        d = __builtin_amdgcn_sdot4(q.y, kv[t].y, d, false);
        d = __builtin_amdgcn_sdot4(q.z, kv[t].z, d, false);
        d = __builtin_amdgcn_sdot4(q.w, kv[t].w, d, false);
        d = group_sum<D>(d);
        const float skt = QB ? quad_bcast(sk[t >> 2], t & 3) : sk[t];
        sc[t] = static_cast<float>(d) * qscale * skt;
        if constexpr (MASKED) {
            if (row0 + t * RS >= j1 || (RS == 2 && row0 + t * RS < jlo)) sc[t] = -INFINITY;
        }
    }

    // Online softmax (log2 domain) for this group's NSLOT rows.
    float mx = sc[0];
#pragma unroll
    for (int t = 1; t < NS; ++t) mx = fmaxf(mx, sc[t]);
    const float m_new = fmaxf(m, mx);
    const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
    const float corr = fast_exp2(m - m_use);
    l *= corr;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] *= corr;
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        const float p = fast_exp2(sc[t] - m_use);
        l += p;
        float w = p * (QB ? quad_bcast(sv[t >> 2], t & 3) : sv[t]);
        if constexpr (MASKED) {
            if (row0 + t * RS >= j1 || (RS == 2 && row0 + t * RS < jlo)) w = 0.f;
        }
        fma_bytes(acc + 0, vv[t].x, w);
        fma_bytes(acc + 4, vv[t].y, w);
        fma_bytes(acc + 8, vv[t].z, w);
        fma_bytes(acc + 12, vv[t].w, w);
    }
    m = m_new;
}

// The registers of one wave iteration: NSLOT rows per group of K, V and scales
// (the scales of this lane's slots; see decode_math).
template <int NS>
struct IterBuf {
    Int4 kv[NS], vv[NS];
    float sk[NS], sv[NS];
};

// The loads of an unmasked wave iteration whose group rows start at row0 and
// lie RS rows apart.  QUAD: one scale per lane and 4 slots (see decode_math).  The
// contiguous kernels load consecutive rows' scales as vectors instead: the 16 quad
// reads of an iteration at D = 128 show where a CU has few waves (one chunk of 5000
// rows 69.3 -> 66.9 us, B6 H32 D128 2048 rows 17.2 -> 16.6; the paged D = 128 kernel,
// whose scales are 8 rows of one page, is 1-2% faster with them).
template <int D, int NS, int FL, int RS, bool QUAD>
__device__ __forceinline__ void load_iter(IterBuf<NS>& b, const int8_t* __restrict__ Kbh,
                                          const int8_t* __restrict__ Vbh,
                                          const float* __restrict__ sKbh,
                                          const float* __restrict__ sVbh, size_t row0, int sub) {
    const int8_t* kp = Kbh + (size_t)row0 * D + sub * 16;
    const int8_t* vp = Vbh + (size_t)row0 * D + sub * 16;
#pragma unroll
    for (int t = 0; t < NS; ++t) b.kv[t] = load_kv16<(FL & kNtKV) != 0>(kp + t * RS * D);
#pragma unroll
    for (int t = 0; t < NS; ++t) b.vv[t] = load_kv16<(FL & kNtKV) != 0>(vp + t * RS * D);
    if constexpr (QUAD) {
#pragma unroll
        for (int i = 0; i < NS / 4; ++i) {
            const size_t r = row0 + RS * ((sub & 3) + 4 * i);
            b.sk[i] = load_f32<(FL & kNtScales) != 0>(sKbh + r);
            b.sv[i] = load_f32<(FL & kNtScales) != 0>(sVbh + r);
        }
    } else {
#pragma unroll
        for (int t = 0; t < NS; t += 4) {
            load_scales4<(FL & kNtScales) != 0>(sKbh + row0 + t, &b.sk[t]);
            load_scales4<(FL & kNtScales) != 0>(sVbh + row0 + t, &b.sv[t]);
        }
    }
}

// A partial wave iteration: rows outside [jlo, j1) get score -inf and weight 0
// (their loads are redirected to a row inside).  RS: rows between slots (2 for
// paired rows; jlo is 0 for the others).  What the scores need is loaded before V,
// and all of it before the math (B519 D128 300 rows 17.9 -> 15.7 us).
template <int D, int NS, int FL, int RS = 1>
__device__ __forceinline__ void decode_tail(
    const int8_t* __restrict__ Kbh, const int8_t* __restrict__ Vbh,
    const float* __restrict__ sKbh, const float* __restrict__ sVbh,
    int row0, int jlo, int j1, int sub, const Int4& q, float qscale,
    float& m, float& l, float* acc) {
    IterBuf<NS> b;
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        const int r = RS == 2 ? max(min(row0 + t * RS, j1 - 1), jlo) : min(row0 + t * RS, j1 - 1);
        b.kv[t] = load_kv16<(FL & kNtKV) != 0>(Kbh + (size_t)r * D + sub * 16);
        b.sk[t] = load_f32<(FL & kNtScales) != 0>(sKbh + r);
    }
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        const int r = RS == 2 ? max(min(row0 + t * RS, j1 - 1), jlo) : min(row0 + t * RS, j1 - 1);
        b.vv[t] = load_kv16<(FL & kNtKV) != 0>(Vbh + (size_t)r * D + sub * 16);
        b.sv[t] = load_f32<(FL & kNtScales) != 0>(sVbh + r);
    }
    __builtin_amdgcn_sched_barrier(0);
    decode_math<D, NS, true, RS>(b.kv, b.vv, b.sk, b.sv, row0, j1, q, qscale, m, l, acc, jlo);
}

// Reductions over the row groups of a wave: the lanes with equal sub (lane % LPR,
// LPR = 4 or 8), every lane getting the result.  On the VALU: rotations inside each
// row of 16 lanes, then the row and half swaps (ds_bpermute, which __shfl_xor uses,
// took 72 LDS operations per wave at D = 64: B16 H12 D64 300 rows 5.8 -> 5.4 us,
// B8 H32 D64 2K 13.4 -> 13.0, kernel time).
template <int N>
__device__ __forceinline__ float row_ror(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + N, 0xF, 0xF, false));
}
template <int LPR, typename Op>
__device__ __forceinline__ float groups_reduce(float x, Op op) {
    if constexpr (LPR == 4) x = op(x, row_ror<4>(x));
    x = op(x, row_ror<8>(x));
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return op(__uint_as_float(h[0]), __uint_as_float(h[1]));
}

// Merges the G row-group states of a wave (lanes with equal `sub`) and writes
// the unit's partial state, or with FINAL the normalised fp16 row (a unit that
// saw no rows, L == 0, gives zeros).
template <int D, bool FINAL>
__device__ __forceinline__ void finish_unit(float m, float l, float* acc, int grp, int sub,
                                            int unit, float* __restrict__ part_ml,
                                            float* __restrict__ part_acc,
                                            uint16_t* __restrict__ out) {
    constexpr int LPR = D / 16;
    auto add = [](float a, float b) { return a + b; };
    const float M = groups_reduce<LPR>(m, [](float a, float b) { return fmaxf(a, b); });
    const float f = (m == -INFINITY) ? 0.f : fast_exp2(m - M);
    const float L = groups_reduce<LPR>(l * f, add);
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = groups_reduce<LPR>(acc[e] * f, add);
    if constexpr (FINAL) {
        if (grp == 0) {
            const float inv = L > 0.f ? 1.f / L : 0.f;
            uint16_t h[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) h[e] = __half_as_ushort(f16_of_f32(acc[e] * inv));
            uint4* dst = reinterpret_cast<uint4*>(out + (size_t)unit * D + sub * 16);
            dst[0] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                                h[6] | (h[7] << 16));
            dst[1] = make_uint4(h[8] | (h[9] << 16), h[10] | (h[11] << 16),
                                h[12] | (h[13] << 16), h[14] | (h[15] << 16));
        }
        return;
    }
    if (grp == 0) {
        float4* dst = reinterpret_cast<float4*>(part_acc + (size_t)unit * D + sub * 16);
        dst[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
        dst[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
        dst[2] = make_float4(acc[8], acc[9], acc[10], acc[11]);
        dst[3] = make_float4(acc[12], acc[13], acc[14], acc[15]);
        if (sub == 0) {
            part_ml[2 * (size_t)unit] = M;
            part_ml[2 * (size_t)unit + 1] = L;
        }
    }
}

// The output row of one (b,h) from the merged accumulator (dims lane*D/64 ..
// +D/64 of this lane) and the merged sum L: the fp16 row, or with qout set the
// per-token int8 quantization of that fp16 row (codes and scale as
// int8k_quantize_per_token gives for it).  A whole wave calls it.
template <int D>
__device__ __forceinline__ void emit_row(const float (&acc)[D / 64], float L, int lane, int bh,
                                         uint16_t* __restrict__ out, int8_t* __restrict__ qout,
                                         float* __restrict__ qscale) {
    constexpr int DPL = D / 64;
    const float inv = L > 0.f ? 1.f / L : 0.f;  // no rows at all (empty sequence): zeros
    float y[DPL];
#pragma unroll
    for (int i = 0; i < DPL; ++i) y[i] = __half2float(f16_of_f32(acc[i] * inv));
    if (qout != nullptr) {
        float am = 0.f;
#pragma unroll
        for (int i = 0; i < DPL; ++i) am = fmaxf(am, fabsf(y[i]));
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) am = fmaxf(am, __shfl_xor(am, off));
        const float sc = fmaxf(am, 1e-8f) / 127.f;
#pragma unroll
        for (int i = 0; i < DPL; ++i)
            qout[(size_t)bh * D + lane * DPL + i] = (int8_t)quant_code(y[i], sc);
        if (lane == 0) qscale[bh] = sc;
        return;
    }
#pragma unroll
    for (int i = 0; i < DPL; ++i)
        out[(size_t)bh * D + lane * DPL + i] = __half_as_ushort(__float2half_rn(y[i]));
}

// Pass 2: one block per bh merges its n partial states into the output row.
// The partials come from other XCDs' writes (a full memory round trip each), so
// the block's 4 waves take every fourth partial, 8 loads in flight per wave, and
// merge in LDS: at n = 235 one wave alone took 15.2 us.
template <int D>
__global__ __launch_bounds__(kBlockThreads) void decode_combine_kernel(
    const float* __restrict__ part_ml, const float* __restrict__ part_acc,
    uint16_t* __restrict__ out, int8_t* __restrict__ qout, float* __restrict__ qscale, int n) {
    constexpr int DPL = D / 64;  // dims per lane
    __shared__ float s_acc[kWavesPerBlock][D];
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int bh = blockIdx.x;
    const float2* ml = reinterpret_cast<const float2*>(part_ml) + (size_t)bh * n;

    float M = -INFINITY;
    for (int s = lane; s < n; s += 64) M = fmaxf(M, ml[s].x);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) M = fmaxf(M, __shfl_xor(M, off));
    const float M_use = (M == -INFINITY) ? 0.f : M;

    float L = 0.f;
    for (int s = lane; s < n; s += 64) L += ml[s].y * fast_exp2(ml[s].x - M_use);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) L += __shfl_xor(L, off);

    float acc[DPL];
#pragma unroll
    for (int i = 0; i < DPL; ++i) acc[i] = 0.f;
    const float* pa = part_acc + (size_t)bh * n * D + lane * DPL;
#pragma unroll 8
    for (int s = w; s < n; s += kWavesPerBlock) {
        const float wt = fast_exp2(ml[s].x - M_use);
#pragma unroll
        for (int i = 0; i < DPL; ++i) acc[i] = fmaf(pa[(size_t)s * D + i], wt, acc[i]);
    }
#pragma unroll
    for (int i = 0; i < DPL; ++i) s_acc[w][lane * DPL + i] = acc[i];
    __syncthreads();
    if (w != 0) return;
#pragma unroll
    for (int i = 0; i < DPL; ++i)
#pragma unroll
        for (int v = 1; v < kWavesPerBlock; ++v) acc[i] += s_acc[v][lane * DPL + i];
    emit_row<D>(acc, L, lane, bh, out, qout, qscale);
}

// The n_full whole iterations of a wave's chunk, starting at iteration `it` and
// wrapping around.  roff(i): the row offset (from the K/V/scale bases) of the
// group's first row in iteration i; RS: rows between its slots.  PIPE: two
// register sets, iteration k+1's loads issued before iteration k is computed
// (the fences keep the compiler from sinking them).
template <int D, int NS, int FL, bool PIPE, int RS, bool QUAD, typename RowOff>
__device__ __forceinline__ void walk_iters(const int8_t* __restrict__ K,
                                           const int8_t* __restrict__ V,
                                           const float* __restrict__ sK,
                                           const float* __restrict__ sV, RowOff roff, int n_full,
                                           int it, int sub, const Int4& q, float qscale, float& m,
                                           float& l, float* acc) {
    auto nxt = [&](int i) { return (i + 1 == n_full) ? 0 : i + 1; };
    auto load = [&](IterBuf<NS>& b, int i) {
        load_iter<D, NS, FL, RS, QUAD>(b, K, V, sK, sV, roff(i), sub);
    };
    auto math = [&](const IterBuf<NS>& b) {
        decode_math<D, NS, false, RS, QUAD>(b.kv, b.vv, b.sk, b.sv, 0, 0, q, qscale, m, l, acc);
    };
    if constexpr (PIPE) {
        IterBuf<NS> ba, bb;
        if (n_full > 0) load(ba, it);
        int k = 0;
        for (; k + 2 < n_full; k += 2) {
            const int it1 = nxt(it);
            load(bb, it1);
            __builtin_amdgcn_sched_barrier(0);
            math(ba);
            it = nxt(it1);
            load(ba, it);
            __builtin_amdgcn_sched_barrier(0);
            math(bb);
        }
        if (n_full - k == 2) {
            load(bb, nxt(it));
            __builtin_amdgcn_sched_barrier(0);
            math(ba);
            math(bb);
        } else if (n_full - k == 1) {
            math(ba);
        }
    } else {
        for (int k = 0; k < n_full; ++k) {
            IterBuf<NS> b;
            load(b, it);
            math(b);
            it = nxt(it);
        }
    }
}

// The end of a one-launch block: each wave merges its row groups (lanes with
// equal `sub`) and leaves (M, L, acc[D]) in LDS; wave 0 merges the nw chunk
// states with the log-sum-exp rule, as decode_combine_kernel, and writes row
// `bh`, or with part_ml set the merged state as partial `bh`.  Every wave of
// the block calls it (it holds the block's barrier).
template <int D, int MAXW>
__device__ __forceinline__ void merge_block(float m, float l, float* acc, int lane, int grp,
                                            int sub, int w, int nw, int bh,
                                            float (&s_ml)[MAXW][2], float (&s_acc)[MAXW][D],
                                            uint16_t* __restrict__ out,
                                            int8_t* __restrict__ qout,
                                            float* __restrict__ qscale,
                                            float* __restrict__ part_ml = nullptr,
                                            float* __restrict__ part_acc = nullptr) {
    constexpr int LPR = D / 16;
    auto add = [](float a, float b) { return a + b; };
    const float M = groups_reduce<LPR>(m, [](float a, float b) { return fmaxf(a, b); });
    const float f = (m == -INFINITY) ? 0.f : fast_exp2(m - M);
    const float Lw = groups_reduce<LPR>(l * f, add);
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = groups_reduce<LPR>(acc[e] * f, add);
    if (grp == 0) {
        float4* dst = reinterpret_cast<float4*>(&s_acc[w][sub * 16]);
        dst[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
        dst[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
        dst[2] = make_float4(acc[8], acc[9], acc[10], acc[11]);
        dst[3] = make_float4(acc[12], acc[13], acc[14], acc[15]);
        if (sub == 0) {
            s_ml[w][0] = M;
            s_ml[w][1] = Lw;
        }
    }
    __syncthreads();
    if (w != 0) return;
    constexpr int DPL = D / 64;
    // The reads are unrolled, so that those of all chunks go out together.  A shorter
    // sequence has fewer chunks; the absent ones are empty states (another chunk's with
    // weight 0 may hold infinities), set in registers: left in LDS by the waves they cost
    // a one-chunk block 0.2 us, and a loop over the chunks 0.2 us at five (300 rows).
    float Mall, L = 0.f, o[DPL];
    auto merge = [&](auto full) {
        constexpr int N = decltype(full)::value ? MAXW : MAXW - 1;
        float mc[N], lc[N], oc[N][DPL];
#pragma unroll
        for (int c = 0; c < N; ++c) {
            mc[c] = -INFINITY, lc[c] = 0.f;
#pragma unroll
            for (int i = 0; i < DPL; ++i) oc[c][i] = 0.f;
        }
#pragma unroll
        for (int c = 0; c < N; ++c) {
            if (!decltype(full)::value && c >= nw) break;
            mc[c] = s_ml[c][0];
            lc[c] = s_ml[c][1];
#pragma unroll
            for (int i = 0; i < DPL; ++i) oc[c][i] = s_acc[c][lane * DPL + i];
        }
        Mall = mc[0];
#pragma unroll
        for (int c = 1; c < N; ++c) Mall = fmaxf(Mall, mc[c]);
        const float M_use = (Mall == -INFINITY) ? 0.f : Mall;
#pragma unroll
        for (int i = 0; i < DPL; ++i) o[i] = 0.f;
#pragma unroll
        for (int c = 0; c < N; ++c) {
            const float wt = fast_exp2(mc[c] - M_use);
            L += lc[c] * wt;
#pragma unroll
            for (int i = 0; i < DPL; ++i) o[i] = fmaf(oc[c][i], wt, o[i]);
        }
    };
    if (nw == MAXW) merge(std::true_type{});
    else merge(std::false_type{});
    if (part_ml != nullptr) {
#pragma unroll
        for (int i = 0; i < DPL; ++i) part_acc[(size_t)bh * D + lane * DPL + i] = o[i];
        if (lane == 0) {
            part_ml[2 * (size_t)bh] = Mall;
            part_ml[2 * (size_t)bh + 1] = L;
        }
        return;
    }
    emit_row<D>(o, L, lane, bh, out, qout, qscale);
}

// One launch for plans of at most kMaxBlockSplits chunks per (b,h): block bh
// runs one wave per chunk (blockDim.x / 64 waves), each wave walks its chunk as
// above, merges its row groups and leaves (m, l, acc[D]) in
// LDS; wave 0 then merges the chunks with the log-sum-exp rule and writes the
// row.  No partial state leaves the chip and there is no second launch.
// MAXW: the most waves the instance is launched with (8 or kMaxBlockSplits).
// The 8-wave instance has twice the registers per wave, which lets it keep the
// next iteration's loads in flight (a second register set, two_sets) while the
// current one computes: at 4 slots a short chunk is only a few dependent load
// rounds, so their latency would show; at D = 128 with 8 slots (204 VGPRs, two
// waves per SIMD) the stream then runs at fewer waves per CU with the same
// bytes in flight, which the HBM read rate prefers.
//
// GROUP (plans of more than kMaxBlockSplits chunks): nb blocks per (b,h), block
// bh * nb + g taking chunks g * waves .. of the (b,h) and leaving their merged
// state as one partial for decode_combine_kernel.  Few (b,h) with long contexts
// run here: against one wave per partial (one register set, grouped rows, 235
// partials per (b,h)) B2 H8 D128 60013 rows of a 64K cache took 60.4 ->
// 43.8 us.
template <int D, int NS, int FL, int MAXW, bool GROUP>
__global__ __launch_bounds__(64 * MAXW) void decode_block_kernel(
    const int8_t* __restrict__ Q, const int8_t* __restrict__ K,
    const int8_t* __restrict__ V, const float* __restrict__ sQ,
    const float* __restrict__ sK, const float* __restrict__ sV, uint16_t* __restrict__ out,
    int8_t* __restrict__ qout, float* __restrict__ qscale, int S, int S_cap, int chunk,
    float qk_scale_log2, int stagger, int nb, float* __restrict__ part_ml,
    float* __restrict__ part_acc) {
    using G = DecodeGeom<D, NS>;
    constexpr int LPR = D / 16;
    __shared__ float s_ml[MAXW][2];
    __shared__ __align__(16) float s_acc[MAXW][D];
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
    const int bh = GROUP ? (int)(blockIdx.x / (unsigned)nb) : (int)blockIdx.x;
    const int c = GROUP ? ((int)blockIdx.x - bh * nb) * nw + w : w;  // chunk of this wave
    const int sub = lane % LPR;
    const int grp = lane / LPR;
    constexpr bool PAIRED = paired_rows(D, NS, MAXW);
    constexpr int RS = PAIRED ? 2 : 1;

    const Int4 q = load16(Q + (size_t)bh * D + sub * 16);
    const float qscale_l = sQ[bh] * qk_scale_log2;
    // Paired rows need the block rows 8h.. to start on a 128-byte line.  Where an odd
    // row stride puts the (b,h)'s first 64-byte row in the middle of one, rows are
    // counted from the row before it (jlo = 1: that row, the last of the previous
    // (b,h), is never used), and the last chunk may run one row past its length.
    const size_t row_bh = (size_t)bh * S_cap;
    const int jlo =
        PAIRED && bh > 0 ? (int)((reinterpret_cast<uintptr_t>(K + row_bh * D) >> 6) & 1) : 0;
    const int8_t* Kbh = K + (row_bh - jlo) * D;
    const int8_t* Vbh = V + (row_bh - jlo) * D;
    const float* sKbh = sK + (row_bh - jlo);
    const float* sVbh = sV + (row_bh - jlo);
    const int end = S + jlo;
    const int j0 = (int)min((long long)c * chunk, (long long)end);
    const bool last = c == nb * nw - 1;
    const int j1 = last ? end : min(end - j0, chunk) + j0;

    float m = -INFINITY, l = 0.f;
    float acc[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.f;
    const int g0 = group_row0<PAIRED, NS>(grp);
    // the first iteration of a (b,h) counted from the row before it is partial
    const int head = (PAIRED && c == 0 && jlo != 0) ? min(G::kRowsPerIter, j1) : 0;
    const int n_full = max(0, j1 - j0 - head) / G::kRowsPerIter;
    const unsigned unit = blockIdx.x * (unsigned)nw + (unsigned)w;
    const int it = stagger ? (int)((unit * 2654435761u) >> 16) % max(n_full, 1) : 0;
    const int jf = j0 + head;
    walk_iters<D, NS, FL, two_sets(D, NS, MAXW), RS, PAIRED>(
        Kbh, Vbh, sKbh, sVbh, [&](int i) { return (size_t)(jf + i * G::kRowsPerIter + g0); },
        n_full, it, sub, q, qscale_l, m, l, acc);
    // partial iterations: the end of the chunk, and the head
    int base = jf + n_full * G::kRowsPerIter, stop = j1;
    for (int part = 0; part < 2; ++part) {
        if (base < stop)
            decode_tail<D, NS, FL, RS>(Kbh, Vbh, sKbh, sVbh, base + g0, jlo, stop, sub, q,
                                       qscale_l, m, l, acc);
        if (!PAIRED || head == 0) break;
        base = 0;
        stop = head;
    }
    merge_block<D, MAXW>(m, l, acc, lane, grp, sub, w, nw, GROUP ? (int)blockIdx.x : bh, s_ml,
                         s_acc, out, qout, qscale, GROUP ? part_ml : nullptr, part_acc);
}

// Paged variant of decode_block_kernel: a block first copies the page ids of
// its rows (clamped to [0, num_pages)) into LDS, so that each iteration's row
// offset is an LDS read instead of a global load in front of its K/V loads; then
// it walks and merges its chunks as decode_block_kernel.  GROUP: nb blocks per
// (b,h), the (b,h) index fastest in the grid; a block past the end of its
// sequence leaves an empty partial.  n_tab: page ids a block's rows can span.
template <int D, int NS, int FL, int MAXW, bool GROUP>
__global__ __launch_bounds__(64 * MAXW) void decode_paged_block_kernel(
    const int8_t* __restrict__ Q, const int8_t* __restrict__ Kp,
    const int8_t* __restrict__ Vp, const float* __restrict__ sQ,
    const float* __restrict__ sKp, const float* __restrict__ sVp,
    const int32_t* __restrict__ block_tables, const int32_t* __restrict__ context_lens,
    uint16_t* __restrict__ out, int8_t* __restrict__ qout, float* __restrict__ qscale, int BH,
    int H, int num_pages, int log2_page, int max_pages, int n_tab, int chunk,
    float qk_scale_log2, int stagger, int nb, float* __restrict__ part_ml,
    float* __restrict__ part_acc) {
    using G = DecodeGeom<D, NS>;
    constexpr int LPR = D / 16;
    extern __shared__ int s_pages[];
    __shared__ float s_ml[MAXW][2];
    __shared__ __align__(16) float s_acc[MAXW][D];
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
    const int g = GROUP ? (int)(blockIdx.x / (unsigned)BH) : 0;
    int bh = (int)blockIdx.x - g * BH;
    // With 16-token pages a head's scales in a page are 64 bytes, and heads 2k
    // and 2k+1 share one 128-byte line.  Blocks go to the 8 XCDs in turn, so
    // with 16 | BH block i of XCD x takes head pair 8 (i / 2) + x: the
    // pair's two heads run at adjacent slots of one XCD (one L2) and walk their
    // pages in the same order (one stagger), and the line is fetched once.
    const bool pair = log2_page < 5 && (BH & 15) == 0;
    if (pair) {
        const int x = bh & 7, i = bh >> 3;
        bh = ((((i >> 1) << 3) + x) << 1) + (i & 1);
    }
    const int b = bh / H, hh = bh - b * H;
    const int page = 1 << log2_page;
    const int32_t* table = block_tables + (size_t)b * max_pages;
    const long long c0 = (long long)g * nw;  // first chunk of the block
    const int p0 = GROUP ? (int)min(c0 * chunk >> log2_page, (long long)max_pages) : 0;
    // the first id of every thread and the query go out beside the length's load
    const int t = (int)threadIdx.x, nt = (int)blockDim.x;
    int id = table[min(p0 + min(t, n_tab - 1), max_pages - 1)];
    const int sub = lane % LPR;
    const int grp = lane / LPR;
    const Int4 q = load16(Q + (size_t)bh * D + sub * 16);
    const float qscale_l = sQ[bh] * qk_scale_log2;
    const int len =
        (int)min((long long)context_lens[b], (long long)max_pages << log2_page);
    const int used = min(((len + page - 1) >> log2_page) - p0, n_tab);  // entries past it: not used
    bool bad = false;
    for (int i = t; i < used; i += nt) {
        if (i != t) id = table[p0 + i];
        bad |= (unsigned)id >= (unsigned)num_pages;
        s_pages[i] = (int)min((unsigned)id, (unsigned)(num_pages - 1));
    }
    if (__syncthreads_or(bad) && threadIdx.x == 0)
        __hip_atomic_fetch_add(&g_paged_bad_ids, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int j0 = (int)min((c0 + w) * chunk, (long long)max(len, 0));
    const int j1 = min(len - j0, chunk) + j0;
    // row offset (in rows of the page arrays) of position r of this head
    auto row_off = [&](int r) -> size_t {
        return ((size_t)s_pages[(r >> log2_page) - p0] * H + hh) * page + (r & (page - 1));
    };

    float m = -INFINITY, l = 0.f;
    float acc[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.f;
    const int n_full = max(0, j1 - j0) / G::kRowsPerIter;
    const unsigned unit =
        ((unsigned)(pair ? bh >> 1 : bh) * (GROUP ? (unsigned)nb : 1u) + (unsigned)g) *
            (unsigned)nw + (unsigned)w;
    const int it = stagger ? (int)((unit * 2654435761u) >> 16) % max(n_full, 1) : 0;
    // a group's rows (NS-aligned, or the 8-aligned pair block) share one page
    constexpr bool PAIRED = paired_rows(D, NS, MAXW);
    constexpr int RS = PAIRED ? 2 : 1;
    const int g0 = group_row0<PAIRED, NS>(grp);
    walk_iters<D, NS, FL, two_sets(D, NS, MAXW), RS, true>(
        Kp, Vp, sKp, sVp, [&](int i) { return row_off(j0 + i * G::kRowsPerIter + g0); },
        n_full, it, sub, q, qscale_l, m, l, acc);
    const int base = j0 + n_full * G::kRowsPerIter;
    if (base < j1) {
        const int row0 = base + g0;
        IterBuf<NS> bt;
#pragma unroll
        for (int t = 0; t < NS; ++t) {
            const size_t r = row_off(min(row0 + t * RS, j1 - 1));
            bt.kv[t] = load_kv16<(FL & kNtKV) != 0>(Kp + r * D + sub * 16);
            bt.sk[t] = load_f32<(FL & kNtScales) != 0>(sKp + r);
        }
#pragma unroll
        for (int t = 0; t < NS; ++t) {
            const size_t r = row_off(min(row0 + t * RS, j1 - 1));
            bt.vv[t] = load_kv16<(FL & kNtKV) != 0>(Vp + r * D + sub * 16);
            bt.sv[t] = load_f32<(FL & kNtScales) != 0>(sVp + r);
        }
        __builtin_amdgcn_sched_barrier(0);
        decode_math<D, NS, true, RS>(bt.kv, bt.vv, bt.sk, bt.sv, row0, j1, q, qscale_l, m, l,
                                     acc);
    }
    merge_block<D, MAXW>(m, l, acc, lane, grp, sub, w, nw, GROUP ? bh * nb + g : bh, s_ml, s_acc,
                         out, qout, qscale, GROUP ? part_ml : nullptr, part_acc);
}

// Paged variant of pass 1.  Unit = (b, h, split) as above, over positions
// [j0, j1) of sequence b (j1 <= context_lens[b]).  A group's NSLOT rows are
// NSLOT-aligned and page_size is a multiple of NSLOT, so they sit in one
// page: one table lookup per group per iteration, then the same immediate
// slot offsets as the contiguous kernel.  Page p of head h holds
// K/V [p][h][page_size][D] and scales [p][h][page_size].  FL: the
// non-temporal load flags of the contiguous kernel's tuning for this D.
template <int D, int NS, bool FINAL, int FL>
__global__ __launch_bounds__(kBlockThreads) void decode_paged_kernel(
    const int8_t* __restrict__ Q, const int8_t* __restrict__ Kp,
    const int8_t* __restrict__ Vp, const float* __restrict__ sQ,
    const float* __restrict__ sKp, const float* __restrict__ sVp,
    const int32_t* __restrict__ block_tables, const int32_t* __restrict__ context_lens,
    float* __restrict__ part_ml, float* __restrict__ part_acc, uint16_t* __restrict__ out,
    int H, int num_pages, int log2_page, int max_pages, int nsplit, int chunk, int units,
    float qk_scale_log2, int stagger) {
    using G = DecodeGeom<D, NS>;
    const int lane = threadIdx.x & 63;
    const int unit = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (unit >= units) return;  // whole wave exits; no block barrier below
    const int bh = unit / nsplit;
    const int sp = unit - bh * nsplit;
    const int b = bh / H, hh = bh - b * H;
    const int page = 1 << log2_page;
    const int len = min(context_lens[b], max_pages << log2_page);
    const int j0 = sp * chunk;
    const int j1 = min(len, j0 + chunk);

    const int sub = lane % G::kLanesPerRow;
    const int grp = lane / G::kLanesPerRow;
    const Int4 q = load16(Q + (size_t)bh * D + sub * 16);
    const float qscale = sQ[bh] * qk_scale_log2;
    const int32_t* table = block_tables + (size_t)b * max_pages;
    // element offset of row r of this head (an id outside [0, num_pages) reads the last page
    // and is counted)
    bool bad = false;
    auto row_off = [&](int r) -> size_t {
        const int id = table[r >> log2_page];
        bad |= (unsigned)id >= (unsigned)num_pages;
        const int pg = min((unsigned)id, (unsigned)(num_pages - 1));
        return ((size_t)pg * H + hh) * page + (r & (page - 1));
    };

    float m = -INFINITY, l = 0.f;
    float acc[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.f;
    const int n_full = max(0, j1 - j0) / G::kRowsPerIter;
    // Iterations start at a unit-dependent rotation (stagger), and the page id of
    // the next iteration is looked up while the current one computes, so the
    // table load is not a dependent load in front of every iteration's K/V loads.
    int it = stagger ? (int)(((unsigned)unit * 2654435761u) >> 16) % max(n_full, 1) : 0;
    size_t r_next = n_full > 0 ? row_off(j0 + it * G::kRowsPerIter + grp * NS) : 0;
    for (int k = 0; k < n_full; ++k) {
        const size_t r0 = r_next;
        it = (it + 1 == n_full) ? 0 : it + 1;
        if (k + 1 < n_full) r_next = row_off(j0 + it * G::kRowsPerIter + grp * NS);
        IterBuf<NS> b;
        load_iter<D, NS, FL, 1, true>(b, Kp, Vp, sKp, sVp, r0, sub);
        decode_math<D, NS, false>(b.kv, b.vv, b.sk, b.sv, 0, 0, q, qscale, m, l, acc);
    }
    const int base = j0 + n_full * G::kRowsPerIter;
    if (base < j1) {
        const int row0 = base + grp * NS;
        Int4 kv[NS], vv[NS];
        float sk[NS], sv[NS];
#pragma unroll
        for (int t = 0; t < NS; ++t) {
            const size_t r = row_off(min(row0 + t, j1 - 1));
            kv[t] = load_kv16<(FL & kNtKV) != 0>(Kp + r * D + sub * 16);
            vv[t] = load_kv16<(FL & kNtKV) != 0>(Vp + r * D + sub * 16);
            sk[t] = load_f32<(FL & kNtScales) != 0>(sKp + r);
            sv[t] = load_f32<(FL & kNtScales) != 0>(sVp + r);
        }
        decode_math<D, NS, true>(kv, vv, sk, sv, row0, j1, q, qscale, m, l, acc);
    }
    if (__ballot(bad) != 0 && lane == 0)
        __hip_atomic_fetch_add(&g_paged_bad_ids, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    finish_unit<D, FINAL>(m, l, acc, grp, sub, unit, part_ml, part_acc, out);
}

struct DecodeWorkspace {
    float* part_ml;
    float* part_acc;
    size_t bytes;
};

DecodeWorkspace carve(void* ws, long long units, int D) {
    const size_t ml_bytes = round_up((size_t)units * 2 * sizeof(float), kWorkspaceAlign);
    const size_t acc_bytes = round_up((size_t)units * D * sizeof(float), kWorkspaceAlign);
    char* p = static_cast<char*>(ws);
    return DecodeWorkspace{reinterpret_cast<float*>(p), reinterpret_cast<float*>(p + ml_bytes),
                           ml_bytes + acc_bytes};
}

// Where a decode writes its rows: fp16 `f16`, or int8 `q` + per-row scale `qs`.
struct DecodeOut {
    uint16_t* f16;
    int8_t* q;
    float* qs;
};

// The arguments of a contiguous decode.
struct DecodeArgs {
    const int8_t *Q, *K, *V;
    const float *sQ, *sK, *sV;
    int BH, S, S_cap;
    float qk;
};

// The 8-wave instance takes the paired-row load flags where it pairs rows.
template <int D, int NS, int MAXW, bool GROUP>
void launch_block(const DecodeTuning& tn, const DecodeArgs& a, const DecodeOut& o,
                  const GroupPlan& g, const DecodeWorkspace& w, hipStream_t stream) {
    const int flags = paired_rows(D, NS, MAXW) ? tn.pair_flags : tn.flags;
    const unsigned blocks = (unsigned)a.BH * (unsigned)g.blocks;
#define INT8K_BLOCK_LAUNCH(FLV)                                                                 \
    decode_block_kernel<D, NS, FLV, MAXW, GROUP><<<blocks, 64 * g.waves, 0, stream>>>(          \
        a.Q, a.K, a.V, a.sQ, a.sK, a.sV, o.f16, o.q, o.qs, a.S, a.S_cap, g.chunk, a.qk,         \
        tn.stagger, g.blocks, w.part_ml, w.part_acc)
    switch (flags & 3) {
        case 0: INT8K_BLOCK_LAUNCH(0); break;
        case 1: INT8K_BLOCK_LAUNCH(1); break;
        case 2: INT8K_BLOCK_LAUNCH(2); break;
        default: INT8K_BLOCK_LAUNCH(3); break;
    }
#undef INT8K_BLOCK_LAUNCH
}

template <int D>
int launch_decode(const DecodeArgs& a, const DecodeOut& o, const SplitPlan& plan,
                  const DecodeWorkspace& w, hipStream_t stream) {
    const DecodeTuning tn = tuning_for(D);
    // f(slots) with the slot count as a compile-time constant
    auto with_ns = [&](auto&& f) {
        if (tn.slots == 4) f(std::integral_constant<int, 4>{});
        else f(std::integral_constant<int, 8>{});
    };
    const GroupPlan& g = plan.g;
    const bool group = g.blocks > 1 || !use_block_kernel();
    with_ns([&](auto ns) {
        if (group)
            launch_block<D, ns.value, kGroupWaves, true>(tn, a, o, g, w, stream);
        else if (g.waves <= kGroupWaves)  // one launch: the waves of one block
            launch_block<D, ns.value, kGroupWaves, false>(tn, a, o, g, w, stream);
        else
            launch_block<D, ns.value, kMaxBlockSplits, false>(tn, a, o, g, w, stream);
    });
    int st = check_launch("decode_block_kernel");
    if (st != INT8K_OK || !group) return st;
    decode_combine_kernel<D><<<(unsigned)a.BH, kBlockThreads, 0, stream>>>(
        w.part_ml, w.part_acc, o.f16, o.q, o.qs, g.blocks);
    return check_launch("decode_combine_kernel");
}

template <int D>
int launch_decode_paged(const int8_t* Q, const int8_t* Kp, const int8_t* Vp, const DecodeOut& o,
                        const float* sQ, const float* sKp, const float* sVp,
                        const int32_t* tables, const int32_t* lens, int B, int H,
                        int num_pages, int log2_page, int max_pages, int max_context,
                        const SplitPlan& plan, const DecodeWorkspace& w, hipStream_t stream) {
    uint16_t* out = o.f16;
    const int BH = B * H;
    const long long units = (long long)BH * plan.nsplit;
    const float qk = (1.0f / std::sqrt((float)D)) * kLog2e;
    const dim3 grid((unsigned)ceil_div(units, kWavesPerBlock));
    constexpr int NS = D == 128 ? 8 : 4;
    const DecodeTuning tn = tuning_for(D);
    const bool one_launch = plan.nsplit <= kGroupWaves && use_block_kernel();
    GroupPlan g;
    if (plan.forced || !use_block_kernel())
        g = plan.g;
    else
        g = plan_groups(BH, max_context, D, NS, plan.nsplit);
    // Short chunks keep the plan's waves: more of them only add merges, and blocks where
    // the (b,h) fill the GPU (page 64, ragged: B32 H32 D64 1000 rows 15.9 us on the
    // plan's 2 waves and 20.1 on 8, B20 H32 1500 rows 16.6 and 20.5 on 4 and 8, B64 H32
    // D128 1500 rows 80 and 89 on 4 and 8).  Past about 32 iterations, or 128 / waves,
    // 8 waves are the faster (B24 H16 D64 2048 rows 19.1 us on 6, 18.3 on 8; B20 H32 4000
    // rows 40.5 on 4, 36.2 on 8).
    const long long iters = ceil_div(max_context, rows_per_iter(D, NS));
    if (g.blocks == 1 && one_launch &&
        (plan.chunk <= 4 * rows_per_iter(D, NS) ||
         (iters <= 4 * kGroupWaves && iters * plan.nsplit <= 16 * kGroupWaves)))
        g = GroupPlan{1, plan.nsplit, plan.chunk};
    // page ids the rows of a block can span, staged in LDS
    const long long rows = (long long)g.waves * g.chunk;
    const long long n_tab = std::min<long long>(
        max_pages, g.blocks == 1 ? ceil_div(rows, 1LL << log2_page) : ((rows - 1) >> log2_page) + 2);
    if (n_tab * 4 <= kPagedLdsTableBytes && (long long)BH * g.blocks * g.waves < (1LL << 26)) {
        const size_t lds = (size_t)n_tab * 4;
        const unsigned blocks = (unsigned)BH * (unsigned)g.blocks;
        const bool group = !(g.blocks == 1 && use_block_kernel());
#define INT8K_PAGED_BLOCK(FLV, GR)                                                          \
    decode_paged_block_kernel<D, NS, FLV, 8, GR><<<blocks, 64 * g.waves, lds, stream>>>(    \
        Q, Kp, Vp, sQ, sKp, sVp, tables, lens, out, o.q, o.qs, BH, H, num_pages, log2_page, \
        max_pages, (int)n_tab, g.chunk, qk, tn.stagger, g.blocks, w.part_ml, w.part_acc)
#define INT8K_PAGED_BLOCK2(FLV)             \
    if (group) INT8K_PAGED_BLOCK(FLV, true); \
    else INT8K_PAGED_BLOCK(FLV, false)
        switch ((paired_rows(D, NS, 8) ? tn.pair_flags : tn.flags) & 3) {
            case 0: INT8K_PAGED_BLOCK2(0); break;
            case 1: INT8K_PAGED_BLOCK2(1); break;
            case 2: INT8K_PAGED_BLOCK2(2); break;
            default: INT8K_PAGED_BLOCK2(3); break;
        }
#undef INT8K_PAGED_BLOCK2
#undef INT8K_PAGED_BLOCK
        int st = check_launch("decode_paged_block_kernel");
        if (st != INT8K_OK || !group) return st;
        decode_combine_kernel<D><<<(unsigned)BH, kBlockThreads, 0, stream>>>(
            w.part_ml, w.part_acc, out, o.q, o.qs, g.blocks);
        return check_launch("decode_combine_kernel");
    }
    const bool final_pass = plan.nsplit == 1 && out != nullptr && aligned_to(out, 16);
#define INT8K_PAGED_LAUNCH(FIN, FLV)                                                     \
    decode_paged_kernel<D, NS, FIN, FLV><<<grid, kBlockThreads, 0, stream>>>(            \
        Q, Kp, Vp, sQ, sKp, sVp, tables, lens, w.part_ml, w.part_acc, out, H, num_pages, \
        log2_page, max_pages, plan.nsplit, plan.chunk, (int)units, qk, tuning_for(D).stagger)
#define INT8K_PAGED_FLAGS(FIN)                          \
    switch (tuning_for(D).flags & 3) {                  \
        case 0: INT8K_PAGED_LAUNCH(FIN, 0); break;      \
        case 1: INT8K_PAGED_LAUNCH(FIN, 1); break;      \
        case 2: INT8K_PAGED_LAUNCH(FIN, 2); break;      \
        default: INT8K_PAGED_LAUNCH(FIN, 3); break;     \
    }
    if (final_pass) {
        INT8K_PAGED_FLAGS(true)
    } else {
        INT8K_PAGED_FLAGS(false)
    }
#undef INT8K_PAGED_FLAGS
#undef INT8K_PAGED_LAUNCH
    int st = check_launch("decode_paged_kernel");
    if (st != INT8K_OK || final_pass) return st;
    decode_combine_kernel<D><<<(unsigned)BH, kBlockThreads, 0, stream>>>(
        w.part_ml, w.part_acc, out, o.q, o.qs, plan.nsplit);
    return check_launch("decode_combine_kernel");
}

}  // namespace
}  // namespace int8k

using namespace int8k;

extern "C" int int8k_decode_attention_num_splits(int BH, int S, int head_dim, int nsplit) {
    if (BH <= 0 || S <= 0 || (head_dim != 64 && head_dim != 128)) return 0;
    return plan_splits(BH, S, head_dim, nsplit).nsplit;
}

// Workspace a contiguous-cache decode with this plan needs: m, l and acc[D] per partial.
static size_t decode_partial_bytes(const SplitPlan& plan, long long BH, int D) {
    return plan.partials > 0 ? carve(nullptr, BH * plan.partials, D).bytes : 0;
}

extern "C" size_t int8k_decode_attention_workspace_bytes(int BH, int S, int head_dim, int nsplit) {
    if (BH <= 0 || S <= 0 || (head_dim != 64 && head_dim != 128)) return 0;
    return decode_partial_bytes(plan_splits(BH, S, head_dim, nsplit), BH, head_dim);
}

// The call's plan with `have` bytes of workspace: an automatic plan whose partials do
// not fit falls back to one block per (b,h) where its chunks merge on chip.
static SplitPlan plan_within(int BH, int S, int D, int nsplit, size_t have) {
    const SplitPlan plan = plan_splits(BH, S, D, nsplit);
    if (plan.forced || have >= decode_partial_bytes(plan, BH, D)) return plan;
    const SplitPlan small = plan_splits(BH, S, D, 0, true);
    return small.partials == 0 ? small : plan;
}

size_t int8k::decode_partials_within(int BH, int S, int head_dim, int nsplit, size_t have) {
    return decode_partial_bytes(plan_within(BH, S, head_dim, nsplit, have), BH, head_dim);
}

static bool out_ok(const DecodeOut& o) {
    return o.f16 ? aligned_to(o.f16, 2) : (o.q != nullptr && o.qs != nullptr && aligned_to(o.qs, 4));
}

static int decode_impl(const int8_t* Q, const int8_t* K, const int8_t* V, const DecodeOut& out,
                       const float* scale_Q, const float* scale_K, const float* scale_V, int BH,
                       int S, int S_cap, int head_dim, int nsplit, void* workspace,
                       size_t workspace_bytes, void* stream) {
    clear_last_error();
    if (!Q || !K || !V || !(out.f16 || out.q) || !scale_Q || !scale_K || !scale_V)
        return INT8K_ERR_INVALID_ARGUMENT;
    if (BH <= 0 || S <= 0 || S_cap < S || nsplit < 0) return INT8K_ERR_INVALID_ARGUMENT;
    if (head_dim != 64 && head_dim != 128) return INT8K_ERR_UNSUPPORTED;
    if (!out.f16 && !out.qs) return INT8K_ERR_INVALID_ARGUMENT;
    if (!aligned_to(Q, 16) || !aligned_to(K, 16) || !aligned_to(V, 16) ||
        !aligned_to(scale_Q, 4) || !aligned_to(scale_K, 4) || !aligned_to(scale_V, 4) ||
        !out_ok(out))
        return INT8K_ERR_MISALIGNED;
    const SplitPlan plan = plan_within(BH, S, head_dim, nsplit, workspace ? workspace_bytes : 0);
    // 64 work-items per unit, < 2^32
    const long long waves = std::max<long long>(plan.forced ? plan.nsplit : 0,
                                                (long long)plan.g.blocks * plan.g.waves);
    if (BH * waves >= (1LL << 26)) return INT8K_ERR_UNSUPPORTED;
    // the one-launch path reads no workspace: a null or short one is accepted there
    if (const size_t need = decode_partial_bytes(plan, BH, head_dim)) {
        if (!workspace || workspace_bytes < need) return INT8K_ERR_WORKSPACE;
        if (!aligned_to(workspace, 16)) return INT8K_ERR_MISALIGNED;
    }
    const DecodeWorkspace w = carve(workspace, (long long)BH * plan.partials, head_dim);
    const DecodeArgs a{Q,  K, V,     scale_Q, scale_K, scale_V,
                       BH, S, S_cap, (1.0f / std::sqrt((float)head_dim)) * kLog2e};
    return head_dim == 128 ? launch_decode<128>(a, out, plan, w, as_stream(stream))
                           : launch_decode<64>(a, out, plan, w, as_stream(stream));
}

extern "C" int int8k_decode_attention_forward(
    const int8_t* Q, const int8_t* K, const int8_t* V, uint16_t* out,
    const float* scale_Q, const float* scale_K, const float* scale_V,
    int BH, int S, int head_dim, int nsplit,
    void* workspace, size_t workspace_bytes, void* stream) {
    if (!out) return INT8K_ERR_INVALID_ARGUMENT;
    return decode_impl(Q, K, V, DecodeOut{out, nullptr, nullptr}, scale_Q, scale_K, scale_V, BH,
                       S, S, head_dim, nsplit, workspace, workspace_bytes, stream);
}

extern "C" int int8k_decode_attention_forward_quant(
    const int8_t* Q, const int8_t* K, const int8_t* V, int8_t* out_q, float* out_scale,
    const float* scale_Q, const float* scale_K, const float* scale_V,
    int BH, int S, int head_dim, int nsplit,
    void* workspace, size_t workspace_bytes, void* stream) {
    if (!out_q || !out_scale) return INT8K_ERR_INVALID_ARGUMENT;
    return decode_impl(Q, K, V, DecodeOut{nullptr, out_q, out_scale}, scale_Q, scale_K, scale_V,
                       BH, S, S, head_dim, nsplit, workspace, workspace_bytes, stream);
}

extern "C" int int8k_decode_attention_forward_cache(
    const int8_t* Q, const int8_t* K_cache, const int8_t* V_cache, uint16_t* out,
    const float* scale_Q, const float* sK_cache, const float* sV_cache,
    int BH, int S, int capacity, int head_dim, int nsplit,
    void* workspace, size_t workspace_bytes, void* stream) {
    if (!out) return INT8K_ERR_INVALID_ARGUMENT;
    return decode_impl(Q, K_cache, V_cache, DecodeOut{out, nullptr, nullptr}, scale_Q, sK_cache,
                       sV_cache, BH, S, capacity, head_dim, nsplit, workspace, workspace_bytes,
                       stream);
}

extern "C" int int8k_decode_attention_forward_cache_quant(
    const int8_t* Q, const int8_t* K_cache, const int8_t* V_cache, int8_t* out_q,
    float* out_scale, const float* scale_Q, const float* sK_cache, const float* sV_cache,
    int BH, int S, int capacity, int head_dim, int nsplit,
    void* workspace, size_t workspace_bytes, void* stream) {
    if (!out_q || !out_scale) return INT8K_ERR_INVALID_ARGUMENT;
    return decode_impl(Q, K_cache, V_cache, DecodeOut{nullptr, out_q, out_scale}, scale_Q,
                       sK_cache, sV_cache, BH, S, capacity, head_dim, nsplit, workspace,
                       workspace_bytes, stream);
}

// The paged kernel always uses 8 slots for D = 128 and 4 for D = 64 (page_size
// is a multiple of both), so its split plan is computed for those slot counts.
static SplitPlan plan_paged(int BH, int max_context, int D, int nsplit_req) {
    const int ns_slots = D == 128 ? 8 : 4;
    const int R = rows_per_iter(D, ns_slots);
    const DecodeTuning tn = tuning_for(D);
    const long long max_split = ceil_div(max_context, R);
    long long ns;
    if (nsplit_req > 0) {
        ns = nsplit_req;
    } else {
        ns = ceil_div(tn.target_units, BH);
        ns = std::min(ns, std::max<long long>(1, ceil_div(max_context, 4LL * R)));
    }
    ns = std::max<long long>(1, std::min(ns, max_split));
    const long long chunk = round_up((size_t)ceil_div(max_context, ns), (size_t)R);
    ns = ceil_div(max_context, chunk);
    const GroupPlan g = ns <= kGroupWaves && use_block_kernel()
                            ? GroupPlan{1, (int)ns, (int)chunk}
                            : forced_groups((int)ns, (int)chunk);
    return SplitPlan{(int)ns, (int)chunk, nsplit_req > 0, g, (int)ns};
}

extern "C" size_t int8k_decode_attention_paged_workspace_bytes(int B, int H, int max_context,
                                                               int head_dim, int nsplit) {
    if (B <= 0 || H <= 0 || max_context <= 0 || (head_dim != 64 && head_dim != 128)) return 0;
    const long long BH = (long long)B * H;
    if (BH >= (1LL << 31)) return 0;
    const SplitPlan plan = plan_paged((int)BH, max_context, head_dim, nsplit);
    return carve(nullptr, BH * plan.nsplit, head_dim).bytes;
}

extern "C" int int8k_decode_attention_paged_num_splits(int B, int H, int max_context,
                                                       int head_dim, int nsplit) {
    if (B <= 0 || H <= 0 || max_context <= 0 || (head_dim != 64 && head_dim != 128)) return 0;
    const long long BH = (long long)B * H;
    if (BH >= (1LL << 31)) return 0;
    return plan_paged((int)BH, max_context, head_dim, nsplit).nsplit;
}

extern "C" int int8k_decode_paged_bad_page_ids(unsigned int* count) {
    clear_last_error();
    if (!count) return INT8K_ERR_INVALID_ARGUMENT;
    const hipError_t e = hipMemcpyFromSymbol(count, HIP_SYMBOL(g_paged_bad_ids),
                                             sizeof(unsigned int), 0, hipMemcpyDeviceToHost);
    if (e != hipSuccess) {
        set_last_error("hipMemcpyFromSymbol(g_paged_bad_ids)", e);
        return INT8K_ERR_HIP;
    }
    return INT8K_OK;
}

static int paged_impl(
    const int8_t* Q, const int8_t* K_pages, const int8_t* V_pages, const DecodeOut& out,
    const float* scale_Q, const float* sK_pages, const float* sV_pages,
    const int32_t* block_tables, const int32_t* context_lens,
    int B, int H, int head_dim, int num_pages, int page_size, int max_pages_per_seq,
    int max_context, int nsplit, void* workspace, size_t workspace_bytes, void* stream) {
    clear_last_error();
    if (!Q || !K_pages || !V_pages || !(out.f16 || (out.q && out.qs)) || !scale_Q || !sK_pages ||
        !sV_pages || !block_tables || !context_lens)
        return INT8K_ERR_INVALID_ARGUMENT;
    if (B <= 0 || H <= 0 || num_pages <= 0 || max_pages_per_seq <= 0 || max_context <= 0 ||
        nsplit < 0)
        return INT8K_ERR_INVALID_ARGUMENT;
    if (head_dim != 64 && head_dim != 128) return INT8K_ERR_UNSUPPORTED;
    if (page_size < 16 || page_size > 1024 || (page_size & (page_size - 1)) != 0)
        return INT8K_ERR_UNSUPPORTED;
    if ((long long)max_context > (long long)max_pages_per_seq * page_size)
        return INT8K_ERR_INVALID_ARGUMENT;
    const long long BH = (long long)B * H;
    if ((long long)num_pages * H * page_size * head_dim >= (1LL << 40)) return INT8K_ERR_UNSUPPORTED;
    if (!aligned_to(Q, 16) || !aligned_to(K_pages, 16) || !aligned_to(V_pages, 16) ||
        !aligned_to(scale_Q, 4) || !aligned_to(sK_pages, 4) || !aligned_to(sV_pages, 4) ||
        !aligned_to(block_tables, 4) || !aligned_to(context_lens, 4) || !out_ok(out))
        return INT8K_ERR_MISALIGNED;
    if (BH >= (1LL << 31)) return INT8K_ERR_UNSUPPORTED;
    const SplitPlan plan = plan_paged((int)BH, max_context, head_dim, nsplit);
    const long long units = BH * plan.nsplit;
    if (units >= (1LL << 26)) return INT8K_ERR_UNSUPPORTED;  // 64 work-items per unit, < 2^32
    const DecodeWorkspace w = carve(workspace, units, head_dim);
    if (!workspace || workspace_bytes < w.bytes) return INT8K_ERR_WORKSPACE;
    if (!aligned_to(workspace, 16)) return INT8K_ERR_MISALIGNED;
    int log2_page = 0;
    while ((1 << log2_page) < page_size) ++log2_page;
    if (head_dim == 128)
        return launch_decode_paged<128>(Q, K_pages, V_pages, out, scale_Q, sK_pages, sV_pages,
                                        block_tables, context_lens, B, H, num_pages, log2_page,
                                        max_pages_per_seq, max_context, plan, w, as_stream(stream));
    return launch_decode_paged<64>(Q, K_pages, V_pages, out, scale_Q, sK_pages, sV_pages,
                                   block_tables, context_lens, B, H, num_pages, log2_page,
                                   max_pages_per_seq, max_context, plan, w, as_stream(stream));
}

extern "C" int int8k_decode_attention_forward_paged(
    const int8_t* Q, const int8_t* K_pages, const int8_t* V_pages, uint16_t* out,
    const float* scale_Q, const float* sK_pages, const float* sV_pages,
    const int32_t* block_tables, const int32_t* context_lens,
    int B, int H, int head_dim, int num_pages, int page_size, int max_pages_per_seq,
    int max_context, int nsplit, void* workspace, size_t workspace_bytes, void* stream) {
    if (!out) return INT8K_ERR_INVALID_ARGUMENT;
    return paged_impl(Q, K_pages, V_pages, DecodeOut{out, nullptr, nullptr}, scale_Q, sK_pages,
                      sV_pages, block_tables, context_lens, B, H, head_dim, num_pages, page_size,
                      max_pages_per_seq, max_context, nsplit, workspace, workspace_bytes, stream);
}

extern "C" int int8k_decode_attention_forward_paged_quant(
    const int8_t* Q, const int8_t* K_pages, const int8_t* V_pages, int8_t* out_q,
    float* out_scale, const float* scale_Q, const float* sK_pages, const float* sV_pages,
    const int32_t* block_tables, const int32_t* context_lens,
    int B, int H, int head_dim, int num_pages, int page_size, int max_pages_per_seq,
    int max_context, int nsplit, void* workspace, size_t workspace_bytes, void* stream) {
    if (!out_q || !out_scale) return INT8K_ERR_INVALID_ARGUMENT;
    return paged_impl(Q, K_pages, V_pages, DecodeOut{nullptr, out_q, out_scale}, scale_Q,
                      sK_pages, sV_pages, block_tables, context_lens, B, H, head_dim, num_pages,
                      page_size, max_pages_per_seq, max_context, nsplit, workspace,
                      workspace_bytes, stream);
}
