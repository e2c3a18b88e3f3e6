// RoPE + fp16 KV-cache write, split-K GQA decode attention and the naive attention baseline.
//
// Semantics (what is computed, which buffers change) follow the reference:
//   rope_kv fused / unfused      src/kernels/rope_kv.cu:10-79  (pairs (i, i+hd/2), angle fp32(pos)*inv_freq[i],
//                                fused leaves the k slice of qkv unrotated)
//   split-K + LSE merge          src/kernels/attention_opt.cu:17-134 (scale 0.125, splits at or past ctx exit at once so
//                                the grid is fixed and graph-capturable)
//   naive                        src/kernels/attention_naive.cu:18-81 (one workgroup per query head)
// How the split-K kernel divides the work is this file's own, described at the kernel.
#include <algorithm>
#include <array>
#include <atomic>
#include <cfloat>
#include <mutex>
#include <random>

#include "../arrival.h"
#include "../kernels.h"
#include "device.h"

namespace cllm {

namespace {

constexpr int kHd = 64;
constexpr int kGroup = 4;

// Rotation of pair (x0, x1) = (v[i], v[i+half]) by angle pos*inv_freq[i].
__device__ __forceinline__ void rotate(float x0, float x1, float ang, float& r0, float& r1) {
    float s, c;
    sincosf(ang, &s, &c);
    r0 = x0 * c - x1 * s;
    r1 = x1 * c + x0 * s;
}

// Work items: [0, (nh+nkv)*half) rotate one pair of a q or k head; then nkv*hd copies of v.
__global__ void __launch_bounds__(256) rope_kv_fused_kernel(float* qkv, const float* inv_freq, uint16_t* kc, uint16_t* vc,
                                                            const int* d_pos, int nh, int nkv, int hd, int max_seq) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int half = hd / 2;
    const int pos = *d_pos;
    const int n_rot = (nh + nkv) * half;
    if (t < n_rot) {
        const int head = t / half, i = t % half;
        float* v = qkv + head * hd;
        float r0, r1;
        rotate(v[i], v[i + half], static_cast<float>(pos) * inv_freq[i], r0, r1);
        if (head < nh) {
            v[i] = r0;
            v[i + half] = r1;
        } else {
            uint16_t* dst = kc + (static_cast<size_t>(head - nh) * max_seq + pos) * hd;
            dst[i] = float_to_half_bits(r0);
            dst[i + half] = float_to_half_bits(r1);
        }
    } else if (t < n_rot + nkv * hd) {
        const int e = t - n_rot;
        const int head = e / hd, d = e % hd;
        vc[(static_cast<size_t>(head) * max_seq + pos) * hd + d] = float_to_half_bits(qkv[(nh + nkv) * hd + e]);
    }
}

__global__ void __launch_bounds__(256) rope_inplace_kernel(float* qkv, const float* inv_freq, const int* d_pos, int nh,
                                                           int nkv, int hd) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int half = hd / 2;
    if (t >= (nh + nkv) * half) return;
    const int head = t / half, i = t % half;
    float* v = qkv + head * hd;
    float r0, r1;
    rotate(v[i], v[i + half], static_cast<float>(*d_pos) * inv_freq[i], r0, r1);
    v[i] = r0;
    v[i + half] = r1;
}

__global__ void __launch_bounds__(256) kv_write_kernel(const float* qkv, uint16_t* kc, uint16_t* vc, const int* d_pos,
                                                       int nh, int nkv, int hd, int max_seq) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 2 * nkv * hd) return;
    const bool is_k = t < nkv * hd;
    const int e = is_k ? t : t - nkv * hd;
    const int head = e / hd, d = e % hd;
    uint16_t* cache = is_k ? kc : vc;
    cache[(static_cast<size_t>(head) * max_seq + *d_pos) * hd + d] = float_to_half_bits(qkv[nh * hd + t]);
}

// ---- split-K attention -------------------------------------------------------------------------------
//
// One kernel.  Bound by the K and V bytes at long contexts, by latency at short ones.  A wave takes whole 32-token
// tiles, straight from the cache into registers in the matrix instructions' layout (no LDS staging), with the next tile's
// 8 KiB in flight while this one is multiplied.  Both products run on v_mfma_f32_16x16x32_f16: the 16 query rows are the kv
// head's 4 query heads times up to 4 fp16 parts of a 32-bit value (11 bits each, three used), so the fp16 keys meet the
// whole query and the fp16 values the whole weight, with products exact and sums in 32 bits.  The weights come out of the
// first product in the lanes in which the second takes them, eight tokens a lane.  About 180 instructions per tile, against
// 480 with mixed-precision FMAs and a sum over lanes per score: that form measured, in one call of a replayed graph, 4.3 us
// at 100 tokens, 10.7 at 8000 and 52.8 at 131071, this one 4.1, 10.0 and 46.5.
//
// A kv head's tiles are dealt evenly to its splits' waves, with only as many splits as give every wave a tile: up to 256
// tokens are one workgroup, which writes the output.  With more, every split stores its (o, m, l), waits until they are in
// memory and counts itself in the kv head's arrival word (arrival.h); the last to arrive merges them all, in split order
// whichever it is, and writes the output.  No workgroup waits for another, so the order in which they run does not matter.
// Polling for the partials instead (each word tagged, the last split's workgroup merging) measured 10.0 us at 8000 tokens
// and 45 at 131071 against 8.9 and 44, and 6.7 against 6.85 at 300.
// Measured on MI355X, 8 kv heads, one call in a replayed graph of 16 (2 at 131071), with 128 tokens per workgroup staged in
// LDS and a second kernel merging the splits one after the other, and now: 100 tokens 6.5 -> 4.1 us, 1000 9.7 -> 7.1, 4000
// 18.4 -> 8.1, 8000 28.0 -> 8.9, 131071 375 -> 44 (6.1 TB/s).
// Workgroups in all: one per CU (2 waves per SIMD).  With the FMA form in workgroups of half the size, 512 measured 57
// against 52 us at 131071 tokens and 12.7 against 11.4 at 8000, 128 measured 82 and 11.7.
constexpr int kSplitBlocks = 256;
constexpr int kMaxSplits = 64;     // splits of one kv head
constexpr int kWaves = 8;          // per workgroup
constexpr int kTile = 32;
constexpr float kScore2 = 0.125f * 1.4426950408889634f;  // score scale times log2(e)

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// A wave's 32 tokens as the matrix instructions take them.  k[a][s]: lane (n, g) = (lane % 16, lane / 16) holds columns
// 32 s + 8 g .. + 7 of token 16 a + n.  v[j]: columns 4 n .. 4 n + 3 of token token_of(g, j).
struct KvTile {
    u32x4 k[2][2];
    u32x2 v[8];
};
__device__ __forceinline__ int token_of(int g, int j) { return 16 * (j / 4) + 4 * g + j % 4; }

__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }
// exp of the difference of two scores, from the dot products.
__device__ __forceinline__ float weight_of(float dot, float m) { return exp2_hw((dot - m) * kScore2); }

// The leading 11 bits (toward zero) of two floats as fp16; the floats keep the rest, 2^11 times.
constexpr float kPart = 2048.f;
__device__ __forceinline__ uint32_t take_f16(float& x, float& y) {
    const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x, y));
    x = fmaf(half_bits_to_float(static_cast<uint16_t>(h)), -kPart, x * kPart);
    y = fmaf(half_bits_to_float(static_cast<uint16_t>(h >> 16)), -kPart, y * kPart);
    return h;
}
// Part p of two floats written as h + m 2^-11 + l 2^-22 with fp16 h, m, l (p = 3: nothing): all 24 bits of a float between
// 2^16 and 2^-24, and 2^-46 at the least, although fp16 itself ends at 2^-24.
__device__ __forceinline__ uint32_t part_f16(float x, float y, int p) {
    const uint32_t h = take_f16(x, y), m = take_f16(x, y);
    const uint32_t l = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x, y));
    return p == 0 ? h : p == 1 ? m : p == 2 ? l : 0u;
}
// Whether the three parts leave anything of them.
__device__ __forceinline__ bool parts_lose(float x, float y) {
    (void)take_f16(x, y), (void)take_f16(x, y), (void)take_f16(x, y);
    return x != 0.f || y != 0.f;
}

// The running softmax of the wave: lane (n, g) holds, for head n / 4, the largest dot product m (starting at the lowest
// float) and its share l of the weights 2^kLift exp(score - largest), and in o[b][i] the sums of part i of head g's weights
// times column 4 n + b.  kLift puts the largest weight at 2^15, so that a weight has all its bits down to 2^-39 of
// that and counts down to 2^-61.
// Weights come from differences of dot products, so they keep their meaning however large the scores are.
constexpr float kLift = 15.f;
struct Running {
    float m, l;
    f32x4 o[4];
};

// One tile at token t0; tokens at or past ctx weigh nothing.  qb: the group's queries, part n % 4 of head n / 4 as fp16 (one
// power-of-two scale per head); ps: that part's scale; sc: the score scale times log2(e) over the head's scale.
__device__ __forceinline__ void attend(const KvTile& kv, const f16x8 (&qb)[2], float ps, float sc, Running& st, int t0, int n,
                                       int g, int ctx) {
    // Scores of tokens 16 a + 4 g + i against (head, part) n; the parts' sum over the head's 4 lanes.
    f32x4 d[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        d[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 2; ++s)
            d[a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, kv.k[a][s]), qb[s], d[a], 0, 0, 0);
    }
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = d[j / 4][j % 4] * ps;
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] += dpp<kDppXor1>(x[j]);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] += dpp<kDppXor2>(x[j]);
    u32x2 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = kv.v[j];
    if (t0 + kTile > ctx) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (t0 + token_of(g, j) >= ctx) x[j] = -INFINITY, v[j] = u32x2{0u, 0u};  // the cache there may hold anything
    }
    float m = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
    m = fmaxf(st.m, max_lanes_xor<32>(max_lanes_xor<16>(m)));
    if (__any(m > st.m)) {  // a new maximum: rare after a wave's first tiles
        const float f = exp2_hw((st.m - m) * sc), fo = __shfl(f, 4 * g);
        st.m = m;
        st.l *= f;
#pragma unroll
        for (int b = 0; b < 4; ++b) st.o[b] *= fo;
    }
    float l[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) l[j] = x[j] = exp2_hw(fmaf(x[j] - m, sc, kLift));
    st.l += ((l[0] + l[1]) + (l[2] + l[3])) + ((l[4] + l[5]) + (l[6] + l[7]));
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = part_f16(x[2 * i], x[2 * i + 1], n % 4);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        u32x4 c;  // column 4 n + b of the 8 tokens
#pragma unroll
        for (int i = 0; i < 4; ++i)
            c[i] = __builtin_amdgcn_perm(v[2 * i + 1][b / 2], v[2 * i][b / 2], b % 2 ? 0x07060302u : 0x05040100u);
        st.o[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, c), st.o[b], 0,
                                                         0, 0);
    }
}

// ---- what the splits exchange ------------------------------------------------------------------------

// Relaxed agent-scope accesses: they pass the XCDs' own L2 caches by and are made in the memory that all of them share.
// Everything the splits exchange goes this way, so a store that has been acknowledged can be read anywhere, and a wave that
// waits for its own stores needs no release fence, which would write back its whole L2 (8000 tokens 8.9 -> 16.0 us).
template <typename T>
using global_ptr = __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ T shared_load(const T* p) {
    return __hip_atomic_load((global_ptr<T>)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void shared_store(T* p, T v) {
    __hip_atomic_store((global_ptr<T>)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// This wave's stores (and its begin()) have been made there.
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

struct ArrivalWord {  // arrival.h's operations
    uint64_t* p;
    __device__ void compare_exchange(uint64_t from, uint64_t to) const {
        (void)__hip_atomic_compare_exchange_strong((global_ptr<uint64_t>)p, &from, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ uint64_t add_one() const {
        return __hip_atomic_fetch_add((global_ptr<uint64_t>)p, uint64_t{1}, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ void store(uint64_t v) const { shared_store(p, v); }
};

// Where the partials of head h's split s lie: o as [h][s][64], then m and l as [h][s][2]; each kv head's arrival word in a
// 128-byte line of its own.
constexpr int kWordStride = 16;
struct Partials {
    float *o, *ml;
    uint64_t* words;
    uint64_t tag;
};

// The splits of head h that fall to this wave, s = half, half + 2, ... below n: their merged (m, l) and the lane's output
// column.  Up to 16 of them, and all of their (m, l), are in flight at once.
__device__ __forceinline__ void merge_half(const Partials& p, int h, int splits, int n, int half, int lane, float& m,
                                           float& l, float& o) {
    constexpr int kRound = 16;
    m = -FLT_MAX, l = 0.f, o = 0.f;
    const float* po = p.o + static_cast<size_t>(h) * splits * kHd + lane;
    const float* pml = p.ml + static_cast<size_t>(h) * splits * 2;
    for (int s0 = half; s0 < n; s0 += 2 * kRound) {
        const int sl = s0 + 2 * (lane % kRound);  // the split whose m (lanes 0-15) or l (16-31) this lane holds
        const bool mine = lane < 2 * kRound && sl < n;
        const float vm = shared_load(pml + (mine ? 2 * sl + lane / kRound : 0));
        float v[kRound];
#pragma unroll
        for (int i = 0; i < kRound; ++i) v[i] = shared_load(po + static_cast<size_t>(min(s0 + 2 * i, n - 1)) * kHd);
        const float sm = mine && lane < kRound ? vm : -FLT_MAX;
        const float sl_ = __shfl(vm, lane + kRound);
        const float mn = fmaxf(m, wave_max(sm)), f = weight_of(m, mn);
        const float e = mine && lane < kRound ? weight_of(sm, mn) : 0.f;
        m = mn;
        l = fmaf(l, f, wave_sum(mine && lane < kRound ? sl_ * e : 0.f));
        o *= f;
#pragma unroll
        for (int i = 0; i < kRound; ++i)
            if (s0 + 2 * i < n) o = fmaf(v[i], __shfl(e, i), o);
    }
}

// The wave's tiles (`first`, then [begin, end)) one token at a time, lane = column: the closed form term by term.
__device__ __forceinline__ void attend_plain(const float* q, const uint16_t* K, const uint16_t* V, int first, int begin,
                                             int end, int ctx, int lane, float (&so)[kGroup][kHd], float (&sml)[kGroup][2]) {
#pragma unroll 1
    for (int h = 0; h < kGroup; ++h) {
        const float qh = q[h * kHd + lane];
        float m = -FLT_MAX, l = 0.f, o = 0.f;
#pragma unroll 1
        for (int t = first; t < end; t = t < begin ? begin : t + 1) {
#pragma unroll 1
            for (int j = t * kTile; j < min((t + 1) * kTile, ctx); ++j) {
                const float s = wave_sum(qh * half_bits_to_float(K[static_cast<size_t>(j) * kHd + lane]));
                const float mn = fmaxf(m, s), f = weight_of(m, mn), p = exp2_hw(fmaf(s - mn, kScore2, kLift));
                l = fmaf(l, f, p);
                o = fmaf(p, half_bits_to_float(V[static_cast<size_t>(j) * kHd + lane]), o * f);
                m = mn;
            }
        }
        so[h][lane] = o;
        if (lane == 0) sml[h][0] = m, sml[h][1] = l;
    }
}

// grid (nkv, splits), block 512.
__global__ void __launch_bounds__(kWaves* kWave) attn_split_kernel(const float* q, const uint16_t* kc, const uint16_t* vc,
                                                                   const int* d_pos, Partials part, float* out, int max_seq) {
    __shared__ float so[kWaves][kGroup][kHd];  // [wave][head][column]
    __shared__ float sml[kWaves][kGroup][2];   // [wave][head] m, l
    __shared__ bool last;

    const int kvh = blockIdx.x, split = blockIdx.y, splits = gridDim.y;
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int n = lane % 16, g = lane / 16;
    // The lane's 16 columns of query n / 4 (as KvTile's k), requested first.
    float qv[2][8];
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(q + (kvh * kGroup + n / 4) * kHd + 32 * (i / 8) + 8 * g + i % 8);
#pragma unroll
        for (int e = 0; e < 4; ++e) qv[i / 8][i % 8 + e] = v[e];
    }
    // A tile (whole tiles lie inside the cache: max_seq is a multiple of 128).
    auto load = [&](KvTile& kv, int tile) {
        const size_t first = (static_cast<size_t>(kvh) * max_seq + static_cast<size_t>(tile) * kTile) * kHd;
        const char* K = reinterpret_cast<const char*>(kc + first);
        const char* V = reinterpret_cast<const char*>(vc + first);
        const uint32_t ko = n * (kHd * 2) + g * 16, vo = 4 * g * (kHd * 2) + n * 8;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int s = 0; s < 2; ++s)
                kv.k[a][s] = gload(reinterpret_cast<const u32x4*>(K + ko + a * 16 * kHd * 2 + s * 64));
#pragma unroll
        for (int j = 0; j < 8; ++j)
            kv.v[j] = __builtin_nontemporal_load((global_ptr<const u32x2>)(V + vo + token_of(0, j) * (kHd * 2)));
    };
    // Wave wi takes tile wi and then its share of the tiles past one for each wave, in one piece (dealt in turn, 60 against
    // 53 us at 131071 tokens).  The first tile does not depend on *d_pos, so the first split's waves request theirs before
    // it has arrived (rows of the cache past ctx weigh nothing), a memory round trip less for short contexts: 100 tokens
    // 5.3 -> 4.1 us.  The other splits wait, for they may have nothing to do.
    const int wi = split * kWaves + w;
    KvTile A, B;
    const bool early = split == 0 && (w + 1) * kTile <= max_seq;
    if (early) load(A, wi);
    const int ctx = *d_pos + 1;
    // At least one split works, so that a position before the first token gives the sums' 0 / 0.
    const int tiles = (ctx + kTile - 1) / kTile;
    const int used = max(1, min(splits, (tiles + kWaves - 1) / kWaves)), waves = kWaves * used;
    if (split >= used) return;
    // Every execution has its own tag: a replayed launch's packet lies elsewhere in the queue.
    const ArrivalWord word{part.words + kvh * kWordStride};
    const uint64_t tag = part.tag ^ reinterpret_cast<uint64_t>(__builtin_amdgcn_dispatch_ptr()) >> 6 << 8;
    uint64_t seen = 0;
    if (used > 1) seen = shared_load(word.p);
    const uint64_t more = max(tiles - waves, 0);
    const int begin = waves + static_cast<int>(more * wi / waves), end = waves + static_cast<int>(more * (wi + 1) / waves);
    Running st{-FLT_MAX, 0.f, {}};
    float m_dot = -FLT_MAX;  // st.m without the query's scale
    bool plain = false;
    if (wi < tiles) {
        if (!early) load(A, wi);
        __builtin_amdgcn_sched_barrier(0);
        // The query's fp16 parts: the head's largest |q| scaled to 2^14 .. 2^15.  Bits below 2^-46 are lost then: 2^-61 of
        // the largest, nothing in a score as long as that is below 2^16.  From there a column that meets zero keys can be
        // so large that the others' bits count, and a wave that lost any does without the parts.
        float big = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) big = fmaxf(big, fabsf(qv[i / 8][i % 8]));
        big = max_lanes_xor<32>(max_lanes_xor<16>(big));
        const int e = big > 0.f && big < INFINITY ? min(14 - ilogbf(big), 110) : 0;
        f16x8 qb[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            u32x4 p;
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = part_f16(ldexpf(qv[s][2 * i], e), ldexpf(qv[s][2 * i + 1], e), n % 4);
            qb[s] = __builtin_bit_cast(f16x8, p);
        }
        if (__builtin_expect(__any(big >= 65536.f), 0)) {
#pragma unroll
            for (int i = 0; i < 16; i += 2)
                plain = plain || parts_lose(ldexpf(qv[i / 8][i % 8], e), ldexpf(qv[i / 8][i % 8 + 1], e));
        }
        const float sc = ldexpf(kScore2, -e), ps = ldexpf(1.f, -11 * (n % 4));
        auto step = [&](const KvTile& kv, int tile) { attend(kv, qb, ps, sc, st, tile * kTile, n, g, ctx); };
        int t = wi, next = begin;
        for (;;) {
            if (next >= end) {
                step(A, t);
                break;
            }
            load(B, next);
            __builtin_amdgcn_sched_barrier(0);  // the next tile's loads go out before this tile's math
            step(A, t);
            t = next++;
            if (next >= end) {
                step(B, t);
                break;
            }
            load(A, next);
            __builtin_amdgcn_sched_barrier(0);
            step(B, t);
            t = next++;
        }
        m_dot = ldexpf(st.m, -e);
    }
    st.l = sum_lanes_xor<32>(sum_lanes_xor<16>(st.l));
    f32x4 y;  // columns 4 n .. 4 n + 3 of head g
#pragma unroll
    for (int b = 0; b < 4; ++b) y[b] = fmaf(fmaf(st.o[b][2], 1.f / kPart, st.o[b][1]), 1.f / kPart, st.o[b][0]);
    *reinterpret_cast<f32x4*>(&so[w][g][4 * n]) = y;
    if (g == 0 && n % 4 == 0) sml[w][n / 4][0] = m_dot, sml[w][n / 4][1] = st.l;
    // An infinity or NaN among the inputs (or a score past the floats) leaves one here, as its parts do not add up to it:
    // such a wave starts over with plain products.
    auto finite = [](float v) { return fabsf(v) < INFINITY; };
    if (__any(plain || !finite(m_dot) || !finite(st.l) || !finite((y[0] + y[1]) + (y[2] + y[3])))) {
        const size_t head = static_cast<size_t>(kvh) * max_seq * kHd;
        attend_plain(q + kvh * kGroup * kHd, kc + head, vc + head, wi, begin, end, ctx, lane, so[w], sml[w]);
    }
    __syncthreads();

    if (used > 1 && tid == 0) arrival::begin(word, seen, tag);
    // Waves 0-3 take a head each: the 8 waves' partials in wave order.
    const int h = kvh * kGroup + w % kGroup;
    if (w < kGroup) {
        float m = -FLT_MAX, l = 0.f, o = 0.f;
#pragma unroll
        for (int i = 0; i < kWaves; ++i) m = fmaxf(m, sml[i][w][0]);
#pragma unroll
        for (int i = 0; i < kWaves; ++i) {
            const float f = weight_of(sml[i][w][0], m);
            l = fmaf(sml[i][w][1], f, l);
            o = fmaf(so[i][w][lane], f, o);
        }
        if (used == 1) {
            out[h * kHd + lane] = o / l;
        } else {
            const size_t slot = static_cast<size_t>(h) * splits + split;
            shared_store(part.o + slot * kHd + lane, o);
            if (lane < 2) shared_store(part.ml + slot * 2 + lane, lane ? l : m);
            stores_done();
        }
    }
    if (used == 1) return;

    __syncthreads();
    if (tid == 0) last = arrival::arrive(word, tag, used);
    __syncthreads();
    if (!last) return;
    // Each head's splits in two halves (waves w and w + 4).
    float m, l, o;
    merge_half(part, h, splits, used, w / kGroup, lane, m, l, o);
    if (w >= kGroup) {
        so[w][0][lane] = o;
        if (lane == 0) sml[w][0][0] = m, sml[w][0][1] = l;
    }
    __syncthreads();
    if (w < kGroup) {
        const float m1 = sml[w + kGroup][0][0], l1 = sml[w + kGroup][0][1], o1 = so[w + kGroup][0][lane];
        const float M = fmaxf(m, m1), f = weight_of(m, M), f1 = weight_of(m1, M);
        out[h * kHd + lane] = (o * f + o1 * f1) / (l * f + l1 * f1);
    }
}

// grid nh, block 256, dynamic LDS max_seq floats of scores + 16 scratch.
__global__ void __launch_bounds__(256) attn_naive_kernel(const float* q, const uint16_t* kc, const uint16_t* vc,
                                                         const int* d_pos, float* out, int nh, int nkv, int hd,
                                                         int max_seq) {
    extern __shared__ float sm[];
    float* sc = sm;
    float* scratch = sm + max_seq;
    const int h = blockIdx.x, kvh = h / (nh / nkv);
    const int ctx = *d_pos + 1;
    const float* qh = q + h * hd;
    const uint16_t* K = kc + static_cast<size_t>(kvh) * max_seq * hd;
    const uint16_t* V = vc + static_cast<size_t>(kvh) * max_seq * hd;
    float mx = -INFINITY;
    for (int t = threadIdx.x; t < ctx; t += blockDim.x) {
        float dot = 0.f;
        for (int d = 0; d < hd; ++d) dot += qh[d] * half_bits_to_float(K[static_cast<size_t>(t) * hd + d]);
        sc[t] = 0.125f * dot;
        mx = fmaxf(mx, sc[t]);
    }
    mx = wave_max(mx);
    if (threadIdx.x % kWave == 0) scratch[threadIdx.x / kWave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(scratch[0], scratch[1]), fmaxf(scratch[2], scratch[3]));
    __syncthreads();
    float sum = 0.f;
    for (int t = threadIdx.x; t < ctx; t += blockDim.x) {
        sc[t] = expf(sc[t] - mx);
        sum += sc[t];
    }
    sum = block_sum(sum, scratch);
    if (threadIdx.x < hd) {
        float acc = 0.f;
        for (int t = 0; t < ctx; ++t) acc += sc[t] * half_bits_to_float(V[static_cast<size_t>(t) * hd + threadIdx.x]);
        out[h * hd + threadIdx.x] = acc / sum;
    }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

void launch_rope_kv_fused(float* qkv, const float* inv_freq, uint16_t* k_cache, uint16_t* v_cache, const int* d_pos,
                          int nh, int nkv, int hd, int max_seq, hipStream_t s) {
    CLLM_REQUIRE(qkv && inv_freq && k_cache && v_cache && d_pos, "rope_kv: null pointer");
    CLLM_REQUIRE(nh > 0 && nkv > 0 && hd > 0 && hd % 2 == 0 && max_seq > 0, "rope_kv: bad dimensions");
    const int items = (nh + nkv) * (hd / 2) + nkv * hd;
    hipLaunchKernelGGL(rope_kv_fused_kernel, dim3((items + 255) / 256), dim3(256), 0, s, qkv, inv_freq, k_cache,
                       v_cache, d_pos, nh, nkv, hd, max_seq);
    CLLM_HIP(hipGetLastError());
}

void launch_rope_inplace(float* qkv, const float* inv_freq, const int* d_pos, int nh, int nkv, int hd, hipStream_t s) {
    CLLM_REQUIRE(qkv && inv_freq && d_pos, "rope: null pointer");
    CLLM_REQUIRE(nh > 0 && nkv > 0 && hd > 0 && hd % 2 == 0, "rope: bad dimensions");
    const int items = (nh + nkv) * (hd / 2);
    hipLaunchKernelGGL(rope_inplace_kernel, dim3((items + 255) / 256), dim3(256), 0, s, qkv, inv_freq, d_pos, nh, nkv,
                       hd);
    CLLM_HIP(hipGetLastError());
}

void launch_kv_write(const float* qkv, uint16_t* k_cache, uint16_t* v_cache, const int* d_pos, int nh, int nkv, int hd,
                     int max_seq, hipStream_t s) {
    CLLM_REQUIRE(qkv && k_cache && v_cache && d_pos, "kv_write: null pointer");
    CLLM_REQUIRE(nh > 0 && nkv > 0 && hd > 0 && max_seq > 0, "kv_write: bad dimensions");
    const int items = 2 * nkv * hd;
    hipLaunchKernelGGL(kv_write_kernel, dim3((items + 255) / 256), dim3(256), 0, s, qkv, k_cache, v_cache, d_pos, nh,
                       nkv, hd, max_seq);
    CLLM_HIP(hipGetLastError());
}

void launch_attention_splitk(const float* q, const uint16_t* k_cache, const uint16_t* v_cache, const int* d_pos,
                             float* part_o, float* part_ml, float* out, int nh, int nkv, int hd, int max_seq,
                             hipStream_t s) {
    CLLM_REQUIRE(q && k_cache && v_cache && d_pos && part_o && part_ml && out, "attention: null pointer");
    CLLM_REQUIRE(nkv > 0 && nh == kGroup * nkv, "attention (split-K): needs nh == 4 * nkv");
    CLLM_REQUIRE(hd == kHd, "attention (split-K): needs head_dim 64");
    CLLM_REQUIRE(max_seq > 0 && max_seq % kAttnChunk == 0, "attention (split-K): max_seq must be a multiple of 128");
    CLLM_REQUIRE(aligned16(q) && aligned16(k_cache) && aligned16(v_cache), "attention: pointers must be 16-byte aligned");
    // Half of the caller's slots at most: the arrival words lie behind the outputs of the others.  (Two splits or more, the
    // only ones that count, leave 8 slots of 64 floats for each kv head's line of 32.)
    const int splits = std::max(1, std::min({max_seq / kAttnChunk / 2, kSplitBlocks / nkv, kMaxSplits}));
    const auto end = reinterpret_cast<uintptr_t>(part_o + static_cast<size_t>(nh) * splits * kHd);
    static const uint64_t salt = std::random_device{}() | static_cast<uint64_t>(std::random_device{}()) << 32;
    static std::atomic<uint64_t> launches{0};
    const Partials part{part_o, part_ml, reinterpret_cast<uint64_t*>((end + 7) & ~uintptr_t{7}),
                        arrival::tag_of(salt, launches.fetch_add(1, std::memory_order_relaxed))};
    hipLaunchKernelGGL(attn_split_kernel, dim3(nkv, splits), dim3(kWaves * kWave), 0, s, q, k_cache, v_cache, d_pos, part, out,
                       max_seq);
    CLLM_HIP(hipGetLastError());
}

void launch_attention_naive(const float* q, const uint16_t* k_cache, const uint16_t* v_cache, const int* d_pos,
                            float* out, int nh, int nkv, int hd, int max_seq, hipStream_t s) {
    CLLM_REQUIRE(q && k_cache && v_cache && d_pos && out, "attention: null pointer");
    CLLM_REQUIRE(nh > 0 && nkv > 0 && nh % nkv == 0, "attention (naive): nh must be a multiple of nkv");
    CLLM_REQUIRE(hd > 0 && hd <= 256 && max_seq > 0, "attention (naive): bad dimensions");
    const size_t smem = (static_cast<size_t>(max_seq) + 16) * sizeof(float);
    CLLM_REQUIRE(smem <= 48 * 1024, "attention (naive): max_seq too large for the LDS score buffer");
    hipLaunchKernelGGL(attn_naive_kernel, dim3(nh), dim3(256), smem, s, q, k_cache, v_cache, d_pos, out, nh, nkv, hd,
                       max_seq);
    CLLM_HIP(hipGetLastError());
}

// ---- split-K attention with the partials in static device memory (no allocation on any call) ----------

namespace {

// The split partials of launch_attention_splitk_static: o [slot][64] then (m, l) [slot][2], slot = head * splits +
// split, for at most kStaticAttnSlots slots.  Each device holds its own copy of this array until the process ends.
// Its name is a host-side stand-in: host code uses only the address hipGetSymbolAddress reports, per device.
__device__ __align__(256) float scratch[kStaticAttnSlots * (kHd + 2)];

std::mutex g_scratch_mu;
std::array<float*, 64> g_scratch{};  // device address of `scratch`, indexed by device (no allocation, host or device)

float* scratch_on_current_device() {
    int dev = 0;
    CLLM_HIP(hipGetDevice(&dev));
    CLLM_REQUIRE(dev >= 0 && dev < static_cast<int>(g_scratch.size()), "attention scratch: device index above 63");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* ptr = nullptr;
        CLLM_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        CLLM_INTERNAL(ptr, "attention scratch: no device address");
        g_scratch[dev] = static_cast<float*>(ptr);
    }
    return g_scratch[dev];
}

}  // namespace

void launch_attention_splitk_static(const float* q, const uint16_t* k_cache, const uint16_t* v_cache, const int* d_pos,
                                    float* out, int nh, int nkv, int hd, int max_seq, hipStream_t s) {
    CLLM_REQUIRE(nh > 0 && max_seq > 0 && max_seq % kAttnChunk == 0,
                 "attention (static scratch): max_seq must be a positive multiple of 128");
    CLLM_REQUIRE(static_cast<long long>(nh) * (max_seq / kAttnChunk) <= kStaticAttnSlots,
                 "attention (static scratch): nh * max_seq / 128 exceeds the 8192 partial slots of the static scratch");
    float* base = scratch_on_current_device();
    // No clearing needed: the partials are written before they are read, and what the arrival words hold does not matter.
    launch_attention_splitk(q, k_cache, v_cache, d_pos, base, base + static_cast<size_t>(kStaticAttnSlots) * kHd, out,
                            nh, nkv, hd, max_seq, s);
}

}  // namespace cllm
