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
// tiles: lane (g, c) = (lane / 8, lane % 8) loads 16 bytes, columns 8c .. 8c + 7, of tokens g, g + 8, g + 16 and g + 24,
// so every load instruction reads 1 KiB of consecutive cache rows straight into registers (no LDS staging), and the next
// tile's 8 KiB are in flight while this one is multiplied.  All 4 query heads of the kv head run on the same registers:
// 8 mixed-precision FMAs per head and token, summed over the 8 column lanes by DPP.  Each token phase g keeps its own
// running softmax (m, l, o), so the loop exchanges nothing between phases; they are merged once, at the wave's end,
// then the workgroup's 8 waves in LDS.
//
// A kv head's tiles are dealt evenly to its splits' waves, with only as many splits as give every wave a tile: up to 256 tokens are one workgroup, which writes the output.  With more, each split publishes its
// (o, m, l) as tagged words (value and tag in one 64-bit word, so a word that carries the tag carries the value) and the
// last split's workgroup polls them and writes the output: one store-to-load hop instead of a second launch.
//  * The workgroups it waits for have smaller indices and wait for nothing, so they have been dispatched before it and
//    always finish.  The wait is bounded besides; should it run out, the outputs are NaN.
//  * The tag is a NaN pattern with the launch's number, which scratch memory does not hold by accident, and the words
//    are zeroed as they are consumed, so a replayed launch (same number) never meets its own earlier words.
// Measured on MI355X, 8 kv heads, one call in a replayed graph of 16 (2 at 131071), before (128 tokens per workgroup
// staged in LDS, a second kernel merging the splits one after the other) and now: 100 tokens 6.5 -> 4.2 us, 1000
// 9.7 -> 7.9, 4000 18.4 -> 9.0, 8000 28.0 -> 10.6, 131071 375 -> 52 (5.2 TB/s).
// Workgroups in all: one per CU (2 waves per SIMD).  With workgroups of half the size, 512 measured 57 against 52 us
// at 131071 tokens and 12.7 against 11.4 at 8000, 128 measured 82 and 11.7.
constexpr int kSplitBlocks = 256;
constexpr int kMaxSplits = 64;     // splits of one kv head
constexpr int kWaves = 8;          // per workgroup
constexpr int kTile = 32;
constexpr int kTileRows = kTile / 8;
constexpr float kScore2 = 0.125f * 1.4426950408889634f;  // score scale times log2(e)

struct KvTile {
    u32x4 k[kTileRows], v[kTileRows];
};

// The running softmax of one token phase: m, l and the lane's 8 output columns for each of the 4 heads, in powers of
// two: m is the largest score times log2(e), a weight is exp2(score log2(e) - m) from one FMA on the raw dot product.
// m starts at the lowest float, not -inf, so that a score of -inf (a cached -inf) weighs exp2(-inf) = 0 and not NaN.
struct Running {
    float m[kGroup], l[kGroup], o[kGroup][8];
};

__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

// Sum over the 8 column lanes of a token (every lane gets it).
__device__ __forceinline__ float sum8(float v) {
    v += dpp<kDppXor1>(v);
    v += dpp<kDppXor2>(v);
    return v + dpp<kDppHalfMirror>(v);
}

// Maximum and sum over the 8 token phases (lane bits 3, 4, 5).
__device__ __forceinline__ float phase_max(float v) {
    v = fmaxf(v, dpp<kDppRor8>(v));
    return max_lanes_xor<32>(max_lanes_xor<16>(v));
}
__device__ __forceinline__ float phase_sum(float v) {
    v += dpp<kDppRor8>(v);
    v = sum_lanes_xor<16>(v);
    return sum_lanes_xor<32>(v);
}

// One tile: tokens t0 + 8 r + g; those at or past ctx weigh nothing.
__device__ __forceinline__ void attend(const KvTile& kv, const float (&q)[kGroup][8], Running& st, int t0, int g, int ctx) {
    float s[kTileRows][kGroup];
#pragma unroll
    for (int r = 0; r < kTileRows; ++r)
#pragma unroll
        for (int h = 0; h < kGroup; ++h) {
            float d = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                d = fmaf(half_bits_to_float(static_cast<uint16_t>(kv.k[r][e])), q[h][2 * e], d);
                d = fmaf(half_bits_to_float(static_cast<uint16_t>(kv.k[r][e] >> 16)), q[h][2 * e + 1], d);
            }
            s[r][h] = sum8(d);
            if (t0 + 8 * r + g >= ctx) s[r][h] = -INFINITY;
        }
    float m[kGroup];
    bool moved = false;
#pragma unroll
    for (int h = 0; h < kGroup; ++h) {
        m[h] = st.m[h];
#pragma unroll
        for (int r = 0; r < kTileRows; ++r) m[h] = fmaxf(m[h], s[r][h] * kScore2);
        moved = moved || m[h] > st.m[h];
    }
    if (__any(moved)) {  // a new maximum somewhere in the wave: rare after a chunk's first tiles
#pragma unroll
        for (int h = 0; h < kGroup; ++h) {
            const float f = exp2_hw(st.m[h] - m[h]);
            st.m[h] = m[h];
            st.l[h] *= f;
#pragma unroll
            for (int e = 0; e < 8; ++e) st.o[h][e] *= f;
        }
    }
#pragma unroll
    for (int r = 0; r < kTileRows; ++r) {
        u32x4 v = kv.v[r];
        if (t0 + 8 * r + g >= ctx) v = u32x4{0, 0, 0, 0};  // the row loaded in its place may hold an inf
#pragma unroll
        for (int h = 0; h < kGroup; ++h) {
            const float p = exp2_hw(fmaf(s[r][h], kScore2, -m[h]));
            st.l[h] += p;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                st.o[h][2 * e] = fmaf(p, half_bits_to_float(static_cast<uint16_t>(v[e])), st.o[h][2 * e]);
                st.o[h][2 * e + 1] = fmaf(p, half_bits_to_float(static_cast<uint16_t>(v[e] >> 16)), st.o[h][2 * e + 1]);
            }
        }
    }
}

// ---- tagged words -----------------------------------------------------------------------------------

typedef __attribute__((address_space(1))) uint64_t global_u64;
__device__ __forceinline__ uint64_t tag_load(const uint64_t* p) {
    return __hip_atomic_load((global_u64*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void tag_store(uint64_t* p, float v, uint32_t tag) {
    __hip_atomic_store((global_u64*)p, static_cast<uint64_t>(tag) << 32 | __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool has_tag(uint64_t v, uint32_t tag) { return static_cast<uint32_t>(v >> 32) == tag; }
__device__ __forceinline__ float value_of(uint64_t v) { return __builtin_bit_cast(float, static_cast<uint32_t>(v)); }

constexpr unsigned kPollCap = 1u << 20;  // about a second

// Where the partials of head h's split s lie: o as [h][s][64], then m and l as [h][s][2].
struct Partials {
    uint64_t *o, *ml;
    uint32_t tag;
};

// The first n (<= used - 1) splits of head h that fall to this wave, s = half, half + 2, ...: their merged (m, l) and the
// lane's output column.  Up to 16 of them, and all of their (m, l), are in flight at once.
__device__ __forceinline__ void merge_half(const Partials& p, int h, int splits, int n, int half, int lane, float& m, float& l,
                                           float& o) {
    constexpr int kRound = 16;
    m = -FLT_MAX, l = 0.f, o = 0.f;
    uint64_t* po = p.o + static_cast<size_t>(h) * splits * kHd + lane;
    uint64_t* pml = p.ml + static_cast<size_t>(h) * splits * 2;
    const uint64_t none = static_cast<uint64_t>(p.tag) << 32;
    for (int s0 = half; s0 < n; s0 += 2 * kRound) {
        const int sl = s0 + 2 * (lane % kRound);  // the split whose m (lanes 0-15) or l (16-31) this lane polls
        const bool mine = lane < 2 * kRound && sl < n;
        uint64_t* const pm = pml + (mine ? 2 * sl + lane / kRound : 0);
        uint64_t vm = mine ? tag_load(pm) : none, v[kRound];
#pragma unroll
        for (int i = 0; i < kRound; ++i) v[i] = s0 + 2 * i < n ? tag_load(po + static_cast<size_t>(s0 + 2 * i) * kHd) : none;
        for (unsigned polls = 0;; ++polls) {
            bool ok = has_tag(vm, p.tag);
#pragma unroll
            for (int i = 0; i < kRound; ++i) ok = ok && has_tag(v[i], p.tag);
            if (__all(ok)) break;
            if (polls == kPollCap) {
                l = __builtin_nanf("");
                return;
            }
            if (!has_tag(vm, p.tag)) vm = tag_load(pm);
#pragma unroll
            for (int i = 0; i < kRound; ++i)
                if (!has_tag(v[i], p.tag)) v[i] = tag_load(po + static_cast<size_t>(s0 + 2 * i) * kHd);
        }
        // Consumed: zeroed for the next launch.
        if (mine) tag_store(pm, 0.f, 0);
#pragma unroll
        for (int i = 0; i < kRound; ++i)
            if (s0 + 2 * i < n) tag_store(po + static_cast<size_t>(s0 + 2 * i) * kHd, 0.f, 0);
        const float sm = mine && lane < kRound ? value_of(vm) : -FLT_MAX;
        const float sl_ = __shfl(value_of(vm), lane + kRound);
        const float mn = fmaxf(m, wave_max(sm)), f = exp2_hw(m - mn);
        const float e = mine && lane < kRound ? exp2_hw(sm - mn) : 0.f;
        m = mn;
        l = fmaf(l, f, wave_sum(mine && lane < kRound ? sl_ * e : 0.f));
        o *= f;
#pragma unroll
        for (int i = 0; i < kRound; ++i)
            if (s0 + 2 * i < n) o = fmaf(value_of(v[i]), __shfl(e, i), o);
    }
}

// grid (nkv, splits), block 512.
__global__ void __launch_bounds__(kWaves* kWave) attn_split_kernel(const float* q, const uint16_t* kc, const uint16_t* vc,
                                                                   const int* d_pos, Partials part, float* out, int max_seq) {
    __shared__ float so[kWaves][kGroup][kHd];  // [wave][head][column]
    __shared__ float sml[kWaves][kGroup][2];   // [wave][head] m, l

    // The group's 4 queries, the lane's 8 columns of each.
    float qr[kGroup][8];
#pragma unroll
    for (int h = 0; h < kGroup; ++h)
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(q + (blockIdx.x * kGroup + h) * kHd + threadIdx.x % 8 * 8 + e);
#pragma unroll
            for (int i = 0; i < 4; ++i) qr[h][e + i] = v[i];
        }
    const int kvh = blockIdx.x, split = blockIdx.y, splits = gridDim.y;
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int g = lane / 8, c = lane % 8;
    // A tile's first row as a uniform base, then the lane's offset; rows past `last` (in the tile) read that one again.
    auto load = [&](KvTile& kv, int tile, int last) {
        const size_t first = (static_cast<size_t>(kvh) * max_seq + static_cast<size_t>(tile) * kTile) * kHd;
        const char* K = reinterpret_cast<const char*>(kc + first);
        const char* V = reinterpret_cast<const char*>(vc + first);
#pragma unroll
        for (int r = 0; r < kTileRows; ++r) {
            const uint32_t off = min(8 * r + g, last) * (kHd * 2) + c * 16;
            kv.k[r] = load_stream(K + off);
            kv.v[r] = load_stream(V + off);
        }
    };
    // Wave wi takes tile wi and then its share of the tiles past one for each wave, in one piece (dealt in turn, 60 against
    // 53 us at 131071 tokens).  The first tile does not depend on *d_pos, so the first split's waves request theirs before
    // it has arrived (rows of the cache past ctx weigh nothing), a memory round trip less for short contexts: 100 tokens
    // 5.3 -> 4.1 us.  The other splits wait, for they may have nothing to do.
    const int wi = split * kWaves + w;
    KvTile A, B;
    const bool early = split == 0 && (w + 1) * kTile <= max_seq;
    if (early) load(A, wi, kTile - 1);
    const int ctx = *d_pos + 1;
    const int tiles = (ctx + kTile - 1) / kTile, used = min(splits, (tiles + kWaves - 1) / kWaves), waves = kWaves * used;
    if (split >= used) return;
    auto last_of = [&](int tile) { return ctx - 1 - tile * kTile; };
    Running st;
#pragma unroll
    for (int h = 0; h < kGroup; ++h) {
        st.m[h] = -FLT_MAX;
        st.l[h] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) st.o[h][e] = 0.f;
    }
    if (wi < tiles) {
        auto step = [&](const KvTile& kv, int tile) { attend(kv, qr, st, tile * kTile, g, ctx); };
        const uint64_t more = max(tiles - waves, 0);
        int t = wi, next = waves + static_cast<int>(more * wi / waves);
        const int end = waves + static_cast<int>(more * (wi + 1) / waves);
        if (!early) load(A, t, last_of(t));
        for (;;) {
            if (next >= end) {
                step(A, t);
                break;
            }
            load(B, next, last_of(next));
            __builtin_amdgcn_sched_barrier(0);  // the next tile's loads go out before this tile's math
            step(A, t);
            t = next++;
            if (next >= end) {
                step(B, t);
                break;
            }
            load(A, next, last_of(next));
            __builtin_amdgcn_sched_barrier(0);
            step(B, t);
            t = next++;
        }
    }

    // The wave's 8 token phases: every phase is rescaled to the head's maximum, then summed by exchanges that halve the
    // values a lane holds: lane bits 5 and 4 pick the head, bit 3 the half of the lane's 8 columns.
    float M[kGroup];
#pragma unroll
    for (int h = 0; h < kGroup; ++h) {
        M[h] = phase_max(st.m[h]);
        const float f = exp2_hw(st.m[h] - M[h]);
        st.l[h] = phase_sum(st.l[h] * f);
#pragma unroll
        for (int e = 0; e < 8; ++e) st.o[h][e] *= f;
    }
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
        x[e] = fold_lanes<16>(fold_lanes<32>(st.o[0][e], st.o[1][e]), fold_lanes<32>(st.o[2][e], st.o[3][e]));
    const bool odd = lane & 8;
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = (odd ? x[e + 4] : x[e]) + dpp<kDppRor8>(odd ? x[e] : x[e + 4]);
    *reinterpret_cast<f32x4*>(&so[w][(lane >> 5) + 2 * ((lane >> 4) & 1)][c * 8 + (odd ? 4 : 0)]) = y;
    if (lane < kGroup) {
        float m = M[0], l = st.l[0];
#pragma unroll
        for (int h = 1; h < kGroup; ++h)
            if (lane == h) m = M[h], l = st.l[h];
        sml[w][lane][0] = m;
        sml[w][lane][1] = l;
    }
    __syncthreads();

    // Waves 0-3 take a head each: the 8 waves' partials in wave order.
    const int h = kvh * kGroup + w % kGroup;
    float m = -FLT_MAX, l = 0.f, o = 0.f;
    if (w < kGroup) {
#pragma unroll
        for (int i = 0; i < kWaves; ++i) m = fmaxf(m, sml[i][w][0]);
#pragma unroll
        for (int i = 0; i < kWaves; ++i) {
            const float f = exp2_hw(sml[i][w][0] - m);
            l = fmaf(sml[i][w][1], f, l);
            o = fmaf(so[i][w][lane], f, o);
        }
        if (used == 1) {
            out[h * kHd + lane] = o / l;
        } else if (split + 1 < used) {
            const size_t slot = static_cast<size_t>(h) * splits + split;
            tag_store(part.o + slot * kHd + lane, o, part.tag);
            if (lane < 2) tag_store(part.ml + slot * 2 + lane, lane ? l : m, part.tag);
        }
    }
    if (split + 1 < used || used == 1) return;

    // The last split: each head's other splits in two halves (waves w and w + 4), then the head's three partials.
    float om, ol, oo;
    merge_half(part, h, splits, used - 1, w / kGroup, lane, om, ol, oo);
    __syncthreads();  // waves 0-3 have read so and sml
    so[w][0][lane] = oo;
    if (lane == 0) sml[w][0][0] = om, sml[w][0][1] = ol;
    __syncthreads();
    if (w < kGroup) {
        const float m1 = sml[w + kGroup][0][0], l1 = sml[w + kGroup][0][1], o1 = so[w + kGroup][0][lane];
        const float M = fmaxf(fmaxf(om, m1), m), f0 = exp2_hw(om - M), f1 = exp2_hw(m1 - M), f = exp2_hw(m - M);
        out[h * kHd + lane] = (oo * f0 + o1 * f1 + o * f) / (ol * f0 + l1 * f1 + l * f);
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
    // A word takes two of the caller's floats (and the first may lie one float further on, at 8 bytes).
    const bool slack = (reinterpret_cast<uintptr_t>(part_o) | reinterpret_cast<uintptr_t>(part_ml)) & 7;
    const int splits = std::max(1, std::min({(max_seq / kAttnChunk - slack) / 2, kSplitBlocks / nkv, kMaxSplits}));
    auto words = [](float* p) { return reinterpret_cast<uint64_t*>((reinterpret_cast<uintptr_t>(p) + 7) & ~uintptr_t{7}); };
    static std::atomic<uint32_t> launches{0};
    const Partials part{words(part_o), words(part_ml), 0xFFC00000u | (launches.fetch_add(1, std::memory_order_relaxed) & 0x3FFFFFu)};
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
    // No clearing needed: every split at or before ctx writes its slots before the merge reads them, and the merge
    // reads no other slot.
    launch_attention_splitk(q, k_cache, v_cache, d_pos, base, base + static_cast<size_t>(kStaticAttnSlots) * kHd, out,
                            nh, nkv, hd, max_seq, s);
}

}  // namespace cllm
