// Batch-1 weight-streaming matvec for gfx950 (wave64), included by one translation unit per weight
// type.  Behaviour follows reference src/kernels/matvec_opt.cu:43-157 (y = W x^ with an fp32
// accumulator, optional fused RMSNorm prologue, STORE / ADD / SWIGLU epilogue, int8 scale per row,
// int4 fp16 scale per 128 columns); the work decomposition is this file's own:
//
//  * A workgroup is 4 waves.  Columns are cut into 2048-wide slices; KS = cols/2048 waves share
//    one row (one slice each), so the 4 waves of a workgroup cover 4/KS row groups.
//  * Every lane owns a fixed set of 32 columns of its slice: the 16-byte chunks lane, lane+64, ...
//    (8 bf16 / 16 int8 / 32 int4 columns per chunk).  Those 32 inputs - normalised when the norm
//    is fused - are read and normalised once per workgroup, handed to the lanes through LDS and kept in
//    VGPRs for every row the wave touches, so the inner loop reads no LDS at all: only 128-bit
//    non-temporal weight loads, 64 lanes x 16 B = 1 KiB contiguous per load instruction.
//  * R rows (rpb) are loaded before any is consumed, for R x (4 KiB bf16 | 2 KiB int8 | 1 KiB int4)
//    of loads per pass; a wave issues the next pass's loads before it multiplies the current one,
//    so up to 2R rows are in flight.  The first pass's weights are requested right after the lane's
//    inputs, before the norm and digit prologue, and with them, for some quantised forms, what is read
//    beside the sums at the end.  No load sits under a branch (rows past the end re-read the last row)
//    and, with KS = 1, no store sits in the loop (each wave's row sums wait in its lanes until its last
//    pass): either made the compiler's wait counts conservative, so that a pass also waited for the next
//    pass's loads (128256 x 2048, bf16 82.5 -> 80.0 us, int8 44.6 -> 40.5,
//    int4 32.2 -> 28.0).  With the launches of small.hip the same shape now takes 76.5, 39.5 and 23.2 us on
//    MI355X: 6.9, 6.7 and 5.8 TB/s, where a plain stream read reaches 7.1.
//  * Quantised 2048-wide rows (KS = 1) use integer digit dots: the workgroup turns the inputs into
//    fixed-point digit words once (with a scale for each 16-byte chunk's columns), and a row then costs
//    24 v_dot8_i32_i4 / v_dot4_i32_i8 per lane instead of a conversion and an FMA per column.  A scale per chunk
//    instead of one per row costs up to 2 % (128256 x 2048 int4 22.8 -> 23.2 us, int8 39.3 -> 39.5; 3072 x 2048
//    2.82 -> 2.83 and 3.21 -> 3.26; 16384 x 2048 SWIGLU 5.23 -> 5.23 and 7.44 -> 7.49).  The 8192-wide down rows (KS = 4) keep the float path.
//  * Row sums are wave64 DPP butterflies (deterministic order); with KS > 1 the slice partials
//    meet in LDS and are added in slice order.  No atomics anywhere.
//  * The grid: min(row blocks, CUs x the shape class's workgroups per CU (grid_per_cu)), but with
//    KS = 1 at least enough workgroups that none takes more than 64 / R passes.
//
// Widths other than 2048 and 8192 (and some of 8192, see pick_shape) use matvec_wide, which stages x in LDS.
#pragma once

#include <algorithm>

#include <hip/hip_ext.h>

#include "../kernels.h"
#include "device.h"
#include "digits.h"
#include "dot.h"

namespace cllm {
namespace mv {

constexpr int kSlice = 2048;
constexpr int kThreads = 256;
// Passes of R rows per wave with KS = 1: the wave's row sums wait in its 64 lanes until the end.
template <int R>
constexpr int kMaxPasses = kWave / R;

template <Epilogue EP>
__device__ __forceinline__ void store_out(float* y, int r, float d, float du) {
    if constexpr (EP == Epilogue::STORE) {
        y[r] = d;
    } else if constexpr (EP == Epilogue::ADD) {
        y[r] = y[r] + d;
    } else {
        y[r] = silu(d) * du;
    }
}

// The fixed-point scale of the digits here fills the digits' whole range (|xi| up to about 2^23, a bit more than the decode
// kernel's words of digits.h hold).  An input is rounded by up to 2^-24 .. 2^-23 of the largest |x^| that shares its scale:
// those of one chunk, 16 columns of int8 or 32 of int4.  Errors against 64 bits, root mean square over 12 seeds, with x^ in
// floats and every weight converted / with one scale for a whole row / with one per chunk:
//                                   normal inputs              one 1000 to 2000 times the rest  it meets zero weights
//   int4  8192 x 4096 norm, SWIGLU  9.4e-7 / 4.2e-7 / 2.7e-7   8.8e-7 / 5.3e-6 / 5.1e-7         2.0e-5 / 1.2e-4 / 1.0e-5
//   int8  4096 x 12288              4.0e-7 / 2.5e-7 / 1.6e-7   3.9e-7 / 5.3e-6 / 2.1e-7         4.8e-6 / 7.1e-5 / 2.5e-6
//   int4  3072 x 2048 norm                 - / 2.8e-7 / 1.7e-7        - / 2.5e-6 / 3.2e-7              - / 7.8e-5 / 9.3e-6
// (The floats lose the bits of the large input's chunk to the bias of the converted weights.)  A scale per row also needed
// the largest |x norm_w| before the norm was known, which is infinite for products past the floats whose x^ are not.
template <WType WT>
__device__ __forceinline__ int wide_exponent(float m) {
    if (!(m > 0.f) || !(m < INFINITY)) return 0;
    constexpr float kMost = WT == WType::INT8 ? 8355700.f : 7829350.f;  // 127 (1 + 256 + 256^2), 7 (1 + 16 + ... + 16^5)
    const int e = min(22 - ilogbf(m), 126);
    return ldexpf(m, e) > kMost ? e - 1 : e;
}
__device__ __forceinline__ uint32_t wide_word(float v, float scale, uint32_t C) {
    return static_cast<uint32_t>(static_cast<int>(rintf(v * scale))) + C;
}

// A thread has 8 neighbouring x^ (thread j columns 8 j ..): the scale of its chunk's fixed-point words, from the chunk's
// largest |x^|; the inverse goes to chunk_scale[chunk] (NaN if one of them is infinite or NaN: the chunk's dots then are).
template <WType WT>
__device__ __forceinline__ float set_chunk_scale(const float* v, int j, float* chunk_scale) {
    constexpr int THREADS = Fmt<WT>::CPC / 8;  // per chunk, neighbours
    float m = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) m = fabsf(v[e]) < INFINITY ? fmaxf(m, fabsf(v[e])) : INFINITY;
    m = fmaxf(m, dpp<kDppXor1>(m));
    if constexpr (THREADS == 4) m = fmaxf(m, dpp<kDppXor2>(m));
    const int e = wide_exponent<WT>(m);
    if (j % THREADS == 0) chunk_scale[j / THREADS] = m < INFINITY ? ldexpf(1.f, -e) : __builtin_nanf("");
    return ldexpf(1.f, e);
}

typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
constexpr int kAuxNt = 2;  // non-temporal

template <WType WT, Epilogue EP, bool NORM, int KS, int R>
__global__ void __launch_bounds__(kThreads) matvec_fast(MatvecArgs a) {
    using F = Fmt<WT>;
    constexpr int NX = F::CPL * F::CPC;  // 32 inputs per lane
    constexpr int GROUPS = 4 / KS;
    constexpr int ROWS_WG = GROUPS * R;
    constexpr bool GLU = EP == Epilogue::SWIGLU;
    constexpr int NP = GLU ? 2 : 1;
    constexpr bool DIG = WT != WType::BF16 && KS == 1;
    // Quantised 8192-wide rows: what the merge of the slices reads (old outputs, int8's scales) comes with the pass's
    // weights instead of after its sums.  20000 rows int8 30.7 -> 27.9 us, int4 22.4 -> 20.9; 2048 rows 5.73 -> 5.59, 5.20 ->
    // 5.10.  bf16, where a pass is twice the bytes, gains nothing (20000 rows 52.6 -> 53.2) and reads them in the merge.
    constexpr bool EARLY = KS > 1 && WT != WType::BF16;
    // Likewise the rows' sums of quantised ADD with KS = 1, once for all passes: 512 rows int8 2.86 -> 2.58 us, int4 2.94 ->
    // 2.67; 2048 rows 3.20 -> 3.15, 3.08 -> 2.92; 20483 rows 8.81 -> 8.68, 6.22 -> 6.10.  Not int8's scales of STORE (3072 rows
    // 3.24 against 3.27) and SWIGLU (16384 rows 7.48 against 7.66), nor bf16 (512 rows 2.75 against 3.02).
    constexpr bool EARLY_SUM = KS == 1 && WT != WType::BF16 && EP == Epilogue::ADD;
    // x^ by lines of 64 chunks, a lane's 16-byte words of a line at [line][word][lane]: the digits of a chunk, or its
    // floats.  One copy with KS = 1, a slice per wave with KS > 1.
    constexpr int XW = !DIG ? F::CPC / 4 : WT == WType::INT4 ? 6 : 3;
    __shared__ u32x4 xs[KS][F::CPL * XW * kWave];
    __shared__ float chunk_scale[DIG ? kSlice / F::CPC : 1];
    __shared__ float scratch[4];
    __shared__ float part[KS > 1 ? KS * ROWS_WG * NP : 1];

    const int tid = threadIdx.x;
    // The wave index through readfirstlane: the compiler then knows it is uniform, so every row index and weight
    // address derived from it is computed once per wave in scalar registers instead of in every lane.
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int slice = wave % KS, grp = wave / KS;
    const int out_rows = GLU ? a.rows / 2 : a.rows;
    // Row blocks are dealt to the workgroups in turn; base is the same for every wave of a workgroup, so the
    // barriers below (the prologue's, and pass()'s with KS > 1) are reached by all of them.
    const int stride = gridDim.x * ROWS_WG;
    int base = blockIdx.x * ROWS_WG;
    if (base >= out_rows) return;
    int left = (out_rows - base + stride - 1) / stride;  // passes of this workgroup, >= 1

    // The inputs (and norm weights) are requested first, then the first pass's weights, so that the prologue below waits
    // only for the short input loads while the weight bytes are already in flight (loads complete in order, so requesting
    // the weights first would make the prologue wait for them).  They are read in consecutive 16-byte words and change
    // hands in LDS: with KS = 1 thread t takes columns 8 t .. 8 t + 7 of the row that all four waves share, with KS > 1 a
    // wave takes its own slice.  Read the way the lanes use them (32 columns at a stride of 32 to 128 bytes, by every
    // wave), each load touched up to 64 lines: int4 512 x 2048 4.3 us against 2.8 for bf16.
    constexpr int XV = KS == 1 ? 2 : NX / 4;
    f32x4 xin[XV], nwin[NORM ? XV : 1];
#pragma unroll
    for (int i = 0; i < XV; ++i) {
        const int j = KS == 1 ? 2 * tid + i : slice * (kSlice / 4) + i * kWave + lane;
        xin[i] = reinterpret_cast<const f32x4*>(a.x)[j];
        if constexpr (NORM) nwin[i] = reinterpret_cast<const f32x4*>(a.norm_w)[j];
    }
    const size_t rb = row_bytes<WT>(a.cols);
    // Addresses are a row base that is uniform across the wave (scalar registers) plus a 32-bit lane offset, the
    // form of a load with a scalar base: one offset register per lane instead of a 64-bit address per row.
    const char* wbase = static_cast<const char*>(a.w);
    const uint32_t woff = static_cast<uint32_t>(slice * (kSlice * 16 / F::CPC) + lane * 16);
    const int groups_per_row = a.cols / 128;
    // int4: one 128-column group per lane; lanes 4g..4g+3 share scale g of the slice.
    const uint16_t* sbase = static_cast<const uint16_t*>(a.scales);
    const uint32_t soff = static_cast<uint32_t>(slice * (kSlice / 128) + lane / 4);

    // The R rows of one pass: weight chunks and, for int4, the lane's group scales.  Two of these alternate, so the
    // next pass's loads are in flight while this pass is multiplied.
    struct Block {
        u32x4 v[R][F::CPL];
        u32x4 vu[GLU ? R : 1][F::CPL];
        uint16_t g[R], gu[R];
        float y, sc, scu;  // EARLY: of the thread's row in the merge
    };
    // Rows past the end load the last row again (their sums are never stored): with no branch around the loads the
    // compiler counts them exactly, so a pass waits only for its own loads and not for the next pass's as well.
    auto load = [&](Block& b, int r0) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int rc = min(r0 + i, out_rows - 1);
            const char* row = wbase + static_cast<size_t>(rc) * rb;
            const char* row_u = wbase + static_cast<size_t>(rc + out_rows) * rb;
#pragma unroll
            for (int k = 0; k < F::CPL; ++k) {
                b.v[i][k] = load_stream(row + woff + k * 1024);
                if constexpr (GLU) b.vu[i][k] = load_stream(row_u + woff + k * 1024);
            }
            if constexpr (WT == WType::INT4) {
                b.g[i] = gload(sbase + static_cast<size_t>(rc) * groups_per_row + soff);
                if constexpr (GLU) b.gu[i] = gload(sbase + static_cast<size_t>(rc + out_rows) * groups_per_row + soff);
            }
        }
        if constexpr (EARLY) {
            const int rc = min(r0 - grp * R + min(tid, ROWS_WG - 1), out_rows - 1);
            if constexpr (EP == Epilogue::ADD) b.y = a.y[rc];
            if constexpr (WT == WType::INT8) {
                b.sc = static_cast<const float*>(a.scales)[rc];
                if constexpr (GLU) b.scu = static_cast<const float*>(a.scales)[rc + out_rows];
            }
        }
    };
    Block A, B;
    load(A, base + grp * R);
    [[maybe_unused]] float old_y = 0.f, sum_scale = 1.f;
    if constexpr (EARLY_SUM) {  // the row that lane l keeps to the end
        const int rc = min(base + min(lane / R, left - 1) * stride + grp * R + lane % R, out_rows - 1);
        old_y = a.y[rc];
        if constexpr (WT == WType::INT8) sum_scale = static_cast<const float*>(a.scales)[rc];
    }
    __builtin_amdgcn_sched_barrier(0);  // keep the weight loads ahead of the prologue

    if constexpr (NORM) {
        float ss = 0.f;
#pragma unroll
        for (int q = 0; q < XV; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) ss = fmaf(xin[q][e], xin[q][e], ss);
        ss = wave_sum(ss);
        if (lane == 0) scratch[wave] = ss;
        __syncthreads();
        ss = ((scratch[0] + scratch[1]) + scratch[2]) + scratch[3];
        const float inv = rsqrtf(ss / static_cast<float>(a.cols) + a.eps);
#pragma unroll
        for (int q = 0; q < XV; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) xin[q][e] = xin[q][e] * inv * nwin[q][e];
    }
    if constexpr (DIG) {
        // Digit words of the thread's 8 columns in the weight words' layout, with their chunk's scale.
        uint32_t* const xw = reinterpret_cast<uint32_t*>(xs[0]);
        const float v8[8] = {xin[0][0], xin[0][1], xin[0][2], xin[0][3], xin[1][0], xin[1][1], xin[1][2], xin[1][3]};
        const float scale = set_chunk_scale<WT>(v8, tid, chunk_scale);
        if constexpr (WT == WType::INT8) {
            const int at = (tid / 2 / kWave * XW * kWave + tid / 2 % kWave) * 4 + tid % 2 * 2;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t P[3];
                byte_planes(wide_word(xin[h][0], scale, 0x808080u), wide_word(xin[h][1], scale, 0x808080u),
                            wide_word(xin[h][2], scale, 0x808080u), wide_word(xin[h][3], scale, 0x808080u), P);
#pragma unroll
                for (int d = 0; d < 3; ++d) xw[at + d * kWave * 4 + h] = P[d] ^ 0x80808080u;
            }
        } else {
            uint32_t u[8], w[6];
#pragma unroll
            for (int e = 0; e < 8; ++e) u[e] = wide_word(xin[e / 4][e % 4], scale, 0x888888u);
            nibble_words(u, w);
#pragma unroll
            for (int d = 0; d < 6; ++d) xw[d * kWave * 4 + tid] = w[d] ^ 0x88888888u;
        }
    } else {
#pragma unroll
        for (int i = 0; i < XV; ++i) {
            const int j = KS == 1 ? 2 * tid + i : i * kWave + lane, c = j / XW;
            xs[KS == 1 ? 0 : slice][(c / kWave * XW + j % XW) * kWave + c % kWave] = __builtin_bit_cast(u32x4, xin[i]);
        }
    }
    if constexpr (KS == 1) {
        __syncthreads();
    } else {  // a wave reads what it wrote
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }

    // The lane's inputs: digit words (int8 digit k of chunk c, word t (columns 4t .. 4t + 3) at dg[(2k + c) 4 + t]; int4
    // digit k of word t (columns 8t .. 8t + 7) at dg[4k + t]) or 32 floats and their sum.
    [[maybe_unused]] uint32_t dg[DIG ? 24 : 1];
    [[maybe_unused]] float xscale[DIG ? F::CPL : 1];
    if constexpr (DIG)
#pragma unroll
        for (int k = 0; k < F::CPL; ++k) xscale[k] = chunk_scale[k * kWave + lane];
    [[maybe_unused]] float xr[DIG ? 1 : NX], xsum = 0.f;
#pragma unroll
    for (int k = 0; k < F::CPL; ++k)
#pragma unroll
        for (int q = 0; q < XW; ++q) {
            const u32x4 v = xs[KS == 1 ? 0 : slice][(k * XW + q) * kWave + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (DIG) {
                    dg[(q * F::CPL + k) * 4 + e] = v[e];
                } else {
                    xr[k * F::CPC + 4 * q + e] = __builtin_bit_cast(f32x4, v)[e];
                    xsum += xr[k * F::CPC + 4 * q + e];
                }
            }
        }

    // KS = 1: the row sums wait in lanes (lane j: the wave's j-th row) and are stored after the last pass, so no store
    // sits in the loop (a store there made the loop's head wait for the previous pass's loads).  The host keeps every
    // wave within kMaxPasses<R> passes, so 64 lanes hold them all.
    [[maybe_unused]] float acc = 0.f, acc_u = 0.f;
    [[maybe_unused]] int acc_row = -1, held = 0;
    auto pass = [&](const Block& b, int base) {
        const int r0 = base + grp * R;
        float d[R], du[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            if constexpr (DIG) {
                // Per chunk: int8 sum_k 256^k sum(q d_k); int4 sum_k 16^k sum(q d_k) (nibble u = q + 8, so q = u xor 8)
                // times the lane's group scale; times the chunk's scale (and the row's sum times the int8 row scale at the store).
                auto dot = [&](const u32x4* v, uint16_t g) {
                    if constexpr (WT == WType::INT8) {
                        float sum = 0.f;
#pragma unroll
                        for (int c = 0; c < 2; ++c) {
                            int p[3] = {0, 0, 0};
#pragma unroll
                            for (int t = 0; t < 4; ++t)
#pragma unroll
                                for (int k = 0; k < 3; ++k)
                                    p[k] = __builtin_amdgcn_sdot4(static_cast<int>(v[c][t]), static_cast<int>(dg[(2 * k + c) * 4 + t]), p[k], false);
                            // p[0] + 256 p[1] stays below 2^27.
                            sum = fmaf(fmaf(static_cast<float>(p[2]), 65536.f, static_cast<float>(p[0] + 256 * p[1])), xscale[c], sum);
                        }
                        return sum;
                    } else {
                        int ac[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            const int w = static_cast<int>(v[0][t] ^ 0x88888888u);
#pragma unroll
                            for (int k = 0; k < 6; ++k) ac[k] = __builtin_amdgcn_sdot8(w, static_cast<int>(dg[4 * k + t]), ac[k], false);
                        }
                        const int p0 = ac[0] + 16 * ac[1], p1 = ac[2] + 16 * ac[3], p2 = ac[4] + 16 * ac[5];
                        const float p = fmaf(static_cast<float>(p2), 65536.f, static_cast<float>(p0 + 256 * p1));
                        return p * xscale[0] * half_bits_to_float(g);
                    }
                };
                d[i] = dot(b.v[i], b.g[i]);
                du[i] = 0.f;
                if constexpr (GLU) du[i] = dot(b.vu[i], b.gu[i]);
            } else {
                float s = 0.f, su = 0.f;
#pragma unroll
                for (int k = 0; k < F::CPL; ++k) {
                    s += chunk_dot<WT>(b.v[i][k], xr + k * F::CPC);
                    if constexpr (GLU) su += chunk_dot<WT>(b.vu[i][k], xr + k * F::CPC);
                }
                if constexpr (WT == WType::INT8) {
                    s -= kBias<WT> * xsum;
                    if constexpr (GLU) su -= kBias<WT> * xsum;
                }
                if constexpr (WT == WType::INT4) {
                    s = half_bits_to_float(b.g[i]) * (s - 8.f * xsum);
                    if constexpr (GLU) su = half_bits_to_float(b.gu[i]) * (su - 8.f * xsum);
                }
                d[i] = s;
                du[i] = su;
            }
        }
        // Lane l: the sums of row r0 + (l mod R).  int4's 2048-wide rows (1 KiB, the
        // most rows per byte) reduce all R rows at once (rows_sum: int4 lm_head 28.2 -> 26.2 us, gate_up 8.0 -> 7.3 us
        // on MI355X); the other forms keep a full reduction per row, which measured as fast or faster for them (bf16
        // down 7.3 against 8.4 us).
        float tot = 0.f, tot_u = 0.f;
        if constexpr (WT == WType::INT4 && KS == 1) {
            tot = rows_sum<R>(d, lane);
            if constexpr (GLU) tot_u = rows_sum<R>(du, lane);
        } else {
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const float si = wave_sum(d[i]);
                const float sui = GLU ? wave_sum(du[i]) : 0.f;
                if (lane % R == i) {
                    tot = si;
                    tot_u = sui;
                }
            }
        }
        if constexpr (KS == 1) {
            // Lane held + i keeps row r0 + i until the wave's last pass (no store inside the loop); held is a multiple
            // of R, so that lane already holds row i's sum.
            if (lane >= held && lane < held + R) {
                acc = tot;
                acc_u = tot_u;
                acc_row = r0 + lane - held;
            }
            held += R;
        } else {
            // Lane i (< R) holds row r0 + i.
            const float mine = tot, mine_u = tot_u;
            if (lane < R) {
                const int slot = (slice * ROWS_WG + grp * R + lane) * NP;
                part[slot] = mine;
                if constexpr (GLU) part[slot + 1] = mine_u;
            }
            __syncthreads();
            if (tid < ROWS_WG && base + tid < out_rows) {
                const int r = base + tid;
                float s = 0.f, su = 0.f;
#pragma unroll
                for (int q = 0; q < KS; ++q) {
                    s += part[(q * ROWS_WG + tid) * NP];
                    if constexpr (GLU) su += part[(q * ROWS_WG + tid) * NP + 1];
                }
                if constexpr (WT == WType::INT8) {
                    s *= b.sc;
                    if constexpr (GLU) su *= b.scu;
                }
                if constexpr (EARLY && EP == Epilogue::ADD) {
                    a.y[r] = b.y + s;
                } else {
                    store_out<EP>(a.y, r, s, su);
                }
            }
            __syncthreads();
        }
    };

    // One pass's loads are outstanding at the top of each half; the next pass is requested before this one is
    // multiplied.  No load sits under a branch, so each pass waits only for its own loads.
    for (;;) {
        if (left == 1) {
            pass(A, base);
            break;
        }
        load(B, base + stride + grp * R);
        __builtin_amdgcn_sched_barrier(0);  // issue the next pass's loads before this pass's math
        pass(A, base);
        base += stride;
        --left;
        if (left == 1) {
            pass(B, base);
            break;
        }
        load(A, base + stride + grp * R);
        __builtin_amdgcn_sched_barrier(0);
        pass(B, base);
        base += stride;
        --left;
    }
    if constexpr (KS == 1) {
        if (lane < held && acc_row < out_rows) {
            if constexpr (EARLY_SUM) {
                a.y[acc_row] = old_y + acc * sum_scale;
            } else {
                if constexpr (WT == WType::INT8) {
                    const float* sc = static_cast<const float*>(a.scales);
                    acc *= sc[acc_row];
                    if constexpr (GLU) acc_u *= sc[acc_row + out_rows];
                }
                store_out<EP>(a.y, acc_row, acc, acc_u);
            }
        }
    }
}

// ---- any width: cols a multiple of 1024, up to 12288 -----------------------------------------------------
//
// Bound by the weight bytes (int4 by instruction issue beside them).  x^ is staged in LDS once per workgroup in the order
// in which the lanes of a wave read it, so a wave takes whole rows of any width: a step is one 1 KiB line (64 chunks) of
// two rows, the gate and the up row with SWIGLU, else two neighbours, which share the LDS reads of x^.  The quantised
// types stage x^ as digit words (a line's digit d of lane l at [line][d][l], 16 bytes; a third to a half of the
// instructions of converting every weight) with a scale of its own for every lane's chunk (one scale for the row measured
// no faster: 24576 x 4096 int4 11.5 us both, 4096 x 12288 int4 8.6 against 8.5, int8 11.6 against 11.3), bf16 as float4s
// ([line][quad][l]).  The steps of all of a wave's rows
// are one sequence with kDepth steps in flight; the loads are buffer loads, so the ones past the wave's last row and past
// a row's end (widths that are not a whole number of lines) return 0 without a memory access and no load sits under a
// branch.  Row sums wait in LDS for the wave's end, so no store sits in the loop either.
constexpr int kWideWaves = 8, kWideThreads = kWideWaves * kWave;
constexpr int kWideMaxUnits = 64;  // row pairs per wave
constexpr int kXPairs = 12288 / 8 / kWideThreads;  // a thread stages 8 columns at a time
// Steps in flight per wave.  int4 has the most instructions per step, and a third copy of them in the loop costs more
// than it hides: 24576 x 4096 with depths 2, 3 and 4: bf16 35.9 / 34.9 / 34.9 us, int8 21.0 / 19.2 / 19.3, int4 12.3 /
// 13.2 / 14.2; 1000 x 1024: bf16 3.1 / 3.1 / 3.5, int8 3.4 / 3.5 / 3.9, int4 3.6 / 4.0 / 4.2.
template <WType WT>
constexpr int kDepth = WT == WType::INT4 ? 2 : 3;

template <WType WT>
struct Wide {
    using F = Fmt<WT>;
    static constexpr int Q = WT == WType::INT4 ? 6 : WT == WType::INT8 ? 3 : 2;  // 16-byte words of x^ per chunk
    static __host__ __device__ int lines(int cols) { return (cols / F::CPC + kWave - 1) / kWave; }
    // x^, the chunks' scales (quantised types), then the row sums.
    static size_t smem(int cols, int units_per_wave) {
        return static_cast<size_t>(lines(cols)) * kWave * (Q * 16 + (WT != WType::BF16 ? 4 : 0)) +
               sizeof(float) * kWideWaves * 2 * units_per_wave;
    }
};

template <WType WT, Epilogue EP, bool NORM>
__global__ void __launch_bounds__(kWideThreads) matvec_wide(MatvecArgs a, int units, int max_units) {
    using F = Fmt<WT>;
    constexpr bool GLU = EP == Epilogue::SWIGLU, DIG = WT != WType::BF16;
    constexpr int Q = Wide<WT>::Q;
    extern __shared__ u32x4 xs[];  // [line][Q][lane]
    __shared__ float sred[kWideWaves];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int nchunk = a.cols / F::CPC, nk = Wide<WT>::lines(a.cols), rem = nchunk - (nk - 1) * kWave;
    float* const chunk_scale = reinterpret_cast<float*>(xs + nk * Q * kWave);  // DIG: [line][lane]
    float* const sums = chunk_scale + (DIG ? nk * kWave : 0) + wave * 2 * max_units;

    // Units [u0, u0 + n) of this wave.
    const int64_t wi = blockIdx.x * kWideWaves + wave, nw = gridDim.x * kWideWaves;
    const int u0 = static_cast<int>(wi * units / nw), n = static_cast<int>((wi + 1) * units / nw) - u0;
    const int out_rows = GLU ? a.rows / 2 : a.rows;

    // x first, so that its wait does not include the weights.
    f32x4 xv[kXPairs][2], nv[NORM ? kXPairs : 1][2];
    const int pairs = a.cols / 8;  // a multiple of 128: all of a wave's lanes hold one, or none
#pragma unroll
    for (int i = 0; i < kXPairs; ++i) {
        xv[i][0] = xv[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (NORM) nv[i][0] = nv[i][1] = xv[i][0];
        if (i * kWideThreads + wave * kWave < pairs) {
            const int j = 2 * (i * kWideThreads + tid);
            xv[i][0] = reinterpret_cast<const f32x4*>(a.x)[j];
            xv[i][1] = reinterpret_cast<const f32x4*>(a.x)[j + 1];
            if constexpr (NORM) {
                nv[i][0] = reinterpret_cast<const f32x4*>(a.norm_w)[j];
                nv[i][1] = reinterpret_cast<const f32x4*>(a.norm_w)[j + 1];
            }
        }
    }

    // The wave's rows as two buffers: rows r0, r0 + pitch, ... and their partners.
    const uint32_t rb = static_cast<uint32_t>(row_bytes<WT>(a.cols)), pitch = GLU ? rb : 2 * rb;
    const int r0 = GLU ? u0 : 2 * u0;
    const char* w0 = static_cast<const char*>(a.w) + static_cast<size_t>(r0) * rb;
    const int rows_here = GLU ? n : min(2 * n, a.rows - r0);
    const Rsrc wa = make_rsrc(w0, rows_here * rb);
    const Rsrc wb = GLU ? make_rsrc(w0 + static_cast<size_t>(out_rows) * rb, rows_here * rb) : wa;
    const uint32_t second = GLU ? 0 : rb;
    // int4 group scales: one fp16 per 128 columns (4 chunks).
    const uint32_t sb = a.cols / 128 * 2, spitch = GLU ? sb : 2 * sb, ssecond = GLU ? 0 : sb;
    const char* s0 = static_cast<const char*>(a.scales) + static_cast<size_t>(r0) * sb;
    const Rsrc sa = WT == WType::INT4 ? make_rsrc(s0, rows_here * sb) : wa;
    const Rsrc sbu = WT == WType::INT4 && GLU ? make_rsrc(s0 + static_cast<size_t>(out_rows) * sb, rows_here * sb) : sa;

    struct Step {
        u32x4 v[2];
        uint16_t g[2];
    };
    const uint32_t full_off = lane * 16, last_off = lane < rem ? full_off : 0x80000000u;
    const uint32_t full_soff = lane / 4 * 2, last_soff = lane < rem ? full_soff : 0x80000000u;
    uint32_t row_off = 0, row_soff = 0;
    int lk = 0;  // the next step's line
    auto load = [&](Step& b) {
        const bool last = lk == nk - 1;
        const uint32_t off = row_off + lk * 1024 + (last ? last_off : full_off);
        b.v[0] = __builtin_amdgcn_raw_buffer_load_b128(wa, off, 0, kAuxNt);
        b.v[1] = __builtin_amdgcn_raw_buffer_load_b128(wb, off + second, 0, kAuxNt);
        if constexpr (WT == WType::INT4) {
            const uint32_t so = row_soff + lk * 32 + (last ? last_soff : full_soff);
            b.g[0] = __builtin_amdgcn_raw_buffer_load_b16(sa, so, 0, 0);
            b.g[1] = __builtin_amdgcn_raw_buffer_load_b16(sbu, so + ssecond, 0, 0);
        }
        row_off += last ? pitch : 0;
        row_soff += last ? spitch : 0;
        lk = last ? 0 : lk + 1;
    };
    Step st[kDepth<WT>];
#pragma unroll
    for (int d = 0; d < kDepth<WT>; ++d) load(st[d]);
    __builtin_amdgcn_sched_barrier(0);

    [[maybe_unused]] float inv = 1.f;
    if constexpr (NORM) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < kXPairs; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(xv[i][e / 4][e % 4], xv[i][e / 4][e % 4], ss);
        ss = wave_sum(ss);
        if (lane == 0) sred[wave] = ss;
        __syncthreads();
        ss = 0.f;
#pragma unroll
        for (int w = 0; w < kWideWaves; ++w) ss += sred[w];
        inv = rsqrtf(ss / static_cast<float>(a.cols) + a.eps);
    }
#pragma unroll
    for (int i = 0; i < kXPairs; ++i) {
        // A whole number of lines: columns past the row's end stay 0.
        if (i * kWideThreads + wave * kWave >= nk * kWave * F::CPC / 8) continue;
        const int j = i * kWideThreads + tid;  // columns 8 j .. 8 j + 7
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = xv[i][e / 4][e % 4];
            if constexpr (NORM) v[e] = v[e] * inv * nv[i][e / 4][e % 4];
        }
        uint32_t* const xw = reinterpret_cast<uint32_t*>(xs);
        [[maybe_unused]] float scale = 1.f;
        if constexpr (DIG) scale = set_chunk_scale<WT>(v, j, chunk_scale);
        if constexpr (WT == WType::BF16) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
                xs[(j / kWave * Q + q) * kWave + j % kWave] =
                    __builtin_bit_cast(u32x4, f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]});
        } else if constexpr (WT == WType::INT8) {
            const int c = j / 2, at = (c / kWave * Q * kWave + c % kWave) * 4 + j % 2 * 2;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t P[3];
                byte_planes(wide_word(v[4 * h], scale, 0x808080u), wide_word(v[4 * h + 1], scale, 0x808080u),
                            wide_word(v[4 * h + 2], scale, 0x808080u), wide_word(v[4 * h + 3], scale, 0x808080u), P);
#pragma unroll
                for (int d = 0; d < 3; ++d) xw[at + d * kWave * 4 + h] = P[d] ^ 0x80808080u;
            }
        } else {
            const int c = j / 4, at = (c / kWave * Q * kWave + c % kWave) * 4 + j % 4;
            uint32_t u[8], w[6];
#pragma unroll
            for (int e = 0; e < 8; ++e) u[e] = wide_word(v[e], scale, 0x888888u);
            nibble_words(u, w);
#pragma unroll
            for (int d = 0; d < 6; ++d) xw[at + d * kWave * 4] = w[d] ^ 0x88888888u;
        }
    }
    __syncthreads();

    // Row sums: floats, a line's exact integer dots times the chunk's scale (and int4's group scale) added line by line.
    float acc[2] = {0.f, 0.f};
    int k = 0, u = 0;
    auto step = [&](const Step& b) {
        u32x4 x[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) x[q] = xs[(k * Q + q) * kWave + lane];
        [[maybe_unused]] float xscale = 1.f;
        if constexpr (DIG) xscale = chunk_scale[k * kWave + lane];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if constexpr (WT == WType::BF16) {
                float xf[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) xf[e] = __builtin_bit_cast(f32x4, x[e / 4])[e % 4];
                acc[i] += chunk_dot<WT>(b.v[i], xf);
            } else if constexpr (WT == WType::INT8) {
                int c[3] = {0, 0, 0};
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int d = 0; d < 3; ++d)
                        c[d] = __builtin_amdgcn_sdot4(static_cast<int>(b.v[i][t]), static_cast<int>(x[d][t]), c[d], false);
                // c[0] + 256 c[1] stays below 2^27.
                acc[i] = fmaf(fmaf(static_cast<float>(c[2]), 65536.f, static_cast<float>(c[0] + 256 * c[1])), xscale, acc[i]);
            } else {
                int c[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int w = static_cast<int>(b.v[i][t] ^ 0x88888888u);
#pragma unroll
                    for (int d = 0; d < 6; ++d) c[d] = __builtin_amdgcn_sdot8(w, static_cast<int>(x[d][t]), c[d], false);
                }
                const int p0 = c[0] + 16 * c[1], p1 = c[2] + 16 * c[3], p2 = c[4] + 16 * c[5];
                const float p = fmaf(static_cast<float>(p2), 65536.f, static_cast<float>(p0 + 256 * p1));
                acc[i] = fmaf(p * xscale, half_bits_to_float(b.g[i]), acc[i]);
            }
        }
        if (++k == nk) {
            const float t = rows_sum<2>(acc, lane);
            if (lane < 2) sums[2 * u + lane] = t;
            acc[0] = acc[1] = 0.f;
            k = 0;
            ++u;
        }
    };
    for (int s = n * nk; s > 0; s -= kDepth<WT>) {
#pragma unroll
        for (int d = 0; d < kDepth<WT>; ++d) {
            if (d == 0 || s > d) step(st[d]);
            load(st[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int i = lane; i < (GLU ? n : 2 * n); i += kWave) {
        const int r = r0 + i;
        if (r >= out_rows) break;
        float d = sums[GLU ? 2 * i : i], du = GLU ? sums[2 * i + 1] : 0.f;
        if constexpr (WT == WType::INT8) {
            const float* sc = static_cast<const float*>(a.scales);
            d *= sc[r];
            if constexpr (GLU) du *= sc[r + out_rows];
        }
        store_out<EP>(a.y, r, d, du);
    }
}

// Launches a matvec kernel; when the thread has armed kernel events (arm_kernel_events), the dispatch itself
// records them at the kernel's start and end, so a benchmark times the kernel without the launch gap.
template <typename K, typename... Args>
void dispatch(K kernel, int grid, int threads, size_t smem, hipStream_t s, const Args&... args) {
    KernelEvents ev = take_kernel_events();
    if (ev.start)
        hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(threads), static_cast<uint32_t>(smem), s, ev.start, ev.stop, 0u, args...);
    else
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), smem, s, args...);
    CLLM_HIP(hipGetLastError());
}

template <WType WT, Epilogue EP, bool NORM, int KS, int R>
void launch_fast(const MatvecArgs& a, hipStream_t s) {
    auto k = matvec_fast<WT, EP, NORM, KS, R>;
    const int out_rows = EP == Epilogue::SWIGLU ? a.rows / 2 : a.rows;
    constexpr int ROWS_WG = (4 / KS) * R;
    const int need = (out_rows + ROWS_WG - 1) / ROWS_WG;
    // The shape class's workgroups per CU; but with KS = 1 no workgroup may take more than kMaxPasses<R> passes.
    const int grid = std::max(std::min(need, device_cu_count() * grid_per_cu(WT, EP, a.rows, a.cols)),
                              KS == 1 ? (need + kMaxPasses<R> - 1) / kMaxPasses<R> : 0);
    dispatch(k, grid, kThreads, 0, s, a);
}

template <WType WT, Epilogue EP, bool NORM>
void launch_wide(const MatvecArgs& a, hipStream_t s) {
    const int units = EP == Epilogue::SWIGLU ? a.rows / 2 : (a.rows + 1) / 2;
    // Two workgroups per CU, fewer if that leaves the waves with the same number of units, more so that none has over
    // kWideMaxUnits.
    const int most = device_cu_count() * 2 * kWideWaves;
    const int per_wave = std::min((units + most - 1) / most, kWideMaxUnits);
    const int grid = (units + kWideWaves * per_wave - 1) / (kWideWaves * per_wave);
    dispatch(matvec_wide<WT, EP, NORM>, grid, kWideThreads, Wide<WT>::smem(a.cols, per_wave), s, a, units, per_wave);
}

template <WType WT, Epilogue EP, bool NORM, int KS>
void pick_r(int rpb, const MatvecArgs& a, hipStream_t s) {
    switch (rpb) {
        case 1: return launch_fast<WT, EP, NORM, KS, 1>(a, s);
        case 2: return launch_fast<WT, EP, NORM, KS, 2>(a, s);
        case 4: return launch_fast<WT, EP, NORM, KS, 4>(a, s);
        case 8: return launch_fast<WT, EP, NORM, KS, 8>(a, s);
    }
    throw ArgError("matvec: rpb must be 1, 2, 4 or 8");
}

template <WType WT, Epilogue EP, bool NORM>
void pick_shape(int rpb, const MatvecArgs& a, hipStream_t s) {
    if (a.cols == 2048) return pick_r<WT, EP, NORM, 1>(rpb, a, s);
    // Quantised 8192-wide rows convert every weight in matvec_fast, for want of columns per wave to share the digits of
    // x^ with; with two matrices of many rows the any-width kernel's digits are faster for int4: SWIGLU without norm, rows
    // 4096 / 8192 / 30000, 7.3 / 11.9 / 36.0 -> 6.5 / 9.5 / 23.9 us.  int8 is no faster (7.9 / 13.4 / 39.4 against 8.1 /
    // 13.0 / 41.9; 6000 rows 10.8 against 12.1) but has a third of the error against 64 bits (8.0e-7 -> 2.5e-7).
    // Without SWIGLU matvec_fast stays ahead at most row counts (ADD, 2048 / 8192 / 16384 / 30000 rows: int8 5.6 / 12.9 /
    // 22.9 / 37.8 against 6.3 / 13.2 / 25.4 / 39.6, int4 4.9 / 9.9 / 16.4 / 27.0 against 5.8 / 10.3 / 15.7 / 24.0).
    if (a.cols == 8192 && !(WT != WType::BF16 && EP == Epilogue::SWIGLU && a.rows >= 4096)) return pick_r<WT, EP, NORM, 4>(rpb, a, s);
    return launch_wide<WT, EP, NORM>(a, s);
}

template <WType WT>
void launch_wt(Epilogue ep, const MatvecArgs& a, int rpb, hipStream_t s) {
    const bool norm = a.norm_w != nullptr;
    switch (ep) {
        case Epilogue::STORE:
            return norm ? pick_shape<WT, Epilogue::STORE, true>(rpb, a, s) : pick_shape<WT, Epilogue::STORE, false>(rpb, a, s);
        case Epilogue::ADD:
            return norm ? pick_shape<WT, Epilogue::ADD, true>(rpb, a, s) : pick_shape<WT, Epilogue::ADD, false>(rpb, a, s);
        case Epilogue::SWIGLU:
            return norm ? pick_shape<WT, Epilogue::SWIGLU, true>(rpb, a, s) : pick_shape<WT, Epilogue::SWIGLU, false>(rpb, a, s);
    }
    throw ArgError("matvec: bad epilogue");
}

}  // namespace mv

template <WType WT>
void launch_matvec_wt(Epilogue ep, const MatvecArgs& a, int rpb, hipStream_t s);

}  // namespace cllm
