// Config-5 class: S[b*seq + i, :] = softmax((Q[b,i,:] . K[b,:,:]^T) / div +
// bias), the composition of Call(MatMul) (kernel_buffers.cpp:406-432), the
// broadcast elementwise chain Add(Div(S, c), bias[j]) (poly.synth.cpp:
// 231-353) and the stable softmax (kernel_buffers.cpp:290-340).
//
// The output write (4 * batch * seq^2 bytes) bounds the class; the scores are
// a GEMM with K = dim on v_mfma_f32_32x32x16_f16. Forms, best first:
//   * two-pass, query-stationary (dim 128 at any length, dim 64 from 512 keys at
//     multiples of 128; up to 8192 keys): a statistics pass and a
//     recompute-and-write pass (scoreStatsQ / scoreStoreQ), rows' partial
//     statistics in artifact scratch;
//   * scores, then the softmax kernel in place over S (f16, multiples of 128
//     keys, head dims that are multiples of 16);
//   * a scalar f64 path for other dtypes and shapes.
#include <hip/hip_runtime.h>

#include <cstdio>

#include <stdint.h>

#include "exp2_poly.h"
#include "mlk_device_math.h"
#include "runtime_abi.h"
#include "xcd.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void scoresF16(const _Float16* __restrict__ Q,
                                                 const _Float16* __restrict__ K,
                                                 const float* __restrict__ bias,
                                                 float* __restrict__ S, int seq, int dim,
                                                 float div) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int tilesJ = seq / 128;
    const int tilesI = seq / 64;
    const int64_t b = blockIdx.x / (tilesI * tilesJ);
    const int rem = blockIdx.x % (tilesI * tilesJ);
    const int i0 = (rem / tilesJ) * 64 + (wave >> 1) * 32;
    const int j0 = (rem % tilesJ) * 128 + (wave & 1) * 64;
    const _Float16* q = Q + (b * seq + i0 + (lane & 31)) * dim + (lane >> 5) * 8;
    const _Float16* k0 = K + (b * seq + j0 + (lane & 31)) * dim + (lane >> 5) * 8;
    const _Float16* k1 = k0 + static_cast<int64_t>(32) * dim;
    f32x16 acc0, acc1;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        acc0[r] = 0.0f;
        acc1[r] = 0.0f;
    }
    for (int kk = 0; kk < dim; kk += 16) {
        const f16x8 a = *reinterpret_cast<const f16x8*>(q + kk);
        const f16x8 x0 = *reinterpret_cast<const f16x8*>(k0 + kk);
        const f16x8 x1 = *reinterpret_cast<const f16x8*>(k1 + kk);
        acc0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, x0, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, x1, acc1, 0, 0, 0);
    }
    const int col = lane & 31;
    const float bj0 = bias[j0 + col];
    const float bj1 = bias[j0 + 32 + col];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t row = b * seq + i0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        float* dst = S + row * seq + j0 + col;
        dst[0] = acc0[r] / div + bj0;
        dst[32] = acc1[r] / div + bj1;
    }
}

// ------------------------------------------------------------ two pass ----
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

// Query-stationary form of the two passes (head dim D 64 or 128, seq a
// multiple of 128, or at 128 bounded). A wave owns 32 query rows and holds their Q fragments in
// registers for the whole kernel; a workgroup of 4 waves (128 rows) streams one
// of NR ranges of the batch's keys through LDS in 128-key panels, double
// buffered, the next panel's global loads in flight during the current panel's
// MFMAs. Two workgroups share a CU: at most 256 registers per lane, and 68 KiB
// of LDS at D 128 (36 at 64), to which pass 1 adds 4 bytes for each key of its
// range; past 24 panels that leaves room for one. Scores by 64 x 128 tiles and a softmax over S in place read S
// back and each K element once per 64 rows: at D 64, 8 x 1024 took 23.5 us
// and takes 14.5, 16 x 2048 165 and 72.
//   Pass 1 (scoreStatsQ) computes D = K Q^T per panel, so each lane holds 64
//   of its query's scores per panel and keeps a running max and
//   sum(exp(v - max)) in two registers; the lane 32 away holds the other
//   keys of the same query, and the pair is combined once at the end into
//   scratch[row][key range].
//   Pass 2 (scoreStoreQ) computes D = Q K^T per panel and writes
//   softmax of the panel at once, 512 bytes of each of two rows to a store
//   (storeRangeQ), while the other workgroup on the CU computes.
// At D 128 both passes work in base 2 with log2(e) folded into 1/div and the
// bias, so a score costs one fused multiply-add and one v_exp_f32; at D 64 in
// base e, with f64 sums (StatsQ<64>). 16 x 2048 x 128: pass
// 1 takes 29-34 us by the clock, bound by its v_exp_f32 (13 us) and MFMAs (7
// us), which the two waves of a SIMD overlap in part (panels of 64 keys and four
// workgroups a CU: no faster); pass 2 takes 47-50 us, bound by its 256 MiB of
// stores. The pair: 77-87 us from box to box.
constexpr int kPanelQ = 128;                   // keys per streamed panel
constexpr int kMaxRangesQ = 8;                 // key ranges per 128-row block
constexpr float kLog2e = 1.44269504088896340736f;
template <int D>
constexpr int kRowQ = D + 8;                   // halves per LDS panel row
template <int D>
constexpr int kPanelHalvesQ = kPanelQ * kRowQ<D>;
template <int D>
constexpr size_t kLdsStoreQ = 2 * kPanelHalvesQ<D> * sizeof(_Float16);  // pass 1 adds its keys' bias
constexpr int64_t kMaxSeqQ = 8192;             // pass 1's LDS stays <= 100 KiB

/// The max to subtract before exp2: a max of -inf (every score so far -inf)
/// is replaced by 0, so those scores contribute exp2(-inf) = 0 rather than
/// exp2(-inf - -inf) = NaN; the stored max stays -inf.
__device__ __forceinline__ float finiteOr0(float m) { return m == -INFINITY ? 0.0f : m; }

/// The bias in the base of the scores. In base 2 a finite one stays finite, so
/// that keys masked with the lowest float still share a row that has no others.
template <int D>
__device__ __forceinline__ float biasQ(float b) {
    if (D == 64) return b;
    const float t = b * kLog2e;
    return __builtin_isinf(t) && !__builtin_isinf(b) ? __builtin_copysignf(3.402823466e+38f, t) : t;
}

/// A row's max and the sum of its weights over one key range.
template <int D>
struct StatsQ {
    float m, l;
};

/// Head dim 64 keeps the arithmetic of the scores and a softmax over S, its
/// other form: scores in base e, weights exp2((v - max) * log2(e)), their sum in
/// f64 by groups of four. In base 2 with f32 sums, as at 128, a row's sum was
/// off by 5.7e-8 (rms, 8 x 1024; the other form 2.6e-8, so 2.8e-8), and with a
/// bias of 10 the result by 1.7e-7 (16 x 512; 6.6e-8 and 6.6e-8); 8 x 1024 took
/// 14.1 us and takes 14.5, 16 x 2048 68 and 72. A weight as one fused v * log2(e)
/// - k, k whole, saves that, but not 1 at the max: rows of one key are then off
/// by 2e-8.
template <>
struct StatsQ<64> {
    double l;
    float m;
};

/// What a sum of weights against the max `from` is to be multiplied by to be
/// one against the max `to` (finite, or the sum is NaN), no less.
__device__ __forceinline__ double rebase(float from, float to) {
    const double y = (static_cast<double>(from) - static_cast<double>(to)) * 1.4426950408889634074;
    return exp2Poly(y < -1000.0 ? -1000.0 : y, kExp2C10);
}

/// exp2 of a score less a max, in the base of the head dim's scores.
template <int D>
__device__ __forceinline__ float weightQ(float v, float max) {
    return __builtin_amdgcn_exp2f(D == 64 ? (v - max) * kLog2e : v - max);
}

/// 256 threads: global -> registers for the 128-key panel of K (its batch's
/// first row) at row `at`, D / 16 16-byte pieces each, contiguous in K. RAGGED:
/// rows from `rows` on repeat the last one.
template <int D, bool RAGGED>
__device__ __forceinline__ void loadPanelQ(const _Float16* __restrict__ k, int at, int rows, int tid,
                                           u32x4v (&v)[D / 16]) {
    const _Float16* kb = k + static_cast<int64_t>(at) * D;
#pragma unroll
    for (int j = 0; j < D / 16; ++j) {
        const int c = j * 256 + tid;
        const int piece = RAGGED ? min(c / (D / 8), rows - 1 - at) * (D / 8) + c % (D / 8) : c;
        v[j] = *reinterpret_cast<const u32x4v*>(kb + piece * 8);
    }
}

/// Registers -> LDS: key i of the panel to row i, or (QUADS) to row
/// i % 4 * 32 + i / 4.
template <int D, bool QUADS = false>
__device__ __forceinline__ void storePanelQ(_Float16* dst, int tid, const u32x4v (&v)[D / 16]) {
#pragma unroll
    for (int j = 0; j < D / 16; ++j) {
        const int c = j * 256 + tid, key = c / (D / 8);
        const int row = QUADS ? (key & 3) * 32 + (key >> 2) : key;
        *reinterpret_cast<u32x4v*>(dst + row * kRowQ<D> + c % (D / 8) * 8) = v[j];
    }
}

/// Workgroup coordinates: batch, 128-row block, key range of nr, and the
/// range's first key and length: `per` keys, the last range what is left. A
/// batch's workgroups are contiguous within one XCD's share of the grid, a row
/// block's side by side (ranges as the slow dimension: 16 x 2048 x 64 73.5 against
/// 70.2 us, 8 x 1024 x 64 16.0 against 14.5; 16 x 2048 x 128 79.4 against 76.8 on
/// one box, 83 against 85 on another). Grids of no multiple of 8 in grid order: 9 x 640 x 128 13.0
/// against 12.1 us, 13 x 1280 x 64 29.6 against 28.3.
__device__ __forceinline__ void blockOfQ(int seq, int nr, int per, int64_t& b, int& rb, int& kr, int& k0, int& keys) {
    const int panels = seq / kPanelQ;
    int id = xcdShare(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
    kr = id % nr;
    id /= nr;
    b = id / panels;
    rb = id % panels;
    k0 = kr * per;
    keys = min(per, seq - k0);
}

/// Pass-1 statistics of this wave's 32 queries of row block (b, rb) over
/// keys [k0, k0 + keys): D = K Q^T per 128-key panel, so each lane keeps a
/// running max and sum(exp2(v - max)) of its query; the lane 32 away holds
/// the other keys of the same query and the pair is combined at the end.
/// Returns those of query row `qrow` (both half-waves agree).
template <int D, bool RAGGED>
__device__ __forceinline__ StatsQ<D> statsRangeQ(const _Float16* __restrict__ Q, const _Float16* __restrict__ K,
                                              const float* __restrict__ bias, int seq, int sseq, float c2, int64_t b,
                                              int rb, int k0, int keys, _Float16* ldsQ, int64_t& qrow) {
    float* lbias = reinterpret_cast<float*>(ldsQ + 2 * kPanelHalvesQ<D>);  // this key range's bias
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hl = lane >> 5;
    const int np = keys / kPanelQ;
    qrow = b * seq + static_cast<int64_t>(rb) * 128 + wave * 32 + l32;
    constexpr int KS = D / 16;
    const _Float16* qr = Q + (RAGGED ? b * sseq + min(rb * 128 + wave * 32 + l32, sseq - 1) : qrow) * D;
    f16x8 xq[KS];                                 // B operand: this lane's query, KS x 16 head dims
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) xq[ks] = *reinterpret_cast<const f16x8*>(qr + ks * 16 + hl * 8);
    for (int i = tid; i < keys; i += 256) lbias[i] = RAGGED && k0 + i >= sseq ? -INFINITY : biasQ<D>(bias[k0 + i]);
    const _Float16* kb = K + b * (RAGGED ? sseq : seq) * D;
    u32x4v v[D / 16];
    loadPanelQ<D, RAGGED>(kb, k0, sseq, tid, v);
    storePanelQ<D>(ldsQ, tid, v);
    __syncthreads();
    float m = -INFINITY;
    decltype(StatsQ<D>::l) l = 0;
    for (int p = 0; p < np; ++p) {
        if (p + 1 < np) loadPanelQ<D, RAGGED>(kb, k0 + (p + 1) * kPanelQ, sseq, tid, v);
        const _Float16* pk = ldsQ + (p & 1) * kPanelHalvesQ<D>;
        f32x16 acc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f16x8 a = *reinterpret_cast<const f16x8*>(pk + (i * 32 + l32) * kRowQ<D> + ks * 16 + hl * 8);
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, xq[ks], acc[i], 0, 0, 0);
            }
        }
        // acc[i][r]: key p*128 + i*32 + 8*(r/4) + 4*hl + r%4 of this lane's query.
        float mb = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 bb = *reinterpret_cast<const f32x4*>(lbias + p * kPanelQ + i * 32 + 8 * g + 4 * hl);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float x = __builtin_fmaf(acc[i][4 * g + q], c2, bb[q]);
                    acc[i][4 * g + q] = x;
                    mb = fmaxf(mb, x);
                }
            }
        }
        // The lane 32 away agrees on the max, so that f64 sums just add up.
        if constexpr (D == 64) mb = fmaxf(mb, __shfl_xor(mb, 32, 64));
        // A panel whose scores are all -inf adds nothing: its exponentials
        // are taken against a finite stand-in for the -inf max.
        const float mn = fmaxf(m, mb);
        const float ms = finiteOr0(mn);
        if constexpr (D == 64) {
            double sp = 0.0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int r = 0; r < 16; r += 4) {
                    float e[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) e[q] = weightQ<D>(acc[i][r + q], ms);
                    sp += static_cast<double>((e[0] + e[1]) + (e[2] + e[3]));
                }
            }
            l = p > 0 ? l * rebase(m, ms) + sp : sp;
        } else {
            // Eight short sums: a quarter of one long one's rounding.
            float sb[8];
#pragma unroll
            for (int g = 0; g < 8; ++g) {
                sb[g] = weightQ<D>(acc[g / 2][g % 2 * 8], ms);
#pragma unroll
                for (int r = 1; r < 8; ++r) sb[g] += weightQ<D>(acc[g / 2][g % 2 * 8 + r], ms);
            }
            l = l * __builtin_amdgcn_exp2f(m - ms) +
                (((sb[0] + sb[1]) + (sb[2] + sb[3])) + ((sb[4] + sb[5]) + (sb[6] + sb[7])));
        }
        m = mn;
        if (p + 1 < np) storePanelQ<D>(ldsQ + ((p + 1) & 1) * kPanelHalvesQ<D>, tid, v);
        __syncthreads();
    }
    if constexpr (D == 64) {
        StatsQ<D> st;
        st.m = m;
        st.l = l + __shfl_xor(l, 32, 64);
        return st;
    } else {
        const float mo = __shfl_xor(m, 32, 64);
        const float lo = __shfl_xor(l, 32, 64);
        const float mx = fmaxf(m, mo);
        const float ms = finiteOr0(mx);
        return {mx, l * __builtin_amdgcn_exp2f(m - ms) + lo * __builtin_amdgcn_exp2f(mo - ms)};
    }
}

/// Key ranges of a row that a lane merges.
template <int D>
constexpr int kRangesOfLaneQ = D == 64 ? kMaxRangesQ / 2 : kMaxRangesQ;

/// Row statistics of the 16 rows this lane's pass-2 accumulators hold: lane
/// l32 merges row r0 + l32's nr partials pp (those past nr repeat the first)
/// into shift and scale, which the lanes then pass around; at head dim 64 the
/// lane 32 away has half of them. Pass 2 writes exp(v - shift) * scale, scale 1
/// / sum(exp(v - shift)), in the base of the scores. The shift is the row's
/// max, or, at 128, 0 for a row whose max is in [0, 64]: that subtraction has
/// no rounding and is left out, and what then underflows, v < -126, is below
/// float's normal range after the scale too.
/// A log-normalizer max + log2(sum) in one float as the shift would save the
/// multiply, and cost 2^-24 of its magnitude in every value of the row.
/// A row whose scores are all -inf keeps max -inf: exp2(-inf - -inf) writes
/// NaN, as the reference does. Returns whether every row's shift is 0.
template <int D>
__device__ __forceinline__ bool mergeStatsQ(const StatsQ<D> (&pp)[kRangesOfLaneQ<D>], int nr, float (&shift)[16],
                                            float (&scale)[16]) {
    const int hl = (threadIdx.x & 63) >> 5;
    float m = pp[0].m;
#pragma unroll
    for (int i = 1; i < kRangesOfLaneQ<D>; ++i) m = fmaxf(m, pp[i].m);
    float sh, sc;
    bool plain = false;
    if constexpr (D == 64) {
        sh = fmaxf(m, __shfl_xor(m, 32, 64));
        const float ms = finiteOr0(sh);
        double lt = 0.0;
#pragma unroll
        for (int i = 0; i < kRangesOfLaneQ<D>; ++i) {
            const double part = pp[i].l * rebase(pp[i].m, ms);
            lt += hl * kRangesOfLaneQ<D> + i < nr ? part : 0.0;
        }
        sc = static_cast<float>(1.0 / (lt + __shfl_xor(lt, 32, 64)));
    } else {
        plain = m >= 0.0f && m <= 64.0f;
        sh = plain ? 0.0f : m;
        const float ms = finiteOr0(sh);
        float lt = 0.0f;
#pragma unroll
        for (int i = 0; i < kMaxRangesQ; ++i) lt += i < nr ? pp[i].l * __builtin_amdgcn_exp2f(pp[i].m - ms) : 0.0f;
        sc = 1.0f / lt;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        shift[r] = __shfl(sh, 8 * (r >> 2) + 4 * hl + (r & 3), 64);
        scale[r] = __shfl(sc, 8 * (r >> 2) + 4 * hl + (r & 3), 64);
    }
    return D != 64 && __all(plain);
}

/// Pass 2 over keys [k0, k0 + keys) of this wave's 32 rows r0..r0+31 of
/// batch b: D = Q K^T per panel, written as exp2(v - shift) * scale at once.
/// RAGGED: seq is the sequence length sseq of the operands rounded up to whole
/// panels; what is past its end repeats its last row and is not stored. QUADS (S 16-byte aligned, sseq a multiple of 4): MFMA column l
/// of block j is key 4 l + j, so that a lane's four blocks hold four keys in a
/// row and one store writes 512 bytes of each of two rows (8 x 1024 x 64: 15.1
/// -> 13.9 us against 128 bytes); otherwise it is key 32 j + l and a store
/// writes 128.
/// Batches start at different panels: row blocks in step would write the same
/// few columns of rows a power of two apart, which share memory channels (16 x
/// 2048 x 128, both passes: 89.1 -> 76.8 us on one box, 90.7 -> 85.4 on another;
/// x 64: 84 -> 70 on both). Within a batch they stay in step, for K in the L2
/// (each row block apart: 84 us where this takes 77).
template <int D, bool RAGGED, bool QUADS>
__device__ __forceinline__ void storeRangeQ(const _Float16* __restrict__ Q, const _Float16* __restrict__ K,
                                            const float* __restrict__ bias, float* __restrict__ S, int seq,
                                            int sseq, float c2, int64_t b, int rb, int64_t r0, int k0, int keys,
                                            const StatsQ<D>* __restrict__ part, int nr, _Float16* ldsQ) {
    const int ld = RAGGED ? sseq : seq;           // S row length
    const int i0 = static_cast<int>(r0 - b * seq);   // first row within the batch
    const int tid = threadIdx.x;
    const int lane = tid & 63, l32 = lane & 31, hl = lane >> 5;
    const int np = keys / kPanelQ;
    constexpr int KS = D / 16;
    const _Float16* qr = Q + (RAGGED ? b * ld + min(i0 + l32, ld - 1) : r0 + l32) * D;
    f16x8 aq[KS];                                 // A operand: row r0 + l32
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        aq[ks] = *reinterpret_cast<const f16x8*>(qr + ks * 16 + hl * 8);
    }
    const _Float16* kb = K + b * ld * D;
    // Stores: a scalar base per panel (row r0, key kc) plus a fixed lane
    // offset per accumulator register r.
    const int lk = QUADS ? 4 * l32 : l32;         // this lane's key of block 0
    constexpr int jk = QUADS ? 1 : 32;            // from block to block
    uint32_t soff[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        soff[r] = static_cast<uint32_t>(((8 * (r >> 2) + 4 * hl + (r & 3)) * ld + lk) * sizeof(float));
    }
    StatsQ<D> pp[kRangesOfLaneQ<D>];
#pragma unroll
    for (int i = 0; i < kRangesOfLaneQ<D>; ++i) {
        const int range = (D == 64 ? hl * kRangesOfLaneQ<D> : 0) + i;
        pp[i] = part[(r0 + l32) * nr + (range < nr ? range : 0)];
    }
    u32x4v v[D / 16];
    int at = static_cast<int>(b) % np;
    loadPanelQ<D, RAGGED>(kb, k0 + at * kPanelQ, ld, tid, v);
    float shift[16], scale[16];
    const bool plain = mergeStatsQ<D>(pp, nr, shift, scale);
    storePanelQ<D, QUADS>(ldsQ, tid, v);
    __syncthreads();
    for (int p = 0; p < np; ++p) {
        const int kc = k0 + at * kPanelQ;
        if (++at == np) at = 0;
        if (p + 1 < np) loadPanelQ<D, RAGGED>(kb, k0 + at * kPanelQ, ld, tid, v);
        const _Float16* pk = ldsQ + (p & 1) * kPanelHalvesQ<D>;
        f32x16 acc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f16x8 x = *reinterpret_cast<const f16x8*>(pk + (j * 32 + l32) * kRowQ<D> + ks * 16 + hl * 8);
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(aq[ks], x, acc[j], 0, 0, 0);
            }
        }
        float bj[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) bj[j] = biasQ<D>(bias[RAGGED ? min(kc + lk + j * jk, ld - 1) : kc + lk + j * jk]);
        char* sb = reinterpret_cast<char*>(S + (b * ld + i0) * static_cast<int64_t>(ld) + kc);
        auto store = [&](auto value) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (RAGGED && i0 + 8 * (r >> 2) + 4 * hl + (r & 3) >= sseq) continue;
                f32x4 out;
#pragma unroll
                for (int j = 0; j < 4; ++j) out[j] = value(__builtin_fmaf(acc[j][r], c2, bj[j]), r);
                if (QUADS) {
                    if (!RAGGED || kc + lk < sseq) *reinterpret_cast<f32x4*>(sb + soff[r]) = out;
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if (kc + lk + j * jk < sseq) *reinterpret_cast<float*>(sb + soff[r] + j * jk * sizeof(float)) = out[j];
                    }
                }
            }
        };
        if (plain) {
            store([&](float v, int r) { return __builtin_amdgcn_exp2f(v) * scale[r]; });
        } else {
            store([&](float v, int r) { return weightQ<D>(v, shift[r]) * scale[r]; });
        }
        if (p + 1 < np) storePanelQ<D, QUADS>(ldsQ + ((p + 1) & 1) * kPanelHalvesQ<D>, tid, v);
        __syncthreads();
    }
}

template <int D, bool RAGGED>
__global__ __launch_bounds__(256, 2) void scoreStatsQ(const _Float16* __restrict__ Q,
                                                      const _Float16* __restrict__ K,
                                                      const float* __restrict__ bias,
                                                      StatsQ<D>* __restrict__ part, int seq, int sseq, int nr, int per,
                                                      float c2) {
    extern __shared__ __align__(16) _Float16 ldsQ[];
    int64_t b;
    int rb, kr, k0, keys;
    blockOfQ(seq, nr, per, b, rb, kr, k0, keys);
    int64_t qrow;
    const StatsQ<D> st = statsRangeQ<D, RAGGED>(Q, K, bias, seq, sseq, c2, b, rb, k0, keys, ldsQ, qrow);
    if (((threadIdx.x & 63) >> 5) == 0) part[qrow * nr + kr] = st;
}

template <int D, bool RAGGED, bool QUADS>
__global__ __launch_bounds__(256, 2) void scoreStoreQ(const _Float16* __restrict__ Q,
                                                      const _Float16* __restrict__ K,
                                                      const float* __restrict__ bias,
                                                      const StatsQ<D>* __restrict__ part, float* __restrict__ S,
                                                      int seq, int sseq, int nr, int per,
                                                      float c2) {
    extern __shared__ __align__(16) _Float16 ldsQ[];
    int64_t b;
    int rb, kr, k0, keys;
    blockOfQ(seq, nr, per, b, rb, kr, k0, keys);
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int64_t r0 = b * seq + static_cast<int64_t>(rb) * 128 + wave * 32;   // wave-uniform
    storeRangeQ<D, RAGGED, QUADS>(Q, K, bias, S, seq, sseq, c2, b, rb, r0, k0, keys, part, nr, ldsQ);
}

/// Panels of each key range but the last: those that take the fewest panel
/// times, a workgroup's start (Q, its first panel, the statistics) counted as
/// two, over the 512 workgroups the chip holds at once (two ranges against up
/// to eight: 1 x 2048 x 128 36.7 -> 15.4 us, 1 x 1024 x 128 20.8 -> 9.7, 8 x
/// 1024 x 64 19.6 -> 14.4, 4 x 512 x 64 11.0 -> 7.8). `most` is the number of
/// ranges there is room for. Shapes with a choice of launch forms keep to form
/// 0's two ranges below 8 panels.
int panelsPerRange(const mlkd_score_softmax* p, int most) {
    const int64_t panels = p->seq / kPanelQ, rows = p->batch * panels;
    if (p->dim == 128 && p->seq % 256 == 0 && panels < 8) return static_cast<int>(panels / 2);
    int64_t best = 0, per = panels;
    for (int64_t nr = 1; nr <= std::min<int64_t>(most, panels); ++nr) {
        const int64_t each = (panels + nr - 1) / nr;
        const int64_t slots = each <= 24 ? 512 : 256;   // past 24 panels a bias in LDS leaves room for one a CU
        const int64_t t = (rows * ((panels + each - 1) / each) + slots - 1) / slots * (each + 2);
        if (nr > 1 && t >= best) continue;
        best = t;
        per = each;
    }
    return static_cast<int>(per);
}

int rangesQ(const mlkd_score_softmax* p, int most = kMaxRangesQ) {
    const int64_t per = panelsPerRange(p, most);
    return static_cast<int>((p->seq / kPanelQ + per - 1) / per);
}

/// Both passes, at most `most` key ranges per row block with their partials in
/// p->scratch; `ragged` > 0 is the operands' sequence length, p->seq that
/// rounded up to whole panels. Copies of Q, K and the bias, padded by three
/// kernels more, took 16 x 1000 x 128 to 33 us (24 without), 4 x 1000 to 19
/// (12.7), 1 x 300 to 21 (9.9).
template <int D>
int launchQ(const mlkd_score_softmax* p, int most, hipStream_t st, int64_t ragged = 0) {
    auto stats = scoreStatsQ<D, false>;
    auto storeAny = scoreStoreQ<D, true, false>, store = scoreStoreQ<D, false, true>;
    // Once per process; a function-local static initializes thread-safely.
    auto allow = [](auto fn) {
        const int bytes = static_cast<int>(kLdsStoreQ<D> + static_cast<size_t>(kMaxSeqQ) * sizeof(float));
        return hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   bytes) == hipSuccess;
    };
    static const bool attrs = allow(stats) && allow(store) && allow(storeAny);
    if (!attrs) return MLKD_RT_LAUNCH;
    if constexpr (D == 128) {   // dim 64 is not run off the panels
        static const bool raggedAttrs = allow(scoreStatsQ<D, true>) && allow(scoreStoreQ<D, true, true>);
        if (!raggedAttrs) return MLKD_RT_LAUNCH;
        if (ragged > 0) {
            stats = scoreStatsQ<D, true>;
            store = scoreStoreQ<D, true, true>;
        }
    }
    const int64_t sseq = ragged > 0 ? ragged : p->seq;
    if (sseq % 4 != 0 || (reinterpret_cast<uintptr_t>(p->s) & 15u) != 0) store = storeAny;
    const int per = panelsPerRange(p, most) * kPanelQ;
    const size_t ldsStats = kLdsStoreQ<D> + static_cast<size_t>(per) * sizeof(float);
    const int nr = rangesQ(p, most);
    const dim3 grid(static_cast<unsigned>(p->batch * (p->seq / kPanelQ) * nr));
    // At head dim 128 both passes work in base 2: v2 = acc * (log2(e) / div) +
    // bias * log2(e), exp(v - max) = exp2(v2 - max2).
    const float c2 = static_cast<float>((D == 64 ? 1.0 : 1.4426950408889634) / p->div);
    hipLaunchKernelGGL(stats, grid, dim3(256), ldsStats, st, static_cast<const _Float16*>(p->q),
                       static_cast<const _Float16*>(p->k), static_cast<const float*>(p->bias),
                       static_cast<StatsQ<D>*>(p->scratch), static_cast<int>(p->seq),
                       static_cast<int>(sseq), nr, per, c2);
    hipLaunchKernelGGL(store, grid, dim3(256), kLdsStoreQ<D>, st,
                       static_cast<const _Float16*>(p->q), static_cast<const _Float16*>(p->k),
                       static_cast<const float*>(p->bias), static_cast<const StatsQ<D>*>(p->scratch),
                       static_cast<float*>(p->s), static_cast<int>(p->seq),
                       static_cast<int>(sseq), nr, per, c2);
    return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
}

/// `div` is held to where 1 / div times log2(e) is a normal float, the grid to
/// the fewer than 2^32 threads that HIP takes (2^24 batches of a few keys are
/// 4 GiB of Q).
/// Head dim 64 takes it from 512 keys, and more rows than that: with fewer it
/// gains nothing (3 x 256: 7.9 against 7.4 us, 1 x 512: 8.0 and 7.7, 2 x 512:
/// 8.1 and 8.3). Its error is the other form's (2 x 512: 1.39e-7 and 1.39e-7,
/// 8 x 1024: 1.44e-7 and 1.45e-7, 1 x 8192: 1.67e-7 and 1.66e-7).
bool twoPassApplies(const mlkd_score_softmax* p) {
    const double size = p->div < 0 ? -p->div : p->div;
    if (!(size >= 1e-30 && size <= 1e30)) return false;
    return p->qk_dtype == MLKD_F16 && p->bias_dtype == MLKD_F32 && p->s_dtype == MLKD_F32 &&
           (p->dim == 64 || p->dim == 128) && p->seq % kPanelQ == 0 && p->seq > 0 && p->seq <= kMaxSeqQ &&
           (p->dim == 128 || (p->seq >= 512 && p->batch * p->seq > 512)) &&
           (reinterpret_cast<uintptr_t>(p->q) & 15u) == 0 && (reinterpret_cast<uintptr_t>(p->k) & 15u) == 0 &&
           p->batch <= (int64_t{1} << 32) / 256 && p->batch * (p->seq / kPanelQ) * rangesQ(p) < (int64_t{1} << 32) / 256;
}

/// Row statistics partials of nr key ranges: one (max, sum) pair per row and
/// range.
int64_t statsBytes(const mlkd_score_softmax* p, int nr) {
    return p->batch * p->seq * nr * static_cast<int64_t>(p->dim == 64 ? sizeof(StatsQ<64>) : sizeof(StatsQ<128>));
}

template <typename T>
__device__ __forceinline__ double ldAny(const void* p, int dt, int64_t i) {
    if (dt == MLKD_F32) return static_cast<const float*>(p)[i];
    if (dt == MLKD_F16) return static_cast<float>(static_cast<const _Float16*>(p)[i]);
    return static_cast<const double*>(p)[i];
}

__global__ __launch_bounds__(256) void scoresGeneral(mlkd_score_softmax p) {
    const int64_t total = p.batch * p.seq * p.seq;
    for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < total;
         t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t j = t % p.seq;
        const int64_t bi = t / p.seq;  // b*seq + i
        const int64_t b = bi / p.seq;
        double acc = 0.0;
        for (int64_t k = 0; k < p.dim; ++k) {
            acc += ldAny<double>(p.q, p.qk_dtype, bi * p.dim + k) *
                   ldAny<double>(p.k, p.qk_dtype, (b * p.seq + j) * p.dim + k);
        }
        const double v = acc / p.div + ldAny<double>(p.bias, p.bias_dtype, j);
        if (p.s_dtype == MLKD_F32) {
            static_cast<float*>(p.s)[t] = static_cast<float>(v);
        } else if (p.s_dtype == MLKD_F64) {
            static_cast<double*>(p.s)[t] = v;
        } else {
            static_cast<_Float16*>(p.s)[t] = mlk::toHalf(v);
        }
    }
}

/// Workspace bytes of the two passes, for their partials: 0 where they don't
/// run. `q`, if given, is p over whole panels, set up to run in the workspace
/// p->work.
int64_t workBytes(const mlkd_score_softmax* p, mlkd_score_softmax* q = nullptr) {
    mlkd_score_softmax w = *p;
    w.seq = (p->seq + kPanelQ - 1) / kPanelQ * kPanelQ;
    // Off the panels the general kernels, which add in f64, run dim 64.
    if (!twoPassApplies(&w) || (w.seq != p->seq && p->dim != 128)) return 0;
    w.scratch = p->work;
    w.scratch_bytes = statsBytes(&w, rangesQ(&w));
    if (q != nullptr) *q = w;
    return w.scratch_bytes;
}

/// Scratch a run of the two passes is always given: dim 128, whole pairs of
/// panels, for two key ranges. Elsewhere, and for more ranges, they take a
/// workspace where there is one.
int64_t requiredBytes(const mlkd_score_softmax* p) {
    return p->dim == 128 && p->seq % (2 * kPanelQ) == 0 && twoPassApplies(p) ? statsBytes(p, 2) : 0;
}

/// Whether p runs in two passes, with q and the most key ranges set up.
bool runsTwoPass(const mlkd_score_softmax* p, int variant, mlkd_score_softmax& q, int& most) {
    if (variant == 1) return false;
    const int64_t work = workBytes(p, &q);
    if (work > 0 && p->work != nullptr && (reinterpret_cast<uintptr_t>(p->work) & 15u) == 0 && p->work_bytes >= work) {
        most = kMaxRangesQ;
        return true;
    }
    const int64_t need = requiredBytes(p);
    if (need > 0 && p->scratch != nullptr && (reinterpret_cast<uintptr_t>(p->scratch) & 7u) == 0 &&
        p->scratch_bytes >= need) {
        q = *p;
        most = 2;
        return true;
    }
    return false;
}

int launchTwoPass(const mlkd_score_softmax* p, const mlkd_score_softmax& q, int most, hipStream_t st) {
    const int64_t ragged = q.seq == p->seq ? 0 : p->seq;
    return p->dim == 64 ? launchQ<64>(&q, most, st) : launchQ<128>(&q, most, st, ragged);
}

// 0: the best form for the shape (the two-pass query-stationary form where
// it applies); 1: scores, then the softmax kernel in place over S.
int gScoreVariant = 0;

}  // namespace

extern "C" void mlkd_score_set_variant(int variant) { gScoreVariant = variant; }

extern "C" int mlkd_score_ranges(const mlkd_score_softmax* p) {
    mlkd_score_softmax q;
    return workBytes(p, &q) > 0 ? rangesQ(&q) : 0;
}

extern "C" int64_t mlkd_score_scratch_bytes(const mlkd_score_softmax* p) { return p != nullptr ? requiredBytes(p) : 0; }

extern "C" int64_t mlkd_score_pad_bytes(const mlkd_score_softmax* p) {
    const int64_t work = p != nullptr ? workBytes(p) : 0;
    return work > (p != nullptr ? requiredBytes(p) : 0) ? work : 0;
}

extern "C" const char* mlkd_score_kernel_names(const mlkd_score_softmax* p) {
    static thread_local char name[160];
    mlkd_score_softmax q;
    int most;
    if (runsTwoPass(p, p->variant >= 0 ? p->variant : gScoreVariant, q, most)) return "scoreStatsQ+scoreStoreQ";
    const bool fast = p->qk_dtype == MLKD_F16 && p->bias_dtype == MLKD_F32 && p->s_dtype == MLKD_F32 &&
                      p->seq % 128 == 0 && p->dim % 16 == 0 && p->dim > 0 && p->seq < (1 << 20) &&
                      (reinterpret_cast<uintptr_t>(p->q) & 15u) == 0 &&
                      (reinterpret_cast<uintptr_t>(p->k) & 15u) == 0 && p->dim % 8 == 0;
    mlkd_softmax sm;
    sm.variant = -1;
    sm.pad = 0;
    sm.x = p->s;
    sm.y = p->s;
    sm.x_dtype = p->s_dtype;
    sm.y_dtype = p->s_dtype;
    sm.rows = p->batch * p->seq;
    sm.cols = p->seq;
    sm.x_row_stride = p->seq;
    sm.y_row_stride = p->seq;
    std::snprintf(name, sizeof(name), "%s+%s", fast ? "scoresF16" : "scoresGeneral", mlkd_softmax_kernel_name(&sm));
    return name;
}

extern "C" int mlkd_launch_score_softmax(const mlkd_score_softmax* p, void* stream) {
    if (p == nullptr || p->batch < 0 || p->seq < 0 || p->dim < 0) return MLKD_RT_LAUNCH;
    if (p->batch == 0 || p->seq == 0) return 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int variant = p->variant >= 0 ? p->variant : gScoreVariant;
    mlkd_score_softmax q;
    int most;
    if (runsTwoPass(p, variant, q, most)) return launchTwoPass(p, q, most, st);
    const bool fast = p->qk_dtype == MLKD_F16 && p->bias_dtype == MLKD_F32 && p->s_dtype == MLKD_F32 &&
                      p->seq % 128 == 0 && p->dim % 16 == 0 && p->dim > 0 && p->seq < (1 << 20) &&
                      (reinterpret_cast<uintptr_t>(p->q) & 15u) == 0 &&
                      (reinterpret_cast<uintptr_t>(p->k) & 15u) == 0 && p->dim % 8 == 0;
    if (fast) {
        const int64_t blocks = p->batch * (p->seq / 64) * (p->seq / 128);
        if (blocks > 0x7FFFFFFF) return MLKD_RT_LAUNCH;
        hipLaunchKernelGGL(scoresF16, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                           static_cast<const _Float16*>(p->q), static_cast<const _Float16*>(p->k),
                           static_cast<const float*>(p->bias), static_cast<float*>(p->s),
                           static_cast<int>(p->seq), static_cast<int>(p->dim), static_cast<float>(p->div));
    } else {
        hipLaunchKernelGGL(scoresGeneral, dim3(8192), dim3(256), 0, st, *p);
    }
    if (hipGetLastError() != hipSuccess) return MLKD_RT_LAUNCH;
    mlkd_softmax sm;
    sm.variant = -1;
    sm.pad = 0;
    sm.x = p->s;
    sm.y = p->s;
    sm.x_dtype = p->s_dtype;
    sm.y_dtype = p->s_dtype;
    sm.rows = p->batch * p->seq;
    sm.cols = p->seq;
    sm.x_row_stride = p->seq;
    sm.y_row_stride = p->seq;
    return mlkd_launch_softmax(&sm, stream);
}
