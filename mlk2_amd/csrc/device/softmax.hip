// Row-wise stable softmax: Call(Softmax) (runtime/src/execution/
// kernel_buffers.cpp:290-340) and the synthesized six-statement nest of
// compiler/src/passes/poly/poly.synth.cpp:363-523, which computes the same
// values through materialized temps. Per row: r = max over x (a NaN never
// replaces the running max, matching (x > r) ? x : r); y = exp(x - r);
// s = sum y; y = s != 0 ? y / s : 0. The temps are never materialized: the
// row lives in registers between its one HBM read and its one HBM write.
//
// Fast path (f32 in/out, cols % 4 == 0, cols <= 256*CH): one wave per row,
// each lane holds CH float4 of the row (16-byte coalesced loads), the max and
// the sum are wave reductions (ds_swizzle/DPP through __shfl_xor), no LDS and
// no barriers. exp runs in f32 on x - r (x - r is exact whenever x is near r,
// which is where the large outputs are); the row sum accumulates in f64, so
// the normalisation error stays ~1 f32 ULP of each output.
// Longer f32 rows and f16 rows (16 to 65536 columns): softmaxRowWide, the row
// in registers, f64 arithmetic.
// General path (any dtype, any cols): one workgroup per row, three passes over
// the row with LDS reductions, f64 throughout.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>

#include <math.h>
#include <stdint.h>

#include "exp2_poly.h"
#include "mlk_device_math.h"
#include "runtime_abi.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float waveMax(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

__device__ __forceinline__ double waveSum(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

/// Waves a row of softmaxWaveRowScalar<CH> is split over.
template <int CH>
constexpr int kScalarWaves = CH > 16 ? 4 : 1;

/// Loads one row into the lane's CH float4 (columns past `cols` read as -inf,
/// which leaves the max unchanged and adds exp(-inf) = 0 to nothing: the sum
/// skips them). FULL: cols == 256 * CH, so every column is in range and the
/// guards compile away.
template <int CH, bool FULL>
__device__ __forceinline__ void loadRow(const float* xr, int64_t cols, int lane, f32x4 (&v)[CH]) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int64_t col = (static_cast<int64_t>(c) * 64 + lane) * 4;
        if (FULL || col < cols) {
            v[c] = *reinterpret_cast<const f32x4*>(xr + col);
        } else {
            v[c] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        }
    }
}

/// The row max, wave-reduced (every lane returns it).
template <int CH>
__device__ __forceinline__ float rowMax(const f32x4 (&v)[CH]) {
    float m = -INFINITY;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
#pragma unroll
        for (int e = 0; e < 4; ++e) m = fmaxf(m, v[c][e]);
    }
    return waveMax(m);
}

/// exp(v - m), the row sum, and the stores of v / sum. FAST: exp as
/// v_exp_f32 of (x - max) * log2(e), and the row sum as f64 over f32 sums of
/// each 4-element group (the error of either stays below 1e-7 relative of the
/// result, against the class's 1e-6). NT: nontemporal stores.
template <int CH, bool FAST, bool NT, bool FULL>
__device__ __forceinline__ void normalizeRow(f32x4 (&v)[CH], float m, float* yr, int64_t cols, int lane) {
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int64_t col = (static_cast<int64_t>(c) * 64 + lane) * 4;
        if constexpr (FAST) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[c][e] = __builtin_amdgcn_exp2f((v[c][e] - m) * 1.44269504088896340736f);
            if (FULL || col < cols) s += static_cast<double>((v[c][0] + v[c][1]) + (v[c][2] + v[c][3]));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float ex = expf(v[c][e] - m);
                v[c][e] = ex;
                if (FULL || col < cols) s += static_cast<double>(ex);
            }
        }
    }
    s = waveSum(s);
    // The reference's `s != 0 ? y / s : 0` never takes its zero arm here: an
    // in-range element equal to the max m contributes exp(0) = 1, and a row
    // with no such element (m = +-inf, or every element NaN) makes some term
    // NaN (inf - inf, NaN - m). So s >= 1 or s is NaN, and y * (1 / s) is
    // the reference's value without a per-element select.
    const float inv = static_cast<float>(1.0 / s);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int64_t col = (static_cast<int64_t>(c) * 64 + lane) * 4;
        if (FULL || col < cols) {
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = v[c][e] * inv;
            if constexpr (NT) {
                __builtin_nontemporal_store(o, reinterpret_cast<f32x4*>(yr + col));
            } else {
                *reinterpret_cast<f32x4*>(yr + col) = o;
            }
        }
    }
}

template <int CH, bool FAST, bool NT, bool FULL>
__device__ __forceinline__ void finishRow(f32x4 (&v)[CH], float* yr, int64_t cols, int lane) {
    normalizeRow<CH, FAST, NT, FULL>(v, rowMax<CH>(v), yr, cols, lane);
}

/// One row per wave. Always the guarded row body: the guard-free one
/// (FULL) holds 150 VGPRs here against 88, and at 3 waves per SIMD instead
/// of 5 it measured 41.3 us against 40.2 us at 8192 x 4096.
template <int CH, bool FAST = false, bool NT = true>
__global__ __launch_bounds__(256) void softmaxWaveRow(const float* x,
                                                      float* y, int64_t rows,
                                                      int64_t cols, int64_t xs, int64_t ys) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int64_t waves = static_cast<int64_t>(gridDim.x) * 4;
    for (int64_t row = wave; row < rows; row += waves) {
        f32x4 v[CH];
        loadRow<CH, false>(x + row * xs, cols, lane, v);
        finishRow<CH, FAST, NT, false>(v, y + row * ys, cols, lane);
    }
}

/// A workgroup barrier that orders LDS alone: __syncthreads would also wait
/// for every global load and store in flight.
__device__ __forceinline__ void ldsBarrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

/// Max (MAX) or sum of one value per wave over the W waves of a row, in every
/// lane. `slot` is the row's LDS array; a row's max and sum use two arrays, so
/// the barrier of one separates the reads of the other from its next writes.
template <int W, bool MAX, typename T>
__device__ __forceinline__ T acrossWaves(T v, T (&slot)[W]) {
    if constexpr (W > 1) {
        if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = v;
        ldsBarrier();
        v = slot[0];
#pragma unroll
        for (int i = 1; i < W; ++i) {
            if constexpr (MAX) v = fmaxf(v, slot[i]);
            else v += slot[i];
        }
    }
    return v;
}

/// Rows the float4 loads cannot take (cols % 4 != 0, or a row start off 16
/// bytes), up to 256 * CH columns: the arithmetic of softmaxWaveRow<CH, true,
/// true> (f32 max, v_exp_f32, f64 sum of f32 sums of 4-element groups), 4-byte
/// loads and stores that are lane-contiguous per instruction. One wave per row
/// up to 4096 columns; past that the row is split over 4 waves, since one wave
/// would hold 128 row registers beside their addresses and spill. v[c][e]
/// holds element (c * W + wave) * 256 + e * 64 + lane; elements past the row
/// read as -inf and add exp2(-inf) = 0 to their group.
template <int CH>
__global__ __launch_bounds__(256) void softmaxWaveRowScalar(const float* __restrict__ x, float* __restrict__ y,
                                                            int64_t rows, int64_t cols, int64_t xs, int64_t ys) {
    constexpr int W = kScalarWaves<CH>, N = CH / W;
    __shared__ float smax[W];
    __shared__ double ssum[W];
    const int lane = threadIdx.x & 63;
    const int w = W > 1 ? threadIdx.x >> 6 : 0;
    const int64_t rowsPer = 4 / W;
    const int64_t first = static_cast<int64_t>(blockIdx.x) * rowsPer + (W > 1 ? 0 : threadIdx.x >> 6);
    for (int64_t row = first; row < rows; row += static_cast<int64_t>(gridDim.x) * rowsPer) {
        const float* xr = x + row * xs;
        float* yr = y + row * ys;
        f32x4 v[N];
#pragma unroll
        for (int c = 0; c < N; ++c) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t col = static_cast<int64_t>(c * W + w) * 256 + e * 64 + lane;
                v[c][e] = col < cols ? xr[col] : -INFINITY;
            }
        }
        const float m = acrossWaves<W, true>(rowMax<N>(v), smax);
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < N; ++c) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[c][e] = __builtin_amdgcn_exp2f((v[c][e] - m) * 1.44269504088896340736f);
            s += static_cast<double>((v[c][0] + v[c][1]) + (v[c][2] + v[c][3]));
        }
        s = acrossWaves<W, false>(waveSum(s), ssum);
        const float inv = static_cast<float>(1.0 / s);
#pragma unroll
        for (int c = 0; c < N; ++c) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t col = static_cast<int64_t>(c * W + w) * 256 + e * 64 + lane;
                if (col < cols) __builtin_nontemporal_store(v[c][e] * inv, yr + col);
            }
        }
    }
}

/// Two adjacent rows per wave: the second row's loads are issued once the
/// first row's max is known, so they land while the first row is
/// exponentiated, summed and stored. The per-row arithmetic is that of form 0
/// (rowMax, then normalizeRow<CH, true, true>), so the two forms agree bit
/// for bit.
template <int CH, bool FULL>
__global__ __launch_bounds__(256) void softmaxWaveRowPair(const float* x, float* y, int64_t rows, int64_t cols,
                                                          int64_t xs, int64_t ys) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int64_t waves = static_cast<int64_t>(gridDim.x) * 4;
    const int64_t pairs = (rows + 1) / 2;
    for (int64_t pr = wave; pr < pairs; pr += waves) {
        // An odd last row pairs with itself: the same wave computes it twice
        // from the same data and stores the same bits twice. A branch around
        // the second row instead makes the compiler's wait counts assume the
        // second row's loads were issued and drain them all before the first
        // row's reductions, which serialises the pair.
        const int64_t r0 = 2 * pr;
        const int64_t r1 = r0 + 1 < rows ? r0 + 1 : r0;
        f32x4 a[CH], b[CH];
        loadRow<CH, FULL>(x + r0 * xs, cols, lane, a);
        const float ma = rowMax<CH>(a);
        // The barriers fix the order (measured at 8192 x 4096: 39.3 us with
        // it, 39.7 us with both rows' loads first, 40.1 us with the rows'
        // bodies merged by the scheduler, which then waits for both rows
        // before either reduction and holds both rows' temporaries).
        __builtin_amdgcn_sched_barrier(0);
        loadRow<CH, FULL>(x + r1 * xs, cols, lane, b);
        __builtin_amdgcn_sched_barrier(0);
        normalizeRow<CH, true, true, FULL>(a, ma, y + r0 * ys, cols, lane);
        __builtin_amdgcn_sched_barrier(0);
        finishRow<CH, true, true, FULL>(b, y + r1 * ys, cols, lane);
    }
}

/// The row body of form 2 (expf, per-element f64 sums), with each wave
/// walking several rows and the next row's loads issued before the current
/// row's reductions, so HBM reads of row r+1 overlap the exp/sum/stores of
/// row r.
template <int CH>
__global__ __launch_bounds__(256) void softmaxWaveRowPipelined(const float* x, float* y, int64_t rows,
                                                               int64_t cols, int64_t xs, int64_t ys) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int64_t waves = static_cast<int64_t>(gridDim.x) * 4;
    f32x4 cur[CH], nxt[CH];
    if (wave < rows) loadRow<CH, false>(x + wave * xs, cols, lane, cur);
    for (int64_t row = wave; row < rows; row += waves) {
        const int64_t nrow = row + waves;
        if (nrow < rows) loadRow<CH, false>(x + nrow * xs, cols, lane, nxt);
        finishRow<CH, false, true, false>(cur, y + row * ys, cols, lane);
#pragma unroll
        for (int c = 0; c < CH; ++c) cur[c] = nxt[c];
    }
}

template <typename T>
struct WideRow;
template <>
struct WideRow<float> {
    static constexpr int V = 4;
    static constexpr float kMostMax = 1e6f;
    using Vec = f32x4;
    static __device__ __forceinline__ float narrow(double v) { return static_cast<float>(v); }
};
template <>
struct WideRow<_Float16> {
    static constexpr int V = 8;
    static constexpr float kMostMax = 60000.0f;
    using Vec = _Float16 __attribute__((ext_vector_type(8)));
    /// One rounding of v >= 0: to the nearest f32, made round-to-odd (one
    /// step down if that was up, the last bit set if inexact), then to f16.
    static __device__ __forceinline__ _Float16 narrow(double v) {
        const float r = static_cast<float>(v);
        const double d = static_cast<double>(r);
        uint32_t bits = __float_as_uint(r) - (d > v ? 1u : 0u);
        bits |= d != v ? 1u : 0u;
        return static_cast<_Float16>(__uint_as_float(bits));
    }
};

/// softmaxRowWide's row for a max that is infinite or so large that floats
/// near it lie far apart (or, in f16, end): the same arithmetic, element by
/// element from memory, with the exponent itself held at -1000 or more. The
/// max is subtracted before the scale: x * log2(e) + round(-m * log2(e)) is off
/// at x == m by the product's rounding, which leaves [-1000, 1000] from |m| of
/// 1e20 on. x and y may be the same row: each element is read before its
/// thread writes it.
template <typename T, int W>
__device__ __forceinline__ void softmaxOddRow(const T* x, T* y, int cols, float m, int thread, double (&slot)[W]) {
    using R = WideRow<T>;
    auto term = [&](T xv) {
        const double e = (static_cast<double>(static_cast<float>(xv)) - static_cast<double>(m)) * 1.4426950408889634074;
        return exp2Poly(e < -1000.0 ? -1000.0 : e, kExp2C10);
    };
    double s = 0.0;
#pragma unroll 1
    for (int i = thread; i < cols; i += 64 * W) s += term(x[i]);
    s = acrossWaves<W, false>(waveSum(s), slot);
    const double inv = 1.0 / s;
#pragma unroll 1
    for (int i = thread; i < cols; i += 64 * W) y[i] = R::narrow(term(x[i]) * inv);
}

/// Rows past the float4 path's 8192 columns and rows of f16, in f64
/// arithmetic with one rounding to T (the general kernel's precision): W waves
/// per row, CH 16-byte pieces of it in each lane's registers in T, so the row
/// is read once and written once. Pieces start at the row's first 16-byte
/// boundary; the up to V - 1 elements before it and after the last whole
/// piece go one to a lane of the first wave. 2^y takes 15 f64 instructions
/// (which issue at the f32 rate here), so it is computed twice, for the sum
/// and for the output, rather than held in two registers per element. With
/// polynomials of 7 terms for the sum and 8 for the output (2.5e-9 and 5.5e-11
/// off) results were not the exact ones rounded once, 6% of them in rows of two
/// values; those of 10 (1.9e-14) take 1000 x 30001 f32 from 54.5 to 56.1 us,
/// 4.3 TB/s (softmaxBlockRow, which reads the row three times and calls exp
/// twice: 219 us; a copy of the same bytes: 45 us). 8192 x 4096 f16 takes 54 us
/// (160 us). Pieces past the row are skipped, each by a uniform branch: 4000 x
/// 8196 f32 59.5 us (computed for nothing 71.7), 800 x 40000 84.8-88.6 (94), f16
/// 2000 x 20000 73 (79), but 512 x 65536, which has none, 72-75 (70); by twos or
/// fours no faster. The f64 work, about 30 us of each, and the
/// memory traffic overlap only between the two to four rows a CU holds.
/// Summing against a reference of the row's first pieces, so that a piece's
/// terms are computed under the loads of the next, took 72 us; walking rows
/// with the next one's loads in flight 60 us (both need more registers).
template <typename T, int CH, int W>
__global__ __launch_bounds__(W == 1 ? 256 : 64 * W, CH >= 8 ? 4 : 8) void softmaxRowWide(const T* x, T* y, int64_t rows, int cols,
                                                                           int64_t stride) {
    using R = WideRow<T>;
    using Vec = typename R::Vec;
    constexpr int V = R::V;
    constexpr int NOut = sizeof(kExp2C10) / sizeof(double);
    __shared__ float smax[W];
    __shared__ double ssum[W];
    const int lane = threadIdx.x & 63;
    const int w = W > 1 ? threadIdx.x >> 6 : 0;
    const int piece = w * 64 + lane;
    const int64_t row = W > 1 ? static_cast<int64_t>(blockIdx.x)
                              : static_cast<int64_t>(blockIdx.x) * 4 +
                                    __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    if (row >= rows) return;
    const T* xr = x + row * stride;
    T* yr = y + row * stride;
    // The row's first boundary, whole pieces (one or more), and this lane's
    // single element (-1: none).
    const int head = static_cast<int>((-reinterpret_cast<uintptr_t>(xr) & 15) / sizeof(T));
    const int whole = (cols - head) / V;
    const int tail = cols - head - whole * V;
    const int single = piece < head ? piece : (piece < head + tail ? cols - tail + (piece - head) : -1);
    const T kNone = static_cast<T>(-INFINITY);
    T one = kNone;
    if (single >= 0) one = xr[single];
    // A piece past the row is the row's last one again, set to -inf below:
    // with no branch around the loads, the wait for one leaves those behind it
    // in flight.
    Vec v[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int first = c * (W * 64);
        const uint32_t off = static_cast<uint32_t>(min(piece, whole - 1 - first) + first) * 16u;
        v[c] = *reinterpret_cast<const Vec*>(reinterpret_cast<const char*>(xr + head) + off);
    }
    float m = static_cast<float>(one);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        if (whole < (c + 1) * (W * 64)) {
            const bool in = piece < whole - c * (W * 64);
#pragma unroll
            for (int i = 0; i < V; ++i) v[c][i] = in ? v[c][i] : kNone;
        }
#pragma unroll
        for (int i = 0; i < V; ++i) m = fmaxf(m, static_cast<float>(v[c][i]));
    }
    m = acrossWaves<W, true>(waveMax(m), smax);
    // exp(x - m) = 2^(x log2(e) - m log2(e)). Elements more than 300 below
    // the max (and the -inf of elements past the row) become m - 300, whose
    // result rounds to the same zero; NaN stays NaN. Where m - 300 is no value
    // of T near it, or m is infinite, softmaxOddRow runs.
    if (!(fabsf(m) <= R::kMostMax)) {
        softmaxOddRow<T, W>(xr, yr, cols, m, piece, ssum);
        return;
    }
    const T lo = static_cast<T>(m - 300.0f);
    const double mb = static_cast<double>(m) * -1.4426950408889634074;
    auto exponent = [&](T xv) {
        return __builtin_fma(static_cast<double>(static_cast<float>(xv)), 1.4426950408889634074, mb);
    };
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        if (c * (W * 64) >= whole) continue;   // past the row in every lane
#pragma unroll
        for (int i = 0; i < V; ++i) {
            v[c][i] = v[c][i] < lo ? lo : v[c][i];
            s += exp2Poly(exponent(v[c][i]), kExp2C10);
        }
        // The terms are recomputed below, not kept.
        asm volatile("" : "+v"(v[c]), "+v"(s));
    }
    if (w == 0) {
        one = one < lo ? lo : one;
        s += exp2Poly(exponent(one), kExp2C10);
    }
    s = acrossWaves<W, false>(waveSum(s), ssum);
    // s >= 1 or NaN, as in normalizeRow. A NaN row's outputs are all NaN (set
    // at the end: the exponent add would spoil a NaN coefficient).
    const bool bad = !(s > 0.0);
    const double inv = bad ? 0.0 : 1.0 / s;
    double co[NOut];
#pragma unroll
    for (int i = 0; i < NOut; ++i) {   // uniform over the row's waves: scalar registers
        const double k = kExp2C10[i] * inv;
        co[i] = __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(k)),
                                 __builtin_amdgcn_readfirstlane(__double2loint(k)));
    }
    const float nan = static_cast<float>(s);
    auto result = [&](T xv) {
        const T r = R::narrow(exp2Poly(exponent(xv), co));
        return bad ? static_cast<T>(nan) : r;
    };
    if (single >= 0) yr[single] = result(one);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int first = c * (W * 64);
        if (first >= whole) continue;
        Vec o;
#pragma unroll
        for (int i = 0; i < V; ++i) o[i] = result(v[c][i]);
        char* base = reinterpret_cast<char*>(yr + head) + first * 16;
        if (piece < whole - first) {
            __builtin_nontemporal_store(o, reinterpret_cast<Vec*>(base + static_cast<uint32_t>(piece) * 16u));
        }
    }
}

template <typename T>
__device__ __forceinline__ double ld(const void* p, int64_t i) {
    return static_cast<double>(static_cast<const T*>(p)[i]);
}

__device__ __forceinline__ double loadAny(const void* p, int dt, int64_t i) {
    if (dt == MLKD_F32) return ld<float>(p, i);
    if (dt == MLKD_F16) return static_cast<double>(static_cast<float>(static_cast<const _Float16*>(p)[i]));
    return ld<double>(p, i);
}

__device__ __forceinline__ void storeAny(void* p, int dt, int64_t i, double v) {
    if (dt == MLKD_F32) {
        static_cast<float*>(p)[i] = static_cast<float>(v);
    } else if (dt == MLKD_F16) {
        static_cast<_Float16*>(p)[i] = mlk::toHalf(v);
    } else {
        static_cast<double*>(p)[i] = v;
    }
}

__device__ __forceinline__ double blockReduce(double v, bool isMax, double* scratch) {
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double o = __shfl_xor(v, off, 64);
        v = isMax ? ((o > v) ? o : v) : v + o;
    }
    if (lane == 0) scratch[w] = v;
    __syncthreads();
    double r = scratch[0];
    for (int i = 1; i < static_cast<int>(blockDim.x >> 6); ++i) {
        r = isMax ? ((scratch[i] > r) ? scratch[i] : r) : r + scratch[i];
    }
    __syncthreads();
    return r;
}

/// General path: any dtype, any row length. f64 arithmetic as the reference.
__global__ __launch_bounds__(256) void softmaxBlockRow(mlkd_softmax p) {
    __shared__ double scratch[4];
    for (int64_t row = blockIdx.x; row < p.rows; row += gridDim.x) {
        const int64_t xo = row * p.x_row_stride;
        const int64_t yo = row * p.y_row_stride;
        double r = -INFINITY;
        for (int64_t c = threadIdx.x; c < p.cols; c += blockDim.x) {
            const double v = loadAny(p.x, p.x_dtype, xo + c);
            r = (v > r) ? v : r;
        }
        r = blockReduce(r, true, scratch);
        double s = 0.0;
        for (int64_t c = threadIdx.x; c < p.cols; c += blockDim.x) {
            s += exp(loadAny(p.x, p.x_dtype, xo + c) - r);
        }
        s = blockReduce(s, false, scratch);
        for (int64_t c = threadIdx.x; c < p.cols; c += blockDim.x) {
            const double e = exp(loadAny(p.x, p.x_dtype, xo + c) - r);
            storeAny(p.y, p.y_dtype, yo + c, s != 0.0 ? e / s : 0.0);
        }
    }
}

// Launch variant of the wave-per-row path. 0: one row per wave, v_exp_f32 and
// grouped sums, nontemporal stores; 1: rows pipelined over a grid of
// `gSoftmaxWaves` waves; 2: as 0 with the accurate expf and per-element f64
// sums; 3: as 0 with plain stores; 4: as 2 with plain stores; 5: as 0 with two
// adjacent rows per wave (the default: on gfx950 at 8192 x 4096, 38.9 us
// against 39.8 us for form 0 and 37.4 us for a copy of the same bytes). Set
// by the variant search (mlkd_softmax_set_variant).
int gSoftmaxVariant = 5;
int64_t gSoftmaxWaves = 0;

template <int CH>
int launchWave(const mlkd_softmax& p, hipStream_t st) {
    const int variant = p.variant >= 0 ? p.variant : gSoftmaxVariant;
    if (variant == 1) {
        int64_t waves = gSoftmaxWaves > 0 ? gSoftmaxWaves : 2048;
        if (waves > p.rows) waves = p.rows;
        const int64_t blocks = (waves + 3) / 4;
        hipLaunchKernelGGL(softmaxWaveRowPipelined<CH>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                           static_cast<const float*>(p.x), static_cast<float*>(p.y), p.rows, p.cols,
                           p.x_row_stride, p.y_row_stride);
        return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
    }
    const bool full = p.cols == 256 * CH;
    if (variant == 5) {
        int64_t blocks = ((p.rows + 1) / 2 + 3) / 4;
        if (blocks > 8192) blocks = 8192;
        auto pair = full ? softmaxWaveRowPair<CH, true> : softmaxWaveRowPair<CH, false>;
        hipLaunchKernelGGL(pair, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                           static_cast<const float*>(p.x), static_cast<float*>(p.y), p.rows, p.cols,
                           p.x_row_stride, p.y_row_stride);
        return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
    }
    int64_t blocks = (p.rows + 3) / 4;
    if (gSoftmaxWaves > 0 && blocks > (gSoftmaxWaves + 3) / 4) blocks = (gSoftmaxWaves + 3) / 4;
    if (blocks > 8192) blocks = 8192;
    auto kern = softmaxWaveRow<CH, true, true>;
    if (variant == 2) kern = softmaxWaveRow<CH, false, true>;
    if (variant == 3) kern = softmaxWaveRow<CH, true, false>;
    if (variant == 4) kern = softmaxWaveRow<CH, false, false>;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, static_cast<const float*>(p.x),
                       static_cast<float*>(p.y), p.rows, p.cols, p.x_row_stride, p.y_row_stride);
    return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
}

template <int CH>
int launchScalar(const mlkd_softmax& p, hipStream_t st) {
    constexpr int64_t rowsPer = 4 / kScalarWaves<CH>;
    int64_t blocks = (p.rows + rowsPer - 1) / rowsPer;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(softmaxWaveRowScalar<CH>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                       static_cast<const float*>(p.x), static_cast<float*>(p.y), p.rows, p.cols, p.x_row_stride,
                       p.y_row_stride);
    return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
}

/// softmaxRowWide applies to one dtype in and out (f32 or f16), rows of x and
/// y with the same offset from a 16-byte boundary, 16 (a whole piece)
/// to 65536 columns: what the registers of 16 waves hold.
bool wideApplies(const mlkd_softmax* p) {
    const bool f32 = p->x_dtype == MLKD_F32 && p->y_dtype == MLKD_F32;
    const bool f16 = p->x_dtype == MLKD_F16 && p->y_dtype == MLKD_F16;
    const int64_t es = f32 ? 4 : 2;
    return (f32 || f16) && p->cols >= 16 && p->cols <= 65536 &&
           p->x_row_stride == p->y_row_stride &&
           ((reinterpret_cast<uintptr_t>(p->x) ^ reinterpret_cast<uintptr_t>(p->y)) & 15u) == 0 &&
           reinterpret_cast<uintptr_t>(p->x) % static_cast<uintptr_t>(es) == 0;
}

/// A grid holds fewer than 2^32 threads, so fewer than 2^26 rows of one wave
/// (2 GiB of f16 rows of 16 columns) or 2^24 of four: more go in several
/// launches of 2^31 threads, whose own time is nothing beside such rows'.
template <typename T, int CH, int W>
int launchWideAs(const mlkd_softmax& p, hipStream_t st) {
    constexpr int threads = W == 1 ? 256 : 64 * W;
    constexpr int64_t rowsPer = W > 1 ? 1 : 4, most = (int64_t{1} << 31) / threads * rowsPer;
    for (int64_t row = 0; row < p.rows; row += most) {
        const int64_t rows = std::min(p.rows - row, most);
        hipLaunchKernelGGL((softmaxRowWide<T, CH, W>), dim3(static_cast<unsigned>((rows + rowsPer - 1) / rowsPer)),
                           dim3(threads), 0, st, static_cast<const T*>(p.x) + row * p.x_row_stride,
                           static_cast<T*>(p.y) + row * p.x_row_stride, rows, static_cast<int>(p.cols), p.x_row_stride);
    }
    return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
}

/// Waves per row (w) and pieces per lane (ch) by row length. f16 rows up to
/// 2048 columns take one wave and no barrier.
struct WideShape {
    int ch, w;
};

WideShape wideShape(const mlkd_softmax& p) {
    if (p.x_dtype == MLKD_F16) {
        const int64_t c = p.cols;
        if (c <= 512) return {1, 1};
        if (c <= 1024) return {2, 1};
        if (c <= 2048) return {4, 1};
        if (c <= 4096) return {2, 4};
        if (c <= 8192) return {4, 4};
        if (c <= 16384) return {4, 8};
        return c <= 32768 ? WideShape{4, 16} : WideShape{8, 16};
    }
    const int64_t c = p.cols;
    if (c <= 16384) return {16, 4};
    return c <= 32768 ? WideShape{16, 8} : WideShape{16, 16};
}

int launchWide(const mlkd_softmax& p, hipStream_t st) {
    const WideShape f = wideShape(p);
    if (p.x_dtype == MLKD_F16) {
        if (f.w == 1) {
            if (f.ch == 1) return launchWideAs<_Float16, 1, 1>(p, st);
            return f.ch == 2 ? launchWideAs<_Float16, 2, 1>(p, st) : launchWideAs<_Float16, 4, 1>(p, st);
        }
        if (f.w == 4) return f.ch == 2 ? launchWideAs<_Float16, 2, 4>(p, st) : launchWideAs<_Float16, 4, 4>(p, st);
        if (f.w == 8) return launchWideAs<_Float16, 4, 8>(p, st);
        return f.ch == 4 ? launchWideAs<_Float16, 4, 16>(p, st) : launchWideAs<_Float16, 8, 16>(p, st);
    }
    if (f.w == 4) return launchWideAs<float, 16, 4>(p, st);
    return f.w == 8 ? launchWideAs<float, 16, 8>(p, st) : launchWideAs<float, 16, 16>(p, st);
}

/// f32 rows up to 8192 columns that the float4 path does not take.
bool scalarApplies(const mlkd_softmax* p) {
    return p->x_dtype == MLKD_F32 && p->y_dtype == MLKD_F32 && p->cols <= 8192 &&
           (reinterpret_cast<uintptr_t>(p->x) & 3u) == 0 && (reinterpret_cast<uintptr_t>(p->y) & 3u) == 0;
}

}  // namespace

extern "C" void mlkd_softmax_set_variant(int variant, int64_t waves) {
    gSoftmaxVariant = variant;
    gSoftmaxWaves = waves;
}

extern "C" const char* mlkd_softmax_kernel_name(const mlkd_softmax* p) {
    static thread_local char name[96];
    const bool aligned = (reinterpret_cast<uintptr_t>(p->x) & 15u) == 0 &&
                         (reinterpret_cast<uintptr_t>(p->y) & 15u) == 0 &&
                         (p->x_row_stride & 3) == 0 && (p->y_row_stride & 3) == 0;
    int ch = 1;
    while (256 * ch < p->cols) ch *= 2;
    if (!(p->x_dtype == MLKD_F32 && p->y_dtype == MLKD_F32 && (p->cols & 3) == 0 && aligned && p->cols <= 8192)) {
        if (!scalarApplies(p)) {
            if (!wideApplies(p)) return "softmaxBlockRow";
            const WideShape f = wideShape(*p);
            std::snprintf(name, sizeof(name), "softmaxRowWide<%s, %d, %d>", p->x_dtype == MLKD_F16 ? "_Float16" : "float",
                          f.ch, f.w);
            return name;
        }
        std::snprintf(name, sizeof(name), "softmaxWaveRowScalar<%d>", ch);
        return name;
    }
    const int variant = p->variant >= 0 ? p->variant : gSoftmaxVariant;
    if (variant == 1) {
        std::snprintf(name, sizeof(name), "softmaxWaveRowPipelined<%d>", ch);
    } else if (variant == 5) {
        std::snprintf(name, sizeof(name), "softmaxWaveRowPair<%d, %s>", ch, p->cols == 256 * ch ? "true" : "false");
    } else {
        const bool fastExp = variant != 2 && variant != 4, nt = variant != 3 && variant != 4;
        std::snprintf(name, sizeof(name), "softmaxWaveRow<%d, %s, %s>", ch, fastExp ? "true" : "false",
                      nt ? "true" : "false");
    }
    return name;
}

extern "C" int mlkd_launch_softmax(const mlkd_softmax* p, void* stream) {
    if (p == nullptr || p->rows < 0 || p->cols < 0) return MLKD_RT_LAUNCH;
    if (p->rows == 0 || p->cols == 0) return 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool aligned = (reinterpret_cast<uintptr_t>(p->x) & 15u) == 0 &&
                         (reinterpret_cast<uintptr_t>(p->y) & 15u) == 0 &&
                         (p->x_row_stride & 3) == 0 && (p->y_row_stride & 3) == 0;
    if (p->x_dtype == MLKD_F32 && p->y_dtype == MLKD_F32 && (p->cols & 3) == 0 && aligned) {
        if (p->cols <= 256) return launchWave<1>(*p, st);
        if (p->cols <= 512) return launchWave<2>(*p, st);
        if (p->cols <= 1024) return launchWave<4>(*p, st);
        if (p->cols <= 2048) return launchWave<8>(*p, st);
        if (p->cols <= 4096) return launchWave<16>(*p, st);
        if (p->cols <= 8192) return launchWave<32>(*p, st);
    }
    if (scalarApplies(p)) {
        if (p->cols <= 256) return launchScalar<1>(*p, st);
        if (p->cols <= 512) return launchScalar<2>(*p, st);
        if (p->cols <= 1024) return launchScalar<4>(*p, st);
        if (p->cols <= 2048) return launchScalar<8>(*p, st);
        if (p->cols <= 4096) return launchScalar<16>(*p, st);
        return launchScalar<32>(*p, st);
    }
    if (wideApplies(p)) return launchWide(*p, st);
    int64_t blocks = p->rows < 65536 ? p->rows : 65536;
    hipLaunchKernelGGL(softmaxBlockRow, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, *p);
    return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
}

namespace {

/// Row sum (Call(ReduceSum), kernel_buffers.cpp:237-277, and the poly.synth
/// ReduceSum nest): one wave per row, f64 accumulation (strided per lane,
/// then a wave reduction).
__global__ __launch_bounds__(256) void rowSumWave(mlkd_softmax p) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int64_t waves = static_cast<int64_t>(gridDim.x) * 4;
    for (int64_t row = wave; row < p.rows; row += waves) {
        double s = 0.0;
        for (int64_t c = lane; c < p.cols; c += 64) s += loadAny(p.x, p.x_dtype, row * p.x_row_stride + c);
        s = waveSum(s);
        if (lane == 0) storeAny(p.y, p.y_dtype, row * p.y_row_stride, s);
    }
}

}  // namespace

extern "C" int mlkd_launch_rowsum(const mlkd_softmax* p, void* stream) {
    if (p == nullptr || p->rows < 0 || p->cols < 0) return MLKD_RT_LAUNCH;
    if (p->rows == 0) return 0;
    int64_t blocks = (p->rows + 3) / 4;
    if (blocks > 16384) blocks = 16384;
    hipLaunchKernelGGL(rowSumWave, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), *p);
    return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
}
