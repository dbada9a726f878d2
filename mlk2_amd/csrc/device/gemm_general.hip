// The general GEMM: C[M,N] (+)= A[M,K] * B[K,N], row-major, for the shapes and
// dtypes the tiled MFMA forms of gemm.hip leave.
//
// One operand dtype (f16 with an f32 C, f32, f64): MFMA straight from global
// memory, no LDS staging (directTile). Anything else: a scalar kernel, 64x64
// tiles through LDS.
#include "gemm_general.h"

#include <stdint.h>

#include <algorithm>

#include "mlk_device_math.h"
#include "xcd.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ T ldAny(const void* p, int dt, int64_t i) {
    if (dt == MLKD_F32) return static_cast<T>(static_cast<const float*>(p)[i]);
    if (dt == MLKD_F16) return static_cast<T>(static_cast<float>(static_cast<const _Float16*>(p)[i]));
    return static_cast<T>(static_cast<const double*>(p)[i]);
}

template <typename T>
__device__ __forceinline__ void stAny(void* p, int dt, int64_t i, T v) {
    if (dt == MLKD_F32) {
        static_cast<float*>(p)[i] = static_cast<float>(v);
    } else if (dt == MLKD_F16) {
        if constexpr (sizeof(T) == sizeof(double)) static_cast<_Float16*>(p)[i] = mlk::toHalf(v);
        else static_cast<_Float16*>(p)[i] = static_cast<_Float16>(v);
    } else {
        static_cast<double*>(p)[i] = static_cast<double>(v);
    }
}

// -------------------------------------------------------------- scalar ----
/// One 64x64 output tile by 256 threads, 4x4 per thread, K slabs of 16
/// through LDS; k ascending per output element, starting from C's old value
/// in the accumulate form (the reference's order, kernel_buffers.cpp:
/// 406-432). With skip_zero_a the products of A[i,p] == 0 are left out, as
/// there (:422).
template <typename T>
__device__ __forceinline__ void generalTile(const mlkd_gemm& p, int64_t row0, int64_t col0, T (&As)[16][65],
                                            T (&Bs)[16][65]) {
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    T acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t r = row0 + ty * 4 + i, c = col0 + tx * 4 + j;
            acc[i][j] = (p.accumulate && r < p.m && c < p.n) ? ldAny<T>(p.c, p.c_dtype, r * p.ldc + c) : T(0);
        }
    }
    const bool skip = p.skip_zero_a != 0;
    for (int64_t k0 = 0; k0 < p.k; k0 += 16) {
        for (int e = threadIdx.x; e < 16 * 64; e += 256) {
            const int kk = e / 64, mm = e % 64;
            const int64_t r = row0 + mm, kA = k0 + kk;
            As[kk][mm] = (r < p.m && kA < p.k) ? ldAny<T>(p.a, p.a_dtype, r * p.lda + kA) : T(0);
            const int64_t c = col0 + mm;
            Bs[kk][mm] = (c < p.n && kA < p.k) ? ldAny<T>(p.b, p.b_dtype, kA * p.ldb + c) : T(0);
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            T a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (skip && a[i] == T(0)) continue;
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t r = row0 + ty * 4 + i, c = col0 + tx * 4 + j;
            if (r < p.m && c < p.n) stAny<T>(p.c, p.c_dtype, r * p.ldc + c, acc[i][j]);
        }
    }
}

/// Any shape and dtype mix: one 64x64 tile per workgroup.
template <typename T>
__global__ __launch_bounds__(256) void gemmGeneral(mlkd_gemm p) {
    __shared__ T As[16][65];
    __shared__ T Bs[16][65];
    const int64_t tilesN = (p.n + 63) / 64;
    generalTile<T>(p, (blockIdx.x / tilesN) * 64, (blockIdx.x % tilesN) * 64, As, Bs);
}

// -------------------------------------------------------------- direct ----
/// Per operand type: V elements to 16 bytes and the accumulators of one 16x16
/// MFMA tile (column lane % 16, rows by lane group lane / 16).
template <typename T>
struct Direct;
template <>
struct Direct<_Float16> {
    static constexpr int V = 8;
    using Vec = f16x8;
    using Acc = f32x4;
    using Out = float;
    /// Row q of the tile is accumulator entry(q) in lane group group(q).
    static __device__ __forceinline__ int group(int q) { return q / 4; }
    static __device__ __forceinline__ int entry(int q) { return q % 4; }
    /// acc[j] += a * B over 32 k, for the 8 column tiles j: lane l of tile j
    /// holds column 8 (l % 16) + j. b[i] is 8 columns of k-row i of the
    /// lane's group; column j's 8 k-values are gathered across the b[i].
    static __device__ __forceinline__ void columns(const Vec (&b)[V], Vec (&f)[V]) {
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
            u32x4 o;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                o[q] = __builtin_amdgcn_perm(__builtin_bit_cast(u32x4, b[2 * q + 1])[j >> 1],
                                             __builtin_bit_cast(u32x4, b[2 * q])[j >> 1], sel);
            }
            f[j] = __builtin_bit_cast(Vec, o);
        }
    }
    template <int MT>
    static __device__ __forceinline__ void multiply(const Vec (&a)[MT], const Vec (&b)[V], Acc (&acc)[MT][V]) {
        Vec f[V];
        columns(b, f);
#pragma unroll
        for (int j = 0; j < V; ++j) {
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], f[j], acc[t][j], 0, 0, 0);
        }
    }
};
template <>
struct Direct<float> {
    static constexpr int V = 4;
    using Vec = f32x4;
    using Acc = f32x4;
    using Out = float;
    /// Row q of the tile is accumulator entry(q) in lane group group(q).
    static __device__ __forceinline__ int group(int q) { return q / 4; }
    static __device__ __forceinline__ int entry(int q) { return q % 4; }
    /// 16 k in 4 MFMAs a tile: MFMA i takes k = V g + i from lane group g, so
    /// an A operand is one element of the lane's 16 bytes of its row, a B
    /// operand one of the lane's 16 bytes of its k-row.
    template <int MT>
    static __device__ __forceinline__ void multiply(const Vec (&a)[MT], const Vec (&b)[V], Acc (&acc)[MT][V]) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
#pragma unroll
            for (int j = 0; j < V; ++j) {
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][i], b[i][j], acc[t][j], 0, 0, 0);
                }
            }
        }
    }
};
template <>
struct Direct<double> {
    static constexpr int V = 2;
    using Vec = f64x2;
    using Acc = f64x4;
    using Out = double;
    static __device__ __forceinline__ int group(int q) { return q % 4; }
    static __device__ __forceinline__ int entry(int q) { return q / 4; }
    template <int MT>
    static __device__ __forceinline__ void multiply(const Vec (&a)[MT], const Vec (&b)[V], Acc (&acc)[MT][V]) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
#pragma unroll
            for (int j = 0; j < V; ++j) {
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    acc[t][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t][i], b[i][j], acc[t][j], 0, 0, 0);
                }
            }
        }
    }
};

/// 16 bytes of consecutive elements at any element alignment.
template <typename T>
struct __attribute__((packed, aligned(sizeof(T)))) Packed {
    typename Direct<T>::Vec v;
};

/// Call(MatMul)'s element, as the reference computes it: C_in plus A[i,p] *
/// B[p,j] over p ascending, skipping A[i,p] == 0. The skip changes an element
/// only where its column of B holds an infinity or a NaN, and there the
/// MFMA sum is not finite (0 * inf is NaN), so only such elements take this,
/// or exactTile. The sum is one serial chain, so 16 steps' loads go out ahead
/// of it (16x4096x1024 f64 with one infinity in B: 147 us; one step at a time
/// 1249).
template <typename T, typename O>
__device__ __forceinline__ O exactElement(const T* a, const T* b, int64_t ldb, int k, O c) {
    constexpr int V = Direct<T>::V, U = 16;
    auto step = [&](T at, T bt) {
        const O av = static_cast<O>(at);
        if (av != O(0)) c = c + av * static_cast<O>(bt);
    };
    int p = 0;
#pragma unroll 1
    for (; p + U <= k; p += U) {
        typename Direct<T>::Vec av[U / V];
        T bv[U];
#pragma unroll
        for (int i = 0; i < U / V; ++i) av[i] = reinterpret_cast<const Packed<T>*>(a + p + i * V)->v;
#pragma unroll
        for (int i = 0; i < U; ++i) bv[i] = b[(p + i) * ldb];
#pragma unroll
        for (int i = 0; i < U; ++i) step(av[i / V][i % V], bv[i]);
    }
#pragma unroll 1
    for (; p < k; ++p) step(a[p], b[p * ldb]);
    return c;
}

/// A launch of directTile: a 16 MT x 16 V tile of C per workgroup of `waves`
/// waves and K range of `splitSteps` steps of 4 V k (blockIdx.y); with more
/// than one range the sums go to part[range][m][n].
template <typename T, int MT>
struct DirectArgs {
    const T* a;
    const T* b;
    typename Direct<T>::Out* c;
    typename Direct<T>::Out* part;
    int64_t lda, ldb, ldc;
    int m, n, k;
    int waves, splitSteps, tilesM;
    int accumulate, skip;
};

/// exactElement over a workgroup's whole tile, up to R rows of a column to a
/// thread, K by slabs of KC through LDS. Measured with one infinity in B (each
/// element by itself, one step at a time; the scalar kernel): f64 512^3 84 us
/// (195; 163), 1024^3 308 us (1714; 372).
template <typename T, int MT>
__device__ __forceinline__ void exactTile(const DirectArgs<T, MT>& p, int row0, int col0, unsigned char* lds) {
    using Out = typename Direct<T>::Out;
    constexpr int R = MT == 1 ? 4 : 8, KC = 8, TR = 16 * MT, TC = 16 * Direct<T>::V;
    static_assert(KC * (TR + TC) * sizeof(T) <= MT * Direct<T>::V * 64 * sizeof(typename Direct<T>::Acc),
                  "the slabs fit the sums' LDS");
    T* as = reinterpret_cast<T*>(lds);   // [KC][TR]
    T* bs = as + KC * TR;                // [KC][TC]
    const int rows = min(TR, p.m - row0), cols = min(TC, p.n - col0);
    const int tid = static_cast<int>(threadIdx.x), threads = 64 * p.waves;
    const int cw = min(TC, threads), step = threads / cw;   // columns at once; rows apart of a thread's
    for (int cb = 0; cb < cols; cb += cw) {
        for (int rb = 0; rb < rows; rb += R * step) {
            const int col = cb + tid % cw, row = rb + tid / cw;
            const int staged = min(R * step, TR - rb);
            Out* c = p.c + static_cast<int64_t>(row0) * p.ldc + col0 + col;
            Out s[R];
#pragma unroll
            for (int i = 0; i < R; ++i) {
                s[i] = col < cols && row + i * step < rows ? c[(row + i * step) * p.ldc] : Out(0);
            }
            for (int k0 = 0; k0 < p.k; k0 += KC) {
                __syncthreads();
                for (int e = tid; e < staged * KC; e += threads) {
                    const int r = rb + e / KC, k = k0 + e % KC;
                    as[e % KC * TR + e / KC] = r < rows && k < p.k ? p.a[(row0 + r) * p.lda + k] : T(0);
                }
                for (int e = tid; e < cw * KC; e += threads) {
                    const int k = k0 + e / cw, j = cb + e % cw;
                    bs[e / cw * TC + e % cw] = j < cols && k < p.k ? p.b[k * p.ldb + col0 + j] : T(0);
                }
                __syncthreads();
#pragma unroll
                for (int k = 0; k < KC; ++k) {
                    const Out bv = static_cast<Out>(bs[k * TC + tid % cw]);
#pragma unroll
                    for (int i = 0; i < R; ++i) {
                        const Out av = static_cast<Out>(as[k * TR + min(tid / cw + i * step, TR - 1)]);
                        if (av != Out(0)) s[i] = s[i] + av * bv;
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < R; ++i) {
                if (col < cols && row + i * step < rows) c[(row + i * step) * p.ldc] = s[i];
            }
        }
    }
}

/// One tile, operands straight from global memory into MFMA operand registers
/// (the layouts above make every load 16 bytes of a row), so that a small
/// product needs no staging, no barrier before its sums meet, and can be cut
/// into as many waves as fill the chip: the waves of a workgroup take the K
/// steps round robin and add up through LDS, two halves at a time. DEPTH
/// steps of loads are in flight. Edges: rows past M and columns past N repeat
/// the last ones (the columns as the last V whole ones) and are not stored;
/// a partial last K step is the last 4 V k with zeros for those done already,
/// taken by one wave. Needs n >= V and k >= 4 V.
/// Measured against the scalar kernel: f16 16x4096x4096 12.5 us (1385 us; B
/// alone 34 MB, 6.3 us of HBM), 8x512x512 4.5 us (145 us), f64 512^3 9.5 us
/// (187 us; its MFMAs 3.9 us), 1024^3 39 us, 55 TFLOP/s (370 us). Small ones
/// are bound by the chain of launch, first load and the waves' sum, large
/// ones by the L1's 64 bytes a clock (f16) or the MFMAs (f32, f64). The code is kept short (the
/// store is one loop out of LDS): a small product runs it once, cold.
template <typename T, int MT, int DEPTH>
__device__ __forceinline__ void directTile(const DirectArgs<T, MT>& p) {
    using D = Direct<T>;
    using Vec = typename D::Vec;
    using Acc = typename D::Acc;
    using Out = typename D::Out;
    constexpr int V = D::V, KS = 4 * V;
    extern __shared__ __align__(16) unsigned char ldsG[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int l16 = lane & 15, g = lane >> 4;
    // Each XCD takes a contiguous share of the tiles, down the columns of C,
    // so that a B panel is read into one L2, or two. In grid order instead
    // every L2 reads it, f16 64x4096x8000 (252 tiles) 47.0 us against 18.7,
    // 105x4096x8000 67.4 against 30.1, f32 40x4096x4032 31.4 against 23.6.
    const int id = xcdShare(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
    const int row0 = id % p.tilesM * (16 * MT), col0 = id / p.tilesM * (16 * V);
    const int myCol = col0 + l16 * V;              // nominal first column
    const int useCol = min(myCol, p.n - V);        // first column read
    const int fullSteps = p.k / KS;
    const int s0 = static_cast<int>(blockIdx.y) * p.splitSteps;
    const int s1 = min(s0 + p.splitSteps, fullSteps);   // full steps of this range
    const int count = s1 > s0 + wave ? (s1 - s0 - wave + p.waves - 1) / p.waves : 0;

    uint32_t aOff[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        aOff[t] = static_cast<uint32_t>((min(row0 + t * 16 + l16, p.m - 1) - row0) * p.lda + g * V) * sizeof(T);
    }
    const uint32_t bOff = static_cast<uint32_t>(g * V * p.ldb + (useCol - min(col0, p.n - V))) * sizeof(T);
    const char* aBase = reinterpret_cast<const char*>(p.a + row0 * p.lda);
    const char* bBase = reinterpret_cast<const char*>(p.b + min(col0, p.n - V));

    Acc acc[MT][V];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int j = 0; j < V; ++j) acc[t][j] = Acc{0, 0, 0, 0};
    }
    auto loadAt = [&](int k0, Vec (&av)[MT], Vec (&bv)[V]) {
        const char* ak = aBase + static_cast<int64_t>(k0) * static_cast<int64_t>(sizeof(T));
        const char* bk = bBase + k0 * p.ldb * static_cast<int64_t>(sizeof(T));
#pragma unroll
        for (int t = 0; t < MT; ++t) av[t] = reinterpret_cast<const Packed<T>*>(ak + aOff[t])->v;
#pragma unroll
        for (int r = 0; r < V; ++r) {
            bv[r] = reinterpret_cast<const Packed<T>*>(bk + r * p.ldb * static_cast<int64_t>(sizeof(T)) + bOff)->v;
        }
    };
    if (count > 0) {
        Vec a[DEPTH][MT], b[DEPTH][V];
        // Step i of this wave, or its last one again (which is not used).
        auto load = [&](int i, Vec (&av)[MT], Vec (&bv)[V]) {
            loadAt((s0 + wave + min(i, count - 1) * p.waves) * KS, av, bv);
        };
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) load(d, a[d], b[d]);
        int i = 0;
        for (; i + DEPTH < count; i += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                D::multiply(a[d], b[d], acc);
                load(i + d + DEPTH, a[d], b[d]);
            }
        }
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            if (i + d < count) D::multiply(a[d], b[d], acc);
        }
    }
    const int rest = p.k - fullSteps * KS;
    if (rest > 0 && blockIdx.y == gridDim.y - 1 && wave == p.waves - 1) {
        // The last KS k, those that full steps took set to zero.
        Vec av[MT], bv[V];
        loadAt(p.k - KS, av, bv);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const bool fresh = g * V + e >= KS - rest;
#pragma unroll
            for (int t = 0; t < MT; ++t) av[t][e] = fresh ? av[t][e] : T(0);
            bv[e] = fresh ? bv[e] : Vec(T(0));
        }
        D::multiply(av, bv, acc);
    }
    // The waves' sums: the upper half hands over to the lower, until wave 0
    // has the tile, which all of them then store. 8 spare entries between
    // fragments keep the store's reads at 4 lanes a bank.
    constexpr int F = 64 + 8;
    Acc* red = reinterpret_cast<Acc*>(ldsG);
    auto slot = [&](int w, int t, int j) { return red + ((w * MT + t) * V + j) * F + lane; };
    for (int half = p.waves / 2; half > 0; half /= 2) {
        if (wave >= half && wave < 2 * half) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
#pragma unroll
                for (int j = 0; j < V; ++j) *slot(wave - half, t, j) = acc[t][j];
            }
        }
        __syncthreads();
        if (wave < half) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
#pragma unroll
                for (int j = 0; j < V; ++j) acc[t][j] += *slot(wave, t, j);
            }
        }
        __syncthreads();
    }
    Out* part = gridDim.y > 1 ? p.part + static_cast<int64_t>(blockIdx.y) * p.m * p.n : nullptr;
    const bool exact = p.skip && part == nullptr;   // a sum that is not finite: exactTile
    int* odd = reinterpret_cast<int*>(red + 64);    // in the spare entries
    if (wave == 0) {
        bool bad = false;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int j = 0; j < V; ++j) {
                *slot(0, t, j) = acc[t][j];
#pragma unroll
                for (int e = 0; e < 4; ++e) bad |= exact && !__builtin_isfinite(acc[t][j][e]);
            }
        }
        if (exact) {
            const bool any = __builtin_amdgcn_ballot_w64(bad) != 0;
            if (lane == 0) *odd = any ? 1 : 0;
        }
    }
    __syncthreads();
    if (__builtin_expect(exact && __builtin_amdgcn_readfirstlane(*odd) != 0, 0)) {   // out of the cold path
        exactTile<T, MT>(p, row0, col0, ldsG);
        return;
    }
    const Out* sums = reinterpret_cast<const Out*>(ldsG);
    const int rows = min(16 * MT, p.m - row0), cols = min(16 * V, p.n - col0);
    // Column i of the tile is column i - shift of the ones read (shift > 0
    // in the last lane read of a ragged N: its V columns end at N).
    auto sumAt = [&](int row, int col) {
        const int owner = col / V;
        const int j = col0 + col - min(col0 + owner * V, p.n - V);
        const int q = row % 16;
        return sums[(((row / 16) * V + j) * F + D::group(q) * 16 + owner) * 4 + D::entry(q)];
    };
    const int threads = 64 * p.waves;
    if (p.accumulate && part == nullptr) {
        // Four rows of C read before the first is written (one: f16
        // 200x700x300 with C += A B 7.5 us, four: 6.8).
        constexpr int R = 4;
        const int cw = min(16 * V, threads), step = threads / cw;
        for (int col = static_cast<int>(threadIdx.x) % cw; col < cols; col += cw) {
            for (int row = static_cast<int>(threadIdx.x) / cw; row < rows; row += R * step) {
                Out* dst = p.c + static_cast<int64_t>(row0 + row) * p.ldc + col0 + col;
                Out v[R];
#pragma unroll
                for (int i = 0; i < R; ++i) v[i] = row + i * step < rows ? dst[i * step * p.ldc] : Out(0);
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    if (row + i * step < rows) dst[i * step * p.ldc] = v[i] + sumAt(row + i * step, col);
                }
            }
        }
        return;
    }
    for (int i = static_cast<int>(threadIdx.x); i < rows * (16 * V); i += threads) {
        const int row = i / (16 * V), col = i % (16 * V);
        if (col >= cols) continue;
        const Out v = sumAt(row, col);
        if (part != nullptr) part[static_cast<int64_t>(row0 + row) * p.n + col0 + col] = v;
        else p.c[static_cast<int64_t>(row0 + row) * p.ldc + col0 + col] = v;
    }
}

// The launches of directTile, by operand type and row tiles: overloads of
// gemmGeneral, whose template argument is the accumulators' type. DEPTH: what
// the registers of 2 waves per SIMD (f16, MT 4), or of 4, hold.
#define MLK_GENERAL(T, MT, DEPTH, THREADS, WAVES)                                                   \
    template <typename Sum>                                                                         \
    __global__ __launch_bounds__(THREADS, WAVES) void gemmGeneral(DirectArgs<T, MT> p) {            \
        static_assert(sizeof(Sum) == sizeof(typename Direct<T>::Out));                              \
        directTile<T, MT, DEPTH>(p);                                                                \
    }
MLK_GENERAL(_Float16, 1, 2, 512, 3)
MLK_GENERAL(_Float16, 2, 2, 512, 2)
MLK_GENERAL(_Float16, 4, 2, 512, 2)
MLK_GENERAL(float, 1, 4, 512, 4)
MLK_GENERAL(float, 2, 3, 512, 4)
MLK_GENERAL(float, 4, 2, 512, 3)
MLK_GENERAL(double, 1, 4, 512, 4)
MLK_GENERAL(double, 2, 4, 512, 4)
MLK_GENERAL(double, 4, 2, 512, 3)
#undef MLK_GENERAL

/// C (+)= the sum of the K ranges' parts, in order.
template <typename T>
__global__ __launch_bounds__(256) void gemmSumParts(DirectArgs<T, 1> p, int ranges) {
    using Out = typename Direct<T>::Out;
    const int64_t total = static_cast<int64_t>(p.m) * p.n;
    const int col = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
    if (col >= p.n) return;
    for (int row = static_cast<int>(blockIdx.y); row < p.m; row += static_cast<int>(gridDim.y)) {
        const Out* part = p.part + static_cast<int64_t>(row) * p.n + col;
        Out* dst = p.c + row * p.ldc + col;
        const Out old = p.accumulate ? *dst : Out(0);
        Out v = part[0];
#pragma unroll 8
        for (int s = 1; s < ranges; ++s) v += part[s * total];
        v = old + v;
        if (__builtin_expect(p.skip && !__builtin_isfinite(v), 0)) v = exactElement<T, Out>(p.a + row * p.lda, p.b + col, p.ldb, p.k, old);
        *dst = v;
    }
}

/// How a product runs on directTile: row tiles per workgroup, waves per
/// workgroup, K ranges; mt 0 when it does not (mixed dtypes, fewer columns
/// than one vector, K under one step, strides past the 32-bit lane offsets).
struct DirectPlan {
    int mt = 0, waves = 1, ranges = 1, splitSteps = 0;
    int tilesM = 0, tilesN = 0;
};

DirectPlan directPlan(const mlkd_gemm* p) {
    DirectPlan d;
    const bool f16 = p->a_dtype == MLKD_F16 && p->b_dtype == MLKD_F16 && p->c_dtype == MLKD_F32;
    const bool f32 = p->a_dtype == MLKD_F32 && p->b_dtype == MLKD_F32 && p->c_dtype == MLKD_F32;
    const bool f64 = p->a_dtype == MLKD_F64 && p->b_dtype == MLKD_F64 && p->c_dtype == MLKD_F64;
    if (!(f16 || f32 || f64)) return d;
    const int v = f16 ? 8 : (f32 ? 4 : 2), ks = 4 * v;
    const uintptr_t es = 16u / static_cast<uintptr_t>(v), os = f64 ? 8 : 4;
    if (p->m <= 0 || p->n < v || p->k < ks || p->m >= (1 << 30) || p->n >= (1 << 30) || p->k >= (1 << 30) ||
        p->lda >= (1 << 26) / static_cast<int64_t>(es) || p->ldb >= (1 << 26) || reinterpret_cast<uintptr_t>(p->a) % es != 0 ||
        reinterpret_cast<uintptr_t>(p->b) % es != 0 || reinterpret_cast<uintptr_t>(p->c) % os != 0) {
        return d;
    }
    if (p->skip_zero_a != 0 && p->accumulate == 0) return d;   // no such Call; the scalar kernel skips in order
    const int64_t tilesN = (p->n + 16 * v - 1) / (16 * v);
    const int64_t steps = (p->k + ks - 1) / ks;
    // Row tiles: the fewest that cover M, up to 4; fewer where that leaves
    // under two tiles for each of the 256 CUs.
    int mt = p->m <= 16 ? 1 : (p->m <= 32 ? 2 : 4);
    while (mt > 1 && p->m > 16 * mt / 2 && (p->m + 16 * mt - 1) / (16 * mt) * tilesN < 512 && p->m > 16) mt /= 2;
    const int64_t tilesM = (p->m + 16 * mt - 1) / (16 * mt);
    const int64_t tiles = tilesM * tilesN;
    if (tiles > 0x7FFFFFFF) return d;
    // Waves: towards 2048 on the chip, each with two steps or more. With a
    // long K and tiles to spare CUs, four, and K ranges over more workgroups
    // up to one a CU (their sums meet in a second kernel, about 3 us), each
    // wave keeping 8 steps. Measured, f16 16x4096x4096 (32 tiles, 128 steps):
    // 4 waves x 4 ranges 12.5 us, 1 range 18.9, 8 ranges 14.2, 8 waves x 1-8
    // ranges 14.6-18.6; 4x8192x8191: 4 x 4 27 us, 4 x 1 65; f16 16x1024x8192
    // (64 tiles, 32 steps): 4 x 1 8.4 us, 4 x 2 9.8. f64 512^3 (256 tiles): 1,
    // 2, 4 and 8 waves 13.3, 12.4, 9.5 and 9.9 us.
    int waves = 1;
    int64_t ranges = 1;
    if (steps >= 64 && tiles <= 128) {
        waves = 4;
        while (tiles * ranges * 2 <= 256 && steps >= 8 * waves * ranges * 2) ranges *= 2;
    } else {
        const int most = tiles >= 64 ? 4 : 8;
        while (waves < most && tiles * waves < 2048 && steps >= 4 * waves) waves *= 2;
    }
    d.mt = mt;
    d.waves = waves;
    d.ranges = static_cast<int>(ranges);
    d.splitSteps = static_cast<int>((steps + ranges - 1) / ranges);
    d.tilesM = static_cast<int>(tilesM);
    d.tilesN = static_cast<int>(tilesN);
    return d;
}

template <typename T, int MT>
int launchDirectAs(const mlkd_gemm* p, const DirectPlan& d, int ranges, hipStream_t st) {
    using Out = typename Direct<T>::Out;
    DirectArgs<T, MT> q;
    q.a = static_cast<const T*>(p->a);
    q.b = static_cast<const T*>(p->b);
    q.c = static_cast<Out*>(p->c);
    q.part = static_cast<Out*>(p->work);
    q.lda = p->lda;
    q.ldb = p->ldb;
    q.ldc = p->ldc;
    q.m = static_cast<int>(p->m);
    q.n = static_cast<int>(p->n);
    q.k = static_cast<int>(p->k);
    q.waves = d.waves;
    q.splitSteps = ranges > 1 ? d.splitSteps : 0x7FFFFFFF;
    q.tilesM = d.tilesM;
    q.accumulate = p->accumulate;
    q.skip = p->skip_zero_a;
    void (*kern)(DirectArgs<T, MT>) = gemmGeneral<Out>;
    const size_t lds = static_cast<size_t>(std::max(d.waves / 2, 1)) * MT * Direct<T>::V * 72 *
                       sizeof(typename Direct<T>::Acc);
    if (lds > 65536) {   // once per process and kernel; a function-local static initializes thread-safely
        static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       160 * 1024) == hipSuccess;
        if (!raised) return MLKD_RT_LAUNCH;
    }
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(d.tilesM * d.tilesN), static_cast<unsigned>(ranges)),
                       dim3(static_cast<unsigned>(64 * d.waves)), lds, st, q);
    if (ranges > 1) {
        DirectArgs<T, 1> s;
        s.a = q.a;
        s.b = q.b;
        s.c = q.c;
        s.part = q.part;
        s.lda = q.lda;
        s.ldb = q.ldb;
        s.ldc = q.ldc;
        s.m = q.m;
        s.n = q.n;
        s.k = q.k;
        s.accumulate = q.accumulate;
        s.skip = q.skip;
        hipLaunchKernelGGL(gemmSumParts<T>, dim3(static_cast<unsigned>((p->n + 255) / 256),
                                                 static_cast<unsigned>(std::min<int64_t>(p->m, 16384))),
                           dim3(256), 0, st, s, ranges);
    }
    return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
}

template <typename T>
int launchDirect(const mlkd_gemm* p, const DirectPlan& d, int ranges, hipStream_t st) {
    if (d.mt == 1) return launchDirectAs<T, 1>(p, d, ranges, st);
    return d.mt == 2 ? launchDirectAs<T, 2>(p, d, ranges, st) : launchDirectAs<T, 4>(p, d, ranges, st);
}

int64_t partBytes(const mlkd_gemm* p, const DirectPlan& d) {
    if (d.mt == 0 || d.ranges == 1) return 0;
    return static_cast<int64_t>(d.ranges) * p->m * p->n * (p->c_dtype == MLKD_F64 ? 8 : 4);
}

}  // namespace

void mlkdGemmGeneralTile(const mlkd_gemm* p, int64_t* rows, int64_t* cols) {
    const DirectPlan d = directPlan(p);
    *rows = d.mt == 0 ? 64 : 16 * d.mt;
    *cols = d.mt == 0 ? 64 : 16 * (p->a_dtype == MLKD_F16 ? 8 : (p->a_dtype == MLKD_F32 ? 4 : 2));
}

const char* mlkdGemmGeneralName(const mlkd_gemm* p) {
    const DirectPlan d = directPlan(p);
    if (d.ranges > 1 && p->work != nullptr && p->work_bytes >= partBytes(p, d)) {
        if (p->a_dtype == MLKD_F16) return "gemmGeneral<float>+gemmSumParts<_Float16>";
        return p->a_dtype == MLKD_F32 ? "gemmGeneral<float>+gemmSumParts<float>"
                                      : "gemmGeneral<double>+gemmSumParts<double>";
    }
    const bool wide = p->a_dtype == MLKD_F64 || p->b_dtype == MLKD_F64 || p->c_dtype == MLKD_F64;
    return wide ? "gemmGeneral<double>" : "gemmGeneral<float>";
}

int64_t mlkdGemmGeneralBytes(const mlkd_gemm* p) { return partBytes(p, directPlan(p)); }

int mlkdLaunchGemmGeneral(const mlkd_gemm* p, hipStream_t st) {
    if (const DirectPlan d = directPlan(p); d.mt > 0) {
        const bool room = p->work != nullptr && p->work_bytes >= partBytes(p, d);
        const int ranges = room ? d.ranges : 1;
        if (p->a_dtype == MLKD_F16) return launchDirect<_Float16>(p, d, ranges, st);
        return p->a_dtype == MLKD_F32 ? launchDirect<float>(p, d, ranges, st) : launchDirect<double>(p, d, ranges, st);
    }
    const int64_t tiles = ((p->m + 63) / 64) * ((p->n + 63) / 64);
    if (tiles > 0x7FFFFFFF) return MLKD_RT_LAUNCH;
    const bool wide = p->a_dtype == MLKD_F64 || p->b_dtype == MLKD_F64 || p->c_dtype == MLKD_F64;
    void (*kern)(mlkd_gemm) = gemmGeneral<float>;
    if (wide) kern = gemmGeneral<double>;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(tiles)), dim3(256), 0, st, *p);
    return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
}
