// Dense C[M,N] (+)= A[M,K] * B[K,N], row-major: Call(MatMul)
// (runtime/src/execution/kernel_buffers.cpp:406-432, C accumulated in place)
// and the poly.synth init+accumulate nest (compiler/src/passes/poly/
// poly.synth.cpp:58-147, C = 0 then +=).
//
// f16 x f16 -> f32 (tensor_f16_gpu), 256x256 workgroup tiles, launch forms 0-8.
// The default, form 8 (gemmF16Dma8s, or gemmF16Dma8 when a lane offset
// needs more than 32 bits), moves both operands global -> LDS by
// the direct path into a 4-deep ring of K steps and runs 8 waves of
// v_mfma_f32_16x16x32_f16 tiles; form 7 (gemmF16Dma) is the same data path
// with 4 waves of 32x32x16 tiles. Form 0, the first: v_mfma_f32_32x32x16_f16,
// K step 64, 512 threads = 8 waves as 2 (M) x 4 (N); each wave owns
// 128x64 = 4x2 MFMA tiles (128 accumulator VGPRs). A and B tiles are double
// buffered in LDS (2 x 72 KiB): the next K step's global loads are issued
// before the current step's MFMAs and written to the other buffer after
// them, one barrier per step. A is stored as loaded ([m][k], k contiguous);
// B is transposed in registers on its way to LDS ([n][k]) so that both MFMA
// operands are single 16-byte LDS reads (8 consecutive k per lane). Rows of
// both LDS tiles are padded by 16 bytes. Workgroups are mapped XCD-aware:
// consecutive workgroup ids go to different XCDs, so the 32 tiles one XCD
// runs form a 4x8 block that shares A and B panels in that XCD's L2.
//
// f32 x f32 -> f32: v_mfma_f32_32x32x2_f32, 64x64 tiles (256 tiles at 1024^2
// fill the 256 CUs). Form 0 (K a multiple of 64, the default) moves both
// tiles by the direct path into a 4-deep LDS ring; form 1 (K a multiple of
// 32) stages them through registers, A transposed into LDS ([k][m]) and B
// stored as loaded ([k][n]) so each MFMA operand is one conflict-free 4-byte
// read.
//
// Any other shape or dtype mix runs the general kernels (gemm_general.hip).
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "gemm_general.h"
#include "mlk_device_math.h"
#include "runtime_abi.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- f16 ----
constexpr int kBM = 256, kBN = 256, kBK = 64;
constexpr int kPadK = kBK + 8;           // halves per LDS row (16-byte pad)
constexpr int kTileHalves = 256 * kPadK;  // one LDS tile (A or B)

/// Skip-zero-A Call form (kernel_buffers.cpp:406-432 skips A[i,p] == 0):
/// the skip changes a result beyond the sign of a zero sum only where B
/// holds an infinity or a NaN, since 0 * inf and 0 * NaN are NaN, and then
/// every accumulator of that column is non-finite (inf * a or 0 * inf; finite
/// f16 products cannot overflow f32). So after the MFMA loop a wave checks
/// its own accumulators for an infinity or a NaN. A wave that finds one
/// recomputes its block exactly (exactWaveBlock); the
/// others store the MFMA result. f32 operands can also overflow to inf from
/// finite values; those blocks take the exact path too, which computes the
/// same overflow.
template <typename V, int I, int J>
__device__ __forceinline__ bool waveNonFinite(const V (&acc)[I][J]) {
    constexpr int E = sizeof(V) / sizeof(float);
    // A class test per value into a lane mask: no vector registers beyond
    // the accumulators, which the 4-wave forms hold in all 512.
    bool bad = false;
#pragma unroll
    for (int i = 0; i < I; ++i) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
#pragma unroll
            for (int e = 0; e < E; ++e) bad |= !__builtin_isfinite(acc[i][j][e]);
        }
    }
    return __builtin_amdgcn_ballot_w64(bad) != 0;
}

template <typename V>
__device__ __forceinline__ bool waveNonFinite(const V& acc) {
    const V one[1][1] = {{acc}};
    return waveNonFinite(one);
}

/// The exact Call(MatMul) form over one wave's rows x cols block: C_in (when
/// accumulating) plus A[i,p] * B[p,j] over p ascending, skipping A[i,p] ==
/// 0, in f32 with separate multiply and add, as the general kernel computes
/// it. Lane l takes column c0 + cb + l; rows go 4 at a time. Only a block
/// whose MFMA accumulators met a non-finite value runs it.
template <typename TA, typename TB>
__device__ __forceinline__ void exactWaveBlock(const TA* __restrict__ A, const TB* __restrict__ B,
                                               float* __restrict__ C, int64_t lda, int64_t ldb, int64_t ldc,
                                               int K, int64_t r0, int64_t c0, int rows, int cols, bool acc) {
    const int lane = threadIdx.x & 63;
    for (int cb = 0; cb < cols; cb += 64) {
        const bool on = cb + lane < cols;
        const int64_t c = c0 + cb + lane;
        for (int rb = 0; rb < rows; rb += 4) {
            float s[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] = (acc && on) ? C[(r0 + rb + r) * ldc + c] : 0.0f;
            for (int k = 0; k < K; ++k) {
                const float b = on ? static_cast<float>(B[k * ldb + c]) : 0.0f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float a = static_cast<float>(A[(r0 + rb + r) * lda + k]);
                    if (a != 0.0f) s[r] = s[r] + a * b;
                }
            }
            if (on) {
#pragma unroll
                for (int r = 0; r < 4; ++r) C[(r0 + rb + r) * ldc + c] = s[r];
            }
        }
    }
}

__device__ __forceinline__ void xcdTile(int tilesM, int tilesN, int& tm, int& tn) {
    const int id = blockIdx.x;
    const int total = tilesM * tilesN;
    // Group tiles 4 (M) x 8 (N) per XCD when the grid is a multiple of that.
    if (tilesM % 4 == 0 && tilesN % 8 == 0 && total % 256 == 0) {
        const int xcd = id % 8;
        const int local = id / 8;            // 0 .. total/8-1
        const int groupsN = tilesN / 8;
        const int roundTiles = 256;          // 8 XCDs x 32 tiles per round
        const int round = (id / roundTiles);
        const int localInRound = local % 32;
        const int groupId = round * 8 + xcd;
        const int gm = groupId / groupsN;
        const int gn = groupId % groupsN;
        tm = gm * 4 + localInRound / 8;
        tn = gn * 8 + localInRound % 8;
        return;
    }
    tm = id / tilesN;
    tn = id % tilesN;
}

template <bool ACC>
__global__ __launch_bounds__(512) void gemmF16Mfma(const _Float16* __restrict__ A,
                                                   const _Float16* __restrict__ B,
                                                   float* __restrict__ C, int M, int N, int K,
                                                   int64_t lda, int64_t ldb, int64_t ldc,
                                                   int /*accumulate: template ACC*/, int skipZeroA) {
    extern __shared__ __align__(16) _Float16 lds[];
    _Float16* As = lds;                      // [2][256][kPadK]
    _Float16* Bs = lds + 2 * kTileHalves;    // [2][256][kPadK]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave >> 2;   // 0..1
    const int wn = wave & 3;    // 0..3
    int tm, tn;
    xcdTile(M / kBM, N / kBN, tm, tn);
    const int64_t row0 = static_cast<int64_t>(tm) * kBM;
    const int64_t col0 = static_cast<int64_t>(tn) * kBN;

    // Loader roles: threads 0..255 load A (8 x 16 B each), 256..511 load a
    // 8 (k) x 8 (n) block of B each.
    const bool loadsA = tid < 256;
    const int t = tid & 255;
    // k-block fastest across lanes: the 8 lanes that share an n-block
    // write one LDS row's 8 chunks, so transposed writes are conflict-free.
    const int bk = t & 7;      // B block: k rows bk*8 .. +7
    const int bn = t >> 3;     // B block: n cols bn*8 .. +7
    u32x4 reg[8];

    auto globalLoad = [&](int k0) {
        if (loadsA) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int c = j * 256 + t;      // 16-byte chunk of the 256x64 tile
                const int r = c >> 3;
                const int ch = c & 7;
                reg[j] = *reinterpret_cast<const u32x4*>(A + (row0 + r) * lda + k0 + ch * 8);
            }
        } else {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                reg[r] = *reinterpret_cast<const u32x4*>(B + static_cast<int64_t>(k0 + bk * 8 + r) * ldb +
                                                        col0 + bn * 8);
            }
        }
    };
    auto ldsStore = [&](int buf) {
        if (loadsA) {
            _Float16* dst = As + buf * kTileHalves;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int c = j * 256 + t;
                const int r = c >> 3;
                const int ch = c & 7;
                *reinterpret_cast<u32x4*>(dst + r * kPadK + ch * 8) = reg[j];
            }
        } else {
            _Float16* dst = Bs + buf * kTileHalves;
            // 8x8 transpose of 16-bit values: column n of the block becomes
            // 8 consecutive k values.
#pragma unroll
            for (int n = 0; n < 8; ++n) {
                const int p = n >> 1;
                const uint32_t sel = (n & 1) ? 0x07060302u : 0x05040100u;
                u32x4 o;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    o[j] = __builtin_amdgcn_perm(reg[2 * j + 1][p], reg[2 * j][p], sel);
                }
                *reinterpret_cast<u32x4*>(dst + (bn * 8 + n) * kPadK + bk * 8) = o;
            }
        }
    };

    f32x16 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
        }
    }

    const int steps = K / kBK;
    globalLoad(0);
    ldsStore(0);
    __syncthreads();
    const int lrow = lane & 31;
    const int lk = (lane >> 5) * 8;
    for (int s = 0; s < steps; ++s) {
        const int buf = s & 1;
        if (s + 1 < steps) globalLoad((s + 1) * kBK);
        const _Float16* as = As + buf * kTileHalves + (wm * 128 + lrow) * kPadK + lk;
        const _Float16* bs = Bs + buf * kTileHalves + (wn * 64 + lrow) * kPadK + lk;
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 16) {
            f16x8 a[4], b[2];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const f16x8*>(as + i * 32 * kPadK + kk);
#pragma unroll
            for (int j = 0; j < 2; ++j) b[j] = *reinterpret_cast<const f16x8*>(bs + j * 32 * kPadK + kk);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], acc[i][j], 0, 0, 0);
                }
            }
        }
        if (s + 1 < steps) {
            ldsStore(buf ^ 1);
        }
        __syncthreads();
    }

    if (ACC && skipZeroA && waveNonFinite(acc)) {
        exactWaveBlock<_Float16, _Float16>(A, B, C, lda, ldb, ldc, K, row0 + wm * 128, col0 + wn * 64, 128, 64, ACC);
        return;
    }
    // D layout of a 32x32 MFMA tile: lane l, register r holds
    // row 8*(r/4) + 4*(l/32) + r%4, column l%32.
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int64_t cBase = col0 + wn * 64 + j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t row = row0 + wm * 128 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                float* dst = C + row * ldc + cBase;
                const float v = acc[i][j][r];
                *dst = ACC ? *dst + v : v;
            }
        }
    }
}

/// Two-per-CU variant: a 128 x 256 workgroup tile of 4 waves (each 64 x 128 =
/// 2 x 4 MFMA tiles), K step 32, LDS tiles double buffered in 60 KiB, so
/// two workgroups share a CU and one's load waits overlap the other's MFMAs.
/// Global loads run two steps ahead in two register sets (the K loop is
/// unrolled by two so the sets are static; AHEAD2 = false loads one step
/// ahead in one set). A is staged as loaded ([m][k]);
/// B arrives as 4 (k) x 8 (n) blocks and is transposed in registers to
/// [n][k]; LDS rows are 40 halves (80 bytes), which keeps the 16-byte
/// operand reads conflict-free.
constexpr int kBM2 = 128, kBN2 = 256, kBK2 = 32, kPad2 = kBK2 + 8;
constexpr int kTileA2 = kBM2 * kPad2, kTileB2 = kBN2 * kPad2;
constexpr size_t kLdsGemm2 = 2 * (kTileA2 + kTileB2) * sizeof(_Float16);

__device__ __forceinline__ void xcdTile2(int tilesM, int tilesN, int& tm, int& tn) {
    // Consecutive ids go to different XCDs: give each XCD a contiguous block
    // of tile ids, row-major over (tm, tn) within the block.
    const int total = tilesM * tilesN;
    int id = blockIdx.x;
    if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
    tm = id / tilesN;
    tn = id % tilesN;
}

template <bool ACC, bool AHEAD2>
__global__ __launch_bounds__(256, 2) void gemmF16Mfma2cu(const _Float16* __restrict__ A,
                                                         const _Float16* __restrict__ B,
                                                         float* __restrict__ C, int M, int N, int K,
                                                         int64_t lda, int64_t ldb, int64_t ldc, int skipZeroA) {
    extern __shared__ __align__(16) _Float16 lds[];
    _Float16* As = lds;                     // [2][128][40]
    _Float16* Bs = lds + 2 * kTileA2;       // [2][256][40]
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6, l32 = lane & 31, hl = lane >> 5;
    const int wm = wave >> 1, wn = wave & 1;
    int tm, tn;
    xcdTile2(M / kBM2, N / kBN2, tm, tn);
    const int64_t row0 = static_cast<int64_t>(tm) * kBM2;
    const int64_t col0 = static_cast<int64_t>(tn) * kBN2;
    const int bk = t & 7;    // B block: k rows bk*4 .. +3
    const int bn = t >> 3;   // B block: n cols bn*8 .. +7
    u32x4 ra0[2], rb0[4], ra1[2], rb1[4];
    auto load = [&](int k0, u32x4(&ra)[2], u32x4(&rb)[4]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int c = j * 256 + t;   // 512 chunks: 128 rows x 4
            ra[j] = *reinterpret_cast<const u32x4*>(A + (row0 + (c >> 2)) * lda + k0 + (c & 3) * 8);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            rb[r] = *reinterpret_cast<const u32x4*>(B + static_cast<int64_t>(k0 + bk * 4 + r) * ldb + col0 + bn * 8);
        }
    };
    auto store = [&](int buf, const u32x4(&ra)[2], const u32x4(&rb)[4]) {
        _Float16* da = As + buf * kTileA2;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int c = j * 256 + t;
            *reinterpret_cast<u32x4*>(da + (c >> 2) * kPad2 + (c & 3) * 8) = ra[j];
        }
        _Float16* db = Bs + buf * kTileB2;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const int pp = n >> 1;
            const uint32_t sel = (n & 1) ? 0x07060302u : 0x05040100u;
            uint32_t o0 = __builtin_amdgcn_perm(rb[1][pp], rb[0][pp], sel);
            uint32_t o1 = __builtin_amdgcn_perm(rb[3][pp], rb[2][pp], sel);
            typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
            u32x2 o;
            o[0] = o0;
            o[1] = o1;
            *reinterpret_cast<u32x2*>(db + (bn * 8 + n) * kPad2 + bk * 4) = o;
        }
    };
    f32x16 acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
        }
    }
    auto mfmaStep = [&](int buf) {
        const _Float16* as = As + buf * kTileA2 + (wm * 64 + l32) * kPad2 + hl * 8;
        const _Float16* bs = Bs + buf * kTileB2 + (wn * 128 + l32) * kPad2 + hl * 8;
#pragma unroll
        for (int kk = 0; kk < kBK2; kk += 16) {
            f16x8 a[2], b[4];
#pragma unroll
            for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const f16x8*>(as + i * 32 * kPad2 + kk);
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const f16x8*>(bs + j * 32 * kPad2 + kk);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], acc[i][j], 0, 0, 0);
                }
            }
        }
    };
    // K / kBK2 is even (the launcher requires K % 64 == 0).
    const int steps = K / kBK2;
    load(0, ra0, rb0);
    store(0, ra0, rb0);
    if (AHEAD2) {
        load(kBK2, ra1, rb1);
        __syncthreads();
        for (int s = 0; s < steps; s += 2) {
            if (s + 2 < steps) load((s + 2) * kBK2, ra0, rb0);
            mfmaStep(0);
            store(1, ra1, rb1);
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
            if (s + 3 < steps) load((s + 3) * kBK2, ra1, rb1);
            mfmaStep(1);
            if (s + 2 < steps) store(0, ra0, rb0);
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        __syncthreads();
        for (int s = 0; s < steps; ++s) {
            if (s + 1 < steps) load((s + 1) * kBK2, ra0, rb0);
            mfmaStep(s & 1);
            if (s + 1 < steps) store((s + 1) & 1, ra0, rb0);
            __syncthreads();
        }
    }
    if (ACC && skipZeroA && waveNonFinite(acc)) {
        exactWaveBlock<_Float16, _Float16>(A, B, C, lda, ldb, ldc, K, row0 + wm * 64, col0 + wn * 128, 64, 128, ACC);
        return;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t cBase = col0 + wn * 128 + j * 32 + l32;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t row = row0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * hl + (r & 3);
                float* dst = C + row * ldc + cBase;
                const float v = acc[i][j][r];
                *dst = ACC ? *dst + v : v;
            }
        }
    }
}

/// 4-wave variant: the same 256x256x64 workgroup tile with each wave owning a
/// 128x128 quadrant (4x4 MFMA tiles, 256 accumulators in AGPRs), so every
/// kk step issues 8 LDS operand reads for 16 MFMAs. Thread t loads 8 A chunks
/// and one 8x8 B block per K step.
template <bool ACC>
__global__ __launch_bounds__(256) void gemmF16Mfma4w(const _Float16* __restrict__ A,
                                                     const _Float16* __restrict__ B,
                                                     float* __restrict__ C, int M, int N, int K,
                                                     int64_t lda, int64_t ldb, int64_t ldc,
                                                     int /*accumulate: template ACC*/, int skipZeroA) {
    extern __shared__ __align__(16) _Float16 lds[];
    _Float16* As = lds;
    _Float16* Bs = lds + 2 * kTileHalves;
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = t >> 6;
    const int wm = wave >> 1;   // 0..1
    const int wn = wave & 1;    // 0..1
    int tm, tn;
    xcdTile(M / kBM, N / kBN, tm, tn);
    const int64_t row0 = static_cast<int64_t>(tm) * kBM;
    const int64_t col0 = static_cast<int64_t>(tn) * kBN;
    const int bk = t & 7;
    const int bn = t >> 3;
    u32x4 ra[8], rb[8];
    auto globalLoad = [&](int k0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int c = j * 256 + t;
            ra[j] = *reinterpret_cast<const u32x4*>(A + (row0 + (c >> 3)) * lda + k0 + (c & 7) * 8);
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            rb[r] = *reinterpret_cast<const u32x4*>(B + static_cast<int64_t>(k0 + bk * 8 + r) * ldb + col0 + bn * 8);
        }
    };
    auto ldsStore = [&](int buf) {
        _Float16* da = As + buf * kTileHalves;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int c = j * 256 + t;
            *reinterpret_cast<u32x4*>(da + (c >> 3) * kPadK + (c & 7) * 8) = ra[j];
        }
        _Float16* db = Bs + buf * kTileHalves;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const int p = n >> 1;
            const uint32_t sel = (n & 1) ? 0x07060302u : 0x05040100u;
            u32x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = __builtin_amdgcn_perm(rb[2 * j + 1][p], rb[2 * j][p], sel);
            *reinterpret_cast<u32x4*>(db + (bn * 8 + n) * kPadK + bk * 8) = o;
        }
    };
    f32x16 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
        }
    }
    const int steps = K / kBK;
    globalLoad(0);
    ldsStore(0);
    __syncthreads();
    const int lrow = lane & 31;
    const int lk = (lane >> 5) * 8;
    for (int s = 0; s < steps; ++s) {
        const int buf = s & 1;
        if (s + 1 < steps) globalLoad((s + 1) * kBK);
        const _Float16* as = As + buf * kTileHalves + (wm * 128 + lrow) * kPadK + lk;
        const _Float16* bs = Bs + buf * kTileHalves + (wn * 128 + lrow) * kPadK + lk;
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 16) {
            f16x8 a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const f16x8*>(as + i * 32 * kPadK + kk);
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const f16x8*>(bs + j * 32 * kPadK + kk);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], acc[i][j], 0, 0, 0);
                }
            }
        }
        if (s + 1 < steps) ldsStore(buf ^ 1);
        __syncthreads();
    }
    if (ACC && skipZeroA && waveNonFinite(acc)) {
        exactWaveBlock<_Float16, _Float16>(A, B, C, lda, ldb, ldc, K, row0 + wm * 128, col0 + wn * 128, 128, 128, ACC);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t cBase = col0 + wn * 128 + j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t row = row0 + wm * 128 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                float* dst = C + row * ldc + cBase;
                const float v = acc[i][j][r];
                *dst = ACC ? *dst + v : v;
            }
        }
    }
}

/// 4-wave variant with A moved by the gfx950 direct global->LDS path
/// (global_load_lds_dwordx4): A never occupies VGPRs, which leaves room for
/// the 256 accumulators plus B's register staging without spills. A's LDS
/// tile is unpadded [256][64] with 16-byte chunks XOR-swizzled by
/// (row >> 1) & 7, so the 16 rows one quarter-wave reads hit 16 distinct
/// chunk slots. Each direct-load instruction writes 64 consecutive 16-byte
/// slots (lane i -> slot i); the lane chooses the global chunk that belongs
/// in that slot.
constexpr int kTileA = 256 * kBK;  // halves, unpadded

__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }

template <bool ACC>
__global__ __launch_bounds__(256) void gemmF16Mfma4wDirect(const _Float16* __restrict__ A,
                                                           const _Float16* __restrict__ B,
                                                           float* __restrict__ C, int M, int N, int K,
                                                           int64_t lda, int64_t ldb, int64_t ldc,
                                                           int /*accumulate: template ACC*/, int skipZeroA) {
    extern __shared__ __align__(16) _Float16 lds[];
    _Float16* As = lds;                    // [2][256][64] swizzled
    _Float16* Bs = lds + 2 * kTileA;       // [2][256][kPadK]
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = t >> 6;
    const int wm = wave >> 1;
    const int wn = wave & 1;
    int tm, tn;
    xcdTile(M / kBM, N / kBN, tm, tn);
    const int64_t row0 = static_cast<int64_t>(tm) * kBM;
    const int64_t col0 = static_cast<int64_t>(tn) * kBN;
    const int bk = t & 7;
    const int bn = t >> 3;
    u32x4 rb[8];
    auto directA = [&](int k0, int buf) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int slot0 = (wave * 8 + j) * 64;          // first slot of this instruction
            const int q = slot0 + lane;
            const int row = q >> 3;
            const int c = (q & 7) ^ swz(row);               // logical chunk stored in slot q
            const _Float16* src = A + (row0 + row) * lda + k0 + c * 8;
            _Float16* dst = As + buf * kTileA + slot0 * 8;  // wave-uniform
            __builtin_amdgcn_global_load_lds(src, reinterpret_cast<__attribute__((address_space(3))) void*>(
                                                       reinterpret_cast<uintptr_t>(dst)),
                                             16, 0, 0);
        }
    };
    auto loadB = [&](int k0) {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            rb[r] = *reinterpret_cast<const u32x4*>(B + static_cast<int64_t>(k0 + bk * 8 + r) * ldb + col0 + bn * 8);
        }
    };
    auto storeB = [&](int buf) {
        _Float16* db = Bs + buf * kTileHalves;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const int p = n >> 1;
            const uint32_t sel = (n & 1) ? 0x07060302u : 0x05040100u;
            u32x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = __builtin_amdgcn_perm(rb[2 * j + 1][p], rb[2 * j][p], sel);
            *reinterpret_cast<u32x4*>(db + (bn * 8 + n) * kPadK + bk * 8) = o;
        }
    };
    f32x16 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
        }
    }
    const int steps = K / kBK;
    directA(0, 0);
    loadB(0);
    storeB(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const int lrow = lane & 31;
    const int lhalf = lane >> 5;
    for (int s = 0; s < steps; ++s) {
        const int buf = s & 1;
        if (s + 1 < steps) {
            directA((s + 1) * kBK, buf ^ 1);
            loadB((s + 1) * kBK);
        }
        const _Float16* as = As + buf * kTileA;
        const _Float16* bs = Bs + buf * kTileHalves + (wn * 128 + lrow) * kPadK + lhalf * 8;
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 16) {
            f16x8 a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = wm * 128 + i * 32 + lrow;
                const int c = (kk >> 3) + lhalf;
                a[i] = *reinterpret_cast<const f16x8*>(as + row * kBK + ((c ^ swz(row)) * 8));
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const f16x8*>(bs + j * 32 * kPadK + kk);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], acc[i][j], 0, 0, 0);
                }
            }
        }
        if (s + 1 < steps) storeB(buf ^ 1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    if (ACC && skipZeroA && waveNonFinite(acc)) {
        exactWaveBlock<_Float16, _Float16>(A, B, C, lda, ldb, ldc, K, row0 + wm * 128, col0 + wn * 128, 128, 128, ACC);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t cBase = col0 + wn * 128 + j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t row = row0 + wm * 128 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                float* dst = C + row * ldc + cBase;
                const float v = acc[i][j][r];
                *dst = ACC ? *dst + v : v;
            }
        }
    }
}

/// Variant 3: variant 2's data movement with an explicit software pipeline
/// inside the K step. Operand fragments are double buffered in registers:
/// the 8 LDS reads for kk+1 are issued while the 16 MFMAs of kk run, and
/// sched_group_barrier pins the interleave (1 DS read per 2 MFMAs; the next
/// step's global loads spread over the first kk; the B transpose and its LDS
/// writes over the last kk), so the MFMA pipe never waits on LDS latency
/// except once after each barrier.
template <bool ACC>
__global__ __launch_bounds__(256) void gemmF16Mfma4wPipe(const _Float16* __restrict__ A,
                                                         const _Float16* __restrict__ B,
                                                         float* __restrict__ C, int M, int N, int K,
                                                         int64_t lda, int64_t ldb, int64_t ldc, int skipZeroA) {
    extern __shared__ __align__(16) _Float16 lds[];
    _Float16* As = lds;
    _Float16* Bs = lds + 2 * kTileA;
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = t >> 6;
    const int wm = wave >> 1;
    const int wn = wave & 1;
    int tm, tn;
    xcdTile(M / kBM, N / kBN, tm, tn);
    const int64_t row0 = static_cast<int64_t>(tm) * kBM;
    const int64_t col0 = static_cast<int64_t>(tn) * kBN;
    const int bk = t & 7;
    const int bn = t >> 3;
    const int lrow = lane & 31;
    const int lhalf = lane >> 5;
    u32x4 rb[8];
    auto directA = [&](int k0, int buf) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int slot0 = (wave * 8 + j) * 64;
            const int q = slot0 + lane;
            const int row = q >> 3;
            const int c = (q & 7) ^ swz(row);
            const _Float16* src = A + (row0 + row) * lda + k0 + c * 8;
            _Float16* dst = As + buf * kTileA + slot0 * 8;
            __builtin_amdgcn_global_load_lds(src, reinterpret_cast<__attribute__((address_space(3))) void*>(
                                                       reinterpret_cast<uintptr_t>(dst)),
                                             16, 0, 0);
        }
    };
    auto loadB = [&](int k0) {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            rb[r] = *reinterpret_cast<const u32x4*>(B + static_cast<int64_t>(k0 + bk * 8 + r) * ldb + col0 + bn * 8);
        }
    };
    auto storeB = [&](int buf) {
        _Float16* db = Bs + buf * kTileHalves;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const int p = n >> 1;
            const uint32_t sel = (n & 1) ? 0x07060302u : 0x05040100u;
            u32x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = __builtin_amdgcn_perm(rb[2 * j + 1][p], rb[2 * j][p], sel);
            *reinterpret_cast<u32x4*>(db + (bn * 8 + n) * kPadK + bk * 8) = o;
        }
    };
    f16x8 fa[2][4], fb[2][4];
    auto readFrags = [&](int buf, int kk, int slot) {
        const _Float16* as = As + buf * kTileA;
        const _Float16* bs = Bs + buf * kTileHalves + (wn * 128 + lrow) * kPadK + lhalf * 8 + kk;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = wm * 128 + i * 32 + lrow;
            const int c = (kk >> 3) + lhalf;
            fa[slot][i] = *reinterpret_cast<const f16x8*>(as + row * kBK + ((c ^ swz(row)) * 8));
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) fb[slot][j] = *reinterpret_cast<const f16x8*>(bs + j * 32 * kPadK);
    };
    f32x16 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
        }
    }
    auto mfmas = [&](int slot) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[slot][i], fb[slot][j], acc[i][j], 0, 0, 0);
            }
        }
    };
    const int steps = K / kBK;
    directA(0, 0);
    loadB(0);
    storeB(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (int s = 0; s < steps; ++s) {
        const int buf = s & 1;
        // Branch-free step body (one scheduling region): the last step
        // re-loads its own, in-bounds K slice into the idle buffer.
        const int kNext = (s + 1 < steps ? s + 1 : s) * kBK;
        readFrags(buf, 0, 0);
        directA(kNext, buf ^ 1);
        loadB(kNext);
        // kk = 0: next fragments + the next step's global loads.
        readFrags(buf, 16, 1);
        mfmas(0);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // 1 DS read
            __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);   // 2 VMEM reads
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);   // 2 MFMA
        }
        readFrags(buf, 32, 0);
        mfmas(1);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        }
        readFrags(buf, 48, 1);
        mfmas(0);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        }
        mfmas(1);
        storeB(buf ^ 1);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);   // 4 VALU (transpose)
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);   // 1 DS write
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);   // 2 MFMA
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    if (ACC && skipZeroA && waveNonFinite(acc)) {
        exactWaveBlock<_Float16, _Float16>(A, B, C, lda, ldb, ldc, K, row0 + wm * 128, col0 + wn * 128, 128, 128, ACC);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t cBase = col0 + wn * 128 + j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t row = row0 + wm * 128 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                float* dst = C + row * ldc + cBase;
                const float v = acc[i][j][r];
                *dst = ACC ? *dst + v : v;
            }
        }
    }
}

/// Variant 7: both operands moved global -> LDS by the gfx950 direct path
/// (global_load_lds_dwordx4, no VGPR staging) into a 4-deep ring of K steps
/// of 32; B is kept as loaded ([k][n]) and read with ds_read_b64_tr_b16,
/// which hands each lane 4 consecutive k of one column, i.e. the MFMA B
/// operand without a register transpose. 4 waves (2 x 2), each owning a
/// 128 x 128 quadrant (4 x 4 MFMA tiles, 256 accumulators). The fragments of
/// the next 16-deep sub-step are read while the current one's 16 MFMAs run
/// (one LDS read per MFMA). One barrier per K step certifies the next stage;
/// every step issues exactly one stage (past the end a harmless reload into
/// a slot nothing reads), so the wait before the barrier is a constant
/// vmcnt. The direct loads are inline asm: the kernel accounts for them
/// itself, so the compiler adds no conservative waits on them.
/// LDS swizzles: A rows are 64 bytes (4 chunks), chunk c of row r sits at
/// c ^ ((r >> 2) & 3); B rows are 512 bytes, chunk c of k-row r sits at
/// c ^ ((r & 3) * 4). Both measured conflict-free (SQ_LDS_BANK_CONFLICT 0).
constexpr int kDmaBK = 32, kDmaStages = 4;
constexpr int kDmaA = 256 * kDmaBK;                   // halves per A stage
constexpr int kDmaStage = 2 * kDmaA;                  // A then B
constexpr size_t kLdsDma = static_cast<size_t>(kDmaStages) * kDmaStage * sizeof(_Float16);   // 128 KiB

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __fp16 fp16x4 __attribute__((__vector_size__(4 * sizeof(__fp16))));

__device__ __forceinline__ uint32_t ldsOffset(const void* p) {
    // Generic pointers into LDS carry the LDS offset in their low 32 bits.
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p));
}

/// 16 bytes per lane from `src` to LDS `dst` + 16 * lane; `dst` is the same
/// for the whole wave and goes through M0. M0 is a reserved register: naming
/// it as a clobber only draws a warning that reserved registers are not
/// preserved, so it is left out. The asm sets M0 itself right before the
/// load, and in the kernels that use these loads every M0 write comes from
/// these asm statements (the compiled code holds no other value in M0).
__device__ __forceinline__ void dmaLoad16(const _Float16* src, const _Float16* dst) {
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(ldsOffset(dst));
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(m0) : "memory");
}

struct DmaFrag {
    f16x8 a[4];
    f16x4 b[4][2];
};

template <bool ACC>
__global__ __launch_bounds__(256, 1) void gemmF16Dma(const _Float16* __restrict__ A,
                                                     const _Float16* __restrict__ B,
                                                     float* __restrict__ C, int M, int N, int K,
                                                     int64_t lda, int64_t ldb, int64_t ldc, int skipZeroA) {
    extern __shared__ __align__(16) _Float16 lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    int tm, tn;
    xcdTile(M / kBM, N / kBN, tm, tn);
    const int64_t row0 = static_cast<int64_t>(tm) * kBM;
    const int64_t col0 = static_cast<int64_t>(tn) * kBN;
    const int steps = K / kDmaBK;

    // Stage `slot` receives K step min(slot, steps - 1) in ring slot
    // slot % kDmaStages. Wave w issues A instructions 4w..4w+3 (16 rows
    // each) and B instructions 4w..4w+3 (2 k-rows each).
    auto issue = [&](int slot) {
        const int k0 = min(slot, steps - 1) * kDmaBK;
        const _Float16* st = lds + (slot % kDmaStages) * kDmaStage;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int ins = wave * 4 + j;
            const int q = ins * 64 + lane;
            const int row = q >> 2;
            const int c = (q & 3) ^ ((row >> 2) & 3);
            dmaLoad16(A + (row0 + row) * lda + k0 + c * 8, st + ins * 512);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int ins = wave * 4 + j;
            const int q = ins * 64 + lane;
            const int krow = q >> 5;
            const int c = (q & 31) ^ ((krow & 3) * 4);
            dmaLoad16(B + static_cast<int64_t>(k0 + krow) * ldb + col0 + c * 8, st + kDmaA + ins * 512);
        }
    };

    f32x16 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
        }
    }
#pragma unroll
    for (int s = 0; s < kDmaStages - 1; ++s) issue(s);

    const int l32 = lane & 31, hl = lane >> 5;
    const int g = lane >> 4, sl = lane & 15;
    // Lane byte offsets inside a stage. A: per sub-step kk (tile i adds 32
    // rows = 2048 bytes). B: per (kk, j, h) for the two 4-deep halves of the
    // transposed read (lanes of group g read k-rows 8 * (g >> 1) + sl / 4).
    uint32_t offA[2], offB[2][4][2];
    {
        const int row = wm * 128 + l32;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) offA[kk] = 2u * (row * kDmaBK + (((kk * 2 + hl) ^ ((row >> 2) & 3)) * 8));
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int krow = kk * 16 + 8 * (g >> 1) + (sl >> 2) + 4 * h;
                    const int col = wn * 128 + j * 32 + 16 * (g & 1) + 4 * (sl & 3);
                    offB[kk][j][h] = 2u * (kDmaA + krow * 256 + (((col >> 3) ^ ((krow & 3) * 4)) * 8) + (col & 7));
                }
            }
        }
    }
    const uint32_t ldsBase = ldsOffset(lds);
    // Read r of a sub-step: r 0..3 the A tiles, r 4..11 the B halves (j, h).
    auto readOne = [&](DmaFrag& f, uint32_t base, int kk, int r) {
        if (r < 4) {
            f.a[r] = *reinterpret_cast<const __attribute__((address_space(3))) f16x8*>(base + offA[kk] + 2048u * r);
        } else {
            const int j = (r - 4) >> 1, h = (r - 4) & 1;
            const fp16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
                reinterpret_cast<__attribute__((address_space(3))) fp16x4*>(base + offB[kk][j][h]));
            f.b[j][h] = __builtin_bit_cast(f16x4, v);
        }
    };
    auto mfma = [&](const DmaFrag& f, int idx) {
        const int i = idx >> 2, j = idx & 3;
        const f16x8 bb = __builtin_shufflevector(f.b[j][0], f.b[j][1], 0, 1, 2, 3, 4, 5, 6, 7);
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[i], bb, acc[i][j], 0, 0, 0);
    };
    // 16 MFMAs of `cur` with the 12 reads of the next sub-step between them.
    auto subStep = [&](DmaFrag& cur, DmaFrag& nxt, uint32_t nbase, int nkk) {
#pragma unroll
        for (int idx = 0; idx < 16; ++idx) {
            mfma(cur, idx);
            if (idx < 12) readOne(nxt, nbase, nkk, idx);
        }
#pragma unroll
        for (int idx = 0; idx < 12; ++idx) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    };

    DmaFrag x, y;
    // Stage 0 landed (stages 1 and 2, 8 direct loads each per wave, may be
    // in flight).
    asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int r = 0; r < 12; ++r) readOne(x, ldsBase, 0, r);
    for (int s = 0; s < steps; ++s) {
        const uint32_t cb = ldsBase + 2u * static_cast<uint32_t>((s % kDmaStages) * kDmaStage);
        subStep(x, y, cb, 1);   // sub-step (s, 0); reads (s, 1)
        // Stage s + 1 landed (one later stage, 8 direct loads per wave, may be
        // in flight); after the barrier every wave is past step s - 1, so its
        // slot can be refilled.
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
        issue(s + kDmaStages - 1);
        const uint32_t nb = ldsBase + 2u * static_cast<uint32_t>(((s + 1) % kDmaStages) * kDmaStage);
        subStep(y, x, nb, 0);   // sub-step (s, 1); reads (s + 1, 0)
    }
    // No direct load may still be writing LDS when the workgroup ends.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (ACC && skipZeroA && waveNonFinite(acc)) {
        exactWaveBlock<_Float16, _Float16>(A, B, C, lda, ldb, ldc, K, row0 + wm * 128, col0 + wn * 128, 128, 128, ACC);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t cBase = col0 + wn * 128 + j * 32 + l32;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t row = row0 + wm * 128 + i * 32 + 8 * (r >> 2) + 4 * hl + (r & 3);
                float* dst = C + row * ldc + cBase;
                const float v = acc[i][j][r];
                *dst = ACC ? *dst + v : v;
            }
        }
    }
}

/// Variant 8: variant 7's data movement (the same 4-deep direct-to-LDS ring
/// of K steps of 32, the same swizzles and transposed B reads) with 8 waves
/// (2 per SIMD, 2 (M) x 4 (N)), each owning 128 x 64, and
/// v_mfma_f32_16x16x32_f16 with the operands swapped: each 16 x 16 tile is
/// D = B^T A^T, so a lane holds 4 consecutive columns of one row of C and
/// stores them with one 16-byte write. The 32 tiles of a wave (8 x 4) keep
/// their 128 accumulators in ordinary registers. Under this chip's power
/// limit the smaller MFMA sustains more work per joule (a register-only loop
/// runs 12% faster with it than with 32x32x16). Each K step is two groups of
/// 16 MFMAs (m-tiles 0-3, then 4-7): the first group's MFMAs overlap the
/// reads of the second group's A fragments; the barrier that certifies the
/// next stage sits between the groups, and the second group overlaps the
/// reads of the next step's first group (B fragments double buffered).
/// Every output element takes its products in the same k order as variant
/// 7, and the results match it bit for bit. Needs K a multiple of 64.
template <bool ACC>
__global__ __launch_bounds__(512, 1) void gemmF16Dma8(const _Float16* __restrict__ A,
                                                      const _Float16* __restrict__ B,
                                                      float* __restrict__ C, int M, int N, int K,
                                                      int64_t lda, int64_t ldb, int64_t ldc, int skipZeroA) {
    extern __shared__ __align__(16) _Float16 lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave >> 2, wn = wave & 3;
    int tm, tn;
    xcdTile(M / kBM, N / kBN, tm, tn);
    const int64_t row0 = static_cast<int64_t>(tm) * kBM;
    const int64_t col0 = static_cast<int64_t>(tn) * kBN;
    const int steps = K / kDmaBK;

    // Stage `slot` receives K step min(slot, steps - 1) in ring slot
    // slot % kDmaStages. Wave w issues A instructions 2w, 2w + 1 (16 rows
    // each) and B instructions 2w, 2w + 1 (2 k-rows each).
    auto issue = [&](int slot) {
        const int k0 = min(slot, steps - 1) * kDmaBK;
        const _Float16* st = lds + (slot % kDmaStages) * kDmaStage;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ins = wave * 2 + j;
            const int q = ins * 64 + lane;
            const int row = q >> 2;
            const int c = (q & 3) ^ ((row >> 2) & 3);
            dmaLoad16(A + (row0 + row) * lda + k0 + c * 8, st + ins * 512);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ins = wave * 2 + j;
            const int q = ins * 64 + lane;
            const int krow = q >> 5;
            const int c = (q & 31) ^ ((krow & 3) * 4);
            dmaLoad16(B + static_cast<int64_t>(k0 + krow) * ldb + col0 + c * 8, st + kDmaA + ins * 512);
        }
    };

    f32x4 acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;
        }
    }
#pragma unroll
    for (int s = 0; s < kDmaStages - 1; ++s) issue(s);

    const int l16 = lane & 15, g = lane >> 4;
    // The MFMA's B operand (A^T): row wm * 128 + 16 mt + l16 of A, chunk g
    // (k 8g .. 8g + 7) at its swizzled slot; tile mt adds 1024 bytes.
    uint32_t offA;
    {
        const int row = wm * 128 + l16;
        offA = 2u * (row * kDmaBK + ((g ^ ((row >> 2) & 3)) * 8));
    }
    // The MFMA's A operand (B^T): column wn * 64 + 16 nt + l16 of B, k 8g ..
    // 8g + 7 by two transposed reads (h = 0, 1); lane (g, l16) points at
    // k-row 8g + 4h + l16 / 4, columns 4 (l16 % 4) .. + 3 of the tile.
    uint32_t offB[4][2];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int krow = 8 * g + 4 * h + (l16 >> 2);
            const int col = wn * 64 + nt * 16 + 4 * (l16 & 3);
            offB[nt][h] = 2u * (kDmaA + krow * 256 + (((col >> 3) ^ ((krow & 3) * 4)) * 8) + (col & 7));
        }
    }
    const uint32_t ldsBase = ldsOffset(lds);
    auto readA = [&](f16x8& f, uint32_t base, int mt) {
        f = *reinterpret_cast<const __attribute__((address_space(3))) f16x8*>(base + offA + 1024u * mt);
    };
    auto readB = [&](f16x8& f, uint32_t base, int nt) {
        const fp16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
            reinterpret_cast<__attribute__((address_space(3))) fp16x4*>(base + offB[nt][0]));
        const fp16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
            reinterpret_cast<__attribute__((address_space(3))) fp16x4*>(base + offB[nt][1]));
        f = __builtin_shufflevector(__builtin_bit_cast(f16x4, v0), __builtin_bit_cast(f16x4, v1), 0, 1, 2, 3, 4, 5,
                                    6, 7);
    };
    f16x8 aLo[4], aHi[4], bX[4], bY[4];
    // 16 MFMAs: m-tiles mt0 .. mt0 + 3 against the 4 n-tiles.
    auto group = [&](const f16x8 (&a)[4], const f16x8 (&b)[4], int mt0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[mt0 + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[j], a[i], acc[mt0 + i][j], 0, 0, 0);
            }
        }
    };
    // Stage 0 landed (stages 1 and 2, 4 direct loads each per wave, may be
    // in flight).
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; ++i) readA(aLo[i], ldsBase, i);
#pragma unroll
    for (int j = 0; j < 4; ++j) readB(bX[j], ldsBase, j);
    auto step = [&](int s, f16x8 (&bCur)[4], f16x8 (&bNxt)[4]) {
        const uint32_t cb = ldsBase + 2u * static_cast<uint32_t>((s % kDmaStages) * kDmaStage);
        group(aLo, bCur, 0);                          // m-tiles 0-3 of step s; reads m-tiles 4-7
#pragma unroll
        for (int i = 0; i < 4; ++i) readA(aHi[i], cb, 4 + i);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
            if (i < 4) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        // Stage s + 1 landed (one later stage may be in flight); after the
        // barrier every wave is past step s - 1, so its slot can be refilled.
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
        issue(s + kDmaStages - 1);
        const uint32_t nb = ldsBase + 2u * static_cast<uint32_t>(((s + 1) % kDmaStages) * kDmaStage);
        group(aHi, bCur, 4);                          // m-tiles 4-7 of step s; reads step s + 1's first group
#pragma unroll
        for (int i = 0; i < 4; ++i) readA(aLo[i], nb, i);
#pragma unroll
        for (int j = 0; j < 4; ++j) readB(bNxt[j], nb, j);
#pragma unroll
        for (int i = 0; i < 12; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    };
    for (int s = 0; s < steps; s += 2) {              // steps is even (K % 64 == 0)
        step(s, bX, bY);
        step(s + 1, bY, bX);
    }
    // No direct load may still be writing LDS when the workgroup ends.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (ACC && skipZeroA && waveNonFinite(acc)) {
        exactWaveBlock<_Float16, _Float16>(A, B, C, lda, ldb, ldc, K, row0 + wm * 128, col0 + wn * 64, 128, 64, ACC);
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t row = row0 + wm * 128 + i * 16 + l16;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32x4* dst = reinterpret_cast<f32x4*>(C + row * ldc + col0 + wn * 64 + j * 16 + 4 * g);
            f32x4 v = acc[i][j];
            if (ACC) v += *dst;
            *dst = v;
        }
    }
}

/// Direct load through a scalar base: lane bytes `voff` past `sbase` into LDS
/// at M0 + 16 * lane. The K advance lives in `sbase` (scalar adds), so the
/// per-lane address costs no vector instruction per step.
/// M0 is handled as in dmaLoad16.
__device__ __forceinline__ void dmaLoad16s(const void* sbase, uint32_t voff, uint32_t m0) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(m0) : "memory");
}

// ---------------------------------------------------------- f16 ragged ----
/// Operands of a ragged member (form 8, f32 form 0): C is m x n; A's rows hold
/// ka columns (k, or k rounded up with zeros), B's nb columns (n, or n rounded
/// up), both whole 16-byte pieces at 16-byte aligned rows.
template <typename T>
struct Ragged {
    const T* a;
    const T* b;
    float* c;
    int m, n, k, ka, nb;
    int tilesM, tilesN;
    int64_t lda, ldb, ldc;
    int skip;
};
using RaggedF16 = Ragged<_Float16>;
using RaggedF32 = Ragged<float>;

__device__ __align__(16) const uint32_t kZero16[4] = {0u, 0u, 0u, 0u};

/// exactWaveBlock bounded to m x n. The sums are serial chains, so four rows
/// go together, and 8 steps' loads ahead of their sums (A's by 16-byte pieces,
/// which its rows hold whole): 2000 x 1000 x 3000 with one infinity in B takes
/// 1.0 ms, one row and one step at a time 11.4 (exactWaveBlock around padded
/// copies: 4.6).
template <typename T>
__device__ __forceinline__ void exactRaggedBlock(const Ragged<T>& p, int r0, int c0, int rows, int cols) {
    constexpr int R = 4, U = 8, V = 16 / sizeof(T);
    using Vec = T __attribute__((ext_vector_type(V)));
    const int lane = threadIdx.x & 63;
    rows = min(rows, p.m - r0);
    cols = min(cols, p.n - c0);
    if (lane >= cols) return;
    const T* b = p.b + c0 + lane;
    float* c = p.c + r0 * p.ldc + c0 + lane;
    for (int r = 0; r < rows; r += R) {
        const T* a[R];
        float s[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {   // rows past the last repeat it
            const int row = min(r + i, rows - 1);
            a[i] = p.a + (r0 + row) * p.lda;
            s[i] = c[row * p.ldc];
        }
        auto step = [&](int i, T at, T bt) {
            const float av = static_cast<float>(at);
            if (av != 0.0f) s[i] = s[i] + av * static_cast<float>(bt);
        };
        int k = 0;
        for (; k + U <= p.k; k += U) {
            Vec av[R][U / V];
            T bv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) bv[u] = b[(k + u) * p.ldb];
#pragma unroll
            for (int i = 0; i < R; ++i) {
#pragma unroll
                for (int u = 0; u < U / V; ++u) av[i][u] = *reinterpret_cast<const Vec*>(a[i] + k + u * V);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
                for (int i = 0; i < R; ++i) step(i, av[i][u / V][u % V], bv[u]);
            }
        }
        for (; k < p.k; ++k) {
#pragma unroll
            for (int i = 0; i < R; ++i) step(i, a[i][k], b[k * p.ldb]);
        }
#pragma unroll
        for (int i = 0; i < R; ++i) {
            if (r + i < rows) c[(r + i) * p.ldc] = s[i];
        }
    }
}

/// 16 bytes at 4-byte alignment, all a ragged C has.
struct __attribute__((packed, aligned(4))) Row4 {
    f32x4 v;
};

__device__ __forceinline__ f32x4 loadAny16(const float* p) { return reinterpret_cast<const Row4*>(p)->v; }

/// v (+)= into columns col..col+3 of a row of n.
template <bool ACC>
__device__ __forceinline__ void storeRagged(float* row, int col, int n, f32x4 v) {
    float* dst = row + col;
    if (col + 4 <= n) {
        if (ACC) v += reinterpret_cast<const Row4*>(dst)->v;
        reinterpret_cast<Row4*>(dst)->v = v;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (col + e < n) dst[e] = ACC ? dst[e] + v[e] : v[e];
        }
    }
}

/// Variant 8 (K a multiple of 64): the same tiles, ring, swizzles and
/// per-accumulator MFMAs as gemmF16Dma8 (results identical bit for bit), with
/// no per-step vector address arithmetic and a fixed instruction order.
/// * Vector instructions take issue cycles from the MFMAs of the wave sharing
///   the SIMD (measured on gfx950: 32 v_add_u32 per 32 MFMAs cost 9% of the
///   MFMA rate, 16 v_readfirstlane 18%). gemmF16Dma8 spends about 40 per K
///   step on addresses: 64-bit adds, multiplies by ldb and a readfirstlane
///   per direct load. Here the direct loads take a scalar base plus a fixed
///   32-bit lane offset and M0 comes from scalar registers; the loop is
///   unrolled over the 4 ring slots so that every LDS fragment read is a
///   base register plus an immediate offset (two bases per operand, since
///   DS offsets hold 16 bits).
/// * The compiler does not keep the interleave that sched_group_barrier asks
///   for across the unrolled steps: it hoists the next step's first MFMAs up
///   to the reads that feed them and then waits for those reads every one or
///   two MFMAs. Scheduling fences after each MFMA pin the order, with the
///   memory instructions spread out rather than bunched: the next m-tiles'
///   A reads after every other MFMA of group 1's first half, the next step's
///   fragments after every other MFMA of group 2 in order of first use, and
///   the four direct loads of the stage after every fourth MFMA of group 2
///   from the third (3-4% faster than the same instructions bunched at the
///   start of each group, with identical results).
/// * Within a group the MFMAs walk the 4 x 4 tiles row by row in a snake
///   (n ascending on even m-tiles, descending on odd ones), so every two
///   consecutive MFMAs share an operand register (0.8% faster than plain
///   row order, identical results).
/// Needs lda < 2^23 and ldb < 2^25 (32-bit lane offsets).
/// RAGGED: any m and n, k of any length (rag holds the rest of it); rows past
/// m and columns past n repeat the last ones and are not stored, and lanes
/// past k load zeros in the last K step.
template <bool ACC, bool RAGGED>
__device__ __forceinline__ void dma8sTile(const _Float16* __restrict__ A, const _Float16* __restrict__ B,
                                          float* __restrict__ C, int M, int N, int K, int64_t lda, int64_t ldb,
                                          int64_t ldc, int skipZeroA, const RaggedF16& rag) {
    extern __shared__ __align__(16) _Float16 lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int wm = wave >> 2, wn = wave & 3;
    int tm, tn;
    if constexpr (RAGGED) xcdTile(rag.tilesM, rag.tilesN, tm, tn);
    else xcdTile(M / kBM, N / kBN, tm, tn);
    const int64_t row0 = static_cast<int64_t>(tm) * kBM;
    const int64_t col0 = static_cast<int64_t>(tn) * kBN;
    const int steps = RAGGED ? (K + kDmaBK - 1) / kDmaBK : K / kDmaBK;
    const bool partial = RAGGED && K % kDmaBK != 0;

    // Wave w's direct loads are A instructions 2w, 2w + 1 (16 rows each) and
    // B instructions 2w, 2w + 1 (2 k-rows each) of every stage, as in
    // gemmF16Dma8: lane byte offsets from the tile's A rows / B columns.
    uint32_t gA[2], gB[2];
    int kA[2], kB[2];   // RAGGED: first k of the lane's A piece, k of its B piece, in a step
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int q = (wave * 2 + j) * 64 + lane;
        const int row = q >> 2;
        const int c = (q & 3) ^ ((row >> 2) & 3);
        const int krow = q >> 5;
        const int cb = (q & 31) ^ ((krow & 3) * 4);
        if constexpr (RAGGED) {
            const int r0 = static_cast<int>(row0), c0 = static_cast<int>(col0);
            gA[j] = static_cast<uint32_t>(((min(r0 + row, M - 1) - r0) * lda + c * 8) * 2);
            gB[j] = static_cast<uint32_t>((krow * ldb + min(c0 + cb * 8, rag.nb - 8) - c0) * 2);
        } else {
            gA[j] = static_cast<uint32_t>((row * lda + c * 8) * 2);
            gB[j] = static_cast<uint32_t>((krow * ldb + cb * 8) * 2);
        }
        kA[j] = c * 8;
        kB[j] = krow;
    }
    const char* aTile = reinterpret_cast<const char*>(A + row0 * lda);
    const char* bTile = reinterpret_cast<const char*>(B + col0);
    const uint32_t ldsS = __builtin_amdgcn_readfirstlane(ldsOffset(lds));
    const uint32_t m0Wave = ldsS + static_cast<uint32_t>(wave) * 2048u;
    // Direct load j (A 0, A 1, B 0, B 1) of stage t (K step min(t, steps - 1))
    // into ring slot `slot` = t % 4.
    auto issueOne = [&](int t, const int slot, const int j) {
        if constexpr (RAGGED) {
            if (partial && t >= steps - 1) {
                const int s = steps - 1;
                const char* src = j < 2 ? aTile + static_cast<int64_t>(s) * (kDmaBK * 2) + gA[j & 1]
                                        : bTile + s * ldb * (kDmaBK * 2) + gB[j & 1];
                if ((j < 2 ? kA[j & 1] : kB[j & 1]) >= (j < 2 ? rag.ka : K) - s * kDmaBK) {
                    src = reinterpret_cast<const char*>(kZero16);
                }
                const uint32_t m = m0Wave + static_cast<uint32_t>(slot) * (kDmaStage * 2u) + (j & 1) * 1024u +
                                   (j >= 2 ? kDmaA * 2u : 0u);
                asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(m) : "memory");
                return;
            }
        }
        const int64_t k0 = static_cast<int64_t>(min(t, steps - 1)) * kDmaBK;
        const char* a = aTile + k0 * 2;
        const char* b = bTile + k0 * ldb * 2;
        const uint32_t m = m0Wave + static_cast<uint32_t>(slot) * (kDmaStage * 2u);
        if (j == 0) dmaLoad16s(a, gA[0], m);
        if (j == 1) dmaLoad16s(a, gA[1], m + 1024u);
        if (j == 2) dmaLoad16s(b, gB[0], m + kDmaA * 2u);
        if (j == 3) dmaLoad16s(b, gB[1], m + kDmaA * 2u + 1024u);
    };
    auto issue = [&](int t, const int slot) {
#pragma unroll
        for (int j = 0; j < 4; ++j) issueOne(t, slot, j);
    };

    f32x4 acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    issue(0, 0);
    issue(1, 1);
    issue(2, 2);

    // Fragment bases: slots 0 and 1 from vA0 / vB0, slots 2 and 3 from the
    // bases 64 KiB up; the slot's remaining 0 or 32 KiB, the m-tile (1 KiB)
    // and the second transposed half (4 k-rows, 2 KiB) are immediates.
    const int l16 = lane & 15, g = lane >> 4;
    uint32_t vA0;
    {
        const int row = wm * 128 + l16;
        vA0 = ldsS + 2u * (row * kDmaBK + ((g ^ ((row >> 2) & 3)) * 8));
    }
    uint32_t vB0[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        const int krow = 8 * g + (l16 >> 2);
        const int col = wn * 64 + nt * 16 + 4 * (l16 & 3);
        vB0[nt] = ldsS + 2u * (kDmaA + krow * 256 + (((col >> 3) ^ ((krow & 3) * 4)) * 8) + (col & 7));
    }
    const uint32_t vA2 = vA0 + 65536u;
    uint32_t vB2[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) vB2[nt] = vB0[nt] + 65536u;
    auto readA = [&](f16x8& f, const int slot, int mt) {
        const uint32_t addr = (slot < 2 ? vA0 : vA2) + static_cast<uint32_t>((slot & 1) * kDmaStage * 2 + 1024 * mt);
        f = *reinterpret_cast<const __attribute__((address_space(3))) f16x8*>(addr);
    };
    auto readB = [&](f16x8& f, const int slot, int nt) {
        const uint32_t base = (slot < 2 ? vB0[nt] : vB2[nt]) + static_cast<uint32_t>((slot & 1) * kDmaStage * 2);
        const fp16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
            reinterpret_cast<__attribute__((address_space(3))) fp16x4*>(base));
        const fp16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
            reinterpret_cast<__attribute__((address_space(3))) fp16x4*>(base + 2048u));
        f = __builtin_shufflevector(__builtin_bit_cast(f16x4, v0), __builtin_bit_cast(f16x4, v1), 0, 1, 2, 3, 4, 5,
                                    6, 7);
    };
    f16x8 aLo[4], aHi[4], bX[4], bY[4];
    // Stage 0 landed (stages 1 and 2, 4 direct loads each per wave, may be in
    // flight).
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; ++i) readA(aLo[i], 0, i);
#pragma unroll
    for (int j = 0; j < 4; ++j) readB(bX[j], 0, j);
    auto mfma = [&](const f16x8& a, const f16x8& b, f32x4& c) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, a, c, 0, 0, 0);
    };
    // K step s in ring slot q = s % 4.
    auto step = [&](int s, const int q, f16x8 (&bCur)[4], f16x8 (&bNxt)[4]) {
        const int qn = (q + 1) & 3;
        // Group 1: m-tiles 0-3; the A fragments of m-tiles 4-7 are read
        // behind MFMAs 0, 2, 4 and 6.
#pragma unroll
        for (int idx = 0; idx < 16; ++idx) {
            const int mi = idx >> 2, ni = (mi & 1) ? 3 - (idx & 3) : (idx & 3);
            mfma(aLo[mi], bCur[ni], acc[mi][ni]);
            if (idx < 8 && (idx & 1) == 0) readA(aHi[idx >> 1], q, 4 + (idx >> 1));
            __builtin_amdgcn_sched_barrier(0);
        }
        // Stage s + 1 landed (one later stage may be in flight); after the
        // barrier every wave is past step s - 1, so its slot can be refilled.
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        // Group 2: m-tiles 4-7; step s + 1's fragments read behind the even
        // MFMAs in order of first use (B 0, A 0, B 1-3, A 1-3), and stage
        // s + 3's direct loads into slot (s - 1) % 4 behind MFMAs 2, 6, 10, 14.
#pragma unroll
        for (int idx = 0; idx < 16; ++idx) {
            const int mi = idx >> 2, ni = (mi & 1) ? 3 - (idx & 3) : (idx & 3);
            mfma(aHi[mi], bCur[ni], acc[4 + mi][ni]);
            if (idx == 0) readB(bNxt[0], qn, 0);
            if (idx == 2) readA(aLo[0], qn, 0);
            if (idx >= 4 && idx <= 8 && (idx & 1) == 0) readB(bNxt[(idx - 2) >> 1], qn, (idx - 2) >> 1);
            if (idx >= 10 && (idx & 1) == 0) readA(aLo[(idx - 8) >> 1], qn, (idx - 8) >> 1);
            if ((idx & 3) == 2) issueOne(s + kDmaStages - 1, (q + 3) & 3, idx >> 2);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int s = 0;
    for (; s + 4 <= steps; s += 4) {
        step(s, 0, bX, bY);
        step(s + 1, 1, bY, bX);
        step(s + 2, 2, bX, bY);
        step(s + 3, 3, bY, bX);
    }
    if constexpr (RAGGED) {
        if (s < steps) step(s, 0, bX, bY);
        if (s + 1 < steps) step(s + 1, 1, bY, bX);
        if (s + 2 < steps) step(s + 2, 2, bX, bY);
    } else if (s < steps) {   // K % 128 == 64: two more steps, in slots 0 and 1
        step(s, 0, bX, bY);
        step(s + 1, 1, bY, bX);
    }
    // No direct load may still be writing LDS when the workgroup ends.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (RAGGED) {
        const int r0 = static_cast<int>(row0) + wm * 128, c0 = static_cast<int>(col0) + wn * 64;
        if (ACC && skipZeroA && waveNonFinite(acc)) {
            exactRaggedBlock(rag, r0, c0, 128, 64);
            return;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = r0 + i * 16 + l16;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (row < M) storeRagged<ACC>(C + row * ldc, c0 + j * 16 + 4 * g, N, acc[i][j]);
            }
        }
        return;
    }
    if (ACC && skipZeroA && waveNonFinite(acc)) {
        exactWaveBlock<_Float16, _Float16>(A, B, C, lda, ldb, ldc, K, row0 + wm * 128, col0 + wn * 64, 128, 64, ACC);
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t row = row0 + wm * 128 + i * 16 + l16;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32x4* dst = reinterpret_cast<f32x4*>(C + row * ldc + col0 + wn * 64 + j * 16 + 4 * g);
            f32x4 v = acc[i][j];
            if (ACC) v += *dst;
            *dst = v;
        }
    }
}

template <bool ACC>
__global__ __launch_bounds__(512, 1) void gemmF16Dma8s(const _Float16* __restrict__ A,
                                                       const _Float16* __restrict__ B,
                                                       float* __restrict__ C, int M, int N, int K,
                                                       int64_t lda, int64_t ldb, int64_t ldc,
                                                       int skipZeroA) {
    dma8sTile<ACC, false>(A, B, C, M, N, K, lda, ldb, ldc, skipZeroA, RaggedF16{});
}

/// The ragged member on the same 256 x 256 tiles.
struct RaggedF16Wide : RaggedF16 {};

template <bool ACC>
__global__ __launch_bounds__(512, 1) void gemmF16Dma8s(RaggedF16Wide p) {
    dma8sTile<ACC, true>(p.a, p.b, p.c, p.m, p.n, p.k, p.lda, p.ldb, p.ldc, p.skip, p);
}

constexpr int kRM = 128, kRN = 128;                        // output tile
constexpr int kRA = kRM * kDmaBK;                          // halves per A stage
constexpr int kRStage = kRA + kDmaBK * kRN;                // A, then B
constexpr size_t kLdsRagged = static_cast<size_t>(kDmaStages) * kRStage * sizeof(_Float16);   // 64 KiB

/// The ragged member on tiles of 128 x 128, for shapes that 256 x 256 tiles
/// leave most of the chip idle with: the same direct loads, ring, swizzles,
/// MFMAs and fences, 4 waves of 64 x 64 (16 MFMAs a K step), two workgroups to
/// a CU, bounded as dma8sTile<ACC, true> is. A K step takes 0.31 us for each
/// tile on a CU, one or two: its LDS traffic (32 KiB of reads, half of them
/// transposed, 16 KiB of direct loads; 256 x 128 tiles of 8 waves, a quarter
/// less to load, are no faster). A text of its own, since the schedule is fenced
/// MFMA by MFMA, and 16 a step with 8 fragments to read have other places for
/// the reads, loads and barrier than 32 with 12. 2000 x 1000 x 3000 takes 24.5 us, with C += A
/// B 27.9 us (zero-padded copies of A, B and C around 256 x 256 tiles: 44.4
/// and 59.7 us), 2000^3 25 us (58 us), 1000 x 600 x 1000 10.4 us (28 us).
template <bool ACC>
__global__ __launch_bounds__(256, 2) void gemmF16Dma8s(RaggedF16 p) {
    extern __shared__ __align__(16) _Float16 lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int wm = wave >> 1, wn = wave & 1;
    // Consecutive workgroups go to different XCDs: each takes a contiguous
    // share of the tiles, in columns of 8 tile rows, so that its L2 holds 8 A
    // panels and few B panels.
    const int total = p.tilesM * p.tilesN;
    int id = static_cast<int>(blockIdx.x);
    if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
    const int band = id / (8 * p.tilesN), inBand = id % (8 * p.tilesN);
    const int bandRows = min(8, p.tilesM - band * 8);
    const int tm = band * 8 + inBand % bandRows, tn = inBand / bandRows;
    const int row0 = tm * kRM, col0 = tn * kRN;
    const int steps = (p.k + kDmaBK - 1) / kDmaBK;
    const bool partial = p.k % kDmaBK != 0;

    // Wave w's direct loads are A instructions 2w, 2w + 1 (16 rows each) and
    // B instructions 2w, 2w + 1 (4 k-rows each) of every stage.
    uint32_t gA[2], gB[2];
    int kA[2], kB[2];   // first k of the lane's A piece, k of its B piece, in a step
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int q = (wave * 2 + j) * 64 + lane;
        const int row = q >> 2;
        kA[j] = ((q & 3) ^ ((row >> 2) & 3)) * 8;
        gA[j] = static_cast<uint32_t>(((min(row0 + row, p.m - 1) - row0) * p.lda + kA[j]) * 2);
        kB[j] = q >> 4;
        const int col = ((q & 15) ^ ((kB[j] & 3) * 4)) * 8;
        gB[j] = static_cast<uint32_t>((kB[j] * p.ldb + min(col0 + col, p.nb - 8) - col0) * 2);
    }
    const char* aTile = reinterpret_cast<const char*>(p.a + row0 * p.lda);
    const char* bTile = reinterpret_cast<const char*>(p.b + col0);
    const uint32_t ldsS = __builtin_amdgcn_readfirstlane(ldsOffset(lds));
    const uint32_t m0Wave = ldsS + static_cast<uint32_t>(wave) * 2048u;
    // Direct load j (A 0, A 1, B 0, B 1) of stage t (K step min(t, steps - 1))
    // into ring slot `slot`.
    auto issueOne = [&](int t, const int slot, const int j) {
        const int s = min(t, steps - 1);
        const char* a = aTile + static_cast<int64_t>(s) * (kDmaBK * 2);
        const char* b = bTile + s * p.ldb * (kDmaBK * 2);
        const uint32_t m = m0Wave + static_cast<uint32_t>(slot) * (kRStage * 2u) + (j & 1) * 1024u +
                           (j >= 2 ? kRA * 2u : 0u);
        if (partial && s == steps - 1) {
            const int left = (j < 2 ? p.ka : p.k) - s * kDmaBK;
            const char* src = j < 2 ? a + gA[j & 1] : b + gB[j & 1];
            if ((j < 2 ? kA[j & 1] : kB[j & 1]) >= left) src = reinterpret_cast<const char*>(kZero16);
            asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(m) : "memory");
        } else {
            dmaLoad16s(j < 2 ? a : b, j < 2 ? gA[j & 1] : gB[j & 1], m);
        }
    };
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) {
#pragma unroll
        for (int j = 0; j < 4; ++j) issueOne(t, t, j);
    }
    // Fragment bases; the slot (16 KiB), the m-tile (1 KiB) and the second
    // transposed half (4 k-rows, 1 KiB) are immediates.
    const int l16 = lane & 15, g = lane >> 4;
    uint32_t vA;
    {
        const int row = wm * 64 + l16;
        vA = ldsS + 2u * (row * kDmaBK + ((g ^ ((row >> 2) & 3)) * 8));
    }
    uint32_t vB[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        const int krow = 8 * g + (l16 >> 2);
        const int col = wn * 64 + nt * 16 + 4 * (l16 & 3);
        vB[nt] = ldsS + 2u * (kRA + krow * kRN + (((col >> 3) ^ ((krow & 3) * 4)) * 8) + (col & 7));
    }
    auto readA = [&](f16x8& f, const int slot, int mt) {
        f = *reinterpret_cast<const __attribute__((address_space(3))) f16x8*>(
            vA + static_cast<uint32_t>(slot * kRStage * 2 + 1024 * mt));
    };
    auto readB = [&](f16x8& f, const int slot, int nt) {
        const uint32_t base = vB[nt] + static_cast<uint32_t>(slot * kRStage * 2);
        const fp16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
            reinterpret_cast<__attribute__((address_space(3))) fp16x4*>(base));
        const fp16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
            reinterpret_cast<__attribute__((address_space(3))) fp16x4*>(base + 1024u));
        f = __builtin_shufflevector(__builtin_bit_cast(f16x4, v0), __builtin_bit_cast(f16x4, v1), 0, 1, 2, 3, 4, 5,
                                    6, 7);
    };
    f16x8 aX[4], aY[4], bX[4], bY[4];
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; ++i) readA(aX[i], 0, i);
#pragma unroll
    for (int j = 0; j < 4; ++j) readB(bX[j], 0, j);
    // K step s in ring slot q = s % 4: 6 MFMAs, then the barrier that
    // certifies stage s + 1 (one later stage may be in flight) and frees slot
    // (s - 1) % 4, then step s + 1's fragments and stage s + 3's loads behind
    // the other MFMAs.
    auto step = [&](int s, const int q, f16x8 (&a)[4], f16x8 (&b)[4], f16x8 (&an)[4], f16x8 (&bn)[4]) {
        const int qn = (q + 1) & 3;
#pragma unroll
        for (int idx = 0; idx < 16; ++idx) {
            const int mi = idx >> 2, ni = (mi & 1) ? 3 - (idx & 3) : (idx & 3);
            acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[ni], a[mi], acc[mi][ni], 0, 0, 0);
            if (idx == 5) {
                asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
                asm volatile("s_barrier" ::: "memory");
            }
            if (idx == 6) readB(bn[0], qn, 0);
            if (idx == 7) readA(an[0], qn, 0);
            if (idx >= 8 && idx <= 10) readB(bn[idx - 7], qn, idx - 7);
            if (idx >= 11 && idx <= 13) readA(an[idx - 10], qn, idx - 10);
            if (idx >= 12) issueOne(s + 3, (q + 3) & 3, idx - 12);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int s = 0;
    for (; s + 4 <= steps; s += 4) {
        step(s, 0, aX, bX, aY, bY);
        step(s + 1, 1, aY, bY, aX, bX);
        step(s + 2, 2, aX, bX, aY, bY);
        step(s + 3, 3, aY, bY, aX, bX);
    }
    if (s < steps) step(s, 0, aX, bX, aY, bY);
    if (s + 1 < steps) step(s + 1, 1, aY, bY, aX, bX);
    if (s + 2 < steps) step(s + 2, 2, aX, bX, aY, bY);
    // No direct load may still be writing LDS when the workgroup ends.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int r0 = row0 + wm * 64, c0 = col0 + wn * 64;
    if (ACC && p.skip && waveNonFinite(acc)) {
        exactRaggedBlock(p, r0, c0, 64, 64);
        return;
    }
    // C += reads all of the wave's C before its first store: the reads of a
    // few, each waited for, took 6 us more at 1000 x 600 x 1000.
    f32x4 old[4][4];
    if constexpr (ACC) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float* row = p.c + min(r0 + i * 16 + l16, p.m - 1) * p.ldc;
#pragma unroll
            for (int j = 0; j < 4; ++j) old[i][j] = loadAny16(row + min(c0 + j * 16 + 4 * g, p.n - 4));
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = r0 + i * 16 + l16;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = c0 + j * 16 + 4 * g;
            if (row >= p.m) continue;
            float* dst = p.c + row * p.ldc;
            if (ACC && col + 4 <= p.n) storeRagged<false>(dst, col, p.n, acc[i][j] + old[i][j]);
            else storeRagged<ACC>(dst, col, p.n, acc[i][j]);
        }
    }
}

// ---------------------------------------------------------------- f32 ----
constexpr int kFM = 64, kFN = 64, kFK = 32;
constexpr int kFDepth = 2;   // K steps of global loads in flight ahead of the MFMAs

/// f32 form 1: 64x64 output tile per workgroup of 4 waves (2 x 2 of 32x32),
/// K steps of 32 through double-buffered LDS, v_mfma_f32_32x32x2f32 with k
/// ascending.
/// Global loads run kFDepth steps ahead in registers (slot t % kFDepth holds
/// step t); A is stored transposed ([k][m]) for the MFMA's A operand, and its
/// load mapping gives each wave 16 rows x 4 k-chunks, so every transposed LDS
/// write of a wave hits 64 distinct banks. At 1024^3 on gfx950: 25-26 us,
/// against 29-31 us with one step in flight and the row-major mapping
/// (4-way write conflicts).
template <bool ACC>
__global__ __launch_bounds__(256) void gemmF32Mfma(const float* __restrict__ A,
                                                   const float* __restrict__ B,
                                                   float* __restrict__ C, int /*M: the grid covers it*/, int N,
                                                   int K, int64_t lda, int64_t ldb, int64_t ldc,
                                                   int /*accumulate: template ACC*/, int skipZeroA) {
    __shared__ float At[2][kFK][kFM + 4];   // transposed: [k][m]
    __shared__ float Bs[2][kFK][kFN + 4];   // as loaded: [k][n]
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;   // 2x2 waves, 32x32 each
    const int tilesN = N / kFN;
    const int64_t row0 = static_cast<int64_t>(blockIdx.x / tilesN) * kFM;
    const int64_t col0 = static_cast<int64_t>(blockIdx.x % tilesN) * kFN;

    // A tile 64x32 floats = 512 float4 and B tile 32x64 = 512 float4: 2 of
    // each per thread. Item c of A: wave-slice q = c / 64 covers rows
    // 16 (q / 2) .. +15 and k-chunks 4 (q % 2) .. +3.
    auto aItem = [&](int c, int& r, int& ch) {
        const int q = c >> 6, ln = c & 63;
        r = (q >> 1) * 16 + (ln & 15);
        ch = (q & 1) * 4 + (ln >> 4);
    };
    f32x4 ra[kFDepth][2], rb[kFDepth][2];
    auto globalLoad = [&](int k0, f32x4 (&xa)[2], f32x4 (&xb)[2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int c = j * 256 + tid;
            int r, ch;
            aItem(c, r, ch);
            xa[j] = *reinterpret_cast<const f32x4*>(A + (row0 + r) * lda + k0 + ch * 4);
            const int kr = c >> 4, nc = c & 15;     // B: 32 rows x 16 chunks
            xb[j] = *reinterpret_cast<const f32x4*>(B + static_cast<int64_t>(k0 + kr) * ldb + col0 + nc * 4);
        }
    };
    auto ldsStore = [&](int buf, const f32x4 (&xa)[2], const f32x4 (&xb)[2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int c = j * 256 + tid;
            int r, ch;
            aItem(c, r, ch);
#pragma unroll
            for (int e = 0; e < 4; ++e) At[buf][ch * 4 + e][r] = xa[j][e];
            const int kr = c >> 4, nc = c & 15;
            *reinterpret_cast<f32x4*>(&Bs[buf][kr][nc * 4]) = xb[j];
        }
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const int steps = K / kFK;
#pragma unroll
    for (int d = 0; d < kFDepth; ++d) {
        if (d < steps) globalLoad(d * kFK, ra[d], rb[d]);
    }
    ldsStore(0, ra[0], rb[0]);
    __syncthreads();
    const int lcol = lane & 31;
    const int lk = lane >> 5;
    for (int s0 = 0; s0 < steps; s0 += kFDepth) {
#pragma unroll
        for (int d = 0; d < kFDepth; ++d) {
            const int s = s0 + d;
            if (s < steps) {
                const int buf = s & 1;
                // Slot d held step s, already in LDS: refill it with s + kFDepth.
                if (s + kFDepth < steps) globalLoad((s + kFDepth) * kFK, ra[d], rb[d]);
#pragma unroll
                for (int kk = 0; kk < kFK; kk += 2) {
                    const float a = At[buf][kk + lk][wm * 32 + lcol];
                    const float b = Bs[buf][kk + lk][wn * 32 + lcol];
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
                }
                if (s + 1 < steps) ldsStore(buf ^ 1, ra[(d + 1) % kFDepth], rb[(d + 1) % kFDepth]);
                __syncthreads();
            }
        }
    }
    if (ACC && skipZeroA && waveNonFinite(acc)) {
        exactWaveBlock<float, float>(A, B, C, lda, ldb, ldc, K, row0 + wm * 32, col0 + wn * 32, 32, 32, ACC);
        return;
    }
    const int64_t cBase = col0 + wn * 32 + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t row = row0 + wm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        float* dst = C + row * ldc + cBase;
        *dst = ACC ? *dst + acc[r] : acc[r];
    }
}

/// f32 form 0: both 64x64 tiles move global -> LDS by the direct path
/// (global_load_lds_dwordx4, no register staging and no LDS writes) into a
/// 4-deep ring of K steps of 64 (32 KiB per stage). 8 waves: waves q and
/// q + 4 own the same 32x32 tile (2 x 2 quadrants) on v_mfma_f32_32x32x2_f32
/// and take the two halves of every K step, so each SIMD runs two
/// independent accumulator chains. Within a step the k order is permuted:
/// MFMA t takes k = t from lanes 0-31 and k = 32 + t from lanes 32-63; wave
/// half h takes t = 16h .. 16h + 15. The A operand of 4 consecutive MFMAs is
/// then one 16-byte read of a row of A (16-byte chunk c of row m sits at
/// c ^ (m & 15): the 16 rows a quarter-wave reads hit 16 distinct slots),
/// and the B operand a 4-byte read of 32 consecutive columns. One barrier
/// per K step; every step issues exactly one stage (past the end a harmless
/// reload into a slot nothing reads), so the wait before the barrier is a
/// constant vmcnt. At the end the second half's sums reach the first half's
/// waves through LDS and each output is half 0 + half 1, in that order.
/// Needs K a multiple of 64. Each output's sum runs over k in a different
/// order from form 1's k ascending, within the f32 tolerance.
constexpr int kQK = 64, kQStages = 4;
constexpr int kQA = kFM * kQK;                        // floats per A stage (64 rows x 64 k)
constexpr int kQStage = 2 * kQA;                      // A, then B (64 k x 64 n)
constexpr size_t kLdsF32Dma = static_cast<size_t>(kQStages) * kQStage * sizeof(float);   // 128 KiB

template <bool ACC>
__global__ __launch_bounds__(512, 1) void gemmF32Dma(const float* __restrict__ A, const float* __restrict__ B,
                                                     float* __restrict__ C, int N, int K, int64_t lda,
                                                     int64_t ldb, int64_t ldc, int skipZeroA) {
    extern __shared__ __align__(16) float ldsF[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int quad = wave & 3, h = wave >> 2;   // output quadrant, K-step half
    const int wm = quad >> 1, wn = quad & 1;
    const int tilesN = N / kFN;
    // XCD-blocked map: at 1024^2 each XCD's 32 tiles form a 4 x 8 block, so
    // its L2 holds 4 A and 8 B panels (3 MiB) instead of 16 A panels; the
    // bytes fetched per launch drop by a third (FETCH_SIZE 18470 -> 12330 KiB).
    int tm, tn;
    xcdTile(static_cast<int>(gridDim.x) / tilesN, tilesN, tm, tn);
    const int64_t row0 = static_cast<int64_t>(tm) * kFM;
    const int64_t col0 = static_cast<int64_t>(tn) * kFN;
    const int steps = K / kQK;
    // Stage `slot` receives K step min(slot, steps - 1) in ring slot
    // slot % kQStages. A is 64 rows of 256 bytes and B 64 k-rows of 256
    // bytes, 16 direct loads of 4 rows each: wave w issues instructions
    // 2w and 2w + 1 of each.
    auto issue = [&](int slot) {
        const int k0 = min(slot, steps - 1) * kQK;
        const float* st = ldsF + (slot % kQStages) * kQStage;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ins = wave * 2 + j;
            const int row = ins * 4 + (lane >> 4);
            const int c = (lane & 15) ^ (row & 15);
            dmaLoad16(reinterpret_cast<const _Float16*>(A + (row0 + row) * lda + k0 + c * 4),
                      reinterpret_cast<const _Float16*>(st + ins * 256));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ins = wave * 2 + j;
            const int krow = ins * 4 + (lane >> 4);
            dmaLoad16(reinterpret_cast<const _Float16*>(B + static_cast<int64_t>(k0 + krow) * ldb + col0 +
                                                        (lane & 15) * 4),
                      reinterpret_cast<const _Float16*>(st + kQA + ins * 256));
        }
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int s = 0; s < kQStages - 1; ++s) issue(s);
    const int l32 = lane & 31, hl = lane >> 5;
    const int m = wm * 32 + l32;
    // A: row m, chunks 8 hl + 4 h .. + 3 (k 32 hl + 16 h .. + 15) at their
    // slots.
    uint32_t offA[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int q = 4 * h + i;
        offA[i] = 4u * static_cast<uint32_t>(m * kQK + (((8 * hl + q) ^ (m & 15)) * 4));
    }
    // B: k-row 32 hl + 16 h + t, column wn * 32 + l32.
    const uint32_t offB = 4u * static_cast<uint32_t>(kQA + (32 * hl + 16 * h) * kFN + wn * 32 + l32);
    const uint32_t ldsBase = ldsOffset(ldsF);
    // Stage 0 landed (stages 1 and 2, 4 direct loads each per wave, may be
    // in flight).
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    for (int s = 0; s < steps; ++s) {
        const uint32_t cb = ldsBase + 4u * static_cast<uint32_t>((s % kQStages) * kQStage);
        f32x4 a[4];
        float b[16];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(cb + offA[i]);
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            b[t] = *reinterpret_cast<const __attribute__((address_space(3))) float*>(cb + offB + 4u * kFN * t);
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t >> 2][t & 3], b[t], acc, 0, 0, 0);
        // Stage s + 1 landed (one later stage may be in flight); after the
        // barrier every wave is past step s, so slot (s + 3) % 4, which held
        // step s - 1, can be refilled.
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
        issue(s + kQStages - 1);
    }
    // No direct load may still be writing LDS when the halves meet there.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    float* red = ldsF + quad * (64 * 16);
    if (h == 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) red[r * 64 + lane] = acc[r];
    }
    __syncthreads();
    if (h == 1) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] += red[r * 64 + lane];
    if (ACC && skipZeroA && waveNonFinite(acc)) {
        exactWaveBlock<float, float>(A, B, C, lda, ldb, ldc, K, row0 + wm * 32, col0 + wn * 32, 32, 32, ACC);
        return;
    }
    const int64_t cBase = col0 + wn * 32 + l32;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t row = row0 + wm * 32 + 8 * (r >> 2) + 4 * hl + (r & 3);
        float* dst = C + row * ldc + cBase;
        *dst = ACC ? *dst + acc[r] : acc[r];
    }
}

/// The ragged member: the same ring and reads on any m, n and k. Rows past m
/// and columns past n repeat the last ones and are not stored; in the last K
/// step, lanes past k load zeros. (A text of its own: a shared one moves the
/// instructions of the whole-block kernel, 1% at 1024^3.) 1000^3 takes 22.9
/// us, 700 x 1000 x 900 with C += A B 24.4 us (zero-padded copies of A, B and C
/// around the whole-block kernel: 30.0 and 36.0 us).
template <bool ACC>
__global__ __launch_bounds__(512, 1) void gemmF32Dma(RaggedF32 p) {
    extern __shared__ __align__(16) float ldsF[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int quad = wave & 3, h = wave >> 2;   // output quadrant, K-step half
    const int wm = quad >> 1, wn = quad & 1;
    int tm, tn;
    xcdTile(p.tilesM, p.tilesN, tm, tn);
    const int row0 = tm * kFM, col0 = tn * kFN;
    const int steps = (p.k + kQK - 1) / kQK;
    auto issue = [&](int slot) {
        const int k0 = min(slot, steps - 1) * kQK;
        const float* st = ldsF + (slot % kQStages) * kQStage;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ins = wave * 2 + j;
            const int row = ins * 4 + (lane >> 4);
            const int k = k0 + ((lane & 15) ^ (row & 15)) * 4;
            const void* src = p.a + min(row0 + row, p.m - 1) * p.lda + k;
            if (k >= p.ka) src = kZero16;
            dmaLoad16(static_cast<const _Float16*>(src), reinterpret_cast<const _Float16*>(st + ins * 256));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ins = wave * 2 + j;
            const int k = k0 + ins * 4 + (lane >> 4);
            const void* src = p.b + k * p.ldb + min(col0 + (lane & 15) * 4, p.nb - 4);
            if (k >= p.k) src = kZero16;
            dmaLoad16(static_cast<const _Float16*>(src), reinterpret_cast<const _Float16*>(st + kQA + ins * 256));
        }
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int s = 0; s < kQStages - 1; ++s) issue(s);
    const int l32 = lane & 31, hl = lane >> 5;
    const int m = wm * 32 + l32;
    uint32_t offA[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int q = 4 * h + i;
        offA[i] = 4u * static_cast<uint32_t>(m * kQK + (((8 * hl + q) ^ (m & 15)) * 4));
    }
    const uint32_t offB = 4u * static_cast<uint32_t>(kQA + (32 * hl + 16 * h) * kFN + wn * 32 + l32);
    const uint32_t ldsBase = ldsOffset(ldsF);
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    for (int s = 0; s < steps; ++s) {
        const uint32_t cb = ldsBase + 4u * static_cast<uint32_t>((s % kQStages) * kQStage);
        f32x4 a[4];
        float b[16];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(cb + offA[i]);
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            b[t] = *reinterpret_cast<const __attribute__((address_space(3))) float*>(cb + offB + 4u * kFN * t);
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t >> 2][t & 3], b[t], acc, 0, 0, 0);
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
        issue(s + kQStages - 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    float* red = ldsF + quad * (64 * 16);
    if (h == 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) red[r * 64 + lane] = acc[r];
    }
    __syncthreads();
    if (h == 1) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] += red[r * 64 + lane];
    const int r0 = row0 + wm * 32, c0 = col0 + wn * 32;
    if (ACC && p.skip && waveNonFinite(acc)) {
        exactRaggedBlock(p, r0, c0, 32, 32);
        return;
    }
    const int col = c0 + l32;
    auto rowOf = [&](int r) { return r0 + 8 * (r >> 2) + 4 * hl + (r & 3); };
    if (ACC) {   // all of the lane's C before its first store
        const float* old = p.c + min(col, p.n - 1);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] += old[min(rowOf(r), p.m - 1) * p.ldc];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        if (rowOf(r) < p.m && col < p.n) p.c[rowOf(r) * p.ldc + col] = acc[r];
    }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Process default of the f16 GEMM launch form (a launch's own `variant`
// field overrides it): 0: 8 waves of 128x64; 1: 4 waves of 128x128; 2: 4
// waves with A direct to LDS; 3: 4 waves, explicitly pipelined; 5/6:
// 128x256 tiles, two workgroups per CU, loads two / one step ahead;
// 7: 4 waves, both operands direct to a 4-deep LDS ring, B read transposed;
// 8: variant 7's data path with 8 waves of 16x16x32 MFMA tiles (measured
// fastest on gfx950).
int gGemmF16Variant = 8;

/// The members of gemmF16Dma8s: whole 256 x 256 x 64 blocks, and ragged shapes.
using Tiled8s = void (*)(const _Float16*, const _Float16*, float*, int, int, int, int64_t, int64_t, int64_t, int);
using Ragged8s = void (*)(RaggedF16);
using RaggedWide8s = void (*)(RaggedF16Wide);
/// And of gemmF32Dma.
using TiledF32 = void (*)(const float*, const float*, float*, int, int, int64_t, int64_t, int64_t, int);
using RaggedDma = void (*)(RaggedF32);

/// Raises the dynamic-LDS limit of every form that needs more than the
/// default, once per process (a function-local static: its initialization
/// is thread-safe); returns 0 or MLKD_RT_LAUNCH.
int raiseLdsLimits() {
    static const int rc = [] {
        struct Need {
            const void* fn;
            size_t bytes;
        };
        const size_t ldsBytes = 4 * kTileHalves * sizeof(_Float16);
        const size_t ldsDirect = (2 * kTileA + 2 * kTileHalves) * sizeof(_Float16);
        const Need needs[] = {
            {reinterpret_cast<const void*>(gemmF16Mfma<true>), ldsBytes},
            {reinterpret_cast<const void*>(gemmF16Mfma<false>), ldsBytes},
            {reinterpret_cast<const void*>(gemmF16Mfma4w<true>), ldsBytes},
            {reinterpret_cast<const void*>(gemmF16Mfma4w<false>), ldsBytes},
            {reinterpret_cast<const void*>(gemmF16Mfma4wDirect<true>), ldsDirect},
            {reinterpret_cast<const void*>(gemmF16Mfma4wDirect<false>), ldsDirect},
            {reinterpret_cast<const void*>(gemmF16Mfma4wPipe<true>), ldsDirect},
            {reinterpret_cast<const void*>(gemmF16Mfma4wPipe<false>), ldsDirect},
            {reinterpret_cast<const void*>(gemmF16Dma<true>), kLdsDma},
            {reinterpret_cast<const void*>(gemmF16Dma<false>), kLdsDma},
            {reinterpret_cast<const void*>(gemmF16Dma8<true>), kLdsDma},
            {reinterpret_cast<const void*>(gemmF16Dma8<false>), kLdsDma},
            {reinterpret_cast<const void*>(static_cast<Tiled8s>(gemmF16Dma8s<true>)), kLdsDma},
            {reinterpret_cast<const void*>(static_cast<Tiled8s>(gemmF16Dma8s<false>)), kLdsDma},
            {reinterpret_cast<const void*>(static_cast<RaggedWide8s>(gemmF16Dma8s<true>)), kLdsDma},
            {reinterpret_cast<const void*>(static_cast<RaggedWide8s>(gemmF16Dma8s<false>)), kLdsDma},
            {reinterpret_cast<const void*>(static_cast<TiledF32>(gemmF32Dma<true>)), kLdsF32Dma},
            {reinterpret_cast<const void*>(static_cast<TiledF32>(gemmF32Dma<false>)), kLdsF32Dma},
            {reinterpret_cast<const void*>(static_cast<RaggedDma>(gemmF32Dma<true>)), kLdsF32Dma},
            {reinterpret_cast<const void*>(static_cast<RaggedDma>(gemmF32Dma<false>)), kLdsF32Dma},
        };
        for (const Need& n : needs) {
            if (hipFuncSetAttribute(n.fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(n.bytes)) !=
                hipSuccess) {
                return static_cast<int>(MLKD_RT_LAUNCH);
            }
        }
        return 0;
    }();
    return rc;
}

/// The MFMA form a launch takes: the f16 form (0-3, 5-8) or 100 + the f32
/// form (0, 1); -1 when the shape, dtypes or alignment fit none of them.
int mfmaForm(const mlkd_gemm* p) {
    const bool fits32 = p->m < (1LL << 31) && p->n < (1LL << 31) && p->k < (1LL << 31);
    if (p->k <= 0 || !fits32) return -1;
    if (p->a_dtype == MLKD_F16 && p->b_dtype == MLKD_F16 && p->c_dtype == MLKD_F32 && p->m % kBM == 0 &&
        p->n % kBN == 0 && p->k % kBK == 0 && p->lda % 8 == 0 && p->ldb % 8 == 0 && aligned16(p->a) &&
        aligned16(p->b)) {
        const int v = p->variant >= 0 ? p->variant : gGemmF16Variant;
        if (v == 8) return (p->ldc % 4) == 0 && aligned16(p->c) ? 8 : 7;
        return v == 7 || v == 5 || v == 6 || v == 3 || v == 2 || v == 1 ? v : 0;
    }
    if (p->a_dtype == MLKD_F32 && p->b_dtype == MLKD_F32 && p->c_dtype == MLKD_F32 && p->m % kFM == 0 &&
        p->n % kFN == 0 && p->k % kFK == 0 && p->lda % 4 == 0 && p->ldb % 4 == 0 && aligned16(p->a) &&
        aligned16(p->b)) {
        const int fv = p->variant >= 0 ? p->variant : 0;
        return fv != 1 && p->k % kQK == 0 ? 100 : 101;
    }
    return -1;
}

/// Whether a launch runs on an MFMA form as it is. Only the accumulating
/// (Call) form skips zeros; a non-accumulating launch that asks for the skip
/// takes the general kernel.
bool tiled(const mlkd_gemm* p) { return mfmaForm(p) >= 0 && (p->skip_zero_a == 0 || p->accumulate != 0); }

/// Form 8 takes gemmF16Dma8s when its lane offsets fit 32 bits and
/// gemmF16Dma8 otherwise; the two give identical results.
bool scalarAddressed8(const mlkd_gemm* p) {
    return p->lda < (int64_t{1} << 23) && p->ldb < (int64_t{1} << 25);
}

int launchMfma(const mlkd_gemm* p, int form, hipStream_t st) {
    const int skip = p->skip_zero_a != 0 ? 1 : 0;
    if (raiseLdsLimits() != 0) return MLKD_RT_LAUNCH;
    const _Float16* a16 = static_cast<const _Float16*>(p->a);
    const _Float16* b16 = static_cast<const _Float16*>(p->b);
    float* c = static_cast<float*>(p->c);
    const int m = static_cast<int>(p->m), n = static_cast<int>(p->n), k = static_cast<int>(p->k);
    const bool acc = p->accumulate != 0;
    const int tiles = static_cast<int>((p->m / kBM) * (p->n / kBN));
    const size_t ldsBytes = 4 * kTileHalves * sizeof(_Float16);
    const size_t ldsDirect = (2 * kTileA + 2 * kTileHalves) * sizeof(_Float16);
    switch (form) {
        case 8:
            if (scalarAddressed8(p)) {
                const Tiled8s kern = acc ? Tiled8s{gemmF16Dma8s<true>} : Tiled8s{gemmF16Dma8s<false>};
                hipLaunchKernelGGL(kern, dim3(tiles), dim3(512), kLdsDma, st, a16, b16, c, m, n, k, p->lda, p->ldb,
                                   p->ldc, skip);
            } else {
                hipLaunchKernelGGL((acc ? gemmF16Dma8<true> : gemmF16Dma8<false>), dim3(tiles), dim3(512), kLdsDma,
                                   st, a16, b16, c, m, n, k, p->lda, p->ldb, p->ldc, skip);
            }
            break;
        case 7:
            hipLaunchKernelGGL((acc ? gemmF16Dma<true> : gemmF16Dma<false>), dim3(tiles), dim3(256), kLdsDma, st,
                               a16, b16, c, m, n, k, p->lda, p->ldb, p->ldc, skip);
            break;
        case 5:
        case 6: {
            const int tiles2 = static_cast<int>((p->m / kBM2) * (p->n / kBN2));
            auto kern = form == 5 ? (acc ? gemmF16Mfma2cu<true, true> : gemmF16Mfma2cu<false, true>)
                                  : (acc ? gemmF16Mfma2cu<true, false> : gemmF16Mfma2cu<false, false>);
            hipLaunchKernelGGL(kern, dim3(tiles2), dim3(256), kLdsGemm2, st, a16, b16, c, m, n, k, p->lda, p->ldb,
                               p->ldc, skip);
            break;
        }
        case 3:
            hipLaunchKernelGGL((acc ? gemmF16Mfma4wPipe<true> : gemmF16Mfma4wPipe<false>), dim3(tiles), dim3(256),
                               ldsDirect, st, a16, b16, c, m, n, k, p->lda, p->ldb, p->ldc, skip);
            break;
        case 2:
            hipLaunchKernelGGL((acc ? gemmF16Mfma4wDirect<true> : gemmF16Mfma4wDirect<false>), dim3(tiles),
                               dim3(256), ldsDirect, st, a16, b16, c, m, n, k, p->lda, p->ldb, p->ldc, p->accumulate,
                               skip);
            break;
        case 1:
            hipLaunchKernelGGL((acc ? gemmF16Mfma4w<true> : gemmF16Mfma4w<false>), dim3(tiles), dim3(256), ldsBytes,
                               st, a16, b16, c, m, n, k, p->lda, p->ldb, p->ldc, p->accumulate, skip);
            break;
        case 0:
            hipLaunchKernelGGL((acc ? gemmF16Mfma<true> : gemmF16Mfma<false>), dim3(tiles), dim3(512), ldsBytes, st,
                               a16, b16, c, m, n, k, p->lda, p->ldb, p->ldc, p->accumulate, skip);
            break;
        case 100:
        case 101: {
            const int ftiles = static_cast<int>((p->m / kFM) * (p->n / kFN));
            const float* a32 = static_cast<const float*>(p->a);
            const float* b32 = static_cast<const float*>(p->b);
            if (form == 100) {
                hipLaunchKernelGGL((acc ? TiledF32{gemmF32Dma<true>} : TiledF32{gemmF32Dma<false>}), dim3(ftiles), dim3(512),
                                   kLdsF32Dma, st, a32, b32, c, n, k, p->lda, p->ldb, p->ldc, skip);
            } else {
                hipLaunchKernelGGL((acc ? gemmF32Mfma<true> : gemmF32Mfma<false>), dim3(ftiles), dim3(256), 0, st,
                                   a32, b32, c, m, n, k, p->lda, p->ldb, p->ldc, p->accumulate, skip);
            }
            break;
        }
        default:
            return MLKD_RT_LAUNCH;
    }
    return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
}

/// Whether a product no whole-block form tiles runs on a ragged member: f16
/// operands with an f32 C, or all-f32, at least 2^30 flop or a padding to 256 x
/// 256 (f32: 64 x 64) x 64 blocks of at most 8 times the work. The general
/// kernel has the others.
bool raggedShape(const mlkd_gemm* p) {
    const bool f16 = p->a_dtype == MLKD_F16 && p->b_dtype == MLKD_F16 && p->c_dtype == MLKD_F32;
    const bool f32 = p->a_dtype == MLKD_F32 && p->b_dtype == MLKD_F32 && p->c_dtype == MLKD_F32;
    if (!(f16 || f32) || p->m <= 0 || p->n <= 0 || p->k <= 0) return false;
    if (p->skip_zero_a != 0 && p->accumulate == 0) return false;   // that launch takes the general kernel
    if (mfmaForm(p) >= 0) return false;                             // whole blocks
    if (p->m >= (1 << 30) || p->n >= (1 << 30) || p->k >= (1 << 30)) return false;
    const int64_t tile = f16 ? kBM : kFM;
    const int64_t pm = (p->m + tile - 1) / tile * tile, pn = (p->n + tile - 1) / tile * tile, pk = (p->k + 63) / 64 * 64;
    // A few rows or columns, a quarter of a tile or less: the general kernel
    // fits its tiles to them (f16 64x4096x4096: 15 us; f32 16x4096x4096: 17 us).
    if (pm >= 4 * p->m || pn >= 4 * p->n) return false;
    // Few tiles with a long K: a tile's K loop is serial, and the general
    // kernel cuts K over waves and workgroups (f16 500^3: 5.8 against 11.8 us,
    // 100x4096x4096: 18 against 40 us; f32 500^3: 6.7 against 13.0 us,
    // 200x2000x2000: 29 against 40 us).
    if (f16 && (p->m + kRM - 1) / kRM * ((p->n + kRN - 1) / kRN) < 64 && p->k >= 256) return false;
    if (f32 && pm / kFM * (pn / kFN) <= 128 && p->k >= 128) return false;
    // A grid holds fewer than 2^32 threads (2^23 tiles: a C of 137 GB).
    if (f32 && pm / kFM * (pn / kFN) >= (int64_t{1} << 32) / 512) return false;
    const double work = static_cast<double>(p->m) * static_cast<double>(p->n) * static_cast<double>(p->k);
    return 2.0 * work >= static_cast<double>(int64_t{1} << 30) ||
           static_cast<double>(pm) * static_cast<double>(pn) * static_cast<double>(pk) <= 8.0 * work;
}

size_t align256g(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }

/// One operand's copy for a ragged member: rows x cols elements at stride ld
/// into rows of dcols (whole 16-byte pieces), zeros past cols.
template <typename T>
struct RowCopy {
    const T* src;
    T* dst;
    int64_t rows, cols, ld, dcols;
};

/// Both operands' copies in one launch (blockIdx.z), in 16-byte pieces read at
/// any element alignment; the piece that straddles `cols` element by element.
template <typename T>
__global__ __launch_bounds__(256) void copyRows(RowCopy<T> first, RowCopy<T> second) {
    const RowCopy<T>& c = blockIdx.z == 0 ? first : second;
    constexpr int V = 16 / sizeof(T);
    struct __attribute__((packed, aligned(sizeof(T)))) Any16 {
        u32x4 v;
    };
    const int64_t pieces = c.dcols / V;
    for (int64_t r = blockIdx.y; r < c.rows; r += gridDim.y) {
        for (int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; j < pieces;
             j += static_cast<int64_t>(gridDim.x) * 256) {
            const int64_t c0 = j * V;
            const T* src = c.src + r * c.ld + c0;
            u32x4 v = {0u, 0u, 0u, 0u};
            if (c0 + V <= c.cols) {
                v = reinterpret_cast<const Any16*>(src)->v;
            } else if (c0 < c.cols) {
                T e[V];
#pragma unroll
                for (int i = 0; i < V; ++i) e[i] = c0 + i < c.cols ? src[i] : T{0};
                v = __builtin_bit_cast(u32x4, e);
            }
            *reinterpret_cast<u32x4*>(c.dst + r * c.dcols + c0) = v;
        }
    }
}

/// How such a product runs: an operand off 16 bytes, or with rows that are, is
/// copied to aligned rows first.
struct RaggedPlan {
    bool copyA, copyB;
    bool wide;        // f16 tiles of 256 x 256, not 128 x 128
    int64_t ka, nb;   // columns of A's and B's rows as the kernel reads them
    size_t bytesA, bytesB;
};

bool raggedPlan(const mlkd_gemm* p, RaggedPlan& r) {
    if (!raggedShape(p) || (reinterpret_cast<uintptr_t>(p->c) & 3) != 0) return false;
    const int64_t es = p->a_dtype == MLKD_F16 ? 2 : 4, v = 16 / es;
    r.copyA = p->k % v != 0 || p->lda % v != 0 || !aligned16(p->a);
    r.copyB = p->n % v != 0 || p->ldb % v != 0 || !aligned16(p->b);
    // The tile with the shorter run: rounds over 256 CUs of K steps of 32, each
    // 0.31 us on 128 x 128 and 0.65-0.85 on 256 x 256, and the start and end
    // (2000^3: 25 us against 50, 3000^3: 93 against 71, 4000^3: 160 against 119).
    const auto run = [&](int64_t t, double step, double ends) {
        const int64_t tiles = (p->m + t - 1) / t * ((p->n + t - 1) / t);
        return static_cast<double>((tiles + 255) / 256) * static_cast<double>((p->k + 31) / 32) * step + ends;
    };
    r.wide = es == 2 && run(256, 0.75, 10.0) < run(128, 0.31, 5.0);
    r.ka = r.copyA ? (p->k + v - 1) / v * v : p->k;
    r.nb = r.copyB ? (p->n + v - 1) / v * v : p->n;
    r.bytesA = r.copyA ? align256g(static_cast<size_t>(p->m * r.ka * es)) : 0;
    r.bytesB = r.copyB ? align256g(static_cast<size_t>(p->k * r.nb * es)) : 0;
    // Lane offsets of 32 bits (f16).
    const int64_t lda = r.copyA ? r.ka : p->lda, ldb = r.copyB ? r.nb : p->ldb;
    return es == 4 || (lda < (int64_t{1} << 23) && ldb < (int64_t{1} << 25));
}

/// Whether the copies, if any, have their workspace.
bool roomFor(const mlkd_gemm* p, const RaggedPlan& r) {
    const int64_t need = static_cast<int64_t>(r.bytesA + r.bytesB);
    return need == 0 || (p->work != nullptr && p->work_bytes >= need);
}

template <typename Args, typename T>
Args raggedArgs(const mlkd_gemm* p, const RaggedPlan& r, int tileM, int tileN, hipStream_t st) {
    using Bits = std::conditional_t<sizeof(T) == 2, uint16_t, uint32_t>;
    unsigned char* w = static_cast<unsigned char*>(p->work);
    Args q;
    q.a = r.copyA ? reinterpret_cast<const T*>(w) : static_cast<const T*>(p->a);
    q.b = r.copyB ? reinterpret_cast<const T*>(w + r.bytesA) : static_cast<const T*>(p->b);
    q.c = static_cast<float*>(p->c);
    q.m = static_cast<int>(p->m);
    q.n = static_cast<int>(p->n);
    q.k = static_cast<int>(p->k);
    q.ka = static_cast<int>(r.ka);
    q.nb = static_cast<int>(r.nb);
    q.tilesM = (q.m + tileM - 1) / tileM;
    q.tilesN = (q.n + tileN - 1) / tileN;
    q.lda = r.copyA ? r.ka : p->lda;
    q.ldb = r.copyB ? r.nb : p->ldb;
    q.ldc = p->ldc;
    q.skip = p->skip_zero_a != 0 ? 1 : 0;
    if (r.copyA || r.copyB) {
        const RowCopy<Bits> a = {static_cast<const Bits*>(p->a), reinterpret_cast<Bits*>(w), p->m, p->k, p->lda, r.ka};
        const RowCopy<Bits> b = {static_cast<const Bits*>(p->b), reinterpret_cast<Bits*>(w + r.bytesA), p->k, p->n,
                                 p->ldb, r.nb};
        const int64_t v = 16 / static_cast<int64_t>(sizeof(T));
        const int64_t rows = std::max(r.copyA ? p->m : 0, r.copyB ? p->k : 0);
        const int64_t pieces = std::max(r.copyA ? r.ka / v : 0, r.copyB ? r.nb / v : 0);
        const dim3 grid(static_cast<unsigned>(std::min<int64_t>((pieces + 255) / 256, 64)),
                        static_cast<unsigned>(std::min<int64_t>(rows, 4096)), r.copyA && r.copyB ? 2 : 1);
        hipLaunchKernelGGL(copyRows<Bits>, grid, dim3(256), 0, st, r.copyA ? a : b, b);
    }
    return q;
}

int launchRagged(const mlkd_gemm* p, const RaggedPlan& r, hipStream_t st) {
    if (raiseLdsLimits() != 0) return MLKD_RT_LAUNCH;
    const bool acc = p->accumulate != 0;
    if (p->a_dtype == MLKD_F32) {
        const RaggedF32 q = raggedArgs<RaggedF32, float>(p, r, kFM, kFN, st);
        hipLaunchKernelGGL((acc ? RaggedDma{gemmF32Dma<true>} : RaggedDma{gemmF32Dma<false>}),
                           dim3(static_cast<unsigned>(q.tilesM * q.tilesN)), dim3(512), kLdsF32Dma, st, q);
    } else if (r.wide) {
        const RaggedF16Wide q = raggedArgs<RaggedF16Wide, _Float16>(p, r, kBM, kBN, st);
        hipLaunchKernelGGL((acc ? RaggedWide8s{gemmF16Dma8s<true>} : RaggedWide8s{gemmF16Dma8s<false>}),
                           dim3(static_cast<unsigned>(q.tilesM * q.tilesN)), dim3(512), kLdsDma, st, q);
    } else {
        const RaggedF16 q = raggedArgs<RaggedF16, _Float16>(p, r, kRM, kRN, st);
        hipLaunchKernelGGL((acc ? Ragged8s{gemmF16Dma8s<true>} : Ragged8s{gemmF16Dma8s<false>}),
                           dim3(static_cast<unsigned>(q.tilesM * q.tilesN)), dim3(256), kLdsRagged, st, q);
    }
    return hipGetLastError() == hipSuccess ? 0 : MLKD_RT_LAUNCH;
}

}  // namespace

extern "C" void mlkd_gemm_set_variant(int variant) { gGemmF16Variant = variant; }

extern "C" int64_t mlkd_gemm_pad_bytes(const mlkd_gemm* p) {
    if (p == nullptr || tiled(p)) return 0;
    RaggedPlan r;
    return raggedPlan(p, r) ? static_cast<int64_t>(r.bytesA + r.bytesB) : mlkdGemmGeneralBytes(p);
}

extern "C" void mlkd_gemm_tile(const mlkd_gemm* p, int64_t* rows, int64_t* cols) {
    RaggedPlan r;
    if (!raggedPlan(p, r)) return mlkdGemmGeneralTile(p, rows, cols);
    *rows = *cols = p->a_dtype == MLKD_F32 ? kFM : (r.wide ? kBM : kRM);
}

extern "C" const char* mlkd_gemm_kernel_name(const mlkd_gemm* p) {
    if (RaggedPlan r; raggedPlan(p, r) && roomFor(p, r)) {
        if (p->a_dtype == MLKD_F32) return p->accumulate != 0 ? "gemmF32Dma<true>" : "gemmF32Dma<false>";
        return p->accumulate != 0 ? "gemmF16Dma8s<true>" : "gemmF16Dma8s<false>";
    }
    const bool acc = p->accumulate != 0;
    switch (p->skip_zero_a != 0 && !acc ? -1 : mfmaForm(p)) {
        case 8:
            if (scalarAddressed8(p)) return acc ? "gemmF16Dma8s<true>" : "gemmF16Dma8s<false>";
            return acc ? "gemmF16Dma8<true>" : "gemmF16Dma8<false>";
        case 7: return acc ? "gemmF16Dma<true>" : "gemmF16Dma<false>";
        case 6: return acc ? "gemmF16Mfma2cu<true, false>" : "gemmF16Mfma2cu<false, false>";
        case 5: return acc ? "gemmF16Mfma2cu<true, true>" : "gemmF16Mfma2cu<false, true>";
        case 3: return acc ? "gemmF16Mfma4wPipe<true>" : "gemmF16Mfma4wPipe<false>";
        case 2: return acc ? "gemmF16Mfma4wDirect<true>" : "gemmF16Mfma4wDirect<false>";
        case 1: return acc ? "gemmF16Mfma4w<true>" : "gemmF16Mfma4w<false>";
        case 0: return acc ? "gemmF16Mfma<true>" : "gemmF16Mfma<false>";
        case 100: return acc ? "gemmF32Dma<true>" : "gemmF32Dma<false>";
        case 101: return acc ? "gemmF32Mfma<true>" : "gemmF32Mfma<false>";
        default: break;
    }
    return mlkdGemmGeneralName(p);
}

extern "C" int mlkd_launch_gemm(const mlkd_gemm* p, void* stream) {
    if (p == nullptr || p->m < 0 || p->n < 0 || p->k < 0) return MLKD_RT_LAUNCH;
    if (p->m == 0 || p->n == 0) return 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    // The MFMA forms take the skip-zero-A Call form themselves: a wave whose
    // accumulators met an infinity or a NaN recomputes its block exactly. One
    // launch, no scratch, no host read-back.
    if (tiled(p)) return launchMfma(p, mfmaForm(p), st);
    if (RaggedPlan r; raggedPlan(p, r) && roomFor(p, r)) return launchRagged(p, r, st);
    return mlkdLaunchGemmGeneral(p, st);
}
