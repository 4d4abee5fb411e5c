// Complex GEMM in FP32 on v_mfma_f32_16x16x4f32 with operands staged straight from memory into LDS: the
// design of zgemm64.hip (separate real and imaginary accumulators, two LDS buffers filled by
// global_load_lds while the other is multiplied) for complex64 operands and for complex128 ones that
// are rounded to FP32 as they leave LDS.
//
//   C (m x n) = alpha * op(A) * B + beta * C,   op(A) = A (m x k) or A^H (A stored k x m),
//   alpha, beta real, column-major interleaved; complex64 matrices 8-byte aligned, complex128 ones 16.
//
// A complex128 element is one 16-byte copy of a lane; a complex64 one two 4-byte copies, since a column of
// odd length leaves every other one only 8-byte aligned.  K stages are 16 complex (8 take less time to
// multiply than the next stage takes to arrive).  Slots are permuted by which lane fetches which
// element, so that the 32 lanes of a fragment read that the LDS serves at once spread over its banks:
// element p of matrix column `row` lies at p ^ swizzle(row), and of an A B product's A, rows of
// odd p have their blocks of 16 exchanged.
// ms before -> after (the register-staged 64 x 32 tiles of zgemm.hip): overlap 256 x 160 x 51,627 of complex64
// and complex128 0.250 -> 0.194, update 51,627 x 160 x 256 0.232 -> 0.202; with complex128 operands
// A^H B 96 x 48 x 51,627 0.083 -> 0.043, 864 x 440 x 80,927 3.81 -> 3.01, 32 x 48 x 4,607 0.019 ->
// 0.009, A B 1,000 x 40 x 3,000 0.089 -> 0.030.  The largest reach 80 to 119 TF/s of the 154 that the
// vendor's reach; within 15% whatever the tile, so neither the LDS nor the grid bounds them.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <iterator>
#include <type_traits>

#include "zgemm.h"
#include "zgemm_split.h"

namespace q3x {
namespace {

typedef float acc4 __attribute__((ext_vector_type(4)));
constexpr int KC = 16;  // complex k per stage

template <typename Z>
struct Elem {  // complex64
    static constexpr int lanes = 2;  // that copy one element
    static __device__ __forceinline__ int swizzle(int row) { return 2 * ((row >> 1) & 7); }
    static __device__ __forceinline__ void copy(const Z* src, int part, char* lds) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(&src->x + part),
                                         (__attribute__((address_space(3))) void*)lds, 4, 0, 0);
    }
    static __device__ __forceinline__ void put(const Z* src, int part, char* lds, int lane, bool in) {
        reinterpret_cast<float*>(lds)[lane] = in ? (&src->x)[part] : 0.0f;
    }
};
template <>
struct Elem<double2> {
    static constexpr int lanes = 1;
    static __device__ __forceinline__ int swizzle(int row) { return row & 15; }
    static __device__ __forceinline__ void copy(const double2* src, int, char* lds) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
    }
    static __device__ __forceinline__ void put(const double2* src, int, char* lds, int lane, bool in) {
        reinterpret_cast<double2*>(lds)[lane] = in ? *src : double2{0.0, 0.0};
    }
};
__device__ __forceinline__ float2 to_f32(float2 v) { return v; }
__device__ __forceinline__ float2 to_f32(double2 v) { return {static_cast<float>(v.x), static_cast<float>(v.y)}; }

template <typename ZA, typename ZB, typename ZC, int OPA, int TM, int TN, int WM, int WN>
__global__ void __launch_bounds__(256, 2)
    zgemm32_kernel(int m, int n, int k, int kchunk, const ZA* __restrict__ A, long lda, const ZB* __restrict__ B,
                   long ldb, ZC* __restrict__ C, long ldc, double alpha, double beta, float2* __restrict__ work,
                   int xmap) {
    static_assert(WM * WN == 4, "four waves");
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    constexpr int LA = Elem<ZA>::lanes, LB = Elem<ZB>::lanes;
    constexpr int QA = BM * KC * LA / 256, QB = BN * KC * LB / 256;  // copies per wave and stage
    constexpr int UNIT_A = 64 * sizeof(ZA) / LA, UNIT_B = 64 * sizeof(ZB) / LB;
    static_assert(BM * KC * LA % 256 == 0 && BN * KC * LB % 256 == 0, "whole copies");
    struct alignas(16) Stage {
        ZA a[BM * KC];
        ZB b[BN * KC];
    };
    __shared__ Stage S[2];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int li = lane & 15, lk = lane >> 4;
    // workgroup -> tile and K chunk: xmap 1 keeps the tiles of a K chunk on one XCD, xmap 2 the column
    // tiles of a row block
    int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    if (xmap == 1) {
        const int T = gridDim.x * gridDim.y;
        const int i = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
        const int r = i >> 3, t = r % T;
        bz = (i & 7) + 8 * (r / T);
        bx = t % gridDim.x;
        by = t / gridDim.x;
    } else if (xmap == 2) {
        const int i = blockIdx.x + gridDim.x * blockIdx.y;
        const int r = i >> 3;
        by = r % gridDim.y;
        bx = (i & 7) + 8 * (r / gridDim.y);
        if (bx * BM >= m) return;
    }
    const int m0 = bx * BM, n0 = by * BN;
    const int kbeg = bz * kchunk;
    const int kend = min(k, kbeg + kchunk);

    // LDS slots: of element p of row i
    auto slot_a = [](int i, int p) {
        if (OPA == 0) return p * BM + (LA == 2 ? i ^ ((p & 1) << 4) : i);
        return i * KC + (p ^ Elem<ZA>::swizzle(i));
    };
    auto slot_b = [](int i, int p) { return i * KC + (p ^ Elem<ZB>::swizzle(i)); };
    // and which element this lane's copies fetch
    auto element_a = [&](int q, int& i, int& p) {
        const int e = ((wave + 4 * q) * 64 + lane) / LA;
        if (OPA == 0) {
            p = e / BM;
            i = LA == 2 ? (e % BM) ^ ((p & 1) << 4) : e % BM;
        } else {
            i = e / KC;
            p = (e % KC) ^ Elem<ZA>::swizzle(i);
        }
    };
    auto element_b = [&](int q, int& i, int& p) {
        const int e = ((wave + 4 * q) * 64 + lane) / LB;
        i = e / KC;
        p = (e % KC) ^ Elem<ZB>::swizzle(i);
    };
    const ZA* sa[QA];
    const ZB* sb[QB];
#pragma unroll
    for (int q = 0; q < QA; ++q) {
        int i, p;
        element_a(q, i, p);
        i = min(m0 + i, m - 1);
        sa[q] = OPA == 0 ? A + i + (kbeg + p) * lda : A + kbeg + p + i * lda;
    }
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        int i, p;
        element_b(q, i, p);
        sb[q] = B + kbeg + p + min(n0 + i, n - 1) * ldb;
    }
    auto stage = [&](int buf, int k0) {
        char* la = reinterpret_cast<char*>(S[buf].a);
        char* lb = reinterpret_cast<char*>(S[buf].b);
        const int left = kend - k0;
        if (left >= KC) {
#pragma unroll
            for (int q = 0; q < QA; ++q) {
                Elem<ZA>::copy(sa[q], lane % LA, la + (wave + 4 * q) * UNIT_A);
                sa[q] += OPA == 0 ? KC * lda : KC;
            }
#pragma unroll
            for (int q = 0; q < QB; ++q) {
                Elem<ZB>::copy(sb[q], lane % LB, lb + (wave + 4 * q) * UNIT_B);
                sb[q] += KC;
            }
        } else {  // zeros past the end
#pragma unroll
            for (int q = 0; q < QA; ++q) {
                int i, p;
                element_a(q, i, p);
                Elem<ZA>::put(sa[q], lane % LA, la + (wave + 4 * q) * UNIT_A, lane, p < left);
            }
#pragma unroll
            for (int q = 0; q < QB; ++q) {
                int i, p;
                element_b(q, i, p);
                Elem<ZB>::put(sb[q], lane % LB, lb + (wave + 4 * q) * UNIT_B, lane, p < left);
            }
        }
    };

    acc4 cr[TM][TN], ci[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) cr[a][b] = ci[a][b] = acc4{0, 0, 0, 0};

    if (kbeg < kend) stage(0, kbeg);
    int buf = 0;
    for (int k0 = kbeg; k0 < kend; k0 += KC, buf ^= 1) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const ZA* as = S[buf].a;
        const ZB* bs = S[buf].b;
        constexpr int HK = 2;  // steps of four k whose fragments are read together
#pragma unroll
        for (int j0 = 0; j0 < KC / 4; j0 += HK) {
            float2 fa[HK][TM], fb[HK][TN];
#pragma unroll
            for (int j = 0; j < HK; ++j) {
                const int p = 4 * (j0 + j) + lk;
#pragma unroll
                for (int a = 0; a < TM; ++a) fa[j][a] = to_f32(as[slot_a((wm * TM + a) * 16 + li, p)]);
#pragma unroll
                for (int b = 0; b < TN; ++b) fb[j][b] = to_f32(bs[slot_b((wn * TN + b) * 16 + li, p)]);
            }
            if (j0 + HK == KC / 4 && k0 + KC < kend) stage(buf ^ 1, k0 + KC);
#pragma unroll
            for (int j = 0; j < HK; ++j) {
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b) {
                        cr[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][b].x, fa[j][a].x, cr[a][b], 0, 0, 0);
                        ci[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][b].y, fa[j][a].x, ci[a][b], 0, 0, 0);
                    }
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b) {
                        const float y = fa[j][a].y, yr = OPA == 0 ? -y : y, yi = OPA == 0 ? y : -y;
                        cr[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][b].y, yr, cr[a][b], 0, 0, 0);
                        ci[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][b].x, yi, ci[a][b], 0, 0, 0);
                    }
            }
        }
    }

    // lane li + 16 lk, register r of a tile: row li, column 4 lk + r.  C is read for a row of tiles at a
    // time, before any of it is written.
#pragma unroll
    for (int a = 0; a < TM; ++a) {
        const int gi = m0 + (wm * TM + a) * 16 + li;
        ZC old[TN][4];
        if (!work && beta != 0.0) {
#pragma unroll
            for (int b = 0; b < TN; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    old[b][r] = C[min(gi, m - 1) + min(n0 + (wn * TN + b) * 16 + 4 * lk + r, n - 1) * ldc];
        }
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gj = n0 + (wn * TN + b) * 16 + 4 * lk + r;
                if (gi >= m || gj >= n) continue;
                if (work) {
                    work[(static_cast<long>(bz) * n + gj) * m + gi] = float2{cr[a][b][r], ci[a][b][r]};
                } else {
                    ZC* c = C + gi + gj * ldc;
                    double2 out = {alpha * static_cast<double>(cr[a][b][r]), alpha * static_cast<double>(ci[a][b][r])};
                    if (beta != 0.0) {
                        out.x += beta * static_cast<double>(old[b][r].x);
                        out.y += beta * static_cast<double>(old[b][r].y);
                    }
                    *c = ZC{static_cast<decltype(c->x)>(out.x), static_cast<decltype(c->y)>(out.y)};
                }
            }
    }
}

template <typename ZA, typename ZB, typename ZC>
struct Problem {
    int m, n, k;
    double alpha;
    const ZA* A;
    long lda;
    const ZB* B;
    long ldb;
    double beta;
    ZC* C;
    long ldc;
    float2* work;
    size_t work_bytes;
    hipStream_t st;
};

// The tiles, with the workgroups resident on a CU by registers and the measured rates (4096^3 with
// complex128 operands).
constexpr Tile kTiles[] = {{45, 128, 80, KC, 2, 97.0}, {44, 128, 64, KC, 2, 103.0}, {42, 128, 32, KC, 3, 114.0},
                           {25, 64, 80, KC, 3, 116.0}, {24, 64, 64, KC, 3, 119.0},  {22, 64, 32, KC, 5, 111.0},
                           {21, 64, 16, KC, 6, 99.0},  {12, 32, 32, KC, 7, 98.0}};

template <int OPA, int TM, int TN, int WM, int WN, typename ZA, typename ZB, typename ZC>
hipError_t launch(const Problem<ZA, ZB, ZC>& g, int split) {
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    const int tm = (g.m + BM - 1) / BM, tn = (g.n + BN - 1) / BN;
    const long by_ws = g.work ? static_cast<long>(g.work_bytes / (8ull * g.m * g.n)) : 1;
    int ksplit = static_cast<int>(std::max(1L, std::min<long>({split, by_ws, std::max(1, g.k / KC)})));
    const bool by_xcd = ksplit % 8 == 0;
    int kchunk = (g.k + ksplit - 1) / ksplit;
    kchunk = std::max(1, (kchunk + KC - 1) / KC) * KC;
    if (!by_xcd) ksplit = g.k > 0 ? (g.k + kchunk - 1) / kchunk : 1;
    dim3 grid(tm, tn, ksplit);
    int xmap = by_xcd ? 1 : 0;
    if (OPA == 0 && ksplit == 1 && tn > 1) {
        xmap = 2;
        grid.x = (tm + 7) / 8 * 8;
    }
    hipLaunchKernelGGL((zgemm32_kernel<ZA, ZB, ZC, OPA, TM, TN, WM, WN>), grid, dim3(256), 0, g.st, g.m, g.n, g.k, kchunk,
                       g.A, g.lda, g.B, g.ldb, g.C, g.ldc, g.alpha, g.beta, ksplit > 1 ? g.work : nullptr, xmap);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || ksplit == 1) return e;
    const long total = static_cast<long>(g.m) * g.n;
    hipLaunchKernelGGL((splitk_sum<float2, ZC>), dim3(static_cast<unsigned>((total + 63) / 64)), dim3(256), 0, g.st, g.m,
                       total, ksplit, g.work, g.C, g.ldc, g.alpha, g.beta);
    return hipGetLastError();
}

template <int OPA, typename ZA, typename ZB, typename ZC>
hipError_t run(int tile, int split, int m, int n, int k, double alpha, const void* A, long lda, const void* B, long ldb,
               double beta, void* C, long ldc, void* work, size_t work_bytes, hipStream_t st) {
    const Problem<ZA, ZB, ZC> g{m, n, k, alpha, static_cast<const ZA*>(A), lda, static_cast<const ZB*>(B), ldb, beta,
                                static_cast<ZC*>(C), ldc, static_cast<float2*>(work), work_bytes, st};
    if (tile == 0 || split <= 0) {
        // K chunks are no longer than those of the 64 x 32 tiles of zgemm.hip (eight workgroups per CU),
        // so that no FP32 sum is; 256 x 160 x 51,627: rms error 5.7e-7, with 64 chunks 7.2e-7
        const long tiles = static_cast<long>((m + 63) / 64) * ((n + 31) / 32);
        const long most = work ? std::max(1L, static_cast<long>(work_bytes / (8ull * m * n))) : 1;
        const long by_k = OPA == 0 ? (tiles < 512 ? std::min((k + 511) / 512L, (1024 + tiles - 1) / tiles) : 1)
                                   : std::min<long>(k / 128, 2048 / tiles);
        long fewest = std::max(1L, std::min(most, by_k));
        if (fewest >= 8) fewest = std::min(most, (fewest + 7) / 8 * 8);  // whole rounds of the XCDs
        Tile table[std::size(kTiles)];
        for (size_t i = 0; i < std::size(kTiles); ++i) {
            table[i] = kTiles[i];
            const int lds = 2 * KC * static_cast<int>(table[i].bm * sizeof(ZA) + table[i].bn * sizeof(ZB));
            table[i].resident = std::min(table[i].resident, (160 << 10) / lds);
        }
        const Choice c = choose(table, tile, fewest, OPA == 0 ? fewest : most, 8, m, n, k, cu_count());
        tile = c.tile;
        split = c.split;
    }
    switch (tile) {
        case 45: return launch<OPA, 2, 5, 4, 1>(g, split);
        case 44: return launch<OPA, 4, 2, 2, 2>(g, split);
        case 42: return launch<OPA, 2, 2, 4, 1>(g, split);
        case 25: return launch<OPA, 1, 5, 4, 1>(g, split);
        case 24: return launch<OPA, 2, 2, 2, 2>(g, split);
        case 22: return launch<OPA, 2, 1, 2, 2>(g, split);
        case 21: return launch<OPA, 1, 1, 4, 1>(g, split);
        case 12: return launch<OPA, 1, 1, 2, 2>(g, split);
    }
    return hipErrorInvalidValue;
}

bool aligned(const void* p, unsigned bytes) { return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0; }

}  // namespace

bool zgemm32_has_tile(int tile) {
    return std::any_of(std::begin(kTiles), std::end(kTiles), [tile](const Tile& t) { return t.id == tile; });
}

bool zgemm32_takes(GemmTypes types, int opa, const void* A, const void* B, const void* C, const void* work) {
    if (!aligned(work, 8)) return false;
    switch (types) {
        case GemmTypes::F_D_F_F: return opa == 1 && aligned(A, 8) && aligned(B, 16) && aligned(C, 8);
        case GemmTypes::F_F_F_D: return opa == 0 && aligned(A, 8) && aligned(B, 8) && aligned(C, 16);
        case GemmTypes::D_D_F_D: return aligned(A, 16) && aligned(B, 16) && aligned(C, 16);
        default: return false;
    }
}

hipError_t zgemm32(int tile, int split, GemmTypes types, int opa, int m, int n, int k, double alpha, const void* A,
                   long lda, const void* B, long ldb, double beta, void* C, long ldc, void* work, size_t work_bytes,
                   hipStream_t st) {
    switch (types) {
        case GemmTypes::F_D_F_F:
            return run<1, float2, double2, float2>(tile, split, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, work,
                                                   work_bytes, st);
        case GemmTypes::F_F_F_D:
            return run<0, float2, float2, double2>(tile, split, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, work,
                                                   work_bytes, st);
        case GemmTypes::D_D_F_D:
            return opa == 0 ? run<0, double2, double2, double2>(tile, split, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                                                work, work_bytes, st)
                            : run<1, double2, double2, double2>(tile, split, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                                                work, work_bytes, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace q3x
