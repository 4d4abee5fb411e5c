// FP64 complex GEMM on v_mfma_f64_16x16x4f64 with operands staged straight from memory into LDS.
//
//   C (m x n) = alpha * op(A) * B + beta * C,   op(A) = A (m x k) or A^H (A stored k x m),
//   alpha, beta real, column-major interleaved complex128, every matrix 16-byte aligned.
//
// A wave holds TM x TN tiles of 16 x 16 complex, the real and the imaginary part of each in its own
// accumulator: per four complex k,  Cr += ar br - ai bi  and  Ci += ar bi + ai br  (A^H: the
// products with ai change sign), four MFMA a tile from one 16-byte LDS read per fragment.  The
// operands are passed in the order (B, A), so that a lane's column of the MFMA result is a row of C
// and the 16 lanes of a quarter wave store 256 contiguous bytes.
//
// K runs in stages of KC complex over two LDS buffers.  A stage is copied by global_load_lds (16
// bytes a lane, 64 consecutive LDS slots a wave), which takes neither registers nor VALU issue:
// after the barrier that completes stage s, a wave reads its fragments of s, starts the copy of
// s + 1 and runs the MFMA of s, so the copy has a whole stage of MFMA to arrive.  Operands that are
// contiguous along k (B, and A of A^H B) are copied a row of KC per matrix column; the slot of
// element p in row i is p ^ (i mod min(KC, 16)), by permuting which lane fetches which element, so
// that the fragment reads (lanes walking rows at one p) spread over the banks.  Rows past m or n
// repeat the last one (their results are not stored); a last stage shorter than KC goes through
// registers with zeros past the end.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <iterator>

#include "zgemm.h"
#include "zgemm_split.h"

namespace q3x {
namespace {

typedef double acc4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void copy_to_lds(const double2* src, double2* lds) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

template <int OPA, int TM, int TN, int WM, int WN, int KC, int MINW>
__global__ void __launch_bounds__(256, MINW)
    zgemm64_kernel(int m, int n, int k, int kchunk, const double2* __restrict__ A, long lda,
                   const double2* __restrict__ B, long ldb, double2* __restrict__ C, long ldc, double alpha,
                   double beta, double2* __restrict__ work, int xmap) {
    static_assert(WM * WN == 4, "four waves");
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    constexpr int SW = (KC < 16 ? KC : 16) - 1;
    constexpr int UA = BM * KC / 64, UB = BN * KC / 64;  // wave copies per stage
    constexpr int NU = (UA + UB + 3) / 4;                // at most, per wave
    __shared__ double2 S[2][(BM + BN) * KC];             // A tile, then B tile
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int li = lane & 15, lk = lane >> 4;
    // workgroup -> tile and K chunk, as in zgemm.hip: xmap 1 keeps the tiles of a K chunk on one XCD,
    // xmap 2 the column tiles of a row block
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

    // this lane's element of copy unit u: A^H and B rows are matrix columns (k contiguous); A rows
    // of A B are one p over the tile's rows
    auto place = [&](int u, int& row, int& p) {
        if (OPA == 0 && u < UA) {
            const int e = u * 64 + lane;
            p = e / BM;
            row = e % BM;
        } else {
            const int e = (u < UA ? u : u - UA) * 64 + lane;
            row = e / KC;
            p = (e % KC) ^ (row & SW);
        }
    };
    const double2* src[NU];
#pragma unroll
    for (int q = 0; q < NU; ++q) {
        const int u = wave + 4 * q;
        int row, p;
        place(u, row, p);
        if (u < UA)
            src[q] = OPA == 0 ? A + min(m0 + row, m - 1) + (kbeg + p) * lda : A + kbeg + p + min(m0 + row, m - 1) * lda;
        else
            src[q] = B + kbeg + p + min(n0 + row, n - 1) * ldb;
    }
    auto stage_copy = [&](int buf) {
#pragma unroll
        for (int q = 0; q < NU; ++q) {
            const int u = wave + 4 * q;
            if (u < UA + UB) {
                copy_to_lds(src[q], &S[buf][u * 64]);
                src[q] += OPA == 0 && u < UA ? KC * lda : KC;
            }
        }
    };
    auto stage_tail = [&](int buf, int left) {  // left < KC complex k
#pragma unroll
        for (int q = 0; q < NU; ++q) {
            const int u = wave + 4 * q;
            if (u < UA + UB) {
                int row, p;
                place(u, row, p);
                S[buf][u * 64 + lane] = p < left ? *src[q] : double2{0.0, 0.0};
            }
        }
    };
    auto stage = [&](int buf, int k0) {
        if (kend - k0 >= KC)
            stage_copy(buf);
        else
            stage_tail(buf, kend - k0);
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
        const double2* as = S[buf];
        const double2* bs = S[buf] + BM * KC;
        // the fragments of HK steps of four k at a time; the copy of the next stage starts once the
        // last are read, so that no read waits for it
        constexpr int HK = TM * TN > 1 ? 2 : KC / 4;
#pragma unroll
        for (int j0 = 0; j0 < KC / 4; j0 += HK) {
            double2 fa[HK][TM], fb[HK][TN];
#pragma unroll
            for (int j = 0; j < HK; ++j) {
                const int p = 4 * (j0 + j) + lk;
#pragma unroll
                for (int a = 0; a < TM; ++a) {
                    const int row = (wm * TM + a) * 16 + li;
                    fa[j][a] = OPA == 0 ? as[p * BM + row] : as[row * KC + (p ^ (li & SW))];
                }
#pragma unroll
                for (int b = 0; b < TN; ++b) fb[j][b] = bs[((wn * TN + b) * 16 + li) * KC + (p ^ (li & SW))];
            }
            if (j0 + HK == KC / 4 && k0 + KC < kend) stage(buf ^ 1, k0 + KC);
#pragma unroll
            for (int j = 0; j < HK; ++j) {
                double na[TM];
#pragma unroll
                for (int a = 0; a < TM; ++a) na[a] = -fa[j][a].y;
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b) {
                        cr[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[j][b].x, fa[j][a].x, cr[a][b], 0, 0, 0);
                        ci[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[j][b].y, fa[j][a].x, ci[a][b], 0, 0, 0);
                    }
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b) {
                        const double yr = OPA == 0 ? na[a] : fa[j][a].y, yi = OPA == 0 ? fa[j][a].y : na[a];
                        cr[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[j][b].y, yr, cr[a][b], 0, 0, 0);
                        ci[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[j][b].x, yi, ci[a][b], 0, 0, 0);
                    }
            }
        }
    }

    // lane li + 16 lk, register r of a tile: row li, column 4 r + lk
#pragma unroll
    for (int a = 0; a < TM; ++a) {
        const int gi = m0 + (wm * TM + a) * 16 + li;
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gj = n0 + (wn * TN + b) * 16 + 4 * r + lk;
                if (gi >= m || gj >= n) continue;
                if (work) {
                    work[(static_cast<long>(bz) * n + gj) * m + gi] = double2{cr[a][b][r], ci[a][b][r]};
                } else {
                    double2* c = C + gi + gj * ldc;
                    double2 out = {alpha * cr[a][b][r], alpha * ci[a][b][r]};
                    if (beta != 0.0) {
                        out.x += beta * c->x;
                        out.y += beta * c->y;
                    }
                    *c = out;
                }
            }
    }
}

struct Problem {
    int opa, m, n, k;
    double alpha;
    const double2* A;
    long lda;
    const double2* B;
    long ldb;
    double beta;
    double2* C;
    long ldc;
    double2* work;
    size_t work_bytes;
    hipStream_t st;
};

// The tiles with their measured rates (4096^3: 72.6 TF/s with the two largest, against 61 and 50 TF/s for
// A B and A^H B by the register-staged kernel this took over from, and 76 for the vendor's).  What the
// model of them decides, ms before -> after: overlap 256 x 160 x 51,627 0.349 -> 0.262 (64 x 80, 96
// splits: three full workgroups per CU), update 51,627 x 160 x 256 0.340 -> 0.259 (128 x 32: 160 =
// 5 x 32 exactly); A^H B 864 x 440 x 80,927 6.50 -> 3.9; A^H B 32 x 48 x 4,607 0.019 -> 0.009, A B
// 4,607 x 48 x 96 0.026 -> 0.008 (there the small tiles spread the product over more CUs).
constexpr Tile kTiles[] = {{44, 128, 64, 8, 2, 72.6}, {42, 128, 32, 8, 3, 71.5}, {25, 64, 80, 8, 3, 71.5},
                           {24, 64, 64, 8, 4, 72.0},  {23, 64, 48, 16, 2, 69.0}, {22, 64, 32, 16, 3, 67.5},
                           {21, 64, 16, 16, 3, 61.5}, {12, 32, 32, 16, 4, 62.5}};

template <int OPA, int TM, int TN, int WM, int WN, int KC, int MINW>
hipError_t launch(const Problem& g, int split) {
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    const int tm = (g.m + BM - 1) / BM, tn = (g.n + BN - 1) / BN;
    const long by_ws = g.work ? static_cast<long>(g.work_bytes / (16ull * g.m * g.n)) : 1;
    int ksplit = static_cast<int>(std::max(1L, std::min<long>({split, by_ws, std::max(1, g.k / KC)})));
    // chunks of whole stages; a multiple of 8 of them stays that (those past the end of K are empty),
    // so that each goes to its XCD
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
    hipLaunchKernelGGL((zgemm64_kernel<OPA, TM, TN, WM, WN, KC, MINW>), grid, dim3(256), 0, g.st, g.m, g.n, g.k, kchunk,
                       g.A, g.lda, g.B, g.ldb, g.C, g.ldc, g.alpha, g.beta, ksplit > 1 ? g.work : nullptr, xmap);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || ksplit == 1) return e;
    const long total = static_cast<long>(g.m) * g.n;
    hipLaunchKernelGGL((splitk_sum<double2, double2>), dim3(static_cast<unsigned>((total + 63) / 64)), dim3(256), 0,
                       g.st, g.m, total, ksplit, g.work, g.C, g.ldc, g.alpha, g.beta);
    return hipGetLastError();
}

template <int OPA>
hipError_t by_tile(int tile, const Problem& g, int split) {
    switch (tile) {
        case 44: return launch<OPA, 4, 2, 2, 2, 8, 2>(g, split);
        case 42: return launch<OPA, 2, 2, 4, 1, 8, 2>(g, split);
        case 25: return launch<OPA, 1, 5, 4, 1, 8, 2>(g, split);
        case 24: return launch<OPA, 2, 2, 2, 2, 8, 2>(g, split);
        case 23: return launch<OPA, 1, 3, 4, 1, 16, 2>(g, split);
        case 22: return launch<OPA, 2, 1, 2, 2, 16, 2>(g, split);
        case 21: return launch<OPA, 1, 1, 4, 1, 16, 2>(g, split);
        case 12: return launch<OPA, 1, 1, 2, 2, 16, 2>(g, split);
    }
    return hipErrorInvalidValue;
}

}  // namespace

bool zgemm64_has_tile(int tile) {
    return std::any_of(std::begin(kTiles), std::end(kTiles), [tile](const Tile& t) { return t.id == tile; });
}

bool zgemm64_aligned(const void* A, const void* B, const void* C, const void* work) {
    return ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C) |
             reinterpret_cast<uintptr_t>(work)) & 15) == 0;
}

hipError_t zgemm64(int tile, int split, int opa, int m, int n, int k, double alpha, const void* A, long lda, const void* B,
                   long ldb, double beta, void* C, long ldc, void* work, size_t work_bytes, hipStream_t st) {
    const Problem g{opa, m, n, k, alpha, static_cast<const double2*>(A), lda, static_cast<const double2*>(B), ldb, beta,
                    static_cast<double2*>(C), ldc, static_cast<double2*>(work), work_bytes, st};
    if (tile == 0 || split <= 0) {
        // A B splits too: of few rows and columns and a long k it would else run on a few CUs (32 x 32 x 51,627
        // 2,057 -> 18 us, 160 x 160 x 51,627 2,074 -> 176 us, 320 x 160 x 320 15.5 -> 9.7 us)
        const long most = work ? static_cast<long>(work_bytes / (16ull * m * n)) : 1;
        const Choice c = choose(kTiles, tile, 1, most, 16, m, n, k, cu_count());
        tile = c.tile;
        split = c.split;
    }
    return opa == 0 ? by_tile<0>(tile, g, split) : by_tile<1>(tile, g, split);
}

}  // namespace q3x
