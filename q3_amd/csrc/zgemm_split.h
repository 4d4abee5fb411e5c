// What the LDS-staged complex GEMMs (zgemm64.hip, zgemm32.hip) share: the choice of workgroup tile and K
// split, and the sum of the K chunks' partials.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

namespace q3x {
namespace {

// A workgroup tile: 32 r rows by 16 c columns under the number 10 r + c, K stage KC, workgroups resident
// on a CU (registers and LDS), and the rate of a product that fills the chip, TF/s.
struct Tile {
    int id, bm, bn, kc, resident;
    double rate;
};

// Which tile and K split a product takes: the pair with the least time by a model of one CU's MFMA,
// which is what the kernels are bound by.
//   - a CU runs c = ceil(tiles x splits / CUs) workgroups; its MFMA take c x stages x `mfma`,
//   - a workgroup alone needs `alone` per stage (the barrier and the fragment reads are not hidden,
//     and below 0.55 us the copy of the next stage is not either), resident ones overlap,
//   - each round of resident workgroups costs a prologue and an epilogue, and a split product the
//     traffic and launch of its reduction.
// The constants are measured.  A stage with one workgroup on a CU against its share with several, us: FP64
// 64 x 64 x 8 1.07 / 0.94, 64 x 80 x 8 1.32 / 1.17, 32 x 32 x 16 0.66 / 0.51; FP32 (16 deep) 64 x 64 1.34 / 1.21,
// 64 x 32 0.91 / 0.69, 32 x 32 0.67 / 0.35, 64 x 16 0.71 / 0.38, for which the model takes 0.55.
// only: 0, or the one tile to consider; fewest, most: bounds on the number of K chunks.
struct Choice {
    int tile, split;
};
template <int N>
Choice choose(const Tile (&table)[N], int only, long fewest, long most, int partial_bytes, int m, int n, int k, int cus) {
    Choice best{24, 1};
    double least = 0.0;
    for (const Tile& t : table) {
        if (only != 0 && t.id != only) continue;
        const long tiles = static_cast<long>((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn);
        const double mfma = 8e-6 * t.bm * t.bn * t.kc * cus / t.rate;
        const double alone = std::max(mfma + 0.17, 0.55);
        const long top = std::max(fewest, std::min<long>(most, k / (2 * t.kc)));
        for (int fill = 0; fill <= 12; ++fill) {  // 0: no split; else about fill / 2 + 1/2 workgroups per CU
            long ks = fill == 0 ? 1 : std::min(top, static_cast<long>((fill + 1) / 2) * cus / tiles);
            if (fill > 0 && ks < 2) continue;
            if (fill % 2 == 0 && ks >= 8) ks -= ks % 8;  // whole rounds of the XCDs
            ks = std::max(ks, fewest);
            const long stages = ((k + ks - 1) / ks + t.kc - 1) / t.kc;
            const long c = (tiles * ks + cus - 1) / cus, rounds = (c + t.resident - 1) / t.resident;
            double us = std::max(c * stages * mfma, rounds * stages * alone) + 2.5 * rounds;
            if (ks >= 8 && ks % 8) us *= 1.04;
            if (ks > 1) us += 5.0 + 2e-6 * partial_bytes * m * n * ks / 4.0;
            if (least == 0.0 || us < least) {
                least = us;
                best = {t.id, static_cast<int>(ks)};
            }
        }
    }
    return best;
}

int cu_count() {
    static std::atomic<int> cached{0};  // of the first device used; same value from any thread
    int n = cached.load();
    if (n == 0) {
        int dev = 0;
        (void)hipGetDevice(&dev);
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached.store(n);
    }
    return n;
}

// C = alpha * (sum of the partials) + beta * C.  Four threads an output, each summing a quarter of
// the K chunks in order with eight loads ahead of their adds, then the quarters in
// order.  W, Z: complex types of the partials and of C; the sum is FP64.
template <typename W, typename Z>
__global__ void __launch_bounds__(256) splitk_sum(int m, long total, int ksplit, const W* __restrict__ work,
                                                  Z* __restrict__ C, long ldc, double alpha, double beta) {
    __shared__ double2 part[3][64];
    const int q = threadIdx.x >> 6, l = threadIdx.x & 63;
    const long idx = static_cast<long>(blockIdx.x) * 64 + l;
    const int per = (ksplit + 3) / 4;
    int z = q * per;
    const int z1 = min(ksplit, z + per);
    double2 s = {0.0, 0.0};
    if (idx < total) {
        const W* w = work + idx;
        for (; z + 8 <= z1; z += 8) {
            W v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = w[(z + u) * total];
#pragma unroll
            for (int u = 0; u < 8; ++u) s.x += v[u].x, s.y += v[u].y;
        }
        if (z < z1) {
            W v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = w[min(z + u, z1 - 1) * total];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (z + u < z1) s.x += v[u].x, s.y += v[u].y;
        }
    }
    if (q > 0) part[q - 1][l] = s;
    __syncthreads();
    if (q > 0 || idx >= total) return;
#pragma unroll
    for (int u = 0; u < 3; ++u) s.x += part[u][l].x, s.y += part[u][l].y;
    Z* c = C + idx % m + idx / m * ldc;
    double2 out = {alpha * s.x, alpha * s.y};
    if (beta != 0.0) {
        out.x += beta * c->x;
        out.y += beta * c->y;
    }
    c->x = static_cast<decltype(c->x)>(out.x);
    c->y = static_cast<decltype(c->y)>(out.y);
}

}  // namespace
}  // namespace q3x
