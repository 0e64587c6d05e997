// Host-side choices of the wide-block kernels (exl3_wide.h): row blocks, k-splits, scratch. Plain C++ without device code.
// They follow from the shape alone, never from what the workspace holds: a call gives the same bits eager and captured.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace exl3 {

// Bytes that n elements take in a workspace request (Carve).
inline size_t carve_size(size_t n, size_t elem) { return (n * elem + 255) & ~(size_t)255; }

// The wide kernels address the A rows of a block (`rows` rows, k columns, fp16) by 32-bit offsets from its first byte, in a
// buffer resource of 2^31 - 1 bytes: loads past it return zero. Blocks are cut so that they stay inside.
constexpr bool a_span_ok(int64_t rows, int64_t k) { return 2 * rows * k <= 0x7FFFFFFF; }

// Waves per SIMD (workgroups of four waves per CU) that the kernels of blocks of 32 RG rows are compiled for.
constexpr int wide_occ(int RG, int K) { return RG == 8 ? 1 : RG == 4 ? 2 : RG == 2 ? (K <= 5 ? 3 : 2) : (K <= 5 ? 4 : 3); }

struct LinPlan {
    int RG, P, bps;                                  // row groups of 32 per block, k-splits, 128-blocks of k per split
};

// Row blocks of 32 RG rows that the dense linear has a kernel for, with S shards at K bits.
constexpr bool linear_block_built(int RG, int S, int K) { return RG != 4 || S == 1 || K <= 5; }

// Row block and k-splits P of a dense linear by estimated time: the workgroups spread over the CUs,
// each CU running up to `occ` at a time. Per 32-k step a CU with j workgroups takes kStepUs[RG][j] microseconds, a
// workgroup's start and end kEdgeUs[RG]; several splits add the partials (written once, read once by the reduce kernel)
// and that kernel's launch. Fitted to 878 measured points at K = 4 (1024 x 4096 .. 5376 x 21504, 16 .. 1024 rows, 1 .. 16
// splits): the point it picks is within 1 % of the best on average, 15 % at worst. Few rows and few columns want small
// blocks and many splits (4096 x 4096 at 48 rows: 32-row blocks, 8 splits 15.5 us, 64-row 16.4, 128-row 19.4), many rows
// the wide ones, which decode least (5376 -> 21504 at 2048 rows: 32 / 64 / 128 / 256-row blocks 888 / 616 / 488 / 445 us).
// kBits: the steps at K = 6 and 7 and at K = 8 against K = 4, fitted to 3891 points (1024 -> 3072 .. 5376 -> 21504, one and three
// shards, 12 .. 2048 rows): the point picked is within 0.3 and 0.5 % of the best on average, 9 % at worst; without them 0.7 and
// 2.6 %, 39 % at worst. 128-row blocks of several shards are not built for K > 5: their two A planes and the words spill
// 28 to 55 registers inside the loop (5376 -> 10752 of three shards, 512 rows, K = 7: 32 / 64 / 128 / 256-row blocks 186 / 133 /
// 189 / 117 us).
// `rg` > 0 asks for that row block (halved until there is one and the offsets of its A fit), `cap` bounds the splits.
inline LinPlan linear_plan(int64_t m, int64_t n, int64_t k, int S, int K, int rg, int64_t cap, int cus) {
    const int nblk = (int)(k / 128);
    const int occ[4] = {wide_occ(1, K), wide_occ(2, K), wide_occ(4, K), wide_occ(8, K)};
    static const float kStepUs[4][4] = {{0.29f, 0.52f, 0.77f, 0.84f}, {0.36f, 0.63f, 0.84f, 0.84f},
                                        {0.48f, 0.82f, 0.82f, 0.82f}, {0.75f, 0.75f, 0.75f, 0.75f}};
    static const float kEdgeUs[4] = {4.8f, 7.1f, 8.8f, 11.3f}, kPartUsPerMB[4] = {0.146f, 0.044f, 0.071f, 0.305f};
    static const float kBits[3][4] = {{1.f, 1.f, 1.f, 1.f}, {1.3f, 1.3f, 1.3f, 1.15f}, {1.6f, 1.45f, 1.45f, 0.95f}};
    const float* const bits = kBits[K <= 5 ? 0 : K <= 7 ? 1 : 2];
    const int64_t ncb = (n + 255) / 256;
    const int pmax = nblk / 2 > 1 ? nblk / 2 : 1;
    LinPlan best = {1, 1, nblk};
    float tb = 1e30f;
    for (int g = 0; g < 4; ++g) {
        if ((rg > 0 && rg != 1 << g) || !linear_block_built(1 << g, S, K)) continue;
        const int64_t rows = 32 << g, tiles = (m + rows - 1) / rows * ncb;
        for (int p = 1; p <= pmax && p <= cap; ++p) {
            const int bps = (nblk + p - 1) / p, P = (nblk + bps - 1) / bps;
            if (P != p || !a_span_ok(m < rows ? m : rows, 128LL * bps)) continue;
            const int64_t w = (tiles * P + cus - 1) / cus, full = w / occ[g], rem = w % occ[g];
            const float mb = (float)P * (float)m * (float)n * 4e-6f;
            float t = 4.f * bps * bits[g] * ((float)full * kStepUs[g][occ[g] - 1] + (rem ? kStepUs[g][rem - 1] : 0.f)) +
                      kEdgeUs[g] * (float)(full + (rem ? 1 : 0));
            if (P > 1) t += 3.f + (0.125f + kPartUsPerMB[g]) * mb;
            if (t < tb) {
                tb = t;
                best = {1 << g, P, bps};
            }
        }
    }
    return tb == 1e30f && rg > 1 ? linear_plan(m, n, k, S, K, rg / 2, cap, cus) : best;
}

// Scratch of a dense linear on the MFMA GEMM: transformed rows of S shards, their block sums, partials of P > 1 splits.
inline size_t linear_call_bytes(int64_t m, int64_t n, int64_t k, int S, int P) {
    return carve_size((size_t)S * m * k, 2) + carve_size((size_t)S * m * (k / 128), 4) +
           (P > 1 ? carve_size((size_t)P * m * n, 4) : 0);
}

// Plan of such a call, with at most the splits that cover the device with blocks of 16, 32 or 64 rows (bounds the partials)
// and that fit `most` bytes of scratch. False if not even one split fits.
inline bool linear_call_plan(int64_t m, int64_t n, int64_t k, int S, int K, int rg, int cus, size_t most, LinPlan* pl) {
    const int rs = m <= 16 ? 16 : m <= 32 ? 32 : 64;
    const int64_t ts = (m + rs - 1) / rs * ((n + 255) / 256);
    int64_t cap = ((m <= 32 ? 768 : 512) + ts - 1) / ts;
    while (cap > 1 && linear_call_bytes(m, n, k, S, (int)cap) > most) --cap;
    *pl = linear_plan(m, n, k, S, K, rg, cap, cus);
    return linear_call_bytes(m, n, k, S, pl->P) <= most;
}

// Whether five to eight rows (what the decode GEMV takes in one pass) run on the MFMA GEMM instead. The GEMV's time grows with
// the rows, the GEMM's three launches cost about 15 us on a small matrix, and its decode grows faster with K than the GEMV's. us,
// GEMV / GEMM, at K = 4: 5376 -> 21504 at 5 / 6 / 8 rows 29.9 / 23.6, 32.1 / 23.7, 37.3 / 24.0; 4096 -> 14336 at 6 / 8 rows
// 21.8 / 17.6, 25.9 / 18.0; 8192 x 8192 at 5 rows 19.2 / 18.1; 4096 -> 8192 at 8 rows 16.4 / 17.5. At K = 6 / 7 / 8 the line lies
// higher: 8192 x 8192 at 5 rows 19.6 / 21.9, 20.0 / 22.3, 20.6 / 23.2, at 7 rows 22.3 / 21.8, 22.3 / 22.2, 22.9 / 23.3;
// 4096 -> 14336 at 8 rows 26.5 / 20.5, 26.8 / 21.4, 26.8 / 21.9.
inline bool linear_few_rows(int64_t m, int64_t n, int64_t k, int K) {
    if (m < 5 || m > 8) return false;
    const int64_t least = (K <= 5 ? 200000000 : K == 6 ? 220000000 : K == 7 ? 290000000 : 340000000) / (m - 2);
    return k * n >= (least > 40000000 ? least : 40000000);
}

// Row block of the prefill MoE (M tokens, `npairs` rows over E experts, H -> I -> H; uniform K: 1 .. 8). 32 (one class, one
// launch per projection) up to 64 tokens, 160 where experts take few rows: forking the launches by class costs more there
// (10 to 25 us) than decoding the experts with more rows again; 64 where an expert takes 28 to 64 rows on average (and for
// K > 5, where 128 rows would spill), else 128. Per 32-k step a workgroup of 32 / 64 / 128 rows takes 0.21 / 0.28 / 0.41 us.
// `forced`: 32, 64 or 128 (where it may be taken), or 0.
inline int moe_wide_rows(int64_t M, int64_t E, int64_t npairs, int64_t H, int64_t I, int Kg, int Kd, int forced) {
    const double mean = (double)npairs / (double)E;
    int rows = E > 1 && (M <= 64 || (M <= 160 && mean <= 8)) ? 32 : (mean > 28 && mean <= 64) ? 64 : 128;
    if (forced == 32 || forced == 64 || forced == 128) rows = forced;
    if (rows == 128 && (Kg > 5 || Kd > 5)) rows = 64;
    while (rows > 32 && !a_span_ok(npairs < rows ? npairs : rows, H > I ? H : I)) rows /= 2;
    return rows;
}

// MFMA blocks of a call of npairs rows over E experts, at most: an expert's last block may hold few rows; with 32-row blocks
// and with 128-row ones whose remainder is cut (`whole`: it is not) there is one per 32 rows more.
inline int64_t moe_max_blocks(int64_t npairs, int64_t E, int rows, bool whole) {
    return npairs / (rows == 32 || (rows > 64 && !whole) ? 32 : 64) + (E < npairs ? E : npairs) + 1;
}

// Rows (1, 2 or 4) per workgroup of the router GEMV over [H, E] weights: a CU runs one workgroup at a time, in rounds of 256,
// and a workgroup of 1 / 2 / 4 rows takes 14.3 / 17 / 27.3 us at H = 7168, 5.3 / 6.4 / 11.4 at 2048 (its FMAs bind it from
// two rows on). 512 experts, H = 7168, with 1 / 2 / 4 rows: 8 rows 14.6 / 16.8 / 27.2 us, 64 rows 28.6 / 18.3 / 27.2, 96 rows
// 43 / 33.1 / 27.3.
inline int router_rows(int64_t M, int64_t E, int cus) {
    static const int kCost[3] = {5, 6, 10};
    int best = 1;
    int64_t least = INT64_MAX;
    for (int g = 0; g < 3; ++g) {
        const int64_t wg = (E + 63) / 64 * ((M + (1 << g) - 1) >> g), t = (wg + cus - 1) / cus * kCost[g];
        if (t < least) {
            least = t;
            best = 1 << g;
        }
    }
    return best;
}

}  // namespace exl3
