// Argument blocks of the grouped MoE kernels (device pointers into the caller's tensors and the workspace).
#pragma once

#include <stdint.h>

namespace exl3 {

constexpr int kMoeMaxExperts = 2048;   // expert tables per layer (routed + shared); the align kernel keeps 5 ints each in LDS
constexpr int kMoeSmallRows = 8;       // experts with at most this many rows in a call take the GEMV kernels
constexpr int kMfmaRows = 64;          // row block of the MFMA grouped GEMM with a per-tile K
constexpr int kWideRows = 128;         // largest row block with uniform K

// How an expert's rows are cut into MFMA blocks. Per-tile K: blocks of MB = 64 rows, row classes of up to 16, 32 and 64 rows
// (each runs its own kernel instance, so that small blocks get the register budget and occupancy of a small block).
// Uniform K (wide): blocks of MB = 32, 64 or 128 rows, classes 0: up to 32 rows, 1: more. With MB = 128 a remainder of up to
// 64 rows is cut into blocks of 32 (two 32-row blocks cost what one 128-row block does) unless `whole`: then it stays one
// block (a dense MLP, whose down projection takes its rows in blocks of MB). MB is a power of two (1: no blocks): a division cost
// the one-workgroup align kernel 0.6 of its 5 us.
constexpr int kRowClasses = 3;
struct BlockCut {
    int MB, wide, whole;
    // number of blocks of an expert with c rows
    __host__ __device__ int count(int c) const {
        const int full = c >> __builtin_ctz(MB), rem = c & (MB - 1);
        return full + (split(rem) ? (rem + 31) / 32 : rem > 0);
    }
    // block of the f-th of c rows: its first row and row count
    __host__ __device__ void locate(int c, int f, int& first, int& cnt) const {
        const int full = c & ~(MB - 1), rem = c - full;
        const int sz = f < full || !split(rem) ? MB : 32;
        first = f < full ? f & ~(MB - 1) : full + (sz == 32 ? (f - full) & ~31 : 0);
        cnt = c - first < sz ? c - first : sz;
    }
    __host__ __device__ int row_class(int cnt) const { return wide ? cnt > 32 : cnt <= 16 ? 0 : cnt <= 32 ? 1 : 2; }

private:
    __host__ __device__ bool split(int rem) const { return MB > 64 && !whole && rem <= 64; }
};

// A sorted pair's expert, its row in its MFMA block and the block's rows, in one word.
static_assert(kMoeMaxExperts <= 1 << 11 && kWideRows <= 1 << 7 && kMfmaRows <= 1 << 7, "pair word");
__host__ __device__ constexpr int pair_word(int e, int row, int cnt) { return e | row << 11 | (cnt - 1) << 18; }
__host__ __device__ constexpr int pair_expert(int w) { return w & 0x7FF; }
__host__ __device__ constexpr int pair_row(int w) { return w >> 11 & 0x7F; }
__host__ __device__ constexpr int pair_block_rows(int w) { return (w >> 18 & 0x7F) + 1; }

// One work unit of the GEMV kernels: up to 8 rows (pairs) of one expert, with everything a workgroup needs so that a
// single uniform load replaces the table lookups. Items past the last real one have cnt == 0.
struct alignas(256) ItemDesc {
    int32_t e, p0, cnt, pad;
    int32_t tok[8];                    // token of each row
    float w[8];                        // routing weight of each row (1 for the shared expert)
    int64_t tab[9];                    // the expert's (trellis, suh, svh) addresses for gate, up, down
    int64_t km[6];                     // (kmap, woff) addresses for gate, up, down when K is per tile
};
static_assert(sizeof(ItemDesc) == 256, "item descriptor layout");

struct RouteArgs {
    const int32_t* ids;
    const float* tw;
    int M, topk, slots, E, shared, MR;
    int* counts;                       // optional [E]
    int* n_items;                      // optional: items of <= MR rows
    ItemDesc* items;                   // optional [max_items]
    int max_items;
    const int64_t* tables;             // [9][E] (read when items are built)
    const int64_t* kmaps;              // [6][E] or null
    int use_mfma;                      // experts with more than MR rows -> blocks for the MFMA kernels
    BlockCut cut;                      // (MB a power of two; 1 without blocks)
    ItemDesc* blocks;                  // [max_blocks]
    int max_blocks;
    int* cls_list;                     // optional [kRowClasses][max_blocks]: block indices by row class
    int* cls_cnt;                      // [kRowClasses]
    int* pair_tok;
    float* pair_w;
    int* pair_of;
    int* pair_e;                       // optional [M * slots]: pair_word of each pair in sorted order, -1 past the
                                       // valid pairs
    int* tok_nvalid;                   // optional [M]: valid slots per token; tokens with none get a zero output row
    void* out;
    int64_t out_ld;
    int out_f32, H;
};

constexpr int kFusedRouteMaxE = 512;    // logits per row that the fused layer's in-layer routing handles (8 per lane)
constexpr int kFusedRouteMaxRows = 4;   // tokens up to which the routed entry point ranks inside the fused layer

struct MoeArgs {
    const uint16_t* x;
    int64_t x_ld;
    int M, H, I, topk, slots, E;
    const int32_t* ids;
    const float* tw;
    const int64_t* tables;             // [9][E]
    const int64_t* kmaps;              // [6][E] or null
    int uniform;                       // tables[i][e] == tb[i] + e * ts[i] for every entry (host-known layout)
    int64_t tb[9], ts[9];
    int Kg, Kd;                        // gate/up K, down K (0 = per-tile)
    int gu_tn;                         // tiles per tile-row of the gate and up trellises (uniform K): I / 16, or
                                       // 2 I / 16 for the reference's expert blob (gate and up tiles of a tile-row
                                       // side by side, up at gate + I / 16 tiles)
    int planar;                        // weights in PLANAR4 word order (the reference's blobs at K = 3, 5, 6, 7):
                                       // picks the kernels' PL instantiations (host side only)
    // routing from logits inside the fused layer (null: ids / tw hold the routing): softmax over logits (+ rbias)
    // -> top-k -> renormalised, picks written to ids_out / tw_out
    const float* logits;
    int64_t lg_ld;
    int n_logits;
    const float* rbias;
    int32_t* ids_out;
    float* tw_out;
    int act;
    float limit;
    int shared;
    int MR, max_items;
    // routing (workspace)
    int* n_items;
    const ItemDesc* items;
    const ItemDesc* blocks;            // MFMA row blocks (cnt == 0 past the last)
    int max_blocks;
    const int* cls_list;               // [kRowClasses][max_blocks] block indices by row class
    const int* cls_cnt;                // [kRowClasses] blocks per class
    _Float16* xh;                      // [pairs][2][H] transformed gate / up inputs of MFMA rows; uniform gate|up K:
                                       // per block [2][cnt * H] in block_unit order (exl3_mfma.h)
    float* xsum;                       // [pairs][2][H / 128] block sums of xh (the MFMA rows' affine term)
    float* asum;                       // [pairs][I / 128] block sums of abuf (MFMA rows)
    int* pair_tok;
    float* pair_w;
    int* pair_of;
    int* pair_e;                       // [pairs] pair_word of each pair in sorted order, -1 past the valid pairs
                                       // (MFMA path)
    int block_rows;                    // row block of the call's MFMA blocks (BlockCut::MB)
    int* tok_nvalid;                   // [M] valid slots per token
    int* cnt_tok;                      // [M][H/128] combine arrival counters
    // intermediates (workspace)
    uint16_t* abuf;                    // [pairs][I] fp16, Hadamard-domain down input (MFMA rows at uniform down K: per
                                       // block in block_unit order)
    float* y;                          // [pairs][H] fp32, weighted expert outputs (dense_P > 0: [dense_sets][M][H] down
                                       // partials)
    int dense_P;                       // > 0: one expert takes every token with weight 1 (a dense MLP) on the MFMA
                                       // path: k-splits of its down projection, which runs as a dense linear
    int dense_sets;                    // partials held: dense_P, or 1: the splits run one after another, the later ones
                                       // into xh's memory (a set's size; read no more by then), and add up
    float* part_gu;
    int* cnt_gu;
    int P_gu, nblk_h;
    float* part_d;
    int* cnt_d;
    int P_d, nblk_i;
    // output
    void* out;
    int64_t out_ld;
    int out_f32;
};

}  // namespace exl3
