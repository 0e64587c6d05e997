// What the MFMA kernels (exl3_mfma.hip, exl3_wide.h) share: the windows of a decoded fragment, ordered sums, the order that
// a block's A rows are laid out in, and the dense linear's arguments.
#pragma once

#include "exl3_device.h"

namespace exl3 {

typedef float f4_t __attribute__((ext_vector_type(4)));

// Window of normalised position u' (bits [u'K, u'K + 16) of R, ring words shifted so that the fragment's first bit is bit 0),
// low 16 bits valid.
template <int K>
__device__ __forceinline__ uint32_t frag_window(const uint32_t* R, int up) {
    const int E = up * K + 16;
    const int IW = (E - 1) >> 5;
    const int SH = 32 * (IW + 1) - E;
    if (SH == 0) return R[IW];
    if (E - 16 >= 32 * IW) return R[IW] >> SH;
    return __builtin_amdgcn_alignbit(R[IW - 1], R[IW], SH);
}

// sum over b < n of q[b] (n >= 1), in order, with the loads issued 16 at a time (unconditionally: indices clamped to
// n - 1, so no branch splits a batch into separate round trips)
__device__ __forceinline__ float sum_ordered(const float* q, int n) {
    float v = 0.f;
    for (int b0 = 0; b0 < n; b0 += 16) {
        float t[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) t[i] = ldg(q + (b0 + i < n ? b0 + i : n - 1));
#pragma unroll
        for (int i = 0; i < 16; ++i) v += b0 + i < n ? t[i] : 0.f;
    }
    return v;
}

// ------------------------------------------------------------------------------------------------ dense linear
// A of a block of cnt rows (cnt * k / 8 units of 16 bytes, where the block's rows would lie): the unit holding k unit h
// (half of a 16-k block, see exl3_wide.h) of 16-k block kk of its row r.
__host__ __device__ __forceinline__ constexpr int64_t block_unit(int cnt, int kk, int h, int r) {
    return (int64_t)(2 * kk + h) * cnt + r;
}

// Element of column k in row r of such a block (kperm: the units of k-permuted fragments, K <= 5).
__host__ __device__ __forceinline__ constexpr int64_t unit_elem(int cnt, int k, int r, bool kperm) {
    const int q = (k >> 2) & 3, h = kperm ? q & 1 : q >> 1, hi = kperm ? q >> 1 : q & 1;
    return 8 * block_unit(cnt, k >> 4, h, r) + 4 * hi + (k & 3);
}

struct LinArgs {
    const _Float16* xh;                              // [S][m][k]
    const float* xsum;                               // [S][m][k / 128]
    const int32_t* sonb;                             // shard of each 128-column block (S > 1), else null
    int S;
    const uint32_t* tr;
    const uint16_t* svh;
    void* out;
    int64_t out_ld;
    float* part;                                     // null: the epilogue writes out; else [P][m][n], the splits' partials
    int m, k, n, nblk;
    int nrb, ncb, P, bps;                            // row blocks, 256-column blocks, k-splits of this launch, 128-blocks
                                                     // per split
    int p0;                                          // first split of this launch
    int f32;
    const int64_t* tab;                              // not null: an expert's addresses (ItemDesc::tab), its down projection
                                                     // in place of tr and svh
    const int32_t* rowmap;                           // not null: output row of each row
};

typedef void (*lin_fn)(LinArgs);

__device__ __forceinline__ void linear_store(const LinArgs& a, int row, int col, float v0, float v1) {
    if (a.f32) {
        float* o = reinterpret_cast<float*>(a.out) + (int64_t)row * a.out_ld + col;
        o[0] = v0;
        o[64] = v1;
    } else {
        uint16_t* o = reinterpret_cast<uint16_t*>(a.out) + (int64_t)row * a.out_ld + col;
        o[0] = f2h(v0);
        o[64] = f2h(v1);
    }
}

}  // namespace exl3
