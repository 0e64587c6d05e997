// Wide-block kernels of the dense linear: 32 RG rows x 256 columns per workgroup (exl3_wide.h).
#include <type_traits>

#include "exl3_runtime.h"
#include "exl3_wide.h"

namespace exl3 {

// Tile of this workgroup: ids go round robin over the 8 XCDs; an XCD takes a contiguous run of the tiles (row blocks
// fastest, then column blocks, then k-splits), so that the workgroups it runs at a time share A rows and trellis words
// in its L2.
__device__ __forceinline__ bool wide_tile(const LinArgs& a, int& rb, int& nb, int& p) {
    const int T = a.nrb * a.ncb * a.P, per = (T + 7) / 8;
    const int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (t >= T) return false;
    rb = t % a.nrb;
    const int r = t / a.nrb;
    nb = r % a.ncb;
    p = r / a.ncb;
    return true;
}

// The partials of a block of up to 16 rows (store_tile16's layout), 64 columns from col0.
__device__ __forceinline__ void partials16(const LinArgs& a, int p, int r0, int cnt, int col0, int lane, const f4_t (&acc)[4],
                                           const float* rsum) {
    float* part = a.part + (size_t)p * a.m * a.n + (size_t)r0 * a.n + col0 + (lane & 15);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 4 * (lane >> 4) + i;
        const float sx = kMul1C2 * rsum[r];
        if (r < cnt) {
#pragma unroll
            for (int f = 0; f < 4; ++f) part[(size_t)r * a.n + 16 * f] = kMul1C1 * acc[f][i] + sx;
        }
    }
}

template <int K, int RG, int NPL>
__global__ __launch_bounds__(256, wide_occ(RG, K)) void linear_wide_kernel(LinArgs a) {
    constexpr bool kDirect = RG <= 2;
    typedef std::conditional_t<kDirect, DirectPipe<K, RG>, WidePipe<K, kDirect ? 4 : RG, NPL>> Pipe;
    constexpr int kStage = kDirect ? 0 : WidePipe<K, kDirect ? 4 : RG, NPL>::kStageBytes;
    constexpr int kLoop = kStage + Pipe::kSlotBytes, kC = 32 * kWideCS * 4;
    __shared__ __attribute__((aligned(16))) char smem[kLoop > kC ? kLoop : kC];
    __shared__ float rsum[NPL][32 * RG];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int rb, nb, p;
    if (!wide_tile(a, rb, nb, p)) return;
    const int r0 = rb * 32 * RG;
    const int cnt = a.m - r0 < 32 * RG ? a.m - r0 : 32 * RG;
    const int kb0 = (a.p0 + p) * a.bps, nkb = a.nblk - kb0 < a.bps ? a.nblk - kb0 : a.bps;
    const int tn = a.n / 16;
    const int nhalf = 2 * nb + 1 < a.n / 128 ? 2 : 1;
    int shard[NPL];                                  // shard of each plane (the block's 128-column half; in [0, S))
#pragma unroll
    for (int q = 0; q < NPL; ++q) {
        int v = 0;
        if (NPL > 1) {
            v = a.sonb[2 * nb + (q < nhalf ? q : 0)];
            v = v < 0 ? 0 : (v >= a.S ? a.S - 1 : v);
        }
        shard[q] = v;
    }
#pragma unroll
    for (int q = 0; q < NPL; ++q)
        for (int r = threadIdx.x; r < 32 * RG; r += 256)
            rsum[q][r] = sum_ordered(a.xsum + ((size_t)shard[q] * a.m + r0 + (r < cnt ? r : cnt - 1)) * a.nblk + kb0, nkb);
    Pipe L;
    L.nsteps = nkb * 4;
    L.lane = lane;
    L.setup_w(tn, reinterpret_cast<uint32_t*>(smem + kStage) + wave * 8 * Pipe::TS,
              (a.tab ? reinterpret_cast<const uint32_t*>(a.tab[6]) : a.tr) + (size_t)kb0 * 8 * tn * (8 * K), [&](int pair) {
                  const int ct = nb * 16 + 4 * wave + 2 * pair;
                  return ct < tn ? ct : tn - 2;      // a last half block: in-bounds loads, results unused
              });
    const int hw = wave >> 1;                        // the 128-column half of this wave's columns
    const auto plane = [&](int q) {
        const int sq = (NPL > 1 && q != 0) ? shard[NPL - 1] : shard[0];
        return reinterpret_cast<const u32x4_t*>(a.xh + ((size_t)sq * a.m + r0) * a.k) + block_unit(cnt, kb0 * 8, 0, 0);
    };
    if constexpr (kDirect) {
        L.setup_a(cnt, plane(NPL > 1 ? hw : 0));
    } else {
        L.lds = reinterpret_cast<u32x4_t*>(smem);
        L.apl = NPL > 1 ? hw : 0;
        L.setup_a(cnt, plane);
    }
    float* C = reinterpret_cast<float*>(smem);
    f16_t acc[RG][2];
    bool stored = false;                             // the accumulators are in C already
    if constexpr (RG == 1) {
        if (cnt <= 16) {
            f4_t acc16[4] = {};
            L.run16(cnt, acc16);
            if (a.part) {
                if (hw < nhalf) partials16(a, p, r0, cnt, nb * 256 + 64 * wave, lane, acc16, rsum[NPL > 1 ? hw : 0]);
                return;
            }
            store_tile16(C, acc16, wave, lane);
            stored = true;
        }
    }
    if (!stored) {
#pragma unroll
        for (int rg = 0; rg < RG; ++rg)
#pragma unroll
            for (int np = 0; np < 2; ++np) acc[rg][np] = f16_t{};
        L.run(acc);
    }
    if (a.part) {                                    // fp32 partials, affine applied
        if (hw >= nhalf) return;
        float* part = a.part + (size_t)p * a.m * a.n + (size_t)r0 * a.n + nb * 256 + 64 * wave + (lane & 31);
#pragma unroll
        for (int rg = 0; rg < RG; ++rg)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = 32 * rg + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                const float sx = kMul1C2 * rsum[NPL > 1 ? hw : 0][r];
                if (r < cnt) {
                    part[(size_t)r * a.n] = kMul1C1 * acc[rg][0][i] + sx;
                    part[(size_t)r * a.n + 32] = kMul1C1 * acc[rg][1][i] + sx;
                }
            }
        return;
    }
    // Per 32-row group through LDS: the accumulators' layout has a row's columns across lanes (12 single-rate VALU
    // operations per value for the transform); from LDS a quad of lanes takes a row half, five of seven stages in
    // registers.
    const int rr = threadIdx.x >> 3, half = (threadIdx.x >> 2) & 1, sub = row_sub<4>(lane);
    const int col = nb * 256 + 128 * half + 4 * sub;
    float sd[8][4];
    {
        const uint16_t* sv = (a.tab ? reinterpret_cast<const uint16_t*>(a.tab[8]) : a.svh) + (half < nhalf ? col : col - 128);
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) sd[i][j] = h2f(ldg(sv + 16 * i + j)) * kRsqrt128;
    }
    const bool vec = a.f32 ? ((uintptr_t)a.out & 15) == 0 && (a.out_ld & 3) == 0
                           : ((uintptr_t)a.out & 7) == 0 && (a.out_ld & 3) == 0;
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        if (rg > 0) __syncthreads();
        if (!stored) store_tile(C, acc[rg], wave, lane);
        __syncthreads();
        const int m = 32 * rg + rr;
        if (m >= cnt || half >= nhalf) continue;
        const int64_t orow = a.rowmap ? a.rowmap[r0 + m] : r0 + m;
        const float sx = kMul1C2 * rsum[NPL > 1 ? half : 0][m];
        f4_t v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] = *reinterpret_cast<const f4_t*>(&C[rr * kWideCS + 144 * half + 16 * i + 4 * sub]);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i][j] = kMul1C1 * v[i][j] + sx;
        }
        fwht128_lanes<4>(v, sub);
        if (a.f32) {
            float* o = reinterpret_cast<float*>(a.out) + orow * a.out_ld + col;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                f4_t y;
#pragma unroll
                for (int j = 0; j < 4; ++j) y[j] = v[i][j] * sd[i][j];
                if (vec) {
                    *reinterpret_cast<f4_t*>(o + 16 * i) = y;
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) o[16 * i + j] = y[j];
                }
            }
        } else {
            uint16_t* o = reinterpret_cast<uint16_t*>(a.out) + orow * a.out_ld + col;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                uint32_t y[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) y[j] = f2h(v[i][j] * sd[i][j]);
                if (vec) {
                    *reinterpret_cast<uint2*>(o + 16 * i) = make_uint2(y[0] | y[1] << 16, y[2] | y[3] << 16);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) o[16 * i + j] = (uint16_t)y[j];
                }
            }
        }
    }
}

// (null: no such kernel)
template <int RG, int NPL>
static lin_fn pick_wide(int K) {
    if constexpr (linear_block_built(RG, NPL, 8)) {
        if (K == 6) return linear_wide_kernel<6, RG, NPL>;
        if (K == 7) return linear_wide_kernel<7, RG, NPL>;
        if (K == 8) return linear_wide_kernel<8, RG, NPL>;
    }
    switch (K) {
        case 1: return linear_wide_kernel<1, RG, NPL>;
        case 2: return linear_wide_kernel<2, RG, NPL>;
        case 3: return linear_wide_kernel<3, RG, NPL>;
        case 4: return linear_wide_kernel<4, RG, NPL>;
        case 5: return linear_wide_kernel<5, RG, NPL>;
        default: return nullptr;
    }
}

lin_fn linear_wide_pick(int RG, int S, int K) {
    switch (RG) {
        case 1: return S > 1 ? pick_wide<1, 2>(K) : pick_wide<1, 1>(K);
        case 2: return S > 1 ? pick_wide<2, 2>(K) : pick_wide<2, 1>(K);
        case 4: return S > 1 ? pick_wide<4, 2>(K) : pick_wide<4, 1>(K);
        default: return S > 1 ? pick_wide<8, 2>(K) : pick_wide<8, 1>(K);
    }
}

}  // namespace exl3
