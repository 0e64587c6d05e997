// Grouped GEMM of the prefill MoE path at uniform K, in row blocks of up to 32 RG rows of one expert (exl3_wide.h).
//   gateup  workgroup per (block, 128-column block of I), full H: waves 0, 1 the gate columns, waves 2, 3 the up columns;
//           epilogue: affine, Hadamard * svh, act(gate, up) * suh_down, Hadamard -> the down input (fp16) and its block sums
//   down    workgroup per (block, 256-column block of H), full I; epilogue: affine, Hadamard * svh * w -> y rows
//   combine sums of every token's y rows in slot order -> output
// Up to 64 rows the waves run on their own (no barrier in the loop) and the decode is the bound: VALU 110 instructions per
// step of 64 columns x 32 k, four or three waves per SIMD. The former 16 / 32 / 64-row kernels staged A through the LDS with
// a barrier every second step and spent as many cycles waiting as decoding.
#include <type_traits>

#include "exl3_moe.h"
#include "exl3_moe_dev.h"
#include "exl3_runtime.h"
#include "exl3_wide.h"

namespace exl3 {

// RG: row groups of 32 in a block. Every class accumulates and reduces in the same order, so a row's result does not depend
// on the class its block falls into.

template <int K, int RG, int NPL, bool PL>
struct MoePipe {
    static constexpr bool kDirect = RG <= 2;
    typedef std::conditional_t<kDirect, DirectPipe<K, RG, PL>, WidePipe<K, kDirect ? 4 : RG, NPL, PL>> Pipe;
    static constexpr int kStage = kDirect ? 0 : WidePipe<K, kDirect ? 4 : RG, NPL, PL>::kStageBytes;
    static constexpr int kLoop = kStage + Pipe::kSlotBytes, kC = 32 * kWideCS * 4;
    static constexpr int kSmem = kLoop > kC ? kLoop : kC;
};

// This workgroup's block of class `cl` and column block (null: past the class's work). Ids go round robin over the 8 XCDs;
// an XCD takes a contiguous run of the class's (block, column block) pairs, so that a block's A rows stay in one L2 and
// every XCD has work when the class has fewer than 8 blocks (a dense MLP at 397 rows: three blocks of 128).
__device__ __forceinline__ const ItemDesc* moe_block(const MoeArgs& a, int cl, int ncb, int& nb) {
    const int T = a.cls_cnt[cl] * ncb, per = (T + 7) / 8, j = blockIdx.x >> 3, t = (blockIdx.x & 7) * per + j;
    if (j >= per || t >= T) return nullptr;
    const int idx = t / ncb;
    nb = t - idx * ncb;
    return a.blocks + a.cls_list[cl * a.max_blocks + idx];
}

template <int G>
__device__ __forceinline__ void zero_acc(f16_t (&acc)[G][2]) {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int n = 0; n < 2; ++n) acc[g][n] = f16_t{};
}

template <int K, int RG, bool PL>
__global__ __launch_bounds__(256, wide_occ(RG, K)) void moe_gateup_wide_kernel(MoeArgs a, int cl) {
    typedef MoePipe<K, RG, 2, PL> MP;
    __shared__ __attribute__((aligned(16))) char smem[MP::kSmem];
    __shared__ float rsum[2][32 * RG];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int nb;
    const ItemDesc* d = moe_block(a, cl, a.I / 128, nb);
    if (!d) return;
    const int cnt = d->cnt, p0 = d->p0, nblk = a.H / 128;
    for (int i = threadIdx.x; i < 2 * 32 * RG; i += 256) {   // the rows' sums (block sums in order)
        const int p = i / (32 * RG), m = i - p * (32 * RG);
        rsum[p][m] = sum_ordered(a.xsum + ((size_t)(p0 + (m < cnt ? m : cnt - 1)) * 2 + p) * nblk, nblk);
    }
    const int pw = wave >> 1;                                  // this wave's projection
    typename MP::Pipe L;
    L.nsteps = a.H / 32;
    L.lane = lane;
    L.setup_w(a.gu_tn, reinterpret_cast<uint32_t*>(smem + MP::kStage) + wave * 8 * MP::Pipe::TS,
              reinterpret_cast<const uint32_t*>(d->tab[3 * pw]), [&](int pair) { return nb * 8 + 4 * (wave & 1) + 2 * pair; });
    const auto plane = [&](int p) {
        return reinterpret_cast<const u32x4_t*>(a.xh + ((size_t)p0 * 2 + (size_t)p * cnt) * a.H);
    };
    if constexpr (MP::kDirect) {
        L.setup_a(cnt, plane(pw));
    } else {
        L.lds = reinterpret_cast<u32x4_t*>(smem);
        L.apl = pw;
        L.setup_a(cnt, plane);
    }
    float* C = reinterpret_cast<float*>(smem);
    f16_t acc[RG][2];
    bool stored = false;                                       // the accumulators are in C already
    if constexpr (RG == 1) {
        if (cnt <= 16) {
            f4_t acc16[4] = {};
            L.run16(cnt, acc16);
            store_tile16(C, acc16, wave, lane);
            stored = true;
        }
    }
    if (!stored) {
        zero_acc(acc);
        L.run(acc);
    }

    // per row group: the gate and up columns through LDS, eight lanes to a row
    constexpr int LR = 8, N = 32 / LR;
    const int rr = threadIdx.x / LR, sub = row_sub<LR>(lane), col = nb * 128 + 4 * sub;
    h2_t sg[N][2], su[N][2], sd[N][2];                         // fp16 pairs: as floats they would spill
    {
        const uint16_t *pg = reinterpret_cast<const uint16_t*>(d->tab[2]) + col,
                       *pu = reinterpret_cast<const uint16_t*>(d->tab[5]) + col,
                       *pd = reinterpret_cast<const uint16_t*>(d->tab[7]) + col;
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sg[i][j >> 1][j & 1] = __builtin_bit_cast(_Float16, ldg(pg + 4 * LR * i + j));
                su[i][j >> 1][j & 1] = __builtin_bit_cast(_Float16, ldg(pu + 4 * LR * i + j));
                sd[i][j >> 1][j & 1] = __builtin_bit_cast(_Float16, ldg(pd + 4 * LR * i + j));
            }
    }
    const bool tiled = a.Kd > 0, kp = a.Kd <= 5;               // the down kernel's A: block order (uniform K), or rows
    uint16_t* const ab = a.abuf + (size_t)p0 * a.I;
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        if (32 * rg >= cnt) break;                             // uniform
        if (rg > 0) __syncthreads();
        if (!stored) store_tile(C, acc[rg], wave, lane);
        __syncthreads();
        const int m = 32 * rg + rr;
        if (m >= cnt) continue;
        const float xg = kMul1C2 * rsum[0][m], xu = kMul1C2 * rsum[1][m];
        f4_t g[N], u[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            g[i] = *reinterpret_cast<const f4_t*>(&C[rr * kWideCS + 4 * LR * i + 4 * sub]);
            u[i] = *reinterpret_cast<const f4_t*>(&C[rr * kWideCS + 144 + 4 * LR * i + 4 * sub]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                g[i][j] = kMul1C1 * g[i][j] + xg;
                u[i][j] = kMul1C1 * u[i][j] + xu;
            }
        }
        fwht128_lanes<LR>(g, sub);
        fwht128_lanes<LR>(u, sub);
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float gv = (float)(_Float16)(g[i][j] * kRsqrt128 * (float)sg[i][j >> 1][j & 1]);
                const float uv = (float)(_Float16)(u[i][j] * kRsqrt128 * (float)su[i][j >> 1][j & 1]);
                const float av = (float)(_Float16)act_mul_dev(gv, uv, a.act, a.limit);
                g[i][j] = (float)(_Float16)(av * (float)sd[i][j >> 1][j & 1]);
            }
        fwht128_lanes<LR>(g, sub);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            uint32_t h[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const _Float16 hv = (_Float16)(g[i][j] * kRsqrt128);
                u[i][j] = (float)hv;
                h[j] = __builtin_bit_cast(uint16_t, hv);
            }
            const uint2 v = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
            if (tiled) {
                *reinterpret_cast<uint2*>(ab + unit_elem(cnt, col + 4 * LR * i, m, kp)) = v;
            } else {
                *reinterpret_cast<uint2*>(ab + (size_t)m * a.I + col + 4 * LR * i) = v;
            }
        }
        const float bs = row_sum128<LR>(u);
        if (sub == 0) a.asum[(size_t)(p0 + m) * (a.I / 128) + nb] = bs;
    }
}

template <int K, int RG, bool PL>
__global__ __launch_bounds__(256, wide_occ(RG, K)) void moe_down_wide_kernel(MoeArgs a, int cl) {
    typedef MoePipe<K, RG, 1, PL> MP;
    __shared__ __attribute__((aligned(16))) char smem[MP::kSmem];
    __shared__ float rsum[32 * RG];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nbH = a.H / 128;
    int nb;
    const ItemDesc* d = moe_block(a, cl, (nbH + 1) / 2, nb);
    if (!d) return;
    const int cnt = d->cnt, p0 = d->p0, nbI = a.I / 128, tn = a.H / 16, nhalf = 2 * nb + 1 < nbH ? 2 : 1;
    for (int m = threadIdx.x; m < 32 * RG; m += 256)
        rsum[m] = sum_ordered(a.asum + (size_t)(p0 + (m < cnt ? m : cnt - 1)) * nbI, nbI);
    typename MP::Pipe L;
    L.nsteps = a.I / 32;
    L.lane = lane;
    L.setup_w(tn, reinterpret_cast<uint32_t*>(smem + MP::kStage) + wave * 8 * MP::Pipe::TS,
              reinterpret_cast<const uint32_t*>(d->tab[6]), [&](int pair) {
                  const int ct = nb * 16 + 4 * wave + 2 * pair;
                  return ct < tn ? ct : tn - 2;                // a last half block: in-bounds loads, results unused
              });
    const auto plane = [&](int) { return reinterpret_cast<const u32x4_t*>(a.abuf + (size_t)p0 * a.I); };
    if constexpr (MP::kDirect) {
        L.setup_a(cnt, plane(0));
    } else {
        L.lds = reinterpret_cast<u32x4_t*>(smem);
        L.apl = 0;
        L.setup_a(cnt, plane);
    }
    float* C = reinterpret_cast<float*>(smem);
    f16_t acc[RG][2];
    bool stored = false;                                       // the accumulators are in C already
    if constexpr (RG == 1) {
        if (cnt <= 16) {
            f4_t acc16[4] = {};
            L.run16(cnt, acc16);
            store_tile16(C, acc16, wave, lane);
            stored = true;
        }
    }
    if (!stored) {
        zero_acc(acc);
        L.run(acc);
    }

    constexpr int LR = 4, N = 32 / LR;                         // lanes per 128-column half of a row
    const int rr = threadIdx.x / (2 * LR), half = (threadIdx.x / LR) & 1, sub = row_sub<LR>(lane);
    float sd[N][4];
    {
        const uint16_t* sv = reinterpret_cast<const uint16_t*>(d->tab[8]) + nb * 256 + 128 * (half < nhalf ? half : 0) + 4 * sub;
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) sd[i][j] = h2f(ldg(sv + 4 * LR * i + j));
    }
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        if (32 * rg >= cnt) break;                             // uniform
        if (rg > 0) __syncthreads();
        if (!stored) store_tile(C, acc[rg], wave, lane);
        const int m = 32 * rg + rr;
        const float w = a.pair_w[p0 + (m < cnt ? m : cnt - 1)];
        __syncthreads();
        if (m >= cnt || half >= nhalf) continue;
        const float sx = kMul1C2 * rsum[m];
        f4_t v[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            v[i] = *reinterpret_cast<const f4_t*>(&C[rr * kWideCS + 144 * half + 4 * LR * i + 4 * sub]);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i][j] = kMul1C1 * v[i][j] + sx;
        }
        fwht128_lanes<LR>(v, sub);
        float* dst = a.y + (size_t)(p0 + m) * a.H + nb * 256 + 128 * half + 4 * sub;
#pragma unroll
        for (int i = 0; i < N; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i][j] = v[i][j] * kRsqrt128 * sd[i][j] * w;
            *reinterpret_cast<f4_t*>(dst + 4 * LR * i) = v[i];
        }
    }
}

// out[t] = sum over t's slots in slot order of its y rows (fp32), four columns per thread. Its own launch rather than the
// last arriving down workgroup: counting rows into tokens cost every down workgroup a drain of write-through stores, an
// atomic round trip and the reads.
__global__ __launch_bounds__(256) void moe_combine_kernel(MoeArgs a) {
    const int ncb = (a.H + 1023) / 1024, t = blockIdx.x / ncb, c = 4 * ((blockIdx.x - t * ncb) * 256 + threadIdx.x);
    if (c >= a.H) return;
    f4_t v = {0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < a.slots; j0 += 8) {
        int pr[8];
        f4_t y[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) pr[j] = j0 + j < a.slots ? a.pair_of[t * a.slots + j0 + j] : -1;
#pragma unroll
        for (int j = 0; j < 8; ++j)                            // a missing slot reads pair 0's row and adds zero
            y[j] = ldg(reinterpret_cast<const f4_t*>(a.y + (size_t)(pr[j] >= 0 ? pr[j] : 0) * a.H + c));
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] += pr[j] >= 0 ? y[j][i] : 0.f;
    }
    if (a.out_f32) {
        float* o = reinterpret_cast<float*>(a.out) + (int64_t)t * a.out_ld + c;
        if (((uintptr_t)a.out & 15) == 0 && (a.out_ld & 3) == 0) {
            *reinterpret_cast<f4_t*>(o) = v;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = v[i];
        }
    } else {
        uint16_t* o = reinterpret_cast<uint16_t*>(a.out) + (int64_t)t * a.out_ld + c;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = f2h(v[i]);
    }
}

typedef void (*moe_wide_fn)(MoeArgs, int);

// PLANAR4 instantiations where that order differs from tile order (K = 3, 5, 6, 7); 128-row blocks for K <= 5 only (null: no
// such kernel)
#define EXL3_WIDE_PICK(KERNEL)                              \
    if (pl) {                                               \
        if (K == 3) return KERNEL<3, RG, true>;             \
        if (K == 5) return KERNEL<5, RG, true>;             \
        if constexpr (RG < 4) {                             \
            if (K == 6) return KERNEL<6, RG, true>;         \
            if (K == 7) return KERNEL<7, RG, true>;         \
        }                                                   \
    }                                                       \
    if constexpr (RG < 4) {                                 \
        if (K == 6) return KERNEL<6, RG, false>;            \
        if (K == 7) return KERNEL<7, RG, false>;            \
        if (K == 8) return KERNEL<8, RG, false>;            \
    }                                                       \
    switch (K) {                                            \
        case 1: return KERNEL<1, RG, false>;                \
        case 2: return KERNEL<2, RG, false>;                \
        case 3: return KERNEL<3, RG, false>;                \
        case 4: return KERNEL<4, RG, false>;                \
        case 5: return KERNEL<5, RG, false>;                \
        default: return nullptr;                            \
    }

template <int RG>
static moe_wide_fn pick_gateup(int K, bool pl) {
    EXL3_WIDE_PICK(moe_gateup_wide_kernel)
}
template <int RG>
static moe_wide_fn pick_down(int K, bool pl) {
    EXL3_WIDE_PICK(moe_down_wide_kernel)
}

static int launch_wide(const char* name, moe_wide_fn fn, const MoeArgs& a, int cl, int nblocks, int ncb, hipStream_t st) {
    if (!fn) return fail(EXL3_ERR_INVALID, "exl3_moe_forward: no kernel for blocks of %d rows at K=%d, %d", a.block_rows, a.Kg, a.Kd);
    EXL3_LAUNCH(name, fn, dim3((unsigned)((nblocks + 7) / 8 * 8 * ncb)), dim3(256), 0, st, a, cl);
    return EXL3_OK;
}

// gate|up or down of one row class: 0: blocks of up to 32 rows, 1: up to a.block_rows
int launch_gateup_wide(const MoeArgs& a, int cl, int nblocks, hipStream_t st) {
    moe_wide_fn fn = cl == 0 ? pick_gateup<1>(a.Kg, a.planar)
                   : a.block_rows > 64 ? pick_gateup<4>(a.Kg, a.planar) : pick_gateup<2>(a.Kg, a.planar);
    return launch_wide(cl == 0 ? "moe_gateup_wide_32" : "moe_gateup_wide_big", fn, a, cl, nblocks, a.I / 128, st);
}

int launch_down_wide(const MoeArgs& a, int cl, int nblocks, hipStream_t st) {
    moe_wide_fn fn = cl == 0 ? pick_down<1>(a.Kd, a.planar)
                   : a.block_rows > 64 ? pick_down<4>(a.Kd, a.planar) : pick_down<2>(a.Kd, a.planar);
    return launch_wide(cl == 0 ? "moe_down_wide_32" : "moe_down_wide_big", fn, a, cl, nblocks, (a.H / 128 + 1) / 2, st);
}

int launch_gateup_class(const MoeArgs& a, int cl, hipStream_t st) {
    return launch_wide("moe_gateup_wide", cl == 2 ? pick_gateup<2>(a.Kg, a.planar) : pick_gateup<1>(a.Kg, a.planar), a, cl,
                       a.max_blocks, a.I / 128, st);
}

int launch_down_class(const MoeArgs& a, int cl, hipStream_t st) {
    return launch_wide("moe_down_wide", cl == 2 ? pick_down<2>(a.Kd, a.planar) : pick_down<1>(a.Kd, a.planar), a, cl,
                       a.max_blocks, (a.H / 128 + 1) / 2, st);
}

int launch_moe_combine(const MoeArgs& a, hipStream_t st) {
    EXL3_LAUNCH("moe_combine", moe_combine_kernel, dim3((unsigned)((int64_t)((a.H + 1023) / 1024) * a.M)), dim3(256), 0,
                st, a);
    return EXL3_OK;
}

}  // namespace exl3
