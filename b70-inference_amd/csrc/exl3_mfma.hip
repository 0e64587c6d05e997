// Expert-sorted ragged grouped GEMM on fp16 MFMA for prefill-sized calls.
//
// Rows (token, expert pairs) are grouped by expert and cut into row blocks; in a prefill call every expert with rows gets
// blocks (no GEMV items). Per layer call:
//   pairs_had   transformed gate / up inputs of every block row, fp16(H128(fp16(x * suh)) / sqrt(128)), in the order the
//               gate|up kernel reads them, and their 128-blocks' sums (the codebook affine term)
//   gateup      workgroup per (block, 128-column block of I), full H: decode straight into MFMA B fragments (B holds
//               h = 1024 + bytesum; the affine is applied as c1 * acc + c2 * rowsum(A) in the epilogue), then the fused
//               activation / down-input epilogue (Hadamard * svh, act, * suh_d, Hadamard)
//   down        workgroup per (block, 256-column block of H), full I, epilogue Hadamard * svh_d * w, then the combine
// Uniform K runs in exl3_moe_wide.hip (blocks of up to 128 rows), per-tile K here (blocks of up to 64 rows: A staged
// through a four-stage LDS ring, weight words three steps ahead, one barrier every second step). Workgroup ids are laid
// out so that the column blocks of one row block run on one XCD (shared L2 for its A rows). The dense linear's input
// transform, plan and reduction are here too (its kernel: exl3_wide.hip).
// Semantics: the reference's GateUpDpasKernel / DownDpasKernel / moe_prefill (glm/xpu/csrc/exl3_moe.n128.sycl:
// 472-689, 868-916) and exllamav3's exl3_moe (ext-op-inventory.md:1060-1093).
#include "exl3_device.h"
#include "exl3_gemv.h"
#include "exl3_mfma.h"
#include "exl3_moe.h"
#include "exl3_moe_dev.h"
#include "exl3_plan.h"
#include "exl3_runtime.h"

namespace exl3 {

// ------------------------------------------------------------------------------------------------ input transform
// Eight consecutive fp16 values: one 16-byte load when the address allows it (a wave-uniform choice), else eight.
__device__ __forceinline__ h8_t load_h8(const uint16_t* p, bool vec) {
    if (vec) return __builtin_bit_cast(h8_t, ldg(reinterpret_cast<const u32x4_t*>(p)));
    h8_t v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = __builtin_bit_cast(_Float16, ldg(p + j));
    return v;
}

// B fragment (v_mfma_f32_16x16x32_f16 layout: lane L holds column n = L & 15, rows k = 8 (L >> 4) + j) of the 128-point
// Hadamard matrix H[K][N] = (-1)^popcount(K & N) for K in 32 ks + [0, 32), N in 16 nb + [0, 16). popcount(K & N)
// splits into popcount(k & n) (bits 0-3), bit 4 of k with bit 0 of nb, and bits 0-1 of ks with bits 1-2 of nb: the
// fragment is F_{nb & 1} (lane-dependent, bit 4 of k = L >> 5) times the sign S(ks, nb), a compile-time constant.
__device__ __forceinline__ h8_t had_fragment(int lane, int p) {
    const int n = lane & 15, k0 = 8 * (lane >> 4);
    h8_t f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int odd = (__builtin_popcount((unsigned)((k0 + j) & n)) + p * (lane >> 5)) & 1;
        f[j] = odd ? (_Float16)-1.0f : (_Float16)1.0f;
    }
    return f;
}
__host__ __device__ constexpr bool had_sign_neg(int ks, int nb) {
    return (((ks & 1) & ((nb >> 1) & 1)) ^ (((ks >> 1) & 1) & ((nb >> 2) & 1))) != 0;
}

// fp16(H128(A) / sqrt(128)) of one wave's 16 rows, A = fp16(x * s) in A-fragment layout (lane L: row L & 15, columns
// 32 ks + 8 (L >> 4) + j). The results go to the wave's LDS tile (16 x 128 fp16) and part[i] gets the sum of the fp16
// results of row 4 (L >> 4) + i over this lane's 8 columns (the caller reduces over the 16 lanes of a row). The signs of
// the base fragments sit in B (F, then -F), and four output tiles are in flight at a time: few enough registers for four
// waves per SIMD in the prefill's input transform, which waits on two memory round trips per job.
__device__ __forceinline__ void had16_rows(const h8_t (&A)[4], const h8_t (&F)[4], int lane, _Float16 (*tile)[136],
                                           float (&part)[4]) {
    const int m = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) part[i] = 0.f;
#pragma unroll
    for (int n0 = 0; n0 < 8; n0 += 4) {
        f4_t acc[4];
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            acc[n] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    A[ks], F[(n & 1) + (had_sign_neg(ks, n0 + n) ? 2 : 0)], acc[n], 0, 0, 0);
        }
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const _Float16 h = (_Float16)(acc[n][i] * kRsqrt128);
                part[i] += (float)h;
                tile[4 * g + i][16 * (n0 + n) + m] = h;
            }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ void had_fragments(int lane, h8_t (&F)[4]) {
    F[0] = had_fragment(lane, 0);
    F[1] = had_fragment(lane, 1);
    F[2] = -F[0];
    F[3] = -F[1];
}

// Sum of v over the 16 lanes of a row (lanes with equal L >> 4): quads, then the mirrored lane of the half row and row.
__device__ __forceinline__ float row16_sum(float v) {
#define EXL3_ROW_ADD(ctrl) \
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, false))
    EXL3_ROW_ADD(0xB1);
    EXL3_ROW_ADD(0x4E);
    EXL3_ROW_ADD(0x141);
    EXL3_ROW_ADD(0x140);
#undef EXL3_ROW_ADD
    return v;
}

// One wave per job (16 consecutive pairs of the expert-sorted order, 128-column block kb; jobs row group major, four
// per workgroup): every row's x block times its expert's suh_gate and suh_up, Hadamard / sqrt(128), fp16 (the GEMM
// inputs xh) and their block sums (xsum). Rows are independent here, so a job's rows may belong to several experts
// and no job is empty: the rows' tokens and experts come from the pair arrays in one round trip (no block
// descriptor), then x and the signs in the next. A fragments are fp16(x * suh) (packed fp16 multiplies, one rounding:
// the reference's fp16(x * suh)), the Hadamard is 8 output tiles x 4 k-steps of v_mfma_f32_16x16x32_f16 against the
// two base fragments (fp32 accumulation of exact +-x products), and the sums of the fp16-rounded outputs reduce over
// the 16 lanes of a row.
__global__ __launch_bounds__(256, 4) void pairs_had_kernel(MoeArgs a) {
    __shared__ __attribute__((aligned(16))) _Float16 s_out[4][16][136];    // per wave: 16 rows x 128 (+ pad)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nblk = a.H / 128, np = a.M * a.slots;
    const int job = 4 * blockIdx.x + wave, rg = job / nblk, kb = job - rg * nblk, r0 = 16 * rg;
    if (r0 >= np) return;                                    // past the last row group (uniform)
    const int m = lane & 15, g = lane >> 4;
    const int p = r0 + m < np ? r0 + m : np - 1;
    const int tok = a.pair_tok[p], pw = a.pair_e[p];
    const bool valid = r0 + m < np && pw >= 0;
    const uint32_t vmask = (uint32_t)__builtin_amdgcn_ballot_w64(valid) & 0xFFFFu;   // rows of this job to store
    if (vmask == 0) return;
    const int ec = valid ? pair_expert(pw) : 0;
    const uint16_t* sgn[2];
    if (a.uniform) {
        sgn[0] = reinterpret_cast<const uint16_t*>(a.tb[1] + (int64_t)ec * a.ts[1]);
        sgn[1] = reinterpret_cast<const uint16_t*>(a.tb[4] + (int64_t)ec * a.ts[4]);
    } else {
        sgn[0] = reinterpret_cast<const uint16_t*>(ldg(a.tables + (int64_t)1 * a.E + ec));
        sgn[1] = reinterpret_cast<const uint16_t*>(ldg(a.tables + (int64_t)4 * a.E + ec));
    }
    const uint16_t* xr = a.x + (int64_t)(valid ? tok : 0) * a.x_ld + kb * 128 + 8 * g;
    const bool vx = ((uintptr_t)a.x & 15) == 0 && (a.x_ld & 7) == 0;
    // x and both projections' signs in one round trip
    h8_t xv[4], sg[2][4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) xv[ks] = load_h8(xr + 32 * ks, vx);
#pragma unroll
    for (int proj = 0; proj < 2; ++proj) {
        const uint16_t* sv = sgn[proj] + kb * 128 + 8 * g;
        const bool vs = __builtin_amdgcn_ballot_w64(((uintptr_t)sv & 15) != 0) == 0;   // every row 16-byte aligned
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) sg[proj][ks] = load_h8(sv + 32 * ks, vs);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        sg[0][ks] = xv[ks] * sg[0][ks];                 // A fragments
        sg[1][ks] = xv[ks] * sg[1][ks];
    }
    h8_t F[4];
    had_fragments(lane, F);
#pragma unroll
    for (int proj = 0; proj < 2; ++proj) {
        float part[4];
        had16_rows(sg[proj], F, lane, s_out[wave], part);
        if (a.Kg > 0) {                                 // per block in block_unit order: lane = row, 16-byte units
            const int row = pair_row(pw), cnt = pair_block_rows(pw);
            u32x4_t* dst = reinterpret_cast<u32x4_t*>(a.xh + ((size_t)(r0 + m - row) * 2 + (size_t)proj * cnt) * a.H);
            const bool kp = a.Kg <= 5;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int u = lane + 64 * c, h = (u >> 4) & 1, kk = u >> 5;
                const _Float16* t = &s_out[wave][m][16 * kk];
                typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
                const u2_t lo = *reinterpret_cast<const u2_t*>(t + (kp ? 4 * h : 8 * h));
                const u2_t hi = *reinterpret_cast<const u2_t*>(t + (kp ? 4 * h + 8 : 8 * h + 4));
                if (valid) dst[block_unit(cnt, kb * 8 + kk, h, row)] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
            }
        } else
#pragma unroll
        for (int c = 0; c < 4; ++c) {                   // 16-byte row stores from the tile
            const int u = lane + 64 * c, rr = u >> 4, ch = u & 15;
            const u32x4_t v = *reinterpret_cast<const u32x4_t*>(&s_out[wave][rr][8 * ch]);
            if ((vmask >> rr) & 1)
                *reinterpret_cast<u32x4_t*>(a.xh + ((size_t)(r0 + rr) * 2 + proj) * a.H + kb * 128 + 8 * ch) = v;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float v = row16_sum(part[i]);
            if (m == 0 && ((vmask >> (4 * g + i)) & 1)) a.xsum[((size_t)(r0 + 4 * g + i) * 2 + proj) * nblk + kb] = v;
        }
        __builtin_amdgcn_wave_barrier();                // the tile is rewritten by the next projection
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// Block id and column block of this workgroup under the XCD-aware layout (ids round-robin over 8 XCDs).
__device__ __forceinline__ void xcd_map(int nbc, int& blk, int& nb) {
    const int id = blockIdx.x, xcd = id & 7, j = id >> 3;
    const int q = j / nbc;
    blk = 8 * q + xcd;
    nb = j - q * nbc;
}

// ------------------------------------------------------------------------------------------------ per-tile-K loop
constexpr int kMfT = 4;                              // tile columns per wave

// Workgroups per CU (= waves per SIMD) the per-tile-K kernels are compiled for, by row class (1, 2 or 4 row groups of 16);
// the 1-row-group kernels run five (96 VGPRs), their epilogue buffer aliasing the pipeline's LDS so that five fit.
#ifndef EXL3_MIX_OCC1
#define EXL3_MIX_OCC1 5
#endif
#define EXL3_MIX_OCC(RGA) ((RGA) == 1 ? EXL3_MIX_OCC1 : (RGA) == 2 ? 3 : 2)

// 16-byte unit of (row, chunk) in one staged A plane (16 * RGA rows x four 16-byte chunks = 32 k); the chunk is
// swizzled by row so that the 16 rows of a fragment read hit distinct banks.
__device__ __forceinline__ int a_unit(int row, int ch) { return row * 4 + (ch ^ ((row >> 1) & 3)); }

typedef __attribute__((address_space(3))) const uint32_t* lds_cu32_t;
constexpr int kBufferWord3 = 0x00020000;                     // buffer resource word 3 for raw 32-bit loads (gfx9)
// A wave-uniform buffer resource over `p` (loads at offsets below 2^31 bytes; beyond the range they return zero).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0x7fffffff, kBufferWord3);
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// ------------------------------------------------------------------------------------------------ gate | up
template <int RGA>
__device__ __forceinline__ void gateup_epilogue(const MoeArgs& a, const ItemDesc* d, int nb, int cnt,
                                                const f4_t (&acc)[kMfT][RGA], float* C, const float* rsum);
template <int RGA>
__device__ __forceinline__ void down_epilogue(const MoeArgs& a, const ItemDesc* d, int nb, int cnt,
                                              const f4_t (&acc)[kMfT][RGA], float* C, const float* rsum, int* s_comb);

// Affine, Hadamard * svh, act(g, u) * suh_d, Hadamard of the workgroup's 128 columns per 16-row group -> abuf (fp16)
// and its block sums (the down GEMM's affine term).
template <int RGA>
__device__ __forceinline__ void gateup_epilogue(const MoeArgs& a, const ItemDesc* d, int nb, int cnt,
                                                const f4_t (&acc)[kMfT][RGA], float* C, const float* rsum) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p0 = d->p0;
    const uint16_t* svg = reinterpret_cast<const uint16_t*>(d->tab[2]) + nb * 128;
    const uint16_t* svu = reinterpret_cast<const uint16_t*>(d->tab[5]) + nb * 128;
    const uint16_t* sud = reinterpret_cast<const uint16_t*>(d->tab[7]) + nb * 128;
    const float sg0 = h2f(ldg(svg + lane)), sg1 = h2f(ldg(svg + lane + 64));
    const float su0 = h2f(ldg(svu + lane)), su1 = h2f(ldg(svu + lane + 64));
    const float sd0 = h2f(ldg(sud + lane)), sd1 = h2f(ldg(sud + lane + 64));
    const int nbI = a.I / 128;
#pragma unroll
    for (int rg = 0; rg < RGA; ++rg) {
        // this row group's gate / up columns of the whole workgroup -> C[2][16][128]; wave w holds projection w >> 1,
        // tile columns 4 (w & 1) .. + 3 of the block
#pragma unroll
        for (int t = 0; t < kMfT; ++t) {
            const int p = wave >> 1, col = (4 * (wave & 1) + t) * 16 + (lane & 15);
#pragma unroll
            for (int i = 0; i < 4; ++i) C[(p * 16 + 4 * (lane >> 4) + i) * 128 + col] = acc[t][rg][i];
        }
        __syncthreads();
        for (int j = 0; j < 4; ++j) {
            const int ml = 4 * wave + j, m = 16 * rg + ml;
            if (m >= cnt) break;
            const float sg = kMul1C2 * rsum[m], su = kMul1C2 * rsum[64 + m];
            float g0 = kMul1C1 * C[ml * 128 + lane] + sg, g1 = kMul1C1 * C[ml * 128 + lane + 64] + sg;
            float u0 = kMul1C1 * C[(16 + ml) * 128 + lane] + su, u1 = kMul1C1 * C[(16 + ml) * 128 + lane + 64] + su;
            fwht128_wave(g0, g1, lane);
            fwht128_wave(u0, u1, lane);
            g0 = (float)(_Float16)(g0 * kRsqrt128 * sg0);
            g1 = (float)(_Float16)(g1 * kRsqrt128 * sg1);
            u0 = (float)(_Float16)(u0 * kRsqrt128 * su0);
            u1 = (float)(_Float16)(u1 * kRsqrt128 * su1);
            float a0 = (float)(_Float16)act_mul_dev(g0, u0, a.act, a.limit);
            float a1 = (float)(_Float16)act_mul_dev(g1, u1, a.act, a.limit);
            a0 = (float)(_Float16)(a0 * sd0);
            a1 = (float)(_Float16)(a1 * sd1);
            fwht128_wave(a0, a1, lane);
            const _Float16 h0 = (_Float16)(a0 * kRsqrt128), h1 = (_Float16)(a1 * kRsqrt128);
            if (a.Kd > 0) {                           // uniform down K: the block in block_unit order
                uint16_t* dst = a.abuf + (size_t)p0 * a.I + unit_elem(cnt, nb * 128 + lane, m, a.Kd <= 5);
                dst[0] = __builtin_bit_cast(uint16_t, h0);
                dst[8 * block_unit(cnt, 4, 0, 0)] = __builtin_bit_cast(uint16_t, h1);   // 64 columns on
            } else {
                uint16_t* dst = a.abuf + (size_t)(p0 + m) * a.I + nb * 128;
                dst[lane] = __builtin_bit_cast(uint16_t, h0);
                dst[lane + 64] = __builtin_bit_cast(uint16_t, h1);
            }
            const float bs = wave_sum_f32((float)h0 + (float)h1);
            if (lane == 0) a.asum[(size_t)(p0 + m) * nbI + nb] = bs;
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------------------------ down
// 256 output columns per workgroup (two Hadamard blocks): wave w owns tile columns 4w .. 4w + 3.
// Affine, Hadamard * svh_d * w of the workgroup's 256 columns per 16-row group -> y rows, then the combine.
template <int RGA>
__device__ __forceinline__ void down_epilogue(const MoeArgs& a, const ItemDesc* d, int nb, int cnt,
                                              const f4_t (&acc)[kMfT][RGA], float* C, const float* rsum, int* s_comb) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p0 = d->p0;
    const int nbH = a.H / 128;
    const int nhalf = 2 * nb + 1 < nbH ? 2 : 1;
    const uint16_t* svd = reinterpret_cast<const uint16_t*>(d->tab[8]) + nb * 256;
    float sd[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int hh = h < nhalf ? h : 0;                // unconditional load, unused past nhalf
        sd[h][0] = h2f(ldg(svd + 128 * hh + lane));
        sd[h][1] = h2f(ldg(svd + 128 * hh + lane + 64));
    }
    // row weights of this wave's rows 16 rg + 4 wave + r, all loaded before the first is needed
    float wr[RGA][4];
#pragma unroll
    for (int rg = 0; rg < RGA; ++rg)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = 16 * rg + 4 * wave + r;
            wr[rg][r] = a.pair_w[p0 + (m < cnt ? m : cnt - 1)];
        }
#pragma unroll
    for (int rg = 0; rg < RGA; ++rg) {
#pragma unroll
        for (int t = 0; t < kMfT; ++t) {
            const int col = (4 * wave + t) * 16 + (lane & 15);
#pragma unroll
            for (int i = 0; i < 4; ++i) C[(4 * (lane >> 4) + i) * 256 + col] = acc[t][rg][i];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; ++j) {                 // (row, half) pairs of this wave
            const int ml = 4 * wave + (j >> 1), h = j & 1, m = 16 * rg + ml;
            if (m >= cnt || h >= nhalf) continue;
            const float sx = kMul1C2 * rsum[m];
            float v0 = kMul1C1 * C[ml * 256 + 128 * h + lane] + sx, v1 = kMul1C1 * C[ml * 256 + 128 * h + lane + 64] + sx;
            fwht128_wave(v0, v1, lane);
            const float w = wr[rg][j >> 1];
            float* dst = a.y + (size_t)(p0 + m) * a.H + nb * 256 + 128 * h;
            splitk_store(dst + lane, v0 * kRsqrt128 * sd[h][0] * w);
            splitk_store(dst + lane + 64, v1 * kRsqrt128 * sd[h][1] * w);
        }
        __syncthreads();
    }
    // combine: count rows into their tokens per 128-column block, finish tokens whose slots are all in
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * cnt; i += 256) {
        const int m = i >> 1, h = i & 1;
        int r = -1;
        if (h < nhalf) {
            const int t = a.pair_tok[p0 + m];
            const int old = __hip_atomic_fetch_add(&a.cnt_tok[(size_t)t * nbH + 2 * nb + h], 1, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
            r = (old == a.tok_nvalid[t] - 1) ? t : -1;
        }
        s_comb[i] = r;
    }
    __syncthreads();
    for (int i = wave; i < 2 * cnt; i += 4)
        if (s_comb[i] >= 0) combine_token(a, s_comb[i], 2 * nb + (i & 1), lane);
}

// ------------------------------------------------------------------------------------------------ per-tile K
// Per-tile bitrate (K = 0: tile i of a projection holds 8 kmap[i] words at woff[i]). Each lane decodes 4 k of one
// tile, so the 64 lanes of a wave always share one tile and its K is wave-uniform. Fragment layout (16x16x16): B[k][n]
// lane L holds n = L & 15, k = 4 (L >> 4) + j, j < 4; A[m][k] lane L holds m = L & 15, same k; D[m][n] n = L & 15,
// m = 4 (L >> 4) + i (the tile rows behind the k slots are permuted, see decode4p). Steps whose tiles are all K <= 2
// join the two tile-rows of a column in one 16x16x32 MFMA (8 k per lane: 4 of each tile).
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
constexpr int kMixKMax = 8;
constexpr int kMixTS = 8 * kMixKMax + 4;                    // LDS words per staged tile: 3 pad, w(8K - 1), 64 words

// k-permuted fragments. An MFMA sums over k, so B and A may list a tile-row's 16 k in any common order. In the order
// used here lane L's four k slots are tile rows 2g, 2g + 1, 2g + 8, 2g + 9 (g = L >> 4) of column n = L & 15: the
// positions t0 .. t0 + 3, t0 = 32 (n & 7) + 4 (n >> 3) + 8 g, four consecutive windows (row 8 ((t >> 1) & 1) +
// 2 ((t >> 3) & 3) + (t & 1), column (t >> 5) + 8 ((t >> 2) & 1)). Their bits [(t0 + 1) K - 16, (t0 + 4) K) fit one
// funnel-shifted word for K <= 5: window b sits at bit 16 - b K of it.
// Seen from 3 words into a staged slot (v = slot + 3): v[0] = ring word 8K - 1, v[1 + w] = ring word w. A funnel whose
// first bit is ring bit `start` (>= -16) reads v[(start + 31) >> 5] and the next word, shifted by
// 31 - ((start + 31) & 31). The windows of positions t <= 255 end inside the ring, so a funnel's second word may lie
// past it (any value: none of its bits is used).
__device__ __forceinline__ h4_t decode4p(uint32_t F, int K) {
    const uint32_t w0 = F >> 16;
    const uint32_t w1 = __builtin_amdgcn_ubfe(F, 16 - K, 16);
    const uint32_t w2 = __builtin_amdgcn_ubfe(F, 16 - 2 * K, 16);
    const uint32_t w3 = __builtin_amdgcn_ubfe(F, 16 - 3 * K, 16);
    typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
    const u2_t v = {__builtin_bit_cast(uint32_t, mul1_pair_raw(w0, w1)),
                    __builtin_bit_cast(uint32_t, mul1_pair_raw(w2, w3))};
    return __builtin_bit_cast(h4_t, v);
}

// K = 2 (k2) or 1: decode4p with the window offsets as constants picked by a wave-uniform flag.
__device__ __forceinline__ h4_t decode4p12(uint32_t F, bool k2) {
    const uint32_t w0 = F >> 16;
    const uint32_t w1 = __builtin_amdgcn_ubfe(F, k2 ? 14 : 15, 16);
    const uint32_t w2 = __builtin_amdgcn_ubfe(F, k2 ? 12 : 14, 16);
    const uint32_t w3 = __builtin_amdgcn_ubfe(F, k2 ? 10 : 13, 16);
    typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
    const u2_t v = {__builtin_bit_cast(uint32_t, mul1_pair_raw(w0, w1)),
                    __builtin_bit_cast(uint32_t, mul1_pair_raw(w2, w3))};
    return __builtin_bit_cast(h4_t, v);
}

// Any K (1 .. 8): the funnel origin from the lane's t0 + 1 at run time, and a second funnel for windows 2 and 3.
__device__ __forceinline__ h4_t decode4p_rt(const uint32_t* slot, int K, uint32_t t0p1) {   // slot: v above
    const uint32_t ta = t0p1 * (uint32_t)K + 15u, tb = ta + 2u * (uint32_t)K;     // start + 31 of windows 0 and 2
    const uint32_t* pa = slot + (ta >> 5);
    const uint32_t* pb = slot + (tb >> 5);
    const uint32_t Fa = __builtin_amdgcn_alignbit(pa[0], pa[1], ~ta);
    const uint32_t Fb = __builtin_amdgcn_alignbit(pb[0], pb[1], ~tb);
    typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
    const u2_t v = {__builtin_bit_cast(uint32_t, mul1_pair_raw(Fa >> 16, __builtin_amdgcn_ubfe(Fa, 16 - K, 16))),
                    __builtin_bit_cast(uint32_t, mul1_pair_raw(Fb >> 16, __builtin_amdgcn_ubfe(Fb, 16 - K, 16)))};
    return __builtin_bit_cast(h4_t, v);
}

// One wave, kMfT tile columns (column pair t >> 1: gate|up projection, or down columns c0 + 2 (t >> 1)), RGA row
// groups, 32 k per step = two tile-rows. Per step the wave's 8 tiles (slot 2t + tile-row half) are fetched by 8 lanes
// each (lane i of a tile: words min(4i, 8K - 4) .. + 3, a 16-byte load inside the tile, and for K >= 5 words
// min(32 + 4i, 8K - 4) .. + 3 at staging time) after their (kmap, woff) one step earlier, and staged in a wave-private
// LDS slot per tile at lane-fixed positions: ring word w at slot[4 + w] (lanes past the tile's end leave copies of its
// last words behind it), the last word w(8K - 1) again at slot[3] (written by lane 7, whose last load always ends the
// tile), so that a funnel starting before the ring reads it. The step's 8 bitrates come from its lanes' kmap bytes (wave ballots): a step
// whose tiles are all K <= 2 stages compactly (slot stride kMixTSF, the first load only) and decodes with per-lane funnel origins
// and shifts precomputed for K = 1 and 2 (one select each per tile); other steps stage at stride kMixTS and decode
// with the tile's K at run time. Rings of 4 (first tile words DW - 1 = 2 steps ahead, (K, woff) DW = 3 steps ahead) make
// the loop a 4-step unroll; the step count (H / 32 or I / 32, H and I multiples of 128) is a multiple of 4. A goes
// through four LDS stages written two steps ahead, a barrier every second step, from a register ring of two: loaded
// three steps ahead, stored one step later (the 1-row-group kernels fit five waves per SIMD that way); with
// one row group each wave stages its own plane in a private ring and the loop has no barrier.
constexpr int kMixTSF = 20;                                 // compact slot: 3 pad, w(8K - 1), 16 words (K <= 2)

template <int NPS, int RGA>
struct MfmaPipeMix {
    static constexpr int DW = 3;
    static constexpr int UNITS = NPS * RGA * 64;             // NPS staged A planes; a wave reads plane apl
    // One row group: each wave stages its own plane (64 units, one per lane) in a private ring, so the loop needs no
    // barrier; the loads and LDS writes are those of the shared ring, whose 256 threads stage its units twice or more.
    static constexpr bool PRIV = RGA == 1;
    static constexpr int SU = PRIV ? 64 : UNITS;             // 16-byte units per stage (of the wave's ring if PRIV)
    static constexpr int CPT = PRIV ? 1 : (UNITS + 255) / 256;
    static constexpr int kNT = 2;                            // buffer-load cache policy: nontemporal
    __amdgpu_buffer_rsrc_t wrs, krs, ors;                    // the wave's projection: words, kmap, woff
    int col[2];                                              // per column pair: its first tile column (even)
    int tn, nsteps;
    int apl = 0;
    uint32_t* wl;                                            // the wave's LDS slots [8][kMixTS]
    uint32_t ktile;                                          // this lane's tile entry at step 0 (its slot's tile)
    uint32_t t0p1;                                           // t0 + 1 of the lane's k-permuted positions
    uint32_t fa1, fa2;                                       // fast path: LDS byte address of the lane's funnel
    uint32_t sh1, sh2;                                       // word in compact slot 0 at K = 1 and 2, and the
                                                             // funnel shifts
    __amdgpu_buffer_rsrc_t abuf[CPT];                        // this thread's units of a stage: their plane's rows, offsets
    uint32_t aoff[CPT];                                      // there at step 0, and units in the stage
    int adst[CPT];
    u32x4_t* lds;
    int lane;

    // The step's tile bitrates come from the kmap bytes its lanes loaded (lane 8 sl + i holds slot sl's K), as two
    // wave ballots: `big` (some K > 2: the run-time decode, which reads each K with v_readlane) and `two` (bit 8 sl:
    // slot sl has K = 2, else 1 on the fast path). Scalar loads of the kmap are avoided on purpose: they share the
    // LDS wait counter and may return out of order, so every LDS wait after one would wait for it too.
    __device__ __forceinline__ void load_meta(int (&M)[2], int s) const {
        const int off = (s < nsteps ? s : nsteps - 1) * 2 * tn;
        M[0] = __builtin_amdgcn_raw_buffer_load_b8(krs, ktile, off, 0);
        M[1] = (int)__builtin_amdgcn_raw_buffer_load_b32(ors, 4 * ktile, 4 * off, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ u32x4_t load_words(const int (&M)[2], uint32_t first) const {
        const uint32_t e = 8u * (uint32_t)M[0] - 4u;
        return __builtin_bit_cast(
            u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(wrs, 4u * ((uint32_t)M[1] + (first < e ? first : e)), 0, kNT));
    }
    // the lane's first 16 bytes of its tile: words min(4i, 8K - 4) .. + 3 (all of the tile for K <= 4)
    __device__ __forceinline__ void load_w(u32x4_t& D, const int (&M)[2]) const {
        D = load_words(M, 4u * (uint32_t)(lane & 7));
        __builtin_amdgcn_sched_barrier(0);
    }
    // Stage the step's tiles (M: this lane's (K, woff)). Lane 7's last loaded word ends its tile, so it writes the
    // wrap word. Tiles of K >= 5 (words 32 .. 8K - 1) take a second load here, on the spot: such steps are rare, and
    // keeping a second register ring for them would cost every step occupancy.
    __device__ __forceinline__ void stage_w(const u32x4_t& D, const int (&M)[2], bool fast, bool big) const {
        const int sl = lane >> 3, i = lane & 7;
        if (fast) {
            uint32_t* t = wl + sl * kMixTSF;
            if (i < 4) *reinterpret_cast<u32x4_t*>(t + 4 + 4 * i) = D;
            if (i == 7) t[3] = D[3];
        } else {
            uint32_t* t = wl + sl * kMixTS;
            *reinterpret_cast<u32x4_t*>(t + 4 + 4 * i) = D;
            if (big) {
                const u32x4_t D1 = load_words(M, 32u + 4u * (uint32_t)i);
                *reinterpret_cast<u32x4_t*>(t + 36 + 4 * i) = D1;
                if (i == 7) t[3] = D1[3];
            } else if (i == 7) {
                t[3] = D[3];
            }
        }
    }
    // A fragments (plane apl) of tile-row half sr in the k-permuted order: k 2g, 2g + 1 from chunk 2 sr, 2g + 8, 2g + 9
    // from chunk 2 sr + 1 (4 bytes at 4g in each unit)
    __device__ __forceinline__ void load_af(int stage, int sr, h4_t (&af)[RGA]) const {
        const int g = lane >> 4;
#pragma unroll
        for (int rg = 0; rg < RGA; ++rg) {
            const u32x4_t* base = lds + stage * SU + (PRIV ? 0 : apl * RGA * 64);
            const int row = 16 * rg + (lane & 15);
            typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
            const u2_t v = {reinterpret_cast<const uint32_t*>(base + a_unit(row, 2 * sr))[g],
                            reinterpret_cast<const uint32_t*>(base + a_unit(row, 2 * sr + 1))[g]};
            af[rg] = __builtin_bit_cast(h4_t, v);
        }
    }
    // slot sl = 2 t + sr holds tile column t (pair t >> 1, parity t & 1) of tile-row half sr; m0 = this lane's K
    __device__ __forceinline__ void compute(int stage, f4_t (&acc)[kMfT][RGA], int m0, uint64_t two, bool fast) const {
        if (fast) {
            // both tile-row halves in one 16x16x32 MFMA per tile column: lane group g's eight k slots are its four of
            // half 0 then its four of half 1, in A and B alike
            h4_t af[2][RGA];
            load_af(stage, 0, af[0]);
            load_af(stage, 1, af[1]);
#pragma unroll
            for (int t = 0; t < kMfT; ++t) {
                uint32_t whi[2], wlo[2];                         // the two tiles' funnel words, both reads issued first
#pragma unroll
                for (int sr = 0; sr < 2; ++sr) {
                    const int sl = 2 * t + sr;
                    const bool k2 = (two >> (8 * sl)) & 1;       // wave-uniform select
                    const lds_cu32_t o = (lds_cu32_t)(k2 ? fa2 : fa1);
                    whi[sr] = o[sl * kMixTSF];
                    wlo[sr] = o[sl * kMixTSF + 1];
                }
                h4_t bf[2];
#pragma unroll
                for (int sr = 0; sr < 2; ++sr) {
                    const bool k2 = (two >> (8 * (2 * t + sr))) & 1;
                    bf[sr] = decode4p12(__builtin_amdgcn_alignbit(whi[sr], wlo[sr], k2 ? sh2 : sh1), k2);
                }
                const h8_t b8 = __builtin_shufflevector(bf[0], bf[1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int rg = 0; rg < RGA; ++rg) {
                    const h8_t a8 = __builtin_shufflevector(af[0][rg], af[1][rg], 0, 1, 2, 3, 4, 5, 6, 7);
                    acc[t][rg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a8, b8, acc[t][rg], 0, 0, 0);
                }
            }
        } else {
#pragma unroll
            for (int sr = 0; sr < 2; ++sr) {
                h4_t af[RGA];
                load_af(stage, sr, af);
#pragma unroll
                for (int t = 0; t < kMfT; ++t) {
                    const int sl = 2 * t + sr;
                    const h4_t bf = decode4p_rt(wl + sl * kMixTS + 3, __builtin_amdgcn_readlane(m0, 8 * sl), t0p1);
#pragma unroll
                    for (int rg = 0; rg < RGA; ++rg)
                        acc[t][rg] = __builtin_amdgcn_mfma_f32_16x16x16f16(af[rg], bf, acc[t][rg], 0, 0, 0);
                }
            }
        }
    }
    __device__ __forceinline__ void load_a(u32x4_t (&Ra)[CPT], int s) const {
        const int ss = (s < nsteps ? s : nsteps - 1) * 32;
#pragma unroll
        for (int j = 0; j < CPT; ++j)
            Ra[j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(abuf[j], aoff[j], 2 * ss, 0));
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void store_a(const u32x4_t (&Ra)[CPT], int stage) const {
#pragma unroll
        for (int j = 0; j < CPT; ++j) lds[stage * SU + adst[j]] = Ra[j];
    }
    // step s, R = s mod 4
    template <int R>
    __device__ __forceinline__ void step(int s, u32x4_t (&W)[4], int (&M)[4][2], u32x4_t (&RA)[2][CPT],
                                         f4_t (&acc)[kMfT][RGA]) const {
        load_a(RA[R % 2], s + 3);
        load_meta(M[(R + DW) % 4], s + DW);
        load_w(W[(R + DW - 1) % 4], M[(R + DW - 1) % 4]);
        const int m0 = M[R][0];
        const uint64_t two = __builtin_amdgcn_ballot_w64(m0 == 2);
        const bool fast = __builtin_amdgcn_ballot_w64(m0 > 2) == 0;
        stage_w(W[R], M[R], fast, !fast && __builtin_amdgcn_ballot_w64(m0 > 4) != 0);
        compute(R, acc, m0, two, fast);
        store_a(RA[(R + 1) % 2], (R + 2) % 4);
        if constexpr (!PRIV) {
            if (R % 2 == 0) __syncthreads();
        }
    }
    __device__ __forceinline__ void run(f4_t (&acc)[kMfT][RGA]) const {
        u32x4_t W[4];
        int M[4][2];
        u32x4_t RA[2][CPT];
#pragma unroll
        for (int i = 0; i < DW; ++i) load_meta(M[i], i);
        load_a(RA[0], 0);
        load_a(RA[1], 1);
#pragma unroll
        for (int i = 0; i < DW - 1; ++i) load_w(W[i], M[i]);
        store_a(RA[0], 0);
        store_a(RA[1], 1);
        load_a(RA[1], 2);
        __syncthreads();
        for (int s = 0; s < nsteps; s += 4) {
            step<0>(s, W, M, RA, acc);
            step<1>(s + 1, W, M, RA, acc);
            step<2>(s + 2, W, M, RA, acc);
            step<3>(s + 3, W, M, RA, acc);
        }
        __syncthreads();                                 // every wave's last LDS read done: callers may reuse it
    }
    // After col / tn / wl / lane are set: the lane's tile entry and fast-path origins, and the A staging of `cnt` rows
    // (rowptr(plane, row) -> that row's first element)
    template <typename F>
    __device__ __forceinline__ void setup_a(int cnt, F rowptr) {
        const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if constexpr (PRIV) {                                // the wave's ring: lds + 4 stages * 64 units per wave
            lds += wv * 4 * SU;
            const int row = lane >> 2, ch = lane & 3;
            const _Float16* b = rowptr(apl, 0);
            abuf[0] = buffer_rsrc(b);
            aoff[0] = (uint32_t)(2 * (rowptr(apl, row < cnt ? row : cnt - 1) + 8 * ch - b));
            adst[0] = a_unit(row, ch);
        } else {
#pragma unroll
            for (int j = 0; j < CPT; ++j) {
                const int u0 = (64 * wv + 256 * j) % UNITS, u = u0 + (threadIdx.x & 63);
                const int p = u0 / (RGA * 64), rem = u - p * RGA * 64, row = rem >> 2, ch = rem & 3;
                const _Float16* b = rowptr(p, 0);
                abuf[j] = buffer_rsrc(b);
                aoff[j] = (uint32_t)(2 * (rowptr(p, row < cnt ? row : cnt - 1) + 8 * ch - b));
                adst[j] = p * RGA * 64 + a_unit(row, ch);
            }
        }
        const int sl = lane >> 3, t = sl >> 1, hr = sl & 1, pr = t >> 1;
        ktile = (uint32_t)(hr * tn + (pr ? col[1] : col[0]) + (t & 1));
        const int n = lane & 15, g = lane >> 4;
        t0p1 = (uint32_t)(32 * (n & 7) + 4 * (n >> 3) + 8 * g + 1);
        const uint32_t ta1 = t0p1 + 15u, ta2 = 2u * t0p1 + 15u;           // start + 31 at K = 1, 2
        fa1 = lds_addr(wl) + 4u * (3u + (ta1 >> 5));
        fa2 = lds_addr(wl) + 4u * (3u + (ta2 >> 5));
        sh1 = ~ta1 & 31u;
        sh2 = ~ta2 & 31u;
    }
};

template <int RGA>
__device__ __forceinline__ void gateup_mix_body(const MoeArgs& a, const ItemDesc* d, int nb, int cnt, u32x4_t* stage,
                                                uint32_t* wlds, float* C, float* rsum) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p0 = d->p0;
    MfmaPipeMix<2, RGA> L;
    L.tn = a.I / 16;
    L.nsteps = a.H / 32;
    L.lds = stage;
    L.lane = lane;
    L.wl = wlds + wave * 8 * kMixTS;
    const int pw = wave >> 1;                              // this wave's projection (gate, up), its 4 tile columns
    L.apl = pw;
    L.wrs = buffer_rsrc(reinterpret_cast<const void*>(d->tab[3 * pw]));
    L.krs = buffer_rsrc(reinterpret_cast<const void*>(d->km[2 * pw]));
    L.ors = buffer_rsrc(reinterpret_cast<const void*>(d->km[2 * pw + 1]));
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) L.col[pr] = nb * 8 + 4 * (wave & 1) + 2 * pr;
    L.setup_a(cnt, [&](int p, int row) { return a.xh + ((size_t)(p0 + row) * 2 + p) * a.H; });
    f4_t acc[kMfT][RGA];
#pragma unroll
    for (int t = 0; t < kMfT; ++t)
#pragma unroll
        for (int rg = 0; rg < RGA; ++rg) acc[t][rg] = f4_t{0.f, 0.f, 0.f, 0.f};
    L.run(acc);
    gateup_epilogue<RGA>(a, d, nb, cnt, acc, C, rsum);
}

template <int RGA>
__device__ __forceinline__ void down_mix_body(const MoeArgs& a, const ItemDesc* d, int nb, int cnt, u32x4_t* stage,
                                              uint32_t* wlds, float* C, float* rsum, int* s_comb) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p0 = d->p0;
    const int tn = a.H / 16;
    MfmaPipeMix<1, RGA> L;
    L.tn = tn;
    L.nsteps = a.I / 32;
    L.lds = stage;
    L.lane = lane;
    L.wl = wlds + wave * 8 * kMixTS;
    L.wrs = buffer_rsrc(reinterpret_cast<const void*>(d->tab[6]));
    L.krs = buffer_rsrc(reinterpret_cast<const void*>(d->km[4]));
    L.ors = buffer_rsrc(reinterpret_cast<const void*>(d->km[5]));
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
        int ct = nb * 16 + 4 * wave + 2 * pr;
        L.col[pr] = ct < tn ? ct : tn - 2;             // a last half block: in-bounds loads, results unused
    }
    L.setup_a(cnt, [&](int, int row) { return reinterpret_cast<const _Float16*>(a.abuf) + (size_t)(p0 + row) * a.I; });
    f4_t acc[kMfT][RGA];
#pragma unroll
    for (int t = 0; t < kMfT; ++t)
#pragma unroll
        for (int rg = 0; rg < RGA; ++rg) acc[t][rg] = f4_t{0.f, 0.f, 0.f, 0.f};
    L.run(acc);
    down_epilogue<RGA>(a, d, nb, cnt, acc, C, rsum, s_comb);
}

template <int RGA>
__global__ __launch_bounds__(256, EXL3_MIX_OCC(RGA)) void gateup_mix_kernel(MoeArgs a) {
    constexpr int CL = RGA == 1 ? 0 : RGA == 2 ? 1 : 2;
    // the epilogue's C reuses the pipeline's A stages and weight slots (dead once the pipeline has drained)
    constexpr int kStage = 4 * (RGA == 1 ? 4 : 2 * RGA) * 64 * 16, kW = 4 * 8 * kMixTS * 4, kC = 2 * 16 * 128 * 4;
    __shared__ __attribute__((aligned(16))) char smem[kStage + kW > kC ? kStage + kW : kC];
    u32x4_t* stage = reinterpret_cast<u32x4_t*>(smem);
    uint32_t* wlds = reinterpret_cast<uint32_t*>(smem + kStage);
    float* C = reinterpret_cast<float*>(smem);
    __shared__ float rsum[2 * 64];
    const int nbI = a.I / 128;
    int idx, nb;
    xcd_map(nbI, idx, nb);
    if (idx >= a.cls_cnt[CL]) return;
    const ItemDesc* d = a.blocks + a.cls_list[CL * a.max_blocks + idx];
    const int cnt = d->cnt;
    const int nblk = a.H / 128;
    for (int i = threadIdx.x; i < 2 * 64; i += 256) {
        const int p = i >> 6, m = i & 63;
        rsum[i] = m < cnt ? sum_ordered(a.xsum + ((size_t)(d->p0 + m) * 2 + p) * nblk, nblk) : 0.f;
    }
    __syncthreads();
    gateup_mix_body<RGA>(a, d, nb, cnt, stage, wlds, C, rsum);
}

template <int RGA>
__global__ __launch_bounds__(256, EXL3_MIX_OCC(RGA)) void down_mix_kernel(MoeArgs a) {
    constexpr int CL = RGA == 1 ? 0 : RGA == 2 ? 1 : 2;
    constexpr int kStage = 4 * (RGA == 1 ? 4 : RGA) * 64 * 16, kW = 4 * 8 * kMixTS * 4, kC = 16 * 256 * 4;
    __shared__ __attribute__((aligned(16))) char smem[kStage + kW > kC ? kStage + kW : kC];   // C aliases, as above
    u32x4_t* stage = reinterpret_cast<u32x4_t*>(smem);
    uint32_t* wlds = reinterpret_cast<uint32_t*>(smem + kStage);
    float* C = reinterpret_cast<float*>(smem);
    __shared__ float rsum[64];
    __shared__ int s_comb[2 * 64];
    const int nbH2 = (a.H / 128 + 1) / 2;
    int idx, nb;
    xcd_map(nbH2, idx, nb);
    if (idx >= a.cls_cnt[CL]) return;
    const ItemDesc* d = a.blocks + a.cls_list[CL * a.max_blocks + idx];
    const int cnt = d->cnt;
    const int nbI = a.I / 128;
    for (int m = threadIdx.x; m < 64; m += 256)
        rsum[m] = m < cnt ? sum_ordered(a.asum + (size_t)(d->p0 + m) * nbI, nbI) : 0.f;
    __syncthreads();
    down_mix_body<RGA>(a, d, nb, cnt, stage, wlds, C, rsum, s_comb);
}

// ------------------------------------------------------------------------------------------------ dense linear
// exl3_gemm for more rows than the GEMV takes per pass: y = Hn(Hk(x * suh) @ W_hat) * svh with the trellis decoded
// straight into MFMA B fragments once per row block, as in the reference's large-M linear
// (glm/xpu/csrc/exl3_ops.sycl:643-757), which reconstructs 16384-column fp16 slices and runs a GEMM instead.
//   linear_had   xh[s][m][k] = fp16(H128(fp16(x * suh[s])) / sqrt(128)) and the 128-blocks' sums xsum[s][m][k / 128]
//                (the Hadamard on MFMA, as in the MoE input transform; 16 rows per wave)
//                for every shard s (a fused multi-projection linear: output column blocks of S projections that share
//                the input, each with its own input signs suh[s]; shard_of_nb maps 128-column blocks to shards)
//   linear_wide  (exl3_wide.hip) workgroup per (row block of 32 .. 256 rows, k-split, 256-column block); a wave owns four
//                tile columns. With one split the epilogue writes y; otherwise it writes fp32 partials (affine applied)
//   linear_reduce (k-split only) wave per (row, 128 columns): partials in split order, Hadamard, * svh -> y
// xh in blocks of R rows (a multiple of 32) in block_unit order, the units' k as they are or (kperm) as the two 4-k runs
// of a k-permuted fragment
__global__ __launch_bounds__(256) void linear_had_kernel(const uint16_t* __restrict__ x, int64_t x_ld, int m, int k,
                                                         const uint16_t* __restrict__ suh, _Float16* xh, float* xsum,
                                                         int R, bool kperm) {
    __shared__ __attribute__((aligned(16))) _Float16 s_out[4][16][136];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kb = blockIdx.y, nblk = k / 128;
    suh += (size_t)blockIdx.z * k;                               // shard s = blockIdx.z
    xh += (size_t)blockIdx.z * m * k;
    xsum += (size_t)blockIdx.z * m * nblk;
    const int r0 = blockIdx.x * 64 + 16 * wave;                  // this wave's 16 rows
    if (r0 >= m) return;
    const int mm = lane & 15, g = lane >> 4;
    const int row = r0 + mm < m ? r0 + mm : m - 1;               // rows past m repeat the last one (not stored)
    const uint16_t* xr = x + (int64_t)row * x_ld + kb * 128 + 8 * g;
    const bool vx = ((uintptr_t)x & 15) == 0 && (x_ld & 7) == 0;
    h8_t xv[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) xv[ks] = load_h8(xr + 32 * ks, vx);
    const uint16_t* sv = suh + kb * 128 + 8 * g;
    const bool vs = ((uintptr_t)sv & 15) == 0;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) xv[ks] = xv[ks] * load_h8(sv + 32 * ks, vs);
    h8_t F[4];
    had_fragments(lane, F);
    float part[4];
    had16_rows(xv, F, lane, s_out[wave], part);
    const int b0 = r0 / R * R, cnt = m - b0 < R ? m - b0 : R;    // the block that holds the wave's rows
    u32x4_t* dst = reinterpret_cast<u32x4_t*>(xh + (size_t)b0 * k);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int u = lane + 64 * c, rr = u & 15, h = (u >> 4) & 1, kk = u >> 5;
        const _Float16* t = &s_out[wave][rr][16 * kk];
        typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
        const u2_t lo = *reinterpret_cast<const u2_t*>(t + (kperm ? 4 * h : 8 * h));
        const u2_t hi = *reinterpret_cast<const u2_t*>(t + (kperm ? 4 * h + 8 : 8 * h + 4));
        if (r0 + rr < m) dst[block_unit(cnt, kb * 8 + kk, h, r0 + rr - b0)] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float v = row16_sum(part[i]);
        if (mm == 0 && r0 + 4 * g + i < m) xsum[(size_t)(r0 + 4 * g + i) * nblk + kb] = v;
    }
}

// ------------------------------------------------------------------------------------------------ host
typedef void (*mfma_fn)(MoeArgs);

// Row classes run concurrently: the largest on the caller's stream, the others on the side streams.
template <typename F>
static int fork_classes(hipStream_t st, int ncls, F launch) {
    if (ncls == 1) return launch(0, st);
    if (env_int("EXL3MI_SERIAL_CLASSES", 0)) {            // every class on the caller's stream, one after another
        for (int cl = ncls - 1; cl >= 0; --cl)
            if (const int rc = launch(cl, st)) return rc;
        return EXL3_OK;
    }
    AuxStreams ax;
    int rc = aux_streams(&ax);
    if (rc) return rc;
    EXL3_CHECK_HIP(hipEventRecord(ax.ev[0], st));
    for (int i = 0; i < ncls - 1; ++i) EXL3_CHECK_HIP(hipStreamWaitEvent(ax.s[i], ax.ev[0], 0));
    for (int cl = ncls - 1; cl >= 0; --cl)
        if ((rc = launch(cl, cl == ncls - 1 ? st : ax.s[ncls - 2 - cl]))) return rc;
    for (int i = 0; i < ncls - 1; ++i) {
        EXL3_CHECK_HIP(hipEventRecord(ax.ev[1 + i], ax.s[i]));
        EXL3_CHECK_HIP(hipStreamWaitEvent(st, ax.ev[1 + i], 0));
    }
    return EXL3_OK;
}

// Split-K finish: wave per (row, 128-column block): the split partials summed in split order (eight splits' loads in
// flight at a time), Hadamard, * svh / sqrt(128).
__global__ __launch_bounds__(256) void linear_reduce_kernel(LinArgs a) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = blockIdx.x * 4 + wave;
    if (row >= a.m) return;
    const int col = blockIdx.y * 128 + lane;
    const uint16_t* sv = (a.tab ? reinterpret_cast<const uint16_t*>(a.tab[8]) : a.svh) + col;
    const float s0 = h2f(ldg(sv)) * kRsqrt128, s1 = h2f(ldg(sv + 64)) * kRsqrt128;
    const float* q = a.part + (size_t)row * a.n + col;
    const size_t ps = (size_t)a.m * a.n;
    float v0 = 0.f, v1 = 0.f;
    for (int p0 = 0; p0 < a.P; p0 += 8) {
        float t0[8], t1[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int pp = p0 + i < a.P ? p0 + i : a.P - 1;
            t0[i] = ldg(q + pp * ps);
            t1[i] = ldg(q + pp * ps + 64);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (p0 + i < a.P) {
                v0 += t0[i];
                v1 += t1[i];
            }
    }
    fwht128_wave(v0, v1, lane);
    linear_store(a, a.rowmap ? a.rowmap[row] : row, col, v0 * s0, v1 * s1);
}

lin_fn linear_wide_pick(int RG, int S, int K);           // exl3_wide.hip

// sum += part (n a multiple of 4): the reduce kernel's addition, for splits that run one after another.
__global__ __launch_bounds__(256) void linear_add_kernel(float* sum, const float* __restrict__ part, int64_t n) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    f4_t* s = reinterpret_cast<f4_t*>(sum + i);
    *s = *s + *reinterpret_cast<const f4_t*>(part + i);
}

static int device_cus(int* cus) {
    int dev = 0;
    EXL3_CHECK_HIP(hipGetDevice(&dev));
    EXL3_CHECK_HIP(hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev));
    return EXL3_OK;
}

// k-splits of a dense MLP's down projection (m rows in blocks of `block` rows), at most `cap`.
int dense_down_splits(int64_t m, int64_t n, int64_t k, int K, int block, int64_t cap, int* P) {
    int cus = 0;
    const int rc = device_cus(&cus);
    if (!rc) *P = linear_plan(m, n, k, 1, K, block / 32, cap, cus).P;
    return rc;
}

// The down projection of a dense MLP: the gate|up kernel's output blocks are a dense linear's input. Unlike the grouped
// kernel's, its k is split (5376 <- 21504 at 397 rows: 84 workgroups of 672 steps without).
static int launch_dense_down(const MoeArgs& a, hipStream_t st) {
    LinArgs l = {};
    l.xh = reinterpret_cast<const _Float16*>(a.abuf);
    l.xsum = a.asum;
    l.S = 1;
    l.tab = a.blocks[0].tab;                                       // (address only: device memory)
    l.rowmap = a.pair_tok;
    l.out = a.out;
    l.out_ld = a.out_ld;
    l.f32 = a.out_f32;
    l.m = a.M;
    l.k = a.I;
    l.n = a.H;
    l.nblk = a.I / 128;
    l.nrb = (a.M + a.block_rows - 1) / a.block_rows;
    l.ncb = (a.H + 255) / 256;
    l.bps = (l.nblk + a.dense_P - 1) / a.dense_P;
    const int P = (l.nblk + l.bps - 1) / l.bps;                    // = dense_P
    l.P = a.dense_sets < P ? 1 : P;                                // splits of a launch
    l.part = P > 1 ? a.y : nullptr;
    const int64_t nx = ((int64_t)l.nrb * l.ncb * l.P + 7) / 8 * 8;
    if (nx > 0x7FFFFFFF) return fail(EXL3_ERR_INVALID, "exl3_moe_forward: grid too large");
    const lin_fn fn = linear_wide_pick(a.block_rows / 32, 1, a.Kd);
    if (!fn) return fail(EXL3_ERR_INVALID, "exl3_moe_forward: no kernel for blocks of %d rows at K=%d", a.block_rows, a.Kd);
    const int64_t set = (int64_t)a.M * a.H;
    for (; l.p0 < P; l.p0 += l.P) {                                // one launch, or the first split and the later ones added
        EXL3_LAUNCH("mlp_down_wide", fn, dim3((unsigned)nx), dim3(256), 0, st, l);
        if (l.p0 > 0)
            EXL3_LAUNCH("linear_add", linear_add_kernel, dim3((unsigned)((set / 4 + 255) / 256)), dim3(256), 0, st, a.y, l.part,
                        set);
        if (l.P < P) l.part = reinterpret_cast<float*>(a.xh);
    }
    l.part = a.y;
    if (P > 1)
        EXL3_LAUNCH("linear_reduce", linear_reduce_kernel, dim3((unsigned)((l.m + 3) / 4), (unsigned)(l.n / 128)),
                    dim3(256), 0, st, l);
    return EXL3_OK;
}

int launch_gateup_wide(const MoeArgs& a, int cl, int nblocks, hipStream_t st);  // exl3_moe_wide.hip (uniform K)
int launch_down_wide(const MoeArgs& a, int cl, int nblocks, hipStream_t st);
int launch_moe_combine(const MoeArgs& a, hipStream_t st);
// the same for a uniform projection beside a per-tile-K one (classes of 16, 32 and 64 rows)
int launch_gateup_class(const MoeArgs& a, int cl, hipStream_t st);
int launch_down_class(const MoeArgs& a, int cl, hipStream_t st);

// The grouped GEMM of one layer call: the input transform, then per row class gate|up followed by down on that class's
// stream (a class's down blocks read only the down inputs its own gate|up blocks wrote; tokens whose slots span
// classes are combined by the last slot to finish), so one class's down pass overlaps the others' gate|up.
int launch_moe_mfma(const MoeArgs& a, hipStream_t st) {
    const int nxb = (a.max_blocks + 7) / 8 * 8;
    const int64_t had_jobs = (int64_t)(a.M * a.slots + 15) / 16 * (a.H / 128);
    EXL3_CHECK_ARG(had_jobs / 4 < 0x7FFFFFFF, "exl3_moe_forward: too many rows");
    EXL3_LAUNCH("moe_pairs_had", pairs_had_kernel, dim3((unsigned)((had_jobs + 3) / 4)), dim3(256), 0, st, a);
    const dim3 grid_gu(nxb * (a.I / 128)), grid_dn(nxb * ((a.H / 128 + 1) / 2));
    const bool wide = a.Kg > 0 && a.Kd > 0;
    // uniform K: a block of more than 32 rows leaves room for at most one per 33 rows (65 where smaller remainders are cut)
    const int np = a.M * a.slots, nbig = np / (a.block_rows > 64 && a.dense_P == 0 ? 65 : 33) + 1;
    const int rc = fork_classes(st, wide ? (a.block_rows > 32 ? 2 : 1) : 3, [&](int cl, hipStream_t s) -> int {
        if (wide) {
            const int n = cl == 1 && nbig < a.max_blocks ? nbig : a.max_blocks;
            const int e = launch_gateup_wide(a, cl, n, s);
            return e || a.dense_P > 0 ? e : launch_down_wide(a, cl, n, s);   // (dense: after the classes have joined)
        }
        const int rga = 1 << cl;                       // row groups of 16
        if (a.Kg == 0) {
            mfma_fn gu = rga == 4 ? gateup_mix_kernel<4> : rga == 2 ? gateup_mix_kernel<2> : gateup_mix_kernel<1>;
            EXL3_LAUNCH(rga == 4 ? "moe_gateup_mfma_r4" : rga == 2 ? "moe_gateup_mfma_r2" : "moe_gateup_mfma_r1", gu,
                        grid_gu, dim3(256), 0, s, a);
        } else if (const int e = launch_gateup_class(a, cl, s)) {
            return e;
        }
        if (a.Kd > 0) return launch_down_class(a, cl, s);
        mfma_fn dn = rga == 4 ? down_mix_kernel<4> : rga == 2 ? down_mix_kernel<2> : down_mix_kernel<1>;
        EXL3_LAUNCH(rga == 4 ? "moe_down_mfma_r4" : rga == 2 ? "moe_down_mfma_r2" : "moe_down_mfma_r1", dn, grid_dn,
                    dim3(256), 0, s, a);
        return EXL3_OK;
    });
    if (rc || a.Kd == 0) return rc;
    return a.dense_P > 0 ? launch_dense_down(a, st) : launch_moe_combine(a, st);
}

// Plan of a call of m rows in at most `most` bytes of scratch; *fits: whether there is one.
int linear_mfma_plan(int64_t m, int64_t n, int64_t k, int S, int K, size_t most, LinPlan* pl, bool* fits) {
    int cus = 0;
    if (const int rc = device_cus(&cus)) return rc;
    const int v = env_int("EXL3MI_LINEAR_BLOCK", 0);               // forced row groups of 32 per block: 1, 2, 4 or 8
    *fits = linear_call_plan(m, n, k, S, K, v == 1 || v == 2 || v == 4 || v == 8 ? v : 0, cus, most, pl);
    if (const int jobs = env_int("EXL3MI_LINEAR_JOBS", 0); jobs && *fits) {        // forced workgroup target
        const int nblk = (int)(k / 128);
        const int64_t R = 32 * pl->RG, tiles = (m + R - 1) / R * ((n + 255) / 256), want = (jobs + tiles - 1) / tiles;
        const int pmax = nblk / 2 > 1 ? nblk / 2 : 1;
        pl->bps = (nblk + (int)(want < pmax ? want : pmax) - 1) / (int)(want < pmax ? want : pmax);
        pl->P = (nblk + pl->bps - 1) / pl->bps;
        while (pl->RG > 1 && !(a_span_ok(m < 32 * pl->RG ? m : 32 * pl->RG, 128LL * pl->bps) &&
                               linear_block_built(pl->RG, S, K)))
            pl->RG /= 2;
        *fits = linear_call_bytes(m, n, k, S, pl->P) <= most;
    }
    return EXL3_OK;
}

// Dense linear on MFMA by `pl`: input transform, blocks of 32 .. 256 rows x 256 columns and, with k-splits, the reduction.
// Scratch from the workspace, or `fixed` (fixed_bytes of it; those launches also bypass the opt-in event profiler).
int launch_linear_mfma(const LinPlan& pl, const uint16_t* A, int64_t a_ld, int64_t m, int64_t k, const uint32_t* tr, int64_t n,
                       int K, void* C, int64_t c_ld, bool f32, const uint16_t* suh, int S, const int32_t* sonb,
                       const uint16_t* svh, char* fixed, size_t fixed_bytes, hipStream_t st) {
    const int nblk = (int)(k / 128), R = 32 * pl.RG;
    if (m > 0x7FFFFFFF / 64 || k > 0x7FFFFFFF || n > 0x7FFFFFFF || nblk > 65535)
        return fail(EXL3_ERR_INVALID, "exl3_gemm: shape too large");
    LinArgs a = {};
    a.m = (int)m;
    a.k = (int)k;
    a.n = (int)n;
    a.nblk = nblk;
    a.nrb = (int)((m + R - 1) / R);
    a.ncb = (int)((n + 255) / 256);
    a.bps = pl.bps;
    a.P = pl.P;
    Carve cv{fixed, fixed_bytes};
    if (!fixed) {
        Workspace ws;
        if (const int rc = workspace(linear_call_bytes(m, n, k, S, a.P), 0, st, &ws)) return rc;
        cv = Carve{ws.scratch, ws.scratch_bytes};
    }
    _Float16* xh = cv.take<_Float16>((size_t)S * m * k);
    float* xsum = cv.take<float>((size_t)S * m * nblk);
    a.part = a.P > 1 ? cv.take<float>((size_t)a.P * m * n) : nullptr;
    if (!xh || !xsum || (a.P > 1 && !a.part)) return fail(EXL3_ERR_INVALID, "exl3_gemm: workspace carve failed");
    a.xh = xh;
    a.xsum = xsum;
    a.S = S;
    a.sonb = S > 1 ? sonb : nullptr;
    a.tr = tr;
    a.svh = svh;
    a.out = C;
    a.out_ld = c_ld;
    a.f32 = f32 ? 1 : 0;
    const dim3 hgrid((unsigned)((m + 63) / 64), (unsigned)nblk, (unsigned)S);
    const int64_t nx = ((int64_t)a.nrb * a.ncb * a.P + 7) / 8 * 8;
    if (nx > 0x7FFFFFFF) return fail(EXL3_ERR_INVALID, "exl3_gemm: grid too large");
    const dim3 rgrid((unsigned)((m + 3) / 4), (unsigned)(n / 128));
    const lin_fn fn = linear_wide_pick(pl.RG, S, K);
    if (!fn) return fail(EXL3_ERR_INVALID, "exl3_gemm: no %d-row kernel for %d shards at K=%d", R, S, K);
    if (fixed) {
        hipLaunchKernelGGL(linear_had_kernel, hgrid, dim3(256), 0, st, A, a_ld, (int)m, (int)k, suh, xh, xsum, R, K <= 5);
        hipLaunchKernelGGL(fn, dim3((unsigned)nx), dim3(256), 0, st, a);
        if (a.P > 1) hipLaunchKernelGGL(linear_reduce_kernel, rgrid, dim3(256), 0, st, a);
        EXL3_CHECK_HIP(hipGetLastError());
        return EXL3_OK;
    }
    EXL3_LAUNCH("linear_had", linear_had_kernel, hgrid, dim3(256), 0, st, A, a_ld, (int)m, (int)k, suh, xh, xsum, R,
                K <= 5);
    EXL3_LAUNCH("linear_wide", fn, dim3((unsigned)nx), dim3(256), 0, st, a);
    if (a.P > 1) EXL3_LAUNCH("linear_reduce", linear_reduce_kernel, rgrid, dim3(256), 0, st, a);
    return EXL3_OK;
}

}  // namespace exl3
