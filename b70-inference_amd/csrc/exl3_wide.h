// K loop of the wide-block GEMM kernels: one workgroup of four waves multiplies 32 RG rows by 256 columns.
//
// What bounds it: a 64-row block spends 472 VALU cycles on decoding 64 columns x 32 k for 256 MFMA cycles, so many-row
// calls were bound by the repeated decode and by the serial chain of staging, decode and MFMA in a wave. Here every
// wave owns 64 columns and all 32 RG rows (RG = 8: one wave per SIMD, 256 accumulators per lane): the decode of a step
// (about 110 VALU instructions) is spent once per 256 rows and lies between the MFMAs of the step before
// (32 v_mfma_f32_32x32x16_f16, 1024 cycles), which have no use for its results yet. No value is decoded twice in a
// workgroup and B never touches the LDS as fp16. The LDS carries the A tile (read once per wave: 64 KB per
// workgroup and step, half of what the LDS delivers in the step's MFMA time) and the trellis words.
//
// Fragments (v_mfma_f32_32x32x16_f16): A lane L holds row L & 31, k unit h = L >> 5; B lane L column L & 31 (tile
// (L >> 4) & 1 of a tile pair, column L & 15), the same k; D lane L column L & 31, rows 8 (i >> 2) + 4 h + (i & 3).
// The eight k of unit h in a tile-row of 16: K <= 5: {4h .. 4h + 3, 8 + 4h .. 8 + 4h + 3}, which are two runs of four
// consecutive trellis positions, t0 + {0..3} and t0 + 8 + {0..3} with t0 = 32 (n & 7) + 4 (n >> 3) + 16 h, one funnel
// each; K >= 6: 8h .. 8h + 7 (frag_window's positions). A is laid out in memory to match
// (block_unit).
#pragma once

#include "exl3_device.h"
#include "exl3_mfma.h"

namespace exl3 {

typedef float f16_t __attribute__((ext_vector_type(16)));

// A wave-uniform address kept in scalar registers (64-bit address arithmetic runs on the VALU, and a buffer resource in
// vector registers would be read by a loop over the lanes at every load).
__device__ __forceinline__ void* uniform_ptr(const void* p) {
    const uint64_t u = (uint64_t)(uintptr_t)p;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    return reinterpret_cast<void*>((uintptr_t)(((uint64_t)hi << 32) | lo));
}

// Waits for the loads that a pipe issued past its last step. Without it the compiler waits where an epilogue first reuses one of
// their registers, in every conditional store block that may be the first, and there for the stores before it as well
// (128 rows of 4096 -> 14336, partials: 24.4 -> 30.2 us).
__device__ __forceinline__ void drain_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }      // vmcnt(0)

// Trellis words of one wave: its 64 columns (four tile columns, two pairs of adjacent tiles), 32 k (two tile-rows) per
// step. One coalesced load of K words per lane brings a step in; the words go to wave-private LDS slots (one per tile,
// the ring's last word repeated in front), from which every lane reads the words of its four fragments. LDS operations
// of one wave complete in order, so the slots need no second buffer: step s + 1 is staged when the words of step s have
// been read.
template <int K, bool PL>
struct TileWords {
    static constexpr bool KP = K <= 5;
    static constexpr int TS = 8 * K + 8;                     // words per staged tile: 3 pad, w(8K - 1), w(0) .., 4 past
    static constexpr int NW = KP ? 4 : (48 + 25 * K + 31) / 32;   // words a fragment reads
    static constexpr int kSlotBytes = 4 * 8 * TS * 4;        // of four waves

    const uint32_t* wsrc;                                    // this lane's K words at step 0
    uint32_t wstep;                                          // words between steps (two tile-rows)
    int nsteps;
    uint32_t* wl;                                            // the wave's slots [8][TS]
    int wdst, wwrap;                                         // this lane's staged words, and where its last goes again
    uint32_t fa[2], fsh[2];                                  // first word of each run in slot 0 (LDS address), shift
    int lane;

    __device__ __forceinline__ void load_w(uint32_t (&D)[K], int s) const {
        const uint32_t* p = wsrc + (uint32_t)(s < nsteps ? s : nsteps - 1) * wstep;
#pragma unroll
        for (int i = 0; i < K; ++i) D[i] = ldg(p + WordOrder<K, PL>::word_off(i));
    }
    // lane q of a tile holds words [Kq, Kq + K); its last word goes in front of the tile too if it is the ring's last
    // (the other lanes store theirs where it already is)
    __device__ __forceinline__ void stage_w(const uint32_t (&D)[K]) const {
        uint32_t* t = wl + wdst;
#pragma unroll
        for (int i = 0; i < K; ++i) t[i] = D[i];
        wl[wwrap] = D[K - 1];
    }
    // words of the lane's fragment f (tile-row f >> 1 of the step, tile pair f & 1)
    __device__ __forceinline__ void load_f(uint32_t (&R)[NW], int f) const { load_slot(R, 4 * (f & 1) + 2 * (f >> 1)); }
    __device__ __forceinline__ void load_slot(uint32_t (&R)[NW], int slot) const {
        typedef const __attribute__((address_space(3))) uint32_t* lds_t;
        if constexpr (KP) {
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                R[2 * g] = ((lds_t)fa[g])[slot * TS];
                R[2 * g + 1] = ((lds_t)fa[g])[slot * TS + 1];
            }
        } else {
#pragma unroll
            for (int i = 0; i < NW; ++i) R[i] = ((lds_t)fa[0])[slot * TS + i];
        }
    }
    // pair c (0..3) of a fragment: its k 2c, 2c + 1
    __device__ __forceinline__ uint32_t decode_pair(const uint32_t (&R)[NW], int c) const {
        if constexpr (KP) {
            const int g = c & 1;
            const uint32_t F = __builtin_amdgcn_alignbit(R[2 * g], R[2 * g + 1], fsh[g]);
            if (c < 2)
                return __builtin_bit_cast(uint32_t, mul1_pair_raw(F >> 16, __builtin_amdgcn_ubfe(F, 16 - K, 16)));
            return __builtin_bit_cast(uint32_t, mul1_pair_raw(__builtin_amdgcn_ubfe(F, 16 - 2 * K, 16),
                                                              __builtin_amdgcn_ubfe(F, 16 - 3 * K, 16)));
        } else {
            uint32_t N[NW];
#pragma unroll
            for (int i = 0; i < NW - 1; ++i) N[i] = __builtin_amdgcn_alignbit(R[i], R[i + 1], fsh[0]);
            N[NW - 1] = R[NW - 1];
            return __builtin_bit_cast(uint32_t,
                                      mul1_pair_raw(frag_window<K>(N, 8 * c), frag_window<K>(N, 8 * c + 1)));
        }
    }
    // tr: tile-row 0 of the projection, tile-rows tn tiles apart; pair_col(p): first tile column of the wave's pair p
    template <typename Fn>
    __device__ __forceinline__ void setup_w(int tn, uint32_t* wave_lds, const uint32_t* tr, Fn pair_col) {
        const int g = lane >> 4, pair = g >> 1, hr = g & 1;
        wsrc = tr + (size_t)hr * tn * (8 * K) +
               WordOrder<K, PL>::chunk_base(pair_col(pair) + ((lane & 15) >> 3), lane & 7);
        wstep = (uint32_t)(2 * tn * 8 * K);
        wl = wave_lds;
        const int slot = 2 * g + ((lane & 15) >> 3), q = lane & 7;
        wdst = slot * TS + 4 + q * K;
        wwrap = q == 7 ? slot * TS + 3 : wdst + K - 1;
        setup_f(lane >> 5, (lane >> 4) & 1);
    }
    // the lane reads k unit h of its column, from slots `slot` past the fragment's
    __device__ __forceinline__ void setup_f(int h, int slot) {
        const int n = lane & 15;
        const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)wl +
                              4u * (uint32_t)(slot * TS);
        if constexpr (KP) {
            const int t0 = 32 * (n & 7) + 4 * (n >> 3) + 16 * h;
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int b = (t0 + 8 * r + 1) * K + 15;       // the run's first bit + 31
                fa[r] = base + 4u * (uint32_t)((b >> 5) + 3);
                fsh[r] = (uint32_t)(~b & 31);
            }
        } else {
            const int start = (32 * (n & 7) + 2 * h + 4 * (n >> 3) + 1) * K - 16, w0 = (start - 1) >> 5;
            fa[0] = fa[1] = base + 4u * (uint32_t)(w0 + 4);
            fsh[0] = fsh[1] = (uint32_t)(32 - (start - 32 * w0));
        }
    }
};

template <int K, int RG, int NPL, bool PL = false>
struct WidePipe : TileWords<K, PL> {
    typedef TileWords<K, PL> T;
    using T::decode_pair, T::lane, T::load_f, T::load_w, T::nsteps, T::NW, T::stage_w;
    static constexpr int UNITS = NPL * RG * 128;             // 16-byte A units of one stage (32 k)
    static constexpr int CPT = UNITS / 256;
    static constexpr int ST = 4;                             // A stages
    static constexpr int NG = 2 * RG;                        // groups of two MFMAs in a step
    static constexpr int WR = K <= 5 && NPL == 1 ? 4 : 2;    // steps of words in registers (where four do not spill)
    static constexpr int AD = 4;                             // A fragments in flight (divides NG)
    static_assert(UNITS % 256 == 0 && (RG & (RG - 1)) == 0 && RG >= 2 && RG <= 8, "row groups");
    static constexpr int kStageBytes = ST * UNITS * 16;

    __amdgpu_buffer_rsrc_t abuf[NPL];                        // A of the workgroup's first row group, per plane
    uint32_t aoff[CPT];
    u32x4_t* lds;                                            // [ST][UNITS]
    int apl;                                                 // plane this wave reads
    int astep;                                               // bytes of A between steps

    __device__ __forceinline__ h8_t load_af(int stage, int g) const {        // group g: tile-row g / RG, row group g % RG
        return __builtin_bit_cast(h8_t, lds[stage * UNITS + (apl * RG + g % RG) * 128 + (g / RG) * 64 + lane]);
    }
    __device__ __forceinline__ u32x4_t load_a(int j, int s) const {
        return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                               abuf[2 * j / RG], aoff[j], (s < nsteps ? s : nsteps - 1) * astep, 0));
    }
    __device__ __forceinline__ void store_a(const u32x4_t& v, int j, int stage) const {
        lds[stage * UNITS + 256 * j + threadIdx.x] = v;
    }

    // Step s (R = s mod 4): multiplies stage R by the fragments B while it decodes the next step's from F into Bn. Spread
    // over its groups: the words of step s + 2 are staged and read back into F as its fragments are used up, the words
    // of step s + WR + 1 loaded; A of step s + 2 (loaded two steps ago) is stored to its stage and A of step s + 4 loaded.
    // One barrier per step, which waits for no memory operation but the step's A stores: a stage is written two steps
    // after it was last read and read (its first fragments before its step starts) a barrier after its last write.
    template <int R>
    __device__ __forceinline__ void step(int s, uint32_t (&W)[WR][K], uint32_t (&F)[4][NW], h8_t (&B)[4], h8_t (&Bn)[4],
                                         u32x4_t (&RA)[2][CPT], h8_t (&af)[AD], f16_t (&acc)[RG][2]) const {
        typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
        constexpr int PPG = 16 / NG;                           // pairs decoded per group
        static_assert(PPG * NG == 16 && NG >= CPT + AD, "groups");
        u4_t nb[4];
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int ks = g / RG, rg = g % RG;
            const h8_t a = af[g % AD];
            acc[rg][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, B[2 * ks], acc[rg][0], 0, 0, 0);
            if (g == 0) stage_w(W[(R + 2) % WR]);
            if (g < CPT) {
                store_a(RA[R % 2][g], g, (R + 2) % 4);
                RA[R % 2][g] = load_a(g, s + 4);
            }
            if (g == CPT) load_w(W[(R + 1) % WR], s + WR + 1);
#pragma unroll
            for (int i = 0; i < PPG; ++i) {                    // pairs in the order 0, 2, 1, 3: a run's pairs together
                const int p = g * PPG + i, c = (p & 1) * 2 + ((p >> 1) & 1);
                uint32_t v = decode_pair(F[p >> 2], c);
                asm volatile("" : "+v"(v));                    // decoded in this group: sunk to its use otherwise
                nb[p >> 2][c] = v;
                if ((p & 3) == 3) load_f(F[p >> 2], p >> 2);
            }
            acc[rg][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, B[2 * ks + 1], acc[rg][1], 0, 0, 0);
            const int gn = g + AD;
            af[g % AD] = load_af(gn < NG ? R : (R + 1) % 4, gn % NG);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int f = 0; f < 4; ++f) Bn[f] = __builtin_bit_cast(h8_t, nb[f]);
        asm volatile("" ::: "memory");
        // lgkmcnt(AD): LDS operations complete in order and at least AD reads follow the last A store
        __builtin_amdgcn_s_waitcnt(0xC07F | AD << 8);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ void run(f16_t (&acc)[RG][2]) const {
        uint32_t W[WR][K], F[4][NW];
        h8_t B[2][4], af[AD];
        u32x4_t RA[2][CPT];
        typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int i = 0; i < WR; ++i) load_w(W[i], i);
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            RA[0][j] = load_a(j, 0);
            RA[1][j] = load_a(j, 1);
        }
        stage_w(W[0]);
#pragma unroll
        for (int f = 0; f < 4; ++f) load_f(F[f], f);
        load_w(W[0], WR);
        stage_w(W[1]);
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            u4_t v;
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = decode_pair(F[f], c);
            B[0][f] = __builtin_bit_cast(h8_t, v);
            load_f(F[f], f);
        }
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            store_a(RA[0][j], j, 0);
            store_a(RA[1][j], j, 1);
            RA[0][j] = load_a(j, 2);
            RA[1][j] = load_a(j, 3);
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < AD; ++g) af[g] = load_af(0, g);
        for (int s = 0; s < nsteps; s += 4) {                  // nsteps is a multiple of 4
            step<0>(s, W, F, B[0], B[1], RA, af, acc);
            step<1>(s + 1, W, F, B[1], B[0], RA, af, acc);
            step<2>(s + 2, W, F, B[0], B[1], RA, af, acc);
            step<3>(s + 3, W, F, B[1], B[0], RA, af, acc);
        }
        drain_loads();
        __syncthreads();                                       // every LDS access done: callers may reuse the stages
    }
    // plane(p): the workgroup's rows of plane p at its first k (block_unit order, cnt rows)
    template <typename Fn>
    __device__ __forceinline__ void setup_a(int cnt, Fn plane) {
        const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int p = 0; p < NPL; ++p)
            abuf[p] = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(plane(p)), 0, 0x7fffffff, 0x00020000);
        astep = 64 * cnt;
#pragma unroll
        for (int j = 0; j < CPT; ++j) {                        // two row groups per pass; a wave stages one 16-k block
            const int row = 32 * ((2 * j + (wv >> 1)) % RG) + (lane & 31);
            aoff[j] = 16u * (uint32_t)((2 * (wv & 1) + (lane >> 5)) * cnt + (row < cnt ? row : cnt - 1));
        }
    }
};

// Up to 64 rows (RG = 1, 2): several waves per SIMD, each on its own. A fragments come straight from memory (the block's
// A is read by all workgroups of its row block, so from the L2, and by the workgroup's waves, so from the L1) four
// steps ahead (two with 64 rows): no LDS traffic for A and no barrier in the loop; a fragment's MFMAs run while the next one is decoded.
template <int K, int RG, bool PL = false>
struct DirectPipe : TileWords<K, PL> {
    typedef TileWords<K, PL> T;
    using T::decode_pair, T::lane, T::load_f, T::load_w, T::nsteps, T::NW, T::stage_w;
    static constexpr int AD = RG == 1 ? 4 : 2;               // steps of A in registers
    static constexpr int WR = 4;                             // steps of words in registers
    __amdgpu_buffer_rsrc_t abuf;
    uint32_t aoff[RG];
    int astep, akk;                                          // bytes of A between steps and between 16-k blocks

    __device__ __forceinline__ void load_a(h8_t (&A)[2 * RG], int s) const {
        const int so = (s < nsteps ? s : nsteps - 1) * astep;
#pragma unroll
        for (int i = 0; i < 2 * RG; ++i)
            A[i] = __builtin_bit_cast(h8_t, __builtin_amdgcn_raw_buffer_load_b128(abuf, aoff[i % RG], so + i / RG * akk, 0));
    }
    template <int R>
    __device__ __forceinline__ void step(int s, uint32_t (&W)[WR][K], uint32_t (&F)[4][NW], h8_t (&A)[AD][2 * RG],
                                         f16_t (&acc)[RG][2]) const {
        typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int f = 0; f < 4; ++f) {                         // fragment (tile-row f >> 1, tile pair f & 1)
            u4_t v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int c = (i & 1) * 2 + (i >> 1);          // pairs in the order 0, 2, 1, 3: a run's pairs together
                v[c] = decode_pair(F[f], c);
            }
            load_f(F[f], f);
            const h8_t b = __builtin_bit_cast(h8_t, v);
#pragma unroll
            for (int rg = 0; rg < RG; ++rg)
                acc[rg][f & 1] =
                    __builtin_amdgcn_mfma_f32_32x32x16_f16(A[R % AD][(f >> 1) * RG + rg], b, acc[rg][f & 1], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        stage_w(W[(R + 2) % WR]);
        load_a(A[R % AD], s + AD);
        load_w(W[(R + 2) % WR], s + 2 + WR);
    }
    __device__ __forceinline__ void run(f16_t (&acc)[RG][2]) const {
        uint32_t W[WR][K], F[4][NW];
        h8_t A[AD][2 * RG];
#pragma unroll
        for (int i = 0; i < WR; ++i) load_w(W[i], i);
#pragma unroll
        for (int i = 0; i < AD; ++i) load_a(A[i], i);
        stage_w(W[0]);
#pragma unroll
        for (int f = 0; f < 4; ++f) load_f(F[f], f);
        stage_w(W[1]);
        load_w(W[0], WR);
        load_w(W[1], WR + 1);
        for (int s = 0; s < nsteps; s += 4) {                  // nsteps is a multiple of 4
            step<0>(s, W, F, A, acc);
            step<1>(s + 1, W, F, A, acc);
            step<2>(s + 2, W, F, A, acc);
            step<3>(s + 3, W, F, A, acc);
        }
        drain_loads();
        __syncthreads();                                       // every slot read done: callers may reuse the LDS
    }
    __device__ __forceinline__ void setup_a(int cnt, const void* a) {
        abuf = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(a), 0, 0x7fffffff, 0x00020000);
        akk = 32 * cnt;
        astep = 64 * cnt;
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
            const int row = 32 * rg + (lane & 31);
            aoff[rg] = 16u * (uint32_t)((lane >> 5) * cnt + (row < cnt ? row : cnt - 1));
        }
    }

    // Blocks of up to 16 rows: v_mfma_f32_16x16x32_f16, one tile column and the step's whole k per instruction. The 32-row
    // form with half its rows empty spends 256 MFMA cycles beside 440 VALU cycles a step, this one 64 (us, 32-row form / this:
    // 419 rows over 256 experts of 2304 -> 1280, top-4, K = 4 375 / 334; 9 rows of 5376 -> 21504, K = 8 40.6 / 30.2). Lane L: row
    // or column L & 15, k unit (L >> 4) & 1 of tile-row L >> 5; the instruction adds its k in the order of the two 32x32x16
    // ones it replaces, so that a row's bits do not depend on the form.
    template <int R>
    __device__ __forceinline__ void step16(int s, uint32_t (&W)[WR][K], uint32_t (&F)[4][NW], h8_t (&A)[4],
                                           f4_t (&acc)[4]) const {
        typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int f = 0; f < 4; ++f) {                         // tile column f
            u4_t v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int c = (i & 1) * 2 + (i >> 1);
                v[c] = decode_pair(F[f], c);
            }
            T::load_slot(F[f], 4 * (f >> 1) + (f & 1));
            acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[R], __builtin_bit_cast(h8_t, v), acc[f], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        stage_w(W[(R + 2) % WR]);
        A[R] = load_a16(s + 4);
        load_w(W[(R + 2) % WR], s + 2 + WR);
    }
    __device__ __forceinline__ h8_t load_a16(int s) const {
        const int so = (s < nsteps ? s : nsteps - 1) * astep;
        return __builtin_bit_cast(h8_t, __builtin_amdgcn_raw_buffer_load_b128(abuf, aoff[0], so, 0));
    }
    __device__ __forceinline__ void run16(int cnt, f4_t (&acc)[4]) {
        static_assert(RG == 1 && WR == 4);
        const int h = (lane >> 4) & 1, row = lane & 15;
        T::setup_f(h, 2 * (lane >> 5));
        aoff[0] = 16u * (uint32_t)(h * cnt + (row < cnt ? row : cnt - 1)) + (uint32_t)((lane >> 5) * akk);
        uint32_t W[WR][K], F[4][NW];
        h8_t A[4];
#pragma unroll
        for (int i = 0; i < WR; ++i) load_w(W[i], i);
#pragma unroll
        for (int i = 0; i < 4; ++i) A[i] = load_a16(i);
        stage_w(W[0]);
#pragma unroll
        for (int f = 0; f < 4; ++f) T::load_slot(F[f], 4 * (f >> 1) + (f & 1));
        stage_w(W[1]);
        load_w(W[0], WR);
        load_w(W[1], WR + 1);
        for (int s = 0; s < nsteps; s += 4) {
            step16<0>(s, W, F, A, acc);
            step16<1>(s + 1, W, F, A, acc);
            step16<2>(s + 2, W, F, A, acc);
            step16<3>(s + 3, W, F, A, acc);
        }
        drain_loads();
        __syncthreads();                                       // every slot read done: callers may reuse the LDS
    }
};

// ------------------------------------------------------------------------------------------------ epilogue
// A row of 128 columns spread over L = 4 or 8 adjacent lanes: lane index sub (row_sub) holds columns
// 4 L i + 4 sub + j of v[i][j]. The transform's stages of column bits 0, 1 and of the bits of i are register additions,
// those of sub exchange with the lane whose sub differs in one bit; column bits in ascending order whatever L is (the
// same bits in every row class). sub is not the plain lane number: its bits are chosen
// so that those lanes are at xor distances 1, 2 and 7, each a single DPP move (quad permutes, half-row mirror).
template <int L>
__device__ __forceinline__ int row_sub(int lane) {
    static_assert(L == 4 || L == 8);
    return L == 4 ? lane & 3 : (lane & 7) ^ 3 * ((lane >> 2) & 1);
}
template <int B>                                             // value of the lane whose sub differs in bit B
__device__ __forceinline__ float sub_xor(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                                 B == 0 ? 0xB1 : B == 1 ? 0x4E : 0x141,
                                                                 0xF, 0xF, false));
}
// Sum of a row's 128 values, pairwise by ascending column bit (the same bits whatever L is).
template <int L>
__device__ __forceinline__ float row_sum128(const f4_t (&v)[32 / L]) {
    float t[32 / L];
#pragma unroll
    for (int i = 0; i < 32 / L; ++i) {
        t[i] = (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
        t[i] += sub_xor<0>(t[i]);
        t[i] += sub_xor<1>(t[i]);
        if constexpr (L >= 8) t[i] += sub_xor<2>(t[i]);
    }
#pragma unroll
    for (int n = 16 / L; n > 0; n /= 2)
#pragma unroll
        for (int i = 0; i < n; ++i) t[i] = t[2 * i] + t[2 * i + 1];
    return t[0];
}
template <int L>
__device__ __forceinline__ void fwht128_lanes(f4_t (&v)[32 / L], int sub) {
    constexpr int N = 32 / L;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float a = v[i][0] + v[i][1], b = v[i][0] - v[i][1], c = v[i][2] + v[i][3], d = v[i][2] - v[i][3];
        v[i] = f4_t{a + c, b + d, a - c, b - d};
    }
    const float s0 = sub & 1 ? -1.f : 1.f, s1 = sub & 2 ? -1.f : 1.f, s2 = sub & 4 ? -1.f : 1.f;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float x = v[i][j];
            x = x * s0 + sub_xor<0>(x);
            x = x * s1 + sub_xor<1>(x);
            if constexpr (L >= 8) x = x * s2 + sub_xor<2>(x);
            v[i][j] = x;
        }
#pragma unroll
    for (int st = 1; st < N; st *= 2)
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (!(i & st)) {
                const f4_t a = v[i], b = v[i + st];
                v[i] = a + b;
                v[i + st] = a - b;
            }
}

// Floats per row of a 32 x 256 output tile in LDS, column c at c + 16 (c >> 7): the 16-byte reads of the lanes of a row and
// of the next row hit distinct banks.
constexpr int kWideCS = 288;

// One row group's accumulators of the workgroup (wave w: columns 64 w .. 64 w + 63) into the tile.
__device__ __forceinline__ void store_tile(float* C, const f16_t (&acc)[2], int wave, int lane) {
    const int cl = 64 * wave + (lane & 31) + 16 * (wave >> 1);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        C[r * kWideCS + cl] = acc[0][i];
        C[r * kWideCS + cl + 32] = acc[1][i];
    }
}
// The same of the 16-row form: tile column f, row 4 (lane >> 4) + i, column lane & 15.
__device__ __forceinline__ void store_tile16(float* C, const f4_t (&acc)[4], int wave, int lane) {
    const int cl = 64 * wave + (lane & 15) + 16 * (wave >> 1);
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) C[(4 * (lane >> 4) + i) * kWideCS + cl + 16 * f] = acc[f][i];
}

}  // namespace exl3
