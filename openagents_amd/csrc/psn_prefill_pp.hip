/*
 * psn_prefill_pp.hip -- gfx950 quantized prefill matmul, the kernel that decodes in its loop for tiles of 256 rows of X:
 * Y[m][n] = sum_k h(deq(W)[n][k]) * X[m][k], fp16 MFMA, fp32 accumulation.
 *
 * A workgroup of eight waves (two to a SIMD) owns a BM x BN tile of Y and walks K in steps of 64.  Every wave does every
 * kind of work, a little of it behind each of its MFMAs, so that the two waves of a SIMD fill each other's gaps: while
 * step s is multiplied out of LDS, the wave
 *   - reads the step's operand fragments, half a step before they are multiplied,
 *   - asks for its share of the X tile NS - 1 steps on (direct-to-LDS loads into a ring of NS stages; spread over the
 *     step because four in a row stall their wave for 500 cycles),
 *   - decodes its share of the weights of step s + 1 into the other one of two fp16 tiles.  A weight is decoded once per
 *     workgroup: a thread owns BN / 8 weights of one row per step, and their raw bytes come straight from memory into
 *     registers, asked for a whole 256-wide chunk ahead.
 * One barrier per step.  (Tiles of fewer rows: psn_prefill_frag.hip; its layout needs more registers and LDS than there are for 256 rows.)
 *
 * What bounds it, Q4_K 512 x 14336 x 4096: 69 us; 53 without the decode and its LDS writes, 53 without MFMAs, 57 without loads, so vector instructions, LDS traffic
 * (176 KB per step, 1.3 times as long as the MFMAs) and MFMAs add up; on a full chip power as well (on zero weights, the same instructions, a fifth faster), which is why the MFMAs
 * are 16 x 16 x 32 there (275 us -> 257 at M = 2048).  With fewer than about 180 workgroups power does not bind, the MFMAs that ride shorter do, and the _pp32 kernels multiply
 * 32 x 32 x 16, half as many: Q4_K, weights from memory, five formats and 110 matrices, geometric mean of 32 x 32 over 16 x 16 by workgroups (of 256 compute units): up to 100 1.07 x,
 * 132 .. 150 1.06, 150 .. 165 1.04, 165 .. 180 1.03, 180 .. 195 1.00, 195 .. 256 0.985, more 0.99.  Splitting the roles (eight multiplying and eight staging waves) measured 2-8 % slower, running the two waves of a SIMD in strictly opposite phases 10-15 %, sixteen
 * waves with half the tile each 15 %.
 */
#include "psn_args.h"
#include "psn_device.h"
#include "psn_prefill_common.h"
#include "psn_prefill_formats.h"

/* Which weight row a group of four threads decodes.  The lanes that write to LDS together (sixteen of 16 bytes) should
 * hit sixteen different columns, (row & 1) * 8 + (chunk ^ row bits 1..3); the lanes of one row hold chunks that leave one
 * or two chunk bits to the rows.  So the low bits of the group's number go to row bit 0 and to the row bits that scatter
 * those: SPREAD 0: bits 1, 2, 3 in order; 2: bit 2 first; 3: bit 3 first. */
template <int SPREAD> PSN_DEV int row_of(int idx) {
    const int b0 = idx & 1, b1 = (idx >> 1) & 1, b2 = (idx >> 2) & 1, b3 = (idx >> 3) & 1, high = idx & ~15;
    if constexpr (SPREAD == 2) return high | b0 | (b1 << 2) | (b2 << 1) | (b3 << 3);
    if constexpr (SPREAD == 3) return high | b0 | (b1 << 3) | (b2 << 1) | (b3 << 2);
    return idx;
}

template <int OFF> PSN_DEV void lds_write128o(u32 addr, u32x4 v) { asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(addr), "v"(v), "n"(OFF) : "memory"); }

/* does piece p of a decode (see there) end in an LDS write? */
constexpr bool pp_piece_writes(int p) { return p >= 2 && (p & 3) == 1; }

/* D = W X^T either way; KK: K slices per step */
template <int MF> struct pp_mfma;
template <> struct pp_mfma<16> {
    typedef f32x4 acc;
    static constexpr int KK = 2;
    static PSN_DEV acc mul(u32x4 w, u32x4 x, acc c) { return mfma16(w, x, c); }
    template <int TN> static constexpr int out_bytes() { return wave_out_bytes<TN>(); }
};
template <> struct pp_mfma<32> {
    typedef float16_t acc;
    static constexpr int KK = 4;
    static PSN_DEV acc mul(u32x4 w, u32x4 x, acc c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, w), __builtin_bit_cast(half8_t, x), c, 0, 0, 0); }
    template <int TN> static constexpr int out_bytes() { return wave_out_bytes32<TN>(); }
};

template <typename WF, int BM, int BN, int WM, int MF, int NS>
PSN_DEV void prefill_pp_body(const psn_prefill_args &a) {
    typedef pp_mfma<MF> MMA;
    constexpr int WN = 8 / WM, TM = BM / WM / MF, TN = BN / WN / MF, KK = MMA::KK;
    constexpr int NB = 8, PARTS = 4;                        /* quant bytes per thread and step, threads per weight row */
    static_assert(BN == 128, "512 threads, four to a row");
    constexpr int SPREAD = WF::SPREAD;
    constexpr int XBYTES = BM * 128, WBYTES = BN * 128;
    constexpr int NX = BM / 64;                             /* X loads per wave and step */
    static_assert(TM >= 1 && TN >= 1 && NX >= 1 && NS * XBYTES + 2 * WBYTES == psn_lds_in_loop(WF::FORMAT, BM, BN) && psn_lds_in_loop(WF::FORMAT, BM, BN) <= PSN_LDS_MAX && 8 * MMA::template out_bytes<TN>() <= NS * XBYTES, "tile");
    extern __shared__ uint4 psn_smem[];
    lds_char *const lds_ptr = (lds_char *)psn_smem;
    const u32 lds0 = (u32)(uintptr_t)lds_ptr;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int M = a.M, N = a.N, K = a.K;

    prefill_place at;
    if (!place_workgroup<BM, BN, 512>(a, at)) return;       /* whole workgroup leaves together */
    const int m0 = at.m0, n0 = at.n0, c_begin = at.c0, nq = at.chunks, nsteps = nq * 4;

    typename MMA::acc acc[TM][TN];
    UNROLL for (int i = 0; i < TM; ++i) UNROLL for (int j = 0; j < TN; ++j) acc[i][j] = (typename MMA::acc)(0.f);

    /* X: 16-byte word s of a stage in LDS order is row s / 8, position s % 8, which holds chunk (s % 8) ^ tile_swz(row) */
    u32 xoff[NX];
    UNROLL for (int u = 0; u < NX; ++u) {
        const int s_ = (wave * NX + u) * 64 + lane, row = s_ >> 3, chunk = (s_ & 7) ^ tile_swz(row);
        xoff[u] = (u32)min(m0 + row, M - 1) * (u32)(K * 2) + (u32)(chunk * 16);
    }
    const char *xbase = reinterpret_cast<const char *>(a.X) + (int64_t)c_begin * 512;
    auto issue_x = [&](int g, int u) {                      /* stages past the end repeat the last one, into a slot nothing reads any more */
        const char *xb = xbase + (int64_t)min(g, nsteps - 1) * 128;
        lds_char *xd = lds_ptr + (g % NS) * XBYTES + wave * (NX * 1024);
        __builtin_amdgcn_global_load_lds((const void *)(xb + xoff[u]), (__attribute__((address_space(3))) void *)(xd + u * 1024), 16, 0, 0);
    };

    /* W: this thread's part of its row */
    const int part = tid % PARTS, wrow = row_of<SPREAD>(tid / PARTS);
    const uint8_t *wsrc = a.W + (int64_t)min(n0 + wrow, N - 1) * a.row_bytes + (int64_t)c_begin * WF::BYTES;
    const int woff = WF::template lane_off<NB>(part);
    const u32 wtile = lds0 + (u32)(NS * XBYTES);
    const int kl = WF::template k_lo<NB>(part), kh = WF::template k_hi<NB>(part);
    const u32 wr_lo = wtile + (u32)tile_off(wrow, kl >> 3) + (u32)((kl & 7) * 2), wr_hi = wtile + (u32)tile_off(wrow, kh >> 3) + (u32)((kh & 7) * 2);
    typename WF::template raw<NB> wa, wb;                   /* chunks of even and of odd number */
    WF::template clear<NB>(wa);
    WF::template clear<NB>(wb);
    auto load_chunk = [&](int c, typename WF::template raw<NB> &r) {
        WF::template load<NB>(wsrc + (int64_t)min(c, nq - 1) * WF::BYTES, woff, r);
    };
    /* The decode of step J of a chunk, in pieces: the scales (two), then two per word of four weights; a finished 16 bytes
     * goes to fp16 tile J % 2. */
    constexpr int NW = NB / 4, PIECES = 2 + 4 * NW;
    u32 dec[4];
    half_done dhalf;
    typename WF::scale wscale;
    auto decode = [&](const typename WF::template raw<NB> &w, auto jc, auto pc) {
        constexpr int J = decltype(jc)::value, P = decltype(pc)::value, OFF = (J & 1) * WBYTES;
        if constexpr (P == 0) {
            WF::template scales0<J, NB>(w, part, wscale);
        } else if constexpr (P == 1) {
            WF::template scales1<J, NB>(w, wscale);
        } else {
            constexpr int WORD = (P - 2) >> 1, HI = WORD / NW, I = WORD % NW, B = 2 * I;
            if constexpr ((P & 1) == 0) {
                WF::template first<J, NB, HI>(w, wscale, I, dhalf);
            } else {
                WF::template second<HI>(wscale, dhalf, dec[B], dec[B + 1]);
                if constexpr (B == 2) lds_write128o<OFF>(HI ? wr_hi : wr_lo, (u32x4){dec[0], dec[1], dec[2], dec[3]});
            }
        }
    };

    /* fragment addresses: row (lane % MF) of the wave tile, 16-byte chunk KF kk + lane / MF, swizzled */
    constexpr int KF = 64 / MF;                             /* chunks per K slice: 2 or 4 */
    u32 fx[KK], fw[KK];
    UNROLL for (int kk = 0; kk < KK; ++kk) {
        fx[kk] = lds0 + (u32)tile_off(wm * (BM / WM) + lane % MF, KF * kk + lane / MF);
        fw[kk] = wtile + (u32)tile_off(wn * (BN / WN) + lane % MF, KF * kk + lane / MF);
    }
    /* Operands of a whole step: K slices 0 .. KK - 1 in sets of their own.  They run half a step behind the reads: period p
     * reads step p and multiplies the second half of step p - 1, then the first half of step p, so that a fragment has the
     * time of KK / 2 slices to arrive. */
    constexpr int HK = KK / 2;
    u32x4 xf[KK][TM], wf[KK][TN];
    UNROLL for (int kk = 0; kk < KK; ++kk) { UNROLL for (int i = 0; i < TM; ++i) xf[kk][i] = (u32x4)(0u); UNROLL for (int j = 0; j < TN; ++j) wf[kk][j] = (u32x4)(0u); }
    constexpr int FR = TM + TN, READS = KK * FR;            /* fragments per slice (those of W first) and per step */
    auto read_frag = [&](u32 xslot, auto jc, auto rc) {
        constexpr int R = decltype(rc)::value, kk = R / FR, I = R % FR, OFF = (decltype(jc)::value & 1) * WBYTES;
        if constexpr (I < TN) wf[kk][I] = lds_read128<OFF + I * 128 * MF>(fw[kk]);
        else xf[kk][I - TN] = lds_read128<(I - TN) * 128 * MF>(fx[kk] + xslot);
    };

    /* What rides behind the NPOS MFMAs of a period, spread evenly (a wave that issues several LDS or memory instructions in a
     * row waits for the queue they go into, and its SIMD's matrix pipe with it): the fragment reads of step p, its share of
     * the X loads of step p + NS - 1, the pieces of the decode of step p + 1.  The last few MFMAs carry nothing, so that what
     * the barrier waits for has come in. */
    constexpr int NPOS = KK * TM * TN, NRIDE = NPOS - (NPOS >= 8 ? 2 : 0);
    constexpr auto read_pos = [](int r) constexpr { return r * NRIDE / READS; };
    constexpr auto piece_pos = [](int p) constexpr { return p * NRIDE / PIECES; };
    /* LDS operations issued in front of MFMA `pos` that are younger than the reads of slice kk (in a position: reads first) */
    constexpr auto younger = [](int kk, int pos) constexpr {
        const int last = (kk + 1) * FR - 1, from = last * NRIDE / READS;
        int n = 0;
        for (int r = last + 1; r < READS; ++r) n += r * NRIDE / READS < pos;
        for (int p = 0; p < PIECES; ++p) {
            const int at = p * NRIDE / PIECES;
            n += pp_piece_writes(p) && at >= from && at < pos;
        }
        return n > 15 ? 15 : n;                             /* (four bits of counter: waiting for more than needed is harmless) */
    };
    auto ride = [&](int c, const typename WF::template raw<NB> &w, auto jc, auto qc) {
        constexpr int J = decltype(jc)::value, Q = decltype(qc)::value, NEXT = (J + 1) & 3;
        const u32 xslot = (u32)(((4 * c + J) % NS) * XBYTES);
#define PSN_PP_READ(R) if constexpr (R < READS && read_pos(R) == Q) read_frag(xslot, jc, pf_int<R>());
        PSN_PP_READ(0) PSN_PP_READ(1) PSN_PP_READ(2) PSN_PP_READ(3) PSN_PP_READ(4) PSN_PP_READ(5) PSN_PP_READ(6) PSN_PP_READ(7)
        PSN_PP_READ(8) PSN_PP_READ(9) PSN_PP_READ(10) PSN_PP_READ(11) PSN_PP_READ(12) PSN_PP_READ(13) PSN_PP_READ(14) PSN_PP_READ(15)
#undef PSN_PP_READ
        UNROLL for (int u = 0; u < NX; ++u)
            if (u * NRIDE / NX == Q) issue_x(4 * c + J + NS - 1, u);
#define PSN_PP_PIECE(P) if constexpr (P < PIECES && piece_pos(P) == Q) decode(w, pf_int<NEXT>(), pf_int<P>());
        PSN_PP_PIECE(0) PSN_PP_PIECE(1) PSN_PP_PIECE(2) PSN_PP_PIECE(3) PSN_PP_PIECE(4) PSN_PP_PIECE(5) PSN_PP_PIECE(6) PSN_PP_PIECE(7) PSN_PP_PIECE(8) PSN_PP_PIECE(9)
#undef PSN_PP_PIECE
    };
    static_assert(READS <= 16 && PIECES <= 10, "rides");
    auto multiply = [&](auto kc, auto &&behind) {
        constexpr int kk = decltype(kc)::value;
        UNROLL for (int j = 0; j < TN; ++j) UNROLL for (int i = 0; i < TM; ++i) {
            __builtin_amdgcn_sched_barrier(0);
            acc[i][j] = MMA::mul(wf[kk][j], xf[kk][i], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
            behind(j * TM + i);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    /* slice Q of period p = 4 c + J: multiplies K slice (Q + HK) % KK, of step p - 1 while Q < HK */
    auto slice = [&](int c, const typename WF::template raw<NB> &w, auto jc, auto qc) {
        constexpr int Q = decltype(qc)::value, kk = (Q + HK) % KK;
        if constexpr (Q >= HK) {
            static_assert(((kk + 1) * FR - 1) * NRIDE / READS < Q * TM * TN, "read before it is multiplied");
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(younger(kk, Q * TM * TN)) : "memory");
            tie(xf[kk]);
            tie(wf[kk]);
        }
        multiply(pf_int<kk>(), [&](int pos) {
#define PSN_PP_RIDE(P) if (pos == P) { if constexpr (P < TM * TN) ride(c, w, jc, pf_int<Q * TM * TN + P>()); }
            PSN_PP_RIDE(0) PSN_PP_RIDE(1) PSN_PP_RIDE(2) PSN_PP_RIDE(3) PSN_PP_RIDE(4) PSN_PP_RIDE(5) PSN_PP_RIDE(6) PSN_PP_RIDE(7)
            PSN_PP_RIDE(8) PSN_PP_RIDE(9) PSN_PP_RIDE(10) PSN_PP_RIDE(11) PSN_PP_RIDE(12) PSN_PP_RIDE(13) PSN_PP_RIDE(14) PSN_PP_RIDE(15)
#undef PSN_PP_RIDE
        });
    };
    /* (a set is read into only after its last use: slice kk >= HK is multiplied in slices 0 .. KK - HK - 1 of the period) */
    UNROLL for (int kk = HK; kk < KK; ++kk) {
        constexpr auto ok = [](int k) constexpr { return k * FR * NRIDE / READS >= (k - HK + 1) * TM * TN - 1; };
        static_assert(ok(HK) && ok(KK - 1), "fragment sets overlap");
    }

    load_chunk(0, wa);
    UNROLL for (int g = 0; g < NS - 1; ++g) UNROLL for (int u = 0; u < NX; ++u) issue_x(g, u);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    WF::template landed<NB>(wa);
    load_chunk(1, wb);
#define PSN_PP_PIECE(P) if constexpr (P < PIECES) decode(wa, pf_int<0>(), pf_int<P>());
    PSN_PP_PIECE(0) PSN_PP_PIECE(1) PSN_PP_PIECE(2) PSN_PP_PIECE(3) PSN_PP_PIECE(4) PSN_PP_PIECE(5) PSN_PP_PIECE(6) PSN_PP_PIECE(7) PSN_PP_PIECE(8) PSN_PP_PIECE(9)
#undef PSN_PP_PIECE
    lds_barrier();

    /* Period p = 4 c + J, between two barriers.  Nobody touches the stage of X of step p - 1 nor the fp16 tile of step p - 1
     * any more, which are the ones that X of step p + NS - 1 and the weights of step p + 1 go to.  Its end: X of step p + 1 has
     * landed -- everything but the X loads of the NS - 2 steps after it and, where they are younger, the raw loads (which go
     * first in periods J = 3) -- and this wave's reads and writes of LDS are done. */
#define PSN_PP_STEP(J, w, wother)                                                                                          \
    {                                                                                                                      \
        if constexpr (J == 3) {                                                                                            \
            load_chunk(c + 2, w);                                                                                          \
            WF::template landed<NB>(wother);                                                                               \
        }                                                                                                                  \
        slice(c, J == 3 ? wother : w, pf_int<J>(), pf_int<0>());                                                           \
        slice(c, J == 3 ? wother : w, pf_int<J>(), pf_int<1>());                                                           \
        if constexpr (KK == 4) {                                                                                           \
            slice(c, J == 3 ? wother : w, pf_int<J>(), pf_int<KK - 2>());                                                  \
            slice(c, J == 3 ? wother : w, pf_int<J>(), pf_int<KK - 1>());                                                  \
        }                                                                                                                  \
        constexpr int KEEP = (NS - 2) * NX + ((J + 1) % 4 < NS - 2 ? WF::LOADS : 0);                                       \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(KEEP) : "memory");                               \
        UNROLL for (int kk = HK; kk < KK; ++kk) { tie(xf[kk]); tie(wf[kk]); }                                              \
    }
#define PSN_PP_CHUNK(w, wother) PSN_PP_STEP(0, w, wother) PSN_PP_STEP(1, w, wother) PSN_PP_STEP(2, w, wother) PSN_PP_STEP(3, w, wother)
    int c = 0;
    for (; c + 1 < nq; ++c) {
        PSN_PP_CHUNK(wa, wb)
        ++c;
        PSN_PP_CHUNK(wb, wa)
    }
    if (c < nq) { PSN_PP_CHUNK(wa, wb) }
#undef PSN_PP_CHUNK
#undef PSN_PP_STEP
    multiply(pf_int<HK>(), [](int) {});
    if constexpr (KK == 4) multiply(pf_int<KK - 1>(), [](int) {});
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");       /* nothing is on its way into LDS any more */
    /* the last raw loads were for nothing, but their registers belong to them until they have landed */
    WF::template landed<NB>(wa);
    WF::template landed<NB>(wb);

    /* (worked out again from an opaque thread index, so that nothing of it stays in a register through the loop) */
    int tid_out = threadIdx.x;
    asm volatile("" : "+v"(tid_out));
    const int wm_o = (tid_out >> 6) / WN, wn_o = (tid_out >> 6) % WN, lane_o = tid_out & 63;
    UNROLL for (int i = 0; i < TM; ++i)
        store_tiles<TN>(a, m0 + wm_o * (BM / WM) + MF * i, n0 + wn_o * (BN / WN), lane_o, acc[i], lds0 + (u32)((tid_out >> 6) * MMA::template out_bytes<TN>()));
}


#define PSN_PP(fmt, suffix, WF, BM, BN, WM, MF, NS)                                                                          \
    extern "C" __global__ void __launch_bounds__(512) psn_prefill_##fmt##_m##BM##_n##BN##_pp##suffix(const psn_prefill_args a) { \
        prefill_pp_body<WF, BM, BN, WM, MF, NS>(a);                                                                          \
    }
#define PSN_PP_FAMILY(fmt, WF) PSN_PP(fmt, , WF, 256, 128, 4, 16, 4) PSN_PP(fmt, 32, WF, 256, 128, 4, 32, 4)

#ifdef PSN_BUILD_PP_Q4_0
PSN_PP_FAMILY(q4_0, PpQ4_0)
#endif
#ifdef PSN_BUILD_PP_Q8_0
PSN_PP_FAMILY(q8_0, PpQ8_0)
#endif
#ifdef PSN_BUILD_PP_Q4_K
PSN_PP_FAMILY(q4_K, PpQ4_K)
#endif
#ifdef PSN_BUILD_PP_Q5_K
PSN_PP_FAMILY(q5_K, PpQ5_K)
#endif
#ifdef PSN_BUILD_PP_Q6_K
PSN_PP_FAMILY(q6_K, PpQ6_K)
#endif
