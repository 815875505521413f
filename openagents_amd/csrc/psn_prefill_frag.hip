/*
 * psn_prefill_frag.hip -- gfx950 quantized prefill matmul, the kernels that decode in their loop, tiles of at most 128 rows of X:
 * Y[m][n] = sum_k h(deq(W)[n][k]) * X[m][k], fp16 MFMA, fp32 accumulation.
 *
 * A workgroup of eight waves owns a BM x BN tile of Y.  Four pairs of waves take BN / 4 weight rows each, all BM rows of X; one wave of a pair multiplies the first half of
 * every 256-wide chunk of K, the other the second, and their sums meet in LDS at the end.  So every wave decodes the MFMA operands that it multiplies, and nobody else needs them:
 * decoded weights stay in registers, a weight is decoded once per workgroup, and a fragment of X is read from LDS once per 16 TN weight rows.
 *   - X (a step of 64 k of either half: whole 128-byte lines) and the raw chunks of the weight rows (consecutive lanes on consecutive 16-byte words) arrive by direct-to-LDS loads, two
 *     stages and two chunks deep.
 *   - A period is one step of 64 k of each half.  In its first half a wave multiplies the operands of the step's lower k (the low nibbles), in its second those of the upper; behind every
 *     MFMA ride the reads of the X fragments for the other half, loads, and a piece of the decode of the operand after this one.  One barrier per period, between the
 *     halves, where nobody reads the period's stage of X any more.
 *   - Q4_K and Q5_K: a lane unpacks the scales of one of the chunk's four (tile, step) pairs and hands them to the other lanes of its row through LDS.
 *
 * What bounds it: issue.  Q4_K 256 x 14336 x 4096, 128 x 128 tiles, 48 us with decoded weights in LDS (the kernels before, psn_prefill_pp.hip): 31 us without the decode and its LDS
 * writes, 40 without MFMAs, 40 without loads -- vector instructions, MFMAs and LDS traffic (128 KB per 64 k, as long as the MFMAs twice over) added up instead of
 * overlapping.  Here 39 us: LDS traffic 80 KB, no wait between decode and use, 24 loads of whole words per chunk instead of 40 that touch sixteen rows each (asked
 * for by row from memory, as those kernels do, 44 us).  Against them, us: Q4_K 512 x 4096 x 4096 39 -> 29, 130 x 4096 x 4096 23 -> 19; Q4_0 256 x 14336 x 4096 44 -> 36;
 * Q8_0 52 -> 41; Q5_K 50 -> 42; Q6_K, whose super-blocks need v_perm for every word, 51 -> 47.  Three stages of X instead of two changed nothing.
 */
#include "psn_args.h"
#include "psn_device.h"
#include "psn_prefill_common.h"
#include "psn_prefill_formats.h"

/* ---- what one lane takes out of a weight row's chunk in LDS for one 64-wide step, part `q` of four (the steps 2 half and 2 half + 1 are one wave's) ---- */
struct FragQ4_K {
    typedef PpQ4_K F;
    static constexpr int WORDS = 9, STRIDE = 144;
    static constexpr bool SHARED = true, PASSED = false;
    struct raw { u32x2 q; };
    struct scale { float d[2], m[2]; };
    template <int H> static PSN_DEV void read(u32 chunk, u32, int half, int q, raw &r) { r.q = lds_read64o<16 + 32 * H>(chunk + (u32)(64 * half + 8 * q)); }
    static PSN_DEV void landed(raw &r) { raw_tie(r.q); }
    template <int H> static PSN_DEV void scales(const raw &, u32, int, scale &) {}
    template <int H, int HI> static PSN_DEV void first(const raw &r, const scale &, u32, int, int i, half_done &t) { kq_floats((r.q[i] >> (4 * HI)) & 0x0f0f0f0fu, t); }
    template <int HI> static PSN_DEV void second(const scale &s, const half_done &t, u32 &o0, u32 &o1) { kq_finish(t, s.d[HI], s.m[HI], o0, o1); }
};
struct FragQ5_K {
    typedef PpQ5_K F;
    static constexpr int WORDS = 11, STRIDE = 176;
    static constexpr bool SHARED = true, PASSED = false;
    struct raw { u32x2 q, top; };
    struct scale { float d[2], m[2]; };
    template <int H> static PSN_DEV void read(u32 chunk, u32, int half, int q, raw &r) {
        r.q = lds_read64o<48 + 32 * H>(chunk + (u32)(64 * half + 8 * q));
        r.top = lds_read64o<16>(chunk + (u32)(8 * q));
    }
    static PSN_DEV void landed(raw &r) { raw_tie(r.q); raw_tie(r.top); }
    template <int H> static PSN_DEV void scales(const raw &, u32, int, scale &) {}
    template <int H, int HI> static PSN_DEV void first(const raw &r, const scale &, u32, int half, int i, half_done &t) {
        kq_floats(((r.q[i] >> (4 * HI)) & 0x0f0f0f0fu) | (((r.top[i] >> (4 * half + 2 * H + HI)) & 0x01010101u) << 4), t);
    }
    template <int HI> static PSN_DEV void second(const scale &s, const half_done &t, u32 &o0, u32 &o1) { kq_finish(t, s.d[HI], s.m[HI], o0, o1); }
};
struct FragQ4_0 {
    typedef PpQ4_0 F;
    static constexpr int WORDS = 9, STRIDE = 144;
    static constexpr bool SHARED = false, PASSED = false;
    struct raw { u32x2 q; u32 q2; };
    struct scale { u32 d, q[2]; };
    template <int H> static PSN_DEV void read(u32 chunk, u32, int half, int q, raw &r) {
        const u32 p = chunk + (u32)(72 * half + 8 * q);
        r.q = lds_read2_b32<9 * H, 9 * H + 1>(p);
        r.q2 = lds_read32o<36 * H + 8>(p);
    }
    static PSN_DEV void landed(raw &r) { raw_tie(r.q); raw_tie(r.q2); }
    template <int H> static PSN_DEV void scales(const raw &r, u32, int q, scale &s) {
        typedef pp_blocks<8, 8> B;
        s.d = B::scale<true>(r.q[0], q);
        s.q[0] = __builtin_amdgcn_perm(r.q[1], r.q[0], B::pick(q));
        s.q[1] = __builtin_amdgcn_perm(r.q2, r.q[1], B::pick(q));
    }
    template <int H, int HI> static PSN_DEV void first(const raw &, const scale &s, u32, int, int i, half_done &t) { q0_halves(s.q[i] >> (4 * HI), 0x640f640fu, t); }
    template <int HI> static PSN_DEV void second(const scale &s, const half_done &t, u32 &o0, u32 &o1) { q0_finish(t, 0x64086408u, s.d, o0, o1); }
};

struct FragQ8_0 {
    typedef PpQ8_0 F;
    static constexpr int WORDS = 17, STRIDE = 272;
    static constexpr bool SHARED = false, PASSED = false;
    struct raw { u32x2 a, b; u32 e; };
    struct scale { u32 d, pick; };
    template <int H> static PSN_DEV void read(u32 chunk, u32, int half, int q, raw &r) {
        const u32 p = chunk + (u32)(136 * half + 16 * q);
        r.a = lds_read2_b32<17 * H, 17 * H + 1>(p);
        r.b = lds_read2_b32<17 * H + 2, 17 * H + 3>(p);
        r.e = lds_read32o<68 * H + 16>(p);
    }
    static PSN_DEV void landed(raw &r) { raw_tie(r.a); raw_tie(r.b); raw_tie(r.e); }
    template <int H> static PSN_DEV void scales(const raw &r, u32, int q, scale &s) {
        typedef pp_blocks<16, 8> B;
        s.d = B::scale<true>(r.a[0], q);
        s.pick = B::pick(q);
    }
    template <int H, int HI> static PSN_DEV void first(const raw &r, const scale &s, u32, int, int i, half_done &t) {
        const u32 w[5] = {r.a[0], r.a[1], r.b[0], r.b[1], r.e};
        const int at = HI * 2 + i;
        q0_halves(__builtin_amdgcn_perm(w[at + 1], w[at], s.pick) ^ 0x80808080u, 0x64ff64ffu, t);
    }
    template <int HI> static PSN_DEV void second(const scale &s, const half_done &t, u32 &o0, u32 &o1) { q0_finish(t, 0x64806480u, s.d, o0, o1); }
};

/* Super-blocks of 210 bytes that start on a dword or between two (`pick` takes four bytes out of two dwords accordingly), so they cannot be copied whole: 13 words from the dword on in
 * which the super-block starts, and apart from them (through registers) the dword with its last two scales where it starts two bytes late, and its d. */
struct FragQ6_K {
    typedef PpQ6_K F;
    static constexpr int WORDS = 13, STRIDE = 208;
    static constexpr bool SHARED = false, PASSED = true;
    struct raw { u32x2 a, b, h, sc; u32 a2, b2, h2, sc2, d; };
    struct scale { float d[2], m[2]; };
    template <int H> static PSN_DEV void read(u32 chunk, u32 extra, int half, int q, raw &r) {
        const u32 p = chunk + (u32)(64 * half + 8 * q), h = chunk + (u32)(128 + 32 * half + 8 * q), s = chunk + (u32)(192 + 8 * half);
        r.a = lds_read64o<0>(p);
        r.a2 = lds_read32o<8>(p);
        r.b = lds_read64o<32>(p);
        r.b2 = lds_read32o<40>(p);
        r.h = lds_read64o<0>(h);
        r.h2 = lds_read32o<8>(h);
        r.sc = lds_read64o<0>(s);
        r.sc2 = lds_read32o<0>(half ? extra : s + 8);
        r.d = lds_read32o<4>(extra);
    }
    static PSN_DEV void landed(raw &r) { raw_tie(r.a); raw_tie(r.a2); raw_tie(r.b); raw_tie(r.b2); raw_tie(r.h); raw_tie(r.h2); raw_tie(r.sc); raw_tie(r.sc2); raw_tie(r.d); }
    template <int H> static PSN_DEV void scales(const raw &r, u32 pick, int q, scale &s) {
        const u32 v = __builtin_amdgcn_perm(H ? r.sc2 : r.sc[1], r.sc[H], pick) >> (8 * (q >> 1));
        const float d = h2f_lo(r.d);
        s.d[0] = __fmul_rn(d, (float)(int)(int8_t)(v & 0xffu));
        s.d[1] = __fmul_rn(d, (float)(int)(int8_t)((v >> 16) & 0xffu));
        s.m[0] = s.d[0] * 32.f;
        s.m[1] = s.d[1] * 32.f;
    }
    template <int H, int HI> static PSN_DEV void first(const raw &r, const scale &, u32 pick, int, int i, half_done &t) {
        const u32x2 l = HI ? r.b : r.a;
        const u32 l2 = HI ? r.b2 : r.a2;
        const u32 low = __builtin_amdgcn_perm(i ? l2 : l[1], l[i], pick), high = __builtin_amdgcn_perm(i ? r.h2 : r.h[1], r.h[i], pick);
        kq_floats(((low >> (4 * H)) & 0x0f0f0f0fu) | (((high >> (4 * H + 2 * HI)) & 0x03030303u) << 4), t);
    }
    template <int HI> static PSN_DEV void second(const scale &s, const half_done &t, u32 &o0, u32 &o1) { kq_finish(t, s.d[HI], s.m[HI], o0, o1); }
};

template <typename RF, int TM, int TN>
PSN_DEV void prefill_frag_body(const psn_prefill_args &a) {
    typedef typename RF::F F;
    constexpr int BM = 16 * TM, BN = 64 * TN, XB = BM * 256;          /* a stage of X: one step of either half of a chunk */
    constexpr int STRIDE = RF::STRIDE;
    constexpr int LX = BM / 32, LW = (BN * RF::WORDS + 511) / 512;    /* loads per wave: X per period, W per chunk */
    constexpr int NI = (BN * RF::WORDS + 63) / 64;                    /* 1 KB pieces of a chunk; loads of waves past them go to one more, which nothing reads */
    constexpr int W0 = 2 * XB, WBUF = (NI + 1) * 1024 + (RF::PASSED ? BN * 8 : 0), SC0 = W0 + 2 * WBUF, SCW = RF::SHARED ? TN * 512 : 0;
    static_assert(TM % 4 == 0 && (TN == 1 || TN == 2) && SC0 + 8 * SCW <= PSN_LDS_MAX, "tile");
    static_assert(SC0 + 8 * SCW == psn_lds_in_loop(F::FORMAT, BM, BN) && 4 * TM * TN * 1024 + 8 * wave_out_bytes<TN>() <= SC0 + 8 * SCW, "LDS of the launch; the sums and results at the end");
    static_assert(RF::WORDS == psn_lds_words(F::FORMAT) && RF::SHARED == psn_lds_scales(F::FORMAT), "format");
    extern __shared__ uint4 psn_smem[];
    lds_char *const lds_ptr = (lds_char *)psn_smem;
    const u32 lds0 = (u32)(uintptr_t)lds_ptr;
    const int lane = threadIdx.x & 63, row = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = wave & 1, wn = wave >> 1;
    const int M = a.M, N = a.N, K = a.K;
    prefill_place at;
    if (!place_workgroup<BM, BN, 512>(a, at)) return;                 /* whole workgroup leaves together */
    const int m0 = at.m0, n0 = at.n0, nq = at.chunks;

    f32x4 acc[TM][TN];
    UNROLL for (int i = 0; i < TM; ++i) UNROLL for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4)(0.f);

    u32 xoff[LX];
    UNROLL for (int u = 0; u < LX; ++u) {
        const int c = wave * LX + u, sub = c / (BM / 8), r = (c % (BM / 8)) * 8 + (lane >> 3), piece = (lane & 7) ^ tile_swz(r);
        xoff[u] = (u32)min(m0 + r, M - 1) * (u32)(K * 2) + (u32)(sub * 256 + piece * 16);
    }
    const char *const xb = reinterpret_cast<const char *>(a.X) + (int64_t)at.c0 * 512;
    auto issue_x = [&](int c, int h, u32 slot, int u) {               /* chunks past the end repeat the last one, into slots nothing reads any more */
        load_to_lds(xb + (int64_t)min(c, nq - 1) * 512 + h * 128 + xoff[u], lds_ptr + slot + (wave * LX + u) * 1024);
    };
    /* W: consecutive lanes on consecutive 16-byte words of the tile's rows (words past the last repeat it) */
    u32 woff[LW];
    UNROLL for (int u = 0; u < LW; ++u) {
        const int word = min((wave * LW + u) * 64 + lane, BN * RF::WORDS - 1), r = word / RF::WORDS;
        woff[u] = (u32)min(n0 + r, N - 1) * (u32)a.row_bytes + (u32)(word % RF::WORDS * 16);
    }
    const uint8_t *const wb = a.W + (int64_t)at.c0 * F::BYTES;
    auto issue_w = [&](int c, int buf, int u) {
        load_to_lds((const char *)(wb + (int64_t)min(c, nq - 1) * F::BYTES + woff[u]), lds_ptr + W0 + buf * WBUF + min(wave * LW + u, NI) * 1024);
    };
    /* Q6_K's last words of a row: asked for like the others, written to LDS a period later (a row to a thread; the threads without one repeat the first, which costs no traffic) */
    u32 tail = 0, wd = 0;
    const int trow = (int)threadIdx.x < BN ? (int)threadIdx.x : 0;
    const u32 toff = (u32)min(n0 + trow, N - 1) * (u32)a.row_bytes;
    auto pass_load = [&](int c, int buf, int u) {
        const uint8_t *const at_c = wb + (int64_t)min(c, nq - 1) * F::BYTES;
        if (u < LW) load_to_lds((const char *)((uintptr_t)(at_c + woff[u < LW ? u : 0]) & ~(uintptr_t)3), lds_ptr + W0 + buf * WBUF + min(wave * LW + u, NI) * 1024);
        else if (u == LW) raw_load<204>((const uint8_t *)((uintptr_t)(at_c + toff + 2) & ~(uintptr_t)3), tail);
        else raw_load_u16<208>(at_c + toff, wd);
    };
    auto pass_landed = [&]() { if constexpr (RF::PASSED) { tie1(tail); tie1(wd); } };
    auto pass_store = [&](u32 buf) {
        const u32 to = lds0 + (u32)(W0 + (NI + 1) * 1024 + trow * 8) + buf;
        lds_write32(to, tail);
        lds_write32(to + 4, wd);
    };
    constexpr int NWL = RF::PASSED ? LW + 2 : LW;                     /* loads of W per chunk */
    /* Q6_K: whether this lane's super-blocks start on a dword, by tile; the other way round in the next chunk */
    u32 pick[TN];
    UNROLL for (int t = 0; t < TN; ++t)
        pick[t] = RF::PASSED && ((uintptr_t)(wb + (u32)min(n0 + (wn * TN + t) * 16 + row, N - 1) * (u32)a.row_bytes) & 2) ? 0x05040302u : 0x03020100u;
    /* scales: lane (q, row) works out those of tile q & 1, step 2 half + (q >> 1) (TN = 1: step 2 half + (q & 1)) */
    const int ht = TN == 2 ? q & 1 : 0, hh = TN == 2 ? q >> 1 : q & 1;
    const u32 head = lds0 + (u32)(W0 + ((wn * TN + ht) * 16 + row) * STRIDE), wrow = lds0 + (u32)(W0 + (wn * TN * 16 + row) * STRIDE);
    const u32 erow = lds0 + (u32)(W0 + (NI + 1) * 1024 + (wn * TN * 16 + row) * 8);
    const u32 sc_write = lds0 + (u32)(SC0 + wave * SCW + ((ht * 2 + hh) * 16 + row) * 16), sc_read = lds0 + (u32)(SC0 + wave * SCW + row * 16);
    u32x4 head_words = (u32x4)(0u);
    u32 pick_sc = 0, pick_mn = 0;
    auto read_head = [&](u32 buf) { if constexpr (RF::SHARED) head_words = lds_read128<0>(head + buf); };
    auto own0 = [&]() { if constexpr (RF::SHARED) kq_pick(head_words, 2 * half + hh, pick_sc, pick_mn); };
    auto own1 = [&]() {
        if constexpr (RF::SHARED) {
            float own[4];
            kq_own(head_words, pick_sc, pick_mn, own);
            lds_write128(sc_write, __builtin_bit_cast(u32x4, (f32x4){own[0], own[1], own[2], own[3]}));
        }
    };
    u32x4 sr[2][TN];                                                  /* scales of period h's tiles */
    typename RF::raw raw[2][TN];
    auto read_scale = [&](auto hc, auto tc) {
        constexpr int H = decltype(hc)::value, T = decltype(tc)::value;
        if constexpr (RF::SHARED) sr[H][T] = lds_read128<(T * 2 + H) * 256>(sc_read);
    };
    auto read_raw = [&](u32 buf, auto hc, auto tc) {
        constexpr int H = decltype(hc)::value, T = decltype(tc)::value;
        RF::template read<H>(wrow + buf + (u32)(T * 16 * STRIDE), erow + buf + (u32)(T * 128), half, q, raw[H][T]);
    };

    const u32 flo = lds0 + (u32)(half * (BM * 128) + tile_off(row, F::template k_lo<8>(q) >> 3)), fhi = lds0 + (u32)(half * (BM * 128) + tile_off(row, F::template k_hi<8>(q) >> 3));
    u32x4 xf[2][TM], wf[2];
    typename RF::scale ws[TN];
    half_done hd;
    u32 dec[4];
    /* piece P (0 .. 3) of fragment FR (slice FR / TN, tile FR % TN) of period H */
    auto decode = [&](auto hc, auto fc, auto pc) {
        constexpr int H = decltype(hc)::value, FR = decltype(fc)::value, P = decltype(pc)::value, HI = FR / TN, T = FR % TN, W = P >> 1;
        if constexpr (P == 0 && HI == 0) {
            if constexpr (RF::SHARED) {
                const f32x4 v = __builtin_bit_cast(f32x4, sr[H][T]);
                ws[T].d[0] = v[0]; ws[T].d[1] = v[1]; ws[T].m[0] = v[2]; ws[T].m[1] = v[3];
            } else RF::template scales<H>(raw[H][T], pick[T], q, ws[T]);
        }
        if constexpr ((P & 1) == 0) RF::template first<H, HI>(raw[H][T], ws[T], pick[T], half, W, hd);
        else RF::template second<HI>(ws[T], hd, dec[2 * W], dec[2 * W + 1]);
        if constexpr (P == 3) wf[FR & 1] = (u32x4){dec[0], dec[1], dec[2], dec[3]};
    };

    /* what the first period finds: chunks 0 and 1 of W and both stages of chunk 0 of X asked for, in this order (Q6_K: chunk 0 in LDS, chunk 1 in registers) */
    if constexpr (RF::PASSED) {
        UNROLL for (int u = 0; u < NWL; ++u) pass_load(0, 0, u);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        pass_landed();
        pass_store(0);
    } else UNROLL for (int u = 0; u < LW; ++u) issue_w(0, 0, u);
    UNROLL for (int u = 0; u < LX; ++u) issue_x(0, 0, 0, u);
    if constexpr (RF::PASSED) UNROLL for (int u = 0; u < NWL; ++u) pass_load(1, 1, u);
    else UNROLL for (int u = 0; u < LW; ++u) issue_w(1, 1, u);
    UNROLL for (int u = 0; u < LX; ++u) issue_x(0, 1, XB, u);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(RF::PASSED ? LX : LX + LW) : "memory");
    pass_landed();
    lds_barrier();
    read_head(0);
    static_for<0, TN>([&](auto tc) { read_raw(0, pf_int<0>(), tc); });
    static_for<0, TM>([&](auto ic) { constexpr int i = decltype(ic)::value; xf[0][i] = lds_read128<i * 2048>(flo); });
    lds_wait();
    raw_tie(head_words);
    UNROLL for (int t = 0; t < TN; ++t) RF::landed(raw[0][t]);
    own0();
    own1();
    static_for<0, TN>([&](auto tc) { read_scale(pf_int<0>(), tc); });
    lds_wait();
    tie(xf[0]);
    if constexpr (RF::SHARED) UNROLL for (int t = 0; t < TN; ++t) raw_tie(sr[0][t]);
    static_for<0, 4>([&](auto pc) { decode(pf_int<0>(), pf_int<0>(), pc); });

    u32 xs = 0, wc = 0;                                               /* slot of the period's stage of X, buffer of the chunk */
    constexpr int NPOS = 2 * TN * TM, SL = TN * TM, READ_BY = SL * 3 / 4;
    auto period = [&](int c, auto hc) {
        constexpr int H = decltype(hc)::value;
        const u32 xn = XB - xs, wo = WBUF - wc;
        static_for<0, NPOS>([&](auto pc) {
            constexpr int P = decltype(pc)::value, FR = P / TM, I = P % TM, S = FR / TN, T = FR % TN, PS = P - S * SL;
            if constexpr (S == 1 && PS == 0) {
                /* The next stage of X has landed, in the first period the next chunk of W too; nobody reads this stage any more, nor in the first period this chunk's raw bytes. */
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(H ? NWL : 0) : "memory");
                tie(xf[1]);
                UNROLL for (int t = 0; t < TN; ++t) { if constexpr (RF::SHARED) raw_tie(sr[1 - H][t]); RF::landed(raw[1 - H][t]); }
            }
            __builtin_amdgcn_sched_barrier(0);
            acc[I][T] = mfma16(wf[FR & 1], xf[S][I], acc[I][T]);
            __builtin_amdgcn_sched_barrier(0);
            /* the second period takes the next chunk's scales first: they pass through LDS once more before their first use */
            if constexpr (S == 0 && H == 1 && PS == 0) own0();
            if constexpr (S == 0 && H == 1 && PS == 1) own1();
            if constexpr (RF::PASSED && S == 0 && H == 0 && PS == 0) pass_store(wo);
            static_for<0, TM>([&](auto rc) {                          /* fragments of X: of the stage's second half, then of the next stage's first */
                constexpr int R = decltype(rc)::value;
                if constexpr (R * READ_BY / TM == PS) xf[1 - S][R] = S == 0 ? lds_read128<R * 2048>(fhi + xs) : lds_read128<R * 2048>(flo + xn);
            });
            if constexpr (S == 0) {
                static_for<0, TN>([&](auto tc) {
                    if constexpr (PS == 1 + decltype(tc)::value) read_raw(H ? wo : wc, pf_int<1 - H>(), tc);
                    if constexpr (PS == 2 + decltype(tc)::value) read_scale(pf_int<1 - H>(), tc);
                });
            } else {
                constexpr int NL = H == 0 ? LX + NWL : LX;
                static_for<0, NL>([&](auto uc) {
                    constexpr int U = decltype(uc)::value;
                    if constexpr (PS == U * SL / NL) {
                        if constexpr (H == 1) issue_x(c + 1, 1, xs, U);
                        else if constexpr (U < LX) issue_x(c + 1, 0, xs, U);
                        else if constexpr (RF::PASSED) pass_load(c + 2, wc != 0, U - LX);
                        else issue_w(c + 2, wc != 0, U - LX);
                    }
                });
                if constexpr (H == 0 && PS == 1) read_head(wo);
            }
            if constexpr (RF::PASSED && H == 1 && FR == 2 * TN - 1 && I == 0) UNROLL for (int t = 0; t < TN; ++t) pick[t] ^= 0x05040302u ^ 0x03020100u;     /* from here on the next chunk is decoded */
            static_for<0, 4>([&](auto dc) {
                constexpr int D = decltype(dc)::value;
                if constexpr (D * TM / 4 == I) {
                    if constexpr (FR + 1 < 2 * TN) decode(pf_int<H>(), pf_int<FR + 1>(), dc);
                    else decode(pf_int<1 - H>(), pf_int<0>(), dc);
                }
            });
        });
        __builtin_amdgcn_sched_barrier(0);
        /* (Q6_K: chunk c + 2 of W has landed in its registers: only the stage of X asked for since may be on its way) */
        if constexpr (RF::PASSED && H == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LX) : "memory");
        else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        tie(xf[0]);
        if constexpr (H == 0) raw_tie(head_words);
        else {
            pass_landed();
            wc = wo;
        }
        xs = xn;
    };
    for (int c = 0; c < nq; ++c) {
        period(c, pf_int<0>());
        period(c, pf_int<1>());
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int wave_o = __builtin_amdgcn_readfirstlane(tid >> 6), lane_o = tid & 63, half_o = wave_o & 1, pos = wave_o >> 1;
    constexpr int HT = TM / 2 * TN;
    const u32 give = lds0 + (u32)((pos * 2 * HT + (half_o ? 0 : HT)) * 1024 + lane_o * 16), take = lds0 + (u32)((pos * 2 * HT + (half_o ? HT : 0)) * 1024 + lane_o * 16);
    static_for<0, HT>([&](auto ec) {
        constexpr int e = decltype(ec)::value;
        lds_write128(give + e * 1024u, __builtin_bit_cast(u32x4, half_o ? acc[e / TN][e % TN] : acc[e / TN + TM / 2][e % TN]));
    });
    lds_barrier();
    static_for<0, TM / 2>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        u32x4 o[TN];
        static_for<0, TN>([&](auto jc) { constexpr int j = decltype(jc)::value; o[j] = lds_read128<0>(take + (i * TN + j) * 1024u); });
        lds_wait();
        tie(o);
        f32x4 v[TN];
        static_for<0, TN>([&](auto jc) { constexpr int j = decltype(jc)::value; v[j] = (half_o ? acc[i + TM / 2][j] : acc[i][j]) + __builtin_bit_cast(f32x4, o[j]); });
        store_tiles<TN>(a, m0 + (i + (half_o ? TM / 2 : 0)) * 16, n0 + pos * TN * 16, lane_o, v, lds0 + (u32)(4 * TM * TN * 1024 + wave_o * wave_out_bytes<TN>()));
    });
}

#define PSN_FRAG(fmt, RF, BM, BN)                                                                                            \
    extern "C" __global__ void __launch_bounds__(512) psn_prefill_##fmt##_m##BM##_n##BN##_pp(const psn_prefill_args a) {    \
        prefill_frag_body<RF, BM / 16, BN / 64>(a);                                                                          \
    }
#define PSN_FRAG_FAMILY(fmt, RF) PSN_FRAG(fmt, RF, 64, 64) PSN_FRAG(fmt, RF, 64, 128) PSN_FRAG(fmt, RF, 128, 128)

#ifdef PSN_BUILD_FR_Q4_0
PSN_FRAG_FAMILY(q4_0, FragQ4_0)
#endif
#ifdef PSN_BUILD_FR_Q8_0
PSN_FRAG_FAMILY(q8_0, FragQ8_0)
#endif
#ifdef PSN_BUILD_FR_Q4_K
PSN_FRAG_FAMILY(q4_K, FragQ4_K)
#endif
#ifdef PSN_BUILD_FR_Q5_K
PSN_FRAG_FAMILY(q5_K, FragQ5_K)
#endif
#ifdef PSN_BUILD_FR_Q6_K
PSN_FRAG_FAMILY(q6_K, FragQ6_K)
#endif
