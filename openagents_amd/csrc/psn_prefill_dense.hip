/*
 * psn_prefill_dense.hip -- gfx950 fp16 multiply of the dense prefill family:
 * Y[m][n] = sum_k W[n][k] * X[m][k] over weights that psn_prefill_<fmt>_unpack has turned into fp16 fragments, fp32
 * accumulation on v_mfma_f32_16x16x32_f16.
 *
 * Both operands pass through LDS, put there by direct-to-LDS loads, and are read as 16-byte MFMA fragments one K step ahead;
 * reads and loads are spread behind the MFMAs, one barrier per step, eight waves (two to a SIMD).
 *
 * What bounds it on MI355X: power on a full chip, and the bytes that a compute unit takes in otherwise.
 *   - Power.  4001 x 4096 x 14336 on 256 x 256 tiles, before X came in whole lines: 354 us on real data and 300 on zeros (same instructions); without its loads 288,
 *     without its LDS reads 331, the MFMAs alone 260.  So energy per product is what counts:
 *     16 x 16 x 32 MFMAs instead of 32 x 32 x 16 (384 against 423 us in one run), X fetched in whole 128-byte lines (64 k of a row per stage; a stage
 *     of 32 k fetches every line twice: 354 -> 336, which is what it takes now), and the order of the MFMAs within a step, boustrophedon, so that one operand stays put (1 %).
 *   - Intake.  A compute unit accepts about 40 bytes per cycle of direct-to-LDS loads, whatever the depth of the ring (128 x 128 tiles, rings of four
 *     and five stages: 81.5 and 81.4 us at 512 x 4096 x 14336): 256 x 256 tiles need 31 bytes per cycle of MFMA, 128 x 256 tiles 47, 128 x 128 tiles 63.
 * Against the kernels before (four waves, 32 x 32 x 16 MFMAs, weights from memory straight into registers), 256 x 256 tiles: 4001 x 14336 x 4096
 * 490 -> 393 us (1.20 PFLOP/s), 4001 x 4096 x 14336 410 -> 336 (1.40); 128 x 256: 2048 x 4096 x 4096 69 -> 60, 512 x 14336 x 4096 63 -> 55;
 * the smaller tiles, for few rows on either side: 4001 x 1024 x 4096 69 -> 36, 512 x 4096 x 4096 49 -> 23, 512 x 1024 x 4096 48 -> 13.5.
 * (The largest one on other devices and days: 389 to 395 us, 407 under the profiler.)  Storing Y costs 45 of the 393 us.  Tried without gain: workgroups that walk several tiles and ask for the next one's operands before they store (1-2 %
 * on 128 x 256 tiles, spills on 256 x 256), K ranges rotated against each other per XCD, non-temporal stores.
 */
#include "psn_args.h"
#include "psn_device.h"

#include "psn_prefill_common.h"

/* X: 16-byte piece `lane` of load c (eight rows of 128 bytes in LDS, the pieces of a row at piece ^ tile_swz(row)); rows past the end repeat the last one */
PSN_DEV u32 dense_x_offset(const psn_prefill_args &a, int m0, int c, int lane) {
    const int row = c * 8 + (lane >> 3), piece = (lane & 7) ^ tile_swz(row);
    return (u32)min(m0 + row, a.M - 1) * (u32)(a.K * 2) + (u32)(piece * 16);
}
/* W: the fragment of sixteen rows and 32 k out of the packed order [row / 32][k / 16][(k / 8) & 1][row % 32][8]: lane (q, n) holds k 8 q .. 8 q + 7 of row n.
 * The part of the address that is the same for all lanes (row block and 16-row half) is added by the caller. */
PSN_DEV u32 dense_w_offset(int lane) {
    const int q = lane >> 4;
    return (u32)((q >> 1) * 1024 + (q & 1) * 512 + (lane & 15) * 16);
}

/* Large tiles: WM x WN waves with TM x TN MFMA tiles each, K in steps of 32.  X comes in stages of 64 k (whole lines), a ring of three, W in steps of 32 k, a ring
 * of four: for 256 x 256 tiles that is all 160 KB of LDS.  Step t multiplies what was read during step t - 1, reads the fragments of step t + 1 and asks for W of step t + 4 and
 * half of the stage of X that takes the place of the one read last: the first half of stage (t + 5) / 2 in odd steps, the second of (t + 4) / 2 in even ones.
 * Every load has two to four steps to arrive.  Loads past the end repeat the last step, into slots that nothing reads any more. */
template <int WM, int WN, int TM, int TN> PSN_DEV void dense_large_body(const psn_prefill_args &a) {
    constexpr int WAVES = WM * WN, BM = WM * TM * 16, BN = WN * TN * 16, NX = 3, NW = 4;
    constexpr int XB = BM * 128, WB = BN * 64, W0 = NX * XB;
    constexpr int LXS = BM / 8 / WAVES, LX = LXS / 2, LW = BN / 16 / WAVES, NL = LX + LW;       /* loads per wave: X per stage and step, W per step */
    static_assert(WAVES == 8 && LXS % 2 == 0 && LW >= 1 && W0 + NW * WB == psn_lds_dense(BM, BN) && W0 + NW * WB <= PSN_LDS_MAX && 8 * wave_out_bytes<TN>() <= W0 + NW * WB, "tile");
    extern __shared__ uint4 psn_smem[];
    lds_char *const lds_ptr = (lds_char *)psn_smem;
    const u32 lds0 = (u32)(uintptr_t)lds_ptr;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / WN, wn = wave % WN;
    prefill_place p;
    if (!place_workgroup<BM, BN, 4 * BM>(a, p)) return;                   /* whole workgroup leaves together */
    const int nst = 4 * p.chunks, nsteps = 2 * nst;

    u32 xoff[LXS];
    UNROLL for (int u = 0; u < LXS; ++u) xoff[u] = dense_x_offset(a, p.m0, wave * LXS + u, lane);
    const char *const xb = reinterpret_cast<const char *>(a.X) + (int64_t)p.c0 * 512;
    const u32 wlane = dense_w_offset(lane);
    const int64_t wblock = (int64_t)(a.K >> 4) * 1024;       /* 32 rows */
    const char *const wb = reinterpret_cast<const char *>(a.W) + (p.n0 >> 5) * wblock + (int64_t)p.c0 * 16384;
    auto issue_x = [&](int st, u32 slot, int u) { load_to_lds(xb + (int64_t)min(st, nst - 1) * 128 + xoff[u], lds_ptr + slot + (wave * LXS + u) * 1024); };
    auto issue_w = [&](int t, int slot, int u) {
        const int c = wave * LW + u;                         /* sixteen-row block of the tile */
        load_to_lds(wb + (c >> 1) * wblock + (c & 1) * 256 + (int64_t)min(t, nsteps - 1) * 2048 + wlane, lds_ptr + W0 + slot * WB + c * 1024);
    };

    f32x4 acc[TM][TN];
    UNROLL for (int i = 0; i < TM; ++i) UNROLL for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4)(0.f);
    u32 fx[2];                                               /* fragments of X in the first and second half of a stage */
    UNROLL for (int h = 0; h < 2; ++h) fx[h] = lds0 + (u32)tile_off(wm * TM * 16 + (lane & 15), 4 * h + (lane >> 4));
    const u32 fw = lds0 + (u32)(W0 + wn * TN * 1024 + lane * 16);
    constexpr int FR = TM + TN, NPOS = TM * TN, READ_BY = NPOS * 3 / 4;    /* the last quarter of a step reads nothing: the barrier finds the reads done */
    u32x4 xf[2][TM], wf[2][TN];
    auto read = [&](u32 ax, u32 aw, auto setc, auto rc) {
        constexpr int S = decltype(setc)::value, R = decltype(rc)::value;
        if constexpr (R < TN) wf[S][R] = lds_read128<R * 1024>(aw);
        else xf[S][R - TN] = lds_read128<(R - TN) * 2048>(ax);
    };

    UNROLL for (int u = 0; u < LXS; ++u) issue_x(0, 0, u);
    UNROLL for (int u = 0; u < LW; ++u) issue_w(0, 0, u);
    UNROLL for (int u = 0; u < LW; ++u) issue_w(1, 1, u);
    UNROLL for (int u = 0; u < LXS; ++u) issue_x(1, XB, u);
    UNROLL for (int u = 0; u < LW; ++u) issue_w(2, 2, u);
    UNROLL for (int u = 0; u < LX; ++u) issue_x(2, 2 * XB, u);
    UNROLL for (int u = 0; u < LW; ++u) issue_w(3, 3, u);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LXS + LX + 3 * LW) : "memory");                                /* X stage 0 and W step 0 */
    lds_barrier();
    static_for<0, FR>([&](auto rc) { read(fx[0], fw, pf_int<0>(), rc); });
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LXS + LX + 2 * LW) : "memory");        /* W step 1 */
    tie(xf[0]);
    tie(wf[0]);
    u32 xs = 0;                                              /* slot of X that step t's stage is in */
    auto step = [&](int t, auto slotc) {
        constexpr int SLOT = decltype(slotc)::value, S = SLOT & 1;
        u32 xn = xs, xt = xs;                                /* the slots that step t + 1 reads and that this step's loads of X go to */
        if constexpr (S == 1) xn = xs + XB == NX * XB ? 0 : xs + XB;
        else xt = xs + 2 * XB >= NX * XB ? xs + 2 * XB - NX * XB : xs + 2 * XB;
        const int xst = (t >> 1) + (S ? 3 : 2);
        const u32 ax = fx[1 - S] + xn, aw = fw + (u32)((SLOT + 1) % NW * WB);
        static_for<0, NPOS>([&](auto pc) {
            constexpr int P = decltype(pc)::value, j = P / TM, i = (j & 1) ? TM - 1 - P % TM : P % TM;
            __builtin_amdgcn_sched_barrier(0);
            acc[i][j] = mfma16(wf[S][j], xf[S][i], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, FR>([&](auto rc) { if constexpr (decltype(rc)::value * READ_BY / FR == P) read(ax, aw, pf_int<1 - S>(), rc); });
            static_for<0, NL>([&](auto uc) {
                constexpr int U = decltype(uc)::value;
                if constexpr (U * NPOS / NL + 1 == P) {
                    if constexpr (U < LX) issue_x(xst, xt, S ? U : LX + U);
                    else issue_w(t + NW, SLOT, U - LX);
                }
            });
        });
        __builtin_amdgcn_sched_barrier(0);
        /* W of step t + 2 and X of its stage have landed: at most the loads of this step and the last are on their way */
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * NL) : "memory");
        tie(xf[1 - S]);
        tie(wf[1 - S]);
        xs = xn;
    };
    for (int t = 0; t < nsteps; t += 4) {                    /* (a K range is a multiple of 256) */
        step(t, pf_int<0>());
        step(t + 1, pf_int<1>());
        step(t + 2, pf_int<2>());
        step(t + 3, pf_int<3>());
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");      /* nothing is on its way into LDS any more */

    /* (worked out again from an opaque thread index, so that nothing of it stays in a register through the loop) */
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int wave_o = tid >> 6, lane_o = tid & 63;
    UNROLL for (int i = 0; i < TM; ++i)
        store_tiles<TN>(a, p.m0 + (wave_o / WN * TM + i) * 16, p.n0 + wave_o % WN * TN * 16, lane_o, acc[i], lds0 + (u32)(wave_o * wave_out_bytes<TN>()));
}

/* Small tiles: four pairs of waves, WM x WN, with TM x TN MFMA tiles; one wave of a pair multiplies the first half of every 64-wide stage of K, the other the second, so that a
 * fragment is read once per workgroup row or column of four (64 x 64 outputs to a wave at 128 x 128 tiles) and not of eight; the pair's sums meet in LDS at the end.  Against eight waves
 * with outputs of their own: 4001 x 1024 x 4096 37.3 -> 35.9 us, 512 x 4096 x 14336 85.3 -> 81.5, both on 128 x 128 tiles; on 128 x 256 tiles it gained nothing.  A ring of NS stages holds X and W;
 * period g multiplies stage g, reads the fragments of stage g + 1 and asks for stage g + NS. */
template <int WM, int WN, int TM, int TN, int NS> PSN_DEV void dense_small_body(const psn_prefill_args &a) {
    constexpr int BM = WM * TM * 16, BN = WN * TN * 16, XB = BM * 128, SB = (BM + BN) * 128;
    constexpr int LX = BM / 64, LW = BN / 64, NL = LX + LW;  /* loads per wave and stage */
    static_assert(WM * WN == 4 && LX >= 1 && LW >= 1 && TM % 2 == 0 && NS * SB == psn_lds_dense(BM, BN) && NS * SB <= PSN_LDS_MAX && 4 * TM * TN * 1024 + 8 * wave_out_bytes<TN>() <= NS * SB, "tile");
    extern __shared__ uint4 psn_smem[];
    lds_char *const lds_ptr = (lds_char *)psn_smem;
    const u32 lds0 = (u32)(uintptr_t)lds_ptr;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = wave & 1, wm = (wave >> 1) / WN, wn = (wave >> 1) % WN;
    prefill_place p;
    if (!place_workgroup<BM, BN, 4 * BM>(a, p)) return;                   /* whole workgroup leaves together */
    const int nst = 4 * p.chunks;

    u32 xoff[LX];
    UNROLL for (int u = 0; u < LX; ++u) xoff[u] = dense_x_offset(a, p.m0, wave * LX + u, lane);
    const char *const xb = reinterpret_cast<const char *>(a.X) + (int64_t)p.c0 * 512;
    const u32 wlane = dense_w_offset(lane);
    const int64_t wblock = (int64_t)(a.K >> 4) * 1024;       /* 32 rows */
    const char *const wb = reinterpret_cast<const char *>(a.W) + (p.n0 >> 5) * wblock + (int64_t)p.c0 * 16384;
    auto issue = [&](int st, int slot, auto uc) {            /* stages past the end repeat the last one, into slots that nothing reads any more */
        constexpr int U = decltype(uc)::value;
        const int g = min(st, nst - 1);
        lds_char *const to = lds_ptr + slot * SB;
        if constexpr (U < LX) load_to_lds(xb + (int64_t)g * 128 + xoff[U], to + (wave * LX + U) * 1024);
        else {
            const int c = wave * LW + U - LX, rows = c >> 1; /* sixteen rows and half of the stage's K */
            load_to_lds(wb + (rows >> 1) * wblock + (rows & 1) * 256 + (c & 1) * 2048 + (int64_t)g * 4096 + wlane, to + XB + c * 1024);
        }
    };

    f32x4 acc[TM][TN];
    UNROLL for (int i = 0; i < TM; ++i) UNROLL for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4)(0.f);
    const u32 fx = lds0 + (u32)tile_off(wm * TM * 16 + (lane & 15), 4 * half + (lane >> 4));
    const u32 fw = lds0 + (u32)(XB + wn * TN * 2048 + half * 1024 + lane * 16);
    constexpr int FR = TM + TN, NPOS = TM * TN, READ_BY = NPOS * 3 / 4;
    u32x4 xf[2][TM], wf[2][TN];
    auto read = [&](u32 at, auto setc, auto rc) {
        constexpr int S = decltype(setc)::value, R = decltype(rc)::value;
        if constexpr (R < TN) wf[S][R] = lds_read128<R * 2048>(fw + at);
        else xf[S][R - TN] = lds_read128<(R - TN) * 2048>(fx + at);
    };

    static_for<0, NS>([&](auto sc) { static_for<0, NL>([&](auto uc) { issue(decltype(sc)::value, decltype(sc)::value, uc); }); });
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * NL) : "memory");
    lds_barrier();
    static_for<0, FR>([&](auto rc) { read(0, pf_int<0>(), rc); });
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * NL) : "memory");
    tie(xf[0]);
    tie(wf[0]);
    int slot = 0;                                            /* of stage g */
    auto period = [&](int g, auto setc) {
        constexpr int S = decltype(setc)::value;
        const int next = slot + 1 == NS ? 0 : slot + 1;
        static_for<0, NPOS>([&](auto pc) {
            constexpr int P = decltype(pc)::value, j = P / TM, i = (j & 1) ? TM - 1 - P % TM : P % TM;
            __builtin_amdgcn_sched_barrier(0);
            acc[i][j] = mfma16(wf[S][j], xf[S][i], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, FR>([&](auto rc) { if constexpr (decltype(rc)::value * READ_BY / FR == P) read((u32)(next * SB), pf_int<1 - S>(), rc); });
            static_for<0, NL>([&](auto uc) { if constexpr (decltype(uc)::value * NPOS / NL + 1 == P) issue(g + NS, slot, uc); });
        });
        __builtin_amdgcn_sched_barrier(0);
        /* stage g + 2 has landed: at most the NS - 2 stages after it are on their way */
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * NL) : "memory");
        tie(xf[1 - S]);
        tie(wf[1 - S]);
        slot = next;
    };
    for (int g = 0; g < nst; g += 2) {
        period(g, pf_int<0>());
        period(g + 1, pf_int<1>());
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

    /* a pair's sums: the first wave finishes the upper half of the MFMA tiles, the second the lower, each after taking the other's part out of LDS */
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int wave_o = __builtin_amdgcn_readfirstlane(tid >> 6), lane_o = tid & 63, half_o = wave_o & 1, pos = wave_o >> 1;
    constexpr int H = TM / 2 * TN;
    const u32 give = lds0 + (u32)((pos * 2 * H + (half_o ? 0 : H)) * 1024 + lane_o * 16), take = lds0 + (u32)((pos * 2 * H + (half_o ? H : 0)) * 1024 + lane_o * 16);
    static_for<0, H>([&](auto ec) {
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
        store_tiles<TN>(a, p.m0 + (pos / WN * TM + i + (half_o ? TM / 2 : 0)) * 16, p.n0 + pos % WN * TN * 16, lane_o, v,
                        lds0 + (u32)(4 * TM * TN * 1024 + wave_o * wave_out_bytes<TN>()));
    });
}

extern "C" __global__ void __launch_bounds__(512) psn_prefill_dense_f16(const psn_prefill_args a) { dense_large_body<4, 2, 4, 8>(a); }
extern "C" __global__ void __launch_bounds__(512) psn_prefill_dense_f16_m128(const psn_prefill_args a) { dense_large_body<2, 4, 4, 4>(a); }
extern "C" __global__ void __launch_bounds__(512) psn_prefill_dense_f16_m128_n128(const psn_prefill_args a) { dense_small_body<2, 2, 4, 4, 4>(a); }
extern "C" __global__ void __launch_bounds__(512) psn_prefill_dense_f16_m64_n128(const psn_prefill_args a) { dense_small_body<1, 4, 4, 2, 4>(a); }
extern "C" __global__ void __launch_bounds__(512) psn_prefill_dense_f16_m64_n64(const psn_prefill_args a) { dense_small_body<1, 4, 4, 1, 5>(a); }
