/*
 * psn_prefill_thin.hip -- gfx950 quantized prefill matmul for at most 64 rows of X:
 * Y[m][n] = sum_k h(deq(W)[n][k]) * X[m][k], fp16 MFMA, fp32 accumulation.
 *
 * A workgroup of eight waves owns 16 RT weight rows and all of X (16 TM rows of it, TM = ceil(M / 16)); wave w takes chunks
 * (256 of K) w, w + 8, ... of the range and the eight partial tiles are summed through LDS at the end, always in the order of
 * the waves.  Between start and end no wave waits for another: each has a piece of LDS of its own, through which what it
 * loaded becomes what its lanes multiply:
 *   - W and X are loaded with consecutive lanes on consecutive 16-byte words (asked for in the order the MFMA wants them,
 *     neighbouring lanes sit on different rows and a load takes 64 cycles instead of 16: X alone then cost 10 us per 16 rows of
 *     it at 14336 x 4096), W a whole chunk ahead, X one to four steps of 64 ahead, in registers;
 *   - put into LDS behind the wave's own earlier reads (lds_order() keeps them there), read back as MFMA
 *     operands, W's raw bytes one tile ahead of their decode.
 * Q4_K, Q5_K: a lane unpacks the scales of one of the chunk's four steps for its row and hands them to the row's other lanes through LDS (a sixth of the vector
 * instructions; 14336 x 4096, M = 16: Q4_K 13.6 -> 13.1 us, Q5_K 14.9 -> 14.1; M = 48: Q4_K 18.8 -> 18.0).
 * The loop has one body: past the last chunk every lane asks for the start of the buffer, which costs no traffic.
 *
 * What bounds it: a weight costs about four vector instructions (fp32 d * q - m per weight, then the rounding to fp16), which
 * is 7 us of a 14336 x 4096 launch over all SIMDs, and X, which every workgroup reads whole (RT trades it against workgroups).
 * Two chunks of W on their way instead of one changed nothing (-1 .. +4 %), nor did more of X.  Against the 64 x 64 kernel
 * (psn_prefill.hip), us: Q4_K 4096 x 4096 M = 16 11.4 -> 6.5, M = 33 12.2 -> 9.6, M = 64 13.9 -> 11.3; 1024 x 4096 M = 16 8.8 -> 5.3,
 * M = 48 9.4 -> 6.6; 14336 x 4096 M = 16 21.7 -> 15.1, M = 48 22.4 -> 20.8; 4096 x 14336 M = 16 22.2 -> 16.5.  At 64 rows of a large
 * matrix both take as long.
 */
#include "psn_args.h"
#include "psn_device.h"
#include "psn_prefill_common.h"
#include "psn_prefill_formats.h"

typedef float float4_t __attribute__((ext_vector_type(4)));

/* A row's chunk: WORDS 16-byte words are copied to LDS as they are, rows STRIDE bytes apart; read() takes what step J of part g
 * needs from there. */
template <typename WF> struct Feed;
template <> struct Feed<PpQ4_K> {
    typedef PpQ4_K::raw<8> raw;
    static constexpr int WORDS = 9, STRIDE = 144, SCALES = 1024;
    template <int J, bool SHARED> static PSN_DEV void read(const lds_u8 *row, const lds_u8 *scales, int g, raw &r) {
        fetch<16>(SHARED ? scales + 256 * J : row, r.h);
        fetch<8>(row + 8 * g + (16 + 32 * J), r.q[J]);
    }
};
template <> struct Feed<PpQ5_K> {
    typedef PpQ5_K::raw<8> raw;
    static constexpr int WORDS = 11, STRIDE = 176, SCALES = 1024;
    template <int J, bool SHARED> static PSN_DEV void read(const lds_u8 *row, const lds_u8 *scales, int g, raw &r) {
        fetch<16>(SHARED ? scales + 256 * J : row, r.h);
        fetch<8>(row + 8 * g + 16, r.top);
        fetch<8>(row + 8 * g + (48 + 32 * J), r.q[J]);
    }
};
/* 13 words from the dword on in which the super-block starts; behind them (from 208 on) the dword that holds its last two scales where it
 * starts two bytes late, and its d */
template <> struct Feed<PpQ6_K> {
    typedef PpQ6_K::raw<8> raw;
    static constexpr int WORDS = 13, STRIDE = 224, SCALES = 0;
    template <int J, bool> static PSN_DEV void read(const lds_u8 *row, const lds_u8 *, int g, raw &r) {
        constexpr int H = J >> 1;
        const lds_u8 *const p = row + 8 * g;
        fetch<4>(p + 64 * H, r.ql[2 * H]);
        fetch<4>(p + (64 * H + 32), r.ql[2 * H + 1]);
        fetch<4>(p + (128 + 32 * H), r.qh[H]);
        fetch<16>(row + 192, r.sc);
        fetch<4>(row + 208, r.sc4);
        fetch<4>(row + 212, r.d);
    }
};
template <> struct Feed<PpQ4_0> {
    typedef PpQ4_0::raw<8> raw;
    static constexpr int WORDS = 9, STRIDE = 144, SCALES = 0;
    template <int J, bool> static PSN_DEV void read(const lds_u8 *row, const lds_u8 *, int g, raw &r) { fetch<4>(row + 8 * g + 36 * J, r.q[J]); }
};
template <> struct Feed<PpQ8_0> {
    typedef PpQ8_0::raw<8> raw;
    static constexpr int WORDS = 17, STRIDE = 272, SCALES = 0;
    template <int J, bool> static PSN_DEV void read(const lds_u8 *row, const lds_u8 *, int g, raw &r) {
        fetch<4>(row + 16 * g + 68 * J, r.q[J]);
        fetch<4>(row + 16 * g + (68 * J + 16), r.e[J]);
    }
};

template <typename WF, int TM, int RT>
PSN_DEV void prefill_thin_body(const psn_prefill_args &a) {
    typedef Feed<WF> F;
    constexpr bool ODD = WF::BYTES % 4 != 0;                /* Q6_K: super-blocks start on a dword or between two */
    constexpr bool BIG = ODD || WF::BYTES == 272;           /* a chunk in five or six registers per row and lane instead of three */
    constexpr int XD = RT * TM <= 3 ? 4 : RT * TM <= 8 ? 2 : 1;   /* steps of X on their way */
    constexpr bool AHEAD = TM * (RT + 2) < (BIG ? 16 : 24);       /* registers for the next step's fragments of X */
    constexpr int NI = (16 * F::WORDS + 63) / 64;           /* load instructions per 16 rows and chunk */
    constexpr bool SHARED = psn_lds_thin_scales(WF::FORMAT, TM, RT);                      /* (Q5_K's 48 rows of X by 64 of W leave no room) */
    constexpr int WTILE = 16 * F::STRIDE, MINE = RT * (WTILE + (SHARED ? F::SCALES : 0)) + TM * 2048;
    static_assert(8 * MINE == psn_lds_thin_rings(WF::FORMAT, TM, RT, SHARED) && psn_lds_thin(WF::FORMAT, TM, RT) <= PSN_LDS_MAX && F::WORDS == psn_lds_words(WF::FORMAT) &&
                  (F::SCALES != 0) == psn_lds_scales(WF::FORMAT), "LDS of the launch");
    extern __shared__ uint4 psn_smem[];
    const int tid = threadIdx.x, lane = tid & 63, row = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = a.M, N = a.N, K = a.K, C = K >> 8;
    const int nt = (N + 16 * RT - 1) / (16 * RT), S = a.ksplit;
    const int tile_n = blockIdx.x % nt, split = blockIdx.x / nt;
    const int per_split = (C + S - 1) / S;
    const int c_begin = split * per_split, c_end = min(c_begin + per_split, C);
    if (c_begin >= c_end) return;                           /* whole workgroup leaves together */
    const int n0 = tile_n * 16 * RT, nq = c_end - c_begin;
    /* workgroups that start together would ask for the same lines of X at the same moment: each starts its (cyclic) walk elsewhere */
    const int rot = (int)((blockIdx.x * 5u) % (unsigned)nq);
    auto chunk_of = [&](int i) { const int r = i + rot; return c_begin + (r >= nq ? r - nq : r); };

    lds_u8 *const wl = (lds_u8 *)(__attribute__((address_space(3))) void *)psn_smem + wave * MINE, *const xl = wl + RT * WTILE, *const sl = xl + TM * 2048;

    float4_t acc[RT][TM];
    UNROLL for (int t = 0; t < RT; ++t) UNROLL for (int i = 0; i < TM; ++i) acc[t][i] = (float4_t)(0.f);

    /* W: a tile past the last whole one is moved back so that all its rows exist (with N < 16 the last row repeats) */
    int nb[RT];
    UNROLL for (int t = 0; t < RT; ++t) nb[t] = min(n0 + 16 * t, max(N - 16, 0));
    u32 woff[NI], wdst[NI];
    UNROLL for (int i = 0; i < NI; ++i) {
        const int word = min(i * 64 + lane, 16 * F::WORDS - 1), r = word / F::WORDS, wd = word % F::WORDS;
        woff[i] = (u32)(min(r, N - 1) * (int)a.row_bytes + wd * 16);
        wdst[i] = (u32)(r * F::STRIDE + wd * 16);
    }
    const u32 rowoff = ODD ? (u32)(min(row, N - 1) * (int)a.row_bytes) : 0u;
    u32x4 w[RT][NI];
    u32 tail[ODD ? RT : 1], dd[ODD ? RT : 1];
    /* past the last chunk (valid false) every lane asks for the start of the buffer: no traffic, and the loop has one body */
    auto load_w = [&](int c, bool valid) {
        u32 wo[NI];
        UNROLL for (int i = 0; i < NI; ++i) { wo[i] = valid ? woff[i] : 0u; tie1(wo[i]); }
        UNROLL for (int t = 0; t < RT; ++t) {
            const int64_t at = valid ? (int64_t)nb[t] * a.row_bytes + (int64_t)c * WF::BYTES : 0;
            UNROLL for (int i = 0; i < NI; ++i) {
                if constexpr (ODD) fetch<4>(a.W + (((u32)at + wo[i]) & ~3u), w[t][i]);
                else fetch<16>(a.W + at + wo[i], w[t][i]);
            }
            if constexpr (ODD) {
                const u32 off = (u32)at + (valid ? rowoff : 0u);
                unsigned short d;
                fetch<4>(a.W + ((off + 2) & ~3u) + 204, tail[t]);
                fetch<2>(a.W + off + 208, d);
                dd[t] = d;
            }
        }
    };
    auto put_w = [&]() {
        lds_order();                                        /* the reads of the chunk before */
        UNROLL for (int t = 0; t < RT; ++t) {
            UNROLL for (int i = 0; i < NI; ++i) store<16>(wl + t * WTILE + wdst[i], w[t][i]);
            if constexpr (ODD) {
                store<4>(wl + t * WTILE + row * F::STRIDE + 208, tail[t]);
                store<4>(wl + t * WTILE + row * F::STRIDE + 212, dd[t]);
            }
        }
        lds_order();
        if constexpr (SHARED) {                             /* lane (g, row): the scales of step g */
            u32x4 header[RT];
            UNROLL for (int t = 0; t < RT; ++t) fetch<16>((const lds_u8 *)(wl + t * WTILE + row * F::STRIDE), header[t]);
            lds_order();
            UNROLL for (int t = 0; t < RT; ++t) {
                u32 sc, mn;
                float own[4];
                kq_pick(header[t], g, sc, mn);
                kq_own(header[t], sc, mn, own);
                store<16>(sl + t * F::SCALES + lane * 16, (f32x4){own[0], own[1], own[2], own[3]});
            }
            lds_order();
        }
    };

    /* X: eight rows of 128 bytes per instruction */
    const uint8_t *const xbase = reinterpret_cast<const uint8_t *>(a.X);
    u32 xoff[2 * TM];
    UNROLL for (int u = 0; u < 2 * TM; ++u) xoff[u] = (u32)min(8 * u + (lane >> 3), M - 1) * (u32)(2 * K) + (u32)((lane & 7) * 16);
    u32x4 x[XD][2 * TM];
    auto load_x = [&](int c, bool valid, auto jc, auto sc) {
        constexpr int J = decltype(jc)::value, SLOT = decltype(sc)::value;
        UNROLL for (int u = 0; u < 2 * TM; ++u) {
            u32 o = valid ? xoff[u] : 0u;
            tie1(o);
            fetch<16>(xbase + (int64_t)c * 512 + J * 128 + o, x[SLOT][u]);
        }
    };
    const u32 flo = (u32)tile_off(row, WF::template k_lo<8>(g) >> 3), fhi = (u32)tile_off(row, WF::template k_hi<8>(g) >> 3);
    const u32 xdst = (u32)tile_off(lane >> 3, lane & 7), xdst_odd = (u32)tile_off(8 + (lane >> 3), lane & 7);   /* (the swizzle repeats every sixteen rows) */

    /* X of step J goes through LDS into fragments; its slot takes the step XD further on */
    u32x4 xf[2][2][TM];
    auto stage_x = [&](int c, int next, bool more, auto jc) {
        constexpr int J = decltype(jc)::value, SLOT = J % XD;
        lds_order();                                        /* the reads of the step before */
        UNROLL for (int u = 0; u < 2 * TM; ++u) store<16>(xl + (u >> 1) * 2048 + (u & 1 ? xdst_odd : xdst), x[SLOT][u]);
        lds_order();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (J + XD < 4) load_x(c, true, pf_int<J + XD>(), pf_int<SLOT>());
        else load_x(next, more, pf_int<(J + XD) & 3>(), pf_int<SLOT>());
        UNROLL for (int i = 0; i < TM; ++i) { fetch<16>(xl + i * 2048 + flo, xf[J & 1][0][i]); fetch<16>(xl + i * 2048 + fhi, xf[J & 1][1][i]); }
        __builtin_amdgcn_sched_barrier(0);
    };
    typename F::raw r[2];
    const lds_u8 *const wrow = wl + row * F::STRIDE, *const srow = sl + row * 16;
    /* step J of chunk c; `more`: chunk `next` follows.  What a tile's decode needs is read from LDS one tile, X one step ahead. */
    auto step = [&](int c, int next, bool more, auto jc) {
        constexpr int J = decltype(jc)::value;
        if constexpr (!AHEAD) stage_x(c, next, more, jc);
        else if constexpr (J < 3) stage_x(c, next, more, pf_int<(J + 1) & 3>());
        UNROLL for (int t = 0; t < RT; ++t) {
            typename F::raw &now = r[(J * RT + t) & 1], &then = r[(J * RT + t + 1) & 1];
            if (t + 1 < RT) F::template read<J, SHARED>(wrow + (t + 1) * WTILE, srow + (t + 1) * F::SCALES, g, then);
            else if constexpr (J < 3) F::template read<(J + 1) & 3, SHARED>(wrow, srow, g, then);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (ODD) now.pick = ((u32)nb[t] * (u32)a.row_bytes + (u32)(c * WF::BYTES) + rowoff) & 2u ? 0x05040302u : 0x03020100u;
            u32 lo[4], hi[4];
            typename WF::scale s;
            half_done h;
            if constexpr (F::SCALES != 0 && !SHARED) {
                u32 sc, mn;
                float own[4];
                kq_pick(now.h, J, sc, mn);
                kq_own(now.h, sc, mn, own);
                now.h = __builtin_bit_cast(u32x4, (f32x4){own[0], own[1], own[2], own[3]});
            }
            WF::template scales0<J, 8, true>(now, g, s);
            WF::template scales1<J, 8, true>(now, s);
            UNROLL for (int i = 0; i < 2; ++i) {
                WF::template first<J, 8, 0>(now, s, i, h);
                WF::template second<0>(s, h, lo[2 * i], lo[2 * i + 1]);
                WF::template first<J, 8, 1>(now, s, i, h);
                WF::template second<1>(s, h, hi[2 * i], hi[2 * i + 1]);
            }
            const half8_t wlo = __builtin_bit_cast(half8_t, (u32x4){lo[0], lo[1], lo[2], lo[3]}), whi = __builtin_bit_cast(half8_t, (u32x4){hi[0], hi[1], hi[2], hi[3]});
            UNROLL for (int i = 0; i < TM; ++i) acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, xf[J & 1][0][i]), wlo, acc[t][i], 0, 0, 0);
            UNROLL for (int i = 0; i < TM; ++i) acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, xf[J & 1][1][i]), whi, acc[t][i], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    const int count = (nq - wave + 7) >> 3;                 /* this wave's chunks: wave, wave + 8, ... of the range */
    if (count > 0) {
        /* (loads come back in the order they were asked for: what is needed first goes first) */
        int c = chunk_of(wave);
        load_x(c, true, pf_int<0>(), pf_int<0>());
        if constexpr (XD > 1) load_x(c, true, pf_int<1>(), pf_int<1 % XD>());
        if constexpr (XD > 2) { load_x(c, true, pf_int<2>(), pf_int<2 % XD>()); load_x(c, true, pf_int<3>(), pf_int<3 % XD>()); }
        load_w(c, true);
        __builtin_amdgcn_sched_barrier(0);
        for (int k = 1; k <= count; ++k) {
            const bool more = k < count;
            const int next = more ? chunk_of(wave + 8 * k) : c;
            put_w();
            __builtin_amdgcn_sched_barrier(0);
            load_w(next, more);
            F::template read<0, SHARED>(wrow, srow, g, r[0]);
            if constexpr (AHEAD) stage_x(c, next, more, pf_int<0>());
            __builtin_amdgcn_sched_barrier(0);
            step(c, next, more, pf_int<0>());
            step(c, next, more, pf_int<1>());
            step(c, next, more, pf_int<2>());
            step(c, next, more, pf_int<3>());
            c = next;
        }
    }

    /* partial tiles of the eight waves -> LDS ([wave][tile][register][lane]), then summed in the order of the waves */
    constexpr int TILE = 256, PER_WAVE = RT * TM * TILE;
    static_assert(8 * PER_WAVE * 4 == psn_lds_thin_sums(TM, RT), "the sums at the end");
    float *const part_sums = reinterpret_cast<float *>(psn_smem);
    __syncthreads();
    UNROLL for (int t = 0; t < RT; ++t) UNROLL for (int i = 0; i < TM; ++i) UNROLL for (int r = 0; r < 4; ++r)
        part_sums[wave * PER_WAVE + (t * TM + i) * TILE + r * 64 + lane] = acc[t][i][r];
    __syncthreads();
    UNROLL for (int u = 0; u < (PER_WAVE + 511) / 512; ++u) {
        const int f = u * 512 + tid;
        if (PER_WAVE % 512 != 0 && f >= PER_WAVE) break;
        float sum = part_sums[f];
        UNROLL for (int v = 1; v < 8; ++v) sum += part_sums[v * PER_WAVE + f];
        const int tile = f / TILE, r = (f >> 6) & 3, own = n0 + 16 * (tile / TM);
        const int m = 16 * (tile % TM) + 4 * g + r, n = min(own, max(N - 16, 0)) + row;
        if (m < M && n >= own && n < N) {
            if (S == 1) a.Y[(int64_t)m * N + n] = sum;
            else unsafeAtomicAdd(&a.Y[(int64_t)m * N + n], sum);
        }
    }
}

/* 16 TM rows of X, 16 RT of W.  RT = 4 where LDS and registers hold it (48 rows of X, with Q8_0 sixteen) and two
 * workgroups of RT = 2 do not share a compute unit instead. */
#define PSN_THIN(fmt, WF, TM, RT)                                                                                      \
    extern "C" __global__ void __launch_bounds__(512) psn_prefill_##fmt##_thin_##TM##_##RT(const psn_prefill_args a) { \
        prefill_thin_body<WF, TM, RT>(a);                                                                              \
    }
#define PSN_THIN_FAMILY(fmt, WF)                                                                       \
    PSN_THIN(fmt, WF, 1, 1) PSN_THIN(fmt, WF, 2, 1) PSN_THIN(fmt, WF, 3, 1) PSN_THIN(fmt, WF, 4, 1)    \
    PSN_THIN(fmt, WF, 1, 2) PSN_THIN(fmt, WF, 2, 2) PSN_THIN(fmt, WF, 3, 2) PSN_THIN(fmt, WF, 4, 2)

#ifdef PSN_BUILD_TH_Q4_0
PSN_THIN_FAMILY(q4_0, PpQ4_0)
PSN_THIN(q4_0, PpQ4_0, 2, 4) PSN_THIN(q4_0, PpQ4_0, 3, 4)
#endif
#ifdef PSN_BUILD_TH_Q8_0
PSN_THIN_FAMILY(q8_0, PpQ8_0)
PSN_THIN(q8_0, PpQ8_0, 1, 4)
#endif
#ifdef PSN_BUILD_TH_Q4_K
PSN_THIN_FAMILY(q4_K, PpQ4_K)
PSN_THIN(q4_K, PpQ4_K, 2, 4) PSN_THIN(q4_K, PpQ4_K, 3, 4)
#endif
#ifdef PSN_BUILD_TH_Q5_K
PSN_THIN_FAMILY(q5_K, PpQ5_K)
PSN_THIN(q5_K, PpQ5_K, 2, 4) PSN_THIN(q5_K, PpQ5_K, 3, 4)
#endif
#ifdef PSN_BUILD_TH_Q6_K
PSN_THIN_FAMILY(q6_K, PpQ6_K)
PSN_THIN(q6_K, PpQ6_K, 1, 4) PSN_THIN(q6_K, PpQ6_K, 2, 4) PSN_THIN(q6_K, PpQ6_K, 3, 4)
#endif
