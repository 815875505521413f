/*
 * psn_matvec_batch.hip -- gfx950 decode matvec for up to eight columns (used from three on), scheme Q8, formats whose blocks of 32 carry one scale
 * (Q4_0, Q8_0; Q8_0 activations, quantized beforehand).
 *
 * v_mfma_i32_16x16x32_i8 multiplies one block of 16 weight rows with up to 16 columns (A = the columns' int8, B = the rows'):
 * the integer dot products of the dot4 kernels (psn_matvec.hip) at a cost that does not grow with the batch.  A lane holds four
 * columns of one row and scales them with d_w d_x.  Q4_0: the nibbles are multiplied as they are, and -8 times the sum of the
 * block's activations is what the MFMA starts from.
 *
 * A workgroup of eight waves owns 16 rows; wave w takes chunks (256 of K) w, w + 8, ... and the partial sums meet in LDS at the
 * end, in the order of the waves.  Nothing else is shared: a chunk's weights and activations are loaded a chunk ahead, consecutive
 * lanes on consecutive 16-byte words, and go through the wave's own piece of LDS to the lanes that multiply them.
 *
 * What bounds it: a chunk of a wave is a chain of about 1 us (LDS to MFMA to scaling, eight blocks of it), hidden by the waves of three
 * workgroups on a compute unit with Q4_0 (72 registers) and of two with Q8_0 (55 KB of LDS each, a third would fit without the 2 KB that
 * its activation sums, which it has no use for, are given); the weight stream where rows are many (Q8_0 40000 x 8192, batch 8: 348 MB in 79 us).  Against the
 * register kernels at batch 8: Q4_0 14336 x 4096 21.0 -> 15.7 us, 1000 x 4096 11.2 -> 7.5, 4100 x 16384 92 -> 23.5; Q8_0 25.5 -> 20.1,
 * 11.0 -> 7.5, 90 -> 28.3.  Two tiles per workgroup measured 25-45 % slower (fewer waves), a second chunk on its way 2-15 % slower,
 * rows and columns swapped in the products (fewer LDS reads, 96 registers instead of 68) 0-20 % slower.
 */
#include "psn_args.h"
#include "psn_device.h"

#define UNROLL _Pragma("unroll")
typedef int v4i __attribute__((ext_vector_type(4)));
template <int N> struct ic { static constexpr int value = N; };

/* block J of a row's chunk: what lane part g of four multiplies (eight int8), the block's scale, and the same lane's activations.  Two blocks
 * are a whole number of dwords; the first one's scale is the low half of its first dword, the second one's the high half of the
 * dword before its quants. */
struct BtQ8_0 {
    static constexpr int WORDS = 17, BYTES = 272;
    static constexpr bool SUMS = false;
    template <int J> static PSN_DEV void weights(const lds_u8 *row, int g, u32x2 &b, float &d) {
        const lds_u8 *const p = row + 68 * (J >> 1);
        u32 s;
        if constexpr (J & 1) {
            fetch<4>(p + 36 + 8 * g, b);
            fetch<4>(p + 32, s);
            d = h2f_hi(s);
        } else {
            u32 q0, q1, q2;
            fetch<4>(p + 8 * g, q0);
            fetch<4>(p + 8 * g + 4, q1);
            fetch<4>(p + 8 * g + 8, q2);
            b = (u32x2){align2(q1, q0), align2(q2, q1)};
            fetch<4>(p, s);
            d = h2f_lo(s);
        }
    }
    template <int J> static PSN_DEV void columns(const lds_u8 *x, int g, u32x2 &a) { fetch<8>(x + 32 * J + 8 * g, a); }
};
struct BtQ4_0 {
    static constexpr int WORDS = 9, BYTES = 144;
    static constexpr bool SUMS = true;
    template <int J> static PSN_DEV void weights(const lds_u8 *row, int g, u32x2 &b, float &d) {
        const lds_u8 *const p = row + 36 * (J >> 1);
        u32 s, q;
        if constexpr (J & 1) {
            fetch<4>(p + 20 + 4 * g, q);
            fetch<4>(p + 16, s);
            d = h2f_hi(s);
        } else {
            u32 q0, q1;
            fetch<4>(p + 4 * g, q0);
            fetch<4>(p + 4 * g + 4, q1);
            q = align2(q1, q0);
            fetch<4>(p, s);
            d = h2f_lo(s);
        }
        b = (u32x2){q & 0x0f0f0f0fu, (q >> 4) & 0x0f0f0f0fu};      /* elements 4 g + i and 16 + 4 g + i */
    }
    template <int J> static PSN_DEV void columns(const lds_u8 *x, int g, u32x2 &a) {
        u32 lo, hi;
        fetch<4>(x + 32 * J + 4 * g, lo);
        fetch<4>(x + 32 * J + 16 + 4 * g, hi);
        a = (u32x2){lo, hi};
    }
};

template <typename F>
PSN_DEV void mv_batch(const psn_matvec_args &a) {
    constexpr int NI = (16 * F::WORDS + 63) / 64;           /* load instructions per 16 rows and chunk */
    constexpr int XCOL = 272, MINE = 16 * F::BYTES + 8 * XCOL + 512;   /* (columns 272 bytes apart: other banks) */
    extern __shared__ uint4 psn_smem[];
    const int tid = threadIdx.x, lane = tid & 63, row = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = a.K, C = K >> 8, batch = a.batch;

    /* tiles do not straddle the matrices of a launch */
    const int e0 = a.row_end[0], e1 = a.row_end[1], e2 = a.row_end[2], e3 = a.row_end[3];
    const int t0 = (e0 + 15) >> 4, t1 = t0 + ((e1 - e0 + 15) >> 4), t2 = t1 + ((e2 - e1 + 15) >> 4);
    const int b = blockIdx.x, si = (b >= t0) + (b >= t1) + (b >= t2);
    const uint8_t *const W = si == 0 ? a.W[0] : si == 1 ? a.W[1] : si == 2 ? a.W[2] : a.W[3];
    float *const y = si == 0 ? a.y[0] : si == 1 ? a.y[1] : si == 2 ? a.y[2] : a.y[3];
    const int N = si == 0 ? e0 : si == 1 ? e1 - e0 : si == 2 ? e2 - e1 : e3 - e2;
    const int n0 = (b - (si == 0 ? 0 : si == 1 ? t0 : si == 2 ? t1 : t2)) * 16;

    lds_u8 *const wl = (lds_u8 *)(__attribute__((address_space(3))) void *)psn_smem + wave * MINE, *const xl = wl + 16 * F::BYTES, *const dl = xl + 8 * XCOL;

    float acc[4] = {0.f, 0.f, 0.f, 0.f};

    /* a tile past the last whole one is moved back so that all its rows exist (with N < 16 the last row repeats) */
    const int nb = min(n0, max(N - 16, 0));
    u32 woff[NI], wdst[NI], xoff[2];
    UNROLL for (int i = 0; i < NI; ++i) {
        const int word = min(i * 64 + lane, 16 * F::WORDS - 1), r = word / F::WORDS, wd = word % F::WORDS;
        woff[i] = (u32)(min(r, N - 1) * (int)a.row_bytes + wd * 16);
        wdst[i] = (u32)(r * F::BYTES + wd * 16);
    }
    UNROLL for (int u = 0; u < 2; ++u) xoff[u] = (u32)min(4 * u + (lane >> 4), batch - 1) * (u32)K + (u32)(row * 16);
    const u32 doff = ((u32)min(lane >> 3, batch - 1) * (u32)(K >> 5) + (u32)(lane & 7)) * 4u;    /* lane = column * 8 + block */
    const u32 xdst = (u32)(g * XCOL + row * 16), ddst = (u32)((lane & 7) * 32 + (lane >> 3) * 4);

    u32x4 w[NI], x[2];
    u32 xd, xs = 0;
    /* past the last chunk (valid false) every lane asks for the start of the buffers: no traffic, and the loop has one body */
    auto load = [&](int chunk) {
        const bool valid = chunk < C;
        const int c = valid ? chunk : 0;
        UNROLL for (int i = 0; i < NI; ++i) {
            u32 o = valid ? woff[i] : 0u;
            tie1(o);
            fetch<16>(W + (valid ? (int64_t)nb * a.row_bytes + (int64_t)c * F::BYTES : 0) + o, w[i]);
        }
        UNROLL for (int u = 0; u < 2; ++u) {
            u32 o = valid ? xoff[u] : 0u;
            tie1(o);
            fetch<16>(reinterpret_cast<const uint8_t *>(a.xqs) + (int64_t)c * 256 + o, x[u]);
        }
        u32 o = valid ? doff : 0u;
        tie1(o);
        fetch<4>(reinterpret_cast<const uint8_t *>(a.xd) + (int64_t)c * 32 + o, xd);
        if constexpr (F::SUMS) fetch<4>(reinterpret_cast<const uint8_t *>(a.xs) + (int64_t)c * 32 + o, xs);
    };
    const lds_u8 *const wrow = wl + row * F::BYTES, *const xcol = xl + (row & 7) * XCOL, *const dcol = dl + (g & 1) * 16;
    /* block J of the chunk in LDS; columns past 7 repeat 0..7 and are never stored */
    auto block = [&](auto jc) {
        constexpr int J = decltype(jc)::value;
        u32x2 xa;
        u32x4 dx, xc = (u32x4)(0u);
        F::template columns<J>(xcol, g, xa);
        fetch<16>(dcol + 32 * J, dx);
        if constexpr (F::SUMS) fetch<16>(dcol + (256 + 32 * J), xc);
        u32x2 wb;
        float d;
        F::template weights<J>(wrow, g, wb, d);
        const v4i p = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, xa), __builtin_bit_cast(long, wb), __builtin_bit_cast(v4i, xc), 0, 0, 0);
        UNROLL for (int r = 0; r < 4; ++r) acc[r] = __builtin_fmaf(d * __uint_as_float(dx[r]), (float)p[r], acc[r]);
    };
    if (wave < C) {
        load(wave);
        for (int c = wave; c < C; c += 8) {
            lds_order();                                    /* the reads of the chunk before */
            UNROLL for (int i = 0; i < NI; ++i) store<16>(wl + wdst[i], w[i]);
            UNROLL for (int u = 0; u < 2; ++u) store<16>(xl + u * 4 * XCOL + xdst, x[u]);
            store<4>(dl + ddst, xd);
            if constexpr (F::SUMS) store<4>(dl + 256 + ddst, (u32)(-8 * (int)xs));
            lds_order();
            __builtin_amdgcn_sched_barrier(0);
            load(c + 8);
            __builtin_amdgcn_sched_barrier(0);
            block(ic<0>()); block(ic<1>()); block(ic<2>()); block(ic<3>()); block(ic<4>()); block(ic<5>()); block(ic<6>()); block(ic<7>());
        }
    }

    /* partial tiles of the eight waves -> LDS ([wave][register][lane]), then summed in the order of the waves */
    float *const part_sums = reinterpret_cast<float *>(psn_smem);
    __syncthreads();
    UNROLL for (int r = 0; r < 4; ++r) part_sums[wave * 256 + r * 64 + lane] = acc[r];
    __syncthreads();
    if (tid < 256) {
        float sum = part_sums[tid];
        UNROLL for (int v = 1; v < 8; ++v) sum += part_sums[v * 256 + tid];
        const int n = nb + row, m = 4 * g + (tid >> 6);
        if (m < batch && n >= n0 && n < N) y[(int64_t)m * N + n] = sum;
    }
}

#define PSN_MVB(fmt, F) extern "C" __global__ void __launch_bounds__(512) psn_mvb_##fmt##_q8(const psn_matvec_args a) { mv_batch<F>(a); }
PSN_MVB(q4_0, BtQ4_0)
PSN_MVB(q8_0, BtQ8_0)
