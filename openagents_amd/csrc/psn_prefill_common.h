/*
 * psn_prefill_common.h -- fp16 / MFMA types, the LDS tile layout and the dequantization steps that the prefill kernel
 * families share.
 */
#ifndef PSN_PREFILL_COMMON_H
#define PSN_PREFILL_COMMON_H

#include "psn_args.h"
#include "psn_device.h"
#include "psn_prefill_lds.h"

#define UNROLL _Pragma("unroll")

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char lds_char;

/* An fp16 tile in LDS: rows of 128 bytes (64 k), the eight 16-byte chunks of a row stored at chunk ^ tile_swz(row).  A
 * fragment read takes the same chunk of 16 consecutive rows at a time: over the 64 banks (256 bytes) they must fall into
 * sixteen different 16-byte columns, (row & 1) * 8 + position -- so it is row bits 1..3 that scatter, not bits 0..2, which
 * put rows r and r + 8 into one column and cost every read four extra cycles.  (Q4_K 512 x 14336 x 4096, SQ_LDS_BANK_CONFLICT of
 * SQ_LDS_IDX_ACTIVE: four-wave 128 x 256 kernel 5.5e6 of 1.47e7 with bits 0..2, 3.7e6 of 1.28e7 with bits 1..3; the eight-wave 256 x 128 kernel
 * 1.9e6 of 1.11e7.) */
PSN_DEV int tile_swz(int row) { return (row >> 1) & 7; }
PSN_DEV int tile_off(int row, int chunk) { return row * 128 + ((chunk ^ tile_swz(row)) << 4); }

PSN_DEV u32 h2_bits(half2_t v) { return __builtin_bit_cast(u32, v); }
PSN_DEV half2_t bits_h2(u32 v) { return __builtin_bit_cast(half2_t, v); }

/* four bytes of v (already masked to the wanted 0..255 values) -> four fp16 (1024 + byte) in element
 * order, minus `bias`, times the block scale */
PSN_DEV void bytes_to_h4(u32 v, u32 keep, half2_t bias, half2_t d2, u32 &lo, u32 &hi) {
    const u32 t01 = __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u) & keep;   /* [b0, 0x64, b1, 0x64] */
    const u32 t23 = __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u) & keep;   /* [b2, 0x64, b3, 0x64] */
    lo = h2_bits((bits_h2(t01) - bias) * d2);
    hi = h2_bits((bits_h2(t23) - bias) * d2);
}

PSN_DEV u32 pack_h2_rn(float a, float b) {
    const half2_t v = {(_Float16)a, (_Float16)b};
    return h2_bits(v);
}
PSN_DEV void pf_kq_scales(u32 s0, u32 s1, u32 s2, u32 (&sc)[2], u32 (&mn)[2]) {
    sc[0] = s0 & 0x3f3f3f3fu;
    mn[0] = s1 & 0x3f3f3f3fu;
    sc[1] = (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u);
    mn[1] = ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u);
}
template <int I> PSN_DEV float pf_byte(const u32 (&v)[2]) { return (float)((v[I >> 2] >> (8 * (I & 3))) & 0xffu); }
/* four unsigned byte values of q -> d1 * q - m1, two packed pairs */
PSN_DEV void pf_affine4(u32 q, float d1, float m1, u32 &lo, u32 &hi) {
    const float v0 = __builtin_fmaf(d1, (float)(q & 0xffu), -m1), v1 = __builtin_fmaf(d1, (float)((q >> 8) & 0xffu), -m1);
    const float v2 = __builtin_fmaf(d1, (float)((q >> 16) & 0xffu), -m1), v3 = __builtin_fmaf(d1, (float)(q >> 24), -m1);
    lo = pack_h2_rn(v0, v1);
    hi = pack_h2_rn(v2, v3);
}

template <int N> struct pf_int { static constexpr int value = N; };
template <int I, int N, class F> PSN_DEV void static_for(F &&f) {
    if constexpr (I < N) {
        f(pf_int<I>());
        static_for<I + 1, N>(f);
    }
}

/* 16 bytes per lane from memory to 1 KB of LDS, in the order of the lanes */
PSN_DEV void load_to_lds(const char *from, lds_char *to) {
    __builtin_amdgcn_global_load_lds((const void *)from, (__attribute__((address_space(3))) void *)to, 16, 0, 0);
}

/* Which tile and K range a workgroup takes (kernels of psn_prefill_frag.hip, psn_prefill_pp.hip and psn_prefill_dense.hip).  Workgroups b, b + 8, ... share an XCD and its L2: each XCD gets one contiguous piece of the
 * order "K range, ROWS rows of X, N tile, M tile within the rows", so that the 32 compute units of an XCD share a few panels of X and of W, and no XCD has more than one
 * workgroup more than another (dealing N tiles to the XCDs in turn left 5120 columns in tiles of 256 with three tiles on four of them and two on the others). */
struct prefill_place { int m0, n0, c0, chunks; };            /* corner of the tile; first 256-wide chunk of K and how many */
template <int BM, int BN, int ROWS> PSN_DEV bool place_workgroup(const psn_prefill_args &a, prefill_place &p) {
    constexpr int GROUP = ROWS / BM;
    const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN, tiles = mt * nt, total = tiles * a.ksplit;
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, each = total >> 3, more = total & 7;
    if (local >= each + (xcd < more)) return false;
    const int idx = xcd * each + min(xcd, more) + local, split = idx / tiles, in = idx % tiles;
    const int per = GROUP * nt, g = in / per, r = in % per, rows = min(GROUP, mt - g * GROUP);
    p.m0 = (g * GROUP + r % rows) * BM;
    p.n0 = r / rows * BN;
    const int C = a.K >> 8, range = (C + a.ksplit - 1) / a.ksplit, c1 = min((split + 1) * range, C);
    p.c0 = split * range;
    p.chunks = c1 - p.c0;
    return p.chunks > 0;                                     /* an empty K range adds nothing */
}

/* D = W X^T: lane (q, m) = (lane / 16, lane % 16) ends with rows 4 q .. 4 q + 3 of W for row m of X */
PSN_DEV f32x4 mfma16(u32x4 w, u32x4 x, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, w), __builtin_bit_cast(half8_t, x), c, 0, 0, 0);
}
/* A wave's results of one row of MFMA tiles: lane (q, m) holds columns 16 j + 4 q .. + 3 of row m.  They go through LDS (16 rows of 16 TN + 4 words at `out`, this wave's own), so
 * that an instruction touches whole runs of a row of Y: 16-byte pieces of it where rows are whole 16-byte words and nothing has to be added (stored straight from the
 * MFMA's layout, 64 bytes of sixteen rows at a time: 4001 x 14336 x 4096 7 us more, 4001 x 1024 x 4096 on 256 x 256 tiles 9 more), else words: atomic adds
 * from the MFMA's layout take several times as long (512 x 1024 x 4096 in four ranges, 64 x 128 tiles: 33.3 us instead of 13.5). */
template <int TN> constexpr int wave_out_bytes() { return 16 * (16 * TN + 4) * 4; }
/* the rows' second half of the way: COLS columns of ROWS rows, COLS + 4 words apart at `out`, written by this wave */
template <int ROWS, int COLS> PSN_DEV void store_rows(const psn_prefill_args &a, int row0, int col0, int lane, u32 out) {
    constexpr int PITCH = (COLS + 4) * 4, P16 = COLS / 4, T = ROWS * P16 / 64;
    lds_wait();
    if (a.ksplit == 1 && (a.N & 3) == 0) {
        u32x4 w[T];
        UNROLL for (int t = 0; t < T; ++t) w[t] = lds_read128<0>(out + (u32)((t * 64 + lane) / P16 * PITCH + (t * 64 + lane) % P16 * 16));
        lds_wait();
        tie(w);
        UNROLL for (int t = 0; t < T; ++t) {
            const int row = row0 + (t * 64 + lane) / P16, col = col0 + (t * 64 + lane) % P16 * 4;
            if (row < a.M && col < a.N) *reinterpret_cast<u32x4 *>(a.Y + (int64_t)row * a.N + col) = w[t];
        }
        return;
    }
    u32 w[4 * T];
    UNROLL for (int t = 0; t < 4 * T; ++t) w[t] = lds_read32(out + (u32)((t * 64 + lane) / COLS * PITCH + (t * 64 + lane) % COLS * 4));
    lds_wait();
    UNROLL for (int t = 0; t < 4 * T; ++t) {
        tie1(w[t]);
        const int row = row0 + (t * 64 + lane) / COLS, col = col0 + (t * 64 + lane) % COLS;
        if (row >= a.M || col >= a.N) continue;
        float *y = a.Y + (int64_t)row * a.N + col;
        if (a.ksplit == 1) *y = __uint_as_float(w[t]);
        else unsafeAtomicAdd(y, __uint_as_float(w[t]));
    }
}
template <int TN> PSN_DEV void store_tiles(const psn_prefill_args &a, int row0, int col0, int lane, const f32x4 (&v)[TN], u32 out) {
    constexpr int PITCH = (16 * TN + 4) * 4;
    UNROLL for (int j = 0; j < TN; ++j) lds_write128(out + (u32)((lane & 15) * PITCH + 64 * j + 16 * (lane >> 4)), __builtin_bit_cast(u32x4, v[j]));
    store_rows<16, 16 * TN>(a, row0, col0, lane, out);
}
/* The same from 32 x 32 x 16 products: lane (h, m) = (lane / 32, lane % 32) holds columns 32 j + 8 g + 4 h .. + 3 of row m in registers 4 g .. 4 g + 3; 32 rows of 32 TN + 4 words. */
template <int TN> constexpr int wave_out_bytes32() { return 32 * (32 * TN + 4) * 4; }
template <int TN> PSN_DEV void store_tiles(const psn_prefill_args &a, int row0, int col0, int lane, const float16_t (&v)[TN], u32 out) {
    constexpr int PITCH = (32 * TN + 4) * 4;
    UNROLL for (int j = 0; j < TN; ++j) UNROLL for (int g = 0; g < 4; ++g) {
        const f32x4 p = {v[j][4 * g], v[j][4 * g + 1], v[j][4 * g + 2], v[j][4 * g + 3]};
        lds_write128(out + (u32)((lane & 31) * PITCH + 128 * j + 32 * g + 16 * (lane >> 5)), __builtin_bit_cast(u32x4, p));
    }
    store_rows<32, 32 * TN>(a, row0, col0, lane, out);
}

#endif
