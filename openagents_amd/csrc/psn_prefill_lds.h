/*
 * psn_prefill_lds.h -- LDS that the prefill kernels are launched with, by format and tile.  The host's sizes; every kernel asserts at compile time
 * that its own layout is this large and that what it keeps in LDS at its end fits.
 */
#ifndef PSN_PREFILL_LDS_H
#define PSN_PREFILL_LDS_H

/* formats in the order of the planner's tables */
enum { PSN_F_Q4_0, PSN_F_Q8_0, PSN_F_Q4_K, PSN_F_Q5_K, PSN_F_Q6_K };
constexpr int PSN_LDS_MAX = 160 * 1024;
constexpr bool psn_lds_scales(int f) { return f == PSN_F_Q4_K || f == PSN_F_Q5_K; }                 /* formats whose unpacked scales pass through LDS */

/* 16-byte words of a row's 256-wide chunk, as they come from memory, and bytes between rows in the thin kernels */
constexpr int psn_lds_words(int f) { return f == PSN_F_Q8_0 ? 17 : f == PSN_F_Q5_K ? 11 : f == PSN_F_Q6_K ? 13 : 9; }
constexpr int psn_lds_thin_row(int f) { return f == PSN_F_Q6_K ? 224 : 16 * psn_lds_words(f); }

/* family 4, eight waves.  256 rows (psn_prefill_pp.hip): a ring of four stages of X and two fp16 weight tiles, 128 bytes per row.  Fewer (psn_prefill_frag.hip): two stages of X of 256
 * bytes per row, two chunks of the weight rows in 1 KB pieces and one piece that nobody reads, Q6_K's last words of a row apart, the unpacked scales. */
constexpr int psn_lds_in_loop(int f, int bm, int bn) {
    if (bm == 256) return (4 * bm + 2 * bn) * 128;
    return 2 * (bm * 256 + ((bn * psn_lds_words(f) + 63) / 64 + 1) * 1024 + (f == PSN_F_Q6_K ? bn * 8 : 0)) + (psn_lds_scales(f) ? bn * 64 : 0);
}
/* the dense multiply: three stages of X (64 k) and four steps of W (32 k) with 256 columns, else a ring of four (64 x 64 tiles: five) stages of both */
constexpr int psn_lds_dense(int bm, int bn) { return bn == 256 ? 3 * bm * 128 + 4 * bn * 64 : (bm + bn) * 128 * (bm == 64 && bn == 64 ? 5 : 4); }
/* thin: eight waves with 16 rt weight rows' chunk, their unpacked scales where there is room (64 bytes a row) and 16 tm rows of X (64 k) each; at the end the waves' sums */
constexpr int psn_lds_thin_rings(int f, int tm, int rt, bool scales) { return 8 * (16 * rt * (psn_lds_thin_row(f) + (scales ? 64 : 0)) + tm * 2048); }
constexpr bool psn_lds_thin_scales(int f, int tm, int rt) { return psn_lds_scales(f) && psn_lds_thin_rings(f, tm, rt, true) <= PSN_LDS_MAX; }
constexpr int psn_lds_thin_sums(int tm, int rt) { return 8 * 1024 * rt * tm; }
constexpr int psn_lds_thin(int f, int tm, int rt) {
    return psn_lds_thin_rings(f, tm, rt, psn_lds_thin_scales(f, tm, rt)) > psn_lds_thin_sums(tm, rt) ? psn_lds_thin_rings(f, tm, rt, psn_lds_thin_scales(f, tm, rt)) : psn_lds_thin_sums(tm, rt);
}
/* skinny (Q4_0, Q8_0): three X chunks (64 rows x 256 k) and six or three raw weight chunks (64 rows of 144 or 304 bytes), at the end 8 x 16 KB of sums */
constexpr int psn_lds_skinny_rings(int f) { return 3 * 32768 + (f == PSN_F_Q4_0 ? 6 * 64 * 144 : 3 * 64 * 304); }
constexpr int psn_lds_skinny(int f) { return psn_lds_skinny_rings(f) > 8 * 16384 ? psn_lds_skinny_rings(f) : 8 * 16384; }
/* wide (Q4_0, Q8_0): three stages of X (256 rows x 64 k) and of raw blocks (two per row) */
constexpr int psn_lds_wide(int f) { return 3 * (32768 + 256 * (f == PSN_F_Q4_0 ? 36 : 68)); }
/* the four-wave kernels: two stages of X and of fp16 weights (64 k) */
constexpr int psn_lds_base(int bm, int bn) { return 2 * (bm + bn) * 128; }

#endif
