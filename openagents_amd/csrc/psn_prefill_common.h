/*
 * psn_prefill_common.h -- fp16 / MFMA types, the LDS tile layout and the dequantization steps that the prefill kernel
 * families share.
 */
#ifndef PSN_PREFILL_COMMON_H
#define PSN_PREFILL_COMMON_H

#define UNROLL _Pragma("unroll")

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));

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

#endif
