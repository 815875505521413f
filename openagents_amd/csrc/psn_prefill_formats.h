/*
 * psn_prefill_formats.h -- what a weight format's share of one thread looks like to the prefill kernels that decode in
 * their loop: which bytes a thread asks for, and how they become fp16.
 */
#ifndef PSN_PREFILL_FORMATS_H
#define PSN_PREFILL_FORMATS_H

#include "psn_device.h"
#include "psn_prefill_common.h"

/* ---- raw bytes of a thread, in one to five registers, loaded without a wait.  Every load is aligned to four bytes: 16- and
 *      8-byte loads from odd halfwords (where the quants of Q4_0, Q8_0 and Q6_K blocks start) take two to three times as long
 *      (a whole 14336 x 4096 matrix streamed by 112 workgroups: Q4_0 22.5 us against 9.9, Q8_0 32.9 against 22.4), so those
 *      formats fetch the aligned words around their bytes and pick the bytes out with v_perm.  ("+v": the load's target is the
 *      very register the variable lives in, so that no copy of it is made while the bytes are still on their way.) ---- */
typedef u32 u32x3 __attribute__((ext_vector_type(3)));
template <int NB> struct raw_bytes;
template <> struct raw_bytes<8> { typedef u32x2 t; };
template <> struct raw_bytes<12> { typedef u32x3 t; };
template <> struct raw_bytes<16> { typedef u32x4 t; };
PSN_DEV u32 raw_word(u32 v, int) { return v; }
PSN_DEV u32 raw_word(u32x2 v, int i) { return v[i]; }
PSN_DEV u32 raw_word(u32x3 v, int i) { return v[i]; }
PSN_DEV u32 raw_word(u32x4 v, int i) { return v[i]; }
template <int OFF> PSN_DEV void raw_load(const uint8_t *p, u32 &v) { asm volatile("global_load_dword %0, %1, off offset:%2" : "+v"(v) : "v"(p), "n"(OFF) : "memory"); }
template <int OFF> PSN_DEV void raw_load(const uint8_t *p, u32x2 &v) { asm volatile("global_load_dwordx2 %0, %1, off offset:%2" : "+v"(v) : "v"(p), "n"(OFF) : "memory"); }
template <int OFF> PSN_DEV void raw_load(const uint8_t *p, u32x3 &v) { asm volatile("global_load_dwordx3 %0, %1, off offset:%2" : "+v"(v) : "v"(p), "n"(OFF) : "memory"); }
template <int OFF> PSN_DEV void raw_load(const uint8_t *p, u32x4 &v) { asm volatile("global_load_dwordx4 %0, %1, off offset:%2" : "+v"(v) : "v"(p), "n"(OFF) : "memory"); }
template <int OFF> PSN_DEV void raw_load_u16(const uint8_t *p, u32 &v) { asm volatile("global_load_ushort %0, %1, off offset:%2" : "+v"(v) : "v"(p), "n"(OFF) : "memory"); }
template <typename T> PSN_DEV void raw_tie(T &v) { asm volatile("" : "+v"(v)); }

/* ---- four weights in two pieces of about five instructions each (what fits behind an MFMA): bytes -> `half_done`, then
 *      half_done -> four fp16.  K-quants: the bytes as floats, then d * q - m and the conversion to fp16 (fused multiply-add
 *      and v_cvt_pk_f16_f32 issue in half the cycles of v_fma_mix).  Q4_0 / Q8_0: 1024 + byte as fp16, then minus the bias,
 *      times the scale. ---- */
struct half_done { float f[4]; u32 h[2]; };
PSN_DEV void kq_floats(u32 q, half_done &t) {
    asm volatile("" : "+v"(q));                          /* (else the mask becomes a bit-field extract per byte instead of v_cvt_f32_ubyteN) */
    UNROLL for (int i = 0; i < 4; ++i) t.f[i] = (float)((q >> (8 * i)) & 0xffu);
}
typedef float float2_t __attribute__((ext_vector_type(2)));
PSN_DEV void kq_finish(const half_done &t, float d, float m, u32 &o0, u32 &o1) {
    const float2_t a = {__builtin_fmaf(d, t.f[0], -m), __builtin_fmaf(d, t.f[1], -m)}, b = {__builtin_fmaf(d, t.f[2], -m), __builtin_fmaf(d, t.f[3], -m)};
    o0 = h2_bits(__builtin_convertvector(a, half2_t));
    o1 = h2_bits(__builtin_convertvector(b, half2_t));
}
PSN_DEV void q0_halves(u32 v, u32 keep, half_done &t) {
    t.h[0] = __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u) & keep;
    t.h[1] = __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u) & keep;
}
PSN_DEV void q0_finish(const half_done &t, u32 bias, u32 d2, u32 &o0, u32 &o1) {
    o0 = h2_bits((bits_h2(t.h[0]) - bits_h2(bias)) * bits_h2(d2));
    o1 = h2_bits((bits_h2(t.h[1]) - bits_h2(bias)) * bits_h2(d2));
}

/* ---- a format's share of one thread: part `part` of 32 / NB parts of a row (NB = 8: four).  `base` is the row's chunk plus lane_off(part);
 *      load() asks for everything the four steps of the chunk need (LOADS instructions); step J's bytes are two groups
 *      (HI = 0, 1) of NB weights, which belong at k = k_lo(part) and k_hi(part) of the 64-wide step; first() and second() turn
 *      word i of a group into four fp16, with the step's scales from scales0() and scales1().  SPREAD: row_of() in psn_prefill_pp.hip. ---- */
/* Scales of Q4_K / Q5_K.  Unpacking the two sub-blocks of a 64-wide step costs twenty instructions, as much as decoding seven weights, and four threads share a row: each does
 * it for one of the chunk's four steps (kq_pick: the fields of step j; kq_own: d, d', m, m').  Next to each other (pp kernels) they hand the values round by quad_perm in each step; as
 * the four sixteens of lanes (FAR, thin kernels) through LDS, where the four floats of a step take the header's place in raw. */
PSN_DEV void kq_pick(u32x4 header, int j, u32 &scales, u32 &mins) {
    u32 sc[2], mn[2];
    pf_kq_scales(header.y, header.z, header.w, sc, mn);
    scales = ((j & 2) ? sc[1] : sc[0]) >> (16 * (j & 1));
    mins = ((j & 2) ? mn[1] : mn[0]) >> (16 * (j & 1));
}
PSN_DEV void kq_own(u32x4 header, u32 scales, u32 mins, float (&own)[4]) {
    const float d = h2f_lo(header.x), dm = h2f_hi(header.x);
    own[0] = __fmul_rn(d, (float)(scales & 0xffu));
    own[1] = __fmul_rn(d, (float)((scales >> 8) & 0xffu));
    own[2] = __fmul_rn(dm, (float)(mins & 0xffu));
    own[3] = __fmul_rn(dm, (float)((mins >> 8) & 0xffu));
}
template <int J> PSN_DEV float from_quad(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x55 * J, 0xf, 0xf, true)); }
template <int J, bool FAR, class S> PSN_DEV void kq_scales0(u32x4 header, int part, S &s) {
    if constexpr (FAR) { s.d[0] = __uint_as_float(header.x); s.d[1] = __uint_as_float(header.y); }
    else if constexpr (J == 0) kq_pick(header, part & 3, s.sc, s.mn);
    else { s.d[0] = from_quad<J>(s.own[0]); s.d[1] = from_quad<J>(s.own[1]); }
}
template <int J, bool FAR, class S> PSN_DEV void kq_scales1(u32x4 header, S &s) {
    if constexpr (FAR) { s.m[0] = __uint_as_float(header.z); s.m[1] = __uint_as_float(header.w); }
    else {
        if constexpr (J == 0) {
            kq_own(header, s.sc, s.mn, s.own);
            s.d[0] = from_quad<J>(s.own[0]);
            s.d[1] = from_quad<J>(s.own[1]);
        }
        s.m[0] = from_quad<J>(s.own[2]);
        s.m[1] = from_quad<J>(s.own[3]);
    }
}
struct PpQ4_K {
    static constexpr int FORMAT = PSN_F_Q4_K, BYTES = 144, LOADS = 5;
    template <int NB> struct raw { u32x4 h; typename raw_bytes<NB>::t q[4]; };
    template <int NB> static PSN_DEV int lane_off(int part) { return NB * part; }
    template <int NB> static PSN_DEV void load(const uint8_t *row, int lane, raw<NB> &r) {
        raw_load<0>(row, r.h);
        const uint8_t *p = row + lane;
        raw_load<16>(p, r.q[0]); raw_load<48>(p, r.q[1]); raw_load<80>(p, r.q[2]); raw_load<112>(p, r.q[3]);
    }
    template <int NB> static PSN_DEV void clear(raw<NB> &r) { r.h = (u32x4)(0u); UNROLL for (int j = 0; j < 4; ++j) r.q[j] = 0u; }
    template <int NB> static PSN_DEV void landed(raw<NB> &r) { raw_tie(r.h); UNROLL for (int j = 0; j < 4; ++j) raw_tie(r.q[j]); }
    struct scale { float d[2], m[2]; u32 sc, mn; float own[4]; };
    template <int J, int NB, bool FAR = false> static PSN_DEV void scales0(const raw<NB> &r, int part, scale &s) { kq_scales0<J, FAR>(r.h, part, s); }
    template <int J, int NB, bool FAR = false> static PSN_DEV void scales1(const raw<NB> &r, scale &s) { kq_scales1<J, FAR>(r.h, s); }
    template <int J, int NB, int HI> static PSN_DEV void first(const raw<NB> &r, const scale &, int i, half_done &t) { kq_floats((raw_word(r.q[J], i) >> (4 * HI)) & 0x0f0f0f0fu, t); }
    template <int HI> static PSN_DEV void second(const scale &s, const half_done &t, u32 &o0, u32 &o1) { kq_finish(t, s.d[HI], s.m[HI], o0, o1); }
    template <int NB> static PSN_DEV int k_lo(int part) { return NB * part; }
    template <int NB> static PSN_DEV int k_hi(int part) { return 32 + NB * part; }
    static constexpr int SPREAD = 3;
};
struct PpQ5_K {
    static constexpr int FORMAT = PSN_F_Q5_K, BYTES = 176, LOADS = 6;
    template <int NB> struct raw { u32x4 h; typename raw_bytes<NB>::t top, q[4]; };
    template <int NB> static PSN_DEV int lane_off(int part) { return NB * part; }
    template <int NB> static PSN_DEV void load(const uint8_t *row, int lane, raw<NB> &r) {
        raw_load<0>(row, r.h);
        const uint8_t *p = row + lane;
        raw_load<16>(p, r.top);
        raw_load<48>(p, r.q[0]); raw_load<80>(p, r.q[1]); raw_load<112>(p, r.q[2]); raw_load<144>(p, r.q[3]);
    }
    template <int NB> static PSN_DEV void clear(raw<NB> &r) { r.h = (u32x4)(0u); r.top = 0u; UNROLL for (int j = 0; j < 4; ++j) r.q[j] = 0u; }
    template <int NB> static PSN_DEV void landed(raw<NB> &r) { raw_tie(r.h); raw_tie(r.top); UNROLL for (int j = 0; j < 4; ++j) raw_tie(r.q[j]); }
    struct scale { float d[2], m[2]; u32 sc, mn; float own[4]; };
    template <int J, int NB, bool FAR = false> static PSN_DEV void scales0(const raw<NB> &r, int part, scale &s) { kq_scales0<J, FAR>(r.h, part, s); }
    template <int J, int NB, bool FAR = false> static PSN_DEV void scales1(const raw<NB> &r, scale &s) { kq_scales1<J, FAR>(r.h, s); }
    template <int J, int NB, int HI> static PSN_DEV void first(const raw<NB> &r, const scale &, int i, half_done &t) { kq_floats(((raw_word(r.q[J], i) >> (4 * HI)) & 0x0f0f0f0fu) | (((raw_word(r.top, i) >> (2 * J + HI)) & 0x01010101u) << 4), t); }
    template <int HI> static PSN_DEV void second(const scale &s, const half_done &t, u32 &o0, u32 &o1) { kq_finish(t, s.d[HI], s.m[HI], o0, o1); }
    template <int NB> static PSN_DEV int k_lo(int part) { return NB * part; }
    template <int NB> static PSN_DEV int k_hi(int part) { return 32 + NB * part; }
    static constexpr int SPREAD = 3;
};
/* step J = half J / 2 of the super-block, quarters t = 2 (J & 1) and 2 (J & 1) + 1: the first 32 and the second 32 of
 * the half's 64 low-bit bytes, their low (J even) or high nibbles; bits 4..5 from the half's 32 high-bit bytes.  A
 * super-block (210 bytes) starts on a dword or two bytes behind one: `pick` takes four bytes out of two dwords accordingly. */
struct PpQ6_K {
    static constexpr int FORMAT = PSN_F_Q6_K, BYTES = 210, LOADS = 9;
    template <int NB> struct raw { typename raw_bytes<NB + 4>::t ql[4], qh[2]; u32x4 sc; u32 sc4, d, pick; };
    template <int NB> static PSN_DEV int lane_off(int part) { return NB * part; }
    template <int NB> static PSN_DEV void load(const uint8_t *row, int lane, raw<NB> &r) {
        const uint8_t *d = (const uint8_t *)((uintptr_t)row & ~(uintptr_t)3), *p = d + lane;
        r.pick = ((uintptr_t)row & 2) ? 0x05040302u : 0x03020100u;
        raw_load<0>(p, r.ql[0]); raw_load<32>(p, r.ql[1]); raw_load<64>(p, r.ql[2]); raw_load<96>(p, r.ql[3]);
        raw_load<128>(p, r.qh[0]); raw_load<160>(p, r.qh[1]);
        raw_load<192>(d, r.sc);
        /* the scales' last two bytes where the super-block starts two bytes late (else a dword inside it that nobody uses) */
        raw_load<204>((const uint8_t *)((uintptr_t)(row + 2) & ~(uintptr_t)3), r.sc4);
        raw_load_u16<208>(row, r.d);
    }
    template <int NB> static PSN_DEV void clear(raw<NB> &r) { r.sc = (u32x4)(0u); r.sc4 = r.d = r.pick = 0u; r.qh[0] = r.qh[1] = 0u; UNROLL for (int j = 0; j < 4; ++j) r.ql[j] = 0u; }
    template <int NB> static PSN_DEV void landed(raw<NB> &r) {
        UNROLL for (int j = 0; j < 4; ++j) raw_tie(r.ql[j]);
        raw_tie(r.qh[0]); raw_tie(r.qh[1]); raw_tie(r.sc); raw_tie(r.sc4); raw_tie(r.d);
    }
    struct scale { float d[2], m[2]; };
    template <int J, int NB, bool FAR = false> static PSN_DEV void scales0(const raw<NB> &r, int part, scale &s) {
        /* the scales of quarter t and (16 bits on) of quarter t + 1, each of this part's half */
        constexpr int I = 2 * (J >> 1) + (J & 1);
        const u32 v = __builtin_amdgcn_perm(I == 3 ? r.sc4 : r.sc[(I + 1) & 3], r.sc[I], r.pick) >> (8 * ((NB * part) >> 4));
        s.d[0] = (float)(int)(int8_t)(v & 0xffu);
        s.d[1] = (float)(int)(int8_t)((v >> 16) & 0xffu);
    }
    template <int J, int NB, bool FAR = false> static PSN_DEV void scales1(const raw<NB> &r, scale &s) {
        const float d = h2f_lo(r.d);
        UNROLL for (int i = 0; i < 2; ++i) { s.d[i] = __fmul_rn(d, s.d[i]); s.m[i] = s.d[i] * 32.f; }
    }
    template <int J, int NB, int HI> static PSN_DEV void first(const raw<NB> &r, const scale &, int i, half_done &t) {
        constexpr int H = J >> 1, T = 2 * (J & 1);
        const u32 a = __builtin_amdgcn_perm(raw_word(r.ql[2 * H + HI], i + 1), raw_word(r.ql[2 * H + HI], i), r.pick);
        const u32 b = __builtin_amdgcn_perm(raw_word(r.qh[H], i + 1), raw_word(r.qh[H], i), r.pick);
        kq_floats(((a >> (2 * T)) & 0x0f0f0f0fu) | (((b >> (2 * T + 2 * HI)) & 0x03030303u) << 4), t);
    }
    template <int HI> static PSN_DEV void second(const scale &s, const half_done &t, u32 &o0, u32 &o1) { kq_finish(t, s.d[HI], s.m[HI], o0, o1); }
    template <int NB> static PSN_DEV int k_lo(int part) { return NB * part; }
    template <int NB> static PSN_DEV int k_hi(int part) { return 32 + NB * part; }
    static constexpr int SPREAD = 3;
};
/* Q4_0 and Q8_0: step J = blocks 2 J and 2 J + 1, 36 (68) bytes from a dword on.  The first block's quants start two bytes
 * into its first dword, the second one's on a dword; so the dwords from DW * part on hold a part's bytes two (first block) or
 * four bytes in, its block's scale sits in the low (first block) or high half of the first dword of the block's first
 * part, and one v_perm selector per thread picks either. */
template <int PB, int NB> struct pp_blocks {               /* PB: bytes per part (NB or 2 NB) */
    static constexpr int PARTS = 32 / NB;
    static_assert(PARTS == 4, "a quad, or a part per sixteen lanes");
    static PSN_DEV bool second_block(int part) { return part >= PARTS / 2; }
    static PSN_DEV u32 pick(int part) { return second_block(part) ? 0x07060504u : 0x05040302u; }
    /* the block's scale in both halves.  FAR: the four parts of a row are the four sixteens of lanes, not neighbours */
    template <bool FAR> static PSN_DEV u32 scale(u32 first_dword, int part) {
        u32 v;
        if constexpr (FAR) {
            v = __builtin_amdgcn_permlane16_swap(first_dword, first_dword, false, false)[0];   /* lanes 16..31 get 0..15's, lanes 48..63 get 32..47's */
        } else {
            /* quad_perm: lanes of a quad read their block's first part (parts 0, 0, 2, 2) */
            v = (u32)__builtin_amdgcn_mov_dpp((int)first_dword, 0xA0, 0xf, 0xf, false);
        }
        return __builtin_amdgcn_perm(v, v, second_block(part) ? 0x03020302u : 0x01000100u);
    }
};
struct PpQ4_0 {
    static constexpr int FORMAT = PSN_F_Q4_0, BYTES = 144, LOADS = 4;
    template <int NB> struct raw { typename raw_bytes<NB + 4>::t q[4]; };
    template <int NB> static PSN_DEV int lane_off(int part) { return NB * part; }
    template <int NB> static PSN_DEV void load(const uint8_t *row, int lane, raw<NB> &r) {
        const uint8_t *p = row + lane;
        raw_load<0>(p, r.q[0]); raw_load<36>(p, r.q[1]); raw_load<72>(p, r.q[2]); raw_load<108>(p, r.q[3]);
    }
    template <int NB> static PSN_DEV void clear(raw<NB> &r) { UNROLL for (int j = 0; j < 4; ++j) r.q[j] = 0u; }
    template <int NB> static PSN_DEV void landed(raw<NB> &r) { UNROLL for (int j = 0; j < 4; ++j) raw_tie(r.q[j]); }
    struct scale { u32 d, q[2]; };
    template <int J, int NB, bool FAR = false> static PSN_DEV void scales0(const raw<NB> &r, int part, scale &s) {
        typedef pp_blocks<NB, NB> B;
        s.d = B::template scale<FAR>(raw_word(r.q[J], 0), part);
        UNROLL for (int i = 0; i < NB / 4; ++i) s.q[i] = __builtin_amdgcn_perm(raw_word(r.q[J], i + 1), raw_word(r.q[J], i), B::pick(part));
    }
    template <int J, int NB, bool FAR = false> static PSN_DEV void scales1(const raw<NB> &, scale &) {}
    template <int J, int NB, int HI> static PSN_DEV void first(const raw<NB> &, const scale &s, int i, half_done &t) { q0_halves(s.q[i] >> (4 * HI), 0x640f640fu, t); }
    template <int HI> static PSN_DEV void second(const scale &s, const half_done &t, u32 &o0, u32 &o1) { q0_finish(t, 0x64086408u, s.d, o0, o1); }
    /* low nibbles first, high nibbles sixteen further on */
    template <int NB> static PSN_DEV int k_lo(int part) { return 32 * ((NB * part) >> 4) + ((NB * part) & 15); }
    template <int NB> static PSN_DEV int k_hi(int part) { return k_lo<NB>(part) + 16; }
    static constexpr int SPREAD = 2;
};
struct PpQ8_0 {
    static constexpr int FORMAT = PSN_F_Q8_0, BYTES = 272, LOADS = 8;
    template <int NB> struct raw { typename raw_bytes<2 * NB>::t q[4]; u32 e[4]; };    /* e: the dword behind them */
    template <int NB> static PSN_DEV int lane_off(int part) { return 2 * NB * part; }
    template <int NB> static PSN_DEV void load(const uint8_t *row, int lane, raw<NB> &r) {
        const uint8_t *p = row + lane;
        raw_load<0>(p, r.q[0]); raw_load<2 * NB>(p, r.e[0]); raw_load<68>(p, r.q[1]); raw_load<68 + 2 * NB>(p, r.e[1]);
        raw_load<136>(p, r.q[2]); raw_load<136 + 2 * NB>(p, r.e[2]); raw_load<204>(p, r.q[3]); raw_load<204 + 2 * NB>(p, r.e[3]);
    }
    template <int NB> static PSN_DEV void clear(raw<NB> &r) { UNROLL for (int j = 0; j < 4; ++j) { r.q[j] = 0u; r.e[j] = 0u; } }
    template <int NB> static PSN_DEV void landed(raw<NB> &r) { UNROLL for (int j = 0; j < 4; ++j) { raw_tie(r.q[j]); raw_tie(r.e[j]); } }
    struct scale { u32 d, pick; };
    template <int J, int NB, bool FAR = false> static PSN_DEV void scales0(const raw<NB> &r, int part, scale &s) {
        typedef pp_blocks<2 * NB, NB> B;
        s.d = B::template scale<FAR>(raw_word(r.q[J], 0), part);
        s.pick = B::pick(part);
    }
    template <int J, int NB, bool FAR = false> static PSN_DEV void scales1(const raw<NB> &, scale &) {}
    template <int J, int NB, int HI> static PSN_DEV void first(const raw<NB> &r, const scale &s, int i, half_done &t) {
        const int w = HI * (NB / 4) + i;
        const u32 next = w + 1 < NB / 2 ? raw_word(r.q[J], w + 1 < NB / 2 ? w + 1 : 0) : r.e[J];
        q0_halves(__builtin_amdgcn_perm(next, raw_word(r.q[J], w), s.pick) ^ 0x80808080u, 0x64ff64ffu, t);
    }
    template <int HI> static PSN_DEV void second(const scale &s, const half_done &t, u32 &o0, u32 &o1) { q0_finish(t, 0x64806480u, s.d, o0, o1); }
    template <int NB> static PSN_DEV int k_lo(int part) { return 2 * NB * part; }
    template <int NB> static PSN_DEV int k_hi(int part) { return 2 * NB * part + NB; }
    static constexpr int SPREAD = 0;
};

#endif
