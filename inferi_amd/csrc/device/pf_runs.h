// Weight staging of the prefill GEMMs: half of one weight row's 64 elements of
// a K step read as GGUF block bytes, dequantized with the reference's f32
// arithmetic (crates/inferi/src/quantization.rs:47-392), rounded to f16 and
// stored in a swizzled LDS tile.
#pragma once
#include "gemv.h"

namespace ifr {

// f16 pair of two f32 values, each rounded to nearest from its f32 value
// (v_cvt_pk_f16_f32 written out, so the compiler cannot fuse the producing
// multiply or FMA into one rounding straight to f16, v_fma_mix)
IFR_DEV uint32_t pack_f16x2(float a, float b) {
    uint32_t u;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(u) : "v"(a), "v"(b));
    return u;
}
// f16 of one f32 value (v_cvt_f16_f32 written out, for the same reason)
IFR_DEV _Float16 f16_of(float a) {
    uint32_t u;
    asm("v_cvt_f16_f32 %0, %1" : "=v"(u) : "v"(a));
    const uint16_t b = (uint16_t)u;
    _Float16 h;
    __builtin_memcpy(&h, &b, 2);
    return h;
}

// LDS tiles: 256 rows of 64 halves (128 B) without padding; the 16-byte
// chunk c of row r sits at chunk c ^ s(r), s(r) = ((r / 2) ^ 4 (r % 2)) % 8.
// The sixteen consecutive rows whose 16-byte chunks one read pass serves (64
// banks of 4 bytes, two rows per bank line) fall on distinct banks; the
// dequantized row stores, two threads per row, meet fewer conflicts than
// with s(r) = (r / 2) % 8 (a microbenchmark of the two access patterns:
// reads 5.1 -> 4.7, stores 16.0 -> 14.1 cycles per wave instruction and CU;
// the 4095-token 8B prefill 69.4 -> 69.1 ms, alternated three times).
IFR_DEV uint32_t pg_swz_of(uint32_t r) { return ((r >> 1) ^ ((r & 1u) << 2)) & 7u; }
IFR_DEV uint32_t pg_swz(uint32_t r, uint32_t c) { return r * 64 + 8 * (c ^ pg_swz_of(r)); }

// The block affine map of the step's two sub-blocks 2g, 2g + 1 (g = (k0 %
// 256) / 64): y = d1 q + n1 (low nibbles), d2 q + n2 (high nibbles).
struct Q4kAffine {
    float d1, n1, d2, n2;
};
IFR_DEV Q4kAffine q4k_affine(const u32x4_a16 &hv, uint32_t k0) {
#pragma clang fp contract(off)
    uint32_t sc0, m0s, sc1, m1s;
    scale_min_pair((k0 % 256) / 64, hv.y, hv.z, hv.w, sc0, m0s, sc1, m1s);
    const float d = f16_to_f32(hv.x & 0xFFFFu), dm = f16_to_f32(hv.x >> 16);
    return Q4kAffine{d * (float)sc0, -(dm * (float)m0s), d * (float)sc1, -(dm * (float)m1s)};
}
typedef _Float16 f16x2v __attribute__((ext_vector_type(2)));

// PgRun<FMT>: one thread's half (part p) of a row's 64 elements of a K step.
// load() only loads (nothing is computed on the bytes, so nothing waits for
// them), pin() is where the compiler waits for them and keeps their
// dequantization behind the barrier before it, store() dequantizes into the
// swizzled f16 row r of a 64-wide tile (chunk indices exchanged by x).  The
// values are the reference's f32 ones, rounded to f16 once, with fewer
// instructions per weight than its arithmetic written out:
//  - a code c in the low bits of a 16-bit half is the f16 subnormal c 2^-24,
//    so fma(s 2^24, half, o) is fma(s, c, o), v_fma_mix_f32 reading the half in
//    place (pg_mix4).  Q4_K, Q5_K, Q4_1, Q5_1: s c is exact in f32, and the
//    fused sum rounds once as the reference's separate one does;
//  - Q6_K: the f16 integer c - 32 is exact, and v_fma_mix_f32 reads it in
//    place: fma(d sc, c - 32, -0) is the reference's product (pg_mul4);
//  - Q8_0, Q4_0, Q5_0: d (c - z) is exact in f32 (at most 19 bits), so its
//    rounding to f16 is the only one, and v_pk_mul_f16 of the exact f16
//    integer c - z rounds the same product once (pg_pk4).
// Two-byte aligned fields are read with the hardware's unaligned loads.

// Four codes, the bytes of c: y = s c + o, s given times 2^24, as two f16 pairs.
IFR_DEV void pg_mix4(uint32_t c, float s24, float o, uint32_t &u0, uint32_t &u1) {
    const f16x2v a = __builtin_bit_cast(f16x2v, c & 0x00FF00FFu), b = __builtin_bit_cast(f16x2v, (c >> 8) & 0x00FF00FFu);
    u0 = pack_f16x2(fmaf(s24, (float)a.x, o), fmaf(s24, (float)b.x, o));
    u1 = pack_f16x2(fmaf(s24, (float)a.y, o), fmaf(s24, (float)b.y, o));
}
// Four codes, the bytes of c: y = d (c - z) in f16.  0x6400 | c is 1024 + c.
IFR_DEV void pg_pk4(uint32_t c, _Float16 d, _Float16 z1024, uint32_t &u0, uint32_t &u1) {
    const f16x2v dd = {d, d}, z = {z1024, z1024};
    const f16x2v a = __builtin_bit_cast(f16x2v, __builtin_amdgcn_perm(0x64646464u, c, 0x04010400u));
    const f16x2v b = __builtin_bit_cast(f16x2v, __builtin_amdgcn_perm(0x64646464u, c, 0x04030402u));
    u0 = __builtin_bit_cast(uint32_t, (a - z) * dd);
    u1 = __builtin_bit_cast(uint32_t, (b - z) * dd);
}
// Four codes, the bytes of c: y = s (c - z) in f32, as two f16 pairs.  The
// addend -0 keeps every product's sign; written out, since the compiler takes
// the sum away again and converts each half by itself.
IFR_DEV float pg_mul_lo(float s, uint32_t h) {
    float y;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[0,1,0]" : "=v"(y) : "v"(s), "v"(h), "v"(-0.0f));
    return y;
}
IFR_DEV float pg_mul_hi(float s, uint32_t h) {
    float y;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(y) : "v"(s), "v"(h), "v"(-0.0f));
    return y;
}
IFR_DEV void pg_mul4(uint32_t c, float s, _Float16 z1024, uint32_t &u0, uint32_t &u1) {
    const f16x2v z = {z1024, z1024};
    const f16x2v a = __builtin_bit_cast(f16x2v, __builtin_amdgcn_perm(0x64646464u, c, 0x04010400u)) - z;
    const f16x2v b = __builtin_bit_cast(f16x2v, __builtin_amdgcn_perm(0x64646464u, c, 0x04030402u)) - z;
    const uint32_t ua = __builtin_bit_cast(uint32_t, a), ub = __builtin_bit_cast(uint32_t, b);
    u0 = pack_f16x2(pg_mul_lo(s, ua), pg_mul_hi(s, ua));
    u1 = pack_f16x2(pg_mul_lo(s, ub), pg_mul_hi(s, ub));
}
// 16 values as chunks c and c ^ 1 of tile row r.
IFR_DEV void pg_put16(const uint32_t (&u)[8], _Float16 *tile, uint32_t r, uint32_t c) {
    *(uint4 *)(tile + pg_swz(r, c)) = make_uint4(u[0], u[1], u[2], u[3]);
    *(uint4 *)(tile + pg_swz(r, c ^ 1u)) = make_uint4(u[4], u[5], u[6], u[7]);
}
IFR_DEV _Float16 pg_half(uint32_t b) { return __builtin_bit_cast(_Float16, (uint16_t)b); }

template <int FMT>
struct PgRun;

// Q4_K: the 16 qs bytes [32 g + 16 p, +16) of the step's group g: low nibbles
// to chunks 2p, 2p + 1, high ones to 4 + 2p, 5 + 2p.
template <>
struct PgRun<Q4_K> {
    u32x4_a16 hv, qv;
    IFR_DEV void load(const uint8_t *wrow, uint32_t k0, uint32_t p) {
        const uint8_t *b = wrow + (size_t)(k0 / 256) * 144;
        hv = *(const u32x4_a16 *)b;
        qv = *(const u32x4_a16 *)(b + 16 + 32 * ((k0 % 256) / 64) + 16 * p);
    }
    IFR_DEV void pin() { asm volatile("" : "+v"(hv), "+v"(qv)); }
    template <int H>
    IFR_DEV void store(uint32_t k0, uint32_t p, _Float16 *tile, uint32_t r, uint32_t x) const {
        const Q4kAffine f = q4k_affine(hv, k0);
        uint32_t u[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (H == 0) pg_mix4(qv[i] & 0x0F0F0F0Fu, f.d1 * 0x1p24f, f.n1, u[2 * i], u[2 * i + 1]);
            else pg_mix4(qv[i] & 0xF0F0F0F0u, f.d2 * 0x1p20f, f.n2, u[2 * i], u[2 * i + 1]);
        }
        pg_put16(u, tile, r, (4 * H + 2 * p) ^ x);
    }
};
// Q5_K: the same with the fifth bits, bits 2g and 2g + 1 of qh[16 p, +16).
template <>
struct PgRun<Q5_K> {
    u32x4_a16 hv, ev, qv;
    IFR_DEV void load(const uint8_t *wrow, uint32_t k0, uint32_t p) {
        const uint8_t *b = wrow + (size_t)(k0 / 256) * 176;
        hv = *(const u32x4_a16 *)b;
        ev = *(const u32x4_a16 *)(b + 16 + 16 * p);
        qv = *(const u32x4_a16 *)(b + 48 + 32 * ((k0 % 256) / 64) + 16 * p);
    }
    IFR_DEV void pin() { asm volatile("" : "+v"(hv), "+v"(ev), "+v"(qv)); }
    template <int H>
    IFR_DEV void store(uint32_t k0, uint32_t p, _Float16 *tile, uint32_t r, uint32_t x) const {
        const Q4kAffine f = q4k_affine(hv, k0);
        const uint32_t sh = 2 * ((k0 % 256) / 64);
        uint32_t u[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t e = ev[i] >> sh;
            if constexpr (H == 0)
                pg_mix4((qv[i] & 0x0F0F0F0Fu) | (e & 0x01010101u) << 4, f.d1 * 0x1p24f, f.n1, u[2 * i], u[2 * i + 1]);
            else
                pg_mix4(((qv[i] >> 4) & 0x0F0F0F0Fu) | (e & 0x02020202u) << 3, f.d2 * 0x1p24f, f.n2, u[2 * i], u[2 * i + 1]);
        }
        pg_put16(u, tile, r, (4 * H + 2 * p) ^ x);
    }
};
// Q6_K (quantization.rs:224-257): the step's 64 elements are the low (g even)
// or high nibbles of ql[64 i, +64), i = g / 2, and bits 4 (g % 2) .. + 3 of
// qh[32 i, +32); part p takes bytes 16 p .. + 15 of each 32, whose scales are
// bytes 8 i + 4 (g % 2) + p and + 2.
template <>
struct PgRun<Q6_K> {
    u32x4_a2 q0, q1, hv;
    uint32_t sc, dd;
    IFR_DEV void load(const uint8_t *wrow, uint32_t k0, uint32_t p) {
        const uint32_t g = (k0 % 256) / 64, i = g >> 1;
        const uint8_t *b = wrow + (size_t)(k0 / 256) * 210;
        q0 = *(const u32x4_a2 *)(b + 64 * i + 16 * p);
        q1 = *(const u32x4_a2 *)(b + 64 * i + 32 + 16 * p);
        hv = *(const u32x4_a2 *)(b + 128 + 32 * i + 16 * p);
        sc = *(const u32_a2 *)(b + 192 + 8 * i + 4 * (g & 1u));
        dd = *(const uint16_t *)(b + 208);
    }
    IFR_DEV void pin() { asm volatile("" : "+v"(q0), "+v"(q1), "+v"(hv), "+v"(sc), "+v"(dd)); }
    template <int H>
    IFR_DEV void store(uint32_t k0, uint32_t p, _Float16 *tile, uint32_t r, uint32_t x) const {
#pragma clang fp contract(off)
        const uint32_t s4 = 4 * (((k0 % 256) / 64) & 1u), ss = sc >> (8 * p);
        const float d = f16_to_f32(dd) * (float)(int)(int8_t)((H ? ss >> 16 : ss) & 0xFFu);
        uint32_t u[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t h = hv[i] >> s4;
            if constexpr (H == 0)
                pg_mul4(((q0[i] >> s4) & 0x0F0F0F0Fu) | (h & 0x03030303u) << 4, d, (_Float16)1056.0f, u[2 * i], u[2 * i + 1]);
            else
                pg_mul4(((q1[i] >> s4) & 0x0F0F0F0Fu) | (h & 0x0C0C0C0Cu) << 2, d, (_Float16)1056.0f, u[2 * i], u[2 * i + 1]);
        }
        pg_put16(u, tile, r, (4 * H + 2 * p) ^ x);
    }
};
// Q8_K: its f32 scale times 2^24 could overflow, so each code is converted.
template <>
struct PgRun<Q8_K> {
    u32x4_a4 q0, q1;
    float d;
    IFR_DEV void load(const uint8_t *wrow, uint32_t k0, uint32_t p) {
        const uint8_t *b = wrow + (size_t)(k0 / 256) * 292;
        d = *(const float *)b;
        q0 = *(const u32x4_a4 *)(b + 4 + (k0 % 256) + 32 * p);
        q1 = *(const u32x4_a4 *)(b + 20 + (k0 % 256) + 32 * p);
    }
    IFR_DEV void pin() { asm volatile("" : "+v"(q0), "+v"(q1), "+v"(d)); }
    template <int H>
    IFR_DEV void store(uint32_t, uint32_t p, _Float16 *tile, uint32_t r, uint32_t x) const {
#pragma clang fp contract(off)
        uint32_t u[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int a = (int)(H ? q1[i] : q0[i]);
            u[2 * i] = pack_f16x2(d * (float)(int8_t)a, d * (float)(int8_t)(a >> 8));
            u[2 * i + 1] = pack_f16x2(d * (float)(int8_t)(a >> 16), d * (float)(a >> 24));
        }
        pg_put16(u, tile, r, (4 * p + 2 * H) ^ x);
    }
};
// Unquantized rows: elements [32 p, +32) as they are, or rounded to f16.
template <>
struct PgRun<F16> {
    u32x4_a16 v[4];
    IFR_DEV void load(const uint8_t *wrow, uint32_t k0, uint32_t p) {
        const u32x4_a16 *b = (const u32x4_a16 *)(wrow + 2 * (size_t)(k0 + 32 * p));
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = b[i];
    }
    IFR_DEV void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])); }
    template <int H>
    IFR_DEV void store(uint32_t, uint32_t p, _Float16 *tile, uint32_t r, uint32_t x) const {
#pragma unroll
        for (uint32_t i = 2 * H; i < 2 * H + 2; i++) *(u32x4_a16 *)(tile + pg_swz(r, (4 * p + i) ^ x)) = v[i];
    }
};
template <>
struct PgRun<F32> {
    u32x4_a16 v[8];
    IFR_DEV void load(const uint8_t *wrow, uint32_t k0, uint32_t p) {
        const u32x4_a16 *b = (const u32x4_a16 *)(wrow + 4 * (size_t)(k0 + 32 * p));
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = b[i];
    }
    IFR_DEV void pin() {
        asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
        asm volatile("" : "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
    }
    template <int H>
    IFR_DEV void store(uint32_t, uint32_t p, _Float16 *tile, uint32_t r, uint32_t x) const {
        uint32_t u[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const u32x4_a16 a = v[4 * H + (i >> 1)];
            u[i] = pack_f16x2(__uint_as_float(a[2 * (i & 1)]), __uint_as_float(a[2 * (i & 1) + 1]));
        }
        pg_put16(u, tile, r, (4 * p + 2 * H) ^ x);
    }
};
// The 32-element formats: block k0 / 32 + p.
template <>
struct PgRun<Q8_0> {
    u32x4_a2 q0, q1;
    uint32_t dd;
    IFR_DEV void load(const uint8_t *wrow, uint32_t k0, uint32_t p) {
        const uint8_t *b = wrow + (size_t)(k0 / 32 + p) * 34;
        dd = *(const uint16_t *)b;
        q0 = *(const u32x4_a2 *)(b + 2);
        q1 = *(const u32x4_a2 *)(b + 18);
    }
    IFR_DEV void pin() { asm volatile("" : "+v"(q0), "+v"(q1), "+v"(dd)); }
    template <int H>
    IFR_DEV void store(uint32_t, uint32_t p, _Float16 *tile, uint32_t r, uint32_t x) const {
        uint32_t u[8];
#pragma unroll
        for (int i = 0; i < 4; i++)
            pg_pk4((H ? q1[i] : q0[i]) ^ 0x80808080u, pg_half(dd), (_Float16)1152.0f, u[2 * i], u[2 * i + 1]);
        pg_put16(u, tile, r, (4 * p + 2 * H) ^ x);
    }
};
// Q4_0, Q4_1, Q5_0, Q5_1 (quantization.rs:66-177): element l < 16 the low
// nibble of qs byte l, l >= 16 the high nibble of byte l - 16; the fifth bit
// is bit l of qh.
template <int FMT, int BB, int QS>
struct PgRun32 {
    static constexpr bool AFF = FMT == Q4_1 || FMT == Q5_1, FIVE = FMT == Q5_0 || FMT == Q5_1;
    u32x4_a2 qv;
    uint32_t dm, qh; // d (and m above it), the fifth bits
    IFR_DEV void load(const uint8_t *wrow, uint32_t k0, uint32_t p) {
        const uint8_t *b = wrow + (size_t)(k0 / 32 + p) * BB;
        if constexpr (AFF) dm = *(const u32_a2 *)b;
        else dm = *(const uint16_t *)b;
        if constexpr (FIVE) qh = *(const u32_a2 *)(b + QS - 4);
        else qh = 0;
        qv = *(const u32x4_a2 *)(b + QS);
    }
    IFR_DEV void pin() {
        if constexpr (FIVE) asm volatile("" : "+v"(qv), "+v"(dm), "+v"(qh));
        else asm volatile("" : "+v"(qv), "+v"(dm));
    }
    template <int H>
    IFR_DEV void store(uint32_t, uint32_t p, _Float16 *tile, uint32_t r, uint32_t x) const {
        uint32_t u[8];
        const float s24 = f16_to_f32(dm & 0xFFFFu) * 0x1p24f, m = f16_to_f32(dm >> 16);
        const _Float16 z = (_Float16)(FIVE ? 1040.0f : 1032.0f);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t c = (H ? qv[i] >> 4 : qv[i]) & 0x0F0F0F0Fu;
            if constexpr (FIVE) c |= spread4_b4((qh >> (16 * H + 4 * i)) & 15u);
            if constexpr (AFF) pg_mix4(c, s24, m, u[2 * i], u[2 * i + 1]);
            else pg_pk4(c, pg_half(dm), z, u[2 * i], u[2 * i + 1]);
        }
        pg_put16(u, tile, r, (4 * p + 2 * H) ^ x);
    }
};
template <>
struct PgRun<Q4_0> : PgRun32<Q4_0, 18, 2> {};
template <>
struct PgRun<Q4_1> : PgRun32<Q4_1, 20, 4> {};
template <>
struct PgRun<Q5_0> : PgRun32<Q5_0, 22, 6> {};
template <>
struct PgRun<Q5_1> : PgRun32<Q5_1, 24, 8> {};

} // namespace ifr
