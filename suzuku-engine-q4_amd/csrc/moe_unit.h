// Register-held 64-value units of the decode / verify-window weight rows.
//
// A unit is two adjacent 32-value groups of a row (a quarter of a 256-value
// superblock, two Q8_0 / IQ4_NL blocks, one Q2_0 block).  A lane loads its
// unit's fields straight from global memory into registers and decodes it
// there: LDS holds only the codebook tables, and no weight byte passes
// through it.  Against copying rows to LDS and reading their fields back that
// is 12 of 28 LDS operations per IQ3_S unit less, no ring, no producer waves
// and no hand-off between waves.
//
// Superblocks start on 2-byte boundaries, and a wave's loads at such
// addresses cost the L1 one access per lane and dword crossed (measured per
// wave instruction over consecutive units: dwordx4 at 2-byte offsets 56-72
// accesses, at 4-byte offsets 22-28; dword 56-62 against 14).  So every field
// is loaded as the whole dwords around it and shifted into place by the
// lane's byte shift: 110 instead of 266 accesses per IQ3_S wave unit, adding
// those counts up (a 4-token gate/up launch as a whole, its activations, tables,
// stores and last refills included, has 163 per wave unit).
//
// Unit<TY>:
//   Offs          the dword offsets of the lane's fields from a uniform base
//                 (row starts are whole dwords) and their shifts
//   offs(row, u)  ... of unit u of the row at byte offset `row`
//   step(n)       bytes between unit u and unit u + n, where the two have the
//                 same shifts: n % 4 == 0 for the superblock formats, whose
//                 fields of a quarter are apart, and kEven an even number of
//                 superblocks (blocks)
//   Raw, load     the fields of one unit
//   kRawW         the decoded quads are the loaded registers themselves (the
//                 registers are free only after the dots)
//   kOneD         both groups have the same scale
//   decode        16 signed int8 quads (natural order), the multipliers of
//                 quads 0-3, 4-7, 8-11, 12-15, and the two groups' scales:
//                 group g's exact sum is m[2g] * dot(quads 8g..8g+3) +
//                 m[2g+1] * dot(quads 8g+4..8g+7), its value d[g] * d_x * sum
#pragma once
#include "formats.h"

namespace q4mi {

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3_t __attribute__((ext_vector_type(3)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// Loads of whole dwords at base (uniform) + a 32-bit lane offset + at.  The
// offset is made opaque where it is used, so that the load takes the scalar
// base and the 32-bit offset as they are (a loop-invariant offset is
// otherwise widened ahead of the loop: a second register per offset and a
// 64-bit add per load).  ok (uniform) false: every lane reads the dwords at
// base, a load that costs next to nothing and keeps the count of loads.
typedef const __attribute__((address_space(1))) uint8_t *GPtr;
template <class T>
__device__ inline T ld4_at(GPtr base, uint32_t off, bool ok, uint32_t at = 0) {
    typedef T U __attribute__((aligned(4)));
    off = ok ? off : 0u;
    asm("" : "+v"(off));
    return *(const __attribute__((address_space(1))) U *)(base + off + at);
}

// The dwords around a field: 16 bytes at byte shift s (0 or 2) take five.
struct Win5 { u32x4_t a; uint32_t b; };
__device__ inline void ld_win5(Win5 &w, GPtr b, uint32_t off, bool ok) {
    w.a = ld4_at<u32x4_t>(b, off, ok);
    w.b = ld4_at<uint32_t>(b, off, ok, 16u);
}
__device__ inline u32x4_t win_at(const Win5 &w, uint32_t s) {
    return u32x4_t{__builtin_amdgcn_alignbyte(w.a.y, w.a.x, s), __builtin_amdgcn_alignbyte(w.a.z, w.a.y, s),
                   __builtin_amdgcn_alignbyte(w.a.w, w.a.z, s), __builtin_amdgcn_alignbyte(w.b, w.a.w, s)};
}
__device__ inline u32x2_t win_at(const u32x3_t &w, uint32_t s) {
    return u32x2_t{__builtin_amdgcn_alignbyte(w.y, w.x, s), __builtin_amdgcn_alignbyte(w.z, w.y, s)};
}

// LDS by offset.  The kernels that use these decoders hold their dynamic LDS
// at offset 0 (no static LDS; checked at the first launch), so a table
// lookup's address needs no base added to it.
typedef uint32_t LPtr;
template <class T>
__device__ inline T lds_at(LPtr tab, uint32_t off) {
    typedef const __attribute__((address_space(3))) T *P;
    return *(P)(uintptr_t)(tab + off);
}

struct UnitW {
    int32_t w[16];
    int m[4];
    float d[2];
};

template <uint32_t TY>
struct Unit;

// ------------------------------------------------------------------- IQ3_S
// LDS: the signed quads of every (sign nibble, qh bit, qs byte), 8192 dwords.
// Byte address of an entry: low byte qs & 0xfc, high byte sign nibble << 3 |
// qh bit << 2 | qs & 3, so that the addresses of four quads take two masks
// and one v_perm_b32 each.
template <>
struct Unit<Q4MI_T_IQ3_S> {
    static constexpr uint32_t kTabBytes = 32768;
    static constexpr bool kTwo = false;
    static constexpr bool kOneD = true;
    static constexpr bool kRawW = false;
    struct Offs { uint32_t qs, sg, qh, sc, d, s, hs, ss; };
    struct Raw { Win5 qs; u32x3_t sg; uint32_t qh, sc, d; };
    __device__ static inline Offs offs(uint32_t row, uint32_t u) {
        const uint32_t b = row + (u >> 2) * IQ3S_BYTES, k = u & 3u;
        const uint32_t qs = b + 2u + 16u * k, sg = b + 74u + 8u * k, qh = b + 66u + 2u * k,
                       sc = b + 106u + k;
        // (the last superblock of a row is an odd one, so no window passes
        // the row's end)
        return Offs{qs & ~3u, sg & ~3u, qh & ~3u, sc & ~3u, b & ~3u, qs & 3u, 8u * (qh & 3u), 8u * (sc & 3u)};
    }
    static constexpr uint32_t step(uint32_t n) { return n / 4 * IQ3S_BYTES; }
    static constexpr bool kEven = true;    // step() needs an even superblock count
    __device__ static inline void load(Raw &r, GPtr b, const Offs &o, bool ok) {
        ld_win5(r.qs, b, o.qs, ok);
        r.sg = ld4_at<u32x3_t>(b, o.sg, ok);
        r.qh = ld4_at<uint32_t>(b, o.qh, ok);
        r.sc = ld4_at<uint32_t>(b, o.sc, ok);
        r.d = ld4_at<uint32_t>(b, o.d, ok);
    }
    // The last 512 threads of the block (n >= 512) build one codebook entry
    // each (the first ones have the activations to quantize); a wave's
    // entries are four apart, so its stores fall into distinct banks.
    __device__ static inline uint32_t entry(uint32_t t) {
        return (t & 0x100u) | ((t & 63u) << 2) | ((t >> 6) & 3u);
    }
    // code: this thread's codebook entry, loaded early by the caller
    __device__ static inline uint32_t code(uint32_t tid, uint32_t n) {
        return tid >= n - 512u ? q4mi_iq3s_code_dev[entry(tid - (n - 512u))] : 0u;
    }
    __device__ static inline void init(void *tab, uint32_t c, uint32_t tid, uint32_t n) {
        uint8_t *t = (uint8_t *)tab;
        if (tid >= n - 512u) {
            const uint32_t i = entry(tid - (n - 512u));
            uint32_t g = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) g |= (2u * ((c >> (3 * j)) & 7u) + 1u) << (8 * j);
            uint8_t *e = t + ((i & 0xfcu) | ((i & 3u) << 8) | ((i >> 8) << 10));
#pragma unroll
            for (uint32_t s4 = 0; s4 < 16; s4++)
                *(uint32_t *)(e + (s4 << 11)) = (uint32_t)q4mi_sign4(g, q4mi_expand4(s4));
        }
    }
    // qa, qb: the qh bits of quads 0-3 and 4-7
    __device__ static inline void group(LPtr tab, uint32_t q0, uint32_t q1, uint32_t qa, uint32_t qb,
                                        uint32_t sg, int32_t *w) {
        // byte k of hlo / hhi: sign nibble << 3 | qh bit << 2 of quad k / k+4
        const uint32_t ne = (sg << 3) & 0x78787878u, no = (sg >> 1) & 0x78787878u;
        const uint32_t hlo = __builtin_amdgcn_perm(no, ne, 0x05010400u) |
                             (__umul24(qa, 0x00810204u) & 0x04040404u);
        const uint32_t hhi = __builtin_amdgcn_perm(no, ne, 0x07030602u) |
                             (__umul24(qb, 0x00810204u) & 0x04040404u);
        const uint32_t h0 = hlo | (q0 & 0x03030303u), h1 = hhi | (q1 & 0x03030303u);
        const uint32_t l0 = q0 & 0xfcfcfcfcu, l1 = q1 & 0xfcfcfcfcu;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t sel = 0x0C0C0000u | ((4u + (k & 3)) << 8) | (uint32_t)(k & 3);
            const uint32_t at = __builtin_amdgcn_perm(k < 4 ? h0 : h1, k < 4 ? l0 : l1, sel);
            w[k] = lds_at<int32_t>(tab, at);
        }
    }
    __device__ static inline void decode(LPtr tab, const Raw &r, const Offs &f, UnitW &o) {
        // qs and sg sit 2 bytes into their windows in an even superblock, d in
        // an odd one
        o.d[0] = o.d[1] = q4mi_h2f(r.d >> (16u - 8u * f.s));
        const uint32_t sc = r.sc >> f.ss, qh = r.qh >> f.hs;
        o.m[0] = o.m[1] = 2 * (int)(sc & 15u) + 1;
        o.m[2] = o.m[3] = 2 * (int)((sc >> 4) & 15u) + 1;
        const u32x4_t qs = win_at(r.qs, f.s);
        const u32x2_t sg = win_at(r.sg, f.s);
        group(tab, qs.x, qs.y, qh & 15u, (qh >> 4) & 15u, sg.x, o.w);
        group(tab, qs.z, qs.w, (qh >> 8) & 15u, (qh >> 12) & 15u, sg.y, o.w + 8);
    }
};

// -------------------------------------------------------------------- Q8_0
template <>
struct Unit<Q4MI_T_Q8_0> {
    static constexpr uint32_t kTabBytes = 0;
    static constexpr bool kTwo = false;
    static constexpr bool kOneD = false;
    static constexpr bool kRawW = true;
    struct Offs { uint32_t b; };
    struct Raw { u32x4_t q[4]; uint32_t e; };   // 68 bytes: d | qs[32] | d | qs[32]
    __device__ static inline Offs offs(uint32_t row, uint32_t u) { return Offs{row + 68u * u}; }
    static constexpr uint32_t step(uint32_t n) { return 68u * n; }
    static constexpr bool kEven = false;
    __device__ static inline void load(Raw &r, GPtr b, const Offs &o, bool ok) {
#pragma unroll
        for (int k = 0; k < 4; k++) r.q[k] = ld4_at<u32x4_t>(b, o.b, ok, 16u * k);
        r.e = ld4_at<uint32_t>(b, o.b, ok, 64u);
    }
    __device__ static inline uint32_t code(uint32_t, uint32_t) { return 0; }
    __device__ static inline void init(void *, uint32_t, uint32_t, uint32_t) {}
    __device__ static inline void decode(LPtr, const Raw &r, const Offs &f, UnitW &o) {
        const uint32_t v[17] = {r.q[0].x, r.q[0].y, r.q[0].z, r.q[0].w, r.q[1].x, r.q[1].y,
                                r.q[1].z, r.q[1].w, r.q[2].x, r.q[2].y, r.q[2].z, r.q[2].w,
                                r.q[3].x, r.q[3].y, r.q[3].z, r.q[3].w, r.e};
        o.d[0] = q4mi_h2f(v[0] & 0xffffu);
        o.d[1] = q4mi_h2f(v[8] >> 16);
        o.m[0] = o.m[1] = o.m[2] = o.m[3] = 1;
#pragma unroll
        for (int k = 0; k < 8; k++) {   // block 0: 2 bytes into dword 0; block 1: 4 into dword 8
            o.w[k] = (int32_t)__builtin_amdgcn_alignbyte(v[k + 1], v[k], 2);
            o.w[8 + k] = (int32_t)v[9 + k];
        }
    }
};

// ------------------------------------------------------------------ IQ4_NL
template <>
struct Unit<Q4MI_T_IQ4_NL> {
    static constexpr uint32_t kTabBytes = 0;
    static constexpr bool kTwo = false;
    static constexpr bool kOneD = false;
    static constexpr bool kRawW = false;
    struct Offs { uint32_t b; };
    struct Raw { u32x4_t q[2]; uint32_t e; };   // 36 bytes: d | qs[16] | d | qs[16]
    __device__ static inline Offs offs(uint32_t row, uint32_t u) { return Offs{row + 36u * u}; }
    static constexpr uint32_t step(uint32_t n) { return 36u * n; }
    static constexpr bool kEven = false;
    __device__ static inline void load(Raw &r, GPtr b, const Offs &o, bool ok) {
        r.q[0] = ld4_at<u32x4_t>(b, o.b, ok);
        r.q[1] = ld4_at<u32x4_t>(b, o.b, ok, 16u);
        r.e = ld4_at<uint32_t>(b, o.b, ok, 32u);
    }
    __device__ static inline uint32_t code(uint32_t, uint32_t) { return 0; }
    __device__ static inline void init(void *, uint32_t, uint32_t, uint32_t) {}
    __device__ static inline void decode(LPtr, const Raw &r, const Offs &f, UnitW &o) {
        const uint32_t v[9] = {r.q[0].x, r.q[0].y, r.q[0].z, r.q[0].w, r.q[1].x,
                               r.q[1].y, r.q[1].z, r.q[1].w, r.e};
        o.d[0] = q4mi_h2f(v[0] & 0xffffu);
        o.d[1] = q4mi_h2f(v[4] >> 16);
        o.m[0] = o.m[1] = o.m[2] = o.m[3] = 1;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t a = __builtin_amdgcn_alignbyte(v[k + 1], v[k], 2), b = v[5 + k];
            o.w[k] = iq4nl_map(a & 0x0F0F0F0Fu);
            o.w[4 + k] = iq4nl_map((a >> 4) & 0x0F0F0F0Fu);
            o.w[8 + k] = iq4nl_map(b & 0x0F0F0F0Fu);
            o.w[12 + k] = iq4nl_map((b >> 4) & 0x0F0F0F0Fu);
        }
    }
};

// -------------------------------------------------------------------- Q2_0
template <>
struct Unit<Q4MI_T_Q2_0> {
    static constexpr uint32_t kTabBytes = 0;
    static constexpr bool kTwo = false;
    static constexpr bool kOneD = true;
    static constexpr bool kRawW = false;
    struct Offs { uint32_t b, s; };
    struct Raw { Win5 w; };                     // 18 bytes: d | qs[16]
    __device__ static inline Offs offs(uint32_t row, uint32_t u) {
        const uint32_t b = row + 18u * u;       // (a row's last unit is an odd one)
        return Offs{b & ~3u, b & 3u};
    }
    static constexpr uint32_t step(uint32_t n) { return 18u * n; }
    static constexpr bool kEven = true;
    __device__ static inline void load(Raw &r, GPtr b, const Offs &o, bool ok) { ld_win5(r.w, b, o.b, ok); }
    __device__ static inline uint32_t code(uint32_t, uint32_t) { return 0; }
    __device__ static inline void init(void *, uint32_t, uint32_t, uint32_t) {}
    __device__ static inline void decode(LPtr, const Raw &r, const Offs &f, UnitW &o) {
        // d at byte s of the window (0 or 2), qs at s + 2
        o.d[0] = o.d[1] = q4mi_h2f(r.w.a.x >> (8u * f.s));
        o.m[0] = o.m[1] = o.m[2] = o.m[3] = 1;
        const bool odd = f.s != 0;
        const u32x4_t q = {odd ? r.w.a.y : __builtin_amdgcn_alignbyte(r.w.a.y, r.w.a.x, 2),
                           odd ? r.w.a.z : __builtin_amdgcn_alignbyte(r.w.a.z, r.w.a.y, 2),
                           odd ? r.w.a.w : __builtin_amdgcn_alignbyte(r.w.a.w, r.w.a.z, 2),
                           odd ? r.w.b : __builtin_amdgcn_alignbyte(r.w.b, r.w.a.w, 2)};
#pragma unroll
        for (int k = 0; k < 16; k++) o.w[k] = q20_quad((q[k >> 2] >> (8 * (k & 3))) & 0xffu);
    }
};

// ------------------------------------------------------------------- IQ2_S
template <>
struct Unit<Q4MI_T_IQ2_S> {
    static constexpr uint32_t kTabBytes = sizeof(Iq2sLds);
    static constexpr bool kTwo = true;
    static constexpr bool kOneD = true;
    static constexpr bool kRawW = false;
    struct Offs { uint32_t qs, sg, qh, sc, d, s, hs, ss; };
    struct Raw { u32x3_t qs, sg; uint32_t qh, sc, d; };
    __device__ static inline Offs offs(uint32_t row, uint32_t u) {
        const uint32_t b = row + (u >> 2) * 82u, k = u & 3u;
        const uint32_t qs = b + 2u + 8u * k, sg = b + 34u + 8u * k, qh = b + 66u + 2u * k,
                       sc = b + 74u + 2u * k;
        return Offs{qs & ~3u, sg & ~3u, qh & ~3u, sc & ~3u, b & ~3u, qs & 3u, 8u * (qh & 3u), 8u * (sc & 3u)};
    }
    static constexpr uint32_t step(uint32_t n) { return n / 4 * 82u; }
    static constexpr bool kEven = true;
    __device__ static inline void load(Raw &r, GPtr b, const Offs &o, bool ok) {
        r.qs = ld4_at<u32x3_t>(b, o.qs, ok);
        r.sg = ld4_at<u32x3_t>(b, o.sg, ok);
        r.qh = ld4_at<uint32_t>(b, o.qh, ok);
        r.sc = ld4_at<uint32_t>(b, o.sc, ok);
        r.d = ld4_at<uint32_t>(b, o.d, ok);
    }
    __device__ static inline uint32_t code(uint32_t, uint32_t) { return 0; }
    __device__ static inline void init(void *tab, uint32_t, uint32_t tid, uint32_t n) {
        FmtIQ2S::init(tab, tid, n);
    }
    __device__ static inline void decode(LPtr tab, const Raw &r, const Offs &f, UnitW &o) {
        o.d[0] = o.d[1] = q4mi_h2f(r.d >> (16u - 8u * f.s)) * 0.125f;
        const uint32_t sc = r.sc >> f.ss, qh2 = r.qh >> f.hs;
#pragma unroll
        for (int i = 0; i < 4; i++) o.m[i] = 2 * (int)((sc >> (4 * i)) & 15u) + 1;
        const u32x2_t qs2 = win_at(r.qs, f.s), sg2 = win_at(r.sg, f.s);
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const uint32_t qs = qs2[g], sg = sg2[g], qh = (qh2 >> (8 * g)) & 0xffu;
#pragma unroll
            for (int l = 0; l < 4; l++) {
                const uint32_t idx = ((qs >> (8 * l)) & 0xffu) | ((qh << (8 - 2 * l)) & 0x300u);
                const u32x2_t e = lds_at<u32x2_t>(tab, 8u * idx);
                const u32x2_t m = lds_at<u32x2_t>(tab, 8192u + 8u * ((sg >> (8 * l)) & 0xffu));
                o.w[8 * g + 2 * l] = q4mi_sign4(e.x, m.x);
                o.w[8 * g + 2 * l + 1] = q4mi_sign4(e.y, m.y);
            }
        }
    }
};

// ----------------------------------------------------------------- IQ2_XXS
template <>
struct Unit<Q4MI_T_IQ2_XXS> {
    static constexpr uint32_t kTabBytes = sizeof(Iq2xLds<256>);
    static constexpr bool kTwo = false;
    static constexpr bool kOneD = true;
    static constexpr bool kRawW = false;
    struct Offs { uint32_t qs, d, s; };
    struct Raw { Win5 q; uint32_t d; };         // grid bytes | aux, twice
    __device__ static inline Offs offs(uint32_t row, uint32_t u) {
        const uint32_t b = row + (u >> 2) * 66u, qs = b + 2u + 16u * (u & 3u);
        return Offs{qs & ~3u, b & ~3u, qs & 3u};
    }
    static constexpr uint32_t step(uint32_t n) { return n / 4 * 66u; }
    static constexpr bool kEven = true;
    __device__ static inline void load(Raw &r, GPtr b, const Offs &o, bool ok) {
        r.q.a = ld4_at<u32x4_t>(b, o.qs, ok);
        // (the fifth dword is only needed, and only inside the row, at shift 2)
        r.q.b = ld4_at<uint32_t>(b, o.qs + 8u * o.s, ok);
        r.d = ld4_at<uint32_t>(b, o.d, ok);
    }
    __device__ static inline uint32_t code(uint32_t, uint32_t) { return 0; }
    __device__ static inline void init(void *tab, uint32_t, uint32_t tid, uint32_t n) {
        FmtIQ2XXS::init(tab, tid, n);
    }
    __device__ static inline void decode(LPtr tab, const Raw &r, const Offs &f, UnitW &o) {
        o.d[0] = o.d[1] = q4mi_h2f(r.d >> (16u - 8u * f.s)) * 0.125f;
        const u32x4_t q = win_at(r.q, f.s);
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const uint32_t gi = q[2 * g], aux = q[2 * g + 1];
            o.m[2 * g] = o.m[2 * g + 1] = 2 * (int)(aux >> 28) + 1;
#pragma unroll
            for (int l = 0; l < 4; l++) {
                const u32x2_t e = lds_at<u32x2_t>(tab, 8u * ((gi >> (8 * l)) & 0xffu));
                const u32x2_t m = lds_at<u32x2_t>(tab, 2048u + 8u * ((aux >> (7 * l)) & 127u));
                o.w[8 * g + 2 * l] = q4mi_sign4(e.x, m.x);
                o.w[8 * g + 2 * l + 1] = q4mi_sign4(e.y, m.y);
            }
        }
    }
};

// ------------------------------------------------------------------ IQ2_XS
template <>
struct Unit<Q4MI_T_IQ2_XS> {
    static constexpr uint32_t kTabBytes = sizeof(Iq2xLds<512>);
    static constexpr bool kTwo = true;
    static constexpr bool kOneD = true;
    static constexpr bool kRawW = false;
    struct Offs { uint32_t qs, sc, d, s, ss; };
    struct Raw { Win5 q; uint32_t sc, d; };     // 16-bit grid index | sign index << 9
    __device__ static inline Offs offs(uint32_t row, uint32_t u) {
        const uint32_t b = row + (u >> 2) * 74u, k = u & 3u;
        const uint32_t qs = b + 2u + 16u * k, sc = b + 66u + 2u * k;
        return Offs{qs & ~3u, sc & ~3u, b & ~3u, qs & 3u, 8u * (sc & 3u)};
    }
    static constexpr uint32_t step(uint32_t n) { return n / 4 * 74u; }
    static constexpr bool kEven = true;
    __device__ static inline void load(Raw &r, GPtr b, const Offs &o, bool ok) {
        ld_win5(r.q, b, o.qs, ok);
        r.sc = ld4_at<uint32_t>(b, o.sc, ok);
        r.d = ld4_at<uint32_t>(b, o.d, ok);
    }
    __device__ static inline uint32_t code(uint32_t, uint32_t) { return 0; }
    __device__ static inline void init(void *tab, uint32_t, uint32_t tid, uint32_t n) {
        FmtIQ2XS::init(tab, tid, n);
    }
    __device__ static inline void decode(LPtr tab, const Raw &r, const Offs &f, UnitW &o) {
        o.d[0] = o.d[1] = q4mi_h2f(r.d >> (16u - 8u * f.s)) * 0.125f;
        const uint32_t sc = r.sc >> f.ss;
#pragma unroll
        for (int i = 0; i < 4; i++) o.m[i] = 2 * (int)((sc >> (4 * i)) & 15u) + 1;
        const u32x4_t q = win_at(r.q, f.s);
#pragma unroll
        for (int l = 0; l < 8; l++) {
            const uint32_t v = (q[l >> 1] >> (16 * (l & 1))) & 0xffffu;
            const u32x2_t e = lds_at<u32x2_t>(tab, 8u * (v & 511u));
            const u32x2_t m = lds_at<u32x2_t>(tab, 4096u + 8u * (v >> 9));
            o.w[2 * l] = q4mi_sign4(e.x, m.x);
            o.w[2 * l + 1] = q4mi_sign4(e.y, m.y);
        }
    }
};

// ----------------------------------------------------------------- IQ3_XXS
template <>
struct Unit<Q4MI_T_IQ3_XXS> {
    static constexpr uint32_t kTabBytes = sizeof(Iq3xxsLds);
    static constexpr bool kTwo = false;
    static constexpr bool kOneD = true;
    static constexpr bool kRawW = false;
    struct Offs { uint32_t qs, ax, d, s; };
    struct Raw { Win5 q; u32x3_t ax; uint32_t d; };
    __device__ static inline Offs offs(uint32_t row, uint32_t u) {
        const uint32_t b = row + (u >> 2) * 98u, k = u & 3u;
        const uint32_t qs = b + 2u + 16u * k, ax = b + 66u + 8u * k;
        // (at shift 0 the third dword of ax repeats the second: the window
        // would pass the row's end)
        return Offs{qs & ~3u, ax & ~3u, b & ~3u, qs & 3u};
    }
    static constexpr uint32_t step(uint32_t n) { return n / 4 * 98u; }
    static constexpr bool kEven = true;
    __device__ static inline void load(Raw &r, GPtr b, const Offs &o, bool ok) {
        ld_win5(r.q, b, o.qs, ok);
        const u32x2_t lo = ld4_at<u32x2_t>(b, o.ax, ok);
        r.ax = u32x3_t{lo.x, lo.y, ld4_at<uint32_t>(b, o.ax + 4u + 2u * o.s, ok)};
        r.d = ld4_at<uint32_t>(b, o.d, ok);
    }
    __device__ static inline uint32_t code(uint32_t, uint32_t) { return 0; }
    __device__ static inline void init(void *tab, uint32_t, uint32_t tid, uint32_t n) {
        FmtIQ3XXS::init(tab, tid, n);
    }
    __device__ static inline void decode(LPtr tab, const Raw &r, const Offs &f, UnitW &o) {
        o.d[0] = o.d[1] = q4mi_h2f(r.d >> (16u - 8u * f.s)) * 0.25f;
        const u32x4_t q = win_at(r.q, f.s);
        const u32x2_t ax = win_at(r.ax, f.s);
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const uint32_t aux = ax[g];
            o.m[2 * g] = o.m[2 * g + 1] = 2 * (int)(aux >> 28) + 1;
#pragma unroll
            for (int l = 0; l < 4; l++) {
                const u32x2_t m = lds_at<u32x2_t>(tab, 1024u + 8u * ((aux >> (7 * l)) & 127u));
                const uint32_t q2 = q[2 * g + (l >> 1)] >> (16 * (l & 1));
                o.w[8 * g + 2 * l] = q4mi_sign4(lds_at<uint32_t>(tab, 4u * (q2 & 0xffu)), m.x);
                o.w[8 * g + 2 * l + 1] = q4mi_sign4(lds_at<uint32_t>(tab, 4u * ((q2 >> 8) & 0xffu)), m.y);
            }
        }
    }
};

// ------------------------------------------------------------------ IQ4_XS
template <>
struct Unit<Q4MI_T_IQ4_XS> {
    static constexpr uint32_t kTabBytes = 0;
    static constexpr bool kTwo = false;
    static constexpr bool kOneD = true;
    static constexpr bool kRawW = false;
    struct Offs { uint32_t qs, b, k; };
    struct Raw { u32x4_t q[2]; u32x2_t h; };    // h: d | scales_h, scales_l
    __device__ static inline Offs offs(uint32_t row, uint32_t u) {
        const uint32_t b = row + (u >> 2) * 136u, k = u & 3u;
        return Offs{b + 8u + 32u * k, b, k};
    }
    static constexpr uint32_t step(uint32_t n) { return n / 4 * 136u; }
    static constexpr bool kEven = false;
    __device__ static inline void load(Raw &r, GPtr b, const Offs &o, bool ok) {
        r.q[0] = ld4_at<u32x4_t>(b, o.qs, ok);
        r.q[1] = ld4_at<u32x4_t>(b, o.qs, ok, 16u);
        r.h = ld4_at<u32x2_t>(b, o.b, ok);
    }
    __device__ static inline uint32_t code(uint32_t, uint32_t) { return 0; }
    __device__ static inline void init(void *, uint32_t, uint32_t, uint32_t) {}
    __device__ static inline void decode(LPtr, const Raw &r, const Offs &f, UnitW &o) {
        o.d[0] = o.d[1] = q4mi_h2f(r.h.x & 0xffffu);
        const uint32_t sh = (r.h.x >> (16u + 4u * f.k)) & 15u, sl = r.h.y >> (8u * f.k);
        o.m[0] = o.m[1] = (int)((sl & 15u) | ((sh & 3u) << 4)) - 32;
        o.m[2] = o.m[3] = (int)(((sl >> 4) & 15u) | ((sh >> 2) << 4)) - 32;
#pragma unroll
        for (int g = 0; g < 2; g++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                o.w[8 * g + j] = iq4nl_map(r.q[g][j] & 0x0F0F0F0Fu);
                o.w[8 * g + 4 + j] = iq4nl_map((r.q[g][j] >> 4) & 0x0F0F0F0Fu);
            }
    }
};

// -------------------------------------------------------------------- Q6_K
// A unit is groups 4h + b and 4h + b + 2 of a superblock (half h, b = 0, 1):
// the low and the high nibbles of the same 32 ql bytes, with two bits each of
// the same 32 qh bytes.
template <>
struct Unit<Q4MI_T_Q6_K> {
    static constexpr uint32_t kTabBytes = 0;
    static constexpr bool kTwo = true;
    static constexpr bool kOneD = true;
    static constexpr bool kRawW = false;
    struct Offs { uint32_t ql, qh, sc, d, s, ss, b; };
    struct Raw { u32x4_t l[2], h[2]; uint32_t l8, h8; u32x2_t sc; uint32_t d; };
    __device__ static inline Offs offs(uint32_t row, uint32_t u) {
        const uint32_t p = row + (u >> 2) * 210u, h = (u >> 1) & 1u, b = u & 1u;
        const uint32_t ql = p + 64u * h + 32u * b, qh = p + 128u + 32u * h,
                       sc = p + 192u + 8u * h + 2u * b;
        // (at shift 0 the ninth dwords are not needed; an odd superblock, the
        // row's last among them, sits 2 bytes into its dwords)
        return Offs{ql & ~3u, qh & ~3u, sc & ~3u, (p + 208u) & ~3u, p & 3u, 8u * (sc & 3u), b};
    }
    static constexpr uint32_t step(uint32_t n) { return n / 4 * 210u; }
    static constexpr bool kEven = true;
    __device__ static inline void load(Raw &r, GPtr b, const Offs &o, bool ok) {
        r.l[0] = ld4_at<u32x4_t>(b, o.ql, ok);
        r.l[1] = ld4_at<u32x4_t>(b, o.ql, ok, 16u);
        r.l8 = ld4_at<uint32_t>(b, o.ql, ok, 32u);
        r.h[0] = ld4_at<u32x4_t>(b, o.qh, ok);
        r.h[1] = ld4_at<u32x4_t>(b, o.qh, ok, 16u);
        r.h8 = ld4_at<uint32_t>(b, o.qh, ok, 32u);
        r.sc = ld4_at<u32x2_t>(b, o.sc, ok);
        r.d = ld4_at<uint32_t>(b, o.d, ok);
    }
    __device__ static inline uint32_t code(uint32_t, uint32_t) { return 0; }
    __device__ static inline void init(void *, uint32_t, uint32_t, uint32_t) {}
    __device__ static inline void decode(LPtr, const Raw &r, const Offs &f, UnitW &o) {
        o.d[0] = o.d[1] = q4mi_h2f(r.d >> (8u * f.s));
        // scales sc[8h + 2b], +1 (values 0-15, 16-31) and 4 later
        const uint32_t s0 = r.sc.x >> f.ss, s1 = r.sc.y >> f.ss;
        o.m[0] = (int)(int8_t)(s0 & 0xffu);
        o.m[1] = (int)(int8_t)((s0 >> 8) & 0xffu);
        o.m[2] = (int)(int8_t)(s1 & 0xffu);
        o.m[3] = (int)(int8_t)((s1 >> 8) & 0xffu);
        const uint32_t l[9] = {r.l[0].x, r.l[0].y, r.l[0].z, r.l[0].w, r.l[1].x, r.l[1].y, r.l[1].z, r.l[1].w, r.l8};
        const uint32_t h[9] = {r.h[0].x, r.h[0].y, r.h[0].z, r.h[0].w, r.h[1].x, r.h[1].y, r.h[1].z, r.h[1].w, r.h8};
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t ql = __builtin_amdgcn_alignbyte(l[k + 1], l[k], f.s);
            const uint32_t qh = __builtin_amdgcn_alignbyte(h[k + 1], h[k], f.s) >> (2u * f.b);
            o.w[k] = q6_sub32((ql & 0x0F0F0F0Fu) | ((qh & 0x03030303u) << 4));
            o.w[8 + k] = q6_sub32(((ql >> 4) & 0x0F0F0F0Fu) | (qh & 0x30303030u));
        }
    }
};

// Which unit and half holds group g of a row, and back.
template <uint32_t TY>
__device__ inline uint32_t group_unit(uint32_t g) {
    return TY == Q4MI_T_Q6_K ? (g >> 2) * 2u + (g & 1u) : g >> 1;
}
template <uint32_t TY>
__device__ inline uint32_t group_half(uint32_t g) {
    return TY == Q4MI_T_Q6_K ? (g >> 1) & 1u : g & 1u;
}
template <uint32_t TY>
__device__ inline uint32_t unit_group(uint32_t u, uint32_t half) {
    return TY == Q4MI_T_Q6_K ? (u >> 1) * 4u + (u & 1u) + 2u * half : 2u * u + half;
}

// q8 codes of a run of units in LDS: 16-byte chunk c (0..3) of unit u at
// (c * nu + u) * 16, so that lanes holding consecutive units read
// consecutive 16-byte words (a unit's 64 bytes side by side would put every
// second lane on the same banks); group scales at 2 unit + half.
template <uint32_t TY = 0>
__device__ inline uint32_t code_at(uint32_t oct, uint32_t nu) {   // oct = 8 values
    const uint32_t g = oct >> 2, c = 2u * group_half<TY>(g) + ((oct >> 1) & 1u);
    return (c * nu + group_unit<TY>(g)) * 16u + (oct & 1u) * 8u;
}

// The unit's value against one token: xq / xd = that token's codes (laid out
// as above over nu units) and scales.
struct UnitX {
    int32_t q[16];
    float2 d;
};
__device__ inline void load_unit_q(int32_t (&q)[16], const int8_t *xq, uint32_t nu, uint32_t u) {
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const int4 v = *(const int4 *)(xq + ((uint32_t)c * nu + u) * 16u);
        q[4 * c] = v.x;
        q[4 * c + 1] = v.y;
        q[4 * c + 2] = v.z;
        q[4 * c + 3] = v.w;
    }
}
__device__ inline void load_unit_x(UnitX &x, const int8_t *xq, const float *xd, uint32_t nu,
                                   uint32_t u) {
    load_unit_q(x.q, xq, nu, u);
    x.d = *(const float2 *)(xd + 2u * u);
}
// The two groups' exact integer sums.
template <uint32_t TY>
__device__ inline void unit_sums(const UnitW &o, const int32_t (&q)[16], int (&s)[2]) {
    // exact group sums (24-bit multiplies, full rate: |sums| < 2^20,
    // |multipliers| <= 2^7)
#pragma unroll
    for (int g = 0; g < 2; g++) {
        int a = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) a = q4mi_sdot4(o.w[8 * g + k], q[8 * g + k], a);
        if constexpr (Unit<TY>::kTwo) {
            int b = 0;
#pragma unroll
            for (int k = 4; k < 8; k++) b = q4mi_sdot4(o.w[8 * g + k], q[8 * g + k], b);
            s[g] = __mul24(a, o.m[2 * g]) + __mul24(b, o.m[2 * g + 1]);
        } else {
#pragma unroll
            for (int k = 4; k < 8; k++) a = q4mi_sdot4(o.w[8 * g + k], q[8 * g + k], a);
            s[g] = __mul24(a, o.m[2 * g]);
        }
    }
}
// ... and their values added to acc[0] and acc[1].
template <uint32_t TY>
__device__ inline void unit_dot2(const UnitW &o, const UnitX &x, float (&acc)[2], int (&s)[2]) {
    unit_sums<TY>(o, x.q, s);
    acc[0] = fmaf((float)s[0], o.d[0] * x.d.x, acc[0]);
    acc[1] = fmaf((float)s[1], o.d[1] * x.d.y, acc[1]);
}
template <uint32_t TY>
__device__ inline float unit_dot(const UnitW &o, const int8_t *xq, const float *xd, uint32_t nu,
                                 uint32_t u, float acc) {
    UnitX x;
    load_unit_x(x, xq, xd, nu, u);
    int s[2];
    unit_sums<TY>(o, x.q, s);
    acc = fmaf((float)s[0], o.d[0] * x.d.x, acc);
    return fmaf((float)s[1], o.d[1] * x.d.y, acc);
}
// ... in fp64 (xd: the scales as fp64): every product exact, the sum rounded
// far below fp32.  (fp64 multiply-adds run at fp32's rate here.)
template <uint32_t TY>
__device__ inline double unit_dot64(const UnitW &o, const int8_t *xq, const double *xd, uint32_t nu,
                                    uint32_t u, double acc) {
    int32_t q[16];
    load_unit_q(q, xq, nu, u);
    const double2 dx = *(const double2 *)(xd + 2u * u);
    int s[2];
    unit_sums<TY>(o, q, s);
    if constexpr (Unit<TY>::kOneD)
        return fma((double)o.d[0], fma((double)s[0], dx.x, (double)s[1] * dx.y), acc);
    acc = fma((double)s[0], (double)o.d[0] * dx.x, acc);
    return fma((double)s[1], (double)o.d[1] * dx.y, acc);
}

// Workgroup barrier without the compiler's fence: this wave's LDS operations
// are complete, its loads from global memory stay in flight.
__device__ inline void bar() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Keep a uniform pointer one scalar register pair: the compiler otherwise
// folds its terms into every lane address that is built on it.
__device__ inline GPtr uniform_ptr(const uint8_t *p) {
    uint64_t v = (uint64_t)p;
    asm("" : "+s"(v));
    return (GPtr)v;
}

// Between a unit's decode and the load that refills its registers: every
// field is consumed (the table lookups are issued, multipliers and scales
// formed) before the load, so the new values can take the same registers.
__device__ inline void unit_consumed(UnitW &w) {
    asm volatile("" : "+v"(w.m[0]), "+v"(w.m[1]), "+v"(w.m[2]), "+v"(w.m[3]), "+v"(w.d[0]),
                 "+v"(w.d[1]) :: "memory");
}

// q8 of oct i (values 8i..8i+7) of a row of 32-value groups, codes laid out by
// the row's nu units: the 4 lanes holding octs 4g..4g+3 quantize group g
// together (all 4 must be active).
struct Oct { float4 x, y; };
__device__ inline Oct ld_oct(const float *p, uint32_t i) {
    return Oct{((const float4 *)p)[2 * i], ((const float4 *)p)[2 * i + 1]};
}
template <uint32_t TY = 0, class D>
__device__ inline void quant_oct(const Oct &v, uint32_t i, uint32_t nu, int8_t *q, D *d) {
    float dd;
    *(uint2 *)(q + code_at<TY>(i, nu)) = q4mi_quant_team4(v.x, v.y, &dd);
    const uint32_t g = i >> 2;
    if ((i & 3u) == 0) d[2u * group_unit<TY>(g) + group_half<TY>(g)] = dd;
}

}  // namespace q4mi
