// Device helpers shared by the kernels of libsbvr_hip.so: vector types, fp16 conversions, loads of plane words and
// coefficient lines, and the decode of weights by table look-up.
#ifndef SBVR_DEVICE_H
#define SBVR_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef short v2s __attribute__((ext_vector_type(2)));
__device__ __forceinline__ v2h as_v2h(uint32_t u) { return __builtin_bit_cast(v2h, u); }

__device__ __forceinline__ float h2f(uint16_t h)
{
    return static_cast<float>(__builtin_bit_cast(_Float16, h));
}

__device__ __forceinline__ uint16_t f2h(float f)
{
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(f));
}

// fp16 add of two fp16 values: exact sum rounded once (what __hadd does).
__device__ __forceinline__ uint16_t hadd(uint16_t a, uint16_t b)
{
    return f2h(h2f(a) + h2f(b));
}

// fp16 of a * b + c rounded once (v_fma_mix), which is what a product and a sum converted to fp16 compile to in most
// places, but not in all: for results that have to be another kernel's bit for bit.
__device__ __forceinline__ _Float16 fma_half(float a, float b, float c)
{
    uint32_t r = 0;
    asm("v_fma_mixlo_f16 %0, %1, %2, %3" : "+v"(r) : "v"(a), "v"(b), "v"(c));
    return __builtin_bit_cast(_Float16, static_cast<uint16_t>(r));
}

template <typename IdxT>
__device__ __forceinline__ int load_idx(const void *p, size_t i)
{
    return static_cast<int>(static_cast<const IdxT *>(p)[i]);
}

template <int S>
struct Planes {
    uint32_t w[S];
};

typedef uint32_t v3raw __attribute__((ext_vector_type(3)));
typedef v3raw v3u __attribute__((aligned(4)));          // (as it lies in a row of 3 or 6 plane words)

// The S plane words of one (word of K, column) pair.  kStream: non-temporal loads, for kernels that
// read every plane word once per launch and are bound by that stream (measured on the decode kernel:
// 8.3 us instead of 8.8 us at the 4096 -> 14336 shape, 13.5 instead of 14.5 us at 4096 -> 28672; the
// 32-row, row-dequant and popcount kernels, bound by their arithmetic, gain nothing from it).
template <int S, bool kStream = false>
__device__ __forceinline__ Planes<S> load_planes(const uint32_t *p)
{
    auto ld4 = [](const uint32_t *q) __attribute__((always_inline)) -> v4u {
        return kStream ? __builtin_nontemporal_load(reinterpret_cast<const v4u *>(q)) : *reinterpret_cast<const v4u *>(q);
    };
    auto ld2 = [](const uint32_t *q) __attribute__((always_inline)) -> v2u {
        return kStream ? __builtin_nontemporal_load(reinterpret_cast<const v2u *>(q)) : *reinterpret_cast<const v2u *>(q);
    };
    Planes<S> r;
    if constexpr (S == 4) {
        const v4u v = ld4(p);
        r.w[0] = v.x; r.w[1] = v.y; r.w[2] = v.z; r.w[3] = v.w;
    } else if constexpr (S == 2) {
        const v2u v = ld2(p);
        r.w[0] = v.x; r.w[1] = v.y;
    } else if constexpr (S == 8) {
        const v4u v0 = ld4(p), v1 = ld4(p + 4);
        r.w[0] = v0.x; r.w[1] = v0.y; r.w[2] = v0.z; r.w[3] = v0.w;
        r.w[4] = v1.x; r.w[5] = v1.y; r.w[6] = v1.z; r.w[7] = v1.w;
    } else if constexpr (S == 3) {
        // (12 bytes in one request: a global load wants dword alignment only)
        const v3raw v = kStream ? __builtin_nontemporal_load(reinterpret_cast<const v3u *>(p)) : *reinterpret_cast<const v3u *>(p);
        r.w[0] = v.x; r.w[1] = v.y; r.w[2] = v.z;
    } else if constexpr (S == 6) {
        const v3raw v0 = kStream ? __builtin_nontemporal_load(reinterpret_cast<const v3u *>(p)) : *reinterpret_cast<const v3u *>(p);
        const v3raw v1 = kStream ? __builtin_nontemporal_load(reinterpret_cast<const v3u *>(p + 3)) : *reinterpret_cast<const v3u *>(p + 3);
        r.w[0] = v0.x; r.w[1] = v0.y; r.w[2] = v0.z; r.w[3] = v1.x; r.w[4] = v1.y; r.w[5] = v1.z;
    } else {
#pragma unroll
        for (int j = 0; j < S; ++j)
            r.w[j] = kStream ? __builtin_nontemporal_load(p + j) : p[j];
    }
    return r;
}

// The S fp16 coefficients of table line p as (S + 1) / 2 dwords, in as few loads as the line's alignment allows.
template <int S>
__device__ __forceinline__ void load_line_words(const uint16_t *p, uint32_t (&c)[(S + 1) / 2])
{
    constexpr int CW = (S + 1) / 2;
    if constexpr (S == 4) {
        const uint2 t = *reinterpret_cast<const uint2 *>(p);
        c[0] = t.x; c[1] = t.y;
    } else if constexpr (S == 8) {
        const uint4 t = *reinterpret_cast<const uint4 *>(p);
        c[0] = t.x; c[1] = t.y; c[2] = t.z; c[3] = t.w;
    } else if constexpr (S % 2 == 0) {
#pragma unroll
        for (int j = 0; j < CW; ++j)
            c[j] = reinterpret_cast<const uint32_t *>(p)[j];
    } else {
#pragma unroll
        for (int j = 0; j < CW; ++j)
            c[j] = static_cast<uint32_t>(p[2 * j]) | (2 * j + 1 < S ? static_cast<uint32_t>(p[2 * j + 1]) << 16 : 0u);
    }
}

// ---- decode by table look-up, shared by sbvr_gemm_rows32_lut_kernel and sbvr_gemm_lut_kernel (2, 3 or 4 planes)
template <int S>
struct LutTables {
    static constexpr int TW = S == 4 ? 4 : (S == 3 ? 2 : 1);       // dwords of a byte table
    uint32_t lo[TW], hi[TW];       // low and high bytes of the subset sums 0..3, 4..7, ...
};

// The 2^S subset sums of a coefficient line, entries (2i, 2i + 1) as packed pairs, then as byte tables.  Entry i is
// the sum of the coefficients whose bit is set in i, added up in fp32 and rounded to fp16 once: the reference's
// decode() takes a weight from bin_combs @ coeff (sbvr/core.py:345-366, 927-949), the exact sum rounded once.  The
// fp32 sums are exact, and the entries therefore decode()'s weights bit for bit, whenever the exponents of a line's
// coefficients lie within 11 of each other (every partial sum is then a multiple of the smallest coefficient's
// last place below 2^24 of them); a line that mixes coefficients 2^12 apart and more can differ from decode() in
// the last place of an entry that lands on a rounding tie.
template <int S>
__device__ __forceinline__ void lut_build_tables(const uint32_t (&c)[(S + 1) / 2], LutTables<S> &t)
{
    float cf[S];
#pragma unroll
    for (int q = 0; q < S; ++q)
        cf[q] = h2f(static_cast<uint16_t>(q & 1 ? c[q / 2] >> 16 : c[q / 2] & 0xffffu));
    float s[1 << S];
    s[0] = 0.f;
#pragma unroll
    for (int q = 0; q < S; ++q)
#pragma unroll
        for (int i = 0; i < (1 << q); ++i)
            s[(1 << q) + i] = i == 0 ? cf[q] : s[i] + cf[q];
    v2h e[1 << (S - 1)];
#pragma unroll
    for (int i = 0; i < (1 << (S - 1)); ++i) {
        e[i][0] = static_cast<_Float16>(s[2 * i]);         // (one v_cvt_pk_f16_f32 per pair, round to nearest even)
        e[i][1] = static_cast<_Float16>(s[2 * i + 1]);
    }
#pragma unroll
    for (int i = 0; i < LutTables<S>::TW; ++i) {
        const uint32_t e0 = __builtin_bit_cast(uint32_t, e[2 * i]), e1 = __builtin_bit_cast(uint32_t, e[2 * i + 1]);
        t.lo[i] = __builtin_amdgcn_perm(e1, e0, 0x06040200u);
        t.hi[i] = __builtin_amdgcn_perm(e1, e0, 0x07050301u);
    }
}

// bits of a where mask is set, of b elsewhere (written out: with a constant mask the compiler takes the expression apart
// into two ands and an or)
__device__ __forceinline__ uint32_t bit_select(uint32_t mask, uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "s"(mask), "v"(a), "v"(b));
    return r;
}

// Selector words of one word of K: nibble n of Q[p] holds, in its low min(S, 3) bits, the first planes' bits of element
// p + 4n (the other bits are anything), and top the fourth plane's word.  Two planes at a time: their bits of the even and of the
// odd elements side by side, then these pairs next to the third plane's, 13 operations with 3 and 4 planes, 6 with 2.
template <int S>
struct Nibbles {
    uint32_t Q[4], top;
};

template <int S>
__device__ __forceinline__ void lut_nibble_pairs(const uint32_t (&w)[S], uint32_t (&pair)[2])
{
    pair[0] = bit_select(0x55555555u, w[0], w[1] << 1);
    pair[1] = bit_select(0x55555555u, w[0] >> 1, w[1]);
}

template <int S>
__device__ __forceinline__ void lut_nibble_word(const uint32_t (&w)[S], const uint32_t (&pair)[2], Nibbles<S> &n, int p)
{
    const uint32_t two = p < 2 ? pair[p & 1] : pair[p & 1] >> 2;
    if constexpr (S == 2) {
        n.Q[p] = two;
    } else {
        const uint32_t third = p == 0 ? w[2] << 2 : (p == 1 ? w[2] << 1 : (p == 2 ? w[2] : w[2] >> 1));
        n.Q[p] = bit_select(0x33333333u, two, third);
    }
    if constexpr (S == 4)
        n.top = w[3];
}

template <int S>
__device__ __forceinline__ void lut_nibble_words(const uint32_t (&w)[S], Nibbles<S> &n)
{
    uint32_t pair[2];
    lut_nibble_pairs<S>(w, pair);
#pragma unroll
    for (int p = 0; p < 4; ++p)
        lut_nibble_word<S>(w, pair, n, p);
}

// The selector of v_perm_b32 that takes byte b of its first operand where the fourth plane has element p + 8b, of its
// second elsewhere.
__device__ __forceinline__ uint32_t lut_halves(const Nibbles<4> &n, int p)
{
    uint32_t low = 0x03020100u;
    asm("" : "+v"(low));                 // (in a register: with both constants literal, and and or are two operations)
    return ((p < 2 ? n.top << (2 - p) : n.top >> (p - 2)) & 0x04040404u) | low;
}

// The weights of elements p, p + 8 (w01) and p + 16, p + 24 (w23) of the word, p = 0..7, as packed fp16 pairs.
template <int S>
__device__ __forceinline__ void lut_look_up(const LutTables<S> &t, const Nibbles<S> &n, int p, uint32_t &w01, uint32_t &w23)
{
    const uint32_t qs = p < 4 ? n.Q[p & 3] : n.Q[p & 3] >> 4;
    const uint32_t sel = qs & (S == 2 ? 0x03030303u : 0x07070707u);
    uint32_t lo, hi;
    if constexpr (S == 2) {
        lo = __builtin_amdgcn_perm(t.lo[0], t.lo[0], sel);
        hi = __builtin_amdgcn_perm(t.hi[0], t.hi[0], sel);
    } else {
        lo = __builtin_amdgcn_perm(t.lo[1], t.lo[0], sel);
        hi = __builtin_amdgcn_perm(t.hi[1], t.hi[0], sel);
    }
    if constexpr (S == 4) {
        // byte b of the upper half's look-up where the fourth plane has element p + 8b, of the lower half's elsewhere
        const uint32_t half = lut_halves(n, p);
        lo = __builtin_amdgcn_perm(__builtin_amdgcn_perm(t.lo[3], t.lo[2], sel), lo, half);
        hi = __builtin_amdgcn_perm(__builtin_amdgcn_perm(t.hi[3], t.hi[2], sel), hi, half);
    }
    w01 = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
    w23 = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
}

// The B operand of MFMA q = 0..3 of the word: elements 2q, 2q+8, 2q+16, 2q+24, 2q+1, 2q+9, 2q+17, 2q+25.
template <int S>
__device__ __forceinline__ v4u lut_operand(const LutTables<S> &t, const Nibbles<S> &n, int q)
{
    uint32_t b0, b1, b2, b3;
    lut_look_up<S>(t, n, 2 * q, b0, b1);
    lut_look_up<S>(t, n, 2 * q + 1, b2, b3);
    return v4u{b0, b1, b2, b3};
}

// The same for 2 to 8 planes: up to 4 as above; 6 planes as two tables of three, 8 as two of three and one of two, whose
// entries are added in fp16 (three or five roundings a weight, where the sum plane by plane has one per plane).  A table of
// 16 entries takes 12 operations per four weights, one of 8 or 4 entries 5: 8 planes in two tables of 16 took 0.89 us
// a step of the prefill kernel.
template <int S>
struct WeightTables {
    static constexpr int H = S <= 4 ? S : 3, halves = S <= 4 ? 1 : 2;       // planes of the first table (and the second)
    LutTables<H> t[halves];
    LutTables<2> last;                                                      // (unused, hence no registers, up to 6 planes)
};

template <int S>
struct WeightNibbles {
    Nibbles<WeightTables<S>::H> t[WeightTables<S>::halves];
    Nibbles<2> last;
};

template <int S>
__device__ __forceinline__ void build_weight_tables(const uint32_t (&c)[(S + 1) / 2], WeightTables<S> &t)
{
    if constexpr (S <= 4) {
        lut_build_tables<S>(c, t.t[0]);
    } else {
        const uint32_t first[2] = {c[0], c[1] & 0xffffu}, second[2] = {(c[1] >> 16) | (c[2] << 16), c[2] >> 16};
        lut_build_tables<3>(first, t.t[0]);
        lut_build_tables<3>(second, t.t[1]);
        if constexpr (S == 8) {
            const uint32_t third[1] = {c[3]};
            lut_build_tables<2>(third, t.last);
        }
    }
}

template <int S>
__device__ __forceinline__ void weight_nibbles(const uint32_t (&w)[S], WeightNibbles<S> &n)
{
    if constexpr (S <= 4) {
        lut_nibble_words<S>(w, n.t[0]);
    } else {
        const uint32_t first[3] = {w[0], w[1], w[2]}, second[3] = {w[3], w[4], w[5]};
        lut_nibble_words<3>(first, n.t[0]);
        lut_nibble_words<3>(second, n.t[1]);
        if constexpr (S == 8) {
            const uint32_t third[2] = {w[6], w[7]};
            lut_nibble_words<2>(third, n.last);
        }
    }
}

// The B operand of MFMA q of the word (see lut_operand).
template <int S>
__device__ __forceinline__ v4u weight_operand(const WeightTables<S> &t, const WeightNibbles<S> &n, int q)
{
    v4u r = lut_operand<WeightTables<S>::H>(t.t[0], n.t[0], q);
    // (a line's coefficients grow in magnitude: the largest entries come last, so that one addition rounds at the sum's size)
    auto add = [&](const v4u &u) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            r[i] = __builtin_bit_cast(uint32_t, as_v2h(r[i]) + as_v2h(u[i]));
    };
    if constexpr (S > 4)
        add(lut_operand<3>(t.t[1], n.t[1], q));
    if constexpr (S == 8)
        add(lut_operand<2>(t.last, n.last, q));
    return r;
}

}  // namespace

#endif
