// Goldilocks field p = 2^64 - 2^32 + 1 for gfx950 VALU (and the host).
//
// Values are u64.  "canonical" means in [0, p) -- the representation of the
// reference's BFieldElement (include/types/b_field_element.hpp:31-41) and of
// every buffer crossing the C ABI.  Inside kernels some paths keep values
// "lazy": any u64 congruent to the field element, made canonical before they
// are stored.  Every function says which it takes and returns.
//
// The 64x64 product is built from four 32x32->64 multiply-adds
// (v_mad_u64_u32); the 128-bit result is folded with 2^64 = 2^32 - 1 and
// 2^96 = -1 (mod p).  The kernels take their products and folds from the forms
// that set a rare borrow aside (mul_rare, mul_n, ...) and the exact ones where
// that case is redone, in set-up and on the host.  add_lazy, sqr_wide, mont_sqr,
// mont_mul, lin52 and the shift multiplies (mul_pow2...) have only the native
// checks as callers now.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gl {

typedef uint64_t u64;
typedef uint32_t u32;

constexpr u64 P = 0xFFFFFFFF00000001ull;
constexpr u64 EPS = 0xFFFFFFFFull;  // 2^64 mod p

__host__ __device__ __forceinline__ u64 mk64(u32 lo, u32 hi) { return ((u64)hi << 32) | lo; }

// Starts a carry chain for the device compiler: the value is pinned in a VGPR
// as it stands, so the chain that produced it cannot be merged into the next.
// (The gfx950 compiler of ROCm 7.2 folds a final subtract-with-borrow of 0 into
// a following add-with-carry of 0, as in canon(montyred(..)) or canon(sub(..)),
// and then selects on a wrong carry; the device check
// tests/native/gl64_device_check.hip shows it.)  canon() pins its input.  No
// instruction is emitted; a no-op on the host.
__host__ __device__ __forceinline__ void opaque(u32& x) {
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+v"(x));
#else
    (void)x;
#endif
}

// Explicit 32-bit carry chains (v_add_co/v_addc, v_sub_co/v_subb on gfx950):
// full-rate VALU ops, no 64-bit compares.  The same code serves the host.

// any u64 -> canonical, for an input whose producer is known to compile
// correctly in front of this chain (a 64-bit fold, a load)
__host__ __device__ __forceinline__ u64 canon_raw(u64 x) {
    u32 k, c;
    u32 t0 = __builtin_addc((u32)x, 0xFFFFFFFFu, 0u, &k);  // x + EPS carries out iff x >= p
    u32 t1 = __builtin_addc((u32)(x >> 32), 0u, k, &c);
    return c ? mk64(t0, t1) : x;
}

// any u64 -> canonical.  The input is pinned (opaque) so that the carry chain
// that produced it is never merged into this one.
__host__ __device__ __forceinline__ u64 canon(u64 x) {
    u32 x0 = (u32)x, x1 = (u32)(x >> 32);
    opaque(x0);
    opaque(x1);
    return canon_raw(mk64(x0, x1));
}

// a, b canonical -> canonical
__host__ __device__ __forceinline__ u64 add(u64 a, u64 b) {
    u32 c0, c1, c2, c3;
    u32 s0 = __builtin_addc((u32)a, (u32)b, 0u, &c0);
    u32 s1 = __builtin_addc((u32)(a >> 32), (u32)(b >> 32), c0, &c1);
    u32 t0 = __builtin_addc(s0, 0xFFFFFFFFu, 0u, &c2);
    u32 t1 = __builtin_addc(s1, 0u, c2, &c3);
    return (c1 | c3) ? mk64(t0, t1) : mk64(s0, s1);
}

// a, b canonical -> canonical
__host__ __device__ __forceinline__ u64 sub(u64 a, u64 b) {
    u32 b0, b1, b2, b3;
    u32 d0 = __builtin_subc((u32)a, (u32)b, 0u, &b0);
    u32 d1 = __builtin_subc((u32)(a >> 32), (u32)(b >> 32), b0, &b1);
    u32 e0 = __builtin_subc(d0, 0xFFFFFFFFu, 0u, &b2);   // borrow: add p = subtract EPS
    u32 e1 = __builtin_subc(d1, 0u, b2, &b3);
    return b1 ? mk64(e0, e1) : mk64(d0, d1);
}

// a any u64, b canonical -> lazy (any u64).
__host__ __device__ __forceinline__ u64 add_lazy(u64 a, u64 b) {
    u32 c0, c1, c2, c3;
    u32 s0 = __builtin_addc((u32)a, (u32)b, 0u, &c0);
    u32 s1 = __builtin_addc((u32)(a >> 32), (u32)(b >> 32), c0, &c1);
    // carry: subtract p = add EPS; a + b < 2^65 - 2^32 so this cannot carry again
    u32 t0 = __builtin_addc(s0, c1 ? 0xFFFFFFFFu : 0u, 0u, &c2);
    u32 t1 = __builtin_addc(s1, 0u, c2, &c3);
    return mk64(t0, t1);
}

// 128-bit value (hi:lo) -> lazy u64 congruent to it:
// lo + hl*2^64 + hh*2^96 = lo + hl*(2^32 - 1) - hh  (mod p).
// (Measured on gfx950: the compiler's compare/select form of this fold beats an
// explicit carry chain, whose SGPR carries add wait states.)
__host__ __device__ __forceinline__ u64 fold128(u64 lo, u64 hi) {
    u32 hh = (u32)(hi >> 32), hl = (u32)hi;
    u64 t = lo - hh;
    if (lo < hh) t -= EPS;                 // borrow: add p
    u64 u = ((u64)hl << 32) - hl;          // hl * (2^32 - 1) < 2^64
    u64 r = t + u;
    if (r < u) r += EPS;                   // carry: subtract p
    return r;
}

// a canonical -> canonical
__host__ __device__ __forceinline__ u64 neg(u64 a) { return a ? P - a : 0; }

// 64x64 -> 128 from four independent 32x32 products (v_mad_u64_u32 on the
// device): the cross sum S = a1*b0 + a0*b1 is kept as 64 bits plus a carry c,
// then lo = p00 + (S << 32), hi = p11 + (S >> 32) + (c << 32) + carry(lo).
// No 32-bit half is widened into a fresh register pair (those moves dominated
// the chained form p00 -> a0*b1 + (p00 >> 32) -> ...).  Host code runs the
// same function in the native check against unsigned __int128.
__host__ __device__ __forceinline__ void mul_wide_4mad(u64 a, u64 b, u64& lo, u64& hi) {
    u32 a0 = (u32)a, a1 = (u32)(a >> 32), b0 = (u32)b, b1 = (u32)(b >> 32);
    u64 p00 = (u64)a0 * b0;
    u64 q = (u64)a1 * b1;
    u64 x = (u64)a1 * b0, y = (u64)a0 * b1;
    u32 k0, c, k1, k2, k3, k4;
    u32 S0 = __builtin_addc((u32)x, (u32)y, 0u, &k0);  // cross sum in words: the 64-bit
    u32 S1 = __builtin_addc((u32)(x >> 32), (u32)(y >> 32), k0, &c);  // add + compare costs more
    u32 l1 = __builtin_addc((u32)(p00 >> 32), S0, 0u, &k1);
    u32 h0 = __builtin_addc((u32)q, S1, k1, &k2);
    u32 h1 = __builtin_addc((u32)(q >> 32), 0u, k2, &k3);
    h1 = __builtin_addc(h1, 0u, c, &k4);
    lo = mk64((u32)p00, l1);
    hi = mk64(h0, h1);
}

// a^2 -> 128 bits from three products: the cross term a0*a1 is doubled with
// word shifts (bit 63 becomes the carry into the high word).
__host__ __device__ __forceinline__ void sqr_wide(u64 a, u64& lo, u64& hi) {
    u32 a0 = (u32)a, a1 = (u32)(a >> 32);
    u64 p00 = (u64)a0 * a0;
    u64 q = (u64)a1 * a1;
    u64 x = (u64)a0 * a1;
    u32 x0 = (u32)x, x1 = (u32)(x >> 32);
    u32 s0 = x0 << 1, s1 = (x1 << 1) | (x0 >> 31), c = x1 >> 31;  // 2x = c*2^64 + (s1:s0)
    u32 k1, k2, k3, k4;
    u32 l1 = __builtin_addc((u32)(p00 >> 32), s0, 0u, &k1);
    u32 h0 = __builtin_addc((u32)q, s1, k1, &k2);
    u32 h1 = __builtin_addc((u32)(q >> 32), c, k2, &k3);
    (void)k3;
    (void)k4;
    lo = mk64((u32)p00, l1);
    hi = mk64(h0, h1);
}

__host__ __device__ __forceinline__ void mul_wide(u64 a, u64 b, u64& lo, u64& hi) {
#ifdef __HIP_DEVICE_COMPILE__
    mul_wide_4mad(a, b, lo, hi);
#else
    unsigned __int128 pr = (unsigned __int128)a * b;
    lo = (u64)pr;
    hi = (u64)(pr >> 64);
#endif
}

// Montgomery reduction for R = 2^64: x = hi*2^64 + lo -> x * 2^-64 mod p, for
// any 128-bit x (the reference's montyred, b_field_element.hpp:103).  With
// m = lo * (1 + 2^32) mod 2^64 (lo + (lo << 32), overflow e), x + m*p is a
// multiple of 2^64 and (x + m*p) / 2^64 = hi - b with b = m - (m >> 32) - e;
// a borrow is corrected by adding p (subtracting 2^32 - 1 mod 2^64).  The
// result is < 2^64 and canonical when hi < p.
// In 32-bit words: a = (lo0, lo1 + lo0) with e the carry of the high word,
// b = a - a1 - e, r = hi - b, then r - (2^32 - 1) on a borrow.
__host__ __device__ __forceinline__ u64 montyred(u64 lo, u64 hi) {
    u32 lo0 = (u32)lo, lo1 = (u32)(lo >> 32);
    u32 e, k0, k1, c0, c1, d0, d1;
    u32 a1 = __builtin_addc(lo1, lo0, 0u, &e);
    u32 b0 = __builtin_subc(lo0, a1, e, &k0);
    u32 b1 = __builtin_subc(a1, 0u, k0, &k1);
    u32 r0 = __builtin_subc((u32)hi, b0, 0u, &c0);
    u32 r1 = __builtin_subc((u32)(hi >> 32), b1, c0, &c1);
    r0 = __builtin_subc(r0, 0u - c1, 0u, &d0);
    r1 = __builtin_subc(r1, 0u, d0, &d1);
    return mk64(r0, r1);
}

// L + H * 2^32 mod p for L, H < 2^52 -> < 2^64, in
// 32-bit words: with 2^64 = 2^32 - 1 mod p the value is (L0 - H1) +
// (L1 + H0 + H1) * 2^32; a carry out of the high word is folded back as 2^32 - 1.
__host__ __device__ __forceinline__ u64 lin52(u64 L, u64 H) {
    u32 L0 = (u32)L, L1 = (u32)(L >> 32), H0 = (u32)H, H1 = (u32)(H >> 32);
    u32 b, b2, c, c2, d, d2;
    u32 lo = __builtin_subc(L0, H1, 0u, &b);
    u32 t = __builtin_subc(L1 + H1, 0u, b, &b2);  // L1 + H1 - b >= 0: b = 1 needs H1 > 0
    u32 h = __builtin_addc(H0, t, 0u, &c);       // high word and its carry (value 2^64)
    // carry: add 2^64 = 2^32 - 1 (mod p); then h < 2^21, so h + 1 cannot overflow
    lo = __builtin_subc(lo, 0u, c, &d);
    h = __builtin_addc(h, 0u, c, &c2);
    h = __builtin_subc(h, 0u, d, &d2);
    (void)b2;
    (void)c2;
    (void)d2;
    return mk64(lo, h);
}

// a * a * 2^-64 mod p, any u64 a -> < 2^64
__host__ __device__ __forceinline__ u64 mont_sqr(u64 a) {
    u64 lo, hi;
    sqr_wide(a, lo, hi);
    return montyred(lo, hi);
}

// x * 2^64 mod p (into Montgomery form), any u64 x -> < 2^64:
// x*2^64 = x*(2^32 - 1) = x0*2^32 - x0 - x1 (mod p) for x = x1*2^32 + x0.
__host__ __device__ __forceinline__ u64 to_mont(u64 x) {
    u32 x0 = (u32)x, x1 = (u32)(x >> 32);
    u64 t = (u64)x0 * EPS;  // < 2^64
    u64 r = t - x1;
    if (t < x1) r -= EPS;   // borrow (only when x0 = 0): add p
    return r;
}

// a * b * 2^-64 mod p (Montgomery product), any u64 inputs -> < 2^64
__host__ __device__ __forceinline__ u64 mont_mul(u64 a, u64 b) {
    u64 lo, hi;
    mul_wide(a, b, lo, hi);
    return montyred(lo, hi);
}

// a, b any u64 -> lazy
__host__ __device__ __forceinline__ u64 mul_lazy(u64 a, u64 b) {
    u64 lo, hi;
    mul_wide(a, b, lo, hi);
    return fold128(lo, hi);
}

// a, b any u64 -> canonical
__host__ __device__ __forceinline__ u64 mul(u64 a, u64 b) { return canon_raw(mul_lazy(a, b)); }

// ---- products with the unlikely borrow set aside (device only) -----------------
// The product l + h*2^64 (h = h1:h0) folds to (l + h0*(2^32 - 1)) - h1.  Its
// 64-bit sum u carries about every second time (the carry c adds 2^32 - 1 back),
// but u < h1 with c = 0 needs u below 2^32: one product in 2^32 of random
// operands.  The *_rare forms leave that case to the caller: they add the lane
// to `bad` and their result is then wrong; the caller branches on `bad` once for
// many products and redoes them with the exact forms (mul_lazy, ...).  A fold is
// then 4 VALU operations (a multiply-add and three carry operations) where
// montyred and fold128 take 8 and more.
//
// Carries are lane masks in SGPR pairs, named by asm because the language has
// no word for the carry out of v_mad_u64_u32 and the compiler turns sums with
// two carries in into selects.  gfx950 wants two wait states between a VALU
// write of an SGPR and a VALU read of it, and the compiler does not look into
// asm: the forms take N values at a time and do each step for all of them, so
// that for N >= 3 two other instructions lie between (volatile asm keeps its
// order); fewer values take s_nops.
typedef u64 mask;  // a bit per lane, uniform
template <int N>
__device__ __forceinline__ void carry_wait() {
    if constexpr (N < 3) asm volatile("s_nop %0" ::"n"(N < 3 ? 2 - N : 0));
}

__device__ __forceinline__ bool in_mask(mask m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// r = a + k, a - b, a - b - k, a - k and the carry (borrow) out
#define GL_ADDC_0(r, ko, a, k) \
    asm volatile("v_addc_co_u32 %0, %1, %2, 0, %3" : "=v"(r), "=s"(ko) : "v"(a), "s"(k))
#define GL_SUB_CO(r, k, a, b) \
    asm volatile("v_sub_co_u32 %0, %1, %2, %3" : "=v"(r), "=s"(k) : "v"(a), "v"(b))
#define GL_SUBB_CO(r, ko, a, b, k) \
    asm volatile("v_subb_co_u32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(ko) : "v"(a), "v"(b), "s"(k))
#define GL_SUBB_0(r, ko, a, k) \
    asm volatile("v_subb_co_u32 %0, %1, %2, 0, %3" : "=v"(r), "=s"(ko) : "v"(a), "s"(k))
// r = a * b + c (64 bits) and the carry out; the second form has b = 2^32 - 1
#define GL_MAD_CO(r, k, a, b, c) \
    asm volatile("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(k) : "v"(a), "v"(b), "v"(c))
#define GL_MAD_EPS_CO(r, k, a, c) \
    asm volatile("v_mad_u64_u32 %0, %1, %2, -1, %3" : "=v"(r), "=s"(k) : "v"(a), "v"(c))

// Lanes of value i with k & ~c (k is overwritten), kept on the scalar unit: in a
// mask of its own, or joined to one mask for all values.
template <int N>
__device__ __forceinline__ void note_rare(mask (&bad)[N], int i, mask& k, mask c) {
    asm volatile("s_andn2_b64 %0, %1, %2" : "=s"(bad[i]) : "s"(k), "s"(c) : "scc");
}
__device__ __forceinline__ void note_rare(mask& bad, int, mask& k, mask c) {
    asm volatile("s_andn2_b64 %1, %1, %2\n\ts_or_b64 %0, %0, %1" : "+s"(bad), "+s"(k) : "s"(c) : "scc");
}

// l + (h1:h0) * 2^64 -> lazy u64, or bad: r then has to be lowered by 2^32 - 1
// (u - h1 wrapped to at least 2^64 - 2^32).  Bad: mask[N] or mask.
template <int N, class Bad>
__device__ __forceinline__ void fold128_rare(u64 (&r)[N], const u64 (&l)[N], const u32 (&h0)[N],
                                             const u32 (&h1)[N], Bad& bad) {
    u64 u[N];
    u32 r0[N], r1[N];
    mask c[N], k[N], none;
#pragma unroll
    for (int i = 0; i < N; i++) GL_MAD_EPS_CO(u[i], c[i], h0[i], l[i]);
    carry_wait<N>();
#pragma unroll
    for (int i = 0; i < N; i++) GL_SUBB_CO(r0[i], k[i], (u32)u[i], h1[i], c[i]);  // - h1 - c
    carry_wait<N>();
#pragma unroll
    for (int i = 0; i < N; i++) GL_SUBB_0(r1[i], k[i], (u32)(u[i] >> 32), k[i]);
#pragma unroll
    for (int i = 0; i < N; i++) GL_ADDC_0(r1[i], none, r1[i], c[i]);                // + c * 2^32
#pragma unroll
    for (int i = 0; i < N; i++) {
        note_rare(bad, i, k[i], c[i]);
        r[i] = mk64(r0[i], r1[i]);
    }
}

// r = a * b, any u64 -> lazy u64, or bad.  The partial products are chained through
// the addends of the multiply-adds: 4 of those, 3 moves (the high word of a pair
// to the low one of the next) and one carry, where adding the cross sum word by
// word took four carry operations and a squaring, with its doubling, six of 2 to 4
// cycles (hashing 2^22 rows of 379: 19.9 -> 18.6 ms, LDE 2^20 x 379: 19.1 -> 18.8).
template <int N, class Bad>
__device__ __forceinline__ void mul_rare(u64 (&r)[N], const u64 (&a)[N], const u64 (&b)[N], Bad& bad) {
    u64 l[N], q[N];
    u32 h0[N], h1[N];
    mask cm[N], none;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const u32 a0 = (u32)a[i], a1 = (u32)(a[i] >> 32), b0 = (u32)b[i], b1 = (u32)(b[i] >> 32);
        const u64 p = (u64)a0 * b0, t = (u64)a1 * b0 + (p >> 32);
        u64 y;
        GL_MAD_CO(y, cm[i], a0, b1, t);
        q[i] = (u64)a1 * b1 + (y >> 32);
        l[i] = mk64((u32)p, (u32)y);
        h0[i] = (u32)q[i];
    }
    carry_wait<N>();
#pragma unroll
    for (int i = 0; i < N; i++) GL_ADDC_0(h1[i], none, (u32)(q[i] >> 32), cm[i]);
    fold128_rare(r, l, h0, h1, bad);
}

// r = a * b, any u64 -> lazy u64 (exact; the unlikely borrow in a branch)
template <int N>
__device__ __forceinline__ void mul_n(u64 (&r)[N], const u64 (&a)[N], const u64 (&b)[N]) {
    mask bad[N], any = 0;
    mul_rare(r, a, b, bad);
#pragma unroll
    for (int i = 0; i < N; i++) asm volatile("s_or_b64 %0, %0, %1" : "+s"(any) : "s"(bad[i]) : "scc");
    if (__builtin_expect(in_mask(any), 0)) {
#pragma unroll
        for (int i = 0; i < N; i++)
            if (in_mask(bad[i])) r[i] -= EPS;
    }
}

// lazy -> canonical: p <= x < 2^64 only with a high word of ones
template <int N>
__device__ __forceinline__ void canon_n(u64 (&x)[N]) {
    bool big = false;
#pragma unroll
    for (int i = 0; i < N; i++) big |= (u32)(x[i] >> 32) == 0xFFFFFFFFu;
    if (__builtin_expect(big, 0)) {
#pragma unroll
        for (int i = 0; i < N; i++)
            if (x[i] >= P) x[i] -= P;
    }
}

// x * 2^64 (into Montgomery form), any u64 -> lazy u64, or bad (only when the
// low word of x is 0 and the high one is not)
template <int N>
__device__ __forceinline__ void to_mont_rare(u64 (&r)[N], const u64 (&x)[N], mask& bad) {
    static_assert(N >= 3, "wait states");
    u64 t[N];
    u32 r0[N], r1[N];
    mask k[N];
#pragma unroll
    for (int i = 0; i < N; i++) t[i] = (u64)(u32)x[i] * EPS;
#pragma unroll
    for (int i = 0; i < N; i++) GL_SUB_CO(r0[i], k[i], (u32)t[i], (u32)(x[i] >> 32));
#pragma unroll
    for (int i = 0; i < N; i++) GL_SUBB_0(r1[i], k[i], (u32)(t[i] >> 32), k[i]);
#pragma unroll
    for (int i = 0; i < N; i++) {
        asm volatile("s_or_b64 %0, %0, %1" : "+s"(bad) : "s"(k[i]) : "scc");
        r[i] = mk64(r0[i], r1[i]);
    }
}

// Constants of the joins that the compiler must not see through (it would
// replace the multiply-adds by shifts and carries).
struct JoinConsts {
    u32 two16, eps;
};
__device__ __forceinline__ JoinConsts join_consts() {
    JoinConsts c{65536u, 0xFFFFFFFFu};
    asm volatile("" : "+s"(c.two16), "+s"(c.eps));
    return c;
}

// Sum of d[t] * 256^t over eight byte places whose pair sums A = d[0] + 256 d[1],
// B, C, D lie in [0, 2^31): L + H 2^32 with the halves L = A + B 2^16 and
// H = C + D 2^16, each below 2^48.
__device__ __forceinline__ u64 join_half(const JoinConsts& J, u32 d0, u32 d1, u32 d2, u32 d3) {
    const u32 A = d0 + (d1 << 8), B = d2 + (d3 << 8);
    return (u64)B * J.two16 + A;
}
// L + H 2^32 -> u64 congruent to it: L + H0 2^32 + H1 (2^32 - 1), whose 64-bit
// sum carries only when H0 is within 2^17 of 2^32 (once in 2^15 and less):
// `carry` then says that 2^32 - 1 has to be added.
__device__ __forceinline__ u64 join_rare(const JoinConsts& J, u64 L, u64 H, bool& carry) {
    const u64 L2 = (u64)(u32)(H >> 32) * J.eps + L;
    u32 k;
    const u32 r1 = __builtin_addc((u32)(L2 >> 32), (u32)H, 0u, &k);
    carry = k != 0;
    return mk64((u32)L2, r1);
}

// 2^e mod p for 0 <= e < 192 (compile-time usable)
__host__ __device__ constexpr u64 pow2_mod_p(int e) {
    u64 r = 1;
    for (int i = 0; i < e; i++) r = (r >= P - r) ? r - (P - r) : r + r;
    return r;
}

// x any u64, 0 < E <= 32 -> lazy x * 2^E: lo = x << E, hl = x >> (64 - E) < 2^32
template <int E>
__host__ __device__ __forceinline__ u64 mul_pow2_small(u64 x) {
    static_assert(E > 0 && E <= 32, "small shift");
    u64 lo = x << E;
    u32 hl = (u32)(x >> (64 - E));
    u32 k0, k1, c0, c1, c2, c3;
    u32 u0 = __builtin_subc(0u, hl, 0u, &k0);
    u32 u1 = __builtin_subc(hl, 0u, k0, &k1);
    u32 r0 = __builtin_addc((u32)lo, u0, 0u, &c0);
    u32 r1 = __builtin_addc((u32)(lo >> 32), u1, c0, &c1);
    r0 = __builtin_addc(r0, c1 ? 0xFFFFFFFFu : 0u, 0u, &c2);
    r1 = __builtin_addc(r1, 0u, c2, &c3);
    return mk64(r0, r1);
}

// x * 2^E mod p for a compile-time 0 <= E < 96 and any u64 x -> canonical,
// without a general product.  p divides 2^96 + 1, so with x << E split into
// 32-bit words w0..w4 (E = 32q + r), the 96 low bits count positively and the
// words above bit 96 negatively: x*2^E = lo + w2*2^64 - hi, lo = (w1:w0),
// hi = (w4:w3), and 2^64 = 2^32 - 1 mod p turns w2*2^64 into one
// multiply-add.  The word shuffles are free; r != 0 costs funnel shifts.
template <int E>
__host__ __device__ __forceinline__ u64 mul_pow2(u64 x) {
    static_assert(E >= 0 && E < 96, "exponent");
    constexpr int q = E / 32, r = E % 32;
    const u32 x0 = (u32)x, x1 = (u32)(x >> 32);
    u32 w[5] = {0, 0, 0, 0, 0};
    if (r == 0) {
        w[q] = x0;
        w[q + 1] = x1;
    } else {
        w[q] = x0 << r;
        w[q + 1] = (x1 << r) | (x0 >> (32 - r));
        w[q + 2] = x1 >> (32 - r);
    }
    // In 32-bit words (no 64-bit multiply or compare):
    // m = w2 * (2^32 - 1) = (w2 - [w2 != 0]) : (-w2)
    u32 b0, b1, c0, c1, c2, c3;
    u32 m0 = __builtin_subc(0u, w[2], 0u, &b0);
    u32 m1 = __builtin_subc(w[2], 0u, b0, &b1);
    // t = lo + m < 2^65 - 2^33; a carry (2^64) folds back as EPS and cannot
    // carry again (t mod 2^64 <= 2^64 - 2^33 then)
    u32 t0 = __builtin_addc(w[0], m0, 0u, &c0);
    u32 t1 = __builtin_addc(w[1], m1, c0, &c1);
    t0 = __builtin_addc(t0, c1 ? 0xFFFFFFFFu : 0u, 0u, &c2);
    t1 = __builtin_addc(t1, 0u, c2, &c3);
    // v = t - hi, hi = (w4:w3) = x * 2^E >> 96 < 2^63 (0 when E < 32), so
    // -2^63 < v < 2^64; the canonical result is one of u = v mod 2^64, u + EPS
    // (v >= p: minus p) and u - EPS (v < 0: plus p, which lands in (0, p)),
    // selected at the end (no borrow fix feeding a second carry chain: the
    // gfx950 compiler merges such chains incorrectly, see opaque())
    u32 d1 = 0, u0 = t0, u1 = t1;
    if (q > 0) {
        u32 d0;
        u0 = __builtin_subc(t0, w[3], 0u, &d0);
        u1 = __builtin_subc(t1, w[4], d0, &d1);
    }
    u32 k0, k1, g0, g1;
    u32 a0 = __builtin_addc(u0, 0xFFFFFFFFu, 0u, &k0);  // u + EPS carries iff u >= p
    u32 a1 = __builtin_addc(u1, 0u, k0, &k1);
    u32 s0 = __builtin_subc(u0, 0xFFFFFFFFu, 0u, &g0);  // u - EPS (mod 2^64)
    u32 s1 = __builtin_subc(u1, 0u, g0, &g1);
    (void)b1;
    (void)c3;
    (void)g1;
    return d1 ? mk64(s0, s1) : (k1 ? mk64(a0, a1) : mk64(u0, u1));
}

__host__ __device__ inline u64 pow(u64 b, u64 e) {
    u64 r = 1;
    while (e) {
        if (e & 1) r = mul(r, b);
        b = mul(b, b);
        e >>= 1;
    }
    return r;
}

__host__ __device__ inline u64 inv(u64 a) { return pow(a, P - 2); }

// The reference's primitive 2^k-th root of unity, 7^((p-1)/2^k)
// (src/types/b_field_element.cpp:179-192).
__host__ __device__ inline u64 root_of_unity(u32 k) { return pow(7, (P - 1) >> k); }

}  // namespace gl
