// Tip5 permutation of 16 sponges per wavefront on gfx950, with the MDS layer on
// the matrix cores.
//
// Follows the reference permutation (src/hash/tip5.cpp:92-203): 5 rounds of
// S-box -> circulant MDS -> round constants; S-box = split-and-lookup on lanes
// 0..3 and x^7 on lanes 4..15.  The arithmetic is re-derived for the GPU:
//
//  * Layout.  Lane 16g + n of a wave holds words g, 4 + g, 8 + g, 12 + g of
//    sponge n (registers s[0..3]).  That is where v_mfma_i32_16x16x64_i8 takes
//    its second operand from and leaves its result, so the state never moves
//    between lanes; the four lookup words share register 0, so nothing diverges.
//  * The state is kept in Montgomery form x_M = x * 2^64 mod p (the form the
//    reference's split-and-lookup is defined on): the S-box of words 0..3 is the
//    byte lookup of the canonical value alone.  x^7 takes plain products on the
//    same values: (x 2^64)^7 = x^7 2^64 * 2^384, and 2^192 = 1 (mod p), so no
//    Montgomery reduction occurs at all.  Callers convert absorbed elements in
//    (to_m) and digests out (from_m, canonical).  The 256-byte table sits in LDS.
//  * MDS.  The 16x16 circulant has 16-bit entries m = m0 + 256 m1 + 65536 m2
//    with signed byte digits, the state words are 8 bytes, and 2^64 = 2^32 - 1,
//    so every output word is a sum of eight byte places whose coefficients are
//    fixed signed bytes: twelve 16x16x64 i8 products per round (the low words'
//    bytes reach six of the places, the high words' six).  Bytes are made
//    signed by flipping their top bits (x - kKappa in value); the constant that
//    takes this back, the round constant and a bias that keeps every sum
//    positive start the accumulators.  Sums stay below 2^31 (checked below).
//  * Products and the final join leave their unlikely borrow or carry to one
//    branch per round (gl64.hpp, *_rare).
//  * State words stay "lazy" (any u64 congruent mod p) inside the permutation;
//    callers canonicalise what they store.
//
// What bounds it: VALU issue.  The kernels issue a VALU instruction every 4
// cycles per SIMD (2 for a few plain 32-bit ones); matrix instructions of one
// wave run beside the VALU instructions of the others.  Rows of 2^22 x 379
// (1.6e8 permutations): 19.3 ms, against 29.2 ms with one sponge per lane, the
// MDS in f64 FMAs and Montgomery products.
#pragma once

#include "gl64.hpp"
#include "tip5_constants.hpp"

namespace tip5 {

using gl::u32;
using gl::u64;

constexpr int STATE = 16;
constexpr int RATE = 10;
constexpr int ROUNDS = 5;
constexpr int DIGEST = 5;
constexpr int WORDS = 4;        // state words per lane
constexpr int GROUP = 16;       // sponges per wave

// Round constants of the Tip5 specification: tip5_constants.hpp.
using tip5c::kRoundConstants;

typedef int v4i __attribute__((ext_vector_type(4)));

// 1 in Montgomery form (2^64 mod p)
constexpr u64 kOneM = gl::EPS;

// ---- the MDS layer as byte products (first column: SHA-256 of "Tip5") --------
constexpr int kProducts = 12;
// product p adds to place kPlace[p]; the first six take the low words' bytes
constexpr int kPlace[kProducts] = {0, 1, 2, 3, 4, 5, 0, 1, 4, 5, 6, 7};
constexpr u64 kKappa = 0x8080808080808080ull;
constexpr u32 kBias = 1u << 29;

// signed byte digit d (0..2) of a 16-bit entry: digits 0 and 1 in [-128, 127]
constexpr int mds_digit(int m, int d) {
    int d0 = m & 255;
    if (d0 > 127) d0 -= 256;
    int r = (m - d0) >> 8, d1 = r & 255;
    if (d1 > 127) d1 -= 256;
    return d == 0 ? d0 : d == 1 ? d1 : (r - d1) >> 8;
}
// coefficient of byte b (0..7) of word j in byte place t of output word i:
// 256^(b + d), with places 8 and 9 folded by 2^64 = 2^32 - 1
constexpr int mds_coefficient(int i, int j, int b, int t) {
    const int m = tip5c::kMdsFirstColumn[(i - j) & 15];
    int c = 0;
    for (int d = 0; d < 3; d++) {
        const int pos = b + d;
        if (pos == t) c += mds_digit(m, d);
        if (pos >= 8 && pos - 4 == t) c += mds_digit(m, d);
        if (pos >= 8 && pos - 8 == t) c -= mds_digit(m, d);
    }
    return c;
}

// First operands: lane 16g + r of product p holds row r's coefficients of the
// bytes that lane group g feeds in (register v: word 4v + g).  Row r = 4g' + v'
// is the output word 4v' + g', which lands in register v' of lane group g'.
struct MdsOperands {
    u32 w[kProducts * 64 * 4];
};
constexpr MdsOperands mds_operands() {
    MdsOperands t{};
    for (int p = 0; p < kProducts; p++)
        for (int g = 0; g < 4; g++)
            for (int r = 0; r < 16; r++)
                for (int v = 0; v < 4; v++) {
                    u32 x = 0;
                    for (int b = 0; b < 4; b++)
                        x |= (u32)(mds_coefficient(4 * (r & 3) + (r >> 2), 4 * v + g,
                                                   b + (p < 6 ? 0 : 4), kPlace[p]) &
                                   255)
                             << (8 * b);
                    t.w[(p * 64 + 16 * g + r) * 4 + v] = x;
                }
    return t;
}
__device__ const MdsOperands kMdsOperands = mds_operands();

// Largest magnitude a place's sum can take, over signed bytes.
constexpr int mds_bound(int t) {
    int s = 0;
    for (int j = 0; j < STATE; j++)
        for (int b = 0; b < 8; b++) {
            const int c = mds_coefficient(0, j, b, t);
            s += 128 * (c < 0 ? -c : c);
        }
    return s;
}
constexpr bool mds_fits() {
    for (int t = 0; t < 8; t += 2)
        if ((u64)mds_bound(t) + 256ull * (u64)mds_bound(t + 1) + 65536 >= kBias) return false;
    for (int j = 0; j < STATE; j++)
        for (int b = 0; b < 8; b++)
            for (int t = 0; t < 8; t++) {
                const int c = mds_coefficient(0, j, b, t);
                if (c < -128 || c > 127) return false;
            }
    return true;
}
static_assert(mds_fits(), "MDS byte sums leave their range");

// Accumulator starts of the even byte places: bias + 16 bits of
// (round constant in Montgomery form) + kKappa * (sum of the circulant) - biases.
// start[round][place / 2][g][v] for word 4v + g.
struct MdsStarts {
    u32 w[ROUNDS * 4 * 16];
};
constexpr MdsStarts mds_starts() {
    MdsStarts t{};
    typedef unsigned __int128 u128;
    u64 sum = 0;
    for (int i = 0; i < STATE; i++) sum += tip5c::kMdsFirstColumn[i];
    const u64 back = (u64)(((u128)kKappa * sum) % gl::P);
    const u128 bias = (u128)kBias * (1 + (1ull << 16) + (1ull << 32) + (1ull << 48));
    const u64 minus = gl::P - (u64)(bias % gl::P);
    for (int r = 0; r < ROUNDS; r++)
        for (int i = 0; i < STATE; i++) {
            const u64 rc = (u64)(((u128)kRoundConstants[r * STATE + i] * gl::EPS) % gl::P);
            const u64 c = (u64)(((u128)rc + back + minus) % gl::P);
            for (int q = 0; q < 4; q++)
                t.w[((r * 4 + q) * 4 + (i & 3)) * 4 + (i >> 2)] = kBias + (u32)((c >> (16 * q)) & 0xFFFF);
        }
    return t;
}
__device__ const MdsStarts kMdsStarts = mds_starts();

// ---- LDS tables of a block -----------------------------------------------------
struct alignas(16) Tables {
    u32 start[ROUNDS * 4 * 16];
    uint8_t lut[256];  // the S-box ((x+1)^3 mod 257) - 1, its top bit flipped
};
__device__ __forceinline__ void load_lut(uint8_t* lut) {
    for (u32 x = threadIdx.x; x < 256; x += blockDim.x) {
        u32 t = x + 1;
        lut[x] = (uint8_t)((((t * t % 257) * t % 257) - 1) ^ 0x80);
    }
}
// Fills them (the caller synchronises the block before use).
__device__ __forceinline__ void load_tables(Tables& T) {
    for (u32 i = threadIdx.x; i < ROUNDS * 64; i += blockDim.x) T.start[i] = kMdsStarts.w[i];
    load_lut(T.lut);
}

// The wave's constant operands, and where the lane sits.
struct Wave {
    typedef tip5::Tables Tables;
    static constexpr int kWords = WORDS;    // state words of a lane
    static constexpr u32 kSponges = GROUP;  // sponges of the wave
    __device__ __forceinline__ u32 word(int v) const { return 4 * v + g; }  // register v
    v4i mds[kProducts];
    gl::JoinConsts J;
    const Tables* T;
    u32 g, n;  // lane = 16 g + n
};
__device__ __forceinline__ Wave make_wave(const Tables& T) {
    Wave W;
    const u32 lane = threadIdx.x & 63;
    W.J = gl::join_consts();
    W.T = &T;
    W.g = lane >> 4;
    W.n = lane & 15;
#pragma unroll
    for (int p = 0; p < kProducts; p++)
        W.mds[p] = *(const v4i*)(kMdsOperands.w + (p * 64 + lane) * 4);
    return W;
}

// Montgomery form <-> canonical
__device__ __forceinline__ u64 to_m(u64 x) { return gl::to_mont(x); }
__device__ __forceinline__ u64 from_m(u64 y) { return gl::montyred(y, 0); }

// ---- S-box ----------------------------------------------------------------------
// x^7, exact (the products' unlikely case)
__device__ __forceinline__ u64 pow7(u64 x) {
    const u64 x2 = gl::mul_lazy(x, x), x4 = gl::mul_lazy(x2, x2);
    return gl::mul_lazy(gl::mul_lazy(x, x2), x4);
}
template <int N>
__device__ __forceinline__ void pow7_rare(u64 (&y)[N], const u64 (&x)[N], gl::mask& bad) {
    u64 x2[N], x3[N], x4[N];
    gl::mul_rare(x2, x, x, bad);
    gl::mul_rare(x3, x, x2, bad);
    gl::mul_rare(x4, x2, x2, bad);
    gl::mul_rare(y, x3, x4, bad);
}

// Four bytes through the table.  The loads zero-extend them, which the compiler does
// not make use of (3 operations for its 5: hashing 2^22 rows of 379, 19.3 -> 19.1 ms);
// but it places its own operations behind the x^7, where the loads have arrived,
// which is what a lone wave (LONE) wants.  The last operation is the compiler's: the
// result goes to a matrix product, which wants two wait states after a VALU write of
// its operand, and the compiler does not look into asm.
#define TIP5_LSHL_OR(r, b, n, a) asm("v_lshl_or_b32 %0, %1, " #n ", %2" : "=v"(r) : "v"(b), "v"(a))
template <bool LONE>
__device__ __forceinline__ u32 lookup_bytes(u32 x, const uint8_t* lut) {
    if constexpr (LONE)
        return (u32)lut[x & 0xff] | ((u32)lut[(x >> 8) & 0xff] << 8) |
               ((u32)lut[(x >> 16) & 0xff] << 16) | ((u32)lut[x >> 24] << 24);
    u32 lo, hi;
    TIP5_LSHL_OR(lo, (u32)lut[(x >> 8) & 0xff], 8, (u32)lut[x & 0xff]);
    TIP5_LSHL_OR(hi, (u32)lut[x >> 24], 8, (u32)lut[(x >> 16) & 0xff]);
    return (hi << 16) | lo;
}
#undef TIP5_LSHL_OR

// S-box of words 0..3 on a Montgomery-form value: bytes of the canonical value
// through the table; the result is the Montgomery form of the reference's
// output (tip5.cpp split_and_lookup), less kKappa byte by byte (y ^ kKappa).
__device__ __forceinline__ u64 split_and_lookup(u64 m, const uint8_t* lut) {
    u32 lo = (u32)m, hi = (u32)(m >> 32);
    // p <= m < 2^64 only with a high word of ones and a nonzero low word
    if (__builtin_expect(hi == 0xFFFFFFFFu, 0)) {
        if (lo) {
            lo -= 1;
            hi = 0;
        }
    }
    return gl::mk64(lookup_bytes<false>(lo, lut), lookup_bytes<false>(hi, lut));
}
// ... of m < p, in a lone wave
__device__ __forceinline__ u64 lookup_canonical(u64 m, const uint8_t* lut) {
    return gl::mk64(lookup_bytes<true>((u32)m, lut), lookup_bytes<true>((u32)(m >> 32), lut));
}

// ---- one round, the permutation --------------------------------------------------
// Round r (tip5.cpp:115-125: S-box layer, MDS, round constants) on the wave's
// Montgomery-form states (any u64 words congruent to x_M).  All 64 lanes take
// part; lanes of unused sponges carry any values.
__device__ __forceinline__ void round_m(u64 s[WORDS], int r, const Wave& W) {
    const u64 x[3] = {s[1], s[2], s[3]};
    u64 y7[3];
    gl::mask bad = 0;
    pow7_rare(y7, x, bad);
    const u64 look = split_and_lookup(s[0], W.T->lut);
    if (__builtin_expect(gl::in_mask(bad), 0)) {
#pragma unroll
        for (int i = 0; i < 3; i++) y7[i] = pow7(x[i]);
    }
    v4i lo, hi;
#pragma unroll
    for (int v = 0; v < WORDS; v++) {
        const u64 y = v ? y7[v - 1] ^ kKappa : look;
        lo[v] = (int)(u32)y;
        hi[v] = (int)(u32)(y >> 32);
    }
    const v4i* start = (const v4i*)(W.T->start + r * 64) + W.g;
    v4i y[8];
#pragma unroll
    for (int t = 0; t < 8; t++) y[t] = t & 1 ? v4i{0, 0, 0, 0} : start[2 * t];
#pragma unroll
    for (int p = 0; p < kProducts; p++)
        y[kPlace[p]] = __builtin_amdgcn_mfma_i32_16x16x64_i8(W.mds[p], p < 6 ? lo : hi,
                                                             y[kPlace[p]], 0, 0, 0);
    bool carry[WORDS];
#pragma unroll
    for (int v = 0; v < WORDS; v++)
        s[v] = gl::join_rare(
            W.J, gl::join_half(W.J, (u32)y[0][v], (u32)y[1][v], (u32)y[2][v], (u32)y[3][v]),
            gl::join_half(W.J, (u32)y[4][v], (u32)y[5][v], (u32)y[6][v], (u32)y[7][v]), carry[v]);
    if (__builtin_expect(carry[0] | carry[1] | carry[2] | carry[3], 0)) {
#pragma unroll
        for (int v = 0; v < WORDS; v++)
            if (carry[v]) s[v] += gl::EPS;
    }
}

// The permutation on the wave's Montgomery-form states.
__device__ __forceinline__ void permutation_m(u64 s[WORDS], const Wave& W) {
#pragma unroll 1
    for (int r = 0; r < ROUNDS; r++) round_m(s, r, W);
}

// ---- few sponges: four to a wave ---------------------------------------------------
// Where there are fewer waves of 16 sponges than SIMDs, the time of a permutation is
// the latency of one wave: 300 instructions a round, most of them the products of
// the three x^7 words and the joins of the four words of a lane.  Here a lane has
// one word: lane 16g + 4w + n holds word 4w + g of sponge n < 4.  The other words
// of its row come by row rotations, register v from w + v.  So column 4w + n of the
// matrix product sees its sponge rotated by w, and as the MDS matrix is circulant
// its result is rotated alike: output word g of the column is the lane's own word
// 4w + g.  Only those four rows are needed, so the other rows of a product hold
// other byte places (register v: place v, or 4 + v): four products a round in place
// of twelve, and one join.  A permutation takes 1.9 us where the form above takes
// 4.0, and twice the issue slots per sponge: 16384 rows of 379 163 us against 170,
// 4096 rows 82 against 157.
constexpr int QUAD = 4;  // sponges per wave

// First operands: product 2 P + h, row 4g' + v' is place 4 P + v' of output word g',
// from the bytes of the low (h = 0) or high words.
struct QuadOperands {
    u32 w[4 * 64 * 4];
};
constexpr QuadOperands quad_operands() {
    QuadOperands t{};
    for (int p = 0; p < 4; p++)
        for (int g = 0; g < 4; g++)
            for (int r = 0; r < 16; r++)
                for (int v = 0; v < 4; v++) {
                    u32 x = 0;
                    for (int b = 0; b < 4; b++)
                        x |= (u32)(mds_coefficient(r >> 2, 4 * v + g, b + 4 * (p & 1), 4 * (p >> 1) + (r & 3)) & 255)
                             << (8 * b);
                    t.w[(p * 64 + 16 * g + r) * 4 + v] = x;
                }
    return t;
}
__device__ const QuadOperands kQuadOperands = quad_operands();

struct alignas(16) QuadTables {
    u32 start[ROUNDS * 2 * 16 * 4];  // [round][P][word][v]
    uint8_t lut[256];
};
__device__ __forceinline__ void load_tables(QuadTables& T) {
    for (u32 i = threadIdx.x; i < ROUNDS * 128; i += blockDim.x) {
        const u32 v = i & 3, word = (i >> 2) & 15, P = (i >> 6) & 1, r = i >> 7;
        T.start[i] = v & 1 ? 0 : kMdsStarts.w[((r * 4 + 2 * P + v / 2) * 4 + (word & 3)) * 4 + (word >> 2)];
    }
    load_lut(T.lut);
}

struct QuadWave {
    typedef QuadTables Tables;
    static constexpr int kWords = 1;
    static constexpr u32 kSponges = QUAD;
    __device__ __forceinline__ u32 word(int) const { return own; }
    v4i mds[4];
    gl::JoinConsts J;
    const QuadTables* T;
    u32 own, n;  // the lane's word, of the wave's sponge n
};
__device__ __forceinline__ QuadWave make_wave(const QuadTables& T) {
    QuadWave W;
    const u32 lane = threadIdx.x & 63;
    W.J = gl::join_consts();
    W.T = &T;
    W.own = (lane & 12) + (lane >> 4);
    W.n = lane & 3;
#pragma unroll
    for (int p = 0; p < 4; p++) W.mds[p] = *(const v4i*)(kQuadOperands.w + (p * 64 + lane) * 4);
    return W;
}

__device__ __forceinline__ void round_m(u64 s[1], int r, const QuadWave& W) {
    const u64 x = s[0];
    const v4i* start = (const v4i*)(W.T->start) + r * 32 + W.own;
    v4i ya = start[0], yb = start[16];
    u64 look = lookup_canonical(x, W.T->lut);  // (of use in words 0..3)
    // p <= x < 2^64 only with a high word of ones: left to the branch of the products
    // (with one of its own a permutation took 2.06 us, without 1.94)
    gl::mask bad = __builtin_amdgcn_ballot_w64((u32)(x >> 32) == 0xFFFFFFFFu);
    const u64 x1[1] = {x};
    u64 x2[1], x34[2], y7[1];
    gl::mul_rare(x2, x1, x1, bad);
    const u64 xs[2] = {x, x2[0]}, x22[2] = {x2[0], x2[0]};
    gl::mul_rare(x34, xs, x22, bad);
    const u64 x3[1] = {x34[0]}, x4[1] = {x34[1]};
    gl::mul_rare(y7, x3, x4, bad);
    if (__builtin_expect(gl::in_mask(bad), 0)) {
        y7[0] = pow7(x);
        look = lookup_canonical(gl::canon(x), W.T->lut);
    }
    const u64 y = W.own < 4 ? look : y7[0] ^ kKappa;
    const int l = (int)(u32)y, h = (int)(u32)(y >> 32);
    // (row_ror:n reads lane i - n of the row)
#define TIP5_ROR(a, n) __builtin_amdgcn_mov_dpp(a, 0x120 + n, 0xF, 0xF, true)
    const v4i lo = {l, TIP5_ROR(l, 12), TIP5_ROR(l, 8), TIP5_ROR(l, 4)};
    const v4i hi = {h, TIP5_ROR(h, 12), TIP5_ROR(h, 8), TIP5_ROR(h, 4)};
#undef TIP5_ROR
    ya = __builtin_amdgcn_mfma_i32_16x16x64_i8(W.mds[0], lo, ya, 0, 0, 0);
    yb = __builtin_amdgcn_mfma_i32_16x16x64_i8(W.mds[2], lo, yb, 0, 0, 0);
    ya = __builtin_amdgcn_mfma_i32_16x16x64_i8(W.mds[1], hi, ya, 0, 0, 0);
    yb = __builtin_amdgcn_mfma_i32_16x16x64_i8(W.mds[3], hi, yb, 0, 0, 0);
    bool carry;
    s[0] = gl::join_rare(W.J, gl::join_half(W.J, (u32)ya[0], (u32)ya[1], (u32)ya[2], (u32)ya[3]),
                      gl::join_half(W.J, (u32)yb[0], (u32)yb[1], (u32)yb[2], (u32)yb[3]), carry);
    if (__builtin_expect(carry, 0)) s[0] += gl::EPS;
}
__device__ __forceinline__ void permutation_m(u64 s[1], const QuadWave& W) {
#pragma unroll 1
    for (int r = 0; r < ROUNDS; r++) round_m(s, r, W);
}


}  // namespace tip5
