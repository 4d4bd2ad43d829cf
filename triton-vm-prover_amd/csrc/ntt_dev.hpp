// Batched Goldilocks NTT and coset low-degree extension for gfx950.
//
// Math restated from src/ntt/ntt.cpp:26-131 and src/lde/lde_randomized.cpp:
// the LDE of a column x of length N onto the coset g*<w_M>, M = E*N, is
//   out[E*q + s] = NTT_N(f_s)[q],  f_s[r] = sum_{i = r mod N} p_i (g w_M^s)^i
// where p = INTT_N(x) * o^-i + (X^N - o^N) * rand(X) (o = trace offset).  The
// E cosets replace the reference's zero-pad + size-M NTT (same exact values,
// a quarter of the butterflies at E = 4).
//
// Each size-N transform is a four-step split N = N1 * N2 (N1 = 2^a):
//   step 1: N1-point DFTs down the columns of the N1 x N2 view, twiddle w_N^(n2 k1)
//   step 2: N2-point DFTs along rows (k1 fixed)
// The LDE runs INTT step 2, the coset scaling of all E cosets and forward step 1
// on whole rows in one kernel, with d_out as the only working memory:
//   K1  trace            -> Y   at out[E*N2*k1 + n2]
//   K2  Y (rows k1)      -> Z_s at out[E*(u1 + N2*k1) + s]   (in place per row)
//   K3  Z (u1-tile, all s) -> codewords at out[E*(u1 + N2*u2) + s] (in place)
//
// Sub-DFTs of length L <= 4096 run in LDS as radix-16 passes whose 16-point
// DFTs are matrix products (see Matrix).  Values between the kernels and inside
// them are lazy (any u64 congruent mod p); a kernel whose output leaves the
// library makes it canonical.
//
// This header holds the device code shared by the translation units that
// instantiate the kernels (ntt_step1.hip, ntt_step2.hip, lde_rows.hip,
// lde_step3.hip); the host side (plans, constant tables, launches) is
// ntt_kernels.hip.
//
// Measured on a 2^20 x 379 table to four cosets (3.2 GB in, 12.7 GB out), with
// radix-16 butterflies on the VALU before: K1 1.47 ms (2.2), K2 11.8 (12.2 in two
// kernels, which wrote and read the coefficients in between), K3 5.4 (7.1).  K1 and
// K3 move 4.3 and 4.7 TB/s, near what the memory gives a kernel that reads and
// writes the same amount.  K2 spends most of its time on VALU instructions (per output
// two products for the twiddles between passes, one for the coset, two for the
// twiddle on the way out, and 12 operations in each of three DFT passes): 6.6 cycles
// of a SIMD each, where a saturated SIMD takes 3.7 to 4; the rest is waits on LDS,
// global loads and barriers.
#pragma once

#include <type_traits>

#include "tvh_internal.hpp"

namespace tvh {

// ---------------------------------------------------------------- 16-point DFT
// A wave transforms 16 groups of 16 elements at once: lane 16g + n holds
// elements e = 4v + g (v = 0..3) of group n, before and after (natural order),
// the operand and result layout of v_mfma_i32_16x16x64_i8.
//
// w_64 = 2^39, so a 16-point DFT (and the 2-, 4- and 8-point ones, 2^(4-r) of
// them side by side) has coefficients +-2^x.  With an element split into bytes,
// x = lo + 2^32 hi and 2^64 = 2^32 - 1, every output is a sum of eight byte
// places, s and 4 + s for s < 4, of fixed signed bytes +-2^(x mod 8):
//   place s: P_s lo - Q_s hi,  place 4 + s: Q_s lo + S_s hi,  S_s = P_s + Q_s.
// Bytes are made signed by flipping their top bits; -Q_s hi is taken as Q_s * ~hi.
// The constants this leaves and a bias that keeps the sums positive start the
// accumulators.  16 products on the matrix cores and about 12 VALU operations
// per element for the bytes and the join replace the 39 of the butterflies on
// the VALU, which is what bounded the kernels.  256 elements take 360 cycles of
// a SIMD with four waves on it (a product costs the VALU about 7 of its 16
// cycles); with S_s hi as two products, which saves 16 registers, 440; with 2:4
// sparse products, whose accumulators the VALU has to fill, 370.
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr u32 LOG_TILE = 14;  // log2 elements of the largest tile (128 KB before padding)

// kDftWords u32 per matrix set (direction, r): P, Q, S for s = 0..3, each 64 lanes
// x 4 words; then the accumulator starts of the even places, [4][g][v].
constexpr u32 kDftStarts = 12 * 64 * 4;
constexpr u32 kDftWords = kDftStarts + 64;
constexpr u32 kDftBias = 1u << 25;
constexpr u32 kSignBits = 0x80808080u;

// The matrices stay in registers; the starts are read for each product, into the
// registers of its result.
struct Matrix {
    v4i p[4], q[4], s[4];
    const v4i* start;  // LDS (or global); the lane's first
};
__device__ __forceinline__ Matrix load_matrix(const u32* __restrict__ set, const u32* starts) {
    Matrix M;
    const u32 lane = threadIdx.x & 63;
    const v4i* w = (const v4i*)set;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        M.p[i] = w[i * 64 + lane];
        M.q[i] = w[(4 + i) * 64 + lane];
        M.s[i] = w[(8 + i) * 64 + lane];
    }
    M.start = (const v4i*)starts + (lane >> 4);
    return M;
}

// x any u64 -> lazy.  (The barriers keep other code's asm, whose registers the
// compiler's hazard checks do not see, out of the matrix products; the one in
// the middle halves the accumulators held at a time.)
__device__ __forceinline__ void dft16(const Matrix& M, const gl::JoinConsts& J, u64 (&x)[4]) {
    __builtin_amdgcn_sched_barrier(0);
    v4i lo, hi, nh;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        lo[v] = (int)((u32)x[v] ^ kSignBits);
        hi[v] = (int)((u32)(x[v] >> 32) ^ kSignBits);
        nh[v] = (int)((u32)(x[v] >> 32) ^ ~kSignBits);
    }
    const v4i zero = {0, 0, 0, 0};
    v4i y[4];
    u64 H[4];
#define TVH_MFMA(a, b, c) __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0)
#pragma unroll
    for (int s = 0; s < 4; s++) y[s] = TVH_MFMA(M.q[s], lo, s & 1 ? zero : M.start[8 + 2 * s]);
#pragma unroll
    for (int s = 0; s < 4; s++) y[s] = TVH_MFMA(M.s[s], hi, y[s]);
#pragma unroll
    for (int v = 0; v < 4; v++)
        H[v] = gl::join_half(J, (u32)y[0][v], (u32)y[1][v], (u32)y[2][v], (u32)y[3][v]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 4; s++) y[s] = TVH_MFMA(M.p[s], lo, s & 1 ? zero : M.start[2 * s]);
#pragma unroll
    for (int s = 0; s < 4; s++) y[s] = TVH_MFMA(M.q[s], nh, y[s]);
#undef TVH_MFMA
    bool carry[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const u64 L = gl::join_half(J, (u32)y[0][v], (u32)y[1][v], (u32)y[2][v], (u32)y[3][v]);
        x[v] = gl::join_rare(J, L, H[v], carry[v]);
    }
    if (__builtin_expect(carry[0] | carry[1] | carry[2] | carry[3], 0)) {
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (carry[v]) x[v] += gl::EPS;
    }
    __builtin_amdgcn_sched_barrier(0);
}

// ---------------------------------------------------------------- DFTs of a block
// NT transforms of length L = 2^logL (16 < L <= 4096), NT * L <= 2^LT, in LDS by
// decimation in frequency.  L = 2^rA * 2^rB * 16 with rB = min(4, logL - 4):
//   pass A (L > 256): 2^rA-point DFTs over the top index bits, over the block;
//   passes B, C: the 256-element (or shorter) pieces that remain, each by one
//   wave on its own: no barrier lies between, and the twiddles between B and C
//   are the lane's for the whole kernel.
// A pass takes 16 elements i0 + e*S, S a sixteenth of the sub-transform; for
// r < 4 the low 4 - r bits of e are left alone.  After pass A the result is
// multiplied by w^(rest * digit) and goes back where it came from; pass C leaves
// its piece in natural order.  So result k of the transform is at place
// (k mod 2^rA) * 256 + k / 2^rA (result_place).
//
// A block has 2^(LT-4) threads, 16 elements each: all global loads are in flight
// together, before the matrices take their registers, and the results are
// stored from LDS in the order of global memory.  Tile and length are
// compile-time constants, so that LDS accesses take immediate offsets; global
// ones take a wave-uniform base and a byte offset that the lane keeps
// throughout.  (With both at run time the same code took 1.6 times the VALU
// instructions and spilled registers.)
template <int LT, int LOGL, int LOGQ = 4>
struct Shape {
    static constexpr u32 kThreads = 1u << (LT - LOGQ), kWaves = kThreads / 64;
    static constexpr u32 kPer = 1u << LOGQ;  // elements of a thread
    static constexpr u32 L = 1u << LOGL, logNT = LT - LOGL, NT = 1u << logNT;
    static constexpr u32 rA = LOGL > 8 ? LOGL - 8 : 0;
    static constexpr u32 logP = LOGL < 8 ? LOGL : 8;  // length of a transform's piece
    static constexpr u32 rB = logP - 4;
    // LDS pitch of a transform.  Adjacent lanes take min(NT, 16) transforms and
    // then adjacent elements: the pitch is an odd multiple of 16 / min(NT, 16),
    // which spreads them over the banks.
    static constexpr u32 unit = logNT >= 4 ? 1 : 16u >> logNT;
    static constexpr u32 pitch = unit * (((L + (L >> 4) + (L >> 8) + unit) / unit) | 1);
    static constexpr u32 kStarts = pitch * NT;  // two sets of accumulator starts follow
};

// Element i of transform t: base[(t >> sh) * ts + (t mod 2^sh) * ts2 + i * is].
// (base: the block's first transform.)
template <class T>
struct Place {
    T* base;
    u32 sh, ts, ts2, is;
    __device__ __forceinline__ u32 off(u32 t, u32 i) const {
        return (t >> sh) * ts + (t & ((1u << sh) - 1)) * ts2 + i * is;
    }
};

// Access at a wave-uniform base plus the lane's byte offset (below 2^32: one
// instruction, no address arithmetic).
__device__ __forceinline__ u64 load_at(const u64* base, u32 bytes) {
    return *(const u64*)((const char*)base + bytes);
}
__device__ __forceinline__ void store_at(u64* base, u32 bytes, u64 x) {
    *(u64*)((char*)base + bytes) = x;
}

// LDS place of element i.  (Additive over index parts that share no bit.)
__host__ __device__ constexpr u32 lds_index(u32 i) { return i + (i >> 4) + (i >> 8); }
// Where result k lies.
__host__ __device__ constexpr u32 result_place(u32 k, u32 rA) {
    return ((k & ((1u << rA) - 1)) << 8) | (k >> rA);
}

// Workgroup barrier for LDS hand-offs only: waits for this wave's LDS
// operations, not for its global ones.  No thread of these kernels reads global
// memory that another thread of the block writes before the barrier.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// LDS hand-off between lanes of one wave: its LDS operations execute in order,
// so only the compiler has to keep theirs.
__device__ __forceinline__ void wave_handoff() { asm volatile("" ::: "memory"); }

// The least l with n <= 2^l (n > 0).
__device__ __forceinline__ u32 log_ceil(u32 n) { return n > 1 ? 32 - __builtin_clz(n - 1) : 0; }

__device__ __forceinline__ u32 wave_index() {
    return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

template <u32 LOGS>
__device__ __forceinline__ void lds_put(u64* p, const u64 (&x)[4]) {
#pragma unroll
    for (int v = 0; v < 4; v++) p[lds_index((u32)(4 * v) << LOGS)] = x[v];
}
template <u32 LOGS>
__device__ __forceinline__ void lds_get(const u64* p, u64 (&x)[4]) {
#pragma unroll
    for (int v = 0; v < 4; v++) x[v] = p[lds_index((u32)(4 * v) << LOGS)];
}

// Twiddles w_(16 S)^(rest * digit), rest = (e mod 2^(4-R)) S + jl, digit = e >> (4-R),
// of the elements e = 4v + g of a group with offset jl < S in a pass of digit bits
// R and stride S = 2^LOGS.
template <u32 R, u32 LOGS>
__device__ __forceinline__ void pass_twiddles(u64 (&f)[4], u32 jl, u32 g, const u64* __restrict__ r4096) {
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const u32 e = 4 * v + g;
        f[v] = load_at(r4096, (((e & ((1u << (4 - R)) - 1)) << LOGS) + jl) * ((e >> (4 - R)) << (11 - LOGS)));
    }
}

// Pass A on the first 2^log_t transforms: groups j of stride S = L / 16, lanes
// transform-fastest.  The next group's elements and twiddles are loaded before
// this one is transformed.
template <class Z>
__device__ __forceinline__ void dft_pass_a(u64* buf, u32 log_t, const Matrix& M,
                                           const gl::JoinConsts& J, const u64* __restrict__ r4096) {
    constexpr u32 kStep = 16 * Z::kWaves, kLogS = Z::logP + Z::rA - 4;
    const u32 g = (threadIdx.x & 63) >> 4, n = threadIdx.x & 15;
    const u32 total = 1u << (log_t + kLogS);  // (at least 16: L > 256)
    const u32 mask = (1u << log_t) - 1;
    const u32 jn = n >> log_t;
    u64* const lane_p = buf + (n & mask) * Z::pitch + lds_index(jn) + lds_index(g << kLogS);
    u64 x[4], f[4];
    auto get = [&](u32 w0, u64 (&x)[4], u64 (&f)[4]) -> u64* {
        w0 = w0 < total ? w0 : 0;
        const u32 j = w0 >> log_t;
        u64* p = lane_p + ((w0 & mask) * Z::pitch + lds_index(j));
        lds_get<kLogS>(p, x);
        pass_twiddles<Z::rA, kLogS>(f, j + jn, g, r4096);
        return p;
    };
    u32 w0 = wave_index() * 16;
    if (w0 >= total) return;
    u64* p = get(w0, x, f);
#pragma unroll 1
    for (; w0 < total; w0 += kStep) {
        u64 x2[4], f2[4];
        u64* p2 = get(w0 + kStep, x2, f2);
        dft16(M, J, x);
        gl::mul_n(x, x, f);
        lds_put<kLogS>(p, x);
        p = p2;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            x[v] = x2[v];
            f[v] = f2[v];
        }
    }
}

// Passes B and C of the pieces of the first 2^log_t transforms: M is the matrix
// of rB bits, at first.  From L = 256 on that is the one of pass C too; shorter
// transforms, several to a piece of 256, take the passes one after the other (a
// wave keeps its pieces).  Where 2^log_t transforms do not fill a piece, lanes
// repeat its first groups (equal values go to equal places).
template <class Z>
__device__ __forceinline__ void dft_pieces(u64* buf, u32 log_t, Matrix& M, const u32* mats,
                                           const u32* starts4, const gl::JoinConsts& J,
                                           const u64* __restrict__ r4096) {
    constexpr u32 kLogS = Z::rB, kShare = 8 - Z::logP, kPer = Z::rA;  // log2 transforms, pieces
    const u32 g = (threadIdx.x & 63) >> 4, n = threadIdx.x & 15;
    u32 tl = n >> kLogS;
    const u32 j = n & ((1u << kLogS) - 1);
    if (kShare) tl &= (1u << log_t) - 1;
    u64* const lane_b = buf + tl * Z::pitch + lds_index(j) + lds_index(g << kLogS);  // element j + e * S
    u64* const lane_c = buf + tl * Z::pitch + lds_index(j << 4) + g;  // group kk = j: (kk << 4) + e
    const u32 pieces = log_t + kPer > kShare ? 1u << (log_t + kPer - kShare) : 1;
    auto at = [&](u32 q) -> u32 {  // piece q: its first transform, its place in it
        q = q < pieces ? q : 0;
        return ((q >> kPer) << kShare) * Z::pitch + lds_index((q & ((1u << kPer) - 1)) << 8);
    };
    const u32 q0 = wave_index();
    u64 f[4];
    pass_twiddles<Z::rB, kLogS>(f, j, g, r4096);
    if constexpr (Z::rB == 4) {
        u64 x[4];
        if (q0 < pieces) lds_get<4>(lane_b + at(q0), x);
#pragma unroll 1
        for (u32 q = q0; q < pieces; q += Z::kWaves) {
            const u32 o = at(q);
            u64 x2[4];
            dft16(M, J, x);
            gl::mul_n(x, x, f);
            lds_put<4>(lane_b + o, x);
            wave_handoff();
            lds_get<0>(lane_c + o, x);
            lds_get<4>(lane_b + at(q + Z::kWaves), x2);
            dft16(M, J, x);
            wave_handoff();
            lds_put<4>(lane_b + o, x);  // result kk + 16 e, kk = j
#pragma unroll
            for (int v = 0; v < 4; v++) x[v] = x2[v];
        }
    } else {
#pragma unroll 1
        for (u32 q = q0; q < pieces; q += Z::kWaves) {
            u64* p = lane_b + at(q);
            u64 x[4];
            lds_get<kLogS>(p, x);
            dft16(M, J, x);
            gl::mul_n(x, x, f);
            lds_put<kLogS>(p, x);
        }
        M = load_matrix(mats + 3 * kDftWords, starts4);
        wave_handoff();
#pragma unroll 1
        for (u32 q = q0; q < pieces; q += Z::kWaves) {
            u64 x[4];
            lds_get<0>(lane_c + at(q), x);
            dft16(M, J, x);
            wave_handoff();
            lds_put<kLogS>(lane_b + at(q), x);  // result kk + S * e, kk = j
        }
    }
}

// The accumulator starts to LDS, the matrix of the first pass to registers.
template <class Z>
__device__ __forceinline__ Matrix dft_start(u64* buf, const u32* mats) {
    constexpr u32 r1 = Z::rA ? Z::rA : Z::rB;
    u32* const starts = (u32*)(buf + Z::kStarts);  // of r1 bits, of 4 bits
    if (threadIdx.x < 128)
        starts[threadIdx.x] = (mats + (threadIdx.x < 64 ? r1 - 1 : 3) * kDftWords + kDftStarts)[threadIdx.x & 63];
    return load_matrix(mats + (r1 - 1) * kDftWords, starts);
}
// The first 2^log_t transforms of the block's LDS (elements at lds_index(i), in
// natural order).  M as dft_start left it; it is the same
// afterwards where all passes have 4 bits.  Starts with a barrier, ends without one.
template <class Z>
__device__ __forceinline__ void dft_passes(u64* buf, u32 log_t, Matrix& M, const u32* mats,
                                           const u64* __restrict__ r4096) {
    const gl::JoinConsts J = gl::join_consts();
    const u32* const starts4 = (const u32*)(buf + Z::kStarts) + 64;
    lds_barrier();
    if constexpr (Z::rA != 0) {
        dft_pass_a<Z>(buf, log_t, M, J, r4096);
        if constexpr (Z::rA != 4) M = load_matrix(mats + 3 * kDftWords, starts4);
        lds_barrier();
    }
    dft_pieces<Z>(buf, log_t, M, mats, starts4, J, r4096);
}
template <class Z>
__device__ __forceinline__ void dft_block(u64* buf, u32 log_t, const u32* mats,
                                          const u64* __restrict__ r4096) {
    Matrix M = dft_start<Z>(buf, mats);
    dft_passes<Z>(buf, log_t, M, mats, r4096);
}

// Whether a tile of whole columns that is not full (few columns) takes its passes over
// those that exist: up to 2^8 elements (2^5 x 1, one coset: 9.6 us, 13.5 with passes over
// all 128).  Longer ones are few to a tile, and a fixed count serves them better (2^10
// x 379, four cosets: the commit 137 us, 138.5 with a count at run time).
template <class Z>
constexpr bool part_tile() { return Z::rA == 0; }

// Elements tid + q * kThreads of the tile (q < 16): transform and index, the
// thread's part (t, i) and the part of q (tq, iq), which share no bit.  TF
// (transform-fastest): adjacent threads take adjacent transforms.
template <class Z, bool TF>
struct Tile {
    u32 t, i;
    __device__ __forceinline__ Tile()
        : t(TF ? threadIdx.x & (Z::NT - 1) : threadIdx.x >> (LOGL())),
          i(TF ? threadIdx.x >> Z::logNT : threadIdx.x & (Z::L - 1)) {}
    static constexpr u32 LOGL() { return Z::logP + Z::rA; }
    static constexpr u32 tq(u32 q) { return TF ? 0 : (q * Z::kThreads) >> LOGL(); }
    static constexpr u32 iq(u32 q) {
        return TF ? (q * Z::kThreads) >> Z::logNT : (q * Z::kThreads) & (Z::L - 1);
    }
};

// Global to LDS; scale(t, tq, i, iq, x) changes four elements i + iq[v] of
// transforms t + tq[v] on the way.  valid: transforms of the tile that exist.
// log_e: transforms e*C + u of each run of C * 2^log_e, C = 2^log_c, change places
// to u * 2^log_e + e (TF).
struct Unscaled {
    __device__ __forceinline__ void operator()(u32, const u32 (&)[4], u32, const u32 (&)[4], u64 (&)[4]) const {}
};
template <class Z, bool TF, class Scale>
__device__ __forceinline__ void load_tile(u64* buf, const Place<const u64>& from, u32 valid,
                                          const Scale& scale, u32 log_c = 0, u32 log_e = 0) {
    typedef Tile<Z, TF> Ti;
    const Ti T;
    const u32 lane_o = 8 * from.off(T.t, T.i);
    u64 x[Z::kPer];
    if (valid == Z::NT) {
#pragma unroll
        for (u32 q = 0; q < Z::kPer; q++)
            x[q] = load_at(from.base + from.off(Ti::tq(q), Ti::iq(q)), lane_o);
    } else {
#pragma unroll
        for (u32 q = 0; q < Z::kPer; q++) {
            x[q] = 0;
            if (T.t + Ti::tq(q) < valid)
                x[q] = load_at(from.base + from.off(Ti::tq(q), Ti::iq(q)), lane_o);
        }
    }
    const u32 c1 = (1u << log_c) - 1, e1 = (1u << log_e) - 1;
    const u32 t = (T.t & ~((1u << (log_c + log_e)) - 1)) | ((T.t & c1) << log_e) | ((T.t >> log_c) & e1);
    u64* const lane_p = buf + t * Z::pitch + lds_index(T.i);
#pragma unroll
    for (u32 q = 0; q < Z::kPer; q += 4) {
        u64 y[4] = {x[q], x[q + 1], x[q + 2], x[q + 3]};
        const u32 tq[4] = {Ti::tq(q), Ti::tq(q + 1), Ti::tq(q + 2), Ti::tq(q + 3)};
        const u32 iq[4] = {Ti::iq(q), Ti::iq(q + 1), Ti::iq(q + 2), Ti::iq(q + 3)};
        scale(T.t, tq, T.i, iq, y);
#pragma unroll
        for (u32 v = 0; v < 4; v++) lane_p[Ti::tq(q + v) * Z::pitch + lds_index(iq[v])] = y[v];
    }
}

// LDS results to global; apply(x) changes four results of the thread (elements
// 4j .. 4j + 3 in the j-th call) on the way.  Starts with the barrier after the
// last pass.
template <class Z, bool TF, class To, class Apply>
__device__ __forceinline__ void store_tile(const u64* buf, const To& to, u32 valid,
                                           const Apply& apply) {
    typedef Tile<Z, TF> Ti;
    const Ti T;
    const u32 lane_o = 8 * to.off(T.t, T.i);
    const u64* const lane_p = buf + T.t * Z::pitch + lds_index(result_place(T.i, Z::rA));
    const bool full = valid == Z::NT;
    lds_barrier();
#pragma unroll
    for (u32 q = 0; q < Z::kPer; q += 4) {
        u64 x[4];
#pragma unroll
        for (u32 v = 0; v < 4; v++)
            x[v] = lane_p[Ti::tq(q + v) * Z::pitch + lds_index(result_place(Ti::iq(q + v), Z::rA))];
        apply(x);
#pragma unroll
        for (u32 v = 0; v < 4; v++)
            if (full || T.t + Ti::tq(q + v) < valid)
                store_at(to.base + to.off(Ti::tq(q + v), Ti::iq(q + v)), lane_o, x[v]);
    }
}

// Factors f * s^q of the thread's elements q, four at a time.
struct FactorChain {
    u64 f[4], s4;
    __device__ __forceinline__ FactorChain(u64 f0, u64 s) {
        const u64 s2 = gl::mul_lazy(s, s);
        s4 = gl::mul_lazy(s2, s2);
        f[0] = f0;
        f[1] = gl::mul_lazy(f0, s);
        f[2] = gl::mul_lazy(f0, s2);
        f[3] = gl::mul_lazy(f[1], s2);
    }
    __device__ __forceinline__ void apply(u64 (&x)[4]) {
        const u64 s[4] = {s4, s4, s4, s4};
        gl::mul_n(x, x, f);
        gl::mul_n(f, f, s);
    }
};

// w_N^(+-x) from the two-level 2^24 tables
__device__ __forceinline__ u64 twiddle(const Roots& rt, int dir, u32 x, u32 logN) {
    const u32 y = (x << (kMaxLogN - logN)) & ((1u << kMaxLogN) - 1);
    return gl::mul_lazy(load_at(rt.lo[dir], (y & 4095) * 8), load_at(rt.hi[dir], (y >> 12) * 8));
}

// Per-block segment lookup for multi-table launches: start[i] is the first
// block of segment i (start[nseg] = total blocks); returns the segment of blk.
__device__ __forceinline__ u32 find_segment(const u32* __restrict__ start, u32 nseg, u32 blk) {
    u32 lo = 0, hi = nseg;  // invariant: start[lo] <= blk < start[hi]
    while (hi - lo > 1) {
        u32 mid = (lo + hi) >> 1;
        if (start[mid] <= blk) lo = mid;
        else hi = mid;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// Blocks go to the eight XCDs in turn, each with its own L2.  Of `blocks` blocks,
// 2^lb to a column, the one that XCD x = blk mod 8 runs in turn: a column's blocks
// follow each other on one XCD, the same in every step.  So the cache lines that
// several of them write in part are completed in one L2, and what a step leaves
// in an L2 the next one reads there (NTT 2^20 x 379, rows stored in 32 B runs: 4.5 ->
// 3.9 ms; 2^14 x 60: 20.8 -> 19.0 us.  The LDE's steps, all of which write whole
// lines, gain nothing).
__device__ __forceinline__ u64 column_on_xcd(u32 blk, u32 blocks, u32 lb) {
    const u32 full = (blocks >> (lb + 3)) << (lb + 3);  // of whole groups of eight columns
    if (blk >= full) return blk;
    const u32 y = blk >> 3;
    return ((((y >> lb) << 3) + (blk & 7)) << lb) + (y & ((1u << lb) - 1));
}

// Where a block's transforms are: transform t0 + t of column c, `valid` of them.
// A column of 2^log_per transforms takes max(1, 2^log_per / NT) blocks, so blocks
// never span columns; where every column is a single transform (log_per = 0,
// `flat`), a block takes NT columns.  In-block offsets stay below 2^31 bytes.
struct BlockPlace {
    u64 c;
    u32 t0, valid;
};
// blocks: of a launch whose columns go by XCD, or 0.
__device__ __forceinline__ BlockPlace block_place(u64 blk, u32 log_nt, u32 log_per, u64 cols, bool flat,
                                                  u32 blocks = 0) {
    BlockPlace B;
    if (flat) {
        B.c = blk << log_nt;
        B.t0 = 0;
        B.valid = cols - B.c < (1ull << log_nt) ? (u32)(cols - B.c) : 1u << log_nt;
        return B;
    }
    const u32 lb = log_per > log_nt ? log_per - log_nt : 0;  // log2 blocks of a column
    if (blocks) blk = column_on_xcd((u32)blk, blocks, lb);
    B.c = blk >> lb;
    B.t0 = ((u32)blk & ((1u << lb) - 1)) << log_nt;
    B.valid = 1u << (log_per < log_nt ? log_per : log_nt);
    return B;
}

// Transforms of length 2^logL <= 16: one product, no LDS; 16 / L transforms make a
// group of the matrix product.  A block takes 2^(10 - logL) transforms, a product to
// a wave, `valid` of which exist.  body(t, i) handles elements (t[v], i[v]), v < 4, of
// the lane; results have the same indices.
constexpr u32 kSmallTile = 10, kSmallThreads = 256;
template <class Body>
__device__ __forceinline__ void small_groups(u32 logL, u32 valid, const Body& body) {
    const u32 g = (threadIdx.x & 63) >> 4, n = threadIdx.x & 15, sub = 4 - logL;
    if ((wave_index() * 16) << sub >= valid) return;
    u32 t[4], i[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const u32 e = 4 * v + g;
        t[v] = ((wave_index() * 16 + n) << sub) + (e & ((1u << sub) - 1));
        i[v] = e >> sub;
    }
    body(t, i);
}
// The small DFT of 2^logL points (none for one point).
__device__ __forceinline__ void small_dft(u32 logL, const u32* mats, const gl::JoinConsts& J, u64 (&x)[4]) {
    if (!logL) return;
    const u32* set = mats + (logL - 1) * kDftWords;
    const Matrix M = load_matrix(set, set + kDftStarts);
    dft16(M, J, x);
}

// ---------------------------------------------------------------- step 1
// Transforms n2 of column c, element n1 at src[c*sstride + N2*n1 + n2]; DFT over
// n1 (inverse if INV) -> k1; times w_N^(+-n2*k1) and the constant A.factor; to
// dst[c*dstride + E*N2*k1 + n2].  Adjacent lanes take adjacent transforms
// (adjacent n2: contiguous in HBM).
// SCALED (forward): element i = (n1 << b) + n2 of column c enters as
// (x + [i < k] rand[c*k + i] * delta) * base^i, base^i = p1[n1] * p2[n2]: p1 on
// the way in, p2 (the same for a whole transform) with the output factor, in
// place of a separate read-and-write pass over the table.
template <bool INV, bool SCALED>
struct Step1 {
    const Step1Args& A;
    const NttScaleDev& S;
    const Roots& rt;
    BlockPlace B;
    Place<const u64> in;
    Place<u64> out;
    __device__ __forceinline__ Step1(const Step1Args& A_, const NttScaleDev& S_, const Roots& rt_,
                                     u64 blk, u32 log_nt)
        : A(A_), S(S_), rt(rt_) {
        const u32 b = A.logN - A.a;
        B = block_place(blk, log_nt, b, 0, false, A.by_xcd);
        in = {A.src + B.c * A.sstride + B.t0, 0, 1, 0, 1u << b};
        out = {A.dst + B.c * A.dstride + B.t0, 0, 1, 0, A.E << b};
    }
    __device__ __forceinline__ void scale(u32 t, u32 i, const u32 (&iq)[4], u64 (&x)[4]) const {
        u64 f[4];
#pragma unroll
        for (int v = 0; v < 4; v++) f[v] = load_at(S.p1 + iq[v], i * 8);
        if (S.k) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const u64 pos = ((u64)(iq[v] + i) << (A.logN - A.a)) + B.t0 + t;
                if (pos < S.k)
                    x[v] = gl::add(x[v], gl::mul(S.rand[B.c * S.k + pos], S.delta));
            }
        }
        gl::mul_n(x, x, f);
    }
    __device__ __forceinline__ u64 constant(u32 t) const {  // of transform t's results
        u64 f = A.factor;
        if (SCALED) f = gl::mul_lazy(f, S.p2[(B.t0 + t) & ((1u << (A.logN - A.a)) - 1)]);
        return f;
    }
};
template <bool INV, bool SCALED, int LT, int LOGL>
__device__ __forceinline__ void step1_body(const Step1Args& A, const NttScaleDev& S, u64 blk,
                                           const Roots& rt) {
    extern __shared__ u64 lds[];
    typedef Shape<LT, LOGL> Z;
    const Step1<INV, SCALED> P(A, S, rt, blk, Z::logNT);
    load_tile<Z, true>(lds, P.in, P.B.valid,
                       [&](u32 t, const u32 (&)[4], u32 i, const u32 (&iq)[4], u64 (&x)[4]) {
                           if constexpr (SCALED) P.scale(t, i, iq, x);
                       });
    dft_block<Z>(lds, Z::logNT, rt.dft[INV], rt.r4096[INV]);
    // the thread's results are k = k0 + q * L/16 of one transform
    const Tile<Z, true> T;
    const u32 n2 = P.B.t0 + T.t;
    FactorChain F(gl::mul_lazy(P.constant(T.t), twiddle(rt, INV, n2 * T.i, A.logN)),
                  twiddle(rt, INV, n2 * (Z::L / 16), A.logN));
    store_tile<Z, true>(lds, P.out, P.B.valid, [&](u64 (&x)[4]) { F.apply(x); });
}

// ---------------------------------------------------------------- LDE step 2
// Randomizer r of column c (null: its limb carries none).
__device__ __forceinline__ const u64* rand_at(const RandSpec& rs, u64 c, u64 r) {
    u32 limb = (u32)(c % rs.group);
    if (!((rs.limb_mask >> limb) & 1)) return nullptr;
    return rs.ptr + (c / rs.group) * rs.group_stride + limb * rs.limb_stride + r * rs.elem_stride;
}
// delta_n[s] without a dynamic index (which would copy the by-value kernel argument
// to scratch).  Randomizer r adds *rand_at * rand_delta * o^r to its coefficient.
__device__ __forceinline__ u64 rand_delta(const LdeArgs& A, u32 s) {
    u64 d = A.delta_n[0];
#pragma unroll
    for (u32 i = 1; i < 16; i++)
        if (s == i) d = A.delta_n[i];
    return d;
}

// A block takes NT rows (c, k1) (NT * E * N2 = 2^LT) of Y: inverse row DFT to
// coefficients, which stay in LDS, then all E coset transforms of each row;
// output u1 of coset sl, times N^-1 beta_sl^k1 w_N^(k1*u1), to
// out[c*M + E*N2*k1 + E*u1 + sl].  Coefficient k2 enters coset sl as (C +
// randomizer term) * beta_sl^(N1*k2).  Transforms T = t*E + sl: cosets are the
// fastest index, so the E cosets of one output position are stored by adjacent
// lanes.  The outputs overwrite the row in place (its reads all precede the
// block's first barrier, its writes follow its last one).
struct Rows {
    const LdeArgs& A;
    BlockPlace B;
    Place<const u64> in;
    Place<u64> out;
    __device__ __forceinline__ Rows(const LdeArgs& A_, u64 blk, u32 log_nt) : A(A_) {
        const u32 a = A.a, row = A.E << (A.logN - a);  // (a = 0: M = E*N2)
        B = block_place(blk, log_nt, a, A.cols, a == 0);
        in = {A.src + B.c * A.src_col_stride + B.t0 * A.src_row_stride, 0,
              (u32)(a ? A.src_row_stride : A.src_col_stride), 0, 1};
        out = {A.out + B.c * A.M + (u64)B.t0 * row, A.logE, row, 1, A.E};
    }
    // k1 of row t (a column of its own: 0)
    __device__ __forceinline__ u32 k1(u32 t) const { return A.a ? B.t0 + t : 0; }
    // randomizer term of element k2 of row t in coset sl (canonical): the element is
    // coefficient k1 + k2 * N1, which carries one when below rand_len
    __device__ __forceinline__ u64 rand_term(u32 t, u32 sl, u32 k2) const {
        const u64 r = k1(t) + ((u64)k2 << A.a);
        if (r >= A.rs.k) return 0;
        const u64* p = rand_at(A.rs, A.a ? B.c : B.c + t, r);
        return p ? gl::mul(gl::mul(*p, rand_delta(A, sl)), gl::pow(A.toff, r)) : 0;
    }
    // The randomizer terms of the scaled coefficients of the block's rows in cosets
    // s0 .. s0 + 2^log_s - 1 in LDS (transform t * 2^log_s + s): the few elements
    // that carry one, spread over the block (a term is ~20 dependent products, which
    // would hold up the block in the one wave that has them: 2^16 x 156 with 98
    // randomizers, 0.57 against 0.43 ms), and over the rows that exist (2^7 x 1 with
    // 98, a tile of 32 rows: 47 us with all of them, 15 with one).
    template <class Z>
    __device__ __forceinline__ void add_randomizers(u64* lds, u32 logL, u32 s0, u32 log_s) const {
        const u64 first = A.a ? B.t0 : 0;  // the smallest coefficient index
        if (first >= A.rs.k) return;
        lds_barrier();
        const u64 per = ((A.rs.k - 1 - first) >> A.a) + 1;
        const u32 n = per < Z::L ? (u32)per : Z::L, log_rows = log_ceil(B.valid);
#pragma unroll 1
        for (u32 e = threadIdx.x; e < n << (log_rows + log_s); e += Z::kThreads) {
            const u32 s = e & ((1u << log_s) - 1), t = (e >> log_s) & ((1u << log_rows) - 1);
            const u32 k2 = e >> (log_s + log_rows);
            if (t >= B.valid) continue;
            u64* const p = lds + ((t << log_s) + s) * Z::pitch + lds_index(k2);
            *p = gl::add(gl::canon(*p),
                         gl::mul(rand_term(t, s0 + s, k2), A.pb[((s0 + s) << logL) + k2]));
        }
    }
};
template <int LT, int LOGL>
__device__ __forceinline__ void lde_rows_body(const LdeArgs& A, u64 blk, const Roots& rt) {
    extern __shared__ u64 lds[];
    typedef Shape<LT, LOGL> Z;  // the E * NT coset transforms
    typedef Tile<Z, false> Ti;  // of the rows: elements q < 16 / E
    const Rows P(A, blk, Z::logNT - A.logE);
    const Ti T;
    {
        const u32 lane_o = 8 * P.in.off(T.t, T.i);
        u64 x[16];
#pragma unroll
        for (u32 q = 0; q < 16; q++)
            if ((q << A.logE) < 16) {
                x[q] = 0;
                if (T.t + Ti::tq(q) < P.B.valid)
                    x[q] = load_at(P.in.base + P.in.off(Ti::tq(q), Ti::iq(q)), lane_o);
            }
        u64* const lane_p = lds + T.t * Z::pitch + lds_index(T.i);
#pragma unroll
        for (u32 q = 0; q < 16; q++)
            if ((q << A.logE) < 16 && T.t + Ti::tq(q) < Z::NT >> A.logE)
                lane_p[Ti::tq(q) * Z::pitch + lds_index(Ti::iq(q))] = x[q];
    }
    const u32 log_rows = part_tile<Z>() ? log_ceil(P.B.valid) : Z::logNT - A.logE;
    dft_block<Z>(lds, log_rows, rt.dft[1], rt.r4096[1]);
    // coefficients to registers, then to every coset's transform: product j of
    // the thread is element q = j / E in coset j mod E
    {
        u64 f[16], x[16];
#pragma unroll
        for (u32 j = 0; j < 16; j++) {
            const u32 q = j >> A.logE, sl = j & (A.E - 1);
            f[j] = load_at(A.pb + (sl << LOGL) + Ti::iq(q), T.i * 8);
        }
        lds_barrier();
        const u64* const lane_p = lds + T.t * Z::pitch + lds_index(result_place(T.i, Z::rA));
#pragma unroll
        for (u32 j = 0; j < 16; j++) {
            const u32 q = j >> A.logE;
            x[j] = lane_p[Ti::tq(q) * Z::pitch + lds_index(result_place(Ti::iq(q), Z::rA))];
        }
        lds_barrier();
        u64* const to = lds + (T.t << A.logE) * Z::pitch + lds_index(T.i);
#pragma unroll
        for (u32 j = 0; j < 16; j += 4) {
            u64 y[4] = {x[j], x[j + 1], x[j + 2], x[j + 3]};
            const u64 fj[4] = {f[j], f[j + 1], f[j + 2], f[j + 3]};
            gl::mul_n(y, y, fj);
#pragma unroll
            for (u32 v = 0; v < 4; v++) {
                const u32 q = (j + v) >> A.logE, sl = (j + v) & (A.E - 1);
                to[((Ti::tq(q) << A.logE) + sl) * Z::pitch + lds_index(Ti::iq(q))] = y[v];
            }
        }
    }
    P.template add_randomizers<Z>(lds, LOGL, 0, A.logE);
    dft_block<Z>(lds, part_tile<Z>() ? log_rows + A.logE : Z::logNT, rt.dft[0], rt.r4096[0]);
    // the thread's results are u1 = u0 + q * N2/16 of transform T: the factor
    // advances by w_N^(k1 * N2/16)
    const Tile<Z, true> U;
    const u32 k1 = P.k1(U.t >> A.logE);
    const u32 valid = P.B.valid << A.logE;
    u64 f0 = A.pa[((U.t & (A.E - 1)) << A.a) + (k1 & ((1u << A.a) - 1))];
    if (A.a) {
        FactorChain F(gl::mul_lazy(f0, twiddle(rt, 0, k1 * U.i, A.logN)),
                      twiddle(rt, 0, k1 * (Z::L / 16), A.logN));
        store_tile<Z, true>(lds, P.out, valid, [&](u64 (&x)[4]) { F.apply(x); });
    } else {  // a whole transform per row: no step-1 twiddle, and the codewords
        const u64 f[4] = {f0, f0, f0, f0};
        store_tile<Z, true>(lds, P.out, valid, [&](u64 (&x)[4]) {
            gl::mul_n(x, x, f);
            gl::canon_n(x);
        });
    }
}
// Rows of 2^12 elements: the E coset transforms one after the other, in a tile of
// one transform, from coefficients that wait in LDS.  A block is 8 waves and 70 KB,
// so a CU has two, each at a different place of its work (one tile of 2^14 for four
// cosets is one block of 16 waves, which all meet at every barrier and load
// together).  Output u1 of coset s goes to place (u1 / C) * C*E + s*C + u1 mod C of
// its row, C = 2^log_c: runs of C elements where E*u1 + s would leave gaps of E;
// step 3 puts them in order.
struct CosetPlace {
    u64* base;
    u32 row, log_c, log_e;
    __device__ __forceinline__ u32 off(u32 t, u32 i) const {
        return t * row + ((i >> log_c) << (log_c + log_e)) + (i & ((1u << log_c) - 1));
    }
};
constexpr u32 kCosetsLt = 12, kCosetsThreads = 512;
__device__ __forceinline__ void lde_cosets_body(const LdeArgs& A, u64 blk, const Roots& rt) {
    extern __shared__ u64 lds[];
    typedef Shape<kCosetsLt, kCosetsLt, 3> Z;
    typedef Tile<Z, false> Ti;
    const Rows P(A, blk, Z::logNT);
    const Ti T;
    load_tile<Z, false>(lds, P.in, Z::NT, Unscaled{});
    dft_block<Z>(lds, Z::logNT, rt.dft[1], rt.r4096[1]);
    u64 f[Z::kPer];
    auto factors = [&](u32 s) {
#pragma unroll
        for (u32 q = 0; q < Z::kPer; q++) f[q] = load_at(A.pb + (s << kCosetsLt) + Ti::iq(q), T.i * 8);
    };
    factors(0);
    lds_barrier();
    const u64* const from = lds + T.t * Z::pitch + lds_index(result_place(T.i, Z::rA));
    u64* const coef = lds + Z::kStarts + 64 + threadIdx.x;  // the thread's own
    u64* const to = lds + T.t * Z::pitch + lds_index(T.i);
#pragma unroll
    for (u32 q = 0; q < Z::kPer; q++)
        coef[q * Z::kThreads] = from[Ti::tq(q) * Z::pitch + lds_index(result_place(Ti::iq(q), Z::rA))];
    const Tile<Z, true> U;
    const u32 k1 = P.k1(U.t);
    const u64 w0 = twiddle(rt, 0, k1 * U.i, A.logN), ws = twiddle(rt, 0, k1 * (Z::kThreads >> Z::logNT), A.logN);
    CosetPlace out{P.out.base, P.out.ts, A.log_c, A.logE};
    Matrix M = dft_start<Z>(lds, rt.dft[0]);
#pragma unroll 1
    for (u32 s = 0; s < A.E; s++) {
        lds_barrier();
#pragma unroll
        for (u32 q = 0; q < Z::kPer; q += 4) {
            u64 y[4];
#pragma unroll
            for (u32 v = 0; v < 4; v++) y[v] = coef[(q + v) * Z::kThreads];
            const u64 fq[4] = {f[q], f[q + 1], f[q + 2], f[q + 3]};
            gl::mul_n(y, y, fq);
#pragma unroll
            for (u32 v = 0; v < 4; v++) to[Ti::tq(q + v) * Z::pitch + lds_index(Ti::iq(q + v))] = y[v];
        }
        P.template add_randomizers<Z>(lds, kCosetsLt, s, 0);
        // (opaque: no twiddle is kept in registers from one coset to the next)
        const u64* r4096 = rt.r4096[0];
        asm("" : "+s"(r4096) : "s"(s));
        dft_passes<Z>(lds, Z::logNT, M, rt.dft[0], r4096);
        factors(s + 1 < A.E ? s + 1 : 0);
        FactorChain F(gl::mul_lazy(A.pa[(s << A.a) + k1], w0), ws);
        store_tile<Z, true>(lds, out, Z::NT, [&](u64 (&v)[4]) { F.apply(v); });
        out.base += 1u << A.log_c;
    }
}
// Columns of N <= 16 elements, E * N outputs each (no column step).  One matrix
// product takes 256 outputs, which are whole columns and lie together: its transforms
// are all cosets of 256 / (E N) columns, cosets fastest, each with the column's
// inverse transform of its own (the cosets one after the other in a lane cost their
// latency each: 2^4 rows in 16 cosets took 75 us, here they take 4).  What
// depends on coset and element alone is the lane's for the whole kernel.  The
// outputs go through LDS to be stored in order.  A wave takes A.products of them.
constexpr u32 kShortThreads = 256, kShortOut = 256, kShortPitch = kShortOut + kShortOut / 16;
constexpr u32 kShortLds = (kShortThreads / 64 * kShortPitch + 64) * 8;  // outputs; starts of both matrices
__device__ __forceinline__ void lde_short_body(const LdeArgs& A, u64 blk, const Roots& rt) {
    extern __shared__ u64 lds[];
    const u32 logN = A.logN, sub = 4 - logN;
    const u32 lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    constexpr u32 kWaves = kShortThreads / 64;
    u32* const starts = (u32*)(lds + kWaves * kShortPitch);
    const u32 set = (logN ? logN - 1 : 0) * kDftWords;  // (N = 1: no product)
    if (threadIdx.x < 128)
        starts[threadIdx.x] = (rt.dft[threadIdx.x < 64] + set + kDftStarts)[threadIdx.x & 63];
    const Matrix inv = load_matrix(rt.dft[1] + set, starts), fwd = load_matrix(rt.dft[0] + set, starts + 64);
    const gl::JoinConsts J = gl::join_consts();
    // element i of transform q, in column t of the product's, coset s
    u32 t[4], from[4], to[4];
    u64 pb[4], pa[4], rf[4];
#pragma unroll
    for (u32 v = 0; v < 4; v++) {
        const u32 e = 4 * v + g, q = (n << sub) + (e & ((1u << sub) - 1)), i = e >> sub;
        const u32 s = q & (A.E - 1), o = (((q >> A.logE) << logN) + i) * A.E + s;
        t[v] = q >> A.logE;
        from[v] = ((t[v] << logN) + i) * 8;
        to[v] = o + (o >> 4);
        pb[v] = load_at(A.pb, ((s << logN) + i) * 8);
        pa[v] = load_at(A.pa, s * 8);
        rf[v] = i < A.rs.k ? gl::mul(rand_delta(A, s), gl::pow(A.toff, i)) : 0;
    }
    u64* const buf = lds + wave_index() * kShortPitch;
    const u32 log_cols = 8 - logN - A.logE;  // columns of a product
    __syncthreads();
#pragma unroll 1
    for (u32 j = 0; j < A.products; j++) {
        const u64 p = (blk * A.products + j) * kWaves + wave_index(), c0 = p << log_cols;
        if (c0 >= A.cols) break;
        const u32 valid = A.cols - c0 < 1u << log_cols ? (u32)(A.cols - c0) : 1u << log_cols;
        u64 x[4];
#pragma unroll
        for (u32 v = 0; v < 4; v++) x[v] = t[v] < valid ? load_at(A.src + (c0 << logN), from[v]) : 0;
        if (logN) dft16(inv, J, x);
        if (A.rs.k) {
#pragma unroll
            for (u32 v = 0; v < 4; v++) {
                const u32 i = (4 * v + g) >> sub;
                if (i >= A.rs.k || t[v] >= valid) continue;
                const u64* r = rand_at(A.rs, c0 + t[v], i);
                if (r) x[v] = gl::add(gl::canon(x[v]), gl::mul(*r, rf[v]));
            }
        }
        gl::mul_n(x, x, pb);
        if (logN) dft16(fwd, J, x);
        gl::mul_n(x, x, pa);
        gl::canon_n(x);
#pragma unroll
        for (u32 v = 0; v < 4; v++) buf[to[v]] = x[v];
        wave_handoff();
#pragma unroll
        for (u32 v = 0; v < 4; v++) {
            const u32 o = 64 * v + lane;
            if (o >> (logN + A.logE) < valid) store_at(A.out + p * kShortOut, o * 8, buf[o + (o >> 4)]);
        }
        wave_handoff();
    }
}

// ---------------------------------------------------------------- LDE step 3
// Transforms q = u1*E + s of column c, element k1 at out[c*M + E*N2*k1 + q];
// forward DFT over k1 -> u2, written back to out[c*M + E*N2*u2 + q] (codewords).
template <int LT, int LOGL>
__device__ __forceinline__ void lde_step3_body(const Step3Args& A, u64 blk, const Roots& rt) {
    extern __shared__ u64 lds[];
    typedef Shape<LT, LOGL> Z;
    const u32 logQ = A.logN - A.a + A.logE;  // transforms per column = E*N2
    const BlockPlace B = block_place(blk, Z::logNT, logQ, 0, false);
    u64* col = A.out + B.c * A.M + B.t0;
    // every input of the block is read before any output is written
    load_tile<Z, true>(lds, Place<const u64>{col, 0, 1, 0, 1u << logQ}, B.valid,
                       Unscaled{}, A.log_c, A.log_c ? A.logE : 0);
    dft_block<Z>(lds, Z::logNT, rt.dft[0], rt.r4096[0]);
    store_tile<Z, true>(lds, Place<u64>{col, 0, 1, 0, 1u << logQ}, B.valid,
                        [](u64 (&x)[4]) { gl::canon_n(x); });
}
// Lengths 2^5..2^12 by a compile-time constant: f(std::integral_constant<int, LOGL>).
template <class F>
__host__ __device__ __forceinline__ void with_length(u32 logL, const F& f) {
    switch (logL) {
        case 5: f(std::integral_constant<int, 5>{}); break;
        case 6: f(std::integral_constant<int, 6>{}); break;
        case 7: f(std::integral_constant<int, 7>{}); break;
        case 8: f(std::integral_constant<int, 8>{}); break;
        case 9: f(std::integral_constant<int, 9>{}); break;
        case 10: f(std::integral_constant<int, 10>{}); break;
        case 11: f(std::integral_constant<int, 11>{}); break;
        default: f(std::integral_constant<int, 12>{}); break;
    }
}
// Tiles of 2^12..2^14 elements likewise.
template <class F>
__host__ void with_tile(u32 lt, const F& f) {
    if (lt == 12) f(std::integral_constant<int, 12>{});
    else if (lt == 13) f(std::integral_constant<int, 13>{});
    else f(std::integral_constant<int, 14>{});
}
// Row tile of the NTT: without a column step 2^12, else the shortest that holds 8 rows
// of 2^logL, 2^12 to 2^14.
constexpr u32 ntt_row_tile(u32 logL, bool cols) {
    return cols || logL <= 9 ? 12 : logL == 10 ? 13 : LOG_TILE;
}
// A launch of `cols` columns of 2^log_per transforms (flat: one each, as
// block_place) of length 2^logL in tiles of 2^lt elements; 2^log_e transforms of the
// tile belong to one of a column's.
LaunchShape launch_shape(u32 lt, u32 logL, u32 log_per, u64 cols, bool flat, u32 log_e = 0);

// ---- host launchers of the kernels (one translation unit each) ----
// lt: log2 tile (12..14); blocks, threads and LDS follow from launch_shape.
// ntt_step1.hip
int launch_k_step1(bool inv, u32 lt, const LaunchShape& g, hipStream_t st, const Step1Args& A,
                   const Roots& rt);
int launch_k_step1_multi(const Step1Args* args, const u32* start, u32 nseg, u32 blocks, size_t lds,
                         hipStream_t st, const Roots& rt);
int launch_k_step1_scaled(u32 lt, const LaunchShape& g, hipStream_t st, const Step1Args& A,
                          const NttScaleDev& S, const Roots& rt);
int set_attributes_step1(int lds_bytes);
// ntt_step2.hip
int launch_k_ntt_step2(bool inv, const LaunchShape& g, hipStream_t st, const u64* src, u64* dst, u32 logN,
                       u32 a, u64 cols, u64 ninv, const Roots& rt);
int launch_k_ntt_cols_scaled(const LaunchShape& g, hipStream_t st, const u64* src, u64* dst, u32 logN,
                             u64 cols, const NttScaleDev& S, const Roots& rt);
int set_attributes_step2(int lds_bytes);
// lde_rows.hip
int launch_k_lde_rows(u32 lt, const LaunchShape& g, hipStream_t st, const LdeArgs& A, const Roots& rt);
// lt: as above, or kBatchShort
int launch_k_lde_rows_multi(u32 lt, const LdeArgs* args, const u32* start, u32 nseg, u32 blocks,
                            size_t lds, hipStream_t st, const Roots& rt);
int set_attributes_rows(int lds_bytes);
// lde_step3.hip
int launch_k_lde_step3(u32 lt, const LaunchShape& g, hipStream_t st, const Step3Args& A,
                       const Roots& rt);
int launch_k_lde_step3_multi(const Step3Args* args, const u32* start, u32 nseg, u32 blocks,
                             size_t lds, hipStream_t st, const Roots& rt);
int set_attributes_step3(int lds_bytes);

}  // namespace tvh
