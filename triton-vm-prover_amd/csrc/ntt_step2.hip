// Row step of the batched NTT: kernels and their launchers.
#include "ntt_dev.hpp"

namespace tvh {

// Rows k1 of column c, N2 = 2^b elements at src[c*N + N2*k1 + n2] (the column
// step's output); DFT over n2 -> k2; element k2 to dst[c*N + k1 + N1*k2].  The
// rows are read element-fastest and stored transform-fastest, so adjacent lanes
// write adjacent k1 (runs as long as the block's row count).  COLS: without a
// column step (a = 0) the rows are the columns, read and written alike, in place
// too, and take the factor N^-1 of an inverse transform here.
template <bool INV, bool COLS>
struct RowStep {
    BlockPlace B;
    Place<const u64> in;
    Place<u64> out;
    u64 ninv;
    __device__ __forceinline__ RowStep(const u64* src, u64* dst, u32 logN, u32 a, u64 cols, u64 ninv_,
                                       u64 blk, u32 log_nt, u32 blocks = 0)
        : ninv(ninv_) {
        const u32 b = logN - a;
        B = block_place(blk, log_nt, a, cols, COLS, blocks);
        in = {src + (B.c << logN) + ((u64)B.t0 << b), 0, 1u << b, 0, 1};
        out = {dst + (B.c << logN) + B.t0, 0, COLS ? 1u << logN : 1u, 0, 1u << a};
    }
    __device__ __forceinline__ void finish(u64 (&x)[4]) const {
        if (INV && COLS) {
            const u64 f[4] = {ninv, ninv, ninv, ninv};
            gl::mul_n(x, x, f);
        }
        gl::canon_n(x);
    }
};

template <bool INV, bool COLS, int LOGL>
__global__ void __launch_bounds__(1 << (ntt_row_tile(LOGL, COLS) - 4), 4)
    k_ntt_step2(const u64* src, u64* dst, u32 logN, u32 a, u64 cols, u64 ninv, Roots rt) {
    extern __shared__ u64 lds[];
    typedef Shape<ntt_row_tile(LOGL, COLS), LOGL> Z;
    const RowStep<INV, COLS> P(src, dst, logN, a, cols, ninv, blockIdx.x, Z::logNT, gridDim.x);
    load_tile<Z, false>(lds, P.in, P.B.valid, Unscaled{});
    dft_block<Z>(lds, COLS && part_tile<Z>() ? log_ceil(P.B.valid) : Z::logNT, rt.dft[INV], rt.r4096[INV]);
    store_tile<Z, !COLS>(lds, P.out, P.B.valid, [&](u64 (&x)[4]) { P.finish(x); });
}
// columns of at most 16 elements
template <bool INV>
__global__ void __launch_bounds__(kSmallThreads) k_ntt_step2_small(const u64* src, u64* dst, u32 logN,
                                                                   u64 cols, u64 ninv, Roots rt) {
    const RowStep<INV, true> P(src, dst, logN, 0, cols, ninv, blockIdx.x, kSmallTile - logN);
    const gl::JoinConsts J = gl::join_consts();
    small_groups(logN, P.B.valid, [&](const u32 (&t)[4], const u32 (&i)[4]) {
        u64 x[4];
#pragma unroll
        for (int v = 0; v < 4; v++) x[v] = t[v] < P.B.valid ? P.in.base[P.in.off(t[v], i[v])] : 0;
        small_dft(logN, rt.dft[INV], J, x);
        P.finish(x);
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (t[v] < P.B.valid) P.out.base[P.out.off(t[v], i[v])] = x[v];
    });
}

// Whole transforms of a column each, forward, of a scaled input: element i of
// column c enters as (x + [i < k] rand[c*k + i] * delta) * base^i, base^i = p2[i]
// (NttScaleDev, N1 = 1).  Blocks take as many columns as a tile holds: with the
// column and row steps of longer transforms a block has one column alone, and 2^21
// columns of 4 rows took 9.4 ms.
struct ScaledCols {
    const NttScaleDev& S;
    RowStep<false, true> P;
    __device__ __forceinline__ ScaledCols(const u64* src, u64* dst, u32 logN, u64 cols, const NttScaleDev& S_,
                                          u64 blk, u32 log_nt)
        : S(S_), P(src, dst, logN, 0, cols, 1, blk, log_nt) {}
    __device__ __forceinline__ void scale(u32 t, const u32 (&tq)[4], u32 i, const u32 (&iq)[4],
                                          u64 (&x)[4]) const {
        u64 f[4];
#pragma unroll
        for (int v = 0; v < 4; v++) f[v] = load_at(S.p2 + iq[v], i * 8);
        if (S.k) {
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (iq[v] + i < S.k && t + tq[v] < P.B.valid)
                    x[v] = gl::add(x[v], gl::mul(S.rand[(P.B.c + t + tq[v]) * S.k + iq[v] + i], S.delta));
        }
        gl::mul_n(x, x, f);
    }
};
template <int LOGL>
__global__ void __launch_bounds__(1 << 8, 4) k_ntt_cols_scaled(const u64* src, u64* dst, u64 cols,
                                                               NttScaleDev S, Roots rt) {
    extern __shared__ u64 lds[];
    typedef Shape<12, LOGL> Z;
    const ScaledCols C(src, dst, LOGL, cols, S, blockIdx.x, Z::logNT);
    load_tile<Z, false>(lds, C.P.in, C.P.B.valid,
                        [&](u32 t, const u32 (&tq)[4], u32 i, const u32 (&iq)[4], u64 (&x)[4]) {
                            C.scale(t, tq, i, iq, x);
                        });
    dft_block<Z>(lds, part_tile<Z>() ? log_ceil(C.P.B.valid) : Z::logNT, rt.dft[0], rt.r4096[0]);
    store_tile<Z, false>(lds, C.P.out, C.P.B.valid, [&](u64 (&x)[4]) { C.P.finish(x); });
}
// columns of at most 16 elements
__global__ void __launch_bounds__(kSmallThreads) k_ntt_cols_scaled_small(const u64* src, u64* dst, u32 logN,
                                                                         u64 cols, NttScaleDev S, Roots rt) {
    const ScaledCols C(src, dst, logN, cols, S, blockIdx.x, kSmallTile - logN);
    const gl::JoinConsts J = gl::join_consts();
    small_groups(logN, C.P.B.valid, [&](const u32 (&t)[4], const u32 (&i)[4]) {
        u64 x[4];
#pragma unroll
        for (int v = 0; v < 4; v++) x[v] = t[v] < C.P.B.valid ? C.P.in.base[C.P.in.off(t[v], i[v])] : 0;
        C.scale(0, t, 0, i, x);
        small_dft(logN, rt.dft[0], J, x);
        C.P.finish(x);
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (t[v] < C.P.B.valid) C.P.out.base[C.P.out.off(t[v], i[v])] = x[v];
    });
}

int launch_k_ntt_cols_scaled(const LaunchShape& g, hipStream_t st, const u64* src, u64* dst, u32 logN,
                             u64 cols, const NttScaleDev& S, const Roots& rt) {
    const dim3 blocks(g.blocks), tpb(g.threads);
    if (logN <= 4)
        hipLaunchKernelGGL(k_ntt_cols_scaled_small, blocks, tpb, 0, st, src, dst, logN, cols, S, rt);
    else
        with_length(logN, [&](auto l) {
            hipLaunchKernelGGL(k_ntt_cols_scaled<decltype(l)::value>, blocks, tpb, g.lds, st, src, dst, cols,
                               S, rt);
        });
    return check_launch();
}

// Rows after a column step have 2^7 elements and more (launch_ntt_batched).
template <bool COLS, int LOGL>
constexpr bool kRowShape = COLS || LOGL >= 7;

template <bool INV, bool COLS>
static int launch_step2(const LaunchShape& g, hipStream_t st, const u64* src, u64* dst, u32 logN, u32 a,
                        u64 cols, u64 ninv, const Roots& rt) {
    const dim3 blocks(g.blocks), tpb(g.threads);
    bool done = false;
    if (COLS && logN <= 4) {
        hipLaunchKernelGGL(k_ntt_step2_small<INV>, blocks, tpb, 0, st, src, dst, logN, cols, ninv, rt);
        return check_launch();
    }
    with_length(logN - a, [&](auto l) {
        constexpr int L = decltype(l)::value;
        if constexpr (kRowShape<COLS, L>) {
            hipLaunchKernelGGL((k_ntt_step2<INV, COLS, L>), blocks, tpb, g.lds, st, src, dst, logN, a, cols,
                               ninv, rt);
            done = true;
        }
    });
    return done ? check_launch() : set_error(TVH_ERR_UNSUPPORTED, "row step of 2^%u", logN - a);
}

int launch_k_ntt_step2(bool inv, const LaunchShape& g, hipStream_t st, const u64* src, u64* dst, u32 logN,
                       u32 a, u64 cols, u64 ninv, const Roots& rt) {
    if (a == 0)
        return inv ? launch_step2<true, true>(g, st, src, dst, logN, a, cols, ninv, rt)
                   : launch_step2<false, true>(g, st, src, dst, logN, a, cols, ninv, rt);
    return inv ? launch_step2<true, false>(g, st, src, dst, logN, a, cols, ninv, rt)
               : launch_step2<false, false>(g, st, src, dst, logN, a, cols, ninv, rt);
}

// (2^12 tiles need no more LDS than every kernel has)
int set_attributes_step2(int bytes) {
    std::vector<const void*> fns;
    for (u32 l = 5; l <= 12; l++)
        with_length(l, [&](auto c) {
            constexpr int L = decltype(c)::value;
            if constexpr (ntt_row_tile(L, false) > 12)
                fns.insert(fns.end(), {(const void*)k_ntt_step2<true, false, L>,
                                       (const void*)k_ntt_step2<false, false, L>});
        });
    return set_lds_attribute(fns, bytes);
}

}  // namespace tvh
