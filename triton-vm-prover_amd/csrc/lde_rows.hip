// Row step of the LDE: kernels and launchers.
#include "ntt_dev.hpp"

namespace tvh {

template <int LT, int LOGL>
__global__ void __launch_bounds__(1 << (LT - 4), 4) k_lde_rows(LdeArgs A, Roots rt) {
    lde_rows_body<LT, LOGL>(A, blockIdx.x, rt);
}
__global__ void __launch_bounds__(kCosetsThreads, 4) k_lde_cosets(LdeArgs A, Roots rt) {
    lde_cosets_body(A, blockIdx.x, rt);
}
// columns of at most 16 elements (two waves a SIMD: both matrices stay in registers)
__global__ void __launch_bounds__(kShortThreads, 2) k_lde_short(LdeArgs A, Roots rt) {
    lde_short_body(A, blockIdx.x, rt);
}
__global__ void __launch_bounds__(kShortThreads, 2)
    k_lde_short_multi(const LdeArgs* __restrict__ args, const u32* __restrict__ start, u32 nseg, Roots rt) {
    const u32 seg = find_segment(start, nseg, blockIdx.x);
    lde_short_body(args[seg], blockIdx.x - start[seg], rt);
}

// (longer tiles only where E * N2 needs them: N2 of at least 2^(LT - 4))
template <int LT>
__global__ void __launch_bounds__(1 << (LT - 4), 4)
    k_lde_rows_multi(const LdeArgs* __restrict__ args, const u32* __restrict__ start, u32 nseg, Roots rt) {
    const u32 seg = find_segment(start, nseg, blockIdx.x);
    const LdeArgs& A = args[seg];  // read in place
    const u64 blk = blockIdx.x - start[seg];
    with_length(A.logN - A.a, [&](auto l) {
        constexpr int L = decltype(l)::value;
        if constexpr (LT == 12 || L >= LT - 4) lde_rows_body<LT, L>(A, blk, rt);
    });
}

int launch_k_lde_rows(u32 lt, const LaunchShape& g, hipStream_t st, const LdeArgs& A, const Roots& rt) {
    const dim3 blocks(g.blocks), tpb(g.threads);
    if (A.products) {
        hipLaunchKernelGGL(k_lde_short, blocks, tpb, g.lds, st, A, rt);
        return check_launch();
    }
    if (A.cosets) {
        hipLaunchKernelGGL(k_lde_cosets, blocks, tpb, g.lds, st, A, rt);
        return check_launch();
    }
    with_length(A.logN - A.a, [&](auto l) {
        constexpr int L = decltype(l)::value;
        // (longer tiles only for whole transforms of E * N2 = 2^lt)
        if constexpr (L >= 10) {
            if (lt == 14) hipLaunchKernelGGL((k_lde_rows<14, L>), blocks, tpb, g.lds, st, A, rt);
        }
        if constexpr (L >= 9) {
            if (lt == 13) hipLaunchKernelGGL((k_lde_rows<13, L>), blocks, tpb, g.lds, st, A, rt);
        }
        if (lt == 12) hipLaunchKernelGGL((k_lde_rows<12, L>), blocks, tpb, g.lds, st, A, rt);
    });
    return check_launch();
}

int launch_k_lde_rows_multi(u32 lt, const LdeArgs* args, const u32* start, u32 nseg, u32 blocks,
                            size_t lds, hipStream_t st, const Roots& rt) {
    const dim3 grid(blocks), tpb(lt == kBatchShort ? kShortThreads : 1u << (lt - 4));
    if (lt == kBatchShort) hipLaunchKernelGGL(k_lde_short_multi, grid, tpb, lds, st, args, start, nseg, rt);
    else if (lt == 12) hipLaunchKernelGGL(k_lde_rows_multi<12>, grid, tpb, lds, st, args, start, nseg, rt);
    else if (lt == 13) hipLaunchKernelGGL(k_lde_rows_multi<13>, grid, tpb, lds, st, args, start, nseg, rt);
    else hipLaunchKernelGGL(k_lde_rows_multi<14>, grid, tpb, lds, st, args, start, nseg, rt);
    return check_launch();
}

int set_attributes_rows(int bytes) {
    std::vector<const void*> fns{(const void*)k_lde_rows_multi<12>, (const void*)k_lde_rows_multi<13>,
                                 (const void*)k_lde_rows_multi<14>, (const void*)k_lde_cosets};
    for (u32 l = 5; l <= 12; l++)
        with_length(l, [&](auto c) {
            constexpr int L = decltype(c)::value;
            fns.push_back((const void*)k_lde_rows<12, L>);
            if constexpr (L >= 9)
                fns.push_back((const void*)k_lde_rows<13, L>);
            if constexpr (L >= 10) fns.push_back((const void*)k_lde_rows<14, L>);
        });
    return set_lds_attribute(fns, bytes);
}

}  // namespace tvh
