// Column step of the LDE's forward transforms: kernels and launchers.
#include "ntt_dev.hpp"

namespace tvh {

template <int LT, int LOGL>
__global__ void __launch_bounds__(1 << (LT - 4), 4) k_lde_step3(Step3Args A, Roots rt) {
    lde_step3_body<LT, LOGL>(A, blockIdx.x, rt);
}

template <int LT>
__global__ void __launch_bounds__(1 << (LT - 4), 4) k_lde_step3_multi(const Step3Args* __restrict__ args,
                                                              const u32* __restrict__ start,
                                                              u32 nseg, Roots rt) {
    const u32 seg = find_segment(start, nseg, blockIdx.x);
    const Step3Args& A = args[seg];  // read in place
    const u64 blk = blockIdx.x - start[seg];
    with_length(A.a, [&](auto l) { lde_step3_body<LT, decltype(l)::value>(A, blk, rt); });
}

int launch_k_lde_step3(u32 lt, const LaunchShape& g, hipStream_t st, const Step3Args& A, const Roots& rt) {
    const dim3 blocks(g.blocks), tpb(g.threads);
    with_length(A.a, [&](auto l) {
        constexpr int L = decltype(l)::value;
        if (lt == 12) hipLaunchKernelGGL((k_lde_step3<12, L>), blocks, tpb, g.lds, st, A, rt);
        else if (lt == 13) hipLaunchKernelGGL((k_lde_step3<13, L>), blocks, tpb, g.lds, st, A, rt);
        else hipLaunchKernelGGL((k_lde_step3<14, L>), blocks, tpb, g.lds, st, A, rt);
    });
    return check_launch();
}

int launch_k_lde_step3_multi(const Step3Args* args, const u32* start, u32 nseg, u32 blocks, size_t lds,
                      hipStream_t st, const Roots& rt) {
    hipLaunchKernelGGL(k_lde_step3_multi<kBatchColLt>, dim3(blocks), dim3(1u << (kBatchColLt - 4)), lds, st, args, start, nseg,
                       rt);
    return check_launch();
}

int set_attributes_step3(int bytes) {
    std::vector<const void*> fns{(const void*)k_lde_step3_multi<kBatchColLt>};
    for (u32 l = 5; l <= 12; l++)
        with_length(l, [&](auto c) {
            constexpr int L = decltype(c)::value;
            fns.insert(fns.end(), {(const void*)k_lde_step3<12, L>, (const void*)k_lde_step3<13, L>,
                                   (const void*)k_lde_step3<14, L>});
        });
    return set_lds_attribute(fns, bytes);
}

}  // namespace tvh
