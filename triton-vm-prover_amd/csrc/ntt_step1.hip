// Column (strided) step of the batched NTT and of the LDE's inverse transform:
// kernels and their launchers.
#include "ntt_dev.hpp"

namespace tvh {

template <bool INV, int LT, int LOGL>
__global__ void __launch_bounds__(1 << (LT - 4), 4) k_step1(Step1Args A, Roots rt) {
    step1_body<INV, false, LT, LOGL>(A, NttScaleDev{}, blockIdx.x, rt);
}
template <int LT, int LOGL>
__global__ void __launch_bounds__(1 << (LT - 4), 4) k_step1_scaled(Step1Args A, NttScaleDev S,
                                                                   Roots rt) {
    step1_body<false, true, LT, LOGL>(A, S, blockIdx.x, rt);
}

template <int LT>
__global__ void __launch_bounds__(1 << (LT - 4), 4) k_step1_multi(const Step1Args* __restrict__ args,
                                                                  const u32* __restrict__ start,
                                                                  u32 nseg, Roots rt) {
    const u32 seg = find_segment(start, nseg, blockIdx.x);
    const Step1Args& A = args[seg];
    const u64 blk = blockIdx.x - start[seg];
    with_length(A.a, [&](auto l) {
        step1_body<true, false, LT, decltype(l)::value>(A, NttScaleDev{}, blk, rt);
    });
}

int launch_k_step1(bool inv, u32 lt, const LaunchShape& g, hipStream_t st, const Step1Args& A,
                   const Roots& rt) {
    const dim3 blocks(g.blocks), tpb(g.threads);
    with_length(A.a, [&](auto l) {
        constexpr int L = decltype(l)::value;
#define TVH_STEP1(I, T) hipLaunchKernelGGL((k_step1<I, T, L>), blocks, tpb, g.lds, st, A, rt)
        if (inv) {
            if (lt == 12) TVH_STEP1(true, 12);
            else if (lt == 13) TVH_STEP1(true, 13);
            else TVH_STEP1(true, 14);
        } else {
            if (lt == 12) TVH_STEP1(false, 12);
            else if (lt == 13) TVH_STEP1(false, 13);
            else TVH_STEP1(false, 14);
        }
#undef TVH_STEP1
    });
    return check_launch();
}

int launch_k_step1_scaled(u32 lt, const LaunchShape& g, hipStream_t st, const Step1Args& A,
                          const NttScaleDev& S, const Roots& rt) {
    const dim3 blocks(g.blocks), tpb(g.threads);
    with_length(A.a, [&](auto l) {
        constexpr int L = decltype(l)::value;
#define TVH_STEP1(T) hipLaunchKernelGGL((k_step1_scaled<T, L>), blocks, tpb, g.lds, st, A, S, rt)
        if (lt == 12) TVH_STEP1(12);
        else if (lt == 13) TVH_STEP1(13);
        else TVH_STEP1(14);
#undef TVH_STEP1
    });
    return check_launch();
}

int launch_k_step1_multi(const Step1Args* args, const u32* start, u32 nseg, u32 blocks, size_t lds,
                         hipStream_t st, const Roots& rt) {
    hipLaunchKernelGGL(k_step1_multi<kBatchColLt>, dim3(blocks), dim3(1u << (kBatchColLt - 4)), lds, st,
                       args, start, nseg, rt);
    return check_launch();
}

int set_attributes_step1(int bytes) {
    std::vector<const void*> fns{(const void*)k_step1_multi<kBatchColLt>};
    for (u32 l = 5; l <= 12; l++)
        with_length(l, [&](auto c) {
            constexpr int L = decltype(c)::value;
            fns.insert(fns.end(), {(const void*)k_step1<true, 12, L>, (const void*)k_step1<true, 13, L>,
                                   (const void*)k_step1<true, 14, L>, (const void*)k_step1<false, 12, L>,
                                   (const void*)k_step1<false, 13, L>, (const void*)k_step1<false, 14, L>,
                                   (const void*)k_step1_scaled<12, L>, (const void*)k_step1_scaled<13, L>,
                                   (const void*)k_step1_scaled<14, L>});
        });
    return set_lds_attribute(fns, bytes);
}

}  // namespace tvh
