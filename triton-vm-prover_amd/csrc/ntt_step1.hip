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

// The column lengths that forward transforms have in tiles of 2^LT (launch_ntt_batched):
// 2^6 to 2^10, 2^11 and 2^12 in the largest.  (The LDE's inverse ones: any.)
template <int LT, int LOGL>
constexpr bool kForwardShape = LOGL >= 6 && (LT == 12 ? LOGL <= 9 : LT == 13 ? LOGL <= 10 : LOGL >= 11);

int launch_k_step1(bool inv, u32 lt, const LaunchShape& g, hipStream_t st, const Step1Args& A,
                   const Roots& rt) {
    const dim3 blocks(g.blocks), tpb(g.threads);
    bool done = false;
    auto launch = [&](auto t) {
        constexpr int LT = decltype(t)::value;
        with_length(A.a, [&](auto l) {
            constexpr int L = decltype(l)::value;
            if (inv) {
                hipLaunchKernelGGL((k_step1<true, LT, L>), blocks, tpb, g.lds, st, A, rt);
                done = true;
            } else if constexpr (kForwardShape<LT, L>) {
                hipLaunchKernelGGL((k_step1<false, LT, L>), blocks, tpb, g.lds, st, A, rt);
                done = true;
            }
        });
    };
    with_tile(lt, launch);
    return done ? check_launch() : set_error(TVH_ERR_UNSUPPORTED, "column step of 2^%u in 2^%u tiles", A.a, lt);
}

int launch_k_step1_scaled(u32 lt, const LaunchShape& g, hipStream_t st, const Step1Args& A,
                          const NttScaleDev& S, const Roots& rt) {
    const dim3 blocks(g.blocks), tpb(g.threads);
    bool done = false;
    auto launch = [&](auto t) {
        constexpr int LT = decltype(t)::value;
        with_length(A.a, [&](auto l) {
            constexpr int L = decltype(l)::value;
            if constexpr (kForwardShape<LT, L>) {
                hipLaunchKernelGGL((k_step1_scaled<LT, L>), blocks, tpb, g.lds, st, A, S, rt);
                done = true;
            }
        });
    };
    with_tile(lt, launch);
    return done ? check_launch() : set_error(TVH_ERR_UNSUPPORTED, "column step of 2^%u in 2^%u tiles", A.a, lt);
}

int launch_k_step1_multi(const Step1Args* args, const u32* start, u32 nseg, u32 blocks, size_t lds,
                         hipStream_t st, const Roots& rt) {
    hipLaunchKernelGGL(k_step1_multi<kBatchColLt>, dim3(blocks), dim3(1u << (kBatchColLt - 4)), lds, st,
                       args, start, nseg, rt);
    return check_launch();
}

int set_attributes_step1(int bytes) {
    std::vector<const void*> fns{(const void*)k_step1_multi<kBatchColLt>};
    for (u32 lt = 12; lt <= 14; lt++)
        with_tile(lt, [&](auto t) {
            constexpr int LT = decltype(t)::value;
            for (u32 l = 5; l <= 12; l++)
                with_length(l, [&](auto c) {
                    constexpr int L = decltype(c)::value;
                    fns.push_back((const void*)k_step1<true, LT, L>);
                    if constexpr (kForwardShape<LT, L>)
                        fns.insert(fns.end(), {(const void*)k_step1<false, LT, L>, (const void*)k_step1_scaled<LT, L>});
                });
        });
    return set_lds_attribute(fns, bytes);
}

}  // namespace tvh
