// wm_prefill_kq.hip -- the K-quant instances of the prefill expert GEMMs
// (wm_pf_gemm.h), in a translation unit of their own so that they build in
// parallel with the rest.
#include <hip/hip_runtime.h>

#include "wm_pf_gemm.h"

namespace wm {

// Gate/up: ring slots of two super-blocks (512 columns) for the formats whose
// slots then still fit three deep or more; one super-block else.
template <int WT, int M> static int launch_gu(const PfGemm& g, int n_wg, hipStream_t s) {
    if constexpr (WT == Q2_K || WT == Q3_K || WT == Q4_K)
        if (g.ncol % 512 == 0) return launch_pf_gemm<1, 1, 2, WT, M, 2>(g, n_wg, s);
    return launch_pf_gemm<1, 1, 2, WT, M>(g, n_wg, s);
}

template <int M> static int launch_kq(bool gateup, int wt, const PfGemm& g, int n_wg, hipStream_t s) {
    switch (wt) {
    case Q2_K: return gateup ? launch_gu<Q2_K, M>(g, n_wg, s) : launch_pf_gemm<1, 2, 1, Q2_K, M>(g, n_wg, s);
    case Q3_K: return gateup ? launch_gu<Q3_K, M>(g, n_wg, s) : launch_pf_gemm<1, 2, 1, Q3_K, M>(g, n_wg, s);
    case Q4_K: return gateup ? launch_gu<Q4_K, M>(g, n_wg, s) : launch_pf_gemm<1, 2, 1, Q4_K, M>(g, n_wg, s);
    case Q5_K: return gateup ? launch_gu<Q5_K, M>(g, n_wg, s) : launch_pf_gemm<1, 2, 1, Q5_K, M>(g, n_wg, s);
    case Q6_K: return gateup ? launch_gu<Q6_K, M>(g, n_wg, s) : launch_pf_gemm<1, 2, 1, Q6_K, M>(g, n_wg, s);
    default: return (int)hipErrorInvalidValue;
    }
}

int launch_pf_gemm_kq(int m, bool gateup, int wt, const PfGemm& g, int n_wg, hipStream_t s) {
    if (m == 16) return launch_kq<16>(gateup, wt, g, n_wg, s);
    if (m == 32) return launch_kq<32>(gateup, wt, g, n_wg, s);
    return (int)hipErrorInvalidValue;
}

}  // namespace wm
