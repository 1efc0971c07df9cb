// wm_prefill_kq.hip -- the K-quant instances of the prefill expert GEMMs
// (wm_pf_gemm.h), in a translation unit of their own so that they build in
// parallel with the rest.
#include <hip/hip_runtime.h>

#include "wm_pf_gemm.h"

namespace wm {

// One launch: alone, or with the shared expert's Q8_0 passes behind.
template <int AHL, int WT, int M, int NSB> static int go(const PfGemm& g, const PfGemm* sh, int n_wg, hipStream_t s) {
    if constexpr (AHL == 1 || M == 16)
        if (sh) return launch_pf_gemm2<AHL, WT, M, NSB, Q8_0>(g, *sh, n_wg, s);
    if (sh) return (int)hipErrorInvalidValue;
    return launch_pf_gemm<AHL, WT, M, NSB>(g, n_wg, s);
}

// Gate/up: ring slots of two super-blocks (512 columns) for the formats whose
// slots then still fit three deep or more; one super-block else.
template <int WT, int M> static int launch_one(bool gateup, const PfGemm& g, const PfGemm* sh, int n_wg, hipStream_t s) {
    if (!gateup) return go<2, WT, M, 1>(g, sh, n_wg, s);
    if constexpr (WT == Q2_K || WT == Q3_K || WT == Q4_K)
        if (g.ncol % 512 == 0) return go<1, WT, M, 2>(g, sh, n_wg, s);
    return go<1, WT, M, 1>(g, sh, n_wg, s);
}

template <int M> static int launch_kq(bool gateup, int wt, const PfGemm& g, const PfGemm* sh, int n_wg, hipStream_t s) {
    switch (wt) {
    case Q2_K: return launch_one<Q2_K, M>(gateup, g, sh, n_wg, s);
    case Q3_K: return launch_one<Q3_K, M>(gateup, g, sh, n_wg, s);
    case Q4_K: return launch_one<Q4_K, M>(gateup, g, sh, n_wg, s);
    case Q5_K: return launch_one<Q5_K, M>(gateup, g, sh, n_wg, s);
    case Q6_K: return launch_one<Q6_K, M>(gateup, g, sh, n_wg, s);
    default: return (int)hipErrorInvalidValue;
    }
}

static int launch_m(int m, bool gateup, int wt, const PfGemm& g, const PfGemm* sh, int n_wg, hipStream_t s) {
    if (m == 16) return launch_kq<16>(gateup, wt, g, sh, n_wg, s);
    if (m == 32) return launch_kq<32>(gateup, wt, g, sh, n_wg, s);
    return (int)hipErrorInvalidValue;
}

int launch_pf_gemm_kq(int m, bool gateup, int wt, const PfGemm& g, int n_wg, hipStream_t s) {
    return launch_m(m, gateup, wt, g, nullptr, n_wg, s);
}

int launch_pf_gemm_kq_q8(int m, bool gateup, int wt, const PfGemm& g, const PfGemm& sh, int n_wg, hipStream_t s) {
    return launch_m(m, gateup, wt, g, &sh, n_wg, s);
}

}  // namespace wm
