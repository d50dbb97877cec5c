// psi / local-energy kernels, double bulk precision.
#include "qmc_launch.h"

#ifndef QMC_RAD
#error "compile with -DQMC_RAD=0 (gto_pure) or -DQMC_RAD=1 (sto)"
#endif

namespace qmc {

template <int NM, int RAD>
static void go(const KArgs& a, int mode, hipStream_t s) {
    const dim3 g = grid_for(a.t, a.nw);
    const bool multi = !a.t.identity_conf;
    if (mode == QMC_EVAL_ELOC && multi)
        hipLaunchKernelGGL((wf_kernel<double, NM, RAD, true, true>), g, dim3(kBlock), multi_lds(a.t, true), s, a);
    else if (mode == QMC_EVAL_ELOC)
        hipLaunchKernelGGL((wf_kernel<double, NM, RAD, true, false>), g, dim3(kBlock), 0, s, a);
    else if (multi)
        hipLaunchKernelGGL((wf_kernel<double, NM, RAD, false, true>), g, dim3(kBlock), multi_lds(a.t, false), s, a);
    else if (psi_may_eliminate<NM>() && psi_eliminates(wave_count(a.t, a.nw)))
        hipLaunchKernelGGL((wf_kernel<double, NM, RAD, false, false, AoGeneric, psi_may_eliminate<NM>()>), g,
                           dim3(kBlock), 0, s, a);
    else
        hipLaunchKernelGGL((wf_kernel<double, NM, RAD, false, false>), g, dim3(kBlock), 0, s, a);
}

template <int RAD>
static int bucket(const KArgs& a, int mode, hipStream_t s) {
    switch (nm_bucket_fine(a.t)) {
#define QMC_CASE(K)           \
    case K:                   \
        go<K, RAD>(a, mode, s); \
        return 0;
        QMC_FINE_BUCKETS(QMC_CASE)
#undef QMC_CASE
        default: return -1;
    }
}

template <>
int launch_wf_f64<QMC_RAD>(const KArgs& a, int mode, hipStream_t s) {
    return bucket<QMC_RAD>(a, mode, s);
}

}  // namespace qmc
