// Persistent Metropolis sweep kernels, float bulk precision.
#include "qmc_launch.h"

#ifndef QMC_RAD
#error "compile with -DQMC_RAD=0 (gto_pure) or -DQMC_RAD=1 (sto)"
#endif

namespace qmc {

template <int NM, int RAD>
static void go(const SArgs& a, hipStream_t s) {
    if (a.t.identity_conf)
        hipLaunchKernelGGL((sweep_kernel<float, NM, RAD, false>), grid_for(a.t, a.nw), dim3(kBlock), 0, s, a);
    else
        hipLaunchKernelGGL((sweep_kernel<float, NM, RAD, true>), grid_for(a.t, a.nw), dim3(kBlock), multi_lds(a.t, false), s, a);
}

template <int RAD>
static int bucket(const SArgs& a, hipStream_t s) {
    switch (nm_bucket_fine(a.t)) {
#define QMC_CASE(K)           \
    case K:                   \
        go<K, RAD>(a, s); \
        return 0;
        QMC_FINE_BUCKETS(QMC_CASE)
#undef QMC_CASE
        default: return -1;
    }
}

template <>
int launch_sweep_f32<QMC_RAD>(const SArgs& a, hipStream_t s) {
    return bucket<QMC_RAD>(a, s);
}

}  // namespace qmc
