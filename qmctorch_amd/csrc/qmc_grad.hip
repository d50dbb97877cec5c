// Adjoint-row and AO-layout kernels (FP64).
#include "qmc_adjoint.h"
#include "qmc_launch.h"

#ifndef QMC_RAD
#error "compile with -DQMC_RAD=0 (gto_pure) or -DQMC_RAD=1 (sto)"
#endif
// One unit per kernel family: -DQMC_PART=0 (log|psi| rows, AO layout), 1 (log|psi|
// adjoint), 2 (E_L adjoint), 3 (E_L rows)
#ifndef QMC_PART
#error "compile with -DQMC_PART=0..3"
#endif

namespace qmc {

#if QMC_PART == 0
template <int NM, int RAD>
static void go(const GArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((grad_kernel<NM, RAD>), grid_for(a.t, a.nw), dim3(kBlock), 0, s, a);
}

template <int RAD>
static int bucket(const GArgs& a, hipStream_t s) {
    switch (nm_bucket_fine(a.t)) {
#define QMC_CASE(K)       \
    case K:               \
        go<K, RAD>(a, s); \
        return 0;
        QMC_FINE_BUCKETS(QMC_CASE)
#undef QMC_CASE
        default: return -1;
    }
}

template <>
int launch_grad<QMC_RAD>(const GArgs& a, hipStream_t s) {
    return bucket<QMC_RAD>(a, s);
}

template <>
int launch_ao<QMC_RAD>(const AArgs& a, bool deriv, hipStream_t s) {
    const dim3 g = grid_for(a.t, a.nw);
    if (deriv)
        hipLaunchKernelGGL((ao_kernel<QMC_RAD, true>), g, dim3(kBlock), 0, s, a);
    else
        hipLaunchKernelGGL((ao_kernel<QMC_RAD, false>), g, dim3(kBlock), 0, s, a);
    return 0;
}

#elif QMC_PART == 1
template <>
int launch_grad_reduce<QMC_RAD>(const GRedArgs& a, const RedOut& o, hipStream_t s) {
    const dim3 grid = grid_for_waves(a.r.nslot);
    switch (nm_bucket_fine(a.t)) {
#define QMC_CASE(K)                                                                            \
    case K:                                                                                    \
        if (a.t.identity_conf)                                                                 \
            hipLaunchKernelGGL((grad_reduce_kernel<K, QMC_RAD, false>), grid, dim3(kBlock), 0, s, a);          \
        else                                                                                   \
            hipLaunchKernelGGL((grad_reduce_kernel<K, QMC_RAD, true>), grid, dim3(kBlock), 0, s, a);           \
        break;
        QMC_FINE_BUCKETS(QMC_CASE)
#undef QMC_CASE
        default: return -1;
    }
    red_slot_sum(a.t, a.r, o, s);
    return 0;
}

#elif QMC_PART == 2
template <>
int launch_eloc_reduce<QMC_RAD>(const ERedArgs& a, const RedOut& o, hipStream_t s) {
    const dim3 grid = grid_for_waves(a.r.nslot);
    switch (nm_bucket_fine(a.t)) {
#define QMC_CASE(K)                                                                            \
    case K:                                                                                    \
        if (a.t.identity_conf)                                                                 \
            hipLaunchKernelGGL((eloc_grad_reduce_kernel<K, QMC_RAD, false>), grid, dim3(kBlock), 0, s, a);          \
        else                                                                                   \
            hipLaunchKernelGGL((eloc_grad_reduce_kernel<K, QMC_RAD, true>), grid, dim3(kBlock), 0, s, a);           \
        break;
        QMC_FINE_BUCKETS(QMC_CASE)
#undef QMC_CASE
        default: return -1;
    }
    red_slot_sum(a.t, a.r, o, s);
    return 0;
}

#else
template <int NM, int RAD>
static void go_e(const EArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((eloc_grad_kernel<NM, RAD>), grid_for(a.t, a.nw), dim3(kBlock), 0, s, a);
}

template <int RAD>
static int bucket_e(const EArgs& a, hipStream_t s) {
    switch (nm_bucket_fine(a.t)) {
#define QMC_CASE(K)         \
    case K:                 \
        go_e<K, RAD>(a, s); \
        return 0;
        QMC_FINE_BUCKETS(QMC_CASE)
#undef QMC_CASE
        default: return -1;
    }
}

template <>
int launch_eloc_grad<QMC_RAD>(const EArgs& a, hipStream_t s) {
    return bucket_e<QMC_RAD>(a, s);
}

#endif

}  // namespace qmc
