// sl_high.hip -- the semi-Lagrangian steps of the orders 9..12 (sl_steps.h)
#include "sl_steps.h"

namespace se_sl {

#define SE_SL_HIGH(KERNEL, ...)                                        \
    const dim3 grid(pair_blocks(g.nv0 * g.nv1));                       \
    switch (N) {                                                       \
        case 9: SE_SL_ADV(KERNEL, 9, grid, s, __VA_ARGS__); break;     \
        case 10: SE_SL_ADV(KERNEL, 10, grid, s, __VA_ARGS__); break;   \
        case 11: SE_SL_ADV(KERNEL, 11, grid, s, __VA_ARGS__); break;   \
        default: SE_SL_ADV(KERNEL, 12, grid, s, __VA_ARGS__); break;   \
    }

void sl_first_high(int N, hipStream_t s, const SLGeom& g, const double* q, int nd, const double* vel, double dt,
                   double* qsl, int32_t* dep) {
    SE_SL_HIGH(k_sl_first, g, q, nd, vel, dt, qsl, dep)
}

void sl_second_high(int N, hipStream_t s, const SLGeom& g, const double* q, const double* qp, int nd,
                    const double* vel, const double* vp1, const double* vph, const double* vmh, double dt,
                    double* qsl) {
    SE_SL_HIGH(k_sl_second, g, q, qp, nd, vel, vp1, vph, vmh, dt, qsl)
}

}  // namespace se_sl
