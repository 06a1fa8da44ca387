// tables_cell.h — per-cell material properties from piecewise-linear tables (reference
// kernels.py:1685-1772), shared by the refresh kernel and the fused step.
#pragma once

#include "waam_common.h"

namespace waam {

/* lookup_table_1d — reference kernels.py:1685-1707: clamp outside the knots; inside, every
 * bracketing interval overwrites the result (the last one wins, which matters on a knot). */
__device__ __forceinline__ float lookup_table_1d(float T, const float *t_arr, const float *v_arr,
                                                 int n, float fallback)
{
    float result = fallback;
    if (n > 0) {
        /* the last knot by selects: an array of a kernel's arguments that is indexed by a variable
         * is copied to private memory in a kernel that inlines this twice */
        float t_last = t_arr[0], v_last = v_arr[0];
#pragma unroll
        for (int idx = 1; idx < WAAM_MAX_KNOTS; ++idx) {
            t_last = idx < n ? t_arr[idx] : t_last;
            v_last = idx < n ? v_arr[idx] : v_last;
        }
        if (T <= t_arr[0]) {
            result = v_arr[0];
        } else if (T >= t_last) {
            result = v_last;
        } else {
            /* the last interval that holds T (as the reference's loop leaves it), then one
             * division: a division per interval under its own branch made four lookups of a
             * cell cost more than its thermal update */
            float t0 = 0.0f, t1 = 0.0f, v0 = 0.0f, v1 = 0.0f;
            bool hit = false;
#pragma unroll
            for (int idx = 0; idx < WAAM_MAX_KNOTS - 1; ++idx) {
                if (idx < n - 1) {
                    const bool in = T >= t_arr[idx] && T <= t_arr[idx + 1];
                    t0 = in ? t_arr[idx] : t0;
                    t1 = in ? t_arr[idx + 1] : t1;
                    v0 = in ? v_arr[idx] : v0;
                    v1 = in ? v_arr[idx + 1] : v1;
                    hit = hit || in;
                }
            }
            if (hit) {
                const float w = (T - t0) / (t1 - t0 + 1e-8f);
                result = v0 + w * (v1 - v0);
            }
        }
    }
    return result;
}

/* refresh_thermal_properties for one cell (reference kernels.py:1710-1772): the constants on
 * SOLID and GAS cells, else cp*rho, the lattice diffusivity, the Marangoni coefficient and the
 * relaxation time from the tables at the cell's temperature (use_tables 0: the constants, the
 * Marangoni one scaled) */
struct CellProps {
    float cp_rho, alpha_lu, dgamma_lu, tau;
};

__device__ __forceinline__ CellProps cell_props(const waam_material_tables &tb,
                                                const waam_property_refs &rf, int use_tables,
                                                uint8_t flag, float T_c)
{
    CellProps pr;
    if (flag == SOLID || flag == GAS) {
        pr.cp_rho = rf.cp_rho_ref;
        pr.alpha_lu = rf.alpha_lu_ref;
        pr.dgamma_lu = rf.dgamma_lu_ref;
        pr.tau = rf.tau_ref;
    } else if (use_tables == 1) {
        float cp = lookup_table_1d(T_c, tb.cp_T, tb.cp_V, tb.n_cp, tb.cp_fallback);
        float k_val = lookup_table_1d(T_c, tb.k_T, tb.k_V, tb.n_k, tb.k_fallback);
        float mu_val = lookup_table_1d(T_c, tb.mu_T, tb.mu_V, tb.n_mu, tb.mu_fallback);
        float dgamma = lookup_table_1d(T_c, tb.dgamma_T, tb.dgamma_V, tb.n_dgamma,
                                       tb.dgamma_fallback);
        float alpha_phys = k_val / (rf.rho * cp + 1e-9f);
        float nu_phys = mu_val / (rf.rho + 1e-9f);
        float nu_lu = nu_phys * rf.dt / (rf.dx * rf.dx);
        pr.cp_rho = rf.rho * cp;
        pr.alpha_lu = alpha_phys * rf.dt / (rf.dx * rf.dx);
        pr.dgamma_lu = dgamma * rf.force_scale * rf.marangoni_scale;
        pr.tau = 3.0f * nu_lu + 0.5f;
    } else {
        pr.cp_rho = rf.cp_rho_ref;
        pr.alpha_lu = rf.alpha_lu_ref;
        pr.dgamma_lu = rf.dgamma_lu_ref * rf.marangoni_scale;
        pr.tau = rf.tau_ref;
    }
    return pr;
}

}  // namespace waam
