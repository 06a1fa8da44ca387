/*
 * lorentz.h — the J x B force of one cell and the host side of the Lorentz solve, shared by its own
 * entry and the fused step that adds the force in its collision.
 */
#pragma once

#include "waam_common.h"

namespace waam {

/* apply_lorentz_JxB kernels.py:1480-1513, the increment of one non-GAS cell with f_l >= 0.05 */
__device__ __forceinline__ void lorentz_force(float jx, float jy, float jz, float bx, float by,
                                              float bz, float fl, float dt, float dx, float rho,
                                              float &fx, float &fy, float &fz)
{
    float flw = fl < 1.0f ? fl : 1.0f;
    float scale = flw * dt * dt / (rho * dx);
    fx = (jy * bz - jz * by) * scale;
    fy = (jz * bx - jx * bz) * scale;
    fz = (jx * by - jy * bx) * scale;
}

int check_lorentz(const char *who, const waam_lorentz &q);

/* The solve on q's fields: arc_k from device memory when arc_k_dev is set; force false leaves the
 * force to the caller (J and B are stored either way). Reads the convergence test back after the
 * first chunk of sweeps and after every group of chunks that follows. */
int lorentz_run(const char *who, const waam_lorentz &q, const float *arc_k_dev, bool force,
                waam_lorentz_result &out, hipStream_t st);

}  // namespace waam
