// rollout.hip — the differentiable rollouts' forward steps (frozen flags and phi), a run of steps
// per call.
//
// One step of the reference chain (solvers/coupled_step.py:97-409 with the free surface held) is
// arc injection, ceiling, conduction and advection, losses, floor, phase map, ceiling, phase map,
// then the body forces, their clamp, the MRT collision and the Mach clamp. As one launch per
// reference kernel that was 10 (thermal) or 25 (coupled) launches of 2-5 us of work each from the
// host, at 7 us a launch: the host was the bound (128x64x48: 215 us a thermal step with its
// adjoint, 654 us a coupled one). Here a step is
//   k_rollout_total    the arc weight total and energy per weight (one block)
//   k_rollout_thermal  the whole enthalpy chain of every cell; the arc-weight partial sums of the
//                      next step, whose liquid fraction a cell knows once its own is final
//   k_rollout_flow     forces, collision and Mach clamp of the FLUID/IFACE cells (a list: the
//                      flags are frozen), in the coupled rollout
// launched from one native loop. Saved fields are written where they arise instead of copied: the
// state goes from slot t to slot t + 1 of a stack. Every value is the standalone kernels'
// expression sequence, so the fields are theirs bit for bit.
#include "arc_cell.h"
#include "forces_cell.h"
#include "lbm_cell.h"
#include "rollout.h"

namespace waam {

struct RollConsts {
    PhaseConsts pc;
    float cap_l, cap_s, h_min, cp_rho, alpha_lu;
    LossConsts lc;
    int enable_loss, enable_cap, enable_arc;
    ArcParams ap;          // this step's arc
    float next_i, next_j;  // the next step's arc centre
    int sums;              // form the next step's partial sums
    Dims d;
};

/* 32-bit division: the entries bound the grid by INT_MAX cells */
__device__ __forceinline__ void roll_ijk(size_t c, const Dims &d, int &i, int &j, int &k)
{
    const unsigned cc = (unsigned)c, nf = (unsigned)d.fast(), ny = (unsigned)d.ny;
    const unsigned r = cc / nf;
    const int a = (int)(cc - r * nf), b = (int)(r / ny);
    j = (int)(r - (unsigned)b * ny);
    i = d.layout == kLayoutZYX ? a : b;
    k = d.layout == kLayoutZYX ? b : a;
}

/* enthalpy after arc injection (A); an energy that is no number is kept out by nothing, as in the
 * arc's own entry, so that a run with a bad efficiency does not end in a cold plate */
__device__ __forceinline__ float arc_heated(float h, float fl, float wk, float epw,
                                            const RollConsts &a, int i, int j, int k)
{
    if (epw <= 0.0f) return h;
    const float wdep = fl > 0.55f ? 1.0f : wk;
    const float hot = h + epw * arc_shape(a.ap, i, j, k) * wdep;
    return wdep < 1e-6f ? h : hot;
}

/* a cell's terms of the next step's arc sums W = sum w and S = sum w r^2 */
struct ArcSums {
    double w = 0.0, wc = 0.0, s = 0.0, sc = 0.0;
    __device__ __forceinline__ void add(const ArcParams &ap, float fl, float wk, int i, int j, int k)
    {
        const float wdep = fl > 0.55f ? 1.0f : wk;
        if (wdep < 1e-6f) return;
        const float di = (float)i - ap.arc_i, dj = (float)j - ap.arc_j, dk = (float)k - ap.arc_k;
        const float r2 = di * di + dj * dj + dk * dk * 0.25f;
        const double x = (double)(arc_shape(ap, i, j, k) * wdep);
        double ss, e;
        two_sum(w, x, ss, e);
        w = ss;
        wc += e;
        two_sum(s, x * (double)r2, ss, e);
        s = ss;
        sc += e;
    }
    /* the block's pairs into parts; every thread calls it */
    __device__ __forceinline__ void store(double *parts, double *sh_s, double *sh_c)
    {
        block_reduce_pair(w, wc, sh_s, sh_c);
        __syncthreads();
        block_reduce_pair(s, sc, sh_s, sh_c);
        if (threadIdx.x == 0) {
            parts[4 * blockIdx.x] = w;
            parts[4 * blockIdx.x + 1] = wc;
            parts[4 * blockIdx.x + 2] = s;
            parts[4 * blockIdx.x + 3] = sc;
        }
    }
};

/* the first step's partial sums, and the depth weights of the rollout (its arc_k is fixed) */
__global__ void __launch_bounds__(kBlock) k_rollout_sums(const float *__restrict__ fl,
                                                         const uint8_t *__restrict__ flags,
                                                         float *__restrict__ depth, RollConsts a,
                                                         double *__restrict__ parts)
{
    __shared__ double sh_s[kBlock], sh_c[kBlock];
    const Dims &d = a.d;
    if (blockIdx.x == 0)
        for (int k = threadIdx.x; k < d.nz; k += blockDim.x)
            depth[k] = arc_deposition_weight(k, a.ap.arc_k, 0.0f, a.ap.pen, a.ap.enable);
    ArcSums sums;
    const size_t N = d.n();
    for (size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x; c < N;
         c += (size_t)gridDim.x * blockDim.x) {
        if (flags[c] == GAS) continue;
        int i, j, k;
        roll_ijk(c, d, i, j, k);
        /* the table is being written: the weight itself */
        sums.add(a.ap, fl[c], arc_deposition_weight(k, a.ap.arc_k, 0.0f, a.ap.pen, a.ap.enable),
                 i, j, k);
    }
    sums.store(parts, sh_s, sh_c);
}

/* fixed-order totals of the partial sums: the step's (W, S) in binary64 and, in fp32, the weight
 * total and the energy per unit weight (reference kernels.py:493-496) */
__global__ void __launch_bounds__(kBlock) k_rollout_total(const double *__restrict__ parts,
                                                          float Q_w, float eta, float dt, float dx3,
                                                          float *__restrict__ tot,
                                                          double *__restrict__ sums)
{
    __shared__ double sh_s[kBlock], sh_c[kBlock];
    double out[2];
    for (int g = 0; g < 2; ++g) {
        double s = 0.0, c = 0.0;
        for (int b = threadIdx.x; b < kReduceBlocks; b += blockDim.x) {
            double ss, e;
            two_sum(s, parts[4 * b + 2 * g], ss, e);
            s = ss;
            c += parts[4 * b + 2 * g + 1] + e;
        }
        block_reduce_pair(s, c, sh_s, sh_c);
        out[g] = s + c;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const float w_total = (float)out[0];
        tot[0] = w_total;
        tot[1] = w_total > 1e-9f ? Q_w * eta * dt / (w_total * dx3) : 0.0f;
        sums[0] = out[0];
        sums[1] = out[1];
    }
}

/* One step's enthalpy chain, kReduceBlocks blocks over the cells. ADV: with advection of the
 * heated, capped enthalpy by u. Reads 9 B a cell and its neighbours', writes 12 (28 with saved
 * fields): a grid of a few hundred thousand cells sits in the caches and the launch is bound by
 * its longest lane (two exps for a plain cell, fourteen for a liquid one). */
template <bool ADV>
__global__ void __launch_bounds__(kBlock) k_rollout_thermal(
    const float *__restrict__ H, const float *__restrict__ T, const float *__restrict__ fl,
    const float *__restrict__ ux, const float *__restrict__ uy, const float *__restrict__ uz,
    const uint8_t *__restrict__ flags, const float *__restrict__ depth,
    const float *__restrict__ tot, RollConsts a, float *__restrict__ H_out,
    float *__restrict__ T_out, float *__restrict__ fl_out, float *__restrict__ sA,
    float *__restrict__ sB, float *__restrict__ sE, float *__restrict__ sF,
    double *__restrict__ parts)
{
    __shared__ double sh_s[kBlock], sh_c[kBlock];
    const Dims &d = a.d;
    const size_t N = d.n();
    const float epw = a.enable_arc ? tot[1] : 0.0f;
    ArcParams next = a.ap;
    next.arc_i = a.next_i;
    next.arc_j = a.next_j;
    ArcSums sums;
    for (size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x; c < N;
         c += (size_t)gridDim.x * blockDim.x) {
        const uint8_t flag = flags[c];
        float h = H[c], Tn, fln;
        if (flag == GAS) {
            /* only the phase maps touch it */
            phase_of(h, a.pc, Tn, fln);
            H_out[c] = h;
            T_out[c] = Tn;
            fl_out[c] = fln;
            continue;
        }
        int i, j, k;
        roll_ijk(c, d, i, j, k);
        const float wk = a.enable_arc ? depth[k] : 0.0f;
        const float T_c = T[c];
        const float T_im = masked_at(T, flags, i - 1, j, k, T_c, d);
        const float T_ip = masked_at(T, flags, i + 1, j, k, T_c, d);
        const float T_jm = masked_at(T, flags, i, j - 1, k, T_c, d);
        const float T_jp = masked_at(T, flags, i, j + 1, k, T_c, d);
        const float T_km = masked_at(T, flags, i, j, k - 1, T_c, d);
        const float T_kp = masked_at(T, flags, i, j, k + 1, T_c, d);
        const int n_exp = a.enable_loss ? exposed_faces(flags, i, j, k, d) : 0;
        const float A = arc_heated(h, fl[c], wk, epw, a, i, j, k);
        const float B = a.enable_cap ? ceiling_clamp(A, a.pc.H_liq, a.cap_l, a.cap_s) : A;
        const float lap = T_ip + T_im + T_jp + T_jm + T_kp + T_km - 6.0f * T_c;
        float dH = a.cp_rho * a.alpha_lu * lap * 1.0f;
        if (ADV && flag != SOLID) {
            const float u[3] = {ux[c], uy[c], uz[c]};
            /* the twelve operands along the axes: loads first (masked_at's clamps; a GAS operand
             * gives the next nearer one) */
            float q[12], qf[12], qw[12];
            uint8_t fg[12];
#pragma unroll
            for (int t = 0; t < 12; ++t) {
                const int o = (t & 1 ? 1 : -1) * (t & 2 ? 2 : 1), ax = t >> 2;
                const int ii = imax(0, imin(i + (ax == 0 ? o : 0), d.nx - 1));
                const int jj = imax(0, imin(j + (ax == 1 ? o : 0), d.ny - 1));
                const int kk = imax(0, imin(k + (ax == 2 ? o : 0), d.nz - 1));
                const size_t n = d.idx(ii, jj, kk);
                fg[t] = flags[n];
                q[t] = H[n];
                qf[t] = fl[n];
                qw[t] = a.enable_arc ? depth[kk] : 0.0f;
            }
#pragma unroll
            for (int t = 0; t < 12; ++t) {
                const int o = (t & 1 ? 1 : -1) * (t & 2 ? 2 : 1), ax = t >> 2;
                const int ii = imax(0, imin(i + (ax == 0 ? o : 0), d.nx - 1));
                const int jj = imax(0, imin(j + (ax == 1 ? o : 0), d.ny - 1));
                const int kk = imax(0, imin(k + (ax == 2 ? o : 0), d.nz - 1));
                float v = arc_heated(q[t], qf[t], qw[t], epw, a, ii, jj, kk);
                if (a.enable_cap) v = ceiling_clamp(v, a.pc.H_liq, a.cap_l, a.cap_s);
                q[t] = v;
            }
            float g[3];
#pragma unroll
            for (int ax = 0; ax < 3; ++ax) {
                const float m1 = fg[4 * ax] == GAS ? B : q[4 * ax];
                const float p1 = fg[4 * ax + 1] == GAS ? B : q[4 * ax + 1];
                const float m2 = fg[4 * ax + 2] == GAS ? m1 : q[4 * ax + 2];
                const float p2 = fg[4 * ax + 3] == GAS ? p1 : q[4 * ax + 3];
                g[ax] = upwind_grad(u[ax], m2, m1, B, p1, p2);
            }
            dH -= (u[0] * g[0] + u[1] * g[1] + u[2] * g[2]) * 1.0f;
        }
        h = B + dH;
        if (n_exp != 0) h -= loss_flux(T_c, a.lc) * (float)n_exp * a.lc.dt / a.lc.dx;
        const float E = h;
        if (a.enable_loss && h < a.h_min) h = a.h_min;
        const float F = h;
        if (a.enable_cap) h = ceiling_clamp(h, a.pc.H_liq, a.cap_l, a.cap_s);
        phase_of(h, a.pc, Tn, fln);
        H_out[c] = h;
        T_out[c] = Tn;
        fl_out[c] = fln;
        if (sA) {
            sA[c] = A;
            if (sB) sB[c] = B;
            sE[c] = E;
            sF[c] = F;
        }
        if (a.sums) sums.add(next, fln, wk, i, j, k);
    }
    if (a.sums) sums.store(parts, sh_s, sh_c);
}

struct FlowConsts {
    int enable_csf, wetting, enable_arc, enable_hydro;
    float gamma_lu, cos_t, sin_t, dgamma, g_lu, beta, T_l, F_cap, u_cap, omega_s, omega_b, C_darcy;
    ArcPressure ap;
    Dims d;
};

/* forces, force clamp, MRT collision and Mach clamp of the listed FLUID/IFACE cells, in the
 * reference's order (coupled_step.py:298-409); Fr, Fc (3 arrays each): the force before and after
 * its clamp, when saved */
__global__ void __launch_bounds__(64) k_rollout_flow(
    const int32_t *__restrict__ active, int n_active, const float *__restrict__ f,
    const float *__restrict__ T, const float *__restrict__ fl, const float *__restrict__ phi,
    const uint8_t *__restrict__ flags, FlowConsts a, float *__restrict__ f_out,
    float *__restrict__ u_out, float *__restrict__ Fr, float *__restrict__ Fc)
{
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= n_active) return;
    const Dims &d = a.d;
    const size_t N = d.n(), c = (size_t)active[t];
    int i, j, k;
    roll_ijk(c, d, i, j, k);
    float fin[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) fin[q] = f[(size_t)q * N + c];
    const float flc = fl[c], T_c = T[c];
    ForceStencil fs;
    load_force_stencil(phi, T, flags, i, j, k, d, fs);
    float fx = 0.0f, fy = 0.0f, fz = 0.0f, tx, ty, tz;
    if (a.enable_csf &&
        csf_force(fs, i, j, k, d, a.gamma_lu, a.wetting, a.cos_t, a.sin_t, tx, ty, tz)) {
        fx += tx;
        fy += ty;
        fz += tz;
    }
    if (marangoni_force(fs, flc, a.dgamma, tx, ty, tz)) {
        fx += tx;
        fy += ty;
        fz += tz;
    }
    if (a.enable_arc && arc_pressure_force(fs.phi.c[4], fs.phi.c[5], i, j, k, a.ap, tz)) fz += tz;
    if (a.enable_hydro && flc > 0.0f) fz += -1.0f * a.g_lu * flc;
    if (flc > 0.0f) fz += 1.0f * a.g_lu * a.beta * (T_c - a.T_l) * flc;
    if (Fr) {
        Fr[c] = fx;
        Fr[N + c] = fy;
        Fr[2 * N + c] = fz;
    }
    if (a.F_cap > 0.0f) {
        const float mag = sqrtf(fx * fx + fy * fy + fz * fz);
        if (mag > a.F_cap) {
            const float sc = a.F_cap / (mag + 1e-12f);
            fx = fx * sc;
            fy = fy * sc;
            fz = fz * sc;
        }
    }
    if (Fc) {
        Fc[c] = fx;
        Fc[N + c] = fy;
        Fc[2 * N + c] = fz;
    }
    CellOut o;
    mrt_cell(fin, fx, fy, fz, flc, a.omega_s, a.omega_b, a.C_darcy, o);
#pragma unroll
    for (int q = 0; q < Q; ++q) f_out[(size_t)q * N + c] = o.f[q];
    float u = o.u, v = o.v, w = o.w;
    if (a.u_cap > 0.0f) {
        const float mag = sqrtf(u * u + v * v + w * w);
        if (mag > a.u_cap) {
            const float sc = a.u_cap / (mag + 1e-12f);
            u = u * sc;
            v = v * sc;
            w = w * sc;
        }
    }
    u_out[c] = u;
    u_out[N + c] = v;
    u_out[2 * N + c] = w;
}

int check_rollout(const char *who, const waam_rollout *r, const double *arc_i, const double *arc_j,
                  int n, bool saved)
{
    if (!r || !arc_i || !arc_j) return set_error(WAAM_ERR_INVALID, "%s: NULL argument", who);
    WAAM_RETURN_IF(check_dims(who, r->nx, r->ny, r->nz, r->layout));
    if ((size_t)r->nx * (size_t)r->ny * (size_t)r->nz > (size_t)INT32_MAX)
        return set_error(WAAM_ERR_INVALID, "%s: the grid exceeds 2^31 - 1 cells", who);
    if (n < 1) return set_error(WAAM_ERR_INVALID, "%s: %d steps", who, n);
    if (r->slot0 < 0 || r->slot0 > 1 || (r->stack && r->slot0 != 0))
        return set_error(WAAM_ERR_INVALID, "%s: starting slot %d", who, r->slot0);
    if (r->flow < 0 || r->flow > 2) return set_error(WAAM_ERR_INVALID, "%s: flow %d", who, r->flow);
    WAAM_RETURN_IF(check_ptrs(who, {r->H, r->T, r->fl, r->flags, r->depth, r->sums, r->scratch}));
    if (r->flow && (!r->u || r->n_active < 0 || (r->n_active > 0 && !r->active)))
        return set_error(WAAM_ERR_INVALID, "%s: advection without a velocity or cell list", who);
    if (r->flow == 2) WAAM_RETURN_IF(check_ptrs(who, {r->f, r->phi}));
    if (saved || r->A) {
        WAAM_RETURN_IF(check_ptrs(who, {r->A, r->E, r->F}));
        if (!r->stack) return set_error(WAAM_ERR_INVALID, "%s: saved fields need the stack", who);
        if (r->flow == 2) WAAM_RETURN_IF(check_ptrs(who, {r->Fr, r->Fc}));
    }
    return 0;
}

}  // namespace waam

using namespace waam;

extern "C" int waam_rollout_forward(const waam_rollout *r, const double *arc_i,
                                    const double *arc_j, int n, void *stream)
{
    WAAM_RETURN_IF(check_rollout("waam_rollout_forward", r, arc_i, arc_j, n, false));
    const waam_adj_consts &c = r->c;
    const Dims d{r->nx, r->ny, r->nz, r->layout};
    const size_t N = d.n();
    hipStream_t st = as_stream(stream);
    RollConsts a{};
    a.pc = make_phase_consts(c.cp_rho, c.L_rho, c.T_s, c.T_l);
    a.cap_l = a.pc.H_liq + c.cp_rho * (c.T_cap - c.T_l);
    a.cap_s = c.cp_rho * c.T_cap;
    a.h_min = c.cp_rho * c.T_floor;
    a.cp_rho = c.cp_rho;
    a.alpha_lu = c.alpha_lu;
    a.lc = LossConsts{c.T_amb, r->h_conv, r->eps_rad, c.sigma_sb, c.dt, c.dx, c.enable_conv,
                      c.enable_rad};
    a.enable_loss = c.enable_loss;
    a.enable_cap = c.enable_cap;
    a.enable_arc = c.enable_arc;
    a.ap.kind = 0;
    a.ap.arc_k = c.arc_k;
    a.ap.inv2s2 = 1.0f / (2.0f * c.sigma * c.sigma);
    a.ap.pen = c.pen;
    a.ap.enable = c.surface_weight;
    a.d = d;
    FlowConsts fc{};
    fc.enable_csf = r->enable_csf;
    fc.wetting = r->wetting;
    fc.enable_arc = c.enable_arc;
    fc.enable_hydro = r->enable_hydro;
    fc.gamma_lu = r->gamma_lu;
    fc.cos_t = r->cos_t;
    fc.sin_t = r->sin_t;
    fc.dgamma = r->dgamma;
    fc.g_lu = r->g_lu;
    fc.beta = r->beta;
    fc.T_l = c.T_l;
    fc.F_cap = r->F_cap;
    fc.u_cap = r->u_cap;
    fc.omega_s = r->omega_s;
    fc.omega_b = r->omega_b;
    fc.C_darcy = r->C_darcy;
    fc.ap.arc_k = c.arc_k;
    fc.ap.inv2s2 = 1.0f / (2.0f * r->p_sigma * r->p_sigma + 1e-6f);
    const float F_peak_phys = r->p_pa / (r->rho_phys * c.dx);
    fc.ap.F_peak_lu = F_peak_phys * (c.dt * c.dt) / c.dx;
    fc.d = d;
    double *parts = reinterpret_cast<double *>((char *)r->scratch + kScratchTelemetryParts);
    float *tot = reinterpret_cast<float *>((char *)r->scratch + kScratchTelemetry);
    auto slot = [&](int t) { return (size_t)(r->stack ? t : (r->slot0 + t) & 1); };
    /* only the flow's backward reads the steps' temperatures: two slots do elsewhere */
    auto slot_T = [&](int t) { return r->flow == 2 ? slot(t) : (size_t)((r->slot0 + t) & 1); };
    for (int t = 0; t < n; ++t) {
        const size_t s0 = slot(t), s1 = slot(t + 1);
        a.ap.arc_i = (float)arc_i[t];
        a.ap.arc_j = (float)arc_j[t];
        a.sums = c.enable_arc && t + 1 < n;
        a.next_i = a.sums ? (float)arc_i[t + 1] : 0.0f;
        a.next_j = a.sums ? (float)arc_j[t + 1] : 0.0f;
        if (c.enable_arc) {
            if (t == 0)
                hipLaunchKernelGGL(k_rollout_sums, dim3(kReduceBlocks), dim3(kBlock), 0, st,
                                   r->fl + s0 * N, r->flags, r->depth, a, parts);
            hipLaunchKernelGGL(k_rollout_total, dim3(1), dim3(kBlock), 0, st,
                               (const double *)parts, c.Q_w, c.eta, c.dt, c.dx3, tot,
                               r->sums + (r->A ? 2 * t : 0));
        }
        const float *u = r->flow == 2 ? r->u + 3 * s0 * N : r->u;
        const size_t sv = (size_t)t * N;
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(kReduceBlocks), dim3(kBlock), 0, st,
                               (const float *)r->H + s0 * N, (const float *)r->T + slot_T(t) * N,
                               (const float *)r->fl + s0 * N, u, u ? u + N : u, u ? u + 2 * N : u,
                               r->flags, (const float *)r->depth, (const float *)tot, a,
                               r->H + s1 * N, r->T + slot_T(t + 1) * N, r->fl + s1 * N,
                               r->A ? r->A + sv : nullptr, r->A && r->B ? r->B + sv : nullptr,
                               r->A ? r->E + sv : nullptr, r->A ? r->F + sv : nullptr, parts);
        };
        if (r->flow) launch(k_rollout_thermal<true>);
        else launch(k_rollout_thermal<false>);
        if (r->flow == 2 && r->n_active > 0) {
            fc.ap.arc_i = (float)arc_i[t];
            fc.ap.arc_j = (float)arc_j[t];
            hipLaunchKernelGGL(k_rollout_flow, dim3(grid_for((size_t)r->n_active, 64)), dim3(64),
                               0, st, r->active, r->n_active,
                               (const float *)r->f + (size_t)Q * s0 * N,
                               (const float *)r->T + s1 * N, (const float *)r->fl + s1 * N, r->phi,
                               r->flags, fc, r->f + (size_t)Q * s1 * N, r->u + 3 * s1 * N,
                               r->A ? r->Fr + 3 * sv : nullptr, r->A ? r->Fc + 3 * sv : nullptr);
        }
    }
    return check_launch("waam_rollout_forward");
}
