// cavity.hip — the lid-driven cavity step: D3Q19 pull stream over all cells with half-way
// bounce-back and a moving lid, then the central-moment MRT collision.
//
// The reference's stream has bounce-back only (kernels.py:2982-3010) and, with its buffer
// choreography, never transports momentum between fluid cells; the cavity needs both, so this
// step pulls every FLUID cell from its neighbours every step (all three axes periodic: walls
// are cells). A population that would come from a wall cell is the cell's own opposite
// population (half-way bounce-back); off a LID cell it gains Ladd's moving-wall term
// 6 w_q (e_q . u_w) (wall density 1). The collision is collide_mrt's per-cell map
// (cumulant_kernel.py:28-209) with no force and no Darcy damping.
#include "lbm_cell.h"

namespace waam {

/* A lane per cell of the linear index, so that rows of any length fill their wavefronts (64-lane
 * row tiles left half the wavefronts of the 66-cell rows of 64^3 two cells). The populations and
 * flags of the 19 sources load together; the cell's own populations, which only
 * bounce back, load where a source is a wall. 64^3 fluid cells move 44 MB a step through the
 * Infinity Cache in 15.7 us (2.8 TB/s; 23.3 with the row tiles, every own population loaded and
 * 64-bit indices), 128^3 334 MB in 96 (3.5 TB/s; 143). Bound by the 38 loads a lane issues, half
 * of them flag bytes. */
__global__ void __launch_bounds__(256) k_cavity_step(const float *__restrict__ src,
                                                     float *__restrict__ dst, float *rho,
                                                     float *ux, float *uy, float *uz,
                                                     const uint8_t *__restrict__ flags,
                                                     float omega_s, float omega_b, float uwx,
                                                     float uwy, float uwz, Dims d)
{
    /* 32-bit cell indices (the entry bounds the grid), the wrap of each axis as an offset: 64-bit
     * division and index arithmetic per direction were a third of the kernel's instructions */
    const unsigned N32 = (unsigned)d.n();
    const size_t N = N32;
    const unsigned c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= N32 || flags[c] != FLUID) return;
    const unsigned nf = (unsigned)d.fast(), ny = (unsigned)d.ny, ns = (unsigned)d.slow();
    const unsigned r = c / nf, a = c - r * nf, sl = r / ny, j = r - sl * ny;
    const unsigned row = nf, slab = nf * ny;
    /* offsets of the source one cell down (index 0), none (1) and one up (2) along each axis */
    const unsigned of[3] = {a > 0 ? ~0u : nf - 1, 0u, a + 1 < nf ? 1u : 1u - nf};
    const unsigned oj[3] = {j > 0 ? 0u - row : (ny - 1) * row, 0u, j + 1 < ny ? row : row - slab};
    const unsigned os[3] = {sl > 0 ? 0u - slab : (ns - 1) * slab, 0u,
                            sl + 1 < ns ? slab : slab - ns * slab};
    const bool zyx = d.layout == kLayoutZYX;
    const unsigned ox[3] = {zyx ? of[0] : os[0], 0u, zyx ? of[2] : os[2]};
    const unsigned oz[3] = {zyx ? os[0] : of[0], 0u, zyx ? os[2] : of[2]};
    float fin[Q];
    uint8_t fn[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const unsigned n = c + ox[1 - ex(q)] + oj[1 - ey(q)] + oz[1 - ez(q)];
        fn[q] = flags[n];
        fin[q] = (src + (size_t)q * N)[n];
    }
    bool wall = false;
#pragma unroll
    for (int q = 0; q < Q; ++q) wall = wall || fn[q] != FLUID;
    if (wall) {
        float b[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) b[q] = (src + (size_t)opp(q) * N)[c];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const float eu = (float)ex(q) * uwx + (float)ey(q) * uwy + (float)ez(q) * uwz;
            const float moving = b[q] + 6.0f * wq(q) * eu;
            fin[q] = fn[q] == FLUID ? fin[q] : (fn[q] == WAAM_CAVITY_LID ? moving : b[q]);
        }
    }
    CellOut o;
    mrt_cell(fin, 0.0f, 0.0f, 0.0f, 1.0f, omega_s, omega_b, 0.0f, o);
#pragma unroll
    for (int q = 0; q < Q; ++q) (dst + (size_t)q * N)[c] = o.f[q];
    rho[c] = o.rho;
    ux[c] = o.u;
    uy[c] = o.v;
    uz[c] = o.w;
}

}  // namespace waam

using namespace waam;

extern "C" int waam_cavity_step(const float *f_src, float *f_dst, float *rho, float *ux,
                                float *uy, float *uz, const uint8_t *flags, float omega_s,
                                float omega_b, float uwx, float uwy, float uwz, int nx, int ny,
                                int nz, int layout, void *stream)
{
    WAAM_RETURN_IF(check_dims("waam_cavity_step", nx, ny, nz, layout));
    WAAM_RETURN_IF(check_ptrs("waam_cavity_step", {f_src, f_dst, rho, ux, uy, uz, flags}));
    if (f_src == f_dst) return set_error(WAAM_ERR_INVALID, "waam_cavity_step: f_src aliases f_dst");
    Dims d{nx, ny, nz, layout};
    if (d.n() > (size_t)INT32_MAX)
        return set_error(WAAM_ERR_INVALID, "waam_cavity_step: the grid exceeds 2^31 - 1 cells");
    hipLaunchKernelGGL(k_cavity_step, dim3(grid_for(d.n())), dim3(kBlock), 0, as_stream(stream), f_src, f_dst,
                       rho, ux, uy, uz, flags, omega_s, omega_b, uwx, uwy, uwz, d);
    return check_launch("waam_cavity_step");
}
