// lorentz.hip — the welding-current Lorentz force of the full physics tier (reference
// kernels.py:1236-1513, driven by physics/weld_forces.py:196-281).
//
// One entry per reference kernel: electrical conductivity, the normalised arc current source, a
// weighted Jacobi sweep for the potential with the plate grounded, the L1 change used for the
// convergence test, J = -sigma grad(phi), the axial current binned by radius per z-slab, its
// radial prefix (enclosed current), the axisymmetric self field B_theta = mu0 I_enc / (2 pi r)
// and the J x B body force. The reference's float atomic sums (source total, L1 norms, radial
// bins) become compensated fp64 sums rounded once to fp32, which does not depend on the order
// of the terms.
//
// waam_lorentz_solve runs the same solve as a whole: entry by entry a warm solve took 23 to 63
// launches, each waiting for the one before on a grid that it covers in less than its own latency,
// with a read by the host after every tenth sweep. Its kernels cover several of these each (source
// and its total, on grids of up to 256 tiles the sweeps in LDS, J with the radial bins, prefix with
// B and the force), and the convergence test is taken on the device: there a solve that converges in
// its first chunk of ten is seven launches and one read, with the same values bit for bit. In the
// fused step (waam_step_fused_lorentz) a step of 80x40x30 takes 186 us, 615 to 660 through the
// entries; 400x200x100, which sweeps one by one, 836 and 1600.
#include "arc_cell.h"
#include "lorentz.h"

#include <utility>
#include "waam_common.h"

namespace waam {

constexpr int kLorentzSumBlocks = kReduceBlocks;
constexpr int kBinGroup = 8;  // radial bins per workgroup of the binning kernel

__device__ __forceinline__ float sigma_at(const float *s, int i, int j, int k, const Dims &d)
{
    return s[d.idx(imax(0, imin(d.nx - 1, i)), imax(0, imin(d.ny - 1, j)),
                   imax(0, imin(d.nz - 1, k)))];
}

/* elec_build_sigma kernels.py:1236-1251 */
__global__ void k_elec_build_sigma(float *__restrict__ sigma, const float *__restrict__ f_l,
                                   const uint8_t *__restrict__ flags, float s_liq, float s_sol,
                                   size_t N)
{
    size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= N) return;
    float fl = f_l[c];
    uint8_t f = flags[c];
    sigma[c] = f == GAS ? 1e-8f : (fl > 0.55f ? s_liq : s_sol);
}

__global__ void k_fill(float *__restrict__ a, float v, size_t N)
{
    size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c < N) a[c] = v;
}

struct ElecSource {
    float arc_i, arc_j, arc_k, inv2s2, current, cell_vol;
    int k_min, k_max;
    float sigma_cells;
    const float *arc_k_dev;  // set: the step left arc_k there
};

__host__ __device__ inline void elec_slabs(ElecSource &e, int nz)
{
    int km = (int)(e.arc_k + e.sigma_cells * 4.0f) + 1;
    e.k_max = km < nz ? km : nz;
    int kn = (int)(e.arc_k - e.sigma_cells);
    e.k_min = kn > 0 ? kn : 0;
}

static ElecSource elec_source(float arc_i, float arc_j, float arc_k, float sigma_cells,
                              float current_A, float dx, int nz, const float *arc_k_dev = nullptr)
{
    ElecSource e;
    e.arc_i = arc_i;
    e.arc_j = arc_j;
    e.arc_k = arc_k;
    e.inv2s2 = 1.0f / (2.0f * sigma_cells * sigma_cells + 1e-6f);
    e.current = current_A;
    e.cell_vol = dx * dx * dx;
    e.sigma_cells = sigma_cells;
    e.arc_k_dev = arc_k_dev;
    elec_slabs(e, nz);
    return e;
}

/* the arc's current density before it is normalised: 0 outside the slab range */
__device__ __forceinline__ float elec_source_at(const ElecSource &e, int i, int j, int k)
{
    if (k < e.k_min || k > e.k_max) return 0.0f;
    float di = (float)i - e.arc_i, dj = (float)j - e.arc_j, dk = (float)k - e.arc_k;
    float r2 = di * di + dj * dj + 0.25f * dk * dk;
    float w = waam_expf(-r2 * e.inv2s2);
    return e.current * w / (e.cell_vol + 1e-6f);
}

/* elec_inject_arc_source kernels.py:1260-1286: cells of the slab range get the Gaussian
 * current density, the others keep their value (0 after elec_clear_source) */
__global__ void k_elec_source(float *__restrict__ source, ElecSource e, Dims d)
{
    int i, j, k;
    if (!d.cell(i, j, k)) return;
    if (k < e.k_min || k > e.k_max) return;
    source[d.idx(i, j, k)] = elec_source_at(e, i, j, k);
}

/* elec_normalize_source kernels.py:1289-1301, first loop: compensated partial sums of
 * source * cell volume */
__global__ void __launch_bounds__(kBlock) k_elec_source_sum(const float *__restrict__ source,
                                                            float cell_vol,
                                                            double *__restrict__ parts, size_t N)
{
    __shared__ double sh_s[kBlock], sh_c[kBlock];
    double sum = 0.0, comp = 0.0;
    for (size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x; c < N;
         c += (size_t)gridDim.x * blockDim.x) {
        double ss, er;
        two_sum(sum, (double)(source[c] * cell_vol), ss, er);
        sum = ss;
        comp += er;
    }
    block_reduce_pair(sum, comp, sh_s, sh_c);
    if (threadIdx.x == 0) {
        parts[2 * blockIdx.x] = sum;
        parts[2 * blockIdx.x + 1] = comp;
    }
}

/* fixed-order total of nb partial pairs, rounded to fp32 into out[0] */
__global__ void __launch_bounds__(kBlock) k_pairs_total(const double *__restrict__ parts, int nb,
                                                        float *__restrict__ out)
{
    __shared__ double sh_s[kBlock], sh_c[kBlock];
    double sum = 0.0, comp = 0.0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
        double ss, e;
        two_sum(sum, parts[2 * b], ss, e);
        sum = ss;
        comp += parts[2 * b + 1] + e;
    }
    block_reduce_pair(sum, comp, sh_s, sh_c);
    if (threadIdx.x == 0) out[0] = (float)(sum + comp);
}

/* elec_normalize_source kernels.py:1289-1301, second loop: source *= I / max(total, 1e-12) */
__global__ void k_elec_scale(float *__restrict__ source, const float *__restrict__ total,
                             float target, size_t N)
{
    size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= N) return;
    float t = total[0];
    float scale = target / (t > 1e-12f ? t : 1e-12f);
    source[c] *= scale;
}

/* elec_jacobi_step kernels.py:1315-1356 */
__global__ void k_elec_jacobi(const float *__restrict__ phi_in, float *__restrict__ phi_out,
                              const float *__restrict__ sigma, const float *__restrict__ source,
                              const uint8_t *__restrict__ flags, float dx, float omega,
                              int nz_solid, Dims d)
{
    int i, j, k;
    if (!d.cell(i, j, k)) return;
    size_t c = d.idx(i, j, k);
    uint8_t f = flags[c];
    if (f == GAS || (k <= nz_solid && f == SOLID)) {
        phi_out[c] = 0.0f;
        return;
    }
    const float eps = 1e-12f;
    float sp = sigma_at(sigma, i + 1, j, k, d), sm = sigma_at(sigma, i - 1, j, k, d);
    float sn = sigma_at(sigma, i, j + 1, k, d), ss = sigma_at(sigma, i, j - 1, k, d);
    float st = sigma_at(sigma, i, j, k + 1, d), sb = sigma_at(sigma, i, j, k - 1, d);
    float denom = sp + sm + sn + ss + st + sb + eps;
    float pn = sp * phi_in[d.idx(imin(i + 1, d.nx - 1), j, k)] +
               sm * phi_in[d.idx(imax(i - 1, 0), j, k)] +
               sn * phi_in[d.idx(i, imin(j + 1, d.ny - 1), k)] +
               ss * phi_in[d.idx(i, imax(j - 1, 0), k)] +
               st * phi_in[d.idx(i, j, imin(k + 1, d.nz - 1))] +
               sb * phi_in[d.idx(i, j, imax(k - 1, 0))];
    float phi_new = (pn + source[c] * dx * dx) / denom;
    phi_out[c] = (1.0f - omega) * phi_in[c] + omega * phi_new;
}

/* elec_l1_diff kernels.py:1384-1396: compensated partial sums of |a - b| and |b| */
__global__ void __launch_bounds__(kBlock) k_elec_l1(const float *__restrict__ a,
                                                    const float *__restrict__ b,
                                                    double *__restrict__ parts, size_t N)
{
    __shared__ double sh_s[kBlock], sh_c[kBlock];
    double s0 = 0.0, c0 = 0.0, s1 = 0.0, c1 = 0.0;
    for (size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x; c < N;
         c += (size_t)gridDim.x * blockDim.x) {
        float av = a[c], bv = b[c];
        double ss, e;
        two_sum(s0, (double)fabsf(av - bv), ss, e);
        s0 = ss;
        c0 += e;
        two_sum(s1, (double)fabsf(bv), ss, e);
        s1 = ss;
        c1 += e;
    }
    block_reduce_pair(s0, c0, sh_s, sh_c);
    if (threadIdx.x == 0) {
        parts[2 * blockIdx.x] = s0;
        parts[2 * blockIdx.x + 1] = c0;
    }
    __syncthreads();
    block_reduce_pair(s1, c1, sh_s, sh_c);
    if (threadIdx.x == 0) {
        parts[2 * (gridDim.x + blockIdx.x)] = s1;
        parts[2 * (gridDim.x + blockIdx.x) + 1] = c1;
    }
}

/* elec_compute_J kernels.py:1359-1381 */
__global__ void k_elec_J(float *__restrict__ Jx, float *__restrict__ Jy, float *__restrict__ Jz,
                         const float *__restrict__ phi, const float *__restrict__ sigma,
                         const uint8_t *__restrict__ flags, float dx, Dims d)
{
    int i, j, k;
    if (!d.cell(i, j, k)) return;
    size_t c = d.idx(i, j, k);
    if (flags[c] == GAS) {
        Jx[c] = 0.0f;
        Jy[c] = 0.0f;
        Jz[c] = 0.0f;
        return;
    }
    float sig = sigma[c];
    float gx = (phi[d.idx(imin(i + 1, d.nx - 1), j, k)] - phi[d.idx(imax(i - 1, 0), j, k)]) /
               (2.0f * dx);
    float gy = (phi[d.idx(i, imin(j + 1, d.ny - 1), k)] - phi[d.idx(i, imax(j - 1, 0), k)]) /
               (2.0f * dx);
    float gz = (phi[d.idx(i, j, imin(k + 1, d.nz - 1))] - phi[d.idx(i, j, imax(k - 1, 0))]) /
               (2.0f * dx);
    Jx[c] = -sig * gx;
    Jy[c] = -sig * gy;
    Jz[c] = -sig * gz;
}

__device__ __forceinline__ int radial_bin(int i, int j, float arc_i, float arc_j, float dr,
                                          int n_bins)
{
    float di = (float)i - arc_i, dj = (float)j - arc_j;
    float r = sqrtf(di * di + dj * dj);
    return imin((int)(r / dr), n_bins - 1);
}

/* elec_bin_axial_current kernels.py:1399-1418: bins[k][b] = sum over the slab's cells of
 * radial bin b of Jz dx dx. Workgroup (k, g) sums bins g*kBinGroup.. of slab k: each thread
 * keeps compensated pairs for those bins over a strided part of the slab, then the workgroup
 * combines the threads in a fixed order. */
__global__ void __launch_bounds__(kBlock) k_elec_bins(const float *__restrict__ Jz,
                                                      float *__restrict__ bins, float arc_i,
                                                      float arc_j, float dx, float dr,
                                                      int n_bins, Dims d)
{
    __shared__ double sh_s[kBlock], sh_c[kBlock];
    int k = blockIdx.x;
    int b0 = blockIdx.y * kBinGroup;
    double s[kBinGroup], e[kBinGroup];
#pragma unroll
    for (int g = 0; g < kBinGroup; ++g) s[g] = e[g] = 0.0;
    int nij = d.nx * d.ny;
    for (int t = threadIdx.x; t < nij; t += blockDim.x) {
        int i = t % d.nx, j = t / d.nx;
        int b = radial_bin(i, j, arc_i, arc_j, dr, n_bins) - b0;
        if (b < 0 || b >= kBinGroup) continue;
        float v = Jz[d.idx(i, j, k)] * dx * dx;
#pragma unroll
        for (int g = 0; g < kBinGroup; ++g)
            if (g == b) {
                double ss, er;
                two_sum(s[g], (double)v, ss, er);
                s[g] = ss;
                e[g] += er;
            }
    }
#pragma unroll
    for (int g = 0; g < kBinGroup; ++g) {
        double a = s[g], c = e[g];
        block_reduce_pair(a, c, sh_s, sh_c);
        if (threadIdx.x == 0 && b0 + g < n_bins) bins[(size_t)k * n_bins + b0 + g] = (float)(a + c);
        __syncthreads();
    }
}

/* elec_prefix_bins kernels.py:1421-1432: running fp32 sum along the bins of each slab */
__global__ void k_elec_prefix(float *__restrict__ bins, int n_bins, int nz)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nz) return;
    float acc = 0.0f;
    for (int b = 0; b < n_bins; ++b) {
        acc += bins[(size_t)k * n_bins + b];
        bins[(size_t)k * n_bins + b] = acc;
    }
}

/* elec_B_axisymmetric kernels.py:1435-1477 */
__global__ void k_elec_B(float *__restrict__ Bx, float *__restrict__ By, float *__restrict__ Bz,
                         const float *__restrict__ bins, float arc_i, float arc_j, float dx,
                         float dr, float mu0, int n_bins, Dims d)
{
    int i, j, k;
    if (!d.cell(i, j, k)) return;
    size_t c = d.idx(i, j, k);
    float di = (float)i - arc_i, dj = (float)j - arc_j;
    float r_cells = sqrtf(di * di + dj * dj);
    float bx = 0.0f, by = 0.0f;
    if (r_cells > 1e-3f) {
        int b = imin((int)(r_cells / dr), n_bins - 1);
        float I_enc = bins[(size_t)k * n_bins + b];
        float r_m = r_cells * dx;
        float B_theta = mu0 * I_enc / (2.0f * 3.14159265358979323846f * r_m);
        bx = -B_theta * dj / r_cells;
        by = B_theta * di / r_cells;
    }
    Bx[c] = bx;
    By[c] = by;
    Bz[c] = 0.0f;
}

/* apply_lorentz_JxB kernels.py:1480-1513 */
__global__ void k_lorentz_JxB(float *__restrict__ Fx, float *__restrict__ Fy,
                              float *__restrict__ Fz, const float *__restrict__ Jx,
                              const float *__restrict__ Jy, const float *__restrict__ Jz,
                              const float *__restrict__ Bx, const float *__restrict__ By,
                              const float *__restrict__ Bz, const float *__restrict__ f_l,
                              const uint8_t *__restrict__ flags, float dt, float dx, float rho,
                              size_t N)
{
    size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= N) return;
    float fl = f_l[c];
    if (flags[c] == GAS || fl < 0.05f) return;
    float fx, fy, fz;
    lorentz_force(Jx[c], Jy[c], Jz[c], Bx[c], By[c], Bz[c], fl, dt, dx, rho, fx, fy, fz);
    Fx[c] += fx;
    Fy[c] += fy;
    Fz[c] += fz;
}

/* ---- the whole solve --------------------------------------------------------------------- */

/* what the convergence test leaves in the scratch buffer for the later launches and the host */
struct ElecStatus {
    float res, norm;
    int sweeps, done;
    float arc_k;
    int bead_top;
};
constexpr size_t kElecStatus = kScratchTelemetry + 40;
static_assert(kElecStatus + sizeof(ElecStatus) <= kScratchTelemetryParts, "status in its line");

/* cell of linear index c; 32-bit divisions where the grid allows them */
__device__ __forceinline__ void elec_ijk(size_t c, const Dims &d, bool small, int &i, int &j,
                                         int &k)
{
    if (!small) {
        d.ijk(c, i, j, k);
        return;
    }
    const unsigned u = (unsigned)c, nf = (unsigned)d.fast(), ny = (unsigned)d.ny;
    const unsigned r = u / nf;
    const int a = (int)(u - r * nf), b = (int)(r / ny);
    j = (int)(r - (unsigned)b * ny);
    i = d.layout == kLayoutZYX ? a : b;
    k = d.layout == kLayoutZYX ? b : a;
}

/* conductivity (k_elec_build_sigma) and the partial sums of the source that k_elec_source and
 * k_elec_source_sum give; the source itself is left to the next launch, which knows its scale */
__global__ void __launch_bounds__(kBlock)
k_elec_setup(float *__restrict__ sigma, const float *__restrict__ f_l,
             const uint8_t *__restrict__ flags, float s_liq, float s_sol, ElecSource e,
             double *__restrict__ parts, ElecStatus *__restrict__ status,
             const int *__restrict__ bead_top, Dims d)
{
    __shared__ double sh_s[kBlock], sh_c[kBlock];
    const size_t N = d.n();
    const bool small = N <= 0xffffffffu;
    if (e.arc_k_dev) {
        e.arc_k = *e.arc_k_dev;
        elec_slabs(e, d.nz);
    }
    double sum = 0.0, comp = 0.0;
    for (size_t c = (size_t)blockIdx.x * kBlock + threadIdx.x; c < N;
         c += (size_t)gridDim.x * kBlock) {
        sigma[c] = flags[c] == GAS ? 1e-8f : (f_l[c] > 0.55f ? s_liq : s_sol);
        int i, j, k;
        elec_ijk(c, d, small, i, j, k);
        if (k < e.k_min || k > e.k_max) continue;
        double ss, er;
        two_sum(sum, (double)(elec_source_at(e, i, j, k) * e.cell_vol), ss, er);
        sum = ss;
        comp += er;
    }
    block_reduce_pair(sum, comp, sh_s, sh_c);
    if (threadIdx.x == 0) {
        parts[2 * blockIdx.x] = sum;
        parts[2 * blockIdx.x + 1] = comp;
        if (blockIdx.x == 0) *status = ElecStatus{0.0f, 0.0f, 0, 0, e.arc_k, bead_top ? *bead_top : -1};
    }
}

/* the source scaled to the current: every block totals the partial pairs for itself (the order of
 * k_pairs_total), which costs less than a launch between */
__global__ void __launch_bounds__(kBlock)
k_elec_scaled_source(float *__restrict__ source, ElecSource e, const double *__restrict__ parts,
                     int nb, float target, Dims d)
{
    __shared__ double sh_s[kBlock], sh_c[kBlock];
    __shared__ float s_scale;
    if (e.arc_k_dev) {
        e.arc_k = *e.arc_k_dev;
        elec_slabs(e, d.nz);
    }
    double sum = 0.0, comp = 0.0;
    for (int b = threadIdx.x; b < nb; b += kBlock) {
        double ss, er;
        two_sum(sum, parts[2 * b], ss, er);
        sum = ss;
        comp += parts[2 * b + 1] + er;
    }
    block_reduce_pair(sum, comp, sh_s, sh_c);
    if (threadIdx.x == 0) {
        float t = (float)(sum + comp);
        s_scale = target / (t > 1e-12f ? t : 1e-12f);
    }
    __syncthreads();
    const float scale = s_scale;
    const size_t N = d.n();
    const bool small = N <= 0xffffffffu;
    for (size_t c = (size_t)blockIdx.x * kBlock + threadIdx.x; c < N;
         c += (size_t)gridDim.x * kBlock) {
        int i, j, k;
        elec_ijk(c, d, small, i, j, k);
        source[c] = elec_source_at(e, i, j, k) * scale;
    }
}

struct ElecSweep {
    const float *in;
    float *out;
    const float *sigma, *source;
    const uint8_t *flags;
    const ElecStatus *status;
    double *parts;  // of the last sweep's L1 sums; null: the sums are not wanted
    float dx, omega;
    int nz_solid, sweeps;
    int copy;       // after convergence carry the potential over to `out`
};

constexpr int kSweepTile = 8;
constexpr int kSweepThreads = 1024;
constexpr int kSweepMax = 5;  // sweeps a launch can take
/* Grids of up to this many tiles take their sweeps in tiles: one for each of the 256 CUs, since a
 * workgroup's LDS leaves no room for a second. From there on a chunk's two launches take as many
 * rounds of 12 us as there are tiles for a CU, and single sweeps, bound by their 4 us launches up
 * to about 300 k cells and by memory above, are the shorter: a step of 80x40x30 (200 tiles) takes
 * 193 us in tiles and 207 sweep by sweep (XYZ layout 225, 234), 80x64x32 (320) 217 and 204 (247,
 * 241), 128x64x40 (640) 241 and 199 (295, 280), 160x80x60 (1600) 328 and 230 (430, 372);
 * 400x200x100 took 2390 in tiles and 1610 entry by entry. */
constexpr int kTiledSweepTiles = 256;

static int64_t sweep_tiles(const Dims &d)
{
    constexpr int T = kSweepTile;
    return (int64_t)((d.nx + T - 1) / T) * ((d.ny + T - 1) / T) * ((d.nz + T - 1) / T);
}

/* Up to five Jacobi sweeps (k_elec_jacobi, the same sums in the same order) of an 8^3 tile in LDS:
 * the tile is loaded with a margin of five cells and each sweep computes what the ones after it
 * still need, the last one the tile itself. That is 3.9 updates for one, and still less than the
 * launches it replaces while each tile has a CU: 80x40x30 (200 tiles) 12.4 us for five sweeps,
 * against five dependent launches at 4.5 us and more each. A thread keeps its four cells of the
 * 16^3 that the first sweep computes, so that conductivities, their sum, the source and the neighbours'
 * places are found once and a sweep is seven LDS reads and the arithmetic (all found again in
 * each sweep: 13.8 us). The L1 sums are those of the last sweep. */
template <bool ZYX>
__global__ void __launch_bounds__(kSweepThreads) k_elec_sweeps(ElecSweep e, Dims d)
{
    constexpr int T = kSweepTile, M = kSweepMax, W = T + 2 * M, W3 = W * W * W;
    constexpr int I = W - 2, P = kSweepThreads / (I * I), C = I / P;  // planes at a time; cells
    static_assert(I == 16 && P * I * I == kSweepThreads, "a thread's cells");
    __shared__ float s_sig[W3], s_phi[2][W3];
    __shared__ double sh_s[kSweepThreads], sh_c[kSweepThreads];
    const int tid = (int)threadIdx.x;
    const int nf = d.fast(), ns = d.slow();
    const int tf = (nf + T - 1) / T, tj = (d.ny + T - 1) / T;
    const bool done = e.status->done != 0;
    if (done && !e.copy) return;
    const int x = tid % I, y = (tid / I) % I, z0 = tid / (I * I);
    const int first = M - e.sweeps + 1;  // sweep m leaves a margin of M - m around the tile
    double s0 = 0.0, c0 = 0.0, s1 = 0.0, c1 = 0.0;
    const int tile = (int)blockIdx.x;  // a workgroup each
    const int a0 = (tile % tf) * T - M, b0 = ((tile / tf) % tj) * T - M,
              g0 = (tile / (tf * tj)) * T - M;
    float *in0 = s_phi[first & 1];
    /* every load of the tile is under way before the first is waited for (a place outside the
     * domain loads a cell of its face, which no sweep reads): a load per pass of a loop with
     * the test inside took a trip to memory per pass, ten trips of 0.8 us */
    constexpr int L = (W3 + kSweepThreads - 1) / kSweepThreads;
    float v_in[L], v_sig[L], src[C];
    uint8_t fl[C];
#pragma unroll
    for (int n = 0; n < L; ++n) {
        const int l = imin(tid + n * kSweepThreads, W3 - 1);
        const int a = imax(0, imin(a0 + l % W, nf - 1));
        const int j = imax(0, imin(b0 + (l / W) % W, d.ny - 1));
        const int b = imax(0, imin(g0 + l / (W * W), ns - 1));
        const size_t c = ((size_t)b * d.ny + j) * nf + a;
        v_in[n] = e.in[c];
        v_sig[n] = e.sigma[c];
    }
    const int a = a0 + x + 1, j = b0 + y + 1;
    const bool col = a >= 0 && a < nf && j >= 0 && j < d.ny;
#pragma unroll
    for (int n = 0; n < C; ++n) {
        const int b = imax(0, imin(g0 + z0 + n * P + 1, ns - 1));
        const size_t c = ((size_t)b * d.ny + imax(0, imin(j, d.ny - 1))) * nf +
                         imax(0, imin(a, nf - 1));
        fl[n] = e.flags[c];
        src[n] = e.source[c];
    }
#pragma unroll
    for (int n = 0; n < L; ++n) {
        const int l = tid + n * kSweepThreads;
        if (l >= W3) break;
        in0[l] = v_in[n];
        s_sig[l] = v_sig[n];
    }
    bool zero[C];
#pragma unroll
    for (int n = 0; n < C; ++n) {
        const int b = g0 + z0 + n * P + 1;
        zero[n] = fl[n] == GAS || ((ZYX ? b : a) <= e.nz_solid && fl[n] == SOLID);
        src[n] = src[n] * e.dx * e.dx;
    }
    __syncthreads();
    /* the neighbours' places (the cell's own at the domain's faces) and conductivities */
    const int ap = a + 1 < nf ? 1 : 0, am = a > 0 ? -1 : 0;
    const int jp = j + 1 < d.ny ? W : 0, jm = j > 0 ? -W : 0;
    int bp[C], bm[C];
    float sp[C], sm[C], sn[C], ss[C], st[C], sb[C], denom[C];
#pragma unroll
    for (int n = 0; n < C; ++n) {
        const int zl = z0 + n * P, b = g0 + zl + 1;
        const int l = ((zl + 1) * W + y + 1) * W + x + 1;
        bp[n] = b + 1 < ns ? W * W : 0;
        bm[n] = b > 0 ? -W * W : 0;
        sp[n] = s_sig[l + (ZYX ? ap : bp[n])];
        sm[n] = s_sig[l + (ZYX ? am : bm[n])];
        sn[n] = s_sig[l + jp];
        ss[n] = s_sig[l + jm];
        st[n] = s_sig[l + (ZYX ? bp[n] : ap)];
        sb[n] = s_sig[l + (ZYX ? bm[n] : am)];
        const float eps = 1e-12f;
        denom[n] = sp[n] + sm[n] + sn[n] + ss[n] + st[n] + sb[n] + eps;
    }
    for (int m = first; m <= M; ++m) {
        const float *pin = s_phi[m & 1];
        float *pout = s_phi[(m + 1) & 1];
        const int lo = m - 1, hi = I - m;  // of the cells this sweep computes
        if (col && x >= lo && x <= hi && y >= lo && y <= hi) {
#pragma unroll
            for (int n = 0; n < C; ++n) {
                const int zl = z0 + n * P, b = g0 + zl + 1;
                if (zl < lo || zl > hi || b < 0 || b >= ns) continue;
                const int l = ((zl + 1) * W + y + 1) * W + x + 1;
                const float *q = pin + l;
                const float old = q[0];
                float pn = sp[n] * q[ZYX ? ap : bp[n]] + sm[n] * q[ZYX ? am : bm[n]] +
                           sn[n] * q[jp] + ss[n] * q[jm] + st[n] * q[ZYX ? bp[n] : ap] +
                           sb[n] * q[ZYX ? bm[n] : am];
                float phi_new = (pn + src[n]) / denom[n];
                float now = (1.0f - e.omega) * old + e.omega * phi_new;
                if (zero[n]) now = 0.0f;
                if (m < M) {
                    pout[l] = now;
                    continue;
                }
                if (done) now = old;
                e.out[((size_t)b * d.ny + j) * nf + a] = now;
                if (e.parts) {
                    double sum, er;
                    two_sum(s0, (double)fabsf(now - old), sum, er);
                    s0 = sum;
                    c0 += er;
                    two_sum(s1, (double)fabsf(old), sum, er);
                    s1 = sum;
                    c1 += er;
                }
            }
        }
        __syncthreads();
    }
    if (!e.parts || done) return;
    block_reduce_pair(s0, c0, sh_s, sh_c);
    if (tid == 0) {
        e.parts[2 * blockIdx.x] = s0;
        e.parts[2 * blockIdx.x + 1] = c0;
    }
    __syncthreads();
    block_reduce_pair(s1, c1, sh_s, sh_c);
    if (tid == 0) {
        e.parts[2 * (gridDim.x + blockIdx.x)] = s1;
        e.parts[2 * (gridDim.x + blockIdx.x) + 1] = c1;
    }
}

/* the convergence test after a chunk of sweeps; later launches of a converged solve end at once */
__global__ void __launch_bounds__(kBlock)
k_elec_check(const double *__restrict__ parts, int nb, int sweeps, double tol,
             float *__restrict__ l1, ElecStatus *__restrict__ status)
{
    __shared__ double sh_s[kBlock], sh_c[kBlock];
    if (status->done) return;
    float v[2];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const double *p = parts + 2 * (size_t)w * nb;
        double sum = 0.0, comp = 0.0;
        for (int b = threadIdx.x; b < nb; b += kBlock) {
            double ss, er;
            two_sum(sum, p[2 * b], ss, er);
            sum = ss;
            comp += p[2 * b + 1] + er;
        }
        block_reduce_pair(sum, comp, sh_s, sh_c);
        v[w] = (float)(sum + comp);
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    l1[0] = v[0];
    l1[1] = v[1];
    const double norm = (double)v[1];
    const double rel = (double)v[0] / (1e-30 > norm ? 1e-30 : norm);
    status->res = v[0];
    status->norm = v[1];
    status->sweeps += sweeps;
    status->done = rel < tol ? 1 : 0;
}

constexpr int kJBinGroup = 4;  // radial bins per workgroup of k_elec_J_bins
constexpr int kJBinThreads = 512;
constexpr int kJBinCells = 512;  // cells a wavefront lists before it computes them

/* J (k_elec_J) and the slab's axial current per radius (k_elec_bins) from one read of the
 * potential, x rows contiguous: workgroup (k, g) owns the cells of its slab that lie in its bins.
 * A wavefront goes through its rows without touching memory, lists those cells and computes them
 * with full lanes: what bounds the launch is the looking, so a row beyond the bins is passed over
 * by its j, a cell by its squared radius, and only the rest sees the root and division of the
 * exact test. 80x40x30: 11 us, 17 with the loads in the loop that looks, 14 with the
 * division of a flat index and every cell tested. gate set: only if the potential has converged. */
__global__ void __launch_bounds__(kJBinThreads)
k_elec_J_bins(float *__restrict__ Jx, float *__restrict__ Jy, float *__restrict__ Jz,
              float *__restrict__ bins, const float *__restrict__ phi,
              const float *__restrict__ sigma, const uint8_t *__restrict__ flags, float arc_i,
              float arc_j, float dx, float dr, int n_bins, const ElecStatus *__restrict__ gate,
              Dims d)
{
    constexpr int kWaves = kJBinThreads / 64;
    __shared__ double sh_s[kWaves][kJBinGroup], sh_c[kWaves][kJBinGroup];
    __shared__ uint32_t s_list[kWaves][kJBinCells];
    if (gate && !gate->done) return;
    const int k = blockIdx.x, b0 = blockIdx.y * kJBinGroup;
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    uint32_t *list = s_list[wave];
    double s[kJBinGroup], e[kJBinGroup];
#pragma unroll
    for (int g = 0; g < kJBinGroup; ++g) s[g] = e[g] = 0.0;
    const float *pk = phi + (size_t)k * d.ny * d.nx;
    const int64_t slab = (int64_t)d.ny * d.nx;
    const int64_t up = k + 1 < d.nz ? slab : 0, down = k > 0 ? -slab : 0;
    int n = 0;
    /* the list passes between lanes of one wavefront, whose LDS accesses keep their order: what
     * must not happen is that the compiler moves them past each other */
    auto handover = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    auto compute = [&]() {
        handover();
        for (int q = lane; q < n; q += 64) {
            const uint32_t w = list[q];
            const int b = (int)(w % kJBinGroup), t = (int)(w / kJBinGroup);
            const int j = t / d.nx, i = t - j * d.nx;
            const size_t c = (size_t)k * slab + t;
            const float *p = pk + t;
            const uint8_t f = flags[c];
            float sig = sigma[c];
            float gx = (p[i + 1 < d.nx ? 1 : 0] - p[i > 0 ? -1 : 0]) / (2.0f * dx);
            float gy = (p[j + 1 < d.ny ? d.nx : 0] - p[j > 0 ? -d.nx : 0]) / (2.0f * dx);
            float gz = (p[up] - p[down]) / (2.0f * dx);
            const float jz = f == GAS ? 0.0f : -sig * gz;
            Jx[c] = f == GAS ? 0.0f : -sig * gx;
            Jy[c] = f == GAS ? 0.0f : -sig * gy;
            Jz[c] = jz;
            const float v = jz * dx * dx;
#pragma unroll
            for (int g = 0; g < kJBinGroup; ++g)
                if (g == b) {
                    double ss, er;
                    two_sum(s[g], (double)v, ss, er);
                    s[g] = ss;
                    e[g] += er;
                }
        }
        n = 0;
        handover();
    };
    /* squared radii that the exact test need not see, a little wide; the last bin takes everything
     * beyond it */
    const float lo = fmaxf(((float)b0 - 0.01f) * dr, 0.0f);
    const float hi = ((float)(b0 + kJBinGroup) + 0.01f) * dr;
    const float lo2 = lo * lo * 0.999f;
    const float hi2 = b0 + kJBinGroup >= n_bins ? INFINITY : hi * hi * 1.001f;
    for (int j = wave; j < d.ny; j += kWaves) {
        const float dj = (float)j - arc_j, dj2 = dj * dj;
        if (dj2 > hi2) continue;
        for (int i0 = 0; i0 < d.nx; i0 += 64) {
            const int i = i0 + lane;
            const float di = (float)i - arc_i, r2 = di * di + dj2;
            const bool near = i < d.nx && !(r2 < lo2) && !(r2 > hi2);
            if (__ballot(near) == 0ull) continue;
            const int b = near ? radial_bin(i, j, arc_i, arc_j, dr, n_bins) - b0 : -1;
            const bool mine = b >= 0 && b < kJBinGroup;
            const unsigned long long m = __ballot(mine);
            if (mine)
                list[n + __popcll(m & ((1ull << lane) - 1ull))] =
                    (uint32_t)(j * d.nx + i) * kJBinGroup + (uint32_t)b;
            n += __popcll(m);
            if (n > kJBinCells - 64) compute();
        }
    }
    compute();
    /* the bins' pairs side by side: lanes by shuffles, then wavefronts in order */
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
        for (int g = 0; g < kJBinGroup; ++g) {
            const double os = shfl_down64(s[g], off), oc = shfl_down64(e[g], off);
            double ss, er;
            two_sum(s[g], os, ss, er);
            s[g] = ss;
            e[g] = e[g] + oc + er;
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int g = 0; g < kJBinGroup; ++g) {
            sh_s[wave][g] = s[g];
            sh_c[wave][g] = e[g];
        }
    }
    __syncthreads();
    const int g = (int)threadIdx.x;
    if (g >= kJBinGroup || b0 + g >= n_bins) return;
    double sum = sh_s[0][g], comp = sh_c[0][g];
    for (int w = 1; w < kWaves; ++w) {
        double ss, er;
        two_sum(sum, sh_s[w][g], ss, er);
        sum = ss;
        comp += sh_c[w][g] + er;
    }
    bins[(size_t)k * n_bins + b0 + g] = (float)(sum + comp);
}

constexpr int kForceCells = 1024;  // cells of a slab per workgroup of k_lorentz_force
constexpr int kElecMaxBins = 4096;

struct ElecForce {
    float *Fx, *Fy, *Fz, *Bx, *By, *Bz, *bins;
    const float *raw, *Jx, *Jy, *Jz, *f_l;
    const uint8_t *flags;
    const ElecStatus *gate;  // set: only if the potential has converged
    float arc_i, arc_j, dx, dr, mu0, dt, rho;
    int n_bins, force;       // force 0: J and B are wanted, the step adds the force itself
};

/* enclosed current (k_elec_prefix), self field (k_elec_B) and body force (k_lorentz_JxB) of a piece
 * of a slab: the prefix of the slab's bins is short enough for every workgroup to form it, from
 * the bins as k_elec_J_bins left them (a second array, since the first piece stores the sums) */
__global__ void __launch_bounds__(kBlock) k_lorentz_force(ElecForce e, Dims d)
{
    __shared__ float s_bins[kElecMaxBins];
    if (e.gate && !e.gate->done) return;
    const int k = blockIdx.y;
    for (int b = threadIdx.x; b < e.n_bins; b += kBlock)
        s_bins[b] = e.raw[(size_t)k * e.n_bins + b];
    __syncthreads();
    if (threadIdx.x == 0) {
        float acc = 0.0f;
        for (int b = 0; b < e.n_bins; ++b) {
            acc += s_bins[b];
            s_bins[b] = acc;
        }
    }
    __syncthreads();
    if (blockIdx.x == 0)
        for (int b = threadIdx.x; b < e.n_bins; b += kBlock)
            e.bins[(size_t)k * e.n_bins + b] = s_bins[b];
    const int nij = d.nx * d.ny;
    const int t1 = imin(nij, ((int)blockIdx.x + 1) * kForceCells);
    for (int t = (int)blockIdx.x * kForceCells + (int)threadIdx.x; t < t1; t += kBlock) {
        const int j = t / d.nx, i = t - j * d.nx;
        const size_t c = d.idx(i, j, k);
        float di = (float)i - e.arc_i, dj = (float)j - e.arc_j;
        float r_cells = sqrtf(di * di + dj * dj);
        float bx = 0.0f, by = 0.0f;
        if (r_cells > 1e-3f) {
            int b = imin((int)(r_cells / e.dr), e.n_bins - 1);
            float I_enc = s_bins[b];
            float r_m = r_cells * e.dx;
            float B_theta = e.mu0 * I_enc / (2.0f * 3.14159265358979323846f * r_m);
            bx = -B_theta * dj / r_cells;
            by = B_theta * di / r_cells;
        }
        e.Bx[c] = bx;
        e.By[c] = by;
        e.Bz[c] = 0.0f;
        if (!e.force) continue;
        float fl = e.f_l[c], fx, fy, fz;
        if (e.flags[c] == GAS || fl < 0.05f) continue;
        lorentz_force(e.Jx[c], e.Jy[c], e.Jz[c], bx, by, 0.0f, fl, e.dt, e.dx, e.rho, fx, fy, fz);
        e.Fx[c] += fx;
        e.Fy[c] += fy;
        e.Fz[c] += fz;
    }
}

}  // namespace waam

namespace waam {

int check_lorentz(const char *who, const waam_lorentz &q)
{
    WAAM_RETURN_IF(check_dims(who, q.nx, q.ny, q.nz, q.layout));
    WAAM_RETURN_IF(check_ptrs(who, {q.phi, q.phi_tmp, q.sigma, q.source, q.Jx, q.Jy, q.Jz, q.Bx,
                                    q.By, q.Bz, q.bins, q.l1}));
    if (q.phi == q.phi_tmp || q.bins == q.bins_raw)
        return set_error(WAAM_ERR_INVALID, "%s: buffers alias", who);
    if (q.max_sweeps <= 0)
        return set_error(WAAM_ERR_INVALID, "%s: max_sweeps %d", who, q.max_sweeps);
    if (q.n_bins <= 0 || q.n_bins > kElecMaxBins || !(q.bin_dr > 0.0f))
        return set_error(WAAM_ERR_INVALID, "%s: bins", who);
    return WAAM_OK;
}

/* whether J, the bins, B and the force run in the kernels that take a slab piece by piece. They
 * need x rows contiguous (in the XYZ layout a slab's cells lie a row apart and such a piece would
 * read a line for every cell), the second array of bins and, since k_elec_J_bins lists a cell with
 * its bin in one word, a slab of less than 2^29 cells. Every other solve takes the entries'
 * kernels. */
static bool by_slab(const waam_lorentz &q)
{
    return q.layout == kLayoutZYX && q.bins_raw &&
           (int64_t)q.nx * q.ny <= (int64_t)(0x7fffffff / kJBinGroup);
}

int lorentz_run(const char *who, const waam_lorentz &q, const float *arc_k_dev, bool force,
                waam_lorentz_result &out, hipStream_t st)
{
    Dims d{q.nx, q.ny, q.nz, q.layout};
    const bool zyx = q.layout == kLayoutZYX, slabs = by_slab(q);
    const size_t N = d.n();
    double *src_parts = reinterpret_cast<double *>((char *)q.scratch + kScratchPartials);
    double *l1_parts = reinterpret_cast<double *>((char *)q.scratch + kScratchTelemetryParts);
    ElecStatus *status = reinterpret_cast<ElecStatus *>((char *)q.scratch + kElecStatus);
    ElecSource e = elec_source(q.arc_i, q.arc_j, q.arc_k, q.sigma_cells, q.current, q.dx, q.nz,
                               arc_k_dev);
    const int nb = (int)(grid_for(N) < (unsigned)kReduceBlocks ? grid_for(N) : kReduceBlocks);
    hipLaunchKernelGGL(k_elec_setup, dim3(nb), dim3(kBlock), 0, st, q.sigma, q.f_l, q.flags,
                       q.sigma_liquid, q.sigma_solid, e, src_parts, status, q.bead_top, d);
    hipLaunchKernelGGL(k_elec_scaled_source, dim3(nb), dim3(kBlock), 0, st, q.source, e, src_parts,
                       nb, q.current, d);
    float *in = q.phi, *other = q.phi_tmp;
    if (q.cold)
        hipLaunchKernelGGL(k_fill, dim3(grid_for(N)), dim3(kBlock), 0, st, in, 0.0f, N);
    const int64_t tiles = sweep_tiles(d);
    const bool tiled = tiles <= kTiledSweepTiles;
    const int blocks = tiled ? (int)tiles : kLorentzSumBlocks;  // that leave L1 sums

    auto sweeps = [&](int n) {
        for (int first = 1, m = n; m > 0; first = 0) {
            const int now = first ? (m + 1) / 2 : m;
            m -= now;
            ElecSweep sw{in,
                         other,
                         q.sigma,
                         q.source,
                         q.flags,
                         status,
                         m == 0 ? l1_parts : nullptr,
                         q.dx,
                         q.omega,
                         q.nz_solid,
                         now,
                         n == 1 ? 1 : 0};
            if (zyx)
                hipLaunchKernelGGL(k_elec_sweeps<true>, dim3(blocks), dim3(kSweepThreads), 0, st,
                                   sw, d);
            else
                hipLaunchKernelGGL(k_elec_sweeps<false>, dim3(blocks), dim3(kSweepThreads), 0, st,
                                   sw, d);
            std::swap(in, other);
        }
    };
    auto single_sweeps = [&](int n) {
        for (int m = n; m > 0; --m) {
            hipLaunchKernelGGL(k_elec_jacobi, grid3(d), block3(), 0, st, in, other, q.sigma,
                               q.source, q.flags, q.dx, q.omega, q.nz_solid, d);
            std::swap(in, other);
        }
        hipLaunchKernelGGL(k_elec_l1, dim3(blocks), dim3(kBlock), 0, st, (const float *)in,
                           (const float *)other, l1_parts, N);
    };
    auto sweep_chunk = [&](int n) {
        if (tiled) sweeps(n);
        else single_sweeps(n);
        hipLaunchKernelGGL(k_elec_check, dim3(1), dim3(kBlock), 0, st, l1_parts, blocks, n, q.tol,
                           q.l1, status);
    };
    auto fields = [&](const ElecStatus *gate) {
        const dim3 bins_grid((unsigned)d.nz,
                             (unsigned)((q.n_bins + kJBinGroup - 1) / kJBinGroup));
        if (slabs) {
            hipLaunchKernelGGL(k_elec_J_bins, bins_grid, dim3(kJBinThreads), 0, st, q.Jx, q.Jy,
                               q.Jz, q.bins_raw, in, q.sigma, q.flags, q.arc_i, q.arc_j, q.dx,
                               q.bin_dr, q.n_bins, gate, d);
            ElecForce f{q.Fx,  q.Fy,    q.Fz, q.Bx,    q.By,    q.Bz, q.bins,   q.bins_raw,
                        q.Jx,  q.Jy,    q.Jz, q.f_l,   q.flags, gate, q.arc_i,  q.arc_j,
                        q.dx,  q.bin_dr, q.mu0, q.dt,  q.rho,   q.n_bins, force ? 1 : 0};
            const int64_t nij = (int64_t)d.nx * d.ny;
            hipLaunchKernelGGL(
                k_lorentz_force,
                dim3((unsigned)((nij + kForceCells - 1) / kForceCells), (unsigned)d.nz),
                dim3(kBlock), 0, st, f, d);
            return;
        }
        hipLaunchKernelGGL(k_elec_J, grid3(d), block3(), 0, st, q.Jx, q.Jy, q.Jz, in, q.sigma,
                           q.flags, q.dx, d);
        hipLaunchKernelGGL(k_elec_bins,
                           dim3((unsigned)d.nz, (unsigned)((q.n_bins + kBinGroup - 1) / kBinGroup)),
                           dim3(kBlock), 0, st, q.Jz, q.bins, q.arc_i, q.arc_j, q.dx, q.bin_dr,
                           q.n_bins, d);
        hipLaunchKernelGGL(k_elec_prefix, dim3(grid_for((size_t)d.nz, 64)), dim3(64), 0, st, q.bins,
                           q.n_bins, d.nz);
        hipLaunchKernelGGL(k_elec_B, grid3(d), block3(), 0, st, q.Bx, q.By, q.Bz, q.bins, q.arc_i,
                           q.arc_j, q.dx, q.bin_dr, q.mu0, q.n_bins, d);
        if (force)
            hipLaunchKernelGGL(k_lorentz_JxB, dim3(grid_for(N)), dim3(kBlock), 0, st, q.Fx, q.Fy,
                               q.Fz, q.Jx, q.Jy, q.Jz, q.Bx, q.By, q.Bz, q.f_l, q.flags, q.dt,
                               q.dx, q.rho, N);
    };

    /* A warm solve mostly converges in its first chunk: that one is read by itself, with the field
     * kernels queued behind it (they run only if it did). One that does not is likely to take the
     * rest of a usual limit of 40 sweeps: the chunks after it go out in groups, and a group whose
     * early chunks converge leaves launches that end at once. Single sweeps are read chunk by
     * chunk: they do not look at the test. */
    ElecStatus h{};
    int launched = 0, group = 1;
    while (launched < q.max_sweeps && !h.done) {
        const bool first = launched == 0;
        for (int g = 0; g < group && launched < q.max_sweeps; ++g) {
            const int left = q.max_sweeps - launched, n = left < 10 ? left : 10;
            sweep_chunk(n);
            launched += n;
        }
        if (first && slabs) fields(status);
        WAAM_RETURN_IF(check_launch(who));
        hipError_t rc = hipMemcpyAsync(&h, status, sizeof(h), hipMemcpyDeviceToHost, st);
        if (rc == hipSuccess) rc = hipStreamSynchronize(st);
        if (rc != hipSuccess)
            return set_error(WAAM_ERR_HIP, "%s: %s", who, hipGetErrorString(rc));
        if (!(first && slabs && h.done) && (h.done || launched >= q.max_sweeps)) fields(nullptr);
        group = !tiled ? 1 : (first ? 3 : 4);
    }
    out.res = h.res;
    out.norm = h.norm;
    out.sweeps = h.sweeps;
    out.converged = h.done;
    out.arc_k = h.arc_k;
    out.bead_top = h.bead_top;
    out.in_tmp = in == q.phi_tmp ? 1 : 0;
    return check_launch(who);
}

}  // namespace waam

using namespace waam;

extern "C" {

int waam_elec_build_sigma(float *sigma, const float *f_l, const uint8_t *flags,
                          float sigma_liquid, float sigma_solid, int64_t n, void *stream)
{
    if (n <= 0) return set_error(WAAM_ERR_INVALID, "waam_elec_build_sigma: n <= 0");
    WAAM_RETURN_IF(check_ptrs("waam_elec_build_sigma", {sigma, f_l, flags}));
    hipLaunchKernelGGL(k_elec_build_sigma, dim3(grid_for((size_t)n)), dim3(kBlock), 0,
                       as_stream(stream), sigma, f_l, flags, sigma_liquid, sigma_solid, (size_t)n);
    return check_launch("waam_elec_build_sigma");
}

int waam_elec_clear_source(float *source, int64_t n, void *stream)
{
    if (n <= 0) return set_error(WAAM_ERR_INVALID, "waam_elec_clear_source: n <= 0");
    WAAM_RETURN_IF(check_ptrs("waam_elec_clear_source", {source}));
    hipLaunchKernelGGL(k_fill, dim3(grid_for((size_t)n)), dim3(kBlock), 0, as_stream(stream),
                       source, 0.0f, (size_t)n);
    return check_launch("waam_elec_clear_source");
}

int waam_elec_inject_arc_source(float *source, float arc_i, float arc_j, float arc_k,
                                float sigma_cells, float current_A, float dx, int nx, int ny,
                                int nz, int layout, void *stream)
{
    WAAM_RETURN_IF(check_dims("waam_elec_inject_arc_source", nx, ny, nz, layout));
    WAAM_RETURN_IF(check_ptrs("waam_elec_inject_arc_source", {source}));
    Dims d{nx, ny, nz, layout};
    ElecSource e = elec_source(arc_i, arc_j, arc_k, sigma_cells, current_A, dx, nz);
    hipLaunchKernelGGL(k_elec_source, grid3(d), block3(), 0, as_stream(stream), source, e, d);
    return check_launch("waam_elec_inject_arc_source");
}

int waam_elec_normalize_source(float *source, float target_current_A, float dx, int64_t n,
                               void *scratch, void *stream)
{
    if (n <= 0) return set_error(WAAM_ERR_INVALID, "waam_elec_normalize_source: n <= 0");
    WAAM_RETURN_IF(check_ptrs("waam_elec_normalize_source", {source, scratch}));
    hipStream_t s = as_stream(stream);
    double *parts = reinterpret_cast<double *>((char *)scratch + kScratchPartials);
    float *total = reinterpret_cast<float *>((char *)scratch + kScratchTelemetry) + 8;
    hipLaunchKernelGGL(k_elec_source_sum, dim3(kLorentzSumBlocks), dim3(kBlock), 0, s, source,
                       dx * dx * dx, parts, (size_t)n);
    hipLaunchKernelGGL(k_pairs_total, dim3(1), dim3(kBlock), 0, s, parts, kLorentzSumBlocks,
                       total);
    hipLaunchKernelGGL(k_elec_scale, dim3(grid_for((size_t)n)), dim3(kBlock), 0, s, source, total,
                       target_current_A, (size_t)n);
    return check_launch("waam_elec_normalize_source");
}

int waam_elec_init_ground(float *phi, int64_t n, void *stream)
{
    if (n <= 0) return set_error(WAAM_ERR_INVALID, "waam_elec_init_ground: n <= 0");
    WAAM_RETURN_IF(check_ptrs("waam_elec_init_ground", {phi}));
    hipLaunchKernelGGL(k_fill, dim3(grid_for((size_t)n)), dim3(kBlock), 0, as_stream(stream), phi,
                       0.0f, (size_t)n);
    return check_launch("waam_elec_init_ground");
}

int waam_elec_jacobi_step(const float *phi_in, float *phi_out, const float *sigma,
                          const float *source, const uint8_t *flags, float dx, float omega_j,
                          int nz_solid, int nx, int ny, int nz, int layout, void *stream)
{
    WAAM_RETURN_IF(check_dims("waam_elec_jacobi_step", nx, ny, nz, layout));
    WAAM_RETURN_IF(check_ptrs("waam_elec_jacobi_step", {phi_in, phi_out, sigma, source, flags}));
    if (phi_in == phi_out)
        return set_error(WAAM_ERR_INVALID, "waam_elec_jacobi_step: phi_in aliases phi_out");
    Dims d{nx, ny, nz, layout};
    hipLaunchKernelGGL(k_elec_jacobi, grid3(d), block3(), 0, as_stream(stream), phi_in, phi_out,
                       sigma, source, flags, dx, omega_j, nz_solid, d);
    return check_launch("waam_elec_jacobi_step");
}

int waam_elec_l1_diff(const float *a, const float *b, float *out, int64_t n, void *scratch,
                      void *stream)
{
    if (n <= 0) return set_error(WAAM_ERR_INVALID, "waam_elec_l1_diff: n <= 0");
    WAAM_RETURN_IF(check_ptrs("waam_elec_l1_diff", {a, b, out, scratch}));
    hipStream_t s = as_stream(stream);
    double *parts = reinterpret_cast<double *>((char *)scratch + kScratchTelemetryParts);
    const int nb = kLorentzSumBlocks;
    hipLaunchKernelGGL(k_elec_l1, dim3(nb), dim3(kBlock), 0, s, a, b, parts, (size_t)n);
    hipLaunchKernelGGL(k_pairs_total, dim3(1), dim3(kBlock), 0, s, parts, nb, out);
    hipLaunchKernelGGL(k_pairs_total, dim3(1), dim3(kBlock), 0, s, parts + 2 * nb, nb, out + 1);
    return check_launch("waam_elec_l1_diff");
}

int waam_elec_compute_J(float *Jx, float *Jy, float *Jz, const float *phi, const float *sigma,
                        const uint8_t *flags, float dx, int nx, int ny, int nz, int layout,
                        void *stream)
{
    WAAM_RETURN_IF(check_dims("waam_elec_compute_J", nx, ny, nz, layout));
    WAAM_RETURN_IF(check_ptrs("waam_elec_compute_J", {Jx, Jy, Jz, phi, sigma, flags}));
    Dims d{nx, ny, nz, layout};
    hipLaunchKernelGGL(k_elec_J, grid3(d), block3(), 0, as_stream(stream), Jx, Jy, Jz, phi, sigma,
                       flags, dx, d);
    return check_launch("waam_elec_compute_J");
}

int waam_elec_bin_axial_current(const float *Jz, float *bins, float arc_i, float arc_j, float dx,
                                float bin_dr_cells, int n_bins, int nx, int ny, int nz,
                                int layout, void *stream)
{
    WAAM_RETURN_IF(check_dims("waam_elec_bin_axial_current", nx, ny, nz, layout));
    WAAM_RETURN_IF(check_ptrs("waam_elec_bin_axial_current", {Jz, bins}));
    if (n_bins <= 0 || n_bins > 4096)
        return set_error(WAAM_ERR_INVALID, "waam_elec_bin_axial_current: n_bins %d", n_bins);
    if (!(bin_dr_cells > 0.0f))
        return set_error(WAAM_ERR_INVALID, "waam_elec_bin_axial_current: bin width <= 0");
    Dims d{nx, ny, nz, layout};
    dim3 g((unsigned)nz, (unsigned)((n_bins + kBinGroup - 1) / kBinGroup));
    hipLaunchKernelGGL(k_elec_bins, g, dim3(kBlock), 0, as_stream(stream), Jz, bins, arc_i, arc_j,
                       dx, bin_dr_cells, n_bins, d);
    return check_launch("waam_elec_bin_axial_current");
}

int waam_elec_prefix_bins(float *bins, int n_bins, int nz, void *stream)
{
    if (n_bins <= 0 || nz <= 0) return set_error(WAAM_ERR_INVALID, "waam_elec_prefix_bins: size");
    WAAM_RETURN_IF(check_ptrs("waam_elec_prefix_bins", {bins}));
    hipLaunchKernelGGL(k_elec_prefix, dim3(grid_for((size_t)nz, 64)), dim3(64), 0,
                       as_stream(stream), bins, n_bins, nz);
    return check_launch("waam_elec_prefix_bins");
}

int waam_elec_B_axisymmetric(float *Bx, float *By, float *Bz, const float *bins, float arc_i,
                             float arc_j, float dx, float bin_dr_cells, float mu0, int n_bins,
                             int nx, int ny, int nz, int layout, void *stream)
{
    WAAM_RETURN_IF(check_dims("waam_elec_B_axisymmetric", nx, ny, nz, layout));
    WAAM_RETURN_IF(check_ptrs("waam_elec_B_axisymmetric", {Bx, By, Bz, bins}));
    if (n_bins <= 0 || !(bin_dr_cells > 0.0f))
        return set_error(WAAM_ERR_INVALID, "waam_elec_B_axisymmetric: bins");
    Dims d{nx, ny, nz, layout};
    hipLaunchKernelGGL(k_elec_B, grid3(d), block3(), 0, as_stream(stream), Bx, By, Bz, bins, arc_i,
                       arc_j, dx, bin_dr_cells, mu0, n_bins, d);
    return check_launch("waam_elec_B_axisymmetric");
}

int waam_apply_lorentz_JxB(float *Fx, float *Fy, float *Fz, const float *Jx, const float *Jy,
                           const float *Jz, const float *Bx, const float *By, const float *Bz,
                           const float *f_l, const uint8_t *flags, float dt, float dx,
                           float rho_ref, int64_t n, void *stream)
{
    if (n <= 0) return set_error(WAAM_ERR_INVALID, "waam_apply_lorentz_JxB: n <= 0");
    WAAM_RETURN_IF(check_ptrs("waam_apply_lorentz_JxB", {Fx, Fy, Fz, Jx, Jy, Jz, Bx, By, Bz, f_l,
                                                         flags}));
    hipLaunchKernelGGL(k_lorentz_JxB, dim3(grid_for((size_t)n)), dim3(kBlock), 0,
                       as_stream(stream), Fx, Fy, Fz, Jx, Jy, Jz, Bx, By, Bz, f_l, flags, dt, dx,
                       rho_ref, (size_t)n);
    return check_launch("waam_apply_lorentz_JxB");
}

int waam_lorentz_solve(const waam_lorentz *q, waam_lorentz_result *out, void *stream)
{
    if (!q || !out) return set_error(WAAM_ERR_INVALID, "waam_lorentz_solve: null argument");
    WAAM_RETURN_IF(check_lorentz("waam_lorentz_solve", *q));
    WAAM_RETURN_IF(check_ptrs("waam_lorentz_solve", {q->Fx, q->Fy, q->Fz, q->f_l, q->flags,
                                                     q->scratch}));
    return lorentz_run("waam_lorentz_solve", *q, nullptr, true, *out, as_stream(stream));
}

}  // extern "C"
