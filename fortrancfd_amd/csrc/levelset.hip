// levelset.hip — level-set kernels of the two-phase step on MI355X:
//   * ls_funs / rho_mu / ls_mv        (`.../interface_solver/others.f90:56-176`)
//   * WENO5 flux-split advection with SSP-RK3
//                                     (`.../interface_solver/level_set_rk3_solver.f90:1-219`)
//   * PDE reinitialisation with the mass-constrained lambda
//                                     (`.../interface_solver/level_set_rk3_redis.f90:1-410`)
//   * mass-preserving correction      (`.../interface_solver/mass_preserving_level_set.f90:1-54`)
// Paths are under `Two phase flows/newOpenMP/3D+IBM/` (2D twins under `2D/`).
//
// Layout: reference column-major ghosted arrays.  One thread per interior cell,
// 64 threads along i (the contiguous axis) per wavefront, so every stencil
// load of a wavefront is a contiguous 512-byte run.  Intermediate arrays that
// the reference fills and then ghost-copies with bc() (the flux split s1/s2,
// the backward differences, the lambda numerator/denominator) are recomputed
// or read with clamped indices instead of being stored with ghosts.
#include <algorithm>
#include <mutex>

#include "fcfd_internal.h"
#include "weno.h"

using namespace fcfd;

namespace fcfd {

constexpr double kPi = 3.141592653589793;  // dacos(-1.0_8)

// ls_funs for one value (others.f90:62-87)
__device__ __forceinline__ void lsfun(double phi, double w, double &H, double &D) {
    const double eps = 1.0e-12;
    double x = phi / w;
    if (x > 1.0 - eps) {
        H = 1.0; D = 0.0;
    } else if (x < -1.0 + eps) {
        H = 0.0; D = 0.0;
    } else {
        double s, c;
        sincos(kPi * x, &s, &c);
        H = 0.5 * (1.0 + x + s / kPi);
        D = 0.5 * (1.0 + c) / w;
    }
    H = fmax(fmin(H, 1.0), 0.0);
}

// ------------------------------------------------------------- properties
// ls_funs + rho_mu over the full ghosted box (others.f90:56-120)
// (cp != NULL: a batched 2D stack, case t / slab)
__global__ void k_ls_props(const double *__restrict__ phi, double *__restrict__ H, double *__restrict__ D,
                           double *__restrict__ S, double *__restrict__ R, double *__restrict__ M, long n,
                           double w, double r12, double m12, const fcfd_case *__restrict__ cp, long slab) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    if (cp) {
        const fcfd_case &q = cp[t / slab];
        r12 = q.rho_12;
        m12 = q.mu_12;
    }
    double h, d;
    lsfun(phi[t], w, h, d);
    if (H) H[t] = h;
    if (D) D[t] = d;
    if (S) S[t] = 2.0 * h - 1.0;
    if (R) R[t] = h + r12 * (1.0 - h);
    if (M) M[t] = h + m12 * (1.0 - h);
}

int ls_props(fcfd_ctx *c, const double *phi, double *H, double *D, double *S, double *rho, double *mu) {
    long n = c->G.ntot;
    ProfScope ps_(c, R_MISC);
    hipLaunchKernelGGL(k_ls_props, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, phi, H, D, S, rho, mu,
                       n, c->pr.ls_wid, c->pr.rho_12, c->pr.mu_12, c->cases_dev, c->G.sxy);
    FCFD_CHECK(hipGetLastError());
    return FCFD_OK;
}

// ------------------------------------------------------------- reductions
// Deterministic sums over the interior: a fixed grid of RBLK blocks, each
// thread accumulates a fixed strided subset in order, then fixed-shape tree
// reductions in LDS; a second single-block pass sums the block partials.
constexpr int RBLK = 1024;
constexpr int RTHR = 256;


template <int NS>
__device__ __forceinline__ void block_sum_store(double (&acc)[NS], double *partial, int nblocks) {
    __shared__ double sh[NS][RTHR];
    for (int s = 0; s < NS; ++s) sh[s][threadIdx.x] = acc[s];
    __syncthreads();
    for (int w = RTHR / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int s = 0; s < NS; ++s) sh[s][threadIdx.x] += sh[s][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int s = 0; s < NS; ++s) partial[s * nblocks + blockIdx.x] = sh[s][0];
}

// second pass, one block of RTHR threads per case q (blockIdx.x):
// result[q*RES_STRIDE + s] = sum_b partial[s*nb*ncase + q*nb + b]
__global__ void k_reduce_final(const double *__restrict__ partial, double *__restrict__ result, int ns, int nb) {
    __shared__ double sh[RTHR];
    const long ntot = (long)nb * gridDim.x;
    partial += (long)blockIdx.x * nb;
    result += (long)blockIdx.x * RES_STRIDE;
    for (int s = 0; s < ns; ++s) {
        double a = 0.0;
        for (int b = threadIdx.x; b < nb; b += RTHR) a += partial[s * ntot + b];
        sh[threadIdx.x] = a;
        __syncthreads();
        for (int w = RTHR / 2; w > 0; w >>= 1) {
            if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
            __syncthreads();
        }
        if (threadIdx.x == 0) result[s] = sh[0];
        __syncthreads();
    }
}

// mass / volume (ls_mv, others.f90:129-152) and, with nrm != null, the MPLS
// lambda denominator sum delta^2 |grad phi| (2(1-rho12)H + rho12) dV with
// |grad phi| from the CCD normals, written to grad
// (mass_preserving_level_set.f90:17-34).  blockIdx.y is the case of a
// batched 2D stack (its slice; cp holds its rho_12), 0 otherwise; each case
// reduces over its own RBLK blocks in the same order as a single case.
template <int DIM>
__global__ void k_mass_sums(const double *__restrict__ phi, const double *__restrict__ nx_,
                            const double *__restrict__ ny_, const double *__restrict__ nz_,
                            double *__restrict__ grad, double *__restrict__ partial, Geom G, double w,
                            double r12, int with_lam, const fcfd_case *__restrict__ cp) {
    double acc[3] = {0.0, 0.0, 0.0};
    const int q = blockIdx.y;
    if (cp) r12 = cp[q].rho_12;
    const long n = DIM == 3 ? (long)G.nx * G.ny * G.nz : (long)G.nx * G.ny;
    const double dv = DIM == 3 ? G.dx * G.dy * G.dz : G.dx * G.dy;
    for (long t = (long)blockIdx.x * RTHR + threadIdx.x; t < n; t += (long)RBLK * RTHR) {
        int i, j, k;
        cell_of_index(t, G, i, j, k);
        if (DIM == 2) k = q;
        long id = G.id(i, j, k);
        double h, d;
        lsfun(phi[id], w, h, d);
        double rho = h + r12 * (1.0 - h);
        acc[0] += rho * h * dv;
        acc[1] += h * dv;
        if (with_lam) {
            double fx = nx_[id], fy = ny_[id], g;
            if (DIM == 3) {
                double fz = nz_[id];
                g = sqrt(fx * fx + fy * fy + fz * fz);
            } else {
                g = sqrt(fx * fx + fy * fy);
            }
            grad[id] = g;
            double plam = d * d * g;
            plam = DIM == 3 ? plam * (2.0 * (1.0 - r12) * h + r12) * G.dx * G.dy * G.dz
                            : plam * (2.0 * (1.0 - r12) * h + r12) * G.dx * G.dy;
            acc[2] += plam;
        }
    }
    block_sum_store<3>(acc, partial + (long)q * RBLK, RBLK * gridDim.y);
}

// phi += lambda delta |grad phi|, lambda = (imass - mass) / denominator
// computed here from the reduced sums (mass_preserving_level_set.f90:36-48)
// (per case of a batched stack: its sums, its imass from cp, its lambda slot)
template <int DIM>
__global__ void k_mpls_update(double *__restrict__ phi, const double *__restrict__ grad,
                              const double *__restrict__ sums, double *__restrict__ lam_out, Geom G, double w,
                              double imass, const fcfd_case *__restrict__ cp) {
    int bx_, by_, bz_;
    xcd_block(bx_, by_, bz_);
    int i = bx_ * blockDim.x + threadIdx.x, j = by_ * blockDim.y + threadIdx.y, k = bz_;
    const int q = case_of<DIM>(k);
    sums += (long)q * RES_STRIDE;
    if (cp) imass = cp[q].imass;
    double lam = (imass - sums[0]) / sums[2];
    if (i == 0 && j == 0 && (DIM == 2 || k == 0)) lam_out[(long)q * RES_STRIDE] = lam;
    if (i >= G.nx || j >= G.ny) return;
    long id = G.id(i, j, k);
    double h, d;
    lsfun(phi[id], w, h, d);
    phi[id] = phi[id] + lam * d * grad[id];
}

int mass_sums(fcfd_ctx *c, const double *phi, int with_lam) {
    const Geom &G = c->G;
    ProfScope ps_(c, R_MASS);
    if (G.dim == 3)
        hipLaunchKernelGGL(k_mass_sums<3>, dim3(RBLK), dim3(RTHR), 0, c->stream, phi, c->f[FCFD_NX], c->f[FCFD_NY],
                           c->f[FCFD_NZ], c->f[FCFD_GRAD], c->red.partial, G, c->pr.ls_wid, c->pr.rho_12, with_lam,
                           (const fcfd_case *)nullptr);
    else
        hipLaunchKernelGGL(k_mass_sums<2>, dim3(RBLK, c->nb), dim3(RTHR), 0, c->stream, phi, c->f[FCFD_NX],
                           c->f[FCFD_NY], nullptr, c->f[FCFD_GRAD], c->red.partial, G, c->pr.ls_wid, c->pr.rho_12,
                           with_lam, c->cases_dev);
    FCFD_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_reduce_final, dim3(c->nb), dim3(RTHR), 0, c->stream, c->red.partial, c->red.result, 3,
                       RBLK);
    FCFD_CHECK(hipGetLastError());
    return FCFD_OK;
}

int fetch_result(fcfd_ctx *c, int n) {
    FCFD_CHECK(hipMemcpyAsync(c->red.host, c->red.result, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
    FCFD_CHECK(hipStreamSynchronize(c->stream));
    return FCFD_OK;
}

// ls_mv; mass and vol of case 0 (a batched stack leaves every case's pair at
// red.host[q*RES_STRIDE], [q*RES_STRIDE + 1])
int ls_mv(fcfd_ctx *c, double *mass, double *vol) {
    FCFD_TRY(ls_props(c, c->f[FCFD_PHI], c->f[FCFD_HEAVY], c->f[FCFD_DELTA], c->f[FCFD_SIGN], c->f[FCFD_RHO],
                      c->f[FCFD_MU]));
    FCFD_TRY(mass_sums(c, c->f[FCFD_PHI], 0));
    FCFD_TRY(fetch_result(c, RES_STRIDE * c->nb));
    c->diag.mass = c->red.host[0];
    c->diag.vol = c->red.host[1];
    if (mass) *mass = c->red.host[0];
    if (vol) *vol = c->red.host[1];
    return FCFD_OK;
}

// ------------------------------------------------ ls_mv without allocation
// fcfd_ls_mv_noalloc: the kernels of ls_mv (k_ls_props, k_mass_sums,
// k_reduce_final) on caller-owned fields, with their reduction partials,
// reduced sums and per-case ratios in one file-scope device array instead of
// context memory.  Every call on a device shares that device's copy of the
// array, so calls that overlap on one device (two streams, two threads) race;
// the array keeps the last call's contents, and nothing in it is read before
// this call has written it.
constexpr int NOALLOC_MAX_CASES = FCFD_LS_MV_NOALLOC_MAX_CASES;
constexpr long NA_PARTIAL = 3L * RBLK * NOALLOC_MAX_CASES;            // k_mass_sums block partials
constexpr long NA_RESULT = (long)RES_STRIDE * NOALLOC_MAX_CASES;      // k_reduce_final output
constexpr long NA_CASES = (long)(sizeof(fcfd_case) / sizeof(double)) * NOALLOC_MAX_CASES;
constexpr long NA_WORDS = NA_PARTIAL + NA_RESULT + NA_CASES;          // 1.58 MB
static __device__ __align__(256) double scratch[NA_WORDS];

struct CaseRatios {
    double r12[NOALLOC_MAX_CASES], m12[NOALLOC_MAX_CASES];
};

__global__ void k_put_cases(CaseRatios cr, int n, fcfd_case *__restrict__ dst) {
    const int q = threadIdx.x;
    if (q >= n) return;
    fcfd_case c{};
    c.rho_12 = cr.r12[q];
    c.mu_12 = cr.m12[q];
    dst[q] = c;
}

// sums[2q], sums[2q + 1] = mass, volume of case q
__global__ void k_put_sums(const double *__restrict__ result, int n, double *__restrict__ sums) {
    const int t = threadIdx.x;
    if (t >= 2 * n) return;
    sums[t] = result[(long)(t >> 1) * RES_STRIDE + (t & 1)];
}

}  // namespace fcfd

extern "C" int fcfd_ls_mv_noalloc(const fcfd_grid *grid, const fcfd_params *params, int ncases,
                                  const fcfd_case *cases, const double *phi, double *heavy, double *delta,
                                  double *sign, double *rho, double *mu, double *sums, void *stream) {
    using namespace fcfd;
    if (!grid || !params || !phi || !sums) return FCFD_ERR_ARG;
    if (grid->dim != 2 && grid->dim != 3) return FCFD_ERR_ARG;
    if (grid->ghc != 3 || grid->nx < 4 || grid->ny < 4) return FCFD_ERR_ARG;
    if (grid->dim == 3 && (grid->nz < 4 || ncases != 1 || cases)) return FCFD_ERR_ARG;
    if (grid->dim == 2 && grid->nz != 1) return FCFD_ERR_ARG;
    if (ncases < 1) return FCFD_ERR_ARG;
    if (ncases > NOALLOC_MAX_CASES) {
        fprintf(stderr, "libfcfd: fcfd_ls_mv_noalloc: %d cases exceed its fixed scratch of %d cases\n", ncases,
                NOALLOC_MAX_CASES);
        return FCFD_ERR_ARG;
    }
    if (ncases > 1 && !cases) return FCFD_ERR_ARG;
    // the device address of this device's copy of the scratch array, looked
    // up once per device (the array's name is not a device address on the host)
    static std::mutex mu_;
    static double *dev_scratch[64] = {};
    int dev = 0;
    FCFD_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return FCFD_ERR_ARG;
    double *base;
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (!dev_scratch[dev]) {
            void *ptr = nullptr;
            FCFD_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
            dev_scratch[dev] = (double *)ptr;
        }
        base = dev_scratch[dev];
    }
    double *partial = base, *result = base + NA_PARTIAL;
    fcfd_case *cp = nullptr;
    hipStream_t st = (hipStream_t)stream;
    Geom G;
    G.dim = grid->dim;
    G.nx = grid->nx; G.ny = grid->ny; G.nz = grid->dim == 3 ? grid->nz : ncases;
    G.g = grid->ghc; G.gz = grid->dim == 3 ? grid->ghc : 0;
    G.sx = G.nx + 2 * G.g;
    G.sxy = G.sx * (G.ny + 2 * G.g);
    G.ntot = G.sxy * (G.nz + 2 * G.gz);
    G.dx = (grid->xend - grid->xstart) / G.nx;
    G.dy = (grid->yend - grid->ystart) / G.ny;
    G.dz = grid->dim == 3 ? (grid->zend - grid->zstart) / G.nz : 1.0;
    if (ncases > 1) {
        CaseRatios cr{};
        for (int q = 0; q < ncases; ++q) {
            cr.r12[q] = cases[q].rho_12;
            cr.m12[q] = cases[q].mu_12;
        }
        cp = (fcfd_case *)(base + NA_PARTIAL + NA_RESULT);
        hipLaunchKernelGGL(k_put_cases, dim3(1), dim3(NOALLOC_MAX_CASES), 0, st, cr, ncases, cp);
        FCFD_CHECK(hipGetLastError());
    }
    const long n = G.ntot;
    hipLaunchKernelGGL(k_ls_props, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, phi, heavy, delta, sign,
                       rho, mu, n, params->ls_wid, params->rho_12, params->mu_12, (const fcfd_case *)cp, G.sxy);
    FCFD_CHECK(hipGetLastError());
    if (G.dim == 3)
        hipLaunchKernelGGL(k_mass_sums<3>, dim3(RBLK), dim3(RTHR), 0, st, phi, (const double *)nullptr,
                           (const double *)nullptr, (const double *)nullptr, (double *)nullptr, partial, G,
                           params->ls_wid, params->rho_12, 0, (const fcfd_case *)nullptr);
    else
        hipLaunchKernelGGL(k_mass_sums<2>, dim3(RBLK, ncases), dim3(RTHR), 0, st, phi, (const double *)nullptr,
                           (const double *)nullptr, (const double *)nullptr, (double *)nullptr, partial, G,
                           params->ls_wid, params->rho_12, 0, (const fcfd_case *)cp);
    FCFD_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_reduce_final, dim3(ncases), dim3(RTHR), 0, st, (const double *)partial, result, 3, RBLK);
    FCFD_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_put_sums, dim3(1), dim3(2 * NOALLOC_MAX_CASES), 0, st, (const double *)result, ncases,
                       sums);
    FCFD_CHECK(hipGetLastError());
    return FCFD_OK;
}

namespace fcfd {

int mpls(fcfd_ctx *c) {
    const Geom &G = c->G;
    double *phi = c->f[FCFD_PHI];
    dim3 blk(64, 4), grd = grid_interior(G, blk);
    double *lam_dev = c->red.result + RES_LAMBDA;
    for (int it = 0; it < 2; ++it) {
        // surface_norms: only the first derivatives enter the correction
        FCFD_TRY(ccd_dir(c, 0, phi, c->f[FCFD_NX], c->cx));
        FCFD_TRY(ccd_dir(c, 1, phi, c->f[FCFD_NY], c->cy));
        if (G.dim == 3) FCFD_TRY(ccd_dir(c, 2, phi, c->f[FCFD_NZ], c->cz));
        FCFD_TRY(mass_sums(c, phi, 1));
        {
            ProfScope ps_(c, R_MPLS_UPD);
            if (G.dim == 3)
                hipLaunchKernelGGL(k_mpls_update<3>, grd, blk, 0, c->stream, phi, c->f[FCFD_GRAD], c->red.result,
                                   lam_dev, G, c->pr.ls_wid, c->pr.imass, (const fcfd_case *)nullptr);
            else
                hipLaunchKernelGGL(k_mpls_update<2>, grd, blk, 0, c->stream, phi, c->f[FCFD_GRAD], c->red.result,
                                   lam_dev, G, c->pr.ls_wid, c->pr.imass, c->cases_dev);
            FCFD_CHECK(hipGetLastError());
        }
        FCFD_TRY(bc_scalar(c, phi));
    }
    return FCFD_OK;
}

// ------------------------------------------------------------- advection
// One SSP-RK3 stage of level_set_rk3_solver, fused: velocity flux split
// (source_setup :67-96, with the bc() copy of s1/s2 realised by clamped
// indices), WENO5-JS faces (:162-219), flux divergence (:145-158) and the
// increment-form stage update (:13-60), with every face computed once.
// T = float is the single-precision variant (same operation order, FP32
// weights of weno.h); the velocity is vs (nu, nv, nw).
// A block covers a TX x 256/TX tile and, in 3D, walks kc planes of it (2D:
// the block's slice, a case of a batched stack).  Per plane each thread
// computes the x-face and the y-face below its cell into LDS, the first TX
// threads the tile's last row of y-faces and one thread per row the last
// x-face; then each cell differences them.  The z flux of face k+1/2 is the
// k-1/2 flux of the next plane, from a 7-plane window of (w, phi) splits
// carried in registers.  The LDS plane is double buffered, one barrier per
// plane; what a cell needs besides the faces is loaded before it.  Face value
// F = WENO_left(s1 at f-2..f+2) + WENO_right(s2 at f-1..f+3) at clamped
// positions; L sums F(+1/2) - F(-1/2) per direction.
// With TX = 64 a wave is one row, so a face's six rows (y) or its row (x)
// have scalar bases and one vector offset.  O is the type of a face's byte
// offsets from the first cell its tile reads, OFF_ROWS rows at most: 32 bits,
// or 64 bits where that many rows pass 4 GiB (launch_stage).  Every other
// address is a 64-bit row base and an offset inside the tile's row.
//
// What bounds it: a plane is a chain of memory round trips, the faces one
// after the other and a barrier, about 5 us; a block's planes are serial, so
// the walk is only as long as the grid can afford (stage_planes).  434 us at
// 256^3 (533 with 256 threads striding over the 580 faces at 64-bit
// addresses), 54 us at 128^3 (83 with 16 planes a block whatever the grid), 30
// us in FP32 at 101 x 87 x 117 (90).
template <int TX>
constexpr int OFF_ROWS = 256 / TX + 6;   // rows j0 - 3 .. j0 + TY + 2

template <int DIM, typename T, int TX>
struct StageLds {
    T fx[2][256 / TX][TX + 1], fy[2][256 / TX + 1][TX];
};

template <int DIM, typename T, int TX, typename O>
__device__ __forceinline__ void ls_adv_stage_body(StageLds<DIM, T, TX> &sh, const T *__restrict__ phi,
                                                  T *__restrict__ phin, const T *__restrict__ nu,
                                                  const T *__restrict__ nv, const T *__restrict__ nw,
                                                  T *__restrict__ l1, T *__restrict__ l2, const Geom &G, T dt, T vs,
                                                  int stage, int kc, int bx_, int by_, int bz_) {
    // Products are fused into adds only within one statement here: the flux
    // splits s1, s2 of the z window are formed in the plane that loads them,
    // and with fusion across statements a face whose splits were formed in
    // the same plane (the first face of a walk) rounded differently from the
    // same face formed from carried splits.  A face now has one value
    // wherever a walk starts, which keeps block-by-block runs bit for bit
    // equal to whole-field ones.
#pragma clang fp contract(on)
    constexpr int TY = 256 / TX;
    const int tx = threadIdx.x, t = threadIdx.y * TX + tx;
    const int ty = TX == WAVE ? __builtin_amdgcn_readfirstlane(threadIdx.y) : (int)threadIdx.y;
    const int i0 = bx_ * TX, j0 = by_ * TY, i = i0 + tx, j = j0 + ty;
    // 3D: kc planes per block; 2D: the block's slice (a case of a batched stack)
    const int k0 = DIM == 3 ? bz_ * kc : bz_, k1 = DIM == 3 ? min(k0 + kc, G.nz) : bz_ + 1;
    if (i0 >= G.nx || j0 >= G.ny || k0 >= G.nz) return;   // the whole block
    const bool in = i < G.nx && j < G.ny;
    const int ic = min(i, G.nx - 1), jc = min(j, G.ny - 1);
    const T half = (T)0.5, EPS = (T)1.0e-13;
    const T rhx = (T)(1.0 / G.dx), rhy = (T)(1.0 / G.dy), rhz = (T)(1.0 / G.dz);
    const int xlo = -G.ox0, xhi = G.nx - 1 + G.ox1, ylo = -G.oy0, yhi = G.ny - 1 + G.oy1;
    const int zlo = -G.oz0, zhi = G.nz - 1 + G.oz1;
    auto flux = [&](const T (&u)[6], const T (&p)[6]) -> T {
        T s1[6], s2[6];
#pragma unroll
        for (int m = 0; m < 6; ++m) {
            const T v = vs * u[m];
            s1[m] = half * (v + fabs(v)) * p[m];
            s2[m] = half * (v - fabs(v)) * p[m];
        }
        return weno_left(s1[0], s1[1], s1[2], s1[3], s1[4], EPS) + weno_right(s2[1], s2[2], s2[3], s2[4], s2[5], EPS);
    };
    const unsigned co = (unsigned)(ic - i0) * (unsigned)sizeof(T);   // offset of this column from the tile's first
    // first column and row that the tile's faces read
    const int cb = max(i0 - 3, xlo), rb = max(j0 - 3, ylo);
    // z window of this column: positions clamp(k - 3 + m), m = 0..6
    T s1z[7], s2z[7], Fl = 0;
    if (DIM == 3) {
#pragma unroll
        for (int m = 0; m < 7; ++m) {
            const long row = G.id(i0, jc, clampi(k0 - 3 + m, zlo, zhi));
            const T u = vs * at_bytes(nw + row, co), p = at_bytes(phi + row, co);
            s1z[m] = half * (u + fabs(u)) * p;
            s2z[m] = half * (u - fabs(u)) * p;
        }
        Fl = weno_left(s1z[0], s1z[1], s1z[2], s1z[3], s1z[4], EPS) +
             weno_right(s2z[1], s2z[2], s2z[3], s2z[4], s2z[5], EPS);
    }
    for (int k = k0; k < k1; ++k) {
        const int b = k & 1;
        // this cell's operands and the z window's next plane, ahead of the faces
        const long rc = G.id(i0, jc, k);
        const T pc = at_bytes(phi + rc, co);
        const T l1o = stage >= 1 ? at_bytes(l1 + rc, co) : (T)0, l2o = stage == 2 ? at_bytes(l2 + rc, co) : (T)0;
        T wn = 0, pn = 0;
        if (DIM == 3) {
            const long row = G.id(i0, jc, clampi(k + 4, zlo, zhi));
            wn = at_bytes(nw + row, co);
            pn = at_bytes(phi + row, co);
        }
        // the x-face and the y-face below the cell, then the tile's last
        // y-face row (first TX threads) and last x-faces (TY threads), one
        // after the other: unrolled, their loads take 198 VGPRs.  A face reads
        // positions clamp(f - 2 + m) of its line at byte offsets from cell
        // (cb, rb) of the plane; o0 may be below it (modulo 2^32 or 2^64), the
        // sums never are.
        const long pl = G.id(cb, rb, k);
        const T *pp = phi + pl;
#pragma unroll 1
        for (int r = 0; r < 3; ++r) {
            const bool last = r == 2, xf = r == 0 || (last && t >= 128);
            if (last && !(t < TX || (t >= 128 && t < 128 + TY))) break;
            const T *vp = (xf ? nu : nv) + pl;
            const int row = xf ? (last ? min(j0 + t - 128, G.ny - 1) : jc) : 0;
            const int f = xf ? (last ? i0 + TX - 1 : i - 1) : (last ? j0 + TY - 1 : j - 1);
            const int lo = xf ? xlo : ylo, hi = xf ? xhi : yhi;
            const O st = (xf ? (O)1 : (O)G.sx) * (O)sizeof(T);
            const O o0 = xf ? ((O)(row - rb) * (O)G.sx - (O)cb) * (O)sizeof(T) : (O)(ic - cb) * (O)sizeof(T) - (O)rb * st;
            T u[6], p[6];
#pragma unroll
            for (int m = 0; m < 6; ++m) {
                const O o = o0 + (O)clampi(f - 2 + m, lo, hi) * st;
                u[m] = at_bytes(vp, o);
                p[m] = at_bytes(pp, o);
            }
            const T F = flux(u, p);
            if (xf) sh.fx[b][last ? t - 128 : ty][last ? TX : tx] = F;
            else sh.fy[b][last ? TY : ty][tx] = F;
        }
        __syncthreads();
        // face k + 1/2: gm from s1(k-2..k+2), fp from s2(k-1..k+3)
        T Fr = 0;
        if (DIM == 3)
            Fr = weno_left(s1z[1], s1z[2], s1z[3], s1z[4], s1z[5], EPS) +
                 weno_right(s2z[2], s2z[3], s2z[4], s2z[5], s2z[6], EPS);
        if (in) {
            T L = -(sh.fx[b][ty][tx + 1] - sh.fx[b][ty][tx]) * rhx;
            L = L + (-(sh.fy[b][ty + 1][tx] - sh.fy[b][ty][tx]) * rhy);
            if (DIM == 3) L = L + (-(Fr - Fl) * rhz);
            T src;
            if (stage == 0) {
                at_bytes(l1 + rc, co) = L;
                src = L;
            } else if (stage == 1) {
                at_bytes(l2 + rc, co) = L;
                src = ((T)-3.0 * l1o + L) * (T)0.25;
            } else {
                src = (-l1o - l2o + (T)8.0 * L) / (T)12.0;
            }
            at_bytes(phin + rc, co) = pc + src * dt;
        }
        if (DIM == 3) {
            Fl = Fr;
            // slide the z window to plane k + 1
#pragma unroll
            for (int m = 0; m < 6; ++m) {
                s1z[m] = s1z[m + 1];
                s2z[m] = s2z[m + 1];
            }
            const T u = vs * wn;
            s1z[6] = half * (u + fabs(u)) * pn;
            s2z[6] = half * (u - fabs(u)) * pn;
        }
    }
}

template <int DIM, typename T, int TX, typename O>
__global__ void __launch_bounds__(256) k_ls_adv_stage(const T *__restrict__ phi, T *__restrict__ phin,
                                                      const T *__restrict__ nu, const T *__restrict__ nv,
                                                      const T *__restrict__ nw, T *__restrict__ l1,
                                                      T *__restrict__ l2, Geom G, T dt, T vs, int stage, int kc) {
    __shared__ StageLds<DIM, T, TX> sh;
    int bx_, by_, bz_;
    xcd_block(bx_, by_, bz_);
    ls_adv_stage_body<DIM, T, TX, O>(sh, phi, phin, nu, nv, nw, l1, l2, G, dt, vs, stage, kc, bx_, by_, bz_);
}

// the same stage on every block of a multi-block layout in one launch:
// tab[b] places block b in the stacks; the grid covers the largest block, nz
// walks per block along z.  (A launch per block of 80 x 75 x 85 cells leaves
// the chip nearly empty: 75 us each, eight in a row; together 134 us.)
template <int DIM, int TX, typename O>
__global__ void __launch_bounds__(256) k_ls_adv_stage_blocks(const double *__restrict__ phi,
                                                             double *__restrict__ phin,
                                                             const double *__restrict__ nu,
                                                             const double *__restrict__ nv,
                                                             const double *__restrict__ nw, double *__restrict__ l1,
                                                             double *__restrict__ l2,
                                                             const BlockGeom *__restrict__ tab, double dt, int stage,
                                                             int kc, int nz) {
    __shared__ StageLds<DIM, double, TX> sh;
    int bx_, by_, bz_;
    xcd_block(bx_, by_, bz_);
    const int b = bz_ / nz;
    const Geom G = tab[b].G;
    const long o = tab[b].off;
    ls_adv_stage_body<DIM, double, TX, O>(sh, phi + o, phin + o, nu + o, nv + o, DIM == 3 ? nw + o : nullptr, l1 + o,
                                          l2 + o, G, dt, 1.0, stage, kc, bx_, by_, bz_ - b * nz);
}

// One SSP-RK3 stage with the UCCD source L = -(u phi_x + v phi_y + w phi_z)
// (the reference's commented alternative source,
// `.../interface_solver/level_set_rk3_solver.f90:155-157`), from the upwind
// CCD derivatives fx, fy, fz of the stage input.
template <int DIM>
__global__ void __launch_bounds__(256) k_ls_uccd_stage(const double *__restrict__ phi, double *__restrict__ phin,
                                                       const double *__restrict__ nu, const double *__restrict__ nv,
                                                       const double *__restrict__ nw, const double *__restrict__ fx,
                                                       const double *__restrict__ fy, const double *__restrict__ fz,
                                                       double *__restrict__ l1, double *__restrict__ l2, Geom G,
                                                       double dt, int stage) {
    int bx_, by_, bz_;
    xcd_block(bx_, by_, bz_);
    const int i = bx_ * blockDim.x + threadIdx.x, j = by_ * blockDim.y + threadIdx.y, k = bz_;
    if (i >= G.nx || j >= G.ny) return;
    const long id = G.id(i, j, k);
    double L = -nu[id] * fx[id] - nv[id] * fy[id];
    if (DIM == 3) L = L - nw[id] * fz[id];
    double src;
    if (stage == 0) {
        l1[id] = L;
        src = L;
    } else if (stage == 1) {
        l2[id] = L;
        src = (-3.0 * l1[id] + L) / 4.0;
    } else {
        src = (-l1[id] - l2[id] + 8.0 * L) / 12.0;
    }
    phin[id] = phi[id] + src * dt;
}

// planes a block of the 3D stage walks: 16 (one plane in 17 costs its first
// z-face and window twice), halved while the launch would leave CUs with
// fewer than 8 blocks, down to 4
static int stage_planes(long tiles, int nz, int ncu) {
    int kc = 16;
    while (kc > 4 && tiles * ((nz + kc - 1) / kc) < 8L * ncu) kc /= 2;
    return kc;
}

// whether a stage's face offsets fit 32 bits: OFF_ROWS rows of sx elements
// (rows of up to 53 million cells in FP64 with TX = 64, 38 million with 32)
static bool stage_off32(const dim3 &blk, long sx, size_t size) {
    return (double)(blk.x == 64 ? OFF_ROWS<64> : OFF_ROWS<32>) * (double)sx * (double)size < 4294967296.0;
}

template <int DIM, typename T>
static int launch_stage(hipStream_t st, int ncu, const Geom &G, const T *phi, T *phin, const T *nu, const T *nv,
                        const T *nw, T *l1, T *l2, T dt, T vs, int stage) {
    const bool off32 = stage_off32(tile_rows(G.nx), G.sx, sizeof(T));
    const dim3 blk = off32 ? tile_rows(G.nx) : dim3(64, 4);
    const dim3 tiles((G.nx + blk.x - 1) / blk.x, (G.ny + blk.y - 1) / blk.y, G.nz);
    const int kc = DIM == 3 ? stage_planes((long)tiles.x * tiles.y, G.nz, ncu) : 1;
    const dim3 grd(tiles.x, tiles.y, (G.nz + kc - 1) / kc);
#define FCFD_ST(X_, O_)                                                                                             \
    hipLaunchKernelGGL((k_ls_adv_stage<DIM, T, X_, O_>), grd, blk, 0, st, phi, phin, nu, nv, nw, l1, l2, G, dt, vs, \
                       stage, kc)
    if (!off32) FCFD_ST(64, unsigned long);
    else if (blk.x == 64) FCFD_ST(64, unsigned);
    else FCFD_ST(32, unsigned);
#undef FCFD_ST
    FCFD_CHECK(hipGetLastError());
    return FCFD_OK;
}

// one WENO5 SSP-RK3 stage from phi into phin with the context's velocity
// (the stage sources stay in l1/l2 as in ls_advect); no ghost update
int ls_adv_stage(fcfd_ctx *c, const double *phi, double *phin, int stage) {
    double **F = c->f;
    if (c->G.dim == 3)
        return launch_stage<3, double>(c->stream, c->ncu, c->G, phi, phin, F[FCFD_NU], F[FCFD_NV], F[FCFD_NW], c->l1,
                                       c->l2, c->pr.dt, c->vscale, stage);
    return launch_stage<2, double>(c->stream, c->ncu, c->G, phi, phin, F[FCFD_NU], F[FCFD_NV], nullptr, c->l1, c->l2,
                                   c->pr.dt, c->vscale, stage);
}

int ls_adv_stage_blocks(hipStream_t st, int ncu, const BlockGeom *tab, int nblk, int dim, int nx, int ny, int nz,
                        const double *phi, double *phin, const double *nu, const double *nv, const double *nw,
                        double *l1, double *l2, double dt, int stage) {
    const bool off32 = stage_off32(tile_rows(nx), nx + 6, sizeof(double));   // 3 ghosts a side
    const dim3 blk = off32 ? tile_rows(nx) : dim3(64, 4);
    const dim3 tiles((nx + blk.x - 1) / blk.x, (ny + blk.y - 1) / blk.y);
    int kc = dim == 3 ? stage_planes((long)tiles.x * tiles.y * nblk, nz, ncu) : 1;
    // the blocks' walks share grid.z, whose limit is 65536 (up to 4096 blocks)
    while ((long)nblk * ((nz + kc - 1) / kc) > 65535) kc *= 2;
    const int kz = (nz + kc - 1) / kc;
    const dim3 grd(tiles.x, tiles.y, (unsigned)(nblk * kz));
#define FCFD_SB(D_, X_, O_)                                                                                         \
    hipLaunchKernelGGL((k_ls_adv_stage_blocks<D_, X_, O_>), grd, blk, 0, st, phi, phin, nu, nv, nw, l1, l2, tab, dt, \
                       stage, kc, kz)
    if (dim == 3) {
        if (!off32) FCFD_SB(3, 64, unsigned long);
        else if (blk.x == 64) FCFD_SB(3, 64, unsigned);
        else FCFD_SB(3, 32, unsigned);
    } else {
        if (!off32) FCFD_SB(2, 64, unsigned long);
        else if (blk.x == 64) FCFD_SB(2, 64, unsigned);
        else FCFD_SB(2, 32, unsigned);
    }
#undef FCFD_SB
    FCFD_CHECK(hipGetLastError());
    return FCFD_OK;
}

int ls_advect(fcfd_ctx *c) {
    const Geom &G = c->G;
    dim3 blk(64, 4), grd = grid_interior(G, blk);
    double *a = c->f[FCFD_PHI], *b = c->phiB;
    if (c->pr.ls_scheme == FCFD_LS_UCCD) {
        if (c->vscale != 1.0) {
            fprintf(stderr, "libfcfd: the velocity scale applies to the WENO5 scheme only\n");
            return FCFD_ERR_ARG;
        }
        // upwind-CCD derivatives park in the predictor's spare velocity buffers
        double *d[3] = {c->un, c->vn, c->wn};
        const double *vel[3] = {c->f[FCFD_NU], c->f[FCFD_NV], c->f[FCFD_NW]};
        for (int s = 0; s < 3; ++s) {
            for (int dir = 0; dir < G.dim; ++dir) FCFD_TRY(uccd_dir(c, dir, a, vel[dir], d[dir], nullptr));
            {
                ProfScope ps_(c, R_LS_ADV);
                if (G.dim == 3)
                    hipLaunchKernelGGL(k_ls_uccd_stage<3>, grd, blk, 0, c->stream, a, b, vel[0], vel[1], vel[2], d[0],
                                       d[1], d[2], c->l1, c->l2, G, c->pr.dt, s);
                else
                    hipLaunchKernelGGL(k_ls_uccd_stage<2>, grd, blk, 0, c->stream, a, b, vel[0], vel[1], nullptr, d[0],
                                       d[1], nullptr, c->l1, c->l2, G, c->pr.dt, s);
                FCFD_CHECK(hipGetLastError());
            }
            FCFD_TRY(bc_scalar(c, b));
            double *t = a; a = b; b = t;
        }
        c->phiB = c->f[FCFD_PHI];
        c->f[FCFD_PHI] = a;
        return FCFD_OK;
    }
    for (int s = 0; s < 3; ++s) {
        {
            ProfScope ps_(c, R_LS_ADV);
            FCFD_TRY(ls_adv_stage(c, a, b, s));
        }
        double *t = a; a = b; b = t;
    }
    // the stages read no ghosts (clamped indices): only the result's are filled
    FCFD_TRY(bc_scalar(c, a));
    // three stages end in the buffer that was phiB: swap roles
    c->phiB = c->f[FCFD_PHI];
    c->f[FCFD_PHI] = a;
    return FCFD_OK;
}

// one FP32 WENO5 SSP-RK3 stage from phi into phin with caller arrays (the
// velocity times the context's scale); no ghost update
int ls_adv_stage_f32(fcfd_ctx *c, const float *phi, float *phin, const float *nu, const float *nv, const float *nw,
                     float *l1, float *l2, int stage) {
    const float dt = (float)c->pr.dt, vs = (float)c->vscale;
    if (c->G.dim == 3)
        return launch_stage<3, float>(c->stream, c->ncu, c->G, phi, phin, nu, nv, nw, l1, l2, dt, vs, stage);
    return launch_stage<2, float>(c->stream, c->ncu, c->G, phi, phin, nu, nv, nullptr, l1, l2, dt, vs, stage);
}

// One SSP-RK3 step in FP32 of a caller's level set phi with the caller's
// FP32 cell velocity times the context's scale: stage 0 phi -> B, stage 1
// B -> C, stage 2 C -> phi (each stage reads its input and writes another
// array, no ghosts), then the zero-gradient ghost copy as in ls_advect.
int ls_advect_f32(fcfd_ctx *c, float *phi, const float *nu, const float *nv, const float *nw) {
    const Geom &G = c->G;
    for (auto &p : c->adv32) FCFD_TRY(alloc_once(&p, G.ntot));
    float *B = c->adv32[0], *Cb = c->adv32[1], *l1 = c->adv32[2], *l2 = c->adv32[3];
    float *in[3] = {phi, B, Cb}, *out[3] = {B, Cb, phi};
    for (int s = 0; s < 3; ++s) {
        ProfScope ps_(c, R_LS_ADV);
        FCFD_TRY(ls_adv_stage_f32(c, in[s], out[s], nu, nv, nw, l1, l2, s));
    }
    return bc_scalar_f32(c, phi);
}

// ------------------------------------------------------------- reinit
// Interface band of the reinitialisation: the cells where lsfun's delta can
// be non-zero.  The threshold is tested with the reciprocal width, which may
// differ from lsfun's quotient by an ulp; a cell at the threshold has
// delta = 0 either way (1 + cos(pi x) rounds to 0 within ~1e-8 of |x| = 1).
// NaN counts as inside, as in lsfun.
__device__ __forceinline__ bool in_band(double phi, double iw) {
    const double x = phi * iw;
    return !(x > 1.0 - 1.0e-12) && !(x < -1.0 + 1.0e-12);
}

// source of one stage and the increment-form SSP-RK3 update (redis_solver
// :150-208); l1o, l2o the stored sources of the earlier stages
template <int STAGE>
__device__ __forceinline__ double redis_update(double p0, double l, double l1o, double l2o, double rdt) {
    double src;
    if (STAGE == 0) src = l;
    else if (STAGE == 1) src = (-3.0 * l1o + l) / 4.0;
    else src = (-l1o - l2o + 8.0 * l) / 12.0;
    return p0 - rdt * src;
}

// max|phi - phi_start| of a block into one of NSHARD slots of the case's
// flags (reinit stop test :42-54): a single slot would serialise tens of
// thousands of atomics; the max of non-negative doubles is order
// independent, compared as bit patterns
__device__ __forceinline__ void redis_shard_max(double err, double *sh4, unsigned long long *flags) {
    const double m = block_max256(err, sh4);
    if (threadIdx.x + threadIdx.y == 0) {
        const unsigned b = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
        atomicMax(&flags[FLAG_SHARD0 + b % NSHARD], (unsigned long long)__double_as_longlong(m));
    }
}

struct Recip {
    double x, y, z;   // reciprocal spacings
};
constexpr int REDIS_GRADIENT = 3;  // STAGE of the gradient-only pass

// One reinitialisation stage from phi into out (another array: the stencil
// reads neighbours): backward differences of phi with the bc() ghost copy as
// clamped indices (redis_gradient :219-233), one-sided WENO5 values,
// EPS = 1e-10 (wenojs_flux :295-339), Godunov |grad phi| by the frozen sign
// (:262-291), then the stage source and update.  The mass constraint enters
// as (a / b) delta with delta = 0 outside the interface band, so every cell
// outside it is finished here; a band cell only stores |grad phi| and its
// constraint terms (redis_lambda :366-380; 2D: lambda = delta, 3D: density
// weighted) and its tile is listed for k_redis_band.  The two-pass form stored
// three values per cell and read them back: at 256^3 346 + 355 us a stage
// and a 62 us copy of phi per pseudo step.
// lo: the lowest index phi is read at, -1 where phi's ghosts are valid
// (the first stage: phi(-1) may differ from a copy of phi(0)) and 0 for the
// stage buffers, whose ghosts are not filled; every ghost that bc() would
// fill reads its clamped cell.
template <int DIM, int STAGE, bool BTN>
__global__ void __launch_bounds__(256) k_redis_stage(const double *__restrict__ phi, double *__restrict__ out,
                                                     const double *__restrict__ S0, double *__restrict__ grad,
                                                     double *__restrict__ s2, double *__restrict__ s3,
                                                     double *__restrict__ l1, double *__restrict__ l2,
                                                     BandList band, unsigned long long *flags, Geom G,
                                                     double w, double iw, double r12, double rdt, Recip ih,
                                                     int lo) {
    int bx_, by_, bz_;
    if (DIM == 3) xcd_block_slab(bx_, by_, bz_, 8);
    else xcd_block(bx_, by_, bz_);
    const int i = bx_ * blockDim.x + threadIdx.x, j = by_ * blockDim.y + threadIdx.y, k = bz_;
    flags += (long)case_of<DIM>(k) * FLAG_STRIDE;   // this case's flag block (a block covers one slice)
    if (STAGE != REDIS_GRADIENT && flags[1]) return;
    const bool in = i < G.nx && j < G.ny;
    double err = 0.0;
    int hold = 0;
    if (in) {
        const long id0 = G.id(bx_ * (int)blockDim.x, by_ * (int)blockDim.y, k);   // the block's first cell
        const unsigned off = threadIdx.x + threadIdx.y * (unsigned)G.sx;
        const int n[3] = {G.nx, G.ny, G.nz};
        const int pos[3] = {i, j, k};
        const long st[3] = {1, G.sx, G.sxy};
        const double ihd[3] = {ih.x, ih.y, ih.z};
        // phi at pos-4 .. pos+3 of the three lines and the cell's other
        // operands before any branch that depends on them
        double gw[3][8];
#pragma unroll
        for (int d = 0; d < DIM; ++d) line_load<8, 4>(phi + id0, off, st[d], pos[d], n[d], lo, gw[d]);
        grad += id0; s2 += id0; s3 += id0; l1 += id0; l2 += id0; out += id0;
        const double S = (S0 + id0)[off];
        const double l1o = STAGE == 1 || STAGE == 2 ? l1[off] : 0.0, l2o = STAGE == 2 ? l2[off] : 0.0;
        const double pst = STAGE == 2 ? out[off] : 0.0;   // the last stage writes over phi_start
        const double p0 = gw[0][4];
        const bool pos_sign = S >= 0.0;
        double sel[3];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            // D-phi at pos-3 .. pos+3, ghost entries copying the boundary one:
            // nr[m] = D(clamp(pos - 3 + m, 0, n - 1)) = dw[clamp(m, 3 - pos, n + 2 - pos)]
            // with dw[m] = D(pos - 3 + m) the window's neighbour differences
            double nr[7];
#pragma unroll
            for (int m = 0; m < 7; ++m) nr[m] = (gw[d][m + 1] - gw[d][m]) * ihd[d];
            if (pos[d] < 3 || pos[d] > n[d] - 4) clamp_window(nr, 3 - pos[d], n[d] + 2 - pos[d]);
            const double EPS = 1.0e-10;
            double fm = weno_left(nr[1], nr[2], nr[3], nr[4], nr[5], EPS);   // tdata%s2
            double fp = weno_right(nr[2], nr[3], nr[4], nr[5], nr[6], EPS);  // tdata%s1
            if (pos_sign) sel[d] = fmax(-fmin(fp, 0.0), fmax(fm, 0.0));
            else sel[d] = fmax(fmax(fp, 0.0), -fmin(fm, 0.0));
        }
        const double g = DIM == 3 ? sqrt(sel[0] * sel[0] + sel[1] * sel[1] + sel[2] * sel[2])
                                  : sqrt(sel[0] * sel[0] + sel[1] * sel[1]);
        if (STAGE >= 2) grad[off] = g;   // grad%now holds the last stage's
        if (STAGE != REDIS_GRADIENT) {
            if (BTN && in_band(p0, iw)) {
                double hh, dd;
                lsfun(p0, w, hh, dd);
                const double lam = DIM == 3 ? (2.0 * (1.0 - r12) * hh + r12) * dd : dd;
                grad[off] = g;
                s2[off] = lam * S * (g - 1.0);
                s3[off] = g * dd * lam;
                hold = 1;
            } else {
                const double l = S * g - S;
                const double pn = redis_update<STAGE>(p0, l, l1o, l2o, rdt);
                if (STAGE == 0) l1[off] = l;
                if (STAGE == 1) l2[off] = l;
                out[off] = pn;
                if (STAGE == 2) err = fabs(pst - pn);
            }
        }
    }
    if (BTN && STAGE != REDIS_GRADIENT)
        band.append(STAGE, hold, (unsigned)bx_ + gridDim.x * ((unsigned)by_ + gridDim.y * (unsigned)bz_));
    if (STAGE == 2) {
        __shared__ double sh[4];
        redis_shard_max(err, sh, flags);
    }
}

// The band cells of a stage: 3^d weighted sums of the constraint terms
// (centre weight 16 in 2D, 51 in 3D, bc() copy as clamped indices), the
// correction (redis_lambda :385-408), source and update as in k_redis_stage.
// A term outside the band is 0 (its delta is) and is not stored: it is read
// all the same and not selected, so that the loads of a plane issue together.
// A block takes up to BAND_TILES listed tiles at a time (tiles of gx x gy blocks a
// plane) and works on their band cells with full waves (band_collect): a
// band is a few cells thick, so about a tenth of a listed tile's lanes hold
// one.  18 us at 160 x 144 x 200.  One column of 16 planes per thread, tangent to the band,
// took 350 us at 256^3 for 0.4 % of the cells; one tile per block 53 us at
// 160 x 144 x 200.
template <int DIM, int STAGE>
__global__ void __launch_bounds__(256) k_redis_band(const double *__restrict__ phi, double *__restrict__ out,
                                                    const double *__restrict__ S0, const double *__restrict__ grad,
                                                    const double *__restrict__ s2, const double *__restrict__ s3,
                                                    double *__restrict__ l1, double *__restrict__ l2, BandList band,
                                                    unsigned long long *flags, Geom G, double w, double iw,
                                                    double rdt, unsigned gx, unsigned gy) {
    __shared__ BandCells sh;
    __shared__ unsigned long long s_err[BAND_TILES];
    const int t = threadIdx.x + threadIdx.y * blockDim.x;
    const unsigned total = band.total(STAGE);
    // cell of thread slot th of listed tile number `tile`
    auto cell_of = [&](unsigned tile, int th, int &i, int &j, int &k) {
        const unsigned r = tile / gx, k_ = r / gy;
        const int tx = th % (int)blockDim.x, ty = th / (int)blockDim.x;
        i = (int)((tile - r * gx) * blockDim.x) + tx;
        j = (int)((r - k_ * gy) * blockDim.y) + ty;
        k = (int)k_;
        return i < G.nx && j < G.ny;
    };
    const int per = band_per(band, total);
    for (unsigned g = blockIdx.x * per; g < total; g += gridDim.x * per) {
        if (t < BAND_TILES) s_err[t] = 0ull;
        band_collect(sh, band, STAGE, g, total, per, phi, G, cell_of, [&](double p) { return in_band(p, iw); });
        for (int c = t; c < sh.n; c += 256) {
            const int slot = sh.cell[c] / 256;
            int i, j, k;
            cell_of(sh.tile[slot], sh.cell[c] % 256, i, j, k);
            const long id = G.id(i, j, k);
            const double p0 = phi[id];
            const int is[3] = {max(i - 1, 0), i, min(i + 1, G.nx - 1)};
            const int js[3] = {max(j - 1, 0), j, min(j + 1, G.ny - 1)};
            double hh, dd;
            lsfun(p0, w, hh, dd);
            double a = (DIM == 3 ? 51.0 : 16.0) * s2[id], b = (DIM == 3 ? 51.0 : 16.0) * s3[id];
            const double S = S0[id], gr = grad[id];
            const double l1o = STAGE >= 1 ? l1[id] : 0.0, l2o = STAGE == 2 ? l2[id] : 0.0;
            const double pst = STAGE == 2 ? out[id] : 0.0;
#pragma unroll
            for (int kk = 0; kk < (DIM == 3 ? 3 : 1); ++kk) {
                const int kq = DIM == 3 ? clampi(k + kk - 1, 0, G.nz - 1) : k;
                double ph[9], ta[9], tb[9];
#pragma unroll
                for (int m = 0; m < 9; ++m) {
                    const long o = G.id(is[m % 3], js[m / 3], kq);
                    ph[m] = phi[o];
                    ta[m] = s2[o];
                    tb[m] = s3[o];
                }
                double pa = 0.0, pb = 0.0;
#pragma unroll
                for (int m = 0; m < 9; ++m) {
                    const bool held = in_band(ph[m], iw);
                    const double xa = held ? ta[m] : 0.0, xb = held ? tb[m] : 0.0;
                    if (DIM == 3) {
                        pa += xa;
                        pb += xb;
                    } else {
                        a = a + xa;
                        b = b + xb;
                    }
                }
                if (DIM == 3) {
                    a += pa;
                    b += pb;
                }
            }
            const double s1 = fabs(b) > 1.0e-12 ? a / b * dd : 0.0;
            const double l = (S - s1) * gr - S, pn = redis_update<STAGE>(p0, l, l1o, l2o, rdt);
            if (STAGE == 0) l1[id] = l;
            if (STAGE == 1) l2[id] = l;
            out[id] = pn;
            if (STAGE == 2)   // max of non-negative doubles as bit patterns
                atomicMax(&s_err[slot], (unsigned long long)__double_as_longlong(fabs(pst - pn)));
        }
        __syncthreads();
        if (STAGE == 2 && t < per && g + t < total) {
            const int q = case_of<DIM>((int)(sh.tile[t] / gx / gy));
            atomicMax(&flags[(long)q * FLAG_STRIDE + FLAG_SHARD0 + sh.tile[t] % NSHARD], s_err[t]);
        }
        __syncthreads();
    }
}

// end of one pseudo step: count it, stop when the max over the shards is
// <= tol, clear the shards (one block of NSHARD threads per case); the
// case's done word also goes to poll[case], pinned host memory, so that the
// host's poll needs no copy launch.  Clears the band lists' counters.
__global__ void __launch_bounds__(NSHARD) k_redis_check(unsigned long long *flags, double tol,
                                                        unsigned long long *poll, BandList band) {
    __shared__ double sh[4];
    flags += (long)blockIdx.x * FLAG_STRIDE;
    const int t = threadIdx.x;
    band.clear();
    if (flags[1]) {
        if (t == 0) poll[blockIdx.x] = 1ull;
        return;
    }
    const double e = __longlong_as_double((long long)flags[FLAG_SHARD0 + t]);
    const double err = block_max256(e, sh);
    flags[FLAG_SHARD0 + t] = 0ull;
    if (t == 0) {
        flags[2] += 1;
        if (err <= tol) flags[1] = 1;
        poll[blockIdx.x] = err <= tol ? 1ull : 0ull;
    }
}

__global__ void k_sign_init(const double *__restrict__ phi, double *__restrict__ S0, Geom G, double w, int btn,
                            BandList band) {
    band.clear();
    int bx_, by_, bz_;
    xcd_block(bx_, by_, bz_);
    const int i = bx_ * blockDim.x + threadIdx.x, j = by_ * blockDim.y + threadIdx.y, k = bz_;
    if (i >= G.nx || j >= G.ny) return;
    long id = G.id(i, j, k);
    if (btn == 0) {
        S0[id] = phi[id];
    } else {
        double h, d;
        lsfun(phi[id], w, h, d);
        S0[id] = 2.0 * h - 1.0;
    }
}

// max of grad over the interior into flags[3] (level_set_redis_stable :113-122)
__global__ void k_max_interior(const double *__restrict__ a, unsigned long long *flags, Geom G) {
    int bx_, by_, bz_;
    xcd_block(bx_, by_, bz_);
    const int i = bx_ * blockDim.x + threadIdx.x, j = by_ * blockDim.y + threadIdx.y, k = bz_;
    __shared__ double sh[4];
    double v = 0.0;
    if (i < G.nx && j < G.ny) v = a[G.id(i, j, k)];
    v = block_max256(v, sh);
    const long q = G.dim == 2 ? k : 0;   // the case of a batched stack
    if (threadIdx.x + threadIdx.y == 0)
        atomicMax(&flags[q * FLAG_STRIDE + 3], (unsigned long long)__double_as_longlong(v));
}

__global__ void k_scale_by_flag(double *__restrict__ phi, const unsigned long long *flags, Geom G) {
    int bx_, by_, bz_;
    xcd_block(bx_, by_, bz_);
    const int i = bx_ * blockDim.x + threadIdx.x, j = by_ * blockDim.y + threadIdx.y, k = bz_;
    if (i >= G.nx || j >= G.ny) return;
    double gmax = __longlong_as_double((long long)flags[(G.dim == 2 ? (long)k : 0L) * FLAG_STRIDE + 3]);
    long id = G.id(i, j, k);
    phi[id] = phi[id] / gmax;
}

// one stage: k_redis_stage on every cell, then the listed tiles' band cells
template <int DIM, int STAGE>
static int redis_stage(fcfd_ctx *c, dim3 grd, dim3 blk, int btn, const double *in, double *out, int lo) {
    const Geom &G = c->G;
    const double w = c->pr.ls_wid, iw = 1.0 / w, r12 = c->pr.rho_12, rdt = c->pr.rdt;
    double *grad = c->f[FCFD_GRAD];
    const long nt = (long)grd.x * grd.y * grd.z;
    const BandList band = band_lists(c, nt);
    const Recip ih{1.0 / G.dx, 1.0 / G.dy, 1.0 / G.dz};
    {
        ProfScope ps_(c, R_REDIS_A);
        if (btn)
            hipLaunchKernelGGL((k_redis_stage<DIM, STAGE, true>), grd, blk, 0, c->stream, in, out, c->s0, grad, c->s2,
                               c->s3, c->l1, c->l2, band, c->flag, G, w, iw, r12, rdt, ih, lo);
        else
            hipLaunchKernelGGL((k_redis_stage<DIM, STAGE, false>), grd, blk, 0, c->stream, in, out, c->s0, grad,
                               c->s2, c->s3, c->l1, c->l2, band, c->flag, G, w, iw, r12, rdt, ih, lo);
    }
    FCFD_CHECK(hipGetLastError());
    if constexpr (STAGE != REDIS_GRADIENT) {
        if (btn) {
            ProfScope ps_(c, R_REDIS_B);
            hipLaunchKernelGGL((k_redis_band<DIM, STAGE>), band_grid(c, nt), blk, 0, c->stream, in, out, c->s0, grad,
                               c->s2, c->s3, c->l1, c->l2, band, c->flag, G, w, iw, rdt, grd.x, grd.y);
            FCFD_CHECK(hipGetLastError());
        }
    }
    return FCFD_OK;
}

template <int DIM>
static int redis_pseudo_step(fcfd_ctx *c, dim3 grd, dim3 blk, int btn, int lo) {
    double *phi = c->f[FCFD_PHI];   // phi_start, overwritten by the last stage
    FCFD_TRY((redis_stage<DIM, 0>(c, grd, blk, btn, phi, c->phiB, lo)));
    FCFD_TRY((redis_stage<DIM, 1>(c, grd, blk, btn, c->phiB, c->phiS, 0)));
    return redis_stage<DIM, 2>(c, grd, blk, btn, c->phiS, phi, 0);
}

int redis(fcfd_ctx *c, int btn, int *iters) {
    const Geom &G = c->G;
    const dim3 blk = tile_rows(G.nx), grd = grid_interior(G, blk);
    double *phi = c->f[FCFD_PHI], *grad = c->f[FCFD_GRAD];
    const double w = c->pr.ls_wid, rdt = c->pr.rdt;
    int lo = -1;   // the caller's ghosts until a bc() or a stage has replaced them
    FCFD_CHECK(hipMemsetAsync(c->flag, 0, (size_t)FLAG_STRIDE * c->nb * sizeof(unsigned long long), c->stream));
    // level_set_redis_init / stable (:67-136)
    hipLaunchKernelGGL(k_sign_init, grd, blk, 0, c->stream, phi, c->s0, G, w, btn, band_lists(c, 0));
    if (btn == 0) {
        if (G.dim == 3) FCFD_TRY((redis_stage<3, REDIS_GRADIENT>(c, grd, blk, 0, phi, nullptr, lo)));
        else FCFD_TRY((redis_stage<2, REDIS_GRADIENT>(c, grd, blk, 0, phi, nullptr, lo)));
        hipLaunchKernelGGL(k_max_interior, grd, blk, 0, c->stream, grad, c->flag, G);
        hipLaunchKernelGGL(k_scale_by_flag, grd, blk, 0, c->stream, phi, c->flag, G);
        lo = 0;   // the scaled phi's ghosts are bc() copies
    }
    // pseudo-time budget: the reference stops once the accumulated time exceeds
    // timestop (:18-28,54); replay that accumulation to fix the launch count
    double timestop;
    if (btn == 0) {
        double m = c->gd.xend - c->gd.xstart;
        m = fmax(m, c->gd.yend - c->gd.ystart);
        if (G.dim == 3) m = fmax(m, c->gd.zend - c->gd.zstart);
        timestop = 1.5 * m;
    } else {
        timestop = 3.0 * G.dx;
    }
    int nmax = 0;
    for (double t = 0.0;;) {
        nmax += 1;
        t = t + rdt;
        if (t > timestop) break;
        if (nmax > 10000000) return FCFD_ERR_ARG;
    }
    const double tol = G.dim == 3 ? 1.0e-5 : 1.0e-8;
    // The stop test runs on the device (k_redis_check); a stopped case's
    // kernels return at once.  The done words of pseudo-step `it` reach the
    // host behind it, and before step it+2 is queued the host reads
    // them, so it stops queueing once every case has stopped while one step
    // stays queued ahead.  Slots of flag_host past the 4 nb words read below.
    for (int q = 0; q < 2; ++q)
        if (!c->redis_ev[q]) FCFD_CHECK(hipEventCreateWithFlags(&c->redis_ev[q], hipEventDisableTiming));
    unsigned long long *poll[2] = {c->flag_host + 4 * c->nb, c->flag_host + 5 * c->nb};
    for (int it = 0; it < nmax; ++it) {
        if (it >= 2) {
            FCFD_CHECK(hipEventSynchronize(c->redis_ev[it & 1]));
            bool all = true;
            for (int q = 0; q < c->nb; ++q) all = all && poll[it & 1][q] != 0ull;
            if (all) break;
        }
        if (G.dim == 3) FCFD_TRY(redis_pseudo_step<3>(c, grd, blk, btn, it == 0 ? lo : 0));
        else FCFD_TRY(redis_pseudo_step<2>(c, grd, blk, btn, it == 0 ? lo : 0));
        hipLaunchKernelGGL(k_redis_check, dim3(c->nb), dim3(NSHARD), 0, c->stream, c->flag, tol, poll[it & 1],
                           band_lists(c, 0));
        FCFD_CHECK(hipGetLastError());
        FCFD_CHECK(hipEventRecord(c->redis_ev[it & 1], c->stream));
    }
    FCFD_TRY(bc_scalar(c, phi));
    // words 0..3 of every case's flag block
    FCFD_TRY(gather_to_host(c, c->flag_host, c->flag, FLAG_STRIDE, 4, c->nb));
    FCFD_CHECK(hipStreamSynchronize(c->stream));
    int most = 0;   // a batched stack reports the largest pseudo-step count of its cases
    for (int q = 0; q < c->nb; ++q) most = std::max(most, (int)c->flag_host[4 * q + 2]);
    c->diag.redis_iters = most;
    if (iters) *iters = most;
    return FCFD_OK;
}

}  // namespace fcfd
