// fcfd_internal.h — device context and helpers shared by the HIP sources of
// libfcfd.  Everything here is MI355X (gfx950, wave64) code.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../include/fcfd.h"

#define FCFD_CHECK(call)                                                                \
    do {                                                                                \
        hipError_t e_ = (call);                                                         \
        if (e_ != hipSuccess) {                                                         \
            fprintf(stderr, "libfcfd: HIP error %s at %s:%d\n", hipGetErrorString(e_), \
                    __FILE__, __LINE__);                                                \
            return FCFD_ERR_HIP;                                                        \
        }                                                                               \
    } while (0)

#define FCFD_TRY(expr)              \
    do {                            \
        int rc_ = (expr);           \
        if (rc_ != FCFD_OK) return rc_; \
    } while (0)

namespace fcfd {

constexpr int WAVE = 64;

// Geometry of one ghosted field: interior (nx, ny, nz), ghost width g (gz = 0
// in 2D), strides of the column-major reference layout.
struct Geom {
    int dim, nx, ny, nz, g, gz;
    long sx, sxy, ntot;
    double dx, dy, dz;
    // Ghost depth that holds a neighbour's data on each face (x low / high,
    // y, z): 0 on a physical face, where kernels read clamped indices as the
    // reference's zero-gradient copies; up to g on a face between blocks of
    // a multi-block layout, whose ghosts a halo exchange fills.
    int ox0 = 0, ox1 = 0, oy0 = 0, oy1 = 0, oz0 = 0, oz1 = 0;
    __host__ __device__ long id(int i, int j, int k) const {
        return (long)(i + g) + (long)(j + g) * sx + (long)(k + gz) * sxy;
    }
};

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// d[m] <- d[clamp(m, lo, hi)] for m = 0 .. W-1 (0 <= lo <= hi < W) by
// selects, without indexing registers at run time: the clamped differences
// of a line near a wall taken from the unclamped ones of its load window
template <int W>
__device__ __forceinline__ void clamp_window(double (&d)[W], int lo, int hi) {
    double vlo = d[0], vhi = d[0];
#pragma unroll
    for (int r = 1; r < W; ++r) {
        vlo = lo == r ? d[r] : vlo;
        vhi = hi == r ? d[r] : vhi;
    }
#pragma unroll
    for (int m = 0; m < W; ++m) d[m] = m < lo ? vlo : (m > hi ? vhi : d[m]);
}

// element at a byte offset from a base that is uniform over the wave: the
// load takes the base from scalar registers and 32 offset bits per lane (an
// index would be scaled in 64-bit vector arithmetic for every load).  A
// caller's 32-bit offsets must stay below 4 GiB: inside a tile or a row
// segment, not inside a plane (a 2D plane of 23200 x 23200 cells is larger);
// 64-bit offsets are plain addresses.
template <typename T, typename O>
__device__ __forceinline__ T &at_bytes(T *base, O bytes) {
    return *(T *)((char *)base + bytes);
}
template <typename T, typename O>
__device__ __forceinline__ const T &at_bytes(const T *base, O bytes) {
    return *(const T *)((const char *)base + bytes);
}

// The W values of a field's line around a cell, at pos - BELOW .. of the
// line, indices clamped to [lo, n - 1].  base: the address of the block's
// first cell (uniform over the block), off: the cell's distance from it.  A
// wave whose cells all lie inside the line reads at uniform strides from
// scalar bases (one vector offset for every load of the kernel, where
// per-lane 64-bit addresses take 4-6 instructions a load); the others clamp
// lane by lane.
template <int W, int BELOW>
__device__ __forceinline__ void line_load(const double *__restrict__ base, unsigned off, long st, int pos, int n,
                                          int lo, double (&g)[W]) {
    if (__all(pos - BELOW >= lo && pos + W - 1 - BELOW < n)) {
#pragma unroll
        for (int r = 0; r < W; ++r) g[r] = at_bytes(base + (r - BELOW) * st, off * (unsigned)sizeof(double));
    } else {
#pragma unroll
        for (int r = 0; r < W; ++r) {
            const int q = r < BELOW ? max(pos + r - BELOW, lo) : min(pos + r - BELOW, n - 1);
            g[r] = base[(long)off + (long)(q - pos) * st];
        }
    }
}

// One level of the pressure multigrid hierarchy (see mg.hip).
struct MgLevel {
    int nx, ny, nz;          // cells
    int cx, cy, cz;          // coarsening factor (1|2) to the next level
    double hx, hy, hz;       // spacing
    double wx = 1, wy = 1, wz = 1;   // width of each axis' last cell / spacing (odd axes: see mg.hip)
    long sx, sxy, ntot;      // layout with one ghost layer (finest uses Geom)
    // FP64 arrays (level >= 1): solution/error, rhs, residual, face coeffs
    double *e64, *f64, *r64, *bx64, *by64, *bz64;
    // FP32 mirrors for the mixed-precision inner cycle; e32b is the second
    // error buffer of the fused multi-sweep smoother (read one, write the other)
    float *e32, *f32, *r32, *bx32, *by32, *bz32, *e32b;
    // FP16 face coefficients of level 1 in 3D (params.ppe_rho_half), read by
    // its FP32 smoothing and restriction; NULL elsewhere
    _Float16 *bx16, *by16, *bz16;
};

// Kernel regions timed by the built-in HIP-event profiler (fcfd_prof_*).
enum Region {
    R_LS_ADV, R_REDIS_A, R_REDIS_B, R_MASS, R_MPLS_UPD, R_CCD, R_CURV, R_DIFF, R_PRED, R_PPE_SRC,
    R_PROJ, R_NODE_VEL, R_BC, R_SMOOTH0, R_SMOOTHC, R_RESTRICT0, R_RESTRICTC, R_PROLONG0, R_PROLONGC,
    R_RESID0, R_COARSE, R_FCG, R_MISC, NREG
};

struct ProfRec {
    int reg;
    int ev;   // index of the start event in the pool (end = ev + 1)
};

struct Prof {
    int on = 0;
    std::vector<hipEvent_t> pool;
    std::vector<ProfRec> recs;
    size_t used = 0;
};

struct Reduce {
    double *partial;         // per-block partial results (nslots * nblocks)
    double *partial2;        // second-stage partials (4 slots x 256), inside `partial`
    double *result;          // reduced values (device)
    double *host;            // pinned host mirror
    int nblocks;
};

}  // namespace fcfd

struct fcfd_ctx {
    fcfd_grid gd;
    fcfd_params pr;
    fcfd::Geom G;
    int tile[FCFD_NTILE][3];   // thread-block tile (x, y) and slab rows per enum fcfd_tile_kernel
    hipStream_t stream;
    int device;
    int ncu;                   // compute units of the device
    // ---- state (device, full ghosted arrays) ----
    double *f[FCFD_NFIELDS];   // indexed by enum fcfd_field; NULL when not held
    // ---- scratch ----
    double *phiB, *phiS;       // ping-pong phi buffers / stage start copy
    double *l1, *l2;           // stored RK stage sources
    double *s2, *s3, *s0;      // reinit work: lambda numerator/denominator, frozen sign
    unsigned *band;            // reinit work: counters and lists of the tiles that hold interface-band cells
    double *cx, *cy, *cz;      // CCD second-derivative scratch / cross-derivative temp
    double *dsu, *dsv, *dsw;   // viscous + body force source (sec_part1..3), once per step
    double *un, *vn, *wn;      // predictor output buffer (ping-pong with u, v, w)
    double *ccd_coef[18];      // factorised line matrices [kind * 3 + direction]: CCD, UCCD up / down on
                               // ghosted lines, the same on interior lines (MPLS_RisingBubble set)
    double *ccd_seg[18];       // the same per segment for the partitioned y / z solve, + reduced block LU
    double *ccd_z;             // partitioned solve: segment end values / interface values per line
    double *adj[5];            // advection adjoint: stage states phi1, phi2, adjoints lambda1, lambda2, seed
    float *adv32[4];           // FP32 advection: two stage buffers and the stage sources l1, l2
    float *adj32[7];           // FP32 adjoint: phi1, phi2, lambda1, lambda2, seed, stage sources l1, l2
    double vscale = 1.0;       // factor on NU/NV/NW in the WENO5 advection and its adjoint
    // ---- batched 2D stack (fcfd_create_batch): case q is the slice k = q ----
    int nb = 1;                        // cases in the stack; 1 for an ordinary context
    fcfd_case *cases_dev = nullptr;    // per-case parameters on the device; NULL when nb == 1
    std::vector<fcfd_case> cases;      // host copy
    // ---- reductions ----
    fcfd::Reduce red;
    unsigned long long *flag;  // device flags (reinit error max bits, done, count)
    unsigned long long *flag_host;
    hipEvent_t redis_ev[2] = {nullptr, nullptr};   // reinit stop polls in flight
    // ---- multigrid ----
    std::vector<fcfd::MgLevel> mg;
    float *rho32;              // FP32 copy of rho for the mixed inner cycle
    _Float16 *rho16;           // FP16 copy (params.ppe_rho_half)
    double *mg_scalars;        // device scalars of the solve (norms)
    int mg_ready;
    // level-0 Krylov vectors of the flexible CG (FP64) and FP32 previous z
    double *kr, *kp, *kq, *kz, *kzo;
    float *kzo32;
    // captured V-cycles: [kind][inner cycles 1..4]; kind 0 fp64 on p, 1 fp64 on
    // z with the CG dots, 2 fp32 on e32, 3 fp32 on e32 with the CG dots
    hipGraphExec_t vgraph[2][4][5];                      // [host status slot][kind][inner]
    int *mg_skip;              // device flag: every case's flexible-CG solve has ended
    hipEvent_t cg_ev[2];       // end of the flexible-CG iteration of each host status slot
    std::vector<std::pair<int, int>> vgraph_prof[4][5];  // (region, event) pairs inside each graph
    int capture_kind = -1, capture_inner = 0;            // graph being captured (or -1)
    double prof_gms[fcfd::NREG] = {};                    // timings folded in from graph replays
    int64_t prof_gcnt[fcfd::NREG] = {};
    // ---- bookkeeping ----
    double time;
    int iter;
    int diag_pending;          // step diagnostics of every case waiting in diag_host
    double *diag_host;         // pinned: result words 0..DIAG_W-1 of case q at [q*DIAG_W]
    unsigned long long *pack;  // device staging for per-case values gathered to the host (16 words per case)
    fcfd_diag diag;
    fcfd_m3_state m3 = {{0.0, 0.0}, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 1.0e-5, 0, 0};   // MPLS_RisingBubble step
    fcfd::Prof prof;
};

namespace fcfd {
// Records a start/end HIP event pair on the context stream around the launches
// of its scope when profiling is on.
struct ProfScope {
    fcfd_ctx *c;
    int reg, ev;
    ProfScope(fcfd_ctx *c_, int reg_);
    ~ProfScope();
};
}  // namespace fcfd

namespace fcfd {

// Sum over the threads of a 256-thread block in a fixed order: a butterfly
// inside each wave (lane 0's value is used), then the four wave sums in
// order.  Every thread gets the result; every thread of the block must call
// it; sh4 is LDS scratch of 4 doubles that may be reused after the call.
__device__ __forceinline__ double block_sum256(double v, double *sh4) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
    const int t = threadIdx.x + threadIdx.y * blockDim.x;
    if ((t & (WAVE - 1)) == 0) sh4[t / WAVE] = v;
    __syncthreads();
    const double s = (sh4[0] + sh4[1]) + (sh4[2] + sh4[3]);
    __syncthreads();
    return s;
}

// Workgroups of a launch are dealt to the 8 XCDs round-robin by linear id
// (x fastest, then y, then z).  Renumbering them so that XCD x owns the
// contiguous range of logical blocks [x*nb/8, (x+1)*nb/8) keeps the k-1 and
// k+1 planes a stencil re-reads in the L2 of the XCD that read them first.
// Returns the logical (bx, by, bz) of the calling workgroup.
constexpr unsigned NXCD = 8;
__device__ __forceinline__ void xcd_block(int &bx, int &by, int &bz) {
    const unsigned nbx = gridDim.x, nby = gridDim.y, nb = nbx * nby * gridDim.z;
    const unsigned w = blockIdx.x + nbx * (blockIdx.y + nby * blockIdx.z);
    const unsigned q = nb / NXCD, rem = nb % NXCD, x = w % NXCD;
    const unsigned l = x * q + (x < rem ? x : rem) + w / NXCD;
    bx = (int)(l % nbx);
    const unsigned r = l / nbx;
    by = (int)(r % nby);
    bz = (int)(r / nby);
}

// xcd_block with another order of the logical blocks: with slab = S > 0 the
// tile rows are grouped in slabs of S rows, and an XCD's contiguous range
// walks the planes of one slab (x fastest, then the slab's rows, then the
// planes) before the next slab.  A plane's footprint per XCD is then S tile
// rows instead of the whole plane, so the k-2 .. k+2 planes a z-stencil
// re-reads are still in the XCD's L2.  slab = 0 is xcd_block's order.
__device__ __forceinline__ void xcd_block_slab(int &bx, int &by, int &bz, int slab) {
    const unsigned nbx = gridDim.x, nby = gridDim.y, nbz = gridDim.z, nb = nbx * nby * nbz;
    const unsigned w = blockIdx.x + nbx * (blockIdx.y + nby * blockIdx.z);
    const unsigned q = nb / NXCD, rem = nb % NXCD, x = w % NXCD;
    const unsigned l = x * q + (x < rem ? x : rem) + w / NXCD;
    if (slab <= 0) {
        bx = (int)(l % nbx);
        const unsigned r = l / nbx;
        by = (int)(r % nby);
        bz = (int)(r / nby);
        return;
    }
    const unsigned S = (unsigned)slab, per = nbx * S * nbz;
    const unsigned sl = l / per, rows = min(S, nby - sl * S);
    const unsigned within = l - sl * per;
    bx = (int)(within % nbx);
    const unsigned r = within / nbx;
    by = (int)(sl * S + r % rows);
    bz = (int)(r / rows);
}

// Max over the threads of a 256-thread block (values >= 0 or any order-free
// max); every thread gets the result; every thread of the block must call it.
__device__ __forceinline__ double block_max256(double v, double *sh4) {
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, WAVE));
    const int t = threadIdx.x + threadIdx.y * blockDim.x;
    if ((t & (WAVE - 1)) == 0) sh4[t / WAVE] = v;
    __syncthreads();
    const double m = fmax(fmax(sh4[0], sh4[1]), fmax(sh4[2], sh4[3]));
    __syncthreads();
    return m;
}

// Tiles of 256 cells that hold cells of the interface band, listed by a
// reinitialisation stage for its band pass: NXCD lists of `cap` entries, a
// block appending to list (block id % NXCD), with a counter per stage and
// list (one counter would serialise the appends).  A list can hold every
// block that appends to it.  The order of a list does not matter: every band
// cell is independent of the others.  A grid of no more tiles than CUs is not
// listed: all tiles are taken (all > 0), which saves the append and two
// memory latencies of the band pass.
struct BandList {
    unsigned *cnt;    // [3 stages][NXCD]
    unsigned *tile;   // [NXCD][cap]
    unsigned cap, ncu, all;
    // list the calling block's tile when any of its threads holds a band cell
    __device__ __forceinline__ void append(int stage, int hold, unsigned id) const {
        if (all) return;
        hold = __syncthreads_or(hold);
        if (hold && threadIdx.x + threadIdx.y == 0) {
            const unsigned q = (blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)) % NXCD;
            tile[q * cap + atomicAdd(&cnt[stage * NXCD + q], 1u)] = id;
        }
    }
    __device__ __forceinline__ unsigned total(int stage) const {
        if (all) return all;
        unsigned n = 0;
#pragma unroll
        for (unsigned q = 0; q < NXCD; ++q) n += cnt[stage * NXCD + q];
        return n;
    }
    // entry `at` of the lists taken end to end
    __device__ __forceinline__ unsigned entry(int stage, unsigned at) const {
        if (all) return at;
        for (unsigned q = 0; q < NXCD; ++q) {
            const unsigned n = cnt[stage * NXCD + q];
            if (at < n) return tile[q * cap + at];
            at -= n;
        }
        return 0;
    }
    // all counters of the lists (of one stage): by the first block of a launch
    __device__ __forceinline__ void clear() const {
        const unsigned t = threadIdx.x + threadIdx.y * blockDim.x;
        if (blockIdx.x + blockIdx.y + blockIdx.z == 0 && t < 3 * NXCD) cnt[t] = 0u;
    }
    __device__ __forceinline__ void clear(int stage) const {
        const unsigned t = threadIdx.x + threadIdx.y * blockDim.x;
        if (blockIdx.x + blockIdx.y + blockIdx.z == 0 && t < NXCD) cnt[stage * NXCD + t] = 0u;
    }
};

// the band cells of `per` listed tiles (entries first .. of `total`, at most
// BAND_TILES), collected by a 256-thread block so that it can work on them
// with full waves: cell[0 .. n) = slot * 256 + thread slot within the tile.
// cell_of(tile, thread slot, i, j, k) places a cell (false: none there),
// inside(phi) is the band test.  A block takes no more tiles than give every
// CU a block, so that a short list is spread over the chip: with 8 whatever
// the list, 64 x 128 cells that all lie in the band were 4 blocks, and a
// pseudo step took 82 us instead of 43 (384 x 768, 4 % of the cells: 77
// instead of 53).
constexpr int BAND_TILES = 8;
__device__ __forceinline__ int band_per(const BandList &band, unsigned total) {
    const unsigned n = (total + band.ncu - 1) / band.ncu;
    return n < 1 ? 1 : (n > BAND_TILES ? BAND_TILES : (int)n);
}
struct BandCells {
    unsigned tile[BAND_TILES];
    unsigned short cell[BAND_TILES * 256];
    int n;
};
template <typename CellOf, typename Inside>
__device__ __forceinline__ void band_collect(BandCells &sh, const BandList &band, int stage, unsigned first,
                                             unsigned total, int per, const double *__restrict__ phi, const Geom &G,
                                             CellOf cell_of, Inside inside) {
    const int t = threadIdx.x + threadIdx.y * blockDim.x;
    if (t < BAND_TILES) sh.tile[t] = t < per ? band.entry(stage, first + t) : 0u;
    if (t == 0) sh.n = 0;
    __syncthreads();
    double p[BAND_TILES];
    unsigned have = 0;
#pragma unroll
    for (int s = 0; s < BAND_TILES; ++s) {
        int i, j, k;
        const bool in = cell_of(sh.tile[s], t, i, j, k) && s < per && first + s < total;
        p[s] = phi[in ? G.id(i, j, k) : G.id(0, 0, 0)];
        have |= in ? 1u << s : 0u;
    }
#pragma unroll
    for (int s = 0; s < BAND_TILES; ++s) {
        const bool held = ((have >> s) & 1u) && inside(p[s]);
        const unsigned long long m = __ballot(held);
        int base = 0;
        if (t % WAVE == 0 && m) base = atomicAdd(&sh.n, __popcll(m));
        base = __shfl(base, 0, WAVE);
        if (held) sh.cell[base + __popcll(m & ((1ull << (t % WAVE)) - 1ull))] = (unsigned short)(s * 256 + t);
    }
    __syncthreads();
}

// device flag words: [0] unused, [1] reinit done, [2] reinit pseudo-step
// count, [3] max |grad phi| bits; [FLAG_SHARD0, +NSHARD) per-block max slots.
// A batched stack holds one such block of FLAG_STRIDE words per case.
constexpr int FLAG_SHARD0 = 16, NSHARD = 256, FLAG_STRIDE = FLAG_SHARD0 + NSHARD;
// reduced values per case in Reduce::result: [0..2] mass sums, [RES_LAMBDA]
// the last MPLS multiplier, [RES_VDIV], [RES_VDIV + 1] max / mean |div u|
// (case 0 only); the first DIAG_W words of every case are gathered to the
// host after each step
constexpr int RES_STRIDE = 16, RES_LAMBDA = 8, RES_VDIV = 9, DIAG_W = 11;

// case index of slice k: a batched 2D stack keeps case q in slice k = q;
// 3D contexts hold one case
template <int DIM>
__device__ __forceinline__ int case_of(int k) { return DIM == 2 ? k : 0; }

// n elements on first use, cleared on st where asked.  *p stays null unless
// all of it succeeded, so that a call after one that ran out of memory asks
// again: each array of a set is tested by itself, never the set by its first.
template <typename T>
inline int alloc_once(T **p, long n, bool clear = false, hipStream_t st = nullptr) {
    if (*p) return FCFD_OK;
    T *q = nullptr;
    FCFD_CHECK(hipMalloc((void **)&q, sizeof(T) * n));
    if (clear && hipMemsetAsync(q, 0, sizeof(T) * n, st) != hipSuccess) {
        (void)hipFree(q);
        return FCFD_ERR_HIP;
    }
    *p = q;
    return FCFD_OK;
}

// launch helpers --------------------------------------------------------
// 256-thread block for rows of w threads: 64 x 4, or 32 x 8 where that
// leaves fewer lanes idle past the row end (140 cells: 160 instead of 192
// threads per row; 70 pairs: 96 instead of 128)
inline dim3 tile_rows(int w) {
    const long p64 = (w + 63) / 64 * 64L, p32 = (w + 31) / 32 * 32L;
    return p32 < p64 ? dim3(32, 8) : dim3(64, 4);
}
inline dim3 tile_blk(const fcfd_ctx *c, int kernel) { return dim3(c->tile[kernel][0], c->tile[kernel][1]); }
// interior cell (i, j, k) of a one-dimensional launch over the nx * ny * nz
// interior cells in memory order (x fastest; no idle lanes at the row ends
// as a 2D tile has when nx is not a multiple of its width), the blocks in
// xcd_block's XCD-contiguous order; false past the last cell.  The launch
// (grid_flat) needs nx * ny * nz < 2^32.
__device__ __forceinline__ bool cell_of_flat(const Geom &G, int &i, int &j, int &k) {
    int bx, by, bz;
    xcd_block(bx, by, bz);
    const unsigned t = (unsigned)bx * blockDim.x + threadIdx.x;
    const unsigned nxy = (unsigned)G.nx * (unsigned)G.ny;
    if (t >= nxy * (unsigned)G.nz) return false;
    const unsigned kk = t / nxy, r = t - kk * nxy, jj = r / (unsigned)G.nx;
    i = (int)(r - jj * (unsigned)G.nx);
    j = (int)jj;
    k = (int)kk;
    return true;
}

// cell (i, j, k) of flattened interior index t (i fastest), by 32-bit
// division where t fits (a 64-bit one is several times longer)
__device__ __forceinline__ void cell_of_index(long t, const Geom &G, int &i, int &j, int &k) {
    if (t < 4294967296L) {
        const unsigned tt = (unsigned)t, nx = (unsigned)G.nx, ny = (unsigned)G.ny;
        const unsigned r = tt / nx, kk = r / ny;
        i = (int)(tt - r * nx);
        j = (int)(r - kk * ny);
        k = (int)kk;
    } else {
        i = (int)(t % G.nx);
        const long r = t / G.nx;
        j = (int)(r % G.ny);
        k = (int)(r / G.ny);
    }
}

// cell_of_flat with the index of the block's first cell (id0, uniform) and
// the cell's distance from it (cells of a block follow each other in memory)
__device__ __forceinline__ bool cell_of_flat(const Geom &G, int &i, int &j, int &k, long &id0, unsigned &off) {
    int bx, by, bz;
    xcd_block(bx, by, bz);
    const unsigned nxy = (unsigned)G.nx * (unsigned)G.ny, t0 = (unsigned)bx * blockDim.x, t = t0 + threadIdx.x;
    const unsigned k0 = t0 / nxy, r0 = t0 - k0 * nxy, j0 = r0 / (unsigned)G.nx;
    id0 = G.id((int)(r0 - j0 * (unsigned)G.nx), (int)j0, (int)k0);
    const unsigned kk = t / nxy, r = t - kk * nxy, jj = r / (unsigned)G.nx;
    i = (int)(r - jj * (unsigned)G.nx);
    j = (int)jj;
    k = (int)kk;
    off = (unsigned)(G.id(i, j, k) - id0);
    return t < nxy * (unsigned)G.nz;
}

inline bool flat_fits(const Geom &G) { return (double)G.nx * G.ny * G.nz < 4294967296.0 - 1024.0; }

inline dim3 grid_flat(const Geom &G, int blk) {
    return dim3((unsigned)(((long)G.nx * G.ny * G.nz + blk - 1) / blk));
}

inline dim3 grid_interior(const Geom &G, dim3 blk) {
    return dim3((G.nx + blk.x - 1) / blk.x, (G.ny + blk.y - 1) / blk.y, G.nz);
}

// the band lists of a launch of ntiles 256-thread blocks (the context holds
// room for the larger of its tiled and its flat launch over the interior)
inline BandList band_lists(const fcfd_ctx *c, long ntiles) {
    return BandList{c->band, c->band + 3 * NXCD, (unsigned)((ntiles + NXCD - 1) / NXCD), (unsigned)c->ncu,
                    ntiles <= c->ncu ? (unsigned)ntiles : 0u};
}
// blocks that share the listed tiles: one per tile up to one per CU, then as
// many as BAND_TILES each take, up to 4 per CU
inline dim3 band_grid(const fcfd_ctx *c, long ntiles) {
    const long few = ntiles < c->ncu ? ntiles : c->ncu, n = (ntiles + BAND_TILES - 1) / BAND_TILES, most = 4L * c->ncu;
    return dim3((unsigned)(n < few ? few : (n < most ? n : most)));
}

// kernels implemented in the .hip files (host wrappers)
int upload_cases(fcfd_ctx *c);
// rows of `width` 8-byte words, `pitch` words apart on the device, into
// consecutive host words (one contiguous copy; a gather kernel first when
// there is more than one row); stream ordered
int gather_to_host(fcfd_ctx *c, void *host, const void *dev, long pitch, int width, int rows);
int bc_scalar(fcfd_ctx *c, double *d);
int bc_scalar_f32(fcfd_ctx *c, float *d);
int velbc(fcfd_ctx *c, double *u, double *v, double *w, int nodal);
int ls_props(fcfd_ctx *c, const double *phi, double *H, double *D, double *S, double *rho, double *mu);
int reduce_sums(fcfd_ctx *c, int kind, const double *a, const double *b, const double *cc, const double *d);
int ccd_dir(fcfd_ctx *c, int dir, const double *f, double *fx, double *fxx);
int ccd_lines_set(fcfd_ctx *c, int set, int dir, const double *f, double *fx, double *fxx);
int m3_fields(fcfd_ctx *c);
int uccd_lines_set(fcfd_ctx *c, int set, int dir, const double *f, const double *u, double *fx, double *fxx);
int uccd_dir(fcfd_ctx *c, int dir, const double *f, const double *u, double *fx, double *fxx);
int ls_adv_stage_f32(fcfd_ctx *c, const float *phi, float *phin, const float *nu, const float *nv, const float *nw,
                     float *l1, float *l2, int stage);
// a block of a multi-block layout: its geometry (with open faces) and its
// offset in a stack
struct BlockGeom {
    Geom G;
    long off;
};
// one WENO5 SSP-RK3 stage on every block of a layout in one launch: tab on
// the device, nx, ny, nz the largest block's extents; phin's ghosts are not
// written
int ls_adv_stage_blocks(hipStream_t st, int ncu, const BlockGeom *tab, int nblk, int dim, int nx, int ny, int nz,
                        const double *phi, double *phin, const double *nu, const double *nv, const double *nw,
                        double *l1, double *l2, double dt, int stage);
int ccd_setup(fcfd_ctx *c);
int surface_norms(fcfd_ctx *c, const double *phi, int full);
int curv_kernel(fcfd_ctx *c);
int ls_advect(fcfd_ctx *c);
int ls_adv_stage(fcfd_ctx *c, const double *phi, double *phin, int stage);
int ls_advect_f32(fcfd_ctx *c, float *phi, const float *nu, const float *nv, const float *nw);
int ls_adv_adjoint_step(fcfd_ctx *c, const double *phi, double *lambda, double *ub, double *vb, double *wb);
int redis(fcfd_ctx *c, int btn, int *iters);
int mpls(fcfd_ctx *c);
int ls_mv(fcfd_ctx *c, double *mass, double *vol);
int ns_diff_source(fcfd_ctx *c);
int ns_predictor(fcfd_ctx *c, const double *ut, const double *vt, const double *wt, int write_src = 1);
int ppe_src(fcfd_ctx *c);
int projection(fcfd_ctx *c);
int node_vel(fcfd_ctx *c);
int div_check(fcfd_ctx *c, int to_host);
int mg_setup(fcfd_ctx *c);
int mg_free(fcfd_ctx *c);
int mg_drop_graphs(fcfd_ctx *c);
int prof_graph_accum(fcfd_ctx *c, int kind, int inner);
int ppe_solve(fcfd_ctx *c, double rel_tol, int precision, int *cycles, double *rel, int normalize = 1);
int copy_field(fcfd_ctx *c, double *dst, const double *src);

}  // namespace fcfd
