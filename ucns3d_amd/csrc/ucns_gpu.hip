// libucnsgpu.so -- MI355X (gfx950) residual + SSP-RK3 path behind include/ucns.h.
//
// Per RK stage three kernels run on the library stream:
//   reconstruction  stencil LSQ contraction (P_s dU_s), smoothness indicators
//             and WENO weights, the weighted polynomial at every face Gauss
//             point, CHECKSOL -> MUSCL/Barth -> CHECKSOLX, ULEFT written once
//             per cell (ARBITRARY_ORDER, src/reconstruct_p.f90:2954-3015):
//             recon_tiled.hip (a wave per tile of 8 cells), recon_block.hip
//             and recon_cweno5.hip (a block of waves per tile),
//             recon_muscl.hip (8 lanes per cell), k_recon here (a wave per cell)
//   fluxes    per unique face: rotate, HLLC, rotate back at each Gauss point;
//             the area-weighted sum is written once per face
//             (CALCULATE_FLUXESHI_CONVECTIVE, src/flux_p.f90:478-1030, which
//             solves every face twice; here each face is solved once and
//             scattered atomic-free by the gather below): k_flux_points, or
//             k_flux where faces have one point
//   k_update  one thread per cell: RHS = signed sum of its faces' fluxes, the
//             Shu-Osher stage update (RUNGE_KUTTA3, src/time_p.f90:885-1027),
//             and after the last stage the next dt as a min-reduction
//             (CALCULATE_CFL, src/time_p.f90:27-116)
// Small meshes of one-point faces run fluxes and update as one (k_flux_update).
// Device layouts are chosen for coalescing and differ from the ABI layouts;
// ucns_upload_prestore converts.  FP64 everywhere in UCNS_FP64; in UCNS_MIXED
// the stencil matrices, indicators, Gauss points, reconstruction, weights and
// HLLC run in FP32 while dU formation, conserved->primitive recovery, flux
// accumulation, the RK update and dt stay FP64.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "ucns.h"
#include "ucns_device.h"
#include "ucns_recon.h"
#include "ucns_tiled.h"

using namespace ucns;

namespace {

#define HIP_TRY(expr)                                                                       \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess) {                                                             \
            ctx->err = std::string(#expr) + ": " + hipGetErrorString(e_);                   \
            return UCNS_EHIP;                                                               \
        }                                                                                   \
    } while (0)

template <typename R, int IDEG, int IMAX, int TSMAX>
struct ReconShared {
    static constexpr int NQMAX = 6 * 16;
    union {
        R du[TSMAX * IMAX * NV];  // phase 1
        struct {
            R gh[IDEG * NV];         // combined polynomial
            R beta[TSMAX * NV];
            R omega[TSMAX * NV];
            R ul[NQMAX * NV];        // face-point values
        } late;
    } u;
    R g[TSMAX * IDEG * NV];                 // per-stencil coefficients
    R b[IDEG * IDEG];                // indicator, unpacked
    R mb[IDEG];
    double ui[NV];
};

// Fused reconstruction, one wavefront per cell: WENO-5, the linear central
// polynomial without the limiter (iweno 1, idegfree 3), and shapes and face rules
// the tiled kernels do not hold.
// CH: characteristic-variable WENO, face by face (src/reconstruct_p.f90:497-758).
template <typename R, int IDEG, int IMAX, int TSMAX, bool CH = false>
__global__ __launch_bounds__(WAVE) void k_recon(ReconParams<R> p) {
    constexpr int NROW = (TSMAX * IDEG + WAVE - 1) / WAVE;
    __shared__ ReconShared<R, IDEG, IMAX, TSMAX> sh;
    const int lane = threadIdx.x;
    // XCD-aware order: consecutive blocks go to different XCDs, so give
    // each XCD a contiguous range of cells (its L2 then holds the
    // neighbourhood of its cells)
    const int b = blockIdx.x;
    const int cell = (b % NXCD) * p.per_xcd + b / NXCD;
    if (cell >= p.ncell) return;

    const int info = p.cinfo[cell];
    const int ifca = ci_ifca(info), admis = ci_admis(info), full = ci_full(info);
    const int ts = p.ts;
    const double *Ui = p.U + (size_t)cell * NV;
    double ui[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) ui[v] = Ui[v];
    if (lane < NV) sh.ui[lane] = ui[lane];

    // ---- phase 0: dU of every stencil member (FP64, then rounded to R) ----
    const int32_t *nb = p.nbr + (size_t)cell * ts * IMAX;
    for (int e = lane; e < admis * IMAX; e += WAVE) {
        const double *Un = p.U + (size_t)nb[e] * NV;
#pragma unroll
        for (int v = 0; v < NV; ++v) sh.u.du[e * NV + v] = (R)(Un[v] - ui[v]);
    }
    {
        const R *Bc = p.B + (size_t)cell * (IDEG * (IDEG + 1) / 2);
        for (int e = lane; e < IDEG * (IDEG + 1) / 2; e += WAVE) {
            // packed upper triangle by rows: row k holds l = k..IDEG-1
            int k = 0, base = 0;
            while (e >= base + (IDEG - k)) {
                base += IDEG - k;
                ++k;
            }
            int l = k + (e - base);
            R val = Bc[e];
            sh.b[k * IDEG + l] = val;
            sh.b[l * IDEG + k] = val;
        }
    }
    for (int e = lane; e < IDEG; e += WAVE) sh.mb[e] = p.mbar[(size_t)cell * IDEG + e];
    __syncthreads();

    // ---- phase 1: G_s = P_s dU_s, one (stencil,coefficient) row per lane ----
    R acc[NROW][NV];
    int srow[NROW];
#pragma unroll
    for (int t = 0; t < NROW; ++t) {
        srow[t] = (lane + t * WAVE) / IDEG;
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[t][v] = R(0);
    }
    const int nrows = admis * IDEG;
    const R *Pc = p.P + (size_t)cell * IMAX * ts * IDEG;
#pragma unroll 4
    for (int j = 0; j < IMAX; ++j) {
        const R *Pj = Pc + (size_t)j * ts * IDEG;
#pragma unroll
        for (int t = 0; t < NROW; ++t) {
            const int r = lane + t * WAVE;
            if (r < nrows) {
                const R pv = Pj[r];
                const R *du = &sh.u.du[(srow[t] * IMAX + j) * NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) acc[t][v] += pv * du[v];
            }
        }
    }
#pragma unroll
    for (int t = 0; t < NROW; ++t) {
        const int r = lane + t * WAVE;
        if (r < nrows) {
#pragma unroll
            for (int v = 0; v < NV; ++v) sh.g[r * NV + v] = acc[t][v];
        }
    }
    __syncthreads();

    bool reduce = (full == 0);
    const int nslot = ifca * p.nqm;
    if constexpr (CH) {
        // ---- characteristic WENO: per face, the eigenvectors of the averaged
        // cell / neighbour state in the face frame (WENO_NEIGHBOUR: the ghost of
        // the cell's own average on boundary faces), every stencil's
        // coefficients projected with L, indicators and weights per
        // characteristic variable, the weighted coefficients projected back
        // with R, and that face's values (compute_gradcharv_smoothindicator,
        // diag_At_B_A, src/reconstruct_p.f90:1608-1818) ----
        __shared__ double chR[25], chL[25];
        __shared__ double cbeta[TSMAX * NV];
        __shared__ R wch[TSMAX * IDEG * NV];
        double wi[NV];
        cons2prim_d(p.gamma, ui, wi);
        int trouble = 0;
        const R *qpc = p.qp + (size_t)cell * p.nf * p.nqm * 3;
        for (int f = 0; f < ifca; ++f) {
            if (lane == 0) {
                const int nbf = p.chnb[(size_t)cell * p.nf + f];
                const double *an = p.chang + ((size_t)cell * p.nf + f) * 4;
                double ur[NV], rl[NV], rr[NV];
                if (nbf < 0) {
                    const double *bf = p.bface ? p.bface + (size_t)(p.cface[(size_t)cell * p.nf + f] - 1) * 10 : nullptr;
                    ghost_state(-nbf, p.bc.boundtype, p.gamma, ui, an[0], an[1], an[2], an[3],
                                bf ? bf : p.bc.inflow, bf ? bf + 5 : p.bc.outflow, ur);
                }
                else
#pragma unroll
                    for (int v = 0; v < NV; ++v) ur[v] = p.U[(size_t)nbf * NV + v];
                rotf(ui, an[0], an[1], an[2], an[3], rl);
                rotf(ur, an[0], an[1], an[2], an[3], rr);
                char_eigen_d(p.gamma, rl, rr, chR, chL);
            }
            __syncthreads();
            for (int e = lane; e < admis * IDEG * NV; e += WAVE) {
                const int c = e % NV, sk = e / NV;
                double acc = 0.0;
#pragma unroll
                for (int v = 0; v < NV; ++v) acc += (double)sh.g[sk * NV + v] * chL[c * 5 + v];
                wch[e] = (R)acc;
            }
            __syncthreads();
            if (lane < admis * NV) {
                const int s = lane / NV, c = lane % NV;
                const R *ws = &wch[s * IDEG * NV + c];
                double beta = 0.0;
                for (int a = 0; a < IDEG; ++a) {
                    double ba = 0.0;
                    for (int b2 = 0; b2 < IDEG; ++b2) ba += (double)sh.b[a * IDEG + b2] * (double)ws[b2 * NV];
                    beta += (double)ws[a * NV] * ba;
                }
                cbeta[lane] = beta;
            }
            __syncthreads();
            if (lane < admis * NV) {
                // lambda/(eps+beta)^4 per characteristic variable, in FP64 in both precisions
                const int s = lane / NV, c = lane % NV;
                double sum = 0.0, mine = 0.0;
                for (int t = 0; t < admis; ++t) {
                    const double x = p.eps + cbeta[t * NV + c];
                    const double x2 = x * x;
                    const double w = (t == 0 ? p.lwci1 : 1.0) / (x2 * x2);
                    sum += w;
                    if (t == s) mine = w;
                }
                sh.u.late.omega[lane] = (R)(mine / sum);
            }
            __syncthreads();
            for (int e = lane; e < IDEG * NV; e += WAVE) {
                const int k = e / NV, v = e % NV;
                double acc = 0.0;
#pragma unroll
                for (int c = 0; c < NV; ++c) {
                    double lim = 0.0;
                    for (int s = 0; s < admis; ++s)
                        lim += (double)wch[(s * IDEG + k) * NV + c] * (double)sh.u.late.omega[s * NV + c];
                    acc += chR[v * 5 + c] * lim;
                }
                sh.u.late.gh[e] = (R)acc;
            }
            __syncthreads();
            const int nq = ci_tri(info, f) ? p.qpt : p.qpq;
#pragma unroll 1
            for (int q = lane; q < nq; q += WAVE) {
                asm volatile("" ::: "memory");
                const int e = f * p.nqm + q;
                R x[3] = {qpc[e * 3], qpc[e * 3 + 1], qpc[e * 3 + 2]};
                R phi[IDEG];
                basis_at<R, IDEG>(x, sh.mb, phi);
                double uq[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    R res = R(0);
                    for (int k = 0; k < IDEG; ++k) res += phi[k] * sh.u.late.gh[k * NV + v];
                    uq[v] = ui[v] + (double)res;
                    sh.u.late.ul[e * NV + v] = res;
                }
                if (full && jump_test(p.gamma, wi, uq, 0.85)) trouble = 1;
            }
            __syncthreads();
        }
        reduce = reduce || (__syncthreads_or(trouble) != 0);
    } else {
        // ---- phase 2: beta_{s,v} = g^T (B g) (src/reconstruct_p.f90:995-1004) ----
        if (lane < admis * NV) {
            const int s = lane / NV, v = lane % NV;
            const R *gs = &sh.g[s * IDEG * NV + v];
            R beta = R(0);
            for (int k = 0; k < IDEG; ++k) {
                R bg = R(0);
#pragma unroll
                for (int l = 0; l < IDEG; ++l) bg += sh.b[k * IDEG + l] * gs[l * NV];
                beta += gs[k * NV] * bg;
            }
            sh.u.late.beta[lane] = beta;
        }
        __syncthreads();
        // ---- phase 3: weights (src/reconstruct_p.f90:1031-1049) ----
        if (lane < admis * NV) {
            const int s = lane / NV, v = lane % NV;
            const R eps = (R)p.eps;
            R om;
            if (sizeof(R) == 8) {
                // lambda/(eps+beta)^4 as in the reference
                R sum = R(0), mine = R(0);
                for (int t = 0; t < admis; ++t) {
                    R x = eps + sh.u.late.beta[t * NV + v];
                    R x2 = x * x;
                    R w = (t == 0 ? (R)p.lwci1 : R(1)) / (x2 * x2);
                    sum += w;
                    if (t == s) mine = w;
                }
                om = mine / sum;
            } else {
                // FP32: (eps+beta)^-4 underflows, so scale every weight by
                // (eps+beta_min)^4 first; the normalised weights are unchanged
                R xmin = eps + sh.u.late.beta[v];
                for (int t = 1; t < admis; ++t) xmin = fminf(xmin, eps + sh.u.late.beta[t * NV + v]);
                R sum = R(0), mine = R(0);
                for (int t = 0; t < admis; ++t) {
                    R r = xmin / (eps + sh.u.late.beta[t * NV + v]);
                    R r2 = r * r;
                    R w = (t == 0 ? (R)p.lwci1 : R(1)) * (r2 * r2);
                    sum += w;
                    if (t == s) mine = w;
                }
                om = mine / sum;
            }
            sh.u.late.omega[lane] = om;
        }
        __syncthreads();
        // ---- phase 4: combined coefficients sum_s omega_s G_s ----
        for (int e = lane; e < IDEG * NV; e += WAVE) {
            const int v = e % NV;
            R acc = R(0);
            for (int s = 0; s < admis; ++s) acc += sh.u.late.omega[s * NV + v] * sh.g[s * IDEG * NV + e];
            sh.u.late.gh[e] = acc;
        }
        __syncthreads();
        // ---- phase 5: ULEFT at the face points + CHECKSOL (0.85) ----
        double wi[NV];
        cons2prim_d(p.gamma, ui, wi);
        int trouble = 0;
        const R *qpc = p.qp + (size_t)cell * p.nf * p.nqm * 3;
#pragma unroll 1
        for (int e = lane; e < nslot; e += WAVE) {
            // keep the coefficient loads inside the point loop (hoisted, they
            // would hold IDEG x 5 values in registers across it)
            asm volatile("" ::: "memory");
            const int f = e / p.nqm, q = e % p.nqm;
            const int nq = ci_tri(info, f) ? p.qpt : p.qpq;
            if (q >= nq) continue;
            R x[3] = {qpc[e * 3], qpc[e * 3 + 1], qpc[e * 3 + 2]};
            R phi[IDEG];
            basis_at<R, IDEG>(x, sh.mb, phi);
            double uq[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                R res = R(0);
#pragma unroll
                for (int k = 0; k < IDEG; ++k) res += phi[k] * sh.u.late.gh[k * NV + v];
                // ULEFT is kept as the deviation from the FP64 cell average
                uq[v] = ui[v] + (double)res;
                sh.u.late.ul[e * NV + v] = res;
            }
            if (full && jump_test(p.gamma, wi, uq, 0.85)) trouble = 1;
        }
        reduce = reduce || (__syncthreads_or(trouble) != 0);
    }
    // ---- phase 6: MUSCL + Barth-Jespersen (src/reconstruct_p.f90:2044-2280) ----
    if (reduce) {
        double umin[NV], umax[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) umin[v] = umax[v] = ui[v];
        for (int f = 0; f < ifca; ++f) {
            const int n = p.cnb[(size_t)cell * p.nf + f];
            if (n < 0) continue;
            const double *Un = p.U + (size_t)n * NV;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                umin[v] = fmin(umin[v], Un[v]);
                umax[v] = fmax(umax[v], Un[v]);
            }
        }
        const R *qpc = p.qp + (size_t)cell * p.nf * p.nqm * 3;
        double slope[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) slope[v] = 1.0e16;
#pragma unroll 1
        for (int e = lane; e < nslot; e += WAVE) {
            // keep the coefficient loads inside the point loop (hoisted, they
            // would hold IDEG x 5 values in registers across it)
            asm volatile("" ::: "memory");
            const int f = e / p.nqm, q = e % p.nqm;
            const int nq = ci_tri(info, f) ? p.qpt : p.qpq;
            if (q >= nq) continue;
            R x[3] = {qpc[e * 3], qpc[e * 3 + 1], qpc[e * 3 + 2]};
            R phi[IDEG];
            basis_at<R, IDEG>(x, sh.mb, phi);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                R res = R(0);
#pragma unroll
                for (int k = 0; k < IDEG; ++k) res += phi[k] * sh.g[k * NV + v];
                const double d2 = (double)res;
                double psi;
                if (fabs(d2) <= 0.0)
                    psi = 1.0;
                else if (d2 > 0.0)
                    psi = fmin(1.0, (umax[v] - ui[v]) / d2);
                else
                    psi = fmin(1.0, (umin[v] - ui[v]) / d2);
                slope[v] = fmin(slope[v], psi);
            }
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) slope[v] = wave_min(slope[v]);
#pragma unroll 1
        for (int e = lane; e < nslot; e += WAVE) {
            // keep the coefficient loads inside the point loop (hoisted, they
            // would hold IDEG x 5 values in registers across it)
            asm volatile("" ::: "memory");
            const int f = e / p.nqm, q = e % p.nqm;
            const int nq = ci_tri(info, f) ? p.qpt : p.qpq;
            if (q >= nq) continue;
            R x[3] = {qpc[e * 3], qpc[e * 3 + 1], qpc[e * 3 + 2]};
            R phi[IDEG];
            basis_at<R, IDEG>(x, sh.mb, phi);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                R res = R(0);
#pragma unroll
                for (int k = 0; k < IDEG; ++k) res += phi[k] * sh.g[k * NV + v];
                sh.u.late.ul[e * NV + v] = (R)((double)res * slope[v]);
            }
        }
        __syncthreads();
    }

    bool first = false;
    // ---- phase 7: CHECKSOLX (0.95) -> first order (src/reconstruct_p.f90:3245-3406) ----
    {
        double wi[NV];
        cons2prim_d(p.gamma, ui, wi);
        int trouble = 0;
#pragma unroll 1
        for (int e = lane; e < nslot; e += WAVE) {
            // keep the coefficient loads inside the point loop (hoisted, they
            // would hold IDEG x 5 values in registers across it)
            asm volatile("" ::: "memory");
            const int f = e / p.nqm, q = e % p.nqm;
            const int nq = ci_tri(info, f) ? p.qpt : p.qpq;
            if (q >= nq) continue;
            double uq[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) uq[v] = ui[v] + (double)sh.u.late.ul[e * NV + v];
            if (jump_test(p.gamma, wi, uq, 0.95)) trouble = 1;
        }
        first = __syncthreads_or(trouble) != 0;
        if (first) {
            for (int e = lane; e < nslot; e += WAVE)
#pragma unroll
                for (int v = 0; v < NV; ++v) sh.u.late.ul[e * NV + v] = R(0);
            __syncthreads();
        }
    }

    // a plain store per cell: the counts' atomicAdd on one address took 12 ns
    // each, all of a small MUSCL mesh's time (24^3 cells, 10 RK3 steps: 5.60
    // ms with it, 1.40 ms without)
    if (lane == 0) p.marks[cell] = (reduce ? 1 : 0) + (first ? 65536 : 0);

    // ---- phase 8: ULEFT out, one contiguous block per cell ----
    R *out = p.uleft + (size_t)cell * p.nf * p.nqm * NV;
    for (int e = lane; e < nslot * NV; e += WAVE) out[e] = sh.u.late.ul[e];
}

// upload: pseudo-inverses of cells cell0 .. cell0+cn-1 ([cell][tsa][imax][ideg]
// FP64, the ABI order) into the row stream
template <typename R>
__global__ void k_stream_p(const double *src, unsigned char *stream, int cell0, int cn, int tsa, int ts, int imax,
                           int ideg, int hd, int rd, long long tile_bytes) {
    const size_t n = (size_t)cn * ts * imax * ideg;
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
        const int k = (int)(e % ideg);
        const int j = (int)((e / ideg) % imax);
        const int st = (int)((e / ((size_t)ideg * imax)) % ts);
        const int cl = (int)(e / ((size_t)ideg * imax * ts));
        const int i = cell0 + cl;
        const double v = src[(((size_t)cl * tsa + st) * imax + j) * ideg + k];
        R *row = (R *)(stream + (size_t)(i / 8) * tile_bytes + hd + (size_t)j * rd);
        row[(size_t)k * 8 * ts + (i % 8) * ts + st] = (R)v;
    }
}

// upload: member-index rows [ntile][depth+imax][8 ts] (row r = members j=r,
// zero past imax) into the header (r < depth) and behind the pseudo-inverse
// block of row r - depth
__global__ void k_stream_idx(const int32_t *idx, unsigned char *stream, int ntile, int depth, int imax, int tp, int hd,
                             int pb, int rd, long long tile_bytes) {
    const size_t n = (size_t)ntile * (depth + imax) * tp;
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
        const int q = (int)(e % tp);
        const int r = (int)((e / tp) % (depth + imax));
        const size_t t = e / ((size_t)tp * (depth + imax));
        unsigned char *base = stream + t * tile_bytes;
        int32_t *dst = r < depth ? (int32_t *)(base + (size_t)r * tp * 4) + q
                                 : (int32_t *)(base + hd + (size_t)(r - depth) * rd + pb) + q;
        *dst = idx[e];
    }
}

template <typename R>
__global__ void k_tile_p(const double *src, R *dst, int cell0, int ncells_chunk, int ncell, int ts_in, int ts,
                         int imax, int ideg) {
    // dst covers the tiles of cells [cell0, cell0+ncells_chunk), cell0 % 8 == 0
    const int TP = 8 * ts;
    const size_t per_tile = (size_t)imax * ideg * TP;
    const size_t ntile = ((size_t)ncells_chunk + 7) / 8;
    const size_t total = per_tile * ntile;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
        const size_t t = e / per_tile;
        size_t r = e % per_tile;
        const int pos = (int)(r % TP);
        r /= TP;
        const int k = (int)(r % ideg);
        const int j = (int)(r / ideg);
        const int lc = pos / ts, s = pos % ts;
        const size_t cl = t * 8 + lc;  // cell within the chunk
        R val = R(0);
        if (cl < (size_t)ncells_chunk && cell0 + cl < (size_t)ncell && s < ts_in)
            val = (R)src[((cl * ts_in + s) * imax + j) * ideg + k];
        dst[e] = val;
    }
}

// ---------------------------------------------------------------------------
// HLLC (src/riemann.f90:221-426) on rotated FP64 states.  Primitive recovery
// is FP64.  R=double keeps the reference's arithmetic.  R=float evaluates the
// wave speeds and the star-state correction in FP32 and each side's
// physical flux F_K in FP64:
//   F = F_K + S_K (U*_K - U_K),  K = L if S_M >= 0 else R,
// with U*_K - U_K in its factored form, every component carrying
// (S_M - u_K) / (S_K - S_M):
//   mass rho d, normal momentum rho S_K d, tangential rho v_t d,
//   energy E d + rho chi (S_M - u_K)(S_M + p/(rho (S_K - u_K))),
//   d = (S_M - u_K)/(S_K - S_M), chi = (S_K - u_K)/(S_K - S_M),
// so the FP32 rounding scales with the jump across the face and not with
// the size of the state (the pressure, the energy) as it would if U* and
// U_K were rounded separately and subtracted.
template <class T>
__device__ inline void hllc_t(double gamma, const T *cl, const T *cr, T *flux) {
    T wl[NV], wr[NV];
    cons2prim_t(gamma, cl, wl);
    cons2prim_t(gamma, cr, wr);
    const T rl = wl[0], uL = wl[1], vl = wl[2], zl = wl[3], pl = wl[4], el = cl[4];
    const T rr = wr[0], uR = wr[1], vr = wr[2], zr = wr[3], pr = wr[4], er = cr[4];
    const T ccl = sqrt(gamma * pl / rl), ccr = sqrt(gamma * pr / rr);
    const T srl = sqrt(rl), srr = sqrt(rr);
    const T cc2 = sqrt((((ccl * ccl) * srl) + ((ccr * ccr) * srr)) / (srl + srr) +
                       (0.5 * ((srl * srr) / ((srl + srr) * (srl + srr))) * ((uR - uL) * (uR - uL))));
    const T uu2 = ((uL * srl) + (uR * srr)) / (srl + srr);
    T sl = fmin(uL - ccl, uu2 - cc2), sr = fmax(uR + ccr, uu2 + cc2);
    sl = fmin(sl, 0.0);
    sr = fmax(sr, 0.0);
    const T sm = (pr - pl + (rl * uL * (sl - uL)) - (rr * uR * (sr - uR))) / ((rl * (sl - uL)) - (rr * (sr - uR)));
    const T fl[NV] = {rl * uL, (rl * (uL * uL)) + pl, rl * uL * vl, rl * uL * zl, uL * (el + pl)};
    const T fr[NV] = {rr * uR, (rr * (uR * uR)) + pr, rr * uR * vr, rr * uR * zr, uR * (er + pr)};
    const T mul = rl * ((sl - uL) / (sl - sm));
    const T mur = rr * ((sr - uR) / (sr - sm));
    const T lastl = (el / rl) + ((sm - uL) * (sm + ((pl) / (rl * (sl - uL)))));
    const T lastr = (er / rr) + ((sm - uR) * (sm + ((pr) / (rr * (sr - uR)))));
    const T usl[NV] = {mul, mul * sm, mul * vl, mul * zl, mul * lastl};
    const T usr[NV] = {mur, mur * sm, mur * vr, mur * zr, mur * lastr};
    const double s = copysign(1.0, val(sm));
#pragma unroll
    for (int k = 0; k < NV; ++k)
        flux[k] = (((1.0 + s) / 2.0) * (fl[k] + sl * (usl[k] - cl[k]))) +
                  (((1.0 - s) / 2.0) * (fr[k] + sr * (usr[k] - cr[k])));
}
// The FP64 solver of the flux kernels: hllc_t, term by term, with only the side
// that sign(S_M) picks evaluated (the other is multiplied by 0 there).  The
// kernels spend most of their vector time in FP64 divisions and square roots:
// 11 and 5 of them here, 14 and 5 in hllc_t.
// The other side's terms vanish unless they are not finite: where its wave speed
// is S_M (a division by S - S_M: every component) or its own normal velocity (by
// S - u: the energy), which a state without a sound speed (p <= 0) can bring
// about, hllc_t's 0 times infinity makes the flux NaN.  It does here too, so that
// such a state still ends a march as non-finite.
__device__ inline void hllc64(double gamma, const double *cl, const double *cr, double *flux) {
    double wl[NV], wr[NV];
    cons2prim_d(gamma, cl, wl);
    cons2prim_d(gamma, cr, wr);
    const double rl = wl[0], uL = wl[1], pl = wl[4], rr = wr[0], uR = wr[1], pr = wr[4];
    const double ccl = sqrt(gamma * pl / rl), ccr = sqrt(gamma * pr / rr);
    const double srl = sqrt(rl), srr = sqrt(rr);
    const double cc2 = sqrt((((ccl * ccl) * srl) + ((ccr * ccr) * srr)) / (srl + srr) +
                            (0.5 * ((srl * srr) / ((srl + srr) * (srl + srr))) * ((uR - uL) * (uR - uL))));
    const double uu2 = ((uL * srl) + (uR * srr)) / (srl + srr);
    const double sl = fmin(fmin(uL - ccl, uu2 - cc2), 0.0), sr = fmax(fmax(uR + ccr, uu2 + cc2), 0.0);
    const double sm = (pr - pl + (rl * uL * (sl - uL)) - (rr * uR * (sr - uR))) / ((rl * (sl - uL)) - (rr * (sr - uR)));
    const bool left = copysign(1.0, sm) > 0.0;
    double ck[NV], wk[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        ck[v] = left ? cl[v] : cr[v];
        wk[v] = left ? wl[v] : wr[v];
    }
    const double sk = left ? sl : sr, rk = wk[0], uk = wk[1], pk = wk[4], ek = ck[4];
    const double fk[NV] = {rk * uk, (rk * (uk * uk)) + pk, rk * uk * wk[2], rk * uk * wk[3], uk * (ek + pk)};
    const double mu = rk * ((sk - uk) / (sk - sm));
    const double last = (ek / rk) + ((sm - uk) * (sm + ((pk) / (rk * (sk - uk)))));
    const double us[NV] = {mu, mu * sm, mu * wk[2], mu * wk[3], mu * last};
#pragma unroll
    for (int k = 0; k < NV; ++k) flux[k] = fk[k] + sk * (us[k] - ck[k]);
    const double so = left ? sr : sl, uo = left ? uR : uL;
    if (so == sm || so == uo) {
        flux[4] = (double)NAN;
#pragma unroll
        for (int k = 0; k < NV - 1; ++k) flux[k] = so == sm ? (double)NAN : flux[k];
    }
}

// Reverse mode of hllc_t (FP64): given the flux cotangent hb, the cotangents
// of both rotated states.  The forward values repeat hllc_t; the branches
// (Einfeldt min/max, the clamps of S_L/S_R at 0, the side sign(S_M) picks)
// are taken as hllc_t takes them, ties included, so this is the transpose
// of the derivative the Dual passes of hllc_t compute.
__device__ inline void hllc_vjp(double g, const double *cl, const double *cr, const double *hb, double *clb,
                                double *crb) {
    const double gm = g - 1.0;
    // ---- forward ----
    const double rl = cl[0], ool = 1.0 / rl, uL = cl[1] * ool, vl = cl[2] * ool, zl = cl[3] * ool, el = cl[4];
    const double rr = cr[0], oor = 1.0 / rr, uR = cr[1] * oor, vr = cr[2] * oor, zr = cr[3] * oor, er = cr[4];
    const double ql = uL * uL + vl * vl + zl * zl, qr = uR * uR + vr * vr + zr * zr;
    const double pl = gm * (el - 0.5 * rl * ql), pr = gm * (er - 0.5 * rr * qr);
    const double ccl = sqrt(g * pl / rl), ccr = sqrt(g * pr / rr);
    const double srl = sqrt(rl), srr = sqrt(rr), S = srl + srr;
    const double du = uR - uL;
    const double T1 = ((ccl * ccl) * srl + (ccr * ccr) * srr) / S;
    const double cc2 = sqrt(T1 + (0.5 * ((srl * srr) / (S * S)) * (du * du)));
    const double uu2 = ((uL * srl) + (uR * srr)) / S;
    const double a1 = uL - ccl, a2 = uu2 - cc2, b1 = uR + ccr, b2 = uu2 + cc2;
    const bool selL = a2 < a1, selR = b2 > b1;  // the second argument wins
    double sl = selL ? a2 : a1, sr = selR ? b2 : b1;
    const bool clL = 0.0 < sl, clR = 0.0 > sr;  // clamped to 0
    if (clL) sl = 0.0;
    if (clR) sr = 0.0;
    const double num = pr - pl + (rl * uL * (sl - uL)) - (rr * uR * (sr - uR));
    const double den = (rl * (sl - uL)) - (rr * (sr - uR));
    const double sm = num / den;
    const bool left = copysign(1.0, sm) > 0.0;
    // ---- reverse through the chosen side K: F = F_K + S_K (U*_K - U_K) ----
    const double rK = left ? rl : rr, uK = left ? uL : uR, vK = left ? vl : vr, zK = left ? zl : zr;
    const double pK = left ? pl : pr, eK = left ? el : er, sK = left ? sl : sr;
    const double *cK = left ? cl : cr;
    const double dK = sK - uK, Q = sK - sm, mu = rK * (dK / Q);
    const double D = rK * dK, A = sm - uK, Bq = sm + pK / D;
    const double lastK = (eK / rK) + A * Bq;
    const double us[NV] = {mu, mu * sm, mu * vK, mu * zK, mu * lastK};
    double sKb = 0.0;
#pragma unroll
    for (int k = 0; k < NV; ++k) sKb += hb[k] * (us[k] - cK[k]);
    double usb[NV], cKb[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        usb[k] = sK * hb[k];
        cKb[k] = -sK * hb[k];
    }
    const double mub = usb[0] + usb[1] * sm + usb[2] * vK + usb[3] * zK + usb[4] * lastK;
    double smb = usb[1] * mu;
    double vKb = usb[2] * mu, zKb = usb[3] * mu;
    const double lastb = usb[4] * mu;
    double eKb = lastb / rK, rKb = -lastb * eK / (rK * rK);
    const double Ab = lastb * Bq, Bqb = lastb * A;
    smb += Ab + Bqb;
    double uKb = -Ab;
    double pKb = Bqb / D;
    const double Db = -Bqb * pK / (D * D);
    rKb += Db * dK;
    double dKb = Db * rK;
    rKb += mub * dK / Q;
    dKb += mub * rK / Q;
    const double Qb = -mub * mu / Q;
    sKb += Qb;
    smb -= Qb;
    sKb += dKb;
    uKb -= dKb;
    // F_K = [rK uK, rK uK^2 + pK, rK uK vK, rK uK zK, uK (eK + pK)]
    rKb += hb[0] * uK + hb[1] * uK * uK + hb[2] * uK * vK + hb[3] * uK * zK;
    uKb += hb[0] * rK + hb[1] * 2.0 * rK * uK + hb[2] * rK * vK + hb[3] * rK * zK + hb[4] * (eK + pK);
    pKb += hb[1] + hb[4] * uK;
    vKb += hb[2] * rK * uK;
    zKb += hb[3] * rK * uK;
    eKb += hb[4] * uK;
    // primitive cotangents of both sides
    double rlb = 0, ulb = 0, vlb = 0, zlb = 0, plb = 0, elb = 0, slb = 0;
    double rrb = 0, urb = 0, vrb = 0, zrb = 0, prb = 0, erb = 0, srb = 0;
    if (left) {
        rlb = rKb; ulb = uKb; vlb = vKb; zlb = zKb; plb = pKb; elb = eKb; slb = sKb;
    } else {
        rrb = rKb; urb = uKb; vrb = vKb; zrb = zKb; prb = pKb; erb = eKb; srb = sKb;
    }
    // S_M = num / den
    const double numb = smb / den, denb = -smb * sm / den;
    prb += numb;
    plb -= numb;
    rlb += numb * uL * (sl - uL);
    ulb += numb * rl * (sl - 2.0 * uL);
    slb += numb * rl * uL;
    rrb -= numb * uR * (sr - uR);
    urb -= numb * rr * (sr - 2.0 * uR);
    srb -= numb * rr * uR;
    rlb += denb * (sl - uL);
    slb += denb * rl;
    ulb -= denb * rl;
    rrb -= denb * (sr - uR);
    srb -= denb * rr;
    urb += denb * rr;
    // S_L, S_R: clamps and Einfeldt min / max
    double cclb = 0, ccrb = 0, cc2b = 0, uu2b = 0;
    if (!clL) {
        if (selL) {
            uu2b += slb;
            cc2b -= slb;
        } else {
            ulb += slb;
            cclb -= slb;
        }
    }
    if (!clR) {
        if (selR) {
            uu2b += srb;
            cc2b += srb;
        } else {
            urb += srb;
            ccrb += srb;
        }
    }
    ulb += uu2b * srl / S;
    urb += uu2b * srr / S;
    double srlb = uu2b * (uL - uu2) / S, srrb = uu2b * (uR - uu2) / S;
    const double Xb = cc2b / (2.0 * cc2);
    cclb += Xb * 2.0 * ccl * srl / S;
    ccrb += Xb * 2.0 * ccr * srr / S;
    srlb += Xb * (ccl * ccl - T1) / S;
    srrb += Xb * (ccr * ccr - T1) / S;
    const double S3 = S * S * S, hdu2 = 0.5 * du * du;
    srlb += Xb * hdu2 * srr * (srr - srl) / S3;
    srrb += Xb * hdu2 * srl * (srl - srr) / S3;
    const double dub = Xb * ((srl * srr) / (S * S)) * du;
    urb += dub;
    ulb -= dub;
    rlb += srlb / (2.0 * srl);
    rrb += srrb / (2.0 * srr);
    const double ylb = cclb / (2.0 * ccl), yrb = ccrb / (2.0 * ccr);
    plb += ylb * g / rl;
    rlb -= ylb * g * pl / (rl * rl);
    prb += yrb * g / rr;
    rrb -= yrb * g * pr / (rr * rr);
    // conserved -> primitive: rho = c0, u = c1/c0 ..., p = (g-1)(c4 - c0 q/2)
    auto back = [&](const double *c, double r_b, double u_b, double v_b, double z_b, double p_b, double e_b,
                    double u, double v, double z, double q, double *cb) {
        const double qb = -gm * 0.5 * c[0] * p_b;
        const double ub = u_b + 2.0 * u * qb, vb = v_b + 2.0 * v * qb, zb = z_b + 2.0 * z * qb;
        const double oo = 1.0 / c[0];
        cb[0] += r_b - gm * 0.5 * q * p_b - (ub * u + vb * v + zb * z) * oo;
        cb[1] += ub * oo;
        cb[2] += vb * oo;
        cb[3] += zb * oo;
        cb[4] += gm * p_b + e_b;
    };
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        clb[k] = left ? cKb[k] : 0.0;
        crb[k] = left ? 0.0 : cKb[k];
    }
    back(cl, rlb, ulb, vlb, zlb, plb, elb, uL, vl, zl, ql, clb);
    back(cr, rrb, urb, vrb, zrb, prb, erb, uR, vr, zr, qr, crb);
}

__device__ inline void hllc32(double gamma, const double *cl, const double *cr, double *flux) {
    double wl[NV], wr[NV];
    cons2prim_d(gamma, cl, wl);
    cons2prim_d(gamma, cr, wr);
    const float g = (float)gamma;
    const float rl = (float)wl[0], uL = (float)wl[1], pl = (float)wl[4];
    const float rr = (float)wr[0], uR = (float)wr[1], pr = (float)wr[4];
    const float ccl = sqrtf(g * pl / rl), ccr = sqrtf(g * pr / rr);
    const float srl = sqrtf(rl), srr = sqrtf(rr);
    const float cc2 = sqrtf((((ccl * ccl) * srl) + ((ccr * ccr) * srr)) / (srl + srr) +
                            (0.5f * ((srl * srr) / ((srl + srr) * (srl + srr))) * ((uR - uL) * (uR - uL))));
    const float uu2 = ((uL * srl) + (uR * srr)) / (srl + srr);
    float sl = fminf(uL - ccl, uu2 - cc2), sr = fmaxf(uR + ccr, uu2 + cc2);
    sl = fminf(sl, 0.0f);
    sr = fmaxf(sr, 0.0f);
    const float dp = (float)(wr[4] - wl[4]);
    const float sm = (dp + (rl * uL * (sl - uL)) - (rr * uR * (sr - uR))) / ((rl * (sl - uL)) - (rr * (sr - uR)));
    const bool left = !(copysignf(1.0f, sm) < 0.0f);
    const double *w = left ? wl : wr;
    const double *c = left ? cl : cr;
    const float sk = left ? sl : sr;
    const float rk = (float)w[0], uk = (float)w[1], pk = (float)w[4];
    // physical flux of the upwind side, FP64
    const double fk[NV] = {w[0] * w[1], (w[0] * (w[1] * w[1])) + w[4], w[0] * w[1] * w[2], w[0] * w[1] * w[3],
                           w[1] * (c[4] + w[4])};
    // star-state correction, FP32, factored
    const float den = sk - sm;
    const float d = (sm - uk) / den;
    const float chi = (sk - uk) / den;
    const float du[NV] = {rk * d, rk * sk * d, rk * (float)w[2] * d, rk * (float)w[3] * d,
                          (float)c[4] * d + rk * chi * (sm - uk) * (sm + pk / (rk * (sk - uk)))};
#pragma unroll
    for (int k = 0; k < NV; ++k) flux[k] = fk[k] + (double)(sk * du[k]);
}

template <typename R>
struct FluxParams {
    int nface, nf, nqm, qpq, qpt;
    double gamma;
    const int32_t *fcell;   // [nface][2] left (owner), right
    const int32_t *fslot;   // [nface][2] face slot in left, right; bit 8 of slot 0: triangle
    const double *frot;     // [nface][4] cos a1, sin a1, cos a2, sin a2 of the owner's outward normal
    const double *farea;    // [nface]
    const double *U;        // [ncell][5] cell averages
    const R *uleft;         // face-point deviations from the cell average
    double *fflux;          // [nface][5] outward from the owner
    const double *wq;       // [qpq] quadrilateral-face weights of this context, sum 1
    const double *wt;       // [qpt] triangular-face weights, sum 1
    ucns_boundary_v1 bc;    // free-stream data of the boundary codes
    const double *bface;    // [nface][10] per-face INFLOW(), OUTFLOW() states, or null: bc's
};

template <typename R>
__global__ __launch_bounds__(256) void k_flux(FluxParams<R> p) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= p.nface) return;
    const int cL = p.fcell[2 * f], cR = p.fcell[2 * f + 1];
    const int s0 = p.fslot[2 * f], sR = p.fslot[2 * f + 1];
    const int sL = s0 & 255;
    const bool tri = (s0 >> 8) & 1;
    const int nq = tri ? p.qpt : p.qpq;
    const double *w = tri ? p.wt : p.wq;
    const double c1 = p.frot[4 * f], s1 = p.frot[4 * f + 1], c2 = p.frot[4 * f + 2], s2 = p.frot[4 * f + 3];
    const double area = p.farea[f];
    const bool bnd = cR < 0;  // boundary face: -code
    const double *fin = p.bface ? p.bface + (size_t)f * 10 : p.bc.inflow;
    const double *fout = p.bface ? p.bface + (size_t)f * 10 + 5 : p.bc.outflow;
    double uL[NV], uR[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        uL[v] = p.U[(size_t)cL * NV + v];
        uR[v] = bnd ? 0.0 : p.U[(size_t)cR * NV + v];
    }
    const R *ulL = p.uleft + ((size_t)cL * p.nf + sL) * p.nqm * NV;
    const R *ulR = p.uleft + ((size_t)(bnd ? cL : cR) * p.nf + (bnd ? sL : sR)) * p.nqm * NV;
    double acc[NV] = {0, 0, 0, 0, 0};
    // QB points' deviations are loaded before any is used (indices clamped
    // to the face's nq points; the surplus is not evaluated)
    constexpr int QB = 3;
    R dl[QB][NV], dr[QB][NV];
    for (int q = 0; q < nq; ++q) {
        const int qb = q % QB;
        if (qb == 0) {
#pragma unroll
            for (int u = 0; u < QB; ++u) {
                const int qq = min(q + u, nq - 1);
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    dl[u][v] = ulL[qq * NV + v];
                    dr[u][v] = ulR[qq * NV + v];
                }
            }
        }
        double a[NV], bq[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            R xl = dl[0][v], xr = dr[0][v];
#pragma unroll
            for (int u = 1; u < QB; ++u)
                if (qb == u) {
                    xl = dl[u][v];
                    xr = dr[u][v];
                }
            a[v] = uL[v] + (double)xl;
            bq[v] = uR[v] + (double)xr;
        }
        if (bnd) ghost_state(-cR, p.bc.boundtype, p.gamma, a, c1, s1, c2, s2, fin, fout, bq);  // GET_STATES_BOUNDS
        // ROTATEF (src/grid_t.f90:4217-4258)
        const double la[NV] = {a[0], c1 * s2 * a[1] + s1 * s2 * a[2] + c2 * a[3],
                               c1 * c2 * a[1] + s1 * c2 * a[2] + (-s2) * a[3], (-s1) * a[1] + c1 * a[2], a[4]};
        const double ra[NV] = {bq[0], c1 * s2 * bq[1] + s1 * s2 * bq[2] + c2 * bq[3],
                               c1 * c2 * bq[1] + s1 * c2 * bq[2] + (-s2) * bq[3], (-s1) * bq[1] + c1 * bq[2], bq[4]};
        double hd[NV];
        if (sizeof(R) == 8)
            hllc64(p.gamma, la, ra, hd);
        else
            hllc32(p.gamma, la, ra, hd);
        // ROTATEB (src/grid_t.f90:4261-4305)
        const double rb[NV] = {hd[0], c1 * s2 * hd[1] + c1 * c2 * hd[2] + (-s1) * hd[3],
                               s1 * s2 * hd[1] + s1 * c2 * hd[2] + c1 * hd[3], c2 * hd[1] + (-s2) * hd[2], hd[4]};
        const double wa = w[q] * area;
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] = acc[v] + (rb[v] * wa);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) p.fflux[(size_t)f * NV + v] = acc[v];
}

// The same with one thread per (face, quadrature point), for meshes whose
// faces have several points: nqm times
// the waves, and a point's chain of divisions and square roots runs beside the
// others' instead of after them.  The points' contributions meet in LDS, where
// thread (face, variable) adds them in point order (the order and rounding of
// the one-thread loop).  5,184 hexahedra faces of 9 points: 18.8 -> 6.2 us.
template <typename R>
__global__ __launch_bounds__(256) void k_flux_points(FluxParams<R> p) {
    __shared__ double sh[256][NV + 1];  // per point: the rotated-back flux and its weight times the area
    const int fpb = 256 / p.nqm;        // faces of a block (nqm <= 24: 6 nqm <= 96 points per cell, 4 faces at least)
    const int f0 = blockIdx.x * fpb;
    const int fl = threadIdx.x / p.nqm, q = threadIdx.x - fl * p.nqm;
    const int f = f0 + fl;
    auto point = [&]() {
        const int s0 = p.fslot[2 * f];
        const bool tri = (s0 >> 8) & 1;
        if (q >= (tri ? p.qpt : p.qpq)) return;
        const int cL = p.fcell[2 * f], cR = p.fcell[2 * f + 1];
        const int sL = s0 & 255, sR = p.fslot[2 * f + 1];
        const double *w = tri ? p.wt : p.wq;
        const double c1 = p.frot[4 * f], s1 = p.frot[4 * f + 1], c2 = p.frot[4 * f + 2], s2 = p.frot[4 * f + 3];
        const double area = p.farea[f];
        const bool bnd = cR < 0;  // boundary face: -code
        const size_t oL = (((size_t)cL * p.nf + sL) * p.nqm + q) * NV;
        const size_t oR = bnd ? oL : (((size_t)cR * p.nf + sR) * p.nqm + q) * NV;
        double a[NV], bq[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            a[v] = p.U[(size_t)cL * NV + v] + (double)p.uleft[oL + v];
            bq[v] = bnd ? 0.0 : p.U[(size_t)cR * NV + v] + (double)p.uleft[oR + v];
        }
        if (bnd) {
            const double *fin = p.bface ? p.bface + (size_t)f * 10 : p.bc.inflow;
            const double *fout = p.bface ? p.bface + (size_t)f * 10 + 5 : p.bc.outflow;
            ghost_state(-cR, p.bc.boundtype, p.gamma, a, c1, s1, c2, s2, fin, fout, bq);  // GET_STATES_BOUNDS
        }
        // ROTATEF (src/grid_t.f90:4217-4258)
        const double la[NV] = {a[0], c1 * s2 * a[1] + s1 * s2 * a[2] + c2 * a[3],
                               c1 * c2 * a[1] + s1 * c2 * a[2] + (-s2) * a[3], (-s1) * a[1] + c1 * a[2], a[4]};
        const double ra[NV] = {bq[0], c1 * s2 * bq[1] + s1 * s2 * bq[2] + c2 * bq[3],
                               c1 * c2 * bq[1] + s1 * c2 * bq[2] + (-s2) * bq[3], (-s1) * bq[1] + c1 * bq[2], bq[4]};
        double hd[NV];
        if (sizeof(R) == 8)
            hllc64(p.gamma, la, ra, hd);
        else
            hllc32(p.gamma, la, ra, hd);
        // ROTATEB (src/grid_t.f90:4261-4305)
        double *o = sh[threadIdx.x];
        o[0] = hd[0];
        o[1] = c1 * s2 * hd[1] + c1 * c2 * hd[2] + (-s1) * hd[3];
        o[2] = s1 * s2 * hd[1] + s1 * c2 * hd[2] + c1 * hd[3];
        o[3] = c2 * hd[1] + (-s2) * hd[2];
        o[4] = hd[4];
        o[NV] = w[q] * area;
    };
    if (fl < fpb && f < p.nface) point();
    __syncthreads();
    const int nfb = min(fpb, p.nface - f0);
    for (int e = threadIdx.x; e < nfb * NV; e += 256) {
        const int i = e / NV, v = e - i * NV;
        const int nq = (p.fslot[2 * (f0 + i)] >> 8) & 1 ? p.qpt : p.qpq;
        double acc = 0.0;
        for (int u = 0; u < nq; ++u) acc = acc + (sh[i * p.nqm + u][v] * sh[i * p.nqm + u][NV]);
        p.fflux[(size_t)f0 * NV + e] = acc;
    }
}

struct UpdateParams {
    int ncell, nf, stage;
    double cfl, gamma;
    const int32_t *cface;    // [ncell][nf] +(face+1) owner, -(face+1) neighbour, 0 none
    const double *fflux;
    const double *ovol;      // [ncell] 1/TOTVOLUME
    const double *minedge;
    double *U, *U2;          // U2: u^n; U: the state, updated in place (k_flux_update: the new state alone)
    double *rhs_out;         // optional [ncell][5]
    double *u64;             // optional: the new state as 64-byte records (k_pack64's), for the next reconstruction
    double *copy;            // optional: a copy of the new state, [ncell][5]
    const double *dt;        // this step's dt: one value, or (dt_slots) the slots it is the least of
    int dt_slots;
    unsigned long long *dt_next;  // the next step's slots: cleared to +inf in stage 2, atomic-min targets in stage 3
    double *t;               // advanced by dt in stage 3
};

__device__ inline void atomic_min_pos(unsigned long long *addr, double v) {
    atomicMin(addr, (unsigned long long)__double_as_longlong(v));
}

// A CFL step is the least of DT_SLOTS values on cache lines of their own:
// every block of 256 cells reduces its cells first and then lowers slot
// (block mod DT_SLOTS).  Atomics on one address retire one per 12 ns, so one
// per wave on a single value took 37 us of 196,608 cells' 38 us update (and
// of their k_dt); 16 slots keep a chain of at most 48 atomics there, and a
// reader still loads only 16 lines.
constexpr int DT_SLOTS = 16, DT_STRIDE = 16;  // 128-byte lines

__device__ inline double dt_of(const double *dt, bool slots) {
    if (!slots) return *dt;
    double v = dt[(threadIdx.x & (DT_SLOTS - 1)) * DT_STRIDE];
#pragma unroll
    for (int o = DT_SLOTS / 2; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, WAVE));
    return v;
}

// the block's (256 threads) least d into its slot; every thread takes part
__device__ inline void dt_lower(unsigned long long *slots, double d) {
    __shared__ double sh[256 / WAVE];
    d = wave_min(d);
    if ((threadIdx.x & (WAVE - 1)) == 0) sh[threadIdx.x / WAVE] = d;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 256 / WAVE; ++w) d = fmin(d, sh[w]);
        if (d < 1.0e300) atomic_min_pos(slots + (blockIdx.x & (DT_SLOTS - 1)) * DT_STRIDE, d);
    }
}

// stage 0: gather only (rhs_out); stage 1..3: Shu-Osher update
__global__ __launch_bounds__(256) void k_update(UpdateParams p) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double dtl = 1.0e300;
    const double dt = p.stage > 0 ? dt_of(p.dt, p.dt_slots) : 0.0;
    if (p.stage == 2 && p.dt_next && blockIdx.x == 0) p.dt_next[threadIdx.x] = 0x7FF0000000000000ULL;
    static_assert(DT_SLOTS * DT_STRIDE == 256, "one block of k_update clears the slots");
    if (i < p.ncell) {
        // every face's flux is loaded before the first is summed (face
        // slots past nf, and slots with no face, read face 0 and add nothing)
        constexpr int NFM = 6;
        int cf[NFM];
#pragma unroll
        for (int f = 0; f < NFM; ++f) cf[f] = f < p.nf ? p.cface[(size_t)i * p.nf + f] : 0;
        double F[NFM][NV];
#pragma unroll
        for (int f = 0; f < NFM; ++f) {
            const size_t id = cf[f] != 0 ? (size_t)(abs(cf[f]) - 1) : 0;
#pragma unroll
            for (int v = 0; v < NV; ++v) F[f][v] = p.fflux[id * NV + v];
        }
        double r[NV] = {0, 0, 0, 0, 0};
#pragma unroll
        for (int f = 0; f < NFM; ++f) {
            if (cf[f] > 0) {
#pragma unroll
                for (int v = 0; v < NV; ++v) r[v] = r[v] + F[f][v];
            } else if (cf[f] < 0) {
#pragma unroll
                for (int v = 0; v < NV; ++v) r[v] = r[v] - F[f][v];
            }
        }
        if (p.rhs_out) {
#pragma unroll
            for (int v = 0; v < NV; ++v) p.rhs_out[(size_t)i * NV + v] = r[v];
        }
        if (p.stage > 0) {
            const double oov = p.ovol[i];
            double *u = p.U + (size_t)i * NV, *u2 = p.U2 + (size_t)i * NV;
            const double to4 = 3.0 / 4.0, oo4 = 1.0 / 4.0, to3 = 2.0 / 3.0, oo3 = 1.0 / 3.0;
            double un[NV];
            if (p.stage == 1) {
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    u2[v] = u[v];
                    un[v] = u[v] - (dt * (r[v] * oov));
                }
            } else if (p.stage == 2) {
#pragma unroll
                for (int v = 0; v < NV; ++v) un[v] = (to4 * u2[v]) + (oo4 * u[v]) - (oo4 * (dt * (r[v] * oov)));
            } else {
#pragma unroll
                for (int v = 0; v < NV; ++v) un[v] = (oo3 * u2[v]) + (to3 * u[v]) - (to3 * (dt * (r[v] * oov)));
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) u[v] = un[v];
            if (p.u64) {
                double2 *r64 = (double2 *)(p.u64 + (size_t)i * 8);
                r64[0] = make_double2(un[0], un[1]);
                r64[1] = make_double2(un[2], un[3]);
                r64[2] = make_double2(un[4], 0.0);
                r64[3] = make_double2(0.0, 0.0);
            }
            if (p.copy) {
#pragma unroll
                for (int v = 0; v < NV; ++v) p.copy[(size_t)i * NV + v] = un[v];
            }
            if (p.stage == 3 && p.dt_next) {
                double w[NV];
                cons2prim_d(p.gamma, un, w);
                const double c = sqrt(w[4] * p.gamma / w[0]);
                const double veln = fmax(fmax(fabs(w[1]), fabs(w[2])), fabs(w[3])) + c;
                dtl = (p.cfl / 3.0) * (p.minedge[i] / fabs(veln));
            }
        }
    }
    if (p.stage == 3) {
        if (p.dt_next) dt_lower(p.dt_next, dtl);
        if (i == 0 && p.t) *p.t += dt;
    }
}

// Fluxes and update of a march on one-point faces (MUSCL on hexahedra): 8 lanes
// per cell, a lane per face.  Every flux is formed by both of its cells, in the
// owner's frame and so with the same bits, and the cell's lanes meet in LDS,
// where a lane per variable adds the faces in k_update's order.  The new state
// goes to another buffer (neighbours still read the old one).  Bound: the chain
// face record -> states -> HLLC; k_flux and k_update ran two such chains, a
// launch and the fluxes' way through memory one after the other.
// 24^3 hexahedra: 5.4 and 5.7 us and the gap between them before, 8.5 us this way
// (a march of 10 RK3 steps 0.69 -> 0.65 ms).
// adj [ncell][nf]: other cell or -code, its face slot | 256 triangle | 512 owner,
// face (-1: no face)
template <typename R>
__global__ __launch_bounds__(256) void k_flux_update(FluxParams<R> p, UpdateParams u, const int4 *adj) {
    constexpr int NFM = 6;
    __shared__ double sh[32][NFM][NV];
    const int l8 = threadIdx.x & 7, ci = threadIdx.x >> 3;
    const int i = blockIdx.x * 32 + ci;
    const double dt = dt_of(u.dt, u.dt_slots);
    if (u.stage == 2 && u.dt_next && blockIdx.x == 0) u.dt_next[threadIdx.x] = 0x7FF0000000000000ULL;
    // what the update reads, loaded beside the flux's chain
    const size_t e = (size_t)min(i, u.ncell - 1) * NV + min(l8, NV - 1);
    const double oov = u.ovol[min(i, u.ncell - 1)], us = p.U[e], u0 = u.stage == 1 ? us : u.U2[e];
    const double edge = u.stage == 3 && u.dt_next ? u.minedge[min(i, u.ncell - 1)] : 0.0;
    if (i < u.ncell && l8 < NFM) {
        double acc[NV] = {0, 0, 0, 0, 0};
        const int4 r = l8 < p.nf ? adj[(size_t)i * p.nf + l8] : make_int4(0, 0, -1, 0);
        if (r.z >= 0) {
            const int f = r.z;
            const bool own = (r.y >> 9) & 1, tri = (r.y >> 8) & 1, bnd = r.x < 0;
            const size_t oo = ((size_t)i * p.nf + l8) * NV;
            const size_t on = bnd ? oo : ((size_t)r.x * p.nf + (r.y & 255)) * NV;
            const size_t xo = (size_t)i * NV, xn = bnd ? xo : (size_t)r.x * NV;
            const double c1 = p.frot[4 * f], s1 = p.frot[4 * f + 1], c2 = p.frot[4 * f + 2], s2 = p.frot[4 * f + 3];
            double a[NV], bq[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double me = p.U[xo + v] + (double)p.uleft[oo + v];
                const double ot = bnd ? 0.0 : p.U[xn + v] + (double)p.uleft[on + v];
                a[v] = own ? me : ot;
                bq[v] = own ? ot : me;
            }
            if (bnd) {
                const double *fin = p.bface ? p.bface + (size_t)f * 10 : p.bc.inflow;
                const double *fout = p.bface ? p.bface + (size_t)f * 10 + 5 : p.bc.outflow;
                ghost_state(-r.x, p.bc.boundtype, p.gamma, a, c1, s1, c2, s2, fin, fout, bq);  // GET_STATES_BOUNDS
            }
            // ROTATEF (src/grid_t.f90:4217-4258)
            const double la[NV] = {a[0], c1 * s2 * a[1] + s1 * s2 * a[2] + c2 * a[3],
                                   c1 * c2 * a[1] + s1 * c2 * a[2] + (-s2) * a[3], (-s1) * a[1] + c1 * a[2], a[4]};
            const double ra[NV] = {bq[0], c1 * s2 * bq[1] + s1 * s2 * bq[2] + c2 * bq[3],
                                   c1 * c2 * bq[1] + s1 * c2 * bq[2] + (-s2) * bq[3], (-s1) * bq[1] + c1 * bq[2],
                                   bq[4]};
            double hd[NV];
            if (sizeof(R) == 8)
                hllc64(p.gamma, la, ra, hd);
            else
                hllc32(p.gamma, la, ra, hd);
            // ROTATEB (src/grid_t.f90:4261-4305)
            const double rb[NV] = {hd[0], c1 * s2 * hd[1] + c1 * c2 * hd[2] + (-s1) * hd[3],
                                   s1 * s2 * hd[1] + s1 * c2 * hd[2] + c1 * hd[3], c2 * hd[1] + (-s2) * hd[2], hd[4]};
            const double wa = (tri ? p.wt : p.wq)[0] * p.farea[f];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                acc[v] = acc[v] + (rb[v] * wa);
                if (!own) acc[v] = -acc[v];
            }
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) sh[ci][l8][v] = acc[v];
    }
    __syncthreads();
    double un = 1.0;
    if (i < u.ncell && l8 < NV) {
        double r = 0.0;
#pragma unroll
        for (int f = 0; f < NFM; ++f) r = r + sh[ci][f][l8];
        const double to4 = 3.0 / 4.0, oo4 = 1.0 / 4.0, to3 = 2.0 / 3.0, oo3 = 1.0 / 3.0;
        if (u.stage == 1)
            un = us - (dt * (r * oov));
        else if (u.stage == 2)
            un = (to4 * u0) + (oo4 * us) - (oo4 * (dt * (r * oov)));
        else
            un = (oo3 * u0) + (to3 * us) - (to3 * (dt * (r * oov)));
        u.U[e] = un;
    }
    if (u.stage == 3) {
        if (u.dt_next) {
            double c[NV], w[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) c[v] = __shfl(un, v, 8);
            double dtl = 1.0e300;
            if (i < u.ncell && l8 == 0) {
                cons2prim_d(u.gamma, c, w);
                const double cs = sqrt(w[4] * u.gamma / w[0]);
                const double veln = fmax(fmax(fabs(w[1]), fabs(w[2])), fabs(w[3])) + cs;
                dtl = (u.cfl / 3.0) * (edge / fabs(veln));
            }
            dt_lower(u.dt_next, dtl);
        }
        if (blockIdx.x == 0 && threadIdx.x == 0 && u.t) *u.t += dt;
    }
}

// k_flux_update's adj, once per context
__global__ __launch_bounds__(256) void k_face_records(size_t n, const int32_t *cface, const int32_t *fcell,
                                                      const int32_t *fslot, int4 *adj) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int id = abs(cface[e]) - 1, own = cface[e] > 0;
    adj[e] = id < 0 ? make_int4(0, 0, -1, 0)
                    : make_int4(fcell[2 * id + own], (fslot[2 * id + own] & 255) | (fslot[2 * id] & 256) | own << 9,
                                id, 0);
}

struct DtParams {
    int ncell;
    double cfl, gamma;
    const double *U, *minedge;
    unsigned long long *dt_out;
};

__global__ __launch_bounds__(256) void k_dt(DtParams p) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double d = 1.0e300;
    if (i < p.ncell) {
        double w[NV];
        cons2prim_d(p.gamma, p.U + (size_t)i * NV, w);
        const double c = sqrt(w[4] * p.gamma / w[0]);
        const double veln = fmax(fmax(fabs(w[1]), fabs(w[2])), fabs(w[3])) + c;
        d = (p.cfl / 3.0) * (p.minedge[i] / fabs(veln));
    }
    dt_lower(p.dt_out, d);
}

// the step size of a set of slots
__global__ void k_dt_value(const double *slots, double *out) {
    const double v = dt_of(slots, true);
    if (threadIdx.x == 0) *out = v;
}

// ---------------------------------------------------------------------------
// Adjoint of the residual: vector-Jacobian products w -> (dR/dU)^T w.
//
// The residual is R_i = sum over the faces of cell i of +-F_f, F_f the
// quadrature of ROTATEB(HLLC(ROTATEF(a_q), ROTATEF(b_q))) w_q |f|, with face
// states a_q = U_L + ULEFT_L(q) and b_q = U_R + ULEFT_R(q) (or the ghost
// state of a_q).  A product runs
//   k_flux_vjp  face-parallel: F_bar = w_owner - w_neighbour, and through
//               each quadrature point the cotangents of a_q and b_q, written
//               to the face-point slots of the two cells (each slot belongs
//               to exactly one face, so no atomics);
// then on the row stream
//   k_recon_vjp_s  tile of 8 cells per wave: pulls the face-point cotangents back
//               through the extrapolation, the WENO weights and indicators or the
//               Barth limiter, from the coefficients and decisions that the
//               forward reconstruction stored;
//   k_scatter_s64/s32  P_s^T g_bar_s to the tile's member table, over the rows;
// or on the other layouts (and for geometry cotangents)
//   k_recon_vjp tile of 8 cells per wave, lane = 8 * cell + stencil: repeats
//               the forward decisions of the reconstruction bit for bit
//               (same arithmetic and order), pulls the cotangents back alike,
//               and adds P_s^T g_bar_s to the tile's member table;
// and last
//   k_adj_gather  the member tables summed by cell.
// Discrete decisions (CHECKSOL / CHECKSOLX flags, HLLC and boundary
// regimes, the limiter's arg-min face point and arg-max/min neighbour) are
// those of the state the product is taken at, so the result is the exact
// derivative of the branch the primal takes.

// pseudo-inverse rows and stencil members in whichever device layout the
// forward kernels use: 0 per cell [cell][j][s][k] + [cell][s][j],
// 1 tiled [tile][j][k][8 ts] + [tile][j][8 ts], 2 the row stream
template <typename R>
struct LsqView {
    int mode, ts, tp, imax, ideg, depth, hd, pb, rd;
    long long tile_bytes;
    const int32_t *nbr;
    const R *P;
    const unsigned char *rows;
    __device__ int member(int tile, int cell, int s, int j, int pos) const {
        if (mode == 0) return nbr[((size_t)cell * ts + s) * imax + j];
        if (mode == 1) return nbr[((size_t)tile * imax + j) * tp + pos];
        const unsigned char *b = rows + (size_t)tile * tile_bytes;
        return j < depth ? ((const int32_t *)b)[j * tp + pos]
                         : ((const int32_t *)(b + hd + (size_t)(j - depth) * rd + pb))[pos];
    }
    // coefficient k of member j is row[k * kst]
    __device__ const R *row(int tile, int cell, int s, int j, int pos, int &kst) const {
        if (mode == 0) {
            kst = 1;
            return P + (((size_t)cell * imax + j) * ts + s) * ideg;
        }
        kst = tp;
        if (mode == 1) return P + ((size_t)tile * imax + j) * ideg * tp + pos;
        return (const R *)(rows + (size_t)tile * tile_bytes + hd + (size_t)j * rd) + pos;
    }
};

template <typename R>
struct VjpParams {
    int ncell, ntile, tiles_per_xcd, nf, nqm, qpq, qpt, iweno;
    double gamma, lwci1, eps;
    const double *U;
    LsqView<R> lsq;
    const R *B;            // [ncell][ideg*(ideg+1)/2]
    const R *mbar;         // [ncell][ideg]
    const R *qp;           // [ncell][nf][nqm][3]
    const int32_t *cinfo;
    const int32_t *cnb;    // [ncell][nf]
    const double *ubf;     // [ncell][nf][nqm][5] cotangents of the face-point states
    double *ubar;          // [ncell][5] accumulated
    const R *gload;        // row stream: the forward's stencil coefficients, indicators and
                           // weights [ntile][ideg*5 + 10][8 ts]
    const int *fload;      // row stream: the forward's per-cell flags (1 MUSCL, 2 first order)
    // the tile's distinct stencil members: member (j, pos) of tile t scatters
    // to table row slot[t][j][pos] (UCNS_NOSLOT: straight to HBM), and row r
    // of tile t belongs to cell uq[t][r], r < min(ucount[t], uq_cap); rows
    // past a kernel's LDS table also go straight to HBM and are written as 0
    const uint16_t *slot;
    const int32_t *uq, *ucount;
    int uq_cap;
    double *gbout;         // row stream: each stencil's g_bar [ntile][ideg*5][8 ts], for the scatter
    const int64_t *toff;   // first row of each tile's member table in tab
    double *tab;           // [rows][5] the member tables, summed per cell by k_adj_gather
    // geometry cotangents (k_recon_vjp with GEO, FP64), accumulated: pseudo-
    // inverses [ncell][lsq ts][imax][ideg], indicators [ncell][ideg][ideg]
    // (upper triangle, the part the library reads), basis means [ncell][ideg]
    // and face points [ncell][nf][nqm][3]
    double *gP, *gB, *gM, *gQ;
};

__device__ inline void atomic_add_f64(double *a, double v) { unsafeAtomicAdd(a, v); }


// Distinct members per tile: a wave's scatter goes through an LDS table of
// the tile's distinct member cells (a tile of 8 neighbouring cells shares
// most of its stencil members), flushed with one HBM atomic per member and
// variable instead of one per (stencil, member, variable).
constexpr int HT = 4096;  // hash slots: more than the 8 * 7 * 39 member entries a tile has at most

template <typename R, int IMAX>
__global__ __launch_bounds__(WAVE) void k_tile_members(LsqView<R> L, int ntile, int ncell, const int32_t *cinfo,
                                                       int cap, int32_t *uq, int32_t *ucount, uint16_t *slot) {
    __shared__ int32_t keys[HT];
    __shared__ uint16_t cid[HT];
    __shared__ uint16_t hs[IMAX * 64];
    const int lane = threadIdx.x;
    const int tile = blockIdx.x;
    if (tile >= ntile) return;
    const int ts = L.ts, tp = L.tp;
    for (int h = lane; h < HT; h += WAVE) keys[h] = -1;
    __syncthreads();
    // insert every (member row j, lane position) entry; linear probing
    for (int e = lane; e < IMAX * tp; e += WAVE) {
        const int j = e / tp, pos = e - j * tp;
        const int lc = pos / ts, s = pos - lc * ts;
        const int cell = tile * 8 + lc;
        int h = 0xFFFF;
        if (cell < ncell && s < ci_admis(cinfo[cell])) {
            const int n = L.member(tile, cell, s, j, pos);
            h = (int)(((unsigned)n * 2654435761u) >> 20) & (HT - 1);
            for (int probe = 0; probe < HT; ++probe) {
                const int old = atomicCAS(&keys[h], -1, n);
                if (old == -1 || old == n) break;
                h = (h + 1) & (HT - 1);
            }
        }
        hs[e] = (uint16_t)h;
    }
    __syncthreads();
    // compact: lane l owns hash slots [64 l, 64 l + 64)
    constexpr int PER = HT / WAVE;
    int cnt = 0;
    for (int k = 0; k < PER; ++k) cnt += keys[lane * PER + k] >= 0;
    int incl = cnt;
    for (int o = 1; o < WAVE; o <<= 1) {
        const int t = __shfl_up(incl, o, WAVE);
        if (lane >= o) incl += t;
    }
    int id = incl - cnt;
    for (int k = 0; k < PER; ++k) {
        const int h = lane * PER + k;
        const int key = keys[h];
        if (key >= 0) {
            cid[h] = id < cap ? (uint16_t)id : (uint16_t)UCNS_NOSLOT;
            if (id < cap) uq[(size_t)tile * cap + id] = key;
            ++id;
        }
    }
    if (lane == WAVE - 1) ucount[tile] = incl;
    __syncthreads();
    for (int e = lane; e < IMAX * tp; e += WAVE) {
        const int h = hs[e];
        slot[(size_t)tile * IMAX * tp + e] = h == 0xFFFF ? (uint16_t)UCNS_NOSLOT : cid[h];
    }
}

// pw(x, x^2, x^3, e) = x^e for e = 0..3
template <typename R>
__device__ inline R pw(R x, R x2, R x3, int e) {
    return e == 0 ? R(1) : e == 1 ? x : e == 2 ? x2 : x3;
}

// Reconstruction product on the tiled and per-cell layouts: the forward is
// repeated with its own arithmetic (the same bits, so the same decisions),
// then g_bar of each stencil is scattered through its pseudo-inverse rows.
template <typename R, int IDEG, int IMAX, int NQL, bool GEO = false>
__global__ __launch_bounds__(WAVE) void k_recon_vjp(VjpParams<R> p) {
    constexpr int NP = IDEG * (IDEG + 1) / 2;
    constexpr int KL = (IDEG + 7) / 8;    // coefficients per lane in the face-point pass
    __shared__ double sGb[8][IDEG * NV];  // cotangent of the combined coefficients
    __shared__ R sGh[8][IDEG * NV];       // combined coefficients sum_s omega_s G_s
    __shared__ R sG0[8][IDEG * NV];       // central-stencil coefficients
    __shared__ R sB[8][NP];               // the tile's indicator matrices
    __shared__ double sAcc[UCNS_TILE_UQ][NV];  // scatter to the tile's distinct members
    const int lane = threadIdx.x, lc = lane >> 3, s = lane & 7;
    const int b = blockIdx.x;
    const int tile = (b % NXCD) * p.tiles_per_xcd + b / NXCD;
    if (tile >= p.ntile) return;
    const int nuq = p.slot ? min(p.ucount[tile], p.uq_cap) : 0;
    for (int e = lane; e < min(nuq, UCNS_TILE_UQ) * NV; e += WAVE) (&sAcc[0][0])[e] = 0.0;
    if (p.iweno == 1) {
        const int nvc = min(8, p.ncell - tile * 8);
        const R *Bt = p.B + (size_t)tile * 8 * NP;
        for (int e = lane; e < nvc * NP; e += WAVE) (&sB[0][0])[e] = Bt[e];
    }
    const int cell = tile * 8 + lc;
    const bool cvalid = cell < p.ncell;
    const int cs = cvalid ? cell : 0;
    const int info = cvalid ? p.cinfo[cell] : 0;
    const int ifca = ci_ifca(info), admis = ci_admis(info), full = ci_full(info);
    const bool act = cvalid && s < admis;
    const int pos = lc * p.lsq.ts + s;
    double ui[NV] = {1.0, 0.0, 0.0, 0.0, 1.0};
    if (cvalid) {
#pragma unroll
        for (int v = 0; v < NV; ++v) ui[v] = p.U[(size_t)cell * NV + v];
    }
    const int nslot = ifca * p.nqm;
    const R *qpc = p.qp + (size_t)cs * p.nf * p.nqm * 3;
    const R *mb = p.mbar + (size_t)cs * IDEG;
    const double *ubc = p.ubf + (size_t)cs * p.nf * p.nqm * NV;
    auto qvalid = [&](int q) {
        const int f = q / p.nqm, qq = q - f * p.nqm;
        return cvalid && q < nslot && qq < (ci_tri(info, f) ? p.qpt : p.qpq);
    };

    // ---- A: cotangent of the combined coefficients, sum_q phi_q ubar_q
    // (lane s of a cell takes coefficients s, s+8, s+16 over all its face
    // points), and of the cell average through a_q = U_i + ULEFT(q) ----
    double usum[NV] = {0, 0, 0, 0, 0};
    {
        double ab[KL][NV];
        R mk[KL];
        int ex[KL][3];
#pragma unroll
        for (int t = 0; t < KL; ++t) {
            const int k = s + 8 * t;
            mk[t] = k < IDEG ? mb[k] : R(0);
#pragma unroll
            for (int d = 0; d < 3; ++d) ex[t][d] = k < IDEG ? c_mono[k][d] : 0;
#pragma unroll
            for (int v = 0; v < NV; ++v) ab[t][v] = 0.0;
        }
#pragma unroll 1
        for (int q = 0; q < nslot; ++q) {
            if (!qvalid(q)) continue;
            const R x0 = qpc[q * 3], x1 = qpc[q * 3 + 1], x2 = qpc[q * 3 + 2];
            const R x0s = x0 * x0, x1s = x1 * x1, x2s = x2 * x2;
            const R x0c = x0s * x0, x1c = x1s * x1, x2c = x2s * x2;
            double ub[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                ub[v] = ubc[q * NV + v];
                usum[v] += ub[v];
            }
#pragma unroll
            for (int t = 0; t < KL; ++t) {
                const double ph = (double)(pw(x0, x0s, x0c, ex[t][0]) * pw(x1, x1s, x1c, ex[t][1]) *
                                               pw(x2, x2s, x2c, ex[t][2]) - mk[t]);
#pragma unroll
                for (int v = 0; v < NV; ++v) ab[t][v] += ph * ub[v];
            }
        }
#pragma unroll
        for (int t = 0; t < KL; ++t) {
            const int k = s + 8 * t;
            if (k < IDEG) {
#pragma unroll
                for (int v = 0; v < NV; ++v) sGb[lc][k * NV + v] = ab[t][v];
            }
        }
    }
    __syncthreads();  // sGb, sB

    // ---- B: the stencil coefficients G_s = P_s dU_s, as the forward ----
    R g[IDEG][NV];
#pragma unroll
    for (int k = 0; k < IDEG; ++k)
#pragma unroll
        for (int v = 0; v < NV; ++v) g[k][v] = R(0);
    if (act) {
#pragma unroll 1
        for (int j = 0; j < IMAX; ++j) {
            const int n = p.lsq.member(tile, cell, s, j, pos);
            R du[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) du[v] = (R)(p.U[(size_t)n * NV + v] - ui[v]);
            int kst;
            const R *row = p.lsq.row(tile, cell, s, j, pos, kst);
            R pc[IDEG];
#pragma unroll
            for (int k = 0; k < IDEG; ++k) pc[k] = row[(size_t)k * kst];
#pragma unroll
            for (int k = 0; k < IDEG; ++k)
#pragma unroll
                for (int v = 0; v < NV; ++v) g[k][v] += pc[k] * du[v];
        }
    }
    if (s == 0) {
#pragma unroll
        for (int k = 0; k < IDEG; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) sG0[lc][k * NV + v] = g[k][v];
    }

    // ---- C: indicators, weights and combined coefficients (forward, with
    // its arithmetic: the same bits) ----
    R beta[NV] = {R(0), R(0), R(0), R(0), R(0)};
    R om[NV] = {R(0), R(0), R(0), R(0), R(0)};
    double obar[NV] = {0, 0, 0, 0, 0};
    double wi[NV];
    cons2prim_d(p.gamma, ui, wi);
    bool reduce = cvalid;
    if (p.iweno == 1) {
        if (act) {
#pragma unroll
            for (int k = 0; k < IDEG; ++k) {
                R bg[NV] = {R(0), R(0), R(0), R(0), R(0)};
#pragma unroll
                for (int l = 0; l < IDEG; ++l) {
                    const R bkl = sB[lc][pidx(IDEG, k, l)];
#pragma unroll
                    for (int v = 0; v < NV; ++v) bg[v] += bkl * g[l][v];
                }
#pragma unroll
                for (int v = 0; v < NV; ++v) beta[v] += g[k][v] * bg[v];
            }
        }
        const R lam = (s == 0) ? (R)p.lwci1 : R(1);
        const R eps = (R)p.eps;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            R w;
            if (sizeof(R) == 8) {
                const R x = eps + beta[v];
                const R x2 = x * x;
                w = act ? lam / (x2 * x2) : R(0);
            } else {
                const R x = eps + beta[v];
                const R xmin = grp_min8(act ? x : (R)INFINITY);
                const R r = xmin / x;
                const R r2 = r * r;
                w = act ? lam * (r2 * r2) : R(0);
            }
            const R sum = grp_sum8(w);
            om[v] = act ? w / sum : R(0);
        }
#pragma unroll
        for (int k = 0; k < IDEG; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const R gh = grp_sum8(om[v] * g[k][v]);
                if (s == 0) sGh[lc][k * NV + v] = gh;
                obar[v] += sGb[lc][k * NV + v] * (double)g[k][v];
            }
    }
    __syncthreads();  // sGb, sGh, sG0

    // ---- D: CHECKSOL (0.85) on the WENO face values (forward) ----
    if (p.iweno == 1) {
        int trouble = 0;
#pragma unroll 1
        for (int q = s; q < NQL * 8; q += 8) {
            if (!qvalid(q)) continue;
            R x[3] = {qpc[q * 3], qpc[q * 3 + 1], qpc[q * 3 + 2]};
            R phi[IDEG];
            basis_at<R, IDEG>(x, mb, phi);
            double uq[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                R res = R(0);
#pragma unroll
                for (int k = 0; k < IDEG; ++k) res += phi[k] * sGh[lc][k * NV + v];
                uq[v] = ui[v] + (double)res;
            }
            if (full && jump_test(p.gamma, wi, uq, 0.85)) trouble = 1;
        }
        const int any_trouble = grp_or8(trouble);
        reduce = cvalid && (!full || any_trouble);
    }
    __syncthreads();  // sG0

    // ---- E: MUSCL + Barth (forward), with the limiter's active arguments ----
    bool first = false;
    double slope[NV], d2s[NV];
    int qs[NV], ext[NV];
    R res0[NQL][NV];
    if (reduce) {
        double umin[NV], umax[NV];
        int imin[NV], imax_[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            umin[v] = umax[v] = ui[v];
            imin[v] = imax_[v] = cell;
        }
        for (int f = 0; f < ifca; ++f) {
            const int n = p.cnb[(size_t)cell * p.nf + f];
            if (n < 0) continue;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double un = p.U[(size_t)n * NV + v];
                if (un < umin[v]) imin[v] = n;
                if (un > umax[v]) imax_[v] = n;
                umin[v] = fmin(umin[v], un);
                umax[v] = fmax(umax[v], un);
            }
        }
        double lmin[NV];
        int lq[NV], lw[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            lmin[v] = 1.0e16;
            lq[v] = -1;
            lw[v] = 0;
        }
#pragma unroll
        for (int r = 0; r < NQL; ++r) {
            const int q = s + 8 * r;
#pragma unroll
            for (int v = 0; v < NV; ++v) res0[r][v] = R(0);
            if (qvalid(q)) {
                R x[3] = {qpc[q * 3], qpc[q * 3 + 1], qpc[q * 3 + 2]};
                R phi[IDEG];
                basis_at<R, IDEG>(x, mb, phi);
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    R res = R(0);
#pragma unroll
                    for (int k = 0; k < IDEG; ++k) res += phi[k] * sG0[lc][k * NV + v];
                    res0[r][v] = res;
                    const double d2 = (double)res;
                    double psi;
                    int wsel = 0;
                    if (fabs(d2) <= 0.0)
                        psi = 1.0;
                    else if (d2 > 0.0)
                        psi = fmin(1.0, (umax[v] - ui[v]) / d2);
                    else {
                        psi = fmin(1.0, (umin[v] - ui[v]) / d2);
                        wsel = 1;
                    }
                    if (psi < lmin[v]) {
                        lmin[v] = psi;
                        lq[v] = q;
                        lw[v] = wsel;
                    }
                }
            }
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            slope[v] = grp_min8(lmin[v]);
            // lowest lane of the group holding the minimum
            int cand = (lmin[v] == slope[v]) ? s : 8;
            cand = min(cand, __shfl_xor(cand, 1, WAVE));
            cand = min(cand, __shfl_xor(cand, 2, WAVE));
            cand = min(cand, __shfl_xor(cand, 4, WAVE));
            const int src = lc * 8 + cand;
            qs[v] = lane_bcast(lq[v], src);
            const int wsel = lane_bcast(lw[v], src);
            ext[v] = wsel ? imin[v] : imax_[v];
            d2s[v] = 0.0;
        }
        // the unlimited value at the arg-min point, for the active limiters
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            double mine = 0.0;
#pragma unroll
            for (int r = 0; r < NQL; ++r)
                if (s + 8 * r == qs[v]) mine = (double)res0[r][v];
            d2s[v] = grp_sum8(mine);
        }
        int tr2 = 0;
#pragma unroll
        for (int r = 0; r < NQL; ++r) {
            const int q = s + 8 * r;
            if (qvalid(q)) {
                double uq[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) uq[v] = ui[v] + (double)(R)((double)res0[r][v] * slope[v]);
                if (jump_test(p.gamma, wi, uq, 0.95)) tr2 = 1;
            }
        }
        first = grp_or8(tr2) != 0;
    }

    // ---- F: cotangent of each lane's stencil coefficients ----
    double gb[IDEG][NV];
#pragma unroll
    for (int k = 0; k < IDEG; ++k)
#pragma unroll
        for (int v = 0; v < NV; ++v) gb[k][v] = 0.0;
    auto put = [&](int k, int v, double x) { gb[k][v] = x; };
    double ubi[NV];  // extra cotangent of U_i from the limiter
    double cq[NV], bb[NV];  // limiter correction at the arg-min point; indicator cotangents
    bool scatter = false;
#pragma unroll
    for (int v = 0; v < NV; ++v) ubi[v] = cq[v] = bb[v] = 0.0;
    if (cvalid && !first && reduce) {
        // ULEFT(q) = slope * d2_q: slope_bar = sum_q ubar_q d2_q; through an
        // active limiter slope = (u_ext - u_i) / d2_{q*}
        double sb[NV] = {0, 0, 0, 0, 0};
#pragma unroll
        for (int r = 0; r < NQL; ++r) {
            const int q = s + 8 * r;
            if (qvalid(q)) {
#pragma unroll
                for (int v = 0; v < NV; ++v) sb[v] += ubc[q * NV + v] * (double)res0[r][v];
            }
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            sb[v] = grp_sum8(sb[v]);
            const bool on = slope[v] < 1.0 && qs[v] >= 0;
            const double e = on ? sb[v] / d2s[v] : 0.0;
            cq[v] = on ? e * slope[v] : 0.0;
            ubi[v] = -e;
            if (s == 0 && on) atomic_add_f64(&p.ubar[(size_t)ext[v] * NV + v], e);
        }
        scatter = s == 0;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            R phi[IDEG];
            const bool corr = s == 0 && cq[v] != 0.0;
            if (corr) {
                const int q = qs[v];
                R x[3] = {qpc[q * 3], qpc[q * 3 + 1], qpc[q * 3 + 2]};
                basis_at<R, IDEG>(x, mb, phi);
            }
#pragma unroll
            for (int k = 0; k < IDEG; ++k)
                put(k, v, s == 0 ? slope[v] * sGb[lc][k * NV + v] - (corr ? cq[v] * (double)phi[k] : 0.0) : 0.0);
        }
    } else if (cvalid && !first) {
        // omega_s = lam_s (eps+beta_s)^-4 / sum_t (...):
        // beta_bar_s = -4 omega_s/(eps+beta_s) (obar_s - sum_t omega_t obar_t)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double so = grp_sum8(act ? (double)om[v] * obar[v] : 0.0);
            bb[v] = act ? -4.0 * (double)om[v] / ((double)p.eps + (double)beta[v]) * (obar[v] - so) : 0.0;
        }
        scatter = act;
        // g_bar_s = omega_s gh_bar + 2 beta_bar_s B G_s
#pragma unroll
        for (int v = 0; v < NV; ++v) {
#pragma unroll
            for (int k = 0; k < IDEG; ++k) {
                double hg = 0.0;
#pragma unroll
                for (int l = 0; l < IDEG; ++l) hg += (double)sB[lc][pidx(IDEG, k, l)] * (double)g[l][v];
                put(k, v, act ? (double)om[v] * sGb[lc][k * NV + v] + 2.0 * bb[v] * hg : 0.0);
            }
        }
    } else {
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int k = 0; k < IDEG; ++k) put(k, v, 0.0);
    }

    if constexpr (GEO) {
        // ---- geometry: face points and basis means.  A face value is
        // U_i + sum_k phi_k(x_q) c_k with phi_k = m_k - mbar_k and c the
        // combined WENO coefficients (sGh) or, on the MUSCL path, slope times
        // the central ones (sG0, with the limiter's own dependence on the
        // arg-min point's value); phi_bar_k(q) = sum_v r_bar_v(q) c_kv ----
        const bool weno = cvalid && !first && !reduce && p.iweno == 1;
        const bool muscl = cvalid && !first && reduce;
        double mba[IDEG];
#pragma unroll
        for (int k = 0; k < IDEG; ++k) mba[k] = 0.0;
#pragma unroll
        for (int r = 0; r < NQL; ++r) {
            const int q = s + 8 * r;
            if (!(weno || muscl) || !qvalid(q)) continue;
            const double x[3] = {(double)qpc[q * 3], (double)qpc[q * 3 + 1], (double)qpc[q * 3 + 2]};
            double rb[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double ub = ubc[q * NV + v];
                rb[v] = weno ? ub : slope[v] * ub - (q == qs[v] ? cq[v] : 0.0);
            }
            double xb[3] = {0.0, 0.0, 0.0};
            double pw3[3][4];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                pw3[d][0] = 1.0;
#pragma unroll
                for (int e = 1; e < 4; ++e) pw3[d][e] = pw3[d][e - 1] * x[d];
            }
#pragma unroll
            for (int k = 0; k < IDEG; ++k) {
                double pb = 0.0;
#pragma unroll
                for (int v = 0; v < NV; ++v)
                    pb += rb[v] * (double)(weno ? sGh[lc][k * NV + v] : sG0[lc][k * NV + v]);
                mba[k] -= pb;
                const int e0 = c_mono[k][0], e1 = c_mono[k][1], e2 = c_mono[k][2];
                if (e0 > 0) xb[0] += pb * e0 * pw3[0][e0 - 1] * pw3[1][e1] * pw3[2][e2];
                if (e1 > 0) xb[1] += pb * e1 * pw3[0][e0] * pw3[1][e1 - 1] * pw3[2][e2];
                if (e2 > 0) xb[2] += pb * e2 * pw3[0][e0] * pw3[1][e1] * pw3[2][e2 - 1];
            }
            double *gq = p.gQ + ((size_t)cell * p.nf * p.nqm + q) * 3;
#pragma unroll
            for (int d = 0; d < 3; ++d) gq[d] += xb[d];
        }
#pragma unroll
        for (int k = 0; k < IDEG; ++k) {
            const double t = grp_sum8(mba[k]);
            if (s == 0 && cvalid) p.gM[(size_t)cell * IDEG + k] += t;
        }
        // ---- indicators: beta_s,v = sum_kl B_kl g_k g_l over the full square
        // of the packed upper triangle ----
        if (p.iweno == 1) {
            const bool on = weno && act;
#pragma unroll
            for (int k = 0; k < IDEG; ++k)
#pragma unroll
                for (int l = k; l < IDEG; ++l) {
                    double c = 0.0;
                    if (on) {
#pragma unroll
                        for (int v = 0; v < NV; ++v) c += bb[v] * (double)g[k][v] * (double)g[l][v];
                    }
                    const double t = grp_sum8(k == l ? c : 2.0 * c);
                    if (s == 0 && cvalid) p.gB[((size_t)cell * IDEG + k) * IDEG + l] += t;
                }
        }
    }

    // ---- G: dU_bar_j = P_j^T g_bar to the members, minus the same to U_i ----
    double acc[NV] = {0, 0, 0, 0, 0};
    if (scatter) {
        // member j+1's row and index are in flight while member j is scattered
        int kst;
        int n = p.lsq.member(tile, cell, s, 0, pos);
        const R *row = p.lsq.row(tile, cell, s, 0, pos, kst);
        R pc[IDEG];
#pragma unroll
        for (int k = 0; k < IDEG; ++k) pc[k] = row[(size_t)k * kst];
#pragma unroll 1
        for (int j = 0; j < IMAX; ++j) {
            R pn[IDEG];
            int nn = 0;
            if (j + 1 < IMAX) {
                nn = p.lsq.member(tile, cell, s, j + 1, pos);
                const R *rn = p.lsq.row(tile, cell, s, j + 1, pos, kst);
#pragma unroll
                for (int k = 0; k < IDEG; ++k) pn[k] = rn[(size_t)k * kst];
            }
            double d[NV] = {0, 0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < IDEG; ++k) {
                const double pk = (double)pc[k];
#pragma unroll
                for (int v = 0; v < NV; ++v) d[v] += pk * gb[k][v];
            }
            if constexpr (GEO) {
                // G_s = P_s dU: P_bar(j, k) = sum_v g_bar(k, v) dU_j(v)
                double du[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) du[v] = p.U[(size_t)n * NV + v] - ui[v];
                double *gp = p.gP + (((size_t)cell * p.lsq.ts + s) * IMAX + j) * IDEG;
#pragma unroll
                for (int k = 0; k < IDEG; ++k) {
                    double t = 0.0;
#pragma unroll
                    for (int v = 0; v < NV; ++v) t += gb[k][v] * du[v];
                    gp[k] += t;
                }
            }
            const unsigned sl = p.slot ? p.slot[((size_t)tile * IMAX + j) * p.lsq.tp + pos] : UCNS_NOSLOT;
            if (sl < UCNS_TILE_UQ) {
#pragma unroll
                for (int v = 0; v < NV; ++v)
                    __hip_atomic_fetch_add(&sAcc[sl][v], d[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            } else {
#pragma unroll
                for (int v = 0; v < NV; ++v) atomic_add_f64(&p.ubar[(size_t)n * NV + v], d[v]);
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] -= d[v];
            n = nn;
#pragma unroll
            for (int k = 0; k < IDEG; ++k) pc[k] = pn[k];
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const double t = grp_sum8(acc[v]);
        if (s == 0 && cvalid) atomic_add_f64(&p.ubar[(size_t)cell * NV + v], t + usum[v] + ubi[v]);
    }
    if (nuq > 0) {
        __syncthreads();
        double *tt = p.tab + (size_t)p.toff[tile] * NV;
        for (int e = lane; e < nuq * NV; e += WAVE) tt[e] = e < UCNS_TILE_UQ * NV ? (&sAcc[0][0])[e] : 0.0;
    }
}

// Reconstruction product on the row-stream layouts (TS stencils per cell,
// TP = 8 TS columns per tile row).  The forward kept each stencil's
// coefficients G_s, indicators and weights ([tile][ideg*5 + 10][TP], gload)
// and each cell's flags (fload: 1 MUSCL, 2 first order), so nothing of the
// forward is repeated: the flags pick one of three paths per cell, and g_bar
// of every stencil goes to p.gbout ([tile][ideg*5][TP]) for the row-stream
// scatter.  On the WENO path every step is per variable (indicators and
// weights are), so a lane holds one variable's column of G_s at a time; B G_s
// runs over the packed triangle of B once per variable.
// Bound by latency at two or three waves per SIMD (registers; in FP64 32 bytes a
// lane spill for hexahedra at WENO-4, 16 at WENO-3), and by the issue of
// the face-point pass: with each lane taking a quarter of the coefficients at
// every other point, the monomials of run-time exponents had been most of its
// instructions.  Adjoint of 2 steps on 24,576 tetrahedra 3.34 -> 3.13 ms, on
// 3,375 hexahedra 1.19 -> 1.05 ms, of 3 steps on a 14,000-cell channel 1.76 ->
// 1.71 ms.
template <typename R, int IDEG, int NQL, int TS>
__global__ __launch_bounds__(WAVE, IDEG == 9 ? 3 : 2) void k_recon_vjp_s(VjpParams<R> p) {
    constexpr int NP = IDEG * (IDEG + 1) / 2;
    constexpr int KL = (IDEG + 7) / 8;  // coefficients per lane in the face-point pass
    constexpr int BL = (8 * NP + WAVE - 1) / WAVE;
    // the face-point pass's basis values and cotangents, then the indicators
    constexpr int PHI = 8 * 8 * IDEG * (int)sizeof(R), PASS = PHI + 8 * 8 * NV * 8, BB = 8 * NP * (int)sizeof(R);
    constexpr int TP = 8 * TS;
    constexpr unsigned KS = NV * TP;    // stride of one coefficient row (elements)
    __shared__ double sGb[8][IDEG * NV];  // cotangent of the combined coefficients
    __shared__ __align__(16) char sRaw[PASS > BB ? PASS : BB];
    R(*sB)[NP] = (R(*)[NP])sRaw;                      // the tile's indicator matrices
    R(*sPhi)[8][IDEG] = (R(*)[8][IDEG])sRaw;          // 8 points of each cell: basis values
    double(*sUb)[8][NV] = (double(*)[8][NV])(sRaw + PHI);  // and cotangents (0 where there is no point)
    const int lane = threadIdx.x, lc = lane >> 3, s = lane & 7;
    const int b = blockIdx.x;
    const int tile = (b % NXCD) * p.tiles_per_xcd + b / NXCD;
    if (tile >= p.ntile) return;
    // the indicators wait in registers: their LDS serves the face points first
    R br[BL];
    const int nB = min(8, p.ncell - tile * 8) * NP;
#pragma unroll
    for (int t = 0; t < BL; ++t) br[t] = p.B[(size_t)tile * 8 * NP + min(lane + t * WAVE, nB - 1)];
    const int cell = tile * 8 + lc;
    const bool cvalid = cell < p.ncell;
    const int cs = cvalid ? cell : 0;
    const int info = cvalid ? p.cinfo[cell] : 0;
    const int fl = cvalid ? p.fload[cell] : 0;
    const int ifca = ci_ifca(info), admis = ci_admis(info);
    const bool act = cvalid && s < admis;
    const int nslot = cvalid ? ifca * p.nqm : 0;
    const R *qpc = p.qp + (size_t)cs * p.nf * p.nqm * 3;
    const R *mb = p.mbar + (size_t)cs * IDEG;
    const double *ubc = p.ubf + (size_t)cs * p.nf * p.nqm * NV;
    auto qvalid = [&](int q) {
        const int f = q / p.nqm, qq = q - f * p.nqm;
        return q < nslot && qq < (ci_tri(info, f) ? p.qpt : p.qpq);
    };

    // ---- cotangent of the combined coefficients, sum_q phi_q ubar_q, and of
    // the cell average through a_q = U_i + ULEFT(q), 8 face points of each cell
    // at a time: lane s evaluates the basis at point s and leaves it in LDS with
    // the point's cotangent, then takes coefficients s, s+8, s+16 over the eight ----
    double usum[NV] = {0, 0, 0, 0, 0};
    {
        double ab[KL][NV];
#pragma unroll
        for (int t = 0; t < KL; ++t)
#pragma unroll
            for (int v = 0; v < NV; ++v) ab[t][v] = 0.0;
        const int nq8 = p.nf * p.nqm;
        R x[3];
        double ub[NV];
        auto fetch = [&](int q) {  // indices stay in the cell's block
            const int qc = max(0, min(q, nslot - 1));
#pragma unroll
            for (int d = 0; d < 3; ++d) x[d] = qpc[qc * 3 + d];
#pragma unroll
            for (int v = 0; v < NV; ++v) ub[v] = ubc[qc * NV + v];
        };
        fetch(s);
#pragma unroll 1
        for (int q0 = 0; q0 < nq8; q0 += 8) {
            const bool ok = qvalid(q0 + s);
            {
                // a slot without a point holds whatever the caller left there
                const R xp[3] = {ok ? x[0] : R(0), ok ? x[1] : R(0), ok ? x[2] : R(0)};
                R phi[IDEG];
                basis_at<R, IDEG>(xp, mb, phi);
#pragma unroll
                for (int k = 0; k < IDEG; ++k) sPhi[lc][s][k] = phi[k];
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double u = ok ? ub[v] : 0.0;
                sUb[lc][s][v] = u;
                usum[v] += u;
            }
            fetch(q0 + 8 + s);
            __syncthreads();
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                double uv[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) uv[v] = sUb[lc][u][v];
#pragma unroll
                for (int t = 0; t < KL; ++t) {
                    const double ph = (double)sPhi[lc][u][min(s + 8 * t, IDEG - 1)];
#pragma unroll
                    for (int v = 0; v < NV; ++v) ab[t][v] += ph * uv[v];
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) usum[v] = grp_sum8(usum[v]);
#pragma unroll
        for (int t = 0; t < KL; ++t) {
            const int k = s + 8 * t;
            if (k < IDEG) {
#pragma unroll
                for (int v = 0; v < NV; ++v) sGb[lc][k * NV + v] = ab[t][v];
            }
        }
    }
#pragma unroll
    for (int t = 0; t < BL; ++t)
        if (lane + t * WAVE < nB) sB[0][lane + t * WAVE] = br[t];
    __syncthreads();  // sGb, sB

    const bool reduce = cvalid && (fl & 1), first = (fl & 2) != 0;
    // the tile's blocks (uniform) and this lane's column in them; lanes past
    // the cell's stencils read stencil 0's column and write nothing
    const R *gt = p.gload + (size_t)tile * (IDEG + 2) * KS;
    double *gbt = p.gbout + (size_t)tile * IDEG * KS;
    const unsigned c0 = lc * TS, col = c0 + (s < TS ? s : 0);
    const bool wr = cvalid && s < TS;
    // a MUSCL cell has no use for its indicator matrix: its LDS row takes the
    // central stencil's coefficients
    static_assert(IDEG * NV <= NP, "central coefficients exceed the indicator row");
    R *g0 = &sB[lc][0];
    if (reduce && !first)
        for (int e = s; e < IDEG * NV; e += 8) g0[e] = gt[c0 + (unsigned)e * TP];
    __syncthreads();  // g0
    double ubi[NV] = {0, 0, 0, 0, 0};  // extra cotangent of U_i from the limiter
    if (cvalid && !reduce) {
        // WENO: omega_s = lam_s (eps+beta_s)^-4 / sum_t (...), so with
        // obar_s = gh_bar . G_s:  beta_bar_s = -4 omega_s/(eps+beta_s)
        // (obar_s - sum_t omega_t obar_t),  g_bar_s = omega_s gh_bar + 2 beta_bar_s B G_s
#pragma unroll 1
        for (int v = 0; v < NV; ++v) {
            // B is re-read from LDS per variable: kept in registers across the
            // loop it would take NP of them
            asm volatile("" ::: "memory");
            const unsigned cv = col + (unsigned)v * TP;
            R gv[IDEG];
#pragma unroll
            for (int k = 0; k < IDEG; ++k) gv[k] = act ? gt[cv + k * KS] : R(0);
            const double beta = act ? (double)gt[cv + IDEG * KS] : 0.0;
            const double om = act ? (double)gt[cv + IDEG * KS + NV * TP] : 0.0;
            double obar = 0.0;
#pragma unroll
            for (int k = 0; k < IDEG; ++k) obar += sGb[lc][k * NV + v] * (double)gv[k];
            const double so = grp_sum8(act ? om * obar : 0.0);
            const double bb = act ? -4.0 * om / ((double)p.eps + beta) * (obar - so) : 0.0;
            double hg[IDEG];
#pragma unroll
            for (int k = 0; k < IDEG; ++k) hg[k] = (double)sB[lc][pidx(IDEG, k, k)] * (double)gv[k];
            // one row of B in registers at a time: each row's products are
            // pinned before the next row is read (else the compiler defers
            // them to the stores and keeps all of B live)
#pragma unroll
            for (int k = 0; k < IDEG; ++k) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int l = k + 1; l < IDEG; ++l) {
                    const double bkl = (double)sB[lc][pidx(IDEG, k, l)];
                    hg[k] += bkl * (double)gv[l];
                    hg[l] += bkl * (double)gv[k];
                }
#pragma unroll
                for (int l = k; l < IDEG; ++l) asm volatile("" : "+v"(hg[l]));
            }
            if (wr) {
#pragma unroll
                for (int k = 0; k < IDEG; ++k)
                    gbt[cv + k * KS] = act ? om * sGb[lc][k * NV + v] + 2.0 * bb * hg[k] : 0.0;
            }
        }
    } else if (reduce && !first) {
        // MUSCL + Barth with the forward's arithmetic, for the limiter's
        // active arguments: its arg-min face point and bound neighbour
        double ui[NV], umin[NV], umax[NV];
        int imin[NV], imax_[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            ui[v] = p.U[(size_t)cell * NV + v];
            umin[v] = umax[v] = ui[v];
            imin[v] = imax_[v] = cell;
        }
        for (int f = 0; f < ifca; ++f) {
            const int n = p.cnb[(size_t)cell * p.nf + f];
            if (n < 0) continue;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double un = p.U[(size_t)n * NV + v];
                if (un < umin[v]) imin[v] = n;
                if (un > umax[v]) imax_[v] = n;
                umin[v] = fmin(umin[v], un);
                umax[v] = fmax(umax[v], un);
            }
        }
        double lmin[NV];
        int lq[NV], lw[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            lmin[v] = 1.0e16;
            lq[v] = -1;
            lw[v] = 0;
        }
        R res0[NQL][NV];
#pragma unroll
        for (int r = 0; r < NQL; ++r) {
            const int q = s + 8 * r;
#pragma unroll
            for (int v = 0; v < NV; ++v) res0[r][v] = R(0);
            if (qvalid(q)) {
                R x[3] = {qpc[q * 3], qpc[q * 3 + 1], qpc[q * 3 + 2]};
                R phi[IDEG];
                basis_at<R, IDEG>(x, mb, phi);
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    R res = R(0);
#pragma unroll
                    for (int k = 0; k < IDEG; ++k) res += phi[k] * g0[k * NV + v];
                    res0[r][v] = res;
                    const double d2 = (double)res;
                    double psi;
                    int wsel = 0;
                    if (fabs(d2) <= 0.0)
                        psi = 1.0;
                    else if (d2 > 0.0)
                        psi = fmin(1.0, (umax[v] - ui[v]) / d2);
                    else {
                        psi = fmin(1.0, (umin[v] - ui[v]) / d2);
                        wsel = 1;
                    }
                    if (psi < lmin[v]) {
                        lmin[v] = psi;
                        lq[v] = q;
                        lw[v] = wsel;
                    }
                }
            }
        }
        // ULEFT(q) = slope * d2_q: slope_bar = sum_q ubar_q d2_q; through an
        // active limiter slope = (u_ext - u_i) / d2_{q*}
        double sb[NV] = {0, 0, 0, 0, 0};
#pragma unroll
        for (int r = 0; r < NQL; ++r) {
            const int q = s + 8 * r;
            if (qvalid(q)) {
#pragma unroll
                for (int v = 0; v < NV; ++v) sb[v] += ubc[q * NV + v] * (double)res0[r][v];
            }
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double slope = grp_min8(lmin[v]);
            // lowest lane of the group holding the minimum
            int cand = (lmin[v] == slope) ? s : 8;
            cand = min(cand, __shfl_xor(cand, 1, WAVE));
            cand = min(cand, __shfl_xor(cand, 2, WAVE));
            cand = min(cand, __shfl_xor(cand, 4, WAVE));
            const int src = lc * 8 + cand;
            const int qs = lane_bcast(lq[v], src);
            const int wsel = lane_bcast(lw[v], src);
            const int ext = wsel ? imin[v] : imax_[v];
            // the unlimited value at the arg-min point
            double mine = 0.0;
#pragma unroll
            for (int r = 0; r < NQL; ++r)
                if (s + 8 * r == qs) mine = (double)res0[r][v];
            const double d2s = grp_sum8(mine);
            const double sbv = grp_sum8(sb[v]);
            const bool on = slope < 1.0 && qs >= 0;
            const double e = on ? sbv / d2s : 0.0;
            const double cq = on ? e * slope : 0.0;
            ubi[v] = -e;
            if (s == 0 && on) atomic_add_f64(&p.ubar[(size_t)ext * NV + v], e);
            if (wr) {
                // only the central stencil (lane 0) carries a coefficient cotangent
                R phi[IDEG];
                const bool corr = s == 0 && cq != 0.0;
                if (corr) {
                    R x[3] = {qpc[qs * 3], qpc[qs * 3 + 1], qpc[qs * 3 + 2]};
                    basis_at<R, IDEG>(x, mb, phi);
                }
                const unsigned cv = col + (unsigned)v * TP;
#pragma unroll
                for (int k = 0; k < IDEG; ++k)
                    gbt[cv + k * KS] = s == 0 ? slope * sGb[lc][k * NV + v] - (corr ? cq * (double)phi[k] : 0.0)
                                              : 0.0;
            }
        }
    } else if (wr) {
        // first-order cells: no coefficient cotangent
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int k = 0; k < IDEG; ++k) gbt[col + (unsigned)v * TP + k * KS] = 0.0;
    }
    if (s == 0 && cvalid) {
#pragma unroll
        for (int v = 0; v < NV; ++v) atomic_add_f64(&p.ubar[(size_t)cell * NV + v], usum[v] + ubi[v]);
    }
}

// ubar[n] += the rows of every tile's member table that belong to cell n
// (CSR: rows ent[off[n]] .. ent[off[n+1]-1]); no atomics.  Bound by the
// latency of the dependent loads entry -> row: 8 lanes share a cell, each
// taking every 8th row, so that a cell of WENO-4 tetrahedra (43 rows) is 6
// trips and the launch has 8 times the waves of one thread per cell.
// 24,576 tetrahedra: 54.7 -> 26.0 us (one thread per cell before); a
// 14,000-cell channel: 27.6 -> 9.5 us.
__global__ __launch_bounds__(256) void k_adj_gather(int ncell, const int64_t *off, const int32_t *ent,
                                                    const double *tab, double *ubar) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x, n = t >> 3, s = t & 7;
    double a[NV] = {0, 0, 0, 0, 0};
    if (n < ncell) {
        constexpr int GU = 2;  // rows in flight per lane
        const int64_t e0 = off[n], e1 = off[n + 1];
        for (int64_t e = e0 + s; e < e1; e += 8 * GU) {
            int32_t rr[GU];
#pragma unroll
            for (int u = 0; u < GU; ++u) rr[u] = ent[min(e + 8 * u, e1 - 1)];
            double x[GU][NV];
#pragma unroll
            for (int u = 0; u < GU; ++u)
#pragma unroll
                for (int v = 0; v < NV; ++v) x[u][v] = tab[(size_t)rr[u] * NV + v];
#pragma unroll
            for (int u = 0; u < GU; ++u)
                if (e + 8 * u < e1) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) a[v] += x[u][v];
                }
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) a[v] = grp_sum8(a[v]);
    if (n < ncell && s < NV) {
        double m = a[0];
#pragma unroll
        for (int v = 1; v < NV; ++v) m = s == v ? a[v] : m;
        ubar[(size_t)n * NV + s] += m;
    }
}

// CSR of the member tables by cell: counts, then positions
__global__ void k_adj_csr(int ntile, int cap, const int32_t *uq, const int32_t *ucount, const int64_t *toff,
                          int64_t *cnt, const int64_t *off, int32_t *ent) {
    const int t = blockIdx.x;
    if (t >= ntile) return;
    const int nu = min(ucount[t], cap);
    for (int r = threadIdx.x; r < nu; r += blockDim.x) {
        const int n = uq[(size_t)t * cap + r];
        const unsigned long long k = atomicAdd((unsigned long long *)&cnt[n], 1ull);
        if (off) ent[off[n] + (int64_t)k] = (int32_t)(toff[t] + r);
    }
}

// Face-parallel adjoint of the HLLC flux quadrature: HLLC by its reverse
// mode (hllc_vjp); the ghost state's Jacobian (5 inputs, plus the 10
// free-stream values) from forward-mode passes of the same templated code the
// primal runs, one pass per input; F_bar is pulled back through ROTATEB
// (whose transpose is ROTATEF) and ROTATEF (transpose ROTATEB).
//
// One thread per interior (face, quadrature point): the points are independent,
// their writes are contiguous across lanes, and a small mesh still fills the
// chip (one thread per face left 121 blocks for a 14,000-cell channel).
// Boundary faces, by list, come in the first blocks of the same launch (meshes
// without any get a kernel without their registers) with 16 lanes per point: a
// lane per ghost-state input, where one thread ran the 15 passes one after the
// other.  The block reduces the free-stream cotangents before its atomics
// (same-address atomics retire one per 12 ns).
// 14,000-cell channel: a thread per face 19.4 us and, boundary, 113.7; a thread
// per point 10.6 and 20.6; this launch 19.5.  24,576 tetrahedra: 34.9 -> 22.4 us.
constexpr int BLANES = 16;
// the (face, point) number of a thread, at `lanes` threads per point: a launch may
// hold more than 2^31 threads (from 134 million boundary points on), the points
// stay below that
__host__ __device__ constexpr int vjp_point(int block, int thread, int lanes) {
    return (int)(((long long)block * 256 + thread) / lanes);
}
static_assert(vjp_point(0, 255, BLANES) == 15 && vjp_point(8388607, 255, BLANES) == 134217727 &&
              vjp_point(8388608, 0, BLANES) == 134217728 && vjp_point(134217727, 255, BLANES) == 2147483647 &&
              vjp_point(8388607, 255, 1) == 2147483647);
template <typename R, bool BND>
__device__ __forceinline__ void flux_vjp_block(const FluxParams<R> &p, int block, const int32_t *bfaces, int nbface,
                                               const double *lam, double *ubf, double *bcbar) {
    const int t = vjp_point(block, threadIdx.x, BND ? BLANES : 1);
    const int fi = t / p.nqm, q = t - fi * p.nqm;
    const int f = BND ? (fi < nbface ? bfaces[fi] : p.nface) : fi;
    constexpr bool bnd = BND;
    const int m = threadIdx.x & (BLANES - 1);
    double bcd = 0.0;  // boundary: this lane's free-stream cotangent
    auto point = [&]() {
        const int cL = p.fcell[2 * f], cR = p.fcell[2 * f + 1];
        if ((cR < 0) != BND) return;
        const int s0 = p.fslot[2 * f], sR = p.fslot[2 * f + 1];
        const int sL = s0 & 255;
        const bool tri = (s0 >> 8) & 1;
        if (q >= (tri ? p.qpt : p.qpq)) return;
        const double *w = tri ? p.wt : p.wq;
        const double c1 = p.frot[4 * f], s1 = p.frot[4 * f + 1], c2 = p.frot[4 * f + 2], s2 = p.frot[4 * f + 3];
        const double area = p.farea[f];
        const size_t oL = (((size_t)cL * p.nf + sL) * p.nqm + q) * NV;
        const size_t oR = bnd ? oL : (((size_t)cR * p.nf + sR) * p.nqm + q) * NV;
        double a[NV], bq[NV], Fb[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            a[v] = p.U[(size_t)cL * NV + v] + (double)p.uleft[oL + v];
            bq[v] = bnd ? 0.0 : p.U[(size_t)cR * NV + v] + (double)p.uleft[oR + v];
            Fb[v] = lam[(size_t)cL * NV + v] - (bnd ? 0.0 : lam[(size_t)cR * NV + v]);
        }
        double hb0[NV];
        rotf(Fb, c1, s1, c2, s2, hb0);
        if (bnd) ghost_state(-cR, p.bc.boundtype, p.gamma, a, c1, s1, c2, s2, p.bc.inflow, p.bc.outflow, bq);
        double la[NV], ra[NV];
        rotf(a, c1, s1, c2, s2, la);
        rotf(bq, c1, s1, c2, s2, ra);
        const double wa = w[q] * area;
        double hb[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) hb[v] = wa * hb0[v];
        double lab[NV], rab[NV];
        hllc_vjp(p.gamma, la, ra, hb, lab, rab);
        double ab[NV], bb[NV];
        rotb(lab, c1, s1, c2, s2, ab);
        rotb(rab, c1, s1, c2, s2, bb);
        if (bnd) {
            // lane m: the derivative along the cell's value m (m < 5), the inflow
            // state's m - 5 (an outflow face does not read it) or the outflow
            // state's m - 10 (an inflow face does not); the lanes of a point
            // repeat everything up to here
            const int code = -cR, e = m - NV;
            const bool fs = bcbar && (code == 1 || code == 2 || code == 6) && e < 2 * NV && (e < NV ? code != 2 : code != 1);
            double d = 0.0;
            if (m < NV || fs) {
                Dual A[NV], G[NV], fin[NV], fo[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    A[v] = Dual{a[v], m == v ? 1.0 : 0.0};
                    fin[v] = Dual{p.bc.inflow[v], e == v ? 1.0 : 0.0};
                    fo[v] = Dual{p.bc.outflow[v], e == NV + v ? 1.0 : 0.0};
                }
                ghost_state(code, p.bc.boundtype, p.gamma, A, c1, s1, c2, s2, fin, fo, G);
#pragma unroll
                for (int v = 0; v < NV; ++v) d += bb[v] * G[v].d;
            }
            if (m < NV) {
                double am = ab[0];
#pragma unroll
                for (int v = 1; v < NV; ++v) am = m == v ? ab[v] : am;
                ubf[oL + m] = am + d;
            } else {
                bcd = d;
            }
        } else {
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                ubf[oR + v] = bb[v];
                ubf[oL + v] = ab[v];
            }
        }
    };
    if (f < p.nface) point();
    if constexpr (BND) {
        if (!bcbar) return;
        __shared__ double sh[256 / WAVE][BLANES];
        bcd += __shfl_xor(bcd, 16, WAVE);
        bcd += __shfl_xor(bcd, 32, WAVE);
        if ((threadIdx.x & (WAVE - 1)) < BLANES) sh[threadIdx.x / WAVE][m] = bcd;
        __syncthreads();
        if (threadIdx.x < 2 * NV) {
            double x = 0.0;
            for (int wv = 0; wv < 256 / WAVE; ++wv) x += sh[wv][NV + threadIdx.x];
            if (x != 0.0) atomic_add_f64(&bcbar[threadIdx.x], x);
        }
    }
}

// EDGES: the first nbblock blocks take the boundary faces
template <typename R, bool EDGES>
__global__ __launch_bounds__(256) void k_flux_vjp(FluxParams<R> p, const int32_t *bfaces, int nbface, int nbblock,
                                                  const double *lam, double *ubf, double *bcbar) {
    if constexpr (EDGES) {
        if ((int)blockIdx.x < nbblock) {
            flux_vjp_block<R, true>(p, blockIdx.x, bfaces, nbface, lam, ubf, bcbar);
            return;
        }
    }
    flux_vjp_block<R, false>(p, blockIdx.x - nbblock, bfaces, nbface, lam, ubf, bcbar);
}

// Geometry cotangents of one residual product lam . R(U) on the face side
// (FP64): per face the area (garea), the unit outward normal (gnrm) and the
// cells' 1/TOTVOLUME (govol, through the update term dt R / V that pairs
// with lam).  The face sum S = area sum_q w_q <rotf(Fb), H_q> is linear in
// the area.  It depends on the rotation only through the normal (HLLC and
// the ghost states are invariant under turning the tangents), so its
// normal derivative is taken along two rotations of the whole frame: about
// t1 (n -> n + phi t2, t2 -> t2 - phi n) and about t2 (n -> n + psi t1,
// t1 -> t1 - psi n), each with a dual number; gnrm = area (dS/dphi t2 +
// dS/dpsi t1), the tangential gradient, free of the angles' singularity at
// n = +-z.  Every output is accumulated (+=) over the calls.
template <bool BND>
__global__ __launch_bounds__(256) void k_flux_geom(FluxParams<double> p, const double *lam, const double *ovol,
                                                  double *garea, double *gnrm, double *govol) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= p.nface) return;
    const int cL = p.fcell[2 * f], cR = p.fcell[2 * f + 1];
    if ((cR < 0) != BND) return;
    const int s0 = p.fslot[2 * f], sR = p.fslot[2 * f + 1];
    const int sL = s0 & 255;
    const bool tri = (s0 >> 8) & 1;
    const int nq = tri ? p.qpt : p.qpq;
    const double *w = tri ? p.wt : p.wq;
    const double c1 = p.frot[4 * f], s1 = p.frot[4 * f + 1], c2 = p.frot[4 * f + 2], s2 = p.frot[4 * f + 3];
    const double area = p.farea[f];
    const double nv[3] = {c1 * s2, s1 * s2, c2}, t1[3] = {c1 * c2, s1 * c2, -s2}, t2[3] = {-s1, c1, 0.0};
    double uL[NV], uR[NV], Fb[NV], fbr[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        uL[v] = p.U[(size_t)cL * NV + v];
        uR[v] = BND ? 0.0 : p.U[(size_t)cR * NV + v];
        Fb[v] = lam[(size_t)cL * NV + v] - (BND ? 0.0 : lam[(size_t)cR * NV + v]);
    }
    rotf(Fb, c1, s1, c2, s2, fbr);
    const double *ulL = p.uleft + ((size_t)cL * p.nf + sL) * p.nqm * NV;
    const double *ulR = p.uleft + ((size_t)(BND ? cL : cR) * p.nf + (BND ? sL : sR)) * p.nqm * NV;
    double S = 0.0, dphi = 0.0, dpsi = 0.0, F[NV] = {0, 0, 0, 0, 0};
    for (int q = 0; q < nq; ++q) {
        double a[NV], b[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            a[v] = uL[v] + ulL[q * NV + v];
            b[v] = uR[v] + ulR[q * NV + v];
        }
        if (BND) ghost_state(-cR, p.bc.boundtype, p.gamma, a, c1, s1, c2, s2, p.bc.inflow, p.bc.outflow, b);
        double la[NV], ra[NV], h[NV], hb[NV];
        rotf(a, c1, s1, c2, s2, la);
        rotf(b, c1, s1, c2, s2, ra);
        hllc64(p.gamma, la, ra, h);
        rotb(h, c1, s1, c2, s2, hb);
        double sq = 0.0;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            sq += fbr[v] * h[v];
            F[v] += w[q] * hb[v];
        }
        S += w[q] * sq;
#pragma unroll 1
        for (int seed = 0; seed < 2; ++seed) {
            // seed 0: about t1 (n moves along t2); seed 1: about t2 (n moves along t1)
            VectorFrame<Dual> fr;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                fr.n[d] = Dual{nv[d], seed == 0 ? t2[d] : t1[d]};
                fr.t1[d] = Dual{t1[d], seed == 0 ? 0.0 : -nv[d]};
                fr.t2[d] = Dual{t2[d], seed == 0 ? -nv[d] : 0.0};
            }
            Dual A[NV], B[NV], FB[NV], LA[NV], RA[NV], H[NV], FR[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                A[v] = Dual{a[v], 0.0};
                B[v] = Dual{b[v], 0.0};
                FB[v] = Dual{Fb[v], 0.0};
            }
            if (BND) ghost_state_fr(-cR, p.bc.boundtype, p.gamma, A, fr, p.bc.inflow, p.bc.outflow, B);
            fr.fwd(A, LA);
            fr.fwd(B, RA);
            hllc_t<Dual>(p.gamma, LA, RA, H);
            fr.fwd(FB, FR);
            double d = 0.0;
#pragma unroll
            for (int v = 0; v < NV; ++v) d += (FR[v] * H[v]).d;
            (seed == 0 ? dphi : dpsi) += w[q] * d;
        }
    }
    garea[f] += S;
#pragma unroll
    for (int d = 0; d < 3; ++d) gnrm[(size_t)f * 3 + d] += area * (dphi * t2[d] + dpsi * t1[d]);
    // R_L holds +area F, R_R -area F
    double eL = 0.0, eR = 0.0;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        eL += lam[(size_t)cL * NV + v] * F[v];
        if (!BND) eR += lam[(size_t)cR * NV + v] * F[v];
    }
    atomic_add_f64(&govol[cL], area * eL / ovol[cL]);
    if (!BND) atomic_add_f64(&govol[cR], -area * eR / ovol[cR]);
}

// the state [ncell][5] as 64-byte records [ncell][8] (the last three zero):
// the first reconstruction of a march; the later ones find the records that
// k_update wrote
__global__ __launch_bounds__(256) void k_pack64(size_t n64, const double *U, double *U64) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n64) return;
    const size_t i = e / 8, v = e - i * 8;
    U64[e] = v < NV ? U[i * NV + v] : 0.0;
}

__global__ void k_zero_f64(double *p, size_t n) {
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x)
        p[e] = 0.0;
}

// Reverse of one Shu-Osher stage (the three stage updates are affine in
// the stage state and linear in R):
//   stage 3: u = 1/3 u0 + 2/3 u2 - 2/3 dt R(u2)/V   -> u2_bar, u0_bar
//   stage 2: u2 = 3/4 u0 + 1/4 u1 - 1/4 dt R(u1)/V  -> u1_bar, u0_bar
//   stage 1: u1 = u0 - dt R(u0)/V                    -> u0_bar
// w = -c dt ybar / V is the cotangent handed to the residual product of the
// stage whose output cotangent is ybar.  k_rk3_adj_w forms it for the last
// stage; k_rk3_adj_stage then adds a ybar and the product to the cotangents of
// a stage's inputs, and forms w for the stage before it.  Both clear the
// product's sum for the stage that follows: four launches of 4-5 us a stage
// (clear, w, inputs, and a copy of u0_bar a step) are one.
__global__ void k_rk3_adj_w(int ncell, const double *ybar, const double *ovol, const double *dt, double c, double *w,
                            double *jt) {
    const size_t n = (size_t)ncell * NV;
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
        w[e] = -(c * *dt) * ybar[e] * ovol[e / NV];
        jt[e] = 0.0;
    }
}
// the cotangents of one stage's inputs from its output cotangent y and the
// residual product jt = (dR/du)^T w:
//   stage 3: x = 2/3 y + jt (x = u2_bar), u0_bar = 1/3 y
//   stage 2: x = 1/4 y + jt (x = u1_bar), u0_bar += 3/4 y   (x may alias y)
//   stage 1: a = u0_bar + y + jt (the step's input)
// and from them w of the stage before (dt null: there is none)
__global__ void k_rk3_adj_stage(int ncell, int stage, const double *y, double *jt, double *x, double *u0, double *a,
                                const double *ovol, const double *dt, double c, double *w) {
    const size_t n = (size_t)ncell * NV;
    const double to4 = 3.0 / 4.0, oo4 = 1.0 / 4.0, to3 = 2.0 / 3.0, oo3 = 1.0 / 3.0;
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
        const double ye = y[e], je = jt[e];
        double yn;  // the output cotangent of the stage before
        if (stage == 3) {
            yn = to3 * ye + je;
            x[e] = yn;
            u0[e] = oo3 * ye;
        } else if (stage == 2) {
            u0[e] += to4 * ye;
            yn = oo4 * ye + je;
            x[e] = yn;
        } else {
            yn = u0[e] + (ye + je);
            a[e] = yn;
        }
        if (dt) {
            w[e] = -(c * *dt) * yn * ovol[e / NV];
            jt[e] = 0.0;
        }
    }
}

__global__ void k_fill_u64(unsigned long long *p, unsigned long long v) { p[threadIdx.x] = v; }
// the time and the fixed step of a march
__global__ void k_set2(double *p, double a, double *q, double b) {
    if (threadIdx.x == 0) {
        *p = a;
        *q = b;
    }
}
// What a call hands back to the host, written straight into pinned host memory
// (one launch and one wait where a clear, two sums and three copies through
// pageable memory held the stream for 100 us after a march): the sums of the
// blocks' troubled-cell marks, whether u holds a non-finite value (nu = 0: not
// looked at), and the time.
__global__ __launch_bounds__(256) void k_finish(const int *marks, int n, const double *u, size_t nu, const double *t,
                                                HostResult *out) {
    __shared__ int sh[3][256 / WAVE];
    int a = 0, b = 0, bad = 0;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256) {
        a += marks[e] & 65535;
        b += marks[e] >> 16;
    }
    for (size_t e = blockIdx.x * 256 + threadIdx.x; e < nu; e += gridDim.x * 256)
        if (!isfinite(u[e])) bad = 1;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, WAVE);
        b += __shfl_xor(b, o, WAVE);
        bad |= __shfl_xor(bad, o, WAVE);
    }
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        sh[0][threadIdx.x / WAVE] = a;
        sh[1][threadIdx.x / WAVE] = b;
        sh[2][threadIdx.x / WAVE] = bad;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        int v = 0;
        for (int w = 0; w < 256 / WAVE; ++w) v += sh[threadIdx.x][w];
        out->part[blockIdx.x][threadIdx.x] = v;
    }
    if (t && blockIdx.x == 0 && threadIdx.x == 0) out->t = *t;
}

// Per-cell 5-vectors across the ABI: the caller's cell o = perm[c] (o = c
// without a permutation) in the caller's layout <-> the library's cell c in
// AoS.  src and dst never alias.
__global__ __launch_bounds__(256) void k_cells_in(int ncell, const int32_t *perm, const double *src, int layout,
                                                  double *dst) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    const size_t o = perm ? (size_t)perm[c] : (size_t)c;
#pragma unroll
    for (int v = 0; v < NV; ++v)
        dst[(size_t)c * NV + v] = layout == UCNS_LAYOUT_AOS ? src[o * NV + v] : src[(size_t)v * ncell + o];
}
__global__ __launch_bounds__(256) void k_cells_out(int ncell, const int32_t *perm, const double *src, int layout,
                                                   double *dst) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    const size_t o = perm ? (size_t)perm[c] : (size_t)c;
#pragma unroll
    for (int v = 0; v < NV; ++v)
        dst[layout == UCNS_LAYOUT_AOS ? o * NV + v : (size_t)v * ncell + o] = src[(size_t)c * NV + v];
}

// [cells][ts_in][imax][ideg] (FP64, ABI) -> [cells][imax][ts_out][ideg] (R)
template <typename R>
__global__ void k_relayout_p(const double *src, R *dst, int ncells, int ts_in, int ts_out, int imax, int ideg) {
    const size_t per_out = (size_t)imax * ts_out * ideg;
    const size_t total = per_out * ncells;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
        const size_t c = e / per_out;
        size_t r = e % per_out;
        const int k = (int)(r % ideg);
        r /= ideg;
        const int s = (int)(r % ts_out);
        const int j = (int)(r / ts_out);
        dst[e] = (R)src[((c * ts_in + s) * imax + j) * ideg + k];
    }
}

template <typename T>
int dalloc(ucns_ctx *ctx, T **p, size_t n);

// Scratch of ucns_residual_noalloc: its face fluxes (behind a reserved head
// of 256 bytes), in a file-scope device array that every GPU the
// library runs on holds from the library's first use on it until the process
// ends, so that the call allocates nothing.  In host code the array's name is
// a stand-in, not a device address: scratch_on() takes each device's own
// address once, with hipGetSymbolAddress, and only that address is used.
constexpr size_t UCNS_SCRATCH_BYTES = (size_t)256 << 20;  // 256 MiB: 6.7 M faces
constexpr size_t UCNS_SCRATCH_HEAD = 256;                  // reserved

}  // namespace

static __device__ __align__(256) unsigned char scratch[UCNS_SCRATCH_BYTES];

namespace {
std::mutex g_scratch_mu;
void *g_scratch_ptr[256] = {};

// the address of `scratch` on the current device (taken once per device)
int scratch_on(int device, void **out, std::string &err) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (device < 0 || device >= 256) {
        err = "device ordinal out of range for the scratch table";
        return UCNS_EUNSUPPORTED;
    }
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
            return UCNS_EHIP;
        }
        g_scratch_ptr[device] = p;
    }
    *out = g_scratch_ptr[device];
    return UCNS_OK;
}
}  // namespace

// ---------------------------------------------------------------------------
struct ucns_ctx {
    std::string err;
    int device = 0;
    hipStream_t stream = nullptr;
    // sizes
    int ncell = 0, nf = 0, nqm = 0, nface = 0;
    int precision = UCNS_FP64, iweno = 1, ideg = 0, nnb = 0, imax = 0, ts_abi = 0, ts = 0;
    int qpq = 0, qpt = 0, nf_abi = 0, nqm_abi = 0, index_base = 0;
    double gamma = 1.4, lwci1 = 1.0, eps = 1e-11;
    bool have_prestore = false, have_state = false;
    bool tiled = false;  // WENO-4 lane-per-stencil kernel with the tiled layout
    int smode = 0;      // stencils per cell where the pseudo-inverses are a row stream (0: tiled rows)
    bool bmode = false;  // reconstruction by the block kernels (recon_block.hip)
    bool needs_bc = false, have_bc = false;  // boundary codes 1/2/6 present; ucns_set_boundary called
    double *bface = nullptr;  // [nface][10] per-face INFLOW(), OUTFLOW() states (ucns_set_boundary_faces)
    int nbface = 0;             // faces with a ghost state (codes 1/2/3/4/6)
    int32_t *bfaces = nullptr;  // [nbface] their ids
    ucns_boundary_v1 bc{};
    int ntile = 0;
    // mesh (device)
    int32_t *cinfo = nullptr, *cnb = nullptr, *cface = nullptr, *fcell = nullptr, *fslot = nullptr;
    double *frot = nullptr, *farea = nullptr, *ovol = nullptr, *minedge = nullptr;
    double *wquad = nullptr;  // [128] face weights: [0, 64) quadrilateral, [64, 128) triangle
    std::vector<int32_t> h_cinfo_base;  // ifca + face types (admis/full added at upload)
    // cell order: library cell c is the caller's cell h_perm[c] (both empty:
    // the caller's order); h_iperm is the inverse
    int cell_order = UCNS_ORDER_CALLER;
    std::vector<int32_t> h_perm, h_iperm;
    int32_t *perm = nullptr;    // device copy of h_perm, or null
    double *stage = nullptr;    // [ncell][5] staging buffer of host transfers
    void *scratch = nullptr;    // this device's address of the static scratch array
    // CWENO (ees 5): scheme switches, the caller's low-order data by library
    // cell (ucns_upload_cweno), and on the device the sectors' packed
    // indicators and the means' differences mbar - mbar_c
    int ees = 0, wenoz = 0, ideg2 = 0, imax2 = 0;
    // characteristic WENO (wenwrt 2): per cell face the neighbour or -(boundary
    // code), and the cell's own face angles' cosines and sines
    int wenwrt = 1;
    int32_t *chnb = nullptr;
    double *chang = nullptr;
    bool have_cweno = false;
    std::vector<double> h_cwP, h_cwB, h_cwIB;
    void *Bc = nullptr, *dmb = nullptr;
    // CWENO at WENO-5 (its layouts: Cweno5Params): the sectors' low-order
    // pseudo-inverses and members
    void *Pc = nullptr;
    int32_t *nbc = nullptr;
    bool cw_cell = false;
    // library options of the scheme
    int kernels = UCNS_KERNELS_AUTO;
    int adj_keep_stages = 0;
    double adj_keep_gib = 64.0;
    // prestore (device)
    int32_t *nbr = nullptr;
    void *P = nullptr, *B = nullptr, *mbar = nullptr, *qp = nullptr, *uleft = nullptr;
    unsigned char *rows = nullptr;  // row stream of the DMA reconstruction kernels
    double *u64 = nullptr;          // [ncell][8] the state in 64-byte records, for their gathers
    long long tile_bytes = 0;
    // state (device)
    double *U3 = nullptr;      // second stage state of marches on k_flux_update
    int4 *fadj = nullptr;      // face records by cell of k_flux_update (null: it does not run)
    double *U = nullptr, *U2 = nullptr, *fflux = nullptr, *rhs = nullptr, *t = nullptr, *dtfix = nullptr;
    unsigned long long *dtv = nullptr;  // [2][DT_SLOTS * DT_STRIDE] ping-pong dt slots
    int *marks = nullptr;          // troubled cells per reconstruction block
    HostResult *result = nullptr;  // pinned host memory, written by k_finish
    int nmark = 0;
    // adjoint (allocated on first use): face-point cotangents, state-sized
    // work arrays, the free-stream cotangent, stage checkpoints and step dts
    double *adj_ubf = nullptr, *adj_lam = nullptr, *adj_ubar = nullptr, *adj_x = nullptr, *adj_a = nullptr;
    double *adj_u0 = nullptr, *adj_bc = nullptr, *ckpt = nullptr, *dts = nullptr;
    void *adj_g = nullptr;  // stencil coefficients, indicators, weights of the row-stream reconstruction (R)
    double *adj_gb = nullptr;  // stencil-coefficient cotangents handed to the row stream, [ntile][ideg*5][8 ts]
    // the tiles' distinct stencil members (ensure_members): for the block
    // reconstruction kernels and for the residual product's scatter
    uint16_t *mem_slot = nullptr;                      // [ntile][imax][8 ts] table row of each member entry
    int32_t *mem_uq = nullptr, *mem_count = nullptr;   // [ntile][uq_cap], [ntile]
    int uq_cap = UCNS_TILE_UQ;                         // member-table rows per tile (tile_uq(ts, imax))
    int64_t *adj_toff = nullptr, *adj_off = nullptr;  // table rows per tile, CSR offsets by cell
    int32_t *adj_ent = nullptr;                       // CSR entries: table rows (fewer than 2^31)
    double *adj_tab = nullptr;                          // [rows][5] member tables
    bool adj_g_on = false;  // the next tiled reconstruction stores them
    int *adj_flags = nullptr;  // [ncell] its MUSCL / first-order flags
    bool adj_ready = false;  // every adjoint buffer and member table is in place
    int fail_alloc_in = 0;   // > 0: the fail_alloc_in-th device allocation from now fails (ucns_debug_fail_alloc)
    size_t ckpt_steps = 0;
    // the last stages of a march keep their forward reconstruction for the
    // reverse sweep: face values, and where the product reads them (adj_stores)
    // the stencil coefficients, indicators, weights (as adj_g) and flags
    std::vector<void *> keep_ul, keep_g;
    std::vector<int *> keep_f;
    // geometry cotangents of ucns_rk3_adjoint_geometry (device, FP64, live
    // during that call only): pseudo-inverses, indicators, basis means, face
    // points (k_recon_vjp), face areas, face normals, 1/TOTVOLUME (k_flux_geom)
    double *geo_P = nullptr, *geo_B = nullptr, *geo_M = nullptr, *geo_Q = nullptr;
    double *geo_area = nullptr, *geo_nrm = nullptr, *geo_ovol = nullptr;
    bool geo_on = false;
    // host copies for mapping them back to the caller's arrays: the faces'
    // owner cell and slot, 1/TOTVOLUME and VOLUME(1,1) by library cell
    std::vector<int32_t> h_fcell, h_fslot;
    std::vector<double> h_ovol, h_vol11;
    // stats
    bool timing = false;
    hipEvent_t ev[8] = {};
    ucns_stats_v1 st{};
};

namespace {

template <typename T>
int dalloc(ucns_ctx *ctx, T **p, size_t n) {
    if (ctx->fail_alloc_in > 0 && --ctx->fail_alloc_in == 0) {
        *p = nullptr;
        ctx->err = "device allocation of " + std::to_string(n * sizeof(T)) + " bytes failed (injected)";
        return UCNS_ENOMEM;
    }
    hipError_t e = hipMalloc((void **)p, std::max<size_t>(n, 1) * sizeof(T));
    if (e != hipSuccess) {
        ctx->err = std::string("hipMalloc(") + std::to_string(n * sizeof(T)) + " bytes): " + hipGetErrorString(e);
        return e == hipErrorOutOfMemory ? UCNS_ENOMEM : UCNS_EHIP;
    }
    return UCNS_OK;
}

template <typename T>
void dfree(T *&p) {
    if (p) (void)hipFree((void *)p);
    p = nullptr;
}

int per_xcd(int ncell) { return (ncell + NXCD - 1) / NXCD; }

template <typename R>
LsqView<R> lsq_view(const ucns_ctx *ctx) {
    LsqView<R> L{};
    L.mode = ctx->smode ? 2 : ctx->tiled ? 1 : 0;
    L.ts = ctx->ts;
    L.tp = 8 * ctx->ts;
    L.imax = ctx->imax;
    L.ideg = ctx->ideg;
    L.depth = stream_depth(sizeof(R) == 4, ctx->ts);
    L.pb = ctx->ideg * L.tp * (int)sizeof(R);
    L.rd = L.pb + L.tp * 4;
    L.hd = L.depth * L.tp * 4;
    L.tile_bytes = ctx->tile_bytes;
    L.nbr = ctx->nbr;
    L.P = (const R *)ctx->P;
    L.rows = ctx->rows;
    return L;
}

// kernel selection by (precision, ideg, imax); packed: the last update wrote
// the state's 64-byte records
template <typename R>
int launch_recon_t(ucns_ctx *ctx, bool packed = false) {
    ReconParams<R> p{};
    p.ncell = ctx->ncell;
    p.nf = ctx->nf;
    p.nqm = ctx->nqm;
    p.ts = ctx->ts;
    p.per_xcd = per_xcd(ctx->ncell);
    p.qpq = ctx->qpq;
    p.qpt = ctx->qpt;
    p.gamma = ctx->gamma;
    p.lwci1 = ctx->lwci1;
    p.eps = ctx->eps;
    p.U = ctx->U;
    p.nbr = ctx->nbr;
    p.P = (const R *)ctx->P;
    p.B = (const R *)ctx->B;
    p.mbar = (const R *)ctx->mbar;
    p.qp = (const R *)ctx->qp;
    p.cinfo = ctx->cinfo;
    p.cnb = ctx->cnb;
    p.uleft = (R *)ctx->uleft;
    p.marks = ctx->marks;
    p.chnb = ctx->chnb;
    p.chang = ctx->chang;
    p.bc = ctx->bc;
    p.cface = ctx->cface;
    p.bface = ctx->bface;
    if (ctx->bmode) {
        const LsqView<R> L = lsq_view<R>(ctx);
        ReconBParams<R> w{};
        w.ncell = ctx->ncell;
        w.ntile = ctx->ntile;
        w.tiles_per_xcd = (ctx->ntile + NXCD - 1) / NXCD;
        w.nf = ctx->nf;
        w.nqm = ctx->nqm;
        w.qpq = ctx->qpq;
        w.qpt = ctx->qpt;
        w.gamma = ctx->gamma;
        w.lwci1 = ctx->lwci1;
        w.eps = ctx->eps;
        w.U = ctx->U;
        if (ctx->smode) {
            w.rows = ctx->rows;
            w.tile_bytes = ctx->tile_bytes;
            w.hd = L.hd;
            w.rd = L.rd;
            w.depth = L.depth;
        } else {
            w.rows = (const unsigned char *)ctx->P;
            w.rd = L.pb;
            w.tile_bytes = (long long)ctx->imax * L.pb;
            w.nbr = ctx->nbr;
        }
        w.imax = ctx->imax;
        w.uq_cap = ctx->uq_cap;
        w.uq = ctx->mem_uq;
        w.ucount = ctx->mem_count;
        w.slot = ctx->mem_slot;
        w.B = (const R *)ctx->B;
        w.mbar = (const R *)ctx->mbar;
        w.qp = (const R *)ctx->qp;
        w.cinfo = ctx->cinfo;
        w.cnb = ctx->cnb;
        w.uleft = (R *)ctx->uleft;
        w.marks = ctx->marks;
        w.gstore = ctx->adj_g_on ? (R *)ctx->adj_g : nullptr;
        w.fstore = ctx->adj_g_on ? ctx->adj_flags : nullptr;
        w.chnb = ctx->chnb;
        w.chang = ctx->chang;
        w.bc = ctx->bc;
        w.cface = ctx->cface;
        w.bface = ctx->bface;
        launch_recon_block(w, ctx->ideg, ctx->ts, ctx->wenwrt == 2, ctx->stream);
        return UCNS_OK;
    }
    if (ctx->tiled) {
        ReconWParams<R> w{};
        w.ncell = ctx->ncell;
        w.ntile = ctx->ntile;
        w.tiles_per_xcd = (ctx->ntile + NXCD - 1) / NXCD;
        w.ts = ctx->ts;
        w.nf = ctx->nf;
        w.nqm = ctx->nqm;
        w.qpq = ctx->qpq;
        w.qpt = ctx->qpt;
        w.gamma = ctx->gamma;
        w.lwci1 = ctx->lwci1;
        w.eps = ctx->eps;
        w.U = ctx->U;
        w.nbr = ctx->nbr;
        w.P = (const R *)ctx->P;
        w.B = (const R *)ctx->B;
        w.mbar = (const R *)ctx->mbar;
        w.qp = (const R *)ctx->qp;
        w.cinfo = ctx->cinfo;
        w.cnb = ctx->cnb;
        w.uleft = (R *)ctx->uleft;
        w.marks = ctx->marks;
        const dim3 grid(w.tiles_per_xcd * NXCD), block(WAVE);
        w.stream = ctx->rows;
        w.tile_bytes = ctx->tile_bytes;
        if (ctx->smode) {
            // the row-stream kernels gather the member states from 64-byte records
            const size_t n64 = (size_t)ctx->ncell * 8;
            if (!packed)
                hipLaunchKernelGGL(k_pack64, dim3((unsigned)((n64 + 255) / 256)), dim3(256), 0, ctx->stream, n64,
                                   ctx->U, ctx->u64);
            w.U64 = ctx->u64;
        }
        w.gstore = ctx->adj_g_on ? (R *)ctx->adj_g : nullptr;
        w.fstore = ctx->adj_g_on ? ctx->adj_flags : nullptr;
        if (ctx->ees == 5) {
            w.Bc = (const R *)ctx->Bc;
            w.dmb = (const R *)ctx->dmb;
            w.wenoz = ctx->wenoz;
        }
        launch_recon_tiled(w, ctx->ideg, ctx->smode, ctx->ees == 5, ctx->stream);
        return UCNS_OK;
    }
    if (ctx->iweno == -1) {
        launch_recon_muscl(p, ctx->stream);
        return UCNS_OK;
    }
    const dim3 grid(p.per_xcd * NXCD), block(WAVE);
    if (ctx->wenwrt == 2) {
        // WENO-5, and face rules of more points than the tiled kernels hold
        if (ctx->ideg == 34 && ctx->imax == 69)
            hipLaunchKernelGGL((k_recon<R, 34, 69, 7, true>), grid, block, 0, ctx->stream, p);
        else if (ctx->ideg == 19 && ctx->imax == 39)
            hipLaunchKernelGGL((k_recon<R, 19, 39, 7, true>), grid, block, 0, ctx->stream, p);
        else if (ctx->ideg == 9 && ctx->imax == 19)
            hipLaunchKernelGGL((k_recon<R, 9, 19, 7, true>), grid, block, 0, ctx->stream, p);
        else {
            ctx->err = "no characteristic reconstruction kernel for idegfree=" + std::to_string(ctx->ideg);
            return UCNS_EUNSUPPORTED;
        }
        return UCNS_OK;
    }
    if (ctx->cw_cell) {
        if (ctx->ideg == 34 && ctx->imax == 69 && ctx->ideg2 == 9 && ctx->imax2 == 19) {
            Cweno5Params<R> w{};
            w.ncell = ctx->ncell;
            w.ntile = ctx->ntile;
            w.tiles_per_xcd = (ctx->ntile + NXCD - 1) / NXCD;
            w.ts = ctx->ts;
            w.nf = ctx->nf;
            w.nqm = ctx->nqm;
            w.qpq = ctx->qpq;
            w.qpt = ctx->qpt;
            w.wenoz = ctx->wenoz;
            w.gamma = ctx->gamma;
            w.lwci1 = ctx->lwci1;
            w.eps = ctx->eps;
            w.U = ctx->U;
            w.nbr = ctx->nbr;
            w.nbc = ctx->nbc;
            w.P = (const R *)ctx->P;
            w.Pc = (const R *)ctx->Pc;
            w.B = (const R *)ctx->B;
            w.Bc = (const R *)ctx->Bc;
            w.dmb = (const R *)ctx->dmb;
            w.mbar = (const R *)ctx->mbar;
            w.qp = (const R *)ctx->qp;
            w.cinfo = ctx->cinfo;
            w.cnb = ctx->cnb;
            w.uleft = (R *)ctx->uleft;
            w.marks = ctx->marks;
            launch_recon_cweno5(w, ctx->stream);
            return UCNS_OK;
        }
        ctx->err = "no CWENO kernel for idegfree=" + std::to_string(ctx->ideg) + " idegfree2=" +
                   std::to_string(ctx->ideg2) + " imax2=" + std::to_string(ctx->imax2);
        return UCNS_EUNSUPPORTED;
    }
    if (ctx->ideg == 19 && ctx->imax == 39)
        hipLaunchKernelGGL((k_recon<R, 19, 39, 7>), grid, block, 0, ctx->stream, p);
    else if (ctx->ideg == 34 && ctx->imax == 69)
        hipLaunchKernelGGL((k_recon<R, 34, 69, 7>), grid, block, 0, ctx->stream, p);
    else if (ctx->ideg == 9 && ctx->imax == 19)
        hipLaunchKernelGGL((k_recon<R, 9, 19, 7>), grid, block, 0, ctx->stream, p);
    else if (ctx->ideg == 3 && ctx->imax == 8 && ctx->ts == 1)  // linear, unlimited where CHECKSOL lets it
        hipLaunchKernelGGL((k_recon<R, 3, 8, 1>), grid, block, 0, ctx->stream, p);
    else {
        ctx->err = "no reconstruction kernel for idegfree=" + std::to_string(ctx->ideg) +
                   " imax=" + std::to_string(ctx->imax);
        return UCNS_EUNSUPPORTED;
    }
    return UCNS_OK;
}

template <typename R>
FluxParams<R> flux_params(const ucns_ctx *ctx) {
    FluxParams<R> p{};
    p.nface = ctx->nface;
    p.nf = ctx->nf;
    p.nqm = ctx->nqm;
    p.qpq = ctx->qpq;
    p.qpt = ctx->qpt;
    p.gamma = ctx->gamma;
    p.fcell = ctx->fcell;
    p.fslot = ctx->fslot;
    p.frot = ctx->frot;
    p.farea = ctx->farea;
    p.U = ctx->U;
    p.uleft = (const R *)ctx->uleft;
    p.fflux = ctx->fflux;
    p.wq = ctx->wquad;
    p.wt = ctx->wquad + 64;
    p.bc = ctx->bc;
    p.bface = ctx->bface;
    return p;
}

template <typename R>
void launch_flux_t(ucns_ctx *ctx) {
    const FluxParams<R> p = flux_params<R>(ctx);
    // A thread per point where faces have several: 5,184 hexahedra faces 18.8 ->
    // 6.2 us, 31,000 channel faces 15.9 -> 9 us; marches on 169,000 (channel) to
    // 393,000 (tetrahedra) faces take the same time within 0.3% either way, on
    // 69,000 hexahedra in mixed precision 2.66 -> 2.62 ms.  From a million faces
    // on, where the face values no longer stay in the caches, a thread per face is
    // the faster one (1,080,000 channel faces 147 us against 185, mixed 91 against
    // 136).  Faces of one point gain nothing from it (5.7 against 7.9 us on 41,472).
    if (ctx->nqm > 1 && ctx->nface < 524288) {
        const int fpb = 256 / ctx->nqm;  // faces per block
        hipLaunchKernelGGL((k_flux_points<R>), dim3((ctx->nface + fpb - 1) / fpb), dim3(256), 0, ctx->stream, p);
    } else {
        hipLaunchKernelGGL((k_flux<R>), dim3((ctx->nface + 255) / 256), dim3(256), 0, ctx->stream, p);
    }
}

void tstart(ucns_ctx *ctx, int k) {
    if (ctx->timing) (void)hipEventRecord(ctx->ev[2 * k], ctx->stream);
}
void tstop(ucns_ctx *ctx, int k) {
    if (ctx->timing) (void)hipEventRecord(ctx->ev[2 * k + 1], ctx->stream);
}
void tcollect(ucns_ctx *ctx, int k, double *acc, int64_t *n) {
    if (!ctx->timing) return;
    float ms = 0;
    (void)hipEventSynchronize(ctx->ev[2 * k + 1]);
    if (hipEventElapsedTime(&ms, ctx->ev[2 * k], ctx->ev[2 * k + 1]) == hipSuccess) {
        *acc += ms;
        *n += 1;
    }
}

// reconstruction + face fluxes of the current state (ULEFT and face fluxes on device)
int residual_kernels(ucns_ctx *ctx, bool packed = false) {
    tstart(ctx, 0);
    int rc = ctx->precision == UCNS_MIXED ? launch_recon_t<float>(ctx, packed) : launch_recon_t<double>(ctx, packed);
    if (rc) return rc;
    tstop(ctx, 0);
    tcollect(ctx, 0, &ctx->st.ms_recon, &ctx->st.n_recon);
    tstart(ctx, 1);
    if (ctx->precision == UCNS_MIXED)
        launch_flux_t<float>(ctx);
    else
        launch_flux_t<double>(ctx);
    tstop(ctx, 1);
    tcollect(ctx, 1, &ctx->st.ms_flux, &ctx->st.n_flux);
    return UCNS_OK;
}

// more: another stage follows, so the row-stream kernels' records are written too
int update_kernel(ucns_ctx *ctx, int stage, const double *dt, bool dt_slots, unsigned long long *dt_next, double cfl,
                  double *rhs_out, bool more = false, double *copy = nullptr) {
    UpdateParams p{};
    p.ncell = ctx->ncell;
    p.nf = ctx->nf;
    p.stage = stage;
    p.cfl = cfl;
    p.gamma = ctx->gamma;
    p.cface = ctx->cface;
    p.fflux = ctx->fflux;
    p.ovol = ctx->ovol;
    p.minedge = ctx->minedge;
    p.U = ctx->U;
    p.U2 = ctx->U2;
    p.rhs_out = rhs_out;
    p.u64 = more && ctx->smode && !ctx->bmode ? ctx->u64 : nullptr;
    p.copy = copy;
    p.dt = dt;
    p.dt_slots = dt_slots;
    p.dt_next = dt_next;
    p.t = ctx->t;
    tstart(ctx, 2);
    hipLaunchKernelGGL(k_update, dim3((ctx->ncell + 255) / 256), dim3(256), 0, ctx->stream, p);
    tstop(ctx, 2);
    tcollect(ctx, 2, &ctx->st.ms_update, &ctx->st.n_update);
    return UCNS_OK;
}

// one stage of a march on one-point faces: reconstruction of the state src, then
// fluxes and update into dst (u0: u^n)
template <typename R>
int fused_stage_t(ucns_ctx *ctx, int stage, double *src, const double *u0, double *dst, const double *dt, bool dt_slots,
                  unsigned long long *dt_next, double cfl) {
    double *const state = ctx->U;
    ctx->U = src;
    const int rc = launch_recon_t<R>(ctx);
    const FluxParams<R> p = flux_params<R>(ctx);
    ctx->U = state;
    if (rc) return rc;
    UpdateParams u{};
    u.ncell = ctx->ncell;
    u.nf = ctx->nf;
    u.stage = stage;
    u.cfl = cfl;
    u.gamma = ctx->gamma;
    u.ovol = ctx->ovol;
    u.minedge = ctx->minedge;
    u.U = dst;
    u.U2 = const_cast<double *>(u0);
    u.dt = dt;
    u.dt_slots = dt_slots;
    u.dt_next = dt_next;
    u.t = ctx->t;
    hipLaunchKernelGGL((k_flux_update<R>), dim3((ctx->ncell + 31) / 32), dim3(256), 0, ctx->stream, p, u, ctx->fadj);
    return UCNS_OK;
}

// one SSP-RK3 step of such a march: the state's buffer is read by the first
// stage and written by the last
int fused_step(ucns_ctx *ctx, const double *dt, bool dt_slots, unsigned long long *dt_next, double cfl) {
    double *const u0 = ctx->U, *const dst[4] = {ctx->U, ctx->U2, ctx->U3, ctx->U};
    for (int stage = 1; stage <= 3; ++stage) {
        const int rc = ctx->precision == UCNS_MIXED
                           ? fused_stage_t<float>(ctx, stage, dst[stage - 1], u0, dst[stage], dt, dt_slots, dt_next, cfl)
                           : fused_stage_t<double>(ctx, stage, dst[stage - 1], u0, dst[stage], dt, dt_slots, dt_next,
                                                   cfl);
        if (rc) return rc;
    }
    return UCNS_OK;
}

int finish_blocks(const ucns_ctx *ctx, size_t nu) {
    return (int)std::min<size_t>(NPART, std::max<size_t>(1, (std::max<size_t>(ctx->nmark, nu) + 1023) / 1024));
}

// queues the result of a call; the stream is waited for before it is read
int queue_result(ucns_ctx *ctx, size_t nu, const double *t) {
    hipLaunchKernelGGL(k_finish, dim3(finish_blocks(ctx, nu)), dim3(256), 0, ctx->stream, ctx->marks, ctx->nmark,
                       ctx->U, nu, t, ctx->result);
    HIP_TRY(hipGetLastError());
    return UCNS_OK;
}

// the troubled-cell counts of the last reconstruction into the statistics;
// true if the state was found non-finite
bool read_result(ucns_ctx *ctx, size_t nu) {
    int64_t red = 0, fst = 0;
    int bad = 0;
    for (int b = 0; b < finish_blocks(ctx, nu); ++b) {
        red += ctx->result->part[b][0];
        fst += ctx->result->part[b][1];
        bad += ctx->result->part[b][2];
    }
    ctx->st.n_reduced_last = red;
    ctx->st.n_firstorder_last = fst;
    return bad != 0;
}

int collect_counts(ucns_ctx *ctx) {
    const int rc = queue_result(ctx, 0, nullptr);
    if (rc) return rc;
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    read_result(ctx, 0);
    return UCNS_OK;
}

int dt_kernel(ucns_ctx *ctx, double cfl, unsigned long long *out) {
    hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(DT_SLOTS * DT_STRIDE), 0, ctx->stream, out,
                       (unsigned long long)0x7FF0000000000000ULL);
    DtParams p{};
    p.ncell = ctx->ncell;
    p.cfl = cfl;
    p.gamma = ctx->gamma;
    p.U = ctx->U;
    p.minedge = ctx->minedge;
    p.dt_out = out;
    tstart(ctx, 3);
    hipLaunchKernelGGL(k_dt, dim3((ctx->ncell + 255) / 256), dim3(256), 0, ctx->stream, p);
    tstop(ctx, 3);
    tcollect(ctx, 3, &ctx->st.ms_dt, &ctx->st.n_dt);
    return UCNS_OK;
}

// ---- adjoint -----------------------------------------------------------
void release_members(ucns_ctx *ctx) {
    dfree(ctx->mem_slot);
    dfree(ctx->mem_uq);
    dfree(ctx->mem_count);
}

void release_adjoint(ucns_ctx *ctx) {
    dfree(ctx->adj_ubf);
    dfree(ctx->adj_lam);
    dfree(ctx->adj_ubar);
    dfree(ctx->adj_x);
    dfree(ctx->adj_a);
    dfree(ctx->adj_u0);
    dfree(ctx->adj_bc);
    dfree(ctx->ckpt);
    dfree(ctx->dts);
    if (ctx->adj_g) (void)hipFree(ctx->adj_g);
    ctx->adj_g = nullptr;
    dfree(ctx->adj_flags);
    dfree(ctx->adj_gb);
    dfree(ctx->adj_toff);
    dfree(ctx->adj_off);
    dfree(ctx->adj_ent);
    dfree(ctx->adj_tab);
    if (!ctx->bmode) release_members(ctx);  // the block kernels' are the upload's
    ctx->ckpt_steps = 0;
    ctx->adj_ready = false;
    for (void *q : ctx->keep_ul) (void)hipFree(q);
    for (void *q : ctx->keep_g) (void)hipFree(q);
    for (int *q : ctx->keep_f) (void)hipFree(q);
    ctx->keep_ul.clear();
    ctx->keep_g.clear();
    ctx->keep_f.clear();
}

template <typename R>
void launch_tile_members(ucns_ctx *ctx) {
    const LsqView<R> L = lsq_view<R>(ctx);
    const dim3 grid(ctx->ntile), block(WAVE);
    if (ctx->imax == 39)
        hipLaunchKernelGGL((k_tile_members<R, 39>), grid, block, 0, ctx->stream, L, ctx->ntile, ctx->ncell,
                           ctx->cinfo, ctx->uq_cap, ctx->mem_uq, ctx->mem_count, ctx->mem_slot);
    else if (ctx->imax == 19)
        hipLaunchKernelGGL((k_tile_members<R, 19>), grid, block, 0, ctx->stream, L, ctx->ntile, ctx->ncell,
                           ctx->cinfo, ctx->uq_cap, ctx->mem_uq, ctx->mem_count, ctx->mem_slot);
    else
        hipLaunchKernelGGL((k_tile_members<R, 8>), grid, block, 0, ctx->stream, L, ctx->ntile, ctx->ncell,
                           ctx->cinfo, ctx->uq_cap, ctx->mem_uq, ctx->mem_count, ctx->mem_slot);
}

// the tiles' distinct stencil members, once per upload; all of it or nothing
int ensure_members(ucns_ctx *ctx) {
    if (ctx->mem_slot) return UCNS_OK;
    ctx->uq_cap = tile_uq(ctx->ts, ctx->imax);
    int rc = dalloc(ctx, &ctx->mem_slot, (size_t)ctx->ntile * ctx->imax * 8 * ctx->ts);
    if (!rc) rc = dalloc(ctx, &ctx->mem_uq, (size_t)ctx->ntile * ctx->uq_cap);
    if (!rc) rc = dalloc(ctx, &ctx->mem_count, (size_t)ctx->ntile);
    if (rc) {
        release_members(ctx);
        return rc;
    }
    if (ctx->precision == UCNS_MIXED)
        launch_tile_members<float>(ctx);
    else
        launch_tile_members<double>(ctx);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        release_members(ctx);
        ctx->err = std::string("member tables: ") + hipGetErrorString(e);
        return UCNS_EHIP;
    }
    return UCNS_OK;
}

// frees a temporary device buffer on every exit of the scope
template <typename T>
struct DevTemp {
    T *p = nullptr;
    ~DevTemp() { dfree(p); }
};

// whether the residual product reads what the forward reconstruction stored
// (k_recon_vjp_s); the geometry product (k_recon_vjp) forms it again
bool adj_stores(const ucns_ctx *ctx) { return ctx->smode && !ctx->geo_on; }

// elements of adj_g: the coefficients, indicators and weights of every stencil
size_t adj_g_elems(const ucns_ctx *ctx) { return (size_t)ctx->ntile * (ctx->ideg + 2) * NV * 8 * ctx->ts; }

// the stored forward of one stage, and the coefficients' cotangents
int ensure_stored(ucns_ctx *ctx) {
    if (ctx->adj_gb) return UCNS_OK;
    int rc;
    if ((rc = dalloc(ctx, &ctx->adj_flags, (size_t)ctx->ncell))) return rc;
    if (ctx->precision == UCNS_MIXED)
        rc = dalloc(ctx, (float **)&ctx->adj_g, adj_g_elems(ctx));
    else
        rc = dalloc(ctx, (double **)&ctx->adj_g, adj_g_elems(ctx));
    if (rc) return rc;
    return dalloc(ctx, &ctx->adj_gb, (size_t)ctx->ntile * ctx->ideg * NV * 8 * ctx->ts);
}

int ensure_adjoint_steps(ucns_ctx *ctx) {
    const size_t n = (size_t)ctx->ncell * NV;
    int rc;
    if ((rc = dalloc(ctx, &ctx->adj_ubf, (size_t)ctx->ncell * ctx->nf * ctx->nqm * NV))) return rc;
    if ((rc = dalloc(ctx, &ctx->adj_lam, n))) return rc;
    if ((rc = dalloc(ctx, &ctx->adj_ubar, n))) return rc;
    if ((rc = dalloc(ctx, &ctx->adj_x, n))) return rc;
    if ((rc = dalloc(ctx, &ctx->adj_a, n))) return rc;
    if ((rc = dalloc(ctx, &ctx->adj_u0, n))) return rc;
    if ((rc = dalloc(ctx, &ctx->adj_bc, 2 * NV))) return rc;
    // the tiles' distinct stencil members (once per upload)
    if (ctx->ts <= 8 && (ctx->imax == 39 || ctx->imax == 19 || ctx->imax == 8)) {
        if ((rc = ensure_members(ctx))) return rc;
        // table rows per tile (prefix sums on the host: set-up only).  The
        // library stream is non-blocking: every host read of what its kernels
        // wrote waits for the stream first, and every clear is queued on it.
        const int nt = ctx->ntile, nc = ctx->ncell;
        std::vector<int32_t> uc(nt);
        HIP_TRY(hipMemcpyAsync(uc.data(), ctx->mem_count, nt * sizeof(int32_t), hipMemcpyDeviceToHost,
                               ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
        std::vector<int64_t> toff(nt + 1, 0);
        for (int t = 0; t < nt; ++t) toff[t + 1] = toff[t] + std::min(uc[t], ctx->uq_cap);
        const int64_t rows = toff[nt];
        if (rows >= ((int64_t)1 << 31)) {
            ctx->err = "member tables exceed 2^31 rows";
            return UCNS_EUNSUPPORTED;
        }
        if ((rc = dalloc(ctx, &ctx->adj_toff, (size_t)nt + 1))) return rc;
        if ((rc = dalloc(ctx, &ctx->adj_tab, (size_t)rows * NV))) return rc;
        if ((rc = dalloc(ctx, &ctx->adj_off, (size_t)nc + 1))) return rc;
        if ((rc = dalloc(ctx, &ctx->adj_ent, (size_t)std::max<int64_t>(rows, 1)))) return rc;
        HIP_TRY(hipMemcpyAsync(ctx->adj_toff, toff.data(), (nt + 1) * sizeof(int64_t), hipMemcpyHostToDevice,
                               ctx->stream));
        // CSR by cell: count, scan, fill
        DevTemp<int64_t> cnt_buf;
        if ((rc = dalloc(ctx, &cnt_buf.p, (size_t)nc))) return rc;
        int64_t *cnt = cnt_buf.p;
        HIP_TRY(hipMemsetAsync(cnt, 0, nc * sizeof(int64_t), ctx->stream));
        hipLaunchKernelGGL(k_adj_csr, dim3(nt), dim3(256), 0, ctx->stream, nt, ctx->uq_cap, ctx->mem_uq,
                           ctx->mem_count, ctx->adj_toff, cnt, (const int64_t *)nullptr, (int32_t *)nullptr);
        std::vector<int64_t> hc(nc), off(nc + 1, 0);
        HIP_TRY(hipMemcpyAsync(hc.data(), cnt, nc * sizeof(int64_t), hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
        for (int i = 0; i < nc; ++i) off[i + 1] = off[i] + hc[i];
        if (off[nc] != rows) {  // every table row belongs to exactly one cell
            ctx->err = "member-table index: " + std::to_string(off[nc]) + " entries for " + std::to_string(rows) +
                       " rows";
            return UCNS_EHIP;
        }
        HIP_TRY(hipMemcpyAsync(ctx->adj_off, off.data(), (nc + 1) * sizeof(int64_t), hipMemcpyHostToDevice,
                               ctx->stream));
        HIP_TRY(hipMemsetAsync(cnt, 0, nc * sizeof(int64_t), ctx->stream));
        hipLaunchKernelGGL(k_adj_csr, dim3(nt), dim3(256), 0, ctx->stream, nt, ctx->uq_cap, ctx->mem_uq,
                           ctx->mem_count, ctx->adj_toff, cnt, (const int64_t *)ctx->adj_off, ctx->adj_ent);
        HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    return UCNS_OK;
}

// The adjoint's buffers and member tables, set up on first use.  A context
// counts as set up only once every step has succeeded; a failed step frees
// what the earlier ones allocated, so the next call starts over and returns
// the error again instead of running kernels on missing buffers.
int ensure_adjoint(ucns_ctx *ctx) {
    if (ctx->ees == 5) {
        ctx->err = "the adjoint does not cover CWENO (ees 5)";
        return UCNS_EUNSUPPORTED;
    }
    if (ctx->ideg == 34) {
        ctx->err = "the adjoint covers idegfree 3, 9 and 19 (not WENO-5, idegfree 34)";
        return UCNS_EUNSUPPORTED;
    }
    if (ctx->wenwrt == 2) {
        ctx->err = "the adjoint does not cover characteristic reconstruction (wenwrt 2)";
        return UCNS_EUNSUPPORTED;
    }
    if (ctx->bface) {
        ctx->err = "the adjoint takes uniform boundary states (ucns_set_boundary), not per-face ones";
        return UCNS_EUNSUPPORTED;
    }
    int rc = UCNS_OK;
    if (!ctx->adj_ready) {
        release_adjoint(ctx);
        rc = ensure_adjoint_steps(ctx);
    }
    if (rc == UCNS_OK && adj_stores(ctx)) rc = ensure_stored(ctx);
    if (rc != UCNS_OK) {
        release_adjoint(ctx);
        return rc;
    }
    ctx->adj_ready = true;
    return UCNS_OK;
}

// the member tables of the last scatter into ubar
void adj_gather(ucns_ctx *ctx, double *ubar) {
    hipLaunchKernelGGL(k_adj_gather, dim3((ctx->ncell + 31) / 32), dim3(256), 0, ctx->stream, ctx->ncell,
                       ctx->adj_off, ctx->adj_ent, ctx->adj_tab, ubar);
}

void zero_dev(ucns_ctx *ctx, double *p, size_t n) {
    const int blocks = (int)std::min<size_t>(4096, (n + 255) / 256);
    hipLaunchKernelGGL(k_zero_f64, dim3(std::max(blocks, 1)), dim3(256), 0, ctx->stream, p, n);
}

// P^T g_bar of the last products (adj_gb) onto the row stream, into ubar
template <typename R>
void launch_scatter_t(ucns_ctx *ctx, double *ubar) {
    ReconWParams<R> w{};
    w.ncell = ctx->ncell;
    w.ntile = ctx->ntile;
    w.tiles_per_xcd = (ctx->ntile + NXCD - 1) / NXCD;
    w.ts = ctx->ts;
    w.cinfo = ctx->cinfo;
    w.stream = ctx->rows;
    w.tile_bytes = ctx->tile_bytes;
    w.gbs = ctx->adj_gb;
    w.ubar = ubar;
    w.slot = ctx->mem_slot;
    w.uq_cap = ctx->uq_cap;
    w.ucount = ctx->mem_count;
    w.toff = ctx->adj_toff;
    w.tab = ctx->adj_tab;
    launch_scatter(w, ctx->ideg, ctx->smode, ctx->stream);
}

// the forward reconstruction of the current state for a residual product:
// ULEFT, and in row-stream mode every stencil's coefficients, indicators,
// weights and the cell flags
template <typename R>
int vjp_recon_t(ucns_ctx *ctx) {
    ctx->adj_g_on = adj_stores(ctx);
    tstart(ctx, 3);
    const int rc = launch_recon_t<R>(ctx);
    tstop(ctx, 3);
    tcollect(ctx, 3, &ctx->st.ms_recon_adj, &ctx->st.n_recon_adj);
    ctx->adj_g_on = false;
    return rc;
}

// the products of one residual at the state of the last vjp_recon_t: ubar
// (zeroed here unless the caller did) = the flux product, the reconstruction product and, in
// row-stream mode, the scatter of P^T g_bar (adj_gb) through the member tables
template <typename R>
int vjp_products_t(ucns_ctx *ctx, const double *lam, double *ubar, double *bcbar, bool zeroed = false) {
    const int nfq = ctx->nf * ctx->nqm;
    if (ctx->ts > 8 || nfq > 56) {
        ctx->err = "the residual product needs at most 8 stencils and 56 face points per cell";
        return UCNS_EUNSUPPORTED;
    }
    if (!zeroed) zero_dev(ctx, ubar, (size_t)ctx->ncell * NV);
    FluxParams<R> fp{};
    fp.nface = ctx->nface;
    fp.nf = ctx->nf;
    fp.nqm = ctx->nqm;
    fp.qpq = ctx->qpq;
    fp.qpt = ctx->qpt;
    fp.gamma = ctx->gamma;
    fp.fcell = ctx->fcell;
    fp.fslot = ctx->fslot;
    fp.frot = ctx->frot;
    fp.farea = ctx->farea;
    fp.U = ctx->U;
    fp.uleft = (const R *)ctx->uleft;
    fp.fflux = nullptr;
    fp.wq = ctx->wquad;
    fp.wt = ctx->wquad + 64;
    fp.bc = ctx->bc;
    tstart(ctx, 1);
    const int nint = (int)(((size_t)ctx->nface * ctx->nqm + 255) / 256);
    const int nbblock = (int)(((size_t)ctx->nbface * ctx->nqm * BLANES + 255) / 256);
    if (ctx->nbface)
        hipLaunchKernelGGL((k_flux_vjp<R, true>), dim3(nbblock + nint), dim3(256), 0, ctx->stream, fp, ctx->bfaces,
                           ctx->nbface, nbblock, lam, ctx->adj_ubf, bcbar);
    else
        hipLaunchKernelGGL((k_flux_vjp<R, false>), dim3(nint), dim3(256), 0, ctx->stream, fp,
                           (const int32_t *)nullptr, 0, 0, lam, ctx->adj_ubf, bcbar);
    tstop(ctx, 1);
    tcollect(ctx, 1, &ctx->st.ms_flux_vjp, &ctx->st.n_flux_vjp);
    if constexpr (sizeof(R) == 8) {
        if (ctx->geo_on) {
            hipLaunchKernelGGL(k_flux_geom<false>, dim3((ctx->nface + 255) / 256), dim3(256), 0, ctx->stream, fp, lam,
                               ctx->ovol, ctx->geo_area, ctx->geo_nrm, ctx->geo_ovol);
            if (ctx->nbface)
                hipLaunchKernelGGL(k_flux_geom<true>, dim3((ctx->nface + 255) / 256), dim3(256), 0, ctx->stream, fp,
                                   lam, ctx->ovol, ctx->geo_area, ctx->geo_nrm, ctx->geo_ovol);
        }
    }
    VjpParams<R> vp{};
    vp.ncell = ctx->ncell;
    vp.ntile = ctx->ntile;
    vp.tiles_per_xcd = (ctx->ntile + NXCD - 1) / NXCD;
    vp.nf = ctx->nf;
    vp.nqm = ctx->nqm;
    vp.qpq = ctx->qpq;
    vp.qpt = ctx->qpt;
    vp.iweno = ctx->iweno;
    vp.gamma = ctx->gamma;
    vp.lwci1 = ctx->lwci1;
    vp.eps = ctx->eps;
    vp.U = ctx->U;
    vp.lsq = lsq_view<R>(ctx);
    vp.B = (const R *)ctx->B;
    vp.mbar = (const R *)ctx->mbar;
    vp.qp = (const R *)ctx->qp;
    vp.cinfo = ctx->cinfo;
    vp.cnb = ctx->cnb;
    vp.ubf = ctx->adj_ubf;
    vp.ubar = ubar;
    vp.gload = adj_stores(ctx) ? (const R *)ctx->adj_g : nullptr;
    vp.fload = ctx->adj_flags;
    vp.slot = ctx->mem_slot;
    vp.uq_cap = ctx->uq_cap;
    vp.uq = ctx->mem_uq;
    vp.ucount = ctx->mem_count;
    vp.gbout = adj_stores(ctx) ? ctx->adj_gb : nullptr;
    vp.toff = ctx->adj_toff;
    vp.tab = ctx->adj_tab;
    vp.gP = ctx->geo_P;
    vp.gB = ctx->geo_B;
    vp.gM = ctx->geo_M;
    vp.gQ = ctx->geo_Q;
    const dim3 grid(vp.tiles_per_xcd * NXCD), block(WAVE);
    const bool q3 = nfq <= 24;
    tstart(ctx, 0);
    bool geo_done = false;
    if constexpr (sizeof(R) == 8) {
        if (ctx->geo_on) {
            geo_done = true;
            if (ctx->ideg == 19 && ctx->imax == 39) {
                if (q3)
                    hipLaunchKernelGGL((k_recon_vjp<R, 19, 39, 3, true>), grid, block, 0, ctx->stream, vp);
                else
                    hipLaunchKernelGGL((k_recon_vjp<R, 19, 39, 7, true>), grid, block, 0, ctx->stream, vp);
            } else if (ctx->ideg == 9 && ctx->imax == 19) {
                if (q3)
                    hipLaunchKernelGGL((k_recon_vjp<R, 9, 19, 3, true>), grid, block, 0, ctx->stream, vp);
                else
                    hipLaunchKernelGGL((k_recon_vjp<R, 9, 19, 7, true>), grid, block, 0, ctx->stream, vp);
            } else if (ctx->ideg == 3 && ctx->imax == 8) {
                if (q3)
                    hipLaunchKernelGGL((k_recon_vjp<R, 3, 8, 3, true>), grid, block, 0, ctx->stream, vp);
                else
                    hipLaunchKernelGGL((k_recon_vjp<R, 3, 8, 7, true>), grid, block, 0, ctx->stream, vp);
            } else {
                ctx->err = "no geometry product for idegfree=" + std::to_string(ctx->ideg);
                return UCNS_EUNSUPPORTED;
            }
        }
    }
    if (geo_done) {
    } else if (ctx->smode) {
        // row-stream shapes: from the forward's stored coefficients; the
        // scatter follows on the row stream
        if (!vp.gload || !vp.fload) {
            ctx->err = "the row-stream product needs the forward's stored coefficients";
            return UCNS_EUNSUPPORTED;
        }
        if (ctx->ideg == 19 && ctx->smode == 5)
            hipLaunchKernelGGL((k_recon_vjp_s<R, 19, 3, 5>), grid, block, 0, ctx->stream, vp);
        else if (ctx->ideg == 19)
            hipLaunchKernelGGL((k_recon_vjp_s<R, 19, 7, 7>), grid, block, 0, ctx->stream, vp);
        else if (ctx->smode == 5)
            hipLaunchKernelGGL((k_recon_vjp_s<R, 9, 3, 5>), grid, block, 0, ctx->stream, vp);
        else if (ctx->smode == 6)
            hipLaunchKernelGGL((k_recon_vjp_s<R, 9, 3, 6>), grid, block, 0, ctx->stream, vp);
        else
            hipLaunchKernelGGL((k_recon_vjp_s<R, 9, 3, 7>), grid, block, 0, ctx->stream, vp);
    } else if (ctx->ideg == 19 && ctx->imax == 39) {
        if (q3)
            hipLaunchKernelGGL((k_recon_vjp<R, 19, 39, 3>), grid, block, 0, ctx->stream, vp);
        else
            hipLaunchKernelGGL((k_recon_vjp<R, 19, 39, 7>), grid, block, 0, ctx->stream, vp);
    } else if (ctx->ideg == 9 && ctx->imax == 19) {
        if (q3)
            hipLaunchKernelGGL((k_recon_vjp<R, 9, 19, 3>), grid, block, 0, ctx->stream, vp);
        else
            hipLaunchKernelGGL((k_recon_vjp<R, 9, 19, 7>), grid, block, 0, ctx->stream, vp);
    } else if (ctx->ideg == 3 && ctx->imax == 8) {
        if (q3)
            hipLaunchKernelGGL((k_recon_vjp<R, 3, 8, 3>), grid, block, 0, ctx->stream, vp);
        else
            hipLaunchKernelGGL((k_recon_vjp<R, 3, 8, 7>), grid, block, 0, ctx->stream, vp);
    } else {
        ctx->err = "no residual product for idegfree=" + std::to_string(ctx->ideg);
        return UCNS_EUNSUPPORTED;
    }
    if (ctx->smode && !geo_done) launch_scatter_t<R>(ctx, ubar);  // k_recon_vjp scatters by itself
    if (ctx->mem_slot) adj_gather(ctx, ubar);
    tstop(ctx, 0);
    tcollect(ctx, 0, &ctx->st.ms_recon_vjp, &ctx->st.n_recon_vjp);
    return UCNS_OK;
}

// (dR/dU)^T lam at the current state into ubar; bcbar (device, 10) += the
// free-stream cotangent when non-null
template <typename R>
int residual_vjp_t(ucns_ctx *ctx, const double *lam, double *ubar, double *bcbar) {
    int rc;
    if ((rc = vjp_recon_t<R>(ctx))) return rc;
    return vjp_products_t<R>(ctx, lam, ubar, bcbar);
}

// (dR/dU)^T lam at the current state into ubar; bcbar (device, 10) += the
// free-stream cotangent when non-null
int residual_vjp_dev(ucns_ctx *ctx, const double *lam, double *ubar, double *bcbar) {
    int rc = ensure_adjoint(ctx);
    if (rc) return rc;
    return ctx->precision == UCNS_MIXED ? residual_vjp_t<float>(ctx, lam, ubar, bcbar)
                                        : residual_vjp_t<double>(ctx, lam, ubar, bcbar);
}

// How many of a march's last stages keep their forward reconstruction (at
// most nstage): the scheme's adj_keep_stages caps the count (0: no cap,
// < 0: none), adj_keep_gib the bytes (never more than the free device memory
// less 4 GiB).
// A failed allocation leaves the count at what was had.
int adj_keep(ucns_ctx *ctx, int nstage) {
    const size_t esz = ctx->precision == UCNS_MIXED ? 4 : 8;
    const bool st = adj_stores(ctx);
    const size_t ul = (size_t)ctx->ncell * ctx->nf * ctx->nqm * NV * esz;
    const size_t g = adj_g_elems(ctx) * esz, fl = (size_t)ctx->ncell * sizeof(int);
    const size_t per = ul + (st ? g + fl : 0);
    auto held = [&](size_t nul, size_t ng) { return nul * ul + ng * (g + fl); };
    long want = nstage;
    if (ctx->adj_keep_stages < 0) return 0;
    if (ctx->adj_keep_stages > 0) want = std::min<long>(want, ctx->adj_keep_stages);
    size_t budget = (size_t)(ctx->adj_keep_gib * (double)(1ull << 30));
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) == hipSuccess) {
        const size_t have = fr + held(ctx->keep_ul.size(), ctx->keep_g.size()), margin = 4ull << 30;
        budget = std::min(budget, have > margin ? have - margin : 0);
    }
    want = std::min<long>(want, (long)(budget / per));
    // calls that store and geometry calls share the face values: what one of them
    // holds beyond the other's budget is given back
    const size_t n = (size_t)want;
    if (held(std::max(ctx->keep_ul.size(), n), st ? std::max(ctx->keep_g.size(), n) : ctx->keep_g.size()) > budget) {
        for (; ctx->keep_ul.size() > n; ctx->keep_ul.pop_back()) (void)hipFree(ctx->keep_ul.back());
        for (; ctx->keep_g.size() > (st ? n : 0); ctx->keep_g.pop_back(), ctx->keep_f.pop_back()) {
            (void)hipFree(ctx->keep_g.back());
            (void)hipFree(ctx->keep_f.back());
        }
    }
    size_t got = 0;  // stages in place
    for (; got < n; ++got) {
        if (ctx->keep_ul.size() == got) {
            void *a = nullptr;
            if (hipMalloc(&a, ul) != hipSuccess) break;
            ctx->keep_ul.push_back(a);
        }
        if (st && ctx->keep_g.size() == got) {
            void *b = nullptr;
            int *c = nullptr;
            if (hipMalloc(&b, g) != hipSuccess) break;
            if (hipMalloc((void **)&c, fl) != hipSuccess) {
                (void)hipFree(b);
                break;
            }
            ctx->keep_g.push_back(b);
            ctx->keep_f.push_back(c);
        }
    }
    (void)hipGetLastError();  // a refused allocation only lowers the count
    return (int)got;
}

// Point the reconstruction's outputs (face values; stencil coefficients and
// flags where the product reads them) at kept stage b, and back to the context's
// own buffers on destruction.
struct KeptStage {
    ucns_ctx *ctx;
    void *ul, *g;
    int *f;
    KeptStage(ucns_ctx *c, int b) : ctx(c), ul(c->uleft), g(c->adj_g), f(c->adj_flags) {
        ctx->uleft = ctx->keep_ul[b];
        if (adj_stores(c)) {
            ctx->adj_g = ctx->keep_g[b];
            ctx->adj_flags = ctx->keep_f[b];
        }
    }
    ~KeptStage() {
        ctx->uleft = ul;
        ctx->adj_g = g;
        ctx->adj_flags = f;
    }
};

// step it of nsteps, SSP-RK3 forward from ctx->U with the stage states stored; stages
// 3 it + stage - 1 >= keep0 also keep their reconstruction
int rk3_step_ckpt(ucns_ctx *ctx, int it, int nsteps, const double *dt, unsigned long long *next, double cfl,
                  int keep0) {
    const size_t n = (size_t)ctx->ncell * NV;
    for (int stage = 1; stage <= 3; ++stage) {
        const int q = 3 * it + stage - 1;
        // the stages after the first find their state stored by the update
        if (q == 0)
            HIP_TRY(hipMemcpyAsync(ctx->ckpt, ctx->U, n * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
        int rc;
        if (q >= keep0) {
            KeptStage k(ctx, q - keep0);
            ctx->adj_g_on = adj_stores(ctx);
            rc = residual_kernels(ctx, q > 0);
            ctx->adj_g_on = false;
        } else {
            rc = residual_kernels(ctx, q > 0);
        }
        if (rc) return rc;
        const bool more = q + 1 < 3 * nsteps;
        update_kernel(ctx, stage, dt, next != nullptr, next, cfl, nullptr, more,
                      more ? ctx->ckpt + (size_t)(q + 1) * n : nullptr);
    }
    return UCNS_OK;
}

// The reverse sweep over nsteps stored steps: abar holds the cotangent of
// the final state on entry and of the initial state on return.  Stages are
// reversed in the order (step n: 3, 2, 1), each at its stored state, with
//   w = -c dt ybar / V, jt = (dR/du)^T w, and k_rk3_adj_stage combining ybar
//   and jt into the cotangents of the stage's inputs and the next w.
// In row-stream mode the scatter of a stage's reconstruction product streams the
// pseudo-inverses, and so does the forward reconstruction of a stage that did not
// keep its own.
//
// Stages q = 3 it + stage - 1 >= keep0 kept their forward reconstruction, so
// their products start from it and only the other stages run the
// reconstruction again.
template <typename R>
int rk3_reverse_t(ucns_ctx *ctx, int nsteps, double *abar, double *bcbar, int keep0) {
    const size_t n = (size_t)ctx->ncell * NV;
    const int blocks = (int)std::min<size_t>(8192, (n + 255) / 256);
    double *const ustate = ctx->U;
    double *a = abar, *u0 = ctx->adj_u0, *x = ctx->adj_x, *w = ctx->adj_lam, *jt = ctx->adj_ubar;
    const double cst[4] = {0.0, 1.0, 1.0 / 4.0, 2.0 / 3.0};  // -w / (dt ybar / V) per stage
    int rc = UCNS_OK;
    for (int it = nsteps - 1; it >= 0 && rc == UCNS_OK; --it) {
        const double *dt = ctx->dts + it;
        for (int stage = 3; stage >= 1 && rc == UCNS_OK; --stage) {
            ctx->U = ctx->ckpt + ((size_t)3 * it + stage - 1) * n;
            const double *y = stage == 3 ? a : x;
            if (it == nsteps - 1 && stage == 3)
                hipLaunchKernelGGL(k_rk3_adj_w, dim3(blocks), dim3(256), 0, ctx->stream, ctx->ncell, y, ctx->ovol,
                                   dt, cst[stage], w, jt);
            const int q = 3 * it + stage - 1;
            if (q >= keep0) {
                KeptStage k(ctx, q - keep0);
                if ((rc = vjp_products_t<R>(ctx, w, jt, bcbar, true))) break;
            } else {
                if ((rc = vjp_recon_t<R>(ctx))) break;
                if ((rc = vjp_products_t<R>(ctx, w, jt, bcbar, true))) break;
            }
            // this stage's product is complete: fold it into its input
            // cotangents, and form the cotangent of the stage before
            const double *ndt = stage > 1 ? dt : it > 0 ? dt - 1 : nullptr;
            hipLaunchKernelGGL(k_rk3_adj_stage, dim3(blocks), dim3(256), 0, ctx->stream, ctx->ncell, stage, y, jt, x,
                               u0, a, ctx->ovol, ndt, cst[stage > 1 ? stage - 1 : 3], w);
        }
    }
    ctx->U = ustate;
    if (rc == UCNS_OK) {
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            ctx->err = std::string("rk3 reverse: ") + hipGetErrorString(e);
            rc = UCNS_EHIP;
        }
    }
    return rc;
}

int rk3_reverse(ucns_ctx *ctx, int nsteps, double *abar, double *bcbar, int keep0) {
    return ctx->precision == UCNS_MIXED ? rk3_reverse_t<float>(ctx, nsteps, abar, bcbar, keep0)
                                        : rk3_reverse_t<double>(ctx, nsteps, abar, bcbar, keep0);
}

template <typename R>
int upload_real(ucns_ctx *ctx, void **dst, const std::vector<double> &src) {
    std::vector<R> tmp(src.size());
    for (size_t e = 0; e < src.size(); ++e) tmp[e] = (R)src[e];
    int rc = dalloc(ctx, (R **)dst, tmp.size());
    if (rc) return rc;
    HIP_TRY(hipMemcpy(*dst, tmp.data(), tmp.size() * sizeof(R), hipMemcpyHostToDevice));
    return UCNS_OK;
}

int upload_real_any(ucns_ctx *ctx, void **dst, const std::vector<double> &src) {
    return ctx->precision == UCNS_MIXED ? upload_real<float>(ctx, dst, src) : upload_real<double>(ctx, dst, src);
}

void release_prestore(ucns_ctx *ctx) {
    dfree(ctx->nbr);
    dfree(ctx->nbc);
    dfree(ctx->P);
    dfree(ctx->rows);
    dfree(ctx->u64);
    dfree(ctx->marks);
    release_members(ctx);
    dfree(ctx->B);
    dfree(ctx->mbar);
    if (ctx->Bc) (void)hipFree(ctx->Bc);
    if (ctx->dmb) (void)hipFree(ctx->dmb);
    if (ctx->Pc) (void)hipFree(ctx->Pc);
    ctx->Bc = ctx->dmb = ctx->Pc = nullptr;
    dfree(ctx->qp);
    ctx->have_prestore = false;
}


// ---- cell order -------------------------------------------------------------
// The library may hold the cells in an order of its own, so that a tile of 8
// consecutive cells is a compact cluster whatever order the caller's
// partitioner produced.  perm[c] = the caller's cell of library cell c.

// reverse Cuthill-McKee on the face graph (interior and periodic faces):
// per connected component, breadth-first from a pseudo-peripheral cell of
// least degree, neighbours in increasing degree, then the whole order reversed
void order_rcm(const ucns_mesh_v2 *m, std::vector<int32_t> &perm) {
    const int nc = m->ncell, nfa = m->nface_max, base = m->index_base;
    std::vector<int32_t> deg(nc, 0);
    auto nbr = [&](int i, int f) -> int {
        if (f >= m->ifca[i]) return -1;
        const int bc = m->bcode[(size_t)i * nfa + f];
        if (bc != 0 && bc != 5 && bc != 50) return -1;
        const int j = m->ineigh[(size_t)i * nfa + f] - base;
        return j == i ? -1 : j;
    };
    for (int i = 0; i < nc; ++i)
        for (int f = 0; f < nfa; ++f) deg[i] += nbr(i, f) >= 0;
    std::vector<int32_t> level(nc, -1), q;
    q.reserve(nc);
    // breadth-first levels from r over the cells not yet ordered; returns the
    // cell of least degree in the last level and the number of levels
    std::vector<char> done(nc, 0);
    std::vector<int32_t> touched;
    auto bfs_far = [&](int r, int &nlev) {
        touched.clear();
        std::vector<int32_t> frontier{r}, next;
        level[r] = 0;
        touched.push_back(r);
        nlev = 1;
        int far = r;
        while (!frontier.empty()) {
            next.clear();
            for (int i : frontier)
                for (int f = 0; f < nfa; ++f) {
                    const int j = nbr(i, f);
                    if (j >= 0 && !done[j] && level[j] < 0) {
                        level[j] = level[i] + 1;
                        touched.push_back(j);
                        next.push_back(j);
                    }
                }
            if (next.empty()) {
                far = frontier[0];
                for (int i : frontier)
                    if (deg[i] < deg[far] || (deg[i] == deg[far] && i < far)) far = i;
            } else {
                ++nlev;
            }
            frontier.swap(next);
        }
        for (int i : touched) level[i] = -1;
        return far;
    };
    perm.clear();
    perm.reserve(nc);
    std::vector<int32_t> by_deg(nc);
    for (int i = 0; i < nc; ++i) by_deg[i] = i;
    std::stable_sort(by_deg.begin(), by_deg.end(), [&](int a, int b) { return deg[a] < deg[b]; });
    std::vector<int32_t> cand;
    for (int seed : by_deg) {
        if (done[seed]) continue;
        int r = seed, nlev = 0;
        int far = bfs_far(r, nlev);
        for (int it = 0; it < 8; ++it) {  // pseudo-peripheral cell (George and Liu)
            int nl2 = 0;
            const int far2 = bfs_far(far, nl2);
            if (nl2 <= nlev) break;
            r = far;
            nlev = nl2;
            far = far2;
        }
        size_t head = perm.size();
        perm.push_back(r);
        done[r] = 1;
        while (head < perm.size()) {
            const int i = perm[head++];
            cand.clear();
            for (int f = 0; f < nfa; ++f) {
                const int j = nbr(i, f);
                if (j >= 0 && !done[j]) {
                    done[j] = 1;
                    cand.push_back(j);
                }
            }
            std::sort(cand.begin(), cand.end(),
                      [&](int a, int b) { return deg[a] < deg[b] || (deg[a] == deg[b] && a < b); });
            perm.insert(perm.end(), cand.begin(), cand.end());
        }
    }
    std::reverse(perm.begin(), perm.end());
}

// Morton (Z-order) curve of the centroids: 21 bits per axis over the
// bounding box, ties by the caller's index
void order_morton(const ucns_mesh_v2 *m, std::vector<int32_t> &perm) {
    const int nc = m->ncell;
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (int i = 0; i < nc; ++i)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], m->centroid[(size_t)3 * i + d]);
            hi[d] = std::max(hi[d], m->centroid[(size_t)3 * i + d]);
        }
    auto spread = [](uint64_t x) {  // 21 bits -> every third bit of 63
        x &= 0x1FFFFFull;
        x = (x | x << 32) & 0x1F00000000FFFFull;
        x = (x | x << 16) & 0x1F0000FF0000FFull;
        x = (x | x << 8) & 0x100F00F00F00F00Full;
        x = (x | x << 4) & 0x10C30C30C30C30C3ull;
        x = (x | x << 2) & 0x1249249249249249ull;
        return x;
    };
    std::vector<uint64_t> key(nc);
    for (int i = 0; i < nc; ++i) {
        uint64_t k = 0;
        for (int d = 0; d < 3; ++d) {
            const double ext = hi[d] - lo[d];
            const double t = ext > 0 ? (m->centroid[(size_t)3 * i + d] - lo[d]) / ext : 0.0;
            const uint64_t g = (uint64_t)std::min(2097151.0, std::max(0.0, std::floor(t * 2097152.0)));
            k |= spread(g) << (2 - d);
        }
        key[i] = k;
    }
    perm.resize(nc);
    for (int i = 0; i < nc; ++i) perm[i] = i;
    std::sort(perm.begin(), perm.end(), [&](int a, int b) { return key[a] < key[b] || (key[a] == key[b] && a < b); });
}

// the caller's cell of library cell i, and the library cell of caller cell o
inline size_t src_cell(const ucns_ctx *ctx, int i) { return ctx->h_perm.empty() ? (size_t)i : (size_t)ctx->h_perm[i]; }
inline int lib_cell(const ucns_ctx *ctx, int o) { return ctx->h_iperm.empty() ? o : ctx->h_iperm[o]; }

// caller-order 5-vectors (host or device memory, either layout) -> the
// library's AoS device array dst
int cells_in(ucns_ctx *ctx, const double *src, bool host, int32_t layout, double *dst) {
    if (layout != UCNS_LAYOUT_AOS && layout != UCNS_LAYOUT_SOA) {
        ctx->err = "unknown layout";
        return UCNS_EBADARG;
    }
    const size_t n = (size_t)ctx->ncell * NV;
    if (host) {
        HIP_TRY(hipMemcpyAsync(ctx->stage, src, n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
        src = ctx->stage;
    }
    hipLaunchKernelGGL(k_cells_in, dim3((ctx->ncell + 255) / 256), dim3(256), 0, ctx->stream, ctx->ncell, ctx->perm,
                       src, layout, dst);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return UCNS_OK;
}

// the library's AoS device array src -> caller-order 5-vectors
int cells_out(ucns_ctx *ctx, const double *src, int32_t layout, double *dst, bool host) {
    if (layout != UCNS_LAYOUT_AOS && layout != UCNS_LAYOUT_SOA) {
        ctx->err = "unknown layout";
        return UCNS_EBADARG;
    }
    const size_t n = (size_t)ctx->ncell * NV;
    hipLaunchKernelGGL(k_cells_out, dim3((ctx->ncell + 255) / 256), dim3(256), 0, ctx->stream, ctx->ncell, ctx->perm,
                       src, layout, host ? ctx->stage : dst);
    HIP_TRY(hipGetLastError());
    if (host) HIP_TRY(hipMemcpyAsync(dst, ctx->stage, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return UCNS_OK;
}

// The caller's mesh with its cells in the library's order (per-cell rows
// moved, neighbour ids renumbered); the vectors own the storage the struct
// points into.
struct PermutedMesh {
    ucns_mesh_v2 m{};
    std::vector<int32_t> ifca, ineigh, ineighn, bcode, types;
    std::vector<double> angx, angy, surf, vol, minedge;
    void build(const ucns_mesh_v2 *src, const std::vector<int32_t> &perm, const std::vector<int32_t> &iperm) {
        const int nc = src->ncell, nfa = src->nface_max, base = src->index_base;
        const size_t nfc = (size_t)nc * nfa;
        ifca.resize(nc);
        vol.resize(nc);
        minedge.resize(nc);
        ineigh.resize(nfc);
        ineighn.resize(nfc);
        bcode.resize(nfc);
        types.resize(nfc);
        angx.resize(nfc);
        angy.resize(nfc);
        surf.resize(nfc);
        for (int c = 0; c < nc; ++c) {
            const size_t o = perm[c];
            ifca[c] = src->ifca[o];
            vol[c] = src->totvolume[o];
            minedge[c] = src->minedge[o];
            for (int f = 0; f < nfa; ++f) {
                const size_t d = (size_t)c * nfa + f, sl = o * nfa + f;
                const int bc = src->bcode[sl];
                const int j = src->ineigh[sl] - base;
                const bool link = f < src->ifca[o] && (bc == 0 || bc == 5 || bc == 50) && j >= 0 && j < nc;
                ineigh[d] = link ? iperm[j] + base : src->ineigh[sl];
                ineighn[d] = src->ineighn[sl];
                bcode[d] = bc;
                types[d] = src->types_faces[sl];
                angx[d] = src->faceanglex[sl];
                angy[d] = src->faceangley[sl];
                surf[d] = src->surf[sl];
            }
        }
        m = *src;
        m.ifca = ifca.data();
        m.ineigh = ineigh.data();
        m.ineighn = ineighn.data();
        m.bcode = bcode.data();
        m.types_faces = types.data();
        m.faceanglex = angx.data();
        m.faceangley = angy.data();
        m.surf = surf.data();
        m.totvolume = vol.data();
        m.minedge = minedge.data();
        m.centroid = nullptr;
    }
};

}  // namespace

extern "C" {

int ucns_abi_version(void) { return UCNS_ABI_VERSION; }

const char *ucns_last_error(const ucns_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int ucns_create(const ucns_mesh_v2 *m, const ucns_scheme_v2 *s, ucns_ctx **out) {
    if (!out) return UCNS_EBADARG;
    *out = nullptr;
    if (!m || !s) return UCNS_EBADARG;
    PermutedMesh pm;
    ucns_ctx *ctx = new ucns_ctx();
    *out = ctx;
    auto bad = [&](int code, const std::string &msg) {
        ctx->err = msg;
        return code;
    };
    if (m->abi_version != UCNS_ABI_VERSION || s->abi_version != UCNS_ABI_VERSION)
        return bad(UCNS_EBADARG, "abi_version mismatch");
    if (m->ncell <= 0 || m->nface_max <= 0 || m->nface_max > 6) return bad(UCNS_EBADARG, "bad ncell/nface_max");
    if (!m->ifca || !m->ineigh || !m->ineighn || !m->bcode || !m->types_faces || !m->faceanglex ||
        !m->faceangley || !m->surf || !m->totvolume || !m->minedge)
        return bad(UCNS_EBADARG, "null mesh array");
    if (s->precision != UCNS_FP64 && s->precision != UCNS_MIXED) return bad(UCNS_EBADARG, "bad precision");
    if (s->iweno != 1 && s->iweno != -1) return bad(UCNS_EUNSUPPORTED, "iweno must be 1 (WENO) or -1 (MUSCL)");
    if (s->ees != 0 && s->ees != 5) return bad(UCNS_EUNSUPPORTED, "ees must be 0 (WENO) or 5 (CWENO)");
    if (s->ees == 5 && s->iweno != 1) return bad(UCNS_EBADARG, "CWENO (ees 5) needs iweno 1");
    if (s->wenoz != 0 && s->wenoz != 1) return bad(UCNS_EBADARG, "wenoz must be 0 or 1");
    if (s->wenoz == 1 && s->ees != 5) return bad(UCNS_EUNSUPPORTED, "wenoz 1 is a CWENO option (ees 5)");
    if (s->wenwrt != 1 && s->wenwrt != 2)
        return bad(UCNS_EUNSUPPORTED, "wenwrt must be 1 (conserved) or 2 (characteristic variables)");
    if (s->wenwrt == 2 && (s->iweno != 1 || s->ees != 0))
        return bad(UCNS_EUNSUPPORTED, "characteristic reconstruction (wenwrt 2) is built for WENO with ees 0");
    if (s->limiter != 1) return bad(UCNS_EUNSUPPORTED, "only the Barth-Jespersen limiter (1)");
    if (s->riemann != 1) return bad(UCNS_EUNSUPPORTED, "only the HLLC solver (1)");
    if (s->typesten < 1 || s->typesten > 7) return bad(UCNS_EUNSUPPORTED, "typesten must be 1..7");
    if (s->qp_quad < 1 || s->qp_quad > 64 || s->qp_triangle < 1 || s->qp_triangle > 64 || !s->weights_quad ||
        !s->weights_tri)
        return bad(UCNS_EBADARG, "bad face quadrature");
    if (s->cell_order != UCNS_ORDER_CALLER && s->cell_order != UCNS_ORDER_RCM && s->cell_order != UCNS_ORDER_MORTON)
        return bad(UCNS_EBADARG, "cell_order must be UCNS_ORDER_CALLER, _RCM or _MORTON");
    if (s->cell_order == UCNS_ORDER_MORTON && !m->centroid)
        return bad(UCNS_EBADARG, "UCNS_ORDER_MORTON needs the mesh centroids");
    if (s->kernels != UCNS_KERNELS_AUTO && s->kernels != UCNS_KERNELS_REGISTER)
        return bad(UCNS_EBADARG, "kernels must be UCNS_KERNELS_AUTO or UCNS_KERNELS_REGISTER");
    if (s->reserved != 0) return bad(UCNS_EBADARG, "reserved must be 0");
    if (!std::isfinite(s->adj_keep_gib)) return bad(UCNS_EBADARG, "adj_keep_gib must be finite");
    ctx->cell_order = s->cell_order;
    ctx->kernels = s->kernels;
    ctx->adj_keep_stages = s->adj_keep_stages;
    ctx->adj_keep_gib = s->adj_keep_gib > 0 ? s->adj_keep_gib : 64.0;
    ctx->ncell = m->ncell;
    ctx->nf_abi = m->nface_max;
    ctx->index_base = m->index_base;
    ctx->precision = s->precision;
    ctx->iweno = s->iweno;
    ctx->ees = s->ees;
    ctx->wenwrt = s->wenwrt;
    ctx->wenoz = s->wenoz;
    ctx->ideg = s->idegfree;
    ctx->nnb = s->inumneighbours;
    ctx->imax = s->inumneighbours - 1;
    ctx->ts_abi = s->typesten;
    ctx->qpq = s->qp_quad;
    ctx->qpt = s->qp_triangle;
    ctx->nqm_abi = std::max(s->qp_quad, s->qp_triangle);
    ctx->gamma = s->gamma;
    ctx->lwci1 = s->lwci1;
    ctx->eps = s->weno_eps;
    if (!((ctx->ideg == 34 && ctx->imax == 69) || (ctx->ideg == 19 && ctx->imax == 39) ||
          (ctx->ideg == 9 && ctx->imax == 19) || (ctx->ideg == 3 && ctx->imax == 8)))
        return bad(UCNS_EUNSUPPORTED, "supported (idegfree, inumneighbours): (34, 70) WENO-5, (19, 40) WENO-4, "
                                      "(9, 20) WENO-3 and (3, 9) MUSCL");
    if (ctx->iweno == -1 && ctx->ideg != 3) return bad(UCNS_EUNSUPPORTED, "MUSCL path is linear (idegfree 3)");
    if (m->ncell > 0 && m->ifca)
        for (int i = 0; i < m->ncell; ++i)
            if (m->ifca[i] < 4 || m->ifca[i] > m->nface_max)
                return bad(UCNS_EBADARG, "ifca out of range at cell " + std::to_string(i));
    // the caller's face links, checked before anything reads through them:
    // codes, neighbour ranges and the symmetry of (cell, slot) pairs
    {
        const int nc0 = m->ncell, nfa0 = m->nface_max, b0 = m->index_base;
        for (int i = 0; i < nc0; ++i)
            for (int f = 0; f < m->ifca[i]; ++f) {
                const size_t sl = (size_t)i * nfa0 + f;
                const int bc = m->bcode[sl];
                if (bc == 1 || bc == 2 || bc == 3 || bc == 4 || bc == 6) continue;
                if (bc != 0 && bc != 5 && bc != 50)
                    return bad(UCNS_EUNSUPPORTED, "face codes: 0 interior, 5/50 periodic, 1/2/3/4/6 boundary");
                const int j = m->ineigh[sl] - b0, fj = m->ineighn[sl] - b0;
                if (j < 0 || j >= nc0 || fj < 0 || fj >= m->ifca[j])
                    return bad(UCNS_EBADARG, "face neighbour out of range at cell " + std::to_string(i));
                const size_t slj = (size_t)j * nfa0 + fj;
                if (m->ineigh[slj] - b0 != i || m->ineighn[slj] - b0 != f)
                    return bad(UCNS_EBADARG, "face neighbours are not symmetric at cell " + std::to_string(i));
            }
    }
    if (ctx->cell_order != UCNS_ORDER_CALLER) {
        if (ctx->cell_order == UCNS_ORDER_RCM)
            order_rcm(m, ctx->h_perm);
        else
            order_morton(m, ctx->h_perm);
        ctx->h_iperm.assign(m->ncell, 0);
        for (int c = 0; c < m->ncell; ++c) ctx->h_iperm[ctx->h_perm[c]] = c;
        pm.build(m, ctx->h_perm, ctx->h_iperm);
        m = &pm.m;
    }

    const int nc = m->ncell, nfa = m->nface_max, base = m->index_base;
    // faces in use, Gauss points per face type present
    int nf = 0, nqm = 0;
    bool any_quad = false, any_tri = false;
    for (int i = 0; i < nc; ++i) {
        const int ifca = m->ifca[i];
        if (ifca < 4 || ifca > nfa) return bad(UCNS_EBADARG, "ifca out of range at cell " + std::to_string(i));
        nf = std::max(nf, ifca);
        for (int f = 0; f < ifca; ++f) {
            const int t = m->types_faces[(size_t)i * nfa + f];
            if (t == 5) any_quad = true;
            else if (t == 6) any_tri = true;
            else return bad(UCNS_EBADARG, "types_faces must be 5 or 6");
        }
    }
    if (any_quad) nqm = std::max(nqm, s->qp_quad);
    if (any_tri) nqm = std::max(nqm, s->qp_triangle);
    if (nf > 6) return bad(UCNS_EUNSUPPORTED, "at most 6 faces per cell");
    ctx->nf = nf;
    ctx->nqm = nqm;
    if (nf * nqm > 6 * 16) return bad(UCNS_EUNSUPPORTED, "too many face Gauss points per cell");
    // unique faces: owner = lower cell id (equal ids: lower slot)
    std::vector<int32_t> cinfo(nc, 0), cnb((size_t)nc * nf, -1), cface((size_t)nc * nf, 0);
    std::vector<int32_t> chnb(ctx->wenwrt == 2 ? (size_t)nc * nf : 0, 0);
    std::vector<double> chang(ctx->wenwrt == 2 ? (size_t)nc * nf * 4 : 0, 0.0);
    std::vector<int32_t> fcell, fslot, bfaces;
    std::vector<double> frot, farea;
    for (int i = 0; i < nc; ++i) {
        const int ifca = m->ifca[i];
        int w = ifca;
        for (int f = 0; f < ifca; ++f)
            if (m->types_faces[(size_t)i * nfa + f] == 6) w |= 1 << (8 + f);
        cinfo[i] = w;
        for (int f = 0; f < ifca; ++f) {
            const size_t sl = (size_t)i * nfa + f;
            const int bc = m->bcode[sl];
            if (!chnb.empty()) {
                const bool bnd = bc == 1 || bc == 2 || bc == 3 || bc == 4 || bc == 6;
                chnb[(size_t)i * nf + f] = bnd ? -bc : m->ineigh[sl] - base;
                const double a1 = m->faceanglex[sl], a2 = m->faceangley[sl];
                double *an = &chang[((size_t)i * nf + f) * 4];
                an[0] = std::cos(a1);
                an[1] = std::sin(a1);
                an[2] = std::cos(a2);
                an[3] = std::sin(a2);
            }
            if (bc == 1 || bc == 2 || bc == 3 || bc == 4 || bc == 6) {
                // boundary face: owner only, the right state is a ghost (BOUNDARYS)
                if (bc != 3 && bc != 4) ctx->needs_bc = true;
                cnb[(size_t)i * nf + f] = -1;
                const int id = (int)farea.size();
                bfaces.push_back(id);
                fcell.push_back(i);
                fcell.push_back(-bc);
                fslot.push_back(f | (m->types_faces[sl] == 6 ? 256 : 0));
                fslot.push_back(0);
                const double a1 = m->faceanglex[sl], a2 = m->faceangley[sl];
                frot.push_back(std::cos(a1));
                frot.push_back(std::sin(a1));
                frot.push_back(std::cos(a2));
                frot.push_back(std::sin(a2));
                farea.push_back(m->surf[sl]);
                cface[(size_t)i * nf + f] = id + 1;
                continue;
            }
            if (bc != 0 && bc != 5 && bc != 50)  // periodic: 5 or 50 (src/dg_functions.f90:1786)
                return bad(UCNS_EUNSUPPORTED, "face codes: 0 interior, 5/50 periodic, 1/2/3/4/6 boundary");
            const int j = m->ineigh[sl] - base, fj = m->ineighn[sl] - base;
            if (j < 0 || j >= nc || fj < 0 || fj >= m->ifca[j])
                return bad(UCNS_EBADARG, "face neighbour out of range at cell " + std::to_string(i));
            const size_t slj = (size_t)j * nfa + fj;
            if (m->ineigh[slj] - base != i || m->ineighn[slj] - base != f)
                return bad(UCNS_EBADARG, "face neighbours are not symmetric at cell " + std::to_string(i));
            // MUSCL bounds take the neighbours of interior faces and of periodic
            // faces of code 5, not of code 50 (FIND_BOUNDS, src/reconstruct_p.f90:1871)
            cnb[(size_t)i * nf + f] = bc == 50 ? -1 : j;
            const bool owner = (i < j) || (i == j && f < fj);
            if (!owner) continue;
            const int id = (int)farea.size();
            fcell.push_back(i);
            fcell.push_back(j);
            fslot.push_back(f | (m->types_faces[sl] == 6 ? 256 : 0));
            fslot.push_back(fj);
            const double a1 = m->faceanglex[sl], a2 = m->faceangley[sl];
            frot.push_back(std::cos(a1));
            frot.push_back(std::sin(a1));
            frot.push_back(std::cos(a2));
            frot.push_back(std::sin(a2));
            farea.push_back(m->surf[sl]);
            cface[(size_t)i * nf + f] = id + 1;
            cface[(size_t)j * nf + fj] = -(id + 1);
        }
    }
    ctx->nface = (int)farea.size();
    ctx->nbface = (int)bfaces.size();
    ctx->h_cinfo_base = cinfo;
    std::vector<double> ovol(nc), minedge(nc);
    for (int i = 0; i < nc; ++i) {
        if (!(m->totvolume[i] > 0)) return bad(UCNS_EBADARG, "non-positive volume");
        ovol[i] = 1.0 / m->totvolume[i];
        minedge[i] = m->minedge[i];
    }
    ctx->h_fcell = fcell;
    ctx->h_fslot = fslot;
    ctx->h_ovol = ovol;
    // the device resources, once the host data has been checked
    HIP_TRY(hipGetDevice(&ctx->device));
    HIP_TRY(hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking));
    for (auto &e : ctx->ev) HIP_TRY(hipEventCreate(&e));
    {
        const int rc0 = scratch_on(ctx->device, &ctx->scratch, ctx->err);  // with the device current
        if (rc0) return rc0;
    }
    int rc;
    if ((rc = dalloc(ctx, &ctx->cinfo, nc)) || (rc = dalloc(ctx, &ctx->cnb, cnb.size())) ||
        (rc = dalloc(ctx, &ctx->cface, cface.size())) || (rc = dalloc(ctx, &ctx->fcell, fcell.size())) ||
        (rc = dalloc(ctx, &ctx->fslot, fslot.size())) || (rc = dalloc(ctx, &ctx->frot, frot.size())) ||
        (rc = dalloc(ctx, &ctx->farea, farea.size())) || (rc = dalloc(ctx, &ctx->ovol, nc)) ||
        (rc = dalloc(ctx, &ctx->minedge, nc)) || (rc = dalloc(ctx, &ctx->U, (size_t)nc * NV)) ||
        (rc = dalloc(ctx, &ctx->U2, (size_t)nc * NV)) || (rc = dalloc(ctx, &ctx->rhs, (size_t)nc * NV)) ||
        (rc = dalloc(ctx, &ctx->fflux, (size_t)ctx->nface * NV)) || (rc = dalloc(ctx, &ctx->t, 1)) ||
        (rc = dalloc(ctx, &ctx->dtfix, 1)) || (rc = dalloc(ctx, &ctx->dtv, 2 * DT_SLOTS * DT_STRIDE)) ||
        (rc = dalloc(ctx, &ctx->stage, (size_t)nc * NV)))
        return rc;
    HIP_TRY(hipHostMalloc((void **)&ctx->result, sizeof(HostResult), hipHostMallocDefault));
    if (!bfaces.empty()) {
        if ((rc = dalloc(ctx, &ctx->bfaces, bfaces.size()))) return rc;
        HIP_TRY(hipMemcpy(ctx->bfaces, bfaces.data(), bfaces.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    }
    if (!ctx->h_perm.empty()) {
        if ((rc = dalloc(ctx, &ctx->perm, nc))) return rc;
        HIP_TRY(hipMemcpy(ctx->perm, ctx->h_perm.data(), nc * sizeof(int32_t), hipMemcpyHostToDevice));
    }
    // k_flux_update evaluates every flux twice: 10 steps on 10^3, 18^3, 28^3, 32^3
    // and 36^3 hexahedra take 0.45, 0.49, 0.78, 0.89 and 1.10 ms with it, 0.55,
    // 0.59, 0.84, 0.91 and 1.03 without
    if (nqm == 1 && nc <= 32768 && ((rc = dalloc(ctx, &ctx->fadj, cface.size())) || (rc = dalloc(ctx, &ctx->U3, (size_t)nc * NV))))
        return rc;
    const size_t ul_elems = (size_t)nc * nf * nqm * NV;
    rc = ctx->precision == UCNS_MIXED ? dalloc(ctx, (float **)&ctx->uleft, ul_elems)
                                      : dalloc(ctx, (double **)&ctx->uleft, ul_elems);
    if (rc) return rc;
    HIP_TRY(hipMemset(ctx->uleft, 0, ul_elems * (ctx->precision == UCNS_MIXED ? 4 : 8)));
    HIP_TRY(hipMemcpy(ctx->cinfo, cinfo.data(), nc * sizeof(int32_t), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(ctx->cnb, cnb.data(), cnb.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    if (!chnb.empty()) {
        if ((rc = dalloc(ctx, &ctx->chnb, chnb.size())) || (rc = dalloc(ctx, &ctx->chang, chang.size()))) return rc;
        HIP_TRY(hipMemcpy(ctx->chnb, chnb.data(), chnb.size() * sizeof(int32_t), hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(ctx->chang, chang.data(), chang.size() * sizeof(double), hipMemcpyHostToDevice));
    }
    HIP_TRY(hipMemcpy(ctx->cface, cface.data(), cface.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(ctx->fcell, fcell.data(), fcell.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(ctx->fslot, fslot.data(), fslot.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(ctx->frot, frot.data(), frot.size() * sizeof(double), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(ctx->farea, farea.data(), farea.size() * sizeof(double), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(ctx->ovol, ovol.data(), nc * sizeof(double), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(ctx->minedge, minedge.data(), nc * sizeof(double), hipMemcpyHostToDevice));
    double wq[64] = {0}, wt[64] = {0};
    for (int q = 0; q < s->qp_quad; ++q) wq[q] = s->weights_quad[q];
    for (int q = 0; q < s->qp_triangle; ++q) wt[q] = s->weights_tri[q];
    if ((rc = dalloc(ctx, &ctx->wquad, 128))) return rc;
    HIP_TRY(hipMemcpy(ctx->wquad, wq, sizeof(wq), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(ctx->wquad + 64, wt, sizeof(wt), hipMemcpyHostToDevice));
    HIP_TRY(hipMemset(ctx->t, 0, sizeof(double)));
    if (ctx->fadj) {
        hipLaunchKernelGGL(k_face_records, dim3((unsigned)((cface.size() + 255) / 256)), dim3(256), 0, ctx->stream,
                           cface.size(), ctx->cface, ctx->fcell, ctx->fslot, ctx->fadj);
        HIP_TRY(hipGetLastError());
    }
    return UCNS_OK;
}

int ucns_upload_prestore(ucns_ctx *ctx, const ucns_prestore_v1 *pre) {
    if (!ctx) return UCNS_EBADARG;
    if (!pre || !pre->admis || !pre->full || !pre->ihexl || !pre->invmat || !pre->integ_basis || !pre->volume11 ||
        !pre->qpoints) {
        ctx->err = "null prestore array";
        return UCNS_EBADARG;
    }
    if (ctx->iweno == 1 && !pre->indicator) {
        ctx->err = "WENO needs the indicator matrices";
        return UCNS_EBADARG;
    }
    if (ctx->ees == 5 && !ctx->have_cweno) {
        ctx->err = "CWENO (ees 5): call ucns_upload_cweno before ucns_upload_prestore";
        return UCNS_ESTATE;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    release_prestore(ctx);
    release_adjoint(ctx);  // its buffers are sized by the stencil count
    const int nc = ctx->ncell, ID = ctx->ideg, IM = ctx->imax, NNB = ctx->nnb, TSA = ctx->ts_abi;
    const int base = ctx->index_base;
    // admissible stencils, flags
    int ts = 1;
    std::vector<int32_t> cinfo = ctx->h_cinfo_base;
    for (int i = 0; i < nc; ++i) {
        const size_t o = src_cell(ctx, i);
        const int ad = pre->admis[o];
        if (ad < 1 || ad > TSA) {
            ctx->err = "admis out of range at cell " + std::to_string(o);
            return UCNS_EBADARG;
        }
        ts = std::max(ts, ad);
        cinfo[i] |= (ad << 3) | ((pre->full[o] ? 1 : 0) << 6);
    }
    if (ctx->iweno == -1 && ts != 1) {
        ctx->err = "MUSCL uses the central stencil only (admis must be 1)";
        return UCNS_EUNSUPPORTED;
    }
    ctx->ts = ts;
    const bool mixed = ctx->precision == UCNS_MIXED;
    // the block kernels (recon_block.hip)
    const bool wide = ctx->kernels == UCNS_KERNELS_AUTO && ctx->ees != 5 && ts >= 5 && ts <= 7;
    ctx->tiled = (ctx->iweno == 1 && (ctx->wenwrt == 1 || wide) && ((ID == 19 && IM == 39) || (ID == 9 && IM == 19)) &&
                  ts <= 8 && ctx->nf * ctx->nqm <= 56);
    ctx->cw_cell = ctx->ees == 5 && !ctx->tiled;
    if (ctx->cw_cell && ID != 34) {
        ctx->err = "CWENO (ees 5) runs on the WENO-3 / WENO-4 register kernels (idegfree 9 or 19) or the WENO-5 "
                   "per-cell kernel";
        return UCNS_EUNSUPPORTED;
    }
    {
        // row-stream kernels: tetrahedra (5 stencils, 24 face points) and
        // hexahedra (7 stencils, 54 face points), with WENO-3 also meshes of
        // prisms and pyramids (6 stencils), unless the scheme asks for the
        // register-prefetch kernels.  Channel of 131,000 cells with up to 6,
        // 4 steps: register prefetch 4.77 ms, row stream 4.46 ms (mixed 2.08 and
        // 1.92); the product of 3 steps on 14,000 cells: 2.27 and 1.96 ms
        const int nfq = ctx->nf * ctx->nqm;
        const bool shape_ok = ID == 19 ? ((ts == 5 && nfq <= 24) || (ts == 7 && nfq > 24))
                                       : (ts >= 5 && ts <= 7 && nfq <= 24);
        const bool stream_ok = ctx->kernels == UCNS_KERNELS_AUTO && ctx->tiled && shape_ok && ctx->ees != 5;
        ctx->smode = stream_ok ? ts : 0;
    }
    ctx->ntile = (nc + 7) / 8;
    // WENO-4 of few tiles: there a wave per tile leaves SIMDs idle and its chain of
    // rows bare.  The line is where the blocks no longer all run at once (two a CU
    // in FP64 on hexahedra).  A march's stage in us, row stream and block kernels:
    //   FP64   hexahedra    216 tiles 55.6, 39.4;  512 61.1, 58.9;  615 74.5, 83.2;  1,000 95.4, 111.5
    //          tetrahedra   162 45.8, 31.3;        384 47.5, 42.0;  547 51.3, 53.1;    999 68.4, 77.1
    //   mixed  hexahedra    216 45.4, 32.8;        512 49.4, 43.1;  729 54.5, 55.5;    858 62.4, 64.3
    //          tetrahedra   162 39.3, 27.4;        384 40.2, 31.2;  750 42.8, 39.9;    999 46.4, 47.1
    // (a mesh of hexahedra, pyramids and prisms in FP64, 648 tiles: 84.0, 81.1; the
    // member tables have a say in it below)
    ctx->bmode = ctx->tiled && wide &&
                 (ctx->wenwrt == 2 || (ctx->smode && ID == 19 && ctx->ntile <= (mixed ? 768 : 512)));
    ctx->nmark = ctx->tiled || ctx->cw_cell || ctx->iweno == -1 ? ctx->ntile : nc;
    int rc = dalloc(ctx, &ctx->marks, (size_t)ctx->nmark);
    if (rc) return rc;
    HIP_TRY(hipMemset(ctx->marks, 0, (size_t)ctx->nmark * sizeof(int)));
    // stencil members without the cell itself
    //   tiled: [tile][imax][8*ts], lane position 8-cell-tile local
    //   CWENO at WENO-5: central [tile][imax][8], sectors [tile][imax2][8*(ts-1)]
    //   plain: [cell][ts][imax]
    const int IMC = ctx->cw_cell ? ctx->imax2 : 0, NS = std::max(ts - 1, 1);
    std::vector<int32_t> nbc((size_t)ctx->ntile * IMC * 8 * NS, 0);
    std::vector<int32_t> nbr(ctx->smode     ? (size_t)0
                             : ctx->tiled   ? (size_t)ctx->ntile * IM * 8 * ts
                             : ctx->cw_cell ? (size_t)ctx->ntile * IM * 8
                                            : (size_t)nc * ts * IM,
                             0);
    for (int i = 0; i < nc; ++i) {
        const size_t o = src_cell(ctx, i);
        for (int s = 0; s < pre->admis[o]; ++s) {
            const int32_t *row = pre->ihexl + (o * TSA + s) * NNB;
            if ((size_t)(row[0] - base) != o) {
                ctx->err = "IHEXL(s,1) must be the cell itself (cell " + std::to_string(o) + ")";
                return UCNS_EBADARG;
            }
            for (int k = 0; k < IM; ++k) {
                const int jo = row[k + 1] - base;
                if (jo < 0 || jo >= nc) {
                    ctx->err = "stencil member out of range at cell " + std::to_string(o);
                    return UCNS_EBADARG;
                }
                const int j = lib_cell(ctx, jo);
                if (ctx->smode) {
                    continue;  // carried by the row stream
                } else if (ctx->tiled) {
                    const size_t TP = 8 * (size_t)ts;
                    nbr[((size_t)(i / 8) * IM + k) * TP + (size_t)(i % 8) * ts + s] = j;
                } else if (ctx->cw_cell) {
                    if (s == 0)
                        nbr[((size_t)(i / 8) * IM + k) * 8 + i % 8] = j;
                    else if (k < IMC)
                        nbc[((size_t)(i / 8) * IMC + k) * 8 * NS + (size_t)(i % 8) * NS + s - 1] = j;
                } else {
                    nbr[((size_t)i * ts + s) * IM + k] = j;
                }
            }
        }
    }
    if ((rc = dalloc(ctx, &ctx->nbr, std::max<size_t>(nbr.size(), 1)))) return rc;
    if (!nbr.empty())
        HIP_TRY(hipMemcpy(ctx->nbr, nbr.data(), nbr.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    if (!nbc.empty()) {
        if ((rc = dalloc(ctx, &ctx->nbc, nbc.size()))) return rc;
        HIP_TRY(hipMemcpy(ctx->nbc, nbc.data(), nbc.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    }
    HIP_TRY(hipMemcpy(ctx->cinfo, cinfo.data(), nc * sizeof(int32_t), hipMemcpyHostToDevice));
    // pseudo-inverses: staged in chunks, re-laid out on the device (CWENO at
    // WENO-5: the central stencil's only)
    const int tsP = ctx->cw_cell ? 1 : ts;
    const size_t per_cell_abi = (size_t)TSA * IM * ID, per_cell_dev = (size_t)IM * tsP * ID;
    const size_t dev_elems = ctx->smode ? 1 : ctx->tiled || ctx->cw_cell ? (size_t)ctx->ntile * 8 * per_cell_dev : per_cell_dev * nc;
    rc = mixed ? dalloc(ctx, (float **)&ctx->P, dev_elems) : dalloc(ctx, (double **)&ctx->P, dev_elems);
    if (rc) return rc;
    const int sTP = 8 * ts, sD = stream_depth(mixed, ts), sPB = ID * sTP * (mixed ? 4 : 8);
    const int sRD = sPB + sTP * 4, sHD = sD * sTP * 4;
    if (ctx->smode) {
        ctx->tile_bytes = sHD + (long long)IM * sRD;
        if ((rc = dalloc(ctx, &ctx->rows, (size_t)ctx->ntile * ctx->tile_bytes))) return rc;
        if ((rc = dalloc(ctx, &ctx->u64, (size_t)nc * 8))) return rc;
        // member-index rows: row r holds members j = r (zero past imax)
        const size_t rows = (size_t)sD + IM;
        std::vector<int32_t> idx((size_t)ctx->ntile * rows * sTP, 0);
        for (int i = 0; i < nc; ++i) {
            const size_t o = src_cell(ctx, i);
            for (int s = 0; s < pre->admis[o]; ++s) {
                const int32_t *row = pre->ihexl + (o * TSA + s) * NNB;
                for (int r = 0; r < IM; ++r)
                    idx[((size_t)(i / 8) * rows + r) * sTP + (size_t)(i % 8) * ts + s] = lib_cell(ctx, row[r + 1] - base);
            }
        }
        int32_t *didx = nullptr;
        if ((rc = dalloc(ctx, &didx, idx.size()))) return rc;
        HIP_TRY(hipMemcpy(didx, idx.data(), idx.size() * sizeof(int32_t), hipMemcpyHostToDevice));
        hipLaunchKernelGGL(k_stream_idx, dim3(4096), dim3(256), 0, ctx->stream, didx, ctx->rows, ctx->ntile, sD, IM,
                           sTP, sHD, sPB, sRD, ctx->tile_bytes);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(ctx->stream));
        dfree(didx);
    }
    {
        size_t chunk_cells = std::max<size_t>(8, (size_t)(256u << 20) / (per_cell_abi * sizeof(double)));
        chunk_cells -= chunk_cells % 8;
        double *stage = nullptr, *host_pin = nullptr;
        if ((rc = dalloc(ctx, &stage, chunk_cells * per_cell_abi))) return rc;
        if (hipHostMalloc((void **)&host_pin, chunk_cells * per_cell_abi * sizeof(double), hipHostMallocDefault) !=
            hipSuccess)
            host_pin = nullptr;
        std::vector<double> host_buf;  // pageable staging when pinned memory is refused and cells move
        if (!host_pin && (!ctx->h_perm.empty() || ctx->ees == 5)) host_buf.resize(chunk_cells * per_cell_abi);
        double *gather = host_pin ? host_pin : host_buf.data();
        for (size_t c0 = 0; c0 < (size_t)nc; c0 += chunk_cells) {
            const size_t cn = std::min(chunk_cells, (size_t)nc - c0);
            const size_t bytes = cn * per_cell_abi * sizeof(double);
            const double *src = pre->invmat + c0 * per_cell_abi;
            if (!ctx->h_perm.empty() || ctx->ees == 5) {  // the chunk's cells from their places in the caller's order
                for (size_t c = 0; c < cn; ++c)
                    std::memcpy(gather + c * per_cell_abi, pre->invmat + src_cell(ctx, (int)(c0 + c)) * per_cell_abi,
                                per_cell_abi * sizeof(double));
                if (ctx->ees == 5 && ctx->tiled) {
                    // CWENO: a sector's rows are its low-order pseudo-inverse, zero
                    // past idegfree2 coefficients and imax2 members
                    const int ID2 = ctx->ideg2, IM2 = ctx->imax2;
                    for (size_t c = 0; c < cn; ++c)
                        for (int st = 1; st < TSA; ++st) {
                            double *Pd = gather + c * per_cell_abi + (size_t)st * IM * ID;
                            const double *Pc = ctx->h_cwP.data() + (((c0 + c) * TSA + st) * IM2) * ID2;
                            std::fill(Pd, Pd + (size_t)IM * ID, 0.0);
                            for (int j = 0; j < IM2; ++j)
                                for (int k = 0; k < ID2; ++k) Pd[(size_t)j * ID + k] = Pc[(size_t)j * ID2 + k];
                        }
                }
                src = gather;
            } else if (host_pin) {
                std::memcpy(host_pin, src, bytes);
                src = host_pin;
            }
            HIP_TRY(hipMemcpyAsync(stage, src, bytes, hipMemcpyHostToDevice, ctx->stream));
            if (ctx->smode) {
                const int blocks = (int)std::min<size_t>(4096, (cn * per_cell_dev + 255) / 256);
                if (mixed)
                    hipLaunchKernelGGL(k_stream_p<float>, dim3(blocks), dim3(256), 0, ctx->stream, stage,
                                       ctx->rows, (int)c0, (int)cn, TSA, ts, IM, ID, sHD, sRD, ctx->tile_bytes);
                else
                    hipLaunchKernelGGL(k_stream_p<double>, dim3(blocks), dim3(256), 0, ctx->stream, stage,
                                       ctx->rows, (int)c0, (int)cn, TSA, ts, IM, ID, sHD, sRD, ctx->tile_bytes);
            } else if (ctx->tiled) {
                const size_t out_elems = ((cn + 7) / 8) * 8 * per_cell_dev;
                const int blocks = (int)std::min<size_t>(4096, (out_elems + 255) / 256);
                if (mixed)
                    hipLaunchKernelGGL(k_tile_p<float>, dim3(blocks), dim3(256), 0, ctx->stream, stage,
                                       (float *)ctx->P + c0 * per_cell_dev, (int)c0, (int)cn, nc, TSA, ts, IM, ID);
                else
                    hipLaunchKernelGGL(k_tile_p<double>, dim3(blocks), dim3(256), 0, ctx->stream, stage,
                                       (double *)ctx->P + c0 * per_cell_dev, (int)c0, (int)cn, nc, TSA, ts, IM, ID);
            } else if (ctx->cw_cell) {
                if (mixed)
                    cweno5_rows(stage, (float *)ctx->P, (int)c0, (int)cn, TSA, ctx->stream);
                else
                    cweno5_rows(stage, (double *)ctx->P, (int)c0, (int)cn, TSA, ctx->stream);
            } else {
                const int blocks = (int)std::min<size_t>(4096, (cn * per_cell_dev + 255) / 256);
                if (mixed)
                    hipLaunchKernelGGL(k_relayout_p<float>, dim3(blocks), dim3(256), 0, ctx->stream, stage,
                                       (float *)ctx->P + c0 * per_cell_dev, (int)cn, TSA, tsP, IM, ID);
                else
                    hipLaunchKernelGGL(k_relayout_p<double>, dim3(blocks), dim3(256), 0, ctx->stream, stage,
                                       (double *)ctx->P + c0 * per_cell_dev, (int)cn, TSA, tsP, IM, ID);
            }
            HIP_TRY(hipGetLastError());
            HIP_TRY(hipStreamSynchronize(ctx->stream));
        }
        dfree(stage);
        if (host_pin) (void)hipHostFree(host_pin);
    }
    // indicators, packed upper triangle
    if (ctx->cw_cell) {
        // by columns, entry by entry for the 8 cells of a tile
        const size_t np = (size_t)ID * (ID + 1) / 2;
        std::vector<double> bp((size_t)ctx->ntile * 8 * np, 0.0);
        for (int i = 0; i < nc; ++i) {
            const double *Bi = pre->indicator + src_cell(ctx, i) * ID * ID;
            double *bt = bp.data() + (size_t)(i / 8) * np * 8 + i % 8;
            for (int l = 0; l < ID; ++l)
                for (int k = 0; k <= l; ++k) bt[((size_t)l * (l + 1) / 2 + k) * 8] = Bi[(size_t)k * ID + l];
        }
        if ((rc = upload_real_any(ctx, &ctx->B, bp))) return rc;
    } else if (ctx->iweno == 1) {
        const size_t np = (size_t)ID * (ID + 1) / 2;
        std::vector<double> bp((size_t)nc * np);
        for (int i = 0; i < nc; ++i) {
            const double *Bi = pre->indicator + src_cell(ctx, i) * ID * ID;
            size_t e = (size_t)i * np;
            for (int k = 0; k < ID; ++k)
                for (int l = k; l < ID; ++l) bp[e++] = Bi[(size_t)k * ID + l];
        }
        // zero pad: the tile loads move whole 16-byte pieces, the last of
        // which may reach past the final cell's block
        bp.resize(bp.size() + 512, 0.0);
        if ((rc = upload_real_any(ctx, &ctx->B, bp))) return rc;
    } else {
        std::vector<double> bp(1, 0.0);
        if ((rc = upload_real_any(ctx, &ctx->B, bp))) return rc;
    }
    // basis means
    {
        std::vector<double> mb((size_t)nc * ID);
        ctx->h_vol11.resize(nc);
        for (int i = 0; i < nc; ++i) {
            const size_t o = src_cell(ctx, i);
            ctx->h_vol11[i] = pre->volume11[o];
            const double oov = 1.0 / pre->volume11[o];
            for (int d = 0; d < ID; ++d) mb[(size_t)i * ID + d] = pre->integ_basis[o * ID + d] * oov;
        }
        // zero pad, as B: the row-stream kernels stage a tile's means in LDS
        // with whole 16-byte pieces
        mb.resize(mb.size() + 512, 0.0);
        if ((rc = upload_real_any(ctx, &ctx->mbar, mb))) return rc;
        if (ctx->ees == 5) {
            // the sectors' indicators (packed) and mbar - mbar_c over their coefficients
            const int ID2 = ctx->ideg2, NB2 = ID2 * (ID2 + 1) / 2;
            std::vector<double> bc((size_t)nc * NB2), dm((size_t)nc * ID2);
            for (int i = 0; i < nc; ++i) {
                const double *Bi = ctx->h_cwB.data() + (size_t)i * ID2 * ID2;
                size_t e = (size_t)i * NB2;
                for (int k = 0; k < ID2; ++k)
                    for (int l = k; l < ID2; ++l) bc[e++] = Bi[(size_t)k * ID2 + l];
                const size_t o = src_cell(ctx, i);
                const double oov = 1.0 / pre->volume11[o];
                for (int d = 0; d < ID2; ++d)
                    dm[(size_t)i * ID2 + d] = mb[(size_t)i * ID + d] - ctx->h_cwIB[(size_t)i * ID2 + d] * oov;
            }
            if ((rc = upload_real_any(ctx, &ctx->Bc, bc)) || (rc = upload_real_any(ctx, &ctx->dmb, dm))) return rc;
            if (ctx->cw_cell) {
                // the sectors' low-order pseudo-inverses, stencils 2..ts, as member rows
                const int IM2 = ctx->imax2;
                const size_t pc = (size_t)IM2 * ID2, tp = (size_t)8 * NS;
                std::vector<double> P2((size_t)ctx->ntile * pc * tp, 0.0);
                for (int t = 0; t < ctx->ntile; ++t) {
                    const int i0 = t * 8, nt = std::min(8, nc - i0);
                    double *dst = P2.data() + (size_t)t * pc * tp;
                    for (size_t e = 0; e < pc; ++e, dst += tp)
                        for (int c = 0; c < nt; ++c)
                            for (int st = 1; st < ts; ++st)
                                dst[c * NS + st - 1] = ctx->h_cwP[((size_t)(i0 + c) * TSA + st) * pc + e];
                }
                if ((rc = upload_real_any(ctx, &ctx->Pc, P2))) return rc;
            }
        }
    }
    // Gauss points in the local frames: [cell][nf][nqm][3]
    {
        const int nf = ctx->nf, nqm = ctx->nqm, nfa = ctx->nf_abi, nqa = ctx->nqm_abi;
        std::vector<double> q((size_t)nc * nf * nqm * 3 + 512, 0.0);  // zero pad, as the means
        for (int i = 0; i < nc; ++i)
            for (int f = 0; f < nf; ++f)
                for (int g = 0; g < nqm && g < nqa; ++g)
                    for (int d = 0; d < 3; ++d)
                        q[(((size_t)i * nf + f) * nqm + g) * 3 + d] =
                            pre->qpoints[((src_cell(ctx, i) * nfa + f) * nqa + g) * 3 + d];
        if ((rc = upload_real_any(ctx, &ctx->qp, q))) return rc;
    }
    if (ctx->bmode && (rc = ensure_members(ctx))) return rc;
    if (ctx->bmode && ctx->wenwrt == 1) {
        // A tile with more distinct members than the table in LDS holds (cells in
        // an order without locality) has no rows in flight in the block kernel,
        // and one such tile holds the launch up: 3,375 shuffled hexahedra in FP64
        // take 88.6 us a stage on it, 61.7 on the row stream, which gathers every
        // member and does not care (mixed 75.0 and 50.1).  The characteristic
        // kernel has no such stand-in and stays (2,058 shuffled tetrahedra 72 us,
        // 136 with one wave per cell).
        std::vector<int32_t> uc(ctx->ntile);
        HIP_TRY(hipMemcpyAsync(uc.data(), ctx->mem_count, uc.size() * sizeof(int32_t), hipMemcpyDeviceToHost,
                               ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
        if (*std::max_element(uc.begin(), uc.end()) > ctx->uq_cap) {
            ctx->bmode = false;
            release_members(ctx);
        }
    }
    ctx->have_prestore = true;
    ctx->st.bytes_recon_per_cell =
        (double)((size_t)IM * ts * ID * (mixed ? 4 : 8)) + (ctx->iweno == 1 ? (double)ID * (ID + 1) / 2 * (mixed ? 4 : 8) : 0) +
        (double)ts * IM * 4 + (double)ctx->nf * ctx->nqm * 3 * (mixed ? 4 : 8) + (double)ID * (mixed ? 4 : 8);
    if (ctx->cw_cell) {
        // central P, the sectors' low-order P, both indicators, the members read, mbar - mbar_c
        const int ID2 = ctx->ideg2, IM2 = ctx->imax2, r = mixed ? 4 : 8;
        ctx->st.bytes_recon_per_cell = (double)IM * ID * r + (double)(ts - 1) * IM2 * ID2 * r +
                                       (double)ID * (ID + 1) / 2 * r + (double)ID2 * (ID2 + 1) / 2 * r +
                                       (double)(IM + (ts - 1) * IM2) * 4 + (double)ctx->nf * ctx->nqm * 3 * r +
                                       (double)(ID + ID2) * r;
    }
    return UCNS_OK;
}

int ucns_upload_cweno(ucns_ctx *ctx, const ucns_cweno_v1 *cw) {
    if (!ctx || !cw) return UCNS_EBADARG;
    if (cw->abi_version != UCNS_ABI_VERSION) {
        ctx->err = "ucns_cweno_v1: abi_version mismatch";
        return UCNS_EBADARG;
    }
    if (ctx->ees != 5) {
        ctx->err = "ucns_upload_cweno: the scheme is not CWENO (ees 5)";
        return UCNS_ESTATE;
    }
    if (!cw->invmat_c || !cw->indicator_c || !cw->integ_basis_c) {
        ctx->err = "null CWENO array";
        return UCNS_EBADARG;
    }
    // IORDER <= 3 (idegfree 9 and 19) take linear sectors, IORDER 4 (idegfree
    // 34) quadratic ones (DETERMINE_SIZE, src/grid_p.f90:6151-6161)
    const int want2 = ctx->ideg == 34 ? 9 : 3;
    if (cw->idegfree2 != want2 || cw->inumneighbours2 < want2 + 1 || cw->inumneighbours2 > ctx->nnb) {
        ctx->err = "CWENO sectors: idegfree2 must be " + std::to_string(want2) +
                   " for this idegfree and inumneighbours2 in [idegfree2 + 1, inumneighbours]";
        return UCNS_EUNSUPPORTED;
    }
    const int nc = ctx->ncell, TSA = ctx->ts_abi, ID2 = cw->idegfree2, IM2 = cw->inumneighbours2 - 1;
    const size_t pc = (size_t)TSA * IM2 * ID2;
    ctx->h_cwP.resize((size_t)nc * pc);
    ctx->h_cwB.resize((size_t)nc * ID2 * ID2);
    ctx->h_cwIB.resize((size_t)nc * ID2);
    for (int i = 0; i < nc; ++i) {
        const size_t o = src_cell(ctx, i);
        std::memcpy(ctx->h_cwP.data() + (size_t)i * pc, cw->invmat_c + o * pc, pc * sizeof(double));
        std::memcpy(ctx->h_cwB.data() + (size_t)i * ID2 * ID2, cw->indicator_c + o * ID2 * ID2,
                    (size_t)ID2 * ID2 * sizeof(double));
        std::memcpy(ctx->h_cwIB.data() + (size_t)i * ID2, cw->integ_basis_c + o * ID2, (size_t)ID2 * sizeof(double));
    }
    ctx->ideg2 = ID2;
    ctx->imax2 = IM2;
    ctx->have_cweno = true;
    ctx->have_prestore = false;  // the pseudo-inverses are laid out again by ucns_upload_prestore
    return UCNS_OK;
}

int ucns_set_boundary(ucns_ctx *ctx, const ucns_boundary_v1 *bc) {
    if (!ctx || !bc) return UCNS_EBADARG;
    if (bc->abi_version != UCNS_ABI_VERSION) {
        ctx->err = "abi_version mismatch";
        return UCNS_EBADARG;
    }
    if (bc->boundtype != 0 && bc->boundtype != 1) {
        ctx->err = "boundtype must be 0 or 1";
        return UCNS_EBADARG;
    }
    for (int v = 0; v < NV; ++v)
        if (!std::isfinite(bc->inflow[v]) || !std::isfinite(bc->outflow[v])) {
            ctx->err = "non-finite free-stream state";
            return UCNS_EBADARG;
        }
    if (!(bc->inflow[0] > 0) || !(bc->outflow[0] > 0)) {
        ctx->err = "free-stream density must be positive";
        return UCNS_EBADARG;
    }
    ctx->bc = *bc;
    ctx->have_bc = true;
    return UCNS_OK;
}

int ucns_set_boundary_faces(ucns_ctx *ctx, const double *inflow, const double *outflow) {
    if (!ctx) return UCNS_EBADARG;
    if (!ctx->have_bc) {
        ctx->err = "call ucns_set_boundary first (BOUNDTYPE and the states of the faces not given here)";
        return UCNS_ESTATE;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    dfree(ctx->bface);
    ctx->bface = nullptr;
    if (!inflow && !outflow) return UCNS_OK;
    const int nfa = ctx->nf_abi;
    std::vector<double> h((size_t)ctx->nface * 10);
    for (int f = 0; f < ctx->nface; ++f) {
        const int code = -ctx->h_fcell[2 * f + 1];
        const int ci = ctx->h_fcell[2 * f], sl = ctx->h_fslot[2 * f] & 255;
        const size_t rec = (src_cell(ctx, ci) * nfa + sl) * NV;
        for (int v = 0; v < NV; ++v) {
            h[(size_t)f * 10 + v] = ctx->bc.inflow[v];
            h[(size_t)f * 10 + 5 + v] = ctx->bc.outflow[v];
        }
        if (code <= 0) continue;  // interior and periodic faces: no ghost
        for (int v = 0; v < NV; ++v) {
            if (inflow) h[(size_t)f * 10 + v] = inflow[rec + v];
            if (outflow) h[(size_t)f * 10 + 5 + v] = outflow[rec + v];
        }
        for (int v = 0; v < 10; ++v)
            if (!std::isfinite(h[(size_t)f * 10 + v])) {
                ctx->err = "non-finite boundary state at cell " + std::to_string(src_cell(ctx, ci)) + " face " +
                           std::to_string(sl);
                return UCNS_EBADARG;
            }
        if (!(h[(size_t)f * 10] > 0) || !(h[(size_t)f * 10 + 5] > 0)) {
            ctx->err = "boundary density must be positive (cell " + std::to_string(src_cell(ctx, ci)) + " face " +
                       std::to_string(sl) + ")";
            return UCNS_EBADARG;
        }
    }
    int rc;
    if ((rc = dalloc(ctx, &ctx->bface, h.size()))) return rc;
    HIP_TRY(hipMemcpy(ctx->bface, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
    return UCNS_OK;
}

int ucns_set_state(ucns_ctx *ctx, const double *u, int32_t layout) {
    if (!ctx || !u) return UCNS_EBADARG;
    HIP_TRY(hipSetDevice(ctx->device));
    int rc = cells_in(ctx, u, true, layout, ctx->U);
    if (rc == 0) ctx->have_state = true;
    return rc;
}

int ucns_get_state(ucns_ctx *ctx, double *u, int32_t layout) {
    if (!ctx || !u) return UCNS_EBADARG;
    HIP_TRY(hipSetDevice(ctx->device));
    return cells_out(ctx, ctx->U, layout, u, true);
}

int ucns_set_state_device(ucns_ctx *ctx, const double *u, int32_t layout) {
    if (!ctx || !u) return UCNS_EBADARG;
    HIP_TRY(hipSetDevice(ctx->device));
    int rc = cells_in(ctx, u, false, layout, ctx->U);
    if (rc == 0) ctx->have_state = true;
    return rc;
}

int ucns_get_state_device(ucns_ctx *ctx, double *u, int32_t layout) {
    if (!ctx || !u) return UCNS_EBADARG;
    HIP_TRY(hipSetDevice(ctx->device));
    return cells_out(ctx, ctx->U, layout, u, false);
}

static int ready(ucns_ctx *ctx) {
    if (ctx->needs_bc && !ctx->have_bc) {
        ctx->err = "the mesh has inflow/outflow/farfield faces: call ucns_set_boundary first";
        return UCNS_ESTATE;
    }
    if (!ctx->have_prestore) {
        ctx->err = "ucns_upload_prestore has not been called";
        return UCNS_ESTATE;
    }
    if (!ctx->have_state) {
        ctx->err = "ucns_set_state has not been called";
        return UCNS_ESTATE;
    }
    return UCNS_OK;
}

int ucns_compute_dt(ucns_ctx *ctx, double cfl, double *dt_out) {
    if (!ctx || !dt_out || !(cfl > 0)) return UCNS_EBADARG;
    if (!ctx->have_state) {
        ctx->err = "ucns_set_state has not been called";
        return UCNS_ESTATE;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    dt_kernel(ctx, cfl, ctx->dtv);
    // the least slot straight into the pinned result: a copy of the 2 KiB of slots
    // through pageable memory was up to 1 us slower than one value's had been (512
    // cells 24.2 us with one value, 25.0 with the slots, 16.7 this way)
    hipLaunchKernelGGL(k_dt_value, dim3(1), dim3(WAVE), 0, ctx->stream, (const double *)ctx->dtv, &ctx->result->t);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    *dt_out = ctx->result->t;
    return UCNS_OK;
}

int ucns_reconstruct(ucns_ctx *ctx, double *uleft_out) {
    if (!ctx || !uleft_out) return UCNS_EBADARG;
    int rc = ready(ctx);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(ctx->device));
    rc = ctx->precision == UCNS_MIXED ? launch_recon_t<float>(ctx) : launch_recon_t<double>(ctx);
    if (rc) return rc;
    HIP_TRY(hipGetLastError());
    const size_t n = (size_t)ctx->ncell * ctx->nf * ctx->nqm * NV;
    std::vector<double> d(n);
    if (ctx->precision == UCNS_MIXED) {
        std::vector<float> f(n);
        HIP_TRY(hipMemcpyAsync(f.data(), ctx->uleft, n * 4, hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
        for (size_t e = 0; e < n; ++e) d[e] = f[e];
    } else {
        HIP_TRY(hipMemcpyAsync(d.data(), ctx->uleft, n * 8, hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    // the device keeps deviations from the cell average; hand out states
    std::vector<double> u((size_t)ctx->ncell * NV);
    HIP_TRY(hipMemcpy(u.data(), ctx->U, u.size() * sizeof(double), hipMemcpyDeviceToHost));
    const int nfa = ctx->nf_abi, nqa = ctx->nqm_abi;
    std::memset(uleft_out, 0, sizeof(double) * (size_t)ctx->ncell * nfa * nqa * NV);
    for (int i = 0; i < ctx->ncell; ++i) {
        const size_t o = src_cell(ctx, i);
        for (int f = 0; f < ctx->nf; ++f)
            for (int q = 0; q < ctx->nqm; ++q)
                for (int v = 0; v < NV; ++v)
                    uleft_out[((o * nfa + f) * nqa + q) * NV + v] =
                        u[(size_t)i * NV + v] + d[(((size_t)i * ctx->nf + f) * ctx->nqm + q) * NV + v];
    }
    return collect_counts(ctx);
}

static int residual_to(ucns_ctx *ctx, double *rhs_out, int32_t layout, bool host) {
    if (!ctx) return UCNS_EBADARG;
    if (layout != UCNS_LAYOUT_AOS && layout != UCNS_LAYOUT_SOA) return UCNS_EBADARG;
    int rc = ready(ctx);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(ctx->device));
    if ((rc = residual_kernels(ctx))) return rc;
    update_kernel(ctx, 0, nullptr, false, nullptr, 0.0, ctx->rhs);
    HIP_TRY(hipGetLastError());
    if (!rhs_out) return collect_counts(ctx);
    if ((rc = queue_result(ctx, 0, nullptr))) return rc;
    if ((rc = cells_out(ctx, ctx->rhs, layout, rhs_out, host))) return rc;  // waits for the stream
    read_result(ctx, 0);
    return UCNS_OK;
}

int ucns_residual(ucns_ctx *ctx, double *rhs_out, int32_t layout) { return residual_to(ctx, rhs_out, layout, true); }

int ucns_residual_noalloc(ucns_ctx *ctx, double *rhs_dev, int32_t layout) {
    if (!ctx || !rhs_dev) return UCNS_EBADARG;
    if (layout != UCNS_LAYOUT_AOS && layout != UCNS_LAYOUT_SOA) return UCNS_EBADARG;
    int rc = ready(ctx);
    if (rc) return rc;
    const size_t need = UCNS_SCRATCH_HEAD + (size_t)ctx->nface * NV * sizeof(double);
    if (need > UCNS_SCRATCH_BYTES) {
        ctx->err = "ucns_residual_noalloc: " + std::to_string(ctx->nface) + " faces need " + std::to_string(need) +
                   " bytes of scratch, more than the library's " + std::to_string(UCNS_SCRATCH_BYTES) +
                   " (ucns_residual_device has no such limit)";
        return UCNS_EUNSUPPORTED;
    }
    if (!ctx->scratch) {
        ctx->err = "ucns_residual_noalloc: no scratch address for this device";
        return UCNS_ESTATE;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    // the same kernels as ucns_residual_device, with their face fluxes in the
    // static scratch (every face flux is written before it is read)
    double *const own_fflux = ctx->fflux;
    ctx->fflux = (double *)((unsigned char *)ctx->scratch + UCNS_SCRATCH_HEAD);
    rc = residual_kernels(ctx);
    if (rc == UCNS_OK) update_kernel(ctx, 0, nullptr, false, nullptr, 0.0, ctx->rhs);
    if (rc == UCNS_OK) rc = queue_result(ctx, 0, nullptr);
    if (rc == UCNS_OK) rc = cells_out(ctx, ctx->rhs, layout, rhs_dev, false);  // waits for the stream
    ctx->fflux = own_fflux;
    if (rc) return rc;
    read_result(ctx, 0);
    return UCNS_OK;
}

int ucns_residual_device(ucns_ctx *ctx, double *rhs_dev, int32_t layout) {
    if (!rhs_dev) return UCNS_EBADARG;
    return residual_to(ctx, rhs_dev, layout, false);
}

int ucns_rk3_steps(ucns_ctx *ctx, int32_t nsteps, double cfl, double dt_fixed, double *t_io) {
    if (!ctx || nsteps < 0) return UCNS_EBADARG;
    if (!(dt_fixed > 0) && !(cfl > 0)) {
        ctx->err = "need cfl > 0 or dt_fixed > 0";
        return UCNS_EBADARG;
    }
    int rc = ready(ctx);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(ctx->device));
    const double t0 = t_io ? *t_io : 0.0;
    const bool fixed = dt_fixed > 0;
    hipLaunchKernelGGL(k_set2, dim3(1), dim3(WAVE), 0, ctx->stream, ctx->t, t0, ctx->dtfix, dt_fixed);
    int cur = 0;
    if (!fixed && nsteps > 0) dt_kernel(ctx, cfl, ctx->dtv);
    for (int it = 0; it < nsteps; ++it) {
        const double *dt = fixed ? ctx->dtfix : (const double *)(ctx->dtv + cur * DT_SLOTS * DT_STRIDE);
        unsigned long long *next = fixed ? nullptr : ctx->dtv + (1 - cur) * DT_SLOTS * DT_STRIDE;
        // (timed marches keep the phases apart)
        if (ctx->fadj && !ctx->timing && (rc = fused_step(ctx, dt, !fixed, next, cfl))) return rc;
        for (int stage = 1; stage <= 3 && !(ctx->fadj && !ctx->timing); ++stage) {
            if ((rc = residual_kernels(ctx, it > 0 || stage > 1))) return rc;
            update_kernel(ctx, stage, dt, !fixed, next, cfl, nullptr, it + 1 < nsteps || stage < 3);
        }
        HIP_TRY(hipGetLastError());
        if (!fixed) cur = 1 - cur;
    }
    const size_t nu = (size_t)ctx->ncell * NV;
    if ((rc = queue_result(ctx, nu, ctx->t))) return rc;
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    const bool bad = read_result(ctx, nu);
    if (t_io) *t_io = ctx->result->t;
    if (bad) {
        ctx->err = "non-finite state after the RK3 steps";
        return UCNS_ENONFINITE;
    }
    return UCNS_OK;
}

int ucns_residual_vjp_device(ucns_ctx *ctx, const double *w_dev, double *u_bar_dev, double *bc_bar_dev) {
    if (!ctx || !w_dev || !u_bar_dev) return UCNS_EBADARG;
    int rc = ready(ctx);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(ctx->device));
    if ((rc = ensure_adjoint(ctx))) return rc;
    if ((rc = cells_in(ctx, w_dev, false, UCNS_LAYOUT_AOS, ctx->adj_a))) return rc;
    zero_dev(ctx, ctx->adj_bc, 2 * NV);
    if ((rc = residual_vjp_dev(ctx, ctx->adj_a, ctx->adj_x, ctx->adj_bc))) return rc;
    HIP_TRY(hipGetLastError());
    if (bc_bar_dev)
        HIP_TRY(hipMemcpyAsync(bc_bar_dev, ctx->adj_bc, 2 * NV * sizeof(double), hipMemcpyDeviceToDevice,
                               ctx->stream));
    return cells_out(ctx, ctx->adj_x, UCNS_LAYOUT_AOS, u_bar_dev, false);
}

int ucns_residual_vjp(ucns_ctx *ctx, const double *w, double *u_bar, int32_t layout, double *bc_bar) {
    if (!ctx || !w || !u_bar) return UCNS_EBADARG;
    if (layout != UCNS_LAYOUT_AOS && layout != UCNS_LAYOUT_SOA) return UCNS_EBADARG;
    int rc = ready(ctx);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(ctx->device));
    if ((rc = ensure_adjoint(ctx))) return rc;
    if ((rc = cells_in(ctx, w, true, layout, ctx->adj_a))) return rc;
    zero_dev(ctx, ctx->adj_bc, 2 * NV);
    if ((rc = residual_vjp_dev(ctx, ctx->adj_a, ctx->adj_x, ctx->adj_bc))) return rc;
    HIP_TRY(hipGetLastError());
    double bc[2 * NV];
    HIP_TRY(hipMemcpyAsync(bc, ctx->adj_bc, sizeof(bc), hipMemcpyDeviceToHost, ctx->stream));
    if ((rc = cells_out(ctx, ctx->adj_x, layout, u_bar, true))) return rc;
    if (bc_bar) std::memcpy(bc_bar, bc, sizeof(bc));
    return UCNS_OK;
}

// forward sweep with stage checkpoints + reverse sweep; a_dev holds uN_bar
// on entry and u0_bar on return
static int rk3_adjoint_impl(ucns_ctx *ctx, int32_t nsteps, double cfl, double dt_fixed, double *a_dev, double *t_io) {
    if (nsteps < 1) {
        ctx->err = "nsteps must be >= 1";
        return UCNS_EBADARG;
    }
    if (!(dt_fixed > 0) && !(cfl > 0)) {
        ctx->err = "need cfl > 0 or dt_fixed > 0";
        return UCNS_EBADARG;
    }
    int rc = ensure_adjoint(ctx);
    if (rc) return rc;
    const size_t n = (size_t)ctx->ncell * NV;
    if (ctx->ckpt_steps < (size_t)nsteps) {
        dfree(ctx->ckpt);
        dfree(ctx->dts);
        ctx->ckpt_steps = 0;
        if ((rc = dalloc(ctx, &ctx->ckpt, (size_t)3 * nsteps * n))) return rc;
        if ((rc = dalloc(ctx, &ctx->dts, (size_t)nsteps))) return rc;
        ctx->ckpt_steps = nsteps;
    }
    const int keep0 = 3 * nsteps - adj_keep(ctx, 3 * nsteps);
    const double t0 = t_io ? *t_io : 0.0;
    const bool fixed = dt_fixed > 0;
    hipLaunchKernelGGL(k_set2, dim3(1), dim3(WAVE), 0, ctx->stream, ctx->t, t0, ctx->dtfix, dt_fixed);
    int cur = 0;
    if (!fixed) dt_kernel(ctx, cfl, ctx->dtv);
    for (int it = 0; it < nsteps; ++it) {
        const double *dt = fixed ? ctx->dtfix : (const double *)(ctx->dtv + cur * DT_SLOTS * DT_STRIDE);
        unsigned long long *next = fixed ? nullptr : ctx->dtv + (1 - cur) * DT_SLOTS * DT_STRIDE;
        if (fixed)
            HIP_TRY(hipMemcpyAsync(ctx->dts + it, dt, sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
        else
            hipLaunchKernelGGL(k_dt_value, dim3(1), dim3(WAVE), 0, ctx->stream, dt, ctx->dts + it);
        if ((rc = rk3_step_ckpt(ctx, it, nsteps, dt, next, cfl, keep0))) return rc;
        HIP_TRY(hipGetLastError());
        if (!fixed) cur = 1 - cur;
    }
    zero_dev(ctx, ctx->adj_bc, 2 * NV);
    if ((rc = rk3_reverse(ctx, nsteps, a_dev, ctx->adj_bc, keep0))) return rc;
    if ((rc = queue_result(ctx, 0, ctx->t))) return rc;
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    if (t_io) *t_io = ctx->result->t;
    return UCNS_OK;
}

int ucns_rk3_adjoint_device(ucns_ctx *ctx, int32_t nsteps, double cfl, double dt_fixed, const double *uN_bar_dev,
                            double *u0_bar_dev, double *bc_bar_dev, double *t_io) {
    if (!ctx || !uN_bar_dev || !u0_bar_dev) return UCNS_EBADARG;
    int rc = ready(ctx);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(ctx->device));
    if ((rc = ensure_adjoint(ctx))) return rc;
    if ((rc = cells_in(ctx, uN_bar_dev, false, UCNS_LAYOUT_AOS, ctx->adj_a))) return rc;
    if ((rc = rk3_adjoint_impl(ctx, nsteps, cfl, dt_fixed, ctx->adj_a, t_io))) return rc;
    if (bc_bar_dev)
        HIP_TRY(hipMemcpyAsync(bc_bar_dev, ctx->adj_bc, 2 * NV * sizeof(double), hipMemcpyDeviceToDevice,
                               ctx->stream));
    return cells_out(ctx, ctx->adj_a, UCNS_LAYOUT_AOS, u0_bar_dev, false);
}

int ucns_rk3_adjoint(ucns_ctx *ctx, int32_t nsteps, double cfl, double dt_fixed, const double *uN_bar,
                     double *u0_bar, int32_t layout, double *bc_bar, double *t_io) {
    if (!ctx || !uN_bar || !u0_bar) return UCNS_EBADARG;
    if (layout != UCNS_LAYOUT_AOS && layout != UCNS_LAYOUT_SOA) return UCNS_EBADARG;
    int rc = ready(ctx);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(ctx->device));
    if ((rc = ensure_adjoint(ctx))) return rc;
    if ((rc = cells_in(ctx, uN_bar, true, layout, ctx->adj_a))) return rc;
    if ((rc = rk3_adjoint_impl(ctx, nsteps, cfl, dt_fixed, ctx->adj_a, t_io))) return rc;
    double bc[2 * NV];
    HIP_TRY(hipMemcpyAsync(bc, ctx->adj_bc, sizeof(bc), hipMemcpyDeviceToHost, ctx->stream));
    if ((rc = cells_out(ctx, ctx->adj_a, layout, u0_bar, true))) return rc;
    if (bc_bar) std::memcpy(bc_bar, bc, sizeof(bc));
    return UCNS_OK;
}

namespace {
void release_geometry(ucns_ctx *ctx) {
    dfree(ctx->geo_P);
    dfree(ctx->geo_B);
    dfree(ctx->geo_M);
    dfree(ctx->geo_Q);
    dfree(ctx->geo_area);
    dfree(ctx->geo_nrm);
    dfree(ctx->geo_ovol);
    ctx->geo_on = false;
}

int geo_download(ucns_ctx *ctx, const double *dev, std::vector<double> &host, size_t n) {
    host.resize(n);
    HIP_TRY(hipMemcpyAsync(host.data(), dev, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    return UCNS_OK;
}

// the accumulated device cotangents in the caller's arrays and cell order
int geo_to_caller(ucns_ctx *ctx, const ucns_geometry_bar_v1 *g) {
    const int nc = ctx->ncell, ID = ctx->ideg, IM = ctx->imax, ts = ctx->ts, TSA = ctx->ts_abi;
    const int nf = ctx->nf, nqm = ctx->nqm, nfa = ctx->nf_abi, nqa = ctx->nqm_abi;
    std::vector<double> P, B, M, Q, A, N, V, mb;
    int rc;
    if ((g->invmat && (rc = geo_download(ctx, ctx->geo_P, P, (size_t)nc * ts * IM * ID))) ||
        (g->indicator && ctx->iweno == 1 && (rc = geo_download(ctx, ctx->geo_B, B, (size_t)nc * ID * ID))) ||
        ((g->integ_basis || g->volume11) && (rc = geo_download(ctx, ctx->geo_M, M, (size_t)nc * ID))) ||
        (g->volume11 && (rc = geo_download(ctx, (const double *)ctx->mbar, mb, (size_t)nc * ID))) ||
        (g->qpoints && (rc = geo_download(ctx, ctx->geo_Q, Q, (size_t)nc * nf * nqm * 3))) ||
        (g->surf && (rc = geo_download(ctx, ctx->geo_area, A, (size_t)ctx->nface))) ||
        (g->normal && (rc = geo_download(ctx, ctx->geo_nrm, N, (size_t)ctx->nface * 3))) ||
        (g->totvolume && (rc = geo_download(ctx, ctx->geo_ovol, V, (size_t)nc))))
        return rc;
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    if (g->invmat) std::memset(g->invmat, 0, sizeof(double) * (size_t)nc * TSA * IM * ID);
    if (g->indicator) std::memset(g->indicator, 0, sizeof(double) * (size_t)nc * ID * ID);
    if (g->qpoints) std::memset(g->qpoints, 0, sizeof(double) * (size_t)nc * nfa * nqa * 3);
    if (g->surf) std::memset(g->surf, 0, sizeof(double) * (size_t)nc * nfa);
    if (g->normal) std::memset(g->normal, 0, sizeof(double) * (size_t)nc * nfa * 3);
    for (int i = 0; i < nc; ++i) {
        const size_t o = src_cell(ctx, i);
        if (g->invmat)
            for (int st = 0; st < std::min(ts, TSA); ++st)
                std::memcpy(g->invmat + ((o * TSA + st) * IM) * ID, P.data() + (((size_t)i * ts + st) * IM) * ID,
                            sizeof(double) * IM * ID);
        if (g->indicator && !B.empty())
            std::memcpy(g->indicator + o * ID * ID, B.data() + (size_t)i * ID * ID, sizeof(double) * ID * ID);
        // mbar = INTEG_BASIS / VOLUME(1,1)
        const double v11 = ctx->h_vol11[i];
        double vb = 0.0;
        for (int d = 0; d < ID; ++d) {
            const double m = M.empty() ? 0.0 : M[(size_t)i * ID + d];
            if (g->integ_basis) g->integ_basis[o * ID + d] = m / v11;
            if (g->volume11) vb -= m * mb[(size_t)i * ID + d] / v11;
        }
        if (g->volume11) g->volume11[o] = vb;
        if (g->qpoints)
            for (int f = 0; f < std::min(nf, nfa); ++f)
                for (int q = 0; q < std::min(nqm, nqa); ++q)
                    for (int d = 0; d < 3; ++d)
                        g->qpoints[((o * nfa + f) * nqa + q) * 3 + d] = Q[(((size_t)i * nf + f) * nqm + q) * 3 + d];
        // 1/TOTVOLUME
        if (g->totvolume) g->totvolume[o] = -V[i] * ctx->h_ovol[i] * ctx->h_ovol[i];
    }
    for (int f = 0; f < ctx->nface; ++f) {
        const size_t o = src_cell(ctx, ctx->h_fcell[2 * f]);
        const int sl = ctx->h_fslot[2 * f] & 255;
        if (g->surf) g->surf[o * nfa + sl] = A[f];
        if (g->normal)
            for (int d = 0; d < 3; ++d) g->normal[(o * nfa + sl) * 3 + d] = N[(size_t)f * 3 + d];
    }
    return UCNS_OK;
}
}  // namespace

int ucns_rk3_adjoint_geometry(ucns_ctx *ctx, int32_t nsteps, double dt_fixed, const double *uN_bar, double *u0_bar,
                              int32_t layout, double *bc_bar, const ucns_geometry_bar_v1 *gbar, double *t_io) {
    if (!ctx || !uN_bar || !u0_bar || !gbar) return UCNS_EBADARG;
    if (layout != UCNS_LAYOUT_AOS && layout != UCNS_LAYOUT_SOA) return UCNS_EBADARG;
    if (gbar->abi_version != UCNS_ABI_VERSION) {
        ctx->err = "ucns_geometry_bar_v1: abi_version mismatch";
        return UCNS_EBADARG;
    }
    if (!(dt_fixed > 0)) {
        ctx->err = "ucns_rk3_adjoint_geometry: needs dt_fixed > 0 (the step size is held fixed under the geometry)";
        return UCNS_EBADARG;
    }
    int rc = ready(ctx);
    if (rc) return rc;
    // k_recon_vjp reads any layout of the pseudo-inverses (LsqView); it takes
    // the row stream of 6 stencils, not those of 5 and 7
    if (ctx->precision != UCNS_FP64 || (ctx->smode && ctx->smode != 6)) {
        ctx->err = "ucns_rk3_adjoint_geometry: needs an FP64 context on the register kernels "
                   "(precision UCNS_FP64; kernels UCNS_KERNELS_REGISTER where the row-stream kernels would run)";
        return UCNS_EUNSUPPORTED;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    // from here on every product is the geometry product; its arrays go with the call
    struct Scope {
        ucns_ctx *ctx;
        explicit Scope(ucns_ctx *c) : ctx(c) { c->geo_on = true; }
        ~Scope() { release_geometry(ctx); }
    } scope(ctx);
    if ((rc = ensure_adjoint(ctx))) return rc;
    const size_t nc = ctx->ncell;
    if ((rc = dalloc(ctx, &ctx->geo_P, nc * ctx->ts * ctx->imax * ctx->ideg)) ||
        (rc = dalloc(ctx, &ctx->geo_B, nc * ctx->ideg * ctx->ideg)) || (rc = dalloc(ctx, &ctx->geo_M, nc * ctx->ideg)) ||
        (rc = dalloc(ctx, &ctx->geo_Q, nc * ctx->nf * ctx->nqm * 3)) ||
        (rc = dalloc(ctx, &ctx->geo_area, (size_t)ctx->nface)) ||
        (rc = dalloc(ctx, &ctx->geo_nrm, (size_t)ctx->nface * 3)) || (rc = dalloc(ctx, &ctx->geo_ovol, nc)))
        return rc;
    zero_dev(ctx, ctx->geo_P, nc * ctx->ts * ctx->imax * ctx->ideg);
    zero_dev(ctx, ctx->geo_B, nc * ctx->ideg * ctx->ideg);
    zero_dev(ctx, ctx->geo_M, nc * ctx->ideg);
    zero_dev(ctx, ctx->geo_Q, nc * ctx->nf * ctx->nqm * 3);
    zero_dev(ctx, ctx->geo_area, (size_t)ctx->nface);
    zero_dev(ctx, ctx->geo_nrm, (size_t)ctx->nface * 3);
    zero_dev(ctx, ctx->geo_ovol, nc);
    if ((rc = cells_in(ctx, uN_bar, true, layout, ctx->adj_a)) == UCNS_OK)
        rc = rk3_adjoint_impl(ctx, nsteps, 0.0, dt_fixed, ctx->adj_a, t_io);
    double bc[2 * NV];
    if (rc == UCNS_OK && hipMemcpyAsync(bc, ctx->adj_bc, sizeof(bc), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess)
        rc = UCNS_EHIP;
    if (rc == UCNS_OK) rc = cells_out(ctx, ctx->adj_a, layout, u0_bar, true);
    if (rc == UCNS_OK) rc = geo_to_caller(ctx, gbar);
    if (rc == UCNS_EHIP && ctx->err.empty()) ctx->err = "ucns_rk3_adjoint_geometry: HIP error";
    if (rc) return rc;
    if (bc_bar) std::memcpy(bc_bar, bc, sizeof(bc));
    return UCNS_OK;
}

int ucns_stats(ucns_ctx *ctx, ucns_stats_v1 *out) {
    if (!ctx || !out) return UCNS_EBADARG;
    *out = ctx->st;
    return UCNS_OK;
}

int ucns_debug_fail_alloc(ucns_ctx *ctx, int32_t nth) {
    if (!ctx || nth < 0) return UCNS_EBADARG;
    ctx->fail_alloc_in = nth;
    return UCNS_OK;
}

int ucns_reset_stats(ucns_ctx *ctx) {
    if (!ctx) return UCNS_EBADARG;
    const double b = ctx->st.bytes_recon_per_cell;
    ctx->st = ucns_stats_v1{};
    ctx->st.bytes_recon_per_cell = b;
    ctx->timing = true;
    return UCNS_OK;
}

void ucns_destroy(ucns_ctx *ctx) {
    if (!ctx) return;
    if (!ctx->stream) {  // rejected before any device resource was created
        delete ctx;
        return;
    }
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    release_prestore(ctx);
    release_adjoint(ctx);
    dfree(ctx->cinfo);
    dfree(ctx->cnb);
    dfree(ctx->chnb);
    dfree(ctx->chang);
    dfree(ctx->bface);
    dfree(ctx->cface);
    dfree(ctx->fcell);
    dfree(ctx->fslot);
    dfree(ctx->frot);
    dfree(ctx->farea);
    dfree(ctx->ovol);
    dfree(ctx->minedge);
    dfree(ctx->wquad);
    dfree(ctx->stage);
    dfree(ctx->perm);
    dfree(ctx->U);
    dfree(ctx->U2);
    dfree(ctx->U3);
    dfree(ctx->fadj);
    dfree(ctx->rhs);
    dfree(ctx->fflux);
    dfree(ctx->t);
    dfree(ctx->dtfix);
    dfree(ctx->dtv);
    if (ctx->result) (void)hipHostFree(ctx->result);
    ctx->result = nullptr;
    dfree(ctx->bfaces);
    dfree(ctx->uleft);
    for (auto &e : ctx->ev)
        if (e) (void)hipEventDestroy(e);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

}  // extern "C"
