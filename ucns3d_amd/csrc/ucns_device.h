// Device code shared by the library's translation units: constants, kernel
// parameter blocks, the basis, dual numbers, face frames and boundary states,
// lane-group helpers and direct global->LDS loads.
#ifndef UCNS_DEVICE_H
#define UCNS_DEVICE_H

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ucns.h"

namespace ucns {

constexpr int NV = 5;
constexpr int WAVE = 64;
constexpr int NXCD = 8;
// distinct stencil members of a tile held in LDS by the residual product's scatter
#define UCNS_TILE_UQ 512
#define UCNS_NOSLOT 0xFFFFu
// rows of a tile's member table: 8 neighbouring cells share about 343
// distinct members with WENO-4 on tets (5 stencils), 373 with WENO-3 on
// hexes, 660 with WENO-4 on hexes (7 stencils of 39 members)
constexpr int tile_uq(int ts, int imax) { return ts > 5 && imax > 19 ? 768 : UCNS_TILE_UQ; }
constexpr int NPART = 256;  // blocks (and results) of k_finish
struct HostResult {
    int part[NPART][4];  // per block: reduced cells, first-order cells, non-finite values, 0
    double t;
};
// monomial exponents of BASIS_REC (src/basis.f90:11-102), cubic max here
static __constant__ int8_t c_mono[34][3] = {
    {1, 0, 0}, {0, 1, 0}, {0, 0, 1},
    {2, 0, 0}, {1, 1, 0}, {0, 2, 0}, {1, 0, 1}, {0, 1, 1}, {0, 0, 2},
    {3, 0, 0}, {2, 1, 0}, {1, 2, 0}, {0, 3, 0}, {2, 0, 1}, {1, 1, 1}, {0, 2, 1}, {1, 0, 2}, {0, 1, 2}, {0, 0, 3},
    {4, 0, 0}, {3, 1, 0}, {2, 2, 0}, {1, 3, 0}, {0, 4, 0}, {3, 0, 1}, {2, 1, 1}, {1, 2, 1}, {0, 3, 1},
    {2, 0, 2}, {1, 1, 2}, {0, 2, 2}, {1, 0, 3}, {0, 1, 3}, {0, 0, 4}};


// per-cell info word
//   bits 0-2 ifca, 3-5 admis, 6 full, 8-13 face k is a triangle
__host__ __device__ inline int ci_ifca(int w) { return w & 7; }
__host__ __device__ inline int ci_admis(int w) { return (w >> 3) & 7; }
__host__ __device__ inline int ci_full(int w) { return (w >> 6) & 1; }
__host__ __device__ inline int ci_tri(int w, int f) { return (w >> (8 + f)) & 1; }

template <typename R>
struct ReconParams {
    int ncell, nf, nqm, ts, per_xcd;
    int qpq, qpt;
    double gamma, lwci1, eps;
    const double *U;       // [ncell][5]
    const int32_t *nbr;    // [ncell][ts][imax]
    const R *P;            // [ncell][imax][ts][ideg]
    const R *B;            // [ncell][ideg*(ideg+1)/2] packed upper triangle by rows
    const R *mbar;         // [ncell][ideg] INTEG_BASIS/VOLUME(1,1)
    const R *qp;           // [ncell][nf][nqm][3]
    const int32_t *cinfo;  // [ncell]
    const int32_t *cnb;    // [ncell][nf] face neighbours
    R *uleft;              // [ncell][nf][nqm][5]
    int *marks;            // [ncell], or per tile: MUSCL cells + 65536 * first-order cells (summed by k_finish)
    // characteristic WENO (wenwrt 2): per cell face the neighbour (negative:
    // the boundary code) and the cell's own face angles (cos a1, sin a1, cos
    // a2, sin a2); the free-stream data of the boundary ghosts
    const int32_t *chnb;   // [ncell][nf]
    const double *chang;   // [ncell][nf][4]
    ucns_boundary_v1 bc;
    const int32_t *cface;  // [ncell][nf] +(face+1) where the cell owns the face
    const double *bface;   // [nface][10] per-face INFLOW(), OUTFLOW() states, or null: bc's
};

__device__ inline void cons2prim_d(double gamma, const double *u, double *w) {
    double oo = 1.0 / u[0];
    w[0] = u[0];
    w[1] = u[1] * oo;
    w[2] = u[2] * oo;
    w[3] = u[3] * oo;
    w[4] = (gamma - 1.0) * (u[4] - 0.5 * u[0] * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]));
}

// ---------------------------------------------------------------------------
// Forward-mode dual numbers for the adjoint: the same scalar code as the
// primal, run on (value, one directional derivative).  Branches follow the
// value, so the derivative is the one of the branch the primal takes.
struct Dual {
    double v, d;
};
// the Dual overloads below would otherwise hide the global math functions
using ::fabs;
using ::fmax;
using ::fmin;
using ::sqrt;
__device__ inline double val(double x) { return x; }
__device__ inline double val(const Dual &x) { return x.v; }
__device__ inline Dual operator+(Dual a, Dual b) { return {a.v + b.v, a.d + b.d}; }
__device__ inline Dual operator-(Dual a, Dual b) { return {a.v - b.v, a.d - b.d}; }
__device__ inline Dual operator-(Dual a) { return {-a.v, -a.d}; }
__device__ inline Dual operator*(Dual a, Dual b) { return {a.v * b.v, a.d * b.v + a.v * b.d}; }
__device__ inline Dual operator/(Dual a, Dual b) {
    const double q = a.v / b.v;
    return {q, (a.d - q * b.d) / b.v};
}
__device__ inline Dual operator+(double a, Dual b) { return {a + b.v, b.d}; }
__device__ inline Dual operator+(Dual a, double b) { return {a.v + b, a.d}; }
__device__ inline Dual operator-(double a, Dual b) { return {a - b.v, -b.d}; }
__device__ inline Dual operator-(Dual a, double b) { return {a.v - b, a.d}; }
__device__ inline Dual operator*(double a, Dual b) { return {a * b.v, a * b.d}; }
__device__ inline Dual operator*(Dual a, double b) { return {a.v * b, a.d * b}; }
__device__ inline Dual operator/(Dual a, double b) { return {a.v / b, a.d / b}; }
__device__ inline Dual operator/(double a, Dual b) {
    const double q = a / b.v;
    return {q, -q * b.d / b.v};
}
__device__ inline Dual sqrt(Dual a) {
    const double r = ::sqrt(a.v);
    return {r, a.d / (2.0 * r)};
}
__device__ inline Dual fabs(Dual a) { return a.v < 0.0 ? -a : a; }
__device__ inline Dual fmin(Dual a, Dual b) { return (b.v < a.v) ? b : a; }
__device__ inline Dual fmax(Dual a, Dual b) { return (b.v > a.v) ? b : a; }
__device__ inline Dual fmin(Dual a, double b) { return (b < a.v) ? Dual{b, 0.0} : a; }
__device__ inline Dual fmax(Dual a, double b) { return (b > a.v) ? Dual{b, 0.0} : a; }

template <class T>
__device__ inline void cons2prim_t(double gamma, const T *u, T *w) {
    T oo = 1.0 / u[0];
    w[0] = u[0];
    w[1] = u[1] * oo;
    w[2] = u[2] * oo;
    w[3] = u[3] * oo;
    w[4] = (gamma - 1.0) * (u[4] - 0.5 * u[0] * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]));
}

// CHECKSOL / CHECKSOLX test of one face point against the cell average
// (src/reconstruct_p.f90:3183-3196): primitive recovery in FP64.
__device__ inline bool jump_test(double gamma, const double *wi, const double *uq, double jump) {
    double wq[NV];
    cons2prim_d(gamma, uq, wq);
    if (fabs(wq[0] - wi[0]) >= jump * wi[0]) return true;
    if (fabs(wq[4] - wi[4]) >= jump * wi[4]) return true;
    if (wq[4] < 0.0 || wq[0] < 0.0) return true;
    return false;
}

template <typename R, int IDEG>
__device__ inline void basis_at(const R *x, const R *mbar, R *phi) {
    R px[5], py[5], pz[5];
    px[0] = py[0] = pz[0] = R(1);
#pragma unroll
    for (int k = 1; k < 5; ++k) {
        px[k] = px[k - 1] * x[0];
        py[k] = py[k - 1] * x[1];
        pz[k] = pz[k - 1] * x[2];
    }
#pragma unroll
    for (int d = 0; d < IDEG; ++d) phi[d] = px[c_mono[d][0]] * py[c_mono[d][1]] * pz[c_mono[d][2]] - mbar[d];
}

__device__ inline double wave_min(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, WAVE));
    return v;
}

// Eigenvectors of the x-split Euler flux Jacobian at the average of two
// rotated states (COMPUTE_EIGENVECTORS, src/flow_operations.f90:3934-3995):
// density, velocity and total energy averaged arithmetically; R columns
// (u-a, u, v-shear, w-shear, u+a), L = R^-1 in the textbook form with
// b = (gamma-1)/a^2.  Row-major [5][5].
__device__ inline void char_eigen_d(double gamma, const double *rl, const double *rr, double *R, double *L) {
    const double rs = 0.5 * (rl[0] + rr[0]);
    const double us = 0.5 * (rl[1] / rl[0] + rr[1] / rr[0]);
    const double vs = 0.5 * (rl[2] / rl[0] + rr[2] / rr[0]);
    const double ws = 0.5 * (rl[3] / rl[0] + rr[3] / rr[0]);
    const double es = 0.5 * (rl[4] + rr[4]);
    const double q2 = us * us + vs * vs + ws * ws;
    const double ps = (gamma - 1.0) * (es - 0.5 * rs * q2);
    const double as = sqrt(gamma * ps / rs);
    const double hs = 0.5 * q2 + as * as / (gamma - 1.0);
    const double b = (gamma - 1.0) / (as * as), bq = 0.5 * b * q2, oa = 1.0 / as;
    const double Rm[25] = {1.0, 1.0, 0.0, 0.0, 1.0,
                           us - as, us, 0.0, 0.0, us + as,
                           vs, vs, 1.0, 0.0, vs,
                           ws, ws, 0.0, 1.0, ws,
                           hs - us * as, 0.5 * q2, vs, ws, hs + us * as};
    const double Lm[25] = {0.5 * (bq + us * oa), -0.5 * (b * us + oa), -0.5 * b * vs, -0.5 * b * ws, 0.5 * b,
                           1.0 - bq, b * us, b * vs, b * ws, -b,
                           -vs, 0.0, 1.0, 0.0, 0.0,
                           -ws, 0.0, 0.0, 1.0, 0.0,
                           0.5 * (bq - us * oa), -0.5 * (b * us - oa), -0.5 * b * vs, -0.5 * b * ws, 0.5 * b};
    for (int e = 0; e < 25; ++e) {
        R[e] = Rm[e];
        L[e] = Lm[e];
    }
}

// ---------------------------------------------------------------------------
// Ghost states of boundary faces: BOUNDARYS (src/flow_operations.f90:2860-3375),
// Euler 3D without a rotating frame, in FP64 in both precisions.
#define UCNS_TOLSMALL 1.0e-13  // src/grid_p.f90:18

template <class T>
__device__ inline void bc_prim2cons(double gamma, const T *s3, T *cr) {
    cr[0] = s3[0];
    cr[1] = s3[1] * s3[0];
    cr[2] = s3[2] * s3[0];
    cr[3] = s3[3] * s3[0];
    const T skins = 0.5 * ((s3[1] * s3[1]) + (s3[2] * s3[2]) + (s3[3] * s3[3]));
    const T ikins = s3[4] / ((gamma - 1.0) * (s3[0]));
    cr[4] = (s3[0] * (ikins)) + (s3[0] * skins);
}

// subsonic inflow (src/flow_operations.f90:2907-2915): s1 free stream, s2 interior
template <class T, class F, class N>
__device__ inline void bc_sub_in(double gamma, const F *s1, const T *s2, T sps, N nx, N ny, N nz, T *cr) {
    T s3[NV];
    s3[4] = 0.5 * ((s1[4]) + (s2[4]) - (s2[0] * sps * ((nx * (s1[1] - s2[1])) + (ny * (s1[2] - s2[2])) + (nz * (s1[3] - s2[3])))));
    s3[0] = s1[0] + (s3[4] - s1[4]) / (sps * sps);
    s3[1] = s1[1] - (nx * (s1[4] - s3[4])) / (sps * s2[0]);
    s3[2] = s1[2] - (ny * (s1[4] - s3[4])) / (sps * s2[0]);
    s3[3] = s1[3] - (nz * (s1[4] - s3[4])) / (sps * s2[0]);
    bc_prim2cons(gamma, s3, cr);
}

// subsonic outflow (src/flow_operations.f90:2995-3010): s1 free stream, s2 interior
template <class T, class F, class N>
__device__ inline void bc_sub_out(double gamma, const F *s1, const T *s2, T sps, N nx, N ny, N nz, T *cr) {
    T s3[NV];
    s3[4] = T{s1[4]};
    s3[0] = s2[0] + (s3[4] - s2[4]) / (sps * sps);
    s3[1] = s2[1] + (nx * (s2[4] - s3[4])) / (sps * s2[0]);
    s3[2] = s2[2] + (ny * (s2[4] - s3[4])) / (sps * s2[0]);
    s3[3] = s2[3] + (nz * (s2[4] - s3[4])) / (sps * s2[0]);
    bc_prim2cons(gamma, s3, cr);
}

// ROTATEF / ROTATEB with precomputed cos/sin of the face angles
template <class T>
__device__ inline void rotf(const T *a, double c1, double s1, double c2, double s2, T *r) {
    r[0] = a[0];
    r[1] = c1 * s2 * a[1] + s1 * s2 * a[2] + c2 * a[3];
    r[2] = c1 * c2 * a[1] + s1 * c2 * a[2] + (-s2) * a[3];
    r[3] = (-s1) * a[1] + c1 * a[2];
    r[4] = a[4];
}
template <class T>
__device__ inline void rotb(const T *h, double c1, double s1, double c2, double s2, T *r) {
    r[0] = h[0];
    r[1] = c1 * s2 * h[1] + c1 * c2 * h[2] + (-s1) * h[3];
    r[2] = s1 * s2 * h[1] + s1 * c2 * h[2] + c1 * h[3];
    r[3] = c2 * h[1] + (-s2) * h[2];
    r[4] = h[4];
}

// The face frame of the rotations: the angles' cosines and sines as the
// primal kernels use them, or the frame vectors themselves (normal n and
// tangents t1, t2, rows of the rotation) in a scalar type C that may carry a
// tangent.  Both give the same rotation: n = (c1 s2, s1 s2, c2),
// t1 = (c1 c2, s1 c2, -s2), t2 = (-s1, c1, 0).
struct AngleFrame {
    double c1, s1, c2, s2;
    template <class T>
    __device__ void fwd(const T *a, T *r) const { rotf(a, c1, s1, c2, s2, r); }
    template <class T>
    __device__ void back(const T *h, T *r) const { rotb(h, c1, s1, c2, s2, r); }
    __device__ double nx() const { return c1 * s2; }
    __device__ double ny() const { return s1 * s2; }
    __device__ double nz() const { return c2; }
};
template <class C>
struct VectorFrame {
    C n[3], t1[3], t2[3];
    template <class T>
    __device__ void fwd(const T *a, T *r) const {
        r[0] = a[0];
        r[1] = n[0] * a[1] + n[1] * a[2] + n[2] * a[3];
        r[2] = t1[0] * a[1] + t1[1] * a[2] + t1[2] * a[3];
        r[3] = t2[0] * a[1] + t2[1] * a[2] + t2[2] * a[3];
        r[4] = a[4];
    }
    template <class T>
    __device__ void back(const T *h, T *r) const {
        r[0] = h[0];
#pragma unroll
        for (int d = 0; d < 3; ++d) r[1 + d] = n[d] * h[1] + t1[d] * h[2] + t2[d] * h[3];
        r[4] = h[4];
    }
    __device__ C nx() const { return n[0]; }
    __device__ C ny() const { return n[1]; }
    __device__ C nz() const { return n[2]; }
};

// fin/fout: the conserved free-stream states (inflow, outflow) of the
// boundary data, of the scalar type F (Dual when their tangent is carried)
template <class T, class F, class Frame>
__device__ inline void ghost_state_fr(int code, int boundtype, double gamma, const T *cl, const Frame &fr,
                                      const F *fin, const F *fout, T *cr) {
    const auto nx = fr.nx(), ny = fr.ny(), nz = fr.nz();
    F f[NV];
    T w[NV];
    switch (code) {
    case 1:  // inflow (src/flow_operations.f90:2880-2925)
        if (boundtype == 0) {
            for (int v = 0; v < NV; ++v) cr[v] = T{fin[v]};
        } else {
            cons2prim_t(gamma, fin, f);
            cons2prim_t(gamma, cl, w);
            const T sps = sqrt((gamma * w[4]) / (w[0]));
            const T vel = sqrt(w[1] * w[1] + w[2] * w[2] + w[3] * w[3]);
            if (val(vel / (sps + UCNS_TOLSMALL)) > 1.0) {
                for (int v = 0; v < NV; ++v) cr[v] = T{fin[v]};
            } else {
                bc_sub_in(gamma, f, w, sps, nx, ny, nz, cr);
            }
        }
        break;
    case 2:  // outflow (src/flow_operations.f90:2965-3013)
        if (boundtype == 0) {
            for (int v = 0; v < NV; ++v) cr[v] = cl[v];
        } else {
            cons2prim_t(gamma, fout, f);
            cons2prim_t(gamma, cl, w);
            const T sps = sqrt((gamma * w[4]) / (w[0]));
            const T vel = sqrt(w[1] * w[1] + w[2] * w[2] + w[3] * w[3]);
            if (val(vel / (sps + UCNS_TOLSMALL)) > 1.0) {
                for (int v = 0; v < NV; ++v) cr[v] = cl[v];
            } else {
                bc_sub_out(gamma, f, w, sps, nx, ny, nz, cr);
            }
        }
        break;
    case 3:  // symmetry (src/flow_operations.f90:3086-3131)
    case 4:  // wall, inviscid branch (src/flow_operations.f90:3132-3160)
    {
        T rot[NV];
        fr.fwd(cl, rot);
        rot[1] = -rot[1];
        fr.back(rot, cr);
        break;
    }
    default:  // 6, farfield (src/flow_operations.f90:3203-3296)
    {
        T rot[NV];
        fr.fwd(cl, rot);
        const T vnb = rot[1];
        cons2prim_t(gamma, cl, w);
        const T sps = sqrt((gamma * w[4]) / (w[0]));
        if (val(vnb) <= 0.0) {
            if (val(fabs(vnb)) >= val(sps)) {
                for (int v = 0; v < NV; ++v) cr[v] = T{fin[v]};
            } else {
                cons2prim_t(gamma, fin, f);
                bc_sub_in(gamma, f, w, sps, nx, ny, nz, cr);
            }
        } else {
            if (val(fabs(vnb)) >= val(sps)) {
                for (int v = 0; v < NV; ++v) cr[v] = cl[v];
            } else {
                cons2prim_t(gamma, fout, f);
                bc_sub_out(gamma, f, w, sps, nx, ny, nz, cr);
            }
        }
    }
    }
}

template <class T, class F>
__device__ inline void ghost_state(int code, int boundtype, double gamma, const T *cl, double c1, double s1, double c2,
                                   double s2, const F *fin, const F *fout, T *cr) {
    ghost_state_fr(code, boundtype, gamma, cl, AngleFrame{c1, s1, c2, s2}, fin, fout, cr);
}

// ---------------------------------------------------------------------------
// WENO reconstruction, lane per (cell, stencil).  A wavefront owns a tile of
// 8 consecutive cells; lane = 8*local_cell + stencil.  Each lane streams its
// stencil's pseudo-inverse from the tiled layout [tile][j][k][8*ts] (one
// contiguous block per load instruction), forms dU_j on the fly from the
// FP64 states and keeps its ideg x 5 coefficients in registers.  The
// indicators, weights and the weighted sum over stencils use shuffles
// inside the 8-lane group of a cell; face points are split over the group.
template <typename R>
struct ReconWParams {
    int ncell, ntile, tiles_per_xcd, ts, nf, nqm, qpq, qpt;
    double gamma, lwci1, eps;
    const double *U;
    const double *U64;     // [ncell][8] the state in 64-byte records (row-stream gathers)
    const int32_t *nbr;    // [ntile][imax][8*ts]
    const R *P;            // [ntile][imax][ideg][8*ts]
    const R *B;            // [ncell][ideg*(ideg+1)/2]
    const R *mbar;         // [ncell][ideg]
    const R *qp;           // [ncell][nf][nqm][3]
    const int32_t *cinfo;
    const int32_t *cnb;    // [ncell][nf]
    R *uleft;              // [ncell][nf][nqm][5] deviations from the cell average
    int *marks;            // [ntile] per tile: MUSCL cells + 65536 * first-order cells (summed by k_finish)
    const unsigned char *stream;  // per-tile row stream of the DMA kernels (StreamShape)
    long long tile_bytes;
    R *gstore;             // optional [ntile][ideg*5 + 10][8*ts]: every stencil's coefficients, then
                           // its indicators beta[5] and weights omega[5], for the adjoint
    int *fstore;           // with gstore: per cell, 1 = MUSCL (CHECKSOL), 2 = first order (CHECKSOLX)
    // scatter of a residual product over the row stream (k_scatter_s64/s32):
    // member j of lane position pos receives P_j^T gbs[.][.][pos]
    const double *gbs;        // [ntile][ideg*5][8*ts] cotangents of the stencil coefficients
    double *ubar;             // [ncell][5] accumulated
    const uint16_t *slot;     // [ntile][imax][8*ts] row of the tile's member table (UCNS_NOSLOT: HBM)
    int uq_cap;               // rows of a member table at most (tile_uq(ts, imax))
    const int32_t *uq, *ucount;
    const int64_t *toff;      // first row of each tile's member table in tab
    double *tab;              // [rows][5] the member tables, summed per cell by k_adj_gather
    // CWENO (ees 5): the sectors' low-order indicators (packed, [ncell][6]) and
    // the differences of the basis means mbar - mbar_c over their 3
    // coefficients ([ncell][3]); the sectors' P rows hold their low-order
    // pseudo-inverses (zero past 3 coefficients and imax2 members)
    const R *Bc;
    const R *dmb;
    int wenoz;
};

template <typename T>
__device__ inline T lane_bcast(T v, int src) {
    return __shfl(v, src, WAVE);
}

// Exchanges inside a cell's 8 lanes by DPP (vector-unit moves: no LDS
// round trip as __shfl_xor's): quad_perm [1,0,3,2] and [2,3,0,1], then
// row_half_mirror, which reaches the other quad once the quad's lanes agree.
template <int CTRL>
__device__ __forceinline__ float dpp8(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp8(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// No contraction: a product passed in must be rounded in every lane alike, or
// the lanes of a cell would hold different sums.
template <typename T>
__device__ __forceinline__ T grp_sum8(T v) {
#pragma clang fp contract(off)
    v += dpp8<0xB1>(v);
    v += dpp8<0x4E>(v);
    v += dpp8<0x141>(v);
    return v;
}
template <typename T>
__device__ __forceinline__ T grp_min8(T v) {
    v = ::fmin(v, dpp8<0xB1>(v));
    v = ::fmin(v, dpp8<0x4E>(v));
    v = ::fmin(v, dpp8<0x141>(v));
    return v;
}
template <typename T>
__device__ __forceinline__ T grp_max8(T v) {
    v = ::fmax(v, dpp8<0xB1>(v));
    v = ::fmax(v, dpp8<0x4E>(v));
    v = ::fmax(v, dpp8<0x141>(v));
    return v;
}
__device__ inline int grp_or8(int v) {
    v |= __shfl_xor(v, 1, WAVE);
    v |= __shfl_xor(v, 2, WAVE);
    v |= __shfl_xor(v, 4, WAVE);
    return v;
}

// index of B(k,l) in the packed upper triangle stored by rows
__host__ __device__ constexpr int pidx(int ideg, int k, int l) {
    return k <= l ? k * ideg - k * (k - 1) / 2 + (l - k) : l * ideg - l * (l - 1) / 2 + (k - l);
}

// Direct global->LDS loads (global_load_lds_dword / _dwordx4): lane l's 4 or
// 16 bytes from its own global address land at LDS byte (M0 + 4 l) or
// (M0 + 16 l).  Issued as inline asm so that the compiler neither counts nor
// waits for them; every reader waits with an explicit s_waitcnt.  The nop
// covers the M0-write hazard ahead of the load.
__device__ __forceinline__ unsigned lds_addr(const void *p) {
    return (unsigned)(size_t)(const __attribute__((address_space(3))) char *)p;
}
__device__ __forceinline__ void lds_load16(const void *g, unsigned lds_base) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(lds_base) : "memory");
}

// Data read once per launch (pseudo-inverses, indicators, face points) is
// loaded non-temporally: streamed through the caches as ordinary lines it evicts
// the states and the face values that the flux kernel reads next.  Channel of
// 131,000 cells, 4 steps: 4.93 -> 4.77 ms (mixed 2.22 -> 2.08); 85,000
// hexahedra, 2 steps: 5.80 -> 5.65 ms; 197,000 tetrahedra: 8.86 -> 8.80 ms; the
// product of 2 steps on 24,576 tetrahedra: 3.70 -> 3.40 ms.  (Where it does not
// pay: stream_nt in recon_tiled.hip.)
__device__ __forceinline__ void lds_load16_nt(const void *g, unsigned lds_base) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" ::"v"(g), "{m0}"(lds_base) : "memory");
}

// one 1 KiB piece: lane l moves bytes [16 l, 16 l + 16) of the chunk when
// they lie below `valid`; NT: non-temporally
template <bool NT = true>
__device__ __forceinline__ void dma_chunk(const char *src, char *lds_dst, int lane, int valid) {
    if (lane * 16 < valid) {
        if constexpr (NT)
            lds_load16_nt(src + lane * 16, lds_addr(lds_dst));
        else
            lds_load16(src + lane * 16, lds_addr(lds_dst));
    }
}

}  // namespace ucns

#endif  // UCNS_DEVICE_H
