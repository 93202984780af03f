// MUSCL reconstruction (IORDER 1, Barth-Jespersen): linear least squares on 8
// members, the limiter over the cell's face points, CHECKSOLX
// (src/gradients.f90:253-497, src/reconstruct_p.f90:2044-2280, 3245-3406).
//
// 8 lanes per cell, 8 cells per wave.  Bound by latency: a cell reads 0.5 KB
// and its chain is members -> states -> slopes -> limiter, so what counts is
// how many cells are in flight and how short the chain is.  Lane j of a cell
// loads member j, its state and its pseudo-inverse row (consecutive lanes,
// consecutive rows), and face j's neighbour for the bounds; the rows meet in
// LDS, where lane e forms entries e and e + 8 of the 15 slopes; the lanes then
// share the cell's face points.  24^3 hexahedra: a march of 10 RK3 steps 1.39
// ms with one wave per cell (15 slopes on 64 lanes, 32.7 us a launch), 0.70 ms
// this way.
#include "ucns_recon.h"

namespace ucns {

template <typename R>
__global__ __launch_bounds__(WAVE) void k_recon_muscl(ReconParams<R> p, int ntile, int tiles_per_xcd) {
    constexpr int IDEG = 3, IMAX = 8;
    __shared__ R sdu[8][IMAX][NV];
    __shared__ R sP[8][IMAX][IDEG];
    __shared__ R sG[8][IDEG * NV];
    const int lane = threadIdx.x, lc = lane >> 3, s = lane & 7;
    const int b = blockIdx.x;
    const int tile = (b % NXCD) * tiles_per_xcd + b / NXCD;
    if (tile >= ntile) return;
    const int cell = tile * 8 + lc;
    const bool cvalid = cell < p.ncell;
    const size_t cc = cvalid ? cell : 0;
    const int n = p.nbr[cc * IMAX + s];
    const int info = cvalid ? p.cinfo[cc] : 0;
    const int ifca = ci_ifca(info);
    const int fn = s < ifca ? p.cnb[cc * p.nf + s] : -1;
    double ui[NV], lo[NV], hi[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) ui[v] = p.U[cc * NV + v];
#pragma unroll
    for (int k = 0; k < IDEG; ++k) sP[lc][s][k] = p.P[(cc * IMAX + s) * IDEG + k];
#pragma unroll
    for (int v = 0; v < NV; ++v) sdu[lc][s][v] = (R)(p.U[(size_t)n * NV + v] - ui[v]);
#pragma unroll
    for (int v = 0; v < NV; ++v) lo[v] = fn >= 0 ? p.U[(size_t)fn * NV + v] : ui[v];
    __syncthreads();
    // ---- slopes: entry e = 5 k + v, members in order ----
#pragma unroll
    for (int e0 = 0; e0 < 16; e0 += 8) {
        const int e = min(e0 + s, IDEG * NV - 1), k = e / NV, v = e - k * NV;
        R acc = R(0);
#pragma unroll
        for (int j = 0; j < IMAX; ++j) acc += sP[lc][j][k] * sdu[lc][j][v];
        sG[lc][e] = acc;  // lane 7 of the second round repeats lane 6's entry
    }
    // ---- bounds over the face neighbours and the cell ----
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        hi[v] = fmax(ui[v], grp_max8(lo[v]));
        lo[v] = fmin(ui[v], grp_min8(lo[v]));
    }
    __syncthreads();
    R g[IDEG][NV], mb[IDEG];
#pragma unroll
    for (int k = 0; k < IDEG; ++k) {
        mb[k] = p.mbar[cc * IDEG + k];
#pragma unroll
        for (int v = 0; v < NV; ++v) g[k][v] = sG[lc][k * NV + v];
    }
    // ---- limiter over the cell's face points ----
    const int nslot = cvalid ? ifca * p.nqm : 0;
    const R *qpc = p.qp + cc * p.nf * p.nqm * 3;
    auto valid = [&](int q) {
        const int f = q / p.nqm;
        return q - f * p.nqm < (ci_tri(info, f) ? p.qpt : p.qpq);
    };
    auto value = [&](int q, R (&res)[NV]) {
        const R x[3] = {qpc[q * 3], qpc[q * 3 + 1], qpc[q * 3 + 2]};
        R phi[IDEG];
        basis_at<R, IDEG>(x, mb, phi);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            res[v] = R(0);
#pragma unroll
            for (int k = 0; k < IDEG; ++k) res[v] += phi[k] * g[k][v];
        }
    };
    double slope[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) slope[v] = 1.0e16;
    R res[NV];
#pragma unroll 1
    for (int q = s; q < nslot; q += 8) {
        if (!valid(q)) continue;
        value(q, res);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double d2 = (double)res[v];
            double psi;
            if (fabs(d2) <= 0.0)
                psi = 1.0;
            else if (d2 > 0.0)
                psi = fmin(1.0, (hi[v] - ui[v]) / d2);
            else
                psi = fmin(1.0, (lo[v] - ui[v]) / d2);
            slope[v] = fmin(slope[v], psi);
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) slope[v] = grp_min8(slope[v]);
    // ---- limited values, CHECKSOLX (0.95) -> first order ----
    double wi[NV];
    cons2prim_d(p.gamma, ui, wi);
    R *out = p.uleft + cc * p.nf * p.nqm * NV;
    int trouble = 0;
#pragma unroll 1
    for (int q = s; q < nslot; q += 8) {
        const bool ok = valid(q);
        if (ok && nslot > 8) value(q, res);  // at most 8 points: the lane still holds its point's value
        double uq[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const R r = ok ? (R)((double)res[v] * slope[v]) : R(0);
            out[q * NV + v] = r;
            uq[v] = ui[v] + (double)r;
        }
        if (ok && jump_test(p.gamma, wi, uq, 0.95)) trouble = 1;
    }
    const bool first = cvalid && grp_or8(trouble) != 0;
    if (first) {
#pragma unroll 1
        for (int q = s; q < nslot; q += 8)
#pragma unroll
            for (int v = 0; v < NV; ++v) out[q * NV + v] = R(0);
    }
    const int nred = __popcll(__ballot(s == 0 && cvalid)), nfst = __popcll(__ballot(s == 0 && first));
    if (lane == 0) p.marks[tile] = nred + 65536 * nfst;
}

template <typename R>
static void launch(const ReconParams<R> &p, hipStream_t stream) {
    const int ntile = (p.ncell + 7) / 8, tpx = (ntile + NXCD - 1) / NXCD;
    hipLaunchKernelGGL(k_recon_muscl<R>, dim3(tpx * NXCD), dim3(WAVE), 0, stream, p, ntile, tpx);
}
void launch_recon_muscl(const ReconParams<double> &p, hipStream_t stream) { launch(p, stream); }
void launch_recon_muscl(const ReconParams<float> &p, hipStream_t stream) { launch(p, stream); }

}  // namespace ucns
