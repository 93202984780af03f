// One block of NW waves per tile of 8 consecutive cells: characteristic WENO-3
// and WENO-4, and WENO-4 in conserved variables on meshes of few tiles
// (src/gradients.f90:253-497, src/reconstruct_p.f90:497-758, 920-1199,
// 2044-2280, 3126-3406).
//
// A wave per tile (ucns_tiled.h) streams at the card's rate once some thousand
// tiles are in flight, but a tile's rows, and the phases behind them, run
// one after the other in it.  Here they spread over four waves:
//   - a wave takes IDEG / NW of the coefficients of all 8 TS (cell, stencil)
//     columns (lane = column), so two or three blocks fit a CU;
//   - pseudo-inverse rows go straight to registers, D rows ahead; a row of one
//     coefficient is 8 TS contiguous values;
//   - the states of the tile's distinct members (343 of 1,560 on tetrahedra, 660
//     of 2,184 on hexahedra) are read once into LDS, and each (row, column) has
//     a 2-byte index into them;
//   - the coefficients then meet in LDS and every later phase spreads over the
//     block: indicators over (column, variable), weighted sums over (cell,
//     coefficient), face points over (cell, point), the limiter over cells.
// Each sum keeps the order and the rounding of the one-wave kernels.
// WENO-4, 1,728 hexahedra (216 tiles): 47 us with a wave per tile, 31 us this
// way; 3,072 tiles of tetrahedra 216 and 218 us; 24,576 tiles 1389 and 1518 us
// (the four waves' index reads, LDS gathers and barriers), so the wave per tile
// keeps the larger meshes (the line, and its measurements, are in
// ucns_upload_prestore).
#include "ucns_recon.h"

namespace ucns {

namespace {

template <typename R, int IDEG, int IMAX, int TS, int NW, bool CH>
struct BlockShape {
    static constexpr int TP = 8 * TS;
    static constexpr int NP = IDEG * (IDEG + 1) / 2;
    static constexpr int GS = IDEG * NV;               // coefficients of a column
    static constexpr int KW = (IDEG + NW - 1) / NW;    // coefficients of a wave
    static constexpr int CAP = tile_uq(TS, IMAX);      // member states held
    static constexpr int TAB = CAP * NV * 8;
    static constexpr int GB = TP * GS * (int)sizeof(R);
    static constexpr int GA = (TAB > GB ? TAB : GB);   // states, then coefficients
    static constexpr int BB = 8 * (CH ? NP : (NP > GS ? NP : GS)) * (int)sizeof(R);  // B, then the weighted sums
};

// ((x0 + x1) + (x2 + x3)) + ((x4 + x5) + (x6 + x7)), absent values 0, every
// product rounded before it is added (the 8-lane exchange's order)
template <int TS, typename R, class F>
__device__ __forceinline__ R tree8(F x) {
#pragma clang fp contract(off)
    R a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = i < TS ? x(i < TS ? i : 0) : R(0);
    return ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
}

// beta_c = w_c^T B w_c over the packed triangle of B for NC columns
// w_c[k] = proj(G[k])_c of one stencil's coefficients in LDS
template <typename R, int IDEG, int NC, class F>
__device__ __forceinline__ void char_beta(const R *G, const R *B, F proj, double (&beta)[NC]) {
    double w[IDEG][NC];
#pragma unroll
    for (int k = 0; k < IDEG; ++k) {
        double x[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) x[v] = (double)G[k * NV + v];
        proj(x, w[k]);
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) beta[c] = 0.0;
#pragma unroll
    for (int k = 0; k < IDEG; ++k) {
        double bg[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) bg[c] = 0.0;
#pragma unroll
        for (int l = k + 1; l < IDEG; ++l) {
            const double bkl = (double)B[pidx(IDEG, k, l)];
#pragma unroll
            for (int c = 0; c < NC; ++c) bg[c] += bkl * w[l][c];
        }
        const double bkk = (double)B[pidx(IDEG, k, k)];
#pragma unroll
        for (int c = 0; c < NC; ++c) beta[c] += w[k][c] * (bkk * w[k][c] + 2.0 * bg[c]);
    }
}

// Characteristic WENO of face f by one wave, lane = 8 * cell + stencil: the
// eigenvectors of the averaged cell / neighbour state in the face frame
// (WENO_NEIGHBOUR: the ghost of the cell's own average on boundary faces),
// indicators and weights per characteristic variable of every stencil's
// projected coefficients (three columns and two at a time, which is what the
// registers hold), and the face's values R sum_s omega_s L p_s(x_q), with
// p_s(x_q) the stencil's polynomial at the point: the sum over stencils is of
// a point's five values, not of the weighted coefficients.  Eigenvectors,
// weights and projections are in FP64 in both precisions
// (compute_gradcharv_smoothindicator, diag_At_B_A, src/reconstruct_p.f90:1608-1818).
// 24,576 tetrahedra, WENO-4: 1289 us with one wave per cell (its lane 0 forming
// the eigenvectors, 25 lanes the indicators), 510 us in the lanes of one wave
// per tile (whose registers spilled), 280 us this way.
template <typename R, int IDEG>
__device__ __forceinline__ bool char_face(const ReconBParams<R> &p, int f, const R *G, const R *B, const R *mb, int s,
                                          size_t cc, bool fv, int info, bool act, const double *ui) {
    const size_t cf = cc * p.nf + (fv ? f : 0);
    double us, vs, ws, as, hs, q2, b, bq, oa;
    {
        const int nbf = p.chnb[cf];
        const double *an = p.chang + cf * 4;
        double u0[NV], ur[NV], rl[NV], rr[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) u0[v] = ui[v];
        if (fv && nbf < 0) {
            const double *bf = p.bface ? p.bface + (size_t)(p.cface[cf] - 1) * 10 : nullptr;
            ghost_state(-nbf, p.bc.boundtype, p.gamma, u0, an[0], an[1], an[2], an[3], bf ? bf : p.bc.inflow,
                        bf ? bf + 5 : p.bc.outflow, ur);
        } else {
#pragma unroll
            for (int v = 0; v < NV; ++v) ur[v] = fv ? p.U[(size_t)nbf * NV + v] : u0[v];
        }
        rotf(u0, an[0], an[1], an[2], an[3], rl);
        rotf(ur, an[0], an[1], an[2], an[3], rr);
        const double rs = 0.5 * (rl[0] + rr[0]);
        us = 0.5 * (rl[1] / rl[0] + rr[1] / rr[0]);
        vs = 0.5 * (rl[2] / rl[0] + rr[2] / rr[0]);
        ws = 0.5 * (rl[3] / rl[0] + rr[3] / rr[0]);
        const double es = 0.5 * (rl[4] + rr[4]);
        q2 = us * us + vs * vs + ws * ws;
        const double ps = (p.gamma - 1.0) * (es - 0.5 * rs * q2);
        as = sqrt(p.gamma * ps / rs);
        hs = 0.5 * q2 + as * as / (p.gamma - 1.0);
        b = (p.gamma - 1.0) / (as * as);
        bq = 0.5 * b * q2;
        oa = 1.0 / as;
    }
    const double l00 = 0.5 * (bq + us * oa), l01 = -0.5 * (b * us + oa), l02 = -0.5 * b * vs, l03 = -0.5 * b * ws,
                 l04 = 0.5 * b;
    const double l10 = 1.0 - bq, l11 = b * us, l12 = b * vs, l13 = b * ws;
    const double l40 = 0.5 * (bq - us * oa), l41 = -0.5 * (b * us - oa);
    double om[NV];
    if (act) {
        // all of it under the condition: arithmetic alone would sink to the
        // weights below and leave its loads here
        double b3[3], b2[2];
        char_beta<R, IDEG, 3>(
            G, B,
            [&](const double(&x)[NV], double(&c)[3]) {
                c[0] = x[0] * l00 + x[1] * l01 + x[2] * l02 + x[3] * l03 + x[4] * l04;
                c[1] = x[0] * l10 + x[1] * l11 + x[2] * l12 + x[3] * l13 - x[4] * b;
                c[2] = x[0] * l40 + x[1] * l41 + x[2] * l02 + x[3] * l03 + x[4] * l04;
            },
            b3);
        // B and the coefficients are read again, not kept
        int zero = 0;
        asm volatile("" : "+v"(zero) : "v"(b3[0]), "v"(b3[1]), "v"(b3[2]));
        char_beta<R, IDEG, 2>(
            G + zero, B + zero,
            [&](const double(&x)[NV], double(&c)[2]) {
                c[0] = x[2] - x[0] * vs;
                c[1] = x[3] - x[0] * ws;
            },
            b2);
        const double lam = s == 0 ? p.lwci1 : 1.0;
        const double beta[NV] = {b3[0], b3[1], b2[0], b2[1], b3[2]};
#pragma unroll
        for (int c = 0; c < NV; ++c) {
            const double x = p.eps + beta[c];
            const double x2 = x * x;
            om[c] = lam / (x2 * x2);
        }
    } else {
#pragma unroll
        for (int c = 0; c < NV; ++c) om[c] = 0.0;
    }
#pragma unroll
    for (int c = 0; c < NV; ++c) {
        const double sum = grp_sum8(om[c]);
        om[c] = act ? om[c] / sum : 0.0;
    }
    // the face's points, QB at a time; lane q mod 8 keeps point q
    constexpr int QB = 3;
    const int nq = fv ? (ci_tri(info, f) ? p.qpt : p.qpq) : 0;
    const R *qf = p.qp + cf * p.nqm * 3;
    R *out = p.uleft + cf * p.nqm * NV;
    bool trouble = false;
    double wi[NV];
    cons2prim_d(p.gamma, ui, wi);
#pragma unroll 1
    for (int q0 = 0; q0 < p.nqm; q0 += 8) {
        double mine[NV] = {0, 0, 0, 0, 0};
        const int q1 = min(q0 + 8, p.nqm);
#pragma unroll 1
        for (int q = q0; q < q1; q += QB) {
            double pv[QB][NV];
            {
                // read in every round, not kept across the loop
                int zq = 0;
                asm volatile("" : "+v"(zq));
                const R *Gq = G + zq, *mq = mb + zq;
                R phi[QB][IDEG];
#pragma unroll
                for (int u = 0; u < QB; ++u) {
                    const R *xq = qf + min(q + u, q1 - 1) * 3;
                    const R x[3] = {xq[0], xq[1], xq[2]};
                    basis_at<R, IDEG>(x, mq, phi[u]);
                }
#pragma unroll
                for (int u = 0; u < QB; ++u)
#pragma unroll
                    for (int v = 0; v < NV; ++v) pv[u][v] = 0.0;
#pragma unroll
                for (int k = 0; k < IDEG; ++k)
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        const double gv = (double)Gq[k * NV + v];  // an idle lane's weight is 0
#pragma unroll
                        for (int u = 0; u < QB; ++u) pv[u][v] += (double)phi[u][k] * gv;
                    }
            }
#pragma unroll
            for (int u = 0; u < QB; ++u) {
                const double *x = pv[u];
                double pc[NV] = {x[0] * l00 + x[1] * l01 + x[2] * l02 + x[3] * l03 + x[4] * l04,
                                 x[0] * l10 + x[1] * l11 + x[2] * l12 + x[3] * l13 - x[4] * b,
                                 x[2] - x[0] * vs, x[3] - x[0] * ws,
                                 x[0] * l40 + x[1] * l41 + x[2] * l02 + x[3] * l03 + x[4] * l04};
#pragma unroll
                for (int c = 0; c < NV; ++c) pc[c] = grp_sum8(om[c] * pc[c]);
                const double rv[NV] = {
                    pc[0] + pc[1] + pc[4],
                    (us - as) * pc[0] + us * pc[1] + (us + as) * pc[4],
                    vs * pc[0] + vs * pc[1] + pc[2] + vs * pc[4],
                    ws * pc[0] + ws * pc[1] + pc[3] + ws * pc[4],
                    (hs - us * as) * pc[0] + 0.5 * q2 * pc[1] + vs * pc[2] + ws * pc[3] + (hs + us * as) * pc[4]};
#pragma unroll
                for (int v = 0; v < NV; ++v) mine[v] = q + u == q0 + s ? rv[v] : mine[v];
            }
        }
        const int q = q0 + s;
        if (fv && q < q1) {
            const bool ok = q < nq;
            double uq[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const R r = ok ? (R)mine[v] : R(0);
                out[q * NV + v] = r;
                uq[v] = ui[v] + (double)r;
            }
            if (ok && ci_full(info) && jump_test(p.gamma, wi, uq, 0.85)) trouble = true;
        }
    }
    return trouble;
}

template <typename R, int IDEG, int IMAX, int TS, int NW, int OCC, int D, bool STORE, bool CH>
__global__ __launch_bounds__(NW *WAVE, OCC) void k_recon_block(ReconBParams<R> p) {
    using S = BlockShape<R, IDEG, IMAX, TS, NW, CH>;
    constexpr int TP = S::TP, NP = S::NP, GS = S::GS, KW = S::KW, NT = NW * WAVE;
    static_assert(!(STORE && CH), "the adjoint does not cover characteristic variables");
    __shared__ __attribute__((aligned(16))) char sMem[S::GA + S::BB];
    __shared__ R sMb[8][IDEG];
    __shared__ double sUi[8][NV];
    __shared__ R sW[CH ? 1 : TP * NV], sOm[CH ? 1 : TP * NV];
    __shared__ int sInfo[8], sTr[8], sRed[8];
    double *const tab = (double *)sMem;
    R *const sG = (R *)sMem;
    R *const sB = (R *)(sMem + S::GA), *const sGh = sB;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int b = blockIdx.x;
    const int tile = (b % NXCD) * p.tiles_per_xcd + b / NXCD;
    if (tile >= p.ntile) return;
    const int cell0 = tile * 8, nvc = min(8, p.ncell - cell0);

    // ---- the tile's own data and the states of its distinct members ----
    const int nu = min(p.ucount[tile], S::CAP);
    const int32_t *uq = p.uq + (size_t)tile * p.uq_cap;
    for (int e = tid; e < nu * NV; e += NT) {
        const int r = e / NV;
        tab[e] = p.U[(size_t)uq[r] * NV + (e - r * NV)];
    }
    for (int e = tid; e < nvc * NP; e += NT) sB[e] = p.B[(size_t)cell0 * NP + e];
    for (int e = tid; e < nvc * IDEG; e += NT) sMb[0][e] = p.mbar[(size_t)cell0 * IDEG + e];
    if (tid < 8 * NV) {
        const double ambient = tid % NV == 0 || tid % NV == NV - 1 ? 1.0 : 0.0;
        sUi[0][tid] = tid < nvc * NV ? p.U[(size_t)cell0 * NV + tid] : ambient;
    }
    if (tid < 8) {
        sInfo[tid] = tid < nvc ? p.cinfo[cell0 + tid] : 0;
        sTr[tid] = 0;
    }
    __syncthreads();

    // ---- least squares: g = P dU, member by member (lane = column) ----
    {
        const int lc = lane / TS, s = lane - lc * TS;
        const bool act = lane < TP && s < ci_admis(sInfo[min(lc, 7)]);
        // the last wave's coefficients end with the last one: one or two may be
        // formed twice, alike
        const int k0 = min(wave * KW, IDEG - KW);
        R g[KW][NV];
#pragma unroll
        for (int k = 0; k < KW; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) g[k][v] = R(0);
        if (act) {
            double ui[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) ui[v] = sUi[lc][v];
            const char *Pt = (const char *)p.rows + (size_t)tile * p.tile_bytes + p.hd + (size_t)k0 * TP * sizeof(R);
            const char *St = (const char *)(p.slot + (size_t)tile * IMAX * TP);
            const unsigned ol = lane * (unsigned)sizeof(R), os = lane * 2u;
            auto fetch = [&](int j, R (&pr)[KW], unsigned &sj) {
                sj = *(const uint16_t *)(St + (size_t)(j * TP * 2) + os);
                const char *row = Pt + (size_t)j * p.rd;
#pragma unroll
                for (int k = 0; k < KW; ++k)
                    pr[k] = __builtin_nontemporal_load((const R *)(row + ol + k * TP * (int)sizeof(R)));
            };
            auto add = [&](const R (&pr)[KW], const double *u) {
                R du[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) du[v] = (R)(u[v] - ui[v]);
#pragma unroll
                for (int k = 0; k < KW; ++k)
#pragma unroll
                    for (int v = 0; v < NV; ++v) g[k][v] += pr[k] * du[v];
            };
            if (nu == p.ucount[tile]) {
                R pb[D][KW];
                unsigned sl[D];
#pragma unroll
                for (int d = 0; d < D; ++d) fetch(d, pb[d], sl[d]);
                // whole rounds of the ring, then the rows that are left
                constexpr int NR = (IMAX - D) / D, TAIL = IMAX - NR * D;
#pragma unroll 1
                for (int j0 = 0; j0 < NR * D; j0 += D) {
#pragma unroll
                    for (int d = 0; d < D; ++d) {
                        R pr[KW];
#pragma unroll
                        for (int k = 0; k < KW; ++k) pr[k] = pb[d][k];
                        const unsigned sj = sl[d];
                        fetch(j0 + d + D, pb[d], sl[d]);
                        add(pr, tab + sj * NV);
                    }
                }
#pragma unroll
                for (int i = 0; i < TAIL; ++i) {
                    R pr[KW];
#pragma unroll
                    for (int k = 0; k < KW; ++k) pr[k] = pb[i % D][k];
                    const unsigned sj = sl[i % D];
                    if (i + D < TAIL) fetch(NR * D + i + D, pb[i % D], sl[i % D]);
                    add(pr, tab + sj * NV);
                }
            } else {
                // more distinct members than the table holds (cells in an
                // order without locality): the others' states from HBM
#pragma unroll 1
                for (int j = 0; j < IMAX; ++j) {
                    R pr[KW];
                    unsigned sj;
                    fetch(j, pr, sj);
                    if (sj < (unsigned)S::CAP)
                        add(pr, tab + sj * NV);
                    else
                        add(pr, p.U + (size_t)p.member(tile, j, lane, TP) * NV);
                }
            }
            if constexpr (STORE) {
                R *gs = p.gstore + ((size_t)tile * (IDEG + 2) + k0) * NV * TP + lane;
#pragma unroll
                for (int k = 0; k < KW; ++k)
#pragma unroll
                    for (int v = 0; v < NV; ++v) gs[(size_t)(k * NV + v) * TP] = g[k][v];
            }
        }
        __syncthreads();  // every wave has read the states
        if (lane < TP) {
#pragma unroll
            for (int k = 0; k < KW; ++k)
#pragma unroll
                for (int v = 0; v < NV; ++v) sG[lane * GS + (k0 + k) * NV + v] = g[k][v];
        }
    }
    __syncthreads();

    const int nfq = p.nf * p.nqm;
    if constexpr (CH) {
        const int lc = lane >> 3, s = lane & 7;
        const int info = sInfo[lc];
        const bool cvalid = lc < nvc;
        const bool act = cvalid && s < ci_admis(info);
        bool trouble = false;
#pragma unroll 1
        for (int f = wave; f < p.nf; f += NW) {
            const bool fv = cvalid && f < ci_ifca(info);
            if (char_face<R, IDEG>(p, f, sG + (lc * TS + (act ? s : 0)) * GS, sB + lc * NP, sMb[lc], s,
                                   (size_t)cell0 + (cvalid ? lc : 0), fv, info, act, sUi[lc]))
                trouble = true;
        }
        if (trouble) sTr[lc] = 1;
    } else {
        // ---- smoothness indicators over the packed triangle of B,
        //   beta = sum_k g_k (B_kk g_k + 2 sum_{l>k} B_kl g_l),
        // one (column, variable) per thread ----
#pragma unroll 1
        for (int it = tid; it < TP * NV; it += NT) {
            const int col = it / NV, v = it - col * NV, lc = col / TS, s = col - lc * TS;
            const bool act = s < ci_admis(sInfo[lc]);
            R x = R(0);
            if (act) {
                R g[IDEG];
#pragma unroll
                for (int k = 0; k < IDEG; ++k) g[k] = sG[col * GS + k * NV + v];
                R beta = R(0);
#pragma unroll
                for (int k = 0; k < IDEG; ++k) {
                    R bg = R(0);
#pragma unroll
                    for (int l = k + 1; l < IDEG; ++l) bg += sB[lc * NP + pidx(IDEG, k, l)] * g[l];
                    beta += g[k] * (sB[lc * NP + pidx(IDEG, k, k)] * g[k] + R(2) * bg);
                }
                if constexpr (STORE) p.gstore[((size_t)tile * (IDEG + 2) + IDEG) * NV * TP + (size_t)v * TP + col] = beta;
                x = (R)p.eps + beta;
            }
            sW[it] = x;
        }
        __syncthreads();
        // ---- weights lambda / (eps + beta)^4, normalised (src/reconstruct_p.f90:1031-1049) ----
#pragma unroll 1
        for (int it = tid; it < TP * NV; it += NT) {
            const int col = it / NV, v = it - col * NV, lc = col / TS, s = col - lc * TS;
            const int admis = ci_admis(sInfo[lc]);
            const R lam = s == 0 ? (R)p.lwci1 : R(1);
            const R x = sW[it];
            R w;
            if (sizeof(R) == 8) {
                const R x2 = x * x;
                w = lam / (x2 * x2);
            } else {
                // FP32: scale by (eps+beta_min)^4 so (eps+beta)^-4 cannot underflow
                R xmin = (R)INFINITY;
#pragma unroll
                for (int t = 0; t < TS; ++t)
                    xmin = fmin(xmin, t < admis ? sW[(lc * TS + t) * NV + v] : (R)INFINITY);
                const R r = xmin / x;
                const R r2 = r * r;
                w = lam * (r2 * r2);
            }
            sOm[it] = s < admis ? w : R(0);
        }
        __syncthreads();
#pragma unroll 1
        for (int it = tid; it < TP * NV; it += NT) {
            const int col = it / NV, v = it - col * NV, lc = col / TS, s = col - lc * TS;
            const R sum = tree8<TS, R>([&](int t) { return sOm[(lc * TS + t) * NV + v]; });
            const R om = s < ci_admis(sInfo[lc]) ? sOm[it] / sum : R(0);
            if constexpr (STORE)
                if (s < ci_admis(sInfo[lc]))
                    p.gstore[((size_t)tile * (IDEG + 2) + IDEG + 1) * NV * TP + (size_t)v * TP + col] = om;
            sW[it] = om;
        }
        __syncthreads();
        // ---- weighted coefficients (B is done with) ----
#pragma unroll 1
        for (int e = tid; e < 8 * GS; e += NT) {
            const int lc = e / GS, kv = e - lc * GS, v = kv % NV;
            sGh[e] = tree8<TS, R>(
                [&](int t) { return sW[(lc * TS + t) * NV + v] * sG[(lc * TS + t) * GS + kv]; });
        }
        __syncthreads();
        // ---- face points: deviation from the average + CHECKSOL (0.85).  A
        // cell that passes it cannot fail CHECKSOLX (its 0.95 jumps imply the
        // 0.85 ones), so only the MUSCL cells below are tested again ----
#pragma unroll 1
        for (int e = tid; e < nvc * nfq; e += NT) {
            const int lc = e / nfq, q = e - lc * nfq, f = q / p.nqm;
            const int info = sInfo[lc];
            if (f >= ci_ifca(info)) continue;
            R *out = p.uleft + ((size_t)cell0 * nfq + e) * NV;
            if (q - f * p.nqm >= (ci_tri(info, f) ? p.qpt : p.qpq)) {
#pragma unroll
                for (int v = 0; v < NV; ++v) out[v] = R(0);
                continue;
            }
            const R *xq = p.qp + ((size_t)cell0 * nfq + e) * 3;
            const R x[3] = {xq[0], xq[1], xq[2]};
            R phi[IDEG];
            basis_at<R, IDEG>(x, sMb[lc], phi);
            double uq[NV], ui[NV], wi[NV];
            R res[NV] = {R(0), R(0), R(0), R(0), R(0)};
#pragma unroll
            for (int k = 0; k < IDEG; ++k)
#pragma unroll
                for (int v = 0; v < NV; ++v) res[v] += phi[k] * sGh[lc * GS + k * NV + v];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                out[v] = res[v];
                ui[v] = sUi[lc][v];
                uq[v] = ui[v] + (double)res[v];
            }
            cons2prim_d(p.gamma, ui, wi);
            if (ci_full(info) && jump_test(p.gamma, wi, uq, 0.85)) sTr[lc] = 1;
        }
    }
    // the unlimited values are written before other waves overwrite them
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    // ---- MUSCL + Barth-Jespersen on the central polynomial of cells that
    // fail (or are not FULL), then CHECKSOLX (0.95) -> first order: one wave
    // per cell, a face point per lane (at most 56) ----
#pragma unroll 1
    for (int lc = wave; lc < 8; lc += NW) {
        const int info = sInfo[lc];
        const bool reduce = lc < nvc && (!ci_full(info) || sTr[lc]);
        bool first = false;
        if (reduce) {
            const size_t cell = (size_t)cell0 + lc;
            const int ifca = ci_ifca(info), f = lane / p.nqm;
            const bool in = f < ifca;
            const bool ok = in && lane - f * p.nqm < (ci_tri(info, f) ? p.qpt : p.qpq);
            R res[NV] = {R(0), R(0), R(0), R(0), R(0)};
            if (ok) {
                const R *xq = p.qp + (cell * nfq + lane) * 3;
                const R x[3] = {xq[0], xq[1], xq[2]};
                R phi[IDEG];
                basis_at<R, IDEG>(x, sMb[lc], phi);
#pragma unroll
                for (int k = 0; k < IDEG; ++k)
#pragma unroll
                    for (int v = 0; v < NV; ++v) res[v] += phi[k] * sG[lc * TS * GS + k * NV + v];
            }
            double ui[NV], lo[NV], hi[NV], slope[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) lo[v] = hi[v] = ui[v] = sUi[lc][v];
            for (int i = 0; i < ifca; ++i) {
                const int n = p.cnb[cell * p.nf + i];
                if (n < 0) continue;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const double un = p.U[(size_t)n * NV + v];
                    lo[v] = fmin(lo[v], un);
                    hi[v] = fmax(hi[v], un);
                }
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) slope[v] = 1.0e16;
            if (ok) {
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
            for (int v = 0; v < NV; ++v) {
                slope[v] = wave_min(slope[v]);
                res[v] = (R)((double)res[v] * slope[v]);
            }
            bool bad = false;
            if (ok) {
                double uq[NV], wi[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) uq[v] = ui[v] + (double)res[v];
                cons2prim_d(p.gamma, ui, wi);
                bad = jump_test(p.gamma, wi, uq, 0.95);
            }
            first = __ballot(bad) != 0;
            if (in) {
                R *out = p.uleft + (cell * nfq + lane) * NV;
#pragma unroll
                for (int v = 0; v < NV; ++v) out[v] = ok && !first ? res[v] : R(0);
            }
        }
        if (lane == 0) {
            sRed[lc] = (reduce ? 1 : 0) | (first ? 2 : 0);
            if (STORE && lc < nvc) p.fstore[cell0 + lc] = (reduce ? 1 : 0) | (first ? 2 : 0);
        }
    }
    __syncthreads();
    if (tid == 0) {
        int m = 0;
#pragma unroll
        for (int lc = 0; lc < 8; ++lc) m += (sRed[lc] & 1) + 65536 * (sRed[lc] >> 1);
        p.marks[tile] = m;
    }
}

// one block per tile; TS stencil columns per cell.  NW waves: 5 or 3
// coefficients of a column each, D rows of them in flight, at OCC waves per SIMD
template <typename R, int IDEG, int IMAX, int TS>
void launch_char(const ReconBParams<R> &p, hipStream_t stream) {
    constexpr int NW = IDEG == 19 ? 4 : 3, D = IDEG == 9 || sizeof(R) == 4 ? 8 : 6;
    const dim3 grid(p.tiles_per_xcd * NXCD), block(NW * WAVE);
    hipLaunchKernelGGL((k_recon_block<R, IDEG, IMAX, TS, NW, 2, D, false, true>), grid, block, 0, stream, p);
}
template <typename R, int TS>
void launch_weno4(const ReconBParams<R> &p, hipStream_t stream) {
    constexpr int OCC = sizeof(R) == 4 ? 4 : TS == 5 ? 3 : 2, D = sizeof(R) == 4 ? 8 : 6;
    const dim3 grid(p.tiles_per_xcd * NXCD), block(4 * WAVE);
    if (p.gstore)
        hipLaunchKernelGGL((k_recon_block<R, 19, 39, TS, 4, OCC, D, true, false>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((k_recon_block<R, 19, 39, TS, 4, OCC, D, false, false>), grid, block, 0, stream, p);
}
template <typename R>
void launch(const ReconBParams<R> &p, int ideg, int ts, bool ch, hipStream_t stream) {
    if (ch && ideg == 19) {
        if (ts == 5) launch_char<R, 19, 39, 5>(p, stream);
        else if (ts == 6) launch_char<R, 19, 39, 6>(p, stream);
        else launch_char<R, 19, 39, 7>(p, stream);
    } else if (ch) {
        if (ts == 5) launch_char<R, 9, 19, 5>(p, stream);
        else if (ts == 6) launch_char<R, 9, 19, 6>(p, stream);
        else launch_char<R, 9, 19, 7>(p, stream);
    } else if (ts == 5) {
        launch_weno4<R, 5>(p, stream);
    } else {
        launch_weno4<R, 7>(p, stream);
    }
}

}  // namespace

void launch_recon_block(const ReconBParams<double> &p, int ideg, int ts, bool ch, hipStream_t stream) {
    launch(p, ideg, ts, ch, stream);
}
void launch_recon_block(const ReconBParams<float> &p, int ideg, int ts, bool ch, hipStream_t stream) {
    launch(p, ideg, ts, ch, stream);
}

}  // namespace ucns
