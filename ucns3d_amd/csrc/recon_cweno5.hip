// CWENO at WENO-5 (EES 5, IORDER 4: a central polynomial of 34 coefficients on
// 69 members, quadratic sectors of 9 coefficients on their first 19), FP64 and
// mixed (src/reconstruct_p.f90:955-1049, 1062-1199, 2044-2280, 3126-3406).
//
// One block of 5 waves per tile of 8 consecutive cells.  The pseudo-inverses are
// 25.6 of the 34 KB a cell needs from HBM, so the design keeps loads in flight and
// every phase spread over the block:
//   - the members' differences are gathered into LDS once, by all threads;
//   - least squares: a thread takes a coefficient of a cell's central polynomial
//     (a member row of the tile is 272 contiguous values), then three of a
//     sector's, whose differences' LDS reads serve all three;
//   - the zero polynomial's indicator: thread (row k, cell) streams the columns
//     of B's packed triangle; sectors: thread (cell, sector, variable);
//   - weights, weighted coefficients and face points over the block, the valid
//     face points of the tile packed.
// Cells whose stencils are incomplete (FULL 0) take the MUSCL values whatever
// the unlimited ones are, so only their central polynomial is formed.
// Blast box of 24,247 cells in FP64: 552 us with one wave per cell, 365 us this
// way (2.3 TB/s of the 34 KB a cell).  Bound by latency: a tile is a dozen
// dependent memory trips with barriers between them, at three blocks a CU.
// Counters at 295,704 cells (4.04 ms): the waves wait in 72% of their cycles, 0.5%
// of them for the LDS to take an instruction; the LDS is busy 25% of the time, and
// HBM moves 2.6 TB/s.  Two central coefficients per thread halve the LDS reads of
// the differences and were slower (520 us: half as many loads in flight); the
// pseudo-inverses are read with non-temporal loads (390 us without: they evict the
// states and face values).
#include "ucns_recon.h"

namespace ucns {

namespace {

constexpr int ID = 34, IM = 69, ID2 = 9, IM2 = 19, NP = ID * (ID + 1) / 2, NP2 = ID2 * (ID2 + 1) / 2;
constexpr int NW = 5, NT = NW * WAVE;
constexpr int GC = ID * NV, GSEC = ID2 * NV;  // coefficients of a central, of a sector polynomial
static_assert(8 * ID <= NT, "a thread per (coefficient, cell)");

// OCC: waves per SIMD
template <typename R, int OCC>
__global__ __launch_bounds__(NT, OCC) void k_recon_cweno5(Cweno5Params<R> p) {
    // members' differences (central, then half of the sectors' at a time),
    // then the sectors' coefficients [c][6][45]: three blocks a CU in FP64
    constexpr int HJ = (IM2 + 1) / 2;
    // behind them, the face neighbours' states for the limiter's bounds
    constexpr int CB = 8 * IM * NV * (int)sizeof(R), HB = 8 * HJ * 6 * NV * (int)sizeof(R), NB = 8 * 6 * NV * 8;
    constexpr int MEM = CB > HB + NB ? CB : HB + NB;
    static_assert(8 * 6 * GSEC * (int)sizeof(R) <= HB, "the sectors' coefficients fit");
    __shared__ __attribute__((aligned(16))) char sMem[MEM];
    __shared__ __attribute__((aligned(16))) R sG[8][GC];  // central coefficients
    __shared__ __attribute__((aligned(16))) R sZ[8][GC];  // zero, then weighted polynomial
    __shared__ R sOm[8][7][NV];
    __shared__ double sBeta[8][7][NV];
    __shared__ double sX[NW][8][NV];                      // the waves' parts of the zero polynomial's indicator
    __shared__ R sCorr[8][NV];
    __shared__ R sMb[8][ID];
    __shared__ double sUi[8][NV];
    __shared__ int sInfo[8], sFirst[9], sTr[8], sRed[8];
    R *const sD = (R *)sMem, *const sS = (R *)sMem;
    double (*const sNb)[6][NV] = (double (*)[6][NV])(sMem + HB);
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
    const int b = blockIdx.x;
    const int tile = (b % NXCD) * p.tiles_per_xcd + b / NXCD;
    if (tile >= p.ntile) return;
    const int cell0 = tile * 8, nvc = min(8, p.ncell - cell0);
    if (tid < 8) {
        sInfo[tid] = tid < nvc ? p.cinfo[cell0 + tid] : 0;
        sTr[tid] = 0;
    }
    if (tid < 8 * NV) sUi[0][tid] = p.U[(size_t)min(cell0 * NV + tid, p.ncell * NV - 1)];
    for (int e = tid; e < nvc * ID; e += NT) sMb[0][e] = p.mbar[(size_t)cell0 * ID + e];
    __syncthreads();
    auto points_of = [&](int info, int f) { return ci_tri(info, f) ? p.qpt : p.qpq; };
    if (tid == 0) {  // where each cell's valid face points start among the tile's
        int n = 0;
        for (int c = 0; c < 8; ++c) {
            sFirst[c] = n;
            for (int f = 0; f < ci_ifca(sInfo[c]); ++f) n += points_of(sInfo[c], f);
        }
        sFirst[8] = n;
    }
    // a face neighbour's state per thread, stored once the central differences
    // have been used
    double un = 0.0;
    if (tid < 8 * 6 * NV) {
        const int c = tid / (6 * NV), f = tid / NV % 6, v = tid % NV;
        if (c < nvc) {
            const int n = f < ci_ifca(sInfo[c]) ? p.cnb[(size_t)(cell0 + c) * p.nf + f] : -1;
            un = n >= 0 ? p.U[(size_t)n * NV + v] : sUi[c][v];
        }
    }
    // differences of the central members, [j][c][v]
    for (int e = tid; e < IM * 8; e += NT) {
        const int c = e & 7;
        if (c < nvc) {
            const size_t n = (size_t)p.nbr[(size_t)tile * IM * 8 + e] * NV;
#pragma unroll
            for (int v = 0; v < NV; ++v) sD[e * NV + v] = (R)(p.U[n + v] - sUi[c][v]);
        }
    }
    __syncthreads();

    // ---- central least squares (src/gradients.f90:253-497) ----
    {
        constexpr int UJ = 23;  // 3 x 23 rows, a third in flight at once
        static_assert(IM % UJ == 0, "whole rounds");
        const int k = tid >> 3, c = tid & 7;
        if (k < ID && c < nvc) {
            R acc[NV] = {R(0), R(0), R(0), R(0), R(0)};
            const R *P = p.P + (size_t)tile * IM * ID * 8 + tid;
#pragma unroll 1
            for (int j0 = 0; j0 < IM; j0 += UJ) {
                R pv[UJ];
#pragma unroll
                for (int u = 0; u < UJ; ++u) pv[u] = __builtin_nontemporal_load(P + (size_t)(j0 + u) * ID * 8);
#pragma unroll
                for (int u = 0; u < UJ; ++u)
#pragma unroll
                    for (int v = 0; v < NV; ++v) acc[v] += pv[u] * sD[((j0 + u) * 8 + c) * NV + v];
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) sG[c][k * NV + v] = acc[v];
        }
    }
    int any_full = 0;
    for (int c = 0; c < nvc; ++c) any_full |= ci_full(sInfo[c]);
    __syncthreads();
    if (tid < 8 * 6 * NV) sNb[0][0][tid] = un;

    // the face point t of the tile's valid ones: its cell and slot
    auto point = [&](int t, int &c, int &slot) {
        c = 0;
#pragma unroll
        for (int i = 1; i < 8; ++i) c += t >= sFirst[i];
        int q = t - sFirst[c], f = 0;
        while (q >= points_of(sInfo[c], f)) q -= points_of(sInfo[c], f++);
        slot = f * p.nqm + q;
    };
    // value of a polynomial (LDS, [34][5]) at a slot of cell c
    auto value = [&](const R *G, int c, int slot, R (&r)[NV]) {
        const R *xq = p.qp + ((size_t)(cell0 + c) * p.nf * p.nqm + slot) * 3;
        const R x[3] = {xq[0], xq[1], xq[2]};
        R phi[ID];
        basis_at<R, ID>(x, sMb[c], phi);
#pragma unroll
        for (int v = 0; v < NV; ++v) r[v] = R(0);
#pragma unroll
        for (int k = 0; k < ID; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) r[v] += phi[k] * G[k * NV + v];
    };
    const int npt = sFirst[8];

    if (any_full) {
        const int ns = max(p.ts - 1, 1), tp = 8 * ns;
        // ---- sectors: their pseudo-inverse columns, then by halves of the
        // members the differences [j][c ns + sector][v] and the sums ----
        // (KS coefficients of a position per thread)
        constexpr int KS = 3;
        static_assert(ID2 % KS == 0 && 8 * 6 * (ID2 / KS) <= NT, "a thread per group and position");
        R g[KS][NV];
        const int grp = tid / tp, pos = tid - grp * tp, sc = pos / ns, ss = pos - sc * ns + 1;
        const bool in = grp < ID2 / KS, on = in && ci_full(sInfo[sc]) && ss < ci_admis(sInfo[sc]);
#pragma unroll
        for (int i = 0; i < KS; ++i)
#pragma unroll
            for (int v = 0; v < NV; ++v) g[i][v] = R(0);
        const R *P = p.Pc + (size_t)tile * IM2 * ID2 * tp + (in ? (size_t)grp * KS * tp + pos : 0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int j0 = h * HJ, nj = h ? IM2 - HJ : HJ;
            R pv[KS][HJ];
#pragma unroll
            for (int j = 0; j < HJ; ++j)
#pragma unroll
                for (int i = 0; i < KS; ++i)
                    pv[i][j] = on && j0 + j < IM2 ? __builtin_nontemporal_load(P + ((size_t)(j0 + j) * ID2 + i) * tp) : R(0);
            for (int e = tid; e < nj * tp; e += NT) {
                const int ps = e % tp, c = ps / ns, s = ps - c * ns + 1, info = sInfo[c];
                if (ci_full(info) && s < ci_admis(info)) {
                    const size_t n = (size_t)p.nbc[(size_t)tile * IM2 * tp + j0 * tp + e] * NV;
#pragma unroll
                    for (int v = 0; v < NV; ++v) sD[e * NV + v] = (R)(p.U[n + v] - sUi[c][v]);
                }
            }
            __syncthreads();
            if (on) {
#pragma unroll
                for (int j = 0; j < HJ; ++j)
                    if (j0 + j < IM2) {
#pragma unroll
                        for (int v = 0; v < NV; ++v) {
                            const R d = sD[(j * tp + pos) * NV + v];
#pragma unroll
                            for (int i = 0; i < KS; ++i) g[i][v] += pv[i][j] * d;
                        }
                    }
            }
            __syncthreads();
        }
        if (in) {
#pragma unroll
            for (int i = 0; i < KS; ++i)
#pragma unroll
                for (int v = 0; v < NV; ++v) sS[(sc * 6 + ss - 1) * GSEC + (grp * KS + i) * NV + v] = g[i][v];
        }
        __syncthreads();
        auto sector = [&](int c, int s) { return sS + (c * 6 + s - 1) * GSEC; };
        // ---- the zero polynomial (G_1 - sum_l lambda_l G_l) / lambda_1,
        // lambda_1 = 1 - 1/LWCI1, lambda_l = (1 - lambda_1)/(ADMIS-1) ----
        const double lam0 = 1.0 - (1.0 / p.lwci1);
        for (int e = tid; e < 8 * GC; e += NT) {
            const int c = e / GC, kv = e - c * GC, admis = ci_admis(sInfo[c]);
            if (!ci_full(sInfo[c])) continue;
            const double laml = admis > 1 ? (1.0 - lam0) / (admis - 1) : 0.0;
            R sl = R(0);
            if (kv < GSEC)
                for (int s = 1; s < admis; ++s) sl += (R)laml * sector(c, s)[kv];
            sZ[c][kv] = (R)(1.0 / lam0) * (sG[c][kv] - sl);
        }
        __syncthreads();
        // ---- indicators in FP64.  The zero polynomial's with INDICATOR: row k
        // of sum_k z_k (B_kk z_k + 2 sum_{l>k} B_kl z_l) by thread (k, cell) ----
        const int kc = tid >> 3, cc = tid & 7;
        double xk[NV] = {0, 0, 0, 0, 0};
        if (kc < ID && cc < nvc && ci_full(sInfo[cc])) {
            const R *Bt = p.B + (size_t)tile * NP * 8 + tid;  // column l: + l (l + 1) / 2 * 8
            double bg[NV] = {0, 0, 0, 0, 0};
            constexpr int UL = 12;
#pragma unroll 1
            for (int l0 = kc / UL * UL; l0 < ID; l0 += UL) {
                double bv[UL];
#pragma unroll
                for (int u = 0; u < UL; ++u) {
                    const int l = l0 + u;
                    bv[u] = l >= kc && l < ID ? (double)Bt[(size_t)(l * (l + 1) / 2) * 8] : 0.0;
                    bv[u] = l == kc ? 0.5 * bv[u] : bv[u];  // the diagonal counts once, the rest twice
                }
#pragma unroll
                for (int u = 0; u < UL; ++u) {
                    const int l = min(l0 + u, ID - 1);
#pragma unroll
                    for (int v = 0; v < NV; ++v) bg[v] += bv[u] * (double)sZ[cc][l * NV + v];
                }
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) xk[v] = (double)sZ[cc][kc * NV + v] * (2.0 * bg[v]);
        }
        // the wave's rows (lanes 8 apart hold one cell's)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
#pragma unroll
            for (int o = 8; o < WAVE; o <<= 1) xk[v] += __shfl_xor(xk[v], o, WAVE);
            if (lane < 8) sX[wave][cc][v] = xk[v];
        }
        // a sector's with INDICATORC, by thread (cell, sector, variable)
        for (int it = tid; it < 8 * 6 * NV; it += NT) {
            const int c = it / (6 * NV), s = it / NV % 6 + 1, v = it % NV, info = sInfo[c];
            if (!ci_full(info) || s >= ci_admis(info)) continue;
            const R *bc = p.Bc + (size_t)(cell0 + c) * NP2, *gs = sector(c, s) + v;
            double bs[NP2];
#pragma unroll
            for (int e = 0; e < NP2; ++e) bs[e] = (double)bc[e];
            double a = 0.0;
#pragma unroll
            for (int k = 0; k < ID2; ++k) {
                double bgk = 0.0;
#pragma unroll
                for (int l = 0; l < ID2; ++l) bgk += bs[pidx(ID2, k, l)] * (double)gs[l * NV];
                a += (double)gs[k * NV] * bgk;
            }
            sBeta[c][s][v] = a;
        }
        __syncthreads();
        if (tid < 8 * NV && ci_full(sInfo[tid / NV])) {
            const int c = tid / NV, v = tid % NV;
            double a = 0.0;
            for (int w = 0; w < NW; ++w) a += sX[w][c][v];
            sBeta[c][0][v] = a;
        }
        __syncthreads();
        // ---- weights in FP64: WENO (power 4) or WENO-Z,
        // tau = sum_l |beta_1 - beta_l| / (ADMIS-1) ----
        for (int it = tid; it < 8 * 7 * NV; it += NT) {
            const int c = it / (7 * NV), s = it / NV % 7, v = it % NV, info = sInfo[c], admis = ci_admis(info);
            if (!ci_full(info) || s >= admis) continue;
            const double laml = admis > 1 ? (1.0 - lam0) / (admis - 1) : 0.0;
            double tau = 0.0;
            if (p.wenoz && admis > 1) {
                for (int t = 1; t < admis; ++t) tau += fabs(sBeta[c][0][v] - sBeta[c][t][v]);
                tau /= (double)(admis - 1);
            }
            double sum = 0.0, mine = 0.0;
            for (int t = 0; t < admis; ++t) {
                const double lam = t == 0 ? lam0 : laml, x = p.eps + sBeta[c][t][v];
                double w;
                if (p.wenoz) {
                    const double r = tau / x, r2 = r * r;
                    w = lam * (1.0 + r2 * r2);
                } else {
                    const double x2 = x * x;
                    w = lam / (x2 * x2);
                }
                sum += w;
                if (t == s) mine = w;
            }
            sOm[c][s][v] = (R)(mine / sum);
        }
        __syncthreads();
        // ---- the weighted polynomial on the high-order basis; the sectors'
        // polynomials use the means of VALUEC: their weighted coefficients
        // times (mbar - mbar_c) shift every face value alike ----
        for (int e = tid; e < 8 * GC; e += NT) {
            const int c = e / GC, kv = e - c * GC, v = kv % NV, admis = ci_admis(sInfo[c]);
            if (!ci_full(sInfo[c])) continue;
            R a = sOm[c][0][v] * sZ[c][kv];
            if (kv < GSEC)
                for (int s = 1; s < admis; ++s) a += sOm[c][s][v] * sector(c, s)[kv];
            sZ[c][kv] = a;
        }
        if (tid < nvc * NV && ci_full(sInfo[tid / NV])) {
            const int c = tid / NV, v = tid % NV, admis = ci_admis(sInfo[c]);
            const R *dm = p.dmb + (size_t)(cell0 + c) * ID2;
            R a = R(0);
#pragma unroll
            for (int k = 0; k < ID2; ++k) {
                R wg = R(0);
                for (int s = 1; s < admis; ++s) wg += sOm[c][s][v] * sector(c, s)[k * NV + v];
                a += dm[k] * wg;
            }
            sCorr[c][v] = a;
        }
        __syncthreads();
        // ---- face values + CHECKSOL (0.85) ----
#pragma unroll 1
        for (int t = tid; t < npt; t += NT) {
            int c, slot;
            point(t, c, slot);
            if (!ci_full(sInfo[c])) continue;
            R r[NV];
            value(sZ[c], c, slot, r);
            R *out = p.uleft + ((size_t)(cell0 + c) * p.nf * p.nqm + slot) * NV;
            double uq[NV], wi[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                r[v] += sCorr[c][v];
                out[v] = r[v];
                uq[v] = sUi[c][v] + (double)r[v];
            }
            cons2prim_d(p.gamma, sUi[c], wi);
            if (jump_test(p.gamma, wi, uq, 0.85)) sTr[c] = 1;
        }
        // the unlimited values are written before other waves overwrite them
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();

    // ---- MUSCL + Barth-Jespersen on the central polynomial of cells that fail
    // (or are not FULL), then CHECKSOLX (0.95) -> first order: one wave per
    // cell, the limited values kept in registers ----
#pragma unroll 1
    for (int c = wave; c < 8; c += NW) {
        const int info = sInfo[c];
        const bool reduce = c < nvc && (!ci_full(info) || sTr[c]);
        bool first = false;
        if (reduce) {
            const size_t cell = (size_t)cell0 + c;
            const int ifca = ci_ifca(info), np = sFirst[c + 1] - sFirst[c];  // at most 96
            double ui[NV], lo[NV], hi[NV], slope[NV];
            R res[2][NV];
            int at[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                at[u] = -1;
                if (lane + u * WAVE < np) {
                    int c2;
                    point(sFirst[c] + lane + u * WAVE, c2, at[u]);
                    value(sG[c], c, at[u], res[u]);
                }
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                lo[v] = hi[v] = ui[v] = sUi[c][v];
                slope[v] = 1.0e16;
            }
            for (int f = 0; f < ifca; ++f) {
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const double un = sNb[c][f][v];
                    lo[v] = fmin(lo[v], un);
                    hi[v] = fmax(hi[v], un);
                }
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
                if (at[u] >= 0) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        const double d2 = (double)res[u][v];
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
            for (int v = 0; v < NV; ++v) slope[v] = wave_min(slope[v]);
            bool bad = false;
            double wi[NV];
            cons2prim_d(p.gamma, ui, wi);
#pragma unroll
            for (int u = 0; u < 2; ++u)
                if (at[u] >= 0) {
                    double uq[NV];
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        res[u][v] = (R)((double)res[u][v] * slope[v]);
                        uq[v] = ui[v] + (double)res[u][v];
                    }
                    if (jump_test(p.gamma, wi, uq, 0.95)) bad = true;
                }
            first = __ballot(bad) != 0;
#pragma unroll
            for (int u = 0; u < 2; ++u)
                if (at[u] >= 0) {
                    R *out = p.uleft + (cell * p.nf * p.nqm + at[u]) * NV;
#pragma unroll
                    for (int v = 0; v < NV; ++v) out[v] = first ? R(0) : res[u][v];
                }
        }
        if (lane == 0) sRed[c] = (reduce ? 1 : 0) + (first ? 65536 : 0);
    }
    __syncthreads();
    if (tid == 0) {
        int m = 0;
        for (int c = 0; c < 8; ++c) m += sRed[c];
        p.marks[tile] = m;
    }
}

// upload: the central pseudo-inverses of cells cell0 .. cell0+cn-1 (cell0 a
// multiple of 8; [cell][tsa][imax][ideg] FP64, the ABI order) into the rows
template <typename R>
__global__ void k_cweno5_rows(const double *src, R *dst, int cell0, int cn, int tsa) {
    const size_t n = (size_t)cn * IM * ID;
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
        const int k = (int)(e % ID), j = (int)(e / ID % IM), c = (int)(e / ((size_t)ID * IM));
        const int i = cell0 + c;
        dst[((size_t)(i / 8) * IM + j) * ID * 8 + k * 8 + i % 8] = (R)src[((size_t)c * tsa * IM + j) * ID + k];
    }
}

template <typename R>
void launch(const Cweno5Params<R> &p, hipStream_t stream) {
    const dim3 grid(p.tiles_per_xcd * NXCD), block(NT);
    // At 4 waves per SIMD three blocks fit a CU (in FP64 the LDS holds no more).
    // The mixed kernel fits a fourth at 5, with 116 bytes of scratch a lane: worth
    // it once the chip's 768 blocks are taken.  Blast box in mixed precision, 2
    // steps: 307 tiles 0.385 ms with 4 waves and 0.412 with 5, 1,370 tiles 1.18
    // and 0.98, 3,030 tiles 2.24 and 1.79; 6 waves (188 bytes) 1.82.
    if (sizeof(R) == 4 && p.ntile > 3 * 256)
        hipLaunchKernelGGL((k_recon_cweno5<R, sizeof(R) == 4 ? 5 : 4>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((k_recon_cweno5<R, 4>), grid, block, 0, stream, p);
}
template <typename R>
void rows(const double *src, R *dst, int cell0, int cn, int tsa, hipStream_t stream) {
    const size_t n = (size_t)cn * IM * ID;
    const unsigned blocks = (unsigned)(n / 256 + 1 < 4096 ? n / 256 + 1 : 4096);
    hipLaunchKernelGGL(k_cweno5_rows<R>, dim3(blocks), dim3(256), 0, stream, src, dst, cell0, cn, tsa);
}

}  // namespace

void launch_recon_cweno5(const Cweno5Params<double> &p, hipStream_t stream) { launch(p, stream); }
void launch_recon_cweno5(const Cweno5Params<float> &p, hipStream_t stream) { launch(p, stream); }
void cweno5_rows(const double *src, double *dst, int cell0, int cn, int tsa, hipStream_t stream) {
    rows(src, dst, cell0, cn, tsa, stream);
}
void cweno5_rows(const double *src, float *dst, int cell0, int cn, int tsa, hipStream_t stream) {
    rows(src, dst, cell0, cn, tsa, stream);
}

}  // namespace ucns
