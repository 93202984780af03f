// Device code of the tiled reconstruction kernels (a wave owns 8 consecutive
// cells, lane = 8 * cell + stencil): the register-prefetch and the row-stream
// least squares and the phases behind them.
#ifndef UCNS_TILED_H
#define UCNS_TILED_H

#include <utility>

#include "ucns_device.h"

namespace ucns {

// STORE: also write every stencil's coefficients to p.gstore (the adjoint's forward pass).
// qpc / mb: the cell's face points and basis means, in HBM or staged in LDS
// by loads still in flight (QWAIT: wait for them before the face points).
// STG: the face values pass through stg (LDS, 8 x 8 x NV values, free once
// the indicators are formed) and leave as coalesced words.
template <typename R, int IDEG, int NQL, bool STORE = false, bool CW = false, bool QWAIT = false, bool STG = false>
__device__ __forceinline__ void recon_late(const ReconWParams<R> &p, R (&g)[IDEG][NV], const double (&ui)[NV],
                                           const R (*sB)[IDEG * (IDEG + 1) / 2], R (*sG0)[IDEG * NV], int lc, int s,
                                           int cell, bool cvalid, int info, bool act, const R *qpc, const R *mb,
                                           R *stg = nullptr) {
    const int ifca = ci_ifca(info), full = ci_full(info);
    if (STORE && act) {
        // coalesced: for each coefficient the 8 ts stencils of the tile are contiguous
        const int TP = 8 * p.ts;
        R *gs = p.gstore + (size_t)(cell >> 3) * (IDEG + 2) * NV * TP + (lc * p.ts + s);
#pragma unroll
        for (int k = 0; k < IDEG; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) gs[(size_t)(k * NV + v) * TP] = g[k][v];
    }
    // central-stencil coefficients kept for the MUSCL fallback
    if (s == 0) {
#pragma unroll
        for (int k = 0; k < IDEG; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) sG0[lc][k * NV + v] = g[k][v];
    }
    __syncthreads();

    R om[NV];
    R corr[NV] = {R(0), R(0), R(0), R(0), R(0)};  // CWENO: the sectors' low-order means
    if constexpr (CW) {
        // ---- CWENO (src/reconstruct_p.f90:955-1029): lambda_1 = 1 - 1/LWCI1 for
        // the central stencil, (1 - lambda_1)/(ADMIS-1) for each sector; lane 0
        // turns its central polynomial into the zero polynomial
        // (G_1 - sum_l lambda_l G_l) / lambda_1 (the sectors' coefficients are
        // zero past the first three) ----
        const int admis = ci_admis(info);
        const double lam0 = 1.0 - (1.0 / p.lwci1);
        const double laml = admis > 1 ? (1.0 - lam0) / (admis - 1) : 0.0;
#pragma unroll
        for (int k = 0; k < IDEG; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const R sl = grp_sum8((s >= 1 && act) ? (R)laml * g[k][v] : R(0));
                if (s == 0) g[k][v] = (R)(1.0 / lam0) * (g[k][v] - sl);
            }
        // indicators: the zero polynomial's with INDICATOR, a sector's with INDICATORC
        double bd[NV] = {0, 0, 0, 0, 0};
        if (act && s == 0) {
#pragma unroll
            for (int k = 0; k < IDEG; ++k) {
                R bg[NV] = {R(0), R(0), R(0), R(0), R(0)};
#pragma unroll
                for (int l = k + 1; l < IDEG; ++l) {
                    const R bkl = sB[lc][pidx(IDEG, k, l)];
#pragma unroll
                    for (int v = 0; v < NV; ++v) bg[v] += bkl * g[l][v];
                }
                const R bkk = sB[lc][pidx(IDEG, k, k)];
#pragma unroll
                for (int v = 0; v < NV; ++v) bd[v] += (double)(g[k][v] * (bkk * g[k][v] + R(2) * bg[v]));
            }
        } else if (act) {
            const R *bc = p.Bc + (size_t)cell * 6;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                R bg[NV] = {R(0), R(0), R(0), R(0), R(0)};
#pragma unroll
                for (int l = k + 1; l < 3; ++l) {
                    const R bkl = bc[pidx(3, k, l)];
#pragma unroll
                    for (int v = 0; v < NV; ++v) bg[v] += bkl * g[l][v];
                }
                const R bkk = bc[pidx(3, k, k)];
#pragma unroll
                for (int v = 0; v < NV; ++v) bd[v] += (double)(g[k][v] * (bkk * g[k][v] + R(2) * bg[v]));
            }
        }
        // weights in FP64 in both precisions: WENO (power 4) or WENO-Z with
        // tau = sum_l |beta_1 - beta_l| / (ADMIS-1)
        const double lam = s == 0 ? lam0 : laml;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double b0 = lane_bcast(bd[v], lc * 8);
            double w = 0.0;
            if (p.wenoz) {
                const double tau = admis > 1 ? grp_sum8((s >= 1 && act) ? fabs(b0 - bd[v]) : 0.0) / (admis - 1) : 0.0;
                const double r = tau / (p.eps + bd[v]);
                const double r2 = r * r;
                w = lam * (1.0 + r2 * r2);
            } else {
                const double x = p.eps + bd[v];
                const double x2 = x * x;
                w = lam / (x2 * x2);
            }
            w = act ? w : 0.0;
            const double sum = grp_sum8(w);
            om[v] = act ? (R)(w / sum) : R(0);
        }
        // the sectors' polynomials use the means of VALUEC: their weighted
        // coefficients times (mbar - mbar_c) shift every face value alike
        const R *dm = p.dmb + (size_t)(cvalid ? cell : 0) * 3;
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) corr[v] += dm[k] * grp_sum8((s >= 1 && act) ? om[v] * g[k][v] : R(0));
    } else {
    // ---- smoothness indicators beta = g^T (B g) (src/reconstruct_p.f90:995-1004),
    // over the packed triangle of the symmetric B:
    //   beta = sum_k g_k (B_kk g_k + 2 sum_{l>k} B_kl g_l) ----
    R beta[NV] = {R(0), R(0), R(0), R(0), R(0)};
    if (act) {
#pragma unroll
        for (int k = 0; k < IDEG; ++k) {
            R bg[NV] = {R(0), R(0), R(0), R(0), R(0)};
#pragma unroll
            for (int l = k + 1; l < IDEG; ++l) {
                const R bkl = sB[lc][pidx(IDEG, k, l)];
#pragma unroll
                for (int v = 0; v < NV; ++v) bg[v] += bkl * g[l][v];
            }
            const R bkk = sB[lc][pidx(IDEG, k, k)];
#pragma unroll
            for (int v = 0; v < NV; ++v) beta[v] += g[k][v] * (bkk * g[k][v] + R(2) * bg[v]);
        }
    }
    // ---- weights (src/reconstruct_p.f90:1031-1049) and the weighted sum ----
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
            // FP32: scale by (eps+beta_min)^4 so (eps+beta)^-4 cannot underflow
            const R x = eps + beta[v];
            const R xmin = grp_min8(act ? x : (R)INFINITY);
            const R r = xmin / x;
            const R r2 = r * r;
            w = act ? lam * (r2 * r2) : R(0);
        }
        const R sum = grp_sum8(w);
        om[v] = act ? w / sum : R(0);
    }
    if (STORE && act) {
        const int TP = 8 * p.ts;
        R *gs = p.gstore + ((size_t)(cell >> 3) * (IDEG + 2) + IDEG) * NV * TP + (lc * p.ts + s);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            gs[(size_t)v * TP] = beta[v];
            gs[(size_t)(NV + v) * TP] = om[v];
        }
    }
    }
#pragma unroll
    for (int k = 0; k < IDEG; ++k)
#pragma unroll
        for (int v = 0; v < NV; ++v) g[k][v] = grp_sum8(om[v] * g[k][v]);

    // ---- face points: deviation from the average + CHECKSOL (0.85) ----
    // Values are stored as they are formed.  A cell that passes CHECKSOL
    // cannot fail CHECKSOLX (its 0.95 jumps imply the 0.85 ones), so only
    // the MUSCL branch below re-tests and overwrites its face points.
    const int nslot = ifca * p.nqm;
    if constexpr (QWAIT) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    R *out = p.uleft + (size_t)(cvalid ? cell : 0) * p.nf * p.nqm * NV;
    double wi[NV];
    cons2prim_d(p.gamma, ui, wi);
    int trouble = 0;
#pragma unroll 1
    for (int q = s; q < NQL * 8; q += 8) {
        const int f = q / p.nqm, qq = q - f * p.nqm;
        const bool ok = cvalid && q < nslot && qq < (ci_tri(info, f) ? p.qpt : p.qpq);
        if (ok) {
            R x[3] = {qpc[q * 3], qpc[q * 3 + 1], qpc[q * 3 + 2]};
            R phi[IDEG];
            basis_at<R, IDEG>(x, mb, phi);
            double uq[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                R res = corr[v];
#pragma unroll
                for (int k = 0; k < IDEG; ++k) res += phi[k] * g[k][v];
                if constexpr (STG)
                    stg[(lc * 8 + s) * NV + v] = res;
                else
                    out[q * NV + v] = res;
                uq[v] = ui[v] + (double)res;
            }
            if (full && jump_test(p.gamma, wi, uq, 0.85)) trouble = 1;
        } else if constexpr (STG) {
#pragma unroll
            for (int v = 0; v < NV; ++v) stg[(lc * 8 + s) * NV + v] = R(0);
        } else if (cvalid && q < nslot) {
#pragma unroll
            for (int v = 0; v < NV; ++v) out[q * NV + v] = R(0);
        }
        if constexpr (STG) {
            // The tile's points q0..q0+7 go out from LDS as whole 8-byte
            // words, consecutive lanes on consecutive words: each cell's
            // 8 points are one contiguous run of its block.  Words past a
            // cell's block (its last points when nf*nqm < NQL*8) stay unwritten.
            asm volatile("" ::: "memory");
            constexpr int WPC = 8 * NV * (int)sizeof(R) / 8;  // words per cell and pass
            const int q0 = q - s;
            const int cbytes = p.nf * p.nqm * NV * (int)sizeof(R);
            const int seg = q0 * NV * (int)sizeof(R);
            const int cell0 = cell - lc;
#pragma unroll
            for (int e = lc * 8 + s; e < 8 * WPC; e += WAVE) {
                const int c = e / WPC, j = e - c * WPC;
                if (cell0 + c < p.ncell && seg + (j + 1) * 8 <= cbytes) {
                    const uint64_t w = ((const uint64_t *)(stg + c * 8 * NV))[j];
                    *(uint64_t *)((char *)p.uleft + (size_t)(cell0 + c) * cbytes + seg + j * 8) = w;
                }
            }
            asm volatile("" ::: "memory");
        }
    }
    const int any_trouble = grp_or8(trouble);  // every lane takes part in the shuffle
    const bool reduce = cvalid && (!full || any_trouble);
    bool first = false;

    // ---- MUSCL + Barth-Jespersen on the central polynomial (src/reconstruct_p.f90:2044-2280) ----
    // then CHECKSOLX (0.95) -> first order (src/reconstruct_p.f90:3245-3406)
    if (reduce) {
        // the staged words of these points are written before they are overwritten
        if constexpr (STG) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        double umin[NV], umax[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) umin[v] = umax[v] = ui[v];
        for (int f = 0; f < ifca; ++f) {
            const int n = p.cnb[(size_t)cell * p.nf + f];
            if (n < 0) continue;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double un = p.U[(size_t)n * NV + v];
                umin[v] = fmin(umin[v], un);
                umax[v] = fmax(umax[v], un);
            }
        }
        double slope[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) slope[v] = 1.0e16;
        R res0[NQL][NV];
#pragma unroll
        for (int r = 0; r < NQL; ++r) {
            const int q = s + 8 * r;
            const int f = q / p.nqm, qq = q - f * p.nqm;
            const bool ok = q < nslot && qq < (ci_tri(info, f) ? p.qpt : p.qpq);
#pragma unroll
            for (int v = 0; v < NV; ++v) res0[r][v] = R(0);
            if (ok) {
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
                    if (fabs(d2) <= 0.0)
                        psi = 1.0;
                    else if (d2 > 0.0)
                        psi = fmin(1.0, (umax[v] - ui[v]) / d2);
                    else
                        psi = fmin(1.0, (umin[v] - ui[v]) / d2);
                    slope[v] = fmin(slope[v], psi);
                }
            }
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) slope[v] = grp_min8(slope[v]);
        int tr2 = 0;
#pragma unroll
        for (int r = 0; r < NQL; ++r) {
            const int q = s + 8 * r;
            const int f = q / p.nqm, qq = q - f * p.nqm;
            const bool ok = q < nslot && qq < (ci_tri(info, f) ? p.qpt : p.qpq);
#pragma unroll
            for (int v = 0; v < NV; ++v) res0[r][v] = (R)((double)res0[r][v] * slope[v]);
            if (ok) {
                double uq[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) uq[v] = ui[v] + (double)res0[r][v];
                if (jump_test(p.gamma, wi, uq, 0.95)) tr2 = 1;
            }
        }
        first = grp_or8(tr2) != 0;
#pragma unroll
        for (int r = 0; r < NQL; ++r) {
            const int q = s + 8 * r;
            if (q < nslot) {
#pragma unroll
                for (int v = 0; v < NV; ++v) out[q * NV + v] = first ? R(0) : res0[r][v];
            }
        }
    }
    {
        // the tile's counts, summed by k_finish when a call returns (same-address
        // atomics retire one per 12 ns on this chip)
        const int nred = __popcll(__ballot(s == 0 && reduce)), nfst = __popcll(__ballot(s == 0 && first));
        if (lc == 0 && s == 0) p.marks[cell >> 3] = nred + 65536 * nfst;
    }
    if (STORE && s == 0 && cvalid) p.fstore[cell] = (reduce ? 1 : 0) | (first ? 2 : 0);
}

// NT: the pseudo-inverses are loaded non-temporally
template <typename R, int IDEG, int IMAX, int NQL, int D, bool CW, bool NT>
__device__ __forceinline__ void recon_w_body(const ReconWParams<R> &p) {
    constexpr int NP = IDEG * (IDEG + 1) / 2;
    __shared__ R sB[8][NP];
    __shared__ R sG0[8][IDEG * NV];
    __shared__ int sN[IMAX * 64];  // stencil members of the tile, [j][pos]
    const int lane = threadIdx.x, lc = lane >> 3, s = lane & 7;
    const int b = blockIdx.x;
    const int tile = (b % NXCD) * p.tiles_per_xcd + b / NXCD;
    if (tile >= p.ntile) return;
    const int cell = tile * 8 + lc;
    const bool cvalid = cell < p.ncell;
    const int info = cvalid ? p.cinfo[cell] : 0;
    const int ifca = ci_ifca(info), admis = ci_admis(info), full = ci_full(info);
    const bool act = cvalid && s < admis;
    const int TP = 8 * p.ts, pos = lc * p.ts + s;
    double ui[NV] = {1.0, 0.0, 0.0, 0.0, 1.0};
    if (cvalid) {
#pragma unroll
        for (int v = 0; v < NV; ++v) ui[v] = p.U[(size_t)cell * NV + v];
    }
    const int nvc = min(8, p.ncell - tile * 8);
    R g[IDEG][NV];
#pragma unroll
    for (int k = 0; k < IDEG; ++k)
#pragma unroll
        for (int v = 0; v < NV; ++v) g[k][v] = R(0);
    {
        // indicators and stencil members of the tile -> LDS (contiguous blocks)
        {
            const R *Bt = p.B + (size_t)tile * 8 * NP;
            for (int e = lane; e < nvc * NP; e += WAVE) (&sB[0][0])[e] = Bt[e];
            const int32_t *nt = p.nbr + (size_t)tile * IMAX * TP;
            for (int e = lane; e < IMAX * TP; e += WAVE) sN[e] = nt[e];
        }
        __syncthreads();
        // ---- LSQ: g_s = P_s dU_s (src/gradients.f90:253-497) ----
        // D members are in flight (their states and pseudo-inverse columns in
        // registers) while one is accumulated.
        if (act) {
            const R *Pt = p.P + (size_t)tile * IMAX * IDEG * TP + pos;
            auto fetch = [](const R *q) {
                if constexpr (NT)
                    return __builtin_nontemporal_load(q);
                else
                    return *q;
            };
            R pb[D][IDEG];
            double ub[D][NV];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const int n = sN[d * TP + pos];
#pragma unroll
                for (int v = 0; v < NV; ++v) ub[d][v] = p.U[(size_t)n * NV + v];
                const R *Pj = Pt + (size_t)d * IDEG * TP;
#pragma unroll
                for (int k = 0; k < IDEG; ++k) pb[d][k] = fetch(Pj + k * TP);
            }
#pragma unroll 1
            for (int j0 = 0; j0 < IMAX; j0 += D) {
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    const int j = j0 + d;
                    if (j < IMAX) {
                        R du[NV], pc[IDEG];
#pragma unroll
                        for (int v = 0; v < NV; ++v) du[v] = (R)(ub[d][v] - ui[v]);
#pragma unroll
                        for (int k = 0; k < IDEG; ++k) pc[k] = pb[d][k];
                        const int jn = j + D;
                        if (jn < IMAX) {
                            const int n = sN[jn * TP + pos];
#pragma unroll
                            for (int v = 0; v < NV; ++v) ub[d][v] = p.U[(size_t)n * NV + v];
                            const R *Pj = Pt + (size_t)jn * IDEG * TP;
#pragma unroll
                            for (int k = 0; k < IDEG; ++k) pb[d][k] = fetch(Pj + k * TP);
                        }
#pragma unroll
                        for (int k = 0; k < IDEG; ++k)
#pragma unroll
                            for (int v = 0; v < NV; ++v) g[k][v] += pc[k] * du[v];
                    }
                }
            }
        }
    }
    const size_t cq = cvalid ? cell : 0;
    recon_late<R, IDEG, NQL, false, CW>(p, g, ui, sB, sG0, lc, s, cell, cvalid, info, act,
                                        p.qp + cq * p.nf * p.nqm * 3, p.mbar + cq * IDEG);
}

// ---------------------------------------------------------------------------
// Row-stream reconstruction: every byte the LSQ loop needs arrives by direct
// global->LDS loads (global_load_lds), so no register load is outstanding
// while rows are in flight.  Vector-memory counters complete in order, and
// the compiler does not count these loads, so the loop waits with explicit
// s_waitcnt vmcnt(N) where N is a lower bound on the loads issued after the
// row it needs.
//
// HBM stream of one tile: header = member indices of rows 0..DEPTH-1, then
// per member row j: the pseudo-inverse block [k][8 ts] (R) followed by the
// member indices of row j + DEPTH ([8 ts] int32), so the indices of a row
// are in LDS one ring turn before its states are fetched.
//
// LDS slot of a row: the row block as streamed, then the member states of
// its TP columns as 48-byte records (5 doubles and a pad), gathered in
// 16-byte pieces from a copy of the state padded to 64-byte records, so a
// record is one cache line; consecutive lanes take consecutive pieces and a
// row is NSI gathers.  After the loop the slots hold the tile's indicators and the
// central coefficients.
constexpr int stream_depth(bool mixed, int ts) { return ts == 5 ? 4 : (mixed ? 2 : 3); }

template <typename R, int IDEG, int IMAX, int TS, int DEPTH>
struct StreamShape {
    static constexpr int NP = IDEG * (IDEG + 1) / 2;
    static constexpr int TP = 8 * TS;
    static constexpr int PB = IDEG * TP * (int)sizeof(R);  // pseudo-inverse bytes of a row
    static constexpr int RD = PB + TP * 4;                 // row bytes in HBM
    static constexpr int HD = DEPTH * TP * 4;              // tile header bytes
    static constexpr int NCH = (RD + 1023) / 1024;         // 1 KiB loads per row
    // the row's member states: the TP columns' 48-byte records, three
    // 16-byte pieces each, gathered by NSI loads of 64 pieces; they start
    // right after the row block (its last 1 KiB load writes only to RD)
    static constexpr int NSI = (3 * TP + 63) / 64;
    static constexpr int UA = (RD + 15) / 16 * 16;
    static constexpr int SB = UA + NSI * 1024;             // slot bytes
    static constexpr int PER = NCH + NSI;                  // loads per row
    static constexpr int BBYTES = 8 * NP * (int)sizeof(R);
    static constexpr int NBC = (BBYTES + 1023) / 1024;
    static constexpr int NB = (BBYTES + SB - 1) / SB;
    static constexpr int S0 = (IMAX - DEPTH) % DEPTH;      // slot of the first tail row
    static constexpr bool TAILB = S0 + NB <= DEPTH && NB < DEPTH;
    static constexpr int TB = NB - 1;                      // tail step after which they are free
    static constexpr int BSLOT = TAILB ? S0 : 0;
    static constexpr int GSLOT = TAILB ? (S0 + NB) % DEPTH : NB;
    static constexpr long long TILE = HD + (long long)IMAX * RD;
    static_assert(RD % 16 == 0 && HD % 16 == 0, "16-byte pieces");
    static_assert(HD <= 1024, "header is one load");
    static_assert(GSLOT < DEPTH && NBC * 1024 <= NB * SB, "late data must fit the ring");
    static_assert(8 * IDEG * NV * (int)sizeof(R) <= SB, "central coefficients exceed a slot");
    static_assert((DEPTH - 1) * PER + NBC <= 63, "vmcnt immediate out of range");
    // after the stream the ring holds B ([B0, B1): every chunk issue_b
    // writes) and the central coefficients ([G0, G1)); the rest is free
    static constexpr int B0 = BSLOT * SB, B1 = B0 + NBC * 1024;
    static constexpr int G0 = GSLOT * SB, G1 = G0 + 8 * IDEG * NV * (int)sizeof(R);
};

// first 1 KiB-aligned offset in [0, ring) where `need` bytes avoid the three
// given ranges; -1 if there is none
constexpr int free_lds(int ring, int need, int a0, int a1, int b0, int b1, int c0, int c1) {
    for (int o = 0; o + need <= ring; o += 1024) {
        const int e = o + need;
        if ((e > a0 && o < a1) || (e > b0 && o < b1) || (e > c0 && o < c1)) continue;
        return o;
    }
    return -1;
}

template <typename R, int IDEG, int IMAX, int NQL, int TS, int DEPTH, bool STORE = false, bool NT = true>
__device__ __forceinline__ void recon_s_body(const ReconWParams<R> &p) {
    using SS = StreamShape<R, IDEG, IMAX, TS, DEPTH>;
    constexpr int NP = SS::NP, TP = SS::TP;
    // ring slots, then the header's index rows
    __shared__ __attribute__((aligned(1024))) char ring[DEPTH * SS::SB + SS::HD];
    const int *hdr = (const int *)(ring + DEPTH * SS::SB);
    const int lane = threadIdx.x, lc = lane >> 3, s = lane & 7;
    const int b = blockIdx.x;
    const int tile = (b % NXCD) * p.tiles_per_xcd + b / NXCD;
    if (tile >= p.ntile) return;
    const int cell = tile * 8 + lc;
    const bool cvalid = cell < p.ncell;
    int info = cvalid ? p.cinfo[cell] : 0;
    double ui[NV] = {1.0, 0.0, 0.0, 0.0, 1.0};
    if (cvalid) {
#pragma unroll
        for (int v = 0; v < NV; ++v) ui[v] = p.U[(size_t)cell * NV + v];
    }
    // the cell's own data is in registers before the first row load
    asm volatile("s_waitcnt vmcnt(0)"
                 : "+v"(info), "+v"(ui[0]), "+v"(ui[1]), "+v"(ui[2]), "+v"(ui[3]), "+v"(ui[4])
                 :
                 : "memory");
    const int admis = ci_admis(info);
    const bool act = cvalid && s < admis;
    const int rl = act ? lc * TS + s : 0;
    const int nvc = min(8, p.ncell - tile * 8);
    const char *T = (const char *)p.stream + (size_t)tile * SS::TILE;

    auto issue_row = [&](int j) {
        const char *src = T + SS::HD + (size_t)j * SS::RD;
        char *dst = ring + (j % DEPTH) * SS::SB;
#pragma unroll
        for (int c = 0; c < SS::NCH; ++c) dma_chunk<NT>(src + c * 1024, dst + c * 1024, lane, SS::RD - c * 1024);
    };
    // piece q = lane + 64 c of a row is bytes [16 (q % 3), +16) of column
    // q / 3's record; pieces past the TP columns re-read cell 0.  Every lane
    // issues every gather, so each row adds exactly NSI loads to the count.
    auto piece_cells = [&](const int *cols, int (&ix)[SS::NSI]) {
#pragma unroll
        for (int c = 0; c < SS::NSI; ++c) {
            const int q = lane + 64 * c;
            ix[c] = q < 3 * TP ? cols[q / 3] : 0;
        }
    };
    auto issue_states = [&](int j, const int (&ix)[SS::NSI]) {
        char *dst = ring + (j % DEPTH) * SS::SB + SS::UA;
#pragma unroll
        for (int c = 0; c < SS::NSI; ++c) {
            const int q = lane + 64 * c;
            const int part = q < 3 * TP ? q % 3 : 0;
            lds_load16(p.U64 + (size_t)ix[c] * 8 + 2 * part, lds_addr(dst + c * 1024));
        }
    };
    // every chunk is issued, also past the last cell's block (lane 0 then
    // re-reads the block's first bytes), so the loads counted below exist
    auto issue_b = [&]() {
        const char *src = (const char *)(p.B + (size_t)tile * 8 * NP);
        char *dst = ring + SS::BSLOT * SS::SB;
        const int bb = nvc * NP * (int)sizeof(R);
#pragma unroll
        for (int c = 0; c < SS::NBC; ++c) {
            const int valid = bb - c * 1024;
            dma_chunk<NT>(valid > 0 ? src + c * 1024 : src, dst + c * 1024, lane, valid > 0 ? valid : 16);
        }
    };


    // prologue: header, then (row, states) pairs for rows 0..DEPTH-1
    dma_chunk<NT>(T, ring + DEPTH * SS::SB, lane, SS::HD);
    issue_row(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(SS::NCH) : "memory");  // header landed
#pragma unroll
    for (int r = 0; r < DEPTH; ++r) {
        if (r > 0) issue_row(r);
        int ix[SS::NSI];
        piece_cells(hdr + r * TP, ix);
        issue_states(r, ix);
    }

    // ---- LSQ: g_s = P_s dU_s (src/gradients.f90:253-497) ----
    R g[IDEG][NV];
#pragma unroll
    for (int k = 0; k < IDEG; ++k)
#pragma unroll
        for (int v = 0; v < NV; ++v) g[k][v] = R(0);
    auto consume = [&](int i) {
        if (act) {
            const char *slot = ring + (i % DEPTH) * SS::SB;
            const double *st = (const double *)(slot + SS::UA + rl * 48);
            const double2 a = *(const double2 *)st;
            const double2 c = *(const double2 *)(st + 2);
            const double u4 = st[4];
            const R du[NV] = {(R)(a.x - ui[0]), (R)(a.y - ui[1]), (R)(c.x - ui[2]), (R)(c.y - ui[3]),
                              (R)(u4 - ui[4])};
            const R *row = (const R *)slot + rl;
            R pc[IDEG];
#pragma unroll
            for (int k = 0; k < IDEG; ++k) pc[k] = row[k * TP];
#pragma unroll
            for (int k = 0; k < IDEG; ++k)
#pragma unroll
                for (int v = 0; v < NV; ++v) g[k][v] += pc[k] * du[v];
        }
    };
#pragma unroll 1
    for (int i = 0; i < IMAX - DEPTH; ++i) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * SS::PER) : "memory");
        consume(i);
        // members of row i+DEPTH, read before that row overwrites this slot
        const int *cols = (const int *)(ring + (i % DEPTH) * SS::SB + SS::PB);
        int ix[SS::NSI];
        piece_cells(cols, ix);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue_row(i + DEPTH);
        issue_states(i + DEPTH, ix);
    }
    // tail: the last DEPTH rows; the indicators follow into the first free slots
    [&]<int... TT>(std::integer_sequence<int, TT...>) {
        (
            [&] {
                constexpr int t = TT;
                constexpr int pend = (DEPTH - 1 - t) * SS::PER + ((SS::TAILB && t > SS::TB) ? SS::NBC : 0);
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(pend) : "memory");
                consume(IMAX - DEPTH + t);
                if constexpr (SS::TAILB && t == SS::TB) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    issue_b();
                }
            }(),
            ...);
    }(std::make_integer_sequence<int, DEPTH>{});
    if constexpr (!SS::TAILB) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue_b();
    }
    // The tile's face points and basis means follow into free LDS, so that
    // the face-point loop reads them there instead of waiting on HBM once
    // per point; the indicators wait for B only.  Where they do not fit
    // (hexahedra in FP32) the loop reads them from HBM.
    constexpr int RING = DEPTH * SS::SB;
    constexpr int NQC = (8 * NQL * 8 * 3 * (int)sizeof(R) + 1023) / 1024;
    constexpr int NMC = (8 * IDEG * (int)sizeof(R) + 1023) / 1024;
    constexpr int QO = free_lds(RING, NQC * 1024, SS::B0, SS::B1, SS::G0, SS::G1, 0, 0);
    constexpr int MO = QO < 0 ? -1 : free_lds(RING, NMC * 1024, SS::B0, SS::B1, SS::G0, SS::G1, QO, QO + NQC * 1024);
    const size_t cq = cvalid ? cell : 0;
    const R *qpc = p.qp + cq * p.nf * p.nqm * 3;
    const R *mb = p.mbar + cq * IDEG;
    if constexpr (QO >= 0) {
        static_assert(NQC + NMC <= 63, "vmcnt immediate out of range");
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the tail's reads of these slots are done
        auto issue_blk = [&](const R *src, int bytes, int off, int nch) {
#pragma unroll 1
            for (int c = 0; c < nch; ++c) {
                const int valid = bytes - c * 1024;
                dma_chunk<NT>(valid > 0 ? (const char *)src + c * 1024 : (const char *)src, ring + off + c * 1024, lane,
                          valid > 0 ? valid : 16);
            }
        };
        const int per = p.nf * p.nqm * 3;
        issue_blk(p.qp + (size_t)tile * 8 * per, nvc * per * (int)sizeof(R), QO, NQC);
        qpc = (const R *)(ring + QO) + lc * per;
        if constexpr (MO >= 0) {
            issue_blk(p.mbar + (size_t)tile * 8 * IDEG, nvc * IDEG * (int)sizeof(R), MO, NMC);
            mb = (const R *)(ring + MO) + lc * IDEG;
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NQC + NMC) : "memory");  // indicators landed
        } else {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NQC) : "memory");
        }
    } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const R (*sB)[NP] = (const R (*)[NP])(ring + SS::BSLOT * SS::SB);
    R (*sG0)[IDEG * NV] = (R (*)[IDEG * NV])(ring + SS::GSLOT * SS::SB);
    // FP64 face values leave through LDS as coalesced words (128^3 hexahedra
    // 20.8 -> 20.1 ms, 64^3 x 6 tetrahedra 10.86 -> 10.71); in FP32 the
    // direct stores measured as fast or faster (hexahedra 10.8 ms direct,
    // 11.6 staged)
    constexpr bool STG = sizeof(R) == 8;
    static_assert(!STG || 8 * 8 * NV * (int)sizeof(R) <= SS::B1 - SS::B0, "face-value staging exceeds the B block");
    recon_late<R, IDEG, NQL, STORE, false, (QO >= 0), STG>(p, g, ui, sB, sG0, lc, s, cell, cvalid, info, act, qpc, mb,
                                                           (R *)(ring + SS::B0));
}

}  // namespace ucns

#endif  // UCNS_TILED_H
