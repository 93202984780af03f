// Host launchers of the reconstruction kernels that live in translation units
// of their own.
#ifndef UCNS_RECON_H
#define UCNS_RECON_H

#include "ucns_device.h"

namespace ucns {

// MUSCL (linear, Barth-Jespersen) reconstruction, recon_muscl.hip
void launch_recon_muscl(const ReconParams<double> &p, hipStream_t stream);
void launch_recon_muscl(const ReconParams<float> &p, hipStream_t stream);

// WENO-3 / WENO-4 (or CWENO) on the tiled layouts, recon_tiled.hip; smode: the
// stencils per cell of the row-stream layout, or 0; w.gstore: also store the
// coefficients for the adjoint
void launch_recon_tiled(const ReconWParams<double> &w, int ideg, int smode, bool cweno, hipStream_t stream);
void launch_recon_tiled(const ReconWParams<float> &w, int ideg, int smode, bool cweno, hipStream_t stream);
// P^T of the stencil-coefficient cotangents on the row stream
void launch_scatter(const ReconWParams<double> &w, int ideg, int smode, hipStream_t stream);
void launch_scatter(const ReconWParams<float> &w, int ideg, int smode, hipStream_t stream);
// CWENO at WENO-5 (idegfree 34, sectors of 9 coefficients on 19 members),
// recon_cweno5.hip.  Device layouts, for tiles of 8 cells (c: the cell in its
// tile) and ns = ts - 1 sector stencils:
//   nbr [tile][69][8]            central members
//   nbc [tile][19][8 ns]         sector members, position c ns + sector
//   P   [tile][69][34 * 8]       central rows (cweno5_rows)
//   Pc  [tile][19][9][8 ns]      sector rows
//   B   [tile][595][8]           packed triangle by columns: entry (k, l >= k) at l (l + 1) / 2 + k
//   Bc  [ncell][45], dmb [ncell][9], and per cell as in ReconParams
template <typename R>
struct Cweno5Params {
    int ncell, ntile, tiles_per_xcd, ts, nf, nqm, qpq, qpt, wenoz;
    double gamma, lwci1, eps;
    const double *U;
    const int32_t *nbr, *nbc;
    const R *P, *Pc, *B, *Bc, *dmb, *mbar, *qp;
    const int32_t *cinfo, *cnb;
    R *uleft;
    int *marks;  // [ntile]
};
void launch_recon_cweno5(const Cweno5Params<double> &p, hipStream_t stream);
void launch_recon_cweno5(const Cweno5Params<float> &p, hipStream_t stream);
// central pseudo-inverses of cells cell0 (a multiple of 8) .. cell0+cn-1 from the ABI order into P
void cweno5_rows(const double *src, double *dst, int cell0, int cn, int tsa, hipStream_t stream);
void cweno5_rows(const double *src, float *dst, int cell0, int cn, int tsa, hipStream_t stream);

// recon_block.hip: characteristic WENO-3 / WENO-4 with 5, 6 or 7 stencils per
// cell (ch), or WENO-4 in conserved variables with 5 or 7
template <typename R>
struct ReconBParams {
    int ncell, ntile, tiles_per_xcd, nf, nqm, qpq, qpt;
    double gamma, lwci1, eps;
    const double *U;
    // pseudo-inverses: tile t's row j is at rows + t tile_bytes + hd + j rd,
    // [ideg][8 ts] R
    const unsigned char *rows;
    long long tile_bytes;
    int hd, rd;
    // distinct members of each tile [ntile][uq_cap] and, per (row, column),
    // the index into them ([ntile][imax][8 ts], UCNS_NOSLOT past uq_cap);
    // the members themselves behind the rows (row stream) or in nbr
    int uq_cap, depth, imax;
    const int32_t *uq, *ucount;
    const uint16_t *slot;
    const int32_t *nbr;
    const R *B, *mbar, *qp;
    const int32_t *cinfo, *cnb;
    R *uleft;
    int *marks;   // [ntile]
    R *gstore;    // as in ReconWParams
    int *fstore;
    const int32_t *chnb;  // characteristic WENO, as in ReconParams
    const double *chang;
    ucns_boundary_v1 bc;
    const int32_t *cface;
    const double *bface;

    // member of row j, column col
    __device__ int member(int tile, int j, int col, int tp) const {
        if (nbr) return nbr[((size_t)tile * imax + j) * tp + col];
        const unsigned char *t = rows + (size_t)tile * tile_bytes;
        const unsigned char *r = j < depth ? t + (size_t)j * tp * 4 : t + hd + (size_t)(j - depth + 1) * rd - tp * 4;
        return ((const int32_t *)r)[col];
    }
};
void launch_recon_block(const ReconBParams<double> &p, int ideg, int ts, bool ch, hipStream_t stream);
void launch_recon_block(const ReconBParams<float> &p, int ideg, int ts, bool ch, hipStream_t stream);

}  // namespace ucns

#endif  // UCNS_RECON_H
