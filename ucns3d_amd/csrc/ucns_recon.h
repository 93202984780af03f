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
// characteristic WENO-3 / WENO-4 on the tiled layouts, recon_char.hip; smode:
// the stencils per cell of the row-stream layout, or 0
void launch_recon_char(const ReconWParams<double> &p, int ideg, int smode, hipStream_t stream);
void launch_recon_char(const ReconWParams<float> &p, int ideg, int smode, hipStream_t stream);

}  // namespace ucns

#endif  // UCNS_RECON_H
