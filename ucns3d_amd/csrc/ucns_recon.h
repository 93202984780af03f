// Host launchers of the reconstruction kernels that live in translation units
// of their own.
#ifndef UCNS_RECON_H
#define UCNS_RECON_H

#include "ucns_device.h"

namespace ucns {

// MUSCL (linear, Barth-Jespersen) reconstruction, recon_muscl.hip
void launch_recon_muscl(const ReconParams<double> &p, hipStream_t stream);
void launch_recon_muscl(const ReconParams<float> &p, hipStream_t stream);

}  // namespace ucns

#endif  // UCNS_RECON_H
