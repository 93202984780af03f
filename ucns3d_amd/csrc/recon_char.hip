// Characteristic-variable WENO-3 and WENO-4 (WENWRT 2) on the tiled kernels:
// the row-stream least squares for tetrahedra and hexahedra (5 or 7
// stencils), the register-prefetch one for other meshes, then the face-by-face
// phase of ucns_tiled.h.
#include "ucns_recon.h"
#include "ucns_tiled.h"

namespace ucns {

template <typename R, int IDEG, int IMAX, int NQL, int TS>
__global__ __launch_bounds__(WAVE) void k_recon_char_s(ReconWParams<R> p) {
    recon_s_body<R, IDEG, IMAX, NQL, TS, stream_depth(sizeof(R) == 4, TS), false, true>(p);
}
template <typename R, int IDEG, int IMAX, int NQL>
__global__ __launch_bounds__(WAVE) void k_recon_char_w(ReconWParams<R> p) {
    recon_w_body<R, IDEG, IMAX, NQL, 1, false, true>(p);
}

template <typename R>
static void launch(const ReconWParams<R> &p, int ideg, int smode, hipStream_t stream) {
    const dim3 grid(p.tiles_per_xcd * NXCD), block(WAVE);
    const bool few = p.nf * p.nqm <= 24;
    if (smode && ideg == 19) {
        if (smode == 5)
            hipLaunchKernelGGL((k_recon_char_s<R, 19, 39, 3, 5>), grid, block, 0, stream, p);
        else
            hipLaunchKernelGGL((k_recon_char_s<R, 19, 39, 7, 7>), grid, block, 0, stream, p);
    } else if (smode) {
        if (smode == 5)
            hipLaunchKernelGGL((k_recon_char_s<R, 9, 19, 3, 5>), grid, block, 0, stream, p);
        else
            hipLaunchKernelGGL((k_recon_char_s<R, 9, 19, 3, 7>), grid, block, 0, stream, p);
    } else if (ideg == 9) {
        if (few)
            hipLaunchKernelGGL((k_recon_char_w<R, 9, 19, 3>), grid, block, 0, stream, p);
        else
            hipLaunchKernelGGL((k_recon_char_w<R, 9, 19, 7>), grid, block, 0, stream, p);
    } else if (few) {
        hipLaunchKernelGGL((k_recon_char_w<R, 19, 39, 3>), grid, block, 0, stream, p);
    } else {
        hipLaunchKernelGGL((k_recon_char_w<R, 19, 39, 7>), grid, block, 0, stream, p);
    }
}
void launch_recon_char(const ReconWParams<double> &p, int ideg, int smode, hipStream_t stream) {
    launch(p, ideg, smode, stream);
}
void launch_recon_char(const ReconWParams<float> &p, int ideg, int smode, hipStream_t stream) {
    launch(p, ideg, smode, stream);
}

}  // namespace ucns
