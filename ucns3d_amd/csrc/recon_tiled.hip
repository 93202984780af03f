// The tiled WENO-3 / WENO-4 kernels in conserved variables: the row-stream
// reconstruction of tetrahedra and hexahedra, and at WENO-3 of meshes with prisms
// and pyramids (with and without the coefficients' copy for the adjoint), its
// transposed scatter, the register-prefetch reconstruction of other meshes, CWENO.
#include "ucns_recon.h"
#include "ucns_tiled.h"

namespace ucns {

// Whether a march's reconstruction loads its pseudo-inverses (`bytes` of them in a
// launch) non-temporally, so that they do not evict the states and face values that
// the next kernels read (ucns_device.h).  That is the faster way, except
//   - where they fit the 256 MB of the memory-side cache: as ordinary lines they
//     stay there from one stage to the next.  us a stage, ordinary and
//     non-temporal, row stream: 32,768 hexahedra WENO-3 mixed (157 MB) 65.6, 84.9;
//     4,913 WENO-4 FP64 (204 MB) 64.8, 75.2; 7,986 tetrahedra WENO-4 FP64 (237 MB)
//     64.2, 69.3; 12,167 hexahedra WENO-4 mixed (252 MB) 89.2, 89.9; 54,872 WENO-3
//     mixed (263 MB) 129.3, 127.1.  Register kernels, WENO-4: 2,058 pyramids mixed
//     (37 MB) 61.7, 58.3; 4,374 FP64 (156 MB) 77.6, 82.1; 11,664 prisms mixed (207
//     MB) 82.3, 97.0; and CWENO on WENO-3, 24,576 tetrahedra (84 MB) 50.3, 60.4;
//   - WENO-4 in FP64 past some 1.3 million cells, which takes as long with them as
//     with ordinary loads, or longer, by where the allocator placed the rows (two
//     contexts created in turn get one placement each).  ms a step, ordinary and
//     non-temporal, in either:
//       tetrahedra 1,170,672 cells   25.3, 25.5   22.7, 23.0
//                  1,361,886         29.6, 29.7   29.0, 30.8
//                  1,971,054         42.9, 43.1   41.8, 44.6
//       hexahedra  1,259,712         40.6, 40.4   36.8, 36.4
//                  1,560,896         50.4, 50.5   50.3, 51.3
//                  2,097,152         68.0, 68.9   67.5, 69.2
//     Why the second placement and the larger mesh do not suit them is not known;
//     on another card the two kinds took the same time in both.
// The kernels of the residual products always load non-temporally: a reversed
// stage streams its rows twice with the stored coefficients between.
template <typename R>
static bool stream_nt(const ReconWParams<R> &w, int ideg, int smode) {
    const long long mib = 1 << 20;
    const long long bytes =
        smode ? w.ntile * w.tile_bytes : (long long)w.ntile * 8 * w.ts * (ideg == 19 ? 39 : 19) * ideg * sizeof(R);
    if (bytes <= 256 * mib) return !smode && ideg == 19 && bytes <= 96 * mib;
    return !(smode && sizeof(R) == 8 && ideg == 19 && w.ncell > 1310720);
}

template <int IDEG, int IMAX, int NQL, int TS, bool NT>
__global__ __launch_bounds__(WAVE) void k_recon_s64(ReconWParams<double> p) {
    recon_s_body<double, IDEG, IMAX, NQL, TS, stream_depth(false, TS), false, NT>(p);
}
// Scatter of a residual product on the row stream, without the
// reconstruction: lane (cell, stencil) holds its g_bar (p.gbs) and streams
// the tile's pseudo-inverse rows through the same LDS ring and layout as the
// reconstruction (no neighbour states); dU_bar_j = P_j^T g_bar goes to the
// tile's member table (then p.tab, summed per cell by k_adj_gather) and
// minus the same to the cell.
template <typename R, int IDEG, int IMAX, int TS, int DEPTH>
__device__ __forceinline__ void scatter_s_body(const ReconWParams<R> &p) {
    using SS = StreamShape<R, IDEG, IMAX, TS, DEPTH>;
    constexpr int TP = SS::TP, NCH = SS::NCH, SL = NCH * 1024;
    constexpr int UQ = tile_uq(TS, IMAX);  // LDS table rows
    __shared__ __attribute__((aligned(1024))) char ring[DEPTH * SL + SS::HD];
    __shared__ double sAcc[UQ][NV];
    __shared__ uint16_t sSlot[IMAX * TP];
    const int *hdr = (const int *)(ring + DEPTH * SL);
    const int lane = threadIdx.x, lc = lane >> 3, s = lane & 7;
    const int b = blockIdx.x;
    const int tile = (b % NXCD) * p.tiles_per_xcd + b / NXCD;
    if (tile >= p.ntile) return;
    const int cell = tile * 8 + lc;
    const bool cvalid = cell < p.ncell;
    int info = cvalid ? p.cinfo[cell] : 0;
    double gb[IDEG][NV];
    {
        const double *gs = p.gbs + (size_t)tile * IDEG * NV * TP + (lc * TS + s);
        const bool in = cvalid && s < TS;
#pragma unroll
        for (int k = 0; k < IDEG; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) gb[k][v] = in ? gs[(size_t)(k * NV + v) * TP] : 0.0;
    }
    const uint16_t *st = p.slot + (size_t)tile * IMAX * TP;
    for (int e = lane; e < IMAX * TP; e += WAVE) sSlot[e] = st[e];
    const int nuq = min(p.ucount[tile], p.uq_cap);
    for (int e = lane; e < min(nuq, UQ) * NV; e += WAVE) (&sAcc[0][0])[e] = 0.0;
    // every cotangent is used before the row stream starts, so the compiler
    // waits for their loads here and not inside the stream
    double gsum = 0.0;
#pragma unroll
    for (int k = 0; k < IDEG; ++k)
#pragma unroll
        for (int v = 0; v < NV; ++v) gsum += gb[k][v];
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(info), "+v"(gsum) : : "memory");
    __syncthreads();  // sSlot, sAcc
    const bool act = cvalid && s < ci_admis(info);
    const int rl = act ? lc * TS + s : 0;
    const char *T = (const char *)p.stream + (size_t)tile * SS::TILE;
    auto issue_row = [&](int j) {
        const char *src = T + SS::HD + (size_t)j * SS::RD;
        char *dst = ring + (j % DEPTH) * SL;
#pragma unroll
        for (int c = 0; c < NCH; ++c) dma_chunk(src + c * 1024, dst + c * 1024, lane, SS::RD - c * 1024);
    };
    int qn[DEPTH];  // members of the next DEPTH rows, oldest first
    double acc[NV] = {0, 0, 0, 0, 0};
    dma_chunk(T, ring + DEPTH * SL, lane, SS::HD);
    issue_row(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NCH) : "memory");  // header landed
#pragma unroll
    for (int r = 0; r < DEPTH; ++r) qn[r] = hdr[r * TP + rl];
#pragma unroll
    for (int r = 1; r < DEPTH; ++r) issue_row(r);
    auto consume = [&](int i) {
        if (act) {
            const R *row = (const R *)(ring + (i % DEPTH) * SL) + rl;
            double d[NV] = {0, 0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < IDEG; ++k) {
                const double pk = (double)row[k * TP];
#pragma unroll
                for (int v = 0; v < NV; ++v) d[v] += pk * gb[k][v];
            }
            const unsigned sl = sSlot[i * TP + rl];
            if (sl < (unsigned)UQ) {
#pragma unroll
                for (int v = 0; v < NV; ++v)
                    __hip_atomic_fetch_add(&sAcc[sl][v], d[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            } else {
#pragma unroll
                for (int v = 0; v < NV; ++v) unsafeAtomicAdd(&p.ubar[(size_t)qn[0] * NV + v], d[v]);
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] -= d[v];
        }
#pragma unroll
        for (int r = 0; r + 1 < DEPTH; ++r) qn[r] = qn[r + 1];
    };
#pragma unroll 1
    for (int i = 0; i < IMAX - DEPTH; ++i) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * NCH) : "memory");
        consume(i);
        const int nn = *(const int *)(ring + (i % DEPTH) * SL + SS::PB + rl * 4);  // members of row i+DEPTH
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue_row(i + DEPTH);
        qn[DEPTH - 1] = nn;
    }
    [&]<int... TT>(std::integer_sequence<int, TT...>) {
        (
            [&] {
                constexpr int t = TT;
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1 - t) * NCH) : "memory");
                consume(IMAX - DEPTH + t);
            }(),
            ...);
    }(std::make_integer_sequence<int, DEPTH>{});
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const double t = grp_sum8(acc[v]);
        if (s == 0 && cvalid) unsafeAtomicAdd(&p.ubar[(size_t)cell * NV + v], t);
    }
    __syncthreads();
    double *tt = p.tab + (size_t)p.toff[tile] * NV;
    for (int e = lane; e < nuq * NV; e += WAVE) tt[e] = e < UQ * NV ? (&sAcc[0][0])[e] : 0.0;
}
template <int IDEG, int IMAX, int TS>
__global__ __launch_bounds__(WAVE) void k_scatter_s64(ReconWParams<double> p) {
    scatter_s_body<double, IDEG, IMAX, TS, stream_depth(false, TS)>(p);
}
template <int IDEG, int IMAX, int TS>
__global__ __launch_bounds__(WAVE) void k_scatter_s32(ReconWParams<float> p) {
    scatter_s_body<float, IDEG, IMAX, TS, stream_depth(true, TS)>(p);
}

// the reconstruction storing every stencil's coefficients for a residual product
template <int IDEG, int IMAX, int NQL, int TS>
__global__ __launch_bounds__(WAVE) void k_recon_sg64(ReconWParams<double> p) {
    recon_s_body<double, IDEG, IMAX, NQL, TS, stream_depth(false, TS), true>(p);
}
template <int IDEG, int IMAX, int NQL, int TS>
__global__ __launch_bounds__(WAVE, 2) void k_recon_sg32(ReconWParams<float> p) {
    recon_s_body<float, IDEG, IMAX, NQL, TS, stream_depth(true, TS), true>(p);
}
template <int IDEG, int IMAX, int NQL, int TS, bool NT>
__global__ __launch_bounds__(WAVE, 2) void k_recon_s32(ReconWParams<float> p) {
    recon_s_body<float, IDEG, IMAX, NQL, TS, stream_depth(true, TS), false, NT>(p);
}

// FP64: registers for the 19x5 coefficients dominate, one wave per SIMD;
// FP32: the compiler is asked for WAVES32 waves per SIMD.
constexpr int WAVES32 = 1;           // waves per SIMD asked for in FP32
constexpr int DEPTH64 = 1, DEPTH32 = 2;  // members in flight of the register-prefetch kernels
template <int IDEG, int IMAX, int NQL, bool NT>
__global__ __launch_bounds__(WAVE) void k_recon_w64(ReconWParams<double> p) {
    recon_w_body<double, IDEG, IMAX, NQL, DEPTH64, false, NT>(p);
}
template <int IDEG, int IMAX, int NQL, bool NT>
__global__ __launch_bounds__(WAVE) void k_recon_cw64(ReconWParams<double> p) {
    recon_w_body<double, IDEG, IMAX, NQL, DEPTH64, true, NT>(p);
}
template <int IDEG, int IMAX, int NQL, bool NT>
__global__ __launch_bounds__(WAVE, WAVES32) void k_recon_cw32(ReconWParams<float> p) {
    recon_w_body<float, IDEG, IMAX, NQL, DEPTH32, true, NT>(p);
}
template <int IDEG, int IMAX, int NQL, bool NT>
__global__ __launch_bounds__(WAVE, WAVES32) void k_recon_w32(ReconWParams<float> p) {
    recon_w_body<float, IDEG, IMAX, NQL, DEPTH32, false, NT>(p);
}

template <typename R, bool NT>
static void launch(const ReconWParams<R> &w, int ideg, int smode, bool cweno, hipStream_t stream) {
    const dim3 grid(w.tiles_per_xcd * NXCD), block(WAVE);
    const bool few = w.nf * w.nqm <= 24;
#define UCNS_LAUNCH(...) hipLaunchKernelGGL((__VA_ARGS__), grid, block, 0, stream, w)
    if (smode) {
        // (ideg, imax, face-point slots, stencils): WENO-4 tets / hexes, WENO-3 tets / prisms and pyramids / hexes
        if constexpr (sizeof(R) == 8) {
            if (ideg == 19 && smode == 5) UCNS_LAUNCH(k_recon_s64<19, 39, 3, 5, NT>);
            else if (ideg == 19) UCNS_LAUNCH(k_recon_s64<19, 39, 7, 7, NT>);
            else if (smode == 5) UCNS_LAUNCH(k_recon_s64<9, 19, 3, 5, NT>);
            else if (smode == 6) UCNS_LAUNCH(k_recon_s64<9, 19, 3, 6, NT>);
            else UCNS_LAUNCH(k_recon_s64<9, 19, 3, 7, NT>);
        } else {
            if (ideg == 19 && smode == 5) UCNS_LAUNCH(k_recon_s32<19, 39, 3, 5, NT>);
            else if (ideg == 19) UCNS_LAUNCH(k_recon_s32<19, 39, 7, 7, NT>);
            else if (smode == 5) UCNS_LAUNCH(k_recon_s32<9, 19, 3, 5, NT>);
            else if (smode == 6) UCNS_LAUNCH(k_recon_s32<9, 19, 3, 6, NT>);
            else UCNS_LAUNCH(k_recon_s32<9, 19, 3, 7, NT>);
        }
    } else if (cweno) {
        if constexpr (sizeof(R) == 8) {
            if (ideg == 9) UCNS_LAUNCH(k_recon_cw64<9, 19, 3, NT>);
            else if (few) UCNS_LAUNCH(k_recon_cw64<19, 39, 3, NT>);
            else UCNS_LAUNCH(k_recon_cw64<19, 39, 7, NT>);
        } else {
            if (ideg == 9) UCNS_LAUNCH(k_recon_cw32<9, 19, 3, NT>);
            else if (few) UCNS_LAUNCH(k_recon_cw32<19, 39, 3, NT>);
            else UCNS_LAUNCH(k_recon_cw32<19, 39, 7, NT>);
        }
    } else if constexpr (sizeof(R) == 8) {
        if (ideg == 9) UCNS_LAUNCH(k_recon_w64<9, 19, 3, NT>);
        else if (few) UCNS_LAUNCH(k_recon_w64<19, 39, 3, NT>);
        else UCNS_LAUNCH(k_recon_w64<19, 39, 7, NT>);
    } else {
        if (ideg == 9) UCNS_LAUNCH(k_recon_w32<9, 19, 3, NT>);
        else if (few) UCNS_LAUNCH(k_recon_w32<19, 39, 3, NT>);
        else UCNS_LAUNCH(k_recon_w32<19, 39, 7, NT>);
    }
}
// the row stream storing every stencil's coefficients (w.gstore)
template <typename R>
static void launch_store(const ReconWParams<R> &w, int ideg, int smode, hipStream_t stream) {
    const dim3 grid(w.tiles_per_xcd * NXCD), block(WAVE);
    if constexpr (sizeof(R) == 8) {
        if (ideg == 19 && smode == 5) UCNS_LAUNCH(k_recon_sg64<19, 39, 3, 5>);
        else if (ideg == 19) UCNS_LAUNCH(k_recon_sg64<19, 39, 7, 7>);
        else if (smode == 5) UCNS_LAUNCH(k_recon_sg64<9, 19, 3, 5>);
        else if (smode == 6) UCNS_LAUNCH(k_recon_sg64<9, 19, 3, 6>);
        else UCNS_LAUNCH(k_recon_sg64<9, 19, 3, 7>);
    } else {
        if (ideg == 19 && smode == 5) UCNS_LAUNCH(k_recon_sg32<19, 39, 3, 5>);
        else if (ideg == 19) UCNS_LAUNCH(k_recon_sg32<19, 39, 7, 7>);
        else if (smode == 5) UCNS_LAUNCH(k_recon_sg32<9, 19, 3, 5>);
        else if (smode == 6) UCNS_LAUNCH(k_recon_sg32<9, 19, 3, 6>);
        else UCNS_LAUNCH(k_recon_sg32<9, 19, 3, 7>);
    }
}
template <typename R>
static void launch_any(const ReconWParams<R> &w, int ideg, int smode, bool cweno, hipStream_t stream) {
    if (smode && w.gstore)
        launch_store(w, ideg, smode, stream);
    else if (stream_nt(w, ideg, smode))
        launch<R, true>(w, ideg, smode, cweno, stream);
    else
        launch<R, false>(w, ideg, smode, cweno, stream);
}
void launch_recon_tiled(const ReconWParams<double> &w, int ideg, int smode, bool cweno, hipStream_t stream) {
    launch_any(w, ideg, smode, cweno, stream);
}
void launch_recon_tiled(const ReconWParams<float> &w, int ideg, int smode, bool cweno, hipStream_t stream) {
    launch_any(w, ideg, smode, cweno, stream);
}

void launch_scatter(const ReconWParams<double> &w, int ideg, int smode, hipStream_t stream) {
    const dim3 grid(w.tiles_per_xcd * NXCD), block(WAVE);
    if (ideg == 19 && smode == 5) UCNS_LAUNCH(k_scatter_s64<19, 39, 5>);
    else if (ideg == 19) UCNS_LAUNCH(k_scatter_s64<19, 39, 7>);
    else if (smode == 5) UCNS_LAUNCH(k_scatter_s64<9, 19, 5>);
    else if (smode == 6) UCNS_LAUNCH(k_scatter_s64<9, 19, 6>);
    else UCNS_LAUNCH(k_scatter_s64<9, 19, 7>);
}
void launch_scatter(const ReconWParams<float> &w, int ideg, int smode, hipStream_t stream) {
    const dim3 grid(w.tiles_per_xcd * NXCD), block(WAVE);
    if (ideg == 19 && smode == 5) UCNS_LAUNCH(k_scatter_s32<19, 39, 5>);
    else if (ideg == 19) UCNS_LAUNCH(k_scatter_s32<19, 39, 7>);
    else if (smode == 5) UCNS_LAUNCH(k_scatter_s32<9, 19, 5>);
    else if (smode == 6) UCNS_LAUNCH(k_scatter_s32<9, 19, 6>);
    else UCNS_LAUNCH(k_scatter_s32<9, 19, 7>);
}
#undef UCNS_LAUNCH

}  // namespace ucns
