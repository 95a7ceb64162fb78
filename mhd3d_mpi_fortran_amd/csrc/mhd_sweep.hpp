// The z sweep of a binary64 Adams-Bashforth stage and the conserved update in one
// kernel: z face fluxes are formed in LDS and consumed there.
#pragma once
#include "mhd_ops.hpp"
#include "mhd_sweep_args.hpp"

namespace mhd {

// A workgroup marches along z in tiles of 4 face planes by 64 x (one wavefront
// a plane) over the faces of `cells` cells: each thread forms its face, passes
// the 8 products on through LDS and updates the cell below the face, whose other
// z face is the wavefront's before it (of the tile before, for the first).  The
// arithmetic is k_flux' and k_update's, the spacings' reciprocals shared by the
// 8 divergences.  Workgroup order: 64-wide x tiles, then rows, then runs along z,
// an eighth of the rows to each XCD (neighbouring rows share their y faces).
//
// The z products need not be read back, nor, but for a call's last step, be
// written (128 bytes a cell), and the update's loads run beside other wavefronts'
// flux arithmetic: at 256^3 (PDM) z flux and update take 1.51 ms for 0.87 + 0.94,
// the step 5.87 ms for 6.21; 128^3 859 us for 901, 1000 x 600 x 5 1.68 ms for 1.79
// (rows that leave lanes idle: sweep_fills); TVD 192^3 2.29 ms for 2.45, WENO5 and
// MPWENO5 128^3 1 to 2 % less.  Bound by memory traffic, 8.1 GB (compulsory 4.6) at the
// 5.3 TB/s that a copy reaches, with 3 wavefronts a SIMD (168 VGPRs; capped at 128
// it took 1.74 ms, and with the x and y differences loaded before the flux 1.80).
// The same in binary32 took 1.48 ms for 0.26 + 0.68 and is not here.
template <int M, int MET>
__global__ void __launch_bounds__(kBlock)
    k_sweep_update(Dims d, Coef<double> c, Prim<double> q, Normals<double> nm, SweepArgs a) {
    __shared__ double ex[8][2 * (kTileN - 1) + 3][kTileX];
    const unsigned ntx = (unsigned)(d.nx0 + kTileX - 1) / kTileX, no = (unsigned)d.ny0;
    const unsigned per = (ntx * no + kXcd / 2) / kXcd;
    const unsigned lb = xcd_map_run(blockIdx.x, gridDim.x, per > 0 ? per : 1u);
    const unsigned tx = lb % ntx;
    const int j = (int)(lb / ntx % no) + 1;
    const int c0 = (int)(lb / ntx / no) * a.cells, c1 = min(c0 + a.cells, d.nz0);
    const int lane = threadIdx.x & (kTileX - 1), w = threadIdx.x / kTileX;
    const int x = (int)tx * kTileX + lane, i = min(x, d.nx0 - 1) + 1;
    const Divisor<double> dxi(a.dx[d.ng + i - 1]), dyj(a.dy[d.ng + j - 1]);
    const double tau = *a.tau_p;
    int p2 = 0, p3 = 0;
#pragma unroll 1
    for (int base = c0; base <= c1; base += kTileN) {
        const int face = base + w;   // 0-based; past the block: its last face, not stored
        const int cell = face - 1;
        const bool live = x < d.nx0 && cell >= c0 && cell < c1;
        double l[8], r[8], fx[8];
        const Taps<double, M, double> tp(ix(d.nx, d.ny, d.ng + i, d.ng + j, d.ng + min(face, d.nz0) + 1),
                                         (ptrdiff_t)d.nx * d.ny);
        recon_taps<double, M>(q.rho, tp, c, l[0], r[0]);
        recon_taps<double, M>(q.vx, tp, c, l[1], r[1]);
        recon_taps<double, M>(q.vy, tp, c, l[2], r[2]);
        recon_taps<double, M>(q.vz, tp, c, l[3], r[3]);
        recon_taps<double, M>(q.p, tp, c, l[4], r[4]);
        recon_taps<double, M>(q.bx, tp, c, l[5], r[5]);
        recon_taps<double, M>(q.by, tp, c, l[6], r[6]);
        recon_taps<double, M>(q.bz, tp, c, l[7], r[7]);
        if constexpr (MET == 1) face_flux_met_vals<double>(c, l, r, nm.n[2], fx);
        else face_flux_vals<double, 3>(c, l, r, fx);
        // products for the wavefront above: two sets in turn, so that one barrier
        // a tile does; the last one's, read in the next tile, three
        const int own = w < kTileN - 1 ? p2 * (kTileN - 1) + w : 2 * (kTileN - 1) + p3;
        const int below = w > 0 ? p2 * (kTileN - 1) + w - 1 : 2 * (kTileN - 1) + (p3 > 0 ? p3 - 1 : 2);
        p2 ^= 1;
        p3 = p3 < 2 ? p3 + 1 : 0;
#pragma unroll
        for (int f = 0; f < 8; ++f) ex[f][own][lane] = fx[f];
        // a call's last step leaves its fluxes, each face once
        if (a.fz && x < d.nx0 && (face < c1 || (face == c1 && c1 == d.nz0))) {
            const ptrdiff_t t = ix(d.nx0, d.ny0, i, j, face + 1);
#pragma unroll
            for (int f = 0; f < 8; ++f) a.fz[f * a.F.nfz + t] = fx[f];
        }
        __syncthreads();
        if (live) {
            const Divisor<double> dzk(a.dz[d.ng + cell]);
            const ptrdiff_t fx0 = ix(d.nx0 + 1, d.ny0, i, j, cell + 1), fy0 = ix(d.nx0, d.ny0 + 1, i, j, cell + 1);
            update_ijk<0, 0, false>(d, a.gm1, tau, a.s, a.so, PrevRK{}, a.dx, a.dy, a.dz, UpdDt{}, i, j, cell + 1, true,
                                    [&](int f) -> double {
                return dxi.under(a.F.x[f * a.F.nfx + fx0 + 1] - a.F.x[f * a.F.nfx + fx0]) +
                       dyj.under(a.F.y[f * a.F.nfy + fy0 + d.nx0] - a.F.y[f * a.F.nfy + fy0]) +
                       dzk.under(fx[f] - ex[f][below][lane]);
            });
        }
    }
}

template <int M>
void sweep_launch_m(mhd_ctx* c, Src<double> s, const SweepArgs& a) {
    const Prim<double> q{s.rho, s.vx, s.vy, s.vz, s.p, s.bx, s.by, s.bz};
    launch(c, MHD_K_UPDATE, dim3(sweep_blocks(c->d)), dim3(kBlock),
           c->met.on ? k_sweep_update<M, 1> : k_sweep_update<M, 0>, c->d, make_coef<double>(c), q,
           make_normals<double>(c), a);
}

inline void sweep_launch(mhd_ctx* c, Src<double> s, const SweepArgs& a) {
    switch (c->p.reconop) {
    case PDM: sweep_launch_m<PDM>(c, s, a); break;
    case TVD: sweep_launch_m<TVD>(c, s, a); break;
    case WENO5: sweep_launch_m<WENO5>(c, s, a); break;
    default: sweep_launch_m<MPWENO5>(c, s, a); break;
    }
}

}  // namespace mhd
