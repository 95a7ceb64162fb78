// Conserved update of an interior cell, for the update kernels and for the
// sweep that forms the z fluxes as well (units that do not contract).
#pragma once
#include "mhd_kernels.hpp"

namespace mhd {

// ------------------------------------------------------------------------
// conserved update of one interior cell: get_conserve + advance_corrector1
// (+ stage combine + pressure) + advance_corrector2 (+ combine + velocity)
// (mhd3d3.f90:1641-1650, 3842-3907, 3648-3792).
//   NST = 0: Adams-Bashforth corrector (no combine, p from the new momentum)
//   NST = 2/3: TVD RK stage ST
// A Runge-Kutta stage 1 holds advance_previous' copies (the conserved state it
// starts from, mhd3d3.f90:3794-3819) in registers and stores them for the
// later stages, which saves the pass that read the state again (k_ct does
// the same for the faces): at 96^3 that pass took 26 us a step.
// ------------------------------------------------------------------------
struct Cells {  // cell primitives written by the update
    double *rho, *vx, *vy, *vz, *p;
};
struct CCells {  // cell primitives the update starts from
    const double *rho, *vx, *vy, *vz, *p;
};
struct PrevRK {  // advance_previous, RK flavour (owned cells)
    double *rho, *mx, *my, *mz, *eng;
};

template <typename TF>
struct FluxSet {
    const TF *x, *y, *z;
    long nfx, nfy, nfz;
};


// CFL partials of the updated state, computed by the update itself (get_dt
// on the new state, mhd3d3.f90:1608-1639): cell B from the stage's new
// faces (CT has written them before the update runs; the affine metric's
// cell-B map when on), the CFL step of every owned cell, one minimum per
// workgroup.  Owned cells only: the caller takes this where every ghost
// cell repeats an owned cell (periodic axes whose ghost spacings repeat the
// owned ones), so the minimum is get_dt's over the ghost-inclusive block.
struct UpdDt {
    const double *bi, *bj, *bk;  // the new faces
    double M[9];                 // affine metric's cell-B map (on != 0)
    int on;
    double gam, cfl;
    double* part;                // one partial per workgroup
};

// GEN: general metric (gm), div = (sum_f F_f |S_f| out) / V; a template
// parameter so that the other grids' kernel carries none of its registers.
// DT: CFL partials of the new state as well (UpdDt)
// Returns the cell's CFL step (DT; else infinity).  div(f): the divergence of flux
// f; live: false leaves the cell alone
template <int NST, int ST, bool DT, typename Div>
__device__ __forceinline__ double update_ijk(const Dims& d, double gm1, double tau, const CCells& s, const Cells& so,
                                            const PrevRK& pv, const double* __restrict__ dx,
                                            const double* __restrict__ dy, const double* __restrict__ dz,
                                            const UpdDt& udt, int i, int j, int k, bool live, Div div) {
    const int ng = d.ng;
    const ptrdiff_t q = ix(d.nx, d.ny, ng + i, ng + j, ng + k);
    // get_conserve from the stage's primitives
    const double r0 = s.rho[q], u = s.vx[q], v = s.vy[q], w = s.vz[q];
    const double mx0 = r0 * u, my0 = r0 * v, mz0 = r0 * w;
    const double e0 = .5 * r0 * (u * u + v * v + w * w) + s.p[q] / gm1;
    double rho = r0 - tau * div(0);
    double eng = e0 - tau * div(4);
    double mx = mx0 - tau * div(1);
    double my = my0 - tau * div(2);
    double mz = mz0 - tau * div(3);
    double hx = mx, hy = my, hz = mz;
    if (NST > 0 && ST == 1) {
        pv.rho[q] = r0;
        pv.mx[q] = mx0;
        pv.my[q] = my0;
        pv.mz[q] = mz0;
        pv.eng[q] = e0;
    } else if (NST == 2 && ST == 2) {
        rho = (pv.rho[q] + rho) / 2.;
        hx = (pv.mx[q] + mx) / 2.;
        hy = (pv.my[q] + my) / 2.;
        hz = (pv.mz[q] + mz) / 2.;
        eng = (pv.eng[q] + eng) / 2.;
    } else if (NST == 3 && ST == 2) {
        rho = (3. * pv.rho[q] + rho) / 4.;
        hx = (3. * pv.mx[q] + mx) / 4.;
        hy = (3. * pv.my[q] + my) / 4.;
        hz = (3. * pv.mz[q] + mz) / 4.;
        eng = (3. * pv.eng[q] + eng) / 4.;
    } else if (NST == 3 && ST == 3) {
        rho = (pv.rho[q] + 2. * rho) / 3.;
        hx = (pv.mx[q] + 2. * mx) / 3.;
        hy = (pv.my[q] + 2. * my) / 3.;
        hz = (pv.mz[q] + 2. * mz) / 3.;
        eng = (pv.eng[q] + 2. * eng) / 3.;
    }
    // pressure from the hydro-only momentum (3685, 3876)
    const double p = gm1 * (eng - .5 * (hx * hx + hy * hy + hz * hz) / rho);
    mx = mx - tau * div(5);
    my = my - tau * div(6);
    mz = mz - tau * div(7);
    if (NST == 2 && ST == 2) {
        mx = (pv.mx[q] + mx) / 2.;
        my = (pv.my[q] + my) / 2.;
        mz = (pv.mz[q] + mz) / 2.;
    } else if (NST == 3 && ST == 2) {
        mx = (3. * pv.mx[q] + mx) / 4.;
        my = (3. * pv.my[q] + my) / 4.;
        mz = (3. * pv.mz[q] + mz) / 4.;
    } else if (NST == 3 && ST == 3) {
        mx = (pv.mx[q] + 2. * mx) / 3.;
        my = (pv.my[q] + 2. * my) / 3.;
        mz = (pv.mz[q] + 2. * mz) / 3.;
    }
    const double un = mx / rho, vn = my / rho, wn = mz / rho;
    if (live) {
        so.rho[q] = rho;
        so.p[q] = p;
        so.vx[q] = un;
        so.vy[q] = vn;
        so.vz[q] = wn;
    }
    double dtc = __builtin_huge_val();
    if constexpr (DT) {
        if (live) {
            // get_bxyz of the new faces, as k_bxyz
            const ptrdiff_t gi = ix(d.nx + 1, d.ny, ng + i, ng + j, ng + k), gj = ix(d.nx, d.ny + 1, ng + i, ng + j, ng + k);
            double x = .5 * (udt.bi[gi + 1] + udt.bi[gi]);
            double y = .5 * (udt.bj[gj + d.nx] + udt.bj[gj]);
            double z = .5 * (udt.bk[q + (ptrdiff_t)d.nx * d.ny] + udt.bk[q]);
            if (udt.on) {
                const double fx = x, fy = y, fz = z;
                x = udt.M[0] * fx + udt.M[1] * fy + udt.M[2] * fz;
                y = udt.M[3] * fx + udt.M[4] * fy + udt.M[5] * fz;
                z = udt.M[6] * fx + udt.M[7] * fy + udt.M[8] * fz;
            }
            dtc = cfl_dt(udt.gam, udt.cfl, un, vn, wn, x, y, z, rho, p, dx[ng + i - 1], dy[ng + j - 1],
                         dz[ng + k - 1]);
        }
    }
    return dtc;
}

// cell t of the block, all fluxes from memory
template <int NST, int ST, typename TF, bool GEN, bool DT = false>
__device__ __forceinline__ double update_cell(const Dims& d, double gm1, const double* __restrict__ tau_p,
                                              const CCells& s, const Cells& so, const PrevRK& pv,
                                              const FluxSet<TF>& F, const double* __restrict__ dx,
                                              const double* __restrict__ dy, const double* __restrict__ dz,
                                              const GMet& gm, long ncell, const UpdDt& udt, long t) {
    if constexpr (!DT) {
        if (t >= ncell) return __builtin_huge_val();
    }
    // with DT every thread reaches the workgroup minimum: threads past the
    // end work on cell 1 and store nothing
    const bool live = t < ncell;
    int i, j, k;
    unflat(live ? t : 0, d.nx0, d.ny0, i, j, k);
    const int ng = d.ng;
    const ptrdiff_t q = ix(d.nx, d.ny, ng + i, ng + j, ng + k);
    const double dxi = dx[ng + i - 1], dyj = dy[ng + j - 1], dzk = dz[ng + k - 1];
    const ptrdiff_t fx0 = ix(d.nx0 + 1, d.ny0, i, j, k);
    const ptrdiff_t fy0 = ix(d.nx0, d.ny0 + 1, i, j, k), fy1 = fy0 + d.nx0;
    const ptrdiff_t fz0 = ix(d.nx0, d.ny0, i, j, k), fz1 = fz0 + (ptrdiff_t)d.nx0 * d.ny0;
    double ar[6] = {0., 0., 0., 0., 0., 0.}, iv = 0.;
    if constexpr (GEN) {
        const ptrdiff_t gi = ix(d.nx + 1, d.ny, ng + i, ng + j, ng + k), gj = ix(d.nx, d.ny + 1, ng + i, ng + j, ng + k);
        ar[0] = gm.af[0][gi];
        ar[1] = gm.af[0][gi + 1];
        ar[2] = gm.af[1][gj];
        ar[3] = gm.af[1][gj + d.nx];
        ar[4] = gm.af[2][q];
        ar[5] = gm.af[2][q + (ptrdiff_t)d.nx * d.ny];
        iv = gm.ivol[q];
    }
    auto div = [&](int f) -> double {
        if constexpr (GEN)
            return ((double(F.x[f * F.nfx + fx0 + 1]) * ar[1] - double(F.x[f * F.nfx + fx0]) * ar[0]) +
                    (double(F.y[f * F.nfy + fy1]) * ar[3] - double(F.y[f * F.nfy + fy0]) * ar[2]) +
                    (double(F.z[f * F.nfz + fz1]) * ar[5] - double(F.z[f * F.nfz + fz0]) * ar[4])) * iv;
        return (double(F.x[f * F.nfx + fx0 + 1]) - double(F.x[f * F.nfx + fx0])) / dxi +
               (double(F.y[f * F.nfy + fy1]) - double(F.y[f * F.nfy + fy0])) / dyj +
               (double(F.z[f * F.nfz + fz1]) - double(F.z[f * F.nfz + fz0])) / dzk;
    };
    return update_ijk<NST, ST, DT>(d, gm1, *tau_p, s, so, pv, dx, dy, dz, udt, i, j, k, live, div);
}

}  // namespace mhd
