// Binary64 edge EMF (get_eijk_LFM, mhd3d3.f90:1754-1856) of the WENO5 and
// MPWENO5 reconstructions, in two kernels.
//
// The corner velocity of an edge (get_vav_center2corner, mhd3d3.f90:1868-2013)
// reconstructs the six lines of its 6x6 footprint along one corner axis, then
// the six left and the six right states along the other, and the same with
// the axes exchanged: 12 line reconstructions and 4 of their states per
// velocity.  A line's reconstruction is the same for the six edges whose
// footprints it crosses, and its states are needed by nothing else, so
//   k_weno_lines  reconstructs every velocity component along every axis once
//                 (3 line reconstructions per cell and component), left and
//                 right states to a scratch array, and
//   k_emf_weno    forms each edge's EMF from those states: 4 reconstructions
//                 per velocity and the two of the face field.
// Per edge that is 13 reconstructions instead of the 34 of a kernel that holds
// the whole footprint, whose window also needs more than 200 VGPRs (two
// wavefronts per SIMD).  Both kernels are bound by VALU issue (the divisions
// of the WENO weights): the states' round trip through memory is 18 words per
// cell.  All three directions of the 96 x 64 x 128 shell (WENO5) took 1154 us
// with that kernel and take 363 us with these (lines 95 us, edges 268 us).
// The operations of each reconstruction, and so the results, are the
// reference's bit for bit.
//
// The scratch holds a slab of z planes (mhd_create sizes it): the launcher
// walks the block slab by slab, reconstructing the 5 planes above and below a
// slab's edges that the z footprints reach into.
#pragma once
#include "mhd_kernels.hpp"

namespace mhd {

// the reconstructed states: component c along axis a, side 0 left, 1 right, at
// the face below cell q of that axis
template <typename R>
struct WenoLines {
    R* s;            // 18 arrays of `stride`
    long stride;     // nx * ny * planes held
    int kz;          // ghost-inclusive plane (1-based) of the first one held
    __device__ __forceinline__ R* at(int c, int a, int side) const {
        return s + (long)((c * 3 + a) * 2 + side) * stride;
    }
};

// one thread per cell of the slab (x fastest, whole ghost-inclusive planes),
// blockIdx.y = 3 * component + axis.  Component c's lines along axis a run
// through the faces a needs (owned + 1); across them they are needed as taps
// of the other corner axis, 3 cells past the owned ones on the axes of the
// corner planes that (c, a) belong to
template <typename R, int M, typename TI>
__global__ void __launch_bounds__(kBlock) k_weno_lines(Dims d, Coef<R> c, const TI* __restrict__ v0,
                                                      const TI* __restrict__ v1, const TI* __restrict__ v2,
                                                      WenoLines<R> ln, int k0, int k1, long ncell) {
    const long t = gtid_xcd();
    if (t >= ncell) return;
    const int cc = blockIdx.y / 3, a = blockIdx.y - 3 * cc;
    int x[3];
    unflat(t, d.nx, d.ny, x[0], x[1], x[2]);
    x[2] += ln.kz - 1;
    const int n[3] = {d.nx0, d.ny0, d.nz0};
    const int ng = d.ng;
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        int lo = ng + 1, hi = ng + n[b];
        if (b == 2) {  // the slab's edges k0..k1
            lo = ng + k0;
            hi = min(hi, ng + k1);
        }
        if (b == a) hi = b == 2 ? ng + k1 : hi + 1;
        else if (cc == a || b == cc) {
            lo -= 3;
            hi = b == 2 ? ng + k1 + 2 : hi + 3;
        }
        if (x[b] < lo || x[b] > hi) return;
    }
    const TI* __restrict__ v = cc == 0 ? v0 : (cc == 1 ? v1 : v2);
    const ptrdiff_t st = a == 0 ? 1 : (a == 1 ? (ptrdiff_t)d.nx : (ptrdiff_t)d.nx * d.ny);
    R l, r;
    recon_line<R, M>(v, ix(d.nx, d.ny, x[0], x[1], x[2]), st, c, l, r);
    ln.at(cc, a, 0)[t] = l;
    ln.at(cc, a, 1)[t] = r;
}

// corner velocity of one edge: component cc, corner axes a1, a2 with strides
// s1, s2; q the edge's base cell in the scratch, f0 the same cell in the field
template <typename R, int M, typename TI>
__device__ __forceinline__ R weno_corner(const WenoLines<R>& ln, const TI* __restrict__ v, const Coef<R>& c, int cc,
                                         int a1, int a2, ptrdiff_t s1, ptrdiff_t s2, ptrdiff_t q, ptrdiff_t f0) {
    R v00_0, v10_0, v01_0, v11_0, v00_1, v01_1, v10_1, v11_1;
    recon_line<R, M>(ln.at(cc, a1, 0), q, s2, c, v00_1, v01_1);
    recon_line<R, M>(ln.at(cc, a1, 1), q, s2, c, v10_1, v11_1);
    recon_line<R, M>(ln.at(cc, a2, 0), q, s1, c, v00_0, v01_0);
    recon_line<R, M>(ln.at(cc, a2, 1), q, s1, c, v10_0, v11_0);
    auto cv = [&](int o1, int o2) { return R(v[f0 + o1 * s1 + o2 * s2]); };
    const R cmm = cv(-1, -1), c0m = cv(0, -1), cm0 = cv(-1, 0), c00 = cv(0, 0);
    const R d00 = sgn1(fabs(cv(-2, -1) - cmm) - fabs(cv(-1, -2) - cmm));
    const R d10 = sgn1(fabs(cv(1, -1) - c0m) - fabs(cv(0, -2) - c0m));
    const R d01 = sgn1(fabs(cv(-2, 0) - cm0) - fabs(cv(-1, 1) - cm0));
    const R d11 = sgn1(fabs(cv(1, 0) - c00) - fabs(cv(0, 1) - c00));
    const R v00 = (R(1) + d00) / R(2) * v00_0 + (R(1) - d00) / R(2) * v00_1;
    const R v10 = (R(1) + d10) / R(2) * v10_0 + (R(1) - d10) / R(2) * v10_1;
    const R v01 = (R(1) + d01) / R(2) * v01_0 + (R(1) - d01) / R(2) * v01_1;
    const R v11 = (R(1) + d11) / R(2) * v11_0 + (R(1) - d11) / R(2) * v11_1;
    return R(.25) * (v00 + v01 + v10 + v11);
}

// EMF of the edges along axis E (0 x, 1 y, 2 z) of the slab k0..k1, one thread
// per edge; v[c] the velocity components, b1 and b2 the faces normal to the
// corner axes
template <typename R, int M, int E, typename TI, typename TF>
__device__ __forceinline__ void emf_weno_edge(const Dims& d, const Coef<R>& c, const TI* const* v,
                                              const TI* const* bf, const TI* __restrict__ vf,
                                              const WenoLines<R>& ln, R ef, const double* __restrict__ efa,
                                              TF* __restrict__ e, int k0, int k1) {
    constexpr int A1 = (E + 1) % 3, A2 = (E + 2) % 3;
    const int ii = d.nx0 + (E != 0), jj = d.ny0 + (E != 1);
    const int kend = min(k1, d.nz0 + (E != 2));
    const long t = gtid_xcd();
    if (t >= (long)ii * jj * (kend - k0 + 1)) return;
    int i, j, k;
    unflat(t, ii, jj, i, j, k);
    k += k0 - 1;
    const int nx = d.nx, ny = d.ny, I = d.ng + i, J = d.ng + j, K = d.ng + k;
    const ptrdiff_t st[3] = {1, (ptrdiff_t)nx, (ptrdiff_t)nx * ny};
    const ptrdiff_t f0 = ix(nx, ny, I, J, K), q = ix(nx, ny, I, J, K - ln.kz + 1);
    const R v1av = weno_corner<R, M>(ln, v[A1], c, A1, A1, A2, st[A1], st[A2], q, f0);
    const R v2av = weno_corner<R, M>(ln, v[A2], c, A2, A1, A2, st[A1], st[A2], q, f0);
    // face normal to A1 along A2, and normal to A2 along A1
    const int n1x = nx + (A1 == 0), n1y = ny + (A1 == 1), n2x = nx + (A2 == 0), n2y = ny + (A2 == 1);
    const ptrdiff_t t1[3] = {1, (ptrdiff_t)n1x, (ptrdiff_t)n1x * n1y}, t2[3] = {1, (ptrdiff_t)n2x, (ptrdiff_t)n2x * n2y};
    R b1l, b1r, b2l, b2r;
    recon_line<R, M>(bf[A1], ix(n1x, n1y, I, J, K), t1[A2], c, b1l, b1r);
    recon_line<R, M>(bf[A2], ix(n2x, n2y, I, J, K), t2[A1], c, b2l, b2r);
    const R sig1 = sgn1(v1av), sig2 = sgn1(v2av);
    const R b1u = pick(sig2, b1l, b1r);
    const R b2u = pick(sig1, b2l, b2r);
    R dum = -v1av * b2u + v2av * b1u;
    // the four cells around the edge, in the reference's order of summation
    const R fuw = R(vf[f0 - st[A1] - st[A2]]), f1 = R(vf[f0 - st[A1]]), f2 = R(vf[f0 - st[A2]]), f00 = R(vf[f0]);
    const R eta = R(.25) * (fuw + f2 + f00 + f1);
    dum = dum + eta * (b1l + b2r - b1r - b2l);
    const ptrdiff_t eo = ix(ii, jj, i, j, k);
    e[eo] = TF(dum * (efa ? R(efa[eo]) : ef));
}

template <typename TI>
struct EmfWenoIn {
    const TI *v[3], *b[3], *vf;   // velocity components (face-normal with a metric), faces, fast speed
    const double* efa[3];         // general metric's factor per edge, or null
};
template <typename R, typename TF>
struct EmfWenoOut {
    TF* e[3];
    R ef[3];
};

// blockIdx.y = edge direction
template <typename R, int M, typename TI, typename TF>
__global__ void __launch_bounds__(kBlock) k_emf_weno(Dims d, Coef<R> c, EmfWenoIn<TI> in, EmfWenoOut<R, TF> o,
                                                    WenoLines<R> ln, int k0, int k1) {
    if (blockIdx.y == 0)
        emf_weno_edge<R, M, 0, TI, TF>(d, c, in.v, in.b, in.vf, ln, o.ef[0], in.efa[0], o.e[0], k0, k1);
    else if (blockIdx.y == 1)
        emf_weno_edge<R, M, 1, TI, TF>(d, c, in.v, in.b, in.vf, ln, o.ef[1], in.efa[1], o.e[1], k0, k1);
    else
        emf_weno_edge<R, M, 2, TI, TF>(d, c, in.v, in.b, in.vf, ln, o.ef[2], in.efa[2], o.e[2], k0, k1);
}

}  // namespace mhd
