// Launchers of the stencil kernels (face flux, edge EMF), instantiated once
// per arithmetic type in its own translation unit so that each can carry its
// own floating-point contract: binary64 without contraction (reference
// parity), fp32 with FMA contraction (mixed precision).
#pragma once
#include "mhd_emf.hpp"
#include "mhd_emf_weno.hpp"
#include "mhd_launch.hpp"

namespace mhd {

// edges handled per thread along the march axis: long runs share the
// sliding stencil windows; a launch whose long-run grid has fewer threads
// than c->emf_fill takes runs of 2 instead, trading window reuse for latency
// hiding.  PDM's ei march (both corner axes strided, its loads the slowest)
// takes runs of 16: at 256^3 0.20 vs 0.22 ms (fp32) and 0.48 vs 0.51 ms
// (binary64), and runs of 32 are slower again (0.23 ms fp32, 0.83 ms
// binary64); for ej and ek runs of 16 measured slower (0.19 vs 0.17 ms
// fp32), and so did runs of 4 (0.17 vs 0.16 ms) and register caps that
// buy a fifth or sixth wavefront per SIMD with spills (EMF class 0.61 and
// 0.72 vs 0.53 ms).
template <int M, int K>
struct EmfSteps {
    static constexpr int T = (scheme(M) == TVD || (M == PDM && K == 1)) ? 16 : 8;
    static constexpr int T_SHORT = 2;
};

// Small and ordinary blocks: the face fluxes and edge EMFs of a stage in one
// launch.  They are independent, and on such blocks each kernel alone neither
// fills the chip (64^3: 500-1100 workgroups of one direction on 256 CUs) nor
// lives long enough to hide its own start and tail, so one after the other they
// take several times what their arithmetic needs.  The grid is the six
// kernels' workgroups end to end, the EMF's (the longest) first; every
// workgroup belongs to one of them.  Its registers are the largest of the six,
// which large blocks would pay for in the flux: blocks past the size to which the
// one launch measured faster (merge_cells) keep the separate kernels, EMF and flux
// on two streams.  A stage of 64^3 (PDM, binary64) took
// 114 us with the six kernels and takes 84 us, 16^3 51 and 12 us.
template <typename R, typename TF>
struct StencilOut {
    TF* flux[3];
    TF* emf[3];
    long nface[3];
    R ef[3];
    const double* efa[3];
    long nthreads[3];      // EMF threads per direction
    unsigned end[6];       // last workgroup + 1 of the EMF's and the flux's directions
};
template <typename R, int M, typename TI, typename TF, int MET, bool EMF, int T>
__global__ void __launch_bounds__(kBlock) k_stencils(Dims d, Coef<R> c, Prim<TI> q, Normals<R> nm, GMet gm,
                                                    EmfIn<TI> e1, EmfIn<TI> e2, EmfIn<TI> e3,
                                                    StencilOut<R, TF> o) {
    __shared__ typename FluxRing<R, M, TI, 1>::Win win;
    const unsigned b = blockIdx.x;
    auto place = [&](int p) {  // place within part p, in its XCD-aware order
        const unsigned lo = p ? o.end[p - 1] : 0;
        return xcd_map(b - lo, o.end[p] - lo);
    };
    if constexpr (EMF) {
        if (b < o.end[0]) {
            emf_block<R, M, 1, T, TI, TF>(d, c, e1, o.ef[0], o.efa[0], o.emf[0], o.nthreads[0], place(0));
            return;
        }
        if (b < o.end[1]) {
            emf_block<R, M, 2, T, TI, TF>(d, c, e2, o.ef[1], o.efa[1], o.emf[1], o.nthreads[1], place(1));
            return;
        }
        if (b < o.end[2]) {
            emf_block<R, M, 3, T, TI, TF>(d, c, e3, o.ef[2], o.efa[2], o.emf[2], o.nthreads[2], place(2));
            return;
        }
    }
    if (b < o.end[3]) flux_block<R, M, 2, TI, TF, MET, 1>(d, c, q, nm, gm, o.flux[1], o.nface[1], place(3), win);
    else if (b < o.end[4]) flux_block<R, M, 3, TI, TF, MET, 1>(d, c, q, nm, gm, o.flux[2], o.nface[2], place(4), win);
    else flux_block<R, M, 1, TI, TF, MET, 1>(d, c, q, nm, gm, o.flux[0], o.nface[0], place(5), win);
}

template <typename R, typename TI, typename TF, int M, int MET>
void flux_launch_mm(mhd_ctx* c, Src<TI> s, bool z) {
    const Coef<R> co = make_coef<R>(c);
    const Prim<TI> q{s.rho, s.vx, s.vy, s.vz, s.p, s.bx, s.by, s.bz};
    const Normals<R> nm = make_normals<R>(c);
    launch(c, MHD_K_FLUX, blocks(c->nf[0]), dim3(kBlock), k_flux<R, M, 1, TI, TF, MET>, c->d, co, q, nm, c->gm,
           (TF*)c->flux[0], c->nf[0]);
    const Dims& d = c->d;
    // fp32 inputs march kFluxRun tiles per workgroup where that still leaves
    // kFluxRunBlocks workgroups, else one tile each (k_flux)
    const unsigned y8 = face_runs<2>(d.nx0, d.ny0 + 1, d.nz0, kFluxRun);
    const unsigned z8 = face_runs<3>(d.nx0, d.ny0, d.nz0 + 1, kFluxRun);
    const bool fp32 = sizeof(TI) == 4;
    if (fp32 && y8 >= (unsigned)kFluxRunBlocks)
        launch(c, MHD_K_FLUX, dim3(y8), dim3(kBlock), k_flux<R, M, 2, TI, TF, MET, kFluxRun>, c->d, co, q, nm,
               c->gm, (TF*)c->flux[1], c->nf[1]);
    else
        launch(c, MHD_K_FLUX, dim3(face_tiles<2>(d.nx0, d.ny0 + 1, d.nz0)), dim3(kBlock),
               k_flux<R, M, 2, TI, TF, MET>, c->d, co, q, nm, c->gm, (TF*)c->flux[1], c->nf[1]);
    if (!z) return;
    if (fp32 && z8 >= (unsigned)kFluxRunBlocks)
        launch(c, MHD_K_FLUX, dim3(z8), dim3(kBlock), k_flux<R, M, 3, TI, TF, MET, kFluxRun>, c->d, co, q, nm,
               c->gm, (TF*)c->flux[2], c->nf[2]);
    else
        launch(c, MHD_K_FLUX, dim3(face_tiles<3>(d.nx0, d.ny0, d.nz0 + 1)), dim3(kBlock),
               k_flux<R, M, 3, TI, TF, MET>, c->d, co, q, nm, c->gm, (TF*)c->flux[2], c->nf[2]);
}

template <typename R, typename TI, typename TF, int M>
void flux_launch_m(mhd_ctx* c, Src<TI> s, bool z) {
    if (c->met.mode == 2) flux_launch_mm<R, TI, TF, M, 2>(c, s, z);
    else if (c->met.on) flux_launch_mm<R, TI, TF, M, 1>(c, s, z);
    else flux_launch_mm<R, TI, TF, M, 0>(c, s, z);
}

template <typename R, typename TI, typename TF>
void flux_launch(mhd_ctx* c, Src<TI> s, bool z) {
    if constexpr (sizeof(R) == 8) {
        switch (recon_code(c)) {
        case TVD_FULL: flux_launch_m<R, TI, TF, TVD_FULL>(c, s, z); return;
        case WENO5_FULL: flux_launch_m<R, TI, TF, WENO5_FULL>(c, s, z); return;
        case MPWENO5_FULL: flux_launch_m<R, TI, TF, MPWENO5_FULL>(c, s, z); return;
        }
    }
    switch (c->p.reconop) {
    case PDM: flux_launch_m<R, TI, TF, PDM>(c, s, z); break;
    case TVD: flux_launch_m<R, TI, TF, TVD>(c, s, z); break;
    case WENO5: flux_launch_m<R, TI, TF, WENO5>(c, s, z); break;
    default: flux_launch_m<R, TI, TF, MPWENO5>(c, s, z); break;
    }
}

// threads and workgroups of direction K's march (k_emf_march)
template <typename R, int M, int K, int T>
long emf_threads(const Dims& d) {
    const long ii = d.nx0 + (K != 1) + (M == PDM && K == 2 && sizeof(R) == 8 ? 7 : 0);
    const long no = K == 3 ? d.nz0 : (K == 1 ? d.ny0 + 1 : d.ny0);
    const long nm = K == 3 ? d.ny0 + 1 : d.nz0 + 1;
    return ii * no * ((nm + T - 1) / T);
}
template <typename R, int M, int K, int T>
unsigned emf_blocks(const Dims& d) {
    if (K == 1) return emf_tiles<T>(d.nx0, d.ny0, d.nz0);
    const long n = emf_threads<R, M, K, T>(d);
    if (M == PDM && K == 2 && sizeof(R) == 8) return (unsigned)((n + kColEdges - 1) / kColEdges);
    return blocks(n).x;
}

template <typename R, int M, int K, int T, typename TI, typename TF>
void emf_launch_kt(mhd_ctx* c, EmfIn<TI> in) {
    const Dims& d = c->d;
    const long n = emf_threads<R, M, K, T>(d);
    const dim3 grid(emf_blocks<R, M, K, T>(d));
    launch(c, MHD_K_EMF, grid, dim3(kBlock), k_emf_march<R, M, K, T, TI, TF>, d, make_coef<R>(c), in,
           R(c->met.ef[K - 1]), c->met.mode == 2 ? c->gm.ef[K - 1] : (const double*)nullptr, (TF*)c->emf[K - 1], n);
}

template <typename R, int M, int K, typename TI, typename TF>
void emf_launch_k(mhd_ctx* c, EmfIn<TI> in) {
    constexpr int T = EmfSteps<M, K>::T;
    const Dims& d = c->d;
    const long ii = d.nx0 + (K != 1);
    const long no = K == 3 ? d.nz0 : (K == 1 ? d.ny0 + 1 : d.ny0);
    const long nm = K == 3 ? d.ny0 + 1 : d.nz0 + 1;
    // a run holds exactly T edges (the last one of a line overlaps its
    // predecessor), so long runs need a march axis of at least T edges; it
    // holds at least 2 = T_SHORT
    if (nm >= T && ii * no * ((nm + T - 1) / T) >= c->emf_fill) emf_launch_kt<R, M, K, T, TI, TF>(c, in);
    else emf_launch_kt<R, M, K, EmfSteps<M, K>::T_SHORT, TI, TF>(c, in);
}

// the binary64 WENO reconstructions' EMF (mhd_emf_weno.hpp), slab by slab of z planes
template <typename R, int M, typename TI, typename TF>
void emf_weno_launch(mhd_ctx* c, const TI* const* u, Src<TI> s) {
    const Dims& d = c->d;
    const Coef<R> co = make_coef<R>(c);
    EmfWenoIn<TI> in{{u[0], u[1], u[2]}, {s.bi, s.bj, s.bk}, s.vf, {}};
    EmfWenoOut<R, TF> out{};
    for (int a = 0; a < 3; ++a) {
        out.e[a] = (TF*)c->emf[a];
        out.ef[a] = R(c->met.ef[a]);
        in.efa[a] = c->met.mode == 2 ? c->gm.ef[a] : nullptr;
    }
    const long plane = (long)d.nx * d.ny;
    const int per = c->weno_planes - kWenoHalo;   // edge planes a slab holds
    for (int k0 = 1; k0 <= d.nz0 + 1; k0 += per) {
        const int k1 = k0 + per - 1 < d.nz0 + 1 ? k0 + per - 1 : d.nz0 + 1;
        const WenoLines<R> ln{(R*)c->weno, plane * c->weno_planes, d.ng + k0 - 3};
        const long nl = plane * (k1 - k0 + 1 + kWenoHalo);
        launch(c, MHD_K_EMF, dim3(blocks(nl).x, 9), dim3(kBlock), k_weno_lines<R, M, TI>, d, co, u[0], u[1], u[2], ln,
               k0, k1, nl);
        // the most edges of the three directions in the slab
        const long nm = (long)(d.nx0 + 1) * (d.ny0 + 1) * (k1 - k0 + 1);
        launch(c, MHD_K_EMF, dim3(blocks(nm).x, 3), dim3(kBlock), k_emf_weno<R, M, TI, TF>, d, co, in, out, ln, k0,
               k1);
    }
}

// edge k: (v1, v2, b1, b2) = (vy, vz, bj, bk), (vz, vx, bk, bi), (vx, vy, bi, bj);
// with a metric the velocities are the face-normal ones w_d = v . n_d
template <typename R, typename TI, typename TF, int M>
void emf_launch_m(mhd_ctx* c, Src<TI> s) {
    const TI* u[3] = {s.vx, s.vy, s.vz};
    if (c->met.on) {
        u[0] = s.w[0];
        u[1] = s.w[1];
        u[2] = s.w[2];
    }
    // in binary64 the WENO footprint's lines are reconstructed once for all the
    // edges they serve; in fp32 the march stays: which products of a line its
    // compiler contracts depends on the line's place in the footprint, so
    // shared lines would round differently by up to 2e-7 of an edge's EMF
    if constexpr ((scheme(M) == WENO5 || scheme(M) == MPWENO5) && sizeof(R) == 8) {
        emf_weno_launch<R, M, TI, TF>(c, u, s);
    } else {
        emf_launch_k<R, M, 1, TI, TF>(c, EmfIn<TI>{u[1], u[2], s.bj, s.bk, s.vf});
        emf_launch_k<R, M, 2, TI, TF>(c, EmfIn<TI>{u[2], u[0], s.bk, s.bi, s.vf});
        emf_launch_k<R, M, 3, TI, TF>(c, EmfIn<TI>{u[0], u[1], s.bi, s.bj, s.vf});
    }
}

template <typename R, typename TI, typename TF>
void emf_launch(mhd_ctx* c, Src<TI> s) {
    if constexpr (sizeof(R) == 8) {
        switch (recon_code(c)) {
        case TVD_FULL: emf_launch_m<R, TI, TF, TVD_FULL>(c, s); return;
        case WENO5_FULL: emf_launch_m<R, TI, TF, WENO5_FULL>(c, s); return;
        case MPWENO5_FULL: emf_launch_m<R, TI, TF, MPWENO5_FULL>(c, s); return;
        }
    }
    switch (c->p.reconop) {
    case PDM: emf_launch_m<R, TI, TF, PDM>(c, s); break;
    case TVD: emf_launch_m<R, TI, TF, TVD>(c, s); break;
    case WENO5: emf_launch_m<R, TI, TF, WENO5>(c, s); break;
    default: emf_launch_m<R, TI, TF, MPWENO5>(c, s); break;
    }
}

// a stage's stencils in one launch (what: kStageFlux | kStageEmf)
template <typename R, typename TI, typename TF, int M, int MET, int T>
void stage_launch_t(mhd_ctx* c, Src<TI> s, int what) {
    const Dims& d = c->d;
    constexpr bool march = M == PDM || M == TVD;
    StencilOut<R, TF> o{};
    unsigned nb[6] = {0, 0, 0, 0, 0, 0};
    for (int a = 0; a < 3; ++a) {
        o.flux[a] = (TF*)c->flux[a];
        o.emf[a] = (TF*)c->emf[a];
        o.nface[a] = c->nf[a];
        o.ef[a] = R(c->met.ef[a]);
        o.efa[a] = c->met.mode == 2 ? c->gm.ef[a] : nullptr;
    }
    if ((what & kStageEmf) && march) {
        o.nthreads[0] = emf_threads<R, M, 1, T>(d);
        o.nthreads[1] = emf_threads<R, M, 2, T>(d);
        o.nthreads[2] = emf_threads<R, M, 3, T>(d);
        nb[0] = emf_blocks<R, M, 1, T>(d);
        nb[1] = emf_blocks<R, M, 2, T>(d);
        nb[2] = emf_blocks<R, M, 3, T>(d);
    }
    if (what & kStageFlux) {
        nb[3] = face_tiles<2>(d.nx0, d.ny0 + 1, d.nz0);
        nb[4] = face_tiles<3>(d.nx0, d.ny0, d.nz0 + 1);
        nb[5] = blocks(c->nf[0]).x;
    }
    unsigned n = 0;
    for (int a = 0; a < 6; ++a) o.end[a] = n += nb[a];
    const Prim<TI> q{s.rho, s.vx, s.vy, s.vz, s.p, s.bx, s.by, s.bz};
    const TI* u[3] = {s.vx, s.vy, s.vz};
    if (c->met.on)
        for (int a = 0; a < 3; ++a) u[a] = s.w[a];
    launch(c, what & kStageFlux ? MHD_K_FLUX : MHD_K_EMF, dim3(n), dim3(kBlock), k_stencils<R, M, TI, TF, MET, march, T>, d,
           make_coef<R>(c), q, make_normals<R>(c), c->gm, EmfIn<TI>{u[1], u[2], s.bj, s.bk, s.vf},
           EmfIn<TI>{u[2], u[0], s.bk, s.bi, s.vf}, EmfIn<TI>{u[0], u[1], s.bi, s.bj, s.vf}, o);
    if constexpr (!march) {
        if (what & kStageEmf) emf_launch_m<R, TI, TF, M>(c, s);
    }
}

// EMF runs of 2 edges per thread; binary64 PDM, whose run start (an 8x8 footprint)
// costs most, takes runs of 4 once runs of 2 give the stage more workgroups than
// there are CUs: below that a stage lasts as long as its longest thread
// (16^3: 44 us a step with runs of 2, 56 with 4, 80 with 8), above as long
// as its arithmetic (24^3: 53 and 52 us; 64^3: 191 and 181; 96^3: 641 and 605; runs
// of 8, at two wavefronts per SIMD, 67, 192 and 642).  TVD's starts are cheap (96^3:
// 566 and 561 us, 32^3: 60 and 61) and fp32 results may depend on the place in a run.
template <typename R, typename TI, typename TF, int M, int MET>
void stage_launch_mm(mhd_ctx* c, Src<TI> s, int what) {
    constexpr int T = EmfSteps<M, 1>::T_SHORT;
    const Dims& d = c->d;
    if constexpr (M == PDM && sizeof(R) == 8) {
        const unsigned n = emf_blocks<R, M, 1, T>(d) + emf_blocks<R, M, 2, T>(d) + emf_blocks<R, M, 3, T>(d) +
                           face_tiles<2>(d.nx0, d.ny0 + 1, d.nz0) + face_tiles<3>(d.nx0, d.ny0, d.nz0 + 1) +
                           blocks(c->nf[0]).x;
        if (n > 256) {
            stage_launch_t<R, TI, TF, M, MET, 4>(c, s, what);
            return;
        }
    }
    stage_launch_t<R, TI, TF, M, MET, T>(c, s, what);
}

template <typename R, typename TI, typename TF, int M>
void stage_launch_m(mhd_ctx* c, Src<TI> s, int what) {
    if (c->met.mode == 2) stage_launch_mm<R, TI, TF, M, 2>(c, s, what);
    else if (c->met.on) stage_launch_mm<R, TI, TF, M, 1>(c, s, what);
    else stage_launch_mm<R, TI, TF, M, 0>(c, s, what);
}

template <typename R, typename TI, typename TF>
void stage_launch(mhd_ctx* c, Src<TI> s, int what) {
    switch (c->p.reconop) {
    case PDM: stage_launch_m<R, TI, TF, PDM>(c, s, what); break;
    case TVD: stage_launch_m<R, TI, TF, TVD>(c, s, what); break;
    case WENO5: stage_launch_m<R, TI, TF, WENO5>(c, s, what); break;
    default: stage_launch_m<R, TI, TF, MPWENO5>(c, s, what); break;
    }
}

// get_v_face (mhd3d3.f90:2594-2615) elementwise in the arithmetic type R of
// the context's flux (binary64 inputs and outputs)
template <typename R>
__global__ void __launch_bounds__(kBlock) k_vface(long n, const double* __restrict__ lam,
                                                 const double* __restrict__ v, double* __restrict__ v0p,
                                                 double* __restrict__ v0n, double* __restrict__ v1p,
                                                 double* __restrict__ v1n, R rspi) {
    const long t = gtid();
    if (t >= n) return;
    R a0, a1, b0, b1;
    vface<R>(R(lam[t]), R(v[t]), +1, rspi, a0, a1);
    vface<R>(R(lam[t]), R(v[t]), -1, rspi, b0, b1);
    v0p[t] = double(a0);
    v1p[t] = double(a1);
    v0n[t] = double(b0);
    v1n[t] = double(b1);
}

template <typename R>
void vface_launch(mhd_ctx* c, long n, const double* lam, const double* v, double* v0p, double* v0n, double* v1p,
                  double* v1n) {
    launch(c, MHD_K_FLUX, blocks(n), dim3(kBlock), k_vface<R>, n, lam, v, v0p, v0n, v1p, v1n, make_coef<R>(c).rspi);
}

}  // namespace mhd
