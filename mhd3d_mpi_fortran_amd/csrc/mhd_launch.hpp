// Context object and launch plumbing shared by the library's translation
// units (binary64 stencil kernels, fp32 stencil kernels, surrogate).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "../../include/mhd_gpu.h"
#include "mhd_kernels.hpp"

namespace mhd {
// stencil inputs of one state: cell primitives, cell B, vf, face B and,
// with a metric, the face-normal velocities w_d = v . n_d
template <typename T>
struct Src {
    const T *rho, *vx, *vy, *vz, *p, *bx, *by, *bz, *vf, *bi, *bj, *bk;
    const T* w[3];
};

// affine metric x_phys = A x_comp (mhd_set_metric); on = false is the
// reference's tensor-product grid, for which every factor below is exactly 1.
// mode 2: the general metric of GMet (mhd_set_metric_nodes)
struct Metric {
    bool on = false;
    int mode = 0;  // 0 tensor product, 1 affine, 2 general
    double A[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};  // row-major
    double n[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};  // unit face normals per computational axis
    double g[3] = {1, 1, 1};    // |C e_d| / det A: flux divergence factor (update, CFL)
    double ct[3] = {1, 1, 1};   // 1 / |C e_d|: constrained-transport factor of face family d
    double ef[3] = {1, 1, 1};   // |C e_a||C e_b| / det A: EMF factor of edges along d
    double M[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};  // A diag(g): face-average B -> cell B
};

// get_eijk_Yee's twelve split fields e<a><s1><s2> of edge direction a (x, y,
// z), s1 the side of the first transverse velocity's moments, s2 the
// second's: e_a = B_b v_b0(s1) v_c1(s2) - B_c v_b1(s1) v_c0(s2), (a, b, c)
// cyclic; index 4*a + YEE_<s1><s2>
enum { YEE_PP = 0, YEE_NP = 1, YEE_PN = 2, YEE_NN = 3 };
}  // namespace mhd

// device scalars: scal[SC_TAU] = tau, scal[SC_TAU0] = tau0, scal[SC_DTCFL] = get_dt result,
// scal[SC_DIVB] = -max |div B| of the last mhd_divb_max
enum { SC_TAU = 0, SC_TAU0 = 1, SC_DTCFL = 2, SC_DIVB = 3 };

struct SurrogateState;

// EMF launches whose long-run grid would leave the chip short of waves
// (fewer than ~8 per SIMD: 256 CUs x 4 SIMDs x 8 waves x 64 lanes) take
// short runs
constexpr long kEmfFillThreads = 256L * 4 * 8 * 64;
// blocks with at least this many owned cells run a stage on two streams by
// default (mhd_set_stage_overlap), smaller ones its stencils in one launch
// (k_stencils)
constexpr long kOverlapCells = 1L << 21;
// Binary64 Runge-Kutta blocks keep the one launch up to the size to which it is the
// faster one by measurement (a launch each on two streams in brackets):
//   PDM   128^3 1393 us a step (1585), 160^3 2889 (3183), 200^3 5875 (6343), 256^3
//         11.23 ms (11.35), 300^3 18.52 (18.57), 320^3 21.78 (21.84)
//   TVD   128^3 1265 us (1299), 144^3 1961 (1997), 160^3 2588 (2591), 200^3 5183
//         (5186), 300^3 16.87 ms (16.63): from 200^3 on the launches of their own
//         take runs of 16 edges, the one launch runs of 2
//   WENO5 and MPWENO5 (whose EMF has launches of its own either way) 128^3 3240 and
//         4522 us (3235, 4555), 200^3 12.98 and 18.16 ms (12.96, 18.17), 256^3 26.03
//         and 36.57 (26.13, 36.69), 300^3 43.32 and 58.90 (43.88, 58.96); long thin
//         blocks of 3 M cells within 1 % either way
// Eight cells along x: PDM 8 x 600 x 600 6.74 ms (8.14), 8 x 1800 x 1800 62.4 (64.8);
// TVD 8 x 600 x 600 5.72 (5.62).  (Binary32 EMFs round with their runs' length, so
// mixed blocks keep theirs.)
constexpr long kMergeCells64 = 1L << 25, kMergeCellsTvd64 = 1L << 22;
// Whether the rows of a binary64 Adams-Bashforth block fill enough of the sweep's
// 64-lane tiles (mhd_sweep.hpp; lanes past a row's end form a flux and drop it).
// Flux and update of their own in brackets.  PDM from 1/2 on: 33 x 260 x 260 1264 us
// (1268; a narrower one takes the one launch, merge_cells: 24 x 320 x 320 1454 for the
// sweep's 1654); TVD from 3/8 on: 24 x 320 x 320 1264 us (1280), 20 x 400 x 400 1795
// (1797), 16 x 400 x 400 1697 (1679), 8 x 400 x 800 2835 (2726); WENO5 and MPWENO5 from
// 3/4 on: 100 x 160 x 160 2145 and 2984 us (2171, 3022), 48 x 220 x 220 2046 and 2856
// (2046, 2842), 65 x 190 x 190 2349 and 3291 (2246, 3184).
inline bool sweep_fills(const mhd_params& p) {
    const int lanes = (p.nx0 + mhd::kTileX - 1) / mhd::kTileX * mhd::kTileX;
    const int eighths = p.reconop == mhd::PDM ? 4 : (p.reconop == mhd::TVD ? 3 : 6);
    return 8 * p.nx0 >= eighths * lanes;
}
// the bound for a block of these parameters.  Adams-Bashforth blocks past it have the
// sweep; PDM ones too narrow for that keep the one launch: 16 x 400 x 400 1941 us
// (sweep 2285, a launch each 2269), 8 x 400 x 800 3213 (3961, 3842), 16 x 1400 x 1400
// 24.5 ms (25.2, 25.5)
inline long merge_cells(const mhd_params& p) {
    if (p.precision == MHD_MIXED) return kOverlapCells;
    if (p.stepop == 1) return p.reconop == mhd::PDM && !sweep_fills(p) ? kMergeCells64 : kOverlapCells;
    return p.reconop == mhd::TVD ? kMergeCellsTvd64 : kMergeCells64;
}

// scratch of the binary64 WENO EMF (mhd_emf_weno.hpp): 18 arrays over a
// slab of whole planes, as many as kWenoScratch bytes hold (it should stay in
// the last-level cache), at least kWenoHalo more than 16 planes of edges -- or
// than one, where the GPU's memory does not hold that (environment
// MHD_WENO_PLANES sets the planes at mhd_create)
constexpr int kWenoHalo = 5;
constexpr size_t kWenoScratch = size_t(160) << 20;

struct mhd_ctx {
    mhd_params p{};
    mhd::Dims d{};
    hipStream_t s = nullptr;
    // second stream: a stage's edge EMF and CT run on it beside the face flux
    // and the cell update (see stage_overlapped).  cur: the stream launch()
    // targets (null = s)
    hipStream_t s2 = nullptr, cur = nullptr;
    hipEvent_t ev_fork = nullptr, ev_emf = nullptr, ev_join = nullptr;
    bool merged = false;   // one launch for a stage's stencils (merge_cells)
    bool overlap = true;   // false: one stream, kernels in the reference's order
    bool fused = false;    // mixed Adams-Bashforth PDM steps: fused face flux + update (mhd_set_fusion)
    char* arena = nullptr;
    size_t arena_bytes = 0;
    bool have_geometry = false;
    long ncell = 0, nbi = 0, nbj = 0, nbk = 0, ninterior = 0, ndtpart = 0, nbxyz = 0, nmax = 0;
    long nf[3] = {0, 0, 0}, ne[3] = {0, 0, 0};
    // EMF launches with fewer long-run threads than this take short runs
    // (environment MHD_EMF_FILL_THREADS overrides it at mhd_create)
    long emf_fill = 0;
    // state (reference layout)
    double *rho = nullptr, *vx = nullptr, *vy = nullptr, *vz = nullptr, *pr = nullptr;
    double *bx = nullptr, *by = nullptr, *bz = nullptr, *vf = nullptr;
    double *bi = nullptr, *bj = nullptr, *bk = nullptr;
    double *dx = nullptr, *dy = nullptr, *dz = nullptr;
    // RK advance_previous
    double *rhop = nullptr, *mxp = nullptr, *myp = nullptr, *mzp = nullptr, *engp = nullptr;
    double *bip = nullptr, *bjp = nullptr, *bkp = nullptr;
    // AB: previous and next state (rotated with the current one each step),
    // extrapolated state (binary64 mode; mixed mode extrapolates into sh)
    // order: rho vx vy vz p bx by bz bi bj bk
    double* xp[11] = {};
    double* xn[11] = {};
    double* xh[11] = {};
    double* vfh = nullptr;
    // fp32 stencil inputs (mixed precision): rho vx vy vz p bx by bz vf bi bj bk
    float* sh[12] = {};
    bool dt_fresh = false;   // dtpart holds the CFL partials of the current state
    long ndt_valid = 0;      // ... that many of them
    bool spacing_mid = false;  // the update's spacings lie within 2^-400 .. 2^400
    bool ghost_twins = false;  // every ghost cell repeats an owned cell (periodic axes, equal ghost spacings)
    // bx,by,bz not stored for the current state (mixed AB steps, all but a call's
    // last stage of mixed RK ones, uploads, advances)
    bool cellb_stale = false;
    bool pred_valid = false;   // the extrapolated state of mhd_predict_ab is held (xh / fp32 copies)
    // per-stage products (binary64, or fp32 in mixed precision)
    void* flux[3] = {nullptr, nullptr, nullptr};
    void* emf[3] = {nullptr, nullptr, nullptr};
    void* weno = nullptr;    // binary64 WENO contexts: the EMF's reconstructed lines, weno_planes planes of 18 arrays
    int weno_planes = 0;
    double* dtpart = nullptr;
    double* divpart = nullptr;   // per-workgroup partials of the div B monitor (apart from the CFL ones)
    double* scal = nullptr;
    int* flags = nullptr;
    double* hscal = nullptr;   // pinned: tau and the CFL minimum of the last step of a call (k_dt_final)
    double tau0_host = 0.;
    hipError_t launch_error = hipSuccess;
    // kernel timing
    bool prof = false;
    unsigned prof_mask = ~0u;   // classes timed while prof is set
    struct Rec {
        int kclass;
        hipEvent_t a, b;
    };
    std::vector<Rec> evs;
    std::vector<hipEvent_t> evpool;
    double prof_ms[MHD_K_NCLASS] = {};
    int prof_n[MHD_K_NCLASS] = {};
    // metric (mhd_set_metric): spacing divided by g_d for the update and the
    // CFL, face-normal velocities (binary64 current / extrapolated state, fp32)
    mhd::Metric met;
    std::vector<double> hdx, hdy, hdz;
    double *dxm = nullptr, *dym = nullptr, *dzm = nullptr;
    char* metbuf = nullptr;
    char* gmetbuf = nullptr;
    mhd::GMet gm{};
    double* w64[3] = {};
    double* wh64[3] = {};
    float* w32[3] = {};
    SurrogateState* sur = nullptr;
    float sur_theta = 0.25f;   // smoothness threshold of the learned reconstruction
    bool sur_stats = false;    // count faces / fallbacks
};

inline dim3 blocks(long n) { return dim3((unsigned)((n + mhd::kBlock - 1) / mhd::kBlock)); }

inline hipEvent_t ev_get(mhd_ctx* c) {
    if (!c->evpool.empty()) {
        hipEvent_t e = c->evpool.back();
        c->evpool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
}

template <typename... KArgs, typename... Args>
inline void launch(mhd_ctx* c, int kclass, dim3 g, dim3 b, void (*k)(KArgs...), Args... args) {
    if (g.x == 0 || g.y == 0) return;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    const bool timed = c->prof && ((c->prof_mask >> kclass) & 1u);
    hipStream_t st = c->cur ? c->cur : c->s;
    auto note = [c](hipError_t err) {
        if (err != hipSuccess && c->launch_error == hipSuccess) c->launch_error = err;
    };
    if (timed) {
        e0 = ev_get(c);
        e1 = ev_get(c);
        if (!e0 || !e1) note(hipErrorOutOfMemory);
        else note(hipEventRecord(e0, st));
    }
    hipLaunchKernelGGL(k, g, b, 0, st, static_cast<KArgs>(args)...);
    note(hipGetLastError());
    if (timed && e0 && e1) {
        note(hipEventRecord(e1, st));
        c->evs.push_back({kclass, e0, e1});
    } else {
        if (e0) c->evpool.push_back(e0);
        if (e1) c->evpool.push_back(e1);
    }
}

// the binary64 reconstruction of a context (mhd::Recon)
inline bool full_division(const mhd_params& p) {  // needed by the limiters, for its eps
    return p.reconop != mhd::PDM && mhd::Coef<double>::full(p.eps);
}
inline int recon_code(const mhd_ctx* c) { return full_division(c->p) ? c->p.reconop + 3 : c->p.reconop; }

template <typename R>
inline mhd::Coef<R> make_coef(const mhd_ctx* c) {
    mhd::Coef<R> k;
    const double pi = 3.141592653589793238462643383279502884;  // binary64 of 4*atan(1)
    k.gam = R(c->p.gam);
    k.gm1 = R(c->p.gam - 1.);
    k.cfl = R(c->p.cfl);
    k.pdmb = R(c->p.pdmb);
    k.eps = R(c->p.eps);
    k.alpha = R(c->p.alpha);
    k.beta = R(c->p.beta);
    k.rspi = R(std::sqrt(pi));
    if constexpr (sizeof(R) == 8) k.set_weno();
    return k;
}

template <typename R>
inline mhd::Normals<R> make_normals(const mhd_ctx* c) {
    mhd::Normals<R> k;
    for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) k.n[a][b] = R(c->met.n[a][b]);
    return k;
}

// per-precision stencil launchers (separate translation units)
// z: the z faces too (false: a sweep forms them, mhd_sweep.hpp)
void launch_flux_fp64(mhd_ctx* c, mhd::Src<double> s, bool z = true);
void launch_emf_fp64(mhd_ctx* c, mhd::Src<double> s);
void launch_recon(mhd_ctx* c, int dir, const double* f, int fn1, int fn2, int lnx, int lny, int lnz, double* fl,
                  double* fr);
void launch_flux_fp32(mhd_ctx* c, mhd::Src<float> s);
// the face fluxes and/or the edge EMFs in one launch (k_stencils)
enum { kStageFlux = 1, kStageEmf = 2 };
void launch_stage_fp64(mhd_ctx* c, mhd::Src<double> s, int what);
void launch_stage_fp32(mhd_ctx* c, mhd::Src<float> s, int what);
void launch_emf_fp32(mhd_ctx* c, mhd::Src<float> s);
void launch_flux_surrogate(mhd_ctx* c, mhd::Src<float> s);
void launch_vface_fp64(mhd_ctx* c, long n, const double* lam, const double* v, double* v0p, double* v0n, double* v1p,
                       double* v1n);
void launch_vface_fp32(mhd_ctx* c, long n, const double* lam, const double* v, double* v0p, double* v0n, double* v1p,
                       double* v1n);
void surrogate_free(mhd_ctx* c);
// get_eijk_Yee's split (12 ghost-inclusive cell arrays, e[4*a + YEE_*]) and
// quadrant sums (mhd_yee.hpp)
void launch_yee_split(mhd_ctx* c, long n, mhd::Prim<double> q, double* const* e);
void launch_yee_sum(mhd_ctx* c, int o1, int o2, int o3, int ax, int n1, int n2, const double* const* e4, double* out);
