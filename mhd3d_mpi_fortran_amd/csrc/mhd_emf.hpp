// Edge EMF (get_eijk_LFM, mhd3d3.f90:1754-1856) as a marching kernel (the
// binary64 WENO reconstructions: mhd_emf_weno.hpp).
//
// Lanes run along x (every tap a coalesced load); each thread walks T edges
// along a transverse axis and keeps the corner-velocity footprint of the
// current edge in a register window, so one step loads a single new
// stencil row of the window instead of the whole 2-D footprint.  The
// arithmetic per edge is exactly that of get_vav_center2corner
// (mhd3d3.f90:1858-2116): same interpolations, limiters and selection in
// the same order, so the binary64 result is bit-identical to the
// reference's.
//
//   K=1  ei: edge along x, corner plane (d1,d2)=(y,z), march along z (= d2)
//   K=2  ej: edge along y, corner plane (d1,d2)=(z,x), march along z (= d1)
//   K=3  ek: edge along z, corner plane (d1,d2)=(x,y), march along y (= d2)
#pragma once
#include "mhd_kernels.hpp"

namespace mhd {

// stencil footprint of the corner velocity per method: offsets LO..LO+N-1
// along both corner axes
template <int M>
struct VavFoot;
template <>
struct VavFoot<TVD> {
    static constexpr int N = 4, LO = -2;
};
template <>
struct VavFoot<TVD_FULL> : VavFoot<TVD> {};
template <>
struct VavFoot<WENO5> {
    static constexpr int N = 6, LO = -3;
};
template <>
struct VavFoot<MPWENO5> {
    static constexpr int N = 6, LO = -3;
};

// register window w[a][b]: a = offset along the march axis, b = along the
// other corner axis, both LO..LO+N-1 relative to the current edge's base cell
template <typename R, int M, bool MARCH_D1, bool UNIT = false>
struct VavWin {
    static constexpr int N = VavFoot<M>::N, LO = VavFoot<M>::LO;
    R w[N][N];
    // value at offset o1 along d1 and o2 along d2
    __device__ __forceinline__ R cv(int o1, int o2) const { return MARCH_D1 ? w[o1 - LO][o2 - LO] : w[o2 - LO][o1 - LO]; }

    // ob, osm, oso: byte offset of the base cell and byte strides along the
    // march and the other axis (32-bit: every array stays below 2^32 bytes);
    // UNIT: the other axis is x, each row of the window is contiguous and
    // loads as wide vectors from one address
    template <typename TI>
    __device__ __forceinline__ void row(const TI* __restrict__ lv, unsigned orow, unsigned oso, R* out) {
        if constexpr (UNIT) {
            const TI* p = reinterpret_cast<const TI*>(reinterpret_cast<const char*>(lv) + orow);
#pragma unroll
            for (int q = 0; q < N; ++q) out[q] = R(p[q + LO]);
        } else {
            // the column offsets are uniform: they go into each load's
            // scalar base, so a row needs one offset register, not N
            const char* b = reinterpret_cast<const char*>(lv);
#pragma unroll
            for (int q = 0; q < N; ++q)
                out[q] = R(load_at(reinterpret_cast<const TI*>(b + (ptrdiff_t)(q + LO) * (ptrdiff_t)oso), orow));
        }
    }
    template <typename TI>
    __device__ __forceinline__ void load(const TI* __restrict__ lv, unsigned ob, unsigned osm, unsigned oso) {
#pragma unroll
        for (int a = 0; a < N; ++a) row(lv, ob + (unsigned)(a + LO) * osm, oso, w[a]);
    }
    // advance one cell along the march axis (ob is the new base cell)
    template <typename TI>
    __device__ __forceinline__ void shift(const TI* __restrict__ lv, unsigned ob, unsigned osm, unsigned oso) {
#pragma unroll
        for (int a = 0; a < N - 1; ++a)
#pragma unroll
            for (int q = 0; q < N; ++q) w[a][q] = w[a + 1][q];
        row(lv, ob + (unsigned)(N - 1 + LO) * osm, oso, w[N - 1]);
    }
    // advance one cell with a row loaded beforehand
    __device__ __forceinline__ void shift_in(const R* nxt) {
#pragma unroll
        for (int a = 0; a < N - 1; ++a)
#pragma unroll
            for (int q = 0; q < N; ++q) w[a][q] = w[a + 1][q];
#pragma unroll
        for (int q = 0; q < N; ++q) w[N - 1][q] = nxt[q];
    }
};

// corner velocity of one edge from its window (mhd3d3.f90:1858-2116), TVD and
// WENO.  (g holds nothing: without it in the marching loop the compiler writes
// 2x as x+x in places of the fp32 MPWENO5 limiter, which then contract
// differently, and the results are to stay what they are.)
template <typename R, int M, bool MD1, bool U>
__device__ __forceinline__ R vav_win(const VavWin<R, M, MD1, U>& W, const Coef<R>& c, const R* g = nullptr) {
    R v00_0, v10_0, v01_0, v11_0, v00_1, v01_1, v10_1, v11_1;
    if constexpr (scheme(M) == TVD) {
        const R vi = (W.cv(-1, -1) + W.cv(0, -1) + W.cv(0, 0) + W.cv(-1, 0)) / R(4);
        constexpr bool FULL = M == TVD_FULL;
        tvd<R, FULL>(W.cv(-2, 0), W.cv(-1, 0), W.cv(0, 0), W.cv(1, 0), vi, c.eps, v00_0, v10_0);
        tvd<R, FULL>(W.cv(0, -2), W.cv(0, -1), W.cv(0, 0), W.cv(0, 1), vi, c.eps, v00_1, v01_1);
        v10_1 = v00_1;
        v11_1 = v01_1;
        v01_0 = v00_0;
        v11_0 = v10_0;
    } else {
        using S = Stencil<R, M>;
        R L[6], Q[6], s[6];
#pragma unroll
        for (int mb = 0; mb < 6; ++mb) {
#pragma unroll
            for (int ma = 0; ma < 6; ++ma) s[ma] = W.cv(ma - 3, mb - 3);
            S::run(s, c, L[mb], Q[mb]);
        }
        S::run(L, c, v00_1, v01_1);
        S::run(Q, c, v10_1, v11_1);
#pragma unroll
        for (int mb = 0; mb < 6; ++mb) {
#pragma unroll
            for (int ma = 0; ma < 6; ++ma) s[ma] = W.cv(mb - 3, ma - 3);
            S::run(s, c, L[mb], Q[mb]);
        }
        S::run(L, c, v00_0, v01_0);
        S::run(Q, c, v10_0, v11_0);
    }
    R d00 = sgn1(fabs(W.cv(-2, -1) - W.cv(-1, -1)) - fabs(W.cv(-1, -2) - W.cv(-1, -1)));
    R d10 = sgn1(fabs(W.cv(1, -1) - W.cv(0, -1)) - fabs(W.cv(0, -2) - W.cv(0, -1)));
    R d01 = sgn1(fabs(W.cv(-2, 0) - W.cv(-1, 0)) - fabs(W.cv(-1, 1) - W.cv(-1, 0)));
    R d11 = sgn1(fabs(W.cv(1, 0) - W.cv(0, 0)) - fabs(W.cv(0, 1) - W.cv(0, 0)));
    R v00 = (R(1) + d00) / R(2) * v00_0 + (R(1) - d00) / R(2) * v00_1;
    R v10 = (R(1) + d10) / R(2) * v10_0 + (R(1) - d10) / R(2) * v10_1;
    R v01 = (R(1) + d01) / R(2) * v01_0 + (R(1) - d01) / R(2) * v01_1;
    R v11 = (R(1) + d11) / R(2) * v11_0 + (R(1) - d11) / R(2) * v11_1;
    return R(.25) * (v00 + v01 + v10 + v11);
}

// Every thread marches exactly T edges (the launcher keeps T <= the march
// axis' edge count, and the last run of a line starts early, overlapping its
// predecessor, whose edges it recomputes but does not store).  With no run-length test the unrolled
// steps form one block and the windows and carried values rename from step
// to step instead of being copied at every conditional join.  A fence ends
// each step: the step's result is pinned there (an empty asm that takes it
// in a register), so the compiler can neither sink the step's arithmetic to
// the result's later use nor hoist the next steps' loads above it -- either
// would keep the whole run's loaded footprint live at once (hundreds of
// registers).
template <typename R>
__device__ __forceinline__ void step_fence(R& v) {
    asm volatile("" : "+v"(v));
    __builtin_amdgcn_sched_barrier(0);
}

// corner velocities of T consecutive edges along the march axis (TVD and WENO)
template <typename R, int M, bool MD1, bool UNIT, int T, typename TI>
__device__ __forceinline__ void vav_march(const TI* __restrict__ lv, ptrdiff_t b, ptrdiff_t s1, ptrdiff_t s2,
                                          const Coef<R>& c, R (&out)[T]) {
    const ptrdiff_t sm = MD1 ? s1 : s2, so = MD1 ? s2 : s1;
    constexpr unsigned E = sizeof(TI);
    unsigned ob = (unsigned)b * E;
    const unsigned osm = (unsigned)sm * E, oso = (unsigned)so * E;
    VavWin<R, M, MD1, UNIT> W;
    W.load(lv, ob, osm, oso);
    R g[8];
    // fp32 UNIT windows (the fewest registers): the next step's row is
    // loaded before the current corner velocity is computed, so its latency
    // hides behind that arithmetic (binary64 windows would lose a wave per
    // SIMD to the extra row)
    constexpr int N = VavWin<R, M, MD1, UNIT>::N, LO = VavWin<R, M, MD1, UNIT>::LO;
    constexpr bool PRE = UNIT && sizeof(R) == 4;
    auto step = [&](int s) {
        R nxt[N];
        if constexpr (PRE) {
            if (s + 1 < T) W.row(lv, ob + osm + (unsigned)(N - 1 + LO) * osm, oso, nxt);
        }
        out[s] = vav_win<R, M>(W, c, g);
        if (s + 1 < T) {
            ob += osm;
            if constexpr (PRE) W.shift_in(nxt);
            else W.shift(lv, ob, osm, oso);
        }
        step_fence(out[s]);
    };
    // MPWENO5 runs the steps as a loop: unrolled they need more registers than
    // it saves
    if constexpr (M == MPWENO5) {
#pragma unroll 1
        for (int s = 0; s < T; ++s) step(s);
    } else {
#pragma unroll
        for (int s = 0; s < T; ++s) step(s);
    }
}

// One PDM2 line through the corner (mhd3d3.f90:1142-1166), held as the raw
// differences of its 4-point stencil (fm2, fm1, f0, fp1): rm = fm1 - fm2,
// r0 = f0 - fm1, rp = fp1 - f0, their slopes pdmb*r and the slopes' signs.
// All of PDM2 but the clamp of the interpolated value depends on these
// alone, so a line that the march slides along itself by one cell keeps two
// of its differences with their slopes and signs, and a line across the
// march is handed on whole to the next edge.  The same operations on the
// same values as PDM2, so the results are bit-identical.
template <typename R>
struct PdmLine {
    R rm, r0, rp, dm, d0, dp, sm, s0, sp, lo, hi;
    __device__ __forceinline__ void set(R fm2, R fm1, R f0, R fp1, R pdmb) {
        hi = dmax(fm1, f0);
        lo = dmin(fm1, f0);
        rm = fm1 - fm2;
        r0 = f0 - fm1;
        rp = fp1 - f0;
        dm = pdmb * rm;
        d0 = pdmb * r0;
        dp = pdmb * rp;
        sm = sgn1(dm);
        s0 = sgn1(d0);
        sp = sgn1(dp);
    }
    // the stencil moved one cell along the line; fm1, f0, fp1 are the new one's
    __device__ __forceinline__ void slide(R fm1, R f0, R fp1, R pdmb) {
        hi = dmax(fm1, f0);
        lo = dmin(fm1, f0);
        rm = r0;
        r0 = rp;
        rp = fp1 - f0;
        dm = d0;
        d0 = dp;
        dp = pdmb * rp;
        sm = s0;
        s0 = sp;
        sp = sgn1(dp);
    }
    // PDM2's left and right states about the interpolated value fi
    __device__ __forceinline__ void finish(R fm1, R f0, R fi, R& fl, R& fr) const {
        const R fii = dmax(lo, dmin(fi, hi));
        const R qm = fabs(sm + s0), qp = fabs(s0 + sp);
        const R dfl = fii - fm1, dfr = f0 - fii;
        fl = fii - s0 * dmax(R(0), fabs(dfl) - qm * fabs(dm));
        fr = fii + s0 * dmax(R(0), fabs(dfr) - qp * fabs(dp));
    }
};

// PDM corner velocities of T consecutive edges (get_vav_center2corner,
// mhd3d3.f90:1858-2116) marching along axis a, the other corner axis being b:
// (a, b) = (d2, d1) for K=1 and K=3, (d1, d2) for K=2.
//   * g[m]: the 8-point interpolation along b of the footprint row at march
//     offset m-4; vi = interp8(g).  A step adds one row, so seven of the eight
//     carry over.  Along d1 first, then d2 is interp2_pdm's order; for K=2
//     (a = d1) that order holds only in fp32, which interpolates along d2 first
//     (the same tensor-product value up to rounding); binary64 K=2 shares its
//     columns between lanes instead (pdm_columns, vav_march_cols).
//   * the four PDM2 lines: two across the march (along b, at a = -1 and 0) and
//     two along it (along a, at b = -1 and 0); a step hands the a = 0 line on
//     as the next a = -1 one and slides the other two (PdmLine).
//   * the corner selection (mhd3d3.f90:2064-2099) compares |rm| and |rp| of
//     the lines: |a - b| = |b - a| exactly.
// Only the 4x5 core of the footprint (b = -2..1, a = -1..3) stays in registers;
// the new row's other taps serve only its interpolation.
template <typename R, bool MD1, bool UNIT, int T, typename TI>
__device__ __forceinline__ void vav_march_pdm(const TI* __restrict__ lv, const Buf<TI>& bv, unsigned ob,
                                              unsigned osm, unsigned oso, const Coef<R>& c,
                                              R (&out)[T]) {
    constexpr unsigned E = sizeof(TI);
    // the 8 taps along b (offsets -4..3) of the row at byte offset orow
    auto row = [&](unsigned orow, R* v) {
        if constexpr (UNIT) {
            const TI* p = reinterpret_cast<const TI*>(reinterpret_cast<const char*>(lv) + orow);
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = R(p[q - 4]);
        } else {
            const unsigned o0 = orow - 4u * oso;
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = R(bv.at(o0, (unsigned)q * oso));
        }
    };
    const R pdmb = c.pdmb;
    R g[8], V[5][4];  // V[a+1][b+2]
    PdmLine<R> C0, C1, L0, L1;
    {
        R w[8][8];  // w[a+4][b+4]
#pragma unroll
        for (int a = 0; a < 8; ++a) row(ob + (unsigned)(a - 4) * osm, w[a]);
#pragma unroll
        for (int a = 0; a < 8; ++a) g[a] = interp8(w[a]);
#pragma unroll
        for (int a = 0; a < 5; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) V[a][b] = w[a + 3][b + 2];
        C0.set(w[3][2], w[3][3], w[3][4], w[3][5], pdmb);
        C1.set(w[4][2], w[4][3], w[4][4], w[4][5], pdmb);
        L0.set(w[2][3], w[3][3], w[4][3], w[5][3], pdmb);
        L1.set(w[2][4], w[3][4], w[4][4], w[5][4], pdmb);
    }
    // fp32: the next row is loaded before the current corner velocity is
    // computed, so its latency hides behind that arithmetic
    constexpr bool PRE = sizeof(R) == 4;
#pragma unroll
    for (int s = 0; s < T; ++s) {
        {
            R nxt[8];
            if constexpr (PRE) {
                if (s + 1 < T) row(ob + (unsigned)(s + 4) * osm, nxt);
            }
            const R vi = interp8(g);
            // X(q): PDM2 along d1 at d2 offset q; Y(p): along d2 at d1 offset p
            const PdmLine<R>& Xm = MD1 ? L0 : C0;
            const PdmLine<R>& X0 = MD1 ? L1 : C1;
            const PdmLine<R>& Ym = MD1 ? C0 : L0;
            const PdmLine<R>& Y0 = MD1 ? C1 : L1;
            // corner values cv(o1, o2) at d1 offset o1, d2 offset o2 (-1, 0)
            auto cv = [&](int o1, int o2) { return MD1 ? V[o1 + 1][o2 + 2] : V[o2 + 1][o1 + 2]; };
            R v00_0, v10_0, v00_1, v01_1, v10_1, v11_1, v01_0, v11_0;
            Xm.finish(cv(-1, -1), cv(0, -1), vi, v00_0, v10_0);
            Ym.finish(cv(-1, -1), cv(-1, 0), vi, v00_1, v01_1);
            Y0.finish(cv(0, -1), cv(0, 0), vi, v10_1, v11_1);
            X0.finish(cv(-1, 0), cv(0, 0), vi, v01_0, v11_0);
            const R d00 = sgn1(fabs(Xm.rm) - fabs(Ym.rm));
            const R d10 = sgn1(fabs(Xm.rp) - fabs(Y0.rm));
            const R d01 = sgn1(fabs(X0.rm) - fabs(Ym.rp));
            const R d11 = sgn1(fabs(X0.rp) - fabs(Y0.rp));
            const R v00 = pick(d00, v00_0, v00_1);
            const R v10 = pick(d10, v10_0, v10_1);
            const R v01 = pick(d01, v01_0, v01_1);
            const R v11 = pick(d11, v11_0, v11_1);
            out[s] = R(.25) * (v00 + v01 + v10 + v11);
            if (s + 1 < T) {
                if constexpr (!PRE) row(ob + (unsigned)(s + 4) * osm, nxt);
                // slide the footprint one cell along a
#pragma unroll
                for (int m = 0; m < 7; ++m) g[m] = g[m + 1];
                g[7] = interp8(nxt);
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int b = 0; b < 4; ++b) V[a][b] = V[a + 1][b];
#pragma unroll
                for (int b = 0; b < 4; ++b) V[4][b] = nxt[b + 2];
                C0 = C1;
                C1.set(V[1][0], V[1][1], V[1][2], V[1][3], pdmb);
                L0.slide(V[0][1], V[1][1], V[2][1], pdmb);
                L1.slide(V[0][2], V[1][2], V[2][2], pdmb);
            }
        }
        step_fence(out[s]);
    }
}

// Binary64 ej (K=2, corner plane (z, x), march along z).  interp2_pdm's order
// interpolates along z first: the eight columns x-4..x+3 of the footprint at every
// edge.  A column is the same for the eight edges along x that it serves, and
// lanes run along x, so each lane interpolates its own column (pdm_columns: one
// load and one interpolation per step and velocity) and the lanes exchange the
// results through LDS.  Lanes stand for columns here: a row of ii edges has
// ii + 7, and a workgroup's outer 4 + 3 only interpolate.  An 8x8 window per lane
// interpolated eight columns per step and needed 206 registers: the three
// directions took 1.49 ms at 256^3, 1.22 ms with this; a 64^3 step 228 and 208 us.
// Bound: VALU issue, at 3 wavefronts per SIMD (160 registers).
constexpr int kColEdges = kBlock - 7;
template <typename R, int T, typename TI>
__device__ __forceinline__ void pdm_columns(const Buf<TI>& bv, unsigned ob, unsigned osm, R (*cols)[kBlock]) {
    const unsigned o0 = ob - 4u * osm;
    R w[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) w[m] = R(bv.at(o0, (unsigned)m * osm));
#pragma unroll
    for (int s = 0; s < T; ++s) {
        cols[s][threadIdx.x] = interp8(w);
        if (s + 1 < T) {
#pragma unroll
            for (int m = 0; m < 7; ++m) w[m] = w[m + 1];
            w[7] = R(bv.at(o0, (unsigned)(s + 8) * osm));
        }
    }
}

// the march's corner velocities from the lanes' columns: V[a+2][b+2] holds the
// footprint's core, a = -2..1 along z, b = -2..1 along x (see vav_march_pdm)
template <typename R, int T, typename TI>
__device__ __forceinline__ void vav_march_cols(const TI* __restrict__ lv, unsigned ob, unsigned osm, const Coef<R>& c,
                                               const R (*cols)[kBlock], R (&out)[T]) {
    auto row = [&](unsigned orow, R* v) {
        const TI* p = reinterpret_cast<const TI*>(reinterpret_cast<const char*>(lv) + orow);
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = R(p[q - 2]);
    };
    const R pdmb = c.pdmb;
    R V[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a) row(ob + (unsigned)(a - 2) * osm, V[a]);
    PdmLine<R> C0, C1, L0, L1;
    C0.set(V[1][0], V[1][1], V[1][2], V[1][3], pdmb);
    C1.set(V[2][0], V[2][1], V[2][2], V[2][3], pdmb);
    L0.set(V[0][1], V[1][1], V[2][1], V[3][1], pdmb);
    L1.set(V[0][2], V[1][2], V[2][2], V[3][2], pdmb);
#pragma unroll
    for (int s = 0; s < T; ++s) {
        R g[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) g[m] = cols[s][(int)threadIdx.x + m - 4];
        const R vi = interp8(g);
        auto cv = [&](int o1, int o2) { return V[o1 + 2][o2 + 2]; };
        R v00_0, v10_0, v00_1, v01_1, v10_1, v11_1, v01_0, v11_0;
        L0.finish(cv(-1, -1), cv(0, -1), vi, v00_0, v10_0);
        C0.finish(cv(-1, -1), cv(-1, 0), vi, v00_1, v01_1);
        C1.finish(cv(0, -1), cv(0, 0), vi, v10_1, v11_1);
        L1.finish(cv(-1, 0), cv(0, 0), vi, v01_0, v11_0);
        const R v00 = pick(sgn1(fabs(L0.rm) - fabs(C0.rm)), v00_0, v00_1);
        const R v10 = pick(sgn1(fabs(L0.rp) - fabs(C1.rm)), v10_0, v10_1);
        const R v01 = pick(sgn1(fabs(L1.rm) - fabs(C0.rp)), v01_0, v01_1);
        const R v11 = pick(sgn1(fabs(L1.rp) - fabs(C1.rp)), v11_0, v11_1);
        out[s] = R(.25) * (v00 + v01 + v10 + v11);
        if (s + 1 < T) {
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) V[a][b] = V[a + 1][b];
            row(ob + (unsigned)(s + 2) * osm, V[3]);
            C0 = C1;
            C1.set(V[2][0], V[2][1], V[2][2], V[2][3], pdmb);
            L0.slide(V[1][1], V[2][1], V[3][1], pdmb);
            L1.slide(V[1][2], V[2][2], V[3][2], pdmb);
        }
        step_fence(out[s]);
    }
}

// workgroups of the ei march: 64 x-lanes by 4 consecutive y edges, one run
// of T edges along z
template <int T>
__host__ __device__ __forceinline__ unsigned emf_tiles(int nx0, int ny0, int nz0) {
    return (unsigned)((nx0 + kTileX - 1) / kTileX) * ((ny0 + 1 + kTileN - 1) / kTileN) * ((nz0 + 1 + T - 1) / T);
}

template <typename T>
struct EmfIn {  // one edge direction's inputs
    const T *v1, *v2, *b1, *b2, *vf;
};

template <int K>
struct EmfGeom {
    // K=1 ei (nx0, ny0+1, nz0+1): other axis y, march z
    // K=2 ej (nx0+1, ny0, nz0+1): other axis y, march z
    // K=3 ek (nx0+1, ny0+1, nz0): other axis z, march y
    static constexpr bool MD1 = (K == 2);
};

// threads = ii * no * ceil(nm / T) (K=2, 3) or emf_tiles workgroups (K=1);
// lanes run along x.  Binary64 PDM's ej: threads = (ii + 7) * no * ceil(nm / T)
// columns, kColEdges of them a workgroup's own
template <typename R, int M, int K, int T, typename TI, typename TF>
__global__ void __launch_bounds__(kBlock) k_emf_march(Dims d, Coef<R> c, EmfIn<TI> in, R ef,
                                                     const double* __restrict__ efa, TF* __restrict__ e,
                                                     long nthreads) {
#define EMF_BLOCK() xcd_block()
#include "mhd_emf_march.inc"
#undef EMF_BLOCK
}

// the same as part of a launch of several directions (k_stencils): workgroup
// `part_block` of the direction
template <typename R, int M, int K, int T, typename TI, typename TF>
__device__ __forceinline__ void emf_block(Dims d, Coef<R> c, EmfIn<TI> in, R ef, const double* __restrict__ efa,
                                          TF* __restrict__ e, long nthreads, unsigned part_block) {
#define EMF_BLOCK() part_block
#include "mhd_emf_march.inc"
#undef EMF_BLOCK
}

}  // namespace mhd
