// vah_stage.h -- the fused Kurganov-Tadmor Heun stage kernel for gfx950.
//
// One launch performs one Euler stage of the reference's rungeKutta2
// (old_cpu-vah_code/src/FullyDiscreteKurganovTadmorScheme.cpp:761-789) for
// every interior cell:
//   out = in + dt*S  (+= x, y, eta flux differences and axis sources)
//   [stage 2: out = (out + q^n)/2]
//   Newton recovery of (e, p, u) at tau + dt, regulation, and the
//   zero-gradient ghost copies of all outputs (DynamicalVariables.cpp:349-489).
//
// Work decomposition.  A workgroup owns a TX x TY tile of cells in (x, y) and
// marches through kz consecutive eta planes.  Its waves have two roles, each
// with one lane per cell of the tile:
//   face waves   solve each x, y and eta face of the tile once and leave the
//                15-component fluxes (and the axis sources, whose pi gradients
//                are differences of values the face has loaded) in LDS;
//   cell waves   form the source terms of the plane meanwhile, then add the
//                fluxes and finish the cell: recovery, regulator, stores.
// The two halves of a cell's work take about the same time, so they run side
// by side instead of one after the other, with one exchange per plane.  In a
// kernel whose every wave did both, a stage of a lattice that does not fill
// the chip was one long serial chain (28 us at 81x81 and at 261x243), four
// barriers a plane kept its four waves in step, and its register need (250,
// two waves per SIMD) was that of the union of both halves.
// Measured, one step: 81x81 57 -> 20 us, 261x243 56 -> 43 us, 611x587 172 ->
// 153 us, 101x101x30 296 -> 194 us, 97x89x33 in split precision 336 -> 180 us,
// 201x201x101 2.55 -> 2.40 ms; with what came later 18, 37, 136, 171, 167 us, 2.01 ms.
// VAH_FLUX_PER_CELL keeps the reference's work split in a kernel of its own:
// every cell solves both of its faces with its own Newton guess.
// Workgroups are mapped to tiles so that the eight XCDs work through the eta
// chunks together (tile_of_block).
#pragma once

#include "vah_device.h"
#include "vah_face.h"
#include "vah_geometry.h"
#include "vah_source.h"

namespace vah {

// Waves per SIMD the register allocation is sized for: 512 registers shared by
// two leave 256 to each.  At three (168 each) the source terms spill and every
// lattice measured slower (101x101x30: 789 against 1058 us for four steps).
constexpr int kWavesPerSimd = 2;

// a tile shape fits NW waves per role when its cells and both face sets do
template <int TX, int TY, int NW>
constexpr bool tile_fits() {
    return TX * TY <= 64 * NW && (TX + 1) * TY <= 64 * NW && TX * (TY + 1) <= 64 * NW;
}

struct StageParams {
    const double *qin;    // 15-field slab the stage reads
    double *qout;         // 15-field slab it writes
    const double *qn;     // q at tau_n (stage 2 convex combination)
    const double *e_in, *p_in;
    double *e_out, *p_out;
    const double *ucur;   // u used for gradients and face Newton guesses
    const double *uprev;  // u one level back (time derivative)
    double *uout;
    long fs;              // elements between fields of a slab
    int nx, ny, nz;       // interior cells
    int ncx, ncy;         // computational extents (interior + 4)
    long sy, sz;          // strides in y and eta
    int tiles_x, tiles_y, zchunks, kz;
    int nblocks;          // tiles of the lattice (tiles_x * tiles_y * zchunks)
    double t_src, t_rec;  // tau of the sources/fluxes, tau of the recovery
    double dt, dt_inv, etabar, etabar_inv;
    double inv_dx, inv_dy, inv_dz;  // 1/d
    double hx, hy, hz;              // (1/d)/2, the reference's centred-difference factor
    double dt_dx, dt_dy, dt_dz;     // dt * (1/d), the weight of a flux difference
    Eos eos;
    unsigned int *counters;  // [0] NaN cells, [1] recovery fallbacks
    unsigned long long *emax;  // running max of the new e (ordered bits), or null
};

// Workgroup -> tile.  The hardware deals workgroups round-robin over the
// eight XCDs (workgroup b runs on XCD b % 8).  All XCDs work through the eta
// chunks together, each on its own slice of a chunk's tiles: XCD x takes the
// tiles x * slice .. (x + 1) * slice - 1 of chunk 0, then of chunk 1, and so
// on.  The planes in flight are then those of a few neighbouring chunks, one
// band that the memory-side cache can hold, and a tile's eta neighbour in the
// next chunk runs on the same XCD shortly after it; giving each XCD a
// contiguous run of all tiles instead keeps eight bands in flight, one per
// XCD (7 % slower at 201x201x101).  The grid holds zchunks * 8 * slice
// workgroups; those past the end of a chunk's tiles get -1.
__device__ __forceinline__ int tile_of_block(const StageParams &P, int b) {
    const int tpl = P.tiles_x * P.tiles_y, slice = (tpl + 7) >> 3;
    const int l = b >> 3, c = l / slice, within = (b & 7) * slice + (l - c * slice);
    return within < tpl && c < P.zchunks ? c * tpl + within : -1;
}

// ---------------------------------------------------------------------------
// KT flux through one cell face (SemiDiscreteKurganovTadmorScheme.cpp:13-57)
// ---------------------------------------------------------------------------

// Newton inputs of one reconstructed face state (EnergyMomentumTensor.cpp:116-143
// with W = Pi = 0): M^mu = T^{tau mu} - pi^{tau mu}, F = M^3/(M^0 + P_L).
struct FaceState {
    double M0, M1, M2, M3, PL, F, Ft, x, MBT;
};

__device__ __forceinline__ FaceState face_state(double t, double ttt, double ttx, double tty, double ttn, double pl,
                                                double pitt, double pitx, double pity, double pitn) {
    FaceState f;
    f.M0 = ttt - pitt;
    f.M1 = ttx - pitx;
    f.M2 = tty - pity;
    f.M3 = ttn - pitn;
    f.PL = pl;
    double M0PL = f.M0 + pl;
    if (M0PL == 0.0) M0PL = 1.e-16;
    f.F = fdiv(f.M3, M0PL);
    f.Ft = t * f.F;
    f.x = sqrt_pos(fabs(1.0 - f.Ft * f.Ft));
    f.MBT = sqrt_pos(f.M1 * f.M1 + f.M2 * f.M2);
    if (f.MBT == 0.0) f.MBT = 1.e-16;
    return f;
}

// One Newton update of u_T for state S from u0 (EnergyMomentumTensor.cpp:45-70),
// evaluated without branches: *u1 receives the update; the status is 1
// converged, -1 failed (e < 0 at u0, or an update that is NaN, infinite,
// negative or above 9.0072e15), 0 continue.  The reference stops before the
// update when e < 0; the update computed here is then discarded, so the
// decisions and the values kept are the reference's.
__device__ __forceinline__ int newton_update(double t, const FaceState &S, double u0, double *u1) {
    const double Ft2 = S.Ft * S.Ft;
    const double xM = S.x * S.MBT;
    const double bL = S.x * S.x * S.M0 - Ft2 * S.PL;
    const double b = S.x * S.x + Ft2;
    const double c0 = S.M0 - t * S.Ft * S.M3;
    double rs = rsqrt(1.0 + u0 * u0);
    double U = u0 * rs;
    double e = c0 - U * xM;
    double iP = rs * rs * rs;
    double g = bL + b * 0.5 * (e - S.PL);
    double f = U * g - xM;
    double fp = iP * g - 0.5 * U * b * xM * iP;
    fp = fabs(fp) == 0.0 ? 1.e-16 : fp;
    double u = u0 - newton_quotient(f, fp);
    *u1 = u;
    // non-short-circuit operators: no branch splits the two sides' chains
    const bool bad = (e < 0.0) | newton_out_of_range(u);
    const bool conv = fabs(u - u0) <= 1.e-7 * fabs(u);
    return bad ? -1 : (int)conv;
}

// Speeds of both sides of a face by the reference's iteration, in one loop
// (independent iterations, each side stops at its own convergence or failure,
// at most 10^4 iterations each), from `guess`.  Every pass evaluates both
// updates and keeps each only while its side is still running, so the two
// dependency chains interleave and the loop body has no branches.  Outputs the
// signed speed v = u^DIR / u^tau of each side; a failed recovery gives the
// reference's fallback u = (1,0,0,0), i.e. v = 0.
template <int DIR>
__device__ __forceinline__ void face_newton(double t, double guess, const FaceState &A, const FaceState &B, double &vA,
                                            double &vB) {
    double ua = guess, ub = guess;
    int sa = 0, sb = 0;
    for (int it = 0; it < 10000 && (sa == 0 || sb == 0); ++it) {
        double na, nb;
        const int ta = newton_update(t, A, ua, &na);
        const int tb = newton_update(t, B, ub, &nb);
        const bool ra = sa == 0, rb = sb == 0;
        ua = ra ? na : ua;
        sa = ra ? ta : sa;
        ub = rb ? nb : ub;
        sb = rb ? tb : sb;
    }
    auto speed = [](const FaceState &S, double u, int st) {
        if (st != 1) return 0.0;
        if (DIR == 3) return S.F;  // u^eta / u^tau = F C/x / (C/x)
        double iC = rsqrt(1.0 + u * u);
        double num = DIR == 1 ? S.M1 : S.M2;
        return u * num * S.x * iC * rcp(S.MBT);  // (u M/MBT) / (C/x)
    };
    vA = speed(A, ua, sa);
    vB = speed(B, ub, sb);
}

// Speeds of both sides of a face, from the start |u_T|^2 = guess2.  With
// ROOT_JUMP they come in closed form (vah_face.h) wherever both sides' Newton
// paths must end on it, which is everywhere but in failing or barely physical
// cells; a lane where one of them need not runs the iteration.
template <int DIR, bool ROOT_JUMP, typename R>
__device__ __forceinline__ void face_speeds(double t, double guess2, const R *qR, const R *qL, double &vR, double &vL,
                                            bool live) {
    if (ROOT_JUMP) {
        const FaceStart s = face_start(guess2);
        auto side = [&](const R *q, double *v) {
            return face_speed<DIR>(t, (double)q[TTT] - (double)q[PITT], (double)q[TTX] - (double)q[PITX],
                                   (double)q[TTY] - (double)q[PITY], (double)q[TTN] - (double)q[PITN], (double)q[PL], s,
                                   v);
        };
        const bool okR = side(qR, &vR), okL = side(qL, &vL);
        if ((okR & okL) | !live) return;
    }
    auto state = [&](const R *q) {
        return face_state(t, q[TTT], q[TTX], q[TTY], q[TTN], q[PL], q[PITT], q[PITX], q[PITY], q[PITN]);
    };
    face_newton<DIR>(t, sqrt_pos(guess2), state(qR), state(qL), vR, vL);
}

// ---------------------------------------------------------------------------
// Field sets seen through buffer resources.  A load or store takes the byte
// offset of the cell (per lane, 32-bit) and the byte offset of the field
// (uniform, an SGPR), so the 15-field stencils need no per-lane 64-bit address
// arithmetic.  An access outside the set's byte range reads 0 and drops the
// store instead of faulting.  A set must stay below 4 GB (checked on the host).
// ---------------------------------------------------------------------------
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kBufWord3 = 0x00020000;  // raw dword access, gfx9 family

struct Buf {
    __amdgpu_buffer_rsrc_t r;
};

__device__ __forceinline__ Buf make_buf(const double *base, int nfields, long fs) {
    Buf b;
    b.r = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)(uint32_t)((long)nfields * fs * 8), kBufWord3);
    return b;
}

__device__ __forceinline__ double ld(const Buf &b, uint32_t cell, uint32_t field) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b.r, (int)cell, (int)field, 0));
}

// The cell at this offset and the next one in x (16 bytes, 8-byte aligned).  The
// vector L1 is the busiest unit of the stage kernels (its data return 68 % of the
// cycles at 611x587, 92 % at 201x201x101) and delivers one such load at 95 bytes per
// clock, two of 8 bytes at 64, whatever the alignment.  The x stencils and the x
// differences with their cell loaded this way: 611x587 142 -> 134 us per step,
// 201x201x101 2.38 -> 2.31 ms, split 97x89x33 173 -> 167 us.
__device__ __forceinline__ void ld2(const Buf &b, uint32_t cell, uint32_t field, double &v0, double &v1) {
    const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(b.r, (int)cell, (int)field, 0);
    const u32x2_t lo = {v.x, v.y}, hi = {v.z, v.w};
    v0 = __builtin_bit_cast(double, lo);
    v1 = __builtin_bit_cast(double, hi);
}

__device__ __forceinline__ void st(const Buf &b, uint32_t cell, uint32_t field, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, v), b.r, (int)cell, (int)field, 0);
}

// the buffers of one stage, and the byte strides of the layout
struct Views {
    Buf qin, qout, qn, e_in, p_in, e_out, p_out, ucur, uprev, uout;
    uint32_t f8;        // field to field
    uint32_t sy8, sz8;  // row to row, plane to plane
};

__device__ __forceinline__ Views make_views(const StageParams &P) {
    Views v;
    v.qin = make_buf(P.qin, NQ, P.fs);
    v.qout = make_buf(P.qout, NQ, P.fs);
    v.qn = make_buf(P.qn, NQ, P.fs);
    v.e_in = make_buf(P.e_in, 1, P.fs);
    v.p_in = make_buf(P.p_in, 1, P.fs);
    v.e_out = make_buf(P.e_out, 1, P.fs);
    v.p_out = make_buf(P.p_out, 1, P.fs);
    v.ucur = make_buf(P.ucur, 4, P.fs);
    v.uprev = make_buf(P.uprev, 4, P.fs);
    v.uout = make_buf(P.uout, 4, P.fs);
    v.f8 = (uint32_t)(P.fs * 8);
    v.sy8 = (uint32_t)(P.sy * 8);
    v.sz8 = (uint32_t)(P.sz * 8);
    return v;
}

// d_i of the pi components entering the axis source of direction DIR
template <int DIR>
struct AxisFields {  // pi^{DIR mu} for mu = x, y, eta
    static constexpr int x = DIR == 1 ? PIXX : DIR == 2 ? PIXY : PIXN;
    static constexpr int y = DIR == 1 ? PIXY : DIR == 2 ? PIYY : PIYN;
    static constexpr int n = DIR == 1 ? PIXN : DIR == 2 ? PIYN : PINN;
};

// Flux through one face.  load(n, v) gives field n at the four stencil positions
// (c-2st .. c+st for the face between cells c-st and c); the left/right
// states are the reference's half-cell extrapolations
// (HalfSiteExtrapolation.cpp:12-26); emit(n, H_n) receives the 15 components in
// order.  start(guess2, v) loads the solves' start |u_T|^2 and, with AX >= 0,
// the velocity u^DIR / u^tau of the cell whose axis source (SourceTerms.cpp:46-176)
// is formed on the way: the cell at stencil position AX + 1, whose centred pi
// differences (times h) are those of positions AX + 2 and AX.  axis(S) receives
// its four components; a lane that is not live gets some flux without ever
// iterating.  The nine components the recovery needs stay in
// registers, the other six are loaded and reconstructed after it, which keeps
// the live state small.
template <int DIR, typename R, bool ROOT_JUMP, int AX, typename Start, typename Load, typename Emit, typename Axis>
__device__ __forceinline__ void face_flux(double t, double h, Start start, Load load, Emit emit, Axis axis,
                                          bool live = true) {
    constexpr int NN = 9;  // TTT..PITN
    // all loads of the nine fields first, so that they are in flight together
    double raw[NN][4];
#pragma unroll
    for (int n = 0; n < NN; ++n) load(n, raw[n]);
    // the start (loads of its own) after the stencil loads, so that one wait
    // covers both
    double guess2, v = 0.0;
    start(guess2, v);
    AxisPi<R> ax;
    if constexpr (AX >= 0) {
        auto d = [&](int n) { return (R)((raw[n][AX + 2] - raw[n][AX]) * h); };
        ax.dtt = d(PITT);
        ax.dtx = d(PITX);
        ax.dty = d(PITY);
        ax.dtn = d(PITN);
    }
    R qL[NN], qR[NN];
#pragma unroll
    for (int n = 0; n < NN; ++n) {
        R q0 = (R)raw[n][0], q1 = (R)raw[n][1], q2 = (R)raw[n][2], q3 = (R)raw[n][3];
        face_values(q0, q1, q2, q3, qL[n], qR[n]);
    }
    // the recovery of both sides runs in double whatever R is
    double vR, vL;
    face_speeds<DIR, ROOT_JUMP, R>(t, guess2, qR, qL, vR, vL, live);
    const double a = fmax(fabs(vL), fabs(vR));
    // (F(qR) + F(qL) - a (qR - qL)) / 2 with F(q) = v q
    const R cR = (R)(0.5 * (vR - a)), cL = (R)(0.5 * (vL + a));
#pragma unroll
    for (int n = 0; n < NN; ++n) emit(n, cR * qR[n] + cL * qL[n]);
    double rest[NQ - NN][4];
#pragma unroll
    for (int n = NN; n < NQ; ++n) load(n, rest[n - NN]);
#pragma unroll
    for (int n = NN; n < NQ; ++n) {
        R q0 = (R)rest[n - NN][0], q1 = (R)rest[n - NN][1], q2 = (R)rest[n - NN][2], q3 = (R)rest[n - NN][3];
        R l, r;
        face_values(q0, q1, q2, q3, l, r);
        emit(n, cR * r + cL * l);
    }
    if constexpr (AX >= 0) {
        auto d = [&](int n) { return (R)((rest[n - NN][AX + 2] - rest[n - NN][AX]) * h); };
        ax.dix = d(AxisFields<DIR>::x);
        ax.diy = d(AxisFields<DIR>::y);
        ax.din = d(AxisFields<DIR>::n);
        R Sa[4];
        axis_source<DIR>(ax, (R)v, Sa);
        axis(Sa);
    }
}

// |u_T|^2 at a cell
__device__ __forceinline__ double uT2_of(const Buf &u, uint32_t f8, uint32_t c) {
    double ux = ld(u, c, f8), uy = ld(u, c, 2 * f8);
    return ux * ux + uy * uy;
}

// d_i of the pi components entering the axis source of direction DIR, from
// memory (all fourteen loads issued before the differences are formed)
template <int DIR, typename R>
__device__ __forceinline__ AxisPi<R> axis_pi(const Buf &q, uint32_t f8, uint32_t s, uint32_t stp, double h) {
    constexpr int F[7] = {PITT, PITX, PITY, PITN, AxisFields<DIR>::x, AxisFields<DIR>::y, AxisFields<DIR>::n};
    double up[7], dn[7];
#pragma unroll
    for (int i = 0; i < 7; ++i) {
        up[i] = ld(q, s + stp, F[i] * f8);
        dn[i] = ld(q, s - stp, F[i] * f8);
    }
    __builtin_amdgcn_sched_barrier(0);  // keep the loads together (not sunk to their uses)
    auto d = [&](int i) { return (R)((up[i] - dn[i]) * h); };
    AxisPi<R> r;
    r.dtt = d(0);
    r.dtx = d(1);
    r.dty = d(2);
    r.dtn = d(3);
    r.dix = d(4);
    r.diy = d(5);
    r.din = d(6);
    return r;
}

// one component of the reference's per-direction update:
// acc += dt * [ (H- - H+)/d  (+ S_axis for the four T^{tau mu} components) ]
__device__ __forceinline__ void add_component(double &acc, int n, double Hm, double Hp, const double (&Sa)[4],
                                              double inv_d, double dt) {
    double r = (Hm - Hp) * inv_d;
    if (n < 4) r += Sa[n];
    acc += r * dt;
}

// the flux part of one component: acc += dt * (H- - H+)/d, the axis sources
// being added separately.  In double one fused multiply-add with dt_d = dt/d
// (precomputed with the stage parameters); in float the difference is formed
// in float and accumulated in double.
__device__ __forceinline__ void add_flux(double &acc, double Hm, double Hp, double /*inv_d*/, double dt_d,
                                         double /*dt*/) {
    acc = __builtin_fma(Hm - Hp, dt_d, acc);
}
__device__ __forceinline__ void add_flux(double &acc, float Hm, float Hp, float inv_d, double /*dt_d*/, double dt) {
    acc += (double)((Hm - Hp) * inv_d) * dt;
}

template <bool D3>
__device__ __forceinline__ void load_src_in(const StageParams &P, const Views &V, uint32_t s, SrcIn &in) {
    const Buf &u = V.ucur;
    const uint32_t f8 = V.f8, sy8 = V.sy8, sz8 = V.sz8;
    in.t = P.t_src;
    in.dt_inv = P.dt_inv;
    in.etabar_inv = P.etabar_inv;
    // The cell together with its left neighbour.  The right neighbours are loaded
    // below, in the order in which the differences enter the source terms: the
    // compiler ranks the operands of its sums by their loads, and with them the
    // products it contracts, which the split precision's float terms would show.
    double el, pl, utl, uxl, uyl, unl;
    ld2(V.e_in, s - 8, 0, el, in.e);
    ld2(V.p_in, s - 8, 0, pl, in.p);
    ld2(u, s - 8, 0, utl, in.ut);
    ld2(u, s - 8, f8, uxl, in.ux);
    ld2(u, s - 8, 2 * f8, uyl, in.uy);
    ld2(u, s - 8, 3 * f8, unl, in.un);
    in.utp = ld(V.uprev, s, 0);
    in.uxp = ld(V.uprev, s, f8);
    in.uyp = ld(V.uprev, s, 2 * f8);
    in.unp = ld(V.uprev, s, 3 * f8);
    auto cd = [&](const Buf &b, uint32_t fo, uint32_t stp, double h) { return (ld(b, s + stp, fo) - ld(b, s - stp, fo)) * h; };
    in.dxut = (ld(u, s + 8, 0) - utl) * P.hx;
    in.dxux = (ld(u, s + 8, f8) - uxl) * P.hx;
    in.dxuy = (ld(u, s + 8, 2 * f8) - uyl) * P.hx;
    in.dxun = (ld(u, s + 8, 3 * f8) - unl) * P.hx;
    in.dyut = cd(u, 0, sy8, P.hy);
    in.dyux = cd(u, f8, sy8, P.hy);
    in.dyuy = cd(u, 2 * f8, sy8, P.hy);
    in.dyun = cd(u, 3 * f8, sy8, P.hy);
    const uint32_t plo = PL * f8;
    in.dxp = (ld(V.p_in, s + 8, 0) - pl) * P.hx;
    in.dyp = cd(V.p_in, 0, sy8, P.hy);
    in.dxe = (ld(V.e_in, s + 8, 0) - el) * P.hx;
    in.dye = cd(V.e_in, 0, sy8, P.hy);
    in.dxpl = cd(V.qin, plo, 8, P.hx);
    in.dypl = cd(V.qin, plo, sy8, P.hy);
    if (D3) {
        in.dnut = cd(u, 0, sz8, P.hz);
        in.dnux = cd(u, f8, sz8, P.hz);
        in.dnuy = cd(u, 2 * f8, sz8, P.hz);
        in.dnun = cd(u, 3 * f8, sz8, P.hz);
        in.dnp = cd(V.p_in, 0, sz8, P.hz);
        in.dne = cd(V.e_in, 0, sz8, P.hz);
        in.dnpl = cd(V.qin, plo, sz8, P.hz);
    } else {
        // one eta cell: the ghost planes equal the cell, the differences are exactly 0
        in.dnut = in.dnux = in.dnuy = in.dnun = 0.0;
        in.dnp = in.dne = in.dnpl = 0.0;
    }
}

// Inputs of a cell's recovery besides its conserved variables: the e its
// fallback scales and the |u_T|^2 its solve starts from.
struct Recovery {
    double e_prev, uT2_guess;
};

// Stage-2 convex combination, recovery, regulation, store with ghost copies.
template <bool D3, bool STAGE2>
__device__ __forceinline__ double finish_cell(const StageParams &P, const Views &V, uint32_t s, int ii, int jj, int kk,
                                              double (&acc)[NQ], const Recovery &rec, bool &nan, bool &fallback) {
    const uint32_t f8 = V.f8;
    if (STAGE2) {
        // all fifteen loads first, so that they are in flight together
        double qn[NQ];
#pragma unroll
        for (int n = 0; n < NQ; ++n) qn[n] = ld(V.qn, s, n * f8);
#pragma unroll
        for (int n = 0; n < NQ; ++n) acc[n] = 0.5 * (acc[n] + qn[n]);
    }
    Prim r = recover(P.t_rec, acc, rec.e_prev, rec.uT2_guess);
    EosP pe;
    pe.begin(P.eos, r.e);
    nan = nan || prim_nan(r);
    fallback = !r.ok;
    double e = r.e, p;
    regulate(P.t_rec, P.eos, pe, acc, e, p, r.ut, r.ux, r.uy, r.un);
    double vals[NQ + 6];
#pragma unroll
    for (int n = 0; n < NQ; ++n) vals[n] = acc[n];
    vals[NQ] = e;
    vals[NQ + 1] = p;
    vals[NQ + 2] = r.ut;
    vals[NQ + 3] = r.ux;
    vals[NQ + 4] = r.uy;
    vals[NQ + 5] = r.un;
    auto store = [&](uint32_t d) {
#pragma unroll
        for (int n = 0; n < NQ; ++n) st(V.qout, d, n * f8, vals[n]);
        st(V.e_out, d, 0, vals[NQ]);
        st(V.p_out, d, 0, vals[NQ + 1]);
#pragma unroll
        for (int m = 0; m < 4; ++m) st(V.uout, d, m * f8, vals[NQ + 2 + m]);
    };
    store(s);
    // face ghosts: copies of the boundary cell (only one index outside)
    if (ii == 0) { store(s - 8); store(s - 16); }
    if (ii == P.nx - 1) { store(s + 8); store(s + 16); }
    if (jj == 0) { store(s - V.sy8); store(s - 2 * V.sy8); }
    if (jj == P.ny - 1) { store(s + V.sy8); store(s + 2 * V.sy8); }
    if (D3) {
        if (kk == 0) { store(s - V.sz8); store(s - 2 * V.sz8); }
        if (kk == P.nz - 1) { store(s + V.sz8); store(s + 2 * V.sz8); }
    }
    return e;
}

// NaN checks of the reference (EnergyMomentumTensor.cpp:178-194 and
// SourceTerms.cpp:658-719 exit there) become a counter the host reads.
// The wave's largest new e goes to P.emax (as ordered bits: e > 0) when set,
// which the batch uses for its freezeout test.
__device__ __forceinline__ void count_flags(const StageParams &P, bool nan, bool fallback, double e) {
    unsigned long long bn = __ballot(nan), bf = __ballot(fallback);
    if ((threadIdx.x & 63) == 0) {
        if (bn) atomicAdd(&P.counters[0], (unsigned)__popcll(bn));
        if (bf) atomicAdd(&P.counters[1], (unsigned)__popcll(bf));
    }
    if (P.emax) {
        double m = e > 0.0 ? e : 0.0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
        if ((threadIdx.x & 63) == 0 && m > 0.0) atomicMax(P.emax, (unsigned long long)__double_as_longlong(m));
    }
}

// The LDS of a stage workgroup: what the face waves hand to the cell waves for
// one plane.  Hx / Hy: fluxes through the tile's x / y faces, slot = the face's
// lane; Dz: difference of the fluxes through a cell's lower and upper eta face;
// Ax: the axis sources of the three directions.
template <bool D3, typename R, int NW>
struct StageLds {
    static constexpr int NL = 64 * NW;  // lanes per role
    R Hx[NQ][NL];
    R Hy[NQ][NL];
    R Dz[D3 ? NQ : 1][D3 ? NL : 1];
    R Ax[D3 ? 3 : 2][4][NL];
};

// a direction as a type
template <int N>
struct Dir {
    static constexpr int value = N;
};

// a workgroup's part of the lattice
struct Tile {
    int i0, j0, k0, k1;
};

template <int TX, int TY>
__device__ __forceinline__ Tile tile_at(const StageParams &P, int tile) {
    const int tpl = P.tiles_x * P.tiles_y;
    const int zc = tile / tpl;
    const int txy = tile - zc * tpl;
    const int ty = txy / P.tiles_x;
    Tile T;
    T.i0 = (txy - ty * P.tiles_x) * TX;
    T.j0 = ty * TY;
    T.k0 = zc * P.kz;
    T.k1 = min(T.k0 + P.kz, P.nz);
    return T;
}

// Byte offset of the cell (i, j) of a plane.  Indices one past either end
// (ghosts) are fine.
__device__ __forceinline__ uint32_t cell_offset(const StageParams &P, uint32_t plane, int i, int j) {
    return (plane + (uint32_t)(j + 2) * (uint32_t)P.sy + (uint32_t)(i + 2)) * 8u;
}

// Source terms of a cell: acc = q + dt S (eulerStepKernelSource), and the
// inputs of its recovery.
template <bool D3, bool STAGE2, typename R>
__device__ __forceinline__ void cell_sources(const StageParams &P, const Views &V, uint32_t s, double (&acc)[NQ],
                                             Recovery &rec, double &iut, bool &nan) {
    const uint32_t f8 = V.f8;
    double Q[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) Q[n] = ld(V.qin, s, n * f8);
    SrcIn in;
    load_src_in<D3>(P, V, s, in);
    R S[NQ];
    source_terms<R>(P.eos, in, Q, S, nan);
#pragma unroll
    for (int n = 0; n < NQ; ++n) acc[n] = Q[n] + P.dt * (double)S[n];
    iut = rcp(in.ut);
    // the cell recovery's inputs come from the same loads: e at the stage's
    // input level (its fallback base) and |u_T| of the velocity that seeds it,
    // u_cur in stage 1 and u_prev in stage 2
    // (FullyDiscreteKurganovTadmorScheme.cpp:761-780)
    rec.e_prev = in.e;
    rec.uT2_guess = STAGE2 ? in.uxp * in.uxp + in.uyp * in.uyp : in.ux * in.ux + in.uy * in.uy;
}

// The cell waves' part of one tile.  Per plane: sources; wait for the plane's
// fluxes; add them; hand the LDS back; finish the cell.
template <bool D3, bool STAGE2, typename R, int TX, int TY, int NW>
__device__ __forceinline__ void cell_role(const StageParams &P, const Views &V, const Tile &T, const StageLds<D3, R, NW> &lds,
                                          int lane) {
    const double dt = P.dt;
    const int ci = lane % TX, cj = lane / TX;
    const int ii = T.i0 + ci, jj = T.j0 + cj;
    const bool cell_ok = cj < TY && ii < P.nx && jj < P.ny;
    for (int kk = T.k0; kk < T.k1; ++kk) {
        const uint32_t s = cell_offset(P, (uint32_t)plane_of(kk, D3) * (uint32_t)P.sz, ii, jj);
        bool nan = false, fallback = false;
        double acc[NQ];
        Recovery rec{0.0, 0.0};
        if (cell_ok) {
            double iut;
            cell_sources<D3, STAGE2, R>(P, V, s, acc, rec, iut, nan);
        }
        __syncthreads();  // the plane's fluxes are in LDS
        if (cell_ok) {
            const R inv_dx = (R)P.inv_dx, inv_dy = (R)P.inv_dy, inv_dz = (R)P.inv_dz;
            const int fx = cj * (TX + 1) + ci, fy = lane;  // the cell's lower x and y face
            // All reads of a direction first: left to itself the compiler waits
            // for each pair of fluxes, 2,700 cycles for the phase.
            constexpr int ND = D3 ? 3 : 2;
            R ax[ND][4], lo[NQ], hi[NQ], dz[D3 ? NQ : 1];
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                ax[0][n] = lds.Ax[0][n][fx];
                ax[1][n] = lds.Ax[1][n][fy];
                if constexpr (D3) ax[2][n] = lds.Ax[2][n][lane];
            }
#pragma unroll
            for (int n = 0; n < NQ; ++n) {
                lo[n] = lds.Hx[n][fx];
                hi[n] = lds.Hx[n][fx + 1];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < 4; ++n) {
#pragma unroll
                for (int d = 0; d < ND; ++d) acc[n] += (double)ax[d][n] * dt;
            }
#pragma unroll
            for (int n = 0; n < NQ; ++n) add_flux(acc[n], lo[n], hi[n], inv_dx, P.dt_dx, dt);
#pragma unroll
            for (int n = 0; n < NQ; ++n) {
                lo[n] = lds.Hy[n][fy];
                hi[n] = lds.Hy[n][fy + TX];
                if constexpr (D3) dz[n] = lds.Dz[n][lane];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < NQ; ++n) {
                add_flux(acc[n], lo[n], hi[n], inv_dy, P.dt_dy, dt);
                if constexpr (D3) add_flux(acc[n], dz[n], R(0), inv_dz, P.dt_dz, dt);
            }
        }
        __syncthreads();  // the face waves may write the next plane
        double e_new = 0.0;
        if (cell_ok) e_new = finish_cell<D3, STAGE2>(P, V, s, ii, jj, kk, acc, rec, nan, fallback);
        count_flags(P, nan, fallback, e_new);
    }
}

// The face waves' part of one tile.  Per plane: the x faces ((TX+1) x TY, face
// f between cells f-1 and f), the y faces (TX x (TY+1)) and each cell's upper
// eta face; the lower one is carried from the plane below.  In 3+1D a lane
// keeps its column's planes k-1, k, k+1 in registers (90 of the 256; the two
// x / y solves need about 150), so that an eta face loads one new plane
// instead of four: 201x201x101 2.68 -> 2.40 ms per step, and the L1 sends a
// third fewer requests to L2.  All lanes with a y face keep a column, also the
// row above the tile, and the y face takes its own cell from it: 2.33 -> 2.28 ms.
// That row's eta faces are formed with the others and used by no one; its
// corner ghosts hold no state, so its lanes never enter the iteration (live).
template <bool D3, typename R, int TX, int TY, int NW>
__device__ __forceinline__ void face_role(const StageParams &P, const Views &V, const Tile &T, StageLds<D3, R, NW> &lds,
                                          int lane) {
    const uint32_t f8 = V.f8, sy8 = V.sy8, sz8 = V.sz8;
    const double t = P.t_src;
    const int ci = lane % TX, cj = lane / TX;              // y face and cell
    const int xi = lane % (TX + 1), xj = lane / (TX + 1);  // x face
    const bool x_ok = xj < TY && T.i0 + xi <= P.nx && T.j0 + xj < P.ny;
    const bool y_ok = cj <= TY && T.i0 + ci < P.nx && T.j0 + cj <= P.ny;
    const bool z_ok = D3 && cj < TY && T.i0 + ci < P.nx && T.j0 + cj < P.ny;
    // a face's start: |u_T|^2 at byte offset g, u^dir / u^tau at c
    auto start = [&](uint32_t g, uint32_t c, int dir) {
        return [&V, f8, g, c, dir](double &guess2, double &v) {
            const double ux = ld(V.ucur, g, f8), uy = ld(V.ucur, g, 2 * f8);
            const double ut = ld(V.ucur, c, 0), ui = ld(V.ucur, c, dir * f8);
            guess2 = ux * ux + uy * uy;
            v = ui * rcp(ut);
        };
    };
    auto axis_to = [&](int d) {
        return [&lds, d, lane](const R (&S)[4]) {
#pragma unroll
            for (int n = 0; n < 4; ++n) lds.Ax[d][n][lane] = S[n];
        };
    };
    R carry[NQ];                                              // flux through the lower eta face
    double below[D3 ? NQ : 1], here[D3 ? NQ : 1], above[D3 ? NQ : 1];  // planes k-1, k, k+1 of this column
    if constexpr (D3) {
        if (y_ok) {
            const uint32_t s = cell_offset(P, (uint32_t)plane_of(T.k0, D3) * (uint32_t)P.sz, T.i0 + ci, T.j0 + cj);
            double far[NQ];
#pragma unroll
            for (int n = 0; n < NQ; ++n) far[n] = ld(V.qin, s - 2u * sz8, n * f8);
#pragma unroll
            for (int n = 0; n < NQ; ++n) below[n] = ld(V.qin, s - sz8, n * f8);
#pragma unroll
            for (int n = 0; n < NQ; ++n) here[n] = ld(V.qin, s, n * f8);
#pragma unroll
            for (int n = 0; n < NQ; ++n) above[n] = ld(V.qin, s + sz8, n * f8);
            face_flux<3, R, true, -1>(
                t, 0.0, [&](double &guess2, double &) { guess2 = uT2_of(V.ucur, f8, s - sz8); },
                [&](int n, double (&v)[4]) { v[0] = far[n], v[1] = below[n], v[2] = here[n], v[3] = above[n]; },
                [&](int n, R h) { carry[n] = h; }, [](const R (&)[4]) {}, z_ok);
        }
    }
    for (int kk = T.k0; kk < T.k1; ++kk) {
        const uint32_t plane = (uint32_t)plane_of(kk, D3) * (uint32_t)P.sz;
        if (x_ok) {
            const uint32_t c = cell_offset(P, plane, T.i0 + xi, T.j0 + xj);
            face_flux<1, R, true, 1>(
                t, P.hx, start(c - 8, c, 1),
                [&](int n, double (&v)[4]) {
                    ld2(V.qin, c - 16u, n * f8, v[0], v[1]);
                    ld2(V.qin, c, n * f8, v[2], v[3]);
                },
                [&](int n, R h) { lds.Hx[n][lane] = h; }, axis_to(0));
        }
        const uint32_t s = cell_offset(P, plane, T.i0 + ci, T.j0 + cj);
        if (y_ok) {
            face_flux<2, R, true, 1>(
                t, P.hy, start(s - sy8, s, 2),
                [&](int n, double (&v)[4]) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if (D3 && j == 2) v[j] = here[n];
                        else v[j] = ld(V.qin, s + (uint32_t)j * sy8 - 2u * sy8, n * f8);
                    }
                },
                [&](int n, R h) { lds.Hy[n][lane] = h; }, axis_to(1));
        }
        if constexpr (D3) {
            if (y_ok) {
                double fresh[NQ];
#pragma unroll
                for (int n = 0; n < NQ; ++n) fresh[n] = ld(V.qin, s + 2u * sz8, n * f8);
                face_flux<3, R, true, 0>(
                    t, P.hz, start(s, s, 3),
                    [&](int n, double (&v)[4]) { v[0] = below[n], v[1] = here[n], v[2] = above[n], v[3] = fresh[n]; },
                    [&](int n, R h) {
                        lds.Dz[n][lane] = carry[n] - h;
                        carry[n] = h;
                    },
                    axis_to(2), z_ok);
#pragma unroll
                for (int n = 0; n < NQ; ++n) {
                    below[n] = here[n];
                    here[n] = above[n];
                    above[n] = fresh[n];
                }
            }
        }
        __syncthreads();  // the plane's fluxes are in LDS
        __syncthreads();  // and have been read
    }
}

// One tile of one stage by a workgroup of 2 x 64 NW lanes: the first half are
// the cell waves, the second the face waves (the split is uniform over each
// wave).  Both run the same number of barriers, two per plane, and the last one
// leaves the LDS free for another tile.
template <bool D3, bool STAGE2, typename R, int TX, int TY, int NW>
__device__ __forceinline__ void stage_tile(const StageParams &P, int tile, StageLds<D3, R, NW> &lds) {
    static_assert(tile_fits<TX, TY, NW>(), "tile does not fit its waves");
    const Views V = make_views(P);
    const Tile T = tile_at<TX, TY>(P, tile);
    const int role = __builtin_amdgcn_readfirstlane((int)threadIdx.x / (64 * NW));
    const int lane = (int)threadIdx.x - role * 64 * NW;
    if (role != 0)
        face_role<D3, R, TX, TY, NW>(P, V, T, lds, lane);
    else
        cell_role<D3, STAGE2, R, TX, TY, NW>(P, V, T, lds, lane);
}

// The parameters are read where they are used, through the kernel-argument
// segment (the kernel's first and only argument, at offset 0), instead of from
// the argument copy the compiler otherwise keeps in scalar registers across
// the plane loop: some ninety uniform values there made it spill about three
// times as many scalar registers and twice as many vector registers as it does
// reading them in place.
__device__ __forceinline__ const StageParams &kernarg_params() {
    typedef __attribute__((address_space(4))) const StageParams KernargParams;
    return *(const StageParams *)(KernargParams *)__builtin_amdgcn_kernarg_segment_ptr();
}

// One event: workgroup -> tile (XCD-aware) -> stage_tile.
template <bool D3, bool STAGE2, typename R, int TX, int NW>
__global__ __launch_bounds__(128 * NW, kWavesPerSimd) void stage_kernel(StageParams P_arg) {
    const StageParams &P = kernarg_params();
    (void)P_arg;
    __shared__ StageLds<D3, R, NW> lds;
    const int tile = tile_of_block(P, (int)blockIdx.x);
    if (tile < 0) return;  // padding workgroups: no barrier reached
    stage_tile<D3, STAGE2, R, TX, kTileY, NW>(P, tile, lds);
}

// The reference's work split (VAH_FLUX_PER_CELL): a lane per cell solves both of
// its faces in each direction with the cell's own Newton guess.
template <bool D3, bool STAGE2>
__global__ __launch_bounds__(kCellThreads, kWavesPerSimd) void stage_per_cell_kernel(StageParams P_arg) {
    const StageParams &P = kernarg_params();
    (void)P_arg;
    __shared__ double Hs[NQ][kCellThreads];  // the lane's forward face
    const int tile = tile_of_block(P, (int)blockIdx.x);
    if (tile < 0) return;
    const Views V = make_views(P);
    const Tile T = tile_at<kCellTileX, kCellTileY>(P, tile);
    const uint32_t f8 = V.f8;
    const double t = P.t_src, dt = P.dt;
    const int tid = (int)threadIdx.x;
    const int ii = T.i0 + tid % kCellTileX, jj = T.j0 + tid / kCellTileX;
    const bool cell_ok = ii < P.nx && jj < P.ny;
    for (int kk = T.k0; kk < T.k1; ++kk) {
        const uint32_t s = cell_offset(P, (uint32_t)plane_of(kk, D3) * (uint32_t)P.sz, ii, jj);
        bool nan = false, fallback = false;
        double e_new = 0.0;
        if (cell_ok) {
            double acc[NQ], iut;
            Recovery rec{0.0, 0.0};
            cell_sources<D3, STAGE2, double>(P, V, s, acc, rec, iut, nan);
            const double uTs = uT2_of(V.ucur, f8, s);
            auto direction = [&](auto dir, uint32_t stp, double h, double inv_d) {
                constexpr int DIR = decltype(dir)::value;
                double Sa[4];
                axis_source<DIR>(axis_pi<DIR, double>(V.qin, f8, s, stp, h), ld(V.ucur, s, DIR * f8) * iut, Sa);
                auto face = [&](uint32_t c, auto emit) {
                    face_flux<DIR, double, false, -1>(
                        t, 0.0, [&](double &guess2, double &) { guess2 = uTs; },
                        [&](int n, double (&v)[4]) {
#pragma unroll
                            for (int j = 0; j < 4; ++j) v[j] = ld(V.qin, c + (uint32_t)j * stp - 2u * stp, n * f8);
                        },
                        emit,
                        [](const double (&)[4]) {});
                };
                face(s + stp, [&](int n, double H) { Hs[n][tid] = H; });
                face(s, [&](int n, double H) { add_component(acc[n], n, H, Hs[n][tid], Sa, inv_d, dt); });
            };
            direction(Dir<1>{}, 8u, P.hx, P.inv_dx);
            direction(Dir<2>{}, V.sy8, P.hy, P.inv_dy);
            if constexpr (D3) direction(Dir<3>{}, V.sz8, P.hz, P.inv_dz);
            e_new = finish_cell<D3, STAGE2>(P, V, s, ii, jj, kk, acc, rec, nan, fallback);
        }
        count_flags(P, nan, fallback, e_new);
    }
}

// Zero-gradient ghost copies of an initial state: every face ghost (one index
// outside; the stencils read no others) takes the value of its boundary cell.
// One thread per ghost cell and field (blockIdx.y), so that all copies are in
// flight at once and the launch holds a few thousand cells of the faces rather
// than the lattice: one thread per lattice cell copying its ghosts' 21 fields
// one after the other took 24 us at 41x37 and 41 us at 101x101x30, this takes
// 3.4 and 8.1 us.  `clear` (or null): four counters set to zero on the way.
static __global__ void ghost_fill_kernel(double *q, double *e, double *p, double *u, long fs, int nx, int ny, int nz,
                                         long sy, long sz, int d3, unsigned int *clear) {
    if (clear && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 4) clear[threadIdx.x] = 0u;
    long m = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long gx = 4L * ny * nz, gy = 4L * nx * nz, gz = d3 ? 4L * nx * ny : 0;
    const int f = (int)blockIdx.y;
    double *a = f < NQ ? q + f * fs : f == NQ ? e : f == NQ + 1 ? p : u + (f - NQ - 2) * fs;
    // g = 0, 1: the two layers below index 0; 2, 3: the two above n - 1
    auto copy = [&](long lo, long n, long st, int g) {
        const long src = g < 2 ? lo : lo + (n - 1) * st;
        a[g < 2 ? lo - (g + 1) * st : src + (g - 1) * st] = a[src];
    };
    auto at = [&](long i, long j, long k) { return (d3 ? k + 2 : 0) * sz + (j + 2) * sy + i + 2; };
    if (m < gx) {
        const long r = m >> 2;  // the four ghosts of a row side by side
        copy(at(0, r % ny, r / ny), nx, 1, (int)(m & 3));
    } else if ((m -= gx) < gy) {
        const long r = m / nx;
        copy(at(m % nx, 0, r >> 2), ny, sy, (int)(r & 3));
    } else if ((m -= gy) < gz) {
        const long r = m / nx;
        copy(at(m % nx, r % ny, 0), nz, sz, (int)(r / ny));
    }
}

// the grid of ghost_fill_kernel for blocks of 256
inline dim3 ghost_grid(int nx, int ny, int nz) {
    const long n = 4L * ny * nz + 4L * nx * nz + (nz > 1 ? 4L * nx * ny : 0);
    return dim3((unsigned)((n + 255) / 256), NQ + 6);
}

// The launches of the 3+1D stage kernels (vah_stage3d.hip): a translation
// unit of their own.
// precision and flux_mode take the values of include/vah.h.
struct StageLaunch {
    int grid;
    hipStream_t stream;
    int precision, flux_mode;
    bool wide;  // 16 x 7 tiles
};
void launch_stage_3d(const StageLaunch &L, int stage, const StageParams &P);

}  // namespace vah
