// Crank-Nicolson propagation with the wavefunction resident on the chip (1DTDSE/sources/prop.c:24-347).
//
// tdse_propagate.hip streams psi through HBM once per step (or two): it runs at the memory's rate
// and, per point, spends more instructions on scans than on the solve.  A grid of up to 16384
// points fits the registers of one compute unit, so here a workgroup of NW waves keeps the whole
// state of its instance in registers for the whole run: every lane owns C consecutive points
// (C = 16, 24 or 32).  Larger grids are covered by overlapping windows of that size, each
// stepped several times between its load and its store.
//
// The step.  With G_j = 1 + i g_j the scaled system B' psi' = A' psi (tdse_internal.h) is
//     M2' G psi' + i K psi' = M2' conj(G) psi - i K psi,   M2' = tridiag(1, 10, 1),  K = 36 dt / dx^2,
// i.e. for phi = G psi' a symmetric system with unit off-diagonals, tridiag(1, c_j, 1) phi = r.  Its
// factorisation needs one number per point, b_j = (1 + i g_j) / beta_j (the pivots of phi):
//     r_j   = (f_{j+1} - f_j) - (f_j - f_{j-1}) + (12 - i (12 g_j + K)) psi_j,   f = conj(G) psi
//     y_j   = r_j - b_{j-1} y_{j-1}            4 FMA a point
//     phi_j = b_j (y_j - phi_{j+1})            6
//     psi'_j = phi_j / (1 + i g_j)             4, from a table
// Both recurrences run twice around a scan over the lanes: once from zero for the carry that leaves
// the lane's chunk, once from the true carry.  Carries decay by rho < 1 per point, below 1e-17 after
// `reach` points, so a scan looks back only as far as that (3 or 4 levels within rows of 16 lanes, one
// step from the row before), a wave takes its carry from the one wave next to it, and windows
// overlap by `reach` points per step.
//
// Where the operands live: psi (r, y and phi in turn) in 4 C registers, b in LDS (up to 19 points a
// lane: 512 lanes x 19 x 16 B = 152 KB) and the rest in registers, both for the whole run; g, V' and
// 1/(1 + i g) come from L2, 32 B a point and step, shared by all instances of a grid.  HBM is idle:
// the FP64 units bound the step (about 57 + 330 / C instructions a point).
//
// Measured under load: a step of 16001 points takes 11.6 us a compute unit, of 12001 8.2, of 8001 6.0, 3.4 to 3.7e11
// points a second on the chip, where the streaming kernels reach 1.75e11.
//
// r_j takes the differences of f first: they cancel exactly, where f_{j-1} + f_{j+1} + (10 - i (10 g_j + K)) psi_j
// rounds three terms of 2 |g| |psi| each (|g| = 75 to 300) for a result of 12 |psi|.  That noise made two solves of one run with
// different lanes differ by 1.1e-12 on the dipole; now by 2e-13.
//
// Observables (prop.c:293-347) of the state a step starts from are summed in its first pass, per
// wave in a fixed order, and collected in LDS for up to TDSE_RES_RING steps.
#include "sincos_reduced.h"
#include "tdse_internal.h"
#include "tdse_wave.h"

namespace {

using namespace tdse;

// points of a lane whose b sits in LDS; the rest are held in registers
constexpr int lds_points(int c) { return c < TDSE_RES_LDS ? c : TDSE_RES_LDS; }

// what neighbouring waves exchange in one step
struct WaveEdge {
    double2 a;    // f and carry of the wave's last point, for the wave after
    double2 nb;   // -b of that point
    double2 f0;   // f of the wave's first point, for the wave before
    double2 up;   // phi of the wave's first point, for the wave before
};

struct Shared {
    WaveEdge edge[TDSE_MAX_WAVES + 1];
    double ring[TDSE_RES_RING + 1][TDSE_MAX_WAVES][5];
    int cur, tried, gate;
};

// a 16-byte table or state row: uniform base, the lane's byte offset, row i of 64 lanes
__device__ inline double2 row(const double2 *base, unsigned lane_off, int i)
{
    const TDSE_GLOBAL char *p = (const TDSE_GLOBAL char *)base + i * 1024;
    const tdse_d2 v = *(const TDSE_GLOBAL tdse_d2 *)(p + lane_off);
    return make_double2(v.x, v.y);
}

// p as a value the compiler knows nothing about: the row addresses of one step are then formed in
// that step, as immediate offsets, and not all kept in registers across the run
__device__ inline const double2 *opaque(const double2 *p)
{
    asm volatile("" : "+s"(p));
    return p;
}

// a + b c, a - b c
__device__ inline double2 cfma(double2 b, double2 c, double2 a)
{
    return make_double2(fma(-b.y, c.y, fma(b.x, c.x, a.x)), fma(b.y, c.x, fma(b.x, c.y, a.y)));
}
__device__ inline double2 cfms(double2 b, double2 c, double2 a)
{
    return make_double2(fma(b.y, c.y, fma(-b.x, c.x, a.x)), fma(-b.y, c.x, fma(-b.x, c.y, a.y)));
}

// lane n of each row of 16 to the whole row
template <int N>
__device__ inline double2 row_bcast(double2 v)
{
    return dpp2_z<0x150 + N>(v);
}

// sum over the wave, in lane 63 (fixed order)
__device__ inline double sum63(double v)
{
    v += dpp_z<kRowShr + 1>(v);
    v += dpp_z<kRowShr + 2>(v);
    v += dpp_z<kRowShr + 4>(v);
    v += dpp_z<kRowShr + 8>(v);
    v += dpp<kRowBcast15, 0xa>(v, 0.0);
    v += dpp<kRowBcast31, 0xc>(v, 0.0);
    return v;
}

// One scan level: z_l += Q_l z_{l -+ D}, Q_l *= Q_{l -+ D} (rows of 16 lanes).
template <int CTRL>
__device__ inline void level(double2 &Q, double2 &z)
{
    const double2 zo = dpp2_z<CTRL>(z), Qo = dpp2_one<CTRL>(Q);
    z = cfma(Q, zo, z);
    Q = cmul(Q, Qo);
}

// The affine maps x_out = z + Q x_in of the lanes' chunks, composed over the lanes before each lane
// (FWD; else those after it) as far as a carry reaches: Q over its own row of 16 lanes, z over the
// row before (after) as well, which hands over its edge lane's total.
template <bool FWD>
__device__ inline void scan_wave(double2 &Q, double2 &z, bool deep)
{
    constexpr int base = FWD ? kRowShr : kRowShl;
    level<base + 1>(Q, z);
    level<base + 2>(Q, z);
    level<base + 4>(Q, z);
    if (deep) level<base + 8>(Q, z);
    const double2 te = dpp2_z<FWD ? kWaveShr1 : kWaveShl1>(z);
    z = cfma(Q, row_bcast<FWD ? 0 : 15>(te), z);  // 0 in the first (last) row
}

// The carry into each lane, Z being what enters the wave: that reaches its first (last) row only.
template <bool FWD>
__device__ inline double2 lane_carry(double2 Q, double2 z, double2 Z, int lane)
{
    const double2 te = dpp2_z<FWD ? kWaveShr1 : kWaveShl1>(z), Qe = dpp2_one<FWD ? kWaveShr1 : kWaveShl1>(Q);
    const bool edge_row = FWD ? lane < 16 : lane >= 48;
    return edge_row ? cfma(Qe, Z, te) : te;
}

// The grid's constants, in scalar registers for the run (read through the geometry they would be
// loaded again after every barrier).
struct StepConst {
    double k36, dt, dx, xmax;
};
__device__ inline StepConst step_const(const TdseGeom &G)
{
    StepConst c = {G.k36, G.dt, G.dx, G.xmax};
    asm volatile("" : "+s"(c.k36), "+s"(c.dt), "+s"(c.dx), "+s"(c.xmax));
    return c;
}

// The state of one lane and what it needs of its grid and window.
template <int C>
struct Lane {
    static constexpr int NL = lds_points(C), NR = C - NL;
    double2 P[C];                    // psi, then r, y, phi in place
    double2 br[NR > 0 ? NR : 1];     // b of points NL .. C - 1
    double2 nQ;                      // product of -b over the chunk (both transfer maps)
    double gl;                       // g of the last point
    unsigned off;                    // byte offset of the lane's first table row
    int j0;                          // grid index of its first point (may lie before the grid)
    bool own;                        // its points belong to this window
};

// b of point i
template <int C>
__device__ inline double2 b_at(const Lane<C> &L, const double2 *lb, int i)
{
    if constexpr (Lane<C>::NR > 0)
        if (i >= Lane<C>::NL) return L.br[i - Lane<C>::NL];
    return lb[i * 64];
}

// byte offset of chunk c's first row in a table or state of tiles of 64 chunks
template <int C>
__device__ inline unsigned row_offset(int c)
{
    return (unsigned)(((c >> 6) * (C * 64) + (c & 63)) * (int)sizeof(double2));
}

// Puts a lane on its chunk of window w: chunks of C points, counted from the table chunk that holds the
// grid's start.  core: the lane's wave holds part of the core table's chunks.
template <int C>
__device__ inline void place_lane(const TdseResident &R, int w, int wave, int lane, Lane<C> &L, int &chunk, bool &core)
{
    const int c0 = w * R.stride, w0 = c0 + wave * 64, c = w0 + lane;
    L.off = row_offset<C>(min(c + R.chunk0, R.chunks));  // (table chunk R.chunks: zeros)
    L.j0 = c * C - R.lead;
    L.own = c >= (w == 0 ? 0 : c0 + R.halo) && (w == R.windows - 1 || c < c0 + R.stride + R.halo);
    chunk = c;
    core = __builtin_amdgcn_readfirstlane(w0 < R.core_chunk0 + R.core_chunks && w0 + 64 > R.core_chunk0);
}

// The lane's b into LDS and registers, with what follows from it.
template <int C>
__device__ inline void load_b(const TdseGeom &G, const TdseResident &R, Lane<C> &L, double2 *lb)
{
    double2 q = make_double2(1.0, 0.0);
    L.gl = row(R.gv, L.off, C - 1).x;
#pragma unroll
    for (int i = 0; i < C; i++) {
        const int j = L.j0 + i;
        double2 b = row(R.b, L.off, i);
        if (j < R.head && j >= 0) b = ld2(R.head_b, j);  // still feels this grid's own left wall
        if (j < 0 || j >= G.nx) b = make_double2(0.0, 0.0);
        if (i < Lane<C>::NL)
            lb[i * 64] = b;
        else
            L.br[i < Lane<C>::NL ? 0 : i - Lane<C>::NL] = b;
        q = cmul(q, make_double2(-b.x, -b.y));
        __builtin_amdgcn_sched_barrier(0);
    }
    L.nQ = q;
}

// The lane's points of a tiled state (zero outside the grid).
template <int C>
__device__ inline void load_tiled(const TdseGeom &G, Lane<C> &L, const double2 *src)
{
#pragma unroll
    for (int i = 0; i < C; i++) {
        const int j = L.j0 + i;
        L.P[i] = j >= 0 && j < G.nx ? ld2(src, tdse_index(j)) : make_double2(0.0, 0.0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Point `index` of a state that leaves the kernel (a row given by the caller, 8-byte aligned).
__device__ inline void put_state(double *dst, long long index, double2 v)
{
    dst[2 * index] = v.x;
    dst[2 * index + 1] = v.y;
}

// Rows of the tables, and of b from LDS, in flight in the first, the last and the passes between.  A
// row costs registers that 32 points a lane do not have: there 3, 6 and 1 / 3 run a step of 16001 points in
// 11.6 us under load, 2 and 6 in 13.4, 3 and 5 in 14, two b rows at the ends in 12.4.  With 16 points 4 rows take 6.0 us
// for 8001 points, 5 or 6 rows 6.4.
constexpr int rows_first(int c) { return c > 24 ? 3 : 4; }
constexpr int rows_last(int c) { return c > 24 ? 6 : 8; }
constexpr int lds_ends(int c) { return c > 24 ? 1 : 2; }
constexpr int lds_between(int c) { return c > 24 ? 3 : 4; }

// Observables over the lane's points (psi in P) that only waves near the atom need: <psi0|psi> and
// PopInt, from the core table: {Re psi0, 1 inside the PopInt window} (and Im psi0 where it is not 0)
// of the chunks that hold either, one row of core_chunks entries per point of a chunk.
template <int C>
__device__ inline void observe_core(const TdseResident &R, const Lane<C> &L, int chunk, Acc &acc)
{
    const int c = chunk - R.core_chunk0, n = R.core_chunks;
    if (c < 0 || c >= n) return;
    const double2 *q = R.core + c;
    constexpr int A = 8;  // rows in flight
    double2 t[A];
#pragma unroll
    for (int i = 0; i < A; i++) t[i] = ld2(q, i * n);
#pragma unroll
    for (int i = 0; i < C; i++) {
        const double2 w = t[i % A], p = L.P[i];
        if (i + A < C) t[i % A] = ld2(q, (i + A) * n);
        acc.pr = fma(p.x, w.x, acc.pr);
        acc.pi = fma(-p.y, w.x, acc.pi);
        acc.pint = fma(fma(p.x, p.x, p.y * p.y), w.y, acc.pint);
        asm volatile("" : "+v"(acc.pr), "+v"(acc.pi), "+v"(acc.pint));
        __builtin_amdgcn_sched_barrier(0);
    }
    if (R.core_im) {
        const double *m = R.core_im + c;
#pragma unroll
        for (int i = 0; i < C; i++) {
            const double v = ld1(m, i * n);
            acc.pr = fma(L.P[i].y, v, acc.pr);
            acc.pi = fma(L.P[i].x, v, acc.pi);
            asm volatile("" : "+v"(acc.pr), "+v"(acc.pi));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// Per-wave sums into a ring entry (lane 63 writes; `add`: onto what earlier windows left there).
__device__ inline void put_observables(Acc &acc, bool own, bool core, bool add, int lane, double *dst)
{
    if (!own) acc = Acc{0.0, 0.0, 0.0, 0.0, 0.0};
    const double pos = sum63(acc.pos), gp = sum63(acc.gp);
    double pr = 0.0, pi = 0.0, pint = 0.0;
    if (core) {
        pr = sum63(acc.pr);
        pi = sum63(acc.pi);
        pint = sum63(acc.pint);
    }
    if (lane == 63) {
        dst[0] = add ? dst[0] + pr : pr;
        dst[1] = add ? dst[1] + pi : pi;
        dst[2] = add ? dst[2] + pint : pint;
        dst[3] = add ? dst[3] + pos : pos;
        dst[4] = add ? dst[4] + gp : gp;
    }
}

// The observables of P alone (the last state of a partial run).
template <int C>
__device__ inline void observe_only(const TdseGeom &G, const Lane<C> &L, int chunk, const double2 *gv, bool core, bool add,
                                    int lane, double *dst)
{
    double s0 = 0.0, s1 = 0.0;
    const TdseResident &R = G.res;
    Acc acc = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (core) observe_core<C>(R, L, chunk, acc);
#pragma unroll
    for (int i = 0; i < C; i++) {
        const double n2 = fma(L.P[i].x, L.P[i].x, L.P[i].y * L.P[i].y);
        s0 += n2;
        s1 = fma((double)i, n2, s1);
        acc.gp = fma(n2, row(gv, L.off, i).y, acc.gp);
        __builtin_amdgcn_sched_barrier(0);
    }
    acc.pos = fma(grid_x(L.j0, G.dx, G.xmax), s0, G.dx * s1);
    put_observables(acc, L.own, core, add, lane, dst);
}

// One time step of the window's points.  ring: this wave's ring entry for the state it starts from.
template <int C>
__device__ inline void step(const TdseResident &R, const StepConst &K, Lane<C> &L, int chunk, const double2 *gv,
                            const double2 *rs, const double2 *lb, Shared &sh, int wave, int lane, double F, bool core,
                            bool deep, bool add, double *ring)
{
    using LN = Lane<C>;
    constexpr int NL = LN::NL, kRows = rows_first(C), kRows4 = rows_last(C), kLds1 = lds_ends(C), kLds = lds_between(C);
    double2 e, rot;  // exp(i F dt x) at the lane's last point; exp(-i F dt dx) - 1, to the point before
    double2 carry;
    {
        // pass 1: observables, r in place, and y from zero
        double2 t[kRows], bq[kLds1];
#pragma unroll
        for (int i = 0; i < kRows && i < C; i++) t[i] = row(gv, L.off, i);
#pragma unroll
        for (int i = 0; i < kLds1 && i < NL; i++) bq[i] = lb[i * 64];
        Acc acc = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (core) observe_core<C>(R, L, chunk, acc);  // a wave that holds part of the atom
        const double2 pl = L.P[C - 1];
        const double2 f0 = make_double2(fma(t[0].x, L.P[0].y, L.P[0].x), fma(-t[0].x, L.P[0].x, L.P[0].y));
        const double2 fl = make_double2(fma(L.gl, pl.y, pl.x), fma(-L.gl, pl.x, pl.y));
        const double2 fR = dpp2_z<kWaveShl1>(f0);
        const double2 fL = dpp2_z<kWaveShr1>(fl);
        double2 dm = make_double2(f0.x - fL.x, f0.y - fL.y), fc = f0;
        double2 y = make_double2(0.0, 0.0), bp = make_double2(0.0, 0.0);
        double s0 = 0.0, s1 = 0.0;
        const double twelve = 12.0;
#pragma unroll
        for (int i = 0; i < C; i++) {
            const double2 p = L.P[i], tt = t[i % kRows];
            const double n2 = fma(p.x, p.x, p.y * p.y);
            s0 += n2;
            s1 = fma((double)i, n2, s1);
            acc.gp = fma(n2, tt.y, acc.gp);
            double2 fp = fR;
            if (i + 1 < C) {
                const double gn = t[(i + 1) % kRows].x;
                fp = make_double2(fma(gn, L.P[i + 1].y, L.P[i + 1].x), fma(-gn, L.P[i + 1].x, L.P[i + 1].y));
            }
            const double2 dp = make_double2(fp.x - fc.x, fp.y - fc.y);
            const double v = fma(twelve, tt.x, K.k36);
            const double2 r = make_double2(fma(v, p.y, fma(twelve, p.x, dp.x - dm.x)), fma(-v, p.x, fma(twelve, p.y, dp.y - dm.y)));
            L.P[i] = r;
            y = i > 0 ? cfms(bp, y, r) : r;
            // summed here, not where the sums are used: that would keep every operand alive
            asm volatile("" : "+v"(y.x), "+v"(y.y), "+v"(s0), "+v"(s1), "+v"(acc.gp));
            dm = dp;
            fc = fp;
            bp = i < NL ? bq[i % kLds1] : b_at<C>(L, lb, i);
            if (i + kRows < C) t[i % kRows] = row(gv, L.off, i + kRows);
            if (i + kLds1 < NL) bq[i % kLds1] = lb[(i + kLds1) * 64];
            __builtin_amdgcn_sched_barrier(0);
        }
        // what the chunk hands to the next lane's first row: -b y of its last point
        const double2 nb = make_double2(-bp.x, -bp.y);
        double2 Q = L.nQ, z = cmul(nb, y);
        scan_wave<true>(Q, z, deep);
        WaveEdge &E = sh.edge[wave];
        if (lane == 63) {
            E.a = make_double2(fl.x + z.x, fl.y + z.y);
            E.nb = nb;
        }
        if (lane == 0) E.f0 = f0;
        // while the other waves arrive: the phase factors and the observables' sums
        {
            const double Fdt = F * K.dt, th = Fdt * grid_x(L.j0 + C - 1, K.dx, K.xmax), d = Fdt * K.dx;
            sincos_wide(th, &e.y, &e.x);
            double hs, hc;
            sincos_wide(-0.5 * d, &hs, &hc);
            rot = make_double2(-2.0 * hs * hs, 2.0 * hs * hc);
        }
        acc.pos = fma(grid_x(L.j0, K.dx, K.xmax), s0, K.dx * s1);
        put_observables(acc, L.own, core, add, lane, ring);
        lds_barrier();
        // from the wave before: its last point's f, and its carry corrected for the f of this wave's
        // first point, which its last row was still missing
        double2 Z = make_double2(0.0, 0.0);
        if (wave > 0) {
            const WaveEdge &B = sh.edge[wave - 1];
            Z = cfma(B.nb, E.f0, B.a);
        }
        carry = lane_carry<true>(Q, z, Z, lane);
        // likewise this wave's last row misses the f of the wave after (0 after the last)
        const double2 fn = sh.edge[wave + 1].f0;
        L.P[C - 1].x += lane == 63 ? fn.x : 0.0;
        L.P[C - 1].y += lane == 63 ? fn.y : 0.0;
    }
    // pass 2: y from the true carry, in place
    {
        double2 bq[kLds];
#pragma unroll
        for (int i = 0; i < kLds && i < NL; i++) bq[i] = lb[i * 64];
        double2 y = make_double2(L.P[0].x + carry.x, L.P[0].y + carry.y);
        L.P[0] = y;
#pragma unroll
        for (int i = 1; i < C; i++) {
            const double2 b = i - 1 < NL ? bq[(i - 1) % kLds] : b_at<C>(L, lb, i - 1);
            y = cfms(b, y, L.P[i]);
            asm volatile("" : "+v"(y.x), "+v"(y.y));
            L.P[i] = y;
            if (i - 1 + kLds < NL) bq[(i - 1) % kLds] = lb[(i - 1 + kLds) * 64];
            if (i % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        }
    }
    // pass 3: phi from zero, for the carry to the lane before
    double2 s[kRows4], bq[kLds];
    {
#pragma unroll
        for (int i = 0; i < kLds; i++)
            if (NL - 1 - i >= 0) bq[(NL - 1 - i) % kLds] = lb[(NL - 1 - i) * 64];
        double2 u = make_double2(0.0, 0.0);
#pragma unroll
        for (int i = C - 1; i >= 0; i--) {
            const double2 b = i < NL ? bq[i % kLds] : b_at<C>(L, lb, i);
            u = cmul(b, make_double2(L.P[i].x - u.x, L.P[i].y - u.y));
            asm volatile("" : "+v"(u.x), "+v"(u.y));
            if (i < NL && i - kLds >= 0) bq[i % kLds] = lb[(i - kLds) * 64];
            if (i % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        }
        double2 Q = L.nQ;
        scan_wave<false>(Q, u, deep);
        if (lane == 0) sh.edge[wave].up = u;
        // the rows of the last pass, in flight across the barrier
#pragma unroll
        for (int i = 0; i < kRows4; i++)
            if (C - 1 - i >= 0) s[(C - 1 - i) % kRows4] = row(rs, L.off, C - 1 - i);
#pragma unroll
        for (int i = 0; i < kLds1; i++)
            if (NL - 1 - i >= 0) bq[(NL - 1 - i) % kLds1] = lb[(NL - 1 - i) * 64];
        lds_barrier();
        carry = lane_carry<false>(Q, u, sh.edge[wave + 1].up, lane);
    }
    // pass 4: phi from the true carry, psi' = phi / (1 + i g), the phase
    {
        double2 u = carry;
#pragma unroll
        for (int i = C - 1; i >= 0; i--) {
            const double2 b = i < NL ? bq[i % kLds1] : b_at<C>(L, lb, i);
            u = cmul(b, make_double2(L.P[i].x - u.x, L.P[i].y - u.y));
            L.P[i] = cmul(e, cmul(s[i % kRows4], u));
            asm volatile("" : "+v"(u.x), "+v"(u.y), "+v"(L.P[i].x), "+v"(L.P[i].y));
            if (i > 0) e = cfma(e, rot, e);  // e + e rot: the rotation's own rounding would change |e| by C steps of it
            if (i < NL && i - kLds1 >= 0) bq[i % kLds1] = lb[(i - kLds1) * 64];
            if (i - kRows4 >= 0) s[i % kRows4] = row(rs, L.off, i - kRows4);
            if (i % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// The whole run of one instance by the waves of a workgroup.
template <int C>
__device__ inline void run_instance(const TdseGeom &G, const TdseInst &I, double2 *work, long long work_stride, double2 *lds,
                                    Shared &sh)
{
    using LN = Lane<C>;
    const TdseResident &R = G.res;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nw = R.waves;
    const bool live = wave < nw;
    const bool deep = R.reach > 8 * C;
    const bool windows = R.windows > 1;
    const int k_start = I.k0, k_stop = I.n_run > 0 ? I.k0 + I.n_run : I.n_steps;
    const bool final_obs = I.src && k_stop < I.n_steps;
    int i_snap = 0;
    int cur = 0;  // multi-window states: the buffer that holds the current state
    // the field is 0 up to and including the first sign change of in_field (prop.c:125-134)
    if (threadIdx.x == 0) sh.gate = I.pregated ? -1 : I.n_steps;
    __syncthreads();
    for (int m0 = 0; !I.pregated && m0 < k_stop; m0 += blockDim.x) {
        const int m = m0 + (int)threadIdx.x;
        if (m < k_stop && I.field[m] * I.field[m + 1] <= 0.0) atomicMin(&sh.gate, m);
        __syncthreads();
        const bool found = sh.gate < I.n_steps;
        __syncthreads();
        if (found) break;
    }
    const int gate = __builtin_amdgcn_readfirstlane(sh.gate);
    auto field = [&](int m) { return m <= gate ? 0.0 : I.field[m]; };
    if (threadIdx.x == 0) {
        const double2 zero = make_double2(0.0, 0.0);
        sh.edge[nw].f0 = zero;  // past the last wave: the wall, or a window's end
        sh.edge[nw].up = zero;
        if (I.src && k_start == 0) {
            I.src[0] = 0.0;
            I.ptot[0] = 1.0;
            I.pint[0] = G.pint0;
            I.expv[0] = 0.0;
            if (I.efield) I.efield[0] = 0.0;
        }
    }
    __syncthreads();
    double2 *const lb = lds + wave * (64 * LN::NL) + lane;  // this lane's b: point i at lb[i * 64]
    LN L;
    const StepConst K = step_const(G);
    const double2 *const gv = R.gv, *const rs = R.s;
    bool core = false;
    int chunk = 0;
    auto place = [&](int w) { place_lane<C>(R, w, wave, lane, L, chunk, core); };
    // chunk c's rows in a window buffer
    auto buf_off = [&](int w) { return row_offset<C>(w * R.stride + wave * 64 + lane); };

    for (int k = k_start; k < k_stop;) {
        int nb = min(R.steps, k_stop - k);
        if (I.save) nb = min(nb, I.save_every - (k - k_start) % I.save_every);
        // prop.c:248-255: snapshot row i_snap gets psi after step m when m % every == 0
        const int snap_step = (k + I.snap_every - 1) / I.snap_every * I.snap_every;
        const bool snaps = I.snap && i_snap < I.n_snap - 1;
        if (snaps) nb = min(nb, snap_step + 1 - k);
        // who gets the state the block ends with: a save (tiled), a snapshot, and after the last step (prop.c:256-262) the
        // last row, if every earlier one was used, and the final state
        double2 *const save = I.save && (k + nb - k_start) % I.save_every == 0
                                  ? I.save + (long long)((k + nb - k_start) / I.save_every - 1) * G.npad
                                  : nullptr;
        double *row_to[3] = {nullptr, nullptr, nullptr};
        if (snaps && k + nb == snap_step + 1) row_to[0] = I.snap + 2ll * G.nx * i_snap++;
        if (k + nb == k_stop) {
            if (I.snap && i_snap == I.n_snap - 1) row_to[1] = I.snap + 2ll * G.nx * i_snap;
            row_to[2] = I.psi_final;
        }
        for (int w = 0; w < R.windows; w++) {
            const bool add = w > 0;
            if (live && (windows || k == k_start)) {
                place(w);
                load_b<C>(G, R, L, lb);
                if (k == k_start) {
                    load_tiled<C>(G, L, I.psi_init ? I.psi_init : G.psi0);
                } else {
                    const double2 *src = work + cur * work_stride;
                    const unsigned o = buf_off(w);
#pragma unroll
                    for (int i = 0; i < C; i++) L.P[i] = row(src, o, i);
                }
            }
            // the block's fields, one per lane
            const double fields = lane < nb ? field(k + lane) : 0.0;
            for (int t = 0; t < nb; t++) {
                if (live) {
                    step<C>(R, K, L, chunk, opaque(gv), opaque(rs), lb, sh, wave, lane, readlane(fields, t), core, deep, add,
                            sh.ring[t][wave]);
                } else {
                    lds_barrier();
                    lds_barrier();
                }
            }
            if (live) {
                if (final_obs && k + nb == k_stop) observe_only<C>(G, L, chunk, gv, core, add, lane, sh.ring[nb][wave]);
                if (windows) {
                    double2 *dst = work + (cur ^ 1) * work_stride;
                    const unsigned o = buf_off(w);
                    if (L.own) {
#pragma unroll
                        for (int i = 0; i < C; i++) st2((double2 *)((char *)dst + o), 64 * i, L.P[i]);
                    }
                } else {
                    for (int m = 0; m < 4; m++) {
                        double *dst = m < 3 ? row_to[m] : reinterpret_cast<double *>(save);
                        if (!dst) continue;
#pragma unroll
                        for (int i = 0; i < C; i++) {
                            const int j = L.j0 + i;
                            if (j >= 0 && j < G.nx) put_state(dst, m < 3 ? j : tdse_index(j), L.P[i]);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
            }
        }
        __syncthreads();  // the ring is complete, a window buffer is in memory
        if (windows) {
            cur ^= 1;
            const double2 *src = work + cur * work_stride;
            for (int m = 0; m < 4; m++) {
                double *dst = m < 3 ? row_to[m] : reinterpret_cast<double *>(save);
                if (!dst) continue;
                for (int j = threadIdx.x; j < G.nx; j += blockDim.x) {
                    const int q = j + R.lead, c = q / C;
                    put_state(dst, m < 3 ? j : tdse_index(j), src[(long long)(c >> 6) * (C * 64) + (q % C) * 64 + (c & 63)]);
                }
            }
        }
        // entries k .. k + nb - 1 of the outputs (and k + nb, the last state of a partial run)
        if (I.src && threadIdx.x <= (unsigned)nb) {
            const int t = threadIdx.x, idx = k + t;
            if (idx > k_start && (t < nb || (final_obs && idx == k_stop))) {
                double sum[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
                for (int w = 0; w < nw; w++)
                    for (int q = 0; q < 5; q++) sum[q] += sh.ring[t][w][q];
                const double F = field(idx - 1);  // the step that produced the state
                I.src[idx] = -sum[4] + F;
                I.ptot[idx] = sum[0] * sum[0] + sum[1] * sum[1];
                I.pint[idx] = sum[2];
                I.expv[idx] = sum[3];
                if (I.efield) I.efield[idx] = F;
            }
        }
        __syncthreads();  // the ring has been read
        k += nb;
    }
}

} // namespace

// Persistent workgroups: instances from the per-XCD queues as in tdse_propagate_kernel, each by
// the chunk length of its geometry.  Dynamic LDS: lds_points(C) complex doubles per lane.
__global__ void __launch_bounds__(64 * TDSE_MAX_WAVES, TDSE_RES_WAVES_PER_SIMD)
tdse_resident_kernel(const TdseGeom *__restrict__ geoms, const TdseInst *__restrict__ insts, const int *__restrict__ order,
                     TdseQueues queues, int *counter, double2 *work, long long work_stride)
{
    __shared__ Shared sh;
    extern __shared__ double2 lds[];
    if (threadIdx.x == 0) sh.tried = 0;
    for (;;) {
        if (threadIdx.x == 0) sh.cur = next_instance(queues, counter, sh.tried);
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(sh.cur);
        __syncthreads();
        if (t < 0) break;
        const TdseInst &I = insts[order[t]];
        const TdseGeom &G = geoms[I.geom];
        double2 *const buf = work + 2 * (long long)blockIdx.x * work_stride;
        switch (G.res.chunk) {
        case 16: run_instance<16>(G, I, buf, work_stride, lds, sh); break;
        case 24: run_instance<24>(G, I, buf, work_stride, lds, sh); break;
        case 32: run_instance<32>(G, I, buf, work_stride, lds, sh); break;
        default: break;
        }
    }
}

// ---- one instance alone -------------------------------------------------------------------
// The windows of one instance side by side, a workgroup each, `nb` steps per launch: with the
// instance on one compute unit a step takes as long as its waves need for all points; with many
// small windows it takes a window's latency, at the price of halos that are solved again.

namespace {

// The observables of entries k .. k + nb - 1 from the windows' sums, part[t][window][5].
__device__ inline void store_entries(const TdseInst &I, const double *part, int windows, int k, int nb)
{
    const int t = threadIdx.x, idx = k + t;
    if (t >= nb || idx == 0) return;
    double sum[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int w = 0; w < windows; w++)
        for (int q = 0; q < 5; q++) sum[q] += part[(t * windows + w) * 5 + q];
    const double F = I.field[idx - 1];
    I.src[idx] = -sum[4] + F;
    I.ptot[idx] = sum[0] * sum[0] + sum[1] * sum[1];
    I.pint[idx] = sum[2];
    I.expv[idx] = sum[3];
    if (I.efield) I.efield[idx] = F;
}

template <int C>
__device__ inline void run_window(const TdseGeom &G, const TdseInst &I, const TdseResident &R, int k, int nb,
                                  const double2 *src, double2 *dst, double *part, double2 *lds, Shared &sh)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, w = blockIdx.x;
    const bool deep = R.reach > 8 * C;
    double2 *const lb = lds + wave * (64 * Lane<C>::NL) + lane;
    Lane<C> L;
    const StepConst K = step_const(G);
    const double2 *const gv = R.gv, *const rs = R.s;
    bool core = false;
    int chunk = 0;
    if (threadIdx.x == 0) {
        sh.edge[R.waves].f0 = make_double2(0.0, 0.0);
        sh.edge[R.waves].up = make_double2(0.0, 0.0);
    }
    place_lane<C>(R, w, wave, lane, L, chunk, core);
    load_b<C>(G, R, L, lb);
    const bool on_grid = L.j0 < G.nx;
    if (src) {
        const unsigned o = row_offset<C>(on_grid ? chunk : 0);
#pragma unroll
        for (int i = 0; i < C; i++) {
            const double2 v = row(src, o, i);
            L.P[i] = make_double2(on_grid ? v.x : 0.0, on_grid ? v.y : 0.0);
        }
    } else {
        load_tiled<C>(G, L, G.psi0);
    }
    const double fields = lane < nb ? I.field[k + lane] : 0.0;
    __syncthreads();
    for (int t = 0; t < nb; t++)
        step<C>(R, K, L, chunk, opaque(gv), opaque(rs), lb, sh, wave, lane, readlane(fields, t), core, deep, false,
                sh.ring[t][wave]);
    if (L.own && on_grid) {
        const unsigned o = row_offset<C>(chunk);
#pragma unroll
        for (int i = 0; i < C; i++) st2((double2 *)((char *)dst + o), 64 * i, L.P[i]);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 5 * nb; e += blockDim.x) {
        double sum = 0.0;
        for (int v = 0; v < R.waves; v++) sum += sh.ring[e / 5][v][e % 5];
        part[((e / 5) * R.windows + w) * 5 + e % 5] = sum;
    }
}

} // namespace

// Steps k .. k + nb - 1 of one instance (gated field) over R.windows workgroups, from src (null: psi0)
// to dst, both in lane-tile order; one more workgroup writes the entries of the launch before
// (nb_prev steps) from its sums.  part: 2 x TDSE_RES_RING x windows x 5 doubles, by the parity of
// `launch`.
__global__ void __launch_bounds__(64 * TDSE_ONE_WAVES)
tdse_window_kernel(const TdseGeom *__restrict__ geom, const TdseInst *__restrict__ inst, TdseResident R, int k, int nb, int nb_prev,
                   int launch, const double2 *src, double2 *dst, double *part)
{
    __shared__ Shared sh;
    extern __shared__ double2 lds[];
    const TdseGeom &G = *geom;
    const TdseInst &I = *inst;
    const long long half = (long long)TDSE_RES_RING * R.windows * 5;
    if ((int)blockIdx.x == R.windows) {
        if (k == 0 && threadIdx.x == 0) {
            I.src[0] = 0.0;
            I.ptot[0] = 1.0;
            I.pint[0] = G.pint0;
            I.expv[0] = 0.0;
            if (I.efield) I.efield[0] = 0.0;
        }
        store_entries(I, part + ((launch - 1) & 1) * half, R.windows, k - nb_prev, nb_prev);
        return;
    }
    double *const mine = part + (launch & 1) * half;
    if (R.chunk == 16)
        run_window<16>(G, I, R, k, nb, src, dst, mine, lds, sh);
    else
        run_window<24>(G, I, R, k, nb, src, dst, mine, lds, sh);
}

// The entries of the run's last launch.
__global__ void tdse_window_finish_kernel(const TdseInst *inst, int windows, int k, int nb, int launch, const double *part)
{
    store_entries(*inst, part + (long long)(launch & 1) * TDSE_RES_RING * windows * 5, windows, k, nb);
}

// A state in lane-tile order (chunks of C points, the grid `lead` points into chunk 0) in natural
// order, interleaved re, im.
__global__ void tdse_window_untile_kernel(const double2 *psi, int C, int lead, int nx, double *dst)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nx) return;
    const int q = j + lead, c = q / C;
    const double2 v = psi[(long long)(c >> 6) * (C * 64) + (q % C) * 64 + (c & 63)];
    dst[2 * j] = v.x;
    dst[2 * j + 1] = v.y;
}

namespace {

// A sum of two doubles, for the tables: their rounding is the same in every step of a run, so its
// effect grows with the steps (a norm drift), where the rounding of the steps themselves averages out.
struct Two {
    double h, l;
};
__device__ inline Two two_sum(double a, double b)
{
    const double s = a + b, t = s - a;
    return {s, (a - (s - t)) + (b - t)};
}
__device__ inline Two norm2(double h, double l)
{
    const double s = h + l;
    return {s, l - (s - h)};
}
__device__ inline Two add2(Two a, Two b)
{
    const Two s = two_sum(a.h, b.h);
    return norm2(s.h, s.l + (a.l + b.l));
}
__device__ inline Two mul2(Two a, Two b)
{
    const double p = a.h * b.h;
    return norm2(p, fma(a.h, b.h, -p) + fma(a.h, b.l, a.l * b.h));
}
__device__ inline Two neg2(Two a) { return {-a.h, -a.l}; }
__device__ inline Two recip2(Two a)
{
    const double q = 1.0 / a.h;
    const Two r = add2({1.0, 0.0}, neg2(mul2({q, 0.0}, a)));  // 1 - q a
    return add2({q, 0.0}, mul2({q, 0.0}, r));
}
// 1 / (1 + i g) and c = (10 + i d) / (1 + i g), d = 10 g + K as the steps' right-hand side has it
// (12 g + K rounded, less 2 g): the two sides of a step are then exact conjugates, which is what
// conserves the norm (with the unrounded 10 g + K here, PopTot drifted by 2e-13 in 1300 steps, ten
// times as much)
__device__ inline void diagonal2(double g, double k36, Two (&s)[2], Two (&c)[2])
{
    const Two G = {g, 0.0}, w = recip2(add2({1.0, 0.0}, mul2(G, G)));
    s[0] = w;
    s[1] = neg2(mul2(G, w));
    const Two d = two_sum(fma(12.0, g, k36), -2.0 * g);
    c[0] = mul2(w, add2({10.0, 0.0}, mul2(d, G)));
    c[1] = mul2(w, add2(d, neg2(mul2({10.0, 0.0}, G))));
}
// b_j = 1 / (c_j - b_{j-1})
__device__ inline void pivot2(const Two (&c)[2], Two (&b)[2])
{
    const Two x = add2(c[0], neg2(b[0])), y = add2(c[1], neg2(b[1]));
    const Two n = recip2(add2(mul2(x, x), mul2(y, y)));
    b[0] = mul2(x, n);
    b[1] = neg2(mul2(y, n));
}

} // namespace

// The pivots b_j = 1 / (c_j - b_{j-1}) forget where they started by rho^2 a point, so any run of points can
// start from the double ones, 1e-16 off, a few points earlier: after `warm` points that is below 1e-20.
__device__ inline void pivots_before(const double *g, const double2 *ib, double k36, int j0, int warm, Two (&b)[2])
{
    const int start = max(0, j0 - warm);
    b[0] = b[1] = {0.0, 0.0};
    if (start > 0) {
        const long long t = tdse_index(start - 1);
        const double gj = g[t];
        const double2 v = ib[t];
        b[0] = {fma(-gj, v.y, v.x), 0.0};
        b[1] = {fma(gj, v.x, v.y), 0.0};
    }
    Two s[2], c[2];
    for (int j = start; j < j0; j++) {
        diagonal2(g[tdse_index(j)], k36, s, c);
        pivot2(c, b);
    }
}

// The resident tables of one lattice (or one grid): chunk c, row i of C points at
// (c >> 6) * 64 C + i * 64 + (c & 63), from the tiled g, V' and 1/beta of nx points; zero past them.  One
// thread per TDSE_RES_GROUP points (a chain of double-double divisions: 24 of them 14 us).
__global__ void tdse_resident_tables_kernel(const double *g, const double *dpot, const double2 *ib, int nx, double k36, int C,
                                            int chunks, int warm, double2 *gv, double2 *s, double2 *b)
{
    const int j0 = (blockIdx.x * blockDim.x + threadIdx.x) * TDSE_RES_GROUP;
    if (j0 >= chunks * C) return;
    Two sj[2], cj[2], bj[2];
    if (j0 < nx) pivots_before(g, ib, k36, j0, warm, bj);
    for (int j = j0; j < j0 + TDSE_RES_GROUP; j++) {
        double2 vg = make_double2(0.0, 0.0), vs = vg, vb = vg;
        if (j < nx) {
            const long long t = tdse_index(j);
            diagonal2(g[t], k36, sj, cj);
            pivot2(cj, bj);
            vg = make_double2(g[t], dpot[t]);
            vs = make_double2(sj[0].h, sj[1].h);
            vb = make_double2(bj[0].h, bj[1].h);
        }
        const int c = j / C, i = j % C;
        const long long q = ((long long)(c >> 6) * C + i) * 64 + (c & 63);
        gv[q] = vg;
        s[q] = vs;
        b[q] = vb;
    }
}

// Per geometry (job blockIdx.y), the core table: entry (i, c) is point (core_chunk0 + c) C + i - lead, {Re psi0,
// 1 in the PopInt window [lo, hi]} and Im psi0, zero outside the grid; and b of its first `head` points,
// which feel its own left wall where the lattice's do not.
__global__ void tdse_resident_core_kernel(const ResidentJob *jobs)
{
    const ResidentJob J = jobs[blockIdx.y];
    const int m = J.C * J.n;
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < m; q += gridDim.x * blockDim.x) {
        const int j = J.first + (q % J.n) * J.C + q / J.n;
        const bool on = j >= 0 && j < J.nx;
        J.core[q] = make_double2(on ? J.psi0[j].x : 0.0, on && j >= J.lo && j <= J.hi ? 1.0 : 0.0);
        J.im[q] = on ? J.psi0[j].y : 0.0;
    }
    const int j0 = (blockIdx.x * blockDim.x + threadIdx.x) * TDSE_RES_GROUP;
    if (j0 >= J.head) return;
    Two s[2], c[2], b[2];
    pivots_before(J.g, J.ib, J.k36, j0, J.warm, b);
    for (int j = j0; j < min(j0 + TDSE_RES_GROUP, J.head); j++) {
        diagonal2(J.g[tdse_index(j)], J.k36, s, c);
        pivot2(c, b);
        J.head_b[j] = make_double2(b[0].h, b[1].h);
    }
}
