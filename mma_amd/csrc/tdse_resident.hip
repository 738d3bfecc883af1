// Crank-Nicolson propagation with the wavefunction resident on the chip (1DTDSE/sources/prop.c:24-347).
//
// tdse_propagate.hip streams psi through HBM once per step (or two): it runs at the memory's rate
// and, per point, spends more instructions on scans than on the solve.  A grid of up to 16353
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
//     y_j   = r_j - b_{j-1} y_{j-1}            4 FMA a point, or w_j = b_j y_j = b_j (r_j - w_{j-1}), 6
//     phi_j = w_j - b_j phi_{j+1}              4
//     psi'_j = phi_j / (1 + i g_j)             4, from a table
// Both recurrences run twice around a scan over the lanes: once from zero for the carry that leaves
// the lane's chunk (as y), once from the true carry (as w).  Carries decay by rho < 1 per point, below 1e-17 after
// `reach` points, so a scan looks back only as far as that (3 or 4 levels within rows of 16 lanes, one
// step from the row before), a wave takes its carry from the one wave next to it, and windows
// overlap by `reach` points per step.
//
// Where the operands live: psi (r, w and psi in turn) in 4 C registers; b of up to 18 points a lane in LDS (512
// lanes x 18 x 16 B = 144 KB), of the others in registers, with 32 points from L2 once a step (far_points); g, V' and
// 1/(1 + i g) come from L2, 32 B a point and step, shared by all instances of a grid.  HBM is idle: the
// FP64 units bound the step (about 46 + 300 / C of their instructions a point, 72 % of the time; the rest is
// waits for LDS and L2 and the two barriers).  No step spills a register: with 22 reloads of spilled values a
// step of 16001 points took 11.7 us, each reload waiting for the table rows in flight before it as well.
//
// Measured under load, 512 instances: a step of 16001 points takes 9.7 us a compute unit (11.7 before the waves
// around the atom had a loop of their own, the sine and cosine that all lanes share were evaluated once
// for eight steps, and the spills were gone), of 12001 7.3 (7.9), of 8001 5.6 (6.0), of 6001 4.0 (5.2, one
// workgroup a CU); 3.6 to 4.2e11 points a second on the chip, where the streaming kernels reach 1.75e11.
//
// r_j takes the differences of f first: they cancel exactly, where f_{j-1} + f_{j+1} + (10 - i (10 g_j + K)) psi_j
// rounds three terms of 2 |g| |psi| each (|g| = 75 to 300) for a result of 12 |psi|.  That noise made two solves of one run with
// different lanes differ by 1.1e-12 on the dipole; now by 2e-13.
//
// Observables (prop.c:293-347) of the state a step starts from are summed in its first pass, per
// wave in a fixed order, and collected in LDS for up to TDSE_RES_RING steps.
#include <type_traits>

#include "sincos_reduced.h"
#include "tdse_internal.h"
#include "tdse_wave.h"

namespace {

using namespace tdse;

// What a workgroup of nw waves shares, in dynamic LDS (tdse_res_lds()).
struct Shared {
    TdseWaveEdge *edge; // nw + 1
    double *ring;       // TDSE_RES_RING + 1 entries of the observables' sums, [nw][5]
    double2 *b;         // the lanes' share of b
    int nw;
    __device__ double *sums(int t, int wave) const { return ring + (t * nw + wave) * 5; }
};
__device__ inline Shared shared_memory(double2 *lds)
{
    Shared sh;
    sh.nw = blockDim.x >> 6;
    sh.edge = reinterpret_cast<TdseWaveEdge *>(lds);
    sh.ring = reinterpret_cast<double *>(sh.edge + sh.nw + 1);
    sh.b = lds + tdse_res_shared(sh.nw) / sizeof(double2);
    return sh;
}
struct Queue {
    int cur, tried, gate;
};

// a 16-byte table or state row: uniform base, the lane's byte offset, row i of 64 lanes
__device__ inline double2 row(const double2 *base, unsigned lane_off, int i)
{
    const TDSE_GLOBAL char *p = (const TDSE_GLOBAL char *)base + i * 1024;
    const tdse_d2 v = *(const TDSE_GLOBAL tdse_d2 *)(p + lane_off);
    return make_double2(v.x, v.y);
}

// r with its fields to be read again from here on, and not kept in registers across what came before
template <typename T>
__device__ inline const T &fresh(const T &r)
{
    typedef const T __attribute__((address_space(4))) const_t;
    const unsigned long long a = reinterpret_cast<unsigned long long>(&r);
    unsigned lo = __builtin_amdgcn_readfirstlane((int)a), hi = __builtin_amdgcn_readfirstlane((int)(a >> 32));
    asm volatile("" : "+s"(lo), "+s"(hi));
    return *(const T *)(const_t *)((unsigned long long)hi << 32 | lo);
}

// a value that all lanes agree on, as one that might differ: branches on it keep the registers' allocation in
// one piece (scalar ones cut it, and b was spilled around them)
__device__ inline int per_lane(int v)
{
    int l;
    asm volatile("v_mov_b32 %0, %1" : "=v"(l) : "s"(v));
    return l;
}

// v as a value the compiler knows nothing about: what follows from it is formed where it is used
__device__ inline int opaque_lane(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// this lane's number, formed anew: kept across a step it would be spilled, and wait for its reload
__device__ inline int lane_id()
{
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(l));
    return l;
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

// With 32 points a lane's registers do not hold psi, b and what the first pass works with.  That pass
// needs no b, so those that LDS does not hold are read from the table again after it, and arrive while y runs
// over the points before (7 B a point and step more from L2).  What is left in registers the compiler spills, and
// each pass waits for the reloads: with the phases of one stage of this kernel a step of 16001 points took 11.1 us
// with all 14, 11.4 with 12, 14 to 18 with 4.
constexpr int far_points(int c) { return c > 24 ? c - tdse_res_lds_points(c) : 0; }

// The state of one lane and what it needs of its grid and window.
template <int C>
struct Lane {
    static constexpr int NL = tdse_res_lds_points(C), NF = far_points(C), NR = C - NL;
    double2 P[C];                    // psi, then r, w, psi in place
    double2 br[NR > 0 ? NR : 1];     // b of points NL .. C - 1
    double2 nQ;                      // product of -b over the chunk (both transfer maps); with 32 points in LDS, lb[64 NL]
    unsigned off;                    // byte offset of the lane's first table row
    int j0;                          // grid index of its first point (may lie before the grid)
    bool own;                        // its points belong to this window
    const TDSE_GLOBAL tdse_d2 *far;  // b of point NL + i at [64 i], where they are not kept all the time
};

// The lane's table rows in registers, for a kernel with one wave per SIMD, which has twice the registers
// and no other wave that computes while it waits: they are the same in every step (one instance of 16001
// points, 4416 steps: 20.1 -> 18.0 ms).  Empty otherwise.
template <int C, bool HOLD>
struct Held {
    double2 gv[HOLD ? C : 1], s[HOLD ? C : 1], b[HOLD ? C : 1];
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
__device__ inline void place_lane(const TdseResident &R, int w, int wave, int lane, Lane<C> &L, int &chunk, int &core)
{
    const int c0 = w * R.stride, w0 = c0 + wave * 64, c = w0 + lane;
    L.off = row_offset<C>(min(c + R.chunk0, R.chunks));  // (table chunk R.chunks: zeros)
    L.j0 = c * C - R.lead;
    L.own = c >= (w == 0 ? 0 : c0 + R.halo) && (w == R.windows - 1 || c < c0 + R.stride + R.halo);
    chunk = c;
    core = __builtin_amdgcn_readfirstlane(w0 < R.core_chunk0 + R.core_chunks && w0 + 64 > R.core_chunk0);
}

// b of point i, where the table (of a lattice that several grids share) has `b`
template <int C>
__device__ inline double2 own_b(const TdseResident &R, const Lane<C> &L, int i, double2 b)
{
    const int j = L.j0 + i;
    if (j < R.head && j >= 0) b = ld2(R.head_b, j);  // still feels this grid's own left wall
    return j < 0 || j >= R.nx ? make_double2(0.0, 0.0) : b;
}

// The lane's b into LDS and registers, and the product of -b.  OWN: some differ from the table's.
template <int C, bool OWN>
__device__ inline double2 load_rows_b(const TdseResident &R, Lane<C> &L, double2 *lb)
{
    using LN = Lane<C>;
    double2 q = make_double2(1.0, 0.0);
    // rows in flight: one at a time, a window's factors took longer to arrive than one of its steps (256
    // instances of 32001 points, two windows, 445 steps: 17.7 ms, with 8 16.2)
    constexpr int kGroup = 8;
#pragma unroll
    for (int i0 = 0; i0 < C; i0 += kGroup) {
        double2 t[kGroup];
#pragma unroll
        for (int m = 0; m < kGroup; m++) t[m] = row(R.b, L.off, i0 + m);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < kGroup; m++) {
            const int i = i0 + m;
            const double2 b = OWN ? own_b<C>(R, L, i, t[m]) : t[m];
            if (i < LN::NL)
                lb[i * 64] = b;
            else
                L.br[i < LN::NL ? 0 : i - LN::NL] = b;
            q = cmul(q, make_double2(-b.x, -b.y));
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    return q;
}

// The lane's b with what follows from it.  Only the waves at the ends of a grid that reads another one's table
// have points whose b is not the table's.
template <int C>
__device__ inline void load_b(const TdseResident &R, Lane<C> &L, double2 *lb, double2 *store)
{
    using LN = Lane<C>;
    const bool own = R.head > 0 && (L.j0 < R.head || L.j0 + C > R.nx);
    const double2 q = __any(own) ? load_rows_b<C, true>(R, L, lb) : load_rows_b<C, false>(R, L, lb);
    if (C > 24)
        lb[64 * LN::NL] = q;
    else
        L.nQ = q;
    if constexpr (LN::NF > 0) {
        // from the table, unless the lane's b are its own
        const double2 *const p = own ? store : R.b + L.off / sizeof(double2) + 64 * LN::NL;
        L.far = (const TDSE_GLOBAL tdse_d2 *)p;
        if (own) {
#pragma unroll
            for (int i = 0; i < LN::NF; i++) st2(store, 64 * i, L.br[i]);
        }
    }
}

// Those of the lane's b that the first pass did not keep.
template <int C>
__device__ inline void fetch_far(Lane<C> &L)
{
    using LN = Lane<C>;
    if constexpr (LN::NF == 0) return;
    unsigned long long at = reinterpret_cast<unsigned long long>(L.far);
    asm volatile("" : "+v"(at));  // the rows' addresses are formed here, not kept (and spilled) across the steps
    const TDSE_GLOBAL tdse_d2 *const far = reinterpret_cast<const TDSE_GLOBAL tdse_d2 *>(at);
#pragma unroll
    for (int i = C - LN::NF; i < C; i++) {
        const tdse_d2 v = far[64 * (i - LN::NL)];
        L.br[i < LN::NL ? 0 : i - LN::NL] = make_double2(v.x, v.y);
    }
}

// v[q] of lane t of each four to v[t] of its lane q.
__device__ inline void transpose_quad(double2 (&v)[4])
{
    const int lane = lane_id();
    const bool odd = lane & 1, high = lane & 2;
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
        const double2 got = dpp2_z<kQuadXor1>(make_double2(odd ? v[q].x : v[q + 1].x, odd ? v[q].y : v[q + 1].y));
        v[q] = make_double2(odd ? got.x : v[q].x, odd ? got.y : v[q].y);
        v[q + 1] = make_double2(odd ? v[q + 1].x : got.x, odd ? v[q + 1].y : got.y);
    }
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const double2 got = dpp2_z<kQuadXor2>(make_double2(high ? v[q].x : v[q + 2].x, high ? v[q].y : v[q + 2].y));
        v[q] = make_double2(high ? got.x : v[q].x, high ? got.y : v[q].y);
        v[q + 2] = make_double2(high ? v[q + 2].x : got.x, high ? v[q + 2].y : got.y);
    }
}

// A lane's points in a tiled state.  Where the grid starts on one of the lane's chunks of 8 points (always, but for
// members of a lattice), a row of 8-point chunks costs one instruction: from one offset per chunk, the rows
// lie at immediate offsets.  A launch of one step executes each path once, so what counts is that all of them
// stay in the instruction cache that two compute units share (64 KiB, the two loops over the steps take 34 of it).
// Rows in turn, and within a row the lane's C / 8 chunks, which are neighbours: a line is done with
// before the next.  With four of them, four lanes take 64 bytes each time, and then exchange them: as 16 bytes
// apiece a state of 16001 points took 18.7 us to leave a compute unit (4096 instances), so 7.6.
template <int C>
struct TiledLane {
    static constexpr int K = C / TDSE_CHUNK;
    static constexpr bool kQuads = K == 4;
    unsigned at[K];        // byte offset of row 4 of each chunk
    int chunk[K];          // which these are
    int j0;                // as in Lane
    bool aligned, inside;  // for the whole wave: as above; all points on the grid
};
template <int C>
__device__ inline TiledLane<C> tiled_lane(const TdseGeom &G, const Lane<C> &L)
{
    typedef TiledLane<C> T;
    T t;
    t.j0 = opaque_lane(L.j0);
    t.aligned = __builtin_amdgcn_readfirstlane(t.j0) % TDSE_CHUNK == 0;  // (the same for every lane)
    t.inside = __all(t.j0 >= 0 && t.j0 + C <= G.nx);
    const int of4 = lane_id() & 3;
#pragma unroll
    for (int q = 0; q < T::K; q++) {
        t.chunk[q] = (t.j0 >> 3) + (T::kQuads ? 4 * (q - of4) + of4 : q);
        // (chunks past the grid: the first of those, which exists)
        t.at[q] = (unsigned)tdse_chunk_base(min(t.chunk[q], G.nchunks)) * (unsigned)sizeof(double2) + 4 * 1024;
    }
    return t;
}
template <typename T>
__device__ inline T *tiled_row(T *base, unsigned at, int r)
{
    typedef typename std::conditional<std::is_const<T>::value, const TDSE_GLOBAL char, TDSE_GLOBAL char>::type byte;
    return (T *)((byte *)base + at + (r - 4) * 1024);
}

// The lane's points of a tiled state (zero outside the grid), all in flight together.
template <int C>
__device__ inline void load_tiled(const TdseGeom &G, Lane<C> &L, const double2 *src)
{
    typedef TiledLane<C> T;
    const T t = tiled_lane<C>(G, L);
    if (t.aligned) {
#pragma unroll
        for (int r = 0; r < TDSE_CHUNK; r++)
#pragma unroll
            for (int q = 0; q < T::K; q++) L.P[TDSE_CHUNK * q + r] = ld2(tiled_row(src, t.at[q], r), 0);
        if constexpr (T::kQuads) {
#pragma unroll
            for (int r = 0; r < TDSE_CHUNK; r++) {
                double2 v[4];
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = L.P[TDSE_CHUNK * q + r];
                transpose_quad(v);
#pragma unroll
                for (int q = 0; q < 4; q++) L.P[TDSE_CHUNK * q + r] = v[q];
            }
        }
    } else {
        const int last = G.nx - 1;
#pragma unroll
        for (int i = 0; i < C; i++) {
            L.P[i] = ld2(src, tdse_index((unsigned)min(max(t.j0 + i, 0), last)));
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (t.inside) return;
#pragma unroll
    for (int i = 0; i < C; i++) {
        const bool on = (unsigned)(t.j0 + i) < (unsigned)G.nx;
        L.P[i] = make_double2(on ? L.P[i].x : 0.0, on ? L.P[i].y : 0.0);
    }
}

// The points of the lanes with `own` into a tiled state (those on the grid).
template <int C>
__device__ inline void store_tiled(const TdseGeom &G, const Lane<C> &L, double2 *dst, bool own)
{
    typedef TiledLane<C> T;
    T t = tiled_lane<C>(G, L);
    const unsigned long long owners = __ballot(own);
    t.inside = t.inside && owners == ~0ull;
    bool mine[T::K];  // whether the lane's entries of chunk[q] are its own, or those of lane q of its four
#pragma unroll
    for (int q = 0; q < T::K; q++) mine[q] = T::kQuads ? owners >> ((lane_id() & ~3) + q) & 1 : own;
    if (t.aligned) {
#pragma unroll
        for (int r = 0; r < TDSE_CHUNK; r++) {
            double2 v[T::K];
#pragma unroll
            for (int q = 0; q < T::K; q++) v[q] = L.P[TDSE_CHUNK * q + r];
            if constexpr (T::kQuads) transpose_quad(v);
#pragma unroll
            for (int q = 0; q < T::K; q++)
                if (t.inside || (mine[q] && (unsigned)(TDSE_CHUNK * t.chunk[q] + r) < (unsigned)G.nx))
                    st2(tiled_row(dst, t.at[q], r), 0, v[q]);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll
        for (int i = 0; i < C; i++) {
            const int j = t.j0 + i;
            if (own && (unsigned)j < (unsigned)G.nx) st2(dst, tdse_index((unsigned)j), L.P[i]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// Where point j of the grid lies in the windows' buffer.
template <int C>
__device__ inline long long window_index(const TdseResident &R, int j)
{
    const int q = j + R.lead, c = q / C;
    return (long long)(c >> 6) * (C * 64) + (q % C) * 64 + (c & 63);
}

// A state from the windows' buffer into a tiled one, by the workgroup: neighbouring threads write neighbouring
// entries, each several of them, all in flight (in the grid's order, one entry of 8 bytes twice at a time, a state of
// 32001 points took 50 us).
template <int C>
__device__ inline void copy_tiled(const TdseGeom &G, const double2 *src, double2 *dst)
{
    constexpr int kGroup = 8;
    const int n = (G.nchunks + 63) / 64 * TDSE_TILE;
    for (int e0 = threadIdx.x; e0 < n; e0 += kGroup * blockDim.x) {
        double2 v[kGroup];
#pragma unroll
        for (int m = 0; m < kGroup; m++) {
            const int e = e0 + m * blockDim.x, j = ((e >> 9) * 64 + (e & 63)) * TDSE_CHUNK + (e >> 6) % TDSE_CHUNK;
            v[m] = ld2(src, window_index<C>(G.res, min(j, G.nx - 1)));
        }
#pragma unroll
        for (int m = 0; m < kGroup; m++) {
            const int e = e0 + m * blockDim.x, j = ((e >> 9) * 64 + (e & 63)) * TDSE_CHUNK + (e >> 6) % TDSE_CHUNK;
            if (j < G.nx) st2(dst, TDSE_TILE + e, v[m]);
        }
    }
}

// Likewise those of each window's points that it left out of a tiled state.
template <int C>
__device__ inline void copy_left_out(const TdseGeom &G, const double2 *src, double2 *dst)
{
    constexpr int kGroup = 8;
    const TdseResident &R = G.res;
    const int each = R.halo * C, n = (R.windows - 1) * each;
    for (int e0 = threadIdx.x; e0 < n; e0 += kGroup * blockDim.x) {
        double2 v[kGroup];
        int j[kGroup];
#pragma unroll
        for (int m = 0; m < kGroup; m++) {
            const int e = min(e0 + m * (int)blockDim.x, n - 1), w = 1 + e / each, i = e % each;
            j[m] = min((w * R.stride + i % R.halo) * C - R.lead + i / R.halo, G.nx - 1);
            v[m] = ld2(src, window_index<C>(R, j[m]));
        }
#pragma unroll
        for (int m = 0; m < kGroup; m++) st2(dst, tdse_index((unsigned)j[m]), v[m]);
    }
}

// Point `index` of a state that leaves the kernel (a row given by the caller, 8-byte aligned).
__device__ inline void put_state(double *dst, long long index, double2 v)
{
    dst[2 * index] = v.x;
    dst[2 * index + 1] = v.y;
}

// Rows of the tables, of the core table, and of b from LDS in flight in the first, the last and the passes
// between.  A row costs registers that 32 points a lane do not have; more of them gain nothing for 16 and 24
// (6 or 8 rows in the first pass, 12 in the last, 4 and 6 of LDS: within 1 % or slower).
constexpr int rows_first(int c) { return c > 24 ? 3 : 4; }
constexpr int rows_last(int c) { return c > 24 ? 4 : 8; }
constexpr int rows_core(int c) { return c > 24 ? 2 : 4; }
constexpr int lds_ends(int c) { return c > 24 ? 1 : 2; }
constexpr int lds_between(int c) { return c > 24 ? 2 : 4; }

// Sine and cosine with the coefficients from memory, into scalar registers: as literals they are moved to
// vector registers before the loop over the steps, where no register is free, and spilled.
__constant__ double kCoef[17] = SINCOS_COEFFICIENTS;
__device__ inline void sincos_lean(double x, double *s, double *c)
{
    typedef const double __attribute__((address_space(4))) coef_t;
    coef_t *k = (coef_t *)kCoef;
    asm volatile("" : "+s"(k));
    sincos_wide(x, s, c, k);
}

// Offset of the lane's rows in the core table: {Re psi0, 1 inside the PopInt window} of the chunks that hold
// either, in tiles as the other tables, then a chunk of zeros for the other lanes of a wave.
template <int C>
__device__ inline unsigned core_offset(const TdseResident &R, const Lane<C> &L)
{
    const int c = (L.j0 + R.lead) / C - R.core_chunk0;
    return row_offset<C>(c < 0 || c > R.core_chunks ? R.core_chunks : c);
}

// The part of Im psi0 in a lane's sums over <psi0|psi>, where there is one.
template <int C>
__device__ inline void core_im(const TdseResident &R, const Lane<C> &L, unsigned off, Acc &acc)
{
    const double *m = R.core_im + off / sizeof(double2);
#pragma unroll
    for (int i = 0; i < C; i++) {
        const double v = ld1(m, 64 * i);
        acc.pr = fma(L.P[i].y, v, acc.pr);
        acc.pi = fma(L.P[i].x, v, acc.pi);
        asm volatile("" : "+v"(acc.pr), "+v"(acc.pi));
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Per-wave sums into a ring entry (lane 63 writes; `add`: onto what earlier windows left there).
__device__ inline void put_observables(Acc &acc, bool own, int core, bool add, int lane, double *dst)
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
        const double v[5] = {pr, pi, pint, pos, gp};
        const int more = per_lane(add);
#pragma unroll
        for (int q = 0; q < 5; q++) {
            const double old = dst[q];
            dst[q] = more ? old + v[q] : v[q];
        }
    }
}

// The observables of P alone (the last state of a partial run), its rows eight at a time.
template <int C>
__device__ inline void observe_only(const TdseGeom &G, const Lane<C> &L, const double2 *gv, int core, bool add,
                                    int lane, double *dst)
{
    constexpr int kGroup = 8;
    double s0 = 0.0, s1 = 0.0;
    const TdseResident &R = G.res;
    Acc acc = {0.0, 0.0, 0.0, 0.0, 0.0};
    const unsigned off = core_offset<C>(R, L);
#pragma unroll
    for (int i0 = 0; i0 < C; i0 += kGroup) {
        double2 t[kGroup];
#pragma unroll
        for (int m = 0; m < kGroup; m++) t[m] = row(gv, L.off, i0 + m);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < kGroup; m++) {
            const double2 p = L.P[i0 + m];
            const double n2 = fma(p.x, p.x, p.y * p.y);
            s0 += n2;
            s1 = fma((double)(i0 + m), n2, s1);
            acc.gp = fma(n2, t[m].y, acc.gp);
        }
        // formed here: put off to the end, the sums would keep every row (in scratch memory)
        asm volatile("" : "+v"(s0), "+v"(s1), "+v"(acc.gp));
        __builtin_amdgcn_sched_barrier(0);
        if (core) {
#pragma unroll
            for (int m = 0; m < kGroup; m++) t[m] = row(R.core, off, i0 + m);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < kGroup; m++) {
                const double2 p = L.P[i0 + m];
                acc.pr = fma(p.x, t[m].x, acc.pr);
                acc.pi = fma(-p.y, t[m].x, acc.pi);
                acc.pint = fma(fma(p.x, p.x, p.y * p.y), t[m].y, acc.pint);
            }
            asm volatile("" : "+v"(acc.pr), "+v"(acc.pi), "+v"(acc.pint));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (core && R.core_im) core_im<C>(R, L, off, acc);
    acc.pos = fma(grid_x(L.j0, G.dx, G.xmax), s0, G.dx * s1);
    put_observables(acc, L.own, core, add, lane, dst);
}

// Observables of the state, and the right-hand side r in its place.  CORE: the wave holds part of the atom.
// What only the wave's edge lanes need later (f of its first and last point) goes to E at once.
template <int C, bool CORE, bool HOLD>
__device__ inline void first_pass(const TdseResident &R, const StepConst &K, Lane<C> &L, const double2 *gv,
                                  const Held<C, HOLD> &H, Acc &acc,
                                  TdseWaveEdge &E)
{
    constexpr int kRows = rows_first(C), kCore = CORE ? rows_core(C) : 1;  // rows in flight
    const double2 *const cq = opaque(R.core);
    auto g_row = [&](int i) {
        if constexpr (HOLD)
            return H.gv[i];
        else
            return row(gv, L.off, i);
    };
    const unsigned coff = CORE ? core_offset<C>(R, L) : 0;
    double2 t[kRows], q[kCore];
    const double gl = g_row(C - 1).x;
#pragma unroll
    for (int i = 0; i < kRows; i++) t[i] = g_row(i);
    if (CORE) {
#pragma unroll
        for (int i = 0; i < kCore; i++) q[i] = row(cq, coff, i);
        if (R.core_im) core_im<C>(R, L, coff, acc);
    }
    const double2 pl = L.P[C - 1];
    const double2 f0 = make_double2(fma(t[0].x, L.P[0].y, L.P[0].x), fma(-t[0].x, L.P[0].x, L.P[0].y));
    const double2 fl = make_double2(fma(gl, pl.y, pl.x), fma(-gl, pl.x, pl.y));
    const int lane = lane_id();
    if (lane == 0) E.f0 = f0;
    if (lane == 63) E.a = fl;
    const double2 fR = dpp2_z<kWaveShl1>(f0);
    const double2 fL = dpp2_z<kWaveShr1>(fl);
    double2 dm = make_double2(f0.x - fL.x, f0.y - fL.y), fc = f0;
    double s0 = 0.0, s1 = 0.0;
    const double twelve = 12.0;
#pragma unroll
    for (int i = 0; i < C; i++) {
        const double2 p = L.P[i], tt = t[i % kRows];
        const double n2 = fma(p.x, p.x, p.y * p.y);
        s0 += n2;
        s1 = fma((double)i, n2, s1);
        acc.gp = fma(n2, tt.y, acc.gp);
        if (CORE) {
            const double2 w = q[i % kCore];
            acc.pr = fma(p.x, w.x, acc.pr);
            acc.pi = fma(-p.y, w.x, acc.pi);
            acc.pint = fma(n2, w.y, acc.pint);
            asm volatile("" : "+v"(acc.pr), "+v"(acc.pi), "+v"(acc.pint));
            if (i + kCore < C) q[i % kCore] = row(cq, coff, i + kCore);
        }
        double2 fp = fR;
        if (i + 1 < C) {
            const double gn = t[(i + 1) % kRows].x;
            fp = make_double2(fma(gn, L.P[i + 1].y, L.P[i + 1].x), fma(-gn, L.P[i + 1].x, L.P[i + 1].y));
        }
        const double2 dp = make_double2(fp.x - fc.x, fp.y - fc.y);
        const double v = fma(twelve, tt.x, K.k36);
        L.P[i] = make_double2(fma(v, p.y, fma(twelve, p.x, dp.x - dm.x)), fma(-v, p.x, fma(twelve, p.y, dp.y - dm.y)));
        // formed here, not where they are used: that would keep every operand alive
        asm volatile("" : "+v"(s0), "+v"(s1), "+v"(acc.gp), "+v"(L.P[i].x), "+v"(L.P[i].y));
        dm = dp;
        fc = fp;
        if (i + kRows < C) t[i % kRows] = g_row(i + kRows);
        __builtin_amdgcn_sched_barrier(0);
    }
    acc.pos = fma(grid_x(L.j0, K.dx, K.xmax), s0, K.dx * s1);
}

// One time step of the window's points.  rot: exp(-i F dt dx) - 1, from a point's phase to the one before.
// ring: this wave's ring entry for the state it starts from.
template <int C, bool CORE, bool HOLD>
__device__ inline void step(const TdseResident &R, const StepConst &K, Lane<C> &L, const double2 *gv,
                            const double2 *rs, const double2 *lb, const Held<C, HOLD> &H, const Shared &sh, int wave, double F, double2 rot, bool deep,
                            bool add, double *ring)
{
    using LN = Lane<C>;
    constexpr int NL = LN::NL, kRows4 = rows_last(C), kLds1 = lds_ends(C), kLds = lds_between(C);
    auto b_row = [&](int i) {
        if constexpr (HOLD)
            return H.b[i];
        else
            return b_at<C>(L, lb, i);
    };
    auto s_row = [&](int i) {
        if constexpr (HOLD)
            return H.s[i];
        else
            return row(rs, L.off, i);
    };
    double2 e;  // exp(i F dt x) at the lane's last point
    double2 carry;
    Acc acc = {0.0, 0.0, 0.0, 0.0, 0.0};
    TdseWaveEdge &E = sh.edge[wave];
    first_pass<C, CORE, HOLD>(R, K, L, gv, H, acc, E);
    __builtin_amdgcn_sched_barrier(0);
    fetch_far<C>(L);
    __builtin_amdgcn_sched_barrier(0);
    {
        // y from zero
        double2 bq[kLds];
#pragma unroll
        for (int i = 0; i < kLds && i < NL; i++) bq[i] = b_row(i);
        double2 y = make_double2(0.0, 0.0), b = y;
#pragma unroll
        for (int i = 0; i < C; i++) {
            y = i > 0 ? cfms(b, y, L.P[i]) : L.P[i];
            asm volatile("" : "+v"(y.x), "+v"(y.y));
            b = i < NL ? bq[i % kLds] : b_row(i);
            if (i + kLds < NL) bq[i % kLds] = b_row(i + kLds);
            if (i % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        }
        // what the chunk hands to the next lane's first row: -b y of its last point
        const double2 nb = make_double2(-b.x, -b.y);
        double2 Q = C > 24 ? lb[64 * NL] : L.nQ, z = cmul(nb, y);
        scan_wave<true>(Q, z, deep);
        const int lane = lane_id();
        if (lane == 63) {
            E.a = make_double2(E.a.x + z.x, E.a.y + z.y);
            E.nb = nb;
        }
        // while the other waves arrive: the phase factors and the observables' sums
        {
            const double th = F * K.dt * grid_x(L.j0 + C - 1, K.dx, K.xmax);
            sincos_lean(th, &e.y, &e.x);
        }
        put_observables(acc, L.own, CORE, add, lane, ring);
        lds_barrier();
        // from the wave before: its last point's f, and its carry corrected for the f of this wave's
        // first point, which its last row was still missing
        double2 Z = make_double2(0.0, 0.0);
        if (per_lane(wave) > 0) {
            const TdseWaveEdge &B = sh.edge[wave - 1];
            Z = cfma(B.nb, E.f0, B.a);
        }
        carry = lane_carry<true>(Q, z, Z, lane);
        // likewise this wave's last row misses the f of the wave after (0 after the last)
        const double2 fn = sh.edge[wave + 1].f0;
        L.P[C - 1].x += lane == 63 ? fn.x : 0.0;
        L.P[C - 1].y += lane == 63 ? fn.y : 0.0;
    }
    // w from the true carry, in place
    {
        double2 bq[kLds];
#pragma unroll
        for (int i = 0; i < kLds && i < NL; i++) bq[i] = b_row(i);
        double2 w = make_double2(-carry.x, -carry.y);
#pragma unroll
        for (int i = 0; i < C; i++) {
            const double2 b = i < NL ? bq[i % kLds] : b_row(i);
            w = cmul(b, make_double2(L.P[i].x - w.x, L.P[i].y - w.y));
            asm volatile("" : "+v"(w.x), "+v"(w.y));
            L.P[i] = w;
            if (i + kLds < NL) bq[i % kLds] = b_row(i + kLds);
            if (i % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        }
    }
    // phi from zero, for the carry to the lane before
    double2 s[kRows4], bq[kLds];
    {
        constexpr int i0 = NL < C - 1 ? NL - 1 : C - 2;  // the first b from LDS
#pragma unroll
        for (int i = 0; i < kLds; i++)
            if (i0 - i >= 0) bq[(i0 - i) % kLds] = b_row(i0 - i);
        double2 u = L.P[C - 1];
#pragma unroll
        for (int i = C - 2; i >= 0; i--) {
            const double2 b = i < NL ? bq[i % kLds] : b_row(i);
            u = cfms(b, u, L.P[i]);
            asm volatile("" : "+v"(u.x), "+v"(u.y));
            if (i < NL && i - kLds >= 0) bq[i % kLds] = b_row(i - kLds);
            if (i % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        }
        double2 Q = C > 24 ? lb[64 * NL] : L.nQ;
        scan_wave<false>(Q, u, deep);
        const int lane = lane_id();
        if (lane == 0) sh.edge[wave].up = u;
        // the rows of the last pass, in flight across the barrier
#pragma unroll
        for (int i = 0; i < kRows4; i++)
            if (C - 1 - i >= 0) s[(C - 1 - i) % kRows4] = s_row(C - 1 - i);
#pragma unroll
        for (int i = 0; i < kLds1; i++)
            if (NL - 1 - i >= 0) bq[(NL - 1 - i) % kLds1] = b_row(NL - 1 - i);
        lds_barrier();
        carry = lane_carry<false>(Q, u, sh.edge[wave + 1].up, lane);
    }
    // phi from the true carry, psi' = phi / (1 + i g), the phase
    {
        double2 u = carry;
#pragma unroll
        for (int i = C - 1; i >= 0; i--) {
            const double2 b = i < NL ? bq[i % kLds1] : b_row(i);
            u = cfms(b, u, L.P[i]);
            L.P[i] = cmul(e, cmul(s[i % kRows4], u));
            asm volatile("" : "+v"(u.x), "+v"(u.y), "+v"(L.P[i].x), "+v"(L.P[i].y));
            if (i > 0) e = cfma(e, rot, e);  // e + e rot: the rotation's own rounding would change |e| by C steps of it
            if (i < NL && i - kLds1 >= 0) bq[i % kLds1] = b_row(i - kLds1);
            if (i - kRows4 >= 0) s[i % kRows4] = s_row(i - kRows4);
            if (i % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// What a run of steps does with its observables: entry t of the ring is sample k + t.
struct Entries {
    const TdseInst *inst;
    int k, k_start, gate, waves;
    bool flush;  // while the steps run (one window)
};

// Samples e.k + t, t0 <= t < t1, from the waves' sums, one per lane of this wave.
__device__ inline void write_entries(const Entries &e, const Shared &sh, int t0, int t1, int mask)
{
    const TdseInst &I = fresh(*e.inst);
    const int t = t0 + lane_id(), idx = e.k + t;
    if (!I.src || t >= t1 || idx <= e.k_start) return;
    double sum[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int w = 0; w < e.waves; w++)
        for (int q = 0; q < 5; q++) sum[q] += sh.sums(t & mask, w)[q];
    const double F = idx - 1 <= e.gate ? 0.0 : I.field[idx - 1];  // the step that produced the state
    I.src[idx] = -sum[4] + F;
    I.ptot[idx] = sum[0] * sum[0] + sum[1] * sum[1];
    I.pint[idx] = sum[2];
    I.expv[idx] = sum[3];
    if (I.efield) I.efield[idx] = F;
}

// nb steps of the window's points.  The ring's halves are written out by the first wave in turn, while the others go
// on: they come back to a half after more barriers than that takes.  The waves that hold part of the atom
// run a loop of their own: with both in one, either the registers or the loads in flight of the others pay for
// what only those need.
template <int C, bool CORE, bool HOLD>
__device__ inline void run_steps(const TdseResident &R, const StepConst &K, Lane<C> &L, const double2 *lb,
                                 const Held<C, HOLD> &H, const Shared &sh,
                                 int wave, const Entries &e, int nb, bool deep, bool add)
{
    constexpr int kHalf = TDSE_RES_RING / 2;
    for (int t0 = 0; t0 < nb; t0 += kHalf) {
        const int m = t0 + lane_id(), t1 = min(nb, t0 + kHalf);
        const double fields = m < t1 && e.k + m > e.gate ? fresh(*e.inst).field[e.k + m] : 0.0;
        double hs, hc;
        sincos_lean(-0.5 * (fields * K.dt * K.dx), &hs, &hc);
        const double2 rots = make_double2(-2.0 * hs * hs, 2.0 * hs * hc);
        for (int t = t0; t < t1; t++)
            step<C, CORE, HOLD>(R, K, L, opaque(R.gv), opaque(R.s), lb, H, sh, wave, readlane(fields, t - t0), readlane2(rots, t - t0), deep,
                          add, sh.sums(t % TDSE_RES_RING, wave));
        if (e.flush && t1 - t0 == kHalf && per_lane(wave) == 0) write_entries(e, sh, t0, t1, TDSE_RES_RING - 1);
    }
}

// The whole run of one instance by the waves of a workgroup.  WINDOWS: over several windows, whose states are loaded
// and stored for every block of steps; else the state stays in registers.  With both in one loop the state was a value that may
// come from either, and went through scratch memory (more than its own 256 KB, each way) in every block.
template <int C, bool WINDOWS>
__device__ inline void run_instance(const TdseGeom &geom, const TdseInst &inst, double2 *work, long long work_stride, double2 *far,
                                    const Shared &sh, Queue &queue)
{
    using LN = Lane<C>;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nw = geom.res.waves;
    const bool live = per_lane(wave) < nw;
    const bool deep = geom.res.reach > 8 * C;
    const int k_start = inst.k0, k_stop = inst.n_run > 0 ? inst.k0 + inst.n_run : inst.n_steps;
    int i_snap = 0;
    int cur = 0;  // multi-window states: the buffer that holds the current state
    {
        const TdseGeom &G = geom;
        const TdseInst &I = inst;
        // the field is 0 up to and including the first sign change of in_field (prop.c:125-134)
        if (threadIdx.x == 0) queue.gate = I.pregated ? -1 : I.n_steps;
        __syncthreads();
        for (int m0 = 0; !I.pregated && m0 < k_stop; m0 += blockDim.x) {
            const int m = m0 + (int)threadIdx.x;
            if (m < k_stop && I.field[m] * I.field[m + 1] <= 0.0) atomicMin(&queue.gate, m);
            __syncthreads();
            const bool found = queue.gate < I.n_steps;
            __syncthreads();
            if (found) break;
        }
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
    }
    const int gate = __builtin_amdgcn_readfirstlane(queue.gate);
    double2 *const lb = sh.b + wave * (64 * tdse_res_lds_rows(C)) + lane;  // this lane's b: point i at lb[i * 64]
    const StepConst K = step_const(fresh(geom));
    // prop.c:248-255: snapshot row i_snap gets psi after step m when m % every == 0; the next such step
    auto snap_step = [&](const TdseInst &I, int k) {
        return I.snap && i_snap < I.n_snap - 1 ? (k + I.snap_every - 1) / I.snap_every * I.snap_every : 0x7ffffffe;
    };

    // the lane's chunk of window w, its b and its points: of the start state (src null) or of the windows' buffer
    auto load_window = [&](LN &L, int &chunk, int &core, int w, const double2 *src) {
        const TdseGeom &G = fresh(geom);
        place_lane<C>(G.res, w, wave, lane, L, chunk, core);
        load_b<C>(G.res, L, lb, far + wave * tdse_res_far(1, C) + lane);
        if (!src) {
            const TdseInst &I = fresh(inst);
            load_tiled<C>(G, L, I.psi_init ? I.psi_init : G.psi0);
        } else {
            const unsigned o = row_offset<C>(chunk);  // (a window's chunks lie in its buffer as in the grid)
#pragma unroll
            for (int i = 0; i < C; i++) L.P[i] = row(src, o, i);
        }
    };
    // nb steps from k of a window's points, and the observables of the last state of a partial run
    auto run_window = [&](LN &L, int core, bool add, int k, int nb) {
        const Entries entries = {&inst, k, k_start, gate, nw, !WINDOWS};
        if (per_lane(core))
            run_steps<C, true, false>(fresh(geom).res, K, L, lb, {}, sh, wave, entries, nb, deep, add);
        else
            run_steps<C, false, false>(fresh(geom).res, K, L, lb, {}, sh, wave, entries, nb, deep, add);
        const TdseGeom &G = fresh(geom);
        const TdseInst &I = fresh(inst);
        if (I.src && k_stop < I.n_steps && k + nb == k_stop)
            observe_only<C>(G, L, G.res.gv, core, add, lane, sh.sums(WINDOWS ? nb : nb % TDSE_RES_RING, wave));
    };
    auto other_waves_steps = [&](int nb) {
        for (int t = 0; t < nb; t++) {
            lds_barrier();
            lds_barrier();
        }
    };
    LN one;
    int one_chunk = 0, one_core = 0;
    if (!WINDOWS && live) load_window(one, one_chunk, one_core, 0, nullptr);

    for (int k = k_start; k < k_stop;) {
        int nb;
        {
            const TdseInst &I = fresh(inst);
            nb = WINDOWS ? min(fresh(geom).res.steps, k_stop - k) : k_stop - k;
            if (I.save) nb = min(nb, I.save_every - (k - k_start) % I.save_every);
            nb = min(nb, snap_step(I, k) + 1 - k);
        }
        // who gets the state the block ends with: a save (tiled), a snapshot, and after the last step (prop.c:256-262) the
        // last row, if every earlier one was used, and the final state
        double *to[4];
        auto receivers = [&] {
            const TdseInst &I = fresh(inst);
            const TdseGeom &G = fresh(geom);
            to[0] = I.save && (k + nb - k_start) % I.save_every == 0
                        ? reinterpret_cast<double *>(I.save + (long long)((k + nb - k_start) / I.save_every - 1) * G.npad)
                        : nullptr;
            const bool at_snap = k + nb == snap_step(I, k) + 1;
            to[1] = at_snap ? I.snap + 2ll * G.nx * i_snap : nullptr;
            to[2] = k + nb == k_stop && I.snap && i_snap + at_snap == I.n_snap - 1 ? I.snap + 2ll * G.nx * (i_snap + at_snap)
                                                                               : nullptr;
            to[3] = k + nb == k_stop ? I.psi_final : nullptr;
            return at_snap;
        };
        bool at_snap = false;
        if constexpr (WINDOWS) {
            // A run's last block goes to its save at once, and not through the windows' buffer.  The save may be the
            // state the run starts from: in its only block a window leaves out what the next has yet to load, the `halo`
            // chunks past the next one's first.
            receivers();
            double2 *const direct = k + nb == k_stop && !to[1] && !to[2] && !to[3] ? reinterpret_cast<double2 *>(to[0]) : nullptr;
            for (int w = 0; w < fresh(geom).res.windows; w++) {
                if (!live) {
                    other_waves_steps(nb);
                    continue;
                }
                LN L;
                int chunk, core;
                load_window(L, chunk, core, w, k == k_start ? nullptr : work + cur * work_stride);
                run_window(L, core, w > 0, k, nb);
                const TdseGeom &G = fresh(geom);
                const bool later = k == k_start && w < G.res.windows - 1 && chunk >= (w + 1) * G.res.stride;
                if (direct) store_tiled<C>(G, L, direct, L.own && !later);
                if (L.own && (later || !direct)) {
                    double2 *dst = work + (cur ^ 1) * work_stride;
                    const unsigned o = row_offset<C>(chunk);
#pragma unroll
                    for (int i = 0; i < C; i++) st2((double2 *)((char *)dst + o), 64 * i, L.P[i]);
                }
            }
            __syncthreads();  // the ring is complete, the windows' buffer is in memory
            const TdseGeom &G = fresh(geom);
            cur ^= 1;
            const double2 *src = work + cur * work_stride;
            if (direct && k == k_start) copy_left_out<C>(G, src, direct);
            if (!direct) at_snap = receivers();
            if (!direct && to[0]) copy_tiled<C>(G, src, reinterpret_cast<double2 *>(to[0]));
            for (int m = 1; m < 4 && !direct; m++) {
                double *dst = to[m];
                if (!dst) continue;
                for (int j = threadIdx.x; j < G.nx; j += blockDim.x) put_state(dst, j, src[window_index<C>(G.res, j)]);
            }
        } else {
            if (live)
                run_window(one, one_core, false, k, nb);
            else
                other_waves_steps(nb);
            at_snap = receivers();
            if (live) {
                const TdseGeom &G = fresh(geom);
                if (to[0]) store_tiled<C>(G, one, reinterpret_cast<double2 *>(to[0]), true);
                for (int m = 1; m < 4; m++) {
                    double *dst = to[m];
                    if (!dst) continue;
                    const int j0 = opaque_lane(one.j0);
#pragma unroll
                    for (int i = 0; i < C; i++) {
                        const int j = j0 + i;
                        if (j >= 0 && j < G.nx) put_state(dst, j, one.P[i]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            __syncthreads();  // the ring is complete
        }
        // what is left in the ring, and the last state of a partial run
        if (wave == 0) {
            const Entries entries = {&inst, k, k_start, gate, nw, false};
            const int from = WINDOWS ? 0 : nb / (TDSE_RES_RING / 2) * (TDSE_RES_RING / 2);
            const bool last = k + nb == k_stop && k_stop < fresh(inst).n_steps;
            write_entries(entries, sh, from, nb + last, WINDOWS ? 31 : TDSE_RES_RING - 1);
        }
        __syncthreads();  // the ring has been read
        i_snap += at_snap;
        k += nb;
    }
}

} // namespace

// Persistent workgroups: instances from the per-XCD queues as in tdse_propagate_kernel, each by
// the chunk length of its geometry.  Dynamic LDS: tdse_res_lds().
__global__ void __launch_bounds__(64 * TDSE_MAX_WAVES, TDSE_RES_WAVES_PER_SIMD)
tdse_resident_kernel(const TdseGeom *__restrict__ geoms, const TdseInst *__restrict__ insts, const int *__restrict__ order,
                     TdseQueues queues, int *counter, double2 *work, long long work_stride)
{
    __shared__ Queue queue;
    extern __shared__ double2 lds[];
    const Shared sh = shared_memory(lds);
    if (threadIdx.x == 0) queue.tried = 0;
    for (;;) {
        if (threadIdx.x == 0) queue.cur = next_instance(queues, counter, queue.tried);
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(queue.cur);
        __syncthreads();
        if (t < 0) break;
        const TdseInst &I = insts[__builtin_amdgcn_readfirstlane(order[t])];
        const TdseGeom &G = geoms[__builtin_amdgcn_readfirstlane(I.geom)];
        // two states of the windows, and the lanes' own b that registers do not hold
        double2 *const buf = work + (long long)blockIdx.x * work_stride;
        const long long states = (work_stride - tdse_res_far(TDSE_MAX_WAVES, 32)) / 2;
        auto run = [&](auto c, auto windows) {
            run_instance<decltype(c)::value, decltype(windows)::value>(G, I, buf, states, buf + 2 * states, sh, queue);
        };
        const std::true_type several{};
        const std::false_type one{};
        switch (G.res.chunk * 2 + (G.res.windows > 1)) {
        case 32: run(std::integral_constant<int, 16>{}, one); break;
        case 33: run(std::integral_constant<int, 16>{}, several); break;
        case 48: run(std::integral_constant<int, 24>{}, one); break;
        case 49: run(std::integral_constant<int, 24>{}, several); break;
        case 64: run(std::integral_constant<int, 32>{}, one); break;
        case 65: run(std::integral_constant<int, 32>{}, several); break;
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
                                  const double2 *src, double2 *dst, double *part, const Shared &sh)
{
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, w = blockIdx.x;
    const bool deep = R.reach > 8 * C;
    double2 *const lb = sh.b + wave * (64 * tdse_res_lds_rows(C)) + lane;
    Lane<C> L;
    const StepConst K = step_const(G);
    const double2 *const gv = R.gv;
    int core = 0;
    int chunk = 0;
    if (threadIdx.x == 0) {
        sh.edge[R.waves].f0 = make_double2(0.0, 0.0);
        sh.edge[R.waves].up = make_double2(0.0, 0.0);
    }
    place_lane<C>(R, w, wave, lane, L, chunk, core);
    load_b<C>(R, L, lb, nullptr);
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
    constexpr bool kHold = C <= 16;  // 24 points' rows do not fit 512 registers
    Held<C, kHold> H;
#pragma unroll
    for (int i = 0; kHold && i < C; i++) {
        H.gv[i] = row(R.gv, L.off, i);
        H.s[i] = row(R.s, L.off, i);
        H.b[i] = b_at<C>(L, lb, i);
    }
    const Entries entries = {&I, k, 0, -1, R.waves, false};
    __syncthreads();
    if (per_lane(core))
        run_steps<C, true, kHold>(R, K, L, lb, H, sh, wave, entries, nb, deep, false);
    else
        run_steps<C, false, kHold>(R, K, L, lb, H, sh, wave, entries, nb, deep, false);
    if (L.own && on_grid) {
        const unsigned o = row_offset<C>(chunk);
#pragma unroll
        for (int i = 0; i < C; i++) st2((double2 *)((char *)dst + o), 64 * i, L.P[i]);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 5 * nb; e += blockDim.x) {
        double sum = 0.0;
        for (int v = 0; v < R.waves; v++) sum += sh.sums(e / 5, v)[e % 5];
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
    extern __shared__ double2 lds[];
    const Shared sh = shared_memory(lds);
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
        run_window<16>(G, I, R, k, nb, src, dst, mine, sh);
    else
        run_window<24>(G, I, R, k, nb, src, dst, mine, sh);
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

// Per geometry (job blockIdx.y), the core table: chunk c of n (n_tiles tiles of 64; zeros from n on), row i, is
// point (core_chunk0 + c) C + i - lead, {Re psi0, 1 in the PopInt window [lo, hi]} and Im psi0, zero outside
// the grid; and b of its first `head` points, which feel its own left wall where the lattice's do not.
__global__ void tdse_resident_core_kernel(const ResidentJob *jobs)
{
    const ResidentJob J = jobs[blockIdx.y];
    const int m = J.C * 64 * J.n_tiles;
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < m; q += gridDim.x * blockDim.x) {
        const int c = q / (64 * J.C) * 64 + q % 64, j = J.first + c * J.C + q / 64 % J.C;
        const bool on = c < J.n && j >= 0 && j < J.nx;
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
