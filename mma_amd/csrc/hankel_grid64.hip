// The FP64 contraction over r and the source planes (Hankel_transform.py:492-514, :641-661) with J0 taken
// from one table for all frequencies and planes.
//
// hk_direct_kernel evaluates J0 for every (plane, omega, rho, r): 45 FP64 instructions each, 1e11 of them on 256
// planes x 768 frequencies x 512 radii x 1024 screen points.  But J0(rho q) depends on (plane, omega, r) only
// through q = K r / D and is band-limited in it, so the sources of one frequency can first be summed
// onto a common grid Q_l = (l - P/2) h by Lagrange interpolation,
//     sum_k w_k sum_j u_kj J0(rho q_kj)  =  sum_l C_l J0(rho Q_l),   C_l = sum_kj w_k u_kj L_l(q_kj / h),
// with P = 16 nodes and rho_max h = 0.23, where the interpolation's error bound (rho h)^P max|prod| / P! is
// 2e-16 of one element: below the rounding of the element itself, whose argument of up to several hundred
// carries 1e-16 of it.  Per source 200 instructions, then a real matrix product in FP64 on the matrix cores,
// C (2 rows a frequency) by J0(rho_m Q_l).
//
// hk64_spread_kernel: one workgroup per (frequency, output).  A wave owns 64 consecutive radii and bins of
// its own for the stretch of q they reach (the radii ascend); a lane walks the planes with the 16
// bins of its current stencil in registers and adds a bin to LDS when the stencil has moved past
// it.  The waves' bins are added in a fixed order: no sum depends on which wave came first.
#include "hankel_internal.h"
#include "hankel_j0.h"
#include "sincos_reduced.h"

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

namespace {

constexpr int P = kNodes64;

__device__ inline double2 cmul(double2 a, double2 b)
{
    return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
__device__ inline double read_lane(double v, int l)
{
    const long long b = __builtin_bit_cast(long long, v);
    const unsigned lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
}
__device__ inline double2 wide(double2 v) { return v; }
__device__ inline double2 wide(float2 v) { return make_double2((double)v.x, (double)v.y); }

// grid position of the largest q of frequency o_max (all radii and planes)
__device__ inline double last_position(const hk_grid64 &g, double o_max) { return o_max * g.inv_c / g.d_min * g.r_max * g.inv_h; }

// bins that the 32 frequencies of a column tile use, in whole stages of the product: both the spread, which
// writes them, and the product, which sums over them, go by this (low frequencies use a part of the grid)
__device__ inline int tile_bins(const hk_grid64 &g, const double *ogrid, int no, int tile)
{
    double o_max = 0.0;
    const int o = tile * (kTile64 / 2) + (threadIdx.x & 31);
    if (o < no) o_max = ogrid[o];
#pragma unroll
    for (int d = 16; d >= 1; d >>= 1) o_max = fmax(o_max, __shfl_xor(o_max, d, 64));
    const int need = (int)last_position(g, o_max) + P + 3;
    return min(g.ld, (need + kStage64 - 1) / kStage64 * kStage64);
}

struct Stencil {
    double re[P], im[P];
    int l0;  // bin of re[0], counted from the block's first; below 0: empty
};

__device__ inline void flush(Stencil &w, double *bre, double *bim)
{
#pragma unroll
    for (int m = 0; m < P; m++) {
        atomicAdd(&bre[w.l0 + m], w.re[m]);
        atomicAdd(&bim[w.l0 + m], w.im[m]);
        w.re[m] = 0.0;
        w.im[m] = 0.0;
    }
}

// moves the stencil to bin l0: one bin up (what ascending planes give) or anywhere
__device__ inline void move_to(Stencil &w, int l0, double *bre, double *bim)
{
    if (l0 == w.l0) return;
    if (l0 == w.l0 + 1 && w.l0 >= 0) {
        atomicAdd(&bre[w.l0], w.re[0]);
        atomicAdd(&bim[w.l0], w.im[0]);
#pragma unroll
        for (int m = 0; m < P - 1; m++) {
            w.re[m] = w.re[m + 1];
            w.im[m] = w.im[m + 1];
        }
        w.re[P - 1] = 0.0;
        w.im[P - 1] = 0.0;
    } else if (w.l0 >= 0) {
        flush(w, bre, bim);
    }
    w.l0 = l0;
}

// 1 / prod_{j != i} (d_i - d_j)
constexpr double node_weight(int i)
{
    double den = 1.0;
    for (int q = 2; q <= i; q++) den *= (double)q;
    for (int q = 2; q <= P - 1 - i; q++) den *= (double)q;
    return ((P - 1 - i) & 1 ? -1.0 : 1.0) / den;
}
template <int... I>
struct Seq {};
template <int N, int... I>
struct MakeSeq : MakeSeq<N - 1, N - 1, I...> {};
template <int... I>
struct MakeSeq<0, I...> {
    using type = Seq<I...>;
};
template <int I>
__device__ inline void add_node(Stencil &w, double &pre, const double (&suf)[P], double f, double2 v)
{
    constexpr double c = node_weight(I);
    const double L = (pre * suf[I]) * c;
    w.re[I] = fma(L, v.x, w.re[I]);
    w.im[I] = fma(L, v.y, w.im[I]);
    pre *= f - (double)(I - (P / 2 - 1));
}
template <int... I>
__device__ inline void add_nodes(Stencil &w, const double (&suf)[P], double f, double2 v, Seq<I...>)
{
    double pre = 1.0;
    (add_node<I>(w, pre, suf, f, v), ...);
}

// adds v times the Lagrange basis of the nodes i - (P/2 - 1) at f in [0, 1)
__device__ inline void add_item(Stencil &w, double f, double2 v)
{
    double suf[P];
    suf[P - 1] = 1.0;
#pragma unroll
    for (int i = P - 2; i >= 0; i--) suf[i] = suf[i + 1] * (f - (double)(i + 1 - (P / 2 - 1)));
    add_nodes(w, suf, f, v, MakeSeq<P>::type());
}

} // namespace

// grid (no, outputs): output q0 + blockIdx.y.  weights: (outputs, nz), or null: output q is plane q.
// Dynamic LDS: g.bins complex doubles.  out: rows 2 (blockIdx.y no + o) and the next, g.ld apart.
template <typename S>
__global__ void __launch_bounds__(kSpread64, 2)
hk64_spread_kernel(hk_planes p, hk_grid64 g, int outputs, const double *weights, int q0, double *out, int *nonfinite)
{
    extern __shared__ double bins[];
    __shared__ int k_range[2], first[kBlocks64], at[kBlocks64 + 1];
    const int o = blockIdx.x, q = q0 + blockIdx.y;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const double K = p.ogrid[o] * g.inv_c;
    const int blocks = (p.nr + 63) / 64;
    if (threadIdx.x == 0) {
        k_range[0] = weights ? p.nz : q;
        k_range[1] = weights ? -1 : q;
    }
    __syncthreads();
    const double *const all = weights;
    if (weights) {
        weights += (long long)q * p.nz;
        for (int k = threadIdx.x; k < p.nz; k += blockDim.x)
            if (weights[k] != 0.0) {
                atomicMin(&k_range[0], k);
                atomicMax(&k_range[1], k);
            }
        __syncthreads();
    }
    // the first output also looks at the planes that no output weighs: 0 times a value that is not finite
    const bool every = weights && q == 0;
    const int k_lo = every ? 0 : k_range[0], k_hi = every ? p.nz - 1 : k_range[1];
    // the stretch of bins of block b: from the least position of its first radius to the largest of its last
    if ((int)threadIdx.x < blocks) {
        const int b = threadIdx.x, f = (int)(K / g.d_max * p.rgrid[b * 64] * g.inv_h);
        first[b] = f;
        at[b + 1] = (int)(K / g.d_min * p.rgrid[min(b * 64 + 63, p.nr - 1)] * g.inv_h) + P + 3 - f;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        at[0] = 0;
        for (int b = 0; b < blocks; b++) at[b + 1] += at[b];
        if (at[blocks] > g.bins) *nonfinite = 1;  // the host sizes the bins so that this never holds
    }
    __syncthreads();
    if (at[blocks] > g.bins) return;
    for (int b = wave; b < blocks; b += blockDim.x >> 6) {
        const int n = at[b + 1] - at[b], f0 = first[b];
        double *bre = bins + at[b], *bim = bre + g.bins;
        for (int l = lane; l < n; l += 64) {
            bre[l] = 0.0;
            bim[l] = 0.0;
        }
        // lanes past the last radius take it again, with no weight
        const int j = min(b * 64 + lane, p.nr - 1);
        const double r = p.rgrid[j], wr = b * 64 + lane < p.nr ? p.tw[j] * r : 0.0, r2 = r * r;
        const S *src = reinterpret_cast<const S *>(p.src) + (long long)k_lo * p.plane_stride + (long long)o * p.nr + j;
        Stencil w;
        w.l0 = -1;
#pragma unroll
        for (int m = 0; m < P; m++) {
            w.re[m] = 0.0;
            w.im[m] = 0.0;
        }
        S ahead = k_lo <= k_hi ? src[0] : S{};
        for (int k0 = k_lo; k0 <= k_hi; k0 += 64) {
            // the factors of 64 planes, one per lane
            const int kl = min(k0 + lane, k_hi);
            const double kd_l = K / (p.distance - p.zgrid[kl]), w_l = weights ? weights[kl] : 1.0;
            unsigned long long skip = __ballot(w_l == 0.0);
            if (every) {
                bool weighed = false;
                for (int i = 0; i < outputs; i++) weighed = weighed || all[(long long)i * p.nz + kl] != 0.0;
                skip &= __ballot(weighed);
            }
            double2 pre_l = make_double2(1.0, 0.0);
            if (p.pre_mode == 1) pre_l = reinterpret_cast<const double2 *>(p.pre)[(long long)kl * p.no + o];
            for (int t0 = 0; t0 < 64 && k0 + t0 <= k_hi; t0++) {
                const int k = k0 + t0;
                const S now = ahead;
                src += p.plane_stride;
                if (k < k_hi) ahead = src[0];  // the next plane's source in flight
                const double wk = read_lane(w_l, t0), KD = read_lane(kd_l, t0);
                if (skip >> t0 & 1) continue;
                double2 v = cmul(make_double2(read_lane(pre_l.x, t0), read_lane(pre_l.y, t0)), wide(now));
                if (p.pre_mode == 2)
                    v = cmul(reinterpret_cast<const double2 *>(p.pre)[((long long)k * p.no + o) * p.nr + j], wide(now));
                if (p.near_field) {
                    double s, c;
                    sincos_wide(-0.5 * KD * r2, &s, &c);
                    v = cmul(make_double2(c, s), v);
                }
                const double wv = wr * wk;
                v.x *= wv;
                v.y *= wv;
                // the position q / h, q = KD r: its integer part as first_bin and width form it, and the fraction
                // with what the two products rounded off
                const double x = KD * r, t = x * g.inv_h, f = floor(t);
                const double rest = fma(-t, g.h, x) + fma(KD, r, -x);
                const int l0 = (int)f + 1 - f0;
                if (l0 < 0 || l0 + P > n) continue;  // every position lies in the block's stretch
                move_to(w, l0, bre, bim);
                add_item(w, fma(rest, g.inv_h, t - f), v);
            }
        }
        if (w.l0 >= 0) flush(w, bre, bim);
    }
    __syncthreads();
    const int used = tile_bins(g, p.ogrid, p.no, o / (kTile64 / 2));
    double *row = out + 2LL * ((long long)blockIdx.y * p.no + o) * g.ld;
    bool finite = true;
    for (int l = threadIdx.x; l < used; l += blockDim.x) {
        double re = 0.0, im = 0.0;
        for (int b = 0; b < blocks; b++) {
            const int i = l - first[b];
            if (i >= 0 && i < at[b + 1] - at[b]) {
                re += bins[at[b] + i];
                im += bins[g.bins + at[b] + i];
            }
        }
        row[l] = re;
        row[g.ld + l] = im;
        finite = finite && isfinite(re) && isfinite(im);
    }
    if (!finite) *nonfinite = 1;
}

template __global__ void hk64_spread_kernel<double2>(hk_planes, hk_grid64, int, const double *, int, double *, int *);
template __global__ void hk64_spread_kernel<float2>(hk_planes, hk_grid64, int, const double *, int, double *, int *);

// J0(rho_m Q_l), Q_l = (l - P/2) h.  h has few enough bits that Q_l is exact, and the rounding of
// rho Q_l, which every source near that bin would share, is put back: cos and sin of the exact product.
__global__ void hk64_bessel_kernel(int nrho, const double *rho, hk_grid64 g, double *out)
{
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= g.ld) return;
    for (int m = blockIdx.y; m < nrho; m += gridDim.y) {  // (a grid has 65535 rows at most)
        const double q = (double)(l - P / 2) * g.h, a = rho[m];
        const double x = a * q, e = fma(a, q, -x);
        double s, c;
        sincos_wide(x, &s, &c);
        out[(long long)m * g.ld + l] = hk::j0(x, fma(-e, s, c), fma(e, c, s));
    }
}

// out[m][n] = sum_l A[m][l] B[n][l] in FP64: A the J0 table (M rows), B the spread sources (N rows per output).
// Tiles of 64 x 64: 16 FLOP for every byte fetched, and 4.5 tiles per CU for 1024 screen points by 4608 rows where 128 x 128
// would leave 1.1.  Eight waves: four of 32 x 32 (2 x 2 of v_mfma_f64_16x16x4) on the even stages of 32 elements
// of the sum and four on the odd ones, whose result is added at the end (with four waves a batch of 240 tiles left
// every SIMD one wave, which waited for its loads).  A stage lies in LDS, the next is in flight.
// A lane of a wave takes the elements 8 s + 2 (lane / 16) and the next of its row, one 16-byte read for two
// products: which elements meet in which product does not matter.  Rows are padded by 2 doubles, so that 16 rows
// start 4 banks apart.  Sums of 64 products are added with their rounding kept: plain sums of 3000 would
// round off 2.7e-15 of the far field, three to five times the direct kernel's error; so it is 1 to 4e-16.
// grid: (outputs x column tiles x row tiles, rounded up to a multiple of 8); tiles next to each other, which share
// their columns, run on one XCD.
__global__ void __launch_bounds__(512, 2)
hk64_gemm_kernel(int M, int N, int outputs, hk_grid64 g, const double *ogrid, const double *A, const double *B, double *out, long long ldo)
{
    constexpr int T = kTile64, KS = kStage64, LD = KS + 2;
    __shared__ __attribute__((aligned(16))) double tile[2][2][T][LD];
    const int half = threadIdx.x >> 8, tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
    double (*ta)[LD] = tile[half][0], (*tb)[LD] = tile[half][1];
    const int mt = (M + T - 1) / T, nt = (N + T - 1) / T;
    // an eighth of all tiles per XCD (consecutive workgroups go to consecutive XCDs)
    const unsigned idx = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8;
    if (idx >= (unsigned)(mt * nt * outputs)) return;
    const int tm = idx % mt, tn = idx / mt % nt, q = idx / mt / nt;
    const int m0 = tm * T, n0 = tn * T;
    B += (long long)q * N * g.ld;
    out += (long long)q * M * ldo;
    const int K = tile_bins(g, ogrid, N / 2, tn);

    // 64 rows x 32 doubles: 16 threads a row, a 16-byte element each, 4 rows of 16 apart
    const int row = tid >> 4, col = (tid & 15) * 2;
    const double *pa[4], *pb[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        pa[i] = A + (long long)min(m0 + row + 16 * i, M - 1) * g.ld + col;
        pb[i] = B + (long long)min(n0 + row + 16 * i, N - 1) * g.ld + col;
    }
    f64x2 ra[4], rb[4];
    auto fetch = [&](int k) {  // zero past the sum's end
        const f64x2 none = {0.0, 0.0};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            ra[i] = k < K ? *reinterpret_cast<const f64x2 *>(pa[i] + k) : none;
            rb[i] = k < K ? *reinterpret_cast<const f64x2 *>(pb[i] + k) : none;
        }
    };
    f64x4 acc[2][2], sum[2][2], rest[2][2];
    const f64x4 zero = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = sum[i][j] = rest[i][j] = zero;
    auto add = [&](int i, int j, f64x4 v) {
        const f64x4 s = sum[i][j] + v, d = s - sum[i][j];
        rest[i][j] += (sum[i][j] - (s - d)) + (v - d);
        sum[i][j] = s;
    };
    const int wm = (wave >> 1) * 32 + (lane & 15), wn = (wave & 1) * 32 + (lane & 15), kq = (lane >> 4) * 2;
    fetch(half * KS);
    for (int k = 0; k < K; k += 2 * KS) {
        __syncthreads();  // the stage before has been read
#pragma unroll
        for (int i = 0; i < 4; i++) {
            *reinterpret_cast<f64x2 *>(&ta[row + 16 * i][col]) = ra[i];
            *reinterpret_cast<f64x2 *>(&tb[row + 16 * i][col]) = rb[i];
        }
        __syncthreads();
        if (k + 2 * KS < K) fetch(k + (2 + half) * KS);
#pragma unroll
        for (int s = 0; s < KS; s += 8) {
            f64x2 a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                a[i] = *reinterpret_cast<const f64x2 *>(&ta[wm + 16 * i][s + kq]);
                b[i] = *reinterpret_cast<const f64x2 *>(&tb[wn + 16 * i][s + kq]);
            }
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
        }
        if ((k / (2 * KS)) % 2 == 1 || k + 2 * KS >= K) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    add(i, j, acc[i][j]);
                    acc[i][j] = zero;
                }
        }
    }
    // the odd stages' sums through LDS, 4 KB a wave and part
    f64x4 *const pass = reinterpret_cast<f64x4 *>(&tile[0][0][0][0]);
    static_assert(sizeof(tile) >= 2 * 4 * 256 * sizeof(f64x4), "room for the odd stages' sums");
    __syncthreads();
    if (half == 1) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            pass[i * 256 + tid] = sum[i >> 1][i & 1];
            pass[(4 + i) * 256 + tid] = rest[i >> 1][i & 1];
        }
    }
    __syncthreads();
    if (half == 1) return;
    // element v of a lane: row 4 v + lane / 16, column lane % 16
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            add(i, j, pass[(2 * i + j) * 256 + tid]);
            rest[i][j] += pass[(4 + 2 * i + j) * 256 + tid];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int m = m0 + (wave >> 1) * 32 + 16 * i + 4 * v + (lane >> 4);
                const int n = n0 + (wave & 1) * 32 + 16 * j + (lane & 15);
                if (m < M && n < N) out[m * ldo + n] = sum[i][j][v] + rest[i][j][v];
            }
        }
}
