// Direct solution of A x = b, A = sigma I~ + tau L, on grids that are
// periodic and uniform in x and z (power-of-two point counts) and walled in
// y -- the channel of the timestep's benchmark.
//
// Row (i, j, k) of the operator (fd/laplacian.h:53-68, fd/identity.h:25-51)
// is sigma Iy_j x + tau (Iy_j Lx x + Ly x + Iy_j Lz x): the identity factors
// of periodic axes are 1 and their 3-point Laplacians are circulant, so the
// discrete Fourier transform in x and z diagonalises them,
//   Lx -> -4 rx^2 sin^2(pi kx / nx),   Lz -> -4 rz^2 sin^2(pi kz / nz),
// and every Fourier mode (kx, kz) leaves one tridiagonal system along y,
//   Iy_j (sigma + tau mu) X_j + tau ry^2 (lo_j X_{j-1} + d_j X_j + hi_j X_{j+1})
//   = B_j,   mu = lambda_x(kx) + lambda_z(kz),
// with the wall rows' ghost coefficients in d_0, d_{n-1} (fd/discretization.h:
// 94-108).  The solve is: real-to-half-complex FFT along x, complex FFT
// along z, one tridiagonal solve per mode (chunks of rows in registers), and
// the inverse transforms -- the exact solution of the same discrete system the
// multigrid iterates on.  The transforms of a y-plane are one memory pass in
// LDS where both point counts are 32 to 128 (three passes per solve) and two
// elsewhere (five).  The singular case (sigma = 0 with
// Neumann walls: the pressure Poisson) solves the mean-free problem, as the
// multigrid does: the (0, 0) mode's right-hand side loses its mean, its last
// unknown is pinned and the solution's mean is removed.
//
// The reference solves these systems with multigrid or PCG
// (solvers/multigrid.h, solvers/pcg.h); this is a different algorithm for the
// same discrete equations, used where the grid allows it.
#include <hip/hip_runtime.h>
#include <cmath>
#include <mutex>
#include <vector>
#include "context.hpp"
#include "fd_kernels.hpp"
#include "fd_ops.hpp"

namespace ibm {
namespace {

constexpr int FFT_THREADS = 256;
constexpr int ZT = 8;              // kx columns per z-transform block
constexpr int MAX_FFT_POINTS = 512;
constexpr int MAX_WALL_POINTS = 800;
constexpr int LINE_THREADS = 256, LINE_MODES = 8, LINE_CHUNKS = LINE_THREADS / LINE_MODES;
constexpr int SHORT_ROWS = 8, SHORT_MODES = 64;      // lines of up to SHORT_ROWS rows: fewer chunks, more modes a block
constexpr size_t MAX_DYNAMIC_LDS = 160 * 1024;

// Row stride of the half-spectrum in coefficients: nh rounded up to 8 (rows
// start on 128-byte boundaries, so the column tiles of the z transform and
// the line solves read whole cache lines).
__host__ __device__ constexpr int spec_ld(int nh) { return (nh + 7) & ~7; }

__device__ inline double2 cmul(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }

__device__ inline int bitrev(int k, int logn) { return (int) (__brev((unsigned) k) >> (32 - logn)); }

// In-place radix-2 transforms of `count` arrays of n points held in LDS in
// bit-reversed order: point k of array t at a[idx(t, k)] holds input
// bitrev(k).  Rows layout (idx = t n + k, the x transforms) maps consecutive
// lanes to consecutive butterflies of one array; columns layout (idx =
// k count + t, the z transforms, whose rows of count arrays are contiguous)
// maps consecutive lanes to consecutive arrays, so that the lanes of a wave
// touch consecutive LDS words either way.  tw[m] = exp(-2 pi i m / n),
// m < n / 2, also in LDS (a stage's twiddle reads would otherwise be
// dependent global loads); `inverse` conjugates the twiddles (no scaling).
// Every thread of the block takes part in every stage.  Stages are done in
// pairs: a thread loads the quad k0, k0 + h, k0 + 2h, k0 + 3h (h = 2^(s-1)),
// does stage s's two butterflies and stage s + 1's two, and stores it -- the
// radix-2 butterflies and twiddles exactly, with one LDS round trip and one
// barrier per two stages.
__device__ inline void butterfly(double2& u, double2& v, double2 w, bool inverse)
{
    if (inverse) w.y = -w.y;
    const double2 t = cmul(v, w);
    v = make_double2(u.x - t.x, u.y - t.y);
    u = make_double2(u.x + t.x, u.y + t.y);
}

template <bool COLS>
__device__ void fft_stages(double2* a, int count, int n, int logn, const double2* tw, bool inverse)
{
    int s = 1;
    const int quads = count * (n >> 2);
    for (; s + 1 <= logn; s += 2) {
        const int h = 1 << (s - 1);
        const int st0 = n >> s, st1 = n >> (s + 1);       // twiddle index steps of stages s and s + 1
        for (int b = threadIdx.x; b < quads; b += blockDim.x) {
            const int t = COLS ? b % count : b / (n >> 2), bb = COLS ? b / count : b - t * (n >> 2);
            const int grp = bb >> (s - 1), pos = bb & (h - 1);
            const int k0 = grp * 4 * h + pos;
            const int i0 = COLS ? k0 * count + t : t * n + k0;
            const int dh = COLS ? h * count : h;
            double2 q0 = a[i0], q1 = a[i0 + dh], q2 = a[i0 + 2 * dh], q3 = a[i0 + 3 * dh];
            const double2 w0 = tw[pos * st0];
            butterfly(q0, q1, w0, inverse);
            butterfly(q2, q3, w0, inverse);
            butterfly(q0, q2, tw[pos * st1], inverse);
            butterfly(q1, q3, tw[(pos + h) * st1], inverse);
            a[i0] = q0;
            a[i0 + dh] = q1;
            a[i0 + 2 * dh] = q2;
            a[i0 + 3 * dh] = q3;
        }
        __syncthreads();
    }
    if (s == logn) {
        const int half_n = n >> 1, half = 1 << (s - 1), stride = n >> s;
        const int total = count * half_n;
        for (int b = threadIdx.x; b < total; b += blockDim.x) {
            const int t = COLS ? b % count : b / half_n, bb = COLS ? b / count : b - t * half_n;
            const int grp = bb >> (s - 1), pos = bb & (half - 1);
            const int k0 = grp * 2 * half + pos, k1 = k0 + half;
            const int i = COLS ? k0 * count + t : t * n + k0, j = COLS ? k1 * count + t : t * n + k1;
            double2 u = a[i], v = a[j];
            butterfly(u, v, tw[pos * stride], inverse);
            a[i] = u;
            a[j] = v;
        }
        __syncthreads();
    }
}

// Forward transform along x of `rows` rows of nx reals into nh = nx / 2 + 1
// coefficients each (row r of x -> row r of s, x fastest in both).  The
// bit reversal is applied to the (cached) global reads, so the LDS writes
// are consecutive.
__global__ void __launch_bounds__(FFT_THREADS) xfft_forward_kernel(int nx, int logn, int rows,
                                                                   const double* __restrict__ x,
                                                                   double2* __restrict__ s,
                                                                   const double2* __restrict__ tw)
{
    extern __shared__ double2 sh[];
    const int rpb = FFT_THREADS / (nx / 2), nh = nx / 2 + 1;
    double2* stw = sh + rpb * nx;
    const int r0 = blockIdx.x * rpb;
    for (int e = threadIdx.x; e < nx / 2; e += blockDim.x) stw[e] = tw[e];
    for (int e = threadIdx.x; e < rpb * nx; e += blockDim.x) {
        const int t = e / nx, k = e - t * nx, row = r0 + t;
        sh[e] = make_double2(row < rows ? x[(size_t) row * nx + bitrev(k, logn)] : 0.0, 0.0);
    }
    __syncthreads();
    fft_stages<false>(sh, rpb, nx, logn, stw, false);
    for (int e = threadIdx.x; e < rpb * nh; e += blockDim.x) {
        const int t = e / nh, k = e - t * nh, row = r0 + t;
        if (row < rows) s[(size_t) row * spec_ld(nh) + k] = sh[t * nx + k];
    }
}

// Inverse of xfft_forward_kernel (the missing coefficients are the
// conjugates of the stored ones), scaled by `scale`.
__global__ void __launch_bounds__(FFT_THREADS) xfft_inverse_kernel(int nx, int logn, int rows,
                                                                   const double2* __restrict__ s,
                                                                   double* __restrict__ x, double scale,
                                                                   const double2* __restrict__ tw)
{
    extern __shared__ double2 sh[];
    const int rpb = FFT_THREADS / (nx / 2), nh = nx / 2 + 1;
    double2* stw = sh + rpb * nx;
    const int r0 = blockIdx.x * rpb;
    for (int e = threadIdx.x; e < nx / 2; e += blockDim.x) stw[e] = tw[e];
    for (int e = threadIdx.x; e < rpb * nx; e += blockDim.x) {
        const int t = e / nx, k = bitrev(e - t * nx, logn), row = r0 + t;
        double2 v = make_double2(0.0, 0.0);
        if (row < rows) {
            if (k < nh) {
                v = s[(size_t) row * spec_ld(nh) + k];
            } else {
                v = s[(size_t) row * spec_ld(nh) + (nx - k)];
                v.y = -v.y;
            }
        }
        sh[e] = v;
    }
    __syncthreads();
    fft_stages<false>(sh, rpb, nx, logn, stw, true);
    for (int e = threadIdx.x; e < rpb * nx; e += blockDim.x) {
        const int t = e / nx, k = e - t * nx, row = r0 + t;
        if (row < rows) x[(size_t) row * nx + k] = sh[t * nx + k].x * scale;
    }
}

// Transform along z, in place, of s laid out [k][j][kx] (kx fastest, nh of
// them in rows of spec_ld(nh)): block (kx tile, j) transforms ZT columns,
// held in LDS as rows of ZT consecutive kx.
__global__ void __launch_bounds__(FFT_THREADS) zfft_kernel(int nh, int ny, int nz, int logn, double2* __restrict__ s,
                                                           const double2* __restrict__ tw, int inverse)
{
    extern __shared__ double2 sh[];
    double2* stw = sh + ZT * nz;
    const int kx0 = blockIdx.x * ZT, j = blockIdx.y;
    const int ld = spec_ld(nh);
    const size_t plane = (size_t) ld * ny;
    for (int e = threadIdx.x; e < nz / 2; e += blockDim.x) stw[e] = tw[e];
    for (int e = threadIdx.x; e < ZT * nz; e += blockDim.x) {
        const int t = e % ZT, k = e / ZT, kx = kx0 + t, kr = bitrev(k, logn);
        sh[e] = kx < nh ? s[(size_t) kr * plane + (size_t) j * ld + kx] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    fft_stages<true>(sh, ZT, nz, logn, stw, inverse != 0);
    for (int e = threadIdx.x; e < ZT * nz; e += blockDim.x) {
        const int t = e % ZT, k = e / ZT, kx = kx0 + t;
        if (kx < nh) s[(size_t) k * plane + (size_t) j * ld + kx] = sh[e];
    }
}

// ----------------------------------------------------------------------
// Both transforms of one y-plane in LDS
// ----------------------------------------------------------------------
// DFT of R values in registers, natural order in and out.
template <int R, bool INV>
__device__ inline void dft(double2 (&v)[R])
{
    if constexpr (R == 2) {
        const double2 u = v[0], w = v[1];
        v[0] = make_double2(u.x + w.x, u.y + w.y);
        v[1] = make_double2(u.x - w.x, u.y - w.y);
    } else {
        // cos(2 pi k / 16), k = 0..4
        constexpr double C[5] = {1.0, 0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.0};
        double2 e[R / 2], o[R / 2];
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {
            e[k] = v[2 * k];
            o[k] = v[2 * k + 1];
        }
        dft<R / 2, INV>(e);
        dft<R / 2, INV>(o);
#pragma unroll
        for (int k = 0; k < R / 2; ++k) {
            const int m = k * (16 / R);                       // exp(-+ 2 pi i m / 16), m < 8
            double2 t = o[k];
            if (m == 4) {
                t = INV ? make_double2(-t.y, t.x) : make_double2(t.y, -t.x);
            } else if (m > 0) {
                const double c = m < 4 ? C[m] : -C[8 - m], sn = m < 4 ? C[4 - m] : C[m - 4];
                t = cmul(t, make_double2(c, INV ? sn : -sn));
            }
            v[k] = make_double2(e[k].x + t.x, e[k].y + t.y);
            v[k + R / 2] = make_double2(e[k].x - t.x, e[k].y - t.y);
        }
    }
}

__device__ inline double2 conj2(double2 a) { return make_double2(a.x, -a.y); }

// LDS position of point n of a row: eight lanes with consecutive n, or with n
// eight apart, lie in different banks.
__device__ inline int swz(int n) { return n ^ ((n >> 3) & 7); }

// Sizes of a plane transform: nx x nz points with nx = 2^LX, nz = 2^LZ.  A row
// of nx reals is transformed as H = nx / 2 complex points, 8 x SX; a column of
// nz as 8 x SZ.
template <int LX, int LZ>
struct plane_size {
    static constexpr int NX = 1 << LX, NZ = 1 << LZ, H = NX / 2, SX = H / 8, SZ = NZ / 8, LD = H + 1;
    static constexpr int THREADS = NX * NZ / 32 < 256 ? 256 : NX * NZ / 32;
    static constexpr size_t LDS = sizeof(double2) * (NZ * LD + NX + NZ);
};

// Tables exp(-2 pi i e / n) for all e < n, from the first halves.
template <class P>
__device__ inline void plane_tables(double2* wx, double2* wz, const double2* __restrict__ twx, const double2* __restrict__ twz)
{
    for (int e = threadIdx.x; e < P::NX; e += P::THREADS) {
        const double2 w = twx[e % (P::NX / 2)];
        wx[e] = e < P::NX / 2 ? w : make_double2(-w.x, -w.y);
    }
    for (int e = threadIdx.x; e < P::NZ; e += P::THREADS) {
        const double2 w = twz[e % (P::NZ / 2)];
        wz[e] = e < P::NZ / 2 ? w : make_double2(-w.x, -w.y);
    }
}

// Two doubles at 8-byte alignment (the caller's vector).
typedef double d2u8 __attribute__((ext_vector_type(2), aligned(8)));

// Forward transforms along x and z of plane j = blockIdx.x, the same values as
// xfft_forward_kernel and zfft_kernel: the half-spectrum stays in LDS between
// them, and every stage takes 8 or 16 points at a time in registers.
// A row's reals are taken as half as many complex points.  Bound by the phases
// of a block, which cannot overlap where one plane fills a CU's LDS (load, four
// LDS round trips, store); two passes wrote and read the half-spectrum once
// more and did radix-2 stages in pairs.  128 x 256 x 128 points, forward /
// inverse: 49 / 49 us by passes, 22 / 18 by planes.
template <int LX, int LZ>
__global__ void __launch_bounds__((plane_size<LX, LZ>::THREADS))
plane_forward_kernel(int ny, const double* __restrict__ x, double2* __restrict__ s, const double2* __restrict__ twx,
                     const double2* __restrict__ twz)
{
    using P = plane_size<LX, LZ>;
    constexpr int NX = P::NX, NZ = P::NZ, H = P::H, SX = P::SX, SZ = P::SZ, LD = P::LD, T = P::THREADS;
    extern __shared__ double2 sh[];
    double2* wx = sh + NZ * LD;
    double2* wz = wx + NX;
    const int j = blockIdx.x, tid = threadIdx.x;
    plane_tables<P>(wx, wz, twx, twz);
    // rows: points m0 + SX i of z[m] = (x[2m], x[2m+1])
    constexpr int ROW_TASKS = NZ * SX, ROW_ITEMS = (ROW_TASKS + T - 1) / T;
    double2 v[ROW_ITEMS][8];
#pragma unroll
    for (int u = 0; u < ROW_ITEMS; ++u) {
        const int e = tid + u * T, row = e / SX, m0 = e % SX;
        if (ROW_TASKS % T == 0 || e < ROW_TASKS) {
            const double* src = x + ((size_t) row * ny + j) * NX + 2 * m0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const d2u8 q = *(const d2u8*) (src + 2 * SX * i);
                v[u][i] = make_double2(q.x, q.y);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < ROW_ITEMS; ++u) {
        const int e = tid + u * T, row = e / SX, m0 = e % SX;
        if (ROW_TASKS % T == 0 || e < ROW_TASKS) {
            dft<8, false>(v[u]);
#pragma unroll
            for (int q = 0; q < 8; ++q)
                sh[row * LD + swz(8 * m0 + q)] = q == 0 ? v[u][q] : cmul(v[u][q], wx[2 * m0 * q]);
        }
    }
    __syncthreads();
    // rows: the SX points of each q, giving Z[8 k + q] in place
    for (int e = tid; e < NZ * 8; e += T) {
        const int row = e >> 3, q = e & 7;
        double2 w[SX];
#pragma unroll
        for (int m = 0; m < SX; ++m) w[m] = sh[row * LD + swz(8 * m + q)];
        dft<SX, false>(w);
#pragma unroll
        for (int m = 0; m < SX; ++m) sh[row * LD + swz(8 * m + q)] = w[m];
    }
    __syncthreads();
    // the rows' coefficients k and H - k from Z[k] and Z[H - k], and the
    // columns' points m0 + SZ i
    for (int e = tid; e < (H / 2 + 1) * SZ; e += T) {
        const int k = e < H / 2 * SZ ? e % (H / 2) : H / 2, m0 = e < H / 2 * SZ ? e / (H / 2) : e - H / 2 * SZ;
        const int at0 = swz(k), at1 = k == 0 ? H : swz(H - k);
        const double2 wk = wx[k];
        double2 a[8], b[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const double2* row = sh + (m0 + SZ * i) * LD;
            const double2 z0 = row[at0], z1 = k == 0 ? z0 : row[at1];
            const double2 ev = make_double2(0.5 * (z0.x + z1.x), 0.5 * (z0.y - z1.y));
            const double2 od = make_double2(0.5 * (z0.y + z1.y), 0.5 * (z1.x - z0.x));
            const double2 t = cmul(od, wk);
            a[i] = make_double2(ev.x + t.x, ev.y + t.y);
            b[i] = make_double2(ev.x - t.x, t.y - ev.y);
        }
        dft<8, false>(a);
        dft<8, false>(b);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            double2* row = sh + (m0 + SZ * q) * LD;
            const double2 w = wz[m0 * q];
            row[at0] = cmul(a[q], w);
            if (k != H / 2) row[at1] = cmul(b[q], w);
        }
    }
    __syncthreads();
    // columns: the SZ points of each q, giving kz = 8 m + q
    for (int e = tid; e < LD * 8; e += T) {
        const int kx = e % LD, q = e / LD, at = kx == H ? H : swz(kx);
        double2 w[SZ];
#pragma unroll
        for (int m = 0; m < SZ; ++m) w[m] = sh[(SZ * q + m) * LD + at];
        dft<SZ, false>(w);
#pragma unroll
        for (int m = 0; m < SZ; ++m) s[((size_t) (8 * m + q) * ny + j) * spec_ld(LD) + kx] = w[m];
    }
}

// Inverse of plane_forward_kernel, scaled by `scale`.
template <int LX, int LZ>
__global__ void __launch_bounds__((plane_size<LX, LZ>::THREADS))
plane_inverse_kernel(int ny, const double2* __restrict__ s, double* __restrict__ x, double scale,
                     const double2* __restrict__ twx, const double2* __restrict__ twz)
{
    using P = plane_size<LX, LZ>;
    constexpr int NX = P::NX, NZ = P::NZ, H = P::H, SX = P::SX, SZ = P::SZ, LD = P::LD, T = P::THREADS;
    extern __shared__ double2 sh[];
    double2* wx = sh + NZ * LD;
    double2* wz = wx + NX;
    const int j = blockIdx.x, tid = threadIdx.x;
    plane_tables<P>(wx, wz, twx, twz);
    __syncthreads();
    // columns: points kz = m0 + 8 i
    for (int e = tid; e < LD * 8; e += T) {
        const int kx = e % LD, m0 = e / LD, at = kx == H ? H : swz(kx);
        double2 w[SZ];
#pragma unroll
        for (int i = 0; i < SZ; ++i) w[i] = s[((size_t) (m0 + 8 * i) * ny + j) * spec_ld(LD) + kx];
        dft<SZ, true>(w);
#pragma unroll
        for (int q = 0; q < SZ; ++q) sh[(SZ * m0 + q) * LD + at] = q == 0 ? w[q] : cmul(w[q], conj2(wz[m0 * q]));
    }
    __syncthreads();
    // columns: the 8 points of each q, giving z = SZ m + q in place, and the
    // rows' Z[k] and Z[H - k] (twice their value) from the coefficients k and
    // H - k
    for (int e = tid; e < (H / 2 + 1) * SZ; e += T) {
        const int k = e < H / 2 * SZ ? e % (H / 2) : H / 2, q = e < H / 2 * SZ ? e / (H / 2) : e - H / 2 * SZ;
        const int at0 = swz(k), at1 = k == 0 ? H : swz(H - k);
        const double2 wk = conj2(wx[k]);
        double2 a[8], b[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const double2* row = sh + (SZ * m + q) * LD;
            a[m] = row[at0];
            b[m] = row[at1];
        }
        dft<8, true>(a);
        dft<8, true>(b);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const double2 ev = make_double2(a[m].x + b[m].x, a[m].y - b[m].y);
            const double2 od = cmul(make_double2(a[m].x - b[m].x, a[m].y + b[m].y), wk);
            double2* row = sh + (SZ * m + q) * LD;
            row[at0] = make_double2(ev.x - od.y, ev.y + od.x);
            if (k != 0 && k != H / 2) row[at1] = make_double2(ev.x + od.y, od.x - ev.y);
        }
    }
    __syncthreads();
    // rows: points m0 + SX i, in place
    for (int e = tid; e < NZ * SX; e += T) {
        const int row = e / SX, m0 = e % SX;
        double2 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = sh[row * LD + swz(m0 + SX * i)];
        dft<8, true>(v);
#pragma unroll
        for (int q = 0; q < 8; ++q)
            sh[row * LD + swz(m0 + SX * q)] = q == 0 ? v[q] : cmul(v[q], conj2(wx[2 * m0 * q]));
    }
    __syncthreads();
    // rows: the SX points of each q, giving z[8 m + q] = (x[2 (8 m + q)], ...)
    for (int e = tid; e < NZ * 8; e += T) {
        const int row = e >> 3, q = e & 7;
        double2 w[SX];
#pragma unroll
        for (int m = 0; m < SX; ++m) w[m] = sh[row * LD + swz(SX * q + m)];
        dft<SX, true>(w);
        double* dst = x + ((size_t) row * ny + j) * NX + 2 * q;
#pragma unroll
        for (int m = 0; m < SX; ++m) *(d2u8*) (dst + 16 * m) = d2u8{w[m].x * scale, w[m].y * scale};
    }
}

struct wall_axis {
    int n;
    double r2, lap_lo, lap_hi, id_lo, id_hi;
};

// Row j's coefficients of mode (kx, kz): sub- and super-diagonal lo, hi and
// the diagonal.
__device__ inline void tri_row(const wall_axis& y, double sigma, double tau, double mu, int j, double& lo, double& hi,
                               double& diag)
{
    const double ty = tau * y.r2;
    lo = j > 0 ? ty : 0.0;
    hi = j < y.n - 1 ? ty : 0.0;
    double d = -2.0, id = 1.0;
    if (j == 0) {
        d += y.lap_lo;
        id += y.id_lo;
    }
    if (j == y.n - 1) {
        d += y.lap_hi;
        id += y.id_hi;
    }
    diag = id * (sigma + tau * mu) + ty * d;
}

// Sum over a workgroup's chunks of the lanes with t = 0.
template <int MODES>
__device__ inline double2 line_sum(double2 v, double2* part)
{
    __syncthreads();
    if (threadIdx.x % MODES == 0) part[threadIdx.x / MODES] = v;
    __syncthreads();
    double2 m = make_double2(0.0, 0.0);
    for (int i = 0; i < LINE_THREADS / MODES; ++i) {
        m.x += part[i].x;
        m.y += part[i].y;
    }
    return m;
}

// Every Fourier mode's tridiagonal system along y: block (tile of MODES kx,
// kz), one thread per mode and chunk of M consecutive rows, which it keeps
// in registers (rows past ny are identity rows).  A forward elimination leaves
// row r as X_r = d_r - c_r X_{r+1} - a_r X_{-1}, with X_{-1} the last row of
// the chunk before, and a backward one gives the first row by the chunk's and
// the previous chunk's last; put into the previous chunk's last row that is
// one equation per chunk, solved by cyclic reduction over them, and a back substitution ends it.  The singular mode's last equation is
// replaced by x = 0 after its right-hand side loses its mean, and its solution
// loses its mean.  Bound by memory (16 bytes per row read and written, whole
// 128-byte lines): cyclic reduction over all rows in LDS took two divisions
// per row and step, eight in all, this one and a fraction.  65 x 256 x 128
// coefficients: 48 us / 17.  Few rows leave most chunks without any: a solve of
// 256 x 2 x 256 points 37 us with 8 modes a block, 30 with 64.
template <int M, int MODES = LINE_MODES>
__global__ void __launch_bounds__(LINE_THREADS) line_kernel(int nh, wall_axis y, double sigma, double tau, int singular,
                                                            const double* __restrict__ lam_x,
                                                            const double* __restrict__ lam_z, double2* __restrict__ s)
{
    __shared__ double2 D[2][LINE_THREADS];
    __shared__ double2 AC[2][LINE_THREADS];
    constexpr int CHUNKS = LINE_THREADS / MODES;
    __shared__ double2 part[CHUNKS];
    const int ny = y.n, t = threadIdx.x % MODES, q = threadIdx.x / MODES;
    const int kx = blockIdx.x * MODES + t, kz = blockIdx.y, j0 = q * M;
    const int ld = spec_ld(nh);
    const bool pin_block = singular && blockIdx.x == 0 && kz == 0;     // holds the singular mode (t = 0)
    const bool pinned = pin_block && t == 0;
    double2* col = s + (size_t) kz * ld * ny + kx;
    double a[M], c[M];
    double2 d[M];
#pragma unroll
    for (int r = 0; r < M; ++r) d[r] = kx < nh && j0 + r < ny ? col[(size_t) (j0 + r) * ld] : make_double2(0.0, 0.0);
    const double mu = kx < nh ? lam_x[kx] + lam_z[kz] : 0.0;
    if (pin_block) {
        double2 own = make_double2(0.0, 0.0);
#pragma unroll
        for (int r = 0; r < M; ++r) own = make_double2(own.x + d[r].x, own.y + d[r].y);
        const double2 sum = line_sum<MODES>(own, part);
        if (pinned) {
#pragma unroll
            for (int r = 0; r < M; ++r)
                if (j0 + r < ny) d[r] = make_double2(d[r].x - sum.x / ny, d[r].y - sum.y / ny);
        }
    }
#pragma unroll
    for (int r = 0; r < M; ++r) {
        const int j = j0 + r;
        double lo = 0.0, hi = 0.0, diag = 1.0;
        if (kx < nh && j < ny) tri_row(y, sigma, tau, mu, j, lo, hi, diag);
        if (pinned && j == ny - 1) {
            lo = hi = 0.0;
            diag = 1.0;
            d[r] = make_double2(0.0, 0.0);
        }
        if (r == 0) {
            const double inv = 1.0 / diag;
            a[r] = lo * inv;
            c[r] = hi * inv;
            d[r] = make_double2(d[r].x * inv, d[r].y * inv);
        } else {
            const double inv = 1.0 / (diag - lo * c[r - 1]);
            a[r] = -lo * a[r - 1] * inv;
            c[r] = hi * inv;
            d[r] = make_double2((d[r].x - lo * d[r - 1].x) * inv, (d[r].y - lo * d[r - 1].y) * inv);
        }
    }
    // the chunk's first row: X_0 = p - f X_{-1} - g X_{M-1}
    double f = a[M - 2], g = c[M - 2];
    double2 p = d[M - 2];
#pragma unroll
    for (int r = M - 3; r >= 0; --r) {
        f = a[r] - c[r] * f;
        p = make_double2(d[r].x - c[r] * p.x, d[r].y - c[r] * p.y);
        g = -c[r] * g;
    }
    // the next chunk's first row in this one's last
    const int id = threadIdx.x;
    D[0][id] = p;
    AC[0][id] = make_double2(f, g);
    __syncthreads();
    double ra = a[M - 1], rc = 0.0;
    double2 rd = d[M - 1];
    if (q + 1 < CHUNKS) {
        const double2 np = D[0][id + MODES], nfg = AC[0][id + MODES];
        const double inv = 1.0 / (1.0 - c[M - 1] * nfg.x);
        ra *= inv;
        rc = -c[M - 1] * nfg.y * inv;
        rd = make_double2((rd.x - c[M - 1] * np.x) * inv, (rd.y - c[M - 1] * np.y) * inv);
    }
    if (q == 0) ra = 0.0;
    // cyclic reduction of X_q + ra X_{q-1} + rc X_{q+1} = rd
    int buf = 1;
#pragma unroll
    for (int sft = 1; sft < CHUNKS; sft <<= 1) {
        D[buf][id] = rd;
        AC[buf][id] = make_double2(ra, rc);
        __syncthreads();
        double2 dm = make_double2(0.0, 0.0), dn = dm, am = dm, an = dm;
        if (q >= sft) {
            dm = D[buf][id - sft * MODES];
            am = AC[buf][id - sft * MODES];
        }
        if (q + sft < CHUNKS) {
            dn = D[buf][id + sft * MODES];
            an = AC[buf][id + sft * MODES];
        }
        const double inv = 1.0 / (1.0 - ra * am.y - rc * an.x);
        rd = make_double2((rd.x - ra * dm.x - rc * dn.x) * inv, (rd.y - ra * dm.y - rc * dn.y) * inv);
        ra = -ra * am.x * inv;
        rc = -rc * an.y * inv;
        buf ^= 1;
    }
    D[buf][id] = rd;
    __syncthreads();
    const double2 before = q > 0 ? D[buf][id - MODES] : make_double2(0.0, 0.0);
    d[M - 1] = rd;
#pragma unroll
    for (int r = M - 2; r >= 0; --r)
        d[r] = make_double2(d[r].x - c[r] * d[r + 1].x - a[r] * before.x, d[r].y - c[r] * d[r + 1].y - a[r] * before.y);
    if (pin_block) {
        double2 own = make_double2(0.0, 0.0);
#pragma unroll
        for (int r = 0; r < M; ++r)
            if (j0 + r < ny) own = make_double2(own.x + d[r].x, own.y + d[r].y);
        const double2 sum = line_sum<MODES>(own, part);
        if (pinned) {
#pragma unroll
            for (int r = 0; r < M; ++r) d[r] = make_double2(d[r].x - sum.x / ny, d[r].y - sum.y / ny);
        }
    }
#pragma unroll
    for (int r = 0; r < M; ++r)
        if (kx < nh && j0 + r < ny) col[(size_t) (j0 + r) * ld] = d[r];
}

int log2_exact(int n)
{
    int l = 0;
    while ((1 << l) < n) ++l;
    return (1 << l) == n ? l : -1;
}

std::vector<double2> twiddles(int n)
{
    std::vector<double2> w(n / 2);
    const long double pi = 3.141592653589793238462643383279502884L;
    for (int m = 0; m < n / 2; ++m) {
        const long double a = -2.0L * pi * m / n;
        w[m] = make_double2((double) cosl(a), (double) sinl(a));
    }
    return w;
}

std::vector<double> eigenvalues(int n, double r2, int count)
{
    std::vector<double> l(count);
    const long double pi = 3.141592653589793238462643383279502884L;
    for (int k = 0; k < count; ++k) {
        const long double sn = sinl(pi * k / n);
        l[k] = (double) (-4.0L * (long double) r2 * sn * sn);
    }
    return l;
}

} // namespace
} // namespace ibm

struct ibm_fft {
    int device;
    int nx, ny, nz, nh, lx, lz;
    ibm::wall_axis y;
    bool neumann;                 // both walls Neumann: sigma = 0 is the singular (mean-free) case
    double2* spec = nullptr;      // nz x ny rows of nh coefficients, row stride spec_ld(nh)
    double2* twx = nullptr;
    double2* twz = nullptr;
    double* lam_x = nullptr;
    double* lam_z = nullptr;
    std::vector<void*> owned;
};

namespace ibm {

// Whether the FFT solver takes grid g (and why not).
static const char* fft_unsupported(const ibm_grid& g)
{
    if (g.axis[0].solid || g.axis[2].solid) return "x and z must be periodic";
    if (!g.axis[1].solid) return "y must be walled";
    const int nx = g.axis[0].points, nz = g.axis[2].points, ny = g.axis[1].points;
    if (log2_exact(nx) < 2 || log2_exact(nz) < 2 || nx > MAX_FFT_POINTS || nz > MAX_FFT_POINTS)
        return "x and z point counts must be powers of two from 4 to 512";
    if (ny < 2 || ny > MAX_WALL_POINTS) return "y must hold 2 to 800 points";
    return nullptr;
}

bool fft_usable(const ibm_grid& g) { return fft_unsupported(g) == nullptr; }

static ibm_status fft_alloc(ibm_ctx* ctx, ibm_fft* p, size_t bytes, void** out)
{
    IBM_HIP(ctx, hipMalloc(out, bytes));
    p->owned.push_back(*out);
    return IBM_OK;
}

// The plane kernels of nx x nz points, or null where the sizes are not among
// theirs: 32 to 128 each.  (256 x 32, 256 x 64, 512 x 32 and their transposes
// would fit the LDS too; they take the five passes.)
struct plane_kernels {
    void (*forward)(int, const double*, double2*, const double2*, const double2*);
    void (*inverse)(int, const double2*, double*, double, const double2*, const double2*);
    int threads;
    size_t lds;
};

template <int LX, int LZ>
static plane_kernels plane_of()
{
    return {plane_forward_kernel<LX, LZ>, plane_inverse_kernel<LX, LZ>, plane_size<LX, LZ>::THREADS, plane_size<LX, LZ>::LDS};
}

constexpr int PLANE_MIN = 5, PLANE_SIZES = 3;
static plane_kernels plane_kernels_of(int lx, int lz)
{
    static const plane_kernels table[PLANE_SIZES][PLANE_SIZES] = {{plane_of<5, 5>(), plane_of<5, 6>(), plane_of<5, 7>()},
                                                                  {plane_of<6, 5>(), plane_of<6, 6>(), plane_of<6, 7>()},
                                                                  {plane_of<7, 5>(), plane_of<7, 6>(), plane_of<7, 7>()}};
    const int i = lx - PLANE_MIN, k = lz - PLANE_MIN;
    return i >= 0 && i < PLANE_SIZES && k >= 0 && k < PLANE_SIZES ? table[i][k] : plane_kernels{};
}

static ibm_status fft_lds_attributes(ibm_ctx* ctx)
{
    // an attribute of a kernel on one device
    static std::mutex lock;
    static std::vector<bool> done;
    std::lock_guard<std::mutex> guard(lock);
    if ((int) done.size() <= ctx->device) done.resize(ctx->device + 1);
    if (done[ctx->device]) return IBM_OK;
    IBM_HIP(ctx, hipFuncSetAttribute((const void*) zfft_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int) MAX_DYNAMIC_LDS));
    for (int lx = PLANE_MIN; lx < PLANE_MIN + PLANE_SIZES; ++lx)
        for (int lz = PLANE_MIN; lz < PLANE_MIN + PLANE_SIZES; ++lz) {
            const plane_kernels k = plane_kernels_of(lx, lz);
            IBM_HIP(ctx, hipFuncSetAttribute((const void*) k.forward, hipFuncAttributeMaxDynamicSharedMemorySize, (int) k.lds));
            IBM_HIP(ctx, hipFuncSetAttribute((const void*) k.inverse, hipFuncAttributeMaxDynamicSharedMemorySize, (int) k.lds));
        }
    done[ctx->device] = true;
    return IBM_OK;
}

ibm_status fft_solve(ibm_ctx* ctx, ibm_fft* p, double sigma, double tau, const double* b, double* x)
{
    if (!ctx || !p) return IBM_ERR_ARG;
    if (!b || !x) return fail(ctx, IBM_ERR_ARG, "null vector");
    if (p->device != ctx->device) return fail(ctx, IBM_ERR_ARG, "FFT solver lives on another device");
    if (!std::isfinite(sigma) || !std::isfinite(tau)) return fail(ctx, IBM_ERR_ARG, "non-finite operator coefficients");
    const int rows = p->ny * p->nz;
    const double points = (double) p->nx * p->ny * p->nz, coeffs = (double) p->nh * p->ny * p->nz;
    const plane_kernels plane = plane_kernels_of(p->lx, p->lz);
    // Planes wherever their sizes fit: both transforms of 128 x ny x 128 points
    // take 27 (planes 14) us at ny = 128, 15 (12) at 32 and 10 (10) at 4; of
    // 32 x ny x 32 7 to 8 (4 to 5) at any ny.
    const bool by_planes = plane.forward != nullptr;
    // b read and x written once; the coefficients written and read twice by
    // planes, four times by passes
    prof_scope prof(ctx, "fft_solve", 8.0 * 2.0 * points + 16.0 * (by_planes ? 4.0 : 8.0) * coeffs);
    const int rpb = FFT_THREADS / (p->nx / 2);
    const size_t xlds = sizeof(double2) * (rpb * p->nx + p->nx / 2);
    const dim3 zgrid((p->nh + ZT - 1) / ZT, p->ny);
    const size_t zlds = sizeof(double2) * (ZT * p->nz + p->nz / 2);
    if (by_planes) {
        plane.forward<<<p->ny, plane.threads, plane.lds, ctx->stream>>>(p->ny, b, p->spec, p->twx, p->twz);
        IBM_LAUNCH_CHECK(ctx);
    } else {
        xfft_forward_kernel<<<(rows + rpb - 1) / rpb, FFT_THREADS, xlds, ctx->stream>>>(p->nx, p->lx, rows, b, p->spec,
                                                                                        p->twx);
        IBM_LAUNCH_CHECK(ctx);
        zfft_kernel<<<zgrid, FFT_THREADS, zlds, ctx->stream>>>(p->nh, p->ny, p->nz, p->lz, p->spec, p->twz, 0);
        IBM_LAUNCH_CHECK(ctx);
    }
    const int singular = sigma == 0.0 && p->neumann;
    auto lines = [&](auto kernel, int modes = LINE_MODES) {
        kernel<<<dim3((p->nh + modes - 1) / modes, p->nz), LINE_THREADS, 0, ctx->stream>>>(p->nh, p->y, sigma, tau, singular, p->lam_x, p->lam_z, p->spec);
    };
    if (p->ny <= SHORT_ROWS) lines(line_kernel<2, SHORT_MODES>, SHORT_MODES);
    else if (p->ny <= 2 * LINE_CHUNKS) lines(line_kernel<2>);
    else if (p->ny <= 4 * LINE_CHUNKS) lines(line_kernel<4>);
    else if (p->ny <= 8 * LINE_CHUNKS) lines(line_kernel<8>);
    else if (p->ny <= 16 * LINE_CHUNKS) lines(line_kernel<16>);
    else lines(line_kernel<(MAX_WALL_POINTS + LINE_CHUNKS - 1) / LINE_CHUNKS>);
    IBM_LAUNCH_CHECK(ctx);
    const double scale = 1.0 / ((double) p->nx * p->nz);
    if (by_planes) {
        plane.inverse<<<p->ny, plane.threads, plane.lds, ctx->stream>>>(p->ny, p->spec, x, scale, p->twx, p->twz);
        IBM_LAUNCH_CHECK(ctx);
        return IBM_OK;
    }
    zfft_kernel<<<zgrid, FFT_THREADS, zlds, ctx->stream>>>(p->nh, p->ny, p->nz, p->lz, p->spec, p->twz, 1);
    IBM_LAUNCH_CHECK(ctx);
    xfft_inverse_kernel<<<(rows + rpb - 1) / rpb, FFT_THREADS, xlds, ctx->stream>>>(p->nx, p->lx, rows, p->spec, x, scale,
                                                                                    p->twx);
    IBM_LAUNCH_CHECK(ctx);
    return IBM_OK;
}

} // namespace ibm

using namespace ibm;

extern "C" {

ibm_status ibm_fft_create(ibm_ctx* ctx, const ibm_grid* g, ibm_fft** out)
{
    if (!ctx || !g || !out) return IBM_ERR_ARG;
    *out = nullptr;
    if (const char* why = fft_unsupported(*g)) return fail(ctx, IBM_ERR_BAD_GRID, "FFT solver: %s", why);
    IBM_TRY(fft_lds_attributes(ctx));
    auto* p = new ibm_fft;
    p->device = ctx->device;
    p->nx = g->axis[0].points;
    p->ny = g->axis[1].points;
    p->nz = g->axis[2].points;
    p->nh = p->nx / 2 + 1;
    p->lx = log2_exact(p->nx);
    p->lz = log2_exact(p->nz);
    const op_axis<double> ya = make_op_axis<double>(g->axis[1]);
    p->y = wall_axis{ya.n, ya.r2, ya.lap_lo, ya.lap_hi, ya.id_lo, ya.id_hi};
    p->neumann = g->axis[1].interior[0] == 1.0 && g->axis[1].interior[1] == 1.0;
    const std::vector<double2> twx = twiddles(p->nx), twz = twiddles(p->nz);
    const std::vector<double> lx = eigenvalues(p->nx, g->axis[0].resolution * g->axis[0].resolution, p->nh);
    const std::vector<double> lz = eigenvalues(p->nz, g->axis[2].resolution * g->axis[2].resolution, p->nz);
    void* m = nullptr;
    ibm_status st = IBM_OK;
    if ((st = fft_alloc(ctx, p, sizeof(double2) * spec_ld(p->nh) * p->ny * (size_t) p->nz, &m)) == IBM_OK) {
        p->spec = (double2*) m;
        st = fft_alloc(ctx, p, sizeof(double2) * twx.size(), &m);
    }
    if (st == IBM_OK) {
        p->twx = (double2*) m;
        st = fft_alloc(ctx, p, sizeof(double2) * twz.size(), &m);
    }
    if (st == IBM_OK) {
        p->twz = (double2*) m;
        st = fft_alloc(ctx, p, sizeof(double) * lx.size(), &m);
    }
    if (st == IBM_OK) {
        p->lam_x = (double*) m;
        st = fft_alloc(ctx, p, sizeof(double) * lz.size(), &m);
    }
    if (st == IBM_OK) {
        p->lam_z = (double*) m;
        if (hipMemcpy(p->twx, twx.data(), sizeof(double2) * twx.size(), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(p->twz, twz.data(), sizeof(double2) * twz.size(), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(p->lam_x, lx.data(), sizeof(double) * lx.size(), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(p->lam_z, lz.data(), sizeof(double) * lz.size(), hipMemcpyHostToDevice) != hipSuccess)
            st = fail(ctx, IBM_ERR_HIP, "FFT solver: table upload failed");
    }
    if (st != IBM_OK) {
        for (void* q : p->owned) hipFree(q);
        delete p;
        return st;
    }
    *out = p;
    return IBM_OK;
}

ibm_status ibm_fft_destroy(ibm_fft* p)
{
    if (!p) return IBM_OK;
    hipDeviceSynchronize();
    for (void* q : p->owned) hipFree(q);
    delete p;
    return IBM_OK;
}

ibm_status ibm_fft_solve(ibm_ctx* ctx, ibm_fft* p, double sigma, double tau, const double* b, double* x)
{
    return ibm::fft_solve(ctx, p, sigma, tau, b, x);
}

} // extern "C"
