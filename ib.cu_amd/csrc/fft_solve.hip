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
// multigrid iterates on, in five memory passes.  The singular case (sigma = 0 with
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

// Sum over a workgroup's LINE_CHUNKS chunks of the lanes with t = 0.
__device__ inline double2 line_sum(double2 v, double2* part)
{
    __syncthreads();
    if (threadIdx.x % LINE_MODES == 0) part[threadIdx.x / LINE_MODES] = v;
    __syncthreads();
    double2 m = make_double2(0.0, 0.0);
    for (int i = 0; i < LINE_CHUNKS; ++i) {
        m.x += part[i].x;
        m.y += part[i].y;
    }
    return m;
}

// Every Fourier mode's tridiagonal system along y: block (tile of LINE_MODES
// kx, kz), one thread per mode and chunk of M consecutive rows, which it keeps
// in registers (rows past ny are identity rows).  A forward elimination leaves
// row r as X_r = d_r - c_r X_{r+1} - a_r X_{-1}, with X_{-1} the last row of
// the chunk before, and a backward one gives the first row by the chunk's and
// the previous chunk's last; put into the previous chunk's last row that is
// one equation per chunk, solved by cyclic reduction over the LINE_CHUNKS of
// them, and a back substitution ends it.  The singular mode's last equation is
// replaced by x = 0 after its right-hand side loses its mean, and its solution
// loses its mean.  Bound by memory (16 bytes per row read and written, whole
// 128-byte lines): cyclic reduction over all rows in LDS took two divisions
// per row and step, eight in all, this one and a fraction.  65 x 256 x 128
// coefficients: 48 us / 17.
template <int M>
__global__ void __launch_bounds__(LINE_THREADS) line_kernel(int nh, wall_axis y, double sigma, double tau, int singular,
                                                            const double* __restrict__ lam_x,
                                                            const double* __restrict__ lam_z, double2* __restrict__ s)
{
    __shared__ double2 D[2][LINE_THREADS];
    __shared__ double2 AC[2][LINE_THREADS];
    __shared__ double2 part[LINE_CHUNKS];
    const int ny = y.n, t = threadIdx.x % LINE_MODES, q = threadIdx.x / LINE_MODES;
    const int kx = blockIdx.x * LINE_MODES + t, kz = blockIdx.y, j0 = q * M;
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
        const double2 sum = line_sum(own, part);
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
    if (q + 1 < LINE_CHUNKS) {
        const double2 np = D[0][id + LINE_MODES], nfg = AC[0][id + LINE_MODES];
        const double inv = 1.0 / (1.0 - c[M - 1] * nfg.x);
        ra *= inv;
        rc = -c[M - 1] * nfg.y * inv;
        rd = make_double2((rd.x - c[M - 1] * np.x) * inv, (rd.y - c[M - 1] * np.y) * inv);
    }
    if (q == 0) ra = 0.0;
    // cyclic reduction of X_q + ra X_{q-1} + rc X_{q+1} = rd
    int buf = 1;
#pragma unroll
    for (int sft = 1; sft < LINE_CHUNKS; sft <<= 1) {
        D[buf][id] = rd;
        AC[buf][id] = make_double2(ra, rc);
        __syncthreads();
        double2 dm = make_double2(0.0, 0.0), dn = dm, am = dm, an = dm;
        if (q >= sft) {
            dm = D[buf][id - sft * LINE_MODES];
            am = AC[buf][id - sft * LINE_MODES];
        }
        if (q + sft < LINE_CHUNKS) {
            dn = D[buf][id + sft * LINE_MODES];
            an = AC[buf][id + sft * LINE_MODES];
        }
        const double inv = 1.0 / (1.0 - ra * am.y - rc * an.x);
        rd = make_double2((rd.x - ra * dm.x - rc * dn.x) * inv, (rd.y - ra * dm.y - rc * dn.y) * inv);
        ra = -ra * am.x * inv;
        rc = -rc * an.y * inv;
        buf ^= 1;
    }
    D[buf][id] = rd;
    __syncthreads();
    const double2 before = q > 0 ? D[buf][id - LINE_MODES] : make_double2(0.0, 0.0);
    d[M - 1] = rd;
#pragma unroll
    for (int r = M - 2; r >= 0; --r)
        d[r] = make_double2(d[r].x - c[r] * d[r + 1].x - a[r] * before.x, d[r].y - c[r] * d[r + 1].y - a[r] * before.y);
    if (pin_block) {
        double2 own = make_double2(0.0, 0.0);
#pragma unroll
        for (int r = 0; r < M; ++r)
            if (j0 + r < ny) own = make_double2(own.x + d[r].x, own.y + d[r].y);
        const double2 sum = line_sum(own, part);
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

static ibm_status fft_lds_attributes(ibm_ctx* ctx)
{
    static std::mutex lock;
    static bool done = false;
    std::lock_guard<std::mutex> guard(lock);
    if (done) return IBM_OK;
    IBM_HIP(ctx, hipFuncSetAttribute((const void*) zfft_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int) MAX_DYNAMIC_LDS));
    done = true;
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
    // b read and x written once; the coefficients written and read four times
    prof_scope prof(ctx, "fft_solve", 8.0 * 2.0 * points + 16.0 * 8.0 * coeffs);
    const int rpb = FFT_THREADS / (p->nx / 2);
    const size_t xlds = sizeof(double2) * (rpb * p->nx + p->nx / 2);
    xfft_forward_kernel<<<(rows + rpb - 1) / rpb, FFT_THREADS, xlds, ctx->stream>>>(p->nx, p->lx, rows, b, p->spec,
                                                                                      p->twx);
    IBM_LAUNCH_CHECK(ctx);
    const dim3 zgrid((p->nh + ZT - 1) / ZT, p->ny);
    const size_t zlds = sizeof(double2) * (ZT * p->nz + p->nz / 2);
    zfft_kernel<<<zgrid, FFT_THREADS, zlds, ctx->stream>>>(p->nh, p->ny, p->nz, p->lz, p->spec, p->twz, 0);
    IBM_LAUNCH_CHECK(ctx);
    const int singular = sigma == 0.0 && p->neumann;
    const dim3 tgrid((p->nh + LINE_MODES - 1) / LINE_MODES, p->nz);
    auto lines = [&](auto kernel) {
        kernel<<<tgrid, LINE_THREADS, 0, ctx->stream>>>(p->nh, p->y, sigma, tau, singular, p->lam_x, p->lam_z, p->spec);
    };
    if (p->ny <= 2 * LINE_CHUNKS) lines(line_kernel<2>);
    else if (p->ny <= 4 * LINE_CHUNKS) lines(line_kernel<4>);
    else if (p->ny <= 8 * LINE_CHUNKS) lines(line_kernel<8>);
    else if (p->ny <= 16 * LINE_CHUNKS) lines(line_kernel<16>);
    else lines(line_kernel<(MAX_WALL_POINTS + LINE_CHUNKS - 1) / LINE_CHUNKS>);
    IBM_LAUNCH_CHECK(ctx);
    zfft_kernel<<<zgrid, FFT_THREADS, zlds, ctx->stream>>>(p->nh, p->ny, p->nz, p->lz, p->spec, p->twz, 1);
    IBM_LAUNCH_CHECK(ctx);
    xfft_inverse_kernel<<<(rows + rpb - 1) / rpb, FFT_THREADS, xlds, ctx->stream>>>(
        p->nx, p->lx, rows, p->spec, x, 1.0 / ((double) p->nx * p->nz), p->twx);
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
