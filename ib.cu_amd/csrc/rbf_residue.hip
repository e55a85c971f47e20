// FP64 matrix products through the INT8 matrix cores (the residue-number
// form of the Ozaki scheme: K. Ozaki, Y. Uchino, T. Imamura, "Ozaki Scheme
// II", 2025).
//
// Row m of the operator and column n of X are scaled by powers of two and
// rounded to integers E'_mk, X'_kn; their exact integer product
//   C_mn = sum_k E'_mk X'_kn
// is found from its residues modulo RES_MODULI coprime moduli p_l <= 256,
// each an INT8 matrix product of the operands' residues (exact in INT32),
// and the Chinese remainder theorem puts C back together; Y = C / (scales).
// The scales are
//   sum_k |E'_mk| <= 2^62,   max_k |X'_kn| <= 2^54,
// so |C| <= 2^116 < P / 2, P = prod p_l = 2^117.8, and the only errors are
// the operands' rounding and one rounding of the result:
//   |Y - E X|_mn <= 2^(ex - 55) sum_k |E_mk| + 2^(e - 63) sum_k |X_kn|
//                   + 2^-53 |Y_mn|,
// 2^e and 2^ex the powers of two above row m's 1-norm and column n's maximum.
// That is a bound on norms.  An FP64 chain of fused multiply-adds is within
// K 2^-53 sum_k |E_mk||X_kn| of each output, which can be far less where a
// row's weight lies on a column's small values; so every column is checked,
// and one that could exceed the chain's bound anywhere (plus the last
// rounding) goes to the FP64 matrix cores:
//   * a column whose values are all of one magnitude, more or less
//     (COLUMN_NARROW; column_scale_kernel), cannot: sum_k |E_mk||X_kn| >=
//     min_k |X_kn| sum_k |E_mk|.  Coordinates of a cell that does not lie
//     across a coordinate plane are such columns;
//   * of others (COLUMN_WIDE) a sixteenth product bounds sum_k |E_mk||X_kn|
//     from below for every output: magnitudes rounded down to seven bits,
//     S = sum_k floor(2^(7 - em) |E_mk|) floor(2^(7 - ex) |X_kn|) in INT32,
//     2^em the power of two above row m's maximum, and
//     S 2^(em + ex - 14) <= sum_k |E_mk||X_kn|.  For the few outputs below
//     their row's threshold the sum itself is formed; one that is too small
//     sends its column to the FP64 products;
//   * columns of mostly negligible values (which would fail), or with a NaN
//     or an infinity, go there at once (COLUMN_F64).
// Measured on the RBC and platelet operators (values and all derivatives, 300
// to 2210 data sites) against long-double products, the error is 0.03 to 0.66
// of the FP64 fused multiply-add chain's in the 2-norm and 0.01 to 0.74 in
// the maximum; one modulus fewer (2^109) would be 4 to 65 times the chain's.
//
// What bounds it: FP64 matrix cores are dense at 78.6 TFLOP/s (measured 72.6
// for a large library product), INT8 at 5.0 POP/s; with random operands the
// card's power budget holds a register-only INT8 loop to 3.9 POP/s
// (16 x 16 x 64; 3.1 with 32 x 32 x 32, which moves twice the accumulators
// per product) and these products to 1.9 to 2.1 (2.3 to 2.9 on operands of
// zeros), so 15 products are worth about 120 FP64 TFLOP/s.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <vector>
#include "rbf_residue.hpp"

namespace ibm {
namespace {

typedef int i4 __attribute__((ext_vector_type(4)));
typedef unsigned __int128 u128;

// The largest fifteen pairwise coprime moduli up to 256: residues fit a
// signed byte (-128 stands for 128 modulo 256).
constexpr int P[RES_MODULI] = {256, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197};

constexpr u128 product()
{
    u128 v = 1;
    for (int p : P) v *= (unsigned) p;
    return v;
}

// W_l = (P / p_l) ((P / p_l)^-1 mod p_l): sum_l W_l r_l = C mod P.
constexpr u128 weight(int l)
{
    const u128 q = product() / (unsigned) P[l];
    const int m = (int) (q % (unsigned) P[l]);
    int inv = 1;
    while (m * inv % P[l] != 1) ++inv;
    return q * (unsigned) inv;
}

// High part: a multiple of 2^77, so that sums of 15 of them times residues
// (below 15 * 2^117.8 * 2^7 < 2^129) and multiples of P's high part are
// exact in FP64; the low parts are below 2^77, their sums below 2^88, and
// enter with FP64 rounding: 2^35 to 2^39 units of C, 2^-77 of its bound or
// less.
constexpr int HIGH = 77;
constexpr double high_part(u128 v) { return (double) (unsigned long long) (v >> HIGH) * 0x1p77; }
constexpr double low_part(u128 v)
{
    const u128 r = v & (((u128) 1 << HIGH) - 1);
    return (double) (unsigned long long) (r >> 40) * 0x1p40 + (double) (unsigned long long) (r & ((1ull << 40) - 1));
}

struct crt_table {
    double hi[RES_MODULI], lo[RES_MODULI];
    double p_hi, p_lo, p_inv;
};

constexpr crt_table make_crt()
{
    crt_table t{};
    for (int l = 0; l < RES_MODULI; ++l) {
        t.hi[l] = high_part(weight(l));
        t.lo[l] = low_part(weight(l));
    }
    t.p_hi = high_part(product());
    t.p_lo = low_part(product());
    t.p_inv = 1.0 / t.p_hi;
    return t;
}

constexpr int SCALE_E = 62, SCALE_X = 54;

// 1.5 * 2^52: x + ROUND holds rint(x) in its low bits (|x| < 2^51), so that
// x + ROUND - ROUND is rint(x) and the low word of x + ROUND, for an integer
// x, is x modulo 2^32.  Additions and fused multiply-adds run at full rate;
// v_rndne_f64 and the conversions between FP64 and integers do not.
constexpr double ROUND = 0x1.8p52;
__device__ inline double nearest(double x, double y) { return fma(x, y, ROUND) - ROUND; }     // rint(x y)
__device__ inline unsigned low_word(double x) { return (unsigned) __double2loint(x + ROUND); }
// (double) v
__device__ inline double from_int(int v)
{
    return __hiloint2double(0x43300000, (int) ((unsigned) v ^ 0x80000000u)) - (0x1p52 + 0x1p31);
}

// 2^31 modulo p in [-p/2, p/2].
constexpr int fold(int l)
{
    const int m = (int) ((1ll << 31) % P[l]);
    return 2 * m > P[l] ? m - P[l] : m;
}

// Sixteen consecutive elements' residues modulo the moduli [L0, L1), one
// 16-byte store each: fragments of the 16 x 16 x 64 INT8 instruction are
// 1 KB, lane (row & 15) + 16 (k / 16), 16 bytes of k each.  An element is
// h 2^31 + d, |h| <= 2^31, |d| <= 2^30: its residue is that of
// h (2^31 mod p) + d, below 2^39 and exact, whose quotient by p is the
// nearest integer exactly (2^39 / p times FP64's rounding is far below the
// distance 1 / (2 p) of a quotient from a tie; p = 256 divides exactly, where
// either end of a tie is the same byte).
template <int L0, int L1>
__device__ inline void store_residues(const double (&h)[16], const double (&d)[16], unsigned char* at, size_t plane)
{
#pragma unroll
    for (int l = L0; l < L1; ++l) {
        const double p = P[l], inv = 1.0 / P[l], f = fold(l);
        i4 w;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            unsigned v = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double t = fma(h[4 * q + i], f, d[4 * q + i]);
                v |= (low_word(fma(-p, nearest(t, inv), t)) & 255) << (8 * i);
            }
            w[q] = (int) v;
        }
        *(i4*) (at + l * plane) = w;
    }
}

// The integer rint(x 2^s), |.| <= 2^62, as h 2^31 + d.
__device__ inline void split_element(double x, int s, double& h, double& d)
{
    const double v = rint(ldexp(x, s));
    h = rint(v * 0x1p-31);
    d = fma(-0x1p31, h, v);
}

// Byte offset of the 16-byte run (row, k0 = 16 run) inside a residue plane.
__device__ inline size_t run_offset(int row, int run, int chunks)
{
    return ((size_t) (row >> 4) * chunks + (run >> 2)) * 1024 + ((row & 15) + 16 * (run & 3)) * 16;
}

// Sixteen consecutive elements' magnitudes in seven bits, |x| < 2^e.
__device__ inline void store_magnitudes(const double (&x)[16], int e, unsigned char* at)
{
    i4 w;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        unsigned v = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) v |= (unsigned) ldexp(fabs(x[4 * q + i]), 7 - e) << (8 * i);
        w[q] = (int) v;
    }
    *(i4*) at = w;
}

// Of operator row m (one wavefront per row): the scale 2^(62 - e), sum |E| <
// 2^e, of its integers; the exponent em of its maximum; and the least
// magnitude product S for which the operands' rounding stays within the
// chain's bound,
//   2^(ex - 55) sum |E| + 2^(e - 63) K 2^ex <= K 2^-53 S 2^(em + ex - 14),
// i.e. S >= 2^(12 - em) sum |E| / K + 2^(e - em + 4).
__global__ __launch_bounds__(256) void operator_scale_kernel(const double* __restrict__ E, long lde, int M, int K,
                                                             int* __restrict__ scale, int* __restrict__ top,
                                                             int* __restrict__ least, int* __restrict__ flag)
{
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (m >= M) return;
    double s = 0, t = 0;
    for (int k = lane; k < K; k += 64) {
        const double v = fabs(E[k + lde * m]);
        s += v;
        t = fmax(t, v);
    }
    for (int off = 32; off > 0; off >>= 1) {
        s += __shfl_xor(s, off, 64);
        t = fmax(t, __shfl_xor(t, off, 64));
    }
    if (lane == 0) {
        int e = 0, em = 0, bound = 0;
        if (!isfinite(s)) {
            *flag = 1;
        } else if (s > 0) {
            frexp(s * (1 + 0x1p-40), &e);      // the sum's own rounding
            frexp(t, &em);
            bound = (int) (ldexp(s, 12 - em) / K + ldexp(16.0, e - em)) + 2;
        }
        scale[m] = SCALE_E - e;
        top[m] = em;
        least[m] = bound;
    }
}

__global__ __launch_bounds__(256) void operator_split_kernel(const double* __restrict__ E, long lde, int M, int K,
                                                             int rows, int chunks, const int* __restrict__ scale,
                                                             const int* __restrict__ top,
                                                             unsigned char* __restrict__ planes, size_t plane)
{
    const long i = (long) blockIdx.x * 256 + threadIdx.x;
    const int runs = chunks * 4;
    if (i >= (long) rows * runs) return;
    // consecutive lanes take the 16 rows of a fragment, then its runs of k
    const int frag_row = (int) (i / ((long) runs * 16)), in = (int) (i - (long) frag_row * runs * 16);
    const int row = frag_row * 16 + (in & 15), run = in >> 4;
    double x[16], h[16], d[16];
    const int s = row < M ? scale[row] : 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int k = run * 16 + j;
        x[j] = row < M && k < K ? E[k + lde * row] : 0.0;
        split_element(x[j], s, h[j], d[j]);
    }
    unsigned char* at = planes + run_offset(row, run, chunks);
    store_residues<0, RES_MODULI>(h, d, at, plane);
    store_magnitudes(x, row < M ? top[row] : 0, at + RES_MODULI * plane);
}

struct column_part {
    const double* X;
    res_packed to;
    int N, K;
};
struct column_set {
    column_part c[RES_MAX_COLUMNS];
};

// Scale 2^(54 - ex) of column n's integers, max |x| < 2^ex, and its class; one
// block per column.  Narrow: the operands' rounding is within the chain's
// bound for every row,
//   2^(ex - 55) + 2^-62 sum |x| <= K 2^-53 min |x|
// (2^e <= 2 sum |E|): 1 : 800 for 2210 values of even distribution.  Columns
// of which more than half lies below 2^-7 of the maximum have no seven-bit
// magnitudes to speak of; those of a maximum below 2^-1000 are left to FP64 as
// the sums here would underflow.
// Also clears the flags of the products that follow.
__global__ __launch_bounds__(256) void column_scale_kernel(column_set set, int* __restrict__ flags, int nflags)
{
    for (int i = (int) (blockIdx.y * gridDim.x + blockIdx.x) * 256 + (int) threadIdx.x; i < nflags;
         i += (int) (gridDim.x * gridDim.y) * 256)
        flags[i] = 0;
    __shared__ double part[3][4];
    __shared__ int small[4];
    const column_part& c = set.c[blockIdx.y];
    const int n = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (n >= c.N) return;                                      // whole block
    const int K = c.K;
    const double* x = c.X + (size_t) n * K;
    double top = 0, low = INFINITY, sum = 0;                   // sum: in units of 2^20, so that it cannot overflow
#pragma unroll 8
    for (int k = threadIdx.x; k < K; k += 256) {
        const double v = fabs(x[k]);
        top = isfinite(v) ? fmax(top, v) : INFINITY;
        low = fmin(low, v);
        sum += v * 0x1p-20;
    }
    for (int off = 32; off > 0; off >>= 1) {
        top = fmax(top, __shfl_xor(top, off, 64));
        low = fmin(low, __shfl_xor(low, off, 64));
        sum += __shfl_xor(sum, off, 64);
    }
    if (lane == 0) {
        part[0][wave] = top;
        part[1][wave] = low;
        part[2][wave] = sum;
    }
    __syncthreads();
    top = fmax(fmax(part[0][0], part[0][1]), fmax(part[0][2], part[0][3]));
    low = fmin(fmin(part[1][0], part[1][1]), fmin(part[1][2], part[1][3]));
    sum = (part[2][0] + part[2][1]) + (part[2][2] + part[2][3]);
    int ex = 0, kind = COLUMN_F64;
    if (top == 0) {
        kind = COLUMN_NARROW;
    } else if (top >= 0x1p-1000 && isfinite(top)) {
        frexp(top, &ex);
        if (ldexp(1.0, ex - 22) + 0x1p-9 * sum <= K * 0x1p-20 * low) {
            kind = COLUMN_NARROW;
        } else {
            int below = 0;
            for (int k = threadIdx.x; k < K; k += 256) below += fabs(x[k]) < 0x1p-7 * top;
            for (int off = 32; off > 0; off >>= 1) below += __shfl_xor(below, off, 64);
            if (lane == 0) small[wave] = below;
            __syncthreads();
            kind = 2 * (small[0] + small[1] + small[2] + small[3]) > K ? COLUMN_F64 : COLUMN_WIDE;
        }
    }
    if (threadIdx.x == 0) {
        c.to.scale[n] = SCALE_X - ex;
        c.to.kind[n] = kind;
    }
}

// Residues of 16 columns x 256 elements for a third of the moduli
// (blockIdx.z; the last third also writes the magnitudes, and the FP64 rows of
// the columns that may need them): rows of 2 KB staged through LDS, so that
// both the loads and the 1 KB fragment stores are contiguous (one block per
// column, whose threads load and store scattered 128- and 16-byte pieces:
// 41 us for 600 columns of 2210 elements).  Padding columns, and those
// without residues, get zeros.
constexpr int SPLIT_PARTS = 3, SPLIT_K = 256, SPLIT_LD = SPLIT_K + SPLIT_K / 16 + 1;
static_assert(RES_MODULI == 15);

__global__ __launch_bounds__(256) void column_split_kernel(column_set set, int k_blocks)
{
    __shared__ double sx[16][SPLIT_LD];                        // element k at k + k / 16
    __shared__ int kinds[16];
    const column_part& c = set.c[blockIdx.y];
    const int N = c.N, K = c.K;
    const int chunks = (K + 63) / 64, runs = chunks * 4;
    const int rows = (N + RES_BN - 1) / RES_BN * RES_BN;
    const int n0 = (int) (blockIdx.x / k_blocks) * 16, k0 = (int) (blockIdx.x % k_blocks) * SPLIT_K;
    if (n0 >= rows || k0 >= K) return;                         // whole block
    for (int i = threadIdx.x; i < 16 * SPLIT_K; i += 256) {
        const int r = i / SPLIT_K, k = i - r * SPLIT_K;
        sx[r][k + (k >> 4)] = n0 + r < N && k0 + k < K ? c.X[(size_t) (n0 + r) * K + k0 + k] : 0.0;
    }
    if (threadIdx.x < 16) kinds[threadIdx.x] = n0 + (int) threadIdx.x < N ? c.to.kind[n0 + threadIdx.x] : -1;
    __syncthreads();
    if (blockIdx.z == 0 && k0 == 0 && threadIdx.x == 0) {
        int live = 0;
        for (int r = 0; r < 16; ++r) live |= (kinds[r] == COLUMN_NARROW || kinds[r] == COLUMN_WIDE) | (kinds[r] == COLUMN_WIDE) << 1;
        c.to.live[n0 / 16] = live;
    }
    if (blockIdx.z == 2)
        for (int r = 0; r < 16; ++r) {
            const int k = threadIdx.x;
            if (kinds[r] > COLUMN_NARROW && k0 + k < (int) c.to.ld)
                c.to.rows[(size_t) (n0 + r) * c.to.ld + k0 + k] = sx[r][k + (k >> 4)];
        }
    const int r = threadIdx.x & 15, run = threadIdx.x >> 4;
    if (k0 / 16 + run >= runs) return;
    const bool has = kinds[r] == COLUMN_NARROW || kinds[r] == COLUMN_WIDE;
    const int s = has ? c.to.scale[n0 + r] : 0;
    double x[16], h[16], d[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        x[j] = has ? sx[r][run * 17 + j] : 0.0;
        split_element(x[j], s, h[j], d[j]);
    }
    unsigned char* at = c.to.planes + run_offset(n0 + r, k0 / 16 + run, chunks);
    const size_t plane = (size_t) rows * chunks * 64;
    if (blockIdx.z == 0) {
        store_residues<0, 5>(h, d, at, plane);
    } else if (blockIdx.z == 1) {
        store_residues<5, 10>(h, d, at, plane);
    } else {
        store_residues<10, 15>(h, d, at, plane);
        store_magnitudes(x, SCALE_X - s, at + RES_MODULI * plane);
    }
}

// ----------------------------------------------------------------------
// The INT8 products.  One block computes one 256 x 128 tile modulo one
// modulus and leaves each output's residue as a byte: eight waves of 64 x 64
// outputs (4 x 4 fragments of 16 x 16), the operands' fragments staged as
// they lie in memory (1 KB each, read conflict-free) by direct-to-LDS loads
// into three buffers, two 64-element chunks ahead of the one multiplied, one
// barrier a chunk.  Units (tile, modulus) rather than whole tiles keep the
// last wave of blocks short.  One operator 8832 x 2210 x 600 takes 0.19 ms (a
// sixth of six); relative to that, four waves of 64 x 128 1.04, 128 x 128
// tiles 1.08, 256 x 256 tiles 1.32 (padding of the 600 columns), 32 x 32 x 32
// instructions with two buffers 1.06.
// ----------------------------------------------------------------------
constexpr int WM = 4, WN = 2, FM = 4, FN = 4;          // waves and fragments per wave
constexpr int WAVES = WM * WN, EF = WM * FM, XF = WN * FN, LOADS = (EF + XF) / WAVES;
constexpr int RES_THREADS = 64 * WAVES;
static_assert(EF * 16 == RES_BM && XF * 16 == RES_BN && LOADS * WAVES == EF + XF);

struct unit_group {
    const unsigned char* E;
    const unsigned char* X;
    const double* E64;           // FP64 rows of the operator and of the wide columns,
    const double* X64;           // 64 * chunks apart
    const int* e_scale;          // per row of the operator
    const int* least;            // per row, see operator_scale_kernel
    const int* x_scale;          // per column
    const int* kind;             // per column
    const int* live;             // per 16 columns
    int* flags;                  // per column: set where an output could exceed the chain's bound
    size_t e_plane, x_plane;     // bytes of one modulus' plane
    int M, N, K;
    int chunks, tiles_n;
    int tile0, tiles;            // tiles [tile0, tile0 + tiles) of the product, here tiles first_tile..
    int first_tile;
};
struct unit_groups {
    unit_group g[RBF_MAX_GROUPS];
    int count, pad;
};

__device__ inline void lds_load16(const void* g, void* l)
{
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) unsigned int*) g,
                                     (__attribute__((address_space(3))) unsigned int*) l, 16, 0, 0);
}

__global__ __launch_bounds__(RES_THREADS, 4) void residue_gemm_kernel(unit_groups G, unsigned* __restrict__ out)
{
    __shared__ __attribute__((aligned(16))) unsigned char s0[EF + XF][1024];
    __shared__ __attribute__((aligned(16))) unsigned char s1[EF + XF][1024];
    __shared__ __attribute__((aligned(16))) unsigned char s2[EF + XF][1024];
    // Blocks reach the XCDs round-robin: XCD x takes the x-th eighth of every
    // group's units, in order (modulus, row tile, column tile), so that the
    // blocks sharing an operator row tile and a modulus' columns share an L2;
    // then its eighth of the magnitude products, most of which have nothing
    // to do.
    const int xcd = blockIdx.x & 7;
    int k = blockIdx.x >> 3, gi = -1, l = 0, local = 0;
    for (int q = 0; q < G.count; ++q) {
        const long n = (long) G.g[q].tiles * RES_MODULI;
        const int lo = (int) (xcd * n / 8), hi = (int) ((xcd + 1) * n / 8);
        if (k < hi - lo) {
            gi = q;
            l = (lo + k) / G.g[q].tiles;
            local = lo + k - l * G.g[q].tiles;
            break;
        }
        k -= hi - lo;
    }
    if (gi < 0)
        for (int q = 0; q < G.count; ++q) {
            const int n = G.g[q].tiles, lo = xcd * n / 8, hi = (xcd + 1) * n / 8;
            if (k < hi - lo) {
                gi = q;
                l = RES_MODULI;
                local = lo + k;
                break;
            }
            k -= hi - lo;
        }
    if (gi < 0) return;                              // whole block exits together
    const unit_group g = G.g[gi];
    const int t = g.tile0 + local, tm = t / g.tiles_n, tn = t - tm * g.tiles_n;
    int live = 0;
#pragma unroll
    for (int i = 0; i < XF; ++i) live |= g.live[tn * XF + i];
    if (!(live & (l == RES_MODULI ? 2 : 1))) return;           // whole block
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const size_t frag_row = (size_t) g.chunks * 1024;
    const unsigned char* src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int f = wave * LOADS + i;
        src[i] = (f < EF ? g.E + l * g.e_plane + ((size_t) tm * EF + f) * frag_row
                         : g.X + l * g.x_plane + ((size_t) tn * XF + (f - EF)) * frag_row) + lane * 16;
    }
    i4 acc[FM][FN];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b) acc[a][b] = i4{};
    // Chunk c into a buffer; past the end the last chunk again (not used), so
    // that every chunk issues LOADS loads and the counted wait below holds.
    auto load = [&](int c, unsigned char (*buf)[1024]) {
        const size_t o = (size_t) min(c, g.chunks - 1) * 1024;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) lds_load16(src[i] + o, &buf[wave * LOADS + i][0]);
    };
    // One chunk: wait until this wave's loads of it have landed (those of the
    // next chunk stay in flight) and its fragment reads of the previous chunk
    // are done, then for every wave; the loads two chunks ahead may then
    // overwrite the previous chunk's buffer.
    auto chunk = [&](int c, unsigned char (*buf)[1024], unsigned char (*ahead)[1024]) {
        __builtin_amdgcn_s_waitcnt(LOADS | (7 << 4));          // vmcnt(LOADS), lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        load(c + 2, ahead);
        __builtin_amdgcn_sched_barrier(0);
        i4 e[FM];
#pragma unroll
        for (int a = 0; a < FM; ++a) e[a] = *(const i4*) (&buf[wm * FM + a][lane * 16]);
#pragma unroll
        for (int b = 0; b < FN; ++b) {
            const i4 x = *(const i4*) (&buf[EF + wn * FN + b][lane * 16]);
#pragma unroll
            for (int a = 0; a < FM; ++a) acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x, e[a], acc[a][b], 0, 0, 0);
        }
    };
    load(0, s0);
    load(1, s1);
    int c = 0;
    for (; c + 3 <= g.chunks; c += 3) {
        chunk(c, s0, s2);
        chunk(c + 1, s1, s0);
        chunk(c + 2, s2, s1);
    }
    if (c < g.chunks) {
        chunk(c, s0, s2);
        if (c + 1 < g.chunks) chunk(c + 1, s1, s0);
    }
    __builtin_amdgcn_s_waitcnt(7 << 4);                        // no load into LDS outlives the block
    // The first operand's rows are columns of Y: a lane holds rows
    // 4 (lane / 16) + i of X's fragment at sample lane % 16.
    if (l == RES_MODULI) {
        // Magnitudes: outputs of wide columns below their row's bound.  Mostly
        // that is the seven bits' doing (a sample beside a data site whose
        // value is below 2^-7 of the column's largest: some tens among the
        // five million outputs of an operator on cells that lie across a
        // coordinate plane), and the FP64 pass for a single column costs a
        // fifth of the whole evaluation.  So a wavefront lists its outputs and
        // forms their sums, all lanes together.  A column with more than
        // REFINED of them among the wavefront's 64 rows is flagged at once
        // (its own outputs decide, whatever its neighbours hold).
        constexpr int REFINED = 4;
        static_assert(REFINED * 16 * FN * sizeof(int) <= sizeof(s0[0]));
        __syncthreads();                                       // s0 is free
        int* listed = (int*) s0[wave];
        int count = 0;
#pragma unroll
        for (int b = 0; b < FN; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = tn * RES_BN + (wn * FN + b) * 16 + 4 * (lane >> 4) + i;
                const bool wide = n < g.N && g.kind[n] == COLUMN_WIDE;
                unsigned long long below[FM];
                int found = 0;                                 // of column n
#pragma unroll
                for (int a = 0; a < FM; ++a) {
                    const int m = tm * RES_BM + (wm * FM + a) * 16 + (lane & 15);
                    below[a] = __ballot(wide && m < g.M && acc[a][b][i] < g.least[m]);
                    found += __popcll(below[a] >> (lane & 48) & 0xffff);
                }
                const bool many = found > REFINED;
                if (many && (lane & 15) == 0) g.flags[n] = 1;
#pragma unroll
                for (int a = 0; a < FM; ++a) {
                    const bool own = !many && (below[a] >> lane & 1);
                    const unsigned long long mask = __ballot(own);
                    if (own)
                        listed[count + __popcll(mask & ((1ull << lane) - 1))] =
                            (wm * FM + a) * 16 + (lane & 15) | (n - tn * RES_BN) << 8;
                    count += __popcll(mask);
                }
            }
        __syncthreads();
        const int K = g.K;
        const size_t ld = (size_t) g.chunks * 64;
        for (int r = 0; r < count; ++r) {
            const int entry = __builtin_amdgcn_readfirstlane(listed[r]);
            const int m = tm * RES_BM + (entry & 255), n = tn * RES_BN + (entry >> 8);
            if (__hip_atomic_load(&g.flags[n], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) continue;
            const double* e = g.E64 + ld * m;
            const double* x = g.X64 + ld * n;
            double se = 0, sx = 0, ex = 0;
#pragma unroll 8
            for (int k = lane; k < K; k += 64) {
                const double ve = fabs(e[k]), vx = fabs(x[k]);
                se += ve;
                sx += vx;
                ex = fma(ve, vx, ex);
            }
            for (int off = 32; off > 0; off >>= 1) {
                se += __shfl_xor(se, off, 64);
                sx += __shfl_xor(sx, off, 64);
                ex += __shfl_xor(ex, off, 64);
            }
            // half a unit of X's integers times sum |E|, half a unit of E's
            // times sum |X| (the units are 2^-scale), against the chain's
            // bound; 2^-30 for the sums' own rounding
            if (ldexp(se, -1 - g.x_scale[n]) + ldexp(sx, -1 - g.e_scale[m]) > (1 - 0x1p-30) * 0x1p-53 * K * ex && lane == 0)
                __hip_atomic_store(&g.flags[n], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
    }
    // residues: those of the four rows make one word
    const double p = P[l], inv = 1.0 / p;
    const size_t tile = (size_t) (g.first_tile + local);
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b) {
            unsigned w = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double d = from_int(acc[a][b][i]);
                w |= (low_word(fma(-p, nearest(d, inv), d)) & 255) << (8 * i);
            }
            out[(((tile * (FM * FN) + (a * FN + b)) * WAVES + wave) * RES_MODULI + l) * 64 + lane] = w;
        }
}

// Clears the flags of every product's columns.
__global__ __launch_bounds__(256) void clear_flags_kernel(int* __restrict__ flags, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) flags[i] = 0;
}

struct list_group {
    const int* kind;
    const int* flags;
    int* list;
    int N, pad;
};
struct list_groups {
    list_group g[RBF_MAX_GROUPS];
};

// Each product's columns that need FP64 products, in order (one block per product).
__global__ __launch_bounds__(256) void list_kernel(list_groups G)
{
    __shared__ int wave_count[4];
    const list_group g = G.g[blockIdx.x];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int found = 0;
    for (int n0 = 0; n0 < g.N; n0 += 256) {
        const int n = n0 + (int) threadIdx.x;
        const bool on = n < g.N && (g.kind[n] == COLUMN_F64 || (g.kind[n] == COLUMN_WIDE && g.flags[n]));
        const unsigned long long mask = __ballot(on);
        if (lane == 0) wave_count[wave] = __popcll(mask);
        __syncthreads();
        int at = found;
        for (int w = 0; w < wave; ++w) at += wave_count[w];
        if (on) g.list[1 + at + __popcll(mask & ((1ull << lane) - 1))] = n;
        found += wave_count[0] + wave_count[1] + wave_count[2] + wave_count[3];
        __syncthreads();
    }
    if (threadIdx.x == 0) g.list[0] = found;
}

struct crt_group {
    const int* e_scale;
    const int* x_scale;
    const int* live;             // per 16 columns
    double* Y;
    int M, N, tiles_n, tile0, first_tile, pad;
};
struct crt_groups {
    crt_group g[RBF_MAX_GROUPS];
    int count, pad;
};

// Y from the residues: HBM-bound (15 bytes read and 8 written per output).
// A thread takes four outputs (columns 4 (lane / 16) + 0..3 at one sample);
// block (tile, column fragment b of wave row wn): its four waves x FM row
// fragments cover the tile's 256 samples, so that every column is stored in
// one run of 2 KB.  What it leaves in a column without residues is overwritten
// by the FP64 product.
__global__ __launch_bounds__(256) void crt_kernel(crt_groups G, const unsigned* __restrict__ res)
{
    constexpr crt_table T = make_crt();
    const int tile = blockIdx.x / XF, xf = blockIdx.x - tile * XF;
    int q = 0;
    while (q + 1 < G.count && tile >= G.g[q + 1].first_tile) ++q;
    const crt_group g = G.g[q];
    const int t = g.tile0 + (tile - g.first_tile), tm = t / g.tiles_n, tn = t - tm * g.tiles_n;
    const int lane = threadIdx.x & 63, wm = threadIdx.x >> 6;
    const int wn = xf / FN, b = xf - wn * FN, wave = wn * WM + wm;
    const int n0 = tn * RES_BN + xf * 16 + 4 * (lane >> 4);
    if (tn * RES_BN + xf * 16 >= g.N || !(g.live[tn * XF + xf] & 1)) return;
    int xs[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) xs[i] = n0 + i < g.N ? g.x_scale[n0 + i] : 0;
#pragma unroll
    for (int a = 0; a < FM; ++a) {
        const int m = tm * RES_BM + (wm * FM + a) * 16 + (lane & 15);
        const unsigned* r = res + ((((size_t) tile * (FM * FN) + (a * FN + b)) * WAVES + wave) * RES_MODULI) * 64 + lane;
        unsigned w[RES_MODULI];
#pragma unroll
        for (int l = 0; l < RES_MODULI; ++l) w[l] = r[l * 64];
        if (m >= g.M) continue;
        const int es = g.e_scale[m];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (n0 + i >= g.N) continue;
            double h = 0.0, lo = 0.0;
#pragma unroll
            for (int l = 0; l < RES_MODULI; ++l) {
                const double d = from_int((int) (signed char) (w[l] >> (8 * i)));
                h = fma(T.hi[l], d, h);
                lo = fma(T.lo[l], d, lo);
            }
            const double Q = nearest(h, T.p_inv);
            const double y = ldexp(fma(-Q, T.p_hi, h) + fma(-Q, T.p_lo, lo), -(es + xs[i]));
            g.Y[m + (size_t) g.M * (n0 + i)] = y;
        }
    }
}

struct span { int product, tile0, tiles; };

int tiles_of(const res_product& p) { return res_ceil(p.M, RES_BM) * res_ceil(p.N, RES_BN); }

} // namespace

void res_pack_operator(hipStream_t s, const double* E, long lde, int M, int K, unsigned char* planes, int* flag)
{
    const size_t plane = res_plane_bytes(M, RES_BM, K);
    const int rows = res_ceil(M, RES_BM) * RES_BM, chunks = res_chunks(K);
    int* scale = (int*) (planes + RES_PLANES * plane);
    operator_scale_kernel<<<res_ceil(M, 4), 256, 0, s>>>(E, lde, M, K, scale, scale + M, scale + 2 * (size_t) M, flag);
    const long runs = (long) rows * chunks * 4;
    operator_split_kernel<<<(unsigned) ((runs + 255) / 256), 256, 0, s>>>(E, lde, M, K, rows, chunks, scale, scale + M,
                                                                          planes, plane);
}

static size_t tile_bytes(int count, const res_product* p)
{
    long tiles = 0;
    for (int i = 0; i < count; ++i) tiles += tiles_of(p[i]);
    return (size_t) std::min<long>(tiles, RES_LAUNCH_TILES) * RES_TILE_BYTES;
}

int* res_flags(int count, const res_product* p, unsigned char* work, int* n)
{
    *n = 0;
    for (int i = 0; i < count; ++i) *n += p[i].N;
    return (int*) (work + tile_bytes(count, p));
}

void res_pack_columns(hipStream_t s, int count, const res_columns* c, int* flags, int nflags)
{
    column_set set{};
    int n = 0, k = 0;
    for (int i = 0; i < count; ++i) {
        set.c[i] = column_part{c[i].X, res_columns_at(c[i].packed, c[i].N, c[i].K), c[i].N, c[i].K};
        n = std::max(n, c[i].N);
        k = std::max(k, c[i].K);
    }
    const int k_blocks = res_ceil(k, SPLIT_K), rows = res_ceil(n, RES_BN) * RES_BN;
    column_scale_kernel<<<dim3((unsigned) n, (unsigned) count), 256, 0, s>>>(set, flags, nflags);
    column_split_kernel<<<dim3((unsigned) (rows / 16 * k_blocks), (unsigned) count, SPLIT_PARTS), 256, 0, s>>>(set, k_blocks);
}

size_t res_work_bytes(int count, const res_product* p)
{
    size_t columns = 0;
    for (int i = 0; i < count; ++i) columns += (size_t) p[i].N;
    return tile_bytes(count, p) + sizeof(int) * (2 * columns + (size_t) count);
}

ibm_status res_products(ibm_ctx* ctx, hipStream_t s, int count, res_product* p, unsigned char* work, bool cleared)
{
    int columns;
    int* const flags = res_flags(count, p, work, &columns);
    int* flags_of[RBF_MAX_GROUPS];
    list_groups L{};
    for (int i = 0, at = 0; i < count; at += p[i++].N) {
        const res_packed x = res_columns_at(p[i].X, p[i].N, p[i].K);
        flags_of[i] = flags + at;
        int* list = flags + columns + at + i;
        p[i].list = list;
        L.g[i] = list_group{x.kind, flags_of[i], list, p[i].N, 0};
    }
    if (!cleared) {
        clear_flags_kernel<<<(unsigned) res_ceil(columns, 256), 256, 0, s>>>(flags, columns);
        IBM_LAUNCH_CHECK(ctx);
    }
    // Launches of equal parts, at most RES_LAUNCH_TILES tiles (the residues of
    // a launch are recombined before the next overwrites them), longest
    // contraction first: the short units come last and fill the tail.
    long total = 0;
    for (int i = 0; i < count; ++i) total += tiles_of(p[i]);
    const int launches = (int) ((total + RES_LAUNCH_TILES - 1) / RES_LAUNCH_TILES);
    const int most = launches ? (int) ((total + launches - 1) / launches) : 0;
    std::vector<int> order(count);
    for (int i = 0; i < count; ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return p[a].K > p[b].K; });
    std::vector<span> spans;
    int at = 0, taken = 0;
    auto flush = [&]() -> ibm_status {
        if (spans.empty()) return IBM_OK;
        unit_groups U{};
        crt_groups C{};
        int first = 0;
        long per_xcd = 0;
        for (const span& sp : spans) {
            const res_product& r = p[sp.product];
            const size_t ep = res_plane_bytes(r.M, RES_BM, r.K), xp = res_plane_bytes(r.N, RES_BN, r.K);
            const int* e_scale = (const int*) (r.E + RES_PLANES * ep);
            const res_packed x = res_columns_at(r.X, r.N, r.K);
            const int tn = res_ceil(r.N, RES_BN);
            U.g[U.count++] = unit_group{r.E, r.X, r.E64, x.rows, e_scale, e_scale + 2 * (size_t) r.M, x.scale, x.kind,
                                        x.live, flags_of[sp.product], ep, xp, r.M, r.N, r.K, res_chunks(r.K), tn,
                                        sp.tile0, sp.tiles, first};
            C.g[C.count++] = crt_group{e_scale, x.scale, x.live, r.Y, r.M, r.N, tn, sp.tile0, first, 0};
            first += sp.tiles;
        }
        for (int x = 0; x < 8; ++x) {
            long n = 0;
            for (int q = 0; q < U.count; ++q) {
                const long tiles = U.g[q].tiles, units = tiles * RES_MODULI;
                n += (x + 1) * units / 8 - x * units / 8 + (x + 1) * tiles / 8 - x * tiles / 8;
            }
            per_xcd = std::max(per_xcd, n);
        }
        residue_gemm_kernel<<<(unsigned) (8 * per_xcd), RES_THREADS, 0, s>>>(U, (unsigned*) work);
        IBM_LAUNCH_CHECK(ctx);
        crt_kernel<<<(unsigned) (first * XF), 256, 0, s>>>(C, (const unsigned*) work);
        IBM_LAUNCH_CHECK(ctx);
        spans.clear();
        taken = 0;
        return IBM_OK;
    };
    for (int i : order) {
        const int tiles = tiles_of(p[i]);
        for (at = 0; at < tiles;) {
            const int n = std::min(tiles - at, most - taken);
            spans.push_back(span{i, at, n});
            at += n;
            taken += n;
            if (taken == most || (int) spans.size() == RBF_MAX_GROUPS) IBM_TRY(flush());
        }
    }
    IBM_TRY(flush());
    list_kernel<<<(unsigned) count, 256, 0, s>>>(L);
    IBM_LAUNCH_CHECK(ctx);
    return IBM_OK;
}

} // namespace ibm
