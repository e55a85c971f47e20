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
// the operands' rounding (2^-62 of the row's 1-norm, 2^-54 of the column's
// maximum) and one rounding of the result.  Measured on the RBC and platelet
// operators (values and all derivatives, 300 to 2210 data sites) against
// long-double products, the error is 0.03 to 0.66 of the FP64 fused
// multiply-add chain's in the 2-norm and 0.01 to 0.74 in the maximum; one
// modulus fewer (2^109) would be 4 to 65 times the chain's.
//
// What bounds it: FP64 matrix cores are dense at 78.6 TFLOP/s (measured 72.6
// for a large library product), INT8 at 5.0 POP/s; with random operands the
// card's power budget holds a register-only INT8 loop to 3.9 POP/s
// (16 x 16 x 64; 3.1 with 32 x 32 x 32, which moves twice the accumulators
// per product) and these products to 1.9 to 2.1 (2.3 to 2.9 on operands of
// zeros), so 15 products are worth about 120 FP64 TFLOP/s.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <climits>
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
// exact in FP64; the low parts are below 2^77 and enter with FP64 rounding,
// 2^-60 of an integer of C's unit size or less.
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
constexpr int BAD_COLUMN = INT_MIN;           // scale of a column with a NaN or an infinity

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

// Scale of operator row m (one wavefront per row): 2^(62 - e), sum |E| < 2^e.
__global__ __launch_bounds__(256) void operator_scale_kernel(const double* __restrict__ E, long lde, int M, int K,
                                                             int* __restrict__ scale, int* __restrict__ flag)
{
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (m >= M) return;
    double s = 0;
    for (int k = lane; k < K; k += 64) s += fabs(E[k + lde * m]);
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) {
        int e = 0;
        if (!isfinite(s)) *flag = 1;
        else if (s > 0) frexp(s * (1 + 0x1p-40), &e);      // the sum's own rounding
        scale[m] = SCALE_E - e;
    }
}

__global__ __launch_bounds__(256) void operator_split_kernel(const double* __restrict__ E, long lde, int M, int K,
                                                             int rows, int chunks, const int* __restrict__ scale,
                                                             unsigned char* __restrict__ planes, size_t plane)
{
    const long i = (long) blockIdx.x * 256 + threadIdx.x;
    const int runs = chunks * 4;
    if (i >= (long) rows * runs) return;
    // consecutive lanes take the 16 rows of a fragment, then its runs of k
    const int frag_row = (int) (i / ((long) runs * 16)), in = (int) (i - (long) frag_row * runs * 16);
    const int row = frag_row * 16 + (in & 15), run = in >> 4;
    double h[16], d[16];
    const int s = row < M ? scale[row] : 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int k = run * 16 + j;
        split_element(row < M && k < K ? E[k + lde * row] : 0.0, s, h[j], d[j]);
    }
    store_residues<0, RES_MODULI>(h, d, planes + run_offset(row, run, chunks), plane);
}

struct column_set {
    res_columns c[RES_MAX_COLUMNS];
};

__device__ inline int* column_scales(const res_columns& c, int chunks)
{
    const size_t rows = (size_t) ((c.N + RES_BN - 1) / RES_BN) * RES_BN;
    return (int*) (c.planes + RES_MODULI * rows * chunks * 64);
}

// Scale of column n: 2^(54 - e), max |x| < 2^e; one block per column.
__global__ __launch_bounds__(256) void column_scale_kernel(column_set set)
{
    __shared__ double part[4];
    const res_columns c = set.c[blockIdx.y];
    const int n = blockIdx.x;
    if (n >= c.N) return;                                      // whole block
    const double* x = c.X + (size_t) n * c.K;
    double m = 0;
#pragma unroll 8
    for (int k = threadIdx.x; k < c.K; k += 256) {
        const double v = fabs(x[k]);
        m = isfinite(v) ? fmax(m, v) : INFINITY;
    }
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmax(fmax(part[0], part[1]), fmax(part[2], part[3]));
        int e = 0;
        if (isfinite(m) && m > 0) frexp(m, &e);
        column_scales(c, (c.K + 63) / 64)[n] = isfinite(m) ? SCALE_X - e : BAD_COLUMN;
    }
}

// Residues of 16 columns x 256 elements for a third of the moduli
// (blockIdx.z): rows of 2 KB staged through LDS, so that both the loads and
// the 1 KB fragment stores are contiguous (one block per column, whose
// threads load and store scattered 128- and 16-byte pieces: 41 us for 600
// columns of 2210 elements).  Padding columns get zeros.
constexpr int SPLIT_PARTS = 3, SPLIT_K = 256, SPLIT_LD = SPLIT_K + SPLIT_K / 16 + 1;
static_assert(RES_MODULI == 15);

__global__ __launch_bounds__(256) void column_split_kernel(column_set set, int k_blocks)
{
    __shared__ double sx[16][SPLIT_LD];                        // element k at k + k / 16
    const res_columns c = set.c[blockIdx.y];
    const int chunks = (c.K + 63) / 64, runs = chunks * 4;
    const int rows = (c.N + RES_BN - 1) / RES_BN * RES_BN;
    const int n0 = (int) (blockIdx.x / k_blocks) * 16, k0 = (int) (blockIdx.x % k_blocks) * SPLIT_K;
    if (n0 >= rows || k0 >= c.K) return;                       // whole block
    for (int i = threadIdx.x; i < 16 * SPLIT_K; i += 256) {
        const int r = i / SPLIT_K, k = i - r * SPLIT_K;
        sx[r][k + (k >> 4)] = n0 + r < c.N && k0 + k < c.K ? c.X[(size_t) (n0 + r) * c.K + k0 + k] : 0.0;
    }
    __syncthreads();
    const int r = threadIdx.x & 15, run = threadIdx.x >> 4;
    if (k0 / 16 + run >= runs) return;
    const int s = n0 + r < c.N ? column_scales(c, chunks)[n0 + r] : BAD_COLUMN;
    double h[16], d[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) split_element(s != BAD_COLUMN ? sx[r][run * 17 + j] : 0.0, s, h[j], d[j]);
    unsigned char* at = c.planes + run_offset(n0 + r, k0 / 16 + run, chunks);
    const size_t plane = (size_t) rows * chunks * 64;
    if (blockIdx.z == 0) store_residues<0, 5>(h, d, at, plane);
    else if (blockIdx.z == 1) store_residues<5, 10>(h, d, at, plane);
    else store_residues<10, 15>(h, d, at, plane);
}

// ----------------------------------------------------------------------
// The INT8 products.  One block computes one 256 x 128 tile modulo one
// modulus and leaves each output's residue as a byte: eight waves of 64 x 64
// outputs (4 x 4 fragments of 16 x 16), the operands' fragments staged as
// they lie in memory (1 KB each, read conflict-free) by direct-to-LDS loads
// into three buffers, two 64-element chunks ahead of the one multiplied, one
// barrier a chunk.  Units (tile, modulus) rather than whole tiles keep the
// last wave of blocks short.  Measured for 8832 x 2210 x 600 (16 moduli):
// 0.219 ms; four waves of 64 x 128 0.228, 128 x 128 tiles 0.237, 256 x 256
// tiles 0.289 (padding of the 600 columns), 32 x 32 x 32 instructions with
// two buffers 0.232.
// ----------------------------------------------------------------------
constexpr int WM = 4, WN = 2, FM = 4, FN = 4;          // waves and fragments per wave
constexpr int WAVES = WM * WN, EF = WM * FM, XF = WN * FN, LOADS = (EF + XF) / WAVES;
constexpr int RES_THREADS = 64 * WAVES;
static_assert(EF * 16 == RES_BM && XF * 16 == RES_BN && LOADS * WAVES == EF + XF);

struct unit_group {
    const unsigned char* E;
    const unsigned char* X;
    size_t e_plane, x_plane;     // bytes of one modulus' plane
    int chunks, tiles_n;
    int tile0, tiles;            // tiles [tile0, tile0 + tiles) of the product, here tiles first_tile..
    int first_tile;
    int pad;
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
    // blocks sharing an operator row tile and a modulus' columns share an L2.
    const int xcd = blockIdx.x & 7;
    int k = blockIdx.x >> 3, gi = -1, u = 0;
    for (int q = 0; q < G.count; ++q) {
        const long n = (long) G.g[q].tiles * RES_MODULI;
        const int lo = (int) (xcd * n / 8), hi = (int) ((xcd + 1) * n / 8);
        if (k < hi - lo) {
            gi = q;
            u = lo + k;
            break;
        }
        k -= hi - lo;
    }
    if (gi < 0) return;                              // whole block exits together
    const unit_group g = G.g[gi];
    const int l = u / g.tiles, local = u - l * g.tiles, t = g.tile0 + local;
    const int tm = t / g.tiles_n, tn = t - tm * g.tiles_n;
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
    // 4 (lane / 16) + i of X's fragment at sample lane % 16; their four
    // residues make one word.
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

struct crt_group {
    const int* e_scale;
    const int* x_scale;
    const double* E64;
    const double* X64;
    double* Y;
    long ld64;
    int M, N, K, tiles_n, tile0, first_tile;
};
struct crt_groups {
    crt_group g[RBF_MAX_GROUPS];
    int count, pad;
};

// Y from the residues: HBM-bound (15 bytes read and 8 written per output).
// A thread takes four outputs (columns 4 (lane / 16) + 0..3 at one sample);
// block (tile, column fragment b of wave row wn): its four waves x FM row
// fragments cover the tile's 256 samples, so that every column is stored in
// one run of 2 KB.
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
    if (tn * RES_BN + xf * 16 >= g.N) return;
    int xs[4];
    bool bad[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        xs[i] = n0 + i < g.N ? g.x_scale[n0 + i] : 0;
        bad[i] = xs[i] == BAD_COLUMN;
        xs[i] = bad[i] ? 0 : xs[i];
    }
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
            double y = ldexp(fma(-Q, T.p_hi, h) + fma(-Q, T.p_lo, lo), -(es + xs[i]));
            if (bad[i]) {
                // a NaN or an infinity in the column: the plain product
                const double* e = g.E64 + g.ld64 * m;
                const double* x = g.X64 + (size_t) (n0 + i) * g.K;
                y = 0.0;
                for (int k = 0; k < g.K; ++k) y = fma(e[k], x[k], y);
            }
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
    int* scale = (int*) (planes + RES_MODULI * plane);
    operator_scale_kernel<<<res_ceil(M, 4), 256, 0, s>>>(E, lde, M, K, scale, flag);
    const long runs = (long) rows * chunks * 4;
    operator_split_kernel<<<(unsigned) ((runs + 255) / 256), 256, 0, s>>>(E, lde, M, K, rows, chunks, scale, planes, plane);
}

void res_pack_columns(hipStream_t s, int count, const res_columns* c)
{
    column_set set{};
    int n = 0, k = 0;
    for (int i = 0; i < count; ++i) {
        set.c[i] = c[i];
        n = std::max(n, c[i].N);
        k = std::max(k, c[i].K);
    }
    const int k_blocks = res_ceil(k, SPLIT_K), rows = res_ceil(n, RES_BN) * RES_BN;
    column_scale_kernel<<<dim3((unsigned) n, (unsigned) count), 256, 0, s>>>(set);
    column_split_kernel<<<dim3((unsigned) (rows / 16 * k_blocks), (unsigned) count, SPLIT_PARTS), 256, 0, s>>>(set, k_blocks);
}

size_t res_work_bytes(int count, const res_product* p)
{
    long tiles = 0;
    for (int i = 0; i < count; ++i) tiles += tiles_of(p[i]);
    return (size_t) std::min<long>(tiles, RES_LAUNCH_TILES) * RES_TILE_BYTES;
}

ibm_status res_products(ibm_ctx* ctx, hipStream_t s, int count, const res_product* p, unsigned char* work)
{
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
            const int tn = res_ceil(r.N, RES_BN);
            U.g[U.count++] = unit_group{r.E, r.X, ep, xp, res_chunks(r.K), tn, sp.tile0, sp.tiles, first, 0};
            C.g[C.count++] = crt_group{(const int*) (r.E + RES_MODULI * ep), (const int*) (r.X + RES_MODULI * xp), r.E64,
                                       r.X64, r.Y, r.ld64, r.M, r.N, r.K, tn, sp.tile0, first};
            first += sp.tiles;
        }
        for (int x = 0; x < 8; ++x) {
            long n = 0;
            for (int q = 0; q < U.count; ++q) {
                const long units = (long) U.g[q].tiles * RES_MODULI;
                n += (x + 1) * units / 8 - x * units / 8;
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
    return flush();
}

} // namespace ibm
