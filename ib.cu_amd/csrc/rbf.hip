// RBF surface evaluation on the matrix cores: Y = E^T X for every cell of a
// cell type at once, and the per-sample surface geometry derived from it.
//
// Restates:
//   bases::impl::slice * matrix (bases/operators.h:95-109): a DGEMM
//     Y[ns x 3nc] = E[0:nd, 0:ns]^T X[nd x 3nc], E being the (nd+np) x ns
//     LU-solved evaluator (or derivative) matrix, X the data-site
//     coordinates with column comp*nc + cell (bases/container.h:54).
//   bases::geometry::compute (bases/geometry.h:74-123): unit normal
//     n = t1 x t2 / |t1 x t2| and patch area sigma = w |t1 x t2|, plus the
//     cell area sum(sigma) and enclosed volume sum(x . n sigma) / 3.
//
// Both operands of E^T X are contiguous along the contraction index, so
// each is packed once into "rows x Kp" tiles (k fastest, zero padded):
// the operator at creation, X per call.  One launch covers every
// (cell type, operator) pair.  Precisions:
//   64  few columns and short contractions on v_mfma_f64_16x16x4
//       (rbf_thin_kernel where few blocks do, else 128 x 128 tiles); the
//       others through residues on the INT8 matrix cores (rbf_residue.hip),
//       but for the columns that residues do not hold as well and for
//       operators without residue planes;
//   32  v_mfma_f32_16x16x4 on FP32 operands, FP32 accumulation;
//   16  split BF16: a = a_hi + a_lo with a_hi = bf16(a), a_lo = bf16(a -
//       a_hi); a b ~ a_hi b_hi + a_hi b_lo + a_lo b_hi with
//       v_mfma_f32_16x16x32_bf16 and FP32 accumulation.
// The block tile is 128 (samples) x 128 (columns), or 64 x 64 (FP32, and split
// BF16 of few tiles), with the contraction staged through LDS in 128-byte rows
// (144-byte stride, conflict-free for the 16-byte fragment reads), four waves
// each owning a quadrant.
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstring>
#include <algorithm>
#include <atomic>
#include <climits>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>
#include "context.hpp"
#include "rbf_residue.hpp"

namespace ibm {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

constexpr int TILE = 128;        // rows of a block tile (samples and columns)
constexpr int ROWB = 128;        // bytes of one LDS row per contraction chunk
constexpr int NTHREADS = 256;
constexpr int KPAD = 64;         // contraction padded to a multiple of 64 elements
constexpr int MAX_GROUPS = RBF_MAX_GROUPS;

enum { MODE_F64 = 0, MODE_F32 = 1, MODE_BF16X3 = 2 };

__host__ __device__ constexpr int elem_bytes(int mode) { return mode == MODE_F64 ? 8 : mode == MODE_F32 ? 4 : 2; }
__host__ __device__ constexpr int planes(int mode) { return mode == MODE_BF16X3 ? 2 : 1; }

struct gemm_group {
    const unsigned char* E[2];   // operator planes: rows_pad x Kp elements
    const unsigned char* X[2];   // data-site planes: cols_pad x Kp elements
    double* Y;                   // M x N, column-major, ld = M
    const int* list;             // LISTED: the number of columns to take of X and Y, then their indices
    int M, N, Kp, tiles_n, first_tile;
};

struct gemm_groups {
    gemm_group g[MAX_GROUPS];
    int count, total_tiles;
};

// Listed columns up to this many run in listed_thin_kernel.
constexpr int LISTED_THIN = 64;

__device__ inline uint16_t bf16_bits(float f)
{
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);     // round to nearest even (finite inputs)
    return (uint16_t) (u >> 16);
}

__device__ inline float bf16_value(uint16_t b) { return __uint_as_float(((uint32_t) b) << 16); }

// Packs src (column-major, element (k, r) at src[k + ld r]) into dst planes
// laid out as rows_pad x Kp with k fastest, zero outside rows x K.
template <int MODE>
__global__ __launch_bounds__(256) void pack_kernel(const double* __restrict__ src, long ld, int rows, int K,
                                                   int rows_pad, int Kp, unsigned char* __restrict__ hi,
                                                   unsigned char* __restrict__ lo)
{
    long total = (long) rows_pad * Kp;
    for (long i = blockIdx.x * (long) blockDim.x + threadIdx.x; i < total; i += (long) gridDim.x * blockDim.x) {
        // 32-bit quotient where the index fits (a 64-bit division is a long
        // instruction sequence)
        int r, k;
        if (total <= 0xffffffffl) {
            const unsigned u = (unsigned) i;
            r = (int) (u / (unsigned) Kp);
            k = (int) (u - (unsigned) r * (unsigned) Kp);
        } else {
            r = (int) (i / Kp);
            k = (int) (i - (long) r * Kp);
        }
        double v = (r < rows && k < K) ? src[k + ld * r] : 0.0;
        if constexpr (MODE == MODE_F64) {
            ((double*) hi)[i] = v;
        } else if constexpr (MODE == MODE_F32) {
            ((float*) hi)[i] = (float) v;
        } else {
            uint16_t h = bf16_bits((float) v);
            double rest = v - (double) bf16_value(h);
            ((uint16_t*) hi)[i] = h;
            ((uint16_t*) lo)[i] = bf16_bits((float) rest);
        }
    }
}

template <int MODE>
__device__ inline void mfma_step(const u4& xa, const u4& eb, const u4& xa_lo, const u4& eb_lo,
                                 typename std::conditional<MODE == MODE_F64, d4, f4>::type& acc)
{
    if constexpr (MODE == MODE_F64) {
        double a[2], b[2];
        __builtin_memcpy(a, &xa, 16);
        __builtin_memcpy(b, &eb, 16);
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[0], b[0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[1], b[1], acc, 0, 0, 0);
    } else if constexpr (MODE == MODE_F32) {
        float a[4], b[4];
        __builtin_memcpy(a, &xa, 16);
        __builtin_memcpy(b, &eb, 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc, 0, 0, 0);
    } else {
        bf8 ah, bh, al, bl;
        __builtin_memcpy(&ah, &xa, 16);
        __builtin_memcpy(&bh, &eb, 16);
        __builtin_memcpy(&al, &xa_lo, 16);
        __builtin_memcpy(&bl, &eb_lo, 16);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, acc, 0, 0, 0);
    }
}

// One T x T tile of Y per block.  The MFMA "A" operand is the X tile
// (output rows = columns of Y) and "B" the operator tile, so a lane's four
// results are four columns of Y at one sample row and the 16 lanes of a
// group store 16 consecutive samples (128 contiguous bytes).
//
// Fragment convention (16 x 16 x 4 and 16 x 16 x 32 alike): lane l supplies
// row l % 16 of its operand and the contraction slice owned by lane group
// l / 16; both operands use the same slice assignment, so the sum over the
// chunk is complete whatever order the hardware pairs the slices in.
// Results: lane l holds four rows of column l % 16: rows 4 (l / 16) + r,
// r = 0..3, for the FP32-accumulating instructions, but rows (l / 16) + 4 r
// for v_mfma_f64_16x16x4 (both measured on gfx950).
//
// LISTED: columns [0, N) of the group's list.
template <int MODE, int WN, int RB, int NB, int T, bool LISTED>
__device__ inline void gemm_tile(const gemm_group& g, int N, int tm, int tn)
{
    constexpr int PL = planes(MODE);
    constexpr int THREADS = 128 * WN;                // waves: 2 along the samples x WN along the columns
    constexpr int IN = T / 32, JN = T / 16 / WN;     // 16-sample and 16-column blocks per wave
    constexpr int RS = RB + 16;                      // LDS row stride: 16-row fragment reads hit disjoint banks
    constexpr int LOADS = T * RB / 16 / THREADS;     // 16-byte staging loads per thread, tile and plane
    using acc_t = typename std::conditional<MODE == MODE_F64, d4, f4>::type;
    __shared__ __attribute__((aligned(16))) unsigned char ldsb[NB][PL][2][T * RS];

    const long row_bytes = (long) g.Kp * elem_bytes(MODE);
    const int nchunks = (int) (row_bytes / RB);

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;

    // Global -> register staging: LOADS x 16 bytes per thread per tile and plane.
    const unsigned char* srcE[PL];
    const unsigned char* srcX[PL];
#pragma unroll
    for (int p = 0; p < PL; ++p) {
        srcE[p] = g.E[p] + (long) tm * T * row_bytes;
        srcX[p] = g.X[p] + (LISTED ? 0 : (long) tn * T * row_bytes);
    }
    u4 pe[PL][LOADS], px[PL][LOADS];
    long goff[LOADS], xoff[LOADS];
    int loff[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        int idx = tid + THREADS * i;
        int r = idx / (RB / 16), q = idx % (RB / 16);
        goff[i] = (long) r * row_bytes + q * 16;
        // past the list's end its last column again (not stored)
        xoff[i] = LISTED ? (long) g.list[1 + min(tn * T + r, N - 1)] * row_bytes + q * 16 : goff[i];
        loff[i] = r * RS + q * 16;
    }
#define RBF_LOAD(c)                                                                   \
    _Pragma("unroll") for (int p = 0; p < PL; ++p)                                    \
        _Pragma("unroll") for (int i = 0; i < LOADS; ++i) {                           \
            pe[p][i] = *(const u4*) (srcE[p] + goff[i] + (long) (c) * RB);         \
            px[p][i] = *(const u4*) (srcX[p] + xoff[i] + (long) (c) * RB);         \
        }

    acc_t acc[JN][IN];
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int i = 0; i < IN; ++i) acc[j][i] = acc_t{};

    const int frow = lane & 15, fgrp = lane >> 4;
#define RBF_STORE(buf)                                                                \
    _Pragma("unroll") for (int p = 0; p < PL; ++p)                                    \
        _Pragma("unroll") for (int i = 0; i < LOADS; ++i) {                           \
            *(u4*) (&ldsb[buf][p][0][loff[i]]) = pe[p][i];                            \
            *(u4*) (&ldsb[buf][p][1][loff[i]]) = px[p][i];                            \
        }
    RBF_LOAD(0);
    if constexpr (NB == 2) {
        // Two LDS buffers, one barrier per chunk: chunk c + 1 is stored into
        // the buffer chunk c - 1 used (every wave left it at the last
        // barrier) while chunk c is multiplied from the other.
        RBF_STORE(0);
        if (nchunks > 1) {
            RBF_LOAD(1);
        }
        __syncthreads();
    }
    for (int c = 0; c < nchunks; ++c) {
        const int buf = NB == 2 ? (c & 1) : 0;
        if constexpr (NB == 2) {
            if (c + 1 < nchunks) {
                RBF_STORE(buf ^ 1);
            }
            if (c + 2 < nchunks) {
                RBF_LOAD(c + 2);
            }
        } else {
            __syncthreads();
            RBF_STORE(0);
            __syncthreads();
            if (c + 1 < nchunks) {
                RBF_LOAD(c + 1);
            }
        }
        const unsigned char (*lds)[2][T * RS] = ldsb[buf];
#pragma unroll
        for (int s = 0; s < RB / 64; ++s) {
            u4 ef[PL][IN], xf[PL][JN];
            const int off = s * 64 + fgrp * 16;
#pragma unroll
            for (int p = 0; p < PL; ++p) {
#pragma unroll
                for (int i = 0; i < IN; ++i)
                    ef[p][i] = *(const u4*) (&lds[p][0][(wm * 16 * IN + i * 16 + frow) * RS + off]);
#pragma unroll
                for (int j = 0; j < JN; ++j)
                    xf[p][j] = *(const u4*) (&lds[p][1][(wn * 16 * JN + j * 16 + frow) * RS + off]);
            }
#pragma unroll
            for (int j = 0; j < JN; ++j)
#pragma unroll
                for (int i = 0; i < IN; ++i)
                    mfma_step<MODE>(xf[0][j], ef[0][i], xf[PL - 1][j], ef[PL - 1][i], acc[j][i]);
        }
        if constexpr (NB == 2) __syncthreads();
    }
#undef RBF_LOAD
#undef RBF_STORE

    const int m_base = tm * T + wm * 16 * IN + frow;
    const int n_base = tn * T + wn * 16 * JN + (MODE == MODE_F64 ? fgrp : fgrp * 4);
    constexpr int RSTEP = MODE == MODE_F64 ? 4 : 1;
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int i = 0; i < IN; ++i) {
            int m = m_base + i * 16;
            if (m >= g.M) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int n = n_base + j * 16 + r * RSTEP;
                if (n < N) g.Y[m + (long) g.M * (LISTED ? g.list[1 + n] : n)] = (double) acc[j][i][r];
            }
        }
}

template <int MODE, int WN, int RB = ROWB, int NB = 1, int T = TILE>
__global__ __launch_bounds__(128 * WN, 2) void rbf_gemm_kernel(gemm_groups G)
{
    // Blocks reach the XCDs round-robin (block i on XCD i % 8).  XCD x takes
    // the x-th eighth of every group's tiles, in order, so that the XCDs get
    // equal work however the groups' contraction lengths differ, and the
    // tiles sharing an operator row block share an L2.
    const int xcd = blockIdx.x & 7;
    int k = blockIdx.x >> 3, gi = -1, t = 0;
    for (int q = 0; q < G.count; ++q) {
        const int tq = (q + 1 < G.count ? G.g[q + 1].first_tile : G.total_tiles) - G.g[q].first_tile;
        const int lo = xcd * tq / 8, hi = (xcd + 1) * tq / 8;
        if (k < hi - lo) {
            gi = q;
            t = lo + k;
            break;
        }
        k -= hi - lo;
    }
    if (gi < 0) return;                              // whole block exits together
    const gemm_group g = G.g[gi];
    const int tm = t / g.tiles_n, tn = t - tm * g.tiles_n;
    gemm_tile<MODE, WN, RB, NB, T, false>(g, g.N, tm, tn);
}

// The next of a block's tiles of the listed columns, turn by turn: XCD x takes
// the x-th eighth of every group's tiles.  The lists' lengths are known on
// the device alone, so the blocks of a launch of one size share out the tiles
// that there are (a block for each tile that there could be, most often for
// none: 39 us of the suspension step in a kernel trace; so 27, five to ten a
// launch).  Lists of [least, most] columns count, in tiles of `rows` x `cols`.
__device__ inline bool listed_tile(const gemm_groups& G, int turn, int rows, int cols, int least, int most, int& group,
                                   int& tm, int& tn)
{
    const int xcd = blockIdx.x & 7;
    int k = turn;
    for (int q = 0; q < G.count; ++q) {
        const int N = G.g[q].list[0];
        if (N < least || N > most) continue;
        const int tiles_n = (N + cols - 1) / cols, tq = (G.g[q].M + rows - 1) / rows * tiles_n;
        const int lo = (int) ((long) xcd * tq / 8), hi = (int) ((long) (xcd + 1) * tq / 8);
        if (k < hi - lo) {
            group = q;
            tm = (lo + k) / tiles_n;
            tn = lo + k - tm * tiles_n;
            return true;
        }
        k -= hi - lo;
    }
    return false;
}

// Whether any list has [least, most] columns: a lane for each (the walk above
// is a chain of loads).
__device__ inline bool any_listed(const gemm_groups& G, int least, int most)
{
    static_assert(MAX_GROUPS <= 64);
    const int lane = threadIdx.x & 63, N = lane < G.count ? G.g[lane].list[0] : 0;
    return __ballot(N >= least && N <= most) != 0;
}

constexpr int LISTED_WAVES_N = 4, LISTED_BLOCKS = 512;       // two blocks per CU

// FP64 tiles of the lists that are too long for listed_thin_kernel.
__global__ __launch_bounds__(128 * LISTED_WAVES_N, 4) void listed_gemm_kernel(gemm_groups G)
{
    if (!any_listed(G, LISTED_THIN + 1, INT_MAX)) return;        // whole block
    int q, tm, tn;
    for (int turn = blockIdx.x >> 3; listed_tile(G, turn, TILE, TILE, LISTED_THIN + 1, INT_MAX, q, tm, tn);
         turn += gridDim.x >> 3) {
        const gemm_group g = G.g[q];
        gemm_tile<MODE_F64, LISTED_WAVES_N, ROWB, 2, TILE, true>(g, g.list[0], tm, tn);
        __syncthreads();
    }
}

// FP64 products of few columns, in column tiles of at most 64: bound by
// reading the operator (once; its matrix-core time is 0.3 NB of that).  A
// wave owns 16 samples and the tile's columns, so that operator rows go
// straight from memory to the wave that multiplies them, THIN_AHEAD chunks
// ahead (4 KB each: the 1656 waves of three 8832 x 2210 operators keep 20 MB
// in flight), and only the columns are shared, through two LDS buffers.  The
// multiply sequence of every output is rbf_gemm_kernel's.  Measured against
// its 128-column tiles (us): three operators 8832 x 2210, 3 / 24 / 64 columns
// 294 / 303 / 295 -> 110 / 135 / 203 (the operators alone take 97 at the
// copy rate); 715 x 503, 24 columns 70 -> 15.
constexpr int THIN_ROWS = 32, THIN_RB = 256, THIN_RS = THIN_RB + 16, THIN_AHEAD = 3, THIN_THREADS = 128;

// LISTED: columns [0, N) of the group's list.
template <int NB, bool LISTED>
__device__ inline void thin_tile(const gemm_group& g, int N, int row_tile, int col0)
{
    constexpr int XLOADS = NB * 16 * THIN_RB / 16 / THIN_THREADS;    // 16-byte staging loads per thread
    __shared__ __attribute__((aligned(16))) unsigned char lds[2][NB * 16 * THIN_RS];
    const int row0 = row_tile * THIN_ROWS + (threadIdx.x >> 6) * 16;
    const long row_bytes = (long) g.Kp * 8;
    const int nchunks = (int) (row_bytes / THIN_RB);
    const int lane = threadIdx.x & 63, frow = lane & 15, fgrp = lane >> 4;
    const unsigned char* e = g.E[0] + (long) (row0 + frow) * row_bytes + fgrp * 16;
    const unsigned char* x[XLOADS];
    int xo[XLOADS];
#pragma unroll
    for (int i = 0; i < XLOADS; ++i) {
        const int idx = threadIdx.x + THIN_THREADS * i, r = idx / (THIN_RB / 16), q = idx % (THIN_RB / 16);
        x[i] = g.X[0] + (long) (LISTED ? g.list[1 + min(col0 + r, N - 1)] : col0 + r) * row_bytes + q * 16;
        xo[i] = r * THIN_RS + q * 16;
    }
    u4 pe[THIN_AHEAD][4], px[XLOADS];
    d4 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = d4{};
    // Loads past the last chunk repeat it (not used).
    auto load_e = [&](int c, u4 (&to)[4]) {
#pragma unroll
        for (int s = 0; s < 4; ++s) to[s] = *(const u4*) (e + (long) min(c, nchunks - 1) * THIN_RB + s * 64);
    };
    auto load_x = [&](int c) {
#pragma unroll
        for (int i = 0; i < XLOADS; ++i) px[i] = *(const u4*) (x[i] + (long) min(c, nchunks - 1) * THIN_RB);
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int i = 0; i < XLOADS; ++i) *(u4*) (&lds[buf][xo[i]]) = px[i];
    };
#pragma unroll
    for (int a = 0; a < THIN_AHEAD; ++a) load_e(a, pe[a]);
    load_x(0);
    store_x(0);
    load_x(1);
    __syncthreads();
    auto chunk = [&](int c, u4 (&ce)[4]) {
        const int buf = c & 1;
        u4 ef[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) ef[s] = ce[s];
        store_x(buf ^ 1);                       // chunk c + 1, read after the barrier below
        load_x(c + 2);
        load_e(c + THIN_AHEAD, ce);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const u4 xf = *(const u4*) (&lds[buf][(b * 16 + frow) * THIN_RS + s * 64 + fgrp * 16]);
                mfma_step<MODE_F64>(xf, ef[s], xf, ef[s], acc[b]);
            }
        __syncthreads();
    };
    int c = 0;
    for (; c + THIN_AHEAD <= nchunks; c += THIN_AHEAD) {
#pragma unroll
        for (int a = 0; a < THIN_AHEAD; ++a) chunk(c + a, pe[a]);
    }
#pragma unroll
    for (int a = 0; a < THIN_AHEAD; ++a)
        if (c + a < nchunks) chunk(c + a, pe[a]);
    const int m = row0 + frow;
    if (m >= g.M) return;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n = col0 + b * 16 + fgrp + 4 * r;
            if (n < N) g.Y[m + (long) g.M * (LISTED ? g.list[1 + n] : n)] = acc[b][r];
        }
}

template <int NB>
__global__ __launch_bounds__(THIN_THREADS) void rbf_thin_kernel(gemm_groups G)
{
    int gi = 0;
    while (gi + 1 < G.count && (int) blockIdx.x >= G.g[gi + 1].first_tile) ++gi;
    const gemm_group g = G.g[gi];
    const int tile = (int) blockIdx.x - g.first_tile, row_tile = tile / g.tiles_n;
    thin_tile<NB, false>(g, g.N, row_tile, (tile - row_tile * g.tiles_n) * (16 * NB));
}

// Lists of up to LISTED_THIN columns, in column tiles of 32.
constexpr int LISTED_NB = 2, LISTED_THIN_BLOCKS = 1024;      // four blocks per CU
__global__ __launch_bounds__(THIN_THREADS) void listed_thin_kernel(gemm_groups G)
{
    if (!any_listed(G, 1, LISTED_THIN)) return;                  // whole block
    int q, tm, tn;
    for (int turn = blockIdx.x >> 3; listed_tile(G, turn, THIN_ROWS, 16 * LISTED_NB, 1, LISTED_THIN, q, tm, tn);
         turn += gridDim.x >> 3) {
        const gemm_group g = G.g[q];
        thin_tile<LISTED_NB, true>(g, g.list[0], tm, tn * 16 * LISTED_NB);
        __syncthreads();
    }
}

// Surface geometry of one cell per block from the evaluated position and
// the two tangent blocks (each ns x 3nc, column comp*nc + cell).
__global__ __launch_bounds__(256) void geometry_kernel(int ns, int nc, const double* __restrict__ y,
                                                       const double* __restrict__ t1, const double* __restrict__ t2,
                                                       const double* __restrict__ w, double* __restrict__ normal,
                                                       double* __restrict__ sigma, double* __restrict__ area,
                                                       double* __restrict__ volume)
{
    __shared__ double red[2][256];
    const int cell = blockIdx.x;
    const long count = (long) ns * nc;
    double a_sum = 0, v_sum = 0;
    for (int s = threadIdx.x; s < ns; s += blockDim.x) {
        long at = (long) cell * ns + s;
        double a[3], b[3], x[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            a[i] = t1[count * i + at];
            b[i] = t2[count * i + at];
            x[i] = y[count * i + at];
        }
        double n0 = a[1] * b[2] - a[2] * b[1];
        double n1 = a[2] * b[0] - a[0] * b[2];
        double n2 = a[0] * b[1] - a[1] * b[0];
        double det = sqrt(n0 * n0 + n1 * n1 + n2 * n2);
        normal[count * 0 + at] = n0 / det;
        normal[count * 1 + at] = n1 / det;
        normal[count * 2 + at] = n2 / det;
        double sg = w[s] * det;
        sigma[at] = sg;
        a_sum += sg;
        v_sum += w[s] * (x[0] * n0 + x[1] * n1 + x[2] * n2);
    }
    red[0][threadIdx.x] = a_sum;
    red[1][threadIdx.x] = v_sum;
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if (threadIdx.x < h) {
            red[0][threadIdx.x] += red[0][threadIdx.x + h];
            red[1][threadIdx.x] += red[1][threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        area[cell] = red[0][0];
        volume[cell] = red[1][0] / 3.0;
    }
}

__global__ void clear_flag_kernel(int* flag) { *flag = 0; }

int mode_of(int precision)
{
    return precision == 64 ? MODE_F64 : precision == 32 ? MODE_F32 : precision == 16 ? MODE_BF16X3 : -1;
}

int round_up(int a, int b) { return (a + b - 1) / b * b; }

template <int MODE>
void launch_pack(hipStream_t s, const double* src, long ld, int rows, int K, int rows_pad, int Kp,
                 unsigned char* hi, unsigned char* lo)
{
    long total = (long) rows_pad * Kp;
    int blocks = (int) std::min<long>((total + 255) / 256, 8192);
    pack_kernel<MODE><<<blocks, 256, 0, s>>>(src, ld, rows, K, rows_pad, Kp, hi, lo);
}

void pack(int mode, hipStream_t s, const double* src, long ld, int rows, int K, int rows_pad, int Kp,
          unsigned char* hi, unsigned char* lo)
{
    if (mode == MODE_F64) launch_pack<MODE_F64>(s, src, ld, rows, K, rows_pad, Kp, hi, lo);
    else if (mode == MODE_F32) launch_pack<MODE_F32>(s, src, ld, rows, K, rows_pad, Kp, hi, lo);
    else launch_pack<MODE_BF16X3>(s, src, ld, rows, K, rows_pad, Kp, hi, lo);
}

} // namespace
} // namespace ibm

using namespace ibm;

struct ibm_rbf {
    int device;
    int mode, M, K, Kp, rows_pad, nops;
    size_t plane_bytes;                  // bytes of one operator plane
    unsigned char* mem;                  // nops x planes(mode) planes
    unsigned char* res;                  // FP64: nops x res_bytes of residue planes, or null
    size_t res_bytes;
    const unsigned char* plane(int op, int p) const { return mem + (size_t) (op * planes(mode) + p) * plane_bytes; }
};

namespace ibm {

int rbf_nops(const ibm_rbf* op) { return op ? op->nops : 0; }

// FP64 GEMM variants, by waves along the columns: 2 (64 x 64 wave tiles,
// about 250 registers, two waves per SIMD) or 4 (64 x 32, at most 128
// registers, four waves per SIMD, and two LDS buffers so that a chunk takes
// one barrier: 57 against 51 TFLOP/s at the C4 RBC shape; single-buffered it
// reached 55, with 256-byte chunks 52).
// Both give every output the same MFMA sequence over the same chunks, so
// their results are bitwise equal.  Unless forced, the first eager launch of
// a shape (tiles, summed contraction length) times both and keeps the faster
// for the process; launches under graph capture use the recorded choice or
// the 4-wave default.
std::atomic<int> forced_waves_n{0};
std::mutex variant_lock;
std::map<std::pair<int, long>, int> variant_table;
constexpr int DEFAULT_WAVES_N = 4;

void launch_f64(int wn, const gemm_groups& G, int blocks, hipStream_t stream)
{
    if (wn == 4) rbf_gemm_kernel<MODE_F64, 4, ROWB, 2><<<blocks, 512, 0, stream>>>(G);
    else rbf_gemm_kernel<MODE_F64, 2><<<blocks, NTHREADS, 0, stream>>>(G);
}

// FP32 products, and split-BF16 ones of few tiles, take 64 x 64 tiles with two
// LDS buffers: a quarter of the work per tile fills the chip evenly where 128 x
// 128 tiles leave CUs with one tile more than others or with none (a CU runs
// 8832 x 2210 operators at 165 us a 128-column FP32 tile, however few there
// are), and pads the columns to 64.  128 / 64, us, three operators 8832 x 2210:
// FP32 with 24 / 192 / 600 / 1200 columns 167 / 304 / 748 / 1333 -> 91 / 212 /
// 652 / 1185; split BF16 with 24 / 192 / 600 71 / 122 / 270 -> 45 / 114 / 328.
// A small split-BF16 tile takes 0.38 of the time of a large one (measured on
// operators from 330 x 300 to 8832 x 2210, 3 to 1200 columns), and the large
// ones run in rounds of 256: the smaller estimate is taken.  The multiply
// sequence of an output is the same either way.
// FP32 contractions of a single chunk of 64 elements are bound by storing their
// outputs, where the large tiles' longer runs are faster once there are many
// (six operators 8832 x 40: 600 columns, 2070 tiles, 67 / 78; 1200 130 / 163).
constexpr int SMALL_TILE = 64, SHORT_LARGE_TILES = 1536;
bool small_tiles(int mode, const gemm_groups& G)
{
    long large = 0, small = 0;
    int kp = 0;
    for (int q = 0; q < G.count; ++q) {
        const gemm_group& g = G.g[q];
        kp = std::max(kp, g.Kp);
        large += (long) ((g.M + TILE - 1) / TILE) * ((g.N + TILE - 1) / TILE);
        small += (long) ((g.M + SMALL_TILE - 1) / SMALL_TILE) * ((g.N + SMALL_TILE - 1) / SMALL_TILE);
    }
    if (mode == MODE_F32) return kp > KPAD || large < SHORT_LARGE_TILES;
    return 0.38 * small < 256.0 * ((large + 255) / 256);
}

constexpr int THIN_COLUMNS = 64;       // columns of a full tile of rbf_thin_kernel

void launch_thin(int k, const gemm_groups& T, hipStream_t stream)
{
    if (k == 0) rbf_thin_kernel<1><<<T.total_tiles, THIN_THREADS, 0, stream>>>(T);
    else if (k == 1) rbf_thin_kernel<2><<<T.total_tiles, THIN_THREADS, 0, stream>>>(T);
    else if (k == 2) rbf_thin_kernel<3><<<T.total_tiles, THIN_THREADS, 0, stream>>>(T);
    else rbf_thin_kernel<4><<<T.total_tiles, THIN_THREADS, 0, stream>>>(T);
}

int f64_variant(ibm_ctx* ctx, hipStream_t stream, const gemm_groups& G, int blocks)
{
    (void) ctx;
    const int forced = forced_waves_n.load();
    if (forced) return forced;
    long ksum = 0;
    for (int i = 0; i < G.count; ++i) ksum += G.g[i].Kp;
    const std::pair<int, long> key{G.total_tiles, ksum};
    {
        std::lock_guard<std::mutex> guard(variant_lock);
        auto it = variant_table.find(key);
        if (it != variant_table.end()) return it->second;
    }
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) return DEFAULT_WAVES_N;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        if (e0) hipEventDestroy(e0);
        return DEFAULT_WAVES_N;
    }
    float ms[2] = {0, 0};
    bool ok = true;
    const int cand[2] = {2, 4};
    for (int c = 0; c < 2 && ok; ++c) {
        launch_f64(cand[c], G, blocks, stream);   // warm-up; every launch writes the same outputs
        ok = hipEventRecord(e0, stream) == hipSuccess;
        for (int r = 0; r < 2 && ok; ++r) launch_f64(cand[c], G, blocks, stream);
        ok = ok && hipGetLastError() == hipSuccess && hipEventRecord(e1, stream) == hipSuccess &&
             hipEventSynchronize(e1) == hipSuccess && hipEventElapsedTime(&ms[c], e0, e1) == hipSuccess;
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    const int pick = !ok ? DEFAULT_WAVES_N : (ms[1] <= ms[0] ? 4 : 2);
    if (ok) {
        std::lock_guard<std::mutex> guard(variant_lock);
        variant_table[key] = pick;
    }
    return pick;
}

// Whether an FP64 evaluation of N columns goes through residues
// (rbf_residue.hip) if the operator has them.  Those cost about 40 us of
// launches and 40 bytes an output beside the products, so short contractions
// do not gain by them (K = 440: equal to the FP64 tiles' time; K = 120, 600
// columns, six operators of 8832 rows 405 us against 166; K = 40 four times
// the tiles'), nor do few columns, nor a single column tile of a large output
// while K is middling (three operators 8832 x 560, 65 columns 94 us against
// 81, 8832 x 700 111 / 98, 8832 x 900 133 / 130).  The rule looks at one
// operator's shape only: an entry's path (and so every bit of its result)
// does not depend on what it is batched with.
constexpr int RESIDUE_N = 65, RESIDUE_K = 551, RESIDUE_ONE_TILE_K = 801;
constexpr long RESIDUE_ONE_TILE_OUTPUTS = 500000;
bool by_residues(const ibm_rbf* op, int N)
{
    if (!op->res || N < RESIDUE_N || op->K < RESIDUE_K) return false;
    return op->K >= RESIDUE_ONE_TILE_K || N > TILE || (long) op->M * N < RESIDUE_ONE_TILE_OUTPUTS;
}

// Whether a launch's FP64 products of more than 64 columns run in
// rbf_thin_kernel too, in tiles of 64 columns, or in the FP64 tiles: there as
// long as all blocks are resident at once (four per CU), which keeps more of
// the chip busy than few long tiles; beyond, the tiles' greater reuse wins.
// Thin / tiles, us: six operators of 715 x 503, 192 columns (414 blocks)
// 29 / 74; of 1500 x 440, 192 columns (846) 46 / 67; of 4000 x 440, 65
// columns (1500) 66 / 65; three of 8832 x 440, 65 columns (1656) 83 / 65.  Over
// 1000 shapes of 1 to 6 operators none was slower than in tiles.  Both give
// the same bits.
constexpr long THIN_MOST_BLOCKS = 1024;

// Offset of entry b's packed columns in the evaluation's packed operand and,
// at b = count, its total; entries with the same columns share a packing
// (first: the entry that owns it).
size_t packed_offset(int count, ibm_rbf* const* ops, const int* N, const double* const* X, int b, int* first)
{
    size_t at = 0;
    for (int i = 0; i < count; ++i) {
        const ibm_rbf& op = *ops[i];
        const bool res = by_residues(&op, N[i]);
        int owner = i;
        for (int j = 0; j < i && owner == i; ++j)
            if (X[j] == X[i] && N[j] == N[i] && ops[j]->K == op.K && by_residues(ops[j], N[j]) == res) owner = j;
        if (i == b) {
            if (first) *first = owner;
            return owner == i ? at : packed_offset(count, ops, N, X, owner, nullptr);
        }
        if (owner != i) continue;
        at += res ? (res_columns_bytes(N[i], op.K) + 255) / 256 * 256
                  : (size_t) round_up(std::max(N[i], 1), TILE) * op.Kp * elem_bytes(op.mode) * planes(op.mode);
    }
    return at;
}

// FP64 products of the columns that the residue path has listed.
ibm_status listed_products(ibm_ctx* ctx, hipStream_t stream, int count, const res_product* p)
{
    gemm_groups G{};
    bool long_lists = false;
    for (int i = 0; i < count; ++i) {
        const res_packed x = res_columns_at(p[i].X, p[i].N, p[i].K);
        gemm_group& g = G.g[G.count++];
        g.E[0] = g.E[1] = (const unsigned char*) p[i].E64;
        g.X[0] = g.X[1] = (const unsigned char*) x.rows;
        g.Y = p[i].Y;
        g.list = p[i].list;
        g.M = p[i].M;
        g.N = p[i].N;
        g.Kp = (int) x.ld;
        long_lists = long_lists || p[i].N > LISTED_THIN;
    }
    listed_thin_kernel<<<LISTED_THIN_BLOCKS, THIN_THREADS, 0, stream>>>(G);
    IBM_LAUNCH_CHECK(ctx);
    if (long_lists) listed_gemm_kernel<<<LISTED_BLOCKS, 128 * LISTED_WAVES_N, 0, stream>>>(G);
    IBM_LAUNCH_CHECK(ctx);
    return IBM_OK;
}

// The residue path's products of operators [j0, j1) (operands and outputs
// unset without X / Y: for sizes only).
int residue_products(int count, ibm_rbf* const* ops, const int* N, const double* const* X, double* const* Y, int j0,
                     int j1, unsigned char* packed, res_product* out)
{
    int n = 0;
    for (int b = 0; b < count; ++b) {
        const ibm_rbf& op = *ops[b];
        if (N[b] == 0 || !by_residues(&op, N[b])) continue;
        for (int j = j0; j < std::min(j1, op.nops); ++j)
            out[n++] = res_product{op.res + (size_t) j * op.res_bytes, (const double*) op.plane(j, 0),
                                   X ? packed + packed_offset(count, ops, N, X, b, nullptr) : nullptr,
                                   Y ? Y[b] + (size_t) j * op.M * N[b] : nullptr, op.M, N[b], op.K, nullptr};
    }
    return n;
}

ibm_status rbf_reserve(ibm_ctx* ctx, int count, ibm_rbf* const* ops, const int* N, int j0, int j1)
{
    res_product products[MAX_GROUPS];
    int groups = 0;
    for (int b = 0; b < count; ++b) groups += std::max(0, std::min(j1, ops[b]->nops) - j0);
    if (groups > MAX_GROUPS) return IBM_OK;          // refused by the evaluation itself
    const int n = residue_products(count, ops, N, nullptr, nullptr, j0, j1, nullptr, products);
    void* mem;
    return n ? scratch(ctx, SLOT_RBF_WORK, res_work_bytes(n, products), &mem) : IBM_OK;
}

ibm_status rbf_eval_range(ibm_ctx* ctx, hipStream_t stream, int count, ibm_rbf* const* ops, const int* N,
                          const double* const* X, double* const* Y, int j0, int j1, bool do_pack,
                          unsigned char** packed)
{
    if (!ctx) return IBM_ERR_ARG;
    if (count <= 0 || !ops || !N || !X || !Y) return fail(ctx, IBM_ERR_ARG, "empty or null batch");
    int mode = ops[0] ? ops[0]->mode : -1;
    int groups = 0;
    for (int b = 0; b < count; ++b) {
        if (!ops[b] || !X[b] || !Y[b] || N[b] < 0) return fail(ctx, IBM_ERR_ARG, "bad batch entry %d", b);
        if (ops[b]->mode != mode) return fail(ctx, IBM_ERR_ARG, "batch mixes precisions");
        if (ops[b]->device != ctx->device) return fail(ctx, IBM_ERR_ARG, "operator %d lives on another device", b);
        groups += std::max(0, std::min(j1, ops[b]->nops) - j0);
    }
    if (groups > MAX_GROUPS) return fail(ctx, IBM_ERR_SIZE, "at most %d operator blocks per launch", MAX_GROUPS);
    if (do_pack) {
        void* scratch_mem;
        IBM_TRY(scratch(ctx, SLOT_RBF_X, packed_offset(count, ops, N, X, count, nullptr), &scratch_mem));
        *packed = (unsigned char*) scratch_mem;
    } else if (!*packed) {
        return fail(ctx, IBM_ERR_ARG, "no packed operand");
    }

    res_product products[MAX_GROUPS];
    const int nres = residue_products(count, ops, N, X, Y, j0, j1, *packed, products);
    void* work = nullptr;
    int* flags = nullptr;
    int nflags = 0;
    if (nres) {
        IBM_TRY(scratch(ctx, SLOT_RBF_WORK, res_work_bytes(nres, products), &work));
        flags = res_flags(nres, products, (unsigned char*) work, &nflags);
    }
    long thin_blocks = 0;
    for (int b = 0; b < count && mode == MODE_F64; ++b)
        if (N[b] > THIN_COLUMNS && !by_residues(ops[b], N[b]))
            thin_blocks += (long) ((ops[b]->M + THIN_ROWS - 1) / THIN_ROWS) * ((N[b] + THIN_COLUMNS - 1) / THIN_COLUMNS) *
                           std::max(0, std::min(j1, ops[b]->nops) - j0);
    gemm_groups G{}, thin[4]{};        // thin[k]: rbf_thin_kernel's entries with tiles of 16 (k + 1) columns
    int tiles = 0, ncols = 0;
    res_columns cols[RES_MAX_COLUMNS];
    for (int b = 0; b < count; ++b) {
        const ibm_rbf& op = *ops[b];
        if (N[b] == 0) continue;
        int owner = b;
        unsigned char* hi = *packed + packed_offset(count, ops, N, X, b, &owner);
        if (by_residues(&op, N[b])) {
            if (do_pack && owner == b) {
                cols[ncols++] = res_columns{X[b], hi, N[b], op.K};
                if (ncols == RES_MAX_COLUMNS) {
                    res_pack_columns(stream, ncols, cols, nullptr, 0);
                    ncols = 0;
                }
            }
            continue;
        }
        int cols_pad = round_up(N[b], TILE);
        unsigned char* lo = planes(mode) > 1 ? hi + (size_t) cols_pad * op.Kp * elem_bytes(mode) : nullptr;
        if (do_pack && owner == b) pack(mode, stream, X[b], op.K, N[b], op.K, cols_pad, op.Kp, hi, lo);
        const bool is_thin = mode == MODE_F64 && (N[b] <= THIN_COLUMNS || thin_blocks <= THIN_MOST_BLOCKS);
        for (int j = j0; j < std::min(j1, op.nops); ++j) {
            gemm_groups& to = is_thin ? thin[std::min(N[b] - 1, THIN_COLUMNS - 1) / 16] : G;
            gemm_group& g = to.g[to.count++];
            g.E[0] = op.plane(j, 0);
            g.E[1] = planes(mode) > 1 ? op.plane(j, 1) : g.E[0];
            g.X[0] = hi;
            g.X[1] = lo ? lo : hi;
            g.Y = Y[b] + (size_t) j * op.M * N[b];
            g.M = op.M;
            g.N = N[b];
            g.Kp = op.Kp;
            g.tiles_n = is_thin ? (N[b] + THIN_COLUMNS - 1) / THIN_COLUMNS : cols_pad / TILE;
            g.first_tile = tiles;
            if (!is_thin) tiles += (op.rows_pad / TILE) * g.tiles_n;
        }
    }
    if (ncols) res_pack_columns(stream, ncols, cols, flags, nflags);
    IBM_LAUNCH_CHECK(ctx);
    double flops = 0;
    for (int b = 0; b < count; ++b)
        flops += 2.0 * ops[b]->M * (double) N[b] * ops[b]->K * std::max(0, std::min(j1, ops[b]->nops) - j0);
    int blocks = 0, edge = TILE;
    if (tiles) {
        // Longest contraction first: each XCD takes its share of the groups
        // in group order, so the short tiles come last and fill the tail.
        std::stable_sort(G.g, G.g + G.count, [](const gemm_group& a, const gemm_group& b) { return a.Kp > b.Kp; });
        if (mode != MODE_F64 && small_tiles(mode, G)) edge = SMALL_TILE;
        tiles = 0;
        for (int q = 0; q < G.count; ++q) {
            G.g[q].first_tile = tiles;
            G.g[q].tiles_n = (G.g[q].N + edge - 1) / edge;
            tiles += (G.g[q].M + edge - 1) / edge * G.g[q].tiles_n;
        }
        G.total_tiles = tiles;
        // blocks: 8 x the most tiles any XCD takes (its share of every group)
        int per_xcd = 0;
        for (int x = 0; x < 8; ++x) {
            int n = 0;
            for (int q = 0; q < G.count; ++q) {
                const int tq = (q + 1 < G.count ? G.g[q + 1].first_tile : tiles) - G.g[q].first_tile;
                n += (x + 1) * tq / 8 - x * tq / 8;
            }
            per_xcd = std::max(per_xcd, n);
        }
        blocks = 8 * per_xcd;
    }
    const int wn = mode == MODE_F64 && tiles ? f64_variant(ctx, stream, G, blocks) : 2;
    prof_scope prof(ctx, "rbf_gemm", flops);
    if (nres) {
        IBM_TRY(res_products(ctx, stream, nres, products, (unsigned char*) work, ncols > 0));
        IBM_TRY(listed_products(ctx, stream, nres, products));
    }
    for (int k = 0; k < 4; ++k) {
        gemm_groups& T = thin[k];
        if (!T.count) continue;
        std::stable_sort(T.g, T.g + T.count, [](const gemm_group& a, const gemm_group& b) { return a.Kp > b.Kp; });
        for (int q = 0; q < T.count; ++q) {
            T.g[q].first_tile = T.total_tiles;
            T.total_tiles += (T.g[q].M + THIN_ROWS - 1) / THIN_ROWS * T.g[q].tiles_n;
        }
        launch_thin(k, T, stream);
    }
    IBM_LAUNCH_CHECK(ctx);
    if (!tiles) return IBM_OK;
    if (mode == MODE_F64) {
        launch_f64(wn, G, blocks, stream);
    } else if (mode == MODE_F32) {
        if (edge == SMALL_TILE) rbf_gemm_kernel<MODE_F32, 2, ROWB, 2, SMALL_TILE><<<blocks, NTHREADS, 0, stream>>>(G);
        else rbf_gemm_kernel<MODE_F32, 2><<<blocks, NTHREADS, 0, stream>>>(G);
    } else {
        if (edge == SMALL_TILE) rbf_gemm_kernel<MODE_BF16X3, 2, ROWB, 2, SMALL_TILE><<<blocks, NTHREADS, 0, stream>>>(G);
        else rbf_gemm_kernel<MODE_BF16X3, 2><<<blocks, NTHREADS, 0, stream>>>(G);
    }
    IBM_LAUNCH_CHECK(ctx);
    return IBM_OK;
}

} // namespace ibm

extern "C" {

ibm_status ibm_rbf_create(ibm_ctx* ctx, int precision, int M, int K, int nops, const double* const* E, int lde,
                          ibm_rbf** out)
{
    if (!ctx || !out) return IBM_ERR_ARG;
    *out = nullptr;
    int mode = mode_of(precision);
    if (mode < 0) return fail(ctx, IBM_ERR_ARG, "precision must be 64, 32 or 16 (split bf16), got %d", precision);
    if (M <= 0 || K <= 0 || nops <= 0 || nops > 8 || lde < K || !E)
        return fail(ctx, IBM_ERR_ARG, "bad operator shape M=%d K=%d nops=%d lde=%d", M, K, nops, lde);
    for (int j = 0; j < nops; ++j)
        if (!E[j]) return fail(ctx, IBM_ERR_ARG, "null operator %d", j);
    ibm_rbf* op = new ibm_rbf{};
    op->device = ctx->device;
    op->mode = mode;
    op->M = M;
    op->K = K;
    op->Kp = round_up(K, KPAD);
    op->rows_pad = round_up(M, TILE);
    op->nops = nops;
    op->plane_bytes = (size_t) op->rows_pad * op->Kp * elem_bytes(mode);
    size_t bytes = op->plane_bytes * nops * planes(mode);
    if (hipMalloc(&op->mem, bytes) != hipSuccess) {
        delete op;
        return fail(ctx, IBM_ERR_HIP, "out of device memory for a %zu-byte operator", bytes);
    }
    // FP64 operators also keep their residue planes (sixteen bytes per
    // element beside the eight); without the memory for them, or with
    // elements they cannot represent, every product runs on the FP64 matrix
    // cores.
    int* flag = nullptr;
    if (mode == MODE_F64 && res_fits(K)) {
        op->res_bytes = (res_operator_bytes(M, K) + 255) / 256 * 256;
        if (hipMalloc(&op->res, op->res_bytes * nops + sizeof(int)) != hipSuccess) {
            (void) hipGetLastError();
            op->res = nullptr;
        } else {
            flag = (int*) (op->res + op->res_bytes * nops);
            clear_flag_kernel<<<1, 1, 0, ctx->stream>>>(flag);
            for (int j = 0; j < nops; ++j) res_pack_operator(ctx->stream, E[j], lde, M, K, op->res + op->res_bytes * j, flag);
        }
    }
    for (int j = 0; j < nops; ++j)
        pack(mode, ctx->stream, E[j], lde, M, K, op->rows_pad, op->Kp, (unsigned char*) op->plane(j, 0),
             planes(mode) > 1 ? (unsigned char*) op->plane(j, 1) : nullptr);
    int unfit = 0;
    if (hipGetLastError() != hipSuccess ||
        (flag && hipMemcpyAsync(&unfit, flag, sizeof(int), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess) ||
        hipStreamSynchronize(ctx->stream) != hipSuccess) {
        hipFree(op->mem);
        hipFree(op->res);
        delete op;
        return fail(ctx, IBM_ERR_HIP, "operator packing failed");
    }
    if (unfit) {
        hipFree(op->res);
        op->res = nullptr;
    }
    *out = op;
    return IBM_OK;
}

ibm_status ibm_rbf_gemm_variant(int waves_n)
{
    if (waves_n != 0 && waves_n != 2 && waves_n != 4) return IBM_ERR_ARG;
    ibm::forced_waves_n.store(waves_n);
    return IBM_OK;
}

ibm_status ibm_rbf_destroy(ibm_rbf* op)
{
    if (!op) return IBM_OK;
    hipFree(op->mem);
    hipFree(op->res);
    delete op;
    return IBM_OK;
}

ibm_status ibm_rbf_eval(ibm_ctx* ctx, int count, ibm_rbf* const* ops, const int* N, const double* const* X,
                        double* const* Y)
{
    if (!ctx) return IBM_ERR_ARG;
    unsigned char* packed = nullptr;
    return ibm::rbf_eval_range(ctx, ctx->stream, count, ops, N, X, Y, 0, 8, true, &packed);
}

ibm_status ibm_surface_geometry(ibm_ctx* ctx, int ns, int nc, const double* y, const double* t1, const double* t2,
                                const double* w, double* normal, double* sigma, double* area, double* volume)
{
    if (!ctx) return IBM_ERR_ARG;
    if (ns <= 0 || nc < 0) return fail(ctx, IBM_ERR_ARG, "bad sizes ns=%d nc=%d", ns, nc);
    if (!nc) return IBM_OK;
    if (!y || !t1 || !t2 || !w || !normal || !sigma || !area || !volume) return fail(ctx, IBM_ERR_ARG, "null array");
    // y, t1, t2 and w read; normals, sigma, area, volume written
    prof_scope prof(ctx, "geometry", 8.0 * ((double) ns * nc * 13 + ns + 2.0 * nc));
    geometry_kernel<<<nc, 256, 0, ctx->stream>>>(ns, nc, y, t1, t2, w, normal, sigma, area, volume);
    IBM_LAUNCH_CHECK(ctx);
    return IBM_OK;
}

} // extern "C"
