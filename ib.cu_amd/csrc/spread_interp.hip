// Spreading and interpolation between Lagrangian markers and the MAC grid.
//
// Reference algorithm (ib/novel.h:58-168, ib/interpolate.h:49-76): per
// component, sort markers by cell, segmented-sum 8 stencil values per sweep
// into 8 plane buffers, combine the planes; interpolation is a per-marker
// 64-point gather.  The values computed are the same:
//     spread:  fe_c(g) = h^-3 sum_m f_c(m) prod_j phi(g_j - X_j(m)/h)
//     interp:  U_c(m)  = sum_g u_c(g) prod_j phi(g_j - X_j(m)/h)
// with the reference's index conventions (geometry.hpp).
//
// MI355X design:
//   * markers are counting-sorted into bins of 4 x 4 x 4 cells, and one
//     workgroup per brick of 8 x 8 x 8 cells adds its markers' stencils, each
//     visited once, to a tile of 64-bit fixed-point integers in LDS; a merge
//     pass sums the tiles.  Integer sums do not depend on scheduling: bitwise
//     reproducible without global atomics or an order inside a bin;
//   * grids whose tiles would not fit the fixed workspace although their bins
//     do are spread owner-computes: one workgroup per 8x8x8 brick of grid
//     points gathers the (canonically ordered) markers of the bins whose
//     stencils reach the brick into an LDS tile of the same integers;
//   * few scattered markers on a large grid are gathered by the bricks of points
//     (the same integers, no tiles in memory);
//   * interpolation is two lanes per marker and component, each with half of
//     every row of the separable sum sum_z wz sum_y wy sum_x wx u.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <algorithm>
#include <climits>
#include <mutex>
#include "context.hpp"
#include "deltas.hpp"


// ----------------------------------------------------------------------
// Fixed workspace of ibm_spread_sets_noalloc: the buffers of one spread of at
// most STATIC_MAX_MARKERS markers onto grids of at most STATIC_MAX_BINS bins
// (a 128 x 129 x 128 cell grid), 184 MB per device, held from the first
// ibm_create until the process ends: the tiles of STATIC_MAX_BRICKS bricks (as many as
// such a grid has, unless an axis is so short that its bricks are mostly
// empty: those grids take the brick kernel, which needs 36.6 MB) or that
// kernel's bins.
// ----------------------------------------------------------------------
namespace ibm_fixed {
constexpr size_t STATIC_MAX_MARKERS = size_t(1) << 18;
constexpr size_t STATIC_MAX_BINS = size_t(128) * 129 * 128;
constexpr size_t STATIC_MAX_BRICKS = size_t(16) * 17 * 16;
constexpr size_t STATIC_SCAN_BYTES = size_t(1) << 20;
constexpr size_t STATIC_STATS_BYTES = 4096;
constexpr size_t TILE_BYTES = sizeof(long long) * 3 * 12 * 12 * 12;      // one brick's tiles

constexpr size_t align256(size_t b) { return (b + 255) & ~size_t(255); }
constexpr size_t STATIC_BIN_WORDS = align256(sizeof(int) * (STATIC_MAX_BINS + 1));
constexpr size_t STATIC_INT_ARRAY = align256(sizeof(int) * STATIC_MAX_MARKERS);
constexpr size_t STATIC_BRICK_KERNEL_BYTES =
    2 * STATIC_BIN_WORDS +                                   // count, start
    4 * STATIC_INT_ARRAY +                                   // key, rank, perm, code
    align256(sizeof(long long) * STATIC_MAX_MARKERS) +       // tmp
    align256(sizeof(double) * 6 * STATIC_MAX_MARKERS) +      // sorted positions and forces
    STATIC_STATS_BYTES + STATIC_SCAN_BYTES;
constexpr size_t STATIC_TILE_KERNEL_BYTES =
    2 * align256(sizeof(int) * (8 * STATIC_MAX_BRICKS + 1)) +    // count, start
    3 * STATIC_INT_ARRAY +                                   // key, rank, perm
    STATIC_STATS_BYTES + 256 + align256(sizeof(int) * STATIC_MAX_BRICKS) +   // statistics, quantum, flags
    TILE_BYTES * STATIC_MAX_BRICKS;
constexpr size_t STATIC_SCRATCH_BYTES =
    STATIC_TILE_KERNEL_BYTES > STATIC_BRICK_KERNEL_BYTES ? STATIC_TILE_KERNEL_BYTES : STATIC_BRICK_KERNEL_BYTES;
} // namespace ibm_fixed

namespace ibm {
namespace {

constexpr int MAX_SETS = 16;
constexpr int CHUNK = 64;
constexpr int SPREAD_THREADS = 256;

struct kaxis {
    double length, resolution, shift;
    double s_over_r;   // shift / resolution, rounded once as fd::discretization::units does per call
    int cells, points, solid, pad;
};

struct kgrids {
    kaxis a[3][3];     // [component][dimension]
    double res3[3];    // product of the resolutions of each component grid
    int points[3][3];
    int cand[2][3];    // per dimension, the components whose axes are the (at most two) distinct ones
    int sel[3][3];     // sel[c][j]: which candidate component c uses along dimension j
};

struct marker_sets {
    int nsets;
    int total;
    int offset[MAX_SETS + 1];
    const double* x[MAX_SETS];
    const double* f[MAX_SETS];
    double* out[MAX_SETS];
};

struct bin_desc {
    int nb[3];
    int qmin[3];
    int fc[3];
    int fs[3];
    int lo[3], hi[3];
    int nbins;
};

// Statistics gathered while binning; they bound the spread accumulators.
// Maxima are spread over STAT_SLOTS words (by block index) so the atomics
// do not all hit one address; readers reduce the slots.
constexpr int STAT_SLOTS = 64;
struct bin_stats {
    unsigned long long max_abs_f[STAT_SLOTS];   // bit patterns of max |f| (non-negative doubles order as integers)
    unsigned long long max_count[STAT_SLOTS];   // largest number of markers in one bin
};

__device__ inline int set_of(const marker_sets& s, int m)
{
    int k = 0;
    while (k + 1 < s.nsets && m >= s.offset[k + 1]) ++k;
    return k;
}

// axis_stencil() with the per-axis quotient shift/resolution precomputed and
// the periodic wrap (i + cells) % cells written for i in [-cells, 2 cells).
__device__ inline stencil_axis kstencil(const kaxis& a, double x)
{
#pragma clang fp contract(off)
    double y = x - a.s_over_r;
    if (!a.solid) {
        // For y in [-L, 2L), floor(y / L) is decided by comparisons alone
        // (correctly rounded division is monotone and y / L < 1 whenever
        // y < L), so modulo(y, L) = y - L * floor(y / L) is reproduced
        // exactly without the division.
        double L = a.length;
        if (y >= 0 && y < L) {
        } else if (y < 0 && y >= -L) {
            y = y + L;
        } else if (y >= L && y < 2 * L) {
            y = y - L;
        } else {
            y = ref_modulo(y, L);
        }
    }
    double diff = (y * a.resolution + a.shift) - a.shift;
    double fl = ref_floor(diff);
    int i = (int) fl;
    int j = i;
    if (!a.solid) j = i < 0 ? i + a.cells : (i >= a.cells ? i - a.cells : i);
    int w = a.points + a.solid;
    int k = j + a.solid;
    k = k < 0 ? 0 : (k >= w ? w - 1 : k);
    stencil_axis s;
    s.base = k - a.solid;
    s.d = fl - diff;
    return s;
}

// Maximum over the 64 lanes of a wavefront (all lanes must be active).
__device__ inline unsigned long long wave_max(unsigned long long v)
{
    for (int off = 32; off > 0; off >>= 1) {
        unsigned long long o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    return v;
}

// ----------------------------------------------------------------------
// Binning: key = bin of the marker's face-aligned cell.  For dimension j the
// face component fc[j] is aligned on cell faces there; its (clamped) base
// cell plus the integer part of its shift is q_j.  Every component's base
// cell then lies in q_j + [lo_j, hi_j], which bounds the bins a brick reads.
// ----------------------------------------------------------------------
// Clears n 32-bit words (used in place of hipMemsetAsync so that a binning
// pass can be recorded in a HIP graph).
__global__ void zero_words_kernel(unsigned int* __restrict__ p, size_t n)
{
    for (size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t) gridDim.x * blockDim.x)
        p[i] = 0u;
}

__global__ void bin_count_kernel(marker_sets sets, kgrids g, bin_desc bd, int with_forces,
                                 int* __restrict__ key, int* __restrict__ rank,
                                 int* __restrict__ code, int* __restrict__ count,
                                 bin_stats* __restrict__ stats)
{
    // No early return: every lane takes part in the wavefront reduction and
    // in the grouping of the rank atomics.
    int m = blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long fbits = 0;
    const bool valid = m < sets.total;
    int bin = -1;
    if (valid) {
        int k = set_of(sets, m);
        int l = m - sets.offset[k];
        int n = sets.offset[k + 1] - sets.offset[k];
        const double* x = sets.x[k];
        double p[3] = {x[l], x[n + l], x[2 * n + l]};
        int q[3];
        bin = 0;
        bool placed = true;                 // false at a NaN or infinite position
        int stride = 1;
        for (int j = 0; j < 3; ++j) {
            stencil_axis st = kstencil(g.a[bd.fc[j]][j], p[j]);
            placed = placed && isfinite(st.d);
            q[j] = st.base + bd.fs[j];
            int qb = q[j] - bd.qmin[j];
            qb = qb < 0 ? 0 : (qb >= bd.nb[j] ? bd.nb[j] - 1 : qb);
            bin += qb * stride;
            stride *= bd.nb[j];
        }
        int c9 = 0;
        for (int c = 0; c < 3; ++c)
            for (int j = 0; j < 3; ++j) {
                stencil_axis st = kstencil(g.a[c][j], p[j]);
                c9 |= ((st.base - q[j]) & 1) << (3 * c + j);
            }
        key[m] = bin;
        code[m] = c9;
        if (with_forces) {
            const double* f = sets.f[k];
            const double f0 = fabs(f[l]), f1 = fabs(f[n + l]), f2 = fabs(f[2 * n + l]);
            double a = f0 > f1 ? f0 : f1;
            a = a > f2 ? a : f2;
            // A non-finite force or position is recorded as the canonical NaN,
            // whose bit pattern exceeds every finite and infinite one, so it
            // survives the integer maxima below and poisons the spread result.
            if (!(placed && isfinite(f0) && isfinite(f1) && isfinite(f2))) a = __longlong_as_double(0x7ff8000000000000ll);
            fbits = (unsigned long long) __double_as_longlong(a);
        }
    }
    // Ranks inside a bin: consecutive markers mostly share a bin, so the
    // lanes of a wavefront are grouped by bin (one ballot per distinct bin)
    // and each group's first lane takes the group's ranks with one atomic;
    // the groups' atomics go out together, to distinct addresses.
    {
        const int lane = threadIdx.x & 63;
        const unsigned long long lt = (1ull << lane) - 1;
        unsigned long long todo = __ballot(valid);
        int leader = lane, before = 0, size = 0;
        while (todo) {
            const int l = __ffsll((long long) todo) - 1;
            const int lb = __shfl(bin, l, 64);
            const unsigned long long grp = __ballot(valid && bin == lb) & todo;
            if ((grp >> lane) & 1) {
                leader = l;
                before = __popcll(grp & lt);
            }
            if (lane == l) size = __popcll(grp);
            todo &= ~grp;
        }
        int base = 0;
        if (valid && leader == lane) base = atomicAdd(&count[bin], size);
        base = __shfl(base, leader, 64);
        if (valid) rank[m] = base + before;
    }
    if (with_forces) {
        fbits = wave_max(fbits);
        if ((threadIdx.x & 63) == 0 && fbits) atomicMax(&stats->max_abs_f[blockIdx.x % STAT_SLOTS], fbits);
    }
}

// Places each marker's ordering key (code, marker id) in its bin's range.
__global__ void bin_scatter_kernel(int total, const int* __restrict__ key, const int* __restrict__ rank,
                                   const int* __restrict__ code, const int* __restrict__ start,
                                   long long* __restrict__ tmp)
{
    int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= total) return;
    tmp[start[key[m]] + rank[m]] = ((long long) code[m] << 32) | (unsigned) m;
}

// Canonical order inside a bin: by (code, marker id).  Writes the permutation
// and sorted copies of positions and forces (SoA, 6 * total doubles).
__global__ void bin_canon_kernel(marker_sets sets, int with_forces,
                                 const int* __restrict__ key, const int* __restrict__ start,
                                 const long long* __restrict__ tmp,
                                 int* __restrict__ perm, double* __restrict__ sorted,
                                 bin_stats* __restrict__ stats)
{
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    int total = sets.total;
    unsigned long long cnt = 0;
    if (p < total) {
        const long long mine = tmp[p];
        int m = (int) (mine & 0xffffffffll);
        int b = key[m];
        int s = start[b], e = start[b + 1];
        int r = 0;
        for (int i = s; i < e; ++i) r += tmp[i] < mine;
        int dst = s + r;
        perm[dst] = m;
        cnt = (unsigned long long) (e - s);
        int k = set_of(sets, m);
        int l = m - sets.offset[k];
        int n = sets.offset[k + 1] - sets.offset[k];
        for (int j = 0; j < 3; ++j) sorted[(size_t) j * total + dst] = sets.x[k][(size_t) j * n + l];
        if (with_forces)
            for (int j = 0; j < 3; ++j) sorted[(size_t) (3 + j) * total + dst] = sets.f[k][(size_t) j * n + l];
    }
    cnt = wave_max(cnt);
    if ((threadIdx.x & 63) == 0 && cnt) atomicMax(&stats->max_count[blockIdx.x % STAT_SLOTS], cnt);
}

// ----------------------------------------------------------------------
// Spreading
//
// One workgroup per brick of BX x BY x BZ grid points (all three
// components).  The markers of the bins whose stencils reach the brick are
// walked in canonical order in chunks of 64; every wavefront owns a stream
// of chunks.  For a chunk, lanes are markers: each computes its separable
// weights once and, if its stencil meets the brick, stores them in the
// wavefront's LDS slice (compacted with a ballot).  Then each quarter of the
// wavefront walks a quarter of the compacted markers with lanes = the 16
// (sy, sz) rows of the stencil, four x points per lane: it sums the
// contributions of consecutive markers of one cell in registers and adds
// them to the brick tile when the cell changes.
//
// The tile holds 64-bit fixed-point integers (two's complement): integer
// addition is associative, so the four wavefronts may add in any order and
// the result is still bitwise reproducible.  The quantum q is a power of
// two chosen so that |sum| < 2^62 q for every point:
//     sum <= 64 cells * max_count * max|f| * h^-3 * max phi^3  (phi^3 <= 0.3),
// and each added cell sum is rounded to the nearest multiple of q, so a
// point's error is at most 64 * q / 2 per flush group, about 2^-55 of that
// bound.
// ----------------------------------------------------------------------
struct region_dim {
    int first;   // first bin coordinate (may be negative before wrapping)
    int count;   // number of bins
    int wrap;    // periodic wrap modulus (0 = none)
};

template <int B>
__device__ inline region_dim brick_region(const bin_desc& bd, const kaxis& fa, int j, int P0)
{
    region_dim r;
    int nb = bd.nb[j];
    if (!fa.solid) {
        int lo = P0 - 2 - bd.hi[j];
        int hi = P0 + B - bd.lo[j];
        if (hi - lo + 1 >= nb) { r.first = 0; r.count = nb; r.wrap = 0; }
        else { r.first = lo - bd.qmin[j]; r.count = hi - lo + 1; r.wrap = nb; }
    } else {
        int lo = P0 - 2 - bd.hi[j] - bd.qmin[j];
        int hi = P0 + B - bd.lo[j] - bd.qmin[j];
        lo = lo < 0 ? 0 : lo;
        hi = hi >= nb ? nb - 1 : hi;
        r.first = lo; r.count = hi >= lo ? hi - lo + 1 : 0; r.wrap = 0;
    }
    return r;
}

// Offset of stencil point (base + o - 1) inside the brick along one axis, or -1.
template <int B>
__device__ inline int brick_offset(const kaxis& a, int base, int o, int P0)
{
    int v = base + o - 1 - P0;
    if (!a.solid) {
        if (v < 0) v += a.cells;
        else if (v >= a.cells) v -= a.cells;
    }
    int lim = a.points - P0;
    lim = lim < B ? lim : B;
    return (v >= 0 && v < lim) ? v : -1;
}

__device__ inline void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int BX = 8, BY = 8, BZ = 8;
constexpr int BRICK_PTS = BX * BY * BZ;
constexpr int WAVES = SPREAD_THREADS / 64;
constexpr int MAX_ROWS = (BY + 4) * (BZ + 4);
constexpr int MAX_SEG2 = 2 * MAX_ROWS;
// Padded weight row: 2*WROW dwords is 2 mod 4, so any 16 consecutive rows
// start in distinct LDS banks, and the 8 extra entries absorb the reads of a
// final partial batch.
constexpr int WROW = CHUNK + 9;
constexpr int VISIT_BATCH = 4;
// Wx row of 6 doubles (48 bytes): the 16-byte stores of 16 consecutive lanes
// start 12 banks apart and cover distinct banks.
constexpr int WX_STRIDE = 6;
constexpr int POS_LIST = 2048;      // region markers listed in LDS; larger regions search the segments
// FAST: every periodic axis has at least BX + 8 cells, so a stencil that
// reaches the brick has a unique brick-relative origin in [-3, B).
constexpr int MIN_FAST_CELLS = BX + 8;
// Bias that keeps the flat brick index of a stencil origin in [-3, B)^3 positive (12 bits).
constexpr int ORG_BIAS = 3 + BX * (3 + BY * 3);
static_assert(ORG_BIAS + BRICK_PTS < 4096, "flat origin must fit in 12 bits");

// Whether the stencil of base cell `base` meets the brick along one axis;
// with FAST, also its brick-relative origin (offset of stencil point 0).
template <bool FAST, int B>
__device__ inline bool axis_hit(const kaxis& a, int base, int P0, int& origin)
{
    int lim = a.points - P0;
    lim = lim < B ? lim : B;
    if (FAST) {
        int v = base - 1 - P0;
        if (!a.solid) {
            if (v < -4) v += a.cells;
            else if (v >= a.cells - 4) v -= a.cells;
        }
        origin = v;
        return v + 3 >= 0 && v < lim;
    } else {
        origin = 0;
        bool m = false;
#pragma unroll
        for (int o = 0; o < 4; ++o) m = m || brick_offset<B>(a, base, o, P0) >= 0;
        return m;
    }
}

template <bool MAC, bool FAST>
__global__ void __launch_bounds__(SPREAD_THREADS)
spread_brick_kernel(kgrids g, bin_desc bd, int delta, int total,
                    const int* __restrict__ start, const double* __restrict__ sorted,
                    const bin_stats* __restrict__ stats,
                    double* __restrict__ fe0, double* __restrict__ fe1, double* __restrict__ fe2,
                    int bricks_x, int bricks_y, int nbricks, int xcd_chunk)
{
    __shared__ unsigned long long acc[3][BRICK_PTS];
    __shared__ double W[WAVES][16][WROW];     // wz[a] * wy[b] * f at row 4a + b
    __shared__ __attribute__((aligned(16))) double Wx[WAVES][CHUNK + VISIT_BATCH][WX_STRIDE];   // wx[0..3]
    __shared__ int org[WAVES][CHUNK + VISIT_BATCH];
    __shared__ int seg_begin[MAX_SEG2];
    __shared__ int seg_pref[MAX_SEG2 + 1];
    __shared__ int pos_list[POS_LIST];
    __shared__ double bound_s;

    const int tid = threadIdx.x;
    int bid = blockIdx.x;
    if (xcd_chunk > 0) bid = (bid & 7) * xcd_chunk + (bid >> 3);
    if (bid >= nbricks) return;
    const int P0x = (bid % bricks_x) * BX;
    const int P0y = ((bid / bricks_x) % bricks_y) * BY;
    const int P0z = (bid / (bricks_x * bricks_y)) * BZ;

    for (int i = tid; i < 3 * BRICK_PTS; i += SPREAD_THREADS) (&acc[0][0])[i] = 0ull;

    region_dim rx = brick_region<BX>(bd, g.a[bd.fc[0]][0], 0, P0x);
    region_dim ry = brick_region<BY>(bd, g.a[bd.fc[1]][1], 1, P0y);
    region_dim rz = brick_region<BZ>(bd, g.a[bd.fc[2]][2], 2, P0z);
    const int rows = ry.count * rz.count;          // <= MAX_ROWS (checked on the host)
    const int nseg = 2 * rows;
    for (int r = tid; r < rows; r += SPREAD_THREADS) {
        int yy = ry.first + r % ry.count;
        int zz = rz.first + r / ry.count;
        if (ry.wrap) yy = (yy % ry.wrap + ry.wrap) % ry.wrap;
        if (rz.wrap) zz = (zz % rz.wrap + rz.wrap) % rz.wrap;
        int row = (zz * bd.nb[1] + yy) * bd.nb[0];
        int x0 = rx.first;
        if (rx.wrap) x0 = (x0 % rx.wrap + rx.wrap) % rx.wrap;
        int c0 = rx.count, c1 = 0;
        if (rx.wrap && x0 + rx.count > bd.nb[0]) { c0 = bd.nb[0] - x0; c1 = rx.count - c0; }
        int s0 = start[row + x0], e0 = start[row + x0 + c0];
        int s1 = start[row], e1 = c1 ? start[row + c1] : s1;
        seg_begin[2 * r] = s0;     seg_pref[2 * r + 1] = e0 - s0;
        seg_begin[2 * r + 1] = s1; seg_pref[2 * r + 2] = e1 - s1;
    }
    __syncthreads();
    if (tid < 64) {
        constexpr int PER = (MAX_SEG2 + 63) / 64;
        int vals[PER];
        int sum = 0;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int idx = tid * PER + i;
            vals[i] = idx < nseg ? seg_pref[idx + 1] : 0;
            sum += vals[i];
        }
        int incl = sum;
        for (int off = 1; off < 64; off <<= 1) {
            int y = __shfl_up(incl, off, 64);
            if (tid >= off) incl += y;
        }
        int run = incl - sum;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int idx = tid * PER + i;
            run += vals[i];
            if (idx < nseg) seg_pref[idx + 1] = run;
        }
        if (tid == 0) seg_pref[0] = 0;
        unsigned long long fb = wave_max(stats->max_abs_f[tid]);
        unsigned long long cm = wave_max(stats->max_count[tid]);
        if (tid == 0) {
            double res3 = fmax(g.res3[0], fmax(g.res3[1], g.res3[2]));
            bound_s = 64.0 * (double) cm * __longlong_as_double((long long) fb) * res3 * 0.3;
        }
    }
    __syncthreads();
    const int T = seg_pref[nseg];
    // Flattened sorted positions of the region's markers (when they fit).
    const bool listed = T <= POS_LIST;
    if (listed)
        for (int i = tid; i < nseg; i += SPREAD_THREADS) {
            int b = seg_begin[i], o = seg_pref[i], n = seg_pref[i + 1] - o;
            for (int k = 0; k < n; ++k) pos_list[o + k] = b + k;
        }
    __syncthreads();
    // A NaN or infinite force or position makes the bound non-finite: every point is then
    // written as NaN (the accumulation below still runs, on a dummy quantum).
    const bool poisoned = !(bound_s <= 1.7976931348623157e308);
    int e2 = 0;
    if (!poisoned && bound_s > 0) frexp(bound_s, &e2);
    const double inv_q = ldexp(1.0, 62 - e2);

    const int wave = tid >> 6;
    const int lane = tid & 63;
    const unsigned long long lanemask_lt = (1ull << lane) - 1;

    // Sorted position of region marker idx (binary search over the segments).
    auto locate = [&](int idx) {
        if (listed) return pos_list[idx];
        int lo = 0, hi = nseg;
        while (hi - lo > 1) {
            int mid = (lo + hi) >> 1;
            if (seg_pref[mid] <= idx) lo = mid; else hi = mid;
        }
        return seg_begin[lo] + (idx - seg_pref[lo]);
    };
    // Positions and forces of the next chunk are loaded while the current
    // one is processed.
    double np_[3] = {0, 0, 0}, nf_[3] = {0, 0, 0};
    {
        int idx = wave * CHUNK + lane;
        if (idx < T) {
            int pp = locate(idx);
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                np_[j] = sorted[(size_t) j * total + pp];
                nf_[j] = sorted[(size_t) (3 + j) * total + pp];
            }
        }
    }
    for (int cb = wave * CHUNK; cb < T; cb += WAVES * CHUNK) {
        // ---- lanes are markers ----
        int idx = cb + lane;
        bool valid = idx < T;
        double p[3] = {np_[0], np_[1], np_[2]}, fv[3] = {nf_[0], nf_[1], nf_[2]};
        {
            int nidx = idx + WAVES * CHUNK;
            if (nidx < T) {
                int pp = locate(nidx);
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    np_[j] = sorted[(size_t) j * total + pp];
                    nf_[j] = sorted[(size_t) (3 + j) * total + pp];
                }
            }
        }
        double w0[3][4], w1[3][4];
        int b0[3], b1[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            stencil_axis st = kstencil(g.a[g.cand[0][j]][j], p[j]);
            b0[j] = st.base;
            delta4(delta, st.d, w0[j]);
            if (MAC || g.cand[1][j] != g.cand[0][j]) {
                st = kstencil(g.a[g.cand[1][j]][j], p[j]);
                b1[j] = st.base;
                delta4(delta, st.d, w1[j]);
            } else {
                b1[j] = b0[j];
#pragma unroll
                for (int o = 0; o < 4; ++o) w1[j][o] = w0[j][o];
            }
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const bool s0 = MAC ? (c == 0) : (g.sel[c][0] != 0);
            const bool s1 = MAC ? (c == 1) : (g.sel[c][1] != 0);
            const bool s2 = MAC ? (c == 2) : (g.sel[c][2] != 0);
            const int bb0 = s0 ? b1[0] : b0[0];
            const int bb1 = s1 ? b1[1] : b0[1];
            const int bb2 = s2 ? b1[2] : b0[2];
            double w[3][4];
#pragma unroll
            for (int o = 0; o < 4; ++o) {
                w[0][o] = s0 ? w1[0][o] : w0[0][o];
                w[1][o] = s1 ? w1[1][o] : w0[1][o];
                w[2][o] = s2 ? w1[2][o] : w0[2][o];
            }
            // Does the stencil meet the brick?  Brick-relative origin of stencil point 0.
            int ow0, ow1, ow2;
            bool hit = valid && axis_hit<FAST, BX>(g.a[c][0], bb0, P0x, ow0)
                             && axis_hit<FAST, BY>(g.a[c][1], bb1, P0y, ow1)
                             && axis_hit<FAST, BZ>(g.a[c][2], bb2, P0z, ow2);
            const unsigned long long hits = __ballot(hit);
            const int nh = __popcll(hits);
            const int slot = __popcll(hits & lanemask_lt);
            if (hit) {
                double fc = fv[c] * g.res3[c];
                double2* wxp = reinterpret_cast<double2*>(&Wx[wave][slot][0]);
                wxp[0] = make_double2(w[0][0], w[0][1]);
                wxp[1] = make_double2(w[0][2], w[0][3]);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    double wyf = w[1][b] * fc;
#pragma unroll
                    for (int a = 0; a < 4; ++a) W[wave][4 * a + b][slot] = w[2][a] * wyf;
                }
                if (FAST) {
                    // flat brick index of stencil point 0 (biased to stay positive) and,
                    // per axis, which of the four offsets fall inside the brick
                    int lx = min(g.a[c][0].points - P0x, BX), ly = min(g.a[c][1].points - P0y, BY);
                    int lz = min(g.a[c][2].points - P0z, BZ);
                    int mx = 0, my = 0, mz = 0;
#pragma unroll
                    for (int o = 0; o < 4; ++o) {
                        mx |= ((unsigned) (ow0 + o) < (unsigned) lx) << o;
                        my |= ((unsigned) (ow1 + o) < (unsigned) ly) << o;
                        mz |= ((unsigned) (ow2 + o) < (unsigned) lz) << o;
                    }
                    int flat = ow0 + BX * (ow1 + BY * ow2) + ORG_BIAS;
                    org[wave][slot] = flat | (mx << 12) | (my << 16) | (mz << 20);
                } else {
                    org[wave][slot] = (bb0 + 1) | ((bb1 + 1) << 10) | ((bb2 + 1) << 20);
                }
            }
            wave_sync();
            // ---- lanes are (quarter q, sy, sz), each for the four x points ----
            // Quarter q walks compacted markers [q per, (q+1) per) and sums
            // the contributions of consecutive markers of one cell in four
            // registers; a change of cell (stencil origin) adds them to the tile.
            const kaxis& ax = g.a[c][0];
            const kaxis& ay = g.a[c][1];
            const kaxis& az = g.a[c][2];
            const int qy = lane & 3, qz = (lane >> 2) & 3, quarter = lane >> 4;
            const double* wrow = &W[wave][4 * qz + qy][0];
            const int per = (nh + 3) >> 2;
            const int kbeg = quarter * per;
            const int kend = min(kbeg + per, nh);
            const int lane_off = BX * (qy + BY * qz) - ORG_BIAS;
            double P[4] = {0.0, 0.0, 0.0, 0.0};
            int cur = -1;
            auto flush = [&]() {
                if (cur < 0) return;
                if (FAST) {
                    const int o = cur;
                    if ((o >> (16 + qy)) & (o >> (20 + qz)) & 1) {
                        const int t0 = (o & 4095) + lane_off;
#pragma unroll
                        for (int sx = 0; sx < 4; ++sx)
                            if ((o >> (12 + sx)) & 1)
                                atomicAdd(&acc[c][t0 + sx], (unsigned long long) __double2ll_rn(P[sx] * inv_q));
                    }
                } else {
                    const int o = cur;
                    int oy = brick_offset<BY>(ay, ((o >> 10) & 1023) - 1, qy, P0y);
                    int oz = brick_offset<BZ>(az, ((o >> 20) & 1023) - 1, qz, P0z);
                    if (oy >= 0 && oz >= 0) {
#pragma unroll
                        for (int sx = 0; sx < 4; ++sx) {
                            int ox = brick_offset<BX>(ax, (o & 1023) - 1, sx, P0x);
                            if (ox >= 0)
                                atomicAdd(&acc[c][ox + BX * (oy + BY * oz)],
                                          (unsigned long long) __double2ll_rn(P[sx] * inv_q));
                        }
                    }
                }
            };
            for (int k0 = kbeg; k0 < kend; k0 += VISIT_BATCH) {
                // all loads of the batch first (entries past kend are never used)
                int ov[VISIT_BATCH];
                double pv[VISIT_BATCH];
                double2 xa[VISIT_BATCH], xb[VISIT_BATCH];
#pragma unroll
                for (int i = 0; i < VISIT_BATCH; ++i) {
                    ov[i] = org[wave][k0 + i];
                    pv[i] = wrow[k0 + i];
                    const double2* wxp = reinterpret_cast<const double2*>(&Wx[wave][k0 + i][0]);
                    xa[i] = wxp[0];
                    xb[i] = wxp[1];
                }
#pragma unroll
                for (int i = 0; i < VISIT_BATCH; ++i) {
                    if (k0 + i < kend) {
                        if (ov[i] != cur) {
                            flush();
                            P[0] = P[1] = P[2] = P[3] = 0.0;
                            cur = ov[i];
                        }
                        P[0] = fma(xa[i].x, pv[i], P[0]);
                        P[1] = fma(xa[i].y, pv[i], P[1]);
                        P[2] = fma(xb[i].x, pv[i], P[2]);
                        P[3] = fma(xb[i].y, pv[i], P[3]);
                    }
                }
            }
            flush();
            wave_sync();
        }
    }
    __syncthreads();

    // Each grid point belongs to exactly one brick: plain stores.
    const double q = poisoned ? __longlong_as_double(0x7ff8000000000000ll) : ldexp(1.0, e2 - 62);
    double* fe[3] = {fe0, fe1, fe2};
    for (int i = tid; i < BRICK_PTS; i += SPREAD_THREADS) {
        int tx = i % BX, ty = (i / BX) % BY, tz = i / (BX * BY);
        int X = P0x + tx, Y = P0y + ty, Z = P0z + tz;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int* pt = g.points[c];
            if (X < pt[0] && Y < pt[1] && Z < pt[2])
                fe[c][(size_t) X + (size_t) pt[0] * ((size_t) Y + (size_t) pt[1] * Z)] =
                    (double) (long long) acc[c][i] * q;
        }
    }
}

// ----------------------------------------------------------------------
// Host side
// ----------------------------------------------------------------------
kaxis to_kaxis(const ibm_axis& a)
{
    kaxis k;
    k.length = a.length; k.resolution = a.resolution; k.shift = a.shift;
    k.s_over_r = a.shift / a.resolution;
    k.cells = a.cells; k.points = a.points; k.solid = a.solid; k.pad = 0;
    return k;
}

ibm_status make_kgrids(ibm_ctx* ctx, const ibm_grid* grids, kgrids* out)
{
    if (!grids) return fail(ctx, IBM_ERR_ARG, "grids is null");
    for (int c = 0; c < 3; ++c) {
        if (grids[c].dims != 3)
            return fail(ctx, IBM_ERR_ARG, "spread/interpolate support 3-dimensional grids (got %d)", grids[c].dims);
        double r = 1.0;
        for (int j = 0; j < 3; ++j) {
            out->a[c][j] = to_kaxis(grids[c].axis[j]);
            out->points[c][j] = grids[c].axis[j].points;
            r *= grids[c].axis[j].resolution;
            if (grids[c].axis[j].cells < 1 || grids[c].axis[j].points < 1)
                return fail(ctx, IBM_ERR_BAD_GRID, "empty grid axis");
        }
        out->res3[c] = r;
        if ((long long) grids[c].axis[0].points * grids[c].axis[1].points * grids[c].axis[2].points > INT_MAX)
            return fail(ctx, IBM_ERR_SIZE, "spread/interpolate grids hold at most %d points", INT_MAX);
    }
    // Along each dimension the component grids may use at most two distinct
    // discretisations (MAC: the face-aligned one and the centred one).
    for (int j = 0; j < 3; ++j) {
        out->cand[0][j] = 0;
        out->cand[1][j] = 0;
        int ncand = 1;
        for (int c = 0; c < 3; ++c) {
            const ibm_axis& a = grids[c].axis[j];
            int found = -1;
            for (int k = 0; k < ncand; ++k) {
                const ibm_axis& b = grids[out->cand[k][j]].axis[j];
                if (a.shift == b.shift && a.resolution == b.resolution && a.cells == b.cells &&
                    a.points == b.points && a.solid == b.solid && a.length == b.length) {
                    found = k;
                    break;
                }
            }
            if (found < 0) {
                if (ncand == 2)
                    return fail(ctx, IBM_ERR_BAD_GRID, "more than two staggerings along dimension %d", j);
                out->cand[1][j] = c;
                found = ncand++;
            }
            out->sel[c][j] = found;
        }
        // Canonical order for a MAC-shaped axis (component j alone differs):
        // candidate 1 is component j, candidate 0 the shared centred axis.
        if (ncand == 2) {
            int other = (j + 1) % 3, third = (j + 2) % 3;
            if (out->sel[j][j] != out->sel[other][j] && out->sel[other][j] == out->sel[third][j]) {
                out->cand[0][j] = other;
                out->cand[1][j] = j;
                for (int c = 0; c < 3; ++c) out->sel[c][j] = (c == j) ? 1 : 0;
            }
        }
    }
    return IBM_OK;
}

ibm_status make_sets(ibm_ctx* ctx, int nsets, const int* n, const double* const* x,
                     const double* const* f, double* const* out, marker_sets* s)
{
    if (nsets < 0 || nsets > MAX_SETS) return fail(ctx, IBM_ERR_ARG, "nsets must be in [0, %d]", MAX_SETS);
    if (nsets > 0 && (!n || !x)) return fail(ctx, IBM_ERR_ARG, "null marker arrays");
    s->nsets = nsets;
    long long total = 0;
    s->offset[0] = 0;
    for (int k = 0; k < nsets; ++k) {
        if (n[k] < 0) return fail(ctx, IBM_ERR_SIZE, "negative marker count");
        if (n[k] > 0 && !x[k]) return fail(ctx, IBM_ERR_ARG, "null positions for set %d", k);
        if (n[k] > 0 && f && !f[k]) return fail(ctx, IBM_ERR_ARG, "null forces for set %d", k);
        if (n[k] > 0 && out && !out[k]) return fail(ctx, IBM_ERR_ARG, "null output for set %d", k);
        s->x[k] = x[k];
        s->f[k] = f ? f[k] : nullptr;
        s->out[k] = out ? out[k] : nullptr;
        total += n[k];
        s->offset[k + 1] = (int) total;
    }
    if (total > (1LL << 30)) return fail(ctx, IBM_ERR_SIZE, "too many markers");
    s->total = (int) total;
    return IBM_OK;
}

bin_desc make_bins(const ibm_grid* grids)
{
    bin_desc bd;
    long long nbins = 1;
    for (int j = 0; j < 3; ++j) {
        int fc = -1;
        for (int c = 0; c < 3; ++c)
            if (grids[c].axis[j].alignment == 0.0) { fc = c; break; }
        if (fc < 0) fc = 0;
        const ibm_axis& fa = grids[fc].axis[j];
        int fs = (int) fa.shift;                  // 0 or 1 for face grids, 0 otherwise
        bd.fc[j] = fc;
        bd.fs[j] = fs;
        if (fa.solid) { bd.qmin[j] = -1 + fs; bd.nb[j] = fa.points + 1; }
        else { bd.qmin[j] = 0; bd.nb[j] = fa.cells; }
        // base_c - q = floor(y - D) - floor(y) - fs with y = x/h - fs and
        // D = shift_c - fs, i.e. in {-ceil(D) - fs, -floor(D) - fs}.
        int lo = INT_MAX, hi = INT_MIN;
        for (int c = 0; c < 3; ++c) {
            double delta = grids[c].axis[j].shift - fs;
            int a = -(int) ceil(delta) - fs, b = -(int) floor(delta) - fs;
            lo = a < lo ? a : lo;
            hi = b > hi ? b : hi;
        }
        bd.lo[j] = lo;
        bd.hi[j] = hi;
        nbins *= bd.nb[j];
    }
    // Grids are limited to INT_MAX points (make_kgrids), so this only fails
    // with walls adding a bin row; callers check nbins > 0.
    bd.nbins = nbins <= INT_MAX - 1 ? (int) nbins : -1;
    return bd;
}

int blocks_for(long long n, int threads) { return (int) ((n + threads - 1) / threads); }

// Device buffers of one binning pass.
struct bin_work {
    int *count, *start, *key, *rank, *perm, *code;
    long long* tmp;
    double* sorted;          // 6 * total doubles: positions, then forces (SoA)
    bin_stats* stats;
    void* scan_tmp;
    size_t scan_bytes;
};

// The binning buffers in the context's scratch slots (grown on demand).
ibm_status ctx_bin_work(ibm_ctx* ctx, int total, int nbins, bin_work* w)
{
    void* p;
    IBM_TRY(scratch(ctx, SLOT_BIN_COUNT, sizeof(int) * (size_t) (nbins + 1), &p)); w->count = (int*) p;
    IBM_TRY(scratch(ctx, SLOT_BIN_START, sizeof(int) * (size_t) (nbins + 1), &p)); w->start = (int*) p;
    IBM_TRY(scratch(ctx, SLOT_KEY, sizeof(int) * (size_t) total, &p)); w->key = (int*) p;
    IBM_TRY(scratch(ctx, SLOT_RANK, sizeof(int) * (size_t) total, &p)); w->rank = (int*) p;
    IBM_TRY(scratch(ctx, SLOT_TMP, sizeof(long long) * (size_t) total, &p)); w->tmp = (long long*) p;
    IBM_TRY(scratch(ctx, SLOT_PERM, sizeof(int) * (size_t) total, &p)); w->perm = (int*) p;
    IBM_TRY(scratch(ctx, SLOT_CODE, sizeof(int) * (size_t) total, &p)); w->code = (int*) p;
    IBM_TRY(scratch(ctx, SLOT_SORTED, sizeof(double) * 6 * (size_t) total, &p)); w->sorted = (double*) p;
    IBM_TRY(scratch(ctx, SLOT_FLAGS, sizeof(bin_stats), &p)); w->stats = (bin_stats*) p;
    size_t tbytes = 0;
    IBM_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, tbytes, w->count, w->start, nbins + 1, ctx->stream));
    IBM_TRY(scratch(ctx, SLOT_SCAN_TMP, tbytes, &p));
    w->scan_tmp = p;
    w->scan_bytes = tbytes;
    return IBM_OK;
}

// Counting sort of all markers into bins: leaves the bin starts (nbins+1),
// the permutation and sorted positions (and forces) in `w`.  Every buffer
// that must start at zero is cleared here, by kernels (no memset), so the
// pass can be recorded in a HIP graph and run on reused memory.
ibm_status bin_markers(ibm_ctx* ctx, const marker_sets& sets, const kgrids& kg, const bin_desc& bd,
                       int with_forces, const bin_work& w, bool timed)
{
    const int total = sets.total;
    const int nbins = bd.nbins;
    prof_scope prof(ctx, timed ? "bin" : nullptr);
    {
        size_t words = (size_t) nbins + 1;
        zero_words_kernel<<<blocks_for((long) std::min<size_t>(words, 1u << 22), 256), 256, 0, ctx->stream>>>(
            (unsigned int*) w.count, words);
        IBM_LAUNCH_CHECK(ctx);
        zero_words_kernel<<<1, 256, 0, ctx->stream>>>((unsigned int*) w.stats, sizeof(bin_stats) / 4);
        IBM_LAUNCH_CHECK(ctx);
    }
    if (total > 0) {
        bin_count_kernel<<<blocks_for(total, 256), 256, 0, ctx->stream>>>(sets, kg, bd, with_forces, w.key, w.rank,
                                                                           w.code, w.count, w.stats);
        IBM_LAUNCH_CHECK(ctx);
    }
    size_t tbytes = w.scan_bytes;
    IBM_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(w.scan_tmp, tbytes, w.count, w.start, nbins + 1, ctx->stream));
    if (total > 0) {
        bin_scatter_kernel<<<blocks_for(total, 256), 256, 0, ctx->stream>>>(total, w.key, w.rank, w.code, w.start,
                                                                             w.tmp);
        IBM_LAUNCH_CHECK(ctx);
        bin_canon_kernel<<<blocks_for(total, 256), 256, 0, ctx->stream>>>(sets, with_forces, w.key, w.start, w.tmp,
                                                                           w.perm, w.sorted, w.stats);
        IBM_LAUNCH_CHECK(ctx);
    }
    return IBM_OK;
}

ibm_status check_delta(ibm_ctx* ctx, int delta)
{
    if (delta != IBM_DELTA_COSINE && delta != IBM_DELTA_PESKIN && delta != IBM_DELTA_BSPLINE3)
        return fail(ctx, IBM_ERR_ARG, "unknown delta kind %d", delta);
    return IBM_OK;
}

using namespace ibm_fixed;
static_assert(sizeof(bin_stats) <= STATIC_STATS_BYTES, "binning statistics exceed their fixed slot");
constexpr int STATIC_MAX_DEVICES = 64;
std::mutex static_scratch_mutex;
void* static_scratch_ptr[STATIC_MAX_DEVICES] = {};

ibm_status static_limits(ibm_ctx* ctx, int total, int nbins)
{
    if ((size_t) total > STATIC_MAX_MARKERS)
        return fail(ctx, IBM_ERR_SIZE, "ibm_spread_sets_noalloc takes at most %zu markers (got %d)",
                    STATIC_MAX_MARKERS, total);
    if ((size_t) nbins > STATIC_MAX_BINS)
        return fail(ctx, IBM_ERR_SIZE, "ibm_spread_sets_noalloc takes grids of at most %zu bins (got %d)",
                    STATIC_MAX_BINS, nbins);
    return IBM_OK;
}

// Carves the binning buffers of the brick kernel out of the fixed workspace
// at `base` (a device address of `scratch`).
ibm_status static_bin_work(ibm_ctx* ctx, unsigned char* base, int nbins, bin_work* w)
{
    size_t off = 0;
    auto take = [&](size_t bytes) { unsigned char* p = base + off; off += align256(bytes); return p; };
    w->count = (int*) take(STATIC_BIN_WORDS);
    w->start = (int*) take(STATIC_BIN_WORDS);
    w->key = (int*) take(STATIC_INT_ARRAY);
    w->rank = (int*) take(STATIC_INT_ARRAY);
    w->perm = (int*) take(STATIC_INT_ARRAY);
    w->code = (int*) take(STATIC_INT_ARRAY);
    w->tmp = (long long*) take(sizeof(long long) * STATIC_MAX_MARKERS);
    w->sorted = (double*) take(sizeof(double) * 6 * STATIC_MAX_MARKERS);
    w->stats = (bin_stats*) take(STATIC_STATS_BYTES);
    w->scan_tmp = base + off;
    size_t tbytes = 0;
    // A size query: rocPRIM neither allocates nor launches anything here.
    IBM_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, tbytes, w->count, w->start, nbins + 1, ctx->stream));
    if (tbytes > STATIC_SCAN_BYTES)
        return fail(ctx, IBM_ERR_SIZE, "scan workspace of %zu bytes exceeds the fixed %zu", tbytes, STATIC_SCAN_BYTES);
    w->scan_bytes = tbytes;
    return IBM_OK;
}

// ----------------------------------------------------------------------
// Tile spreading: every marker is visited once.
//
// The markers of nboxes independent boxes (one set of component grids,
// repeated; the C4 channel is one box, the small periodic boxes of a batch
// are many) are counting-sorted into bins of 4 x 4 x 4 face-aligned cells,
// eight to a "brick" of 8 x 8 x 8, brick-major.  One workgroup per brick adds
// each of its markers' 64 stencil values per component into a 12 x 12 x 12
// tile of 64-bit fixed-point integers in LDS (the brick's points plus the
// reach of its stencils), and stores the tile once.  A merge pass then forms
// every grid point from the tiles that cover it.  Integer addition is
// associative, so the result does not depend on scheduling nor on the order
// inside a bin: no floating-point atomics, no global atomics on the grid,
// bitwise reproducible.
//
// Tile geometry along axis j: brick b covers bins q in [8 b, 8 b + 8) (bin
// coordinates relative to qmin; the last brick of an axis may be partial); a
// marker of bin q has base cell base_c = q + qmin + d_c for component c with
// d_c in [lo_j, hi_j] (hi_j - lo_j <= 1), and touches points base_c - 1 ..
// base_c + 2, so the tile starts at point T0 = 8 b + qmin + lo - 1 and a
// marker's stencil origin lies at tile index (q - 8 b) + (d_c - lo) in
// [0, 8].  On a periodic axis the tile index of a point is its distance from
// T0 modulo the cells, plus any multiple of them that stays in the tile.
// ----------------------------------------------------------------------
constexpr int TB = 8;                       // brick edge in cells
constexpr int SUB = 8;                      // bins (of 4 x 4 x 4 cells) per brick
constexpr int TT = 12;                      // tile edge in points
constexpr int TILE_PTS = TT * TT * TT;
constexpr int TILE_THREADS = 256;

struct tile_desc {
    int nbr[3];         // bricks per axis
    int bricks;         // bricks per box
    int nboxes;
    int keys;           // nboxes * bricks * SUB
    int box_points[3];  // points of one box's component grid
};

// Box of marker m: offsets holds nboxes + 1 increasing marker indices.  All 64
// lanes call it together, the first with the smallest m, whose box is found by
// comparing 64 offsets at a time (a wavefront's markers mostly lie in one box,
// and a bisection per lane is log2(nboxes) dependent loads); lanes beyond that
// box bisect the rest.
__device__ inline int box_of(const int* __restrict__ off, int nboxes, int m)
{
    const int m0 = __builtin_amdgcn_readfirstlane(m), lane = threadIdx.x & 63;
    int lo = 0, n = nboxes;
    while (n > 1) {
        const int step = (n + 63) / 64;
        const int before = __popcll(__ballot(lane * step < n && off[lo + min(lane * step, n - 1)] <= m0));
        lo += (before - 1) * step;
        n = min(step, n - (before - 1) * step);
    }
    if (lo + 1 < nboxes && off[lo + 1] <= m) {
        int hi = nboxes;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (off[mid] <= m) lo = mid; else hi = mid;
        }
    }
    return lo;
}

// Global load through a pointer that comes out of an indexed table (which
// would otherwise compile to a flat load).
__device__ inline double gload(const double* p, size_t i)
{
    return ((const __attribute__((address_space(1))) double*) p)[i];
}

__device__ inline void load_marker(const marker_sets& sets, int m, double (&p)[3])
{
    const int k = set_of(sets, m), l = m - sets.offset[k];
    const size_t n = (size_t) (sets.offset[k + 1] - sets.offset[k]);
#pragma unroll
    for (int j = 0; j < 3; ++j) p[j] = gload(sets.x[k], j * n + l);
}

__device__ inline void load_force(const marker_sets& sets, int m, double (&f)[3])
{
    const int k = set_of(sets, m), l = m - sets.offset[k];
    const size_t n = (size_t) (sets.offset[k + 1] - sets.offset[k]);
#pragma unroll
    for (int j = 0; j < 3; ++j) f[j] = gload(sets.f[k], j * n + l);
}

__device__ inline double load_force(const marker_sets& sets, int m, int c)
{
    const int k = set_of(sets, m), l = m - sets.offset[k];
    return gload(sets.f[k], (size_t) c * (sets.offset[k + 1] - sets.offset[k]) + l);
}

// Clears the bin counts and the statistics of a tile spread.
__global__ void __launch_bounds__(256) tile_clear_kernel(int* __restrict__ count, int keys, bin_stats* __restrict__ stats)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < keys + 1) count[i] = 0;
    if (blockIdx.x == 0)
        for (int w = threadIdx.x; w < (int) (sizeof(bin_stats) / 4); w += 256) ((unsigned*) stats)[w] = 0u;
}

// Bin of every marker, its rank inside the bin and the force maximum.  Bound
// by latency (positions and forces, then the returning atomics): a thread
// takes COUNT_ITEMS markers, 64 apart, so that their loads and atomics are in
// flight together.  Consecutive markers mostly share a bin, so a wavefront
// finds its few distinct bins by ballots and takes each one's ranks with one
// atomic.  2.39 M markers: 134 us with single-cell bins (a wavefront meets
// twenty or more), 102 with 4 x 4 x 4-cell bins, 58 with four markers a
// thread.  Scattered markers share no bins: a round of ballots for each of a
// wavefront's 256 would be a chain of 33 us (2000 markers; 13 so), so only the
// first COUNT_GROUPS bins of 64 markers are found that way.
constexpr int COUNT_ITEMS = 4, COUNT_GROUPS = 24;

__global__ void __launch_bounds__(256)
tile_count_kernel(marker_sets sets, kgrids g, bin_desc bd, tile_desc td, const int* __restrict__ box_off,
                  int* __restrict__ key, int* __restrict__ rank, int* __restrict__ count, bin_stats* __restrict__ stats)
{
    const int lane = threadIdx.x & 63;
    const int m0 = (blockIdx.x * 4 + (int) (threadIdx.x >> 6)) * (64 * COUNT_ITEMS) + lane;
    double p[COUNT_ITEMS][3], f[COUNT_ITEMS][3];
#pragma unroll
    for (int i = 0; i < COUNT_ITEMS; ++i) {
        const int m = min(m0 + 64 * i, sets.total - 1);
        load_marker(sets, m, p[i]);
        load_force(sets, m, f[i]);
    }
    unsigned long long fbits = 0;
    int groups = COUNT_GROUPS;
    int bin[COUNT_ITEMS], leader[COUNT_ITEMS], before[COUNT_ITEMS], base[COUNT_ITEMS];
#pragma unroll
    for (int i = 0; i < COUNT_ITEMS; ++i) {
        const int m = m0 + 64 * i;
        const bool valid = m < sets.total;
        int br[3], sub = 0;
        bool placed = true;                 // false at a NaN or infinite position, whose weights are NaN
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            stencil_axis st = kstencil(g.a[bd.fc[j]][j], p[i][j]);
            placed = placed && isfinite(st.d);
            int qb = st.base + bd.fs[j] - bd.qmin[j];
            qb = qb < 0 ? 0 : (qb >= bd.nb[j] ? bd.nb[j] - 1 : qb);
            br[j] = qb / TB;
            sub |= ((qb >> 2) & 1) << j;
        }
        const int box = td.nboxes > 1 ? box_of(box_off, td.nboxes, min(m, sets.total - 1)) : 0;
        bin[i] = (((box * td.nbr[2] + br[2]) * td.nbr[1] + br[1]) * td.nbr[0] + br[0]) * SUB + sub;
        const double f0 = fabs(f[i][0]), f1 = fabs(f[i][1]), f2 = fabs(f[i][2]);
        double a = f0 > f1 ? f0 : f1;
        a = a > f2 ? a : f2;
        // A non-finite force or position is recorded as the canonical NaN,
        // whose bit pattern exceeds every finite and infinite one, so it
        // survives the integer maxima and poisons the spread result (the
        // integers below cannot carry a NaN).
        if (!(placed && isfinite(f0) && isfinite(f1) && isfinite(f2))) a = __longlong_as_double(0x7ff8000000000000ll);
        if (valid) {
            key[m] = bin[i];
            const unsigned long long bits = (unsigned long long) __double_as_longlong(a);
            fbits = bits > fbits ? bits : fbits;
        }
        // ranks inside a bin, one atomic per group of lanes sharing a bin;
        // lanes beyond the first bins take theirs alone
        const unsigned long long lt = (1ull << lane) - 1;
        unsigned long long todo = __ballot(valid);
        int size = 0;
        leader[i] = lane;
        before[i] = 0;
        for (int group = 0; todo && group < groups; ++group) {
            const int l = __ffsll((long long) todo) - 1;
            const int lbin = __shfl(bin[i], l, 64);
            const unsigned long long grp = __ballot(valid && bin[i] == lbin) & todo;
            if ((grp >> lane) & 1) {
                leader[i] = l;
                before[i] = __popcll(grp & lt);
            }
            if (lane == l) size = __popcll(grp);
            todo &= ~grp;
        }
        if (todo >> lane & 1) size = 1;
        if (todo) groups = 2;                                // scattered markers: the next are, too
        base[i] = 0;
        if (valid && leader[i] == lane) base[i] = atomicAdd(&count[bin[i]], size);
    }
#pragma unroll
    for (int i = 0; i < COUNT_ITEMS; ++i) {
        const int r = __shfl(base[i], leader[i], 64) + before[i];
        if (m0 + 64 * i < sets.total) rank[m0 + 64 * i] = r;
    }
    fbits = wave_max(fbits);
    if (lane == 0 && fbits) atomicMax(&stats->max_abs_f[blockIdx.x % STAT_SLOTS], fbits);
}

// The marker indices in bin order (start[key] + rank).
__global__ void __launch_bounds__(256)
tile_place_kernel(int total, const int* __restrict__ key, const int* __restrict__ rank, const int* __restrict__ start,
                  int* __restrict__ perm)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < total) perm[start[key[m]] + rank[m]] = m;
}

// The fixed-point quantum q = 2^(e - 62), e the exponent of a bound on any
// point's sum: the base cells whose stencils reach a point lie in five
// consecutive face-aligned cells per axis, so in `reach` bins (two per axis,
// three where the last bin of a periodic axis is partial), and |sum| <= reach
// max_count max|f| max_c res3_c phi^3, phi the delta kernel's maximum.  A
// non-finite bound marks the result as poisoned (all NaN).
//
// It also decides whether tile_gather_kernel takes the spread: where no bin
// holds more than gather_most markers (0: never).
struct tile_scale {
    double inv_q, q;
    int poisoned, gather;
};

__device__ inline void make_scale(const kgrids& g, int delta, int reach, int gather_most, unsigned long long max_f,
                                  unsigned long long max_count, tile_scale* out)
{
    const double phi3 = delta == IBM_DELTA_BSPLINE3 ? 0.3 : 0.126;     // (2/3)^3, (1/2)^3 with room for rounding
    const double res3 = fmax(g.res3[0], fmax(g.res3[1], g.res3[2]));
    const double one = __longlong_as_double((long long) max_f) * res3 * phi3;
    const double bound = (double) reach * (double) max_count * one;
    tile_scale s;
    s.poisoned = !(bound <= 1.7976931348623157e308);
    int e2 = 0;
    if (!s.poisoned && bound > 0) frexp(bound, &e2);
    s.inv_q = ldexp(1.0, 62 - e2);
    s.q = s.poisoned ? __longlong_as_double(0x7ff8000000000000ll) : ldexp(1.0, e2 - 62);
    s.gather = gather_most > 0 && max_count <= (unsigned long long) gather_most;
    *out = s;
}

__global__ void tile_scale_kernel(kgrids g, int delta, int reach, int gather_most, const bin_stats* __restrict__ stats,
                                  tile_scale* __restrict__ out)
{
    const int tid = threadIdx.x;      // one wavefront
    unsigned long long fb = wave_max(stats->max_abs_f[tid]);
    unsigned long long cm = wave_max(stats->max_count[tid]);
    if (tid == 0) make_scale(g, delta, reach, gather_most, fb, cm, out);
}

__global__ void __launch_bounds__(256) tile_max_kernel(const int* __restrict__ count, int keys, bin_stats* __restrict__ stats)
{
    unsigned long long m = 0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < keys; i += gridDim.x * 256)
        m = (unsigned long long) count[i] > m ? (unsigned long long) count[i] : m;
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0 && m) atomicMax(&stats->max_count[blockIdx.x % STAT_SLOTS], m);
}

// Bin starts (keys + 1), the largest bin and the quantum, in one workgroup:
// up to SCAN_MAX bins this is one launch instead of the two of a device-wide
// scan and the quantum's own.  Wave w takes the w-th sixteenth of the bins, in
// steps of 256: once for its sum, once for the starts (67,584 bins of the C4
// channel: 8 us; 32 with a thread on 66 consecutive bins).
constexpr int SCAN_THREADS = 1024, SCAN_WAVES = SCAN_THREADS / 64, SCAN_MAX = 1 << 17;

__device__ inline int4 load_counts(const int* __restrict__ count, int i, int end)
{
    if (i + 4 <= end) return *(const int4*) (count + i);
    return make_int4(i < end ? count[i] : 0, i + 1 < end ? count[i + 1] : 0, i + 2 < end ? count[i + 2] : 0, 0);
}

__global__ void __launch_bounds__(SCAN_THREADS)
tile_scan_kernel(kgrids g, int delta, int reach, int gather_most, const int* __restrict__ count, int keys, const bin_stats* __restrict__ stats,
                 int* __restrict__ start, tile_scale* __restrict__ out)
{
    __shared__ int wave_sum[SCAN_WAVES];
    __shared__ int wave_top[SCAN_WAVES];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per = (keys + SCAN_WAVES * 256 - 1) / (SCAN_WAVES * 256) * 256;
    const int i0 = wave * per + lane * 4, end = min(wave * per + per, keys);
    int sum = 0, top = 0;
#pragma unroll 4
    for (int i = i0; i < end; i += 256) {
        const int4 v = load_counts(count, i, end);
        sum += v.x + v.y + v.z + v.w;
        top = max(max(top, max(v.x, v.y)), max(v.z, v.w));
    }
    for (int off = 32; off > 0; off >>= 1) {
        sum += __shfl_xor(sum, off, 64);
        top = max(top, __shfl_xor(top, off, 64));
    }
    if (lane == 0) {
        wave_sum[wave] = sum;
        wave_top[wave] = top;
    }
    __syncthreads();
    int run = 0;
    for (int w = 0; w < wave; ++w) run += wave_sum[w];
    int4 next = load_counts(count, i0, end);
    for (int step = 0; step < per; step += 256) {
        const int i = i0 + step;
        const int4 v = next;
        next = load_counts(count, i + 256, end);
        const int own = v.x + v.y + v.z + v.w;
        int incl = own;
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(incl, off, 64);
            if (lane >= off) incl += y;
        }
        const int s0 = run + incl - own, s1 = s0 + v.x, s2 = s1 + v.y, s3 = s2 + v.z;
        if (i + 4 <= end) {
            *(int4*) (start + i) = make_int4(s0, s1, s2, s3);
        } else {
            if (i < end) start[i] = s0;
            if (i + 1 < end) start[i + 1] = s1;
            if (i + 2 < end) start[i + 2] = s2;
        }
        run += __shfl(incl, 63, 64);
    }
    if (wave == SCAN_WAVES - 1 && lane == 0) start[keys] = run;          // the last wave ends at the total
    if (wave == 0) {
        const unsigned long long fb = wave_max(stats->max_abs_f[lane]);
        const unsigned long long cm = wave_max((unsigned long long) (lane < SCAN_WAVES ? wave_top[lane] : 0));
        if (lane == 0) make_scale(g, delta, reach, gather_most, fb, cm, out);
    }
}

// Adds the integer nearest to w v (in quanta) to a tile entry.  FAST: the
// integer is below 2^51, so one fused multiply-add with 1.5 * 2^52 leaves it
// in the low bits (the constant's own bits are the high word's).  Otherwise
// the same in two parts: the multiple of 2^12 nearest to w v, taken with a
// constant whose mantissa bits, shifted up by 12, cancel those that the exact
// remainder's constant brings along (the mantissa field holds 2^52 - 0x4338
// 2^36 plus an integer below 2^50 in magnitude: no carry leaves it).  A plain
// conversion to a 64-bit integer is about ten instructions, several of them
// at a fraction of the rate.
template <bool FAST>
__device__ inline void add_value(unsigned long long* at, double w, double v)
{
    constexpr double ROUND = 0x1.8p52;                        // bits 0x4338 << 48
    if (FAST) {
        const double t = fma(w, v, ROUND);
        atomicAdd(at, (unsigned long long) __double_as_longlong(t) - 0x4338000000000000ull);
    } else {
        constexpr double C = ((double) (1ull << 52) + (double) ((1ull << 52) - (0x4338ull << 36))) * 0x1p12;
        const double t = fma(w, v, C);
        const double rest = fma(w, v, C - t) + ROUND;
        atomicAdd(at, ((unsigned long long) __double_as_longlong(t) << 12) + (unsigned long long) __double_as_longlong(rest));
    }
}

// The 64 values of one component of a marker, plane by plane.
template <bool FAST>
__device__ inline void add_stencil(unsigned long long* t, const double (&wx)[4], const double (&wy)[4],
                                   const double (&wz)[4], double fq)
{
    double z0 = wz[0], z1 = wz[1], z2 = wz[2], z3 = wz[3];
#pragma unroll 1
    for (int sz = 0; sz < 4; ++sz) {
#pragma unroll
        for (int sy = 0; sy < 4; ++sy) {
            const double wyz = z0 * (wy[sy] * fq);
#pragma unroll
            for (int sx = 0; sx < 4; ++sx) add_value<FAST>(t + sx + TT * sy, wx[sx], wyz);
        }
        t += TT * TT;
        z0 = z1;
        z1 = z2;
        z2 = z3;
    }
}

// One workgroup per brick and component: its markers' stencils into the
// component's tile in LDS, which is then stored (flags[brick] = 0 for a brick
// without markers, whose tiles are not written).  Bound by the LDS atomics
// (52 % of the cycles at C4, two thirds of them bank conflicts), the vector
// ALU that feeds them (47 %) and the loads' latency.  Lanes of one atomic
// that hit one address serialise, so each chunk of markers is first listed by
// its rank among the markers of one stencil origin: 64 consecutive entries
// then nearly always have 64 different origins.  What a marker needs (its
// three offsets inside a cell, its scaled force) waits in LDS meanwhile, so
// that memory is read once, in the bin order.  One component per block gives
// three times the blocks where bricks are few, and four blocks per CU where
// they are many; the short code (the planes of the stencil in a loop) matters
// where a block runs once, since most of 35 us on a 32^3 grid with 2562
// markers went into fetching straight-line code for three components and both
// conversions.  Measured in us, C4 channel with 2.39 M markers / that sphere /
// 64 boxes of 32^3 with 0.26 M markers: three components per block in bin order
// 398 / 28 / 188; listed by rank and origin, per component 458 / 20 / 133; by
// rank alone 384 to 399 / 17.5 / 94.
constexpr int CHUNK_MARKERS = 512, ORIGINS = 9 * 9 * 9, THREAD_MARKERS = CHUNK_MARKERS / TILE_THREADS;

__global__ void __launch_bounds__(TILE_THREADS, 4)
tile_spread_kernel(marker_sets sets, kgrids g, bin_desc bd, tile_desc td, int delta, const int* __restrict__ start,
                   const int* __restrict__ perm, const tile_scale* __restrict__ scale,
                   unsigned long long* __restrict__ tiles, int* __restrict__ flags, int blocks, int chunk, int may_gather)
{
    __shared__ __attribute__((aligned(16))) unsigned long long acc[TILE_PTS];
    __shared__ __attribute__((aligned(16))) double2 offsets01[CHUNK_MARKERS], offset2_force[CHUNK_MARKERS];
    __shared__ int count[ORIGINS];
    __shared__ int level[64];                                // markers of rank r (63: and beyond)
    __shared__ unsigned short order[CHUNK_MARKERS];
    __shared__ unsigned short corner[CHUNK_MARKERS];         // tile index of a marker's stencil origin
    // XCD x takes the x-th eighth: a brick's components share its L2's markers
    const int block = (int) (blockIdx.x & 7) * chunk + (int) (blockIdx.x >> 3);
    if ((int) (blockIdx.x >> 3) >= chunk || block >= blocks) return;
    const int brick = block / 3, c = block - 3 * brick;
    const int s0 = start[(size_t) brick * SUB];
    const int s1 = start[(size_t) (brick + 1) * SUB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (may_gather && scale->gather) return;
    if (s1 == s0) {
        if (tid == 0 && c == 0) flags[brick] = 0;
        return;                                      // whole block
    }
    for (int i = tid; i < TILE_PTS; i += TILE_THREADS) acc[i] = 0ull;
    const int r = brick % td.bricks;
    const int b0 = r % td.nbr[0];
    const int b1 = (r / td.nbr[0]) % td.nbr[1];
    const int b2 = r / (td.nbr[0] * td.nbr[1]);
    const int bq[3] = {b0 * TB, b1 * TB, b2 * TB};
    // The quantum's inverse is a power of two: applied to the scaled force, it
    // scales every product exactly as it would scale the finished one (a
    // product that ends at 1/2 or more has no subnormal factor on the way).
    // Not to res3 alone: for forces near 1e-288 the inverse is near the end of
    // the range and the product would be infinite.
    const double inv_q = scale->inv_q, res3 = g.res3[c];
    // values of a force below this (in quanta) stay below 2^51: see make_scale
    const double fast_below = 0x1p51 / (delta == IBM_DELTA_BSPLINE3 ? 0.3 : 0.126);
#pragma unroll 1
    for (int c0 = s0; c0 < s1; c0 += CHUNK_MARKERS) {
        const int n = min(s1 - c0, CHUNK_MARKERS);
        double p[THREAD_MARKERS][3], f[THREAD_MARKERS];
#pragma unroll
        for (int k = 0; k < THREAD_MARKERS; ++k) {
            const int m = perm[c0 + min(tid + k * TILE_THREADS, n - 1)];
            load_marker(sets, m, p[k]);
            f[k] = load_force(sets, m, c);
        }
        for (int i = tid; i < ORIGINS; i += TILE_THREADS) count[i] = 0;
        if (tid < 64) level[tid] = 0;
        __syncthreads();
        int at[THREAD_MARKERS];                              // rank and place among its markers, or -1
#pragma unroll
        for (int k = 0; k < THREAD_MARKERS; ++k) {
            const int i = tid + k * TILE_THREADS;
            int o[3];
            double d[3];
            bool on = i < n;
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const kaxis& a = g.a[c][j];
                const int q = kstencil(g.a[bd.fc[j]][j], p[k][j]).base + bd.fs[j];
                int qb = q - bd.qmin[j];
                qb = qb < 0 ? 0 : (qb >= bd.nb[j] ? bd.nb[j] - 1 : qb);
                const stencil_axis st = kstencil(a, p[k][j]);
                // base_c - q, unwrapped across a periodic seam
                int s = st.base - q;
                if (!a.solid) {
                    if (s > 2) s -= a.cells;
                    else if (s < -3) s += a.cells;
                }
                o[j] = qb - bq[j] + s - bd.lo[j];
                d[j] = st.d;
                // A marker outside a walled axis's range (clamped by the
                // index policy) can have an origin off the tile: its points
                // lie outside the grid, which drops them, so it is skipped.
                on = on && o[j] >= 0 && o[j] <= TT - 4;
            }
            at[k] = -1;
            if (on) {
                const int rank = min(atomicAdd(&count[o[0] + 9 * (o[1] + 9 * o[2])], 1), 63);
                at[k] = rank << 16 | atomicAdd(&level[rank], 1);
                offsets01[i] = make_double2(d[0], d[1]);
                offset2_force[i] = make_double2(d[2], f[k] * res3 * inv_q);
                corner[i] = (unsigned short) (o[0] + TT * (o[1] + TT * o[2]));
            }
        }
        __syncthreads();
        // list of the markers by rank
        const int members = level[lane];
        int incl = members;
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(incl, off, 64);
            if (lane >= off) incl += y;
        }
        const int listed = __shfl(incl, 63, 64);
#pragma unroll
        for (int k = 0; k < THREAD_MARKERS; ++k) {
            const int to = __shfl(incl - members, at[k] >= 0 ? at[k] >> 16 : 0, 64) + (at[k] & 0xffff);
            if (at[k] >= 0) order[to] = (unsigned short) (tid + k * TILE_THREADS);
        }
        __syncthreads();
        for (int i0 = wave * 64; i0 < listed; i0 += TILE_THREADS) {
            if (i0 + lane >= listed) continue;
            const int i = order[i0 + lane];
            const double2 d01 = offsets01[i], d2f = offset2_force[i];
            double wx[4], wy[4], wz[4];
            delta4(delta, d01.x, wx);
            delta4(delta, d01.y, wy);
            delta4(delta, d2f.x, wz);
            unsigned long long* t = acc + corner[i];
            if (fabs(d2f.y) < fast_below) add_stencil<true>(t, wx, wy, wz, d2f.y);
            else add_stencil<false>(t, wx, wy, wz, d2f.y);
        }
        __syncthreads();
    }
    ulonglong2* dst = (ulonglong2*) (tiles + ((size_t) brick * 3 + c) * TILE_PTS);
    for (int i = tid; i < TILE_PTS / 2; i += TILE_THREADS) dst[i] = ((const ulonglong2*) acc)[i];
    if (tid == 0 && c == 0) flags[brick] = 1;
}

// Every grid point of every box and component: the sum of the tile entries
// that cover it, times the quantum.  HBM-bound in its traffic (3.4 entries a
// point), latency-bound if the entries are loaded one after another: all of a
// thread's flags are loaded first, then all its entries, absent ones from the
// first entry's address.  A thread takes one point of one component
// (consecutive threads consecutive points, whatever the row length: a block
// per grid row left 96 of its 128 threads idle on boxes of 32 cells), XCD x
// the x-th eighth of them, so that rows that share tiles share an L2.
//
// Per axis a point is covered by the tiles b with 8 b + t = v, t < 12, v its
// distance from the first tile's start: on walled axes one v, on periodic
// ones every v = rel + k cells up to the last tile's end.  Walls and whole
// bricks (WHOLE) leave at most two tiles: b = v / 8 and, for the first four
// points of a brick, the one before it (the last one before the first).
// Other periodic axes have up to six: those grids loop over them.
constexpr int MERGE_THREADS = 256;

struct cover {
    int rel, cells, nbr, solid;
};

template <typename F>
__device__ inline void visit(const cover& a, F&& f)
{
    for (int v = a.rel; v < (a.nbr - 1) * TB + TT; v += a.cells) {
        if (v >= 0) {
            const int b = v / TB, t = v - b * TB;
            if (b < a.nbr) f(b, t);
            if (b > 0 && b - 1 < a.nbr && t + TB < TT) f(b - 1, t + TB);
        }
        if (a.solid) break;
    }
}

template <bool WHOLE>
__global__ void __launch_bounds__(MERGE_THREADS)
tile_merge_kernel(kgrids g, bin_desc bd, tile_desc td, int box0, unsigned chunk,
                  const unsigned long long* __restrict__ tiles, const int* __restrict__ flags,
                  const tile_scale* __restrict__ scale, double* __restrict__ fe0, double* __restrict__ fe1,
                  double* __restrict__ fe2, int may_gather)
{
    if (may_gather && scale->gather) return;
    const int bz = blockIdx.y / 3, c = blockIdx.y - 3 * bz, box = box0 + bz;
    const unsigned block = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
    const unsigned at = block * MERGE_THREADS + threadIdx.x;
    if (at >= (unsigned) td.box_points[c]) return;
    const unsigned n0 = g.points[c][0], n1 = g.points[c][1];
    const unsigned row = at / n0, z = row / n1;
    const int pp[3] = {(int) (at - row * n0), (int) (row - z * n1), (int) z};
    cover cv[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const kaxis& a = g.a[c][j];
        int rel = pp[j] - (bd.qmin[j] + bd.lo[j] - 1);       // from the first tile point of brick 0
        if (!a.solid) rel = rel < 0 ? rel + a.cells : (rel >= a.cells ? rel - a.cells : rel);
        cv[j] = cover{rel, a.cells, td.nbr[j], a.solid};
    }
    long long sum = 0;
    if (WHOLE) {
        int b[3][2], t[3][2];
        bool ok[3][2];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int v = cv[j].rel < 0 ? 0 : cv[j].rel, b0 = v / TB, t0 = v - b0 * TB;
            b[j][0] = b0;
            t[j][0] = t0;
            ok[j][0] = cv[j].rel >= 0 && b0 < cv[j].nbr;
            b[j][1] = b0 > 0 ? b0 - 1 : (cv[j].solid ? 0 : cv[j].nbr - 1);
            t[j][1] = t0 + TB;
            ok[j][1] = cv[j].rel >= 0 && t0 + TB < TT && b[j][1] < cv[j].nbr && (b0 > 0 || !cv[j].solid);
        }
        unsigned brick[8];
        bool has[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int x = k & 1, y = k >> 1 & 1, w = k >> 2;
            has[k] = ok[0][x] && ok[1][y] && ok[2][w];
            brick[k] = ((unsigned) (box * td.nbr[2] + b[2][w]) * td.nbr[1] + b[1][y]) * td.nbr[0] + b[0][x];
            brick[k] = has[k] ? brick[k] : 0u;
        }
        int fl[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) fl[k] = flags[brick[k]];
        unsigned long long e[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int x = k & 1, y = k >> 1 & 1, w = k >> 2;
            has[k] = has[k] && fl[k];
            const size_t i = ((size_t) brick[k] * 3 + c) * TILE_PTS + t[0][x] + TT * (t[1][y] + TT * t[2][w]);
            e[k] = tiles[has[k] ? i : (size_t) 0];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) sum += has[k] ? (long long) e[k] : 0ll;
    } else {
        visit(cv[2], [&](int b2, int t2) {
            visit(cv[1], [&](int b1, int t1) {
                const unsigned brick_row = ((unsigned) (box * td.nbr[2] + b2) * td.nbr[1] + b1) * td.nbr[0];
                const unsigned tile_row = TT * (t1 + TT * t2);
                visit(cv[0], [&](int b0, int t0) {
                    const unsigned brick = brick_row + b0;
                    if (flags[brick]) sum += (long long) tiles[((size_t) brick * 3 + c) * TILE_PTS + tile_row + t0];
                });
            });
        });
    }
    double* fe = c == 0 ? fe0 : (c == 1 ? fe1 : fe2);
    fe[(size_t) box * td.box_points[c] + at] = (double) sum * scale->q;
}

// Few scattered markers on a large grid: every brick would hold a marker or
// some, and its tiles of 12^3 points be cleared, stored and merged for them.
// Instead one workgroup per 8 x 8 x 8 points visits the markers of the bins
// that reach them, adds what falls on them to an LDS tile and writes the
// points: the same integers, so the same bits, without tiles in memory.  A
// marker is visited by eight workgroups, so bins must hold few (GATHER_MOST,
// looked at on the device when the bins are counted: clumped markers keep the
// tiles; the launches of the path not taken leave at once), and the kernel is
// launched where the grid has GATHER_BRICKS bricks (fewer are bound by their
// launches) and on average at most GATHER_PER_BRICK markers a brick.  Bound by
// the latency of its chain of loads and by writing the grids.  Scattered
// markers, whole spread, us, brick kernel / tiles / this: 20,000 on
// 128 x 256 x 128 244 / 376 / 193, 200,000 on 256^3 1031 / 1489 / 737, 20,000
// on 100^3 (9 a brick) 121 / 155 / 97, 2000 on 64^3 50 / 55 / 44; above the
// limit 20,000 on 64^3 (39 a brick) 63 / 57 / 101, 200,000 on 128^3 (49)
// 278 / 224 / 383.
constexpr int GATHER_MOST = 24, GATHER_BRICKS = 100, GATHER_PER_BRICK = 12;
constexpr int GATHER_AXIS = 8, GATHER_THREADS = 256, GATHER_CHUNK = 128, GATHER_ENTRIES = 3 * GATHER_CHUNK;

__global__ void __launch_bounds__(GATHER_THREADS, 4)
tile_gather_kernel(marker_sets sets, kgrids g, bin_desc bd, tile_desc td, int delta, const int* __restrict__ start,
                   const int* __restrict__ perm, const tile_scale* __restrict__ scale, double* __restrict__ fe0,
                   double* __restrict__ fe1, double* __restrict__ fe2, int bricks_x, int bricks_y, int nbricks, int chunk)
{
    __shared__ unsigned long long acc[3][BRICK_PTS];
    __shared__ __attribute__((aligned(16))) double2 offsets01[GATHER_ENTRIES], offset2_force[GATHER_ENTRIES];
    __shared__ int bases[3][GATHER_ENTRIES];
    __shared__ unsigned char component[GATHER_ENTRIES];
    __shared__ int axis_bin[3][GATHER_AXIS], axis_bins[3], entries;
    __shared__ int first[GATHER_THREADS], before[GATHER_THREADS + 1], wave_sum[GATHER_THREADS / 64];
    // XCD x takes the x-th eighth: neighbouring bricks share its L2's markers
    const int bid = (int) (blockIdx.x & 7) * chunk + (int) (blockIdx.x >> 3);
    if ((int) (blockIdx.x >> 3) >= chunk || bid >= nbricks || !scale->gather) return;       // whole block
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int P0x = bid % bricks_x * BX, P0y = bid / bricks_x % bricks_y * BY, P0z = bid / (bricks_x * bricks_y) * BZ;
    // per axis, the bins of four cells that hold any of the (up to 12) cells
    // whose stencils reach the brick, each once
    if (tid < 3) {
        const int j = tid;
        const region_dim r = brick_region<BX>(bd, g.a[bd.fc[j]][j], j, j == 0 ? P0x : (j == 1 ? P0y : P0z));
        int n = 0;
        for (int i = 0; i < r.count;) {
            int q = r.first + i;
            if (r.wrap) q = q < 0 ? q + r.wrap : (q >= r.wrap ? q - r.wrap : q);
            const int end = r.wrap && q + 4 - (q & 3) > r.wrap ? r.wrap : q + 4 - (q & 3);
            if (n == 0 || q >> 2 != axis_bin[j][0]) axis_bin[j][n++] = q >> 2;
            i += end - q;
        }
        axis_bins[j] = n;
    }
    __syncthreads();
    const int nx = axis_bins[0], ny = axis_bins[1], bins = nx * ny * axis_bins[2];     // at most 6 per axis
    // the bins' markers, flattened
    int own = 0;
    if (tid < bins) {
        const int cx = axis_bin[0][tid % nx], cy = axis_bin[1][tid / nx % ny], cz = axis_bin[2][tid / (nx * ny)];
        const int key = (((cz >> 1) * td.nbr[1] + (cy >> 1)) * td.nbr[0] + (cx >> 1)) * SUB + ((cx & 1) | (cy & 1) << 1 | (cz & 1) << 2);
        first[tid] = start[key];
        own = start[key + 1] - first[tid];
    }
    int incl = own;
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(incl, off, 64);
        if (lane >= off) incl += y;
    }
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    for (int w = 0; w < wave; ++w) incl += wave_sum[w];
    before[tid + 1] = incl;
    if (tid == 0) before[0] = 0;
    int T = 0;
    for (int w = 0; w < GATHER_THREADS / 64; ++w) T += wave_sum[w];
    if (T > 0) {
        for (int i = tid; i < 3 * BRICK_PTS; i += GATHER_THREADS) (&acc[0][0])[i] = 0ull;
        const double inv_q = scale->inv_q;
        const double fast_below = 0x1p51 / (delta == IBM_DELTA_BSPLINE3 ? 0.3 : 0.126);
        for (int c0 = 0; c0 < T; c0 += GATHER_CHUNK) {
            if (tid == 0) entries = 0;
            __syncthreads();
            // a thread per marker: its components whose stencils meet the brick
            const int at = c0 + tid;
            if (tid < GATHER_CHUNK && at < T) {
                int lo = 0, hi = GATHER_THREADS;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (before[mid] <= at) lo = mid; else hi = mid;
                }
                const int m = perm[first[lo] + (at - before[lo])];
                double p[3], f[3];
                load_marker(sets, m, p);
                load_force(sets, m, f);
                int q[3], qb[3];
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    q[j] = kstencil(g.a[bd.fc[j]][j], p[j]).base + bd.fs[j];
                    const int b = q[j] - bd.qmin[j];
                    qb[j] = b < 0 ? 0 : (b >= bd.nb[j] ? bd.nb[j] - 1 : b);
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    double d[3];
                    int base[3];
                    bool hit = true;
#pragma unroll
                    for (int j = 0; j < 3; ++j) {
                        const kaxis& a = g.a[c][j];
                        const stencil_axis st = kstencil(a, p[j]);
                        d[j] = st.d;
                        base[j] = st.base;
                        int s = st.base - q[j];
                        if (!a.solid) {
                            if (s > 2) s -= a.cells;
                            else if (s < -3) s += a.cells;
                        }
                        const int o = (qb[j] & (TB - 1)) + s - bd.lo[j];
                        bool any = false;
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            any = any || brick_offset<BX>(a, st.base, k, j == 0 ? P0x : (j == 1 ? P0y : P0z)) >= 0;
                        hit = hit && any && o >= 0 && o <= TT - 4;           // o: as in tile_spread_kernel
                    }
                    if (hit) {
                        const int e = atomicAdd(&entries, 1);
                        offsets01[e] = make_double2(d[0], d[1]);
                        offset2_force[e] = make_double2(d[2], f[c] * g.res3[c] * inv_q);
#pragma unroll
                        for (int j = 0; j < 3; ++j) bases[j][e] = base[j];
                        component[e] = (unsigned char) c;
                    }
                }
            }
            __syncthreads();
            // four lanes per component of a marker, one plane of its stencil each
            for (int i = tid; i < 4 * entries; i += GATHER_THREADS) {
                const int e = i >> 2, sz = i & 3, c = component[e];
                const int oz = brick_offset<BZ>(g.a[c][2], bases[2][e], sz, P0z);
                if (oz < 0) continue;
                int ox[4], oy[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    ox[k] = brick_offset<BX>(g.a[c][0], bases[0][e], k, P0x);
                    oy[k] = brick_offset<BY>(g.a[c][1], bases[1][e], k, P0y);
                }
                const double2 d01 = offsets01[e], d2f = offset2_force[e];
                double wx[4], wy[4], wz[4];
                delta4(delta, d01.x, wx);
                delta4(delta, d01.y, wy);
                delta4(delta, d2f.x, wz);
                const double z = sz == 0 ? wz[0] : (sz == 1 ? wz[1] : (sz == 2 ? wz[2] : wz[3]));
                const bool fast = fabs(d2f.y) < fast_below;
#pragma unroll
                for (int sy = 0; sy < 4; ++sy) {
                    if (oy[sy] < 0) continue;
                    const double wyz = z * (wy[sy] * d2f.y);
                    unsigned long long* row = &acc[c][BX * (oy[sy] + BY * oz)];
#pragma unroll
                    for (int sx = 0; sx < 4; ++sx) {
                        if (ox[sx] < 0) continue;
                        if (fast) add_value<true>(row + ox[sx], wx[sx], wyz);
                        else add_value<false>(row + ox[sx], wx[sx], wyz);
                    }
                }
            }
            __syncthreads();
        }
    }
    const double q = scale->q;
    for (int i = tid; i < 3 * BRICK_PTS; i += GATHER_THREADS) {
        const int c = i / BRICK_PTS, k = i - c * BRICK_PTS;
        const int X = P0x + k % BX, Y = P0y + k / BX % BY, Z = P0z + k / (BX * BY);
        const int* pt = g.points[c];
        double* fe = c == 0 ? fe0 : (c == 1 ? fe1 : fe2);
        if (X < pt[0] && Y < pt[1] && Z < pt[2])
            fe[(size_t) X + (size_t) pt[0] * ((size_t) Y + (size_t) pt[1] * Z)] = T > 0 ? (double) (long long) acc[c][k] * q : 0.0 * q;
    }
}

// Two doubles at 8-byte alignment (global loads need only dword alignment).
typedef double d2u8 __attribute__((ext_vector_type(2), aligned(8)));

// Grid index of stencil point p for interpolation (ib/interpolate.h:16-22):
// axis_interp_index() for p in [-2, points + 1], its modulo by comparisons.
__device__ inline int kinterp_index(const kaxis& a, int p)
{
    if (!a.solid) {
        p = p < 0 ? p + a.cells : p;
        p = p >= a.cells ? p - a.cells : p;
        p = p >= a.cells ? p - a.cells : p;
    }
    return p < 0 ? 0 : (p >= a.points ? a.points - 1 : p);
}

// Interpolation (ib/interpolate.h:49-76), two lanes per marker and component,
// each with two points of the 16 stencil rows; with BOXES, box b's grids lie
// at b * box_points.
// Bound by the vector L1's handling of scattered rows and, at half its issue
// rate, the vector ALU: lanes of a pair share a row's line, so a load has 32
// rows to look up instead of 64, and all 16 rows of a component are on their
// way at once (no branch between them, the weights computed meanwhile), which
// also meets each line of neighbouring markers while it is in the cache (16.5
// to 7.6 million L2 requests at the size below).  One lane for a marker's
// three components, rows one after another / one lane per marker and
// component / this, us: 2210 markers 19 / 7.6 / 6.8, 46,400 on 100^3
// 25 / 19 / 15, 684,000 in the 128 x 256 x 128 channel 138 / 156 / 135, 64
// boxes of 32^3 with 264,000 69 / 41 / 42.
constexpr int INTERP_THREADS = 256, INTERP_MARKERS = INTERP_THREADS / 2;

template <bool BOXES>
__global__ void __launch_bounds__(INTERP_THREADS, 4)
interp_kernel(marker_sets sets, kgrids g, int delta, const int* __restrict__ box_off, int nboxes, int blocks, int chunk,
              const double* __restrict__ u0, const double* __restrict__ u1, const double* __restrict__ u2)
{
    // XCD x takes the x-th eighth: neighbouring markers share its L2's rows
    const int nth = (int) (blockIdx.x >> 3), c = nth / chunk, block = (int) (blockIdx.x & 7) * chunk + nth % chunk;
    if (block >= blocks) return;
    const int half = threadIdx.x & 1, own = block * INTERP_MARKERS + (int) (threadIdx.x >> 1);
    const int m = min(own, sets.total - 1);
    double p[3];
    load_marker(sets, m, p);
    const kaxis* a = g.a[c];
    double d[3];
    int at[3][4];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const stencil_axis st = kstencil(a[j], p[j]);
        d[j] = st.d;
#pragma unroll
        for (int o = 0; o < 4; ++o) at[j][o] = kinterp_index(a[j], st.base + o - 1);
    }
    const int x0 = half ? at[0][2] : at[0][0], x1 = half ? at[0][3] : at[0][1];
    const int px = g.points[c][0], py = g.points[c][1];
    const double* u = c == 0 ? u0 : (c == 1 ? u1 : u2);    // global loads (an indexed array would be flat)
    if (BOXES) u += (size_t) box_of(box_off, nboxes, m) * px * py * g.points[c][2];
    d2u8 v[4][4];
    // the two points are adjacent except across a periodic seam or a clamped
    // wall: then one 16-byte load per row instead of two
    if (x1 == x0 + 1) {
        u += x0;
#pragma unroll
        for (int z = 0; z < 4; ++z)
#pragma unroll
            for (int y = 0; y < 4; ++y) v[z][y] = *(const d2u8*) (u + px * (at[1][y] + py * at[2][z]));
    } else {
#pragma unroll
        for (int z = 0; z < 4; ++z)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                const double* row = u + px * (at[1][y] + py * at[2][z]);
                v[z][y] = d2u8{row[x0], row[x1]};
            }
    }
    __builtin_amdgcn_sched_barrier(0);
    // the weights while the rows are on their way
    double w[3][4], sum = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) delta4(delta, d[j], w[j]);
    const double w0 = half ? w[0][2] : w[0][0], w1 = half ? w[0][3] : w[0][1];
#pragma unroll
    for (int z = 0; z < 4; ++z) {
        double sy = 0.0;
#pragma unroll
        for (int y = 0; y < 4; ++y) sy = fma(w[1][y], fma(w1, v[z][y].y, w0 * v[z][y].x), sy);
        sum = fma(w[2][z], sy, sum);
    }
    sum += __shfl_xor(sum, 1, 64);
    const int k = set_of(sets, m);
    if (own < sets.total && half == 0)
        sets.out[k][(size_t) c * (sets.offset[k + 1] - sets.offset[k]) + (m - sets.offset[k])] = sum;
}

} // namespace

// Allocates the fixed workspace of `device` (made current by the caller) once
// per device; ibm_create calls it.  (As a __device__ array the loader fills it
// from the host, 73 ms in the first ibm_create of a process instead of 1.)
ibm_status static_scratch_init(ibm_ctx* ctx, int device)
{
    if (device < 0 || device >= STATIC_MAX_DEVICES)
        return fail(ctx, IBM_ERR_ARG, "device %d beyond the fixed-workspace table", device);
    std::lock_guard<std::mutex> lock(static_scratch_mutex);
    if (!static_scratch_ptr[device]) IBM_HIP(ctx, hipMalloc(&static_scratch_ptr[device], STATIC_SCRATCH_BYTES));
    return IBM_OK;
}

// Checked inputs of a spread and its bins.
ibm_status spread_setup(ibm_ctx* ctx, const ibm_grid* grids, int delta, double* const* fe, kgrids* kg, bin_desc* bd)
{
    IBM_TRY(make_kgrids(ctx, grids, kg));
    IBM_TRY(check_delta(ctx, delta));
    if (!fe || !fe[0] || !fe[1] || !fe[2]) return fail(ctx, IBM_ERR_ARG, "null output grid");
    for (int c = 0; c < 3; ++c)
        for (int j = 0; j < 3; ++j)
            if (!kg->a[c][j].solid && kg->a[c][j].cells < 4)
                return fail(ctx, IBM_ERR_BAD_GRID, "periodic dimension needs at least 4 cells for a 4-point stencil");
    *bd = make_bins(grids);
    if (bd->nbins <= 0) return fail(ctx, IBM_ERR_SIZE, "too many grid bins");
    for (int j = 0; j < 3; ++j)
        if (bd->hi[j] - bd->lo[j] > 1 || bd->hi[j] < bd->lo[j])
            return fail(ctx, IBM_ERR_BAD_GRID, "component grids are not a staggering of one cell grid");
    return IBM_OK;
}

// Component j alone differs along axis j.
bool mac_shaped(const kgrids& kg)
{
    for (int c = 0; c < 3; ++c)
        for (int j = 0; j < 3; ++j)
            if (kg.sel[c][j] != (c == j ? 1 : 0) || kg.cand[1][j] != j || kg.cand[0][j] == j) return false;
    return true;
}

// Every periodic axis long enough for the brick kernel's division-free wrap.
bool wide_axes(const kgrids& kg)
{
    for (int c = 0; c < 3; ++c)
        for (int j = 0; j < 3; ++j)
            if (!kg.a[c][j].solid && kg.a[c][j].cells < MIN_FAST_CELLS) return false;
    return true;
}

// The general wrap of the brick kernel packs point indices into 10 bits; the
// entry points refuse such grids whichever path takes the call.
ibm_status narrow_axes_limit(ibm_ctx* ctx, const kgrids& kg)
{
    if (wide_axes(kg)) return IBM_OK;
    for (int c = 0; c < 3; ++c)
        for (int j = 0; j < 3; ++j)
            if (kg.a[c][j].points > 1022)
                return fail(ctx, IBM_ERR_SIZE, "small periodic axes with more than 1022 points on another axis");
    return IBM_OK;
}

bool whole_bricks(const kgrids& kg)
{
    for (int c = 0; c < 3; ++c)
        for (int j = 0; j < 3; ++j)
            if (!kg.a[c][j].solid && kg.a[c][j].cells % TB != 0) return false;
    return true;
}

// The brick kernel's spread.
ibm_status spread_bricks(ibm_ctx* ctx, const kgrids& kg, const bin_desc& bd, int delta, const marker_sets& sets,
                         double* const* fe, unsigned char* fixed_workspace)
{
    bin_work w;
    if (fixed_workspace) IBM_TRY(static_bin_work(ctx, fixed_workspace, bd.nbins, &w));
    else IBM_TRY(ctx_bin_work(ctx, sets.total, bd.nbins, &w));
    IBM_TRY(bin_markers(ctx, sets, kg, bd, 1, w, fixed_workspace == nullptr));
    int maxp[3] = {0, 0, 0};
    for (int c = 0; c < 3; ++c)
        for (int j = 0; j < 3; ++j) maxp[j] = kg.points[c][j] > maxp[j] ? kg.points[c][j] : maxp[j];
    int bx = (maxp[0] + BX - 1) / BX, by = (maxp[1] + BY - 1) / BY, bz = (maxp[2] + BZ - 1) / BZ;
    long long nbricks = (long long) bx * by * bz;
    if (nbricks > 0x7fffffff) return fail(ctx, IBM_ERR_SIZE, "grid too large");
    int xcd_chunk = (nbricks % 8 == 0) ? (int) (nbricks / 8) : 0;
    const bool mac = mac_shaped(kg), fast = wide_axes(kg);
    double grid_points = 0;
    for (int c = 0; c < 3; ++c) grid_points += (double) kg.points[c][0] * kg.points[c][1] * kg.points[c][2];
    // positions + forces read once, three grids written once
    prof_scope prof(ctx, fixed_workspace ? nullptr : "spread_brick", 48.0 * sets.total + 8.0 * grid_points);
    auto launch = [&](auto kernel) {
        kernel<<<(int) nbricks, SPREAD_THREADS, 0, ctx->stream>>>(
            kg, bd, delta, sets.total, w.start, w.sorted, w.stats, fe[0], fe[1], fe[2], bx, by, (int) nbricks,
            xcd_chunk);
    };
    if (mac && fast) launch(spread_brick_kernel<true, true>);
    else if (mac) launch(spread_brick_kernel<true, false>);
    else if (fast) launch(spread_brick_kernel<false, true>);
    else launch(spread_brick_kernel<false, false>);
    IBM_LAUNCH_CHECK(ctx);
    return IBM_OK;
}

// Bricks of one box, and whether every brick's tiles of nboxes boxes may be
// held (16 GiB) and numbered.
long long bricks_of(const bin_desc& bd)
{
    long long n = 1;
    for (int j = 0; j < 3; ++j) n *= (bd.nb[j] + TB - 1) / TB;
    return n;
}

constexpr long long TILE_MAX_BYTES = 1ll << 34;
bool tiles_fit(const bin_desc& bd, int nboxes)
{
    const long long bricks = bricks_of(bd);
    return bricks <= TILE_MAX_BYTES / (long long) TILE_BYTES / nboxes && bricks * nboxes * SUB <= INT_MAX - 1;
}

// Spread of the markers of nboxes boxes (box b: markers [off[b], off[b+1])
// of the sets' concatenation, off on the device) into nboxes consecutive
// copies of each component grid, by bricks and tiles.
ibm_status spread_tiles(ibm_ctx* ctx, const kgrids& kg, const bin_desc& bd, int delta, const marker_sets& sets, int nboxes,
                        const int* box_off, double* const* fe, unsigned char* fixed_workspace)
{
    tile_desc td{};
    int reach = 1;
    for (int j = 0; j < 3; ++j) {
        const kaxis& a = kg.a[bd.fc[j]][j];
        td.nbr[j] = (bd.nb[j] + TB - 1) / TB;
        reach *= !a.solid && a.cells % 4 != 0 ? 3 : 2;
    }
    td.bricks = (int) bricks_of(bd);
    td.nboxes = nboxes;
    td.keys = td.bricks * nboxes * SUB;
    double grid_points = 0;
    unsigned most = 0;
    for (int c = 0; c < 3; ++c) {
        td.box_points[c] = kg.points[c][0] * kg.points[c][1] * kg.points[c][2];
        most = std::max(most, (unsigned) td.box_points[c]);
        grid_points += (double) td.box_points[c] * nboxes;
    }
    const size_t nbricks = (size_t) td.bricks * nboxes, total = (size_t) sets.total;
    const size_t key_words = sizeof(int) * ((size_t) td.keys + 1);
    int *count, *start, *key, *rank, *perm, *flags;
    bin_stats* stats;
    tile_scale* sc;
    unsigned long long* tiles;
    void *p, *scan_tmp = nullptr;
    size_t scan_bytes = 0;
    if (fixed_workspace) {
        size_t off = 0;
        auto take = [&](size_t bytes) { unsigned char* q = fixed_workspace + off; off += align256(bytes); return q; };
        count = (int*) take(key_words);
        start = (int*) take(key_words);
        key = (int*) take(sizeof(int) * total);
        rank = (int*) take(sizeof(int) * total);
        perm = (int*) take(sizeof(int) * total);
        stats = (bin_stats*) take(STATIC_STATS_BYTES);
        sc = (tile_scale*) take(sizeof(tile_scale));
        flags = (int*) take(sizeof(int) * nbricks);
        tiles = (unsigned long long*) take(TILE_BYTES * nbricks);
    } else {
        IBM_TRY(scratch(ctx, SLOT_BIN_COUNT, key_words, &p)); count = (int*) p;
        IBM_TRY(scratch(ctx, SLOT_BIN_START, key_words, &p)); start = (int*) p;
        IBM_TRY(scratch(ctx, SLOT_KEY, sizeof(int) * total, &p)); key = (int*) p;
        IBM_TRY(scratch(ctx, SLOT_RANK, sizeof(int) * total, &p)); rank = (int*) p;
        IBM_TRY(scratch(ctx, SLOT_PERM, sizeof(int) * total, &p)); perm = (int*) p;
        IBM_TRY(scratch(ctx, SLOT_FLAGS, sizeof(bin_stats), &p)); stats = (bin_stats*) p;
        IBM_TRY(scratch(ctx, SLOT_TILES, TILE_BYTES * nbricks, &p)); tiles = (unsigned long long*) p;
        IBM_TRY(scratch(ctx, SLOT_TILE_FLAGS, align256(sizeof(tile_scale)) + sizeof(int) * nbricks, &p));
        sc = (tile_scale*) p;
        flags = (int*) ((unsigned char*) p + align256(sizeof(tile_scale)));
        if (td.keys > SCAN_MAX) {
            IBM_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, count, start, td.keys + 1, ctx->stream));
            IBM_TRY(scratch(ctx, SLOT_SCAN_TMP, scan_bytes, &scan_tmp));
        }
    }
    const bool timed = fixed_workspace == nullptr;
    const bool may_gather = nboxes == 1 && td.bricks >= GATHER_BRICKS && (long long) sets.total <= (long long) GATHER_PER_BRICK * td.bricks;
    const int gather_most = may_gather ? GATHER_MOST : 0;
    {
        prof_scope prof(ctx, timed ? "bin" : nullptr);
        tile_clear_kernel<<<blocks_for((long long) td.keys + 1, 256), 256, 0, ctx->stream>>>(count, td.keys, stats);
        IBM_LAUNCH_CHECK(ctx);
        if (total > 0) {
            tile_count_kernel<<<blocks_for(sets.total, 256 * COUNT_ITEMS), 256, 0, ctx->stream>>>(
                sets, kg, bd, td, box_off, key, rank, count, stats);
            IBM_LAUNCH_CHECK(ctx);
        }
        if (td.keys <= SCAN_MAX) {
            tile_scan_kernel<<<1, SCAN_THREADS, 0, ctx->stream>>>(kg, delta, reach, gather_most, count, td.keys, stats, start, sc);
            IBM_LAUNCH_CHECK(ctx);
        } else {
            IBM_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(scan_tmp, scan_bytes, count, start, td.keys + 1, ctx->stream));
            tile_max_kernel<<<std::min(blocks_for(td.keys, 256), 1024), 256, 0, ctx->stream>>>(count, td.keys, stats);
            IBM_LAUNCH_CHECK(ctx);
            tile_scale_kernel<<<1, 64, 0, ctx->stream>>>(kg, delta, reach, gather_most, stats, sc);
            IBM_LAUNCH_CHECK(ctx);
        }
        if (total > 0) {
            tile_place_kernel<<<blocks_for(sets.total, 256), 256, 0, ctx->stream>>>(sets.total, key, rank, start, perm);
            IBM_LAUNCH_CHECK(ctx);
        }
    }
    {
        prof_scope prof(ctx, timed ? "spread_tile" : nullptr, 48.0 * sets.total);
        const int blocks = (int) nbricks * 3, chunk = (blocks + 7) / 8;
        tile_spread_kernel<<<(unsigned) (8 * chunk), TILE_THREADS, 0, ctx->stream>>>(sets, kg, bd, td, delta, start, perm, sc,
                                                                                     tiles, flags, blocks, chunk, may_gather);
        IBM_LAUNCH_CHECK(ctx);
    }
    {
        prof_scope prof(ctx, timed ? "spread_merge" : nullptr, 8.0 * grid_points);
        if (may_gather) {
            int bricks[3] = {0, 0, 0};
            for (int c = 0; c < 3; ++c)
                for (int j = 0; j < 3; ++j) bricks[j] = std::max(bricks[j], (kg.points[c][j] + BX - 1) / BX);
            const int n = bricks[0] * bricks[1] * bricks[2], chunk = (n + 7) / 8;
            tile_gather_kernel<<<(unsigned) (8 * chunk), GATHER_THREADS, 0, ctx->stream>>>(
                sets, kg, bd, td, delta, start, perm, sc, fe[0], fe[1], fe[2], bricks[0], bricks[1], n, chunk);
            IBM_LAUNCH_CHECK(ctx);
        }
        bool whole = true;
        for (int c = 0; c < 3; ++c)
            for (int j = 0; j < 3; ++j) whole = whole && (kg.a[c][j].solid || kg.a[c][j].cells % TB == 0);
        const unsigned blocks = (most + MERGE_THREADS - 1) / MERGE_THREADS, chunk = (blocks + 7) / 8;
        constexpr int BOXES_PER_LAUNCH = 65535 / 3;
        for (int b0 = 0; most > 0 && b0 < nboxes; b0 += BOXES_PER_LAUNCH) {
            const int nb = std::min(BOXES_PER_LAUNCH, nboxes - b0);
            const dim3 grid(8 * chunk, (unsigned) (3 * nb));
            if (whole)
                tile_merge_kernel<true><<<grid, MERGE_THREADS, 0, ctx->stream>>>(kg, bd, td, b0, chunk, tiles, flags, sc,
                                                                                 fe[0], fe[1], fe[2], may_gather);
            else
                tile_merge_kernel<false><<<grid, MERGE_THREADS, 0, ctx->stream>>>(kg, bd, td, b0, chunk, tiles, flags, sc,
                                                                                  fe[0], fe[1], fe[2], may_gather);
            IBM_LAUNCH_CHECK(ctx);
        }
    }
    return IBM_OK;
}

// Whether the tiles of one box's bricks can be held in the context's scratch
// (up to 16 GiB, kept like every scratch buffer): false, with the failure
// cleared, where the device's memory is taken.
bool tiles_held(ibm_ctx* ctx, const bin_desc& bd)
{
    void* p;
    const std::string before = ctx->error;
    if (scratch(ctx, SLOT_TILES, TILE_BYTES * (size_t) bricks_of(bd), &p) == IBM_OK) return true;
    (void) hipGetLastError();
    ctx->error = before;
    return false;
}

// The public spread.  ibm_spread_sets and ibm_spread_sets_noalloc give the
// same bits, so the path depends on the markers and grids alone: tiles where
// a brick's tiles for the whole grid fit the fixed workspace, or where the
// input is beyond what the fixed workspace takes at all; else (grids of few
// bins and many mostly empty bricks, or no memory left for the tiles, where
// the results are as accurate but not the same bits) the brick kernel.
// Measured (us, brick kernel / tiles, binning included): C4 channel with
// 2.39 M markers 1802 / 580, 100^3 periodic with 176,000 markers 268 / 120,
// one sphere of 2562 markers on 32^3 89 / 41.
ibm_status spread_sets(ibm_ctx* ctx, const ibm_grid* grids, int delta, const marker_sets& sets,
                       double* const* fe, unsigned char* fixed_workspace = nullptr)
{
    kgrids kg;
    bin_desc bd;
    IBM_TRY(spread_setup(ctx, grids, delta, fe, &kg, &bd));
    if (fixed_workspace) IBM_TRY(static_limits(ctx, sets.total, bd.nbins));
    IBM_TRY(narrow_axes_limit(ctx, kg));
    const bool beyond = (size_t) sets.total > STATIC_MAX_MARKERS || (size_t) bd.nbins > STATIC_MAX_BINS;
    const bool by_tiles = bricks_of(bd) <= (long long) STATIC_MAX_BRICKS || (beyond && tiles_fit(bd, 1));
    if (by_tiles && (fixed_workspace || tiles_held(ctx, bd)))
        return spread_tiles(ctx, kg, bd, delta, sets, 1, nullptr, fe, fixed_workspace);
    return spread_bricks(ctx, kg, bd, delta, sets, fe, fixed_workspace);
}

// The timestep's spread of several marker sets: by tiles wherever they fit.
ibm_status spread_sets_step(ibm_ctx* ctx, const ibm_grid* grids, int delta, int nsets, const int* n,
                            const double* const* x, const double* const* f, double* const* fe)
{
    marker_sets s;
    IBM_TRY(make_sets(ctx, nsets, n, x, f, nullptr, &s));
    kgrids kg;
    bin_desc bd;
    IBM_TRY(spread_setup(ctx, grids, delta, fe, &kg, &bd));
    const bool fit = tiles_fit(bd, 1) && tiles_held(ctx, bd);
    if (!fit || !whole_bricks(kg)) IBM_TRY(narrow_axes_limit(ctx, kg));
    if (fit) return spread_tiles(ctx, kg, bd, delta, s, 1, nullptr, fe, nullptr);
    return spread_bricks(ctx, kg, bd, delta, s, fe, nullptr);
}

// ibm_spread_boxes' grids: every periodic axis a multiple of the brick edge.
ibm_status spread_boxes(ibm_ctx* ctx, const ibm_grid* grids, int delta, const marker_sets& sets, int nboxes,
                        const int* box_off, double* const* fe)
{
    kgrids kg;
    bin_desc bd;
    IBM_TRY(make_kgrids(ctx, grids, &kg));
    if (!whole_bricks(kg))
        return fail(ctx, IBM_ERR_BAD_GRID, "batched spreading needs periodic axes of a multiple of %d cells", TB);
    IBM_TRY(spread_setup(ctx, grids, delta, fe, &kg, &bd));
    if (bricks_of(bd) * nboxes > (INT_MAX - 1) / SUB)
        return fail(ctx, IBM_ERR_SIZE, "too many boxes or bins for one batched spread");
    return spread_tiles(ctx, kg, bd, delta, sets, nboxes, box_off, fe, nullptr);
}

ibm_status interp_sets(ibm_ctx* ctx, const ibm_grid* grids, int delta, const marker_sets& sets,
                       const double* const* ue)
{
    kgrids kg;
    IBM_TRY(make_kgrids(ctx, grids, &kg));
    IBM_TRY(check_delta(ctx, delta));
    if (!ue || !ue[0] || !ue[1] || !ue[2]) return fail(ctx, IBM_ERR_ARG, "null input grid");
    if (sets.total == 0) return IBM_OK;
    prof_scope prof(ctx, "interp");
    const int blocks = blocks_for(sets.total, INTERP_MARKERS), chunk = (blocks + 7) / 8;
    interp_kernel<false><<<24 * chunk, INTERP_THREADS, 0, ctx->stream>>>(sets, kg, delta, nullptr, 1, blocks, chunk, ue[0],
                                                                        ue[1], ue[2]);
    IBM_LAUNCH_CHECK(ctx);
    return IBM_OK;
}


// The box offsets (host, nboxes + 1) in the context's scratch.  Up to
// OFFSET_LAUNCHES parts travel as kernel arguments, which the launch copies:
// the caller's array is free at once, without a copy and a synchronisation of
// the stream (64 boxes: a spread, an interpolation and a check of the solution
// 326 us with the two copies, 298 without).
constexpr int OFFSET_PART = 512, OFFSET_LAUNCHES = 4;
struct offset_part {
    int v[OFFSET_PART];
};

__global__ void __launch_bounds__(OFFSET_PART) offsets_kernel(offset_part p, int n, int* __restrict__ out)
{
    if ((int) threadIdx.x < n) out[threadIdx.x] = p.v[threadIdx.x];
}

ibm_status upload_box_offsets(ibm_ctx* ctx, int nboxes, const int* offsets, int total, const int** dev)
{
    if (!offsets) return fail(ctx, IBM_ERR_ARG, "null box offsets");
    if (offsets[0] != 0 || offsets[nboxes] != total)
        return fail(ctx, IBM_ERR_SIZE, "box offsets must run from 0 to the marker count %d", total);
    for (int b = 0; b < nboxes; ++b)
        if (offsets[b + 1] < offsets[b]) return fail(ctx, IBM_ERR_SIZE, "box offsets must not decrease");
    void* p;
    IBM_TRY(scratch(ctx, SLOT_BOX_OFF, sizeof(int) * (size_t) (nboxes + 1), &p));
    *dev = (const int*) p;
    if (nboxes < OFFSET_PART * OFFSET_LAUNCHES) {
        for (int at = 0; at <= nboxes; at += OFFSET_PART) {
            offset_part part;
            const int n = std::min(OFFSET_PART, nboxes + 1 - at);
            std::copy_n(offsets + at, n, part.v);
            offsets_kernel<<<1, OFFSET_PART, 0, ctx->stream>>>(part, n, (int*) p + at);
            IBM_LAUNCH_CHECK(ctx);
        }
        return IBM_OK;
    }
    IBM_HIP(ctx, hipMemcpyAsync(p, offsets, sizeof(int) * (size_t) (nboxes + 1), hipMemcpyHostToDevice, ctx->stream));
    // the host array may be reused once the call returns
    IBM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return IBM_OK;
}

ibm_status interp_boxes(ibm_ctx* ctx, const ibm_grid* grids, int delta, const marker_sets& sets, int nboxes,
                        const int* box_off, const double* const* ue)
{
    kgrids kg;
    IBM_TRY(make_kgrids(ctx, grids, &kg));
    IBM_TRY(check_delta(ctx, delta));
    if (!ue || !ue[0] || !ue[1] || !ue[2]) return fail(ctx, IBM_ERR_ARG, "null input grid");
    if (sets.total == 0) return IBM_OK;
    prof_scope prof(ctx, "interp");
    const int blocks = blocks_for(sets.total, INTERP_MARKERS), chunk = (blocks + 7) / 8;
    interp_kernel<true><<<24 * chunk, INTERP_THREADS, 0, ctx->stream>>>(sets, kg, delta, box_off, nboxes, blocks, chunk, ue[0],
                                                                       ue[1], ue[2]);
    IBM_LAUNCH_CHECK(ctx);
    return IBM_OK;
}
} // namespace ibm

extern "C" {

ibm_status ibm_spread_sets(ibm_ctx* ctx, const ibm_grid* grids, ibm_delta delta, int nsets,
                           const int* n, const double* const* x, const double* const* f,
                           double* const* fe)
{
    if (!ctx) return IBM_ERR_ARG;
    if (nsets > 0 && !f) return ibm::fail(ctx, IBM_ERR_ARG, "null force arrays");
    ibm::marker_sets s;
    IBM_TRY(ibm::make_sets(ctx, nsets, n, x, f, nullptr, &s));
    return ibm::spread_sets(ctx, grids, (int) delta, s, fe);
}

ibm_status ibm_spread_sets_noalloc(ibm_ctx* ctx, const ibm_grid* grids, ibm_delta delta, int nsets,
                                   const int* n, const double* const* x, const double* const* f,
                                   double* const* fe)
{
    if (!ctx) return IBM_ERR_ARG;
    if (nsets > 0 && !f) return ibm::fail(ctx, IBM_ERR_ARG, "null force arrays");
    if (ctx->device < 0 || ctx->device >= ibm::STATIC_MAX_DEVICES || !ibm::static_scratch_ptr[ctx->device])
        return ibm::fail(ctx, IBM_ERR_HIP, "the fixed spreading workspace of device %d is not set up", ctx->device);
    ibm::marker_sets s;
    IBM_TRY(ibm::make_sets(ctx, nsets, n, x, f, nullptr, &s));
    return ibm::spread_sets(ctx, grids, (int) delta, s, fe, (unsigned char*) ibm::static_scratch_ptr[ctx->device]);
}

ibm_status ibm_spread(ibm_ctx* ctx, const ibm_grid* grids, ibm_delta delta, int n,
                      const double* x, const double* f, double* const* fe)
{
    return ibm_spread_sets(ctx, grids, delta, 1, &n, &x, &f, fe);
}

ibm_status ibm_interpolate_sets(ibm_ctx* ctx, const ibm_grid* grids, ibm_delta delta, int nsets,
                                const int* n, const double* const* x, const double* const* ue,
                                double* const* ul)
{
    if (!ctx) return IBM_ERR_ARG;
    if (nsets > 0 && !ul) return ibm::fail(ctx, IBM_ERR_ARG, "null output arrays");
    ibm::marker_sets s;
    IBM_TRY(ibm::make_sets(ctx, nsets, n, x, nullptr, ul, &s));
    return ibm::interp_sets(ctx, grids, (int) delta, s, ue);
}

ibm_status ibm_interpolate(ibm_ctx* ctx, const ibm_grid* grids, ibm_delta delta, int n,
                           const double* x, const double* const* ue, double* ul)
{
    return ibm_interpolate_sets(ctx, grids, delta, 1, &n, &x, ue, &ul);
}

ibm_status ibm_spread_boxes(ibm_ctx* ctx, const ibm_grid* grids, ibm_delta delta, int nboxes, const int* offsets,
                            const double* x, const double* f, double* const* fe)
{
    if (!ctx) return IBM_ERR_ARG;
    if (nboxes < 1) return ibm::fail(ctx, IBM_ERR_ARG, "at least one box");
    if (!offsets) return ibm::fail(ctx, IBM_ERR_ARG, "null box offsets");
    int n = offsets[nboxes];
    ibm::marker_sets s;
    IBM_TRY(ibm::make_sets(ctx, 1, &n, &x, &f, nullptr, &s));
    const int* dev_off = nullptr;
    IBM_TRY(ibm::upload_box_offsets(ctx, nboxes, offsets, s.total, &dev_off));
    return ibm::spread_boxes(ctx, grids, (int) delta, s, nboxes, dev_off, fe);
}

ibm_status ibm_interpolate_boxes(ibm_ctx* ctx, const ibm_grid* grids, ibm_delta delta, int nboxes, const int* offsets,
                                 const double* x, const double* const* ue, double* ul)
{
    if (!ctx) return IBM_ERR_ARG;
    if (nboxes < 1) return ibm::fail(ctx, IBM_ERR_ARG, "at least one box");
    if (!offsets) return ibm::fail(ctx, IBM_ERR_ARG, "null box offsets");
    int n = offsets[nboxes];
    ibm::marker_sets s;
    IBM_TRY(ibm::make_sets(ctx, 1, &n, &x, nullptr, &ul, &s));
    const int* dev_off = nullptr;
    IBM_TRY(ibm::upload_box_offsets(ctx, nboxes, offsets, s.total, &dev_off));
    return ibm::interp_boxes(ctx, grids, (int) delta, s, nboxes, dev_off, ue);
}

} // extern "C"
