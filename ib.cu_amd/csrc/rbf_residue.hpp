// FP64 products of an RBF evaluation on the INT8 matrix cores
// (rbf_residue.hip): Y = E^T X through residues modulo fifteen coprime
// moduli, and the columns that need FP64 products instead.  rbf.hip decides
// which batch entries take this path, owns the buffers and multiplies those
// columns.
#pragma once
#include "context.hpp"

namespace ibm {

constexpr int RES_MODULI = 15;
constexpr int RES_BM = 256, RES_BN = 128;      // block tile: samples x columns
// Bytes of residues a tile leaves for the recombination, and the most tiles
// one launch leaves (half a GiB).
constexpr size_t RES_TILE_BYTES = (size_t) RES_BM * RES_BN * RES_MODULI;
constexpr int RES_LAUNCH_TILES = 1024;

inline int res_ceil(int a, int b) { return (a + b - 1) / b; }
// 64-element contraction chunks of K.
inline int res_chunks(int K) { return res_ceil(K, 64); }
// Whether an operator of contraction length K may take the path: INT32 sums
// of K products of residues of at most 128 stay below 2^31.
inline bool res_fits(int K) { return K <= 131000; }
inline size_t res_plane_bytes(int rows, int block, int K)
{
    return (size_t) res_ceil(rows, block) * block * (size_t) res_chunks(K) * 64;
}
// One plane per modulus and one of seven-bit magnitudes.
constexpr int RES_PLANES = RES_MODULI + 1;
inline size_t res_align(size_t b) { return (b + 255) & ~size_t(255); }

// An M x K operator: its planes, and per row the scale of its integers, the
// exponent of its largest element and the least magnitude product that the
// integers are good for (see operator_scale_kernel).
inline size_t res_operator_bytes(int M, int K) { return RES_PLANES * res_plane_bytes(M, RES_BM, K) + 3 * sizeof(int) * (size_t) M; }

// Classes of a column.
enum { COLUMN_NARROW = 0, COLUMN_WIDE = 1, COLUMN_F64 = 2 };

// N packed columns of K elements: the planes; per column its integers' scale
// and its class; per 16 columns bit 0 if one has residues, bit 1 if one is
// wide; and the columns themselves, rows of `ld` doubles, zero past K (written
// where the class is not COLUMN_NARROW).
struct res_packed {
    unsigned char* planes;
    int *scale, *kind, *live;
    double* rows;
    size_t ld, bytes;
};
inline res_packed res_columns_at(unsigned char* base, int N, int K)
{
    res_packed p;
    const size_t n = (size_t) N, planes = RES_PLANES * res_plane_bytes(N, RES_BN, K), ints = res_align(sizeof(int) * n);
    p.planes = base;
    p.scale = (int*) (base + planes);
    p.kind = (int*) (base + planes + ints);
    p.live = (int*) (base + planes + 2 * ints);
    const size_t head = planes + 2 * ints + res_align(sizeof(int) * (size_t) (res_ceil(N, RES_BN) * (RES_BN / 16)));
    p.rows = (double*) (base + head);
    p.ld = (size_t) res_chunks(K) * 64;
    p.bytes = head + sizeof(double) * n * p.ld;
    return p;
}
inline size_t res_columns_bytes(int N, int K) { return res_columns_at(nullptr, N, K).bytes; }

// Rows [0, M) of E (element k of row m at E[k + lde m]) into `planes`;
// *flag (device, cleared by the caller) is set when a row cannot be
// represented (a non-finite element or row sum).
void res_pack_operator(hipStream_t s, const double* E, long lde, int M, int K, unsigned char* planes, int* flag);

struct res_columns {
    const double* X;           // N columns of K elements
    unsigned char* packed;     // res_columns_bytes
    int N, K;
};
constexpr int RES_MAX_COLUMNS = 2 * IBM_MAX_CELL_TYPES;
// Also clears `flags` (those of res_flags, or none).
void res_pack_columns(hipStream_t s, int count, const res_columns* c, int* flags, int nflags);

struct res_product {
    const unsigned char* E;    // operator planes
    const double* E64;         // its FP64 rows, zero past K, 64 res_chunks(K) apart
    unsigned char* X;          // packed columns
    double* Y;                 // M x N, column-major
    int M, N, K;
    const int* list;           // out: [0] the number of columns that need FP64 products, then their indices
};
// Every product, but for the columns in its list; `work` holds
// res_work_bytes: the tiles' residues, the lists and their flags (*n of them),
// which are cleared first unless the packing has done so.
size_t res_work_bytes(int count, const res_product* p);
int* res_flags(int count, const res_product* p, unsigned char* work, int* n);
ibm_status res_products(ibm_ctx* ctx, hipStream_t s, int count, res_product* p, unsigned char* work, bool cleared);

} // namespace ibm
