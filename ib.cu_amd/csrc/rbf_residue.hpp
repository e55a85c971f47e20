// FP64 products of an RBF evaluation on the INT8 matrix cores
// (rbf_residue.hip): Y = E^T X through residues modulo fifteen coprime
// moduli.  rbf.hip decides which batch entries take this path and owns the
// buffers.
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
// Residue planes of an M x K operator / of N columns, and one int of scale
// per row / column behind them.
inline size_t res_operator_bytes(int M, int K) { return RES_MODULI * res_plane_bytes(M, RES_BM, K) + sizeof(int) * (size_t) M; }
inline size_t res_columns_bytes(int N, int K)
{
    return RES_MODULI * res_plane_bytes(N, RES_BN, K) + (sizeof(int) * (size_t) N + 255) / 256 * 256;
}

// Rows [0, M) of E (element k of row m at E[k + lde m]) into `planes`;
// *flag (device, cleared by the caller) is set when a row cannot be
// represented (a non-finite element or row sum).
void res_pack_operator(hipStream_t s, const double* E, long lde, int M, int K, unsigned char* planes, int* flag);

struct res_columns {
    const double* X;           // N columns of K elements
    unsigned char* planes;     // res_columns_bytes
    int N, K;
};
constexpr int RES_MAX_COLUMNS = 2 * IBM_MAX_CELL_TYPES;
void res_pack_columns(hipStream_t s, int count, const res_columns* c);

struct res_product {
    const unsigned char* E;    // operator planes
    const unsigned char* X;    // column planes
    const double* E64;         // FP64 rows of the operator (stride ld64) and
    const double* X64;         // the columns: for columns that hold a NaN or an infinity
    double* Y;                 // M x N, column-major
    int M, N, K;
    long ld64;
};
// Every product; `work` holds res_work_bytes of their tiles.
size_t res_work_bytes(int count, const res_product* p);
ibm_status res_products(ibm_ctx* ctx, hipStream_t s, int count, const res_product* p, unsigned char* work);

} // namespace ibm
