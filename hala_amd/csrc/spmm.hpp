// spmm.hpp -- sparse matrix times several vectors, the four scalar types.
//
// A workgroup owns 256 rows, a thread a row.  The rows' entries are staged in
// LDS tile by tile (values, and the byte offset each column has in a vector:
// coalesced reads), and each thread walks its row in CSR order over up to G
// vectors at once: a matrix entry is read once per G vectors instead of once
// per vector, and a wavefront's gathers of one entry position go to
// neighbouring elements of the vectors wherever neighbouring rows have
// neighbouring columns.  A few workgroups of long rows, and rows that fill
// tiles by themselves, are walked in memory instead (walk_rows in gather.hpp).
#pragma once
#include "scalar.hpp"
#include "spmv.hpp"

namespace hala_amd {

template <class S>
struct spmm_tile {
    static constexpr int value = sizeof(S) == 16 ? 1024 : 2048;  // entries staged (16 to 20 KiB of values)
};

// acc[k] = op over the row's entries, k < G: acc + v * x_k (N), acc + (alpha * x_k) * v (TRANS).
// x_k(c) is at xb[k] + c * step bytes (TO: uint64_t where gather_wide() of the vector, else unsigned).  TI = short: columns as offsets from
// the block's first row.
// WALK: each thread reads its row's entries from memory itself (walk_rows), nothing is staged.
// Must be called by all 256 threads of the block; sv, so: spmm_tile entries of LDS each (WALK: unused).
template <class S, int G, class TI, bool TRANS, class TO, bool WALK>
__device__ __forceinline__ void csr_block_rowsums(int nrows, const int *__restrict__ pntr, const TI *__restrict__ indx,
                                                  const int *__restrict__ tmap, const S *__restrict__ vals,
                                                  const char *const (&xb)[G], TO step, S alpha, bool conjv,
                                                  bool conjx, S *sv, TO *so, S (&acc)[G]) {
    constexpr int TILE = spmm_tile<S>::value;
    const int r0 = blockIdx.x * SPMV_ROWS;
    const int cb = sizeof(TI) == 2 ? r0 : 0;
    const int row = r0 + threadIdx.x;
    const int bstart = pntr[r0], bend = pntr[min(r0 + SPMV_ROWS, nrows)];
    int rs = 0, re = 0;
    if (row < nrows) {
        rs = pntr[row];
        re = pntr[row + 1];
    }
    // one entry into the G sums
    auto add = [&](const S v, const TO o) {
        S x[G];
#pragma unroll
        for (int k = 0; k < G; k++) x[k] = *reinterpret_cast<const S *>(xb[k] + o);
#pragma unroll
        for (int k = 0; k < G; k++) {
            if (is_complex<S>::value && conjx) x[k] = cconj(x[k]);
            acc[k] = cadd(acc[k], TRANS ? cmul(cmul(alpha, x[k]), v) : cmul(v, x[k]));
        }
    };
    if constexpr (WALK) {
#pragma unroll 4
        for (int j = rs; j < re; j++) {
            S v = vals[TRANS ? tmap[j] : j];
            if (is_complex<S>::value && conjv) v = cconj(v);
            add(v, gather_offset<TO>(cb + (int)indx[j], step));
        }
        return;
    }
    for (int base = bstart; base < bend; base = tile_next(base, bend, TILE)) {
        const int cnt = min(TILE, bend - base);
#pragma unroll 4
        for (int e = threadIdx.x; e < cnt; e += SPMV_ROWS) {
            const int j = base + e;
            S v = vals[TRANS ? tmap[j] : j];
            if (is_complex<S>::value && conjv) v = cconj(v);
            sv[e] = v;
            so[e] = gather_offset<TO>(cb + (int)indx[j], step);
        }
        __syncthreads();
        const int a = max(rs, base) - base, b = min(re, base + cnt) - base;
#pragma unroll 2
        for (int j = a; j < b; j++) add(sv[j], so[j]);
        __syncthreads();
    }
}

// y_k = alpha op(A) x_k + beta y_k for k < ncols (beta zero: y not read), op(A)
// by trans ('N', 'T', 'C'); x_k(c) at x[k sg + c sc], y_k at y + k ldy, each row
// (transposed: column) summed in the order of the single product.
template <class S>
void spmm_columns(hala_csr A, char trans, S alpha, const S *vals, const S *x, int64_t sg, int64_t sc, bool conjx, S beta,
                  S *y, int64_t ldy, int ncols);

// C = alpha op(A) op(B) + beta C, column-major, with hala_spmm_*'s argument checks
// (sparse/hala_sparse_utils.hpp:127-167).  op(B) column i is B's column i ('N')
// or row i ('T', 'C': conjugated).
template <class S>
void spmm(hala_csr A, char transa, char transb, int b_rows, int b_cols, S alpha, const S *vals, const S *B, int ldb,
          S beta, S *C, int ldc);

}  // namespace hala_amd
