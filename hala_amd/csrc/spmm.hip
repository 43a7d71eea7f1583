// spmm.hip -- sparse matrix times dense matrix (see spmm.hpp) and the
// transposed product.
//
// Bound by the gathers out of the caches (the matrix comes once per group of G
// columns, the vectors once): 64^3 27-point FP64 times 16 vectors 121 us, one
// product per column 333 us; 701^2 5-point complex FP64 times 5 vectors 38 us,
// one product per column (a thread per row, no staging) 184 us.  Groups of 8:
// the row sums and the operands of two entries then fit 96 registers.  Few
// workgroups of long rows are not staged (walk_rows): 2000 rows of 45 random
// entries, complex FP64, 66 -> 10 us (19 us with a thread per row before).
#include <algorithm>
#include <type_traits>

#include "spmm.hpp"

namespace hala_amd {

namespace {

template <class S, int G, class TI, bool TRANS, class TO, bool WALK>
__global__ __launch_bounds__(256) void spmm_rows_kernel(int nrows, const int *__restrict__ pntr,
                                                        const TI *__restrict__ indx, const int *__restrict__ tmap,
                                                        const S *__restrict__ vals, const S *__restrict__ x, int64_t sg,
                                                        TO step, S alpha, S beta, int conjv, int conjx, S *y,
                                                        int64_t ldy, int nc) {
    __shared__ S sv[WALK ? 1 : spmm_tile<S>::value];
    __shared__ TO so[WALK ? 1 : spmm_tile<S>::value];
    const int row = blockIdx.x * SPMV_ROWS + threadIdx.x;
    const char *xb[G];  // columns past nc repeat the last one (its loads hit in the cache); nothing is stored for them
#pragma unroll
    for (int k = 0; k < G; k++) xb[k] = reinterpret_cast<const char *>(x + (int64_t)min(k, nc - 1) * sg);
    const bool bz = czero(beta);
    S acc[G];
#pragma unroll
    for (int k = 0; k < G; k++) {
        acc[k] = S{};
        if (TRANS && !bz && k < nc && row < nrows) acc[k] = cmul(beta, y[k * ldy + row]);
    }
    csr_block_rowsums<S, G, TI, TRANS, TO, WALK>(nrows, pntr, indx, tmap, vals, xb, step, alpha, conjv != 0, conjx != 0,
                                                 sv, so, acc);
    if (row >= nrows) return;
#pragma unroll
    for (int k = 0; k < G; k++) {
        if (k >= nc) break;
        S *o = y + k * ldy + row;
        if (TRANS) {
            *o = acc[k];
        } else if (is_complex<S>::value) {
            S v = cmul(alpha, acc[k]);
            if (!bz) v = cadd(v, cmul(beta, *o));
            *o = v;
        } else {
            *o = bz ? cadd(cmul(alpha, acc[k]), S{}) : cadd(cmul(alpha, acc[k]), cmul(beta, *o));
        }
    }
}

// One transposed product: the terms (alpha x_i) v of 256 output rows are formed
// in entry order (coalesced indices, many gathers in flight) into LDS, then each
// thread adds its row's terms in increasing source row, starting from beta y.
// (400009 x 320014 FP32 operator of 4.5 M entries: 158 us with a thread per
// output row walking its entries alone, a chain of two dependent gathers per
// entry, 64 us with this kernel; its values are gathered through tmap, which
// is what is left.)
template <class T>
__global__ __launch_bounds__(256) void spmv_t_rows_kernel(int nrows, const int *__restrict__ tpntr,
                                                          const int *__restrict__ trow, const int *__restrict__ tmap,
                                                          const T *__restrict__ vals, const T *__restrict__ x, T alpha,
                                                          T beta, T *__restrict__ y) {
    constexpr int TILE = spmv_tile<T>::value;
    __shared__ T prod[TILE];
    const int r0 = blockIdx.x * SPMV_ROWS, row = r0 + threadIdx.x;
    const int bstart = tpntr[r0], bend = tpntr[min(r0 + SPMV_ROWS, nrows)];
    int rs = 0, re = 0;
    T acc = T(0);
    if (row < nrows) {
        rs = tpntr[row];
        re = tpntr[row + 1];
        if (beta != T(0)) acc = beta * y[row];
    }
    for (int base = bstart; base < bend; base = tile_next(base, bend, TILE)) {
        const int cnt = min(TILE, bend - base);
        int e = threadIdx.x;
        for (; e + 3 * SPMV_ROWS < cnt; e += 4 * SPMV_ROWS) {
            int m[4], r[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                m[q] = tmap[base + e + q * SPMV_ROWS];
                r[q] = trow[base + e + q * SPMV_ROWS];
            }
            T v[4], w[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                v[q] = vals[m[q]];
                w[q] = x[r[q]];
            }
#pragma unroll
            for (int q = 0; q < 4; q++) prod[e + q * SPMV_ROWS] = (alpha * w[q]) * v[q];
        }
        for (; e < cnt; e += SPMV_ROWS) prod[e] = (alpha * x[trow[base + e]]) * vals[tmap[base + e]];
        __syncthreads();
        const int a = max(rs, base), b = min(re, base + cnt);
        for (int j = a; j < b; j++) acc = acc + prod[j - base];
        __syncthreads();
    }
    if (row < nrows) y[row] = acc;
}

template <class S, class TI, bool TRANS>
void launch_group(hala_ctx c, int g, int nrows, const int *pntr, const TI *indx, const int *tmap, const S *vals,
                  const S *x, int64_t sg, int64_t step, S alpha, S beta, int conjv, int conjx, S *y, int64_t ldy,
                  int nc, bool wide, bool walk) {
#define HALA_G(GG, TO, WALK)                                                                                    \
    spmm_rows_kernel<S, GG, TI, TRANS, TO, WALK><<<g, SPMV_ROWS, 0, c->stream>>>(nrows, pntr, indx, tmap, vals, x, sg, \
                                                                                 (TO)step, alpha, beta, conjv,   \
                                                                                 conjx, y, ldy, nc)
    auto group = [&](auto w) {
        constexpr bool WALK = decltype(w)::value;
        if (nc > 6) HALA_G(8, unsigned, WALK);
        else if (nc > 4) HALA_G(6, unsigned, WALK);
        else if (nc > 2) HALA_G(4, unsigned, WALK);
        else if (nc > 1) HALA_G(2, unsigned, WALK);
        else HALA_G(1, unsigned, WALK);
    };
    if (wide) HALA_G(1, uint64_t, false);
    else if (walk) group(std::true_type());
    else group(std::false_type());
#undef HALA_G
    HALA_CHECK_LAUNCH();
}

bool is_n(char t) { return t == 'N' || t == 'n'; }
bool is_c(char t) { return t == 'C' || t == 'c'; }

}  // namespace

template <class S>
void spmm_columns(hala_csr A, char trans, S alpha, const S *vals, const S *x, int64_t sg, int64_t sc, bool conjx, S beta,
                  S *y, int64_t ldy, int ncols) {
    hala_ctx c = A->ctx;
    const bool tr = !is_n(trans);
    const int nrows = tr ? A->ncols : A->nrows, ncin = tr ? A->nrows : A->ncols;
    if (tr) ensure_transpose(A);
    const int g = (nrows + SPMV_ROWS - 1) / SPMV_ROWS;
    const int conjv = is_c(trans) ? 1 : 0;
    const int64_t step = sc * (int64_t)sizeof(S);
    const bool wide = gather_wide(ncin, step);
    const bool walk = !wide && walk_rows(A->nnz, g, tr ? 0 : A->max_row, spmm_tile<S>::value, c->num_cus,
                                         walk_per_cu(sizeof(S), tr, ncols));
    c->path[PATH_PRODUCT] = walk ? 2 : 1;
    if (nrows == 0 || ncols == 0) return;
    const bool apart = A->spread && !tr && !walk && !is_complex<S>::value && sc == 1;
    const int gmax = wide ? 1 : apart ? gather_group(ncin * (int64_t)sizeof(S)) : 8;
    for (int c0 = 0; c0 < ncols; c0 += gmax) {
        const int nc = std::min(gmax, ncols - c0);
        const S *xc = x + c0 * sg;
        S *yc = y + c0 * ldy;
        if (tr)
            launch_group<S, int, true>(c, g, nrows, A->tp.tpntr.as<int>(), A->tp.trow.as<int>(), A->tp.tmap.as<int>(),
                                       vals, xc, sg, step, alpha, beta, conjv, conjx, yc, ldy, nc, wide, walk);
        else if (A->boff.p)
            launch_group<S, short, false>(c, g, nrows, A->pntr, A->boff.as<short>(), nullptr, vals, xc, sg, step, alpha,
                                          beta, 0, conjx, yc, ldy, nc, wide, walk);
        else
            launch_group<S, int, false>(c, g, nrows, A->pntr, A->indx, nullptr, vals, xc, sg, step, alpha, beta, 0,
                                        conjx, yc, ldy, nc, wide, walk);
    }
}

template <class T>
void spmv_trans(hala_csr A, T alpha, const T *vals, const T *x, T beta, T *y) {
    ensure_transpose(A);
    hala_ctx c = A->ctx;
    if (A->ncols == 0) return;
    // a few workgroups of rows of several tiles each: walked (2000 x 2000, 45 random entries per row in
    // FP64: 26 us staged, 23 us with a thread per row before there were tiles)
    const int blocks = (A->ncols + SPMV_ROWS - 1) / SPMV_ROWS;
    if (blocks <= c->num_cus && A->nnz > (int64_t)blocks * 4 * spmv_tile<T>::value) {
        spmm_columns<T>(A, 'T', alpha, vals, x, 0, 1, false, beta, y, 0, 1);
        return;
    }
    spmv_t_rows_kernel<T><<<(A->ncols + SPMV_ROWS - 1) / SPMV_ROWS, SPMV_ROWS, 0, c->stream>>>(
        A->ncols, A->tp.tpntr.as<int>(), A->tp.trow.as<int>(), A->tp.tmap.as<int>(), vals, x, alpha, beta, y);
    HALA_CHECK_LAUNCH();
}
template void spmv_trans<double>(hala_csr, double, const double *, const double *, double, double *);
template void spmv_trans<float>(hala_csr, float, const float *, const float *, float, float *);

template <class S>
void spmm(hala_csr A, char transa, char transb, int b_rows, int b_cols, S alpha, const S *vals, const S *B, int ldb,
          S beta, S *C, int ldc) {
    auto ok = [&](char t) { return is_n(t) || t == 'T' || t == 't' || is_c(t); };
    HALA_REQUIRE(A && ok(transa) && ok(transb), HALA_ERR_ARG, "spmm: trans must be N, T or C");
    HALA_REQUIRE(b_rows >= 0 && b_cols >= 0, HALA_ERR_ARG, "spmm: negative size");
    const int M = is_n(transa) ? A->nrows : A->ncols;  // rows of C
    const int K = is_n(transa) ? A->ncols : A->nrows;  // rows of op(B)
    const int N = is_n(transb) ? b_cols : b_rows;      // columns of C
    HALA_REQUIRE((is_n(transb) ? b_rows : b_cols) == K, HALA_ERR_ARG, "spmm: op(B) must have op(A)'s column count of rows");
    HALA_REQUIRE(ldb >= std::max(b_rows, 1) && ldc >= std::max(M, 1), HALA_ERR_ARG, "spmm: ldb or ldc below the minimum");
    HALA_REQUIRE(N == 0 || (B && C), HALA_ERR_ARG, "spmm: null pointer");
    HALA_REQUIRE(N == 0 || vals || A->nnz == 0, HALA_ERR_ARG, "spmm: null pointer");
    const bool bn = is_n(transb);
    // one column of a real product (its products are formed in entry order:
    // more gathers in flight), vectors too long for a group of them
    // (gather_group), and rows too long for a thread each (one wavefront per
    // row), run the single product's kernels
    const int64_t sg = bn ? ldb : 1, sc = bn ? 1 : ldb;
    if constexpr (!is_complex<S>::value) {
        const bool alone = bn && is_n(transa) && A->spread && gather_group(K * (int64_t)sizeof(S)) == 1;
        if ((bn && N == 1) || alone || (is_n(transa) && A->kernel == 1)) {
            hala_ctx c = A->ctx;
            c->path[PATH_PRODUCT] = 0;
            tmp_scope ts(c);
            dbuf &t = ts.get();
            if (!bn) t.reserve((size_t)std::max(K, 1) * sizeof(S));
            for (int i = 0; i < N; i++) {
                const S *x = B + (int64_t)i * sg;
                if (!bn) {
                    strided_copy(c, K, sizeof(S), x, ldb, t.p, 1);
                    x = t.as<S>();
                }
                S *y = C + (int64_t)i * ldc;
                if (is_n(transa)) spmv_axpby<S, S, S>(A, vals, x, alpha, beta, y, false);
                else spmv_trans<S>(A, alpha, vals, x, beta, y);
            }
            return;
        }
    }
    spmm_columns<S>(A, transa, alpha, vals, B, sg, sc, is_c(transb), beta, C, ldc, N);
}

#define HALA_SPMM(S)                                                                                             \
    template void spmm_columns<S>(hala_csr, char, S, const S *, const S *, int64_t, int64_t, bool, S, S *, int64_t, \
                                  int);                                                                          \
    template void spmm<S>(hala_csr, char, char, int, int, S, const S *, const S *, int, S, S *, int);
HALA_SPMM(double)
HALA_SPMM(float)
HALA_SPMM(cx<double>)
HALA_SPMM(cx<float>)
#undef HALA_SPMM

}  // namespace hala_amd

using namespace hala_amd;

extern "C" {

int hala_spmm_f64(hala_csr A, char transa, char transb, int b_rows, int b_cols, double alpha, const double *vals,
                  const double *B, int ldb, double beta, double *C, int ldc) {
    HALA_RANGE();
    return guard([&] {
        HALA_REQUIRE(A, HALA_ERR_ARG, "spmm: null matrix");
        set_device(A->ctx);
        spmm<double>(A, transa, transb, b_rows, b_cols, alpha, vals, B, ldb, beta, C, ldc);
    });
}

int hala_spmm_f32(hala_csr A, char transa, char transb, int b_rows, int b_cols, float alpha, const float *vals,
                  const float *B, int ldb, float beta, float *C, int ldc) {
    HALA_RANGE();
    return guard([&] {
        HALA_REQUIRE(A, HALA_ERR_ARG, "spmm: null matrix");
        set_device(A->ctx);
        spmm<float>(A, transa, transb, b_rows, b_cols, alpha, vals, B, ldb, beta, C, ldc);
    });
}

}  // extern "C"
