// tri.hip -- standalone sparse triangular matrix (gpu_triangular_matrix of
// gpu/hala_rocm_sparse_triangular.hpp:29-194) with the semantics of
// sparse_trsv_array (sparse/hala_sparse_utils.hpp:284-335): the CSR holds one
// triangle, the diagonal being the last ('L') or first ('U') entry of a row.
#include <climits>

#include "ilu.hpp"

namespace hala_amd {

// row's diagonal is the last (lower) / first (upper) entry and equals the row index
__global__ void tri_check(int n, int lower, const int *__restrict__ pntr, const int *__restrict__ indx,
                          int *__restrict__ diagpos, int *bad) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int s = pntr[i], e = pntr[i + 1];
    bool ok = e > s;
    int d = -1;
    if (ok) {
        d = lower ? e - 1 : s;
        ok = indx[d] == i;
        if (lower) ok = ok && (s == d || indx[s] < i);
        else ok = ok && (e - 1 == d || indx[e - 1] > i);
    }
    diagpos[i] = d < 0 ? s : d;
    if (!ok) atomicMin(bad, i);
}

__global__ void set_i32_tri(int *p, int v) { *p = v; }

__global__ void f32_to_f64(int64_t n, const float *__restrict__ a, double *__restrict__ b) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (double)a[i];
}

// n elements of E from src (stride ss elements) to dst (stride ds)
template <class E>
__global__ void strided_copy_k(int n, const E *__restrict__ src, int64_t ss, E *__restrict__ dst, int64_t ds) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[(int64_t)i * ds] = src[(int64_t)i * ss];
}

void strided_copy(hala_ctx c, int n, size_t esize, const void *src, int64_t ss, void *dst, int64_t ds) {
    const int g = (n + 255) / 256;
    if (esize == 4)
        strided_copy_k<int><<<g, 256, 0, c->stream>>>(n, (const int *)src, ss, (int *)dst, ds);
    else if (esize == 8)
        strided_copy_k<int2><<<g, 256, 0, c->stream>>>(n, (const int2 *)src, ss, (int2 *)dst, ds);
    else
        strided_copy_k<int4><<<g, 256, 0, c->stream>>>(n, (const int4 *)src, ss, (int4 *)dst, ds);
    HALA_CHECK_LAUNCH();
}

static bool is_n(char t) { return t == 'N' || t == 'n'; }

trsm_layout tri_trsm_layout(hala_tri T, char transb, int nrhs, const void *B, int ldb) {
    HALA_REQUIRE(T && (B || nrhs == 0) && nrhs >= 0, HALA_ERR_ARG, "hala_trsm: bad argument");
    HALA_REQUIRE(is_n(transb) || transb == 'T' || transb == 't' || transb == 'C' || transb == 'c', HALA_ERR_ARG,
                 "hala_trsm: transb must be N, T or C");
    const int n = T->n;
    const bool bn = is_n(transb);
    if (ldb < 0) ldb = bn ? n : nrhs;
    HALA_REQUIRE(ldb >= (bn ? n : nrhs) && ldb >= 1, HALA_ERR_ARG, "hala_trsm: ldb below the minimum");
    // column k of op(B): column k of the stored B, or its row k
    return bn ? trsm_layout{ldb, 1} : trsm_layout{1, ldb};
}

static bool trans_checked(char trans, const char *who) {
    const bool tr = !is_n(trans);
    HALA_REQUIRE(!tr || trans == 'T' || trans == 't' || trans == 'C' || trans == 'c', HALA_ERR_ARG,
                 std::string(who) + ": trans must be N, T or C");
    return tr;
}

// The call's values into the layout that its nrhs vectors run on (one FP64 solve, all three layouts packed ->
// one: 64^3 lower triangle 114 -> 78 us, 16^3 60 -> 34, 27-point 64^3 367 -> 336).
static void load_call(hala_tri T, tri_plan &p, const double *vals, int nrhs) {
    p.loaded64 = 0;
    load_values64(T->ctx, p, vals, tri_route(T->ctx, p, nrhs));
}
// (the plan's loader takes FP64 values; the widening and its narrowing back are exact)
static void load_call(hala_tri T, tri_plan &p, const float *vals, int nrhs) {
    hala_ctx c = T->ctx;
    tmp_scope ts(c);
    dbuf &w = ts.get();
    w.reserve((size_t)T->nnz * sizeof(double));
    f32_to_f64<<<(int)((T->nnz + 255) / 256), 256, 0, c->stream>>>(T->nnz, vals, w.as<double>());
    HALA_CHECK_LAUNCH();
    p.loaded32 = 0;
    load_values32(c, p, w.as<double>(), tri_route(c, p, nrhs));
    HALA_HIP(hipStreamSynchronize(c->stream));
}

}  // namespace hala_amd

using namespace hala_amd;

extern "C" {

int hala_tri_create(hala_ctx c, char uplo, char diag, int n, int64_t nnz, const int *pntr, const int *indx,
                    hala_tri *out) {
    HALA_RANGE();
    return guard([&] {
        HALA_REQUIRE(c && out, HALA_ERR_ARG, "hala_tri_create: null argument");
        *out = nullptr;
        bool lower = (uplo == 'L' || uplo == 'l');
        HALA_REQUIRE(lower || uplo == 'U' || uplo == 'u', HALA_ERR_ARG, "hala_tri_create: uplo must be L or U");
        bool unit = (diag == 'U' || diag == 'u');
        HALA_REQUIRE(unit || diag == 'N' || diag == 'n', HALA_ERR_ARG, "hala_tri_create: diag must be U or N");
        HALA_REQUIRE(n > 0 && nnz > 0 && nnz < INT_MAX && pntr && indx, HALA_ERR_ARG, "hala_tri_create: bad sizes");
        set_device(c);
        int bad = validate_pattern(c, n, n, nnz, pntr, indx, 1);
        HALA_REQUIRE(bad < 0, HALA_ERR_PATTERN, "hala_tri_create: invalid pattern at row " + std::to_string(bad));
        auto *T = new hala_tri_s();
        // the plans' buffers come from the context's cache (hala_tri_destroy synchronises before it returns
        // them): the grid layout's were four allocations and frees more, 30 us each
        alloc_scope as(c->cache.get());
        try {
            T->ctx = c;
            T->n = n;
            T->nnz = nnz;
            T->pntr = pntr;
            T->indx = indx;
            T->uplo = lower ? 'L' : 'U';
            T->diag = unit ? 'U' : 'N';
            dbuf dpos;
            dpos.reserve((size_t)n * sizeof(int));
            int *flag = reinterpret_cast<int *>(c->scal.as<double>() + S_DOT + 7);
            set_i32_tri<<<1, 1, 0, c->stream>>>(flag, INT_MAX);
            tri_check<<<(n + 255) / 256, 256, 0, c->stream>>>(n, lower ? 1 : 0, pntr, indx, dpos.as<int>(), flag);
            HALA_CHECK_LAUNCH();
            int b = fetch_i32(c, flag);
            HALA_REQUIRE(b == INT_MAX, HALA_ERR_PATTERN,
                         "hala_tri_create: row " + std::to_string(b) + " is not " +
                             (lower ? "lower triangular with the diagonal last" : "upper triangular with the diagonal first"));
            build_deps(c, T->N, n, lower ? DEP_ROW_BUT_LAST : DEP_ROW_BUT_FIRST, pntr, indx, dpos.as<int>(), nullptr,
                       unit, !lower);
            build_schedule(c, T->N, false);
            // transposed solve: L^T is upper (backward, source rows descending), U^T lower (forward, ascending)
            build_transpose(c, n, n, nnz, pntr, indx, T->tp);
            build_deps(c, T->T, n, lower ? DEP_T_UPPER : DEP_T_LOWER, pntr, indx, dpos.as<int>(), &T->tp, unit, lower);
            build_schedule(c, T->T, false);
            T->t_built = true;
        } catch (...) {
            delete T;
            throw;
        }
        *out = T;
    });
}

int hala_tri_destroy(hala_tri T) {
    HALA_RANGE();
    return guard([&] {
        if (!T) return;
        (void)hipSetDevice(T->ctx->device);
        (void)hipStreamSynchronize(T->ctx->stream);
        delete T;
    });
}

// x = op(T)^-1 (alpha b): sum of the off-diagonal terms first, then
// (alpha*b_i - s) [/ diag]; the transposed sums add the terms in the source-row
// order of the reference's column sweep.
int hala_trsv_f64(hala_tri T, char trans, double alpha, const double *vals, const double *b, double *x) {
    HALA_RANGE();
    return guard([&] {
        HALA_REQUIRE(T && vals && b && x, HALA_ERR_ARG, "hala_trsv_f64: null argument");
        hala_ctx c = T->ctx;
        set_device(c);
        tri_plan &p = trans_checked(trans, "hala_trsv_f64") ? T->T : T->N;
        load_call(T, p, vals, 1);
        tri_exec<double, double, double>(c, p, TRI_SUM, alpha, b, x);
        if (c->opt.sync_checks) check_wait_error(c);
    });
}

// FP32 values and vectors, FP32 arithmetic in the same term order
int hala_trsv_f32(hala_tri T, char trans, float alpha, const float *vals, const float *b, float *x) {
    HALA_RANGE();
    return guard([&] {
        HALA_REQUIRE(T && vals && b && x, HALA_ERR_ARG, "hala_trsv_f32: null argument");
        hala_ctx c = T->ctx;
        set_device(c);
        tri_plan &p = trans_checked(trans, "hala_trsv_f32") ? T->T : T->N;
        load_call(T, p, vals, 1);
        tri_exec<float, float, float>(c, p, TRI_SUM, alpha, b, x);
        if (c->opt.sync_checks) check_wait_error(c);
    });
}

// B <- op(T)^-1 (alpha B): the values into the plan once, then every column
// (64^3 lower triangle, 8 columns: values, copies, sweep and a host wait per
// column took 1030 us).
int hala_trsm_f64(hala_tri T, char transa, char transb, int nrhs, double alpha, const double *vals, double *B,
                  int ldb) {
    HALA_RANGE();
    return guard([&] {
        HALA_REQUIRE(T && vals, HALA_ERR_ARG, "hala_trsm_f64: null argument");
        hala_ctx c = T->ctx;
        set_device(c);
        const trsm_layout l = tri_trsm_layout(T, transb, nrhs, B, ldb);
        if (nrhs == 0) return;
        tri_plan &p = trans_checked(transa, "hala_trsm_f64") ? T->T : T->N;
        load_call(T, p, vals, nrhs);
        tri_exec_cols<double>(c, p, TRI_SUM, alpha, B, l.ldb, l.inc, nrhs);
        if (c->opt.sync_checks) check_wait_error(c);
    });
}

int hala_trsm_f32(hala_tri T, char transa, char transb, int nrhs, float alpha, const float *vals, float *B, int ldb) {
    HALA_RANGE();
    return guard([&] {
        HALA_REQUIRE(T && vals, HALA_ERR_ARG, "hala_trsm_f32: null argument");
        hala_ctx c = T->ctx;
        set_device(c);
        const trsm_layout l = tri_trsm_layout(T, transb, nrhs, B, ldb);
        if (nrhs == 0) return;
        tri_plan &p = trans_checked(transa, "hala_trsm_f32") ? T->T : T->N;
        load_call(T, p, vals, nrhs);
        tri_exec_cols<float>(c, p, TRI_SUM, alpha, B, l.ldb, l.inc, nrhs);
        if (c->opt.sync_checks) check_wait_error(c);
    });
}

}  // extern "C"
