// cgsmall.hip -- identity / Jacobi CG of a small system in one workgroup.
//
// A pass of the launched loop (cg.hip) on a few thousand rows costs two
// launches and two chip-wide reductions, 9 .. 14 us whatever the size.  Here
// one workgroup keeps the whole iteration: wavefront w owns the canonical
// 256-row block w, lane l of it the rows l, l + 64, l + 128, l + 192, so that a
// block's halving tree is three register adds and six lane shuffles; the
// direction lives in LDS, everything else (x, r, A p, the diagonal and, for
// short rows, the matrix itself) in registers.  Three workgroup barriers per
// pass.  Step order, row sums and reduction order are those of the launched
// loop, so every scalar and vector is the same bit for bit.  What bounds it is
// one CU's chain of LDS gather, tree and barrier.  Per pass, launched -> here
// (identity; Jacobi): 8^2 5-point 9.1 -> 1.5 us; 10.7 -> 2.1, 64^2 5-point
// 11.7 -> 3.5; 13.3 -> 4.6, 16^3 7-point 12.2 -> 4.3; 14.1 -> 6.2.
#include "cgsmall.hpp"

namespace hala_amd {

namespace {

constexpr int BW = 4;        // rows per lane of one block
constexpr int MAX_WAVES = 16;
constexpr int PASSES = 1024;  // passes per launch (the host looks at the stop flag in between)

// column-major copy of the matrix: entry k of row i at k n + i, columns as
// 16-bit; rows shorter than the longest are padded (never used)
__global__ __launch_bounds__(256) void cgs_ell(int n, int len, const int *__restrict__ pntr,
                                               const int *__restrict__ indx, const double *__restrict__ vals,
                                               double *__restrict__ ev, unsigned short *__restrict__ ec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int a = pntr[i], m = pntr[i + 1] - a;
    for (int k = 0; k < len; k++) {
        ev[(size_t)k * n + i] = k < m ? vals[a + k] : 0.0;
        ec[(size_t)k * n + i] = (unsigned short)(k < m ? indx[a + k] : 0);
    }
}

// the canonical tree of one block: a[t] + a[t+128], + a[t+64], then 32 .. 1 (in lane 0)
__device__ __forceinline__ double block_tree(const double *v) {
    double a = (v[0] + v[2]) + (v[1] + v[3]);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) a = a + __shfl_down(a, o, 64);
    return a;
}
// the final pass over nb <= 16 partials, by every wavefront
__device__ __forceinline__ double final_tree(const double *part, int nb) {
    const int l = threadIdx.x & 63;
    double a = 0.0;
    if (l < nb) a = a + part[l];
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) a = a + __shfl_down(a, o, 64);
    return __longlong_as_double(
        ((long long)__builtin_amdgcn_readfirstlane((int)(__double_as_longlong(a) >> 32)) << 32) |
        (unsigned)__builtin_amdgcn_readfirstlane((int)__double_as_longlong(a)));
}

// ML > 0: rows of at most ML entries, held in registers; 0: len entries, re-read each pass.
template <int ML, bool JAC>
__global__ __launch_bounds__(64 * MAX_WAVES) void cg_small_kernel(int n, int len, const int *__restrict__ pntr,
                                                                  const double *__restrict__ ev,
                                                                  const unsigned short *__restrict__ ec,
                                                                  const double *__restrict__ d, double *__restrict__ x,
                                                                  double *__restrict__ rg, double *__restrict__ pg,
                                                                  cg_state *st) {
    if (st->done) return;
    constexpr int R = BW;
    __shared__ double sp[BW * 64 * MAX_WAVES];
    __shared__ double part[3][MAX_WAVES];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nb = blockDim.x >> 6;
    double xv[R], rv[R], dv[R], pv[R];
    double mv[ML > 0 ? R * ML : 1];
    unsigned short mc[ML > 0 ? R * ML : 1];
    int rl[R];
    auto row_of = [&](int q) { return w * CB + q * 64 + lane; };
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int i = row_of(q);
        const bool in = i < n;
        xv[q] = in ? x[i] : 0.0;
        rv[q] = in ? rg[i] : 0.0;
        pv[q] = in ? pg[i] : 0.0;
        dv[q] = JAC && in ? d[i] : 1.0;
        rl[q] = in ? pntr[i + 1] - pntr[i] : 0;
        if (in) sp[i] = pv[q];
        if (ML > 0) {
#pragma unroll
            for (int k = 0; k < ML; k++) {
                const bool e = in && k < len;
                mv[q * ML + k] = e ? ev[(size_t)k * n + i] : 0.0;
                mc[q * ML + k] = e ? ec[(size_t)k * n + i] : 0;
            }
        }
    }
    double zr = st->zr;
    const double tol = st->tol;
    int it = st->it, done = 0, status = 0;
    double rn = st->rn, alpha = st->alpha, beta = st->beta;
    __syncthreads();
    auto publish = [&](const double (&v)[R], int s) {
        const double a = block_tree(v);
        if (lane == 0) part[s][w] = a;
    };
    for (int pass = 0; pass < PASSES && !done; pass++) {
        double ap[R], v[R];
#pragma unroll
        for (int q = 0; q < R; q++) ap[q] = 0.0;
        if (ML > 0) {
#pragma unroll
            for (int k = 0; k < ML; k++)
#pragma unroll
                for (int q = 0; q < R; q++) {
                    const double s = ap[q] + mv[q * ML + k] * sp[mc[q * ML + k]];
                    ap[q] = k < rl[q] ? s : ap[q];
                }
        } else {
            for (int k = 0; k < len; k++)
#pragma unroll
                for (int q = 0; q < R; q++) {
                    const int i = min(row_of(q), n - 1);
                    const double s = ap[q] + ev[(size_t)k * n + i] * sp[ec[(size_t)k * n + i]];
                    ap[q] = k < rl[q] ? s : ap[q];
                }
        }
#pragma unroll
        for (int q = 0; q < R; q++) {
            ap[q] = 1.0 * ap[q] + 0.0;
            v[q] = pv[q] * ap[q];
        }
        publish(v, 0);
        __syncthreads();
        alpha = zr / final_tree(part[0], nb);
        it++;
#pragma unroll
        for (int q = 0; q < R; q++) {
            xv[q] = xv[q] + alpha * pv[q];
            rv[q] = rv[q] + (-alpha) * ap[q];
            v[q] = rv[q] * rv[q];
        }
        publish(v, 1);
        double z[R];
        if (JAC) {
#pragma unroll
            for (int q = 0; q < R; q++) {
                z[q] = rv[q] / dv[q];
                v[q] = rv[q] * z[q];
            }
            publish(v, 2);
        }
        __syncthreads();
        const double rr = final_tree(part[1], nb);
        rn = sqrt(rr);
        if (threadIdx.x == 0 && st->hist && it - 2 < st->max_hist) st->hist[it - 2] = rn;
        if (it == st->max_iter || rn < tol) {
            done = 1;
        } else if (!isfinite(rn)) {
            done = 1;
            status = 1;
        } else {
            const double nzr = JAC ? final_tree(part[2], nb) : rr;
            beta = nzr / zr;
            zr = nzr;
#pragma unroll
            for (int q = 0; q < R; q++) {
                pv[q] = beta * pv[q] + 1.0 * (JAC ? z[q] : rv[q]);
                const int i = row_of(q);
                if (i < n) sp[i] = pv[q];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int i = row_of(q);
        if (i >= n) continue;
        x[i] = xv[q];
        rg[i] = rv[q];
        pg[i] = pv[q];
    }
    if (threadIdx.x == 0) {
        st->zr = zr;
        st->alpha = alpha;
        st->beta = beta;
        st->rn = rn;
        st->it = it;
        st->done = done;
        st->status = status;
    }
}

}  // namespace

// One workgroup holds 16 blocks.  With two blocks per wavefront (tried up to
// 8192 rows) the matrix no longer fits the registers and the re-read costs what
// the launches did: 80^2 9.8 us against 12.2, 20^3 12.6 against 12.6.
// Rows of up to 16 entries: a lane sums its rows one entry at a time, where the
// launched product spreads them over the chip.  Launched -> here per pass: rows
// of 7 on average, 16 at most, 1000 rows 11.4 -> 10.3 us, 4000 rows 13.6 ->
// 12.4; 14 on average, 24 at most, 300 rows 12.6 -> 16.1.  The padded copy
// stays within four times the matrix.
bool cg_small_fits(hala_csr A) {
    return A->nrows > 0 && A->nrows <= MAX_WAVES * CB && A->max_row >= 1 && A->max_row <= 16 &&
           (int64_t)A->max_row * A->nrows <= 4 * A->nnz;
}

void cg_small_passes(hala_ctx c, hala_csr A, const double *vals, const double *pdiag, double *x, double *r, double *p,
                     cg_state *st, const std::function<int()> &done) {
    const int n = A->nrows, len = A->max_row, nw = (n + CB - 1) / CB;
    tmp_scope ts(c);
    dbuf &ev = ts.get(), &ec = ts.get();
    ev.reserve((size_t)n * len * sizeof(double));
    ec.reserve((size_t)n * len * sizeof(unsigned short));
    cgs_ell<<<(n + 255) / 256, 256, 0, c->stream>>>(n, len, A->pntr, A->indx, vals, ev.as<double>(),
                                                    ec.as<unsigned short>());
    HALA_CHECK_LAUNCH();
    do {
#define HALA_CGS(MLV)                                                                                            \
    if (pdiag)                                                                                                  \
        cg_small_kernel<MLV, true><<<1, 64 * nw, 0, c->stream>>>(n, len, A->pntr, ev.as<double>(),               \
                                                                 ec.as<unsigned short>(), pdiag, x, r, p, st);  \
    else                                                                                                        \
        cg_small_kernel<MLV, false><<<1, 64 * nw, 0, c->stream>>>(n, len, A->pntr, ev.as<double>(),              \
                                                                  ec.as<unsigned short>(), nullptr, x, r, p, st)
        // the matrix of short rows fits the registers that 16 wavefronts leave a lane
        if (len <= 5) {
            HALA_CGS(5);
        } else if (len <= 7) {
            HALA_CGS(7);
        } else {
            HALA_CGS(0);
        }
#undef HALA_CGS
        HALA_CHECK_LAUNCH();
    } while (!done());
}

}  // namespace hala_amd
