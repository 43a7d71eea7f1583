// batch.hip -- thousands of independent small SPD systems solved by
// Jacobi-preconditioned CG in one persistent launch, replayed from a HIP graph.
//
// Each workgroup (a "team" of T threads) takes systems from a queue ordered
// largest first and runs the whole CG loop of one system with HALA's step
// order (hex/solvers/hala_solvers_cg.hpp:92-156; Jacobi apply = vdivide,
// wax/hala_blas_extensions.hpp:139-151).  Thread t owns rows t, t+T, ...; team
// dot products: thread t sums its rows in order from 0, then the team is
// reduced with the halving tree (pairs t, t+off).  Two kernels: where the
// systems fit, batch_resident_kernel keeps them whole on the chip (p in LDS,
// the rest in registers); batch_pcg_kernel has only p in LDS and serves longer
// rows and larger systems.
// The team size and workgroups per CU come from hala_batch_tune().
#include <algorithm>
#include <climits>
#include <cmath>
#include <numeric>
#include <vector>

#include "common.hpp"

struct hala_batch_s {
    hala_ctx ctx = nullptr;
    int nsys = 0, n_total = 0, max_n = 0, max_row = 0;
    std::vector<int> sizes;  // rows of each system, largest first (the queue's order)
    int64_t nnz_total = 0;
    const int *row_off = nullptr, *pntr = nullptr, *indx = nullptr;  // device, not owned
    hala_amd::dbuf order, work, iters, ctl;
    int team = 256, wg_per_cu = 2;
    int path = -1;  // what launch_batch last chose (hala_path)
    // graph cache
    hipStream_t cap = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    const void *key[4] = {nullptr, nullptr, nullptr, nullptr};
    double key_rtol = -1.0;
    int key_max_iter = -1, key_team = -1, key_wg = -1;
    ~hala_batch_s() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        if (cap) (void)hipStreamDestroy(cap);
    }
};

namespace hala_amd {

// halving-tree reduction over the team; every thread gets the result
template <int T>
__device__ __forceinline__ double team_sum(double v, double *red) {
    const int t = threadIdx.x;
    if (T > 64) {
        red[t] = v;
        __syncthreads();
#pragma unroll
        for (int off = T / 2; off >= 64; off >>= 1) {
            if (t < off) red[t] = red[t] + red[t + off];
            __syncthreads();
        }
        if (t < 64) v = red[t];
    }
    if (t < 64) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v = v + __shfl_down(v, off, 64);
        if (t == 0) red[0] = v;
    }
    __syncthreads();
    double r = red[0];
    __syncthreads();
    return r;
}

__global__ void batch_reset_kernel(unsigned *ctl) {
    ctl[0] = 0u;
    ctl[1] = 0u;
}

template <int T>
__global__ __launch_bounds__(T) void batch_pcg_kernel(int nsys, int n_total, int max_n, const int *__restrict__ order,
                                                      const int *__restrict__ row_off, const int *__restrict__ pntr,
                                                      const int *__restrict__ indx, const double *__restrict__ vals,
                                                      const double *__restrict__ dvals, const double *__restrict__ b,
                                                      double *__restrict__ x, double *__restrict__ work, double rtol,
                                                      int max_iter, int *__restrict__ iters, unsigned *ctl) {
    extern __shared__ double lds[];
    double *sp = lds;          // p of the current system
    double *red = lds + max_n; // team reduction scratch
    __shared__ int s_q;
    const int t = threadIdx.x;
    for (;;) {
        if (t == 0) s_q = (int)atomicAdd(ctl, 1u);
        __syncthreads();
        const int q = s_q;
        __syncthreads();
        if (q >= nsys) break;
        const int s = order[q];
        const int r0 = row_off[s];
        const int n = row_off[s + 1] - r0;
        const int *P = pntr + r0;
        double *xs = x + r0;
        double *rs = work + r0;
        double *aps = work + n_total + r0;
        const double *bs = b + r0;
        const double *ds = dvals + r0;
        // tol = rtol * norm2(b)
        double acc = 0.0;
        for (int i = t; i < n; i += T) acc = acc + bs[i] * bs[i];
        const double tol = rtol * sqrt(team_sum<T>(acc, red));
        // r = b + (-1)(1*(A x) + 0); z = r ./ d; p = z; zr = <r, z>
        acc = 0.0;
        for (int i = t; i < n; i += T) {
            double sum = 0.0;
            for (int j = P[i]; j < P[i + 1]; j++) sum = sum + vals[j] * xs[indx[j]];
            double ri = bs[i] + (-1.0) * (1.0 * sum + 0.0);
            rs[i] = ri;
            double zi = ri / ds[i];
            sp[i] = zi;
            acc = acc + ri * zi;
        }
        double zr = team_sum<T>(acc, red);  // (its barriers also publish sp)
        int it = 1;
        for (;;) {
            // Ap = A p, <p, Ap>
            acc = 0.0;
            for (int i = t; i < n; i += T) {
                double sum = 0.0;
                for (int j = P[i]; j < P[i + 1]; j++) sum = sum + vals[j] * sp[indx[j]];
                double y = 1.0 * sum + 0.0;
                aps[i] = y;
                acc = acc + sp[i] * y;
            }
            const double pap = team_sum<T>(acc, red);
            it++;
            const double a = zr / pap;
            double rr = 0.0, rz = 0.0;
            for (int i = t; i < n; i += T) {
                xs[i] = xs[i] + a * sp[i];
                double ri = rs[i] + (-a) * aps[i];
                rs[i] = ri;
                rr = rr + ri * ri;
                rz = rz + ri * (ri / ds[i]);
            }
            const double rn = sqrt(team_sum<T>(rr, red));
            const double nzr = team_sum<T>(rz, red);
            if (it == max_iter || rn < tol || !(rn == rn)) break;
            const double beta = nzr / zr;
            for (int i = t; i < n; i += T) sp[i] = beta * sp[i] + 1.0 * (rs[i] / ds[i]);
            zr = nzr;
            __syncthreads();  // p complete before the next product
        }
        if (t == 0) iters[s] = it;
        __syncthreads();
    }
}

// v of lane l + OFF in lane l, for the lanes that lane 0's halving tree needs
template <int OFF>
__device__ __forceinline__ int lane_down(int v) {
    if (OFF == 32) return __builtin_amdgcn_permlane32_swap(v, v, false, false)[1];
    if (OFF == 16) return __builtin_amdgcn_permlane16_swap(v, v, false, false)[1];
    return __builtin_amdgcn_update_dpp(v, v, 0x100 + (OFF & 15), 0xf, 0xf, false);  // row_shl
}
template <int OFF>
__device__ __forceinline__ double add_down(double v) {
    return v + __hiloint2double(lane_down<OFF>(__double2hiint(v)), lane_down<OFF>(__double2loint(v)));
}
// the halving tree over 64 lanes, in lane 0
__device__ __forceinline__ double wave_tree(double v) {
    return add_down<1>(add_down<2>(add_down<4>(add_down<8>(add_down<16>(add_down<32>(v))))));
}
// the halving tree over the team's NW wavefront sums
template <int NW>
__device__ __forceinline__ double waves_tree(const double *red) {
    double v[NW];
#pragma unroll
    for (int j = 0; j < NW; j++) v[j] = red[j];
#pragma unroll
    for (int o = NW / 2; o >= 1; o >>= 1)
#pragma unroll
        for (int j = 0; j < o; j++) v[j] = v[j] + v[j + o];
    return v[0];
}

// The team's loop with the whole system on the chip: at most R T rows of at
// most LEN entries.  Team thread u = l NW + w (l lane, w wavefront, NW
// wavefronts) keeps values and columns of its rows u, u + T, ... and their r,
// x and d in registers; p is in LDS, row q T + u at q T + 64 w + l.  So
//  - an iteration reads no memory, where the loop above reads about 130 B per
//    row, most of it by lanes 40 B apart;
//  - lane l and its neighbours gather p at a stride of 8 B whatever a column's
//    offset: no bank conflicts;
//  - the upper levels of the team's halving tree (u, u + T/2, ...) pair lanes of
//    one wavefront, the lower ones the NW wavefronts' sums: one barrier per
//    reduction, and <r, r> and <r, z> share it.  Three barriers per iteration.
// Unused entries carry value 0 and the column of a slot that holds 0 (the sum,
// never -0, keeps its bits).  What bounds it: FP64 issue and LDS reads, the three
// barriers with their trees and divisions (1.5 us of an iteration's 3.8 for 69^2
// 5-point rows and a team of 512 alone on its CU; 0.5 us for 14^2 in teams of
// 256, 4 per CU), and the load of a system (about 45 us for 69^2).  4096 systems of
// 14^2 .. 70^2, team 512: 6.5 -> 1.87 ms; both give the team's order, so the
// same bits.  Two rounds interleaved, or the matrix loads a round ahead, need
// more registers than there are: 2.06 ms with the spills.
template <int T, int R, int LEN, int WPE>
__global__ __launch_bounds__(T, WPE) void batch_resident_kernel(
    int q0, int q1, const int *__restrict__ order, const int *__restrict__ row_off, const int *__restrict__ pntr,
    const int *__restrict__ indx, const double *__restrict__ vals, const double *__restrict__ dvals,
    const double *__restrict__ b, double *__restrict__ x, double rtol, int max_iter, int *__restrict__ iters,
    unsigned *ctl) {
    extern __shared__ double lds[];
    constexpr int NW = T / 64;
    double *sp = lds + 1 + 3 * NW;  // lds[0] = 0
    double *red = lds + 1;
    double *sv = sp;
    int *si = reinterpret_cast<int *>(sp + T * LEN);
    __shared__ int s_q;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int u = lane * NW + w;                   // the team thread whose rows these are
    const int tpos = (t % NW) * 64 + t / NW;       // p slot of row q T + t
    constexpr unsigned SP = (1 + 3 * NW) * 8;      // byte offset of sp
    auto gather = [&](unsigned off) { return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(lds) + off); };
    if (t == 0) lds[0] = 0.0;
    for (;;) {
        if (t == 0) s_q = q0 + (int)atomicAdd(ctl, 1u);
        __syncthreads();
        const int qs = s_q;
        if (qs >= q1) break;
        const int s = order[qs];
        const int r0 = row_off[s];
        const int n = row_off[s + 1] - r0;
        const int *P = pntr + r0;
        const double *bs = b + r0, *ds = dvals + r0;
        double *xs = x + r0;
        const int nq = (n + T - 1) / T;
        double mv[R * LEN], rv[R], xv[R], dv[R], y[R];
        unsigned mo[(R * LEN + 1) / 2];
        // the vectors in row order (their loads pass under the matrix's), then the matrix, T rows at a time through LDS
#pragma unroll
        for (int q = 0; q < R; q++)
            if (q * T + t < n) {
                rv[q] = bs[q * T + t];
                dv[q] = ds[q * T + t];
                xv[q] = xs[q * T + t];
            }
#pragma unroll
        for (int q = 0; q < R; q++)
            if (q < nq) {
                const int i0 = q * T, i1 = min(n, i0 + T), base = P[i0], m = P[i1] - base;
#pragma unroll
                for (int k = 0; k < LEN; k++) {
                    const int e = k * T + t;
                    if (e >= m) break;
                    sv[e] = vals[base + e];
                    si[e] = indx[base + e];
                }
                const int i = i0 + u;
                const int a = i < n ? P[i] - base : 0, len = i < n ? P[i + 1] - base - a : 0;
                __syncthreads();
#pragma unroll
                for (int k = 0; k < LEN; k++) {
                    const int e = q * LEN + k;
                    double v = 0.0;
                    unsigned o = 0;
                    if (k < len) {
                        v = sv[a + k];
                        const unsigned c = si[a + k], cu = c % T;
                        o = SP + 8 * (c - cu + (cu % NW) * 64 + cu / NW);
                    }
                    mv[e] = v;
                    mo[e / 2] = (e & 1) ? mo[e / 2] | (o << 16) : o;
                }
                __syncthreads();
            }
        // a vector in row order (round q: row q T + t) to the threads that own the rows
        auto spread = [&](double(&v)[R]) {
#pragma unroll
            for (int q = 0; q < R; q++)
                if (q < nq) sp[q * T + tpos] = v[q];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < R; q++)
                if (q < nq) v[q] = sp[q * T + w * 64 + lane];
        };
        // tol = rtol * norm2(b)
        double acc = 0.0;
        spread(rv);
#pragma unroll
        for (int q = 0; q < R; q++)
            if (q < nq) acc = q * T + u < n ? acc + rv[q] * rv[q] : acc;
        acc = wave_tree(acc);
        if (lane == 0) red[w] = acc;
        __syncthreads();
        const double tol = rtol * sqrt(waves_tree<NW>(red));
        spread(dv);
        __syncthreads();
        // r = b + (-1)(1*(A x) + 0); z = r ./ d; p = z; zr = <r, z>
        spread(xv);
        acc = 0.0;
#pragma unroll
        for (int q = 0; q < R; q++)
            if (q < nq) {
                double sum = 0.0;
#pragma unroll
                for (int k = 0; k < LEN; k++) {
                    const int e = q * LEN + k;
                    sum = sum + mv[e] * gather((e & 1) ? mo[e / 2] >> 16 : mo[e / 2] & 0xffffu);
                }
                rv[q] = rv[q] + (-1.0) * (1.0 * sum + 0.0);
                y[q] = rv[q] / dv[q];
                acc = q * T + u < n ? acc + rv[q] * y[q] : acc;
            }
        acc = wave_tree(acc);
        if (lane == 0) red[NW + w] = acc;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < R; q++)
            if (q < nq) sp[q * T + w * 64 + lane] = y[q];
        double zr = waves_tree<NW>(red + NW);
        __syncthreads();
        int it = 1;
        for (;;) {
            // Ap = A p, <p, Ap>; the columns stay packed (unpacked ahead of the loop they'd take twice the registers)
#pragma unroll
            for (int e = 0; e < (R * LEN + 1) / 2; e++) asm volatile("" : "+v"(mo[e]));
            acc = 0.0;
#pragma unroll
            for (int q = 0; q < R; q++)
                if (q < nq) {
                    double sum = 0.0;
#pragma unroll
                    for (int k = 0; k < LEN; k++) {
                        const int e = q * LEN + k;
                        sum = sum + mv[e] * gather((e & 1) ? mo[e / 2] >> 16 : mo[e / 2] & 0xffffu);
                    }
                    y[q] = 1.0 * sum + 0.0;
                    acc = q * T + u < n ? acc + sp[q * T + w * 64 + lane] * y[q] : acc;
                }
            acc = wave_tree(acc);
            if (lane == 0) red[w] = acc;
            __syncthreads();
            it++;
            const double a = zr / waves_tree<NW>(red);
            double rr = 0.0, rz = 0.0;
#pragma unroll
            for (int q = 0; q < R; q++)
                if (q < nq) {
                    const bool in = q * T + u < n;
                    xv[q] = xv[q] + a * sp[q * T + w * 64 + lane];
                    rv[q] = rv[q] + (-a) * y[q];
                    rr = in ? rr + rv[q] * rv[q] : rr;
                    y[q] = rv[q] / dv[q];
                    rz = in ? rz + rv[q] * y[q] : rz;
                }
            rr = wave_tree(rr);
            rz = wave_tree(rz);
            if (lane == 0) {
                red[NW + w] = rr;
                red[2 * NW + w] = rz;
            }
            __syncthreads();
            const double rn = sqrt(waves_tree<NW>(red + NW));
            const double nzr = waves_tree<NW>(red + 2 * NW);
            if (it == max_iter || rn < tol || !(rn == rn)) break;
            const double beta = nzr / zr;
#pragma unroll
            for (int q = 0; q < R; q++)
                if (q < nq) {
                    double *pq = sp + q * T + w * 64 + lane;
                    *pq = beta * *pq + 1.0 * y[q];
                }
            zr = nzr;
            __syncthreads();  // p complete before the next product
        }
        // x back in row order (every wavefront is past its last read of p)
#pragma unroll
        for (int q = 0; q < R; q++)
            if (q < nq) sp[q * T + w * 64 + lane] = xv[q];
        if (t == 0) iters[s] = it;
        __syncthreads();
        for (int q = 0; q < nq; q++)
            if (q * T + t < n) xs[q * T + t] = sp[q * T + tpos];
        __syncthreads();
    }
}

template <int T, int LEN>
constexpr size_t resident_lds(int rows) {
    return (1 + 3 * (T / 64)) * sizeof(double) +
           std::max((size_t)(rows + T - 1) / T * T * sizeof(double), (size_t)T * LEN * 12);
}

static size_t batch_lds(int team, int max_n) { return (size_t)(max_n + team) * sizeof(double); }

// Systems whose rows fit the registers, in two launches: up to R1 rows per
// thread at 128 registers (four wavefronts per SIMD in flight), the larger ones
// up to R2 at 256.  2.5 LEN + 8 registers per row and about 45 others: R1, R2 are
// the largest that do not spill.  Past them the general loop runs (58^2 with a
// team of 256: 21 us per iteration against 3.2 with 512).  Returns whether it ran.
template <int T, int LEN, int R1, int R2>
static bool resident(hala_batch B, hipStream_t s, int wg, const double *vals, const double *dvals, const double *b,
                     double *x, double rtol, int max_iter) {
    if (B->max_n > std::max(R1, R2) * T) return false;
    hala_ctx c = B->ctx;
    // sizes fall: [0, big) need R2
    const int big = (int)(std::partition_point(B->sizes.begin(), B->sizes.end(), [](int n) { return n > R1 * T; }) -
                          B->sizes.begin());
    unsigned *ctl = B->ctl.as<unsigned>();
    B->path = (big ? 4 : 0) + (big < B->nsys ? 2 : 0);
    auto grid = [&](int k) { return std::max(1, std::min(k, c->num_cus * wg)); };
    if (big)
        batch_resident_kernel<T, R2, LEN, 2><<<grid(big), T, resident_lds<T, LEN>(B->sizes[0]), s>>>(
            0, big, B->order.as<int>(), B->row_off, B->pntr, B->indx, vals, dvals, b, x, rtol, max_iter,
            B->iters.as<int>(), ctl);
    if (big < B->nsys)
        batch_resident_kernel<T, R1, LEN, 4><<<grid(B->nsys - big), T, resident_lds<T, LEN>(B->sizes[big]), s>>>(
            big, B->nsys, B->order.as<int>(), B->row_off, B->pntr, B->indx, vals, dvals, b, x, rtol, max_iter,
            B->iters.as<int>(), ctl + 1);
    HALA_CHECK_LAUNCH();
    return true;
}

// A CU's registers hold 16 wavefronts of them, the general loop up to 32: a shape that asks for more on
// systems with few rows per thread, where barriers are all there is to hide, runs faster on the loop.  Team
// 1024, 2 per CU, general -> resident (us, 12 passes): 256 rows 307 -> 447, 512 204 -> 254, 1024 167 -> 159;
// team 512, 4 per CU: 64 rows 476 -> 594, 128 286 -> 311, 200 214 -> 223, 256 185 -> 178; smaller teams gain
// at any size.  (The systems' mean decides: the small ones are the many.)
static bool resident_crowded(hala_batch B, int team, int wg) {
    const int rows = team == 1024 ? 1024 : team == 512 ? 205 : 0;
    return team * wg > 1024 && (int64_t)B->n_total < (int64_t)B->nsys * rows;
}

static bool launch_resident(hala_batch B, hipStream_t s, int team, int wg, const double *vals, const double *dvals,
                            const double *b, double *x, double rtol, int max_iter) {
    if (resident_crowded(B, team, wg)) return false;
#define HALA_RES(T, LEN, R1, R2) resident<T, LEN, R1, R2>(B, s, wg, vals, dvals, b, x, rtol, max_iter)
    if (B->max_row <= 5) switch (team) {
        case 64: return HALA_RES(64, 5, 4, 10);
        case 128: return HALA_RES(128, 5, 4, 10);
        case 256: return HALA_RES(256, 5, 4, 10);
        case 512: return HALA_RES(512, 5, 4, 10);
        case 1024: return HALA_RES(1024, 5, 3, 3);
        }
    else if (B->max_row <= 7) switch (team) {
        case 64: return HALA_RES(64, 7, 3, 8);
        case 128: return HALA_RES(128, 7, 3, 8);
        case 256: return HALA_RES(256, 7, 3, 8);
        case 512: return HALA_RES(512, 7, 3, 8);
        }
#undef HALA_RES
    return false;
}

static void launch_batch(hala_batch B, hipStream_t s, int team, int wg, const double *vals, const double *dvals,
                         const double *b, double *x, double rtol, int max_iter) {
    hala_ctx c = B->ctx;
    unsigned *ctl = B->ctl.as<unsigned>();
    int grid = std::max(1, std::min(B->nsys, c->num_cus * wg));
    size_t lds = batch_lds(team, B->max_n);
    batch_reset_kernel<<<1, 1, 0, s>>>(ctl);
    if (launch_resident(B, s, team, wg, vals, dvals, b, x, rtol, max_iter)) return;
    B->path = 1;
#define HALA_BATCH(TT)                                                                                          \
    batch_pcg_kernel<TT><<<grid, TT, lds, s>>>(B->nsys, B->n_total, B->max_n, B->order.as<int>(), B->row_off,    \
                                               B->pntr, B->indx, vals, dvals, b, x, B->work.as<double>(), rtol,  \
                                               max_iter, B->iters.as<int>(), ctl)
    switch (team) {
    case 64: HALA_BATCH(64); break;
    case 128: HALA_BATCH(128); break;
    case 256: HALA_BATCH(256); break;
    case 512: HALA_BATCH(512); break;
    case 1024: HALA_BATCH(1024); break;
    default: throw status_error{HALA_ERR_ARG, "batch team size must be 64, 128, 256, 512 or 1024"};
    }
#undef HALA_BATCH
    HALA_CHECK_LAUNCH();
}

// one workgroup may use at most 64 KiB of dynamic LDS; a CU holds 160 KiB
static bool fits(hala_batch B, int team, int wg) {
    return batch_lds(team, B->max_n) <= 64 * 1024 && batch_lds(team, B->max_n) * wg <= 160 * 1024;
}

// Runs the batched solve through a captured graph (re-captured when the
// arguments or the launch shape change).
static void run_batch(hala_batch B, const double *vals, const double *dvals, const double *b, double *x, double rtol,
                      int max_iter) {
    hala_ctx c = B->ctx;
    bool same = B->exec && B->key[0] == vals && B->key[1] == dvals && B->key[2] == b && B->key[3] == x &&
                B->key_rtol == rtol && B->key_max_iter == max_iter && B->key_team == B->team &&
                B->key_wg == B->wg_per_cu;
    if (!same) {
        if (B->exec) (void)hipGraphExecDestroy(B->exec);
        if (B->graph) (void)hipGraphDestroy(B->graph);
        B->exec = nullptr;
        B->graph = nullptr;
        if (!B->cap) HALA_HIP(hipStreamCreateWithFlags(&B->cap, hipStreamNonBlocking));
        HALA_HIP(hipStreamBeginCapture(B->cap, hipStreamCaptureModeThreadLocal));
        try {
            launch_batch(B, B->cap, B->team, B->wg_per_cu, vals, dvals, b, x, rtol, max_iter);
        } catch (...) {
            hipGraph_t g = nullptr;
            (void)hipStreamEndCapture(B->cap, &g);
            if (g) (void)hipGraphDestroy(g);
            throw;
        }
        HALA_HIP(hipStreamEndCapture(B->cap, &B->graph));
        HALA_HIP(hipGraphInstantiate(&B->exec, B->graph, nullptr, nullptr, 0));
        B->key[0] = vals;
        B->key[1] = dvals;
        B->key[2] = b;
        B->key[3] = x;
        B->key_rtol = rtol;
        B->key_max_iter = max_iter;
        B->key_team = B->team;
        B->key_wg = B->wg_per_cu;
    }
    c->path[PATH_BATCH] = B->path;
    HALA_HIP(hipGraphLaunch(B->exec, c->stream));
}

}  // namespace hala_amd

using namespace hala_amd;

extern "C" {

int hala_batch_create(hala_ctx c, int nsys, const int *row_off, const int *pntr, const int *indx, hala_batch *out) {
    HALA_RANGE();
    return guard([&] {
        HALA_REQUIRE(c && out && nsys > 0 && row_off && pntr && indx, HALA_ERR_ARG, "hala_batch_create: bad argument");
        *out = nullptr;
        set_device(c);
        std::vector<int> ro(nsys + 1);
        HALA_HIP(hipMemcpyAsync(ro.data(), row_off, (nsys + 1) * sizeof(int), hipMemcpyDeviceToHost, c->stream));
        HALA_HIP(hipStreamSynchronize(c->stream));
        HALA_REQUIRE(ro[0] == 0, HALA_ERR_ARG, "hala_batch_create: row_off[0] must be 0");
        int max_n = 0;
        for (int s = 0; s < nsys; s++) {
            HALA_REQUIRE(ro[s + 1] >= ro[s], HALA_ERR_ARG, "hala_batch_create: decreasing row offsets");
            max_n = std::max(max_n, ro[s + 1] - ro[s]);
        }
        HALA_REQUIRE((size_t)(max_n + 64) * sizeof(double) <= 64 * 1024, HALA_ERR_ARG,
                     "hala_batch_create: a system exceeds the LDS-resident size (8128 rows)");
        const int n_total = ro[nsys];
        // every system's pattern must stay inside its own rows
        int nnz_total = 0;
        HALA_HIP(hipMemcpyAsync(&nnz_total, pntr + n_total, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        HALA_HIP(hipStreamSynchronize(c->stream));
        auto *B = new hala_batch_s();
        try {
            B->ctx = c;
            B->nsys = nsys;
            B->n_total = n_total;
            B->max_n = max_n;
            B->nnz_total = nnz_total;
            B->row_off = row_off;
            B->pntr = pntr;
            B->indx = indx;
            // largest systems first: the dynamic queue then balances the tail
            std::vector<int> ord(nsys);
            std::iota(ord.begin(), ord.end(), 0);
            std::stable_sort(ord.begin(), ord.end(),
                             [&](int a, int b) { return ro[a + 1] - ro[a] > ro[b + 1] - ro[b]; });
            for (int s : ord) B->sizes.push_back(ro[s + 1] - ro[s]);
            B->order.reserve(nsys * sizeof(int));
            HALA_HIP(hipMemcpyAsync(B->order.p, ord.data(), nsys * sizeof(int), hipMemcpyHostToDevice, c->stream));
            B->work.reserve((size_t)2 * std::max(n_total, 1) * sizeof(double));
            B->iters.reserve(nsys * sizeof(int));
            B->ctl.reserve(4 * sizeof(unsigned));
            HALA_HIP(hipStreamSynchronize(c->stream));
            // kernel-side bounds: validate every system's columns
            std::vector<int> hp(n_total + 1), hi(nnz_total);
            HALA_HIP(hipMemcpy(hp.data(), pntr, (n_total + 1) * sizeof(int), hipMemcpyDeviceToHost));
            HALA_HIP(hipMemcpy(hi.data(), indx, (size_t)nnz_total * sizeof(int), hipMemcpyDeviceToHost));
            for (int s = 0; s < nsys; s++) {
                int ns = ro[s + 1] - ro[s];
                for (int i = ro[s]; i < ro[s + 1]; i++) {
                    HALA_REQUIRE(hp[i] <= hp[i + 1] && hp[i + 1] <= nnz_total, HALA_ERR_PATTERN,
                                 "hala_batch_create: bad row pointers at row " + std::to_string(i));
                    B->max_row = std::max(B->max_row, hp[i + 1] - hp[i]);
                    for (int j = hp[i]; j < hp[i + 1]; j++)
                        HALA_REQUIRE(hi[j] >= 0 && hi[j] < ns, HALA_ERR_PATTERN,
                                     "hala_batch_create: column outside its system at row " + std::to_string(i));
                }
            }
        } catch (...) {
            delete B;
            throw;
        }
        *out = B;
    });
}

int hala_batch_destroy(hala_batch B) {
    return guard([&] {
        if (!B) return;
        (void)hipSetDevice(B->ctx->device);
        (void)hipStreamSynchronize(B->ctx->stream);
        delete B;
    });
}

int hala_batch_set_shape(hala_batch B, int team, int wg_per_cu) {
    return guard([&] {
        HALA_REQUIRE(B, HALA_ERR_ARG, "null batch");
        HALA_REQUIRE(team == 64 || team == 128 || team == 256 || team == 512 || team == 1024, HALA_ERR_ARG,
                     "team must be 64..1024 (power of two)");
        HALA_REQUIRE(wg_per_cu >= 1 && wg_per_cu <= 16 && fits(B, team, wg_per_cu), HALA_ERR_ARG,
                     "workgroups per CU do not fit the LDS");
        B->team = team;
        B->wg_per_cu = wg_per_cu;
    });
}

int hala_batch_get_shape(hala_batch B, int *team, int *wg_per_cu) {
    return guard([&] {
        HALA_REQUIRE(B && team && wg_per_cu, HALA_ERR_ARG, "null argument");
        *team = B->team;
        *wg_per_cu = B->wg_per_cu;
    });
}

int hala_batch_pcg_f64(hala_batch B, const double *vals, const double *dvals, const double *b, double *x,
                       double rtol, int max_iter, int *iters) {
    HALA_RANGE();
    return guard([&] {
        HALA_REQUIRE(B && vals && dvals && b && x, HALA_ERR_ARG, "hala_batch_pcg_f64: null argument");
        HALA_REQUIRE(max_iter >= 2, HALA_ERR_ARG, "hala_batch_pcg_f64: max_iter must be >= 2");
        hala_ctx c = B->ctx;
        set_device(c);
        run_batch(B, vals, dvals, b, x, rtol, max_iter);
        if (iters)
            HALA_HIP(hipMemcpyAsync(iters, B->iters.p, B->nsys * sizeof(int), hipMemcpyDeviceToDevice, c->stream));
    });
}

// Autotuner: times every (team, workgroups per CU) shape that fits the LDS on
// the given problem (x reset to zero before each run, best of `reps`) and
// keeps the fastest.  ms_out (host, nullable) receives its time.
int hala_batch_tune(hala_batch B, const double *vals, const double *dvals, const double *b, double *x, double rtol,
                    int max_iter, int reps, int *team_out, int *wg_out, double *ms_out) {
    HALA_RANGE();
    return guard([&] {
        HALA_REQUIRE(B && vals && dvals && b && x && reps >= 1, HALA_ERR_ARG, "hala_batch_tune: bad argument");
        hala_ctx c = B->ctx;
        set_device(c);
        hipEvent_t e0, e1;
        HALA_HIP(hipEventCreate(&e0));
        HALA_HIP(hipEventCreate(&e1));
        float best = 1e30f;
        int bt = B->team, bw = B->wg_per_cu;
        const int teams[] = {64, 128, 256, 512, 1024};
        const int wgs[] = {1, 2, 4, 8};
        try {
            for (int tm : teams)
                for (int wg : wgs) {
                    if (!fits(B, tm, wg) || tm * wg > 2048) continue;
                    float tbest = 1e30f;
                    for (int r = 0; r < reps; r++) {
                        HALA_HIP(hipMemsetAsync(x, 0, (size_t)B->n_total * sizeof(double), c->stream));
                        HALA_HIP(hipEventRecord(e0, c->stream));
                        launch_batch(B, c->stream, tm, wg, vals, dvals, b, x, rtol, max_iter);
                        HALA_HIP(hipEventRecord(e1, c->stream));
                        HALA_HIP(hipEventSynchronize(e1));
                        float ms = 0.f;
                        HALA_HIP(hipEventElapsedTime(&ms, e0, e1));
                        tbest = std::min(tbest, ms);
                    }
                    if (tbest < best) {
                        best = tbest;
                        bt = tm;
                        bw = wg;
                    }
                }
        } catch (...) {
            (void)hipEventDestroy(e0);
            (void)hipEventDestroy(e1);
            throw;
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        B->team = bt;
        B->wg_per_cu = bw;
        if (team_out) *team_out = bt;
        if (wg_out) *wg_out = bw;
        if (ms_out) *ms_out = best;
    });
}

}  // extern "C"
