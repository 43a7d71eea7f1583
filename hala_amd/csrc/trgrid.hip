// trgrid.hip -- register-wavefront sweeps of complete 5- and 7-point grid
// triangles (see trgrid.hpp for the schedule).
//
// What bounds a sweep: its steps and its tile-to-tile hops, one after the
// other (128^3: 382 steps and 30 hops).  A step takes 79 ns in L and 111 ns in
// U (division; one wavefront: 33 ns without its LDS reads, 62 ns with them, the
// rest is the pace of the streaming wave), a hop about 1.4 us (a boundary value
// stored at agent scope, seen by the neighbour's poll one memory round trip
// later, staged, read).  FP64 applies with their gather and scatter, against
// the column-blocked sweeps: 128^3 7-point 196 against 344 us, 64^3 88 against
// 135 us, 127^2 5-point 60 against 125 us, 250^2 111 against about 230 us.
// Tiles of 8 x 8 lines make the fewest hops of a 64-lane tile; the k lag is
// one step although its value comes through LDS (a lag of two takes 509 steps
// of the same length: 272 us on 128^3 when the lag of one took 241).
#include <algorithm>
#include <climits>

#include "tile_order.hpp"
#include "trsolve.hpp"

namespace hala_amd {

namespace {

// Tile shapes.  LAG: the step at which the last line of a tile starts.
template <int DIM>
struct gtile {
    static constexpr int TJ = DIM == 3 ? 8 : 64, TK = DIM == 3 ? 8 : 1;
    static constexpr int LAG = (TJ - 1) + (TK - 1);
    // Boundary results ("frame") of one step of a tile, polled by the tiles
    // behind.  3-D: 16 values, the line row b = TK - 1 by ascending a at 0..7,
    // the line row a = TJ - 1 by descending b at 7..14 (their common line
    // once).  2-D: the last line's value.
    static constexpr int FR = DIM == 3 ? 16 : 1;
    // lanes that poll one step (3-D: 4 for the k-1 tile's row, 4 for the j-1 tile's, two values each)
    static constexpr int LPS = DIM == 3 ? 8 : 1, FV = DIM == 3 ? 2 : 1;
    // ring of steps in LDS: per step the 64 results (read by the next step as the
    // k-1 values) and the frame values (2-D: the frame value alone)
    static constexpr int SLOT = DIM == 3 ? 64 + 16 : 1;
    static constexpr int R = DIM == 3 ? 32 : 256;
    static constexpr int CH = 8;  // steps per unrolled chunk; S is a multiple of it
};
constexpr int RL = 16;            // staged steps (records and input) in LDS = streamed steps in flight
// Frame polls in flight.  One load looks at 64 / LPS steps; two loads in flight
// halve the wait for a value that has just landed (a round trip is about 0.6 us
// here), more only queue behind the poller's own instructions.
constexpr int POLL_ROUNDS = 2;

// A lane's line (a, b) in its tile.  In 3-D the two k of a pair alternate, so
// that the j-1 neighbour is two lanes to the left in a row of 16 lanes and the
// lanes without one are the row's first two, which is what a DPP row shift
// leaves alone.  (a, b) -> (TJ-1-a, TK-1-b) reverses the lanes.
template <int DIM>
__host__ __device__ __forceinline__ int lane_a(int l) {
    return DIM == 3 ? (l & 15) >> 1 : l;
}
template <int DIM>
__host__ __device__ __forceinline__ int lane_b(int l) {
    return DIM == 3 ? (l >> 4) * 2 + (l & 1) : 0;
}
__host__ __device__ __forceinline__ int lane_of(int dim, int a, int b) {
    return dim == 3 ? (b >> 1) * 16 + 2 * a + (b & 1) : a;
}

int lag_of(int dim) { return dim == 3 ? gtile<3>::LAG : gtile<2>::LAG; }

// ---- detection and layout ---------------------------------------------------

struct gdims {
    int nx, ny, nz, backward, TJ, TK, ntj, ntk, S, lag;
};

// Lines of the mirrored grid are counted from the padded end, so that a
// backward tile holds the same lines as the forward one, in reverse.
__device__ __forceinline__ int padded(int m, int t) { return (m + t - 1) / t * t; }

// flag bit 0 / 1: some row's dependencies are not its in-grid neighbours in
// the order k, j, i / i, j, k.  The packed element (forward order) of every
// natural row, and behind them the tile of every ticket.
__global__ __launch_bounds__(256) void grid_check(gdims d, int n, const int *__restrict__ dptr,
                                                  const int *__restrict__ ddep, int *__restrict__ flag,
                                                  int *__restrict__ slot) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < d.ntj * d.ntk) slot[n + tile_ticket(r % d.ntj, r / d.ntj, d.ntj, d.ntk)] = r;
    unsigned bad = 0;
    if (r < n) {
        const int P = d.nx * d.ny;
        const int i = r % d.nx, j = (r / d.nx) % d.ny, k = r / P;
        const int ta = j % d.TJ, tb = k % d.TK;
        slot[r] = (((k / d.TK) * d.ntj + j / d.TJ) * d.S + i + ta + tb) * WAVE + lane_of(d.nz > 1 ? 3 : 2, ta, tb);
        const int s = d.backward ? 1 : -1;
        const bool hx = d.backward ? i < d.nx - 1 : i > 0;
        const bool hy = d.backward ? j < d.ny - 1 : j > 0;
        const bool hz = d.backward ? k < d.nz - 1 : k > 0;
        const int a = dptr[r], m = dptr[r + 1] - a;
        if (m != (int)hx + (int)hy + (int)hz) {
            bad = 3;
        } else {
            int q = a;
            if (hz && ddep[q++] != r + s * P) bad |= 1;
            if (hy && ddep[q++] != r + s * d.nx) bad |= 1;
            if (hx && ddep[q++] != r + s) bad |= 1;
            q = a;
            if (hx && ddep[q++] != r + s) bad |= 2;
            if (hy && ddep[q++] != r + s * d.nx) bad |= 2;
            if (hz && ddep[q++] != r + s * P) bad |= 2;
        }
    }
    // at most one atomic per wavefront and bit, none once the flag holds it
    const unsigned w = (__any(bad & 1) ? 1u : 0u) | (__any(bad & 2) ? 2u : 0u);
    if ((threadIdx.x & (WAVE - 1)) == 0 && w && (w & ~(unsigned)ld_agent(flag))) atomicOr(flag, (int)w);
}

// Step records, processing order: per (tile, step) the terms' coefficients as
// pairs [64] (3-D: k-1 and j-1, 2-D: j-1 and i-1), then per lane the i-1
// coefficient (3-D) and the diagonal (non-unit).  Absent terms and rows off the
// grid hold 0 (diagonal 1).
template <int DIM, class V>
__global__ __launch_bounds__(256) void grid_pack(gdims d, int zyx, int unit, int nstep, const int *__restrict__ dptr,
                                                 const int *__restrict__ dsrc, const int *__restrict__ diag_src,
                                                 const double *__restrict__ f, V *__restrict__ rec) {
    const int ts = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (ts >= nstep) return;
    const int tile = ts / d.S, s = ts % d.S;
    const int a = lane_a<DIM>(lane), b = lane_b<DIM>(lane);
    const int i = s - a - b - (d.backward ? d.S - (d.nx + d.lag) : 0);
    int j = (tile % d.ntj) * d.TJ + a, k = (tile / d.ntj) * d.TK + b, in = i;
    if (d.backward) {
        j = d.ntj * d.TJ - 1 - j;
        k = d.ntk * d.TK - 1 - k;
        in = d.nx - 1 - i;
    }
    V cx = V(0), cy = V(0), cz = V(0), dg = V(1);
    if (i >= 0 && i < d.nx && j >= 0 && j < d.ny && k >= 0 && k < d.nz) {
        const int r = in + d.nx * (j + d.ny * k);
        const bool hx = i > 0;
        const bool hy = d.backward ? j < d.ny - 1 : j > 0;
        const bool hz = d.backward ? k < d.nz - 1 : k > 0;
        int q = dptr[r];
        if (zyx) {
            if (hz) cz = (V)f[dsrc[q++]];
            if (hy) cy = (V)f[dsrc[q++]];
            if (hx) cx = (V)f[dsrc[q++]];
        } else {
            if (hx) cx = (V)f[dsrc[q++]];
            if (hy) cy = (V)f[dsrc[q++]];
            if (hz) cz = (V)f[dsrc[q++]];
        }
        if (!unit) dg = (V)f[diag_src[r]];
    }
    const int W2 = (DIM == 3 ? 1 : 0) + (unit ? 0 : 1);
    V *o = rec + (size_t)ts * WAVE * (2 + W2);
    o[2 * lane] = DIM == 3 ? cz : cy;
    o[2 * lane + 1] = DIM == 3 ? cy : cx;
    V *e = o + 2 * WAVE + lane * W2;
    if (DIM == 3) *e++ = cx;
    if (!unit) *e = dg;
}

template <class T>
__global__ void grid_arm(T *__restrict__ x, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        x[i] = sentinel<T>();
}

// natural -> packed; a thread per row, XCD-contiguous (a line of the packed
// order holds rows of 8 lines, stored by different workgroups).  arm
// (nullable): nf values per vector refilled with sentinels (the sweep's frames).
template <class T, class TIN>
__global__ __launch_bounds__(256) void grid_gather(int n, int64_t N, const int *__restrict__ slot,
                                                   const TIN *__restrict__ in, int64_t ldin, int64_t inc,
                                                   T *__restrict__ xp, T *__restrict__ arm, int64_t nf, const int *gate) {
    if (gate && *gate) return;
    const int r = xcd_block((n + 255) / 256) * 256 + threadIdx.x;
    const int64_t o = (int64_t)blockIdx.y * N;
    if (r < n) xp[o + slot[r]] = (T)in[(int64_t)blockIdx.y * ldin + r * inc];
    if (arm)
        for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nf; e += (int64_t)gridDim.x * 256)
            arm[(int64_t)blockIdx.y * nf + e] = sentinel<T>();
}

// packed -> natural
template <class T, class TOUT>
__global__ __launch_bounds__(256) void grid_scatter(int n, int64_t N, const int *__restrict__ slot,
                                                    const T *__restrict__ xp, TOUT *__restrict__ out, int64_t ldout,
                                                    int64_t inc, const int *gate) {
    if (gate && *gate) return;
    const int r = xcd_block((n + 255) / 256) * 256 + threadIdx.x;
    if (r < n) out[(int64_t)blockIdx.y * ldout + r * inc] = (TOUT)xp[(int64_t)blockIdx.y * N + slot[r]];
}

// ---- the sweep --------------------------------------------------------------

template <class V>
struct gsweep_args {
    int nx, ntj, S, ntiles, nrhs;
    int pad;                 // steps before the tile's first line starts (backward: the rounding of S)
    int jlo, jhi, klo, khi;  // lines on the grid, in processing coordinates
    long long N;
    const int *order;
    const V *rec;
    const V *in;   // packed, forward order
    V *out;        // packed, forward order
    V *frame;      // boundary results, per tile and step (processing order); polled
    V *rearm;      // another sweep's frames, refilled with sentinels
    V alpha;
    unsigned *ticket;  // [0] tiles taken, [1] workgroups done
    int *err;
    const int *gate;
};

constexpr unsigned GRID_SPIN_LIMIT = 1u << 22;

// Waits until an LDS progress counter (two: the smaller of a pair 64 words
// apart) reaches want and returns it (want after GRID_SPIN_LIMIT polls, with bad
// set).  One asm block, so that the compiler's own counting of the LDS
// operations in flight around it stays exact.
__device__ __forceinline__ int lds_wait_ge(const int *flag, int want, bool &bad) {
    const unsigned addr = (unsigned)(size_t)(__attribute__((address_space(3))) const int *)flag;
    int v, s, cnt;
    asm volatile(
        "s_mov_b32 %[cnt], %[lim]\n"
        "Lgw%=:\n"
        "ds_read_b32 %[v], %[a]\n"
        "s_waitcnt lgkmcnt(0)\n"
        "v_readfirstlane_b32 %[s], %[v]\n"
        "s_cmp_ge_i32 %[s], %[w]\n"
        "s_cbranch_scc1 Lgd%=\n"
        "s_sub_u32 %[cnt], %[cnt], 1\n"
        "s_cmp_lg_u32 %[cnt], 0\n"
        "s_cbranch_scc1 Lgw%=\n"
        "Lgd%=:\n"
        : [v] "=&v"(v), [s] "=&s"(s), [cnt] "=&s"(cnt)
        : [a] "v"(addr), [w] "s"(want), [lim] "i"(GRID_SPIN_LIMIT)
        : "memory", "scc");
    if (s < want) {
        bad = true;
        s = want;
    }
    return s;
}
__device__ __forceinline__ int lds_wait_pair(const int *pair, int want, bool &bad) {
    const unsigned addr = (unsigned)(size_t)(__attribute__((address_space(3))) const int *)pair;
    int v, v1, s, cnt;
    asm volatile(
        "s_mov_b32 %[cnt], %[lim]\n"
        "Lgw%=:\n"
        "ds_read_b32 %[v], %[a]\n"
        "ds_read_b32 %[v1], %[a] offset:256\n"
        "s_waitcnt lgkmcnt(0)\n"
        "v_min_i32 %[v], %[v], %[v1]\n"
        "s_nop 1\n"  // a VALU result read by v_readfirstlane needs a wait state
        "v_readfirstlane_b32 %[s], %[v]\n"
        "s_cmp_ge_i32 %[s], %[w]\n"
        "s_cbranch_scc1 Lgd%=\n"
        "s_sub_u32 %[cnt], %[cnt], 1\n"
        "s_cmp_lg_u32 %[cnt], 0\n"
        "s_cbranch_scc1 Lgw%=\n"
        "Lgd%=:\n"
        : [v] "=&v"(v), [v1] "=&v"(v1), [s] "=&s"(s), [cnt] "=&s"(cnt)
        : [a] "v"(addr), [w] "s"(want), [lim] "i"(GRID_SPIN_LIMIT)
        : "memory", "scc");
    if (s < want) {
        bad = true;
        s = want;
    }
    return s;
}

// A progress counter is 64 copies of a word, so that a wave publishes it with
// one plain store.  (A wave's LDS operations take effect in order: what the
// counter stands for has landed when it does.)
__device__ __forceinline__ void lds_publish(int *flag, int v, int lane) {
    __asm__ __volatile__("" ::: "memory");
    __hip_atomic_store(flag + lane, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// the neighbour's value by a DPP shift (CTRL); lanes the shift has no source for keep old
template <int CTRL>
__device__ __forceinline__ double dpp_shr(double old, double src) {
    const long long o = __double_as_longlong(old), s = __double_as_longlong(src);
    const int lo = __builtin_amdgcn_update_dpp((int)o, (int)s, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(s >> 32), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
template <int CTRL>
__device__ __forceinline__ float dpp_shr(float old, float src) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(src), CTRL, 0xf, 0xf, false));
}
constexpr int DPP_ROW_SHR2 = 0x112, DPP_WAVE_SHR1 = 0x138;

// Agent-scope store at a byte offset from a buffer's base; lanes with an
// offset past its end store nothing (no change of the exec mask).
__device__ __forceinline__ void st_agent_buf(__amdgpu_buffer_rsrc_t r, int off, double v) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, off, 0, 16);
}
__device__ __forceinline__ void st_agent_buf(__amdgpu_buffer_rsrc_t r, int off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, 16);
}

// Agent-scope load of W (8, 16 or 4 bytes) at a byte offset; each value of W is one aligned word of the
// memory system.
template <class W>
__device__ __forceinline__ W ld_agent_buf(__amdgpu_buffer_rsrc_t r, int off) {
    constexpr int AUX = 16;
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    if constexpr (sizeof(W) == 16) return __builtin_bit_cast(W, (u4)__builtin_amdgcn_raw_buffer_load_b128(r, off, 0, AUX));
    else if constexpr (sizeof(W) == 8) return __builtin_bit_cast(W, (u2)__builtin_amdgcn_raw_buffer_load_b64(r, off, 0, AUX));
    else return __builtin_bit_cast(W, (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, AUX));
}

// A workgroup sweeps one tile with three waves, so that each wave's waits
// count one kind of traffic only:
//   compute:  one row per lane and step.  The step's operands are read from
//             LDS during the step before; a step then is two DPP moves, the
//             terms in the plan's order, the diagonal, and the stores.
//   streamer: the step records and the input, RL steps ahead, into LDS.
//   poller:   the neighbouring tiles' boundary results (value as flag).  Each
//             round polls a window of steps at once, stages the leading
//             complete ones and publishes their count.
// Tiles are taken by ticket in dependency order (a tile waits only for tiles
// of lower tickets, which are running or done); all waits are bounded.
// Rows off the grid compute 0, so an absent neighbour's term is 0 * 0.
template <int DIM, bool BWD, bool ZYX, bool UNIT, int MODE, class V>
__global__ __launch_bounds__(192) void grid_sweep_kernel(gsweep_args<V> A) {
    using G = gtile<DIM>;
    constexpr int TJ = G::TJ, CH = G::CH, R = G::R, SLOT = G::SLOT;
    constexpr int W2 = (DIM == 3 ? 1 : 0) + (UNIT ? 0 : 1);  // record values per lane after the pair
    constexpr int W2A = W2 > 0 ? W2 : 1;
    typedef V v2 __attribute__((ext_vector_type(2)));
    typedef V vw __attribute__((ext_vector_type(W2A)));
    if (A.gate && *A.gate) return;
    __shared__ __align__(16) v2 s_pair[RL][WAVE];
    // W2 == 1: the value and the input as one pair
    constexpr bool WI = W2 == 1;
    __shared__ __align__(16) v2 s_wi[WI ? RL : 1][WAVE];
    __shared__ __align__(16) vw s_w2[W2 > 1 ? RL : 1][WAVE];
    __shared__ V s_in[WI ? 1 : RL][WAVE];
    __shared__ __align__(16) V s_ring[R * SLOT];
    // steps staged by the streamer and by the poller, steps done by the compute wave
    __shared__ int s_av[2 * WAVE], s_cons[WAVE], s_tk;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (threadIdx.x == 0) {
        s_tk = (int)atomicAdd(A.ticket, 1u);
    }
    if (threadIdx.x < WAVE) {
        s_av[threadIdx.x] = 0;
        s_av[WAVE + threadIdx.x] = 0;
        s_cons[threadIdx.x] = 0;
    }
    for (int e = threadIdx.x; e < R * SLOT; e += 192) s_ring[e] = V(0);
    __syncthreads();
    const int tk = s_tk;
    const int tile = A.order[tk / A.nrhs], rhs = tk % A.nrhs;
    const int tj = tile % A.ntj, tkk = tile / A.ntj;
    const int S = A.S;
    const long long vec = (long long)rhs * A.N;
    const long long base = (long long)tile * S * WAVE;  // first packed element, processing order
    // packed element of processing position p, in the vectors' forward order
    auto fwd = [&](long long p) { return vec + (BWD ? A.N - 1 - p : p); };
    constexpr int FR = G::FR;
    const long long fvec = (long long)rhs * A.ntiles * S * FR;
    bool bad = false;

    if (wave == 1) {
        // ---------------- streamer
        static_assert(RL == 2 * CH, "halves of the staged steps are released chunk by chunk");
        const v2 *rp = reinterpret_cast<const v2 *>(A.rec) + (long long)tile * S * (WAVE * (2 + W2) / 2);
        const V *ip = A.in + fwd(base);
        v2 pr[RL];
        vw w2[RL];
        V bi[RL];
        auto issue = [&](int s, int u) {
            const int sc = min(s, S - 1);
            const v2 *p = rp + sc * (WAVE * (2 + W2) / 2);
            pr[u] = p[lane];
            if (W2 > 0) w2[u] = reinterpret_cast<const vw *>(p + WAVE)[lane];
            bi[u] = ip[(BWD ? -1 : 1) * (sc * WAVE + lane)];
        };
#pragma unroll
        for (int u = 0; u < RL; u++) {
            issue(u, u);
            __builtin_amdgcn_sched_barrier(0);
        }
        V *const rf = A.rearm + fvec + (long long)tile * S * FR;
        int cons = 0;
        auto half = [&](int s0, auto first) {
            constexpr int U0 = decltype(first)::value;
            // these slots are free once the compute wave has read the steps RL before
            if (cons < s0 - CH) cons = lds_wait_ge(s_cons, s0 - CH, bad);
#pragma unroll
            for (int v = 0; v < CH; v++) {
                const int u = U0 + v, s = s0 + v;
                s_pair[u][lane] = pr[u];
                if (WI) {
                    s_wi[u][lane] = v2{w2[u][0], bi[u]};
                } else {
                    if (W2 > 1) s_w2[u][lane] = w2[u];
                    s_in[u][lane] = bi[u];
                }
                issue(s + RL, u);
                if ((v & 3) == 3) lds_publish(s_av, s + 1 < S ? s + 1 : INT_MAX, lane);
            }
            constexpr int NA = CH * FR;  // frame values of these steps, re-armed
#pragma unroll
            for (int e = 0; e < NA; e += WAVE)
                if (NA >= WAVE || lane < NA) rf[s0 * FR + e + lane] = sentinel<V>();
        };
        for (int s0 = 0; s0 < S; s0 += RL) {
            half(s0, std::integral_constant<int, 0>());
            if (s0 + CH < S) half(s0 + CH, std::integral_constant<int, CH>());
        }
        if (bad && lane == 0) atomicOr(A.err, 1);
        return;
    }

    if (wave == 2) {
        // ---------------- poller
        constexpr int LPS = G::LPS, SPB = WAVE / LPS, FV = G::FV;  // lanes per step, steps per load
        constexpr int NR = POLL_ROUNDS;
        const int sub = lane / LPS, f = lane % LPS;
        const bool isk = DIM == 3 && f < LPS / 2;
        const bool have = isk ? tkk > 0 : tj > 0;
        if (!__any(have)) {  // no neighbour: the ring's zeros stand
            lds_publish(s_av + WAVE, INT_MAX, lane);
            return;
        }
        // the neighbour forms a value TJ - 1 = TK - 1 (2-D: TJ - 1) of its steps after this tile's step that
        // reads it; the last `off` steps read nothing and look at its last step instead
        static_assert(DIM == 2 || G::TJ == G::TK, "one offset for both neighbours");
        constexpr int off = TJ - 1, SB = FR * (int)sizeof(V);
        const int stile = isk ? tile - A.ntj : tile - 1, first = max(min(tile - A.ntj, tile - 1), 0);
        const int fv = DIM == 2 ? 0 : (isk ? 2 * f : 7 + 2 * (f - LPS / 2));  // first value of the step's frame
        const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
            A.frame + fvec + (long long)first * S * FR, 0, INT_MAX, 0x00027000);
        // (a lane without a neighbour reads past the end: 0, which is its value)
        const int srco = have ? (stile - first) * S * SB + fv * (int)sizeof(V) : INT_MIN;
        // where a step's values go: its k-1 values beside the results of the step before
        const int rofs = DIM == 2 ? 0 : WAVE + 2 * f, rlag = isk ? 1 : 0;
        typedef V vf __attribute__((ext_vector_type(FV)));
        int head = 0, cons = 0;
        vf v[NR];
        int hq[NR];  // the load's first step
        auto issue = [&](int r) {
            hq[r] = head;
            __asm__ __volatile__("" ::: "memory");  // a repeated look is a new load
            v[r] = ld_agent_buf<vf>(src, srco + min(head + sub + off, S - 1) * SB);
            // loads stay in order, so that looking at one waits for older ones only
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int r = 0; r < NR; r++) issue(r);
        // (the loop has one exit and no memory access on a side path: the
        // waits for a load stay exact counts)
        unsigned rounds = 0;
        do {
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int cnow = __hip_atomic_load(s_cons, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                const unsigned long long miss =
                    __builtin_amdgcn_ballot_w64(is_sent((V)v[r][0])) | __builtin_amdgcn_ballot_w64(is_sent((V)v[r][FV - 1]));
                const int lead = miss ? (int)__builtin_ctzll(miss) / LPS : SPB;
                // the ring holds R - 2 steps past those done
                const int end = min(hq[r] + lead, cons + R - 2);
                // steps below head were staged by an earlier look (and their slots may hold later steps)
                const int s = hq[r] + sub;
                if ((unsigned)(s - head) < (unsigned)(end - head) && end > head)
                    *reinterpret_cast<vf *>(s_ring + ((s - rlag) & (R - 1)) * SLOT + rofs) = v[r];
                head = max(head, end);
                lds_publish(s_av + WAVE, head < S ? head : INT_MAX, lane);
                cons = __builtin_amdgcn_readfirstlane(cnow);
                issue(r);
            }
        } while (head < S && ++rounds < GRID_SPIN_LIMIT);
        if (head < S) {  // give up: let the compute wave run on (its results are reported as an error)
            lds_publish(s_av + WAVE, INT_MAX, lane);
            if (lane == 0) atomicOr(A.err, 1);
        }
        return;
    }

    // ---------------- compute
    __builtin_amdgcn_s_setprio(3);
    const int a = lane_a<DIM>(lane), b = lane_b<DIM>(lane);
    const int jp = tj * TJ + a, kp = tkk * G::TK + b;
    const bool line = jp >= A.jlo && jp < A.jhi && kp >= A.klo && kp < A.khi;
    // row of step s: s - off, on the grid when in [0, nx)
    const int off = line ? a + b + A.pad : INT_MAX / 2;
    const bool all = __all(line);
    // LDS places of the k-1 value (in the slot of the step before) and the j-1 frame value
    const V *zrd = s_ring + (b > 0 ? lane_of(DIM, a, b - 1) : WAVE + a);
    const V *yrd = s_ring + (DIM == 3 ? WAVE + 8 + (7 - b) : 0);
    V *own = s_ring + lane;
    V *outp = A.out + fwd(base + lane);
    // the lanes on the tile's far edges also publish their results to the tiles behind
    const bool edge = DIM == 3 ? (a == TJ - 1 || b == G::TK - 1) : lane == WAVE - 1;
    const __amdgpu_buffer_rsrc_t frame =
        __builtin_amdgcn_make_buffer_rsrc(A.frame + fvec + (long long)tile * S * FR, 0, INT_MAX, 0x00027000);
    int fro = edge ? (int)sizeof(V) * (DIM == 2 ? 0 : (b == G::TK - 1 ? a : 14 - b)) : INT_MIN;
    constexpr int DIR = BWD ? -WAVE : WAVE;
    int avail;  // steps whose records, input and frame values are staged (INT_MAX: all)
    V prev = V(0);
    v2 pr[2];
    vw w2[2];
    V bi[2], yf[2];
    auto fetch = [&](int q, int rl, const V *yp) {
        pr[q] = s_pair[rl][lane];
        if (WI) {
            const v2 t = s_wi[rl][lane];
            w2[q][0] = t[0];
            bi[q] = t[1];
        } else {
            if (W2 > 1) w2[q] = s_w2[rl][lane];
            bi[q] = s_in[rl][lane];
        }
        yf[q] = *yp;
    };
    avail = lds_wait_pair(s_av, 1, bad);
    fetch(0, 0, yrd);
    V zv = V(0);
    if (DIM == 3) zv = zrd[(R - 1) * SLOT];
    auto chunk = [&](int s0, auto masked) {
        constexpr bool MASK = decltype(masked)::value;
        const int c0 = s0 & (R - 1), cn = (s0 + CH) & (R - 1);
        const int rl0 = s0 & (RL - 1), rln = (s0 + CH) & (RL - 1);
        int ahead = avail - s0;
        int a0 = 0, a1 = 0;
#pragma unroll
        for (int u = 0; u < CH; u++) {
            const int q = u & 1, s = s0 + u;
            // the progress counters, looked at once per chunk without waiting for the look
            if (u == 0) {
                a0 = __hip_atomic_load(s_av, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                a1 = __hip_atomic_load(s_av + WAVE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            if (u == 3) ahead = __builtin_amdgcn_readfirstlane(min(a0, a1)) - s0;
            // the next step's operands
            if (__builtin_expect(ahead < u + 2, 0)) ahead = lds_wait_pair(s_av, s + 2, bad) - s0;
            fetch(q ^ 1, u + 1 < CH ? rl0 + u + 1 : rln, yrd + (u + 1 < CH ? c0 + u + 1 : cn) * SLOT);
            __builtin_amdgcn_sched_barrier(0);
            V y;
            if (DIM == 3) {
                y = dpp_shr<DPP_ROW_SHR2>(yf[q], prev);
            } else {
                y = dpp_shr<DPP_WAVE_SHR1>(yf[q], prev);
            }
            const V cy = DIM == 3 ? pr[q][1] : pr[q][0];
            const V cx = DIM == 3 ? w2[q][0] : pr[q][1];
            V acc = MODE == TRI_SUB ? bi[q] : V(0);
            auto term = [&](V cc, V xx) { acc = MODE == TRI_SUB ? acc - cc * xx : acc + cc * xx; };
            if (ZYX) {
                if (DIM == 3) term(pr[q][0], zv);
                term(cy, y);
                term(cx, prev);
            } else {
                term(cx, prev);
                term(cy, y);
                if (DIM == 3) term(pr[q][0], zv);
            }
            if (MODE == TRI_SUM) acc = A.alpha * bi[q] - acc;
            if (!UNIT) acc = acc / w2[q][W2A - 1];
            if (MASK) acc = (unsigned)(s - off) < (unsigned)A.nx ? acc : V(0);
            prev = acc;
            if (DIM == 3) {  // the result, and at once the next step's k-1 value from its slot
                own[(c0 + u) * SLOT] = acc;
                zv = zrd[(c0 + u) * SLOT];
                __builtin_amdgcn_sched_barrier(0);
            }
            st_agent_buf(frame, fro + u * FR * (int)sizeof(V), acc);
            outp[u * DIR] = acc;
        }
        outp += CH * DIR;
        fro += CH * FR * (int)sizeof(V);
        avail = ahead + s0;
        // every LDS read of the chunk's steps has been waited for but the last fetch (step s0 + CH)
        lds_publish(s_cons, s0 + CH, lane);
    };
    for (int s0 = 0; s0 < S; s0 += CH) {
        if (all && s0 >= G::LAG + A.pad && s0 + CH <= A.nx + A.pad) chunk(s0, std::false_type());
        else chunk(s0, std::true_type());
    }
    if (lane == 0) {
        if (bad) atomicOr(A.err, 1);
        const unsigned dn = atomicAdd(A.ticket + 1, 1u);
        if (dn == gridDim.x - 1) {  // the last workgroup to finish re-arms the counters
            st_agent(A.ticket, 0u);
            st_agent(A.ticket + 1, 0u);
        }
    }
}

gdims dims_of(const tri_plan &p) {
    const grid_geom &g = p.grid.g;
    const int dim = g.nz > 1 ? 3 : 2;
    return gdims{g.nx, g.ny, g.nz, p.backward ? 1 : 0, dim == 3 ? 8 : 64, dim == 3 ? 8 : 1, g.ntj, g.ntk, g.S,
                 lag_of(dim)};
}

template <class V>
size_t rec_values(const tri_plan &p) {
    const grid_geom &g = p.grid.g;
    return (size_t)g.N * (2 + (g.nz > 1 ? 1 : 0) + (p.unit ? 0 : 1));
}

template <int DIM, bool BWD, bool ZYX, bool UNIT, class V>
void launch_mode(hala_ctx c, int mode, const gsweep_args<V> &a) {
    const int wg = a.ntiles * a.nrhs;
    if (mode == TRI_SUB) grid_sweep_kernel<DIM, BWD, ZYX, UNIT, TRI_SUB, V><<<wg, 192, 0, c->stream>>>(a);
    else grid_sweep_kernel<DIM, BWD, ZYX, UNIT, TRI_SUM, V><<<wg, 192, 0, c->stream>>>(a);
}
template <int DIM, bool BWD, class V>
void launch_order(hala_ctx c, const tri_plan &p, int mode, const gsweep_args<V> &a) {
    if constexpr (BWD) {
        if (!p.grid.zyx) {
            if (p.unit) launch_mode<DIM, true, false, true, V>(c, mode, a);
            else launch_mode<DIM, true, false, false, V>(c, mode, a);
            return;
        }
    }
    if (p.unit) launch_mode<DIM, BWD, true, true, V>(c, mode, a);
    else launch_mode<DIM, BWD, true, false, V>(c, mode, a);
}

// One sweep over nrhs packed vectors: in -> out through frames `frame` (all
// sentinels at launch); rearm: another frame buffer, refilled with sentinels.
template <class V>
void sweep(hala_ctx c, const tri_plan &p, int mode, V alpha, const V *in, V *out, V *frame, V *rearm, int nrhs,
           const int *gate) {
    const tri_gridplan &q = p.grid;
    const grid_geom &g = q.g;
    const int dim = g.nz > 1 ? 3 : 2, TJ = dim == 3 ? 8 : 64, TK = dim == 3 ? 8 : 1;
    c->path[PATH_SWEEP] = 2;
    gsweep_args<V> a;
    a.nx = g.nx;
    a.ntj = g.ntj;
    a.S = g.S;
    a.ntiles = g.ntj * g.ntk;
    a.nrhs = nrhs;
    a.pad = p.backward ? g.S - (g.nx + lag_of(dim)) : 0;
    a.jlo = p.backward ? g.ntj * TJ - g.ny : 0;
    a.jhi = p.backward ? g.ntj * TJ : g.ny;
    a.klo = p.backward ? g.ntk * TK - g.nz : 0;
    a.khi = p.backward ? g.ntk * TK : g.nz;
    a.N = g.N;
    a.order = q.slot.as<int>() + p.n;
    a.rec = sizeof(V) == 8 ? reinterpret_cast<const V *>(q.rec64.p) : reinterpret_cast<const V *>(q.rec32.p);
    a.in = in;
    a.out = out;
    a.frame = frame;
    a.rearm = rearm;
    a.alpha = alpha;
    a.ticket = counters(c) + 104;
    a.err = wait_error_flag(c);
    a.gate = gate;
    if (dim == 3) {
        if (p.backward) launch_order<3, true, V>(c, p, mode, a);
        else launch_order<3, false, V>(c, p, mode, a);
    } else {
        if (p.backward) launch_order<2, true, V>(c, p, mode, a);
        else launch_order<2, false, V>(c, p, mode, a);
    }
    HALA_CHECK_LAUNCH();
}

// polled boundary values of one vector
int64_t frame_values(const grid_geom &g) {
    return (int64_t)g.ntj * g.ntk * g.S * (g.nz > 1 ? gtile<3>::FR : gtile<2>::FR);
}

}  // namespace

// What grid_probe reads back: dependency count of the row swept last, their distances, a word of the
// caller's; then the check's flag (host side: at PROBE_HOST doubles into the landing zone, past what other
// read-backs use).
constexpr int PROBE_WORDS = 5, PROBE_HOST = 1000;
static int *probe_dev(hala_ctx c) { return reinterpret_cast<int *>(c->scal.as<double>() + S_DOT + 10); }

static __global__ void grid_probe_kernel(int corner, const int *__restrict__ dptr, const int *__restrict__ ddep,
                                         const int *__restrict__ word, int *__restrict__ out) {
    const int a = dptr[corner], m = dptr[corner + 1] - a;
    out[0] = m;
    for (int k = 0; k < 3; k++) out[1 + k] = k < m ? abs(ddep[a + k] - corner) : 0;
    out[4] = *word;
    out[PROBE_WORDS] = 0;
}

int grid_probe(hala_ctx c, tri_plan &p, const int *word) {
    p.grid.ok = false;
    // the last row swept has every neighbour: its offsets are 1, nx (and nx ny)
    grid_probe_kernel<<<1, 1, 0, c->stream>>>(p.backward ? 0 : p.n - 1, p.dptr.as<int>(), p.ddep.as<int>(), word,
                                                probe_dev(c));
    HALA_CHECK_LAUNCH();
    HALA_HIP(hipMemcpyAsync(c->host_pinned + PROBE_HOST, probe_dev(c), PROBE_WORDS * sizeof(int), hipMemcpyDeviceToHost,
                            c->stream));
    HALA_HIP(hipStreamSynchronize(c->stream));
    int v;
    std::memcpy(&v, reinterpret_cast<const int *>(c->host_pinned + PROBE_HOST) + 4, sizeof(int));
    return v;
}

bool grid_layout(hala_ctx c, tri_plan &p) {
    tri_gridplan &q = p.grid;
    const int n = p.n;
    if (n < 4) return false;
    int h[PROBE_WORDS];
    std::memcpy(h, c->host_pinned + PROBE_HOST, sizeof(h));
    const int m = h[0];
    if (m != 2 && m != 3) return false;
    int *o = h + 1;  // m of them
    std::sort(o, o + m);
    grid_geom g;
    if (o[0] != 1 || o[1] < 2) return false;
    g.nx = o[1];
    const int P = m == 3 ? o[2] : n;
    if (P % g.nx != 0 || n % P != 0) return false;
    g.ny = P / g.nx;
    g.nz = n / P;
    if (g.ny < 2 || (m == 3 && g.nz < 2)) return false;
    const int dim = m, TJ = dim == 3 ? 8 : 64, TK = dim == 3 ? 8 : 1;
    g.ntj = (g.ny + TJ - 1) / TJ;
    g.ntk = (g.nz + TK - 1) / TK;
    g.S = (g.nx + lag_of(dim) + 7) / 8 * 8;
    g.N = (int64_t)g.ntj * g.ntk * g.S * WAVE;
    // Tiles of short lines or few lanes are mostly padding.  That costs memory, 32 bytes of record per packed
    // element, so past 2^23 elements (256 MiB of records) a grid has to fill a third of them; it does not cost
    // time, a step takes what it takes.  Applies, columns -> grid: 2 x 20000 (36 elements per row) 7407 -> 4314
    // us, 20000 x 8 (8) 8131 -> 3698, 20 x 60000 (4.4) 31164 -> 13781, 2 x 300 x 300 (8) 345 -> 311, 3 x 500 x
    // 500 (8) 578 -> 562.
    if (g.N > 3 * (int64_t)n && g.N > (1 << 23)) return false;
    if (g.N > (1 << 28)) return false;  // 32-bit byte offsets into a vector's frames
    q.g = g;
    // A hop from tile to tile takes as long as about ten levels of a few rows of the column sweep (1.8 us
    // against 0.19): 3-D grids of short lines, a hop every eight levels, run one vector there.  Applies, column
    // -> grid: 8 x 8 x 4000 1538 -> 1823 us, 9 x 1000 x 9 425 -> 476, 2 x 2 x 2000 775 -> 846; wider levels
    // take the column sweep longer: 3 x 100 x 100 127 -> 124, 5 x 200 x 200 238 -> 227, 12 x 200 x 200 334 -> 237.
    // (Several vectors hide each other's hops.)
    q.thin = dim == 3 && p.col.ok && (int64_t)(g.ntj + g.ntk - 2) * 10 > p.nlev && n < 128 * (int64_t)p.nlev;
    const gdims d = dims_of(p);
    int *flag = probe_dev(c) + PROBE_WORDS;
    const int nt = g.ntj * g.ntk;
    q.slot.reserve(((size_t)n + nt) * sizeof(int));
    grid_check<<<(std::max(n, nt) + 255) / 256, 256, 0, c->stream>>>(d, n, p.dptr.as<int>(), p.ddep.as<int>(), flag,
                                                                     q.slot.as<int>());
    HALA_CHECK_LAUNCH();
    HALA_HIP(hipMemcpyAsync(c->host_pinned + PROBE_HOST, flag, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    return true;
}

void grid_finish(hala_ctx c, tri_plan &p) {
    int bad;
    std::memcpy(&bad, c->host_pinned + PROBE_HOST, sizeof(int));
    // forward plans list a row's terms by ascending column (k-1, j-1, i-1); backward ones either way
    if (bad == 3 || (!p.backward && (bad & 1))) {
        p.grid.slot.release();
        return;
    }
    p.grid.zyx = (bad & 1) == 0;
    p.grid.ok = true;
}

void grid_load_values(hala_ctx c, tri_plan &p, const double *factor, bool f32) {
    tri_gridplan &q = p.grid;
    if (!q.ok) return;
    const gdims d = dims_of(p);
    const int nstep = (int)(q.g.N / WAVE), g = (nstep + 3) / 4;
    auto pack = [&](auto zero, dbuf &rec) {
        using V = decltype(zero);
        if (q.g.nz > 1)
            grid_pack<3, V><<<g, 256, 0, c->stream>>>(d, q.zyx, p.unit, nstep, p.dptr.as<int>(), p.dsrc.as<int>(),
                                                      p.diag_src.as<int>(), factor, rec.as<V>());
        else
            grid_pack<2, V><<<g, 256, 0, c->stream>>>(d, q.zyx, p.unit, nstep, p.dptr.as<int>(), p.dsrc.as<int>(),
                                                      p.diag_src.as<int>(), factor, rec.as<V>());
        HALA_CHECK_LAUNCH();
    };
    grid_reserve_values(p, f32);
    if (f32) pack(0.0f, q.rec32);
    else pack(0.0, q.rec64);
}

void grid_reserve_values(tri_plan &p, bool f32) {
    if (!p.grid.ok) return;
    if (f32) p.grid.rec32.reserve(rec_values<float>(p) * sizeof(float));
    else p.grid.rec64.reserve(rec_values<double>(p) * sizeof(double));
}

bool grid_usable(hala_ctx c, const tri_plan &p, int nrhs) {
    const hala_options &o = c->opt;
    // the column options, where given, ask for the column sweeps
    if (!p.grid.ok || !o.tri_grid || !o.tri_col || o.tri_col_cols || o.tri_col_split) return false;
    return !(p.grid.thin && nrhs == 1);
}

bool grid_pair_usable(hala_ctx c, const tri_plan &first, const tri_plan &second, int nrhs) {
    return grid_usable(c, first, nrhs) && grid_usable(c, second, nrhs) && first.grid.g.same(second.grid.g) &&
           first.backward != second.backward;
}

void grid_reserve(hala_ctx c, tri_plan &p, bool is64, int nrhs, grid_role role) {
    sweep_vecs &v = p.grid.vecs(is64, nrhs);
    const size_t w = is64 ? sizeof(double) : sizeof(float);
    // a sweep re-arms its partner's frames, alone a spare set of its own; a pair's second reads the first's output
    const size_t e = (size_t)p.grid.g.N * w, f = (size_t)frame_values(p.grid.g) * (role == GRID_ALONE ? 2 : 1) * w;
    const bool with_in = role != GRID_SECOND;
    if (nrhs > v.rhs || (with_in && v.in.bytes < e * nrhs) || v.fr.bytes < f * nrhs) {
        if (v.rhs) HALA_HIP(hipStreamSynchronize(c->stream));  // sweeps in flight still use the smaller buffers
        v.drop();
        if (with_in) v.in.reserve(e * nrhs);
        v.out.reserve(e * nrhs);
        v.fr.reserve(f * nrhs);
        const int64_t nf = (int64_t)(f * nrhs / w);
        const int g = grid_for(nf, 256 * 4, 8192);
        if (is64) grid_arm<double><<<g, 256, 0, c->stream>>>(v.fr.as<double>(), nf);
        else grid_arm<float><<<g, 256, 0, c->stream>>>(v.fr.as<float>(), nf);
        HALA_CHECK_LAUNCH();
        v.rhs = nrhs;
    }
    if (capturing(c)) v.pinned = true;
}

template <class T, class TIO>
void grid_exec(hala_ctx c, tri_plan &p, int mode, T alpha, const TIO *in, int64_t ldin, TIO *out, int64_t ldout,
               int nrhs, const int *gate, int64_t inc) {
    tri_gridplan &q = p.grid;
    grid_reserve(c, p, sizeof(T) == 8, nrhs, GRID_ALONE);
    sweep_vecs &v = q.vecs(sizeof(T) == 8, nrhs);
    T *xp = v.in.as<T>(), *op = v.out.as<T>(), *fr = v.fr.as<T>();
    const int64_t nf = frame_values(q.g);
    const dim3 g((unsigned)xcd_grid((p.n + 255) / 256), (unsigned)nrhs);
    grid_gather<T, TIO><<<g, 256, 0, c->stream>>>(p.n, q.g.N, q.slot.as<int>(), in, ldin, inc, xp, fr, nf, gate);
    HALA_CHECK_LAUNCH();
    sweep<T>(c, p, mode, alpha, xp, op, fr, fr + nf * nrhs, nrhs, gate);
    grid_scatter<T, TIO><<<g, 256, 0, c->stream>>>(p.n, q.g.N, q.slot.as<int>(), op, out, ldout, inc, gate);
    HALA_CHECK_LAUNCH();
}

// Between calls both plans' frames are armed or second's hold the last sweep's
// values: first's sweep re-arms second's frames and second's first's.
template <class T>
static void pair_mid(hala_ctx c, tri_plan &first, tri_plan &second, int nrhs, const int *gate) {
    sweep_vecs &u = first.grid.vecs(sizeof(T) == 8, nrhs), &v = second.grid.vecs(sizeof(T) == 8, nrhs);
    T *xp = u.in.as<T>(), *yp = u.out.as<T>(), *zp = v.out.as<T>(), *f1 = u.fr.as<T>(), *f2 = v.fr.as<T>();
    sweep<T>(c, first, TRI_SUB, T(1), xp, yp, f1, f2, nrhs, gate);
    sweep<T>(c, second, TRI_SUB, T(1), yp, zp, f2, f1, nrhs, gate);
}

void grid_pair_mid64(hala_ctx c, tri_plan &first, tri_plan &second, int nrhs, const int *gate) {
    pair_mid<double>(c, first, second, nrhs, gate);
}

template <class T, class TIO>
void grid_exec_pair(hala_ctx c, tri_plan &first, tri_plan &second, const TIO *in, int64_t ldin, TIO *out,
                    int64_t ldout, int nrhs, const int *gate) {
    grid_reserve_pair(c, first, second, sizeof(T) == 8, nrhs);
    const tri_gridplan &q = first.grid;
    const dim3 g((unsigned)xcd_grid((first.n + 255) / 256), (unsigned)nrhs);
    grid_gather<T, TIO><<<g, 256, 0, c->stream>>>(first.n, q.g.N, q.slot.as<int>(), in, ldin, 1,
                                                  first.grid.vecs(sizeof(T) == 8, nrhs).in.template as<T>(), nullptr, 0,
                                                  gate);
    HALA_CHECK_LAUNCH();
    pair_mid<T>(c, first, second, nrhs, gate);
    grid_scatter<T, TIO><<<g, 256, 0, c->stream>>>(first.n, q.g.N, q.slot.as<int>(),
                                                   second.grid.vecs(sizeof(T) == 8, nrhs).out.template as<T>(), out,
                                                   ldout, 1, gate);
    HALA_CHECK_LAUNCH();
}

#define HALA_GRID(T, TIO)                                                                                           \
    template void grid_exec<T, TIO>(hala_ctx, tri_plan &, int, T, const TIO *, int64_t, TIO *, int64_t, int,        \
                                    const int *, int64_t);                                                                  \
    template void grid_exec_pair<T, TIO>(hala_ctx, tri_plan &, tri_plan &, const TIO *, int64_t, TIO *, int64_t,    \
                                         int, const int *);
HALA_GRID(double, double)
HALA_GRID(float, double)
HALA_GRID(float, float)
#undef HALA_GRID

}  // namespace hala_amd
