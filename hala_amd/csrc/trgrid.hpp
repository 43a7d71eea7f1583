// trgrid.hpp -- triangular sweeps of complete 5-point (2-D) and 7-point (3-D)
// grid patterns as register wavefronts.
//
// A plan whose rows are the points (i, j, k) of an nx x ny x nz grid in natural
// order (row = i + nx j + nx ny k) and whose row depends on exactly its in-grid
// neighbours at i-1, j-1 and k-1 (backward plans: the mirrored grid) is swept
// line by line.  A wavefront owns a tile of 8 x 8 lines (64 x 1 in 2-D), one
// lane per line, and a lane computes one row of its line per step, row (i, j, k)
// at step i + a + b (a, b: its line's place in the tile).  The i-1 value is
// then the lane's own previous result, the j-1 value its left neighbour's
// previous result (a DPP move), the k-1 value another lane's previous result,
// through LDS; nothing but that and a few FP operations lies between one step
// and the next, and no barrier is needed.
//
// From i + a + b follow: a tile takes S >= nx + LAG steps, LAG = (TJ - 1) + (TK
// - 1) its last line's start; a value that crosses a tile boundary is formed TJ
// - 1 = TK - 1 steps of its tile after the step that reads it (2-D: TJ - 1), and
// is staged beside the results of the step before the one that reads it (k - 1)
// or of that step (j - 1).
//
// Vectors live in the packed order of the tiles' steps: element
// ((tile * S) + step) * 64 + lane.  A backward plan runs the same kernel on the
// mirrored grid, whose packed order is the forward one reversed, so an ILU's
// two sweeps share one order and need no permutation between them.
#pragma once
#include <vector>

#include "common.hpp"

namespace hala_amd {

struct tri_plan;

struct grid_geom {
    int nx = 0, ny = 0, nz = 0;   // nz == 1: 2-D
    int ntj = 0, ntk = 0, S = 0;  // tiles along j and k, steps per tile
    int64_t N = 0;                // packed elements of a vector
    bool same(const grid_geom &o) const { return nx == o.nx && ny == o.ny && nz == o.nz; }
};

// Buffers of `rhs` vectors in a sweep's order, made on first use: input, output and (grid sweeps) frames, the
// boundary results that the tiles poll, sentinels before a sweep.
struct sweep_vecs {
    dbuf in, out, fr;
    int rhs = 0;
    bool pinned = false;     // a stream capture recorded work on them,
    std::vector<dbuf> kept;  // ... so what larger ones replace stays until the plan goes
    // What a plan keeps for the next call of several vectors; more is given back at the end of the call.
    static constexpr size_t KEEP = size_t(1) << 30;
    void give_back() {
        if (!pinned && in.bytes + out.bytes + fr.bytes > KEEP) drop();
    }
    // for larger ones to take their place
    void drop() {
        if (pinned)
            for (dbuf *b : {&in, &out, &fr})
                if (b->p) kept.emplace_back(std::move(*b));
        in.release();
        out.release();
        fr.release();
        rhs = 0;
        pinned = false;
    }
};

// The grid side of a plan (member of tri_plan).
struct tri_gridplan {
    bool ok = false;
    bool thin = false;  // one vector runs faster on the column sweep (see grid_layout)
    bool zyx = true;  // a row's terms in the order k-1, j-1, i-1 (else i-1, j-1, k-1)
    grid_geom g;
    dbuf slot;          // packed element (forward order) of every natural row, then the tile of every ticket
    dbuf rec64, rec32;  // per (tile, step) the step's coefficients and diagonal (see grid_pack)
    sweep_vecs one64, one32, many64, many32;
    // Several vectors have buffers of their own: those of one vector never move, whatever else the plan
    // solves (a captured apply holds their addresses).
    sweep_vecs &vecs(bool is64, int nrhs) { return nrhs > 1 ? (is64 ? many64 : many32) : (is64 ? one64 : one32); }
};

// Recognises p's pattern from its dependency lists and lays the grid plan out (p.grid.ok tells), in three
// steps that ride on the analysis's own synchronisations (four of their own cost 55 us per triangle):
// grid_probe, which also returns the device word the analysis waits for there; grid_layout (false: no grid),
// launches only; after the next synchronisation grid_finish.
int grid_probe(hala_ctx c, tri_plan &p, const int *word);
bool grid_layout(hala_ctx c, tri_plan &p);
void grid_finish(hala_ctx c, tri_plan &p);
// The factor's values into the step records of one precision.
void grid_load_values(hala_ctx c, tri_plan &p, const double *factor, bool f32);
void grid_reserve_values(tri_plan &p, bool f32);
// The plan runs nrhs vectors on the grid sweep (pattern, options).
bool grid_usable(hala_ctx c, const tri_plan &p, int nrhs = 1);
// ... and so does second, in first's packed order (an ILU's two triangles).
bool grid_pair_usable(hala_ctx c, const tri_plan &first, const tri_plan &second, int nrhs = 1);
// Packed vectors and frames for nrhs right-hand sides of a plan swept alone or in a pair.
enum grid_role { GRID_ALONE, GRID_FIRST, GRID_SECOND };
void grid_reserve(hala_ctx c, tri_plan &p, bool is64, int nrhs, grid_role role);
inline void grid_reserve_pair(hala_ctx c, tri_plan &first, tri_plan &second, bool is64, int nrhs) {
    grid_reserve(c, first, is64, nrhs, GRID_FIRST);
    grid_reserve(c, second, is64, nrhs, GRID_SECOND);
}

// out_k = op^-1 in_k for nrhs vectors in natural order (element r of vector k at in[k ldin + r inc] and
// out[k ldout + r inc]; out may be in), TRI_SUB / TRI_SUM as tri_exec.
template <class T, class TIO>
void grid_exec(hala_ctx c, tri_plan &p, int mode, T alpha, const TIO *in, int64_t ldin, TIO *out, int64_t ldout,
               int nrhs, const int *gate, int64_t inc = 1);
// The two sweeps of an apply (TRI_SUB, first forward, second backward or the
// reverse), natural order in and out.  Plans run as a pair are only run as one.
template <class T, class TIO>
void grid_exec_pair(hala_ctx c, tri_plan &first, tri_plan &second, const TIO *in, int64_t ldin, TIO *out,
                    int64_t ldout, int nrhs, const int *gate);
// The pair without its ends: first's packed input (filled by the caller) to
// second's packed output, both by first's slot map.
void grid_pair_mid64(hala_ctx c, tri_plan &first, tri_plan &second, int nrhs, const int *gate);

}  // namespace hala_amd
