// cgsmall.hpp -- CG of a small system in one workgroup (cgsmall.hip).
#pragma once
#include <functional>

#include "solvers.hpp"

namespace hala_amd {

// The system fits one workgroup.
bool cg_small_fits(hala_csr A);
// Runs passes of identity (pdiag null) or Jacobi CG from the state that the
// start of run_cg left (r, p, zr in st) until done(), which synchronises and
// reads st, says so.
void cg_small_passes(hala_ctx c, hala_csr A, const double *vals, const double *pdiag, double *x, double *r, double *p,
                     cg_state *st, const std::function<int()> &done);

}  // namespace hala_amd
