// tdw_resident.hpp -- the PECE step of lattices whose whole state fits in LDS.
#pragma once
#include "tdw_internal.hpp"

namespace tdw {

static constexpr int RS_NT = 1024;    // most threads per workgroup

struct RsPlan;

// plan and tables of the context's lattice (tdw_create); none where a state
// does not fit, and no error then
int resident_setup(tdw_ctx *c);
void resident_release(tdw_ctx *c);
// constant-mass H in FP64 on a lattice with a plan
bool resident_supported(const tdw_ctx *c);
// 3D lattices with a plan whose step the six passes of tdw_fused.hip do not do
// faster
bool resident_pays3d(const tdw_ctx *c);
// The step of tdw_step (same arrays, complete at its end; lap is not
// written in 3D without gradients).  The adjoint's taped step is the
// same with tape: y to y_out (NULL: in place), the partial corrector to cbuf
// (NULL: the oldest history entry), the new entry to f_next (NULL: the
// dropped oldest entry).
int resident_step(tdw_ctx *c, tdw_state *s, int it, int grad_last, tdw_tape_step *tape = nullptr,
                  tdw_complex *y_out = nullptr, double2 *cbuf = nullptr, tdw_complex *f_next = nullptr);
// 2D planes of 32 or 64 points a side: ddx, ddy and the Laplacian of m arrays
// in one pass (no result may be another's array); *done = 0 elsewhere
int plane_derivatives(tdw_ctx *c, int m, const double2 *in, double2 *ddx, double2 *ddy, double2 *lap, int *done);
// out = H in - e in with <H> of in into qpe, or with use_e the given e (qpe
// is then not written)
int resident_h(tdw_ctx *c, int n, const double2 *in, double2 *out, const double *pots, double *qpe,
               const double *use_e = nullptr);
// out = H in (out is not in); with dotw, d_dot[a] = dv Re <in_a|dotw_a>
int resident_h_only(tdw_ctx *c, int n, const double2 *in, double2 *out, const double *pots,
                    const double2 *dotw = nullptr, double *d_dot = nullptr);
}  // namespace tdw
