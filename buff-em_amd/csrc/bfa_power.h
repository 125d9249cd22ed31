// bfa_power.h -- scattered power from tetrahedron currents (bfa_power.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>

#include "bfa_internal.h"

namespace bfa {
// 32 x 32 tiles of tetrahedron pairs S <= T
int emt_tiles(int nt);
// doubles of work space for npw right-hand sides
size_t emt_work_doubles(int nt, int npw);
// out[j] (device) = Re(J^H Q J) + sum_a |J_a|^2 Q_aa of each right-hand side
void launch_emt_scattered(const DevGeom &g, double omega, const void *J, int64_t ldj, int npw, double *work,
                          double *out, hipStream_t st);
}  // namespace bfa
