// gvh_state.h -- launchers of the state transfer kernels (gvh_state.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace gvh {

struct Extent {
  long long G;  // ghosted cells, below 2^29
  int nx, ny, nz, ncx, ncy;
};
// Device copies of the primitive fields on the interior lattice; pi and Pi
// may be null for zero.
struct InitialFields {
  const double *e, *p, *u[4], *pi[10], *Pi;
};
struct StateBlocks {
  double *q, *e, *p, *u, *up;
};

// spatial_pi: pi^{xx} .. pi^{nn} only; otherwise everything else.
hipError_t launch_state(const InitialFields &F, const StateBlocks &B, const Extent &X, bool mixed,
                        bool spatial_pi, hipStream_t st);
// Block of G floats or doubles as doubles: all of it, or the interior.
hipError_t launch_pack(const void *block, bool is_float, const Extent &X, bool all, double *out,
                       hipStream_t st);

}  // namespace gvh
