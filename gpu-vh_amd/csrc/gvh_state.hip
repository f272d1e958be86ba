// gvh_state.hip -- kernels of the state transfer: primitive fields on the
// interior lattice into the ghosted device state, and one ghosted block of it
// packed for the host.
//
// Only the interior travels over the host link and the host touches each
// value once; laying out, ghost cells, conversion and T^{tau mu} are done
// here.  Built on the host, the 25 ghosted arrays of an initial state took
// 30 ms on a 101x101x51 lattice, now 4 ms, of which the link's share is 2.5;
// read back as a ghosted block and picked on the host, a field took 0.54 ms,
// now 0.32 ms.  Each kernel is one pass over HBM (0.1 ms for all of them on that
// lattice) and the link bounds the transfers.
#include "gvh_internal.h"
#include "gvh_state.h"

#pragma clang fp contract(off)

namespace gvh {
namespace {

constexpr int SBLOCK = 256;

// Ghosted cell s: its interior source (clamped), and whether it is interior
// or a face ghost (edges and corners stay zero, GhostCells.cu:15-144).
struct Source {
  long long cell;
  bool interior, face;
};
__device__ __forceinline__ Source source_of(const Extent &X, unsigned s) {
  const unsigned i = s % (unsigned)X.ncx, r = s / (unsigned)X.ncx;
  const unsigned j = r % (unsigned)X.ncy, k = r / (unsigned)X.ncy;
  auto clamp = [](unsigned g, int n, int &out) {
    const int x = (int)g - NG;
    if (x < 0 || x >= n) ++out;
    return x < 0 ? 0 : (x >= n ? n - 1 : x);
  };
  int out = 0;
  const int x = clamp(i, X.nx, out), y = clamp(j, X.ny, out), z = clamp(k, X.nz, out);
  return Source{x + (long long)X.nx * (y + (long long)X.ny * z), out == 0, out <= 1};
}

// e, p, u, T^{tau mu}, pi^{tau mu} and Pi of one ghosted cell from the
// primitive fields (setConservedVariables, DynamicalVariables.cu:349-392, with
// Ttt..Ttn of EnergyMomentumTensor.cu:159-177; ghost cells,
// HydroPlugin.cpp:220; the previous velocity has zero ghosts,
// DynamicalVariables.cu:280-284).
template <typename PS>
__global__ __launch_bounds__(SBLOCK) void state_kernel(InitialFields F, StateBlocks B, Extent X) {
  const unsigned s = blockIdx.x * SBLOCK + threadIdx.x;
  if (s >= (unsigned)X.G) return;
  const Source c = source_of(X, s);
  const long long G = X.G, a = c.cell;
  double e = 0, p = 0, u[4] = {0, 0, 0, 0}, T[4] = {0, 0, 0, 0}, pi[4] = {0, 0, 0, 0}, Pi = 0;
  if (c.face) {
    e = F.e[a];
    p = F.p[a];
#pragma unroll
    for (int m = 0; m < 4; ++m) u[m] = F.u[m][a];
    if (F.pi[0])
#pragma unroll
      for (int m = 0; m < 4; ++m) pi[m] = F.pi[m][a];
    if (F.Pi) Pi = F.Pi[a];
    const double P = p + Pi;
    T[0] = (e + P) * u[0] * u[0] - P + pi[0];
#pragma unroll
    for (int m = 1; m < 4; ++m) T[m] = (e + P) * u[0] * u[m] + pi[m];
  }
  PS *q = reinterpret_cast<PS *>(B.q + 4 * G);
  B.e[s] = e;
  B.p[s] = p;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    B.q[m * G + s] = T[m];
    q[m * G + s] = (PS)pi[m];
    B.u[m * G + s] = u[m];
    B.up[m * G + s] = c.interior ? u[m] : 0.0;
  }
  q[10 * G + s] = (PS)Pi;
}

// The six spatial pi components.
template <typename PS>
__global__ __launch_bounds__(SBLOCK) void spatial_pi_kernel(InitialFields F, StateBlocks B, Extent X) {
  const unsigned s = blockIdx.x * SBLOCK + threadIdx.x;
  if (s >= (unsigned)X.G) return;
  const Source c = source_of(X, s);
  PS *q = reinterpret_cast<PS *>(B.q + 4 * X.G);
#pragma unroll
  for (int m = 4; m < 10; ++m)
    q[m * X.G + s] = (PS)(c.face && F.pi[m] ? F.pi[m][c.cell] : 0.0);
}

// A ghosted block as doubles: its interior cells, or all of it.
template <typename PS>
__global__ __launch_bounds__(SBLOCK) void pack_kernel(const PS *__restrict__ block, Extent X, int all,
                                                      unsigned n, double *__restrict__ out) {
  const unsigned c = blockIdx.x * SBLOCK + threadIdx.x;
  if (c >= n) return;
  unsigned s = c;
  if (!all) {
    const unsigned i = c % (unsigned)X.nx, r = c / (unsigned)X.nx;
    const unsigned j = r % (unsigned)X.ny, k = r / (unsigned)X.ny;
    s = (i + NG) + (unsigned)X.ncx * ((j + NG) + (unsigned)X.ncy * (k + NG));
  }
  out[c] = (double)block[s];
}

unsigned blocks(long long n) { return (unsigned)((n + SBLOCK - 1) / SBLOCK); }

}  // namespace

hipError_t launch_state(const InitialFields &F, const StateBlocks &B, const Extent &X, bool mixed,
                        bool spatial_pi, hipStream_t st) {
  const unsigned grid = blocks(X.G);
  if (spatial_pi) {
    if (mixed) spatial_pi_kernel<float><<<grid, SBLOCK, 0, st>>>(F, B, X);
    else spatial_pi_kernel<double><<<grid, SBLOCK, 0, st>>>(F, B, X);
  } else {
    if (mixed) state_kernel<float><<<grid, SBLOCK, 0, st>>>(F, B, X);
    else state_kernel<double><<<grid, SBLOCK, 0, st>>>(F, B, X);
  }
  return hipGetLastError();
}

hipError_t launch_pack(const void *block, bool is_float, const Extent &X, bool all, double *out,
                       hipStream_t st) {
  const long long n = all ? X.G : (long long)X.nx * X.ny * X.nz;
  if (is_float)
    pack_kernel<<<blocks(n), SBLOCK, 0, st>>>(static_cast<const float *>(block), X, all, (unsigned)n,
                                              out);
  else
    pack_kernel<<<blocks(n), SBLOCK, 0, st>>>(static_cast<const double *>(block), X, all,
                                              (unsigned)n, out);
  return hipGetLastError();
}

}  // namespace gvh
