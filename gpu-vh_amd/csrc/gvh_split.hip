// gvh_split.hip -- the stage kernel of small lattices: the sources and each
// direction of a cell by a wave of their own.
#include "gvh_stage_body.h"

namespace gvh {

// Blocks of one wave for the sources and one for each direction, on the same
// 64 cells.  The directions' rates meet in LDS and are added by the first wave
// in the order of the one-wave kernel, with the same operations.
//
// What bounds it: the latency of one tile, as all tiles are in flight at once;
// the one-wave kernel works through the sources, the directions and the cell's
// end (its root-find and writes) one after another, here the first two run
// together.  A wave for each interface of a direction (2-D five, 3-D seven)
// gained nothing more: the wave of the sources ends last.  us per step, table
// EoS with bulk, one wave per tile against this: 101x101 42 / 32 FP64 and 36 /
// 29 mixed, 31x31x21 54 / 40 and 50 / 34.
template <int EOS, bool BULK, bool STAGE2, bool HAS_Z, int LOCK, typename R, typename PS>
__global__ __launch_bounds__(64 * (HAS_Z ? 4 : 3), 2) void kt_split_kernel(StageArgs A) {
  __shared__ double part[HAS_Z ? 4 : 3][15 * BLOCK];
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const unsigned b = blockIdx.x, lb = (b & 7u) * (gridDim.x >> 3) + (b >> 3);
  const CellPos c = cell_of_index(A, lb * BLOCK + lane);
  if (wave == 0) {
    stage_cell<EOS, BULK, STAGE2, HAS_Z, true, true, LOCK, R, PS, false, true>(
        A, A.tab, c, part[0] + lane, nullptr, part[1] + lane);
    return;
  }
  if (c.valid) {
    const double *u = A.uin;
    const double e_s = ld_cell(A.ein, c.s);
    const auto g = make_guess<EOS>(A.tab, flux_root_t<EOS, R, LOCK == 3>(e_s));
    const R v = div_st(R(ld_cell(u + wave * A.G, c.s)), R(ld_cell(u, c.s)));
    double *rate = part[wave] + lane;
    if (wave == 1)
      direction_update<EOS, BULK, 0, true, LOCK, R, PS, false, false>(A, A.tab, c.s, e_s, g, v, rate);
    else if (!HAS_Z || wave == 2)
      direction_update<EOS, BULK, 1, true, LOCK, R, PS, false, false>(A, A.tab, c.s, e_s, g, v, rate);
    else if constexpr (HAS_Z)
      direction_update<EOS, BULK, 2, true, LOCK, R, PS, false, false>(A, A.tab, c.s, e_s, g, v, rate);
  }
  __syncthreads();
}

// Up to about as many tiles as blocks are in flight: 512, two per CU, at two
// waves per SIMD (FP64, or half-site root-finds in FP64), and 1536 in FP32.
// Beyond, the waves that wait for the first one hold places.  us per step, one
// wave per tile against split, table EoS with bulk: FP64 171x171 (457 tiles)
// 47 / 41, 201x201 (632) 50 / 50, 301x301 (1416) 73 / 74, 31x31x31 (466) 56 / 42,
// 41x41x31 (815) 63 / 64, 51x51x31 (1260) 84 / 98; mixed 201x201 42 / 36,
// 301x301 53 / 51, 321x321 (1610) 56 / 57, 41x41x31 54 / 45, 51x51x31 66 / 64,
// 61x61x41 (2384) 80 / 83; Wuppertal-Budapest FP64 171x171 56 / 46, 41x41x31
// 73 / 74.
bool split_stage_fits(const StageArgs &A, int eos, int precision) {
  const bool f32 = precision == GVH_MIXED && eos != EOS_WB;
  return A.ntiles <= (f32 ? SPLIT_MAX_TILES_FP32 : SPLIT_MAX_TILES_FP64);
}

template <int EOS, bool BULK, bool STAGE2, bool HAS_Z>
static void launch_s(const StageArgs &A, int precision, hipStream_t st) {
  constexpr int threads = 64 * (HAS_Z ? 4 : 3);
  if (precision == GVH_FP64)
    kt_split_kernel<EOS, BULK, STAGE2, HAS_Z, 1, double, double><<<A.ntiles, threads, 0, st>>>(A);
  else if (precision == GVH_MIXED)
    kt_split_kernel<EOS, BULK, STAGE2, HAS_Z, 1, float, float><<<A.ntiles, threads, 0, st>>>(A);
  else
    kt_split_kernel<EOS, BULK, STAGE2, HAS_Z, 3, float, float><<<A.ntiles, threads, 0, st>>>(A);
}

template <int EOS, bool BULK, bool STAGE2>
static void launch_sz(const StageArgs &A, int precision, hipStream_t st) {
  if (A.nz > 1) launch_s<EOS, BULK, STAGE2, true>(A, precision, st);
  else launch_s<EOS, BULK, STAGE2, false>(A, precision, st);
}

template <int EOS>
static void launch_se(const StageArgs &A, bool bulk, bool stage2, int precision, hipStream_t st) {
  if (bulk) stage2 ? launch_sz<EOS, true, true>(A, precision, st) : launch_sz<EOS, true, false>(A, precision, st);
  else stage2 ? launch_sz<EOS, false, true>(A, precision, st) : launch_sz<EOS, false, false>(A, precision, st);
}

hipError_t launch_split_stage(const StageArgs &A, int eos, bool bulk, bool stage2, int precision,
                              hipStream_t st) {
  switch (eos) {
    case EOS_CONFORMAL: launch_se<EOS_CONFORMAL>(A, bulk, stage2, precision, st); break;
    case EOS_WB: launch_se<EOS_WB>(A, bulk, stage2, precision, st); break;
    default: launch_se<EOS_TABLE>(A, bulk, stage2, precision, st);
  }
  return hipGetLastError();
}

}  // namespace gvh
