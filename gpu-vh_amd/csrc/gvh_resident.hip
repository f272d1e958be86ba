// gvh_resident.hip -- the stage kernel of large lattices with the tabulated
// EoS: one block per CU that stays for the whole stage.
//
// The waves of a block share a copy of the table in LDS and otherwise work
// alone: each takes the next tile of 64 cells from its XCD's counter, so that
// the tiles in flight stay a compact front of the traversal, and there is no
// barrier after the copy.
//
// What bounds it: the VALU (5100 instructions per wave and tile in FP64, 56%
// of the issue slots) and the memory round trips of a tile, at two or three
// waves per SIMD.  The table gathers of the root-finds, some ten round trips
// per tile to L1 or L2, are LDS reads here: 9% of the time.  Tiles handed
// out by counter rather than by a fixed stride are worth another 8% (the
// front stays compact, and no wave waits for a slow neighbour); taking tiles
// from other XCDs at the end cost more round trips than it saved.  201x201x101,
// every cell on the Newton branch, ms per step against one-wave blocks with
// the table in memory: FP64 2.08 -> 2.01, mixed 1.48 -> 1.34; 18% of the
// cells there: 1.99 -> 1.88 and 1.47 -> 1.31.
#include <algorithm>

#include "gvh_stage_body.h"

namespace gvh {

// Waves per block, one block per CU: as many as fit the registers of the
// arithmetic (stage_waves_per_simd; 2 per SIMD in FP64, also with FP64
// root-finds in the mixed form).
template <typename R, int LOCK>
constexpr int resident_waves() {
  return 4 * std::max(2, stage_waves_per_simd<R, LOCK>());
}

// Tile counters: one per XCD and stage, 128 bytes apart.
constexpr int NXCD = 8, TICKET_STRIDE = 32;
static_assert(RESIDENT_TICKETS == 2 * NXCD * TICKET_STRIDE, "counters of two stages");

// FP64 nodes whole where the accumulators leave the room (8 waves), as
// {p, cs2} beside the FP32 nodes of the 12-wave form.
template <bool BULK, bool STAGE2, bool HAS_Z, int LOCK, typename R, typename PS>
__global__ __launch_bounds__((64 * resident_waves<R, LOCK>()), (resident_waves<R, LOCK>() / 4)) void
kt_resident_kernel(StageArgs A0) {
  constexpr int W = resident_waves<R, LOCK>();
  constexpr bool F32 = sizeof(flux_root_t<EOS_TABLE, R, LOCK == 3>) == 4, WIDE = !F32;
  __shared__ double acc_lds[W][15 * 64];
  __shared__ double2 n64[TAB_LDS_NODES * (WIDE ? 2 : 1)];
  __shared__ float4 n32[F32 ? TAB_LDS_NODES : 1];
  for (int k = threadIdx.x; k < A0.tab.n; k += blockDim.x) {
    const double4 v = A0.tab.pc[k];
    if constexpr (WIDE) {
      n64[2 * k] = double2{v.x, v.y};
      n64[2 * k + 1] = double2{v.z, v.w};
    } else {
      n64[k] = double2{v.x, v.z};
    }
    if constexpr (F32) n32[k] = A0.tab.pcf[k];
  }
  // this stage's counters were cleared by the stage before it
  if (blockIdx.x < NXCD && threadIdx.x == 0)
    A0.tickets[((STAGE2 ? 0 : NXCD) + blockIdx.x) * TICKET_STRIDE] = 0;
  __syncthreads();
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const unsigned n8 = A0.ntiles / NXCD;
  double *acc = acc_lds[wave] + lane;
  unsigned *counters = A0.tickets + (STAGE2 ? NXCD : 0) * TICKET_STRIDE;
  // the arguments are read anew for every tile: kept over the loop, what is
  // derived from them would fill the vector registers
  auto args = (const __attribute__((address_space(4))) char *)__builtin_amdgcn_kernarg_segment_ptr();
  // XCD x = block mod 8 sweeps tiles [x n8, (x + 1) n8): a wave's first tile
  // is its own number among the XCD's waves, the later ones come from the
  // counter, each asked for while the one before it is worked on
  const unsigned x = blockIdx.x % NXCD, waves = gridDim.x / NXCD * W;
  auto take = [&]() {
    unsigned v = 0;
    if (lane == 0) v = atomicAdd(counters + x * TICKET_STRIDE, 1u) + waves;
    return v;
  };
  unsigned next = blockIdx.x / NXCD * W + wave;
#pragma unroll 1
  while (true) {
    const unsigned i = __builtin_amdgcn_readfirstlane(next);
    if (i >= n8) break;
    next = take();
    asm("" : "+s"(args));
    const StageArgs &A = *(const StageArgs *)args;
    const LdsTable<WIDE> tab(A.tab, n64, n32);
    const CellPos c = cell_of_index(A, (x * n8 + i) * 64u + lane);
    if (c.valid)
      stage_cell<EOS_TABLE, BULK, STAGE2, HAS_Z, true, true, LOCK, R, PS>(A, tab, c, acc);
  }
}

bool resident_stage_fits(const StageArgs &A) {
  return A.tab.n <= TAB_LDS_NODES && A.ntiles >= RESIDENT_MIN_TILES;
}

template <bool BULK, bool STAGE2, bool HAS_Z>
static void launch_r(const StageArgs &A, int precision, hipStream_t st) {
  const int cus = 256;
  if (precision == GVH_FP64)
    kt_resident_kernel<BULK, STAGE2, HAS_Z, 1, double, double>
        <<<cus, 64 * resident_waves<double, 1>(), 0, st>>>(A);
  else if (precision == GVH_MIXED)
    kt_resident_kernel<BULK, STAGE2, HAS_Z, 1, float, float>
        <<<cus, 64 * resident_waves<float, 1>(), 0, st>>>(A);
  else
    kt_resident_kernel<BULK, STAGE2, HAS_Z, 3, float, float>
        <<<cus, 64 * resident_waves<float, 3>(), 0, st>>>(A);
}

template <bool BULK, bool STAGE2>
static void launch_rz(const StageArgs &A, int precision, hipStream_t st) {
  if (A.nz > 1) launch_r<BULK, STAGE2, true>(A, precision, st);
  else launch_r<BULK, STAGE2, false>(A, precision, st);
}

hipError_t launch_resident_stage(const StageArgs &A, bool bulk, bool stage2, int precision,
                                 hipStream_t st) {
  if (bulk) stage2 ? launch_rz<true, true>(A, precision, st) : launch_rz<true, false>(A, precision, st);
  else stage2 ? launch_rz<false, true>(A, precision, st) : launch_rz<false, false>(A, precision, st);
  return hipGetLastError();
}

}  // namespace gvh
