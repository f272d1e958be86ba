// gvh_device.h -- device math of the KT step for gfx950 (FP64 form).
//
// Reference files are cited per function (paths relative to rhic/src).
// All state arithmetic is double.  Divisions that the reference performs by
// a per-launch constant (dt, dx, t) are replaced by a multiplication with a
// host-computed reciprocal; that, FMA contraction and the flux written as
// (u_dir/u^tau)*q change results at the rounding level only.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace gvh {

constexpr int NG = 2;             // ghost layers (LatticeParameters.h:13-15)
constexpr int MAX_ITERS = 1000000; // EnergyMomentumTensor.cu:15
constexpr double THETA = 2.0;     // FluxLimiter.cu:15
constexpr double EOS_FACTOR = 13.8997; // EquationOfState.cuh:24

enum { EOS_CONFORMAL = 0, EOS_WB = 1, EOS_TABLE = 2 };

// Threads per block of the stage kernels, and cells per tile of a batch.
// One wave per block: a block holds its CU resources until its slowest wave
// ends, and the waves of a block differ in their root-find iteration counts,
// so smaller blocks leave fewer idle slots (the 201x201x101 step: 2.40 ms
// with 64, 2.51 ms with 128, 2.57 ms with 256 threads).
#ifndef GVH_BLOCK
#define GVH_BLOCK 64
#endif

// Lattices of at most this many tiles of 64 cells, by the arithmetic of the
// half-site root-finds, run their stages with several waves per tile
// (gvh_split.hip, split_stage_fits).
#ifndef GVH_SPLIT_MAX_TILES_FP64
#define GVH_SPLIT_MAX_TILES_FP64 512
#define GVH_SPLIT_MAX_TILES_FP32 1536
#endif
constexpr unsigned SPLIT_MAX_TILES_FP64 = GVH_SPLIT_MAX_TILES_FP64;
constexpr unsigned SPLIT_MAX_TILES_FP32 = GVH_SPLIT_MAX_TILES_FP32;

// Lattices of at least this many tiles of 64 cells run their stages in the
// resident kernel (gvh_resident.hip).  Its blocks start with a copy of the
// table and its 2048 (FP64) or 3072 waves end together only if each has
// several tiles.  us per step, one-wave blocks against resident, table EoS
// with bulk: 101x101x31 (4941 tiles) 208 / 219 FP64 and 138 / 145 mixed,
// 101x101x51 (8129) 311 / 308 and 202 / 205, 151x151x41 (14607) 540 / 527
// and 380 / 352, 201x201x101 (63757) 2120 / 2040 and 1469 / 1332.
#ifndef GVH_RESIDENT_MIN_TILES
#define GVH_RESIDENT_MIN_TILES 10240
#endif
constexpr unsigned RESIDENT_MIN_TILES = GVH_RESIDENT_MIN_TILES;
constexpr int RESIDENT_TICKETS = 512;  // its tile counters, 32-bit words

// counters of failure events, indexes into StageArgs::diag
enum { DIAG_NOT_CONVERGED = 0, DIAG_E_NAN = 1, DIAG_E_CLAMPED = 2, DIAG_N = 4 };

// Tabulated EoS on the device.  Node k sits at
// e_k = 2^(emin_exp + k/M) (1 + (k % M)/M); per node the value and the
// difference to node k+1 are stored so that an interpolation is one load.
struct EosTable {
  const double4 *pc;  // {p_k, p_{k+1}-p_k, cs2_k, cs2_{k+1}-cs2_k}
  const double2 *tt;  // {T_k, T_{k+1}-T_k}
  const float4 *pcf;  // pc rounded to FP32 (the mixed form's flux root-finds)
  int n, M, emin_exp;
  double e_first, e_second;  // e_0, e_1
  double e_pen, e_last;      // e_{n-2}, e_{n-1}
  double inv_first_span;     // 1/(e_1 - e_0)
  double inv_last_span;      // 1/(e_{n-1} - e_{n-2})
  float f_first, f_pen, f_last, f_inv_first_span, f_inv_last_span;  // the same in FP32
  // high word (FP64) or bits (FP32) of e_0 = 2^emin_exp, and how far those of
  // e_{n-2} lie above it: the range of the branch-free lookup
  unsigned hi_first, hi_span, fb_first, fb_span;
};

struct StageArgs {
  const double *__restrict__ qin;   // stage input conserved, 15 x G
  const double *__restrict__ qn;    // q^n for the convex average (stage 2)
  double *__restrict__ qout;        // stage output conserved
  const double *__restrict__ uin;   // u of the stage input, 4 x G
  const double *__restrict__ uprev; // u used for the time derivative
  double *__restrict__ uout;
  const double *__restrict__ ein;
  const double *__restrict__ pin;
  double *__restrict__ eout;
  double *__restrict__ pout;
  unsigned long long *__restrict__ diag;
  unsigned *__restrict__ tickets;  // tile counters of the resident kernel (gvh_resident.hip)
  double *__restrict__ reg;  // stage 2 stores the shear regulation factor here if set
  long long G;          // stride between variables
  int nx, ny, nz, ncx, ncy;
  double t;             // time of the Euler step
  double tinf;          // time of the inferred-variable solve
  double dt, inv_dt;
  double h[3], inv_h[3], half_inv_h[3];  // dx, dy, deta and reciprocals
  double etabar;        // eta/s
  double zeta_tpeak;    // zeta/s temperature scale
  double e_reg;         // regulation below this energy density
  EosTable tab;
  int strip, nstrips;   // y rows per traversal strip, number of strips
  unsigned ntiles;      // blocks of 64 cells of the traversal, a multiple of 8
  int variant;          // kernel arrangement of a stage (gvh_stage.hip)
  int max_iters;        // Newton iterations per root-find: MAX_ITERS (the reference's),
                        // or a smaller budget of a batched event
};

// Buffers of one event and their current roles: the reference's pointer
// swaps (FullyDiscreteKurganovTadmorScheme.cu:117-133,
// DynamicalVariables.cu:400-408) as indices.  q[iq] holds q^n, q[1-iq] the
// corrector output Q, q[2] the predictor qS; u[iu] u^n, u[iup] u^{n-1},
// u[3-iu-iup] the predictor u*; (e, p)[ie] the current state.
struct Roles {
  int iq, iu, iup, ie;
};
struct Buffers {
  double *q[3], *u[3], *e[2], *p[2];
};

// State pointers of RK stage 1 or 2 for the given roles.
__host__ __device__ inline void stage_pointers(StageArgs &A, const Buffers &B, const Roles &R,
                                               int stage) {
  const int iqs = 2, iQ = 1 - R.iq, ius = 3 - R.iu - R.iup;
  const int ie_in = stage == 1 ? R.ie : 1 - R.ie;
  A.qin = B.q[stage == 1 ? R.iq : iqs];
  A.qn = B.q[R.iq];
  A.qout = B.q[stage == 1 ? iqs : iQ];
  A.uin = B.u[stage == 1 ? R.iu : ius];
  A.uprev = B.u[stage == 1 ? R.iup : R.iu];
  A.uout = B.u[stage == 1 ? ius : R.iup];
  A.ein = B.e[ie_in];
  A.pin = B.p[ie_in];
  A.eout = B.e[1 - ie_in];
  A.pout = B.p[1 - ie_in];
}

// Times of stage 1 or 2 of the step that starts at t (the predictor's
// inferred variables are solved at t + dt, FullyDiscreteKurganovTadmorScheme.cu:119).
__host__ __device__ inline void stage_times(StageArgs &A, double t, int stage) {
  A.t = stage == 1 ? t : t + A.dt;
  A.tinf = t + A.dt;
}

// Roles after a step: u^{n+1} was written into the u^{n-1} buffer, q^{n+1}
// into Q.
__host__ __device__ inline void rotate_roles(Roles &R) {
  const int old_u = R.iu;
  R.iu = R.iup;
  R.iup = old_u;
  R.iq = 1 - R.iq;
}

// One event of a batch in device memory.
enum { SLOT_FREE = 0, SLOT_RUN = 1, SLOT_DONE = 2 };
struct BatchSlot {
  StageArgs A;        // constants of the event; pointers and times are set per stage
  Buffers B;
  Roles R;
  double t0;
  int steps;          // KT steps done
  int status;         // SLOT_*
  int max_steps;      // the run loop's nt + 1
  int frozen;         // steps seen with no interior cell above e_fo (never reset)
  int fofreq;
  int fo_flags;       // GVH_FO_CURRENT_FIELDS selects the current u, pi for the ring
  int frozen_stop;    // 1 if it ended by the all-frozen rule
  int error;          // 1 if it was retired for a root-find over its iteration budget
  int bulk;           // Pi is evolved
  int tile_first, ntiles;  // its tiles (blocks of cells) in the tile map
  double e_fo;
  unsigned long long above;  // interior cells with e > e_fo in the current state
  double *ring;       // freeze-out history, halves x (fofreq+1) x 10 x nint, or nullptr
  long long nint;
  int halves;         // 2: window m records into ring half m mod 2
};

// ------------------------------------------------------- cell access
// Element s of an array with a uniform (scalar) base: the byte offset is
// formed as a 32-bit product, so a load or store is the scalar-base +
// 32-bit-vector-offset form and needs no 64-bit address per access.  Every
// array of a lattice is below 4 GiB (the context checks the ghosted size).
template <typename T>
__device__ __forceinline__ T ld_cell(const T *base, unsigned s) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) +
                                      s * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ void st_cell(T *base, unsigned s, T v) {
  *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + s * (unsigned)sizeof(T)) = v;
}

// ------------------------------------------------------------ limiter
// approximateDerivative (FluxLimiter.cu:33-39): the nested generalized
// minmod(theta*dl, minmod(dc, theta*dr)) with sgn(0)=+1 equals
// sign * min(|theta dl|, |dc|, |theta dr|) when all three arguments are in the
// same sign class (x < 0 versus x >= 0) and +0 otherwise -- exactly, since
// min and the factors 2 and 1/2 do not round.  That form needs no products
// of signs.  With a = y - x, c = z - y, b = z - x: min(2|a|, |b|/2, 2|c|)
// = 2 min(|a|, |c|, |b|/4) exactly, and a, c in one class force b into it
// (y >= x and z >= y give z >= x, likewise for <), so the class test needs
// only a and c.
//
// Every use takes half of it (the half-site states q +- D/2) or twice the
// half (the gradients), so the kernels evaluate D/2 = sign min(|a|, |c|,
// |b|/4) directly; the factors 2 and 1/2 cancel exactly.
// FP32: the two-argument minmod is the median of (p, q, 0), so
// D/2 = med3(a, med3(b/4, c, 0), 0), two v_med3_f32.
// FP64 (there is no v_med3_f64): the magnitude from two v_min_f64, the sign
// of a inserted into its high word, zero when a and c differ in sign bit.
// A zero a or c makes the magnitude zero, so classing -0 with the negatives
// changes at most the sign of a zero result.
static_assert(THETA == 2.0, "the half-slope form assumes theta = 2");
template <typename R>
__device__ __forceinline__ R half_slope_t(R x, R y, R z);
template <>
__device__ __forceinline__ float half_slope_t<float>(float x, float y, float z) {
  const float a = y - x, b = z - x, c = z - y;
  return __builtin_amdgcn_fmed3f(a, __builtin_amdgcn_fmed3f(b * 0.25f, c, 0.0f), 0.0f);
}
template <>
__device__ __forceinline__ double half_slope_t<double>(double x, double y, double z) {
  const double a = y - x, b = z - x, c = z - y;
  const double m = fmin(fmin(fabs(a), fabs(c)), fabs(b) * 0.25);
  int sx = __double2hiint(a) ^ __double2hiint(c);
  // an empty register constraint keeps the sign test one 32-bit xor and
  // compare; left visible, the combiner widens it to a 64-bit xor and compare
  asm("" : "+v"(sx));
  return sx >= 0 ? copysign(m, a) : 0.0;
}
template <typename R>
__device__ __forceinline__ R slope_t(R x, R y, R z) {
  const R h = half_slope_t<R>(x, y, z);
  return h + h;
}
__device__ __forceinline__ double slope(double x, double y, double z) {
  return slope_t<double>(x, y, z);
}

// ------------------------------------------------ division, square root
// The IEEE-exact expansions of a/b and sqrt(x) on gfx950 cost ~11 and ~15
// VALU instructions.  These start from the hardware approximations
// (v_rcp_f64, v_rsq_f64: at most 4.6e-8 and 5.3e-8 relative, measured on
// 4M inputs over [1e-6, 1e6]) and refine with FMA steps.  A third-order step
// takes the reciprocal to 0.5 ulp; a quotient and a square root end with a
// residual correction, which needs its reciprocal only to 2e-15.  Operands
// here are finite, normal and nonzero in any physical state; special values
// are not treated, except that sqrt_nr(0) is 0 to within 1e-150.
__device__ __forceinline__ double rcp_nr(double b) {
  const double r = __builtin_amdgcn_rcp(b);
  const double e = fma(-b, r, 1.0);
  return fma(r, fma(e, e, e), r);
}
__device__ __forceinline__ double div_nr(double a, double b) {
  double r = __builtin_amdgcn_rcp(b);
  r = fma(fma(-b, r, 1.0), r, r);
  const double q = a * r;
  return fma(fma(-b, q, a), r, q);
}
__device__ __forceinline__ double sqrt_nr(double x) {
  x = fmax(x, 1e-300);
  const double y = __builtin_amdgcn_rsq(x);  // ~ 1/sqrt(x)
  double g = x * y;
  const double h = 0.5 * y;
  g = fma(g, fma(-g, h, 0.5), g);
  return fma(fma(-g, g, x), h, g);
}

// The same operations in the arithmetic type of a root-find: FP64 as above,
// FP32 from the hardware approximations (about 1 ulp).
__device__ __forceinline__ double rcp_t(double b) { return rcp_nr(b); }
__device__ __forceinline__ double div_t(double a, double b) { return div_nr(a, b); }
__device__ __forceinline__ double sqrt_t(double x) { return sqrt_nr(x); }
__device__ __forceinline__ float rcp_t(float b) { return __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ float div_t(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ float sqrt_t(float x) { return __builtin_amdgcn_sqrtf(x); }

// a / b in the stencil and source arithmetic of a stage: the IEEE division
// in FP64 (the reference's expression), the hardware reciprocal (about 1 ulp)
// times a in FP32.
__device__ __forceinline__ double div_st(double a, double b) { return a / b; }
__device__ __forceinline__ float div_st(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

// ---------------------------------------------------------------- EoS
struct TabPos {
  int k;
  double fr;
};

__device__ __forceinline__ TabPos tab_locate(const EosTable &T, double e) {
  TabPos r;
  if (e >= T.e_first && e < T.e_last) {
    int E;
    const double m = frexp(e, &E);  // e = m 2^E, m in [0.5, 1)
    const double f = (2.0 * m - 1.0) * (double)T.M;
    const int j = (int)f;
    r.fr = f - (double)j;
    r.k = (E - 1 - T.emin_exp) * T.M + j;
    if (r.k > T.n - 2) {  // f rounded up onto the last node
      r.k = T.n - 2;
      r.fr += 1.0;
    }
  } else if (e >= T.e_last) {  // beyond the table, +inf included
    r.k = T.n - 2;
    r.fr = (e - T.e_pen) * T.inv_last_span;
  } else {  // below the first node, or NaN
    r.k = 0;
    r.fr = (e - T.e_first) * T.inv_first_span;
  }
  return r;
}

// tab_locate in FP32.
struct TabPosF {
  int k;
  float fr;
};
__device__ __forceinline__ TabPosF tab_locate_f(const EosTable &T, float e) {
  TabPosF r;
  if (e >= T.f_first && e < T.f_last) {
    int E;
    const float m = frexpf(e, &E);
    const float f = (2.0f * m - 1.0f) * (float)T.M;
    const int j = (int)f;
    r.fr = f - (float)j;
    r.k = (E - 1 - T.emin_exp) * T.M + j;
    if (r.k > T.n - 2) {
      r.k = T.n - 2;
      r.fr += 1.0f;
    }
  } else if (e >= T.f_last) {
    r.k = T.n - 2;
    r.fr = (e - T.f_pen) * T.f_inv_last_span;
  } else {
    r.k = 0;
    r.fr = (e - T.f_first) * T.f_inv_first_span;
  }
  return r;
}
// Positions of N energy densities at once: the octave and the place in it come straight from the exponent and mantissa bits, with
// one wave-wide test that all N lie in [e_0, e_{n-2}) and the general lookup
// behind it: 9 VALU instructions per lookup instead of 24, the same node
// and fraction.  Only lanes with an energy density outside that range take
// the general position.
template <int N>
__device__ __forceinline__ void tab_locate_n(const EosTable &T, const double *e, unsigned *k,
                                             double *fr) {
  unsigned d[N], far = 0;
  const double M = (double)T.M;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const unsigned hi = (unsigned)__double2hiint(e[n]);
    d[n] = hi - T.hi_first;
    far = d[n] > far ? d[n] : far;
    const double f = fma(__builtin_amdgcn_frexp_mant(e[n]), M + M, -M);  // (2 m - 1) M
    fr[n] = __builtin_amdgcn_fract(f);
    k[n] = __umul24(d[n] >> 20, (unsigned)T.M) + (unsigned)(int)f;
  }
  if (__any(far >= T.hi_span)) {
#pragma unroll
    for (int n = 0; n < N; ++n)
      if (d[n] >= T.hi_span) {
        const TabPos q = tab_locate(T, e[n]);
        k[n] = (unsigned)q.k;
        fr[n] = q.fr;
      }
  }
}
template <int N>
__device__ __forceinline__ void tab_locate_n(const EosTable &T, const float *e, unsigned *k,
                                             float *fr) {
  unsigned d[N], far = 0;
  const float M = (float)T.M;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const unsigned bits = __float_as_uint(e[n]);
    d[n] = bits - T.fb_first;
    far = d[n] > far ? d[n] : far;
    const float x = fmaf(__builtin_amdgcn_frexp_mantf(e[n]), 2.0f, -1.0f), f = x * M;
    fr[n] = fmaf(x, M, -truncf(f));
    k[n] = __umul24(d[n] >> 23, (unsigned)T.M) + (unsigned)(int)f;
  }
  if (__any(far >= T.fb_span)) {
#pragma unroll
    for (int n = 0; n < N; ++n)
      if (d[n] >= T.fb_span) {
        const TabPosF q = tab_locate_f(T, e[n]);
        k[n] = (unsigned)q.k;
        fr[n] = q.fr;
      }
  }
}

// Node k: {p_k, p_{k+1} - p_k, cs2_k, cs2_{k+1} - cs2_k} (tab_pc), its first
// half (tab_pp) and {T_k, T_{k+1} - T_k} (tab_tt).
__device__ __forceinline__ double4 tab_pc(const EosTable &T, unsigned k) { return ld_cell(T.pc, k); }
__device__ __forceinline__ double2 tab_pp(const EosTable &T, unsigned k) {
  return ld_cell(reinterpret_cast<const double2 *>(T.pc), 2 * k);
}
__device__ __forceinline__ double2 tab_tt(const EosTable &T, unsigned k) { return ld_cell(T.tt, k); }
__device__ __forceinline__ float4 tab_pcf(const EosTable &T, unsigned k) { return ld_cell(T.pcf, k); }
__device__ __forceinline__ float2 tab_ppf(const EosTable &T, unsigned k) {
  return ld_cell(reinterpret_cast<const float2 *>(T.pcf), 2 * k);
}

// The table with copies of its nodes in LDS.  FP64 nodes are either whole
// (WIDE: as in T.pc) or {p_k, cs2_k}, whose differences are taken at the
// lookup (the same subtraction of the same values as in T.pc); FP32 nodes are
// as in T.pcf.  T(e) stays in memory: one lookup per cell and stage.
constexpr int TAB_LDS_NODES = 2048;
template <bool WIDE>
struct LdsTable : EosTable {
  const double2 *n64;
  const float4 *n32;
  __device__ __forceinline__ LdsTable(const EosTable &T, const double2 *a, const float4 *b)
      : EosTable(T), n64(a), n32(b) {}
};
template <bool WIDE>
__device__ __forceinline__ double4 tab_pc(const LdsTable<WIDE> &T, unsigned k) {
  if constexpr (WIDE) {
    const double2 a = T.n64[2 * k], b = T.n64[2 * k + 1];
    return double4{a.x, a.y, b.x, b.y};
  } else {
    const double2 a = T.n64[k], b = T.n64[k + 1];
    return double4{a.x, b.x - a.x, a.y, b.y - a.y};
  }
}
template <bool WIDE>
__device__ __forceinline__ double2 tab_pp(const LdsTable<WIDE> &T, unsigned k) {
  if constexpr (WIDE) return T.n64[2 * k];
  const double a = T.n64[k].x, b = T.n64[k + 1].x;
  return double2{a, b - a};
}
template <bool WIDE>
__device__ __forceinline__ float4 tab_pcf(const LdsTable<WIDE> &T, unsigned k) {
  return T.n32[k];
}
template <bool WIDE>
__device__ __forceinline__ float2 tab_ppf(const LdsTable<WIDE> &T, unsigned k) {
  return *reinterpret_cast<const float2 *>(T.n32 + k);
}

__device__ __forceinline__ TabPos tab_at(const EosTable &T, double e) {
  unsigned k;
  TabPos r;
  tab_locate_n<1>(T, &e, &k, &r.fr);
  r.k = (int)k;
  return r;
}

// c[0] + c[1] x + ... by Horner's rule: one FMA per coefficient.  The WB fits
// of the root-finds are bound by their FMAs; summed over explicit powers of
// e they took 12 multiplications more per evaluation.
template <int N>
__device__ __forceinline__ double horner(const double (&c)[N], double x) {
  double r = c[N - 1];
#pragma unroll
  for (int k = N - 2; k >= 0; --k) r = fma(r, x, c[k]);
  return r;
}

// equilibriumPressure (EquationOfState.cu:31-80) and speedOfSoundSquared
// (:83-116); the conformal c_s^2 is the reference's integer 1/3 == 0.
template <int EOS, typename Tab>
__device__ __forceinline__ void eos_p_cs2(const Tab &T, double e, double &p,
                                          double &cs2) {
  if constexpr (EOS == EOS_CONFORMAL) {
    p = e / 3.0;
    cs2 = 0.0;
  } else if constexpr (EOS == EOS_TABLE) {
    const TabPos q = tab_at(T, e);
    const double4 v = tab_pc(T, (unsigned)q.k);
    p = v.x + q.fr * v.y;
    cs2 = v.z + q.fr * v.w;
  } else {
    constexpr double pn[] = {-0.25181736420168666, 9737.845799644809, 1.077580993288114e6,
        3.1729694865420084e6, 1.6357487344679043e6, 334334.4309240126, 41913.439282708554,
        6340.448389300905, 141.5073484468774, 0.7158279081255019, 0.0009417586777847889,
        3.1188455176941583e-7, 1.9531729608963267e-11};
    constexpr double pd[] = {45829.44617893836, 4.0574329080826794e6, 2.0931169138134286e7,
        1.3512402226067686e7, 1.7851642641834426e6, 278581.2989342773, 26452.34905933697,
        499.04919730607065, 2.3405487982094204, 0.002962497695527404, 9.601103399348206e-7,
        5.928138360995685e-11, 3.2581066229887368e-18};
    p = div_nr(horner(pn, e), horner(pd, e));
    constexpr double cn[] = {5.191934309650155e-32, 4.123605749683891e-23, 3.1955868410879504e-16,
        1.4170364808063119e-10, 6.087136671592452e-6, 0.02969737949090831, 15.382615282179595,
        460.6487249985994, 1612.4245252438795, 275.0492627924299, 58.60283714484669,
        6.504847576502024, 0.03009027913262399, 8.189430244031285e-6};
    constexpr double cd[] = {1.4637868900982493e-30, 6.716598285341542e-22, 3.5477700458515908e-15,
        1.1225580509306008e-9, 0.00003551782901018317, 0.13653226327408863, 60.85769171450653,
        1800.5461219450308, 15190.225535036281, 590.2572000057821, 293.99144775704605,
        21.461303090563028, 0.09301685073435291, 0.000024810902623582917};
    cs2 = div_nr(horner(cn, e), horner(cd, e));
  }
}

template <int EOS, typename Tab>
__device__ __forceinline__ double eos_p(const Tab &T, double e) {
  if constexpr (EOS == EOS_CONFORMAL) {
    return e / 3.0;
  } else if constexpr (EOS == EOS_TABLE) {
    const TabPos q = tab_at(T, e);
    const double2 v = tab_pp(T, (unsigned)q.k);
    return v.x + q.fr * v.y;
  } else {
    double p, c;
    eos_p_cs2<EOS>(T, e, p, c);
    return p;
  }
}

// p and c_s^2 of the table with FP32 node values.
template <typename Tab>
__device__ __forceinline__ void tab_p_cs2_f(const Tab &T, float e, float &p, float &cs2) {
  unsigned k;
  float fr;
  tab_locate_n<1>(T, &e, &k, &fr);
  const float4 v = tab_pcf(T, k);
  p = v.x + fr * v.y;
  cs2 = v.z + fr * v.w;
}

// eos_p_cs2 / eos_p in the arithmetic type F (float only for the conformal
// and tabulated EoS).
template <int EOS, typename F, typename Tab>
__device__ __forceinline__ void eos_p_cs2_t(const Tab &T, F e, F &p, F &cs2) {
  if constexpr (std::is_same<F, double>::value) {
    eos_p_cs2<EOS>(T, e, p, cs2);
  } else {
    static_assert(EOS != EOS_WB, "the WB fits stay in FP64");
    if constexpr (EOS == EOS_CONFORMAL) {
      p = e / 3.0f;
      cs2 = 0.0f;
    } else {
      tab_p_cs2_f(T, e, p, cs2);
    }
  }
}
template <int EOS, typename F, typename Tab>
__device__ __forceinline__ F eos_p_t(const Tab &T, F e) {
  if constexpr (std::is_same<F, double>::value) {
    return eos_p<EOS>(T, e);
  } else {
    F p, c;
    eos_p_cs2_t<EOS, F>(T, e, p, c);
    return p;
  }
}

// effectiveTemperature, EquationOfState.cu:119-148
template <int EOS, typename Tab>
__device__ __forceinline__ double eos_T(const Tab &T, double e) {
  if constexpr (EOS == EOS_CONFORMAL) {
    return pow(e / EOS_FACTOR, 0.25);
  } else if constexpr (EOS == EOS_TABLE) {
    const TabPos q = tab_at(T, e);
    const double2 v = tab_tt(T, (unsigned)q.k);
    return v.x + q.fr * v.y;
  } else {
    constexpr double tn[] = {1.510073201405604e-29, 8.014062800678687e-18, 2.4954778310451065e-10,
        0.000063810382643387, 0.4873490574161924, 207.48582344326206, 6686.07424325115,
        14109.766109389702, 1471.6180520527757, 14.055788949565482, 0.015421252394182246,
        1.5780479034557783e-6};
    constexpr double td[] = {7.558667139355393e-28, 1.3686372302041508e-16, 2.998130743142826e-9,
        0.0005036835870305458, 2.316902328874072, 578.0778724946719, 11179.193315394154,
        17965.67607192861, 1051.0730543534657, 5.916312075925817, 0.003778342768228011,
        1.8472801679382593e-7};
    return div_nr(horner(tn, e), horner(td, e));
  }
}

// bulkViscosityToEntropyDensity, TransportCoefficients.cu:27-36
__device__ __forceinline__ double zeta_over_s(double T, double tpeak) {
  double x = T / tpeak;
  if (x > 1.05) return 0.9 * exp(-(x - 1) / 0.025) + 0.25 * exp(-(x - 1) / 0.13) + 0.001;
  if (x < 0.995) return 0.9 * exp((x - 1) / 0.0025) + 0.22 * exp((x - 1) / 0.022) + 0.03;
  return -13.77 * x * x + 27.55 * x - 13.45;
}
// The same in FP32 for the mixed form's source terms: divisions by the
// constant widths as products with their reciprocals, the hardware exp.
__device__ __forceinline__ float zeta_over_s(float T, float tpeak) {
  const float x = T * __builtin_amdgcn_rcpf(tpeak), d = x - 1.0f;
  if (x > 1.05f) return 0.9f * __expf(d * -40.0f) + 0.25f * __expf(d * (-1.0f / 0.13f)) + 0.001f;
  if (x < 0.995f) return 0.9f * __expf(d * 400.0f) + 0.22f * __expf(d * (1.0f / 0.022f)) + 0.03f;
  return -13.77f * x * x + 27.55f * x - 13.45f;
}

// ------------------------------------------------------------ root-find
// ------------------------------------------------ lookups of a root-find
// p and c_s^2, or p alone, of N energy densities.
template <int EOS, int N, typename F, typename Tab>
__device__ __forceinline__ void eos_p_cs2_n(const Tab &T, const F *e, F *p, F *cs2) {
  if constexpr (EOS == EOS_TABLE) {
    unsigned k[N];
    F fr[N];
    tab_locate_n<N>(T, e, k, fr);
    if constexpr (std::is_same<F, double>::value) {
      double4 v[N];
#pragma unroll
      for (int n = 0; n < N; ++n) v[n] = tab_pc(T, k[n]);
#pragma unroll
      for (int n = 0; n < N; ++n) {
        p[n] = v[n].x + fr[n] * v[n].y;
        cs2[n] = v[n].z + fr[n] * v[n].w;
      }
    } else {
      float4 v[N];
#pragma unroll
      for (int n = 0; n < N; ++n) v[n] = tab_pcf(T, k[n]);
#pragma unroll
      for (int n = 0; n < N; ++n) {
        p[n] = v[n].x + fr[n] * v[n].y;
        cs2[n] = v[n].z + fr[n] * v[n].w;
      }
    }
  } else {
#pragma unroll
    for (int n = 0; n < N; ++n) eos_p_cs2_t<EOS, F>(T, e[n], p[n], cs2[n]);
  }
}
template <int EOS, int N, typename F, typename Tab>
__device__ __forceinline__ void eos_p_n(const Tab &T, const F *e, F *p) {
  if constexpr (EOS == EOS_TABLE) {
    unsigned k[N];
    F fr[N];
    tab_locate_n<N>(T, e, k, fr);
    if constexpr (std::is_same<F, double>::value) {
      double2 v[N];
#pragma unroll
      for (int n = 0; n < N; ++n) v[n] = tab_pp(T, k[n]);
#pragma unroll
      for (int n = 0; n < N; ++n) p[n] = v[n].x + fr[n] * v[n].y;
    } else {
      float2 v[N];
#pragma unroll
      for (int n = 0; n < N; ++n) v[n] = tab_ppf(T, k[n]);
#pragma unroll
      for (int n = 0; n < N; ++n) p[n] = v[n].x + fr[n] * v[n].y;
    }
  } else {
#pragma unroll
    for (int n = 0; n < N; ++n) p[n] = eos_p_t<EOS, F>(T, e[n]);
  }
}

// What a Newton step needs of the iterate e0 alone.
template <typename F>
struct NewtonAt {
  F p, w, om, dc, vi;  // p, w = p/e0, 1 - w, c_s^2 - w, (c_s^2 - w) w/e0
};
template <typename F>
__device__ __forceinline__ NewtonAt<F> newton_at(F e0, F p, F cs2) {
  NewtonAt<F> g;
  const F ie0 = rcp_t(e0);
  g.p = p;
  g.w = p * ie0;
  g.om = F(1) - g.w;
  g.dc = cs2 - g.w;
  g.vi = g.dc * g.w * ie0;
  return g;
}

// Newton step of one root-find (EnergyMomentumTensor.cu:22-44).  With w =
// p/e0, A = M0 (1 - w) + Pi, B = M0 (M0 + Pi) - M, H = sqrt|A^2 + 4 w B| and
// D = (A - H)/(2 w) the reference takes f = e0 + D and f' = 1 - num/(w e0 H),
// num = (c_s^2 - w)(B + D H - (c_s^2 - w) w D M0/e0).  Multiplied through by
// w the quotient has one division instead of three,
//   f/f' = p H (p + d) / (w p H - (c_s^2 - w)(w B + d (H - (c_s^2 - w) w M0/e0))),
// d = w D = (A - H)/2: equal up to rounding, and the halving is exact.
template <typename F>
__device__ __forceinline__ F newton_step(const NewtonAt<F> &g, F M0, F B, F Pi) {
  const F a = fma(M0, g.om, Pi);
  const F q = g.w * B;
  const F h = sqrt_t(fabs(fma(F(4), q, a * a)));
  const F d = F(0.5) * (a - h);
  const F y = fma(d, fma(-g.vi, M0, h), q);
  const F ph = g.p * h;
  return div_t(ph * (g.p + d), fma(-g.dc, y, g.w * ph));
}

// The guess of a cell's root-finds: its own energy density with p and c_s^2
// there.  The cell's own inversion and its 12 half-site ones all start from
// it, so the first iteration of each takes them from here.
template <typename F>
struct Guess {
  F e, p, cs2;
};
template <int EOS, typename F, typename Tab>
__device__ __forceinline__ Guess<F> make_guess(const Tab &T, F e) {
  Guess<F> g;
  g.e = e;
  g.p = g.cs2 = F(0);
  if constexpr (EOS != EOS_CONFORMAL) eos_p_cs2_n<EOS, 1, F>(T, &g.e, &g.p, &g.cs2);
  return g;
}

// energyDensityFromConservedVariables (EnergyMomentumTensor.cu:19-48) for N
// root-finds that share the guess, in lockstep: Newton on e, stopping at
// |de| <= 1e-3 |e|, the step damped by 0.9 after MAX_ITERS/2 iterations.
// max_iters <= MAX_ITERS bounds the iterations (the reference: MAX_ITERS).
// Every iteration evaluates all N steps without branches and a chain keeps
// its iterate once it has converged, so each result equals that of a
// root-find of its own, while the table gathers and the dependency chains of
// the N overlap.  The loop is the wave's: it ends when no lane has a chain
// left.  A NaN iterate never meets the reference's stopping rule and every
// later one is NaN, so its 10^6 iterations return NaN: the chain stops there
// and is counted as not converged.
//
// The first iteration is apart from the loop, since its p and c_s^2 are the
// guess's: no lookup, and 1/e0 and the terms of NewtonAt once for all N.  On
// a 201x201x101 lattice with every cell on this branch the FP64 stage kernel
// issues 5100 VALU instructions per wave against 6450 with three divisions per
// step, the general lookup in every iteration and a divergent loop: 2.05
// against 2.34 ms per step.
template <int EOS, int N, typename F, typename Tab>
__device__ __forceinline__ void solve_e_lockstep(const Tab &T, const Guess<F> &g, const F *M0,
                                                 const F *M, const F *Pi, F *e,
                                                 unsigned long long *diag, int max_iters) {
  if constexpr (EOS == EOS_CONFORMAL) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const F r = fabs(F(4) * M0[k] * M0[k] - F(3) * M[k]);
      e[k] = fabs((std::is_same<F, double>::value ? sqrt(r) : sqrt_t(r)) - M0[k]);
    }
  } else {
    F B[N];
    bool live[N], any = false;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      B[k] = fma(M0[k], M0[k] + Pi[k], -M[k]);
      e[k] = g.e;
      live[k] = true;
    }
    // the scheduler would mix the first steps into the code before them and
    // run out of registers
    __builtin_amdgcn_sched_barrier(0);
    if (max_iters > 0) {
      const NewtonAt<F> at = newton_at(g.e, g.p, g.cs2);
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const F step = newton_step(at, M0[k], B[k], Pi[k]);
        e[k] = g.e - step;
        // a NaN step compares false and ends the chain
        live[k] = fabs(step) > F(0.001) * fabs(e[k]);
        any = any || live[k];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    F scale = F(1), tol = F(0.001);  // of the step; tol = 0.001 / scale
    for (int it = 1; it < max_iters && __builtin_amdgcn_ballot_w64(any); ++it) {
      if (it == MAX_ITERS / 2) {
        scale = F(0.9);
        tol = F(0.001 / 0.9);
      }
      F p[N], cs2[N];
      eos_p_cs2_n<EOS, N, F>(T, e, p, cs2);
      any = false;
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const F step = newton_step(newton_at(e[k], p[k], cs2[k]), M0[k], B[k], Pi[k]);
        const F ek = fma(-scale, step, e[k]);
        e[k] = live[k] ? ek : e[k];
        live[k] = live[k] && fabs(step) > tol * fabs(ek);
        any = any || live[k];
      }
    }
#pragma unroll
    for (int k = 0; k < N; ++k) any = any || isnan(e[k]);
    if (any) {
      int bad = 0;
#pragma unroll
      for (int k = 0; k < N; ++k) bad += (live[k] || isnan(e[k])) ? 1 : 0;
      atomicAdd(&diag[DIAG_NOT_CONVERGED], (unsigned long long)bad);
    }
  }
}

template <int EOS, typename Tab>
__device__ __forceinline__ double solve_e(const Tab &T, const Guess<double> &g, double M0,
                                          double M, double Pi, unsigned long long *diag,
                                          int max_iters) {
  double e;
  solve_e_lockstep<EOS, 1, double>(T, g, &M0, &M, &Pi, &e, diag, max_iters);
  return e;
}

struct Prim {
  double e, p, ut, ux, uy, un;
};

// getInferredVariables, EnergyMomentumTensor.cu:51-108 (the '#ifdef Pi'
// consistency fix at :82-85 is never compiled in the reference; omitted)
template <int EOS, typename Tab>
__device__ __forceinline__ Prim inferred(const Tab &T, double t, double ttt,
                                         double ttx, double tty, double ttn,
                                         double pitt, double pitx, double pity,
                                         double pitn, double Pi, const Guess<double> &g,
                                         unsigned long long *diag, int max_iters) {
  double M0 = ttt - pitt, M1 = ttx - pitx, M2 = tty - pity, M3 = ttn - pitn;
  double M = M1 * M1 + M2 * M2 + t * t * M3 * M3;
  Prim r;
  r.e = (g.e <= 0.1) ? M0 - M / M0 : solve_e<EOS>(T, g, M0, M, Pi, diag, max_iters);
  if (isnan(r.e)) atomicAdd(&diag[DIAG_E_NAN], 1ull);
  r.p = eos_p<EOS>(T, r.e);
  if (r.e < 1.e-7) {
    r.e = 1.e-7;
    r.p = 1.e-7;
    atomicAdd(&diag[DIAG_E_CLAMPED], 1ull);
  }
  double P = r.p + Pi;
  double E = 1.0 / (r.e + P);
  r.ut = sqrt(fabs((M0 + P) * E));
  double E2 = E / r.ut;
  r.ux = M1 * E2;
  r.uy = M2 * E2;
  r.un = M3 * E2;
  return r;
}

// Flux velocity v = u_dir/u^tau of a half-site state, as getInferredVariables
// (EnergyMomentumTensor.cu:51-108) followed by u_dir/u^tau
// (SpectralRadius.cu, FluxFunctions.cu).  With E = 1/(e+P),
// u^tau = sqrt|(M0+P)E| and u_dir = M_dir E/u^tau, so
// v = M_dir E/|(M0+P)E| = sign(e+P) M_dir/|M0+P|: one division and no square
// root, equal up to rounding wherever e+P is finite and nonzero.
template <int EOS, int DIR, typename Tab>
__device__ __forceinline__ double flux_velocity(const Tab &T, double t, double ttt,
                                                double ttx, double tty, double ttn, double pitt,
                                                double pitx, double pity, double pitn,
                                                double Pi, const Guess<double> &g,
                                                unsigned long long *diag, int max_iters) {
  const double M0 = ttt - pitt, M1 = ttx - pitx, M2 = tty - pity, M3 = ttn - pitn;
  const double M = M1 * M1 + M2 * M2 + t * t * M3 * M3;
  double e = (g.e <= 0.1) ? M0 - M / M0 : solve_e<EOS>(T, g, M0, M, Pi, diag, max_iters);
  if (isnan(e)) atomicAdd(&diag[DIAG_E_NAN], 1ull);
  double p = eos_p<EOS>(T, e);
  if (e < 1.e-7) {
    e = 1.e-7;
    p = 1.e-7;
    atomicAdd(&diag[DIAG_E_CLAMPED], 1ull);
  }
  const double P = p + Pi;
  const double Md = DIR == 0 ? M1 : (DIR == 1 ? M2 : M3);
  return ((e + P > 0.0) ? Md : -Md) / fabs(M0 + P);
}

// flux_velocity of N half-site states of one direction that share the
// guess g, with their root-finds in lockstep (solve_e_lockstep); vacuum: the
// guess is at most 0.1 fm^-4, where the reference takes the closed form.
// W[k] = (T^tt, T^tx, T^ty, T^tn, pi^tt, pi^tx, pi^ty, pi^tn, Pi).
// In the mixed form (R = float) the root-finds of the flux states run in FP32
// for the conformal and tabulated EoS: their results only set the flux
// velocities of FP32 fluxes.  The WB fits (powers up to e^13) overflow FP32
// and stay FP64, as does every cell's own inversion.
// ROOT64 keeps them in FP64 in every form (the mixed form's split as the
// GVH_MIXED_F64_ROOTS precision states it).
template <int EOS, typename R, bool ROOT64 = false>
using flux_root_t =
    typename std::conditional<(sizeof(R) == 4 && EOS != EOS_WB && !ROOT64), float, double>::type;

template <int EOS, int DIR, int N, typename R, bool ROOT64, typename Tab>
__device__ __forceinline__ void flux_velocity_lockstep(const Tab &T, double t,
                                                       const R (*W)[9], bool vacuum,
                                                       const Guess<flux_root_t<EOS, R, ROOT64>> &g,
                                                       unsigned long long *diag, int max_iters,
                                                       double *v) {
  using F = flux_root_t<EOS, R, ROOT64>;
  F M0[N], M[N], Md[N], Pi[N], e[N];
  const F tf = F(t);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    M0[k] = (F)W[k][0] - (F)W[k][4];
    const F M1 = (F)W[k][1] - (F)W[k][5], M2 = (F)W[k][2] - (F)W[k][6],
            M3 = (F)W[k][3] - (F)W[k][7];
    M[k] = M1 * M1 + M2 * M2 + tf * tf * M3 * M3;
    Md[k] = DIR == 0 ? M1 : (DIR == 1 ? M2 : M3);
    Pi[k] = (F)W[k][8];
  }
  if (vacuum) {
#pragma unroll
    for (int k = 0; k < N; ++k) e[k] = M0[k] - div_t(M[k], M0[k]);
  } else {
    solve_e_lockstep<EOS, N, F>(T, g, M0, M, Pi, e, diag, max_iters);
  }
  F p[N];
  eos_p_n<EOS, N, F>(T, e, p);
  // NaN and clamped states are rare: one test for all N
  bool plain = true;
#pragma unroll
  for (int k = 0; k < N; ++k) plain = plain && e[k] >= F(1.e-7);
  if (!plain) {
    int nan = 0, low = 0;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      nan += isnan(e[k]) ? 1 : 0;
      if (e[k] < F(1.e-7)) {
        e[k] = p[k] = F(1.e-7);
        ++low;
      }
    }
    if (nan) atomicAdd(&diag[DIAG_E_NAN], (unsigned long long)nan);
    if (low) atomicAdd(&diag[DIAG_E_CLAMPED], (unsigned long long)low);
  }
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const F P = p[k] + Pi[k];
    v[k] = (double)div_t((e[k] + P > F(0)) ? Md[k] : -Md[k], fabs(M0[k] + P));
  }
}

}  // namespace gvh
