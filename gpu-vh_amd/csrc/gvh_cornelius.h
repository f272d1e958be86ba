// gvh_cornelius.h -- freeze-out surface elements of one lattice cell on the
// GPU: one wave (64 lanes) per cell, the cell's lines, polygons and
// polyhedra in LDS.
//
// Behaviour of the cornelius v1.3 surface finder (freezeout/cornelius-c++-1.3/
// cornelius.cpp; Huovinen & Petersen, arXiv:1206.3371):
//  * a cell has elements iff 0 < #corners(value >= v0) < 2^d
//    (cornelius.cpp:2201-2214, 2257-2272);
//  * each square (2-D face) is cut on its edges in the order (x2=0), (x1=0),
//    (x1=dx), (x2=dx) by the linear zero of value - v0; a corner exactly at
//    v0 next to one below is moved 1e-9 dx along the edge; four cuts are
//    paired by the mean corner value (cornelius.cpp:1192-1345);
//  * the lines of a cube are joined into polygons only when the cube is
//    ambiguous (a square with four cuts, or six lines), by end points within
//    1e-10 in the L1 norm, reversing a line whose end meets
//    (cornelius.cpp:436-476, 1552-1650); polygons of a hypercube are joined
//    into polyhedra only when it is ambiguous (cornelius.cpp:743-813,
//    1858-1970);
//  * polygon centroid: vertex mean for three lines, else the area-weighted
//    mean of the triangles (line, vertex mean); polyhedron centroid: the
//    volume-weighted mean of the tetrahedra (line, polygon centroid, vertex
//    mean); normals are sums of triangle / tetrahedron normals each turned
//    away from its outside point (cornelius.cpp:91-106, 478-617, 815-987).
//
// Work split: lanes 0..6*ncubes-1 cut one square each (the 8 cubes of a
// hypercube cut their squares separately, as each cube owns its squares); a
// prefix over the wave places the lines; lane q joins the lines of cube q;
// lane g builds polygon g; lane h builds polyhedron h.  The sequential parts
// keep the summation order above and the arithmetic is free of
// contractions, so results equal a plain IEEE-754 double evaluation term by
// term.
#pragma once
#include <hip/hip_runtime.h>

#pragma clang fp contract(off)

namespace gvh {
namespace corn {

constexpr int D = 4;
constexpr int MAXL = 96;    // 8 cubes x 6 squares x 2 lines
constexpr int MAXCP = 12;   // polygons of one cube (one line each at worst)
constexpr int MAXP = 96;    // polygons of a cell
constexpr int MAXE = 10;    // elements of a cell (cornelius.cpp:1703, 2004)

// A line: start, end, and the free-axis components of a point on the outside
// (its two held-axis components equal the start's; the free axes are in
// Work::oax).
struct LineRec {
  double s[D], e[D], o2[2];
};

struct Work {
  LineRec L[MAXL];
  double pcen[MAXP][D];
  unsigned char oax[MAXL];          // free axes x1 | x2 << 2 of each line
  unsigned char ord[MAXL];          // absolute line indices, polygon by polygon
  unsigned char pstart[MAXP], plen[MAXP], pcube[MAXP];
  unsigned char cpst[8][MAXCP], cplen[8][MAXCP];
  unsigned char hlist[MAXP], hfirst[MAXE], hlen[MAXE];
  short hntet[MAXE];
  unsigned char cfirst[8], cnl[8], camb[8], cnp[8];
  int np, nh, nlines, overflow;
  union {
    double tet[MAXL][D + 1];  // per-tetrahedron terms of one polyhedron (4-D cells)
    double pnrm[MAXCP][D];    // polygon normals (3-D cells)
  };
  double v[16];
  double dx[D];
  double v0;
  int dim;
};

// Component i of a 4-vector held in registers, by selects (a run-time index
// into a private array would put the array in scratch memory).
__device__ __forceinline__ double pick(const double *v, int i) {
  return i == 0 ? v[0] : (i == 1 ? v[1] : (i == 2 ? v[2] : v[3]));
}

// Cube q of a cell: the axis held constant, its value and the three free
// axes x0 < x1 < x2.  A 3-D cell is the cube with axis 0 held at 0.
__device__ __forceinline__ void cube_axes(const Work &W, int q, int &cst, double &cv, int &x0,
                                          int &x1, int &x2) {
  if (W.dim == 4) {
    cst = q >> 1;
    cv = (q & 1) * W.dx[cst];
    x0 = cst == 0 ? 1 : 0;
    x1 = cst <= 1 ? 2 : 1;
    x2 = cst <= 2 ? 3 : 2;
  } else {
    cst = 0;
    cv = 0.0;
    x0 = 1;
    x1 = 2;
    x2 = 3;
  }
}

// Corner (a, b, c) of cube q over its free axes: axis k takes q's side j if
// it is the held axis, else the next of a, b, c.
__device__ __forceinline__ double cube_value(const Work &W, int q, int a, int b, int c) {
  if (W.dim == 3) return W.v[4 * a + 2 * b + c];
  const int cst = q >> 1, j = q & 1;
  const int i0 = cst == 0 ? j : a;
  const int i1 = cst == 1 ? j : (cst == 0 ? a : b);
  const int i2 = cst == 2 ? j : (cst <= 1 ? b : c);
  const int i3 = cst == 3 ? j : c;
  return W.v[8 * i0 + 4 * i1 + 2 * i2 + i3];
}

// Cut points of one square with values sq[a][b] at (a h1, b h2) along its
// free axes x1 < x2, in the coordinates of those axes: up to four, in the
// edge order below, and the outside point of each of its nl lines (half the
// number of cut points).  Every index is fixed at compile time, so the
// result stays in registers.
struct SquareCut {
  double cut[4][2];
  double opt[2][2];
  int nl;
};

__device__ __forceinline__ SquareCut square_cut(const double sq[2][2], double h1, double h2,
                                                double v0) {
  SquareCut r;
  r.nl = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) r.cut[k][0] = r.cut[k][1] = 0.0;
  r.opt[0][0] = r.opt[0][1] = r.opt[1][0] = r.opt[1][1] = 0.0;
  int above = 0;
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b) above += sq[a][b] >= v0;
  if (above == 0 || above == 4) return r;
  // edges from corner value a to corner value b: along x1 at x2 = 0, along
  // x2 at x1 = 0, along x2 at x1 = h1, along x1 at x2 = h2
  const double ea[4] = {sq[0][0], sq[0][0], sq[1][0], sq[0][1]};
  const double eb[4] = {sq[1][0], sq[0][1], sq[1][1], sq[1][1]};
  const double fix[4] = {0.0, 0.0, h1, h2};
  const double hh[4] = {h1, h2, h2, h1};
  const bool along1[4] = {true, false, false, true};
  int nc = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const double a = ea[e], b = eb[e], h = hh[e];
    double s = 0.0;
    bool cut = true;
    if ((a - v0) * (b - v0) < 0) s = (a - v0) / (a - b) * h;
    else if (a == v0 && b < v0) s = 1e-9 * h;
    else if (b == v0 && a < v0) s = (1.0 - 1e-9) * h;
    else cut = false;
    if (cut) {
      const double p0 = along1[e] ? s : fix[e], p1 = along1[e] ? fix[e] : s;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k == nc) {
          r.cut[k][0] = p0;
          r.cut[k][1] = p1;
        }
      ++nc;
    }
  }
  if (nc == 4) {
    double mid = 0;
    for (int a = 0; a < 2; ++a)
      for (int b = 0; b < 2; ++b) mid += 0.25 * sq[a][b];
    if ((sq[0][0] < v0 && mid < v0) || (sq[0][0] > v0 && mid > v0))
      for (int k = 0; k < 2; ++k) {
        const double t = r.cut[1][k];
        r.cut[1][k] = r.cut[2][k];
        r.cut[2][k] = t;
      }
    if (mid - v0 < 0) {
      r.opt[0][0] = r.opt[1][0] = 0.5 * h1;
      r.opt[0][1] = r.opt[1][1] = 0.5 * h2;
    } else if (sq[0][0] - v0 < 0) {
      r.opt[1][0] = h1;
      r.opt[1][1] = h2;
    } else {
      r.opt[0][0] = h1;
      r.opt[1][1] = h2;
    }
  } else if (nc == 2) {
    int nout = 0;
    for (int a = 0; a < 2; ++a)
      for (int b = 0; b < 2; ++b)
        if (sq[a][b] < v0) {
          r.opt[0][0] += a * h1;
          r.opt[0][1] += b * h2;
          ++nout;
        }
    if (nout > 0) {
      r.opt[0][0] /= nout;
      r.opt[0][1] /= nout;
    }
  }
  r.nl = nc >> 1;
  return r;
}

// Line K of a square into W.L[i]: free axes x1, x2 take the cut
// coordinates, constant axes c0, c1 the values cv0, cv1.
template <int K>
__device__ __forceinline__ void store_line(Work &W, int i, const SquareCut &r, int c0, int c1,
                                           double cv0, double cv1, int x1, int x2) {
  LineRec &l = W.L[i];
  l.s[x1] = r.cut[2 * K][0];
  l.s[x2] = r.cut[2 * K][1];
  l.s[c0] = cv0;
  l.s[c1] = cv1;
  l.e[x1] = r.cut[2 * K + 1][0];
  l.e[x2] = r.cut[2 * K + 1][1];
  l.e[c0] = cv0;
  l.e[c1] = cv1;
  l.o2[0] = r.opt[K][0];
  l.o2[1] = r.opt[K][1];
  W.oax[i] = (unsigned char)(x1 | (x2 << 2));
}

// Component k of the outside point of line i.
__device__ __forceinline__ double outside(const Work &W, int i, int k) {
  const int a = W.oax[i];
  const LineRec &l = W.L[i];
  return k == (a & 3) ? l.o2[0] : (k == (a >> 2) ? l.o2[1] : l.s[k]);
}

__device__ __forceinline__ bool same_point_lt(const double *a, const double *b) {
  double d = 0;
  for (int i = 0; i < D; ++i) d += fabs(a[i] - b[i]);
  return d < 1e-10;
}

__device__ __forceinline__ bool same_point_le(const double *a, const double *b) {
  double d = 0;
  for (int i = 0; i < D; ++i) d += fabs(a[i] - b[i]);
  return d <= 1e-10;
}

__device__ __forceinline__ void orient(double *nrm, const double *outdir) {
  double dot = 0;
  for (int i = 0; i < D; ++i) dot += outdir[i] * nrm[i];
  if (dot < 0)
    for (int i = 0; i < D; ++i) nrm[i] = -nrm[i];
}

__device__ __forceinline__ void tetra_normal(const double *a, const double *b, const double *c,
                                             double *n) {
  const double bc01 = b[0] * c[1] - b[1] * c[0];
  const double bc02 = b[0] * c[2] - b[2] * c[0];
  const double bc03 = b[0] * c[3] - b[3] * c[0];
  const double bc12 = b[1] * c[2] - b[2] * c[1];
  const double bc13 = b[1] * c[3] - b[3] * c[1];
  const double bc23 = b[2] * c[3] - b[3] * c[2];
  n[0] = 1.0 / 6.0 * (a[1] * bc23 - a[2] * bc13 + a[3] * bc12);
  n[1] = -1.0 / 6.0 * (a[0] * bc23 - a[2] * bc03 + a[3] * bc02);
  n[2] = 1.0 / 6.0 * (a[0] * bc13 - a[1] * bc03 + a[3] * bc01);
  n[3] = -1.0 / 6.0 * (a[0] * bc12 - a[1] * bc02 + a[2] * bc01);
}

__device__ __forceinline__ int pline_index(const Work &W, int g, int k) {
  return W.ord[W.pstart[g] + k];
}
__device__ __forceinline__ const LineRec &pline(const Work &W, int g, int k) {
  return W.L[pline_index(W, g, k)];
}

// Centroid (and, for 3-D cells, normal) of polygon g.
__device__ void polygon_geometry(Work &W, int g, bool want_normal) {
  const int n = W.plen[g];
  int cst, x1, x2, x3;
  double cv;
  cube_axes(W, W.pcube[g], cst, cv, x1, x2, x3);
  double mean[D] = {0, 0, 0, 0};
  for (int i = 0; i < n; ++i) {
    const LineRec &l = pline(W, g, i);
    for (int j = 0; j < D; ++j) mean[j] += l.s[j] + l.e[j];
  }
  for (int j = 0; j < D; ++j) mean[j] = mean[j] / double(2.0 * n);
  double cen[D];
  if (n == 3) {
    for (int j = 0; j < D; ++j) cen[j] = mean[j];
  } else {
    double up[D] = {0, 0, 0, 0}, down = 0;
    for (int i = 0; i < n; ++i) {
      const LineRec &l = pline(W, g, i);
      double a[D], b[D], cm[D];
      for (int j = 0; j < D; ++j) {
        cm[j] = (l.s[j] + l.e[j] + mean[j]) / 3.0;
        a[j] = l.s[j] - mean[j];
        b[j] = l.e[j] - mean[j];
      }
      const double u1 = pick(a, x2) * pick(b, x3) - pick(a, x3) * pick(b, x2);
      const double u2 = pick(a, x1) * pick(b, x3) - pick(a, x3) * pick(b, x1);
      const double u3 = pick(a, x2) * pick(b, x1) - pick(a, x1) * pick(b, x2);
      const double A = 0.5 * sqrt(u1 * u1 + u2 * u2 + u3 * u3);
      for (int j = 0; j < D; ++j) up[j] += cm[j] * A;
      down += A;
    }
    for (int j = 0; j < D; ++j) cen[j] = up[j] / down;
  }
  for (int j = 0; j < D; ++j) W.pcen[g][j] = cen[j];
  if (!want_normal) return;
  double nsum[D] = {0, 0, 0, 0};
  for (int i = 0; i < n; ++i) {
    const int li = pline_index(W, g, i);
    const LineRec &l = W.L[li];
    double a[D], b[D], nrm[D], o[D];
    for (int j = 0; j < D; ++j) {
      a[j] = l.s[j] - cen[j];
      b[j] = l.e[j] - cen[j];
    }
    const double n1 = 0.5 * (pick(a, x2) * pick(b, x3) - pick(a, x3) * pick(b, x2));
    const double n2 = -0.5 * (pick(a, x1) * pick(b, x3) - pick(a, x3) * pick(b, x1));
    const double n3 = 0.5 * (pick(a, x1) * pick(b, x2) - pick(a, x2) * pick(b, x1));
    for (int j = 0; j < D; ++j) nrm[j] = j == x1 ? n1 : (j == x2 ? n2 : (j == x3 ? n3 : 0.0));
    for (int j = 0; j < D; ++j) o[j] = outside(W, li, j) - cen[j];
    orient(nrm, o);
    for (int j = 0; j < D; ++j) nsum[j] += nrm[j];
  }
  for (int j = 0; j < D; ++j) W.pnrm[g][j] = nsum[j];
}

// Polygon g and line j of tetrahedron t of a polyhedron whose np polygons
// are listed from W.hlist[first]: its lines polygon by polygon.
__device__ __forceinline__ void tet_line(const Work &W, int first, int np, int t, int &g, int &j) {
  g = W.hlist[first];
  j = 0;
  for (int i = 0; i < np; ++i) {
    const int gi = W.hlist[first + i];
    const int n = W.plen[gi];
    if (t < n) {
      g = gi;
      j = t;
      return;
    }
    t -= n;
  }
}

// Centroid and normal of polyhedron h, called by all lanes of the wave.  The
// tetrahedra (one per line of each polygon, at most 96) are spread over the
// lanes, lane l taking tetrahedra l and l + 64; their terms go to W.tet and
// every lane sums the rows in tetrahedron order, the order of the
// reference's serial loops, so the sums round the same way.
__device__ void polyhedron_geometry(Work &W, int h, int lane, double *cen_out, double *nrm_out) {
  const int first = W.hfirst[h], np = W.hlen[h], ntet = W.hntet[h];
  static_assert(MAXL <= 128, "two tetrahedra per lane");
  int g[2] = {0, 0}, j[2] = {0, 0}, li[2] = {0, 0};
  const LineRec *ln[2] = {nullptr, nullptr};
#pragma unroll
  for (int r = 0; r < 2; ++r)
    if (lane + 64 * r < ntet) {
      tet_line(W, first, np, lane + 64 * r, g[r], j[r]);
      li[r] = pline_index(W, g[r], j[r]);
      ln[r] = &W.L[li[r]];
    }
  // mean of the line end points
#pragma unroll
  for (int r = 0; r < 2; ++r)
    if (ln[r])
      for (int k = 0; k < D; ++k) W.tet[lane + 64 * r][k] = ln[r]->s[k] + ln[r]->e[k];
  __syncthreads();
  double mean[D] = {0, 0, 0, 0};
#pragma unroll 4
  for (int t = 0; t < ntet; ++t)
    for (int k = 0; k < D; ++k) mean[k] += W.tet[t][k];
  for (int k = 0; k < D; ++k) mean[k] = mean[k] / double(2.0 * ntet);
  __syncthreads();
  // volume-weighted centroid
#pragma unroll
  for (int r = 0; r < 2; ++r)
    if (ln[r]) {
      const LineRec &l = *ln[r];
      const double *pc = W.pcen[g[r]];
      double a[D], b[D], c[D], n[D], cm[D];
      for (int k = 0; k < D; ++k) {
        cm[k] = (l.s[k] + l.e[k] + pc[k] + mean[k]) / 4.0;
        a[k] = l.s[k] - mean[k];
        b[k] = l.e[k] - mean[k];
        c[k] = pc[k] - mean[k];
      }
      tetra_normal(a, b, c, n);
      double V = 0;
      for (int k = 0; k < D; ++k) V += n[k] * n[k];
      V = sqrt(V);
      for (int k = 0; k < D; ++k) W.tet[lane + 64 * r][k] = cm[k] * V;
      W.tet[lane + 64 * r][D] = V;
    }
  __syncthreads();
  double up[D] = {0, 0, 0, 0}, down = 0;
#pragma unroll 4
  for (int t = 0; t < ntet; ++t) {
    for (int k = 0; k < D; ++k) up[k] += W.tet[t][k];
    down += W.tet[t][D];
  }
  double cen[D];
  for (int k = 0; k < D; ++k) cen[k] = up[k] / down;
  __syncthreads();
  // normal: the oriented tetrahedron normals about the centroid
#pragma unroll
  for (int r = 0; r < 2; ++r)
    if (ln[r]) {
      const LineRec &l = *ln[r];
      const double *pc = W.pcen[g[r]];
      double a[D], b[D], c[D], n[D], o[D];
      for (int k = 0; k < D; ++k) {
        a[k] = l.s[k] - cen[k];
        b[k] = l.e[k] - cen[k];
        c[k] = pc[k] - cen[k];
        o[k] = outside(W, li[r], k) - cen[k];
      }
      tetra_normal(a, b, c, n);
      orient(n, o);
      for (int k = 0; k < D; ++k) W.tet[lane + 64 * r][k] = n[k];
    }
  __syncthreads();
  double nrm[D] = {0, 0, 0, 0};
#pragma unroll 4
  for (int t = 0; t < ntet; ++t)
    for (int k = 0; k < D; ++k) nrm[k] += W.tet[t][k];
  if (lane == 0)
    for (int k = 0; k < D; ++k) {
      cen_out[k] = cen[k];
      nrm_out[k] = nrm[k];
    }
  __syncthreads();
}

// Lines joined into polyhedra when the start or the end of a line of the
// candidate polygon is the start of a line already in the polyhedron.
__device__ bool polygons_touch(const Work &W, int gi, int gq) {
  for (int a = 0; a < W.plen[gi]; ++a) {
    const LineRec &l1 = pline(W, gi, a);
    for (int b = 0; b < W.plen[gq]; ++b) {
      const LineRec &l2 = pline(W, gq, b);
      if (same_point_le(l1.s, l2.s) || same_point_le(l1.e, l2.s)) return true;
    }
  }
  return false;
}

// Elements of the cell whose corners W.v, spacings W.dx, iso-value W.v0 and
// dimension W.dim are set.  Called by all 64 lanes of a one-wave workgroup;
// returns the element count (<= MAXE) to every lane and leaves centroid i /
// normal i in cen[i], nrm[i] (4-vectors; a 3-D cell uses axes 1..3).
__device__ int cell_elements(Work &W, double (*cen)[D], double (*nrm)[D]) {
  const int lane = threadIdx.x;
  const int ncube = W.dim == 4 ? 8 : 1;
  // no element unless the cell has corners on both sides
  {
    const int nc = 1 << W.dim;
    int above = 0;
    for (int i = 0; i < nc; ++i) above += W.v[i] >= W.v0;
    if (above == 0 || above == nc) return 0;
  }
  // --- 1: squares -> lines
  SquareCut sc;
  sc.nl = 0;
  int c0 = 0, c1 = 0, x1 = 0, x2 = 0;
  double cv0 = 0.0, cv1 = 0.0;
  const int q = lane / 6, r = lane % 6, f = r >> 1, jj = r & 1;
  if (lane < 6 * ncube) {
    // square (f, jj) of cube q: free axis f held at side jj
    int cst, a0, a1, a2;
    double cv;
    cube_axes(W, q, cst, cv, a0, a1, a2);
    double sq[2][2];
    for (int a = 0; a < 2; ++a)
      for (int b = 0; b < 2; ++b)
        sq[a][b] = f == 0 ? cube_value(W, q, jj, a, b)
                          : (f == 1 ? cube_value(W, q, a, jj, b) : cube_value(W, q, a, b, jj));
    const int xf = f == 0 ? a0 : (f == 1 ? a1 : a2);
    x1 = f == 0 ? a1 : a0;
    x2 = f == 2 ? a1 : a2;
    c0 = cst;
    c1 = xf;
    cv0 = cv;
    cv1 = jj * W.dx[xf];
    sc = square_cut(sq, W.dx[x1], W.dx[x2], W.v0);
  }
  const int cnt = sc.nl;
  const unsigned long long b1 = __ballot(cnt >= 1), b2 = __ballot(cnt == 2);
  const unsigned long long lt = (1ull << lane) - 1ull;
  const int pos = __popcll(b1 & lt) + __popcll(b2 & lt);
  if (cnt >= 1) store_line<0>(W, pos, sc, c0, c1, cv0, cv1, x1, x2);
  if (cnt == 2) store_line<1>(W, pos + 1, sc, c0, c1, cv0, cv1, x1, x2);
  if (lane < ncube) {
    const unsigned long long below = (1ull << (6 * lane)) - 1ull;
    const unsigned long long mine = 0x3full << (6 * lane);
    W.cfirst[lane] = __popcll(b1 & below) + __popcll(b2 & below);
    W.cnl[lane] = __popcll(b1 & mine) + __popcll(b2 & mine);
    W.camb[lane] = __popcll(b2 & mine);
  }
  if (lane == 0) W.nlines = __popcll(b1) + __popcll(b2);
  __syncthreads();
  // --- 2: lines of each cube -> polygons
  if (lane < ncube) {
    const int nl = W.cnl[lane], first = W.cfirst[lane];
    int amb = W.camb[lane], np = 0;
    if (nl > 0) {
      if (amb == 0 && nl == 6) amb = 1;
      if (amb > 0) {
        unsigned freem = (1u << nl) - 1u;
        int used = 0, pos2 = 0;
        do {
          const int start = pos2;
          int n = 0;
          double le[D] = {0, 0, 0, 0};
          // after an addition the scan restarts; the reference resets its
          // counter to 0 and the loop increment resumes it at 1
          for (int i = 0; i < nl; ++i) {
            if (!((freem >> i) & 1u)) continue;
            LineRec &l = W.L[first + i];
            bool add = n == 0;
            if (!add) {
              const bool sm = same_point_lt(l.s, le), em = same_point_lt(l.e, le);
              if (sm || em) {
                if (em)
                  for (int k = 0; k < D; ++k) {
                    const double t = l.s[k];
                    l.s[k] = l.e[k];
                    l.e[k] = t;
                  }
                add = true;
              }
            }
            if (add) {
              W.ord[first + pos2++] = (unsigned char)(first + i);
              freem &= ~(1u << i);
              ++used;
              ++n;
              for (int k = 0; k < D; ++k) le[k] = l.e[k];
              i = 0;
            }
          }
          W.cpst[lane][np] = (unsigned char)(first + start);
          W.cplen[lane][np] = (unsigned char)n;
          ++np;
        } while (used < nl);
      } else {
        for (int i = 0; i < nl; ++i) W.ord[first + i] = (unsigned char)(first + i);
        W.cpst[lane][0] = (unsigned char)first;
        W.cplen[lane][0] = (unsigned char)nl;
        np = 1;
      }
    }
    W.camb[lane] = amb;
    W.cnp[lane] = np;
  }
  __syncthreads();
  if (lane == 0) {
    int g = 0;
    for (int c = 0; c < ncube; ++c)
      for (int p = 0; p < W.cnp[c]; ++p, ++g) {
        W.pstart[g] = W.cpst[c][p];
        W.plen[g] = W.cplen[c][p];
        W.pcube[g] = (unsigned char)c;
      }
    W.np = g;
  }
  __syncthreads();
  // --- 3: polygon centroids (and normals of a 3-D cell's polygons)
  for (int g = lane; g < W.np; g += 64) polygon_geometry(W, g, W.dim == 3);
  __syncthreads();
  if (W.dim == 3) {
    const int ne = W.np < MAXE ? W.np : MAXE;
    if (lane < ne)
      for (int k = 0; k < D; ++k) {
        cen[lane][k] = W.pcen[lane][k];
        nrm[lane][k] = W.pnrm[lane][k];
      }
    if (lane == 0 && W.np > MAXE) W.overflow = 1;
    return ne;
  }
  // --- 4: polygons -> polyhedra
  // ambiguous: the cubes that are, or the 24-line pattern of two corners
  bool joins = __ballot(lane < 8 && W.camb[lane < 8 ? lane : 0]) != 0ull;
  if (!joins && W.nlines == 24) {
    const int below = __popcll(__ballot(lane < 16 && W.v[lane < 16 ? lane : 0] < W.v0));
    joins = below == 2 || below == 14;
  }
  const int np = W.np;
  // Row j: the polygons that touch polygon j, all pairs at once.  Scanned by
  // one lane, line against line, the joining was 80 of a cell's 125 us.
  auto touching = reinterpret_cast<unsigned long long(*)[2]>(W.tet);
  if (joins) {
    for (int j = lane; j < np; j += 64) touching[j][0] = touching[j][1] = 0ull;
    __syncthreads();
    for (int t = lane; t < np * np; t += 64) {
      const int i = t / np, j = t - i * np;
      if (i != j && polygons_touch(W, i, j)) atomicOr(&touching[j][i >> 6], 1ull << (i & 63));
    }
    __syncthreads();
  }
  if (lane == 0) {
    int nh = 0;
    if (joins) {
      // a polyhedron begins with the first polygon that is left and takes, one
      // by one, the first left that touches any of its own
      unsigned long long left0 = np >= 64 ? ~0ull : (1ull << np) - 1ull;
      unsigned long long left1 = np > 64 ? (1ull << (np - 64)) - 1ull : 0ull;
      int pos3 = 0;
      do {
        const int first = pos3;
        int ntet = 0;
        unsigned long long t0 = ~0ull, t1 = ~0ull;
        while ((t0 & left0) | (t1 & left1)) {
          const int i = t0 & left0 ? __builtin_ctzll(t0 & left0) : 64 + __builtin_ctzll(t1 & left1);
          if (pos3 == first) t0 = t1 = 0ull;
          t0 |= touching[i][0];
          t1 |= touching[i][1];
          if (i < 64) left0 &= ~(1ull << i);
          else left1 &= ~(1ull << (i - 64));
          W.hlist[pos3++] = (unsigned char)i;
          ntet += W.plen[i];
        }
        W.hfirst[nh] = (unsigned char)first;
        W.hlen[nh] = (unsigned char)(pos3 - first);
        W.hntet[nh] = (short)ntet;
        ++nh;
      } while ((left0 | left1) && nh < MAXE);
      if (left0 | left1) W.overflow = 1;
    } else {
      int ntet = 0;
      for (int i = 0; i < np; ++i) {
        W.hlist[i] = (unsigned char)i;
        ntet += W.plen[i];
      }
      W.hfirst[0] = 0;
      W.hlen[0] = (unsigned char)np;
      W.hntet[0] = (short)ntet;
      nh = 1;
    }
    W.nh = nh;
  }
  __syncthreads();
  // --- 5: polyhedron centroids and normals
  const int nh = W.nh;
  for (int h = 0; h < nh; ++h) polyhedron_geometry(W, h, lane, cen[h], nrm[h]);
  return nh;
}

// ------------------------------------------------ plain cells, one per lane
// A plain cell has no square with four cuts, no cube whose six lines are two
// triangles, and polygons that are one polyhedron: nearly every cell of a
// smooth surface.  Which lines it has, and the order in which the general
// search lists them, then follow from the corner pattern alone:
//  * a cube with three to five lines is one polygon, its lines in square
//    order; one with six is a hexagon, followed from its first line around,
//    turning lines whose end meets;
//  * the polygons come in cube order, or, where a hexagon (or the 24-line
//    pattern of two corners) makes the cell ambiguous, each time the first
//    one that shares a square with those before it.
// So a lane takes a whole cell: it lists its lines by its cubes' patterns, computes the
// cut of each of the 32 edges once (the squares that share an edge cut it at
// the same point) and goes over the list four times, summing in the general
// search's order: the element equals its bit by bit.  End points are matched
// by edge where the general search matches coordinates within 1e-10; cells
// with a cut that near a corner are left to it.

// Corner pattern of a cell (corner c = sum of side * 2^(d-1-axis)): bit c is
// set where the value is at least v0.  False for values that are no number,
// or so near v0 that the product of two differences could vanish.
template <int NC>
__device__ __forceinline__ bool corner_mask(const double *v, double v0, unsigned &above) {
  bool odd = false;
  above = 0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const double d = v[c] - v0;
    above |= (v[c] >= v0 ? 1u : 0u) << c;
    odd = odd || !(fabs(d) >= 1e-140 || d == 0.0);
  }
  return !odd;
}

// Cut of the edge from value a to value b (exactly one of them below v0).
__device__ __forceinline__ double edge_cut(double a, double b, double v0, double h) {
  if (a == v0) return 1e-9 * h;
  if (b == v0) return (1.0 - 1e-9) * h;
  return (a - v0) / (a - b) * h;
}

// x / 3, correctly rounded: quotient by the rounded reciprocal and one
// residual correction (Markstein).
__device__ __forceinline__ double third(double x) {
  const double r = 1.0 / 3.0, q = x * r;
  return fma(fma(-3.0, q, x), r, q);
}

// 1 / (2 n) for a polygon of n = 3..6 lines, and x / (2 n) from it, correctly
// rounded in the same way.
__device__ __forceinline__ double one_over_twice(int n) {
  int hi = n == 3 ? 0x3fc55555 : (n == 4 ? 0x3fc00000 : (n == 5 ? 0x3fb99999 : 0x3fb55555));
  int lo = n == 4 ? 0 : (n == 5 ? (int)0x9999999au : 0x55555555);
  // the words stay selects; seen as a double, they become four branches
  asm("" : "+v"(hi), "+v"(lo));
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double over_twice(double x, int n, double r) {
  const double q = x * r;
  return fma(fma(-double(2 * n), q, x), r, q);
}

// x / b, correctly rounded, from r = 1 / b correctly rounded: one residual
// correction makes the quotient faithful, a second one exact.
__device__ __forceinline__ double quotient(double x, double b, double r) {
  double q = x * r;
  q = fma(fma(-b, q, x), r, q);
  return fma(fma(-b, q, x), r, q);
}

// Squares of a cell: number 6 q + r, q = 2 a + j the cube that holds axis a
// at side j, r = 2 f + jj its square that holds the cube's f-th free axis at
// side jj.  A 3-D cell is the cube q = 0 with corners 0..7.
struct SquareInfo {
  unsigned base, w1, w2;  // corner (0, 0); corner weights of the free axes
  unsigned x1, x2;        // free axes x1 < x2
  unsigned edge[4];       // edges (x2 = 0), (x1 = 0), (x1 = h1), (x2 = h2)
};
// Edge number: axis * 8 + the corner's sides along the other axes.
__host__ __device__ constexpr unsigned edge_number(unsigned d, unsigned corner) {
  return d * 8 + ((corner >> (4 - d)) << (3 - d) | (corner & ((8u >> d) - 1u)));
}
__host__ __device__ constexpr SquareInfo square_info(unsigned n) {
  const unsigned q = n / 6, r = n - 6 * q, a = q >> 1, j = q & 1, f = r >> 1, jj = r & 1;
  const unsigned i1 = f == 0 ? 1 : 0, i2 = f == 2 ? 1 : 2;
  const unsigned xf = f + (f >= a ? 1u : 0u), x1 = i1 + (i1 >= a ? 1u : 0u), x2 = i2 + (i2 >= a ? 1u : 0u);
  const unsigned base = j * (8u >> a) + jj * (8u >> xf), w1 = 8u >> x1, w2 = 8u >> x2;
  return SquareInfo{base, w1, w2, x1, x2,
                    {edge_number(x1, base), edge_number(x2, base), edge_number(x2, base + w1),
                     edge_number(x1, base + w2)}};
}
// Corners (0,0), (0,1), (1,0), (1,1) of a square above v0, as bits 0..3.
__host__ __device__ constexpr unsigned square_bits(unsigned base, unsigned w1, unsigned w2, unsigned m) {
  const unsigned b = m >> base;
  return (b & 1u) | ((b >> w2) & 1u) << 1 | ((b >> w1) & 1u) << 2 | ((b >> (w1 + w2)) & 1u) << 3;
}

// What the pattern of a cube's eight corners says of it: its lines in the
// order and direction in which the general search joins them, each as start
// edge | end edge << 5 | square << 10.
struct alignas(16) CubeLines {
  unsigned short line[6];
  unsigned info;  // number of lines; flags; the squares that are cut << 8
};
constexpr unsigned CUBE_NLINES = 7u, CUBE_NOT_PLAIN = 8u, CUBE_HEXAGON = 16u;
struct CubePatterns {
  CubeLines p[256];
};
constexpr CubePatterns cube_patterns(unsigned q) {
  CubePatterns T{};
  const unsigned a = q >> 1;
  SquareInfo sq[6] = {};
  for (unsigned r = 0; r < 6; ++r) sq[r] = square_info(6 * q + r);
  for (unsigned pat = 0; pat < 256; ++pat) {
    // the cell's corners on this cube
    unsigned m = 0, above = 0;
    for (unsigned i = 0; i < 8; ++i) {
      const unsigned low = i & ((8u >> a) - 1u), c = (i - low) << 1 | (q & 1 ? 8u >> a : 0u) | low;
      m |= ((pat >> i) & 1u) << c;
      above += (pat >> i) & 1u;
    }
    unsigned first[6] = {}, last[6] = {}, cut = 0, n = 0;
    bool crossed = false;
    for (unsigned r = 0; r < 6; ++r) {
      const unsigned b = square_bits(sq[r].base, sq[r].w1, sq[r].w2, m);
      if (b == 0 || b == 15) continue;
      if (b == 6 || b == 9) crossed = true;
      const unsigned c[4] = {((b >> 2) ^ b) & 1u, ((b >> 1) ^ b) & 1u, ((b >> 3) ^ (b >> 2)) & 1u,
                             ((b >> 3) ^ (b >> 1)) & 1u};
      first[r] = sq[r].edge[c[0] ? 0 : (c[1] ? 1 : 2)];
      last[r] = sq[r].edge[c[3] ? 3 : (c[2] ? 2 : 1)];
      cut |= 1u << r;
      ++n;
    }
    CubeLines &L = T.p[pat];
    // two opposite corners apart from the six others: two triangles
    if (crossed || (n == 6 && (above == 2 || above == 6))) {
      L.info = CUBE_NOT_PLAIN;
      continue;
    }
    L.info = n | (n == 6 ? CUBE_HEXAGON : 0u) | cut << 8;
    unsigned left = cut, end = 0;
    for (unsigned k = 0; k < n; ++k) {
      unsigned r = 0;
      while (!((left >> r) & 1u)) ++r;
      bool turned = false;
      if (n == 6 && k > 0) {
        // around the hexagon: the first line left that begins or ends here
        while (!(((left >> r) & 1u) && (first[r] == end || last[r] == end))) ++r;
        turned = last[r] == end;
      }
      left &= ~(1u << r);
      end = turned ? first[r] : last[r];
      L.line[k] = (unsigned short)((turned ? last[r] : first[r]) | end << 5 | (6 * q + r) << 10);
    }
  }
  return T;
}
constexpr CubePatterns CUBE0 = cube_patterns(0), CUBE1 = cube_patterns(1), CUBE2 = cube_patterns(2),
                       CUBE3 = cube_patterns(3), CUBE4 = cube_patterns(4), CUBE5 = cube_patterns(5),
                       CUBE6 = cube_patterns(6), CUBE7 = cube_patterns(7);
__device__ const CubePatterns CUBES[8] = {CUBE0, CUBE1, CUBE2, CUBE3, CUBE4, CUBE5, CUBE6, CUBE7};

// The eight corners of the cube that holds axis a at side j, as bits.
__device__ __forceinline__ unsigned cube_corners(unsigned m, unsigned a, unsigned j) {
  unsigned x = m >> (j * (8u >> a));
  if (a == 0) return x & 255u;
  if (a == 1) return (x & 15u) | ((x >> 4) & 0xf0u);
  if (a == 3) {
    x &= 0x5555u;
    x = (x | x >> 1) & 0x3333u;
  } else {
    x &= 0x3333u;
  }
  x = (x | x >> 2) & 0x0f0fu;
  return (x | x >> 4) & 255u;
}

// LDS of a wave of plain cells; columns are lanes.  A line in the list is its
// two edges and its square.
template <int DIM>
struct PlainLds {
  static constexpr int LINES = DIM == 4 ? MAXL / 2 : 6;
  double E[32 * 64];                     // edge cuts
  double pc[DIM == 4 ? 8 * D * 64 : 1];  // polygon centroids, by cube
  double2 at[32][2];                     // position of an edge: its held coordinates
  double mean[5][4];                     // by class and axis: mean of corners below v0
  unsigned sq[48];                       // base | w1 << 4 | w2 << 8 | x1 << 12 | x2 << 14
  unsigned short list[(LINES + 1) * 64]; // start edge | end edge << 5 | square << 10; a row to spare
};

// Mean of the corners of a square below v0 along one of its free axes, of
// length h, by how many of them lie on the far side and how many there are:
// 0, h/2, h, h/3, 2h/3 (classes 0..4; MEAN_CLASS1 and 2 hold those of the
// square's two axes, three bits for each pattern of corners below).
__device__ __forceinline__ double class_mean(unsigned k, double h) {
  return k == 0 ? 0.0 : (k == 1 ? 0.5 * h : (k == 2 ? h : third(k == 3 ? h : h + h)));
}
constexpr unsigned long long mean_classes(unsigned far) {
  unsigned long long t = 0;
  for (unsigned low = 1; low < 15; ++low) {
    unsigned n = 0, n1 = 0;
    for (unsigned i = 0; i < 4; ++i) {
      n += (low >> i) & 1u;
      n1 += ((low & far) >> i) & 1u;
    }
    const unsigned k = n1 == 0 ? 0 : (n == 3 ? 2 + n1 : (n == 2 && n1 == 1 ? 1 : 2));
    t |= (unsigned long long)k << (3 * low);
  }
  return t;
}
constexpr unsigned long long MEAN_CLASS1 = mean_classes(12u), MEAN_CLASS2 = mean_classes(10u);

template <int DIM>
__device__ __forceinline__ void plain_tables(PlainLds<DIM> &S, int lane, const double *h) {
  if (lane < (DIM == 4 ? 48 : 6)) {
    const SquareInfo q = square_info(lane);
    S.sq[lane] = q.base | q.w1 << 4 | q.w2 << 8 | q.x1 << 12 | q.x2 << 14;
  }
  if (lane < 20) {
    const unsigned x = lane & 3u;
    S.mean[lane >> 2][x] = class_mean(lane >> 2, x == 0 ? h[0] : (x == 1 ? h[1] : (x == 2 ? h[2] : h[3])));
  }
  if (lane < 32) {
    const unsigned d = lane >> 3, pos = lane & 7u;
    const unsigned c = (pos >> (3 - d)) << (4 - d) | (pos & ((8u >> d) - 1u));
    S.at[lane][0] = double2{c & 8u ? h[0] : 0.0, c & 4u ? h[1] : 0.0};
    S.at[lane][1] = double2{c & 2u ? h[2] : 0.0, c & 1u ? h[3] : 0.0};
  }
}

// The cut point of an edge in four coordinates.
template <int DIM>
__device__ __forceinline__ void edge_point(const PlainLds<DIM> &S, int lane, unsigned edge,
                                           double *x) {
  const double2 a = S.at[edge][0], b = S.at[edge][1];
  const double c = S.E[64 * edge + lane];
  const unsigned d = edge >> 3;
  x[0] = d == 0 ? c : a.x;
  x[1] = d == 1 ? c : a.y;
  x[2] = d == 2 ? c : b.x;
  x[3] = d == 3 ? c : b.y;
}
struct Line4 {
  double s[D], e[D];
};
template <int DIM>
__device__ __forceinline__ Line4 plain_line(const PlainLds<DIM> &S, int lane, unsigned id) {
  Line4 l;
  edge_point(S, lane, id & 31u, l.s);
  edge_point(S, lane, (id >> 5) & 31u, l.e);
  return l;
}
// body(line, id, whether it is a polygon's last) for the lines of the lane's
// list; bit i of ends is set for a polygon's last line.  The next line and the
// number of the one after it are fetched while the body works on this one: a
// line is two dependent LDS reads, and few waves fit a CU to hide them.
template <int DIM, typename B>
__device__ __forceinline__ void for_lines(const PlainLds<DIM> &S, int lane, int nl,
                                          unsigned long long ends, B &&body) {
  auto number = [&](int i) -> unsigned { return S.list[64 * (i < nl ? i : 0) + lane]; };
  unsigned id = number(0), idn = number(1);
  Line4 l = plain_line(S, lane, id);
#pragma unroll 1
  for (int i = 2; i <= nl + 1; ++i) {
    const unsigned idnn = number(i);
    const Line4 ln = plain_line(S, lane, idn);
    body(l, id, (bool)(ends & 1ull));
    ends >>= 1;
    l = ln;
    id = idn;
    idn = idnn;
  }
}

// Outside point of a line (outside() of the general search).
template <int DIM>
__device__ __forceinline__ void plain_outside(const PlainLds<DIM> &S, unsigned id, unsigned m,
                                              const double *s, double *o) {
  const unsigned q = S.sq[id >> 10], x1 = (q >> 12) & 3u, x2 = q >> 14;
  const unsigned low = ~square_bits(q & 15u, (q >> 4) & 15u, (q >> 8) & 15u, m) & 15u;
  const double o1 = S.mean[(unsigned)(MEAN_CLASS1 >> (3 * low)) & 7u][x1];
  const double o2 = S.mean[(unsigned)(MEAN_CLASS2 >> (3 * low)) & 7u][x2];
#pragma unroll
  for (unsigned k = 0; k < D; ++k) o[k] = k == x1 ? o1 : (k == x2 ? o2 : s[k]);
}

// Lists the lines of the lane's cell (corner pattern m; near: an edge cut
// within 1e-10 of a corner); the number of lines, or 0 if the cell is not
// plain.  ends: the last lines of polygons.  The eight cubes are looked up
// together and written without branches: following the lines of one cube
// after another, each lane through its own cubes, took 24 000 cycles of a
// window's 188 000 per wave, and 56 000 where one cell in ten has a hexagon.
template <int DIM>
__device__ __forceinline__ int list_lines(PlainLds<DIM> &S, int lane, unsigned m, bool near,
                                          unsigned long long &ends) {
  constexpr unsigned NQ = DIM == 4 ? 8 : 1;
  CubeLines c[NQ];
#pragma unroll
  for (unsigned q = 0; q < NQ; ++q) c[q] = CUBES[q].p[cube_corners(m, q >> 1, q & 1)];
  unsigned any = 0, present = 0, nlines = 0;
#pragma unroll
  for (unsigned q = 0; q < NQ; ++q) {
    const unsigned n = c[q].info & CUBE_NLINES;
    any |= c[q].info;
    present |= (n ? 1u : 0u) << q;
    nlines += n;
  }
  if (any & CUBE_NOT_PLAIN) return 0;
  bool joined = any & CUBE_HEXAGON;
  if constexpr (DIM == 4) {
    const int na = __popc(m);
    joined = joined || (nlines == 24 && (na == 2 || na == 14));
  }
  if (joined && near) return 0;
  unsigned pos[NQ];  // of the cube's first line
  unsigned at = 0;
#pragma unroll
  for (unsigned q = 0; q < NQ; ++q) {
    pos[q] = at;
    at += c[q].info & CUBE_NLINES;
  }
  if constexpr (DIM == 4)
    if (joined) {
      // cubes in the order in which they touch those before, the lowest first:
      // bytes by cube of the cubes that share a cut square with it (the held
      // axes of its cut squares) and of its lines; bytes by cube of positions
      unsigned long long touching = 0, lengths = 0, posq = 0;
#pragma unroll
      for (unsigned q = 0; q < NQ; ++q) {
        const unsigned f = (c[q].info >> 8) & 63u, a2 = q & ~1u;
        touching |= (unsigned long long)((f & ((1u << a2) - 1u)) | (f >> a2) << (a2 + 2)) << (8 * q);
        lengths |= (unsigned long long)(c[q].info & CUBE_NLINES) << (8 * q);
      }
      unsigned left = present, touch = 255u;
      at = 0;
#pragma unroll 1
      while (left & touch) {
        const unsigned q = (unsigned)__builtin_ctz(left & touch);
        posq |= (unsigned long long)at << (8 * q);
        at += (unsigned)(lengths >> (8 * q)) & 255u;
        touch = (left == present ? 0u : touch) | ((unsigned)(touching >> (8 * q)) & 255u);
        left &= ~(1u << q);
      }
      if (left) return 0;
#pragma unroll
      for (unsigned q = 0; q < NQ; ++q) pos[q] = (unsigned)(posq >> (8 * q)) & 255u;
    }
  ends = 0;
#pragma unroll
  for (unsigned q = 0; q < NQ; ++q) {
    const unsigned n = c[q].info & CUBE_NLINES;
    if constexpr (DIM == 4) ends |= n ? 1ull << (pos[q] + n - 1) : 0ull;
#pragma unroll
    for (unsigned k = 0; k < 6; ++k)
      S.list[64 * (k < n ? pos[q] + k : (unsigned)PlainLds<DIM>::LINES) + lane] = c[q].line[k];
  }
  return (int)nlines;
}

// Element of the lane's plain 4-D cell of nl lines.  The sums are those of
// polygon_geometry and polyhedron_geometry, term by term.
__device__ __forceinline__ void plain_element4(PlainLds<4> &S, int lane, unsigned m, int nl,
                                               unsigned long long ends, const double *h, double *cen,
                                               double *nrm) {
  auto pc = [&](unsigned id, int k) -> double & { return S.pc[64 * ((id >> 10) / 6 * D + k) + lane]; };
  // polygon means and the mean of all lines
  double mean[D] = {0, 0, 0, 0}, pm[D] = {0, 0, 0, 0};
  int n = 0;
  for_lines(S, lane, nl, ends, [&](const Line4 &l, unsigned id, bool last) {
    for (int k = 0; k < D; ++k) {
      const double t = l.s[k] + l.e[k];
      pm[k] += t;
      mean[k] += t;
    }
    ++n;
    if (last) {
      const double r = one_over_twice(n);
      for (int k = 0; k < D; ++k) {
        pc(id, k) = over_twice(pm[k], n, r);
        pm[k] = 0;
      }
      n = 0;
    }
  });
  for (int k = 0; k < D; ++k) mean[k] = mean[k] / double(2.0 * nl);
  // area-weighted centroids of the polygons with more than three lines
  double up[D] = {0, 0, 0, 0}, down = 0;
  for_lines(S, lane, nl, ends, [&](const Line4 &l, unsigned id, bool last) {
    double a[D], b[D], c[D];
    for (int k = 0; k < D; ++k) {
      c[k] = pc(id, k);
      a[k] = l.s[k] - c[k];
      b[k] = l.e[k] - c[k];
    }
    // the cube's free axes in order
    const unsigned held = (id >> 10) / 12;
    auto free_axis = [&](const double *v, int i) {
      return (unsigned)i < held ? v[i] : v[i + 1];
    };
    const double a1 = free_axis(a, 0), a2 = free_axis(a, 1), a3 = free_axis(a, 2);
    const double b1 = free_axis(b, 0), b2 = free_axis(b, 1), b3 = free_axis(b, 2);
    const double u1 = a2 * b3 - a3 * b2;
    const double u2 = a1 * b3 - a3 * b1;
    const double u3 = a2 * b1 - a1 * b2;
    const double ar = 0.5 * sqrt(u1 * u1 + u2 * u2 + u3 * u3);
    for (int k = 0; k < D; ++k) up[k] += third(l.s[k] + l.e[k] + c[k]) * ar;
    down += ar;
    ++n;
    if (last) {
      if (n > 3) {
        const double r = 1.0 / down;
        for (int k = 0; k < D; ++k) pc(id, k) = quotient(up[k], down, r);
      }
      for (int k = 0; k < D; ++k) up[k] = 0;
      down = 0;
      n = 0;
    }
  });
  // volume-weighted centroid of the polyhedron
  for_lines(S, lane, nl, ends, [&](const Line4 &l, unsigned id, bool) {
    double a[D], b[D], c[D], t[D];
    for (int k = 0; k < D; ++k) {
      t[k] = pc(id, k);
      a[k] = l.s[k] - mean[k];
      b[k] = l.e[k] - mean[k];
      c[k] = t[k] - mean[k];
      t[k] = (l.s[k] + l.e[k] + t[k] + mean[k]) / 4.0;
    }
    double nv[D];
    tetra_normal(a, b, c, nv);
    double V = 0;
    for (int k = 0; k < D; ++k) V += nv[k] * nv[k];
    V = sqrt(V);
    for (int k = 0; k < D; ++k) up[k] += t[k] * V;
    down += V;
  });
  for (int k = 0; k < D; ++k) cen[k] = up[k] / down;
  // oriented normal
  for (int k = 0; k < D; ++k) nrm[k] = 0;
  for_lines(S, lane, nl, ends, [&](const Line4 &l, unsigned id, bool) {
    double a[D], b[D], c[D], o[D], nv[D];
    plain_outside(S, id, m, l.s, o);
    for (int k = 0; k < D; ++k) {
      a[k] = l.s[k] - cen[k];
      b[k] = l.e[k] - cen[k];
      c[k] = pc(id, k) - cen[k];
      o[k] = o[k] - cen[k];
    }
    tetra_normal(a, b, c, nv);
    orient(nv, o);
    for (int k = 0; k < D; ++k) nrm[k] += nv[k];
  });
}

// The same for a plain 3-D cell, the cube with axis 0 held at 0.
__device__ __forceinline__ void plain_element3(PlainLds<3> &S, int lane, unsigned m, int nl,
                                               const double *h, double *cen, double *nrm) {
  double pm[D] = {0, 0, 0, 0};
  for_lines(S, lane, nl, 0, [&](const Line4 &l, unsigned, bool) {
    for (int k = 0; k < D; ++k) pm[k] += l.s[k] + l.e[k];
  });
  for (int k = 0; k < D; ++k) pm[k] = pm[k] / double(2.0 * nl);
  if (nl > 3) {
    double up[D] = {0, 0, 0, 0}, down = 0;
    for_lines(S, lane, nl, 0, [&](const Line4 &l, unsigned, bool) {
      double a[D], b[D];
      for (int k = 0; k < D; ++k) {
        a[k] = l.s[k] - pm[k];
        b[k] = l.e[k] - pm[k];
      }
      const double u1 = a[2] * b[3] - a[3] * b[2];
      const double u2 = a[1] * b[3] - a[3] * b[1];
      const double u3 = a[2] * b[1] - a[1] * b[2];
      const double ar = 0.5 * sqrt(u1 * u1 + u2 * u2 + u3 * u3);
      for (int k = 0; k < D; ++k) up[k] += third(l.s[k] + l.e[k] + pm[k]) * ar;
      down += ar;
    });
    for (int k = 0; k < D; ++k) pm[k] = up[k] / down;
  }
  for (int k = 0; k < D; ++k) {
    cen[k] = pm[k];
    nrm[k] = 0;
  }
  for_lines(S, lane, nl, 0, [&](const Line4 &l, unsigned id, bool) {
    double a[D], b[D], o[D], t[D];
    plain_outside(S, id, m, l.s, o);
    for (int k = 0; k < D; ++k) {
      a[k] = l.s[k] - pm[k];
      b[k] = l.e[k] - pm[k];
      o[k] = o[k] - pm[k];
    }
    t[0] = 0.0;
    t[1] = 0.5 * (a[2] * b[3] - a[3] * b[2]);
    t[2] = -0.5 * (a[1] * b[3] - a[3] * b[1]);
    t[3] = 0.5 * (a[1] * b[2] - a[2] * b[1]);
    orient(t, o);
    for (int k = 0; k < D; ++k) nrm[k] += t[k];
  });
}

}  // namespace corn
}  // namespace gvh
