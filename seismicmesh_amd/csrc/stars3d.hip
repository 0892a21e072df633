// Device 3D Delaunay tetrahedralisation.
//
// Replaces the role of CGAL's insert / get_finite_cells
// (SeismicMesh/generation/cpp/delaunay_class3.cpp:116-129, :276-344) in the
// 3D loop, as delaunay3d.cpp does on the host.  With the symbolic
// perturbation of the in-sphere test (delaunay3d.cpp) the tetrahedralisation
// is a function of the point set, and so is the star of each vertex: every
// star can be found on its own, and all of them agree.
//
// One wave finds one star.  The star of v is kept as its link, a closed
// triangulated surface around v: each lane holds one triangle (a, b, c) of
// it, i.e. the tetrahedron (v, a, b, c), or the hull facet (v, a, b) when c
// is the symbolic vertex at infinity.  A new point q is tested against all
// triangles at once: with v as the origin the lifted in-sphere determinant is
// linear in (q, |q|^2), so a triangle carries its four cofactors and their
// permanents, and a test is eight multiply-adds against a forward error
// bound.  The triangles in conflict are replaced by the cone from q over the
// rim of their hole.
//   near (k_stars<false, false>): the points of the grid cells around v,
//     sorted by distance, until every circumsphere lies in the part of the
//     grid already seen: 85 % of the vertices of the 76-primitive solid end
//     here, after ~12 insertions and ~30 candidates;
//   far (k_stars<true, false>): the triangles still open (hull facets, the
//     wide spheres over concave parts of a boundary) search the rest of the
//     points through a tree over the grid with 4 x 4 x 4 children a node,
//     one child per lane; a node is entered when the largest value of the
//     conflict polynomial over its points' box (separable by axis) is not
//     negative.  All open triangles share one traversal.
// Points already refused never come back: the Voronoi cell of v only
// shrinks.  Stars with a test inside its error bound are found again with
// exact integer predicates (k_stars<true, true>); with too many of them (a
// lattice: most_exact_stars) the build goes to the host.  Vertices of more than 64 link triangles
// ("hubs", 0.1 % of the vertices) get no star: their cells are found in
// their neighbours' stars, and cells of four hubs from the triangulation of
// the hubs alone, checked by one tree search each.  Every star emits the
// cells whose lowest id it is, sorted; an offset scan places them, so the
// output is canonical and sorted like the host's.
//
// Bound: instruction issue -- FP64 vector arithmetic, and in the tree the
// chain of dependent node reads -- with 3 to 4 waves a SIMD to hide it.
// Measured on MI355X, whole build (16 host threads in brackets): 523 k
// points of the 76-primitive solid just off their lattice 27 ms (120-150), of
// which near 7.7, far 17.5, and at the twentieth iteration, whose points lie
// in the boundary, 46, of which near 7.8, far 33; 138 k points of a graded box
// model 9.6 ms (45); 3 k points of a ball 0.5 ms (6.4, one thread).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

#include "common.h"
#include "delaunay3d.h"
#include "predicates.h"
#include "stars3d.h"

namespace smk {

namespace {

using smpred::kEps;

constexpr int kMaxLevels = 6;
constexpr int kCellsPerPoint = 6;
constexpr int kMaxHubs = 8192;
// Points of a cell beyond this many are crowded.  A star's first candidates
// are any 64 of the cells around it, and where those hold many times more,
// hardly one of the 64 is a neighbour: the link outgrows 64 triangles, so
// that there are about as many hubs as crowded points (60 k points, a
// twentieth of them 64, 256, 1024 to a cell: 1.6, 2.3, 2.5 k hubs of 1.9,
// 2.7, 2.9 k crowded points).  The build is therefore left at once when
// there are more of them than it may have hubs.  This also bounds what a cell
// can hold, and with it the loops over a cell's points.  Half of 60 k points
// some thousands to a cell: 83 ms before, 40 of them for near and far passes
// that ended with 28 k hubs; the host's 30 now.
constexpr int kCrowded = 24;
constexpr int kPoolPerPoint = 32;  // link triangles per vertex (24.5 on average)

struct SPt {  // a point in grid order
  double x, y, z;
  int32_t id;
  int32_t dup;  // a point with the same coordinates has a lower id
};

// A node of the occupancy tree: the box of its points and which of its
// 4 x 4 x 4 children hold any.
struct Node {
  double lo[3], hi[3];
  uint64_t mask;
  uint64_t pad;
};

struct StarGrid {
  double lo[3], hi[3], s, inv, slack;
  int32_t g[3];
  int32_t nlev;
  int32_t dim[kMaxLevels][3];
  int64_t moff[kMaxLevels];
};

// status words (device, then pinned host)
enum {
  kStX = 0,
  kStF = 1,
  kStHub = 2,
  kStFail = 3,
  kStPool = 4,
  kStTotal = 5,
  kStCrowd = 6,
  kStWords = 8
};

__device__ inline uint64_t enc(double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  return (u >> 63) ? ~u : u | (1ull << 63);
}
__device__ inline double dec(uint64_t u) {
  return __longlong_as_double((long long)((u >> 63) ? u & ~(1ull << 63) : ~u));
}

__global__ void k_star_init(uint64_t *bb, int32_t *status) {
  if (threadIdx.x < 3) bb[threadIdx.x] = ~0ull;
  else if (threadIdx.x < 6) bb[threadIdx.x] = 0ull;
  if (threadIdx.x < kStWords) status[threadIdx.x] = 0;
}

__global__ void k_star_bbox(int64_t n, const double *p, uint64_t *bb, int32_t *status) {
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  bool bad = false;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double x = p[3 * i + k];
      bad |= !(fabs(x) < 1e150);
      lo[k] = fmin(lo[k], x);
      hi[k] = fmax(hi[k], x);
    }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      lo[k] = fmin(lo[k], __shfl_xor(lo[k], off));
      hi[k] = fmax(hi[k], __shfl_xor(hi[k], off));
    }
  if (__ballot(bad) && threadIdx.x % 64 == 0) status[kStFail] = kLeftInput;
  if (threadIdx.x % 64 == 0)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      atomicMin((unsigned long long *)&bb[k], (unsigned long long)enc(lo[k]));
      atomicMax((unsigned long long *)&bb[3 + k], (unsigned long long)enc(hi[k]));
    }
}

// Cell size: the given spacing, but no more than the mean spacing of the
// points in their box and no more cells than allocated.
__global__ void k_star_grid(int64_t n, double spacing, int64_t cap_cells, int64_t cap_nodes,
                            const uint64_t *bb, StarGrid *g, int32_t *status) {
  double ext[3], vol = 1.0, big = 0.0;
  bool ok = status[kStFail] == 0;
  for (int k = 0; k < 3; ++k) {
    const double lo = dec(bb[k]), hi = dec(bb[3 + k]);
    g->lo[k] = lo;
    g->hi[k] = hi;
    ext[k] = hi - lo;
    ok = ok && ext[k] > 0.0;
    vol *= ext[k];
    big = fmax(big, fmax(fabs(lo), fabs(hi)));
  }
  double s = cbrt(vol / (double)n);
  ok = ok && s > 0.0;
  if (!ok) {
    s = 1.0;
    status[kStFail] = kLeftInput;
  }
  if (spacing > 0.0 && spacing < s) s = spacing;
  for (int it = 0; it < 4096; ++it) {
    double c = 1.0, m = 0.0;
    for (int k = 0; k < 3; ++k) {
      const double e = ok ? floor(ext[k] / s) + 1.0 : 1.0;
      c *= e;
      m = fmax(m, e);
    }
    if (c <= (double)cap_cells && m <= 1024.0) break;
    s *= 1.05;
  }
  // squared distances are compared in FP32
  if (!(s > 1e-15 && s < 1e15)) status[kStFail] = kLeftInput;
  g->s = s;
  g->inv = 1.0 / s;
  // rounding of a cell's corner, and of the cell a point falls into
  g->slack = 1e-9 * s + 1e-15 * big;
  int64_t d[3], c = 1;
  for (int k = 0; k < 3; ++k) {
    d[k] = ok ? (int64_t)floor(ext[k] / s) + 1 : 1;
    if (d[k] > 1024) {
      d[k] = 1;
      status[kStFail] = kLeftInput;
    }
    g->g[k] = (int32_t)d[k];
    c *= d[k];
  }
  if (c > cap_cells) {
    for (int k = 0; k < 3; ++k) g->g[k] = (int32_t)(d[k] = 1);
    status[kStFail] = kLeftInput;
  }
  int l = 0;
  int64_t off = 0;
  do {
    for (int k = 0; k < 3; ++k) g->dim[l][k] = (int32_t)(d[k] = (d[k] + 3) / 4);
    g->moff[l] = off;
    off += d[0] * d[1] * d[2];
    ++l;
  } while (d[0] * d[1] * d[2] > 1 && l < kMaxLevels);
  g->nlev = l;
  if (off > cap_nodes) {
    // no room (a grid one or two cells wide): nothing may be written
    for (int k = 0; k < 3; ++k) g->g[k] = g->dim[0][k] = 1;
    g->nlev = 1;
    status[kStFail] = kLeftInput;
  }
}

__device__ inline int cell_coord(const StarGrid &g, double x, int k) {
  const int c = (int)((x - g.lo[k]) * g.inv);
  return c < 0 ? 0 : (c >= g.g[k] ? g.g[k] - 1 : c);
}
__device__ inline int64_t cell_index(const StarGrid &g, int i, int j, int k) {
  return ((int64_t)i * g.g[1] + j) * g.g[2] + k;
}

__global__ void k_star_count(int64_t n, const double *p, const StarGrid *gp, int32_t *cnt,
                             int32_t *cell, int32_t *status) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (status[kStFail]) {
    cell[i] = 0;
    return;
  }
  const StarGrid &g = *gp;
  const int32_t c = (int32_t)cell_index(g, cell_coord(g, p[3 * i], 0), cell_coord(g, p[3 * i + 1], 1),
                                        cell_coord(g, p[3 * i + 2], 2));
  cell[i] = c;
  const uint64_t m = __ballot(atomicAdd(&cnt[c], 1) >= kCrowded);
  if (m && threadIdx.x % 64 == __builtin_ctzll(m))
    atomicAdd(&status[kStCrowd], (int32_t)__builtin_popcountll(m));
}

// the counts are consumed from the top, so they are zero again afterwards
__global__ void k_star_scatter(int64_t n, const double *p, const int32_t *cell,
                               const int32_t *start, int32_t *cnt, SPt *ps, int32_t most,
                               int32_t *status) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool crowded = status[kStCrowd] > most;
  if (crowded && i == 0) status[kStFail] = kLeftCrowded;
  if (i >= n || crowded || status[kStFail]) return;
  const int32_t c = cell[i];
  SPt q;
  q.x = p[3 * i];
  q.y = p[3 * i + 1];
  q.z = p[3 * i + 2];
  q.id = (int32_t)i;
  q.dup = 0;
  ps[start[c] + atomicSub(&cnt[c], 1) - 1] = q;
}

__global__ void k_star_dups(int64_t n, const StarGrid *gp, const int32_t *start, SPt *ps,
                            const int32_t *status) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || status[kStFail]) return;
  const StarGrid &g = *gp;
  const double x = ps[i].x, y = ps[i].y, z = ps[i].z;
  const int32_t id = ps[i].id;
  const int64_t c = cell_index(g, cell_coord(g, x, 0), cell_coord(g, y, 1), cell_coord(g, z, 2));
  for (int32_t e = start[c], ee = start[c + 1]; e < ee; ++e)
    if (ps[e].x == x && ps[e].y == y && ps[e].z == z && ps[e].id < id) {
      ps[i].dup = 1;
      return;
    }
}

// The nodes of one level: a wave per node, a child per lane.  The boxes are
// those of the points, not of the cells: a flat side of a domain then has
// boxes as thin as the rounding noise of its points, which is what lets the
// search pass over them (with cell boxes every facet in such a side entered
// every cell of the side).
__global__ void k_star_nodes(const StarGrid *gp, int level, const int32_t *start, const SPt *ps,
                             Node *nodes, const int32_t *status) {
  const StarGrid &g = *gp;
  if (level >= g.nlev || status[kStFail]) return;
  const int lane = threadIdx.x % 64;
  const int32_t *d = g.dim[level];
  const int64_t count = (int64_t)d[0] * d[1] * d[2];
  const int32_t *cd = level == 0 ? g.g : g.dim[level - 1];
  for (int64_t w = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64; w < count;
       w += (int64_t)gridDim.x * blockDim.x / 64) {
    const int k = (int)(w % d[2]), j = (int)((w / d[2]) % d[1]), i = (int)(w / d[2] / d[1]);
    const int ci = 4 * i + lane / 16, cj = 4 * j + (lane / 4) % 4, ck = 4 * k + lane % 4;
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    bool occ = false;
    if (ci < cd[0] && cj < cd[1] && ck < cd[2]) {
      const int64_t c = ((int64_t)ci * cd[1] + cj) * cd[2] + ck;
      if (level == 0) {
        for (int32_t e = start[c], ee = start[c + 1]; e < ee; ++e) {
          const double x[3] = {ps[e].x, ps[e].y, ps[e].z};
          occ = true;
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            lo[a] = fmin(lo[a], x[a]);
            hi[a] = fmax(hi[a], x[a]);
          }
        }
      } else {
        const Node &n = nodes[g.moff[level - 1] + c];
        occ = n.mask != 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          lo[a] = n.lo[a];
          hi[a] = n.hi[a];
        }
      }
    }
    const uint64_t m = __ballot(occ);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        lo[a] = fmin(lo[a], __shfl_xor(lo[a], off));
        hi[a] = fmax(hi[a], __shfl_xor(hi[a], off));
      }
    if (lane == 0) {
      Node n;
      for (int a = 0; a < 3; ++a) {
        n.lo[a] = lo[a];
        n.hi[a] = hi[a];
      }
      n.mask = m;
      n.pad = 0;
      nodes[g.moff[level] + w] = n;
    }
  }
}

// ------------------------------------------------------------ predicates
__device__ inline bool lex_greater(const double *a, const double *b) {
  if (a[0] != b[0]) return a[0] > b[0];
  if (a[1] != b[1]) return a[1] > b[1];
  return a[2] > b[2];
}

__device__ inline int orient_fix(const double *a, const double *b, const double *c,
                                 const double *d) {
  const int s = smpred::orient3d_filter(a, b, c, d);
  return s != SM_PRED_UNRESOLVED ? s : smpred::orient3d_fix(a, b, c, d);
}

struct P3 {
  double v[3];
};

// Signs of orient3d(a, b, c, d), and of the perturbed in-sphere test of
// delaunay3d.cpp; SM_PRED_UNRESOLVED outside the integer stage's range.
// Not inlined: their registers and stack stay out of the filtered path.
__device__ __noinline__ int orient_exact_call(P3 a, P3 b, P3 c, P3 d) {
  return orient_fix(a.v, b.v, c.v, d.v);
}

__device__ __noinline__ int insphere_exact_call(P3 a, P3 b, P3 c, P3 d, P3 e) {
  const int s = smpred::insphere_fix(a.v, b.v, c.v, d.v, e.v);
  if (s != 0) return s;
  P3 pt[5] = {a, b, c, d, e};
  unsigned left = 31;
  for (int k = 0; k < 5; ++k) {
    int top = -1;
    for (int i = 0; i < 5; ++i)
      if ((left >> i & 1) && (top < 0 || lex_greater(pt[i].v, pt[top].v))) top = i;
    left &= ~(1u << top);
    if (top == 4) return -1;
    P3 w[4] = {a, b, c, d};
    w[top] = e;
    const int o = orient_fix(w[0].v, w[1].v, w[2].v, w[3].v);
    if (o != 0) return o;
  }
  return -1;
}

// ------------------------------------------------------------- the stars
constexpr int kInfV = 0xffff;  // the vertex at infinity in a triangle
constexpr int kDead = -1;      // an unused triangle slot (in .a)
constexpr int kTab = 64;       // points held for one link
constexpr int kStack = 64 * kMaxLevels;

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ inline int lane_of() { return (int)__lane_id(); }
__device__ inline int below(uint64_t m) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}
__device__ inline int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ inline int rdl(int x, int lane) { return __builtin_amdgcn_readlane(x, lane); }
__device__ inline double rdl(double x, int lane) {
  const int64_t u = __double_as_longlong(x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(u >> 32), lane);
  return __longlong_as_double((int64_t)((uint64_t)hi << 32 | lo));
}

// One wave's share of LDS.
struct StarLds {
  double tx[kTab], ty[kTab], tz[kTab];  // inserted points
  int32_t tid[kTab];                    // their positions in grid order
  double cx[64], cy[64], cz[64];        // candidates of a chunk
  int32_t ci[64];
  int32_t run0[64], runp[64];  // runs of grid points, inclusive prefix of lengths
  int32_t used[kTab];
  uint32_t rim[66];            // directed edges of a hole's rim
};
struct FarLds {
  uint32_t stack[kStack];  // tree nodes: level (3 bits), then i, j, k (9 bits each)
};

struct Tri {
  int32_t a, b, c;  // table indices; a = kDead: unused; c = kInfV: hull facet
  double N[3], D, P[3], Pd;
  double half;  // 1 / (2 D) for the tree search
  float diam;   // upper bound of the sphere's diameter (inf: none)
};

enum { kOk = 0, kUncertain = 1, kOverflow = 2, kUnresolved = 3, kFar = 4, kVoid = 5 };

// FAR: with the tree search.  EXACT: uncertain tests settled by the integer
// stage (else they end the star with kUncertain).
template <bool FAR, bool EXACT>
struct Star {
  StarLds &sh;
  FarLds *fsh;
  const StarGrid &g;
  const SPt *ps;
  const int32_t *start;
  const Node *nodes;
  const int32_t *fail;  // EXACT: set once the whole build is void
  double vx, vy, vz;
  int self;
  Tri t;
  bool conf;
  int ntab = 0;
  float need2 = INFINITY;  // square of the largest diameter

  __device__ Star(StarLds &s, FarLds *f, const StarGrid &gg, const SPt *p, const int32_t *st,
                  const Node *m, const int32_t *fl)
      : sh(s), fsh(f), g(gg), ps(p), start(st), nodes(m), fail(fl) {}

  // A star of a lattice takes milliseconds of exact predicates, one after
  // the other: after each of them it looks whether another star has met one
  // that cannot be settled.  (One read a predicate of tens of microseconds.
  // With all stars in flight finished first, the exact pass of such an
  // attempt took 4-5 ms on 138 k points; 2-3 now.)
  __device__ bool voided() const {
    return uni(__hip_atomic_load(fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;
  }

  __device__ P3 tab(int i) const { return P3{{sh.tx[i], sh.ty[i], sh.tz[i]}}; }
  __device__ P3 vert() const { return P3{{vx, vy, vz}}; }

  __device__ bool on_side(double a, double b, double v, int k) const {
    return a == v && b == v && (v == g.lo[k] || v == g.hi[k]);
  }

  // cofactors, permanents and diameter of the lane's triangle
  __device__ void coef() {
    Tri &r = t;
    const double a[3] = {sh.tx[r.a] - vx, sh.ty[r.a] - vy, sh.tz[r.a] - vz};
    const double b[3] = {sh.tx[r.b] - vx, sh.ty[r.b] - vy, sh.tz[r.b] - vz};
    double ab[3], abp[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int i = (k + 1) % 3, j = (k + 2) % 3;
      const double u = a[i] * b[j], w = a[j] * b[i];
      ab[k] = u - w;
      abp[k] = fabs(u) + fabs(w);
    }
    if (r.c == kInfV) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        r.N[k] = ab[k];
        r.P[k] = abp[k];
      }
      r.D = r.Pd = 0.0;
      r.half = INFINITY;
      // a facet in a side of the points' box has no point beyond it; a
      // point in its plane is decided by the sphere behind it
      const bool closed = on_side(sh.tx[r.a], sh.tx[r.b], vx, 0) ||
                          on_side(sh.ty[r.a], sh.ty[r.b], vy, 1) ||
                          on_side(sh.tz[r.a], sh.tz[r.b], vz, 2);
      r.diam = closed ? 0.0f : INFINITY;
      return;
    }
    const double c[3] = {sh.tx[r.c] - vx, sh.ty[r.c] - vy, sh.tz[r.c] - vz};
    const double la = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
    const double lb = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
    const double lc = c[0] * c[0] + c[1] * c[1] + c[2] * c[2];
    r.D = 0.0;
    r.Pd = 0.0;
    double n2 = 0.0, p2 = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int i = (k + 1) % 3, j = (k + 2) % 3;
      const double u1 = b[i] * c[j], w1 = b[j] * c[i];
      const double u2 = c[i] * a[j], w2 = c[j] * a[i];
      const double bc = u1 - w1, bcp = fabs(u1) + fabs(w1);
      const double ca = u2 - w2, cap = fabs(u2) + fabs(w2);
      r.N[k] = (la * bc + lb * ca) + lc * ab[k];
      r.P[k] = (la * bcp + lb * cap) + lc * abp[k];
      r.D += a[k] * bc;
      r.Pd += fabs(a[k]) * bcp;
      n2 += r.N[k] * r.N[k];
      p2 += r.P[k] * r.P[k];
    }
    // |N| / D; a D that its rounding error could change by 1e-6 counts as a
    // sphere without bound (the tree search then decides)
    if (!(r.D > 1e6 * (16.0 * kEps) * r.Pd)) r.diam = INFINITY;
    else r.diam = (float)((sqrt(n2) + 24.0 * kEps * sqrt(p2)) / r.D) * 1.00001f;
    if (FAR) r.half = 0.5 / fmax(r.D, 0.0);
  }

  __device__ void update_need() {
    float m = t.a != kDead ? t.diam : 0.0f;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    need2 = m * m * 1.00001f;
  }

  // v, a, b (of a hull facet) and q are exactly coplanar: they share a
  // coordinate, or (EXACT) three of them, q included, share two, a row along
  // an axis.  On the edges of a box this settles what the exact stage cannot:
  // rows with a coordinate 0 next to neighbours at 1e-13.  (138 k points of a
  // graded box, 8 iterations from their lattice: 403 ms without the rows, 2
  // of the last 5 builds tried on the device in vain; 327 with them, all 5
  // made there; 375 with every build on 16 host threads.  Looked for in the
  // far pass too, whose uncertain points are mostly in a side, they cost it 4
  // %.)
  __device__ bool same_plane(int a, int b, double x, double y, double z) const {
    if ((vx == x && sh.tx[a] == x && sh.tx[b] == x) ||
        (vy == y && sh.ty[a] == y && sh.ty[b] == y) ||
        (vz == z && sh.tz[a] == z && sh.tz[b] == z))
      return true;
    if (!EXACT) return false;
    const bool vq[3] = {vx == x, vy == y, vz == z};
    const bool aq[3] = {sh.tx[a] == x, sh.ty[a] == y, sh.tz[a] == z};
    const bool bq[3] = {sh.tx[b] == x, sh.ty[b] == y, sh.tz[b] == z};
    int va = 0, vb = 0, ab = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      va += vq[k] && aq[k];
      vb += vq[k] && bq[k];
      ab += aq[k] && bq[k];
    }
    return va > 1 || vb > 1 || ab > 1;
  }

  // lane of the finite triangle across the edge (a, b) of a hull facet
  __device__ int behind(int a, int b) const {
    const bool nb = t.a != kDead && t.c != kInfV &&
                    ((t.a == b && t.b == a) || (t.b == b && t.c == a) || (t.c == b && t.a == a));
    const uint64_t m = __ballot(nb);
    return m ? __builtin_ctzll(m) : 0;
  }

  // conf: which triangles (x, y, z) is in conflict with; returns kOk,
  // kUncertain or kUnresolved (wave-uniform)
  __device__ int test(double x, double y, double z) {
    const double qx = x - vx, qy = y - vy, qz = z - vz;
    const double l = qx * qx + qy * qy + qz * qz;
    const double val = (qx * t.N[0] + qy * t.N[1]) + (qz * t.N[2] - l * t.D);
    const double err = (24.0 * kEps) * ((fabs(qx) * t.P[0] + fabs(qy) * t.P[1]) +
                                        (fabs(qz) * t.P[2] + l * t.Pd));
    const bool live = t.a != kDead;
    conf = live && val > err;
    bool unc = live && !(val > err) && !(val < -err);
    if (__ballot(unc) == 0) return kOk;
    bool flat = false, bad = false;
    if (unc && t.c == kInfV && same_plane(t.a, t.b, x, y, z)) {
      flat = true;
      unc = false;
    }
    if (!EXACT) {
      if (__ballot(unc)) return kUncertain;
    } else if (unc) {
      const P3 q{{x, y, z}};
      int o;
      if (t.c == kInfV) {
        o = orient_exact_call(vert(), tab(t.a), tab(t.b), q);
        flat = o == 0;
      } else {
        o = insphere_exact_call(vert(), tab(t.a), tab(t.b), tab(t.c), q);
      }
      bad = o == SM_PRED_UNRESOLVED;
      conf = o > 0 && !bad;
    }
    if (EXACT && __ballot(bad)) return kUnresolved;
    if (EXACT && voided()) return kVoid;
    // a point in a hull facet's plane: as the finite tetrahedron behind it
    uint64_t m = __ballot(flat);
    while (m) {
      const int ln = __builtin_ctzll(m);
      m &= m - 1;
      const int nb = behind(rdl(t.a, ln), rdl(t.b, ln));
      const bool inb = (__ballot(conf) >> nb & 1) != 0;
      if (lane_of() == ln) conf = inb;
    }
    return kOk;
  }

  // a table entry no triangle refers to (64 triangles have at most 34
  // vertices)
  __device__ int recycle() {
    const int lane = lane_of();
    sh.used[lane] = 0;
    wave_sync();
    if (t.a != kDead) {
      sh.used[t.a] = 1;
      sh.used[t.b] = 1;
      if (t.c != kInfV) sh.used[t.c] = 1;
    }
    wave_sync();
    return __builtin_ctzll(__ballot(sh.used[lane] == 0));
  }

  // the triangles in conf replaced by the cone from (x, y, z)
  __device__ int insert(double x, double y, double z, int32_t idx) {
    const int lane = lane_of();
    const int q = ntab < kTab ? ntab++ : recycle();
    if (lane == 0) {
      sh.tx[q] = x;
      sh.ty[q] = y;
      sh.tz[q] = z;
      sh.tid[q] = idx;
    }
    // rim: directed edges whose twin belongs to no triangle in conflict
    const uint32_t a16 = (uint32_t)t.a & 0xffffu, b16 = (uint32_t)t.b, c16 = (uint32_t)t.c;
    const uint32_t e[3] = {a16 << 16 | b16, b16 << 16 | c16, c16 << 16 | a16};
    const uint32_t w[3] = {b16 << 16 | a16, c16 << 16 | b16, a16 << 16 | c16};
    bool rim[3] = {conf, conf, conf};
    uint64_t m = __ballot(conf);
    while (m) {
      const int ln = __builtin_ctzll(m);
      m &= m - 1;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const uint32_t o = (uint32_t)rdl((int)e[j], ln);
#pragma unroll
        for (int i = 0; i < 3; ++i) rim[i] = rim[i] && w[i] != o;
      }
    }
    int nb = 0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const uint64_t rm = __ballot(rim[j]);
      const int pos = nb + below(rm);
      if (rim[j] && pos < 64) sh.rim[pos] = e[j];
      nb += __builtin_popcountll(rm);
    }
    if (conf) t.a = kDead;
    const uint64_t room = __ballot(t.a == kDead);
    if (nb > __builtin_popcountll(room)) return kOverflow;
    wave_sync();
    const int r = below(room);
    if (t.a == kDead && r < nb) {
      const uint32_t ed = sh.rim[r];
      const int a = (int)(ed >> 16), b = (int)(ed & 0xffffu);
      t.a = a == kInfV ? b : (b == kInfV ? q : a);
      t.b = a == kInfV ? q : (b == kInfV ? a : b);
      t.c = (a == kInfV || b == kInfV) ? kInfV : q;
      coef();
    }
    wave_sync();
    update_need();
    return kOk;
  }

  // ------------------------------------------------ candidates near v
  uint32_t key;        // lane k: the k-th nearest candidate (squared distance | its lane)
  int cnt = 0, pos = 0;

  // candidate lanes (ok) sorted by distance into key / cnt
  __device__ void sort_chunk(bool ok, const SPt &q, int32_t idx) {
    const int lane = lane_of();
    const double dx = q.x - vx, dy = q.y - vy, dz = q.z - vz;
    const float d2 = (float)(dx * dx + dy * dy + dz * dz);
    // 26 bits of the squared distance (rounded down), then the lane
    key = ok ? ((__float_as_uint(d2) & ~63u) | (uint32_t)lane) : 0xffffffffu;
    sh.cx[lane] = q.x;
    sh.cy[lane] = q.y;
    sh.cz[lane] = q.z;
    sh.ci[lane] = idx;
    cnt = __builtin_popcountll(__ballot(ok));
    pos = 0;
#pragma unroll
    for (int size = 2; size <= 64; size <<= 1)
#pragma unroll
      for (int str = size >> 1; str > 0; str >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)key, str);
        const bool up = (lane & size) == 0, low = (lane & str) == 0;
        key = (low == up) ? (key < o ? key : o) : (key < o ? o : key);
      }
    wave_sync();
  }

  // The initial link from the sorted chunk: the nearest point and the first
  // pair spanning a volume with it (all third points at once for each
  // second).  Returns the mask of the three used, 0 when there is none.
  __device__ uint64_t start_link() {
    if (cnt < 3) return 0;
    const int lane = lane_of();
    const P3 v = vert();
    const int sa = rdl((int)key, 0) & 63, own = (int)(key & 63u);
    const P3 A{{sh.cx[sa], sh.cy[sa], sh.cz[sa]}};
    const P3 C{{sh.cx[own], sh.cy[own], sh.cz[own]}};
    int ib = 1, ic = -1, o = 0;
    for (; ib < cnt - 1 && ib < 8; ++ib) {
      const int sb = rdl((int)key, ib) & 63;
      const P3 B{{sh.cx[sb], sh.cy[sb], sh.cz[sb]}};
      const int r = smpred::orient3d_filter(v.v, A.v, B.v, C.v);
      const bool good = lane > ib && lane < cnt && r != SM_PRED_UNRESOLVED && r != 0;
      const uint64_t m = __ballot(good);
      if (m) {
        ic = __builtin_ctzll(m);
        o = rdl(r, ic);
        break;
      }
    }
    if (ic < 0) return 0;
    const int sb = rdl((int)key, ib) & 63, sc = rdl((int)key, ic) & 63;
    const int srt[3] = {sa, o > 0 ? sb : sc, o > 0 ? sc : sb};
    if (lane == 0)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        sh.tx[k] = sh.cx[srt[k]];
        sh.ty[k] = sh.cy[srt[k]];
        sh.tz[k] = sh.cz[srt[k]];
        sh.tid[k] = sh.ci[srt[k]];
      }
    ntab = 3;
    wave_sync();
    // (0 1 2) and the hull facets behind its edges
    if (lane < 4) {
      t.a = lane == 0 ? 0 : (lane == 1 ? 1 : (lane == 2 ? 2 : 0));
      t.b = lane == 0 ? 1 : (lane == 1 ? 0 : (lane == 2 ? 1 : 2));
      t.c = lane == 0 ? 2 : kInfV;
      coef();
    }
    update_need();
    return 1ull | 1ull << ib | 1ull << ic;
  }

  // wave prefix of run lengths into LDS; returns the total
  __device__ int runs(int32_t s0, int32_t len) {
    const int lane = lane_of();
    int pre = len;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(pre, off);
      if (lane >= off) pre += o;
    }
    sh.run0[lane] = s0 - (pre - len);
    sh.runp[lane] = pre;
    wave_sync();
    return rdl(pre, 63);
  }
  // grid position of the k-th point of the runs
  __device__ int32_t run_point(int k) const {
    int lo = 0;  // first run whose prefix exceeds k
#pragma unroll
    for (int w = 32; w > 0; w >>= 1)
      if (sh.runp[lo + w - 1] <= k) lo += w;
    return sh.run0[lo] + k;
  }

  // Runs of the cells within R cells of c along each axis but not within
  // Rin (entries e0 .. e0 + 63 of them); returns the number of points.
  __device__ int ring_runs(const int *c, int R, int Rin, int e0) {
    const int side = 2 * R + 1;
    const int e = e0 + lane_of();
    int32_t s0 = 0, len = 0;
    if (e < 2 * side * side) {
      const int row = e >> 1, half = e & 1;
      const int di = row / side - R, dj = row % side - R;
      const int i = c[0] + di, j = c[1] + dj;
      const int ad = abs(di) > abs(dj) ? abs(di) : abs(dj);
      int k0 = c[2] - R, k1 = c[2] + R;
      bool use = i >= 0 && i < g.g[0] && j >= 0 && j < g.g[1];
      if (ad > Rin) use = use && half == 0;
      else if (half == 0) k1 = c[2] - Rin - 1;
      else k0 = c[2] + Rin + 1;
      k0 = k0 < 0 ? 0 : k0;
      k1 = k1 >= g.g[2] ? g.g[2] - 1 : k1;
      if (use && k0 <= k1) {
        // nearest point of the run's box
        double d2 = 0.0;
        const double lo[3] = {g.lo[0] + i * g.s, g.lo[1] + j * g.s, g.lo[2] + k0 * g.s};
        const double hi[3] = {lo[0] + g.s, lo[1] + g.s, g.lo[2] + (k1 + 1) * g.s};
        const double v[3] = {vx, vy, vz};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double d = fmax(0.0, fmax(lo[a] - v[a], v[a] - hi[a]) - g.slack);
          d2 += d * d;
        }
        if (!(d2 > (double)need2)) {
          s0 = start[cell_index(g, i, j, k0)];
          len = start[cell_index(g, i, j, k1) + 1] - s0;
        }
      }
    }
    return runs(s0, len);
  }

  // distance from v within which every point has been a candidate after
  // the cells within R of v's cell
  __device__ double coverage(const int *c, int R) const {
    double m = INFINITY;
    const double v[3] = {vx, vy, vz};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if (c[k] - R > 0) m = fmin(m, v[k] - (g.lo[k] + (c[k] - R) * g.s));
      if (c[k] + R + 1 < g.g[k]) m = fmin(m, g.lo[k] + (c[k] + R + 1) * g.s - v[k]);
    }
    return fmax((m - g.slack) * (1.0 - 1e-9), 0.0);
  }

  // ------------------------------------------------ the tree search
  // One traversal checks all triangles of `set` (a lane mask) at once.  It
  // stops at a leaf that holds a point in conflict with one of them: the
  // one nearest to v becomes the only candidate of the chunk, and the leaf
  // goes back on the stack.  kOk with cnt = 0: the stack is empty.
  int sp = 0;
  __device__ void push_root() {
    if (lane_of() == 0) fsh->stack[0] = (uint32_t)(g.nlev - 1) << 27;
    sp = 1;
    wave_sync();
  }

  __device__ int search(uint64_t set) {
    const int lane = lane_of();
    cnt = pos = 0;
    while (sp > 0) {
      const uint32_t nd = (uint32_t)uni((int)fsh->stack[--sp]);
      wave_sync();
      const int lev = (int)(nd >> 27);
      const int i = (int)(nd >> 18 & 511u), j = (int)(nd >> 9 & 511u), k = (int)(nd & 511u);
      const int32_t *d = g.dim[lev];
      const Node &node = nodes[g.moff[lev] + ((int64_t)i * d[1] + j) * d[2] + k];
      const uint64_t m = node.mask;
      const double v[3] = {vx, vy, vz};
      double nlo[3], nhi[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        nlo[a] = node.lo[a] - v[a];
        nhi[a] = node.hi[a] - v[a];
      }
      // which triangles reach the node at all: a triangle per lane
      uint64_t sub;
      {
        double val = 0.0, pe = 0.0, M2 = 0.0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double M = fmax(fabs(nlo[a]), fabs(nhi[a]));
          const double x = fmax(nlo[a], fmin(t.N[a] * t.half, nhi[a]));
          val += x * (t.N[a] - t.D * x);
          pe += M * t.P[a];
          M2 += M * M;
        }
        sub = set & __ballot(t.a != kDead && !(val < -40.0 * kEps * (pe + M2 * t.Pd)));
      }
      if (sub == 0) continue;
      const bool occ = (m >> lane & 1) != 0;
      const int cc[3] = {4 * i + lane / 16, 4 * j + (lane / 4) % 4, 4 * k + lane % 4};
      double lo[3], hi[3], M[3], d2 = 0.0, M2 = 0.0;
      if (lev > 0) {
        const int32_t *cd = g.dim[lev - 1];
        const Node &child =
            nodes[g.moff[lev - 1] +
                  (occ ? ((int64_t)cc[0] * cd[1] + cc[1]) * cd[2] + cc[2] : (int64_t)0)];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          lo[a] = child.lo[a] - v[a];
          hi[a] = child.hi[a] - v[a];
        }
      } else {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double c0 = g.lo[a] + cc[a] * g.s - v[a] - g.slack;
          lo[a] = fmax(c0, nlo[a]);
          hi[a] = fmin(c0 + g.s + 2.0 * g.slack, nhi[a]);
        }
      }
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        M[a] = fmax(fabs(lo[a]), fabs(hi[a]));
        M2 += M[a] * M[a];
        const double dd = fmax(0.0, fmax(lo[a], -hi[a]));
        d2 += dd * dd;
      }
      bool hit = false;
      uint64_t near = 0;  // the triangles that reach some child
      for (uint64_t sm = sub; sm; sm &= sm - 1) {
        const int s = __builtin_ctzll(sm);
        const double D = rdl(t.D, s), hf = rdl(t.half, s);
        double val = 0.0, pe = M2 * rdl(t.Pd, s);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          // the largest value of N x - D x^2 over [lo, hi]
          const double N = rdl(t.N[a], s);
          const double x = fmax(lo[a], fmin(N * hf, hi[a]));
          val += x * (N - D * x);
          pe += M[a] * rdl(t.P[a], s);
        }
        const bool h = occ && !(val < -40.0 * kEps * pe);
        near |= __ballot(h) ? 1ull << s : 0;
        hit = hit || h;
      }
      const uint64_t hm = __ballot(hit);
      if (hm == 0) continue;
      if (lev > 0) {
        // children onto the stack, the nearest on top
        const uint32_t kk = (__float_as_uint((float)d2) & ~63u) | (uint32_t)lane;
        const int n = __builtin_popcountll(hm);
        if (sp + n > kStack) return kOverflow;
        int rank = 0;  // by decreasing distance
        for (uint64_t o = hm; o; o &= o - 1)
          rank += (uint32_t)rdl((int)kk, __builtin_ctzll(o)) > kk;
        if (hit)
          fsh->stack[sp + rank] = (uint32_t)(lev - 1) << 27 | (uint32_t)cc[0] << 18 |
                                  (uint32_t)cc[1] << 9 | (uint32_t)cc[2];
        sp += n;
        wave_sync();
        continue;
      }
      // leaf cells: their points, one per lane
      int32_t s0 = 0, len = 0;
      if (hit) {
        const int64_t c = cell_index(g, cc[0], cc[1], cc[2]);
        s0 = start[c];
        len = start[c + 1] - s0;
      }
      const int total = runs(s0, len);
      for (int b = 0; b < total; b += 64) {
        SPt q;
        q.x = vx;
        q.y = vy;
        q.z = vz;
        int32_t idx = -1;
        bool ok = b + lane < total, in = false, bad = false;
        if (ok) {
          idx = run_point(b + lane);
          q = ps[idx];
          ok = idx != self && q.dup == 0;
        }
        const double qx = q.x - vx, qy = q.y - vy, qz = q.z - vz;
        const double l = qx * qx + qy * qy + qz * qz;
        const auto side = [&](int s, bool &unc) {  // filtered conflict with triangle s
          const double val = (qx * rdl(t.N[0], s) + qy * rdl(t.N[1], s)) +
                             (qz * rdl(t.N[2], s) - l * rdl(t.D, s));
          const double err =
              (24.0 * kEps) * ((fabs(qx) * rdl(t.P[0], s) + fabs(qy) * rdl(t.P[1], s)) +
                               (fabs(qz) * rdl(t.P[2], s) + l * rdl(t.Pd, s)));
          unc = !(val > err) && !(val < -err);
          return val > err;
        };
        for (uint64_t sm = near; sm; sm &= sm - 1) {
          const int s = __builtin_ctzll(sm);
          bool unc, in1 = side(s, unc);
          if (__ballot(ok && (in1 || unc)) == 0) continue;
          // vertices of the triangle itself are no candidates
          const int ta = rdl(t.a, s), tb = rdl(t.b, s), tc = rdl(t.c, s);
          const bool use = ok && idx != sh.tid[ta] && idx != sh.tid[tb] &&
                           (tc == kInfV || idx != sh.tid[tc == kInfV ? 0 : tc]);
          in = in || (use && in1);
          unc = unc && use;
          if (__ballot(unc) == 0) continue;
          // a point in a hull facet's plane is the concern of the sphere
          // behind the facet, which is searched or closed by itself
          unc = unc && !(tc == kInfV && same_plane(ta, tb, q.x, q.y, q.z));
          if (!EXACT) {
            if (__ballot(unc)) return kUncertain;
          } else if (unc) {
            const P3 qq{{q.x, q.y, q.z}};
            const int o = tc == kInfV ? orient_exact_call(vert(), tab(ta), tab(tb), qq)
                                      : insphere_exact_call(vert(), tab(ta), tab(tb), tab(tc), qq);
            bad = bad || o == SM_PRED_UNRESOLVED;
            in = in || (o > 0 && o != SM_PRED_UNRESOLVED);
          }
          if (EXACT && __ballot(bad)) return kUnresolved;
          if (EXACT && voided()) return kVoid;
        }
        if (__ballot(in) == 0) continue;
        float best = in ? (float)l : INFINITY;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) best = fminf(best, __shfl_xor(best, off));
        const int o = __builtin_ctzll(__ballot(in && (float)l == best));
        if (lane == o) {
          sh.cx[0] = q.x;
          sh.cy[0] = q.y;
          sh.cz[0] = q.z;
          sh.ci[0] = idx;
        }
        key = 0;
        cnt = 1;
        if (lane == 0) fsh->stack[sp] = nd;
        ++sp;
        wave_sync();
        return kOk;
      }
      wave_sync();
    }
    return kOk;
  }

  __device__ int build() {
    t.a = kDead;
    t.b = t.c = 0;
    const int c[3] = {cell_coord(g, vx, 0), cell_coord(g, vy, 1), cell_coord(g, vz, 2)};
    const int lane = lane_of();
    bool built = false, far = false;
    int R = 1, Rin = -1, e0 = 0, at = 0, total = ring_runs(c, 1, -1, 0);
    double cov = 0.0;
    uint64_t skip = 0, seen = 0, set = 0;
    for (int guard = 0; guard < 1 << 20; ++guard) {
      if (pos < cnt) {
        // the one place where points are tested and inserted
        const int k = pos++;
        if (skip >> k & 1) continue;
        const uint32_t kk = (uint32_t)rdl((int)key, k);
        if (!far && __uint_as_float(kk & ~63u) > need2) {
          pos = cnt;  // sorted: all later ones are farther
          continue;
        }
        const int src = (int)(kk & 63u);
        const double x = sh.cx[src], y = sh.cy[src], z = sh.cz[src];
        int rc = test(x, y, z);
        if (rc) return rc;
        const uint64_t cm = __ballot(conf);
        if (cm == 0) {
          if (far) return kOverflow;  // the search and the test disagree: leave it
          continue;
        }
        if ((rc = insert(x, y, z, sh.ci[src]))) return rc;
        const uint64_t live = __ballot(t.a != kDead);
        seen &= ~cm & live;
        set &= ~cm & live;
        continue;
      }
      if (!far) {
        if (at < total) {
          // next chunk of the ring's points
          SPt q;
          q.x = vx;
          q.y = vy;
          q.z = vz;
          int32_t idx = -1;
          bool ok = at + lane < total;
          if (ok) {
            idx = run_point(at + lane);
            q = ps[idx];
            const double dx = q.x - vx, dy = q.y - vy, dz = q.z - vz;
            ok = idx != self && q.dup == 0 &&
                 !((float)(dx * dx + dy * dy + dz * dz) * 0.9999f > need2);
          }
          at += 64;
          skip = 0;
          cnt = pos = 0;
          if (__ballot(ok) == 0) continue;
          sort_chunk(ok, q, idx);
          if (!built) {
            skip = start_link();
            built = skip != 0;
            if (!built) {
              // too few points, or all in one plane: a wider region
              if (++R > 4) return kOverflow;
              pos = cnt = 0;
              e0 = at = 0;
              total = ring_runs(c, R, -1, 0);
            }
          }
          continue;
        }
        if (e0 + 64 < 2 * (2 * R + 1) * (2 * R + 1)) {
          e0 += 64;
          at = 0;
          wave_sync();
          total = ring_runs(c, R, Rin, e0);
          continue;
        }
        if (!built) {
          if (++R > 4) return kOverflow;
          e0 = at = 0;
          wave_sync();
          total = ring_runs(c, R, -1, 0);
          continue;
        }
        cov = coverage(c, R);
        if (!((double)need2 > cov * cov)) return kOk;
        // wide spheres (hull facets above all) are left to the tree: more
        // rings do not close them
        if (R < 4 && (R < 2 || (double)need2 < 64.0 * g.s * g.s)) {
          Rin = R++;
          e0 = at = 0;
          wave_sync();
          total = ring_runs(c, R, Rin, 0);
          continue;
        }
        if (!FAR) return kFar;
        far = true;
        skip = 0;
        sp = 0;
      }
      if (FAR) {
        const float cf = (float)(cov * (1.0 - 1e-6));
        const uint64_t open = __ballot(t.a != kDead && !(t.diam <= cf)) & ~seen;
        if (sp == 0 || set == 0) {
          // the last traversal found no more: its triangles are done
          seen |= set;
          set = open & ~set;
          if (set == 0) return kOk;
          push_root();
        }
        const int rc = search(set);
        if (rc) return rc;
      }
    }
    return kOverflow;
  }
};

constexpr int kStarWaves = 4;
template <bool FAR, bool EXACT>
__global__ __launch_bounds__(64 * kStarWaves, EXACT ? 1 : (FAR ? 3 : 4)) void k_stars(
    int64_t n, const StarGrid *gp, const SPt *ps, const int32_t *start, const Node *nodes,
    const int32_t *list, const int32_t *nlist, int32_t most, int32_t *far, int32_t *exact,
    int32_t *hubs, int32_t *pool, int64_t pool_cap, int32_t *poff, int32_t *pcnt,
    int32_t *rowcnt, int32_t *status, int32_t most_exact) {
  __shared__ StarLds shm[kStarWaves];
  __shared__ FarLds fshm[FAR ? kStarWaves : 1];
  if (status[kStFail]) return;
  // too many uncertain stars after the near pass: the rest is no use
  if (FAR && status[kStX] > most_exact) {
    if (threadIdx.x == 0) status[kStFail] = kLeftUncertain;
    return;
  }
  const int lane = threadIdx.x % 64;
  const int64_t items = list ? (int64_t)*nlist : n;
  if (list && items > most) {
    if (blockIdx.x == 0 && threadIdx.x == 0) status[kStFail] = kLeftUncertain;
    return;
  }
  const int64_t nw = (int64_t)gridDim.x * kStarWaves;
  const unsigned blk = list ? blockIdx.x : xcd_block();
  const int wv = uni(threadIdx.x / 64);
  for (int64_t w = (int64_t)blk * kStarWaves + wv; w < items; w += nw) {
    if (EXACT &&
        __hip_atomic_load(&status[kStFail], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return;
    const int self = uni(list ? list[w] : (int)w);
    const SPt q = ps[self];
    const int32_t id = uni(q.id);
    if (uni(q.dup)) {
      if (lane == 0) pcnt[id] = rowcnt[id] = poff[id] = 0;
      continue;
    }
    Star<FAR, EXACT> st(shm[wv], &fshm[FAR ? wv : 0], *gp, ps, start, nodes, status + kStFail);
    st.vx = q.x;
    st.vy = q.y;
    st.vz = q.z;
    st.self = self;
    const int rc = st.build();
    if (rc != kOk) {
      if (lane == 0) {
        pcnt[id] = rowcnt[id] = 0;
        poff[id] = -1;  // no star
        if (rc == kFar) far[atomicAdd(&status[kStF], 1)] = self;
        else if (rc == kUncertain) exact[atomicAdd(&status[kStX], 1)] = self;
        else if (rc == kOverflow) hubs[atomicAdd(&status[kStHub], 1)] = id;
        else if (rc == kUnresolved)
          __hip_atomic_store(&status[kStFail], kLeftUnresolved, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      }
      wave_sync();
      continue;
    }
    // the link's finite triangles, and how many of them have v lowest
    const Tri &t = st.t;
    const bool fin = t.a != kDead && t.c != kInfV;
    int32_t ia = 0, ib = 0, ic = 0;
    if (fin) {
      ia = ps[st.sh.tid[t.a]].id;
      ib = ps[st.sh.tid[t.b]].id;
      ic = ps[st.sh.tid[t.c]].id;
    }
    const uint64_t fm = __ballot(fin);
    const int total = __builtin_popcountll(fm);
    const int mine = __builtin_popcountll(__ballot(fin && id < ia && id < ib && id < ic));
    int32_t off = 0;
    if (lane == 0) off = atomicAdd(&status[kStPool], total);
    off = uni(off);
    if ((int64_t)off + total > pool_cap || off < 0) {
      if (lane == 0) status[kStFail] = kLeftPool;
      return;
    }
    if (lane == 0) {
      poff[id] = off;
      pcnt[id] = total;
      rowcnt[id] = mine;
    }
    if (fin) {
      const int64_t o = 3 * ((int64_t)off + below(fm));
      pool[o] = ia;
      pool[o + 1] = ib;
      pool[o + 2] = ic;
    }
    wave_sync();
  }
}

// bad[c] = 1 when some point lies in the sphere of cell c, 2 when that
// cannot be told: one tree search per cell (a wave each).  pos: position in
// grid order of each point id.
__global__ __launch_bounds__(64 * kStarWaves) void k_star_check(
    const StarGrid *gp, const SPt *ps, const int32_t *start, const Node *nodes,
    const int32_t *cells, int nc, const int32_t *pos, int32_t *bad, const int32_t *status) {
  __shared__ StarLds shm[kStarWaves];
  __shared__ FarLds fshm[kStarWaves];
  const int wv = uni(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int c = blockIdx.x * kStarWaves + wv;
  if (c >= nc) return;
  Star<true, true> st(shm[wv], &fshm[wv], *gp, ps, start, nodes, status + kStFail);
  const int self = uni(pos[cells[4 * c]]);
  st.vx = ps[self].x;
  st.vy = ps[self].y;
  st.vz = ps[self].z;
  st.self = self;
  if (lane < 3) {
    const int32_t o = pos[cells[4 * c + 1 + lane]];
    shm[wv].tx[lane] = ps[o].x;
    shm[wv].ty[lane] = ps[o].y;
    shm[wv].tz[lane] = ps[o].z;
    shm[wv].tid[lane] = o;
  }
  wave_sync();
  st.t.a = lane == 0 ? 0 : kDead;
  st.t.b = 1;
  st.t.c = 2;
  if (lane == 0) st.coef();
  st.push_root();
  const int rc = st.search(1ull);
  if (lane == 0) bad[c] = rc != kOk ? 2 : (st.cnt > 0 ? 1 : 0);
}

__global__ void k_star_positions(int64_t n, const SPt *ps, int32_t *pos) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) pos[ps[i].id] = (int32_t)i;
}

// Each vertex's row of the output: its cells in which it is the lowest id,
// (v, a, b, c) with a the lowest of the rest, sorted.  (a, b) is a directed
// edge of v's link, so it orders a row by itself.
constexpr int kRowWaves = 4, kRowMax = 64;
__global__ __launch_bounds__(64 * kRowWaves) void k_star_rows(
    int64_t n, const int32_t *pool, const int32_t *poff, const int32_t *pcnt,
    const int32_t *rowptr, int32_t *tet, int64_t cap, int32_t *status) {
  __shared__ uint64_t key[kRowWaves][kRowMax];
  __shared__ int32_t last[kRowWaves][kRowMax];
  if (status[kStFail]) return;
  const int lane = threadIdx.x % 64, wv = threadIdx.x / 64;
  const int64_t v = (int64_t)blockIdx.x * kRowWaves + wv;
  if (v >= n) return;
  const int cnt = pcnt[v];
  if (cnt == 0 || cnt > kRowMax) return;
  const int64_t off = poff[v];
  int r = 0;
  for (int b = 0; b < cnt; b += 64) {
    int32_t a = 0, bb = 0, c = 0;
    bool low = false;
    if (b + lane < cnt) {
      const int32_t *e = pool + 3 * (off + b + lane);
      a = e[0];
      bb = e[1];
      c = e[2];
      low = (int32_t)v < a && (int32_t)v < bb && (int32_t)v < c;
      // rotate the smallest to the front (an even permutation)
      if (bb < a && bb < c) {
        const int32_t x = a;
        a = bb;
        bb = c;
        c = x;
      } else if (c < a && c < bb) {
        const int32_t x = c;
        c = bb;
        bb = a;
        a = x;
      }
    }
    const uint64_t m = __ballot(low);
    if (low) {
      const int p = r + below(m);
      key[wv][p] = (uint64_t)(uint32_t)a << 32 | (uint32_t)bb;
      last[wv][p] = c;
    }
    r += __builtin_popcountll(m);
  }
  wave_sync();
  const int64_t row = rowptr[v];
  if (row + r > cap) {
    if (lane == 0) status[kStFail] = kLeftCells;
    return;
  }
  for (int p = lane; p < r; p += 64) {
    const uint64_t k = key[wv][p];
    int rank = 0;
    for (int o = 0; o < r; ++o) rank += key[wv][o] < k;
    int4 out;
    out.x = (int32_t)v;
    out.y = (int32_t)(k >> 32);
    out.z = (int32_t)(k & 0xffffffffu);
    out.w = last[wv][p];
    *reinterpret_cast<int4 *>(tet + 4 * (row + rank)) = out;
  }
}

// Cells whose lowest id is a hub (a vertex without a star: poff = -1), from
// the star of their lowest other vertex.
__global__ void k_star_hub_cells(int64_t n, const int32_t *pool, const int32_t *poff,
                                 const int32_t *pcnt, int32_t *out, int32_t cap,
                                 int32_t *count) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  const int cnt = pcnt[v];
  const int64_t off = poff[v];
  for (int k = 0; k < cnt; ++k) {
    const int32_t *e = pool + 3 * (off + k);
    int32_t lo = (int32_t)v;
    bool own = true;
    for (int j = 0; j < 3; ++j) {
      lo = e[j] < lo ? e[j] : lo;
      if (e[j] < (int32_t)v && poff[e[j]] >= 0) own = false;
    }
    if (lo == (int32_t)v || !own) continue;
    const int32_t at = atomicAdd(count, 1);
    if (at < cap) {
      out[4 * at] = (int32_t)v;
      out[4 * at + 1] = e[0];
      out[4 * at + 2] = e[1];
      out[4 * at + 3] = e[2];
    }
  }
}

__global__ void k_star_gather(int n, const int32_t *ids, const double *p, double *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 3 * n) out[i] = p[3 * (int64_t)ids[i / 3] + i % 3];
}

// out[i] = a[ids[i]], or a[ids[i]] = in[i]
__global__ void k_star_read(int n, const int32_t *ids, const int32_t *a, int32_t *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = a[ids[i]];
}
__global__ void k_star_write(int n, const int32_t *ids, const int32_t *in, int32_t *a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[ids[i]] = in[i];
}
// cell c of the hubs' cells to place `to[c]`
__global__ void k_star_place(int n, const int32_t *to, const int4 *cells, int4 *tet) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) tet[to[i]] = cells[i];
}

inline size_t al(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace

void stars_free(StarScratch *s) {
  if (s->mem) (void)hipFree(s->mem);
  if (s->h_status) (void)hipHostFree(s->h_status);
  s->mem = nullptr;
  s->h_status = nullptr;
  s->bytes = 0;
}

// The most vertices whose stars may need exact predicates: where the exact
// pass takes as long as the host build would.  Measured with a share x of n
// vertices (exact cubes in part of a box, jittered elsewhere): the pass takes
// 1 + 35 x ms whatever n is up to 64 k, since the longest star decides (x =
// 0.04 0.1 0.16 0.31 0.48: 1.9 2.9 4.5 8 15-18 ms); where moved vertices are
// scattered among lattice ones, 1 + 9 x.  The other passes take 0.8 ms, the
// host 2.2 us a point on one thread (4.3 on a whole lattice) and a quarter of
// that or less on several.  Between the two slopes the lines meet at x =
// (host - 1.8 ms) / 20 ms; a thirty-second costs at most 0.7 ms in any case,
// and beyond a half whole lattices come, 20 ms and more for the longest star
// and, on the 523 k points of the 76-primitive solid, 119 ms at x = 0.65 with
// 16 host threads at 105-130.  Examples, device and host: 512 points, x =
// 0.36, 7 ms and 1.3 (now left to the host); 3 k points from a ball's
// lattice, x = 0.18, 2.7 and 7; 27 k, x = 0.41, 6.2 and 18 on 16 threads.
int32_t most_exact_stars(int64_t n, int host_threads) {
  const double host_ms = 2.2e-3 * (double)n / (host_threads > 1 ? 4.0 : 1.0);
  const double share = std::min(0.5, std::max(1.0 / 32.0, (host_ms - 1.8) / 20.0));
  return (int32_t)(share * (double)n);
}

int device_delaunay3d(StarScratch *sc, const double *p, int64_t n, double spacing,
                      int host_threads, int32_t *tet, int64_t cap, int64_t *count, bool *done,
                      hipStream_t s) {
  *done = false;
  if (n < kStarMinPoints || n > (int64_t)1 << 25) {
    sc->left = kLeftInput;
    return SM_OK;
  }
  if (sc->skip > 0) {
    --sc->skip;
    return SM_OK;
  }
  const int64_t cells = kCellsPerPoint * n + 4096;
  const int64_t pool_cap = kPoolPerPoint * n + 4096;
  // one allocation: layout below
  size_t off = 0;
  const auto take = [&](size_t b) {
    const size_t o = off;
    off += al(b);
    return o;
  };
  const size_t o_bb = take(6 * 8), o_grid = take(sizeof(StarGrid)), o_st = take(kStWords * 4);
  const size_t o_ps = take((size_t)n * sizeof(SPt)), o_cell = take((size_t)n * 4);
  const size_t o_cnt = take((size_t)(cells + 1) * 4), o_start = take((size_t)(cells + 1) * 4);
  const int64_t node_cap = cells / 4 + 64;
  const size_t o_node = take((size_t)node_cap * sizeof(Node));
  const size_t o_lf = take((size_t)n * 4), o_lx = take((size_t)n * 4);
  const size_t o_hub = take((size_t)n * 4);
  const size_t o_poff = take((size_t)n * 4), o_pcnt = take((size_t)n * 4);
  const size_t o_row = take((size_t)(n + 1) * 4), o_rowp = take((size_t)(n + 1) * 4);
  const size_t o_pool = take((size_t)pool_cap * 12);
  const size_t o_ws = take(scan_workspace(std::max(cells, n) + 1));
  // without room for the scratch the host build does it, which needs none
  // on the device
  const auto no_room = [&]() {
    (void)hipGetLastError();
    sc->left = kLeftMemory;
    sc->skip = 3;
    return SM_OK;
  };
  if (off > sc->max_bytes) return no_room();
  if (sc->bytes < off) {
    if (sc->mem) (void)hipFree(sc->mem);
    sc->mem = nullptr;
    sc->bytes = 0;
    if (hipMalloc(&sc->mem, off) != hipSuccess) {
      sc->mem = nullptr;
      return no_room();
    }
    sc->bytes = off;
  }
  if (!sc->h_status && hipHostMalloc((void **)&sc->h_status, kStWords * sizeof(int32_t),
                                     hipHostMallocDefault) != hipSuccess) {
    sc->h_status = nullptr;
    return no_room();
  }
  char *b = reinterpret_cast<char *>(sc->mem);
  uint64_t *bb = reinterpret_cast<uint64_t *>(b + o_bb);
  StarGrid *g = reinterpret_cast<StarGrid *>(b + o_grid);
  int32_t *st = reinterpret_cast<int32_t *>(b + o_st);
  SPt *ps = reinterpret_cast<SPt *>(b + o_ps);
  int32_t *cell = reinterpret_cast<int32_t *>(b + o_cell);
  int32_t *cnt = reinterpret_cast<int32_t *>(b + o_cnt);
  int32_t *start = reinterpret_cast<int32_t *>(b + o_start);
  Node *nodes = reinterpret_cast<Node *>(b + o_node);
  int32_t *lx = reinterpret_cast<int32_t *>(b + o_lx);
  int32_t *lf = reinterpret_cast<int32_t *>(b + o_lf);
  int32_t *hub = reinterpret_cast<int32_t *>(b + o_hub);
  int32_t *poff = reinterpret_cast<int32_t *>(b + o_poff);
  int32_t *pcnt = reinterpret_cast<int32_t *>(b + o_pcnt);
  int32_t *row = reinterpret_cast<int32_t *>(b + o_row);
  int32_t *rowp = reinterpret_cast<int32_t *>(b + o_rowp);
  int32_t *pool = reinterpret_cast<int32_t *>(b + o_pool);
  void *ws = b + o_ws;

  const int B = 256;
  const unsigned gn = blocks_for(n, B);
  // the hubs are settled on one host thread, which has the whole set done in
  // eight times what an eighth of it takes (8 k points with 1.3 k hubs: 25 ms
  // against the host's 18, and 4.2 with 174)
  const int32_t most_hubs = (int32_t)std::min<int64_t>(kMaxHubs, n / 8);
  int rc;
  hipLaunchKernelGGL(k_star_init, dim3(1), dim3(64), 0, s, bb, st);
  hipLaunchKernelGGL(k_star_bbox, dim3(std::min(gn, 256u)), dim3(B), 0, s, n, p, bb, st);
  hipLaunchKernelGGL(k_star_grid, dim3(1), dim3(1), 0, s, n, spacing, cells, node_cap, bb, g, st);
  if ((rc = fill<int32_t>(cnt, cells + 1, 0, s))) return rc;
  hipLaunchKernelGGL(k_star_count, dim3(gn), dim3(B), 0, s, n, p, g, cnt, cell, st);
  if ((rc = scan_exclusive(cnt, start, cells + 1, nullptr, ws, s))) return rc;
  hipLaunchKernelGGL(k_star_scatter, dim3(gn), dim3(B), 0, s, n, p, cell, start, cnt, ps, most_hubs,
                     st);
  hipLaunchKernelGGL(k_star_dups, dim3(gn), dim3(B), 0, s, n, g, start, ps, st);
  for (int l = 0; l < kMaxLevels; ++l) {
    const int64_t most = std::max<int64_t>(1, cells >> (5 * l));
    hipLaunchKernelGGL(k_star_nodes, dim3((unsigned)std::min<int64_t>(2048, blocks_for(most, 4))),
                       dim3(B), 0, s, g, l, start, ps, nodes, st);
  }
  const int32_t most_exact = most_exact_stars(n, host_threads);
  constexpr int W = kStarWaves;
  hipLaunchKernelGGL((k_stars<false, false>), dim3(blocks_for(n, W)), dim3(64 * W), 0, s, n, g, ps,
                     start, nodes, (const int32_t *)nullptr, (const int32_t *)nullptr, 0, lf, lx,
                     hub, pool, pool_cap, poff, pcnt, row, st, most_exact);
  hipLaunchKernelGGL((k_stars<true, false>), dim3(blocks_for(n, 4 * W)), dim3(64 * W), 0, s, n, g,
                     ps, start, nodes, lf, st + kStF, (int32_t)n, lf, lx, hub, pool, pool_cap,
                     poff, pcnt, row, st, most_exact);
  hipLaunchKernelGGL((k_stars<true, true>), dim3((unsigned)std::min<int64_t>(1024, gn)),
                     dim3(64 * W), 0, s, n, g, ps, start, nodes, lx, st + kStX, most_exact, lf, lx,
                     hub, pool, pool_cap, poff, pcnt, row, st, most_exact);
  SM_LAUNCH_CHECK();
  const auto place = [&]() -> int {
    if ((rc = fill<int32_t>(row + n, 1, 0, s))) return rc;
    if ((rc = scan_exclusive(row, rowp, n + 1, st + kStTotal, ws, s))) return rc;
    hipLaunchKernelGGL(k_star_rows, dim3(blocks_for(n, kRowWaves)), dim3(64 * kRowWaves), 0, s, n,
                       pool, poff, pcnt, rowp, tet, cap, st);
    SM_LAUNCH_CHECK();
    SM_HIP(hipMemcpyAsync(sc->h_status, st, kStWords * 4, hipMemcpyDeviceToHost, s));
    SM_HIP(hipStreamSynchronize(s));
    return SM_OK;
  };
  if ((rc = place())) return rc;
  const int32_t *hs = sc->h_status;
  const auto leave = [&](int why = kLeftHubs) {
    sc->left = sc->h_status[kStFail] ? sc->h_status[kStFail] : why;
    // what fails now (a degenerate lattice) likely fails again; but a large
    // one is known for it early (5 of 130 ms) and loses a share of its
    // uncertain stars with every move
    sc->skip = sc->left == kLeftUncertain && n >= 65536 ? 2 : 3;
    return SM_OK;
  };
  if (hs[kStFail] || hs[kStHub] > most_hubs) return leave();
  if (hs[kStTotal] > cap || hs[kStTotal] < 0) return leave(kLeftCells);
  // Hubs: their rows from their neighbours' stars and, for cells of four
  // hubs, from the hubs' own triangulation, each cell checked against every
  // point; some thousand cells, ordered on the host.  The host arrays outlive
  // the copies on the stream, also where memory runs out.
  struct Cell {
    int32_t v[4];
  };
  std::vector<int32_t> hv, hc, own, hb, rows, to, r0;
  std::vector<double> hp;
  std::vector<Cell> all;
  if (hs[kStHub] > 0) try {
    const int nh = hs[kStHub];
    hv.resize((size_t)nh);
    SM_HIP(hipMemcpyAsync(hv.data(), hub, nh * 4, hipMemcpyDeviceToHost, s));
    SM_HIP(hipStreamSynchronize(s));
    std::sort(hv.begin(), hv.end());
    const int32_t hcap = (int32_t)n;
    int32_t *hcells = pool + 3 * (int64_t)hs[kStPool];  // behind the stars
    int32_t *hcount = lx, *posn = lf, *tmp = cell;
    if (3 * (int64_t)hs[kStPool] + 4 * (int64_t)hcap > 3 * pool_cap) return leave();
    double *hpts = reinterpret_cast<double *>(cnt);  // cells + 1 >= 6 nh ints
    SM_HIP(hipMemcpyAsync(hub, hv.data(), nh * 4, hipMemcpyHostToDevice, s));
    if ((rc = fill<int32_t>(hcount, 1, 0, s))) return rc;
    hipLaunchKernelGGL(k_star_hub_cells, dim3(gn), dim3(B), 0, s, n, pool, poff, pcnt, hcells,
                       hcap, hcount);
    hipLaunchKernelGGL(k_star_gather, dim3(blocks_for(3 * nh, B)), dim3(B), 0, s, nh, hub, p,
                       hpts);
    SM_LAUNCH_CHECK();
    int32_t nc = 0;
    hp.resize((size_t)nh * 3);
    SM_HIP(hipMemcpyAsync(&nc, hcount, 4, hipMemcpyDeviceToHost, s));
    SM_HIP(hipMemcpyAsync(hp.data(), hpts, hp.size() * 8, hipMemcpyDeviceToHost, s));
    SM_HIP(hipStreamSynchronize(s));
    if (nc < 0 || nc > hcap) return leave();
    hc.resize((size_t)nc * 4);
    if (nc) SM_HIP(hipMemcpyAsync(hc.data(), hcells, hc.size() * 4, hipMemcpyDeviceToHost, s));
    if (nh >= 4) {
      smdt::DT3 dt;
      rc = dt.run(hp.data(), nh, 0, 1, 1, [&](int, const int32_t *c, int64_t k) {
        for (int64_t i = 0; i < 4 * k; ++i) own.push_back(hv[(size_t)c[i]]);
      });
      if (rc) {
        SM_HIP(hipStreamSynchronize(s));
        return leave();
      }
    }
    SM_HIP(hipStreamSynchronize(s));
    if (!own.empty()) {
      const int no = (int)(own.size() / 4);
      if (no > n || 4 * (int64_t)no > 4 * (int64_t)hcap) return leave();
      int32_t *dc = hcells, *bad = tmp;
      SM_HIP(hipMemcpyAsync(dc, own.data(), own.size() * 4, hipMemcpyHostToDevice, s));
      hipLaunchKernelGGL(k_star_positions, dim3(gn), dim3(B), 0, s, n, ps, posn);
      hipLaunchKernelGGL(k_star_check, dim3(blocks_for(no, W)), dim3(64 * W), 0, s, g, ps, start,
                         nodes, dc, no, posn, bad, st);
      SM_LAUNCH_CHECK();
      hb.resize((size_t)no);
      SM_HIP(hipMemcpyAsync(hb.data(), bad, no * 4, hipMemcpyDeviceToHost, s));
      SM_HIP(hipStreamSynchronize(s));
      for (int c = 0; c < no; ++c) {
        if (hb[(size_t)c] & 2) return leave();
        if (hb[(size_t)c] == 0)
          hc.insert(hc.end(), own.begin() + 4 * (size_t)c, own.begin() + 4 * (size_t)c + 4);
      }
    }
    all.resize(hc.size() / 4);
    for (size_t i = 0; i < all.size(); ++i) {
      std::memcpy(all[i].v, hc.data() + 4 * i, 16);
      smdt::canonical_tet(all[i].v);
    }
    std::sort(all.begin(), all.end(), [](const Cell &x, const Cell &y) {
      return std::lexicographical_compare(x.v, x.v + 4, y.v, y.v + 4);
    });
    // the hubs' rows were empty so far: count, place, fill
    rows.assign((size_t)nh, 0);
    to.resize(all.size());
    for (const Cell &c : all) {
      const auto it = std::lower_bound(hv.begin(), hv.end(), c.v[0]);
      if (it == hv.end() || *it != c.v[0]) return leave();
      ++rows[(size_t)(it - hv.begin())];
    }
    SM_HIP(hipMemcpyAsync(tmp, rows.data(), nh * 4, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_star_write, dim3(blocks_for(nh, B)), dim3(B), 0, s, nh, hub, tmp, row);
    if ((rc = place())) return rc;
    // (the rows kernel does not see the hubs' rows)
    if (hs[kStFail] || hs[kStTotal] > cap || hs[kStTotal] < 0) return leave(kLeftCells);
    hipLaunchKernelGGL(k_star_read, dim3(blocks_for(nh, B)), dim3(B), 0, s, nh, hub, rowp, tmp);
    SM_LAUNCH_CHECK();
    r0.resize((size_t)nh);
    SM_HIP(hipMemcpyAsync(r0.data(), tmp, nh * 4, hipMemcpyDeviceToHost, s));
    SM_HIP(hipStreamSynchronize(s));
    size_t at = 0;
    for (int h = 0; h < nh; ++h)
      for (int32_t k = 0; k < rows[(size_t)h]; ++k) to[at++] = r0[(size_t)h] + k;
    if (!all.empty()) {
      const int na = (int)all.size();
      // cells behind the stars again (16-byte aligned), their places before
      int32_t *dto = reinterpret_cast<int32_t *>(cnt);
      int4 *dall = reinterpret_cast<int4 *>(nodes);
      if (na > cells || (int64_t)na * 16 > node_cap * (int64_t)sizeof(Node)) return leave();
      SM_HIP(hipMemcpyAsync(dto, to.data(), (size_t)na * 4, hipMemcpyHostToDevice, s));
      SM_HIP(hipMemcpyAsync(dall, all.data(), (size_t)na * 16, hipMemcpyHostToDevice, s));
      hipLaunchKernelGGL(k_star_place, dim3(blocks_for(na, B)), dim3(B), 0, s, na, dto, dall,
                         reinterpret_cast<int4 *>(tet));
      SM_LAUNCH_CHECK();
      SM_HIP(hipStreamSynchronize(s));
    }
  } catch (const std::bad_alloc &) {
    SM_HIP(hipStreamSynchronize(s));
    return leave();
  }
  *count = hs[kStTotal];
  sc->left = kLeftNot;
  *done = true;
  return SM_OK;
}

}  // namespace smk
