// wb_classify.hip -- shape queries and the SCAN / POSTSCAN / CLASSIFY pass.
//
// Equivalences used (each is exact, not approximate):
//  * A point's class depends only on its own point, the hyperboloid size of
//    the last tile (flowsnake counter order) whose pointsIn(cylinder) holds
//    it, and the set D of directions to the other points of
//    pointsIn(downward hyperboloid) (classify.cpp:96-173).  surround()'s
//    pruning only removes directions whose two neighbour gaps are both under
//    30 deg and never the first or last one, so it never creates or removes
//    a gap of 144 deg; and the first loop over the previous point's
//    downPoints only inserts directions of points that the second loop
//    inserts too.  So class 1 <=> |D|>1 and every gap between successive
//    sorted directions, and the wrap-around gap, is < DEG144.
//  * When every direction is in [-2^30, 2^30), those gaps are the circular
//    gaps of the directions mod 2^31, and adding directions only shrinks
//    them: the test may stop as soon as the directions seen so far pass.
//    The host checks the cloud extent (< 1e7 scale units) that guarantees
//    the smallest non-zero dy/|dx| keeps every direction >= 30 units below
//    +180 deg.
//  * Gaps are tracked with a 64-bit occupancy mask of 2^25-unit bins.  A
//    longest circular run of <= 23 empty bins bounds every gap by
//    25*2^25 < DEG144 (pass); >= 26 empty bins gives a gap > 26*2^25 > DEG144
//    (fail); a run of 24 or 25 is decided in a second pass that records the
//    exact extreme directions in the two bins bordering the run.
//  * Skipping a 32-point group whose bounding box fails the shape test is
//    exact: clamping the shape centre into the box makes each coordinate
//    difference no larger than for any point inside, and every predicate is
//    monotone in those differences.
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>

#include "wb_flowsnake.h"
#include "wb_internal.h"
#include "wb_wave.h"
#include "../../include/wb_gpu.h"

#define WAVE 64
// waves per SIMD the ground-test kernel is compiled for
#ifndef WB_GROUND_MINW
#define WB_GROUND_MINW 5
#endif
constexpr double kSqrt34 = 0.86602540378443864676372317;  // eisenstein.h:33
constexpr double kSqrt7 = 2.6457513110645905905016;       // scan.h:23

// lane values: the first active lane's, and lane l's (l wave-uniform)
__device__ inline int rfl(int v) { return __builtin_amdgcn_readfirstlane(v); }
// lane l's value of v (l wave-uniform)
__device__ inline double rdl(double v, uint32_t l)
{
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, (int)l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), (int)l);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// The device hands consecutive workgroups to its 8 XCDs in turn, and each
// XCD has its own L2.  xcd_block(b, nb) renumbers the nb blocks of a grid so
// that the blocks one XCD runs take one contiguous range of the work: kernels
// whose neighbouring blocks read the same leaves then find them in that XCD's
// L2.  A permutation of [0, nb): results do not depend on it.
__device__ inline uint32_t xcd_block(uint32_t b, uint32_t nb)
{
  const uint32_t x = b % 8, per = nb / 8, extra = nb % 8;
  return x * per + (x < extra ? x : extra) + b / 8;
}

struct TreeView {
  const double *px, *py, *pz;
  const uint32_t *leaf_start;
  const double *leaf_cube;
  const int32_t *leaf_parent;
  const double *node_cube;
  const int32_t *node_child, *node_parent;
  const double *chunk_box;
  const uint32_t *chunk_low;
  const double *chunk_sx, *chunk_sy, *chunk_sz;
  const float4 *oct_xy;
  const float *oct_z, *leaf_low;
  double ox, oy, oz, side;  // the root cube
  const uint2 *node_crange;
  const double *child_zlow;
  const uint8_t *leaf_out;
  const uint32_t *pt_leaf, *canon, *crank, *sidx;
  uint32_t nleaves, nnodes;
  uint64_t n;
};

static TreeView view(const wb_tree *t)
{
  TreeView v;
  v.px = t->px; v.py = t->py; v.pz = t->pz;
  v.leaf_start = t->leaf_start; v.leaf_cube = t->leaf_cube; v.leaf_parent = t->leaf_parent;
  v.node_cube = t->node_cube; v.node_child = t->node_child; v.node_parent = t->node_parent;
  v.chunk_box = t->chunk_box; v.chunk_low = t->chunk_low;
  v.oct_xy = t->oct_xy; v.oct_z = t->oct_z; v.leaf_low = t->leaf_low;
  v.ox = t->center[0]; v.oy = t->center[1]; v.oz = t->center[2]; v.side = t->side;
  v.chunk_sx = t->chunk_sx; v.chunk_sy = t->chunk_sy; v.chunk_sz = t->chunk_sz; v.node_crange = t->node_crange;
  v.child_zlow = t->child_zlow;
  v.leaf_out = t->leaf_out;  // (null without a point outside the root)
  v.pt_leaf = t->pt_leaf; v.canon = t->canon; v.crank = t->crank;
  v.sidx = t->sidx; v.nleaves = t->nleaves; v.nnodes = t->nnodes; v.n = t->n;
  return v;
}

// every point of the leaf lies in its cube (a tree of a batch may have no
// leaf_out where another one has)
__device__ inline bool leaf_inside(const TreeView &T, uint32_t leaf)
{
  return !T.leaf_out || T.leaf_out[leaf] == 0;
}

// ---------------------------------------------------------------------------
// Batched countPointsIn / pointsIn: one wave per shape.  The walk expands up
// to eight nodes of its stack per round, lane 8i+k testing child k of the
// i-th node from the top; the children that pass take the nodes' places in
// the order of the lanes, so the stack holds leaves and nodes in DFS order
// (octree.cpp:234-251) from its top down, and leaves come off it in that
// order.  They are served in batches of up to 64.
// What bounds it: the latency of a round's loads (child links and the nodes'
// cubes, read together) and of a batch's, at about 20 waves per CU.
// ---------------------------------------------------------------------------
// Entries a wave's stack holds.  A round takes up to eight nodes while that
// leaves room for what one node per round (the plain depth-first walk: at
// most 7 waiting entries per level and 8 children) can still add.
#define WB_WSTK 512
#define WB_WSTK_WIDE (WB_WSTK - 8 * 8 - 7 * (WB_MAX_LEVEL + 1) - 8)
struct ShapeWalk {
  int stk[WB_WSTK];
  int leaf[2 * WAVE];
  uint32_t pre[WAVE], b[WAVE], e[WAVE], mask[WAVE];
};

template <int KIND>
__device__ inline wb::Shape query_shape(const double *p)
{
  if (KIND == wb::SHAPE_CYLINDER) return wb::make_cylinder(p[0], p[1], p[2]);
  if (KIND == wb::SHAPE_SPHERE) return wb::make_sphere(p[0], p[1], p[2], p[3]);
  return wb::make_hyperboloid(p[0], p[1], p[2], p[3], p[4]);
}

// Octree::cube (octree.cpp:349-358) of child k of the cube (cx, cy, cz, side):
// the operations the build used for the stored cubes
__device__ inline void child_cube(double cx, double cy, double cz, double side, int k,
                                  double &x, double &y, double &z, double &sd)
{
  x = cx + (double)(2 * (k & 1) - 1) * side / 4;
  y = cy + (double)(2 * ((k >> 1) & 1) - 1) * side / 4;
  z = cz + (double)(2 * (k >> 2) - 1) * side / 4;
  sd = side / 2;
}

// serve(nb): the leaves K.leaf[0 .. nb) (nb <= 64), in DFS order
template <class Serve>
__device__ inline void shape_walk(const TreeView &T, const wb::Shape &S, ShapeWalk &K,
                                  Serve &&serve)
{
  if (T.nleaves == 0) return;
  if (!wb::shape_intersect(S, T.node_cube[0], T.node_cube[1], T.node_cube[2], T.node_cube[3]))
    return;
  const int lane = threadIdx.x;
  const uint64_t lt = (1ull << lane) - 1ull;
  if (lane == 0) K.stk[0] = 0;
  int sp = 1, nb = 0;
  while (sp > 0) {
    __syncthreads();
    const bool have = lane < sp;
    const int code = have ? K.stk[sp - 1 - lane] : 0;
    const uint64_t isleaf = __ballot(have && code < 0), isnode = __ballot(have && code >= 0);
    // the leaves above the first node
    const int nl = isnode ? __builtin_ctzll(isnode) : __popcll(isleaf);
    if (lane < nl) K.leaf[nb + lane] = -2 - code;
    nb += nl;
    sp -= nl;
    if (isnode) {
      // the nodes down to the next leaf
      const uint64_t rest = ~(isnode >> nl);
      int run = rest ? __builtin_ctzll(rest) : WAVE;
      run = sp > WB_WSTK_WIDE ? 1 : run < 8 ? run : 8;
      const bool on = (lane >> 3) < run;
      int ch = -1;
      bool hit = false;
      if (on) {
        const int nd = K.stk[sp - 1 - (lane >> 3)];
        const double *nc = T.node_cube + 4 * (size_t)nd;
        ch = T.node_child[8 * (size_t)nd + (lane & 7)];
        double x, y, z, sd;
        child_cube(nc[0], nc[1], nc[2], nc[3], lane & 7, x, y, z, sd);
        hit = ch != -1 && wb::shape_intersect(S, x, y, z, sd);
      }
      const uint64_t hits = __ballot(hit);
      sp += __popcll(hits) - run;
      __syncthreads();
      if (hit) K.stk[sp - 1 - __popcll(hits & lt)] = ch;
    }
    while (nb >= WAVE || (sp == 0 && nb > 0)) {
      __syncthreads();
      serve(nb < WAVE ? nb : WAVE);
      nb = nb < WAVE ? 0 : nb - WAVE;
      __syncthreads();
      const int left = K.leaf[WAVE + lane];
      __syncthreads();
      K.leaf[lane] = left;
    }
  }
}

// exclusive running sum over the wave's lanes, and the total
__device__ inline uint32_t wave_prefix(uint32_t v, uint32_t &total)
{
  const int lane = threadIdx.x;
  uint32_t s = v;
#pragma unroll
  for (int d = 1; d < WAVE; d <<= 1) {
    const uint32_t w = __shfl_up(s, d, WAVE);
    if (lane >= d) s += w;
  }
  total = (uint32_t)__builtin_amdgcn_readlane((int)s, 63);
  return s - v;
}

// the last of pre[0..nb) (ascending from 0) that is at most t
__device__ inline int prefix_find(const uint32_t *pre, int nb, uint32_t t)
{
  int lo = 0;
#pragma unroll
  for (int d = WAVE / 2; d > 0; d >>= 1)
    if (lo + d < nb && pre[lo + d] <= t) lo += d;
  return lo;
}

// The 32-point groups of the leaves K.b..K.e (K.pre: running sums of their
// numbers, tot in all), 64 at a time, a lane each: f(q, g, hit) with the leaf,
// the group and whether the shape may reach its box.
template <class F>
__device__ inline void leaf_groups(const TreeView &T, const wb::Shape &S, const ShapeWalk &K,
                                   int nb, uint32_t tot, F &&f)
{
  for (uint32_t t0 = 0; t0 < tot; t0 += WAVE) {
    const uint32_t t = t0 + threadIdx.x;
    bool hit = false;
    int q = 0;
    uint32_t g = 0;
    if (t < tot) {
      q = prefix_find(K.pre, nb, t);
      g = K.b[q] / WB_CHUNK + (t - K.pre[q]);
      const double *bx = T.chunk_box + 6 * (size_t)g;
      hit = wb::shape_may_hit_box(S, bx[0], bx[1], bx[2], bx[3], bx[4], bx[5]);
    }
    f(q, g, hit);
  }
}

// countPointsIn of shape blockIdx.x.  A leaf whose corners are all in the
// shape counts whole (octree.cpp:1226-1231, 1256-1257); of the others the
// groups whose box the shape may reach are read, four per step.
template <int KIND>
__global__ void __launch_bounds__(64) k_count_points_in(TreeView T, const double *params,
                                                        uint64_t nshapes, uint64_t *counts)
{
  __shared__ ShapeWalk K;
  const uint64_t s = blockIdx.x;
  if (s >= nshapes) return;
  const int lane = threadIdx.x;
  const wb::Shape S = query_shape<KIND>(params + WB_SHAPE_NPARAMS * s);
  uint64_t cnt = 0;  // this lane's share
  shape_walk(T, S, K, [&](int nb) {
    uint32_t b = 0, e = 0, ng = 0;
    if (lane < nb) {
      const int l = K.leaf[lane];
      const double *lc = T.leaf_cube + 4 * (size_t)l;
      b = T.leaf_start[l];
      e = T.leaf_start[l + 1];
      if (wb::shape_in_cube(S, lc[0], lc[1], lc[2], lc[3])) cnt += e - b;
      else if (e > b) ng = (e - 1) / WB_CHUNK - b / WB_CHUNK + 1;
    }
    uint32_t tot;
    K.pre[lane] = wave_prefix(ng, tot);
    K.b[lane] = b;
    K.e[lane] = e;
    __syncthreads();
    leaf_groups(T, S, K, nb, tot, [&](int q, uint32_t g, bool hit) {
      const uint32_t gb = K.b[q], ge = K.e[q];
      uint64_t own = __ballot(hit);
      while (own) {
        // four groups per step, two loads in flight per lane
        uint32_t j[2];
        bool ok[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const bool any = own != 0;
          const int o1 = any ? __builtin_ctzll(own) : 0;
          own &= own - 1;
          const bool two = own != 0;
          const int o2 = two ? __builtin_ctzll(own) : o1;
          own &= own - 1;
          const int o = lane < 32 ? o1 : o2;
          const uint32_t gg = (uint32_t)__shfl((int)g, o, WAVE);
          const uint32_t bb = (uint32_t)__shfl((int)gb, o, WAVE);
          const uint32_t ee = (uint32_t)__shfl((int)ge, o, WAVE);
          j[u] = gg * WB_CHUNK + (lane & 31);
          ok[u] = (lane < 32 ? any : two) && j[u] >= bb && j[u] < ee;
          if (!ok[u]) j[u] = bb;
        }
        double x[2], y[2], z[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          x[u] = T.px[j[u]];
          y[u] = T.py[j[u]];
          z[u] = T.pz[j[u]];
        }
#pragma unroll
        for (int u = 0; u < 2; u++) cnt += ok[u] && wb::shape_in(S, x[u], y[u], z[u]);
      }
    });
    __syncthreads();
  });
  for (int d = WAVE / 2; d > 0; d >>= 1) cnt += __shfl_xor(cnt, d, WAVE);
  if (lane == 0) counts[s] = cnt;
}

// pointsIn of shape blockIdx.x: its input indices from offs[s] on, leaf by
// leaf in DFS order and in canonical (input) order inside a leaf.  The leaves
// of a batch that lie whole in the shape or have a group the shape may reach
// are read as one sequence, four points per lane and step; of a leaf not whole
// in the shape only the points of such groups are tested.
template <int KIND>
__global__ void __launch_bounds__(64) k_points_in(TreeView T, const double *params,
                                                  uint64_t nshapes, const uint64_t *offs,
                                                  uint32_t *out)
{
  __shared__ ShapeWalk K;
  const uint64_t s = blockIdx.x;
  if (s >= nshapes) return;
  const int lane = threadIdx.x;
  const uint64_t lt = (1ull << lane) - 1ull;
  const wb::Shape S = query_shape<KIND>(params + WB_SHAPE_NPARAMS * s);
  // the writes stay inside the shape's own range whatever the walk finds
  uint64_t pos = offs[s];
  const uint64_t lim = offs[s + 1];
  shape_walk(T, S, K, [&](int nb) {
    uint32_t b = 0, e = 0, ng = 0;
    bool all = false, wide = false;
    if (lane < nb) {
      const int l = K.leaf[lane];
      const double *lc = T.leaf_cube + 4 * (size_t)l;
      b = T.leaf_start[l];
      e = T.leaf_start[l + 1];
      all = wb::shape_in_cube(S, lc[0], lc[1], lc[2], lc[3]);
      if (!all && e > b) ng = (e - 1) / WB_CHUNK - b / WB_CHUNK + 1;
      // a leaf of at most 537 points spans at most 18 groups; a longer one is
      // not pruned
      wide = ng > 32;
      if (wide) ng = 0;
    }
    uint32_t tot;
    K.pre[lane] = wave_prefix(ng, tot);
    K.b[lane] = b;
    K.e[lane] = e;
    K.mask[lane] = wide ? ~0u : 0u;
    __syncthreads();
    leaf_groups(T, S, K, nb, tot, [&](int q, uint32_t g, bool hit) {
      if (hit) atomicOr(&K.mask[q], 1u << (g - K.b[q] / WB_CHUNK));
    });
    __syncthreads();
    // K.e: first group of a leaf whose points are tested, all ones for whole
    const uint32_t np = all || K.mask[lane] ? e - b : 0u;
    K.pre[lane] = wave_prefix(np, tot);
    const uint32_t g0 = all ? ~0u : wide ? ~0u - 1 : b / WB_CHUNK;
    K.e[lane] = g0;
    __syncthreads();
    constexpr int U = 4;
    for (uint32_t t0 = 0; t0 < tot; t0 += U * WAVE) {
      uint32_t slot[U];
      int q[U];
      bool in[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const uint32_t t = t0 + u * WAVE + lane;
        in[u] = t < tot;
        q[u] = prefix_find(K.pre, nb, in[u] ? t : 0u);
        slot[u] = in[u] ? T.canon[K.b[q[u]] + (t - K.pre[q[u]])] : 0u;
      }
      double x[U], y[U], z[U];
      bool test[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const uint32_t gq = K.e[q[u]];
        test[u] = in[u] && gq != ~0u;
        if (test[u] && gq != ~0u - 1) test[u] = in[u] = (K.mask[q[u]] >> (slot[u] / WB_CHUNK - gq)) & 1u;
        if (test[u]) {
          x[u] = T.px[slot[u]];
          y[u] = T.py[slot[u]];
          z[u] = T.pz[slot[u]];
        }
      }
      uint32_t id[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        if (test[u]) in[u] = wb::shape_in(S, x[u], y[u], z[u]);
        if (in[u]) id[u] = T.sidx[slot[u]];
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const uint64_t bal = __ballot(in[u]);
        const uint64_t w = pos + (uint64_t)__popcll(bal & lt);
        if (in[u] && w < lim) out[w] = id[u];
        pos += (uint64_t)__popcll(bal);
      }
    }
    __syncthreads();
  });
}

// ---------------------------------------------------------------------------
// Batched countPointsIn / pointsIn with a lane per shape.  The shapes are
// taken in Morton order of their centres (k_query_keys + the radix sort), so
// the 64 shapes of a wave are neighbours and share most of their leaves.
// A wave walks the octree once for its 64 shapes: findBlocks
// (octree.cpp:234-251) with an explicit stack whose entries carry the mask of
// lanes for which the node and every ancestor intersect the lane's shape, so
// each lane sees exactly the leaves findBlocks returns for its own shape, in
// the same (DFS) order.  A leaf whose eight corners are all in a lane's shape
// counts whole for that lane (octree.cpp:1226-1231, 1256-1257); otherwise the
// lane tests the leaf's points, skipping 32-point groups whose bounding box
// no point of the shape can reach (wb::shape_may_hit_box: exact).  A group's
// points are read once per wave with one vector load and handed to every
// lane by readlane.
// ---------------------------------------------------------------------------
// pending entries at one time: at most 7 siblings per level on the path plus
// 8 children (internal nodes sit at levels 0..WB_MAX_LEVEL)
#define WB_QSTK (7 * (WB_MAX_LEVEL + 1) + 8 + 2)
struct QueryStack {
  int code[WB_QSTK];
  uint32_t lo[WB_QSTK], hi[WB_QSTK];
};

// The walk: leaf(l, on) for every leaf some lane reaches, in DFS order; `on`
// tells whether this lane's findBlocks returns it.
template <class Leaf>
__device__ inline void query_walk(const TreeView &T, const wb::Shape &S, bool active,
                                  QueryStack &K, Leaf &&leaf)
{
  if (T.nleaves == 0) return;
  const uint64_t m0 = __ballot(active && wb::shape_intersect(S, T.node_cube[0], T.node_cube[1],
                                                             T.node_cube[2], T.node_cube[3]));
  if (!m0) return;
  K.code[0] = 0;
  K.lo[0] = (uint32_t)m0;
  K.hi[0] = (uint32_t)(m0 >> 32);
  int sp = 1;
  const uint32_t lane = __lane_id();
  while (sp > 0) {
    sp--;
    const int code = rfl(K.code[sp]);
    const uint32_t mlo = (uint32_t)rfl((int)K.lo[sp]), mhi = (uint32_t)rfl((int)K.hi[sp]);
    const bool on = ((lane < 32 ? mlo >> lane : mhi >> (lane - 32)) & 1u) != 0;
    if (code < 0) {
      leaf(-2 - code, on);
      continue;
    }
    const double *nc = T.node_cube + 4 * (size_t)code;
    const double cx = nc[0], cy = nc[1], cz = nc[2], side = nc[3];
    const int *chp = T.node_child + 8 * (size_t)code;
    int ck[8];
    uint64_t mk[8];
    uint32_t pushed = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) ck[k] = rfl(chp[k]);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      mk[k] = 0;
      if (ck[k] != -1) {
        double x, y, z, sd;
        child_cube(cx, cy, cz, side, k, x, y, z, sd);
        mk[k] = __ballot(on && wb::shape_intersect(S, x, y, z, sd));
        if (mk[k]) pushed |= 1u << k;
      }
    }
    // child 0 on top: a child's entry sits below those of the smaller indices
#pragma unroll
    for (int k = 0; k < 8; k++) {
      if (mk[k]) {
        const int pos = sp + __popc(pushed >> (k + 1));
        K.code[pos] = ck[k];
        K.lo[pos] = (uint32_t)mk[k];
        K.hi[pos] = (uint32_t)(mk[k] >> 32);
      }
    }
    sp += __popc(pushed);
  }
}

// Morton key of a shape's centre in the tree's root cube (21 bits per axis,
// z, y, x interleaved as the octree's child index): the visiting order of the
// lane-per-shape kernels.  A cylinder has no z.
__device__ inline uint32_t query_cell(double d, double inv_cell)
{
  const double u = d * inv_cell;
  if (!(u >= 0.0)) return 0;
  if (u >= (double)(1u << WB_MAX_LEVEL)) return (1u << WB_MAX_LEVEL) - 1;
  return (uint32_t)u;
}

__device__ inline uint64_t spread3(uint32_t v)
{
  uint64_t x = v & 0x1fffffull;
  x = (x | (x << 32)) & 0x1f00000000ffffull;
  x = (x | (x << 16)) & 0x1f0000ff0000ffull;
  x = (x | (x << 8)) & 0x100f00f00f00f00full;
  x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
  x = (x | (x << 2)) & 0x1249249249249249ull;
  return x;
}

__global__ void k_query_keys(const double *params, uint64_t ns, int kind, double lox, double loy,
                             double loz, double inv_cell, uint32_t *key, uint32_t *val)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ns) return;
  const double *p = params + WB_SHAPE_NPARAMS * i;
  const uint32_t cx = query_cell(p[0] - lox, inv_cell), cy = query_cell(p[1] - loy, inv_cell);
  const uint32_t cz = kind == wb::SHAPE_CYLINDER ? 0u : query_cell(p[2] - loz, inv_cell);
  // the top 32 of the 63 key bits (cells of side/1024 in x and y) give the
  // locality that matters
  key[i] = (uint32_t)((spread3(cx) | (spread3(cy) << 1) | (spread3(cz) << 2)) >> 31);
  val[i] = (uint32_t)i;
}

// lane o's value of v (o wave-uniform)
__device__ inline uint64_t rdl64(uint64_t v, uint32_t o)
{
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, (int)o);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), (int)o);
  return ((uint64_t)hi << 32) | lo;
}

// lane o's shape (o wave-uniform), read from the lane that holds it
__device__ inline wb::Shape lane_shape(const wb::Shape &S, uint32_t o)
{
  wb::Shape R = S;
  R.cx = rdl(S.cx, o);
  R.cy = rdl(S.cy, o);
  R.cz = rdl(S.cz, o);
  R.r = rdl(S.r, o);
  R.por2 = rdl(S.por2, o);
  R.slope = rdl(S.slope, o);
  return R;
}

// countPointsIn of shapes order[64w .. 64w+63] by wave w.  Inside a leaf,
// each 32-point group is loaded once (lanes 0-31 and 32-63 both hold it)
// and tested against the shapes of the lanes that may reach it ("owners"),
// two per step: lanes 0-31 against the first owner's shape, lanes 32-63
// against the second's, the two ballot halves counted for their owners.
template <int KIND>
__global__ void __launch_bounds__(256) k_query_count(TreeView T, const double *params,
                                                     const uint32_t *order, uint64_t ns,
                                                     uint64_t *counts)
{
  __shared__ QueryStack stk[4];
  QueryStack &K = stk[threadIdx.x / WAVE];
  const uint32_t lane = __lane_id();
  const uint64_t q = (uint64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const bool active = q < ns;
  const uint32_t si = active ? order[q] : 0u;
  const wb::Shape S = query_shape<KIND>(params + WB_SHAPE_NPARAMS * (uint64_t)si);
  uint64_t cnt = 0;
  const bool hi_half = lane >= WAVE / 2;
  query_walk(T, S, active, K, [&](int l, bool on) {
    const double *lc = T.leaf_cube + 4 * (size_t)l;
    const uint32_t b = T.leaf_start[l], e = T.leaf_start[l + 1];
    if (e <= b) return;
    const bool all = on && wb::shape_in_cube(S, lc[0], lc[1], lc[2], lc[3]);
    if (all) cnt += e - b;
    const bool rest = on && !all;
    if (!__ballot(rest)) return;
    const uint32_t g1 = (e - 1) / WB_CHUNK;
    for (uint32_t g = b / WB_CHUNK; g <= g1; g++) {
      const double *bx = T.chunk_box + 6 * (size_t)g;
      const bool hit = rest && wb::shape_may_hit_box(S, bx[0], bx[1], bx[2], bx[3], bx[4], bx[5]);
      uint64_t own = __ballot(hit);
      if (!own) continue;
      const uint32_t base = g * WB_CHUNK;
      const uint32_t j = base + (lane & (WB_CHUNK - 1));
      const bool valid = j >= b && j < e;
      double x = 0, y = 0, z = 0;
      if (valid) {
        x = T.px[j];
        y = T.py[j];
        z = T.pz[j];
      }
      while (own) {
        const uint32_t o1 = (uint32_t)__ffsll((long long)own) - 1;
        own &= own - 1;
        const bool two = own != 0;
        const uint32_t o2 = two ? (uint32_t)__ffsll((long long)own) - 1 : o1;
        own &= own - 1;
        const wb::Shape A = lane_shape(S, o1), B = lane_shape(S, o2);
        const wb::Shape &H = hi_half ? B : A;
        const uint64_t in = __ballot(valid && wb::shape_in(H, x, y, z));
        if (lane == o1) cnt += __popcll(in & 0xffffffffull);
        if (two && lane == o2) cnt += __popcll(in >> 32);
      }
    }
  });
  if (active) counts[si] = cnt;
}

// pointsIn of shapes order[64w .. 64w+63] by wave w: each shape's input
// indices from offs[shape] on, leaf by leaf in DFS order and in canonical
// (input) order inside a leaf, as k_points_in writes them.  A leaf is read
// in canonical order 64 points at a time; each such group is tested against
// the shape of every lane that takes the leaf (one owner per step, its
// indices written by consecutive lanes).
template <int KIND>
__global__ void __launch_bounds__(256) k_query_points(TreeView T, const double *params,
                                                      const uint32_t *order, uint64_t ns,
                                                      const uint64_t *offs, uint32_t *out)
{
  __shared__ QueryStack stk[4];
  QueryStack &K = stk[threadIdx.x / WAVE];
  const uint32_t lane = __lane_id();
  const uint64_t q = (uint64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const bool active = q < ns;
  const uint32_t si = active ? order[q] : 0u;
  const wb::Shape S = query_shape<KIND>(params + WB_SHAPE_NPARAMS * (uint64_t)si);
  // the writes stay inside the shape's own range whatever the walk finds
  uint64_t pos = active ? offs[si] : 0;
  const uint64_t lim = active ? offs[si + 1] : 0;
  const uint64_t lt = (1ull << lane) - 1ull;
  query_walk(T, S, active, K, [&](int l, bool on) {
    const double *lc = T.leaf_cube + 4 * (size_t)l;
    const uint32_t b = T.leaf_start[l], e = T.leaf_start[l + 1];
    if (e <= b) return;
    const bool all = on && wb::shape_in_cube(S, lc[0], lc[1], lc[2], lc[3]);
    const bool rest = on && !all;
    // bit g - g0: the lane's shape may reach 32-point group g (a leaf of at
    // most 537 points spans at most 18 groups; a longer one is not pruned)
    const uint32_t g0 = b / WB_CHUNK, g1 = (e - 1) / WB_CHUNK;
    const bool wide = g1 - g0 >= 32;
    uint32_t gm = 0;
    if (wide) {
      gm = rest ? ~0u : 0u;
    } else if (__ballot(rest)) {
      for (uint32_t g = g0; g <= g1; g++) {
        const double *bx = T.chunk_box + 6 * (size_t)g;
        if (rest && wb::shape_may_hit_box(S, bx[0], bx[1], bx[2], bx[3], bx[4], bx[5]))
          gm |= 1u << (g - g0);
      }
    }
    const uint64_t owners = __ballot(all || gm != 0);
    if (!owners) return;
    for (uint32_t c0 = b; c0 < e; c0 += WAVE) {
      const uint32_t c = c0 + lane;
      const bool valid = c < e;
      uint32_t slot = 0, id = 0;
      double x = 0, y = 0, z = 0;
      if (valid) {
        slot = T.canon[c];
        id = T.sidx[slot];
        x = T.px[slot];
        y = T.py[slot];
        z = T.pz[slot];
      }
      const uint32_t gb = valid && !wide ? slot / WB_CHUNK - g0 : 0;
      uint64_t own = owners;
      while (own) {
        const uint32_t o = (uint32_t)__ffsll((long long)own) - 1;
        own &= own - 1;
        const bool ao = __builtin_amdgcn_readlane((int)all, (int)o) != 0;
        const uint32_t go = (uint32_t)__builtin_amdgcn_readlane((int)gm, (int)o);
        bool in = valid && ao;
        if (!ao) {
          const wb::Shape H = lane_shape(S, o);
          in = valid && ((go >> gb) & 1u) && wb::shape_in(H, x, y, z);
        }
        const uint64_t bal = __ballot(in);
        if (!bal) continue;
        const uint64_t p0 = rdl64(pos, o), l0 = rdl64(lim, o);
        const uint64_t w = p0 + (uint64_t)__popcll(bal & lt);
        if (in && w < l0) out[w] = id;
        if (lane == o) pos = p0 + (uint64_t)__popcll(bal);
      }
    }
  });
}

// ---------------------------------------------------------------------------
// Tiles
// ---------------------------------------------------------------------------
struct TileGeo {
  double scx, scy, spacing, r;
  int lo, hi;
  uint32_t ntiles;
  // dense Eisenstein-address -> counter index map over the island's box
  int gx0, gy0, gw, gh;
  const int32_t *grid;
};

// counter of the tile at Eisenstein (ex, ey), false if it is not a tile
__device__ inline bool tile_at(const TileGeo &g, int ex, int ey, int *cnt)
{
  int gx = ex - g.gx0, gy = ey - g.gy0;
  if (gx < 0 || gy < 0 || gx >= g.gw || gy >= g.gh) return false;
  int k = g.grid[(int64_t)gy * g.gw + gx];
  if (k < 0) return false;
  *cnt = g.lo + k;
  return true;
}

// Flowsnake::cyl, flowsnake.cpp:263-271
__device__ inline void tile_center(const TileGeo &g, int ex, int ey, double *cx, double *cy)
{
  double zr = ex - ey / 2., zi = ey * kSqrt34;
  zr *= g.spacing;
  zi *= g.spacing;
  *cx = zr + g.scx;
  *cy = zi + g.scy;
}

__global__ void k_tile_geo(TileGeo g, int32_t *tex, int32_t *tey, int *bounds)
{
  uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  int ex = 0, ey = 0;
  bool ok = k < g.ntiles;
  if (ok) {
    wb::to_flowsnake_dev((int64_t)g.lo + k, &ex, &ey);
    tex[k] = ex;
    tey[k] = ey;
  }
  int x0 = ok ? ex : INT32_MAX, x1 = ok ? ex : INT32_MIN, y0 = ok ? ey : INT32_MAX, y1 = ok ? ey : INT32_MIN;
  for (int s = 1; s < 64; s <<= 1) {
    x0 = min(x0, __shfl_xor(x0, s, 64));
    x1 = max(x1, __shfl_xor(x1, s, 64));
    y0 = min(y0, __shfl_xor(y0, s, 64));
    y1 = max(y1, __shfl_xor(y1, s, 64));
  }
  // one atomic per block and bound
  __shared__ int wb4[4][256 / 64];
  const int w = threadIdx.x / 64;
  if (__lane_id() == 0) {
    wb4[0][w] = x0; wb4[1][w] = x1; wb4[2][w] = y0; wb4[3][w] = y1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < (int)blockDim.x / 64; k++) {
      x0 = min(x0, wb4[0][k]); x1 = max(x1, wb4[1][k]);
      y0 = min(y0, wb4[2][k]); y1 = max(y1, wb4[3][k]);
    }
    atomicMin(&bounds[0], x0);
    atomicMax(&bounds[1], x1);
    atomicMin(&bounds[2], y0);
    atomicMax(&bounds[3], y1);
  }
}

// clears a pass's counters: per tile the points, the list places taken and the
// state (0 empty, 1 scanned, 2 a tree tile), and the 64 words of err (one launch: a memset of an odd size is two)
__global__ void __launch_bounds__(256) k_pass_init(uint32_t ntiles, uint32_t *tile_cnt,
                                                   uint32_t *tile_fill, uint32_t *state,
                                                   uint32_t *err)
{
  const uint32_t b = blockIdx.x * 1024 + threadIdx.x;
#pragma unroll
  for (uint32_t k = 0; k < 4; k++)
    if (b + 256 * k < ntiles) {
      tile_cnt[b + 256 * k] = 0;
      tile_fill[b + 256 * k] = 0;
    }
  const uint32_t w = blockIdx.x * 256 + threadIdx.x;
  if (w < ntiles / 4 + 1) state[w] = 0;
  if (b < 64) err[b] = 0;
}

__global__ void k_fill_i32(int32_t *p, uint64_t n, int32_t v)
{
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_bounds_init(int *b)
{
  if (threadIdx.x == 0) {
    b[0] = INT32_MAX;
    b[1] = INT32_MIN;
    b[2] = INT32_MAX;
    b[3] = INT32_MIN;
  }
}

__global__ void k_tile_grid(TileGeo g, const int32_t *tex, const int32_t *tey, int32_t *grid)
{
  uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= g.ntiles) return;
  grid[(int64_t)(tey[k] - g.gy0) * g.gw + (tex[k] - g.gx0)] = (int32_t)k;
}

#define MAX_MEMB 4

// the lanes with `has` whose key equals this lane's (0 without `has`)
__device__ inline uint64_t wave_peers(bool has, int key)
{
  uint64_t todo = __ballot(has), peers = 0;
  while (todo) {
    const int kl = __builtin_amdgcn_readlane(key, __ffsll((long long)todo) - 1);
    const bool same = has && key == kl;
    const uint64_t m = __ballot(same);
    if (same) peers = m;
    todo &= ~m;
  }
  return peers;
}

// cnt[key] += 1 for every active lane with `has`: the peer masks first, then
// one atomic per distinct key from its first lane, none of them waited for
// (no slot is returned)
__device__ inline void wave_count_inc(uint32_t *cnt, bool has, int key)
{
  const uint64_t peers = wave_peers(has, key);
  if (has && __ffsll((long long)peers) - 1 == (int)__lane_id())
    atomicAdd(&cnt[key], (uint32_t)__popcll(peers));
}

// Slot claims of a wave, K keys per lane: for each k, one atomic on
// cnt[key[k]] per distinct key from its first lane, each lane's base read
// from that lane, lanes with the same key given consecutive slots in lane
// order (slot[k], where has[k]).  The atomics of all K keys are issued
// before any is waited for: one round trip per wave.
template <int K>
__device__ inline void wave_claim_n(uint32_t *cnt, const bool (&has)[K], const int (&key)[K],
                                    uint32_t (&slot)[K])
{
  const uint32_t lane = __lane_id();
  uint64_t peers[K];
  int first[K];
  uint32_t base[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    peers[k] = wave_peers(has[k], key[k]);
    first[k] = has[k] ? __ffsll((long long)peers[k]) - 1 : (int)lane;
  }
#pragma unroll
  for (int k = 0; k < K; k++) {
    base[k] = 0;
    if (has[k] && first[k] == (int)lane)
      base[k] = atomicAdd(&cnt[key[k]], (uint32_t)__popcll(peers[k]));
  }
#pragma unroll
  for (int k = 0; k < K; k++)
    slot[k] = (uint32_t)__shfl((int)base[k], first[k], 64) +
              (uint32_t)__popcll(peers[k] & ((1ull << lane) - 1));
}

// The (leaf, tile) part of the membership test, once per leaf for the
// lattice cells near it: a window of cells (ex, ey), ex in [x0, x0+w), ey in
// [y0, y0+h), w*h <= LEAF_WIN, covering every cell whose centre can lie
// within the candidate bound of a point inside the leaf's square (one cell
// of slack on each side).  Flag bit 0: a tile whose cylinder findBlocks
// reaches this leaf through (every ancestor cube and the leaf cube intersect
// it); bit 1: all eight leaf corners in the cylinder.  w = 0: the leaf's
// window is too large and its points take the full test.
#define LEAF_WIN 256
struct LeafWin {
  int x0, y0, w, h;
};

__global__ void __launch_bounds__(64) k_leaf_tiles(TreeView T, TileGeo g, LeafWin *win,
                                                   uint8_t *flags)
{
  const uint32_t l = blockIdx.x;
  if (l >= T.nleaves) return;
  const double *lc = T.leaf_cube + 4 * (size_t)l;
  const double h = lc[3] / 2, lim = g.r * (1 + 1e-9) + 1e-9;
  const double fy0 = ((lc[1] - h - lim) - g.scy) / g.spacing / kSqrt34;
  const double fy1 = ((lc[1] + h + lim) - g.scy) / g.spacing / kSqrt34;
  const double u0 = ((lc[0] - h - lim) - g.scx) / g.spacing;
  const double u1 = ((lc[0] + h + lim) - g.scx) / g.spacing;
  LeafWin wl = {0, 0, 0, 0};
  if (fabs(fy0) < 1e9 && fabs(fy1) < 1e9 && fabs(u0) < 1e9 && fabs(u1) < 1e9) {
    wl.y0 = (int)floor(fy0) - 1;
    const int y1 = (int)ceil(fy1) + 1;
    wl.x0 = (int)floor(u0 + wl.y0 / 2.0) - 1;
    const int x1 = (int)ceil(u1 + y1 / 2.0) + 1;
    wl.w = x1 - wl.x0 + 1;
    wl.h = y1 - wl.y0 + 1;
    if (wl.w <= 0 || wl.h <= 0 || wl.w * wl.h > LEAF_WIN) wl.w = wl.h = 0;
  }
  if (threadIdx.x == 0) win[l] = wl;
  const int ncell = wl.w * wl.h;
  // the ancestors' cubes: their numbers one after the other, the cubes read
  // together.  (Read cell by cell, two loads per ancestor in turn, the walk up
  // was the kernel: 23.7M points 0.22 ms, 0.15 so.)
  __shared__ double anc[WB_MAX_LEVEL + 1][4];
  int na = 0, mine = -1;
  for (int nd = rfl(T.leaf_parent[l]); nd >= 0; nd = rfl(T.node_parent[nd])) {
    if ((int)threadIdx.x == na) mine = nd;
    na++;
  }
  if (mine >= 0) {
#pragma unroll
    for (int k = 0; k < 4; k++) anc[threadIdx.x][k] = T.node_cube[4 * (size_t)mine + k];
  }
  __syncthreads();
  for (int c = threadIdx.x; c < ncell; c += 64) {
    const int ex = wl.x0 + c % wl.w, ey = wl.y0 + c / wl.w;
    uint8_t f = 0;
    int cnt;
    if (tile_at(g, ex, ey, &cnt)) {
      double cx, cy;
      tile_center(g, ex, ey, &cx, &cy);
      const wb::Shape cyl = wb::make_cylinder(cx, cy, g.r);
      bool reach = wb::shape_intersect(cyl, lc[0], lc[1], lc[2], lc[3]);
      for (int a = 0; reach && a < na; a++)
        reach = wb::shape_intersect(cyl, anc[a][0], anc[a][1], anc[a][2], anc[a][3]);
      if (reach) f = 1 | (wb::shape_in_cube(cyl, lc[0], lc[1], lc[2], lc[3]) ? 2 : 0);
    }
    flags[(size_t)l * LEAF_WIN + c] = f;
  }
}

// the lattice point itself (k = 0) and its six neighbours
__device__ inline int near_a(int k) { return (int)((0x949u >> (2 * k)) & 3u) - 1; }
__device__ inline int near_b(int k) { return (int)((0x895u >> (2 * k)) & 3u) - 1; }

// pointsIn(cylinder) membership of every point, evaluated from the point's
// side: the candidates are the lattice tiles near it; a tile holds the point
// iff findBlocks reaches its leaf (every ancestor cube and the leaf cube
// intersect the cylinder) and either all eight leaf corners are in or the
// point itself is.  The leaf's part comes from its k_leaf_tiles window;
// candidates outside the window (points outside their leaf's cube) take the
// whole test.
__global__ void __launch_bounds__(256, 5) k_membership(TreeView T, TileGeo g, const LeafWin *win,
                                                       const uint8_t *flags, int32_t *memb,
                                                       uint32_t *nmemb, uint32_t *tile_cnt,
                                                       uint32_t *err)
{
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= T.n) return;
  const double x = T.px[i], y = T.py[i];
  const uint32_t leaf = T.pt_leaf[i];
  const double *lc = T.leaf_cube + 4 * leaf;
  const LeafWin wl = win[leaf];
  // The lattice point nearest to p (Eisenstein coordinates a + b*omega,
  // centre spacing*(a - b/2, b*sqrt3/2)) by rounding the cube coordinates
  // (a - b, b, -a) and fixing the one rounded farthest.  A centre within the
  // candidate bound (spacing*41/71, a hair over the hexagon's circumradius
  // spacing/sqrt3) of p lies within 1.16 spacings of that point, so it is the
  // point itself or one of its six neighbours (the next ring is sqrt3
  // spacings away); a rounding near a tie that picks a neighbour of the
  // nearest point still leaves every such centre in the seven.
  // (u and v only choose the seven: products with the reciprocals do)
  const double inv = 1 / g.spacing;
  const double u = (x - g.scx) * inv, v = (y - g.scy) * inv;
  const double fb = v * (1 / kSqrt34), fa = u + fb / 2;
  double rx = __builtin_rint(fa - fb), ry = __builtin_rint(fb), rz = __builtin_rint(-fa);
  const double ddx = fabs(rx - (fa - fb)), ddy = fabs(ry - fb), ddz = fabs(rz + fa);
  if (ddy > ddx && ddy > ddz) ry = -rx - rz;
  else if (ddz >= ddx && ddz >= ddy) rz = -rx - ry;
  const int X = (int)-rz, Y = (int)ry;
  const double lim = g.r * (1 + 1e-9) + 1e-9;
  // The candidates of the seven within the bound: one to three.  Each lane's
  // own are then looked up side by side, three at a time: the tiles' numbers,
  // the leaf's flags of them and the tests.  One candidate of the seven after
  // the other, for whichever lanes had it, every wave waited for all seven
  // pairs of loads (23.7M points 0.79 ms, 0.43 so).
  uint32_t cand = 0;
#pragma unroll
  for (int k = 0; k < 7; k++) {
    double cx, cy;
    tile_center(g, X + near_a(k), Y + near_b(k), &cx, &cy);
    const double dx = cx - x, dy = cy - y;
    if (dx * dx + dy * dy <= lim * lim) cand |= 1u << k;
  }
  int nm = 0;
  int32_t mem[MAX_MEMB] = {INT32_MIN, INT32_MIN, INT32_MIN, INT32_MIN};
  while (cand) {
    constexpr int P = 3;
    int ex[P], ey[P], cnt[P];
    uint8_t f[P];  // bit 0 a tile that reaches the leaf, bit 1 holds it whole, 128 outside the window
    bool at[P];
#pragma unroll
    for (int j = 0; j < P; j++) {
      at[j] = cand != 0;
      const int k = cand ? __builtin_ctz(cand) : 0;
      cand &= cand - 1;
      ex[j] = X + near_a(k);
      ey[j] = Y + near_b(k);
    }
#pragma unroll
    for (int j = 0; j < P; j++) at[j] = at[j] && tile_at(g, ex[j], ey[j], &cnt[j]);
#pragma unroll
    for (int j = 0; j < P; j++) {
      const int gx = ex[j] - wl.x0, gy = ey[j] - wl.y0;
      const bool inside = gx >= 0 && gy >= 0 && gx < wl.w && gy < wl.h;
      f[j] = 0;
      if (at[j]) f[j] = inside ? flags[(size_t)leaf * LEAF_WIN + gy * wl.w + gx] : 128;
    }
#pragma unroll
    for (int j = 0; j < P; j++) {
      if (!f[j]) continue;
      double cx, cy;
      tile_center(g, ex[j], ey[j], &cx, &cy);
      const wb::Shape cyl = wb::make_cylinder(cx, cy, g.r);
      bool in = (f[j] & 1) && ((f[j] & 2) || wb::cyl_in(cyl, x, y));
      if (f[j] & 128) {
        in = wb::shape_in_cube(cyl, lc[0], lc[1], lc[2], lc[3]) || wb::cyl_in(cyl, x, y);
        in = in && wb::shape_intersect(cyl, lc[0], lc[1], lc[2], lc[3]);
        for (int nd = T.leaf_parent[leaf]; in && nd >= 0; nd = T.node_parent[nd]) {
          const double *q = T.node_cube + 4 * nd;
          in = wb::shape_intersect(cyl, q[0], q[1], q[2], q[3]);
        }
      }
      if (in) {
#pragma unroll
        for (int k = 0; k < MAX_MEMB; k++)
          if (k == nm) mem[k] = cnt[j];
        nm++;
      }
    }
  }
  if (nm > MAX_MEMB) {
    atomicOr(err, 1u);
    nm = MAX_MEMB;
  }
  ((int4 *)memb)[i] = make_int4(mem[0], mem[1], mem[2], mem[3]);
  nmemb[i] = nm;
#pragma unroll
  for (int k = 0; k < MAX_MEMB; k++) wave_count_inc(tile_cnt, k < nm, k < nm ? mem[k] - g.lo : 0);
}

__global__ void k_tile_lists(uint64_t n, const int32_t *memb, const uint32_t *nmemb, int lo,
                             const uint32_t *crank, const uint32_t *tile_off, uint32_t *tile_fill,
                             uint32_t *lists)
{
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t nm = nmemb[i];
  bool has[MAX_MEMB];
  int t[MAX_MEMB];
  uint32_t slot[MAX_MEMB];
#pragma unroll
  for (uint32_t k = 0; k < MAX_MEMB; k++) {
    has[k] = k < nm;
    t[k] = has[k] ? memb[MAX_MEMB * i + k] - lo : 0;
  }
  // the slot claims of all memberships in one round of atomics
  wave_claim_n<MAX_MEMB>(tile_fill, has, t, slot);
  const uint32_t cr = crank[i];
#pragma unroll
  for (uint32_t k = 0; k < MAX_MEMB; k++)
    if (has[k]) lists[tile_off[t[k]] + slot[k]] = cr;
}

// ---------------------------------------------------------------------------
// SCAN: one wave per tile (scanCylinder, scan.cpp:31-140)
// ---------------------------------------------------------------------------
#define SCAN_CAP 1024

// pairwisesum (manysum.cpp:120-154) of m <= SCAN_CAP values produced by
// val(j): one balanced tree per set bit of m, over the aligned block that
// bit owns (largest block first), block sums added to 0 in ascending bit
// order.  Balanced trees of up to 64 values are xor butterflies across the
// wave; larger blocks combine their 64-value chunk sums the same way.
template <class V>
__device__ inline double wave_pairwise(uint32_t m, V &&val)
{
  const int lane = __lane_id();
  double acc = 0;
  for (int k = 0; k < 11; k++) {
    if (!((m >> k) & 1u)) continue;
    uint32_t off = (m >> (k + 1)) << (k + 1);
    uint32_t sz = 1u << k;
    double blk;
    if (sz <= 64) {
      double v = (uint32_t)lane < sz ? val(off + lane) : 0.0;
      for (uint32_t s = 1; s < sz; s <<= 1) v = v + __shfl_xor(v, (int)s, WAVE);
      blk = __shfl(v, 0, WAVE);
    } else {
      // chunk sums of 64, then a balanced tree over the chunks
      uint32_t nch = sz / 64;
      double mine = 0;
      for (uint32_t ch = 0; ch < nch; ch++) {
        double v = val(off + ch * 64 + lane);
        for (int s = 1; s < 64; s <<= 1) v = v + __shfl_xor(v, s, WAVE);
        if ((uint32_t)lane == ch) mine = v;
      }
      for (uint32_t s = 1; s < nch; s <<= 1) mine = mine + __shfl_xor(mine, (int)s, WAVE);
      blk = __shfl(mine, 0, WAVE);
    }
    acc += blk;
  }
  return acc;
}

__device__ inline double pw3(double a0, double a1, double a2, int n)
{
  // pairwisesum of n <= 3 values
  if (n == 1) return 0 + a0;
  if (n == 2) return 0 + (a0 + a1);
  return (0 + a2) + (a0 + a1);
}

// 3x3 Gauss-Jordan of matrix.cpp:262-422 on a (3x3, row-major) and b (3x1).
// Every row and column index is a compile-time constant, so the system stays
// in registers; the pivot choices made at run time select among them.
// rows R0 and R1 exchanged when `c`, by selects (no indexed access)
template <int R0, int R1>
__device__ __attribute__((always_inline)) inline void swap_rows_s(double (&a)[9], double (&b)[3],
                                                                  bool c)
{
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const double x = a[3 * R0 + k], y = a[3 * R1 + k];
    a[3 * R0 + k] = c ? y : x;
    a[3 * R1 + k] = c ? x : y;
  }
  const double x = b[R0], y = b[R1];
  b[R0] = c ? y : x;
  b[R1] = c ? x : y;
}

__device__ inline double sel3(double r0, double r1, double r2, int k)
{
  return k == 0 ? r0 : (k == 1 ? r1 : r2);
}

// rowop(row0, row1, piv) of matrix.cpp
template <int ROW0, int ROW1, int PIV>
__device__ __attribute__((always_inline)) inline void rowop_s(double (&a)[9], double (&b)[3])
{
  double slope = 0, minslope = __builtin_inf(), det;
  int flags = 0, pivot;
  bool piv_ok = true;  // piv >= 0
  if (a[3 * ROW0 + PIV] == 0 && a[3 * ROW1 + PIV] == 0) piv_ok = false;
  pivot = piv_ok ? PIV : -1;
  if (piv_ok && a[3 * ROW0 + PIV] == 0) flags = 9;
  if (!piv_ok) {
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const double x0 = a[3 * ROW0 + i], x1 = a[3 * ROW1 + i];
      if (x0 != 0 || x1 != 0) {
        if (wb::dabs(x0) > wb::dabs(x1) || ROW0 >= ROW1) {
          slope = wb::dabs(x1 / x0);
          flags &= ~8;
        } else {
          slope = wb::dabs(x0 / x1);
          flags |= 8;
        }
        if (slope < minslope) {
          minslope = slope;
          flags = (flags >> 3) * 9;
          pivot = i;
        }
      }
    }
  }
  flags &= 1;
  swap_rows_s<ROW0, ROW1>(a, b, flags != 0);
  det = (pivot < 0) ? 0 : sel3(a[3 * ROW0], a[3 * ROW0 + 1], a[3 * ROW0 + 2], pivot);
  if (det != 0 && det != 1) {
#pragma unroll
    for (int i = 0; i < 3; i++) a[3 * ROW0 + i] /= det;
    b[ROW0] /= det;
  }
  if (pivot >= 0) slope = sel3(a[3 * ROW1], a[3 * ROW1 + 1], a[3 * ROW1 + 2], pivot);
  if (slope != 0 && ROW0 != ROW1) {
#pragma unroll
    for (int i = 0; i < 3; i++) a[3 * ROW1 + i] -= a[3 * ROW0 + i] * slope;
    b[ROW1] -= b[ROW0] * slope;
  }
}

// findpivot(row, column) of matrix.cpp
template <int ROW>
__device__ __attribute__((always_inline)) inline void findpivot_s(double (&a)[9], double (&b)[3])
{
  int pivotrow = -1;
  double maxratio = 0;
  // the column loop runs while pivotrow < ROW; pivotrow, once set, is >= ROW
#pragma unroll
  for (int column = ROW; column < 3; column++) {
    if (pivotrow < ROW) {
#pragma unroll
      for (int i = ROW; i < 3; i++) {
        const double s0 = column + 1 < 3 ? a[3 * i + column + 1] * a[3 * i + column + 1] : 0.0;
        const double s1 = column + 2 < 3 ? a[3 * i + column + 2] * a[3 * i + column + 2] : 0.0;
        const double piv = a[3 * i + column];
        const double ratio = (piv * piv) / pw3(s0, s1, 0.0, 3 - column);
        if (ratio > maxratio) {
          pivotrow = i;
          maxratio = ratio;
        }
      }
    }
  }
  if constexpr (ROW < 1) swap_rows_s<1, ROW>(a, b, pivotrow == 1);
  if constexpr (ROW < 2) swap_rows_s<2, ROW>(a, b, pivotrow == 2);
}

__device__ __attribute__((always_inline)) inline void gausselim_s(double (&a)[9], double (&b)[3])
{
  findpivot_s<0>(a, b);
  rowop_s<0, 0, 0>(a, b); rowop_s<0, 1, 0>(a, b); rowop_s<0, 2, 0>(a, b);
  findpivot_s<1>(a, b);
  rowop_s<1, 0, 1>(a, b); rowop_s<1, 1, 1>(a, b); rowop_s<1, 2, 1>(a, b);
  findpivot_s<2>(a, b);
  rowop_s<2, 0, 2>(a, b); rowop_s<2, 1, 2>(a, b); rowop_s<2, 2, 2>(a, b);
  // back substitution
  rowop_s<2, 0, 2>(a, b); rowop_s<2, 1, 2>(a, b);
  rowop_s<1, 0, 1>(a, b);
}

// the tilt (sx, sy) of the least-squares plane z = sx*x + sy*y + c through
// the normal equations (scan.cpp:53-73, leastsquares.cpp); every lane holds the same sums and
// gets the same answer
__device__ __attribute__((always_inline)) inline void plane_tilt(double sxx, double syx, double syy, double s1x, double s1y,
                                  double s11, double sxz, double syz, double s1z, double *sx,
                                  double *sy)
{
  double a[9] = {sxx, syx, s1x, syx, syy, s1y, s1x, s1y, s11};
  double b[3] = {sxz, syz, s1z};
  gausselim_s(a, b);
  if (a[0] == 0) b[0] = __builtin_nan("");
  if (a[4] == 0) b[1] = __builtin_nan("");
  if (a[8] == 0) b[2] = __builtin_nan("");
  double p = b[0], q = b[1];
  const double len = wb::hypot(p, q);
  if (len > 1) { p /= len; q /= len; }
  if (wb::disnan(p) || wb::disnan(q)) { p = 0; q = 0; }
  *sx = p;
  *sy = q;
}

// Slot s of a K-slot per-lane array, s wave-uniform.
template <int K, class V>
__device__ inline V slot_sel(const V (&v)[K], uint32_t s)
{
  V r = v[0];
#pragma unroll
  for (int k = 1; k < K; k++)
    if (s == (uint32_t)k) r = v[k];
  return r;
}

// v moved across the lanes of each row of 16 by the DPP control CTRL (every
// lane active; the controls used here read inside the row)
template <int CTRL>
__device__ inline double dpp_d(double v)
{
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf,
                                                            false);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Pairwise sum of lanes base .. base+sz-1 (sz a wave-uniform power of two up
// to 64, base a multiple of sz): lanes 2i and 2i+1 are added, then pairs of
// those sums, and so on.  Each level inside a row pairs every lane with a
// lane of the sibling group (quad_perm 1,0,3,2 and 2,3,0,1, then the
// half-row and row mirrors), whose lanes all hold that group's sum, so
// every addition has the operands of the xor butterfly; the row sums are
// then read and added in the same tree.
__device__ inline double lanes_pairwise(double b, uint32_t sz, uint32_t base)
{
  if (sz >= 2) b = b + dpp_d<0xb1>(b);
  if (sz >= 4) b = b + dpp_d<0x4e>(b);
  if (sz >= 8) b = b + dpp_d<0x141>(b);
  if (sz >= 16) b = b + dpp_d<0x140>(b);
  if (sz == 64) return (rdl(b, 0) + rdl(b, 16)) + (rdl(b, 32) + rdl(b, 48));
  if (sz == 32) return rdl(b, base) + rdl(b, base + 16);
  return rdl(b, base);
}

// minimum and maximum over the wave: the row steps by DPP, the four row
// results read
__device__ inline double wave_dmin(double v)
{
  v = fmin(v, dpp_d<0xb1>(v));
  v = fmin(v, dpp_d<0x4e>(v));
  v = fmin(v, dpp_d<0x141>(v));
  v = fmin(v, dpp_d<0x140>(v));
  return fmin(fmin(rdl(v, 0), rdl(v, 16)), fmin(rdl(v, 32), rdl(v, 48)));
}
__device__ inline double wave_dmax(double v)
{
  v = fmax(v, dpp_d<0xb1>(v));
  v = fmax(v, dpp_d<0x4e>(v));
  v = fmax(v, dpp_d<0x141>(v));
  v = fmax(v, dpp_d<0x140>(v));
  return fmax(fmax(rdl(v, 0), rdl(v, 16)), fmax(rdl(v, 32), rdl(v, 48)));
}

// wave_pairwise for m <= 64*K values held K per lane (value e in slot e/64
// of lane e%64): the same block trees and block order.  The blocks of up to 64
// values lie in the last slot that is not full, aligned to their size, so one
// pass over that slot's levels meets them in ascending order; the larger ones
// are balanced trees over the full slots before it.
template <int K>
__device__ inline double wave_pairwise_reg(uint32_t m, const double (&v)[K])
{
  static_assert(K <= 4, "blocks of up to 256 values");
  double acc = 0;
  const uint32_t full = m / WAVE, rest = m % WAVE;
  if (rest) {
    double b = slot_sel<K>(v, full);
    if (rest & 1) acc += rdl(b, rest & ~1u);
    b = b + dpp_d<0xb1>(b);
    if (rest & 2) acc += rdl(b, rest & ~3u);
    b = b + dpp_d<0x4e>(b);
    if (rest & 4) acc += rdl(b, rest & ~7u);
    b = b + dpp_d<0x141>(b);
    if (rest & 8) acc += rdl(b, rest & ~15u);
    if (rest >= 16) {
      b = b + dpp_d<0x140>(b);
      if (rest & 16) acc += rdl(b, rest & ~31u);
      if (rest & 32) acc += rdl(b, 0) + rdl(b, 16);
    }
  }
  if (full & 1) acc += lanes_pairwise(slot_sel<K>(v, full - 1), WAVE, 0);
  if constexpr (K >= 2) {
    if (full & 2) {
      acc += lanes_pairwise(v[0], WAVE, 0) + lanes_pairwise(v[1], WAVE, 0);
    }
  }
  if constexpr (K >= 4) {
    if (full & 4)
      acc += (lanes_pairwise(v[0], WAVE, 0) + lanes_pairwise(v[1], WAVE, 0)) +
             (lanes_pairwise(v[2], WAVE, 0) + lanes_pairwise(v[3], WAVE, 0));
  }
  return acc;
}

// Sum over the wave of K float slots per lane: plain (naive), or with each
// lane's slots added by Neumaier's compensated sum and the lanes' (sum,
// error) pairs merged by Knuth's TwoSum, so the rounding errors of every
// addition are carried and added once at the end.
template <int K>
__device__ inline float wave_fsum(const float (&v)[K], bool comp)
{
  float s = 0, e = 0;
#pragma unroll
  for (int k = 0; k < K; k++) {
    const float t = s + v[k];
    if (comp) e += wb::dabs(s) >= wb::dabs(v[k]) ? (s - t) + v[k] : (v[k] - t) + s;
    s = t;
  }
  for (int o = 1; o < WAVE; o <<= 1) {
    const float s2 = __shfl_xor(s, o, WAVE), e2 = __shfl_xor(e, o, WAVE);
    const float t = s + s2;
    if (comp) {
      const float bp = t - s;
      e = e + e2 + ((s - (t - bp)) + (s2 - bp));
    }
    s = t;
  }
  return s + e;
}

// The plane tilt from FP32 moments of (x, y, z - z0) (a shift of z leaves the
// tilt unchanged), solved through the centred 2x2 normal equations in FP32.
// Returns false when the xy spread is too close to collinear for FP32
// (det < 1e-3 trace^2 of the centred xy moments, or fewer than 3 points); the
// caller then fits in FP64.
template <int K>
__device__ inline bool plane_tilt_f32(uint32_t m, const double (&vx)[K], const double (&vy)[K],
                                      const double (&vz)[K], const bool (&mine)[K], bool comp,
                                      double *sx, double *sy)
{
  const double z0 = rdl(vz[0], 0);
  float fx[K], fy[K], fz[K], t[K];
#pragma unroll
  for (int s = 0; s < K; s++) {
    fx[s] = mine[s] ? (float)vx[s] : 0.0f;
    fy[s] = mine[s] ? (float)vy[s] : 0.0f;
    fz[s] = mine[s] ? (float)(vz[s] - z0) : 0.0f;
  }
  const float Sx = wave_fsum<K>(fx, comp), Sy = wave_fsum<K>(fy, comp);
  const float Sz = wave_fsum<K>(fz, comp);
#pragma unroll
  for (int s = 0; s < K; s++) t[s] = fx[s] * fx[s];
  const float Sxx = wave_fsum<K>(t, comp);
#pragma unroll
  for (int s = 0; s < K; s++) t[s] = fx[s] * fy[s];
  const float Sxy = wave_fsum<K>(t, comp);
#pragma unroll
  for (int s = 0; s < K; s++) t[s] = fy[s] * fy[s];
  const float Syy = wave_fsum<K>(t, comp);
#pragma unroll
  for (int s = 0; s < K; s++) t[s] = fx[s] * fz[s];
  const float Sxz = wave_fsum<K>(t, comp);
#pragma unroll
  for (int s = 0; s < K; s++) t[s] = fy[s] * fz[s];
  const float Syz = wave_fsum<K>(t, comp);
  const float n = (float)m;
  const float mx = Sx / n, my = Sy / n, mz = Sz / n;
  const float cxx = Sxx - Sx * mx, cyy = Syy - Sy * my, cxy = Sxy - Sx * my;
  const float cxz = Sxz - Sx * mz, cyz = Syz - Sy * mz;
  const float det = cxx * cyy - cxy * cxy, tr = cxx + cyy;
  const bool well = m >= 3 && det > 1e-3f * tr * tr;
  double p = (double)((cxz * cyy - cyz * cxy) / det), q = (double)((cyz * cxx - cxz * cxy) / det);
  const double len = wb::hypot(p, q);
  if (len > 1) { p /= len; q /= len; }
  if (wb::disnan(p) || wb::disnan(q)) { p = 0; q = 0; }
  *sx = p;
  *sy = q;
  return well;
}

// What a tile's scan ends in, one tile per lane: the sums of the normal
// equations, the plane's tilt, the extremes of the untilted heights and the
// bottom layer's sectors.  The solution and the record, a few hundred
// instructions of divisions and square roots, are then done for all the
// wave's tiles at once.
struct TileFit {
  double sxx, syx, syy, s1x, s1y, sxz, syz, s1z;
  double sx, sy, bottom, top;
  uint32_t m, nbottom, hist[7];
};

__device__ __attribute__((always_inline)) inline void fit_solve(TileFit &F)
{
  // (the sum of m ones is exact in any order)
  plane_tilt(F.sxx, F.syx, F.syy, F.s1x, F.s1y, (double)F.m, F.sxz, F.syz, F.s1z, &F.sx, &F.sy);
}

__device__ __attribute__((always_inline)) inline void fit_record(const TileFit &F, double r,
                                                                 double min_hs, int fit_fp64,
                                                                 TileRec *out, uint8_t *state)
{
  double density = 0;
  int tree = 0;
  for (int i = 0; i < 7; i++) density += (int)F.hist[i] * (int)F.hist[i];
  if (F.m > F.nbottom && density < 7) tree = 1;
  density = sqrt(density) * kSqrt7 / (r * r) / M_PI;
  if (F.m > F.nbottom && density < 0.5) tree = 1;
  if (F.top - F.bottom > 1.5) tree = 1;
  TileRec rr;
  rr.npoints = (int32_t)F.m;
  rr.nground = 0;
  rr.tree_flags = tree;
  rr.fit_fp64 = fit_fp64;
  rr.density = density;
  rr.hs_scan = sqrt(1 / density + min_hs * min_hs);
  rr.hs = rr.hs_scan;
  rr.height = F.top - F.bottom;
  rr.tilt_x = F.sx;
  rr.tilt_y = F.sy;
  *out = rr;
  *state = (uint8_t)(1 + tree);
}

// The scan of up to T tiles of at most 64*K points each by one wave, K points
// per lane (point e in slot e/64 of lane e%64): the operations and summation
// order of the general path of k_scan, with the canonical sort done by a
// bitonic network over lanes and slots and every point read once.  Tile j's
// fit is lane j's.  One tile at a time, every lane solving the same equations
// and the sums' levels walked once per block, took 0.80 and 0.76 ms for the
// tiles of up to 64 and 128 points of 23.7M points, against 0.54 and
// 0.67 ms.
template <int K, bool F32, int T>
__device__ __attribute__((always_inline)) inline void scan_reg(
    const TreeView &V, const TileGeo &g, const uint32_t (&t)[T], const uint32_t (&m)[T],
    const int32_t *tex, const int32_t *tey, const uint32_t *tile_off, const uint32_t *lists,
    double min_hs, int prec, TileRec *rec, uint8_t *state, unsigned long long *ctr)
{
  const uint32_t lane = __lane_id();
  uint32_t c[T][K];
#pragma unroll
  for (int j = 0; j < T; j++) {
    const uint32_t off = m[j] ? tile_off[t[j]] : 0u;
#pragma unroll
    for (int s = 0; s < K; s++) {
      const uint32_t e = s * WAVE + lane;
      c[j][s] = e < m[j] ? lists[off + e] : 0xffffffffu;
    }
  }
#pragma unroll
  for (int j = 0; j < T; j++) {
    // canonical order: the m ranks ascending (pads last), sorted only as far
    // as the next power of two
    uint32_t unused[K];
    wbw::wave_sort<K, false>(c[j], unused, wbw::pow2_ceil(m[j]));
  }
  const double r = g.r;
  double vx[T][K], vy[T][K], vz[T][K];
  uint32_t q[T][K];
#pragma unroll
  for (int j = 0; j < T; j++)
#pragma unroll
    for (int s = 0; s < K; s++) q[j][s] = s * WAVE + lane < m[j] ? V.canon[c[j][s]] : 0u;
#pragma unroll
  for (int j = 0; j < T; j++) {
    double cx = 0, cy = 0;
    if (m[j]) tile_center(g, tex[t[j]], tey[t[j]], &cx, &cy);
#pragma unroll
    for (int s = 0; s < K; s++) {
      vx[j][s] = 0; vy[j][s] = 0; vz[j][s] = 0;
      if (s * WAVE + lane < m[j]) {
        vx[j][s] = V.px[q[j][s]] - cx;
        vy[j][s] = V.py[q[j][s]] - cy;
        vz[j][s] = V.pz[q[j][s]] - 0;
      }
    }
  }
  TileFit F;
  F.m = 0;
  F.sxx = F.syx = F.syy = F.s1x = F.s1y = F.sxz = F.syz = F.s1z = 0;
  double px = 0, py = 0;  // lane j's tilt from FP32 moments
  bool fit64 = true;
  int fell_back = 0;
#pragma unroll
  for (int j = 0; j < T; j++) {
    const bool me = lane == (uint32_t)j;
    if (me) F.m = m[j];
    // FP32 fits are an option for the precision study; FP64 is the reference
    if (F32 && prec != WB_FIT_FP64) {
      bool mine[K];
#pragma unroll
      for (int s = 0; s < K; s++) mine[s] = s * WAVE + lane < m[j];
      double fx, fy;
      const bool well =
          plane_tilt_f32<K>(m[j], vx[j], vy[j], vz[j], mine, prec == WB_FIT_FP32_COMP, &fx, &fy);
      const bool back = !well && prec == WB_FIT_FP32_COMP;
      if (me) {
        px = fx;
        py = fy;
        fit64 = back;
        fell_back = back;
      }
      if (!back) continue;
    }
    double a[K];
#define WB_SUM(dst, expr)                            \
  {                                                  \
    _Pragma("unroll") for (int s = 0; s < K; s++) {  \
      const double x = vx[j][s], y = vy[j][s], z = vz[j][s]; \
      (void)x, (void)y, (void)z;                     \
      a[s] = (expr);                                 \
    }                                                \
    const double sum = wave_pairwise_reg<K>(m[j], a); \
    if (me) dst = sum;                               \
  }
    WB_SUM(F.sxx, x * x)
    WB_SUM(F.syx, y * x)
    WB_SUM(F.syy, y * y)
    WB_SUM(F.s1x, 1.0 * x)
    WB_SUM(F.s1y, 1.0 * y)
    WB_SUM(F.sxz, x * z)
    WB_SUM(F.syz, y * z)
    WB_SUM(F.s1z, 1.0 * z)
#undef WB_SUM
  }
  // (with the FP32 options only a tile that fell back has sums to solve)
  if (!F32 || prec == WB_FIT_FP64 || __ballot(fell_back != 0)) fit_solve(F);
  if (F32 && !fit64) {
    F.sx = px;
    F.sy = py;
  }
  uint32_t inexact = 0;  // points whose sector the exact form decides, bit K*j+s
#pragma unroll
  for (int j = 0; j < T; j++) {
    const bool me = lane == (uint32_t)j;
    const double sx = rdl(F.sx, j), sy = rdl(F.sy, j);
    double u[K];
    double bottom = __builtin_inf(), top = -__builtin_inf();
#pragma unroll
    for (int s = 0; s < K; s++) {
      u[s] = vz[j][s] - (sy * vy[j][s] + sx * vx[j][s]);
      if (s * WAVE + lane < m[j]) {
        bottom = fmin(bottom, u[s]);
        top = fmax(top, u[s]);
      }
    }
    bottom = wave_dmin(bottom);
    top = wave_dmax(top);
    uint32_t first = 0xffffffffu;
#pragma unroll
    for (int s = K - 1; s >= 0; s--) {
      const uint64_t atb = __ballot(s * WAVE + lane < m[j] && u[s] == bottom);
      if (atb) first = s * WAVE + (uint32_t)(__ffsll((long long)atb) - 1);
    }
    double bottom2 = __builtin_inf();
#pragma unroll
    for (int s = 0; s < K; s++)
      if (s * WAVE + lane < m[j] && s * WAVE + lane < first) bottom2 = fmin(bottom2, u[s]);
    bottom2 = wave_dmin(bottom2);
    if (wb::disinf(bottom2)) bottom2 = bottom;
    if (me) {
      F.bottom = bottom;
      F.top = top;
    }
    // 7-sector histogram of the bottom layer
    uint32_t nbottom = 0, hist[7] = {0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < K; s++) {
      int sec = -1;
      const bool low = s * WAVE + lane < m[j] && u[s] < bottom2 + 2 * r;
      if (low) {
        sec = wb::scan_sector_est(vx[j][s], vy[j][s], r);
        if (sec < 0) inexact |= 1u << (K * j + s);
      }
      nbottom += (uint32_t)__popcll(__ballot(low));
#pragma unroll
      for (int k = 0; k < 7; k++) hist[k] += (uint32_t)__popcll(__ballot(sec == k));
    }
    if (me) {
      F.nbottom = nbottom;
#pragma unroll
      for (int k = 0; k < 7; k++) F.hist[k] = hist[k];
    }
  }
  if (__ballot(inexact != 0)) {
    uint32_t nedge = 0;
#pragma unroll
    for (int j = 0; j < T; j++)
#pragma unroll
      for (int s = 0; s < K; s++) {
        const bool ask = (inexact >> (K * j + s)) & 1u;
        if (!__ballot(ask)) continue;
        int sec = -1, edge = 0;
        if (ask) {
          double cx, cy;
          tile_center(g, tex[t[j]], tey[t[j]], &cx, &cy);
          sec = wb::scan_sector_exact(V.px[q[j][s]] - cx, V.py[q[j][s]] - cy, r, &edge);
        }
        nedge += (uint32_t)__popcll(__ballot(edge != 0));
#pragma unroll
        for (int k = 0; k < 7; k++) {
          const uint32_t h = (uint32_t)__popcll(__ballot(sec == k));
          if (lane == (uint32_t)j) F.hist[k] += h;
        }
      }
    if (nedge && lane == 0) atomicAdd(&ctr[0], (unsigned long long)nedge);
  }
  uint32_t tl = 0;
#pragma unroll
  for (int j = 0; j < T; j++)
    if (lane == (uint32_t)j) tl = t[j];
  if (lane < T && F.m) {
    fit_record(F, r, min_hs, fell_back, rec + tl, state + tl);
    if (fell_back) atomicAdd(&ctr[7], 1ull);
  }
}

// Size classes of the scan: 0 = 1..tiny points, 1 = up to 16, 2 = 17-32, 3 = 33-64,
// 4 = 65-128, 5 = 129-256, 6 = more.  One thread per tile: every tile with
// points goes on its class's list (the lists of classes 0 and 6 fill la from
// the front and the back, 1 and 5 lb, 2 and 4 lc, 3 ld; ncls[c] the lengths),
// so each class kernel visits only its own tiles.  The order inside a list
// does not matter: every tile's record depends on that tile alone.  An empty
// tile has no record: 64 B for each of 27.8M tile numbers, most of them empty,
// took 0.5 ms.
#define SCAN_NCLS 7
// Points from which each class takes its own launch, several tiles per step
// (and tiny tiles a lane each).  Mixed and own launches, scan and postscan in
// ms: 300k points 0.075 and 0.17, 1.17M 0.195 and 0.22, 2.4M 0.31 and 0.28,
// 2.4M at 8 points per m2 0.48 and 0.28, 10M 1.10 and 0.80 to 0.90.
#define SCAN_MANY (3u << 19)
// blocks of a scan launch (resident ones take more than one step; launching
// 65536 empty blocks takes 15 us)
#define SCAN_GRID 8192
__device__ inline int scan_class(uint32_t m, uint32_t tiny)
{
  return m == 0          ? -1
         : m <= tiny     ? 0
         : m <= 16       ? 1
         : m <= 32       ? 2
         : m <= WAVE     ? 3
         : m <= 2 * WAVE ? 4
         : m <= 4 * WAVE ? 5
                         : 6;
}

__global__ void __launch_bounds__(1024) k_scan_classes(uint32_t ntiles, const uint32_t *tile_cnt,
                                                      uint32_t *la, uint32_t *lb, uint32_t *lc,
                                                      uint32_t *ld, uint32_t *ncls,
                                                      uint32_t tiny)
{
  // slots are claimed per block: the waves' class counts summed in LDS, one
  // atomic per class and block (atomics on the list counters are
  // serialised, so one per wave would cost more than the pass)
  __shared__ uint32_t wcnt[SCAN_NCLS][1024 / WAVE];
  __shared__ uint32_t bbase[SCAN_NCLS];
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t m = t < ntiles ? tile_cnt[t] : 0u;
  const int c = scan_class(m, tiny);
  const uint32_t lane = __lane_id(), w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  uint64_t mk[SCAN_NCLS];
#pragma unroll
  for (int k = 0; k < SCAN_NCLS; k++) {
    mk[k] = __ballot(c == k);
    if (lane == 0) wcnt[k][w] = (uint32_t)__popcll(mk[k]);
  }
  __syncthreads();
  if (threadIdx.x < SCAN_NCLS) {
    const int k = threadIdx.x;
    uint32_t tot = 0;
    for (uint32_t v = 0; v < nw; v++) {
      const uint32_t x = wcnt[k][v];
      wcnt[k][v] = tot;  // exclusive prefix over the block's waves
      tot += x;
    }
    bbase[k] = tot ? atomicAdd(&ncls[k], tot) : 0u;
  }
  __syncthreads();
  if (c < 0) return;
  const uint32_t pos = bbase[c] + wcnt[c][w] + (uint32_t)__popcll(mk[c] & ((1ull << lane) - 1));
  switch (c) {
  case 0: la[pos] = t; break;
  case 1: lb[pos] = t; break;
  case 2: lc[pos] = t; break;
  case 3: ld[pos] = t; break;
  case 4: lc[ntiles - 1 - pos] = t; break;
  case 5: lb[ntiles - 1 - pos] = t; break;
  default: la[ntiles - 1 - pos] = t; break;
  }
}

// A class list: entry i at list[step * i] (step +1 for a list filled from
// the front of its buffer, -1 from the back), n entries.
struct ClassList {
  const uint32_t *list;
  int32_t step;
  const uint32_t *n;
  __device__ uint32_t at(uint32_t i) const { return list[(int64_t)step * i]; }
};

// T tiles per wave and step, over the tiles of one size class: up to 64,
// 65-128 and 129-256 points (K = 1, 2, 4 points per lane).  Each class has its
// own register budget.  The next tiles' numbers are read before these tiles'
// scan.
// F32: the kernel of the FP32 fit options (the precision study); the FP64
// kernel does not carry their code or registers.
template <int K, bool F32, int T, int MINW>
__global__ void __launch_bounds__(64, MINW) k_scan_reg(TreeView V, TileGeo g, const int32_t *tex,
                                                 const int32_t *tey, const uint32_t *tile_off,
                                                 const uint32_t *tile_cnt, const uint32_t *lists,
                                                 ClassList cl, double min_hs, int prec,
                                                 TileRec *rec, uint8_t *state, unsigned long long *ctr)
{
  const uint32_t n = (uint32_t)rfl((int)*cl.n);
  uint32_t i = blockIdx.x * T;
  if (i >= n) return;
  uint32_t next[T];
#pragma unroll
  for (int j = 0; j < T; j++) next[j] = i + j < n ? cl.at(i + j) : 0xffffffffu;
  for (; i < n; i += gridDim.x * T) {
    uint32_t t[T], m[T];
#pragma unroll
    for (int j = 0; j < T; j++) {
      const bool live = next[j] != 0xffffffffu;
      t[j] = live ? next[j] : 0u;
      m[j] = live ? tile_cnt[t[j]] : 0u;
      const uint32_t k = i + gridDim.x * T + j;
      next[j] = k < n ? cl.at(k) : 0xffffffffu;
    }
    scan_reg<K, F32, T>(V, g, t, m, tex, tey, tile_off, lists, min_hs, prec, rec, state, ctr);
  }
}

// ---------------------------------------------------------------------------
// Tiles of at most GS = 16 or 32 points, WAVE/GS of them per wave: group
// q (lanes GS*q .. GS*q+GS-1) scans one tile with the operations of
// scan_reg<1> in the same order (FP64 fit only).  Every exchange stays
// inside a group: the canonical sort is the register network on GS lanes,
// the pairwise sums are the xor butterflies of lanes_pairwise (DPP inside a
// row, one ds_bpermute across the two rows of a 32-lane group) with each
// group's blocks read from the lanes its own point count names, and the
// minima, the first bottom point and the sector counts are taken per group.
// ---------------------------------------------------------------------------
// pairwisesum (manysum.cpp:120-154) of the first m values of this lane's
// group of GS lanes (m may differ between groups; every lane active)
template <int GS>
__device__ inline double group_pairwise(double v, uint32_t m, uint32_t gbase)
{
  constexpr int LV = GS == 16 ? 5 : 6;
  double L[LV];
  L[0] = v;
  L[1] = L[0] + dpp_d<0xb1>(L[0]);
  L[2] = L[1] + dpp_d<0x4e>(L[1]);
  L[3] = L[2] + dpp_d<0x141>(L[2]);
  L[4] = L[3] + dpp_d<0x140>(L[3]);
  if constexpr (GS == 32) L[5] = L[4] + __shfl_xor(L[4], 16, WAVE);
  // the block of bit k of m starts at (m >> (k+1)) << (k+1); block sums are
  // added to 0 in ascending bit order, as wave_pairwise_reg does
  double acc = 0;
#pragma unroll
  for (int k = 0; k < LV; k++) {
    const uint32_t off = (m >> (k + 1)) << (k + 1);
    const double b = __shfl(L[k], (int)(gbase + (off & (GS - 1))), WAVE);
    if ((m >> k) & 1u) acc = acc + b;
  }
  return acc;
}

// minimum / maximum over this lane's group of GS lanes
template <int GS>
__device__ inline double group_dmin(double v)
{
  v = fmin(v, dpp_d<0xb1>(v));
  v = fmin(v, dpp_d<0x4e>(v));
  v = fmin(v, dpp_d<0x141>(v));
  v = fmin(v, dpp_d<0x140>(v));
  if constexpr (GS == 32) v = fmin(v, __shfl_xor(v, 16, WAVE));
  return v;
}
template <int GS>
__device__ inline double group_dmax(double v)
{
  v = fmax(v, dpp_d<0xb1>(v));
  v = fmax(v, dpp_d<0x4e>(v));
  v = fmax(v, dpp_d<0x141>(v));
  v = fmax(v, dpp_d<0x140>(v));
  if constexpr (GS == 32) v = fmax(v, __shfl_xor(v, 16, WAVE));
  return v;
}

// WAVE/GS tiles of the class list at a time and R rounds of them per wave and
// step (the FP64 fit; the FP32 options take these tiles through
// k_scan_reg<1>): entries i0 on of the n.  Lane NG*j + q takes the fit of
// round j's group q.
template <int GS, int R>
__device__ __attribute__((always_inline)) inline void scan_rows(
    const TreeView &V, const TileGeo &g, const int32_t *tex, const int32_t *tey,
    const uint32_t *tile_off, const uint32_t *tile_cnt, const uint32_t *lists, const ClassList &cl,
    uint32_t n, uint32_t i0, double min_hs, TileRec *rec, uint8_t *state, unsigned long long *ctr)
{
  constexpr uint32_t NG = WAVE / GS;
  const uint32_t lane = __lane_id(), grp = lane / GS, gl = lane % GS, gbase = lane - gl;
  const uint64_t gmask = ((1ull << GS) - 1) << gbase;
  const int src = (int)(lane % NG * GS);  // a lane of the group whose fit this one takes
  const double r = g.r;
  uint32_t t[R], m[R], q[R];
  double vx[R], vy[R], vz[R];
#pragma unroll
  for (int j = 0; j < R; j++) {
    const uint32_t i = i0 + j * NG + grp;
    t[j] = i < n ? cl.at(i) : 0u;
    m[j] = i < n ? tile_cnt[t[j]] : 0u;
  }
#pragma unroll
  for (int j = 0; j < R; j++) {
    uint32_t c[1] = {gl < m[j] ? lists[tile_off[t[j]] + gl] : 0xffffffffu};
    // canonical order inside each group: the network on GS lanes sorts every
    // aligned group of GS lanes on its own (pads last)
    uint32_t unused[1];
    wbw::wave_sort<1, false>(c, unused, GS);
    q[j] = gl < m[j] ? V.canon[c[0]] : 0u;
  }
  TileFit F;
  F.m = 0;
  F.sxx = F.syx = F.syy = F.s1x = F.s1y = F.sxz = F.syz = F.s1z = 0;
  uint32_t tl = 0;
#pragma unroll
  for (int j = 0; j < R; j++) {
    vx[j] = vy[j] = vz[j] = 0;
    if (gl < m[j]) {
      double cx, cy;
      tile_center(g, tex[t[j]], tey[t[j]], &cx, &cy);
      vx[j] = V.px[q[j]] - cx;
      vy[j] = V.py[q[j]] - cy;
      vz[j] = V.pz[q[j]] - 0;
    }
  }
#pragma unroll
  for (int j = 0; j < R; j++) {
    const bool me = lane / NG == (uint32_t)j;
    const uint32_t mj = (uint32_t)__shfl((int)m[j], src, WAVE);
    const uint32_t tj = (uint32_t)__shfl((int)t[j], src, WAVE);
    if (me) {
      F.m = mj;
      tl = tj;
    }
#define WB_SUM(dst, expr)                                           \
{                                                                 \
  const double x = vx[j], y = vy[j], z = vz[j];                   \
  (void)x, (void)y, (void)z;                                      \
  const double sum = __shfl(group_pairwise<GS>((expr), m[j], gbase), src, WAVE); \
  if (me) dst = sum;                                              \
}
    WB_SUM(F.sxx, x * x)
    WB_SUM(F.syx, y * x)
    WB_SUM(F.syy, y * y)
    WB_SUM(F.s1x, 1.0 * x)
    WB_SUM(F.s1y, 1.0 * y)
    WB_SUM(F.sxz, x * z)
    WB_SUM(F.syz, y * z)
    WB_SUM(F.s1z, 1.0 * z)
#undef WB_SUM
  }
  fit_solve(F);
  uint32_t inexact = 0;
#pragma unroll
  for (int j = 0; j < R; j++) {
    const bool me = lane / NG == (uint32_t)j;
    const double sx = __shfl(F.sx, (int)(j * NG + grp), WAVE);
    const double sy = __shfl(F.sy, (int)(j * NG + grp), WAVE);
    const bool mine = gl < m[j];
    const double u = vz[j] - (sy * vy[j] + sx * vx[j]);
    const double bottom = group_dmin<GS>(mine ? u : __builtin_inf());
    const double top = group_dmax<GS>(mine ? u : -__builtin_inf());
    const uint64_t atb = __ballot(mine && u == bottom) & gmask;
    const uint32_t first = atb ? (uint32_t)(__ffsll((long long)atb) - 1) - gbase : 0xffffffffu;
    double bottom2 = group_dmin<GS>(mine && gl < first ? u : __builtin_inf());
    if (wb::disinf(bottom2)) bottom2 = bottom;
    // 7-sector histogram of the bottom layer
    int sec = -1;
    const bool low = mine && u < bottom2 + 2 * r;
    if (low) {
      sec = wb::scan_sector_est(vx[j], vy[j], r);
      if (sec < 0) inexact |= 1u << j;
    }
    const double bs = __shfl(bottom, src, WAVE), ts = __shfl(top, src, WAVE);
    const uint64_t smask = ((1ull << GS) - 1) << src;
    const uint32_t nb = (uint32_t)__popcll(__ballot(low) & smask);
    if (me) {
      F.bottom = bs;
      F.top = ts;
      F.nbottom = nb;
    }
#pragma unroll
    for (int k = 0; k < 7; k++) {
      const uint32_t h = (uint32_t)__popcll(__ballot(sec == k) & smask);
      if (me) F.hist[k] = h;
    }
  }
  if (__ballot(inexact != 0)) {
    uint32_t nedge = 0;
#pragma unroll
    for (int j = 0; j < R; j++) {
      const bool ask = (inexact >> j) & 1u;
      if (!__ballot(ask)) continue;
      int sec = -1, edge = 0;
      if (ask) {
        double cx, cy;
        tile_center(g, tex[t[j]], tey[t[j]], &cx, &cy);
        sec = wb::scan_sector_exact(V.px[q[j]] - cx, V.py[q[j]] - cy, r, &edge);
      }
      nedge += (uint32_t)__popcll(__ballot(edge != 0));
      const uint64_t smask = ((1ull << GS) - 1) << src;
#pragma unroll
      for (int k = 0; k < 7; k++) {
        const uint32_t h = (uint32_t)__popcll(__ballot(sec == k) & smask);
        if (lane / NG == (uint32_t)j) F.hist[k] += h;
      }
    }
    if (nedge && lane == 0) atomicAdd(&ctr[0], (unsigned long long)nedge);
  }
  if (lane < NG * R && F.m) fit_record(F, r, min_hs, 0, rec + tl, state + tl);
}

template <int GS, int R, int MINW>
__global__ void __launch_bounds__(64, MINW) k_scan_row(TreeView V, TileGeo g, const int32_t *tex,
                                                       const int32_t *tey, const uint32_t *tile_off,
                                                       const uint32_t *tile_cnt,
                                                       const uint32_t *lists, ClassList cl,
                                                       double min_hs, TileRec *rec, uint8_t *state,
                                                       unsigned long long *ctr)
{
  constexpr uint32_t per = WAVE / GS * R;
  const uint32_t n = (uint32_t)rfl((int)*cl.n);
  for (uint32_t i0 = blockIdx.x * per; i0 < n; i0 += gridDim.x * per)
    scan_rows<GS, R>(V, g, tex, tey, tile_off, tile_cnt, lists, cl, n, i0, min_hs, rec, state, ctr);
}

// The classes of 1 to 256 points in one launch, for the clouds whose classes
// do not fill the chip one by one: a step of a class per block (16-lane groups
// for up to 16 points, 32-lane groups, then a wave per tile).  As five
// launches the chain took the longest tile of each in turn (18.5k points 65
// us, 300k points 126 us, scan and postscan, against 50 and 75 us).
__global__ void __launch_bounds__(64, 4) k_scan_mixed(TreeView V, TileGeo g, const int32_t *tex,
                                                      const int32_t *tey, const uint32_t *tile_off,
                                                      const uint32_t *tile_cnt,
                                                      const uint32_t *lists, ClassList c16,
                                                      ClassList c32, ClassList c64, ClassList c128,
                                                      ClassList c256, double min_hs, TileRec *rec, uint8_t *state,
                                                      unsigned long long *ctr)
{
  const uint32_t n16 = (uint32_t)rfl((int)*c16.n), n32 = (uint32_t)rfl((int)*c32.n);
  const uint32_t n64 = (uint32_t)rfl((int)*c64.n), n128 = (uint32_t)rfl((int)*c128.n);
  const uint32_t n256 = (uint32_t)rfl((int)*c256.n);
  // the longest steps first
  const uint32_t e256 = n256, e128 = e256 + n128, e64 = e128 + n64, e32 = e64 + (n32 + 1) / 2;
  const uint32_t end = e32 + (n16 + 3) / 4;
  for (uint32_t u = blockIdx.x; u < end; u += gridDim.x) {
    if (u >= e32) {
      scan_rows<16, 1>(V, g, tex, tey, tile_off, tile_cnt, lists, c16, n16, 4 * (u - e32), min_hs,
                       rec, state, ctr);
    } else if (u >= e64) {
      scan_rows<32, 1>(V, g, tex, tey, tile_off, tile_cnt, lists, c32, n32, 2 * (u - e64), min_hs,
                       rec, state, ctr);
    } else {
      const uint32_t t[1] = {u >= e128 ? c64.at(u - e128) : u >= e256 ? c128.at(u - e256) : c256.at(u)};
      const uint32_t m[1] = {tile_cnt[t[0]]};
      if (u >= e128)
        scan_reg<1, false, 1>(V, g, t, m, tex, tey, tile_off, lists, min_hs, WB_FIT_FP64, rec, state, ctr);
      else if (u >= e256)
        scan_reg<2, false, 1>(V, g, t, m, tex, tey, tile_off, lists, min_hs, WB_FIT_FP64, rec, state, ctr);
      else
        scan_reg<4, false, 1>(V, g, t, m, tex, tey, tile_off, lists, min_hs, WB_FIT_FP64, rec, state, ctr);
    }
  }
}

// ---------------------------------------------------------------------------
// Tiles of at most 8 points, a lane each (the FP64 fit): the operations of
// scan_reg<1> in the same order on one lane's registers.  Sixteen lanes per
// tile took 1.62 ms for the 2.0M such tiles of a sparse 4M-point cloud, this
// 0.26 ms.
// ---------------------------------------------------------------------------
// pairwisesum of the first m (1..8) of v
__device__ inline double lane_pairwise(const double (&v)[8], uint32_t m)
{
  const double p01 = v[0] + v[1], p23 = v[2] + v[3], p45 = v[4] + v[5], p67 = v[6] + v[7];
  const double q03 = p01 + p23;
  double acc = 0;
  if (m & 1) acc = acc + (m == 1 ? v[0] : m == 3 ? v[2] : m == 5 ? v[4] : v[6]);
  if (m & 2) acc = acc + (m & 4 ? p45 : p01);
  if (m & 4) acc = acc + q03;
  if (m & 8) acc = acc + (q03 + (p45 + p67));
  return acc;
}

__global__ void __launch_bounds__(64) k_scan_lane(TreeView V, TileGeo g, const int32_t *tex,
                                                  const int32_t *tey, const uint32_t *tile_off,
                                                  const uint32_t *tile_cnt, const uint32_t *lists,
                                                  ClassList cl, double min_hs, TileRec *rec, uint8_t *state,
                                                  unsigned long long *ctr)
{
  const uint32_t n = *cl.n;
  const double r = g.r;
  for (uint32_t i = blockIdx.x * WAVE + threadIdx.x; i < n; i += gridDim.x * WAVE) {
    const uint32_t t = cl.at(i), m = tile_cnt[t], off = tile_off[t];
    uint32_t c[8];
#pragma unroll
    for (int s = 0; s < 8; s++) c[s] = (uint32_t)s < m ? lists[off + s] : 0xffffffffu;
    // canonical order (Batcher's network for eight)
    constexpr int net[19][2] = {{0, 1}, {2, 3}, {4, 5}, {6, 7}, {0, 2}, {1, 3}, {4, 6},
                                {5, 7}, {1, 2}, {5, 6}, {0, 4}, {1, 5}, {2, 6}, {3, 7},
                                {2, 4}, {3, 5}, {1, 2}, {3, 4}, {5, 6}};
#pragma unroll
    for (int k = 0; k < 19; k++) {
      const uint32_t lo = min(c[net[k][0]], c[net[k][1]]), hi = max(c[net[k][0]], c[net[k][1]]);
      c[net[k][0]] = lo;
      c[net[k][1]] = hi;
    }
    double cx, cy, x[8], y[8], z[8], a[8];
    tile_center(g, tex[t], tey[t], &cx, &cy);
#pragma unroll
    for (int s = 0; s < 8; s++) {
      x[s] = y[s] = z[s] = 0;
      if ((uint32_t)s < m) {
        const uint32_t q = V.canon[c[s]];
        x[s] = V.px[q] - cx;
        y[s] = V.py[q] - cy;
        z[s] = V.pz[q] - 0;
      }
    }
    TileFit F;
    F.m = m;
#define WB_SUM(dst, expr)                                     \
  {                                                           \
    _Pragma("unroll") for (int s = 0; s < 8; s++) a[s] = (expr); \
    dst = lane_pairwise(a, m);                                \
  }
    WB_SUM(F.sxx, x[s] * x[s])
    WB_SUM(F.syx, y[s] * x[s])
    WB_SUM(F.syy, y[s] * y[s])
    WB_SUM(F.s1x, 1.0 * x[s])
    WB_SUM(F.s1y, 1.0 * y[s])
    WB_SUM(F.sxz, x[s] * z[s])
    WB_SUM(F.syz, y[s] * z[s])
    WB_SUM(F.s1z, 1.0 * z[s])
#undef WB_SUM
    fit_solve(F);
    F.bottom = __builtin_inf();
    F.top = -__builtin_inf();
#pragma unroll
    for (int s = 0; s < 8; s++) {
      a[s] = z[s] - (F.sy * y[s] + F.sx * x[s]);
      if ((uint32_t)s < m) {
        F.bottom = fmin(F.bottom, a[s]);
        F.top = fmax(F.top, a[s]);
      }
    }
    // the lowest of the points before the first that is at the bottom
    double bottom2 = __builtin_inf();
    bool before = true;
#pragma unroll
    for (int s = 0; s < 8; s++) {
      before = before && (uint32_t)s < m && a[s] != F.bottom;
      if (before) bottom2 = fmin(bottom2, a[s]);
    }
    if (wb::disinf(bottom2)) bottom2 = F.bottom;
    // 7-sector histogram of the bottom layer, four bits a sector
    uint32_t h = 0, inexact = 0;
    F.nbottom = 0;
#pragma unroll
    for (int s = 0; s < 8; s++)
      if ((uint32_t)s < m && a[s] < bottom2 + 2 * r) {
        F.nbottom++;
        const int sec = wb::scan_sector_est(x[s], y[s], r);
        if (sec < 0) inexact |= 1u << s;
        else h += 1u << (4 * sec);
      }
    if (inexact) {
      uint32_t nedge = 0;
      for (int s = 0; s < 8; s++)
        if ((inexact >> s) & 1u) {
          const uint32_t cs = s == 0   ? c[0]
                              : s == 1 ? c[1]
                              : s == 2 ? c[2]
                              : s == 3 ? c[3]
                              : s == 4 ? c[4]
                              : s == 5 ? c[5]
                              : s == 6 ? c[6]
                                       : c[7];
          const uint32_t q = V.canon[cs];
          int edge = 0;
          h += 1u << (4 * wb::scan_sector_exact(V.px[q] - cx, V.py[q] - cy, r, &edge));
          nedge += edge != 0;
        }
      if (nedge) atomicAdd(&ctr[0], (unsigned long long)nedge);
    }
#pragma unroll
    for (int k = 0; k < 7; k++) F.hist[k] = (h >> (4 * k)) & 15u;
    fit_record(F, r, min_hs, 0, rec + t, state + t);
  }
}

// the scan of one tile of up to SCAN_CAP points by one wave (LDS sort)
__device__ void scan_big(const TreeView &T, const TileGeo &g, int ex, int ey, uint32_t off,
                         uint32_t m, const uint32_t *lists, double min_hs, int prec,
                         TileRec *out, uint8_t *state, unsigned long long *ctr, uint32_t *cp,
                         int *histo)
{
  const int lane = threadIdx.x;
  uint32_t P = 1;
  while (P < m) P <<= 1;
  for (uint32_t j = lane; j < P; j += WAVE) cp[j] = j < m ? lists[off + j] : 0xffffffffu;
  if (lane < 7) histo[lane] = 0;
  __syncthreads();
  // canonical order of the tile's points = ascending canonical position
  for (uint32_t k = 2; k <= P; k <<= 1)
    for (uint32_t j = k >> 1; j > 0; j >>= 1) {
      for (uint32_t i = lane; i < P; i += WAVE) {
        uint32_t ixj = i ^ j;
        if (ixj > i) {
          bool up = (i & k) == 0;
          uint32_t a = cp[i], b = cp[ixj];
          if ((a > b) == up) { cp[i] = b; cp[ixj] = a; }
        }
      }
      __syncthreads();
    }
  double cx, cy;
  tile_center(g, ex, ey, &cx, &cy);
  const double r = g.r;
  // the tile's points relative to the cylinder axis, in canonical order
  // (location - xyz(cyl centre, 0)); read through the canonical map
  auto VX = [&](uint32_t j) { return T.px[T.canon[cp[j]]] - cx; };
  auto VY = [&](uint32_t j) { return T.py[T.canon[cp[j]]] - cy; };
  auto VZ = [&](uint32_t j) { return T.pz[T.canon[cp[j]]] - 0; };
  // normal equations of [x y 1] z (transmult and operator*, matrix.cpp:181-215)
  double sxx = wave_pairwise(m, [&](uint32_t j) { double v = VX(j); return v * v; });
  double syx = wave_pairwise(m, [&](uint32_t j) { return VY(j) * VX(j); });
  double syy = wave_pairwise(m, [&](uint32_t j) { double v = VY(j); return v * v; });
  double s1x = wave_pairwise(m, [&](uint32_t j) { return 1.0 * VX(j); });
  double s1y = wave_pairwise(m, [&](uint32_t j) { return 1.0 * VY(j); });
  double s11 = wave_pairwise(m, [&](uint32_t j) { (void)j; return 1.0 * 1.0; });
  double sxz = wave_pairwise(m, [&](uint32_t j) { return VX(j) * VZ(j); });
  double syz = wave_pairwise(m, [&](uint32_t j) { return VY(j) * VZ(j); });
  double s1z = wave_pairwise(m, [&](uint32_t j) { return 1.0 * VZ(j); });
  double sx, sy;
  plane_tilt(sxx, syx, syy, s1x, s1y, s11, sxz, syz, s1z, &sx, &sy);
  // untilted height; bottom, bottom2 (the running minimum before its last
  // update), top
  auto U = [&](uint32_t j) { return VZ(j) - (sy * VY(j) + sx * VX(j)); };
  double bottom = __builtin_inf(), top = -__builtin_inf();
  for (uint32_t j = lane; j < m; j += WAVE) {
    double u = U(j);
    bottom = fmin(bottom, u);
    top = fmax(top, u);
  }
  for (int s = 1; s < WAVE; s <<= 1) {
    bottom = fmin(bottom, __shfl_xor(bottom, s, WAVE));
    top = fmax(top, __shfl_xor(top, s, WAVE));
  }
  uint32_t first = 0xffffffffu;
  for (uint32_t j = lane; j < m; j += WAVE)
    if (U(j) == bottom && j < first) first = j;
  for (int s = 1; s < WAVE; s <<= 1) first = min(first, (uint32_t)__shfl_xor((int)first, s, WAVE));
  double bottom2 = __builtin_inf();
  for (uint32_t j = lane; j < first; j += WAVE) bottom2 = fmin(bottom2, U(j));
  for (int s = 1; s < WAVE; s <<= 1) bottom2 = fmin(bottom2, __shfl_xor(bottom2, s, WAVE));
  if (wb::disinf(bottom2)) bottom2 = bottom;
  // 7-sector histogram of the bottom layer
  uint32_t nbottom = 0;
  for (uint32_t j = lane; j < m; j += WAVE) {
    if (!(U(j) < bottom2 + 2 * r)) continue;
    nbottom++;
    const double vx = VX(j), vy = VY(j);
    int edge = 0;
    const int sec = wb::scan_sector(vx, vy, r, &edge);
    if (edge) atomicAdd(&ctr[0], 1ull);
    atomicAdd(&histo[sec], 1);
  }
  for (int s = 1; s < WAVE; s <<= 1) nbottom += __shfl_xor((int)nbottom, s, WAVE);
  __syncthreads();
  if (lane == 0) {
    double density = 0;
    int tree = 0;
    for (int i = 0; i < 7; i++) density += histo[i] * histo[i];
    if (m > nbottom && density < 7) tree = 1;
    density = sqrt(density) * kSqrt7 / (r * r) / M_PI;
    if (m > nbottom && density < 0.5) tree = 1;
    if (top - bottom > 1.5) tree = 1;
    TileRec rr;
    rr.npoints = (int32_t)m;
    rr.nground = 0;
    rr.tree_flags = tree;
    rr.fit_fp64 = prec != WB_FIT_FP64;  // tiles of this size always fit in FP64
    rr.density = density;
    rr.hs_scan = sqrt(1 / density + min_hs * min_hs);
    rr.hs = rr.hs_scan;
    rr.height = top - bottom;
    rr.tilt_x = sx;
    rr.tilt_y = sy;
    *out = rr;
    *state = (uint8_t)(1 + tree);
    if (prec != WB_FIT_FP64) atomicAdd(&ctr[7], 1ull);
  }
  __syncthreads();
}

// Tiles of more than 256 points: the canonical sort in LDS and every value
// read through the canonical map.
__global__ void __launch_bounds__(64) k_scan(TreeView T, TileGeo g, const int32_t *tex,
                                             const int32_t *tey, const uint32_t *tile_off,
                                             const uint32_t *tile_cnt, const uint32_t *lists,
                                             ClassList cl, double min_hs, int prec, TileRec *rec,
                                             uint8_t *state, uint32_t *err,
                                             unsigned long long *ctr)
{
  __shared__ uint32_t cp[SCAN_CAP];
  __shared__ int histo[7];
  const uint32_t n = *cl.n;
  for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
    const uint32_t t = cl.at(i);
    const uint32_t m = tile_cnt[t];
    if (m > SCAN_CAP) {
      if (threadIdx.x == 0) atomicOr(err, 2u);
      continue;
    }
    scan_big(T, g, tex[t], tey[t], tile_off[t], m, lists, min_hs, prec, rec + t, state + t,
             ctr, cp, histo);
  }
}

// POSTSCAN (scan.cpp:142-179): tree tiles widen their hyperboloid by the
// number of tree tiles met along six rays before an empty ring or a
// non-tree tile.
__global__ void k_postscan(TileGeo g, const int32_t *tex, const int32_t *tey,
                           const uint8_t *state, TileRec *rec, int32_t *nground,
                           unsigned long long *nonempty)
{
  // the non-empty tiles counted per block (one atomic on the counter per
  // block: atomics on one address are serialised)
  __shared__ uint32_t bcount;
  if (threadIdx.x == 0) bcount = 0;
  __syncthreads();
  uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < g.ntiles) nground[t] = 0;
  const uint8_t mine = t < g.ntiles ? state[t] : 0;
  const bool live = mine != 0;
  const uint64_t lv = __ballot(live);
  if (__lane_id() == 0 && lv) atomicAdd(&bcount, (uint32_t)__popcll(lv));
  __syncthreads();
  if (threadIdx.x == 0 && bcount) atomicAdd(nonempty, (unsigned long long)bcount);
  if (!live) return;
  const double hs_scan = rec[t].hs_scan;
  const int r1x[6] = {1, 1, 0, -1, -1, 0}, r1y[6] = {0, 1, 1, 0, -1, -1};  // root1, eisenstein.cpp:51
  int i = 1, ring, nontree, count = 0;
  if (mine == 2) {
    // a ring's six tiles are read together, each by its place and its state:
    // the longest chain of rings is the kernel (18.5k points 22 us with the
    // count and the record read tile by tile, 10 so; 1.17M 41 and 22)
    const int ex = tex[t], ey = tey[t];
    do {
      ring = nontree = 0;
      int o[6];
      uint8_t q[6];
#pragma unroll
      for (int j = 0; j < 6; j++) {
        int cnt;
        o[j] = tile_at(g, ex + r1x[j] * i, ey + r1y[j] * i, &cnt) ? cnt - g.lo : -1;
      }
#pragma unroll
      for (int j = 0; j < 6; j++) q[j] = o[j] >= 0 ? state[o[j]] : 0;
#pragma unroll
      for (int j = 0; j < 6; j++) {
        ring += q[j] != 0;
        count += q[j] == 2;
        nontree += q[j] == 1;
      }
      ++i;
    } while (ring && !nontree);
  }
  double w = count * g.spacing / 6;
  rec[t].hs = sqrt(hs_scan * hs_scan + w * w);
}

// The tiles' records in the caller's layout, empty tiles zero but for their
// address; a block's 256 records pass through LDS and leave in whole lines.
__global__ void __launch_bounds__(256) k_tile_out(uint32_t ntiles, const uint32_t *tile_cnt,
                                                  const TileRec *rec, const int32_t *tex,
                                                  const int32_t *tey, const int32_t *nground,
                                                  wb_tile *out)
{
  constexpr uint32_t W = sizeof(wb_tile) / 4;
  __shared__ __align__(16) wb_tile s[256];
  const uint32_t t0 = blockIdx.x * 256, t = t0 + threadIdx.x;
  if (t < ntiles) {
    wb_tile o = {};
    o.flowsnake_x = tex[t];
    o.flowsnake_y = tey[t];
    if (tile_cnt[t]) {
      const TileRec r = rec[t];
      o.npoints = r.npoints;
      o.nground = nground ? nground[t] : r.nground;
      o.tree_flags = r.tree_flags;
      o.fit_fp64 = r.fit_fp64;
      o.density = r.density;
      o.hs_scan = r.hs_scan;
      o.hs = r.hs;
      o.height = r.height;
      o.tilt_x = r.tilt_x;
      o.tilt_y = r.tilt_y;
    }
    s[threadIdx.x] = o;
  }
  __syncthreads();
  const uint32_t n = min(256u, ntiles - t0) * W;
  const uint32_t *src = (const uint32_t *)s;
  uint32_t *dst = (uint32_t *)(out + t0);
  for (uint32_t k = threadIdx.x; k < n; k += 256) dst[k] = src[k];
}

// ---------------------------------------------------------------------------
// CLASSIFY
// ---------------------------------------------------------------------------
// a point handed to the wave-per-point kernel, with the directions found
// so far and the walk it continues with
struct HeavyRec {
  uint64_t occ;
  uint32_t i;
  uint32_t start;  // walk to start from: 0 A, 1 B, 2 the exact border pass
};

struct ClassifyArgs {
  TreeView T;
  TileGeo g;
  const int32_t *memb;
  const uint32_t *nmemb;
  const TileRec *rec;
  double thickness, max_slope;
  // 1: every point lies in its leaf's cube, so the care wedges may skip a
  // node or leaf by its cube and a child cube's bottom face may be raised to
  // the lowest point stored under it; 0 (a point outside the root cube):
  // only the 32-point groups' boxes, which bound the points themselves, are
  // tested
  int cube_wedges;
  const double *tab;     // tan[511], cos[512], sin[512] packed
  const float *edges;    // bin-edge directions (wb::fill_edge_table)
  wb::AtanConst K;
  uint8_t *cls;          // per sorted slot
  uint8_t *cls_in;       // per input index (the caller's class bytes)
  uint32_t *nslow;       // points decided by the exact gap pass
  HeavyRec *heavy;       // points handed to the wave-per-point kernel
  uint32_t *nheavy, *heavy_next;
  unsigned long long *atan_exact;
  // What walk A leaves to walk B: per wave with open lanes units of up to
  // open_per of them: the place in pool (and upper 16 bits of y) and length
  // of its leaf list, its records and the first one.  Records lie at the
  // wave's own place; a list of up to OPEN_LIST leaves does too, a longer one
  // past pool_shared (npool: entries taken).
  // open_classes: the units of class k lie from unit_cap * k on (nopen: of
  // each class; open_next: units the resident kernel has taken); else unit w is wave w's, with no
  // records when it left no lane open.
  HeavyRec *open;
  uint4 *open_unit;
  uint32_t *pool;
  uint64_t pool_shared, pool_cap;
  uint32_t unit_cap, open_per;
  uint32_t walk_per;  // points of a wave of walk A (at least open_per)
  uint32_t leaf_cap;  // leaves a wave of walk A lists at most
  int open_budget;  // groups and rounds of candidates a unit of walk B takes at most
  int open_classes;
  uint32_t *nopen, *open_next;
  unsigned long long *npool;
  // work items in place of the points (nullptr: work index k is sorted slot
  // k with the hyperboloid size of its deciding tile): item k is (slot,
  // tile record index), and its verdict goes to item_cls[k] only
  const uint2 *items;
  uint64_t n_items;
  uint8_t *item_cls;
};

// the slot and hyperboloid size of work index k; false for a point in no tile
__device__ inline bool work_point(const ClassifyArgs &A, uint64_t k, uint32_t &slot, double &hs)
{
  if (A.items) {
    const uint2 it = A.items[k];
    slot = it.x;
    hs = A.rec[it.y].hs;
    return true;
  }
  slot = (uint32_t)k;
  if (A.nmemb[k] == 0) return false;
  int w = INT32_MIN;
  for (uint32_t j = 0; j < A.nmemb[k]; j++) w = max(w, A.memb[MAX_MEMB * k + j]);
  hs = A.rec[w - A.g.lo].hs;
  return true;
}

// the verdict of work index k: the class byte of the point (per sorted slot
// and at its input index), or of the work item
__device__ inline void work_verdict(const ClassifyArgs &A, uint64_t k, uint32_t slot, uint8_t v)
{
  if (A.items) {
    A.item_cls[k] = v;
    return;
  }
  A.cls[k] = v;
  A.cls_in[A.T.sidx[slot]] = v;
}

__device__ inline uint64_t rotr64(uint64_t x, int a) { return (x >> a) | (x << (64 - a)); }

// classification of the empty-bin mask: 1 pass, 2 fail, 0 undecided
__device__ inline int gap_verdict(uint64_t occupied)
{
  uint64_t e = ~occupied;
  uint64_t r2 = e & rotr64(e, 1);
  uint64_t r4 = r2 & rotr64(r2, 2);
  uint64_t r8 = r4 & rotr64(r4, 4);
  uint64_t r16 = r8 & rotr64(r8, 8);
  uint64_t r24 = r16 & rotr64(r8, 16);
  if (r24 == 0) return 1;
  uint64_t r26 = r24 & rotr64(e, 24) & rotr64(e, 25);
  if (r26 != 0) return 2;
  return 0;
}

__device__ inline int dir_bin_pos(int a) { return (int)(((uint32_t)a + 0x40000000u) & 0x7fffffffu); }

// OR over the 64 lanes by DPP row operations: lanes of a row swap within
// quads, then rotate by 4 and 8, so every lane holds its row's OR; the two
// row broadcasts fold row r-1 into row r and row 1 into rows 2 and 3, so
// lane 63 holds the OR of all lanes.  Lanes a broadcast does not write add 0.
template <int CTRL, int ROWS>
__device__ inline uint32_t dpp_or(uint32_t v)
{
  return v | (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
__device__ inline uint32_t wave_or32(uint32_t v)
{
  v = dpp_or<0xb1, 0xf>(v);   // quad_perm 1,0,3,2
  v = dpp_or<0x4e, 0xf>(v);   // quad_perm 2,3,0,1
  v = dpp_or<0x124, 0xf>(v);  // row_ror 4
  v = dpp_or<0x128, 0xf>(v);  // row_ror 8
  v = dpp_or<0x142, 0xa>(v);  // row_bcast 15 into rows 1 and 3
  v = dpp_or<0x143, 0xc>(v);  // row_bcast 31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ inline uint64_t wave_or(uint64_t v)
{
  return ((uint64_t)wave_or32((uint32_t)(v >> 32)) << 32) | wave_or32((uint32_t)v);
}

// ---------------------------------------------------------------------------
// Ground-test walk: findBlocks (octree.cpp:234-251) for 64 hyperboloids at
// once, with an explicit stack.  The 64 lanes of a wave hold 64 consecutive
// points of the sorted order (spatial neighbours), each with its own
// hyperboloid.  A stack entry is a node or leaf code and the mask of lanes
// for which it and every ancestor intersect the lane's hyperboloid, so each
// lane sees exactly the leaves findBlocks returns for its own shape.
// Expanding a node tests its eight children at once; their cubes follow from
// the parent's by Octree::cube (octree.cpp:349-358), the operations the
// build used, so no child cube is loaded.
// Visiting order: the children of a node are taken starting with the xy
// quadrant that holds the wave's first point, then its x, y and diagonal
// neighbours, the lower half (where a downward hyperboloid lies) first.
// Leaves near the point in every direction come early, which lets the early
// exit of the ground test come early.  The order changes no result: a pass
// on a subset of D is a pass on D, and a fail or an exact gap needs all of D.
// ---------------------------------------------------------------------------
// Entries pending at one time: at most 7 siblings per level on the path
// (internal nodes sit at levels 0..WB_MAX_LEVEL) plus 8 children.  All
// entries of one level are children of one node (a node is expanded when it
// is popped, and its children are taken before its siblings), so the lanes
// that reach them are kept per level.
#define WB_STK (7 * (WB_MAX_LEVEL + 1) + 8 + 2)
// leaves walk A takes at most before it hands its open lanes to
// k_ground_heavy (ClassifyArgs::leaf_cap is the number), or, of all entries it
// takes from its stack
#define GROUND_LEAVES 256
#define GROUND_STEPS 1024
struct WaveStack {
  // x: node or leaf code; y: level, and the point count of a leaf << 8; z: a
  // leaf's first slot; w: (float) at most the lowest z stored under the entry
  uint4 ent[WB_STK];
  uint2 mask[WB_MAX_LEVEL + 2];  // lanes whose walk reached the parent
  uint32_t leaf[GROUND_LEAVES];  // the leaves walk A took, in its order
};

// A value every lane of the wave reads from the same address, fetched by the
// scalar unit into scalar registers (i wave-uniform; nothing writes the
// tree's arrays while a ground kernel runs).
__device__ inline double uload(const double *p, size_t i)
{
  return ((const __attribute__((address_space(4))) double *)p)[i];
}

// a value every lane reads from the same address, as uload
__device__ inline float uloadf(const float *p, size_t i)
{
  return ((const __attribute__((address_space(4))) float *)p)[i];
}
__device__ inline uint32_t uloadu(const uint32_t *p, size_t i)
{
  return ((const __attribute__((address_space(4))) uint32_t *)p)[i];
}

// A lane's hyperboloid as hyp_near reads it
struct Near {
  double x, y, cz, por2, thr;  // thr = por2 * wb::kNearShrink
};

__device__ inline double near_t(const Near &P, double s2, double qx, double qy, double qz)
{
  return wb::hyp_near(s2, qx - P.x, qy - P.y, P.cz - qz);
}

// What holds every hyperboloid of the wave's open lanes: the box of their
// axes, the highest centre and the lowest threshold (wave-uniform).  A box
// that fails union_hits meets none of them: its distance from the axes' box
// is at most its distance from any lane's axis (each difference rounds
// monotonically), so near_t's bound holds for the union too.
struct Union {
  double x0, x1, y0, y1, cz, thr;
};

__device__ inline Union wave_union(const Near &P, bool open)
{
  const double inf = __builtin_inf();
  Union U;
  U.x0 = wave_dmin(open ? P.x : inf);
  U.x1 = wave_dmax(open ? P.x : -inf);
  U.y0 = wave_dmin(open ? P.y : inf);
  U.y1 = wave_dmax(open ? P.y : -inf);
  U.cz = wave_dmax(open ? P.cz : -inf);
  U.thr = wave_dmin(open ? P.thr : inf);
  return U;
}

__device__ inline bool union_hits(const Union &U, double s2, double x0, double x1, double y0,
                                  double y1, double z0)
{
  const double dx = fmax(fmax(x0 - U.x1, U.x0 - x1), 0.0);
  const double dy = fmax(fmax(y0 - U.y1, U.y0 - y1), 0.0);
  const double dz = U.cz - z0;
  return wb::hyp_near(s2, dx, dy, dz) >= U.thr;
}

// bit k of the result is bit k ^ r of the 8-bit mask m (r < 8)
__device__ inline uint32_t xor_bits8(uint32_t m, int r)
{
  if (r & 1) m = ((m & 0x55) << 1) | ((m >> 1) & 0x55);
  if (r & 2) m = ((m & 0x33) << 2) | ((m >> 2) & 0x33);
  if (r & 4) m = ((m & 0x0f) << 4) | (m >> 4);
  return m;
}

// visiting order: child k has rank k ^ o (o: the xy quadrant taken first; the
// lower half, bit 2 clear, comes first, since the hyperboloids open downwards)
__device__ inline int child_rank(int k, int o) { return k ^ o; }

// Pushes the children of node `code` (cube cx, cy, cz, side at level lvl)
// that may meet the hyperboloid of an open lane, in reverse visiting order:
// lane k < 8 tests child k (its cube by Octree::cube, octree.cpp:349-358,
// the operations of the build; its bottom face raised to the lowest point
// stored under it when every point lies in its leaf's cube) against the
// wave's union.  The lanes' own tests follow when a child is popped.
// Returns the new stack depth.
template <bool IN>
__device__ inline int push_children(const TreeView &T, WaveStack &S, int sp, int code, int lvl,
                                    double cx, double cy, double cz, double side, uint64_t mk,
                                    const Union &U, double s2, double rx, double ry)
{
  const uint32_t lane = __lane_id();
  const int o = rfl((rx >= cx ? 1 : 0) | (ry >= cy ? 2 : 0));
  int ck = -1;
  uint2 cr = make_uint2(0u, 0u);
  double zl = -__builtin_inf();
  if (lane < 8) {
    const size_t at = 8 * (size_t)code + lane;
    ck = T.node_child[at];
    cr = T.node_crange[at];
    if (IN) zl = T.child_zlow[at];
  }
  const double h = side / 4;
  const double x = cx + ((lane & 1) ? h : -h), y = cy + ((lane & 2) ? h : -h);
  const double z = cz + ((lane & 4) ? h : -h);
  const bool hit = ck != -1 && union_hits(U, s2, x - h, x + h, y - h, y + h, fmax(z - h, zl));
  const uint32_t pm = (uint32_t)__ballot(hit);
  if (hit) {
    const uint32_t above = xor_bits8(pm, o) >> (((int)lane ^ o) + 1);  // taken after this one
    S.ent[sp + __popc(above)] =
        make_uint4((uint32_t)ck, (uint32_t)(lvl + 1) | ((cr.y - cr.x) << 8), cr.x,
                   __float_as_uint((float)(zl - __builtin_fabs(zl) * 0x1p-22)));
  }
  S.mask[lvl + 1] = make_uint2((uint32_t)mk, (uint32_t)(mk >> 32));
  return sp + __popc(pm);
}

// classes of walk B's units by the length of their leaf lists
#define OPEN_CLASSES 4
// leaf list entries kept at a wave's own place
#define OPEN_LIST 64
#ifndef OPEN_P1
#define OPEN_P1 16
#endif
#ifndef OPEN_P2
#define OPEN_P2 32
#endif
// candidates of one 32-point group from which on a lane's care wedges are
// taken anew before the next group
#ifndef OPEN_REFRESH
#define OPEN_REFRESH 4
#endif
// lanes that need a 32-point group up to which it is tested two lanes at a
// time, half a wave of slots each
#ifndef OPEN_PAIR
#define OPEN_PAIR 12
#endif
// a lane whose walk A entered leaves with more groups than this is finished
// by k_ground_heavy, a wave to the point
#define HEAVY_B_GROUPS 1024u
// blocks of the heavy kernel at most: 4 waves on each SIMD of 256 CUs
#define HEAVY_GRID 4096u

// the lanes' hyperboloids: Hyperboloid(p - (0,0,thickness), hs, slope)
// (shape.cpp:119-125) with its axis at x, y instead of x + 0, y + 0: the two
// differ only in the sign of a zero, which no test can see (every use is a
// difference that is squared, compared or passed to hypot)
__device__ inline Near make_near(const ClassifyArgs &A, double x, double y, double z, double hs)
{
  const double sl = A.max_slope, por = hs * (sl * sl);
  Near P;
  P.x = x;
  P.y = y;
  P.cz = (z - A.thickness) + por;
  P.por2 = por * por;
  P.thr = P.por2 * wb::kNearShrink;
  return P;
}

// A point this far inside (near_t less 2^-39 of a reaches por2 + sure_slack)
// is in, and findBlocks reaches its leaf, whatever the roundings: a cube that
// holds the point lies no farther from the axis than the point but for the
// rounding of clamp_axis's difference (2^-53 of the root's side), and 2^-39
// of a covers those of the products.
__device__ inline double sure_slack(const ClassifyArgs &A)
{
  const double d = A.max_slope * (A.T.side * 0x1p-52);
  return 2 * d * d;
}

__device__ __forceinline__ void ground_setup(const ClassifyArgs &A, float *edges)
{
  for (int k = threadIdx.x; k < 3 * 128; k += blockDim.x) edges[k] = A.edges[k];
  __syncthreads();
}

// Walk A for 64 points, one per lane: the lowest point of each 32-point group
// of every leaf findBlocks returns (a subset of D, so only a pass is decided
// here).  The lanes left open go to walk B (k_ground_open) in units of
// at most 64 with the directions found and the list of the leaves taken here,
// which holds every leaf B needs: what A left out by a hyperboloid or by care
// wedges (which only shrink) no open lane needs.  A wave that fills its list
// and a lane with many groups go to k_ground_heavy.
//
// What bounds it: VALU issue (the tests of boxes and samples), and the wait
// for a popped cube.  So a node's children are tested by eight lanes at once
// against the wave's union instead of by every lane in turn, the lanes' own
// test of a cube is the eight-operation near_t, and walk B, whose work per
// point varies most, is a kernel of its own.
// IN: every point lies in its leaf's cube (the build flags the other case),
// so the care wedges may skip a node or leaf by its cube and a cube's bottom
// face may be raised to the lowest point stored under it.
template <bool IN>
__device__ __forceinline__ void walk_body(const ClassifyArgs &A, uint64_t unit, WaveStack &S,
                                          const float *edges)
{
  const TreeView &T = A.T;
  const uint32_t lane = __lane_id();
  // work index: a sorted slot, or a work item
  const uint64_t i = unit * A.walk_per + lane;
  const bool inrange = lane < A.walk_per && i < (A.items ? A.n_items : T.n);
  // lane state: 0 undecided, 1 not ground, 3 no tile; handed on: 5 to the
  // heavy kernel, walk A cut short
  int state = 3;
  double x = 0, y = 0, z = 0, hs = 0;
  uint32_t slot = 0;
  if (inrange && work_point(A, i, slot, hs)) {
    x = T.px[slot]; y = T.py[slot]; z = T.pz[slot];
    state = 0;
  }
  const double sl = A.max_slope, s2 = (sl * sl) * wb::kNearShrink;
  const Near P = make_near(A, x, y, z, hs);
  // a subset of D will do here, so a sample that rounding might put either
  // side of the surface, or of a bin's edge, is left to walk B
  const double sure = P.por2 + sure_slack(A);
  wb::LaneWedges W;
  W.n = -1;
  uint64_t occ = 0, checked = 0;
  uint32_t groups_a = 0, nleaf = 0;
  uint64_t alive = __ballot(state == 0);
  if (alive) {
    Union U = wave_union(P, state == 0);
    int ualive = __popcll(alive);
    // the wave's first point orders the children
    const int ld = __ffsll((long long)alive) - 1;
    const double rx = rdl(x, ld), ry = rdl(y, ld);
    int sp = 1;
    S.ent[0] = make_uint4(0u, 0u, 0u, __float_as_uint(-__builtin_inff()));
    S.mask[0] = make_uint2((uint32_t)alive, (uint32_t)(alive >> 32));
    for (uint32_t steps = 0; sp > 0; steps++) {
      if (steps == GROUND_STEPS) {
        if (state == 0) state = 5;
        break;
      }
      const uint4 en = S.ent[--sp];
      const int code = rfl((int)en.x), lvl = rfl((int)(en.y & 255u));
      const uint2 mw = S.mask[lvl];
      uint64_t m = (((uint64_t)(uint32_t)rfl((int)mw.y) << 32) | (uint32_t)rfl((int)mw.x)) & alive;
      if (m == 0) continue;
      const double *cb = code >= 0 ? T.node_cube + 4 * (size_t)code
                                   : T.leaf_cube + 4 * (size_t)(-2 - code);
      const double cx = uload(cb, 0), cy = uload(cb, 1), cz = uload(cb, 2), side = uload(cb, 3);
      // the lanes' own tests: whether the cube, its bottom face raised, may
      // meet the lane's hyperboloid and care wedges
      bool on = (m >> lane) & 1;
      // a leaf whose points lie in its cube, also where not every leaf's do
      const bool lin = IN || (code < 0 && leaf_inside(T, (uint32_t)(-2 - code)));
      const bool anyw = lin && __ballot(on && W.n >= 0) != 0;
      const double hh = side / 2, x0 = cx - hh, x1 = cx + hh, y0 = cy - hh, y1 = cy + hh;
      if (!lin) {
        // a point may lie outside its leaf's cube, so reaching the leaf does
        // not follow from the point: findBlocks' own test, cube by cube
        wb::Shape H = wb::make_cylinder(x, y, 0);
        H.kind = wb::SHAPE_HYPERBOLOID;
        H.cz = P.cz;
        H.por2 = P.por2;
        H.slope = sl;
        on = on && wb::hyp_intersect(H, cx, cy, cz, side);
        m = __ballot(on);
      } else if (code < 0 || anyw) {
        const double zb = fmax(cz - hh, IN ? (double)__uint_as_float((uint32_t)rfl((int)en.w))
                                           : (double)uloadf(T.leaf_low, (uint32_t)(-2 - code)));
        on = on && near_t(P, s2, fmin(fmax(x, x0), x1), fmin(fmax(y, y0), y1), zb) >= P.thr;
        if (anyw) on = on && wb::lane_hit(W, x, y, x0, x1, y0, y1);
        m = __ballot(on);
      }
      if (m == 0) continue;
      if (code >= 0) {
        sp = push_children<IN>(T, S, sp, code, lvl, cx, cy, cz, side, m, U, s2, rx, ry);
        continue;
      }
      if (nleaf == A.leaf_cap) {
        if (state == 0) state = 5;
        break;
      }
      const uint32_t b = (uint32_t)rfl((int)en.z), e = b + ((uint32_t)rfl((int)en.y) >> 8);
      S.leaf[nleaf++] = (uint32_t)(-2 - code);
      // the lowest point of each group (the likeliest to lie in a downward
      // hyperboloid), or the group's first slot in the leaf when the lowest
      // one belongs to the neighbouring leaf: lane g fetches the sample of
      // group g and tests it against the wave's union, and the samples that
      // pass are tested by every lane
      const uint32_t g0 = b / WB_CHUNK, ng = (e - 1) / WB_CHUNK - g0 + 1;
      if (on) groups_a += ng;
      for (uint32_t gb = 0; gb < ng; gb += WAVE) {
        const uint32_t g = gb + lane;
        double sx = 0, sy = 0, sz = 0;
        if (g < ng) {
          // the group's lowest point from the per-group copy (consecutive
          // lanes, consecutive words)
          const uint32_t j = T.chunk_low[g0 + g];
          if (j < b || j >= e) {
            const uint32_t jf = g == 0 ? b : (g0 + g) * WB_CHUNK;
            sx = T.px[jf]; sy = T.py[jf]; sz = T.pz[jf];
          } else {
            sx = T.chunk_sx[g0 + g]; sy = T.chunk_sy[g0 + g]; sz = T.chunk_sz[g0 + g];
          }
        }
        uint64_t todo = __ballot(g < ng && union_hits(U, s2, sx, sx, sy, sy, sz));
        while (todo) {
          const uint32_t s = (uint32_t)__ffsll((long long)todo) - 1;
          todo &= todo - 1;
          const double qx = rdl(sx, s), qy = rdl(sy, s), qz = rdl(sz, s);
          const double dx = qx - x, dy = qy - y, dz = P.cz - qz;
          const double t = wb::hyp_near(s2, dx, dy, dz), a = dz * __builtin_fabs(dz);
          const bool in = on & ((qx != x) | (qy != y)) & (__builtin_fma(-0x1p-39, a, t) >= sure);
          if (!__ballot(in)) continue;
          bool ok;
          const int bin = wb::dir_bin_est(dy, dx, &ok);
          if (in & ok) occ |= 1ull << bin;
        }
      }
      if (state == 0 && occ != checked) {
        checked = occ;
        if (gap_verdict(occ) == 1) state = 1;
        else wb::lane_wedges_update(occ, edges, W, 1);
      }
      alive = __ballot(state == 0);
      if (alive == 0) break;
      // the union shrinks with the open lanes: taken again once a quarter of
      // them are decided
      const int na = __popcll(alive);
      if (4 * na <= 3 * ualive) {
        U = wave_union(P, state == 0);
        ualive = na;
      }
    }
  }
  if (state == 0 && groups_a > HEAVY_B_GROUPS) state = 6;
  // hand the open lanes over, with the directions found so far
  const uint64_t hb = __ballot(state >= 5), ob = __ballot(state == 0);
  const uint64_t lt = (1ull << lane) - 1;
  if (!ob && !A.open_classes && lane == 0) A.open_unit[unit] = make_uint4(0u, 0u, 0u, 0u);
  if (hb | ob) {
    // where units are few, those with the longest leaf lists come first
    // (class 0), so that the longest ones don't start last
    const uint32_t no = (uint32_t)__popcll(ob), wave = (uint32_t)unit;
    const uint32_t cls = nleaf >= 64 ? 0 : nleaf >= 32 ? 1 : nleaf >= 16 ? 2 : 3;
    const uint32_t per = A.open_per, nu = (no + per - 1) / per;
    uint32_t hbase = 0, uat = wave;
    uint64_t pbase = (uint64_t)wave * OPEN_LIST;
    if (lane == 0) {
      if (hb) hbase = atomicAdd(A.nheavy, (uint32_t)__popcll(hb));
      if (ob && A.open_classes) uat = atomicAdd(A.nopen + cls, nu) + cls * A.unit_cap;
      // a longer list takes its place from the pool's shared end
      if (ob && nleaf > OPEN_LIST) pbase = A.pool_shared + atomicAdd(A.npool, (unsigned long long)nleaf);
    }
    hbase = (uint32_t)rfl((int)hbase);
    uat = (uint32_t)rfl((int)uat);
    pbase = rdl64(pbase, 0);
    HeavyRec r;
    r.occ = occ;
    r.i = (uint32_t)i;
    r.start = 0;
    if (state >= 5) {
      r.start = (uint32_t)(state - 5);
      A.heavy[hbase + __popcll(hb & lt)] = r;
    }
    if (ob) {
      const uint32_t rec = wave * WAVE + lane * per;
      uint4 desc = make_uint4((uint32_t)pbase, nleaf | (uint32_t)(pbase >> 32) << 16,
                              min(per, no - min(no, lane * per)), rec);
      if (pbase + nleaf > A.pool_cap) {
        // the shared end is full: the wave-per-point kernel takes the lanes
        if (lane == 0) hbase = atomicAdd(A.nheavy, no);
        hbase = (uint32_t)rfl((int)hbase);
        r.start = 1;
        if (state == 0) A.heavy[hbase + __popcll(ob & lt)] = r;
        desc = make_uint4(0u, 0u, 0u, 0u);
      } else {
        for (uint32_t k = lane; k < nleaf; k += WAVE) A.pool[pbase + k] = S.leaf[k];
        if (state == 0) A.open[(size_t)wave * WAVE + __popcll(ob & lt)] = r;
      }
      if (lane < nu) A.open_unit[uat + lane] = desc;
    }
  }
  if (inrange && (state == 1 || state == 3)) work_verdict(A, i, slot, state == 1 ? 1 : 0);
}

// Walk B for a unit of up to 64 points, a lane each: every point of D that
// can change the verdict, from the leaves walk A listed.  64 leaves at a time
// are tested against the unit's union, a lane each; in a leaf that passes,
// its octets (8 slots), a lane each; then every lane tests the 32-point group
// of an octet that passed (its box against the lane's hyperboloid and care
// wedges), the octet's box, and the octet's points one after the other, a
// point in scalar registers, into a mask of its candidates; last each lane
// takes its own candidates, so lanes with different ones work together.
// A point left with a longest empty run of 24 or 25 bins takes the leaves
// once more (GAP) for the exact extreme directions in the two bins bordering
// the run.  A point that meets a neighbour so near its surface that rounding
// decides goes to the heavy kernel, which tests as the reference does.
// What bounds it: VALU issue (the points' tests, 45k instructions per unit of
// the 23.7M-point tile with all outliers above the surface).  Walks A and B
// and the gap pass in one kernel, with every lane testing every child, sample
// and box by hyp_in and the gap pass left to the heavy kernel, took 41.5 and
// 12.7 ms on that tile against 9 + 19 and 0.3 ms now, 4.9 and 0.32 against
// 4.3 and 0.08 ms on the one with low outliers, 2.7 and 0.67 against 2.0 and
// 0.08 ms on 1.17M points, 0.46 and 0.04 against 0.25 and 0.01 ms on 18.5k.
struct OpenPoint {
  int state;  // 0 undecided, 1 not ground, 2 ground, 3 none, 4 the exact gap
              // decides; to the heavy kernel: 6 walk B, 7 the exact gap
  uint64_t occ;
  wb::LaneWedges W;
  // of the gap pass: the bins bordering the runs (8 bits each: before and
  // after the first, the second), the largest position in a bin before a run
  // and the smallest in a bin after it
  uint32_t border;
  int hi[2], lo[2];
};

// CAP: a long unit's open lanes go to the heavy kernel (A.open_budget).
template <bool IN, bool GAP, bool CAP>
__device__ __forceinline__ void open_pass(const ClassifyArgs &A, const uint32_t *pool, uint32_t nleaf,
                                          const Near &P, OpenPoint &O, const float *edges,
                                          double2 *edge, int &nexact)
{
  const TreeView &T = A.T;
  const uint32_t lane = __lane_id();
  const double sl = A.max_slope, s2 = (sl * sl) * wb::kNearShrink, x = P.x, y = P.y;
  const double slack = sure_slack(A);
  const int want = GAP ? 4 : 0;
  bool pend = false;
  uint32_t work = 0;  // groups, and rounds of candidates
  uint64_t checked = O.occ;
  uint64_t alive = __ballot(O.state == want);
  if (alive == 0) return;
  Union U = wave_union(P, O.state == want);
  int ualive = __popcll(alive);
  for (uint32_t lb = 0; lb < nleaf && alive; lb += WAVE) {
    uint32_t leaf_l = 0;
    bool lh = lb + lane < nleaf;
    if (lh) {
      leaf_l = pool[lb + lane];
      const double *c = T.leaf_cube + 4 * (size_t)leaf_l;
      const double h = c[3] / 2;
      lh = union_hits(U, s2, c[0] - h, c[0] + h, c[1] - h, c[1] + h,
                      IN || leaf_inside(T, leaf_l) ? fmax(c[2] - h, (double)T.leaf_low[leaf_l])
                                                : c[2] - h);
    }
    uint64_t ltodo = __ballot(lh);
    while (ltodo) {
      const uint32_t ls = (uint32_t)__ffsll((long long)ltodo) - 1;
      ltodo &= ltodo - 1;
      const uint32_t leaf = (uint32_t)__builtin_amdgcn_readlane((int)leaf_l, (int)ls);
      const uint32_t b = uloadu(T.leaf_start, leaf), e = uloadu(T.leaf_start, leaf + 1);
      bool on = O.state == want, all = false;
      bool anyw = __ballot(on && O.W.n >= 0) != 0;
      {
        const double *c = T.leaf_cube + 4 * (size_t)leaf;
        const double cx = uload(c, 0), cy = uload(c, 1), cz = uload(c, 2), hh = uload(c, 3) / 2;
        if (IN || leaf_inside(T, leaf)) {
          const double x0 = cx - hh, x1 = cx + hh, y0 = cy - hh, y1 = cy + hh;
          on = on && near_t(P, s2, fmin(fmax(x, x0), x1), fmin(fmax(y, y0), y1),
                            fmax(cz - hh, (double)uloadf(T.leaf_low, leaf))) >= P.thr;
          if (anyw && __ballot(on))
            on = on & wb::wedge_hit2(min(O.W.n, 2), O.W.ax, O.W.ay, O.W.bx, O.W.by, (float)(x0 - x),
                                     (float)(x1 - x), (float)(y0 - y), (float)(y1 - y));
        } else {
          // points outside their leaf's cube: findBlocks' own tests, and the
          // leaf whose eight corners are all in
          wb::Shape H = wb::make_cylinder(x, y, 0);
          H.kind = wb::SHAPE_HYPERBOLOID;
          H.cz = P.cz;
          H.por2 = P.por2;
          H.slope = sl;
          on = on && wb::hyp_intersect(H, cx, cy, cz, 2 * hh);
          all = on && wb::hyp_in_cube(H, cx, cy, cz, 2 * hh);
          for (int nd = T.leaf_parent[leaf]; nd >= 0; nd = T.node_parent[nd]) {
            const double *q = T.node_cube + 4 * (size_t)nd;
            on = on && wb::hyp_intersect(H, q[0], q[1], q[2], q[3]);
          }
          all = all && on;
        }
      }
      if (!__ballot(on)) continue;
      const bool anyall = !IN && __ballot(all) != 0;
      const uint32_t q0 = b / WB_OCT, nq = (e - 1) / WB_OCT - q0 + 1;
      for (uint32_t qb = 0; qb < nq; qb += WAVE) {
        bool h = qb + lane < nq;
        // (a lane that takes the whole leaf takes points outside its box's reach)
        if (h && (IN || !anyall)) {
          const Union R = {U.x0 - T.ox, U.x1 - T.ox, U.y0 - T.oy, U.y1 - T.oy, U.cz - T.oz, U.thr};
          const float4 bx = T.oct_xy[q0 + qb + lane];
          h = union_hits(R, s2, bx.x, bx.y, bx.z, bx.w, T.oct_z[q0 + qb + lane]);
        }
        uint64_t todo = __ballot(h);
        while (todo) {
          // the group of the next octet, and its octets that passed
          const uint32_t qf = q0 + qb + (uint32_t)__ffsll((long long)todo) - 1;
          const uint32_t chk = qf / (WB_CHUNK / WB_OCT);
          bool hit = on;
          {
            const double *bx = T.chunk_box + 6 * (size_t)chk;
            const double x0 = uload(bx, 0), x1 = uload(bx, 1), y0 = uload(bx, 2), y1 = uload(bx, 3),
                         z0 = uload(bx, 4);
            hit = on & (all | (near_t(P, s2, fmin(fmax(x, x0), x1), fmin(fmax(y, y0), y1), z0) >=
                               P.thr));
            if (anyw && __ballot(hit))
              hit = hit & wb::wedge_hit2(min(O.W.n, 2), O.W.ax, O.W.ay, O.W.bx, O.W.by,
                                         (float)(x0 - x), (float)(x1 - x), (float)(y0 - y),
                                         (float)(y1 - y));
          }
          const uint64_t hb = __ballot(hit);
          // lanes j and j + 32 fetch slot j of the group (the arrays are padded
          // to whole groups)
          double gx = 0, gy = 0, gz = 0;
          if (hb) {
            const uint32_t j = chk * WB_CHUNK + (lane & (WB_CHUNK - 1));
            gx = T.px[j]; gy = T.py[j]; gz = T.pz[j];
          }
          uint32_t cand = 0;  // this lane's candidates among the group's slots
          if (hb && __popcll(hb) <= OPEN_PAIR) {
            // few lanes need the group: two at a time, lanes 0-31 test its
            // slots against the first one's hyperboloid and care run, lanes
            // 32-63 against the second's
            uint64_t own = hb;
            while (own) {
              const uint32_t o1 = (uint32_t)__ffsll((long long)own) - 1;
              own &= own - 1;
              const uint32_t o2 = own ? (uint32_t)__ffsll((long long)own) - 1 : o1;
              own &= own - 1;
              const bool up = lane >= WAVE / 2;
              const double ox = rdl(x, o1), oy = rdl(y, o1), oz = rdl(P.cz, o1), ot = rdl(P.thr, o1);
              const double qx = rdl(x, o2), qy = rdl(y, o2), qz = rdl(P.cz, o2), qt = rdl(P.thr, o2);
              const double dx = gx - (up ? qx : ox), dy = gy - (up ? qy : oy);
              const double dz = (up ? qz : oz) - gz;
              bool c = wb::hyp_near(s2, dx, dy, dz) >= (up ? qt : ot);
              if (!IN) c = c | (__shfl((int)all, (int)(up ? o2 : o1), WAVE) != 0);
              if (anyw && __ballot(c)) {
                wb::LaneWedges V;
                const int o = (int)(up ? o2 : o1);
                V.ax[0] = __shfl(O.W.ax[0], o, WAVE); V.ay[0] = __shfl(O.W.ay[0], o, WAVE);
                V.bx[0] = __shfl(O.W.bx[0], o, WAVE); V.by[0] = __shfl(O.W.by[0], o, WAVE);
                V.bx[1] = __shfl(O.W.bx[1], o, WAVE); V.by[1] = __shfl(O.W.by[1], o, WAVE);
                V.n = __shfl(O.W.n, o, WAVE);
                c = c & wb::lane_dir(V, (float)dx, (float)dy);
              }
              const uint64_t cm = __ballot(c);
              if (lane == o1) cand = (uint32_t)cm;
              if (lane == o2 && o2 != o1) cand = (uint32_t)(cm >> 32);
            }
            // the group's slots inside the leaf
            const uint32_t s0 = chk * WB_CHUNK;
            if (b > s0) cand &= ~0u << (b - s0);
            if (e < s0 + WB_CHUNK) cand &= (1u << (e - s0)) - 1;
            const uint32_t past = (chk + 1) * (WB_CHUNK / WB_OCT) - (q0 + qb);
            todo = past < WAVE ? (todo >> past) << past : 0;
          }
          // otherwise octet by octet, every lane tests a point at a time
          for (uint32_t q = qf; todo && q0 + qb + (uint32_t)__ffsll((long long)todo) - 1 <
                                            (chk + 1) * (WB_CHUNK / WB_OCT);) {
            q = q0 + qb + (uint32_t)__ffsll((long long)todo) - 1;
            todo &= todo - 1;
            if (!hb) continue;
            uint32_t c8 = 0;
#pragma unroll
            for (uint32_t k = 0; k < WB_OCT; k++) {
              const uint32_t j = WB_OCT * (q % (WB_CHUNK / WB_OCT)) + k;
              const double dx = rdl(gx, j) - x, dy = rdl(gy, j) - y, dz = P.cz - rdl(gz, j);
              bool c = hit & (all | (wb::hyp_near(s2, dx, dy, dz) >= P.thr));
              if (!__ballot(c)) continue;
              if (anyw) c = c & wb::lane_dir(O.W, (float)dx, (float)dy);
              c8 |= c ? 1u << k : 0u;
            }
            // the octet's slots inside the leaf
            const uint32_t k0 = b > q * WB_OCT ? b - q * WB_OCT : 0;
            const uint32_t k1 = e < (q + 1) * WB_OCT ? e - q * WB_OCT : WB_OCT;
            const uint32_t in8 = ((1u << k1) - 1) & ~((1u << k0) - 1);
            cand |= (c8 & in8) << (WB_OCT * (q % (WB_CHUNK / WB_OCT)));
          }
          if (!hit) cand = 0;
          uint32_t taken = 0;
          while (__ballot(cand != 0)) {
            taken++;
            const bool has = cand != 0;
            const uint32_t j = chk * WB_CHUNK + (has ? (uint32_t)__ffs((int)cand) - 1 : 0u);
            cand &= cand - 1;
            double dx = 0, dy = 0, dz = 0;
            if (has) {
              dx = T.px[j] - x;
              dy = T.py[j] - y;
              dz = P.cz - T.pz[j];
            }
            // (a difference is zero only between equal coordinates)
            const bool c = has & ((dx != 0) | (dy != 0));
            if (!__ballot(c)) continue;
            const double t = wb::hyp_near(s2, dx, dy, dz), a = dz * __builtin_fabs(dz);
            const bool in = c & (all | (__builtin_fma(-0x1p-39, a, t) >= P.por2 + slack));
            if (c & !in) O.state = GAP ? 7 : 6;
            if (!GAP) {
              // a direction near a bin's edge waits for the leaf's end (the
              // call of the exact form would cost every lane registers in
              // this loop); a second one in the same leaf is left to the
              // heavy kernel
              bool ok;
              const int bin = wb::dir_bin_est(dy, dx, &ok);
              if (in & ok) O.occ |= 1ull << bin;
              if (in & !ok) {
                if (pend) O.state = 6;
                pend = true;
                edge[lane] = make_double2(dx, dy);
              }
            } else {
              // only a direction that may be a border bin's extreme one is
              // taken exactly: by the float position, within 2^11 units of the
              // exact one
              bool ok;
              float q;
              const uint32_t bin = (uint32_t)wb::dir_bin_est(dy, dx, &ok, &q), bd = O.border;
              const int est = (int)(q * 0x1p25f);
              const bool b0 = bin == (bd & 255u), a0 = bin == ((bd >> 8) & 255u);
              const bool b1 = bin == ((bd >> 16) & 255u), a1 = bin == (bd >> 24);
              const bool may = (b0 & (est > O.hi[0] - 4096)) | (a0 & (est - 4096 < O.lo[0])) |
                               (b1 & (est > O.hi[1] - 4096)) | (a1 & (est - 4096 < O.lo[1]));
              if (__builtin_expect(in & (!ok | may), 0)) {
                const double *ttan = A.tab, *tcos = A.tab + 511, *tsin = A.tab + 1023;
                const int p = dir_bin_pos(wb::atan2i_ext(dy, dx, ttan, tcos, tsin, A.K, &nexact));
                const uint32_t xb = (uint32_t)p >> 25;
                if (xb == (bd & 255u)) O.hi[0] = max(O.hi[0], p);
                if (xb == ((bd >> 16) & 255u)) O.hi[1] = max(O.hi[1], p);
                if (xb == ((bd >> 8) & 255u)) O.lo[0] = min(O.lo[0], p);
                if (xb == (bd >> 24)) O.lo[1] = min(O.lo[1], p);
              }
            }
          }
          if (CAP) work += taken + 1;
          // many candidates: the directions just found may leave out the next
          // group's
          if (!GAP && taken >= OPEN_REFRESH && O.occ != checked && O.state == 0) {
            checked = O.occ;
            if (gap_verdict(O.occ) == 1) {
              O.state = 1;
              on = false;
            } else {
              wb::lane_wedges_update(O.occ, edges, O.W);
            }
          }
          if (!GAP && taken >= OPEN_REFRESH) anyw = __ballot(on && O.W.n >= 0) != 0;
        }
      }
      if (!GAP) {
        if (__builtin_expect(__ballot(pend) != 0, 0)) {
          const double *ttan = A.tab, *tcos = A.tab + 511, *tsin = A.tab + 1023;
          if (pend) {
            const double2 d = edge[lane];
            O.occ |= 1ull << wb::dir_bin(d.y, d.x, ttan, tcos, tsin, A.K, &nexact);
          }
          pend = false;
        }
        if (O.state == 0 && O.occ != checked) {
          checked = O.occ;
          if (gap_verdict(O.occ) == 1) O.state = 1;
          else wb::lane_wedges_update(O.occ, edges, O.W);
        }
      }
      if (CAP && __builtin_expect(rfl((int)work) > A.open_budget, 0))
        O.state = O.state == want ? (GAP ? 7 : 6) : O.state;
      alive = __ballot(O.state == want);
      if (alive == 0) break;
      const int na = __popcll(alive);
      if (4 * na <= 3 * ualive) {
        U = wave_union(P, O.state == want);
        ualive = na;
      }
    }
  }
}

template <bool IN, bool CAP>
__device__ __forceinline__ void open_body(const ClassifyArgs &A, uint32_t u, const float *edges,
                                          double2 *edge)
{
  const TreeView &T = A.T;
  const uint32_t lane = __lane_id();
  const uint4 un = A.open_unit[u];
  const uint32_t *pool = A.pool + (((uint64_t)((uint32_t)rfl((int)un.y) >> 16) << 32) |
                                   (uint32_t)rfl((int)un.x));
  const uint32_t nleaf = (uint32_t)rfl((int)un.y) & 0xffffu;
  const uint32_t npt = (uint32_t)rfl((int)un.z);
  if (npt == 0) return;
  const bool live = lane < npt;
  const size_t at = (size_t)un.w + lane;
  OpenPoint O;
  O.state = live ? 0 : 3;
  O.occ = 0;
  double x = 0, y = 0, z = 0, hs = 0;
  if (live) {
    const HeavyRec r = A.open[at];
    uint32_t slot = 0;
    work_point(A, r.i, slot, hs);
    x = T.px[slot]; y = T.py[slot]; z = T.pz[slot];
    O.occ = r.occ;
  }
  const Near P = make_near(A, x, y, z, hs);
  int nexact = 0;
  wb::lane_wedges_update(O.occ, edges, O.W);
  open_pass<IN, false, CAP>(A, pool, nleaf, P, O, edges, edge, nexact);
  if (O.state == 0) {
    O.state = gap_verdict(O.occ);
    if (O.state == 0) O.state = 4;
  }
  if (__ballot(O.state == 4)) {
    int before[2] = {255, 255}, after[2] = {255, 255}, nr = 0;
    if (O.state == 4) {
      for (int st = 0; st < 64; st++) {
        if ((O.occ >> st) & 1) continue;
        if (!((O.occ >> ((st + 63) & 63)) & 1)) continue;
        int len = 0;
        while (len < 64 && !((O.occ >> ((st + len) & 63)) & 1)) len++;
        if (len >= 24 && nr < 2) {
          const int bf = (st + 63) & 63, af = (st + len) & 63;
          if (nr == 0) { before[0] = bf; after[0] = af; }
          else { before[1] = bf; after[1] = af; }
          nr++;
        }
      }
      // the border wedges span at most 27 bins: each one wedge
      wb::Wedges w;
      wb::border_wedges(before, after, nr, w, edges);
      O.W.ax[0] = w.ax[0]; O.W.ay[0] = w.ay[0]; O.W.bx[0] = w.bx[0]; O.W.by[0] = w.by[0];
      O.W.ax[1] = w.ax[2]; O.W.ay[1] = w.ay[2]; O.W.bx[1] = w.bx[2]; O.W.by[1] = w.by[2];
      O.W.n = nr ? nr == 2 ? 3 : 1 : -1;
    }
    O.border = (uint32_t)before[0] | (uint32_t)after[0] << 8 | (uint32_t)before[1] << 16 |
               (uint32_t)after[1] << 24;
    O.hi[0] = O.hi[1] = -1;
    O.lo[0] = O.lo[1] = 0x7fffffff;
    open_pass<IN, true, CAP>(A, pool, nleaf, P, O, edges, edge, nexact);
    if (O.state == 4) {
      const int g0 = (int)(((uint32_t)O.lo[0] - (uint32_t)O.hi[0]) & 0x7fffffffu);
      const int g1 = (int)(((uint32_t)O.lo[1] - (uint32_t)O.hi[1]) & 0x7fffffffu);
      O.state = (g0 >= wb::DEG144) | ((nr > 1) & (g1 >= wb::DEG144)) ? 2 : 1;
      atomicAdd(A.nslow, 1u);
    }
  }
  if (nexact) atomicAdd(A.atan_exact, (unsigned long long)nexact);
  if (live) {
    HeavyRec r = A.open[at];
    if (O.state >= 6) {
      r.occ = O.occ;
      r.start = (uint32_t)(O.state - 5);
      A.heavy[atomicAdd(A.nheavy, 1u)] = r;
    } else {
      uint32_t slot = 0;
      work_point(A, r.i, slot, hs);
      work_verdict(A, r.i, slot, (uint8_t)O.state);
    }
  }
}

#ifndef WB_OPEN_MINW
#define WB_OPEN_MINW 5
#endif

template <bool IN, int MINW>
__global__ void __launch_bounds__(WAVE, MINW) k_ground(ClassifyArgs A)
{
  __shared__ WaveStack S;
  __shared__ float edges[3 * 128];
  ground_setup(A, edges);
  walk_body<IN>(A, blockIdx.x, S, edges);
}

// The same walk on a grid that stays resident: each wave takes its first
// unit of 64 items by its place in the grid, then the next unit no wave has
// taken (*next counts the units taken beyond the grid's; zero before the
// launch), until none is left.  Launched with fewer blocks than fit on the
// device, it leaves room on every CU for the kernels of other streams,
// which a kernel of many short blocks does not: each freed slot goes to its
// next block.
template <bool IN, int MINW>
__global__ void __launch_bounds__(WAVE, MINW) k_ground_resident(ClassifyArgs A, uint32_t *next)
{
  __shared__ WaveStack S;
  __shared__ float edges[3 * 128];
  ground_setup(A, edges);
  const uint64_t nunits = ((A.items ? A.n_items : A.T.n) + A.walk_per - 1) / A.walk_per;
  uint64_t unit = blockIdx.x;
  while (unit < nunits) {
    walk_body<IN>(A, unit, S, edges);
    uint32_t u = 0;
    if (__lane_id() == 0) u = atomicAdd(next, 1u);
    unit = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)u) + gridDim.x;
  }
}

// Walk A of several trees in one launch: blocks boff[k] .. boff[k+1]-1 take
// tree k, whose arguments are AA[k].
template <bool IN, int MINW>
__global__ void __launch_bounds__(WAVE, MINW) k_ground_batch(const ClassifyArgs *AA,
                                                             const uint32_t *boff, int ntrees)
{
  __shared__ WaveStack S;
  __shared__ float edges[3 * 128];
  int lo = 0, hi = ntrees;  // boff[lo] <= blockIdx.x < boff[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (boff[mid] <= blockIdx.x) lo = mid;
    else hi = mid;
  }
  ground_setup(AA[lo], edges);
  walk_body<IN>(AA[lo], blockIdx.x - boff[lo], S, edges);
}

// Unit u of walk B in the order of the classes (those with the longest leaf
// lists first); false past the last.
template <bool IN, bool CAP>
__device__ __forceinline__ bool open_unit(const ClassifyArgs &A, uint32_t u, const float *edges,
                                          double2 *edge)
{
  uint32_t cls = 0;
#pragma unroll
  for (int k = 0; k < OPEN_CLASSES; k++) {
    const uint32_t nk = (uint32_t)rfl((int)A.nopen[k]);
    if (cls == (uint32_t)k && u >= nk) {
      u -= nk;
      cls++;
    }
  }
  if (cls == OPEN_CLASSES) return false;
  open_body<IN, CAP>(A, cls * A.unit_cap + u, edges, edge);
  return true;
}

// Walk B over the units walk A left, a block per unit there can be: with
// classes block u takes unit u of their order, else wave u's.  (A resident
// grid that takes the units by a counter was 3 to 7% slower on 40k to 300k
// points: every claim waits for the counter's word.)
template <bool IN, bool CAP, int MINW>
__global__ void __launch_bounds__(WAVE, MINW) k_ground_open(ClassifyArgs A)
{
  __shared__ float edges[3 * 128];
  __shared__ double2 edge[WAVE];
  ground_setup(A, edges);
  if (A.open_classes) open_unit<IN, CAP>(A, blockIdx.x, edges, edge);
  else if (blockIdx.x < A.unit_cap) open_body<IN, CAP>(A, blockIdx.x, edges, edge);
}

// The same as a grid that stays resident and takes the units by a counter
// (A.open_next, zero before the launch): with the context's sharing switch.
template <bool IN, bool CAP>
__global__ void __launch_bounds__(WAVE, WB_OPEN_MINW) k_ground_open_resident(ClassifyArgs A)
{
  __shared__ float edges[3 * 128];
  __shared__ double2 edge[WAVE];
  ground_setup(A, edges);
  for (;;) {
    uint32_t u = 0;
    if (threadIdx.x == 0) u = atomicAdd(A.open_next, 1u);
    if (!open_unit<IN, CAP>(A, (uint32_t)rfl((int)u), edges, edge)) return;
  }
}

// The entry of off[0..m] (ascending) that holds u: off[e] <= u < off[e+1]; m
// past the last.
__device__ __forceinline__ int batch_find(const uint32_t *off, int m, uint32_t u)
{
  for (int b = 0; b < m; b += WAVE) {
    const int k = b + (int)threadIdx.x;
    const uint64_t past = __ballot(k < m && off[k + 1] > u);
    if (past) return b + __builtin_ctzll(past);
  }
  return m;
}

// off[0..m]: the running sums of what the batch's trees counted: units of
// walk B by class and then tree (open), or heavy points by tree.
__global__ void __launch_bounds__(WAVE) k_batch_sums(const ClassifyArgs *AA, int ntrees, int open,
                                                     uint32_t *off)
{
  const int m = open ? ntrees * OPEN_CLASSES : ntrees;
  const int lane = threadIdx.x;
  uint32_t sum = 0;
  if (lane == 0) off[0] = 0;
  for (int b = 0; b < m; b += WAVE) {
    const int k = b + lane;
    uint32_t v = 0;
    if (k < m) v = open ? AA[k % ntrees].nopen[k / ntrees] : *AA[k].nheavy;
    for (int d = 1; d < WAVE; d <<= 1) {
      const uint32_t w = __shfl_up(v, d, WAVE);
      if (lane >= d) v += w;
    }
    if (k < m) off[k + 1] = sum + v;
    sum += (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
  }
}

// Walk B over several trees: block u takes unit u of the batch, those with
// the longest lists of every tree first (uoff: k_batch_sums).  A grid of as
// many blocks as there can be units needs no counter: taking the units tree by
// tree, each wave by each tree's counter, took 12 trees of 150k points 4.4 ms.
template <bool IN, bool CAP>
__global__ void __launch_bounds__(WAVE, WB_OPEN_MINW) k_ground_open_batch(const ClassifyArgs *AA,
                                                                          const uint32_t *uoff,
                                                                          int ntrees)
{
  __shared__ float edges[3 * 128];
  __shared__ double2 edge[WAVE];
  const int e = batch_find(uoff, ntrees * OPEN_CLASSES, blockIdx.x);
  if (e == ntrees * OPEN_CLASSES) return;
  const ClassifyArgs &A = AA[e % ntrees];
  ground_setup(A, edges);
  open_body<IN, CAP>(A, (uint32_t)(e / ntrees) * A.unit_cap + blockIdx.x - uoff[e], edges, edge);
}

// One heavy point per 64-lane block.  The shape is the same in every lane,
// so the lanes split the work.  The walk pops up to eight nodes at a time
// (lane 8i+k tests child k of the i-th node from the top; children in the
// visiting order of k_ground, the popped nodes' children stacked so the top
// node's come out first) and collects the leaves it reaches into a batch of
// up to HB_LEAVES.  A batch is served lane-parallel: per
// leaf its bounds, whether its cube lies inside the hyperboloid and which
// 32-point groups' boxes may meet it; then 64 of the batch's samples (walk
// A: the lowest point of each group) or slots (walk B, and C, the exact
// border pass for a longest empty run of 24 or 25 bins) per step, with the
// early exit checked after every step.
#ifndef HB_LEAVES
#define HB_LEAVES 256
#endif
// The heavy walk's stack.  Its levels never decrease from bottom to top
// (the children of the i-th popped node sit above those of the (i+1)-th, one
// level deeper than their parents).  So a round that pops a level-(m-1) node
// also pops every level >= m entry, and afterwards the level-m entries are
// that round's children, at most 8 x 8 = 64; until the next such round they
// only decrease.  Internal nodes sit at levels 0..20: at most 64 entries at
// each of levels 1..20.
#define HB_STK (64 * WB_MAX_LEVEL - 64)

#ifndef WB_HEAVY_MINW
#define WB_HEAVY_MINW 4
#endif
// The block's shared arrays: the walk's stack, the leaf batch (leaf,
// bounds, group mask, prefix of counts), the care wedges of walks A and B
// (uniform).
struct HeavyShared {
  int stk[HB_STK];
  uint32_t lq[HB_LEAVES], lb[HB_LEAVES], le[HB_LEAVES], lmask[HB_LEAVES];
  uint32_t lpre[HB_LEAVES + 1];
  wb::Wedges wg;
};

__device__ __forceinline__ void heavy_body(const ClassifyArgs &A, const HeavyRec hr,
                                           HeavyShared &SH)
{
  int *stk = SH.stk;
  uint32_t *lq = SH.lq, *lb = SH.lb, *le = SH.le, *lmask = SH.lmask, *lpre = SH.lpre;
  wb::Wedges &wg = SH.wg;
  const TreeView &T = A.T;
  const uint32_t i = hr.i;  // work index (k_ground hands over only lanes with a tile)
  const uint32_t lane = threadIdx.x;
  const double *ttan = A.tab, *tcos = A.tab + 511, *tsin = A.tab + 1023;
  uint32_t slot = 0;
  double hs = 0;
  work_point(A, i, slot, hs);
  const double x = T.px[slot], y = T.py[slot], z = T.pz[slot];
  const wb::Shape H = wb::make_hyperboloid(x - 0, y - 0, z - A.thickness, hs, A.max_slope);
  int nexact = 0;
  // the directions k_ground found are a subset of D; the walks it completed
  // did not pass and are not repeated
  uint64_t occ = lane == 0 ? hr.occ : 0, checked = hr.occ;
  int verdict = 0;  // 1 pass, 2 fail, 4 ambiguous
  int before[2] = {-1, -1}, afterb[2] = {-1, -1}, nr = 0;
  int hi[2] = {-1, -1}, lo[2] = {0x7fffffff, 0x7fffffff};
  for (int phase = rfl((int)hr.start); phase < 3 && verdict != 1 && verdict != 2; phase++) {
    if (phase == 2) {
      const uint64_t occw = wave_or(occ);
      verdict = gap_verdict(occw);
      if (verdict != 0) break;
      verdict = 4;
      for (int st = 0; st < 64; st++) {
        if ((occw >> st) & 1) continue;
        if (!((occw >> ((st + 63) & 63)) & 1)) continue;
        int len = 0;
        while (len < 64 && !((occw >> ((st + len) & 63)) & 1)) len++;
        if (len >= 24 && nr < 2) {
          before[nr] = (st + 63) & 63;
          afterb[nr] = (st + len) & 63;
          nr++;
        }
      }
    }
    int sp = 0;
    {
      const double *rc = T.node_cube;
      if (wb::hyp_intersect(H, rc[0], rc[1], rc[2], rc[3])) {
        if (lane == 0) stk[0] = 0;
        sp = 1;
      }
    }
    if (lane == 0) {
      if (phase < 2) wb::care_wedges(checked, wg, A.edges);
      else wb::border_wedges(before, afterb, nr, wg, A.edges);
    }
    __syncthreads();
    bool done = false;
    // batches grow 16, 64, 256 leaves: an early pass stops after few leaves
    uint32_t lim = 16;
    while (!done) {
      // collect the leaves of the next part of the walk
      uint32_t nq = 0;
      while (sp > 0 && nq + 8 <= lim) {
        // P nodes from the top of the stack, with room for their leaves in
        // the batch (the stack's own room follows from HB_STK)
        const int P = min(min(8, sp), (int)((lim - nq) / 8));
        const int gi = (int)(lane >> 3), k = (int)(lane & 7);
        const int code = gi < P ? stk[sp - 1 - gi] : 0;
        __syncthreads();
        bool h = false;
        int ck = -1, t = 0;
        if (gi < P) {
          const double *nc = T.node_cube + 4 * (size_t)code;
          const double cx = nc[0], cy = nc[1], cz = nc[2], side = nc[3];
          const int o = (x >= cx ? 1 : 0) | (y >= cy ? 2 : 0);
          ck = T.node_child[8 * (size_t)code + k];
          t = child_rank(k, o);
          if (ck != -1) {
            const double ncx = cx + (double)(2 * (k & 1) - 1) * side / 4;
            const double ncy = cy + (double)(2 * ((k & 2) / 2) - 1) * side / 4;
            const double ncz = cz + (double)(2 * ((k & 4) / 4) - 1) * side / 4;
            const double zl = A.cube_wedges ? T.child_zlow[8 * (size_t)code + k] : -__builtin_inf();
            h = wb::hyp_intersect_low(H, ncx, ncy, ncz, side / 2, zl) &&
                (!A.cube_wedges || wb::wedge_hit(wg, x, y, ncx - side / 4, ncx + side / 4,
                                                 ncy - side / 4, ncy + side / 4));
          }
        }
        // per popped node: node children and leaf children by rank
        // (OR over each group of 8 lanes: quad swaps, then the half-row mirror)
        uint32_t rn = h && ck >= 0 ? 1u << t : 0u, rl = h && ck < -1 ? 1u << t : 0u;
        rn = dpp_or<0xb1, 0xf>(rn);
        rl = dpp_or<0xb1, 0xf>(rl);
        rn = dpp_or<0x4e, 0xf>(rn);
        rl = dpp_or<0x4e, 0xf>(rl);
        rn = dpp_or<0x141, 0xf>(rn);
        rl = dpp_or<0x141, 0xf>(rl);
        // node i's children go above those of nodes i+1..P-1; its leaves
        // after those of nodes 0..i-1
        const int base = sp - P;
        int nabove = 0, lbefore = 0, ntot = 0, ltot = 0;
        for (int i = 0; i < P; i++) {
          const int cn = __popc((uint32_t)__builtin_amdgcn_readlane((int)rn, 8 * i));
          const int cl = __popc((uint32_t)__builtin_amdgcn_readlane((int)rl, 8 * i));
          if (i > gi) nabove += cn;
          if (i < gi) lbefore += cl;
          ntot += cn;
          ltot += cl;
        }
        if (h && ck >= 0) stk[base + nabove + __popc(rn >> (t + 1))] = ck;
        if (h && ck < -1) lq[nq + lbefore + __popc(rl & ((1u << t) - 1))] = (uint32_t)(-2 - ck);
        sp = base + ntot;
        nq += ltot;
        __syncthreads();
      }
      if (nq == 0) break;
      lim = min(4 * lim, (uint32_t)HB_LEAVES);
      // per-leaf bounds, inside flag (bit 31 of lmask) and group mask, and
      // the prefix of the leaves' sample counts (walk A) or selected-group
      // counts (walks B and C)
      uint32_t carry = 0;
      for (uint32_t k0 = 0; k0 < nq; k0 += WAVE) {
        const uint32_t k = k0 + lane;
        uint32_t cnt = 0;
        if (k < nq) {
          const uint32_t leaf = lq[k];
          const uint32_t b = T.leaf_start[leaf], e = T.leaf_start[leaf + 1];
          const uint32_t g0 = b / WB_CHUNK, ng = (e - 1) / WB_CHUNK - g0 + 1;
          // bits 0-30: the groups to read (groups past the 31st are always
          // read); bit 31: the leaf cube lies inside the hyperboloid
          uint32_t mask = 0x7fffffffu;
          const double *lc = T.leaf_cube + 4 * (size_t)leaf;
          const double h2 = lc[3] / 2;
          // the wedges may have narrowed since the leaf was collected
          const bool seen =
              !A.cube_wedges || wb::wedge_hit(wg, x, y, lc[0] - h2, lc[0] + h2, lc[1] - h2, lc[1] + h2);
          if (phase != 0 && seen) {
            const bool inside = wb::hyp_in_cube(H, lc[0], lc[1], lc[2], lc[3]);
            mask = inside ? 0x80000000u : 0u;
            for (uint32_t g = 0; g < ng && g < 31; g++) {
              const double *bx = T.chunk_box + 6 * (uint64_t)(g0 + g);
              if ((inside || wb::hyp_may_hit_box(H, bx[0], bx[1], bx[2], bx[3], bx[4], bx[5])) &&
                  wb::wedge_hit(wg, x, y, bx[0], bx[1], bx[2], bx[3]))
                mask |= 1u << g;
            }
          }
          lb[k] = b;
          le[k] = e;
          lmask[k] = mask;
          cnt = !seen ? 0 : phase == 0 ? ng
                                       : __popc(mask & 0x7fffffffu) + (ng > 31 ? ng - 31 : 0);
        }
        uint32_t incl = cnt;
        for (int s = 1; s < WAVE; s <<= 1) {
          const uint32_t v = (uint32_t)__shfl_up((int)incl, s, WAVE);
          if ((int)lane >= s) incl += v;
        }
        if (k < nq) lpre[k + 1] = carry + incl;
        carry += (uint32_t)__shfl((int)incl, WAVE - 1, WAVE);
      }
      if (lane == 0) lpre[0] = 0;
      __syncthreads();
      const uint32_t S = carry;
      uint32_t kc = 0;  // this lane's leaf in the batch
      // walk A: a sample per lane; walks B and C: two selected groups per
      // step, lanes 0-31 the slots of the first, 32-63 of the second
      const uint32_t per = phase == 0 ? WAVE : WAVE / WB_CHUNK;
      for (uint32_t f0 = 0; f0 < S && !done; f0 += per) {
        const uint32_t f = phase == 0 ? f0 + lane : f0 + lane / WB_CHUNK;
        while (kc + 1 < nq && lpre[kc + 1] <= f) kc++;
        if (f < S) {
          const uint32_t b = lb[kc], e = le[kc], mask = lmask[kc], o = f - lpre[kc];
          const uint32_t g0 = b / WB_CHUNK;
          uint32_t j;
          bool test = true;
          if (phase == 0) {
            j = T.chunk_low[g0 + o];
            if (j < b || j >= e) j = o == 0 ? b : (g0 + o) * WB_CHUNK;
          } else {
            // the o-th selected group of the leaf: a set bit of the mask,
            // or one of the groups past the 31st
            const uint32_t m31 = mask & 0x7fffffffu, pc = __popc(m31);
            uint32_t g;
            if (o < pc) {
              uint32_t m = m31;
              for (uint32_t q = 0; q < o; q++) m &= m - 1;
              g = __ffs(m) - 1;
            } else {
              g = 31 + (o - pc);
            }
            j = (g0 + g) * WB_CHUNK + (lane & (WB_CHUNK - 1));
            test = j >= b && j < e;
          }
          if (test) {
            const double qx = T.px[j], qy = T.py[j], qz = T.pz[j];
            const bool in = (phase != 0 && (mask >> 31)) || wb::hyp_in(H, qx, qy, qz);
            if (in && (qx != x || qy != y)) {
              const int bin = wb::dir_bin(qy - y, qx - x, ttan, tcos, tsin, A.K, &nexact);
              if (phase < 2) {
                occ |= 1ull << bin;
              } else if (bin == before[0] || bin == afterb[0] || bin == before[1] ||
                         bin == afterb[1]) {
                const int pos =
                    dir_bin_pos(wb::atan2i_ext(qy - y, qx - x, ttan, tcos, tsin, A.K, &nexact));
                for (int q = 0; q < 2; q++) {
                  if (bin == before[q] && pos > hi[q]) hi[q] = pos;
                  if (bin == afterb[q] && pos < lo[q]) lo[q] = pos;
                }
              }
            }
          }
        }
        if (phase < 2) {
          const uint64_t occw = wave_or(occ);
          if (occw != checked) {
            checked = occw;
            if (gap_verdict(occw) == 1) {
              verdict = 1;
              done = true;
            }
            __syncthreads();
            if (lane == 0) wb::care_wedges(occw, wg, A.edges);
            __syncthreads();
          }
        }
      }
      __syncthreads();
    }
  }
  if (verdict == 0) verdict = gap_verdict(wave_or(occ));
  if (verdict == 4) {
    bool pass = true;
    for (int k = 0; k < nr; k++) {
      int h = hi[k], l = lo[k];
      for (int s = 1; s < 64; s <<= 1) {
        h = max(h, __shfl_xor(h, s, 64));
        l = min(l, __shfl_xor(l, s, 64));
      }
      const int gap = (int)(((uint32_t)l - (uint32_t)h) & 0x7fffffffu);
      if (gap >= wb::DEG144) pass = false;
    }
    verdict = pass ? 1 : 2;
    if (lane == 0) atomicAdd(A.nslow, 1u);
  }
  for (int s = 1; s < 64; s <<= 1) nexact += __shfl_xor(nexact, s, 64);
  if (lane == 0) {
    work_verdict(A, i, slot, (uint8_t)verdict);
    if (nexact) atomicAdd(A.atan_exact, (unsigned long long)nexact);
  }
}


// The handed-over points, as many as the ground kernel counted (*nheavy,
// read on the device, so the host does not wait for the count): block b
// takes record b, then the next record not yet taken (*next counts the
// records taken beyond the first gridDim.x; zero before the launch).
__global__ void __launch_bounds__(64, WB_HEAVY_MINW) k_ground_heavy(ClassifyArgs A, const HeavyRec *heavy,
                                                                    const uint32_t *nheavy,
                                                                    uint32_t *next)
{
  __shared__ HeavyShared SH;
  __shared__ uint32_t take;
  const uint32_t nh = *nheavy;
  uint32_t r = blockIdx.x;
  while (r < nh) {
    heavy_body(A, heavy[r], SH);
    __syncthreads();
    if (threadIdx.x == 0) take = atomicAdd(next, 1u) + gridDim.x;
    __syncthreads();
    r = take;
  }
}

// the same over several trees (hoff: k_batch_sums; the first tree's counter
// counts the records taken)
__global__ void __launch_bounds__(64, WB_HEAVY_MINW) k_ground_heavy_batch(const ClassifyArgs *AA,
                                                                          const uint32_t *hoff,
                                                                          int ntrees)
{
  __shared__ HeavyShared SH;
  __shared__ uint32_t take;
  uint32_t r = blockIdx.x;
  for (;;) {
    const int k = batch_find(hoff, ntrees, r);
    if (k == ntrees) return;
    heavy_body(AA[k], AA[k].heavy[r - hoff[k]], SH);
    __syncthreads();
    if (threadIdx.x == 0) take = atomicAdd(AA[0].heavy_next, 1u) + gridDim.x;
    __syncthreads();
    r = take;
  }
}

// an input merged into an earlier point at its location gets that point's class
__global__ void k_dup_class(uint64_t ndup, const uint32_t *pairs, uint8_t *out)
{
  uint64_t d = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= ndup) return;
  out[pairs[2 * d]] = out[pairs[2 * d + 1]];
}

// class histogram (per-block partials, summed by k_sum_hist) and, when tile
// records are wanted, the number of ground points each deciding tile
// classified
// Class totals, and Tile::nGround (classify.cpp:151-155): CLASSIFY tests
// every point of a tile with that tile's hyperboloid size and counts the
// ground verdicts, so a point in several tiles counts once in each tile
// that finds it ground.  The point's final class is its deciding tile's
// verdict, which every tile of the same size shares; the other tiles'
// verdicts come from k_ground over work items (k_overlap_items,
// k_item_ground).
__global__ void __launch_bounds__(256) k_count_ground(uint64_t n, const uint8_t *cls,
                                                       const int32_t *memb, const uint32_t *nmemb,
                                                       const TileRec *rec, int lo,
                                                       int32_t *nground, uint32_t *partial,
                                                       int per_tile)
{
  __shared__ uint32_t h[3];
  if (threadIdx.x < 3) h[threadIdx.x] = 0;
  __syncthreads();
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint8_t c = i < n ? cls[i] : 255;
  for (int k = 0; k < 3; k++) {
    uint64_t b = __ballot(c == k);
    if (__lane_id() == 0 && b) atomicAdd(&h[k], (uint32_t)__popcll(b));
  }
  if (per_tile && c == 2) {
    int w = INT32_MIN;
    for (uint32_t k = 0; k < nmemb[i]; k++) w = max(w, memb[MAX_MEMB * i + k]);
    const double hw = rec[w - lo].hs;
    for (uint32_t k = 0; k < nmemb[i]; k++) {
      const int t = memb[MAX_MEMB * i + k];
      if (t == w || rec[t - lo].hs == hw) atomicAdd(&nground[t - lo], 1);
    }
  }
  __syncthreads();
  if (threadIdx.x < 3) partial[3 * (uint64_t)blockIdx.x + threadIdx.x] = h[threadIdx.x];
}

// A point's tiles whose hyperboloid size differs from its deciding tile's:
// with items == nullptr, off[i] receives their number; otherwise the items
// (slot, tile record index) are written from off[i] on.
__global__ void k_overlap_items(uint64_t n, const int32_t *memb, const uint32_t *nmemb,
                                const TileRec *rec, int lo, uint32_t *off, uint2 *items)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t m = nmemb[i];
  int w = INT32_MIN;
  for (uint32_t k = 0; k < m; k++) w = max(w, memb[MAX_MEMB * i + k]);
  uint32_t c = 0;
  const uint32_t base = items ? off[i] : 0;
  for (uint32_t k = 0; k < m; k++) {
    const int t = memb[MAX_MEMB * i + k];
    if (t != w && rec[t - lo].hs != rec[w - lo].hs) {
      if (items) items[base + c] = make_uint2((uint32_t)i, (uint32_t)(t - lo));
      c++;
    }
  }
  if (!items) off[i] = c;
}

__global__ void k_item_ground(uint64_t nitems, const uint2 *items, const uint8_t *item_cls,
                              int32_t *nground)
{
  const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < nitems && item_cls[k] == 2) atomicAdd(&nground[items[k].y], 1);
}

__global__ void __launch_bounds__(256) k_sum_hist(const uint32_t *partial, uint32_t nblocks,
                                                   unsigned long long *hist3)
{
  uint64_t s[3] = {0, 0, 0};
  for (uint32_t b = blockIdx.x * blockDim.x + threadIdx.x; b < nblocks; b += gridDim.x * blockDim.x)
    for (int k = 0; k < 3; k++) s[k] += partial[3 * (uint64_t)b + k];
  for (int k = 0; k < 3; k++) {
    uint64_t v = s[k];
    for (int sh = 1; sh < 64; sh <<= 1) v += __shfl_xor(v, sh, 64);
    if (__lane_id() == 0) atomicAdd(&hist3[k], (unsigned long long)v);
  }
}

// ---------------------------------------------------------------------------
// host drivers
// ---------------------------------------------------------------------------
uint32_t *wb_query_order(wb_tree *t, int kind, const double *dparams, uint64_t ns)
{
  wb_ctx *c = t->ctx;
  uint32_t *key = (uint32_t *)wb_alloc(c, 4 * ns);
  uint32_t *val = (uint32_t *)wb_alloc(c, 4 * ns);
  const double h = t->side / 2;
  hipLaunchKernelGGL(k_query_keys, dim3(wb_blocks(ns, 256)), dim3(256), 0, c->stream, dparams, ns,
                     kind, t->center[0] - h, t->center[1] - h, t->center[2] - h,
                     (double)(1u << WB_MAX_LEVEL) / t->side, key, val);
  wb_radix_sort_u32_prefix(c, key, val, ns, 4);
  wb_free(c, key, 4 * ns);
  return val;
}

void wb_run_count(wb_tree *t, int kind, const double *dparams, uint64_t ns, uint64_t *dcounts,
                  const uint32_t *order)
{
  if (ns == 0) return;
  hipStream_t st = t->ctx->stream;
  if (!order) {
    const dim3 grid((unsigned)ns), blk(WAVE);
    if (kind == wb::SHAPE_CYLINDER)
      hipLaunchKernelGGL(k_count_points_in<wb::SHAPE_CYLINDER>, grid, blk, 0, st, view(t), dparams, ns, dcounts);
    else if (kind == wb::SHAPE_SPHERE)
      hipLaunchKernelGGL(k_count_points_in<wb::SHAPE_SPHERE>, grid, blk, 0, st, view(t), dparams, ns, dcounts);
    else
      hipLaunchKernelGGL(k_count_points_in<wb::SHAPE_HYPERBOLOID>, grid, blk, 0, st, view(t), dparams, ns, dcounts);
    return;
  }
  const dim3 grid(wb_blocks(ns, 256)), blk(256);
  if (kind == wb::SHAPE_CYLINDER)
    hipLaunchKernelGGL(k_query_count<wb::SHAPE_CYLINDER>, grid, blk, 0, st, view(t), dparams,
                       order, ns, dcounts);
  else if (kind == wb::SHAPE_SPHERE)
    hipLaunchKernelGGL(k_query_count<wb::SHAPE_SPHERE>, grid, blk, 0, st, view(t), dparams,
                       order, ns, dcounts);
  else
    hipLaunchKernelGGL(k_query_count<wb::SHAPE_HYPERBOLOID>, grid, blk, 0, st, view(t), dparams,
                       order, ns, dcounts);
}

void wb_run_points(wb_tree *t, int kind, const double *dparams, uint64_t ns, const uint64_t *doffs,
                   uint32_t *dout, const uint32_t *order)
{
  if (ns == 0) return;
  hipStream_t st = t->ctx->stream;
  if (!order) {
    const dim3 grid((unsigned)ns), blk(WAVE);
    if (kind == wb::SHAPE_CYLINDER)
      hipLaunchKernelGGL(k_points_in<wb::SHAPE_CYLINDER>, grid, blk, 0, st, view(t), dparams, ns, doffs, dout);
    else if (kind == wb::SHAPE_SPHERE)
      hipLaunchKernelGGL(k_points_in<wb::SHAPE_SPHERE>, grid, blk, 0, st, view(t), dparams, ns, doffs, dout);
    else
      hipLaunchKernelGGL(k_points_in<wb::SHAPE_HYPERBOLOID>, grid, blk, 0, st, view(t), dparams, ns, doffs, dout);
    return;
  }
  const dim3 grid(wb_blocks(ns, 256)), blk(256);
  if (kind == wb::SHAPE_CYLINDER)
    hipLaunchKernelGGL(k_query_points<wb::SHAPE_CYLINDER>, grid, blk, 0, st, view(t), dparams,
                       order, ns, doffs, dout);
  else if (kind == wb::SHAPE_SPHERE)
    hipLaunchKernelGGL(k_query_points<wb::SHAPE_SPHERE>, grid, blk, 0, st, view(t), dparams,
                       order, ns, doffs, dout);
  else
    hipLaunchKernelGGL(k_query_points<wb::SHAPE_HYPERBOLOID>, grid, blk, 0, st, view(t), dparams,
                       order, ns, doffs, dout);
}

// Room for what walk A of n work indices leaves to walk B: units of every
// wave (in each class), and leaf lists of OPEN_LIST entries a wave, with a
// shared end for the longer ones (a list that finds no room there sends its
// lanes to the heavy kernel).
struct OpenBuffers {
  HeavyRec *open;
  uint4 *unit;
  uint32_t *pool;
  size_t nrec, nunit, npool;
};

// The state of one tree's classification pass between its phases:
// classify_prepare (tile geometry, membership, SCAN, POSTSCAN, the ground
// test's arguments), the ground test (one tree, or several in one launch),
// classify_finish (counts, Tile::nGround, tile records, timings, release).
struct ClassifyRun {
  wb_tree *t;
  wb_ctx *c;  // allocations and stream (the tree's context, or a batch's)
  hipStream_t st;
  const wb_classify_params *p;
  uint8_t *d_class_out;
  wb_tile *tiles_out;  // host, or null
  bool scan_only;
  ClassifyOut *out;
  uint64_t n;
  TileGeo g;
  hipEvent_t ev[8];
  int32_t *tex, *tey, *memb, *grid;
  uint32_t *tile_cnt, *tile_fill, *nmemb, *err, *nslow, *tile_off, *lists;
  TileRec *rec;
  uint8_t *state;
  unsigned long long *ctr;
  uint64_t gcells, total;
  uint8_t *cls;
  HeavyRec *heavy;
  OpenBuffers open;
  ClassifyArgs A;
  uint32_t h_nheavy, h_nslow;
  uint32_t *heavy_next;  // records the heavy kernel has taken beyond its grid
};

// The flowsnake coordinates of tiles lo .. lo+ntiles-1 and the address
// grid over them (k_tile_geo, k_tile_grid) depend on nothing else, so the
// context keeps those of its last WB_GEO_CACHE tilings: a pass over a tiling
// seen before neither recomputes them nor waits for the grid's bounds.
static const wb_ctx::TileGeoCache &tile_geometry(wb_ctx *c, const TileGeo &g0)
{
  for (size_t k = 0; k < c->geo.size(); k++)
    if (c->geo[k].lo == g0.lo && c->geo[k].ntiles == g0.ntiles) {
      if (k + 1 != c->geo.size()) std::rotate(c->geo.begin() + k, c->geo.begin() + k + 1, c->geo.end());
      return c->geo.back();
    }
  hipStream_t st = c->stream;
  wb_ctx::TileGeoCache e;
  e.lo = g0.lo;
  e.ntiles = g0.ntiles;
  e.tex = (int32_t *)wb_alloc(c, 4ull * g0.ntiles);
  e.tey = (int32_t *)wb_alloc(c, 4ull * g0.ntiles);
  int *dbounds = (int *)wb_alloc(c, 16);
  hipLaunchKernelGGL(k_bounds_init, dim3(1), dim3(64), 0, st, dbounds);
  hipLaunchKernelGGL(k_tile_geo, dim3(wb_blocks(g0.ntiles, 256)), dim3(256), 0, st, g0, e.tex,
                     e.tey, dbounds);
  int *hb = (int *)(c->hbox + WB_HBOX_GEO);
  WB_CHECK(hipMemcpyAsync(hb, dbounds, 16, hipMemcpyDeviceToHost, st));
  WB_CHECK(hipStreamSynchronize(st));
  wb_free(c, dbounds, 16);
  TileGeo g = g0;
  e.gx0 = g.gx0 = hb[0];
  e.gy0 = g.gy0 = hb[2];
  e.gw = g.gw = hb[1] - hb[0] + 1;
  e.gh = g.gh = hb[3] - hb[2] + 1;
  const uint64_t gcells = (uint64_t)g.gw * (uint64_t)g.gh;
  e.grid = (int32_t *)wb_alloc(c, 4 * gcells);
  hipLaunchKernelGGL(k_fill_i32, dim3(wb_blocks(gcells, 256)), dim3(256), 0, st, e.grid, gcells, -1);
  hipLaunchKernelGGL(k_tile_grid, dim3(wb_blocks(g.ntiles, 256)), dim3(256), 0, st, g, e.tex, e.tey,
                     e.grid);
  if (c->geo.size() >= WB_GEO_CACHE) {
    // the oldest tiling's arrays go back to the pool (stream-ordered reuse)
    wb_ctx::TileGeoCache &o = c->geo.front();
    wb_free(c, o.tex, 4ull * o.ntiles);
    wb_free(c, o.tey, 4ull * o.ntiles);
    wb_free(c, o.grid, 4 * (uint64_t)o.gw * (uint64_t)o.gh);
    c->geo.erase(c->geo.begin());
  }
  c->geo.push_back(e);
  return c->geo.back();
}

static void open_buffers(wb_ctx *c, ClassifyArgs &A, uint64_t n, uint64_t nbatch, OpenBuffers &B)
{
  const uint64_t resident = 20 * (uint64_t)c->ncu;
  // Points of a wave of walk A and of a unit of walk B.  A wave of 16 takes
  // more than a quarter of the time of one of 64 (lanes that need the same
  // nodes and points share their tests), but with few waves the longest one is
  // the kernel (ground test of 18.5k points 0.27 ms with waves of 64, 0.25
  // with 16; 150k with outliers above 1.60 and 1.31; 300k, waves of 32, 1.77
  // and 1.65).
  const uint64_t all = (nbatch ? nbatch : n) / WAVE;
  A.walk_per = 2 * all < resident ? 16 : all < resident ? 32 : WAVE;
  A.open_per = WAVE;
  // How long a wave may go on before its open lanes go to the wave-per-point
  // kernel: the leaves walk A lists, and the groups and rounds of candidates
  // walk B takes.  Hyperboloids of a shallow slope reach many leaves and hold
  // most of their points, and points outside the root lie in leaves that no
  // cube bounds; the longest waves are then the kernels of all but the largest
  // clouds, and the heavy kernel, 30 to 60 ns a point, has the chip to itself.
  // The three kernels in ms with 256 leaves and no budget, and so: slope 0.1,
  // high outliers, 35k points 0.99 0.78, 60k 3.12 1.7, 150k 2.6 1.6, 400k 4.1 2.2,
  // 1.17M 5.4 3.8, 2.4M 7.2 5.2, 7M 16.4 13.4, 23.7M 34.3 35.6; low ones, 150k 1.4
  // 1.0, 1.17M 3.2 1.9, 7M 4.4 3.6, 23.7M 9.3 7.5; slope 1 with points outside the
  // root, 60k 1.66 1.14, 70k 1.65 1.33.  At slope 1 in a root that holds all, the
  // walks' longest waves cost less than the heavy kernel's start in some clouds
  // and more in others (150k points, low outliers, 0.66 0.62; none 0.91 0.98).
  // (Slope 0.3, 7M and more, is as slope 1: 16.1 and, handing over, 17.3.)
  const bool shallow = A.max_slope < (all < 12 * resident ? 0.5 : 0.2);
  A.leaf_cap = GROUND_LEAVES;
  A.open_budget = INT32_MAX;
  if (shallow || !A.cube_wedges) {
    if (16 * all < resident) A.leaf_cap = 96;
    else if (3 * all < resident) A.leaf_cap = shallow ? 32 : 64;
    else if (all < 3 * resident) A.leaf_cap = 96;
    else if (shallow) A.leaf_cap = all < 12 * resident ? 128 : 160;
    A.open_budget = all < (shallow ? 12 : 3) * resident ? 512 : shallow ? 1024 : 2048;
  }
  const uint64_t waves = (n + A.walk_per - 1) / A.walk_per;
  B.nrec = (size_t)waves * WAVE;
  const uint32_t ucap = (uint32_t)std::min<uint64_t>(waves * 4, 0x3fffffffull);
  A.pool_shared = waves * OPEN_LIST;
  B.npool = (size_t)(waves * (OPEN_LIST + 16) + 65536);
  A.pool_cap = B.npool;
  A.unit_cap = (uint32_t)waves;
  // The longest first while a long one is a large part of the whole (1.17M
  // points 3.07 to 2.49 ms); with more points neighbours in space stay
  // neighbours in time, which the caches gain from, and no place in a class is
  // claimed (23.7M points, mostly ground: 31.8 to 29.8 ms).
  A.open_classes = nbatch || c->sharing || waves < 20 * resident;
  if (A.open_classes) {
    A.unit_cap = ucap;
    A.open_per = 2 * all < resident ? OPEN_P1 : 3 * all < 4 * resident ? OPEN_P2 : WAVE;
    A.open_per = std::min(A.open_per, A.walk_per);
  }
  B.nunit = (size_t)A.unit_cap * (A.open_classes ? OPEN_CLASSES : 1);
  A.open = B.open = (HeavyRec *)wb_alloc(c, sizeof(HeavyRec) * B.nrec + 16);
  A.open_unit = B.unit = (uint4 *)wb_alloc(c, sizeof(uint4) * B.nunit + 16);
  A.pool = B.pool = (uint32_t *)wb_alloc(c, 4 * B.npool);
}

static void open_release(wb_ctx *c, OpenBuffers &B)
{
  wb_free(c, B.open, sizeof(HeavyRec) * B.nrec + 16);
  wb_free(c, B.unit, sizeof(uint4) * B.nunit + 16);
  wb_free(c, B.pool, 4 * B.npool);
}

static void classify_prepare(ClassifyRun &R, wb_tree *t, wb_ctx *c, const double *corners,
                             int ncorners, const wb_classify_params *p, uint8_t *d_class_out,
                             wb_tile *tiles_out, bool scan_only, uint64_t nbatch,
                             ClassifyOut *out)
{
  R.t = t; R.c = c; R.st = c->stream; R.p = p; R.d_class_out = d_class_out;
  R.tiles_out = tiles_out; R.scan_only = scan_only; R.out = out;
  R.cls = nullptr; R.heavy = nullptr; R.h_nheavy = 0; R.h_nslow = 0;
  hipStream_t st = R.st;
  const uint64_t n = R.n = t->n;
  wb::SnakeSetup ss = wb::snake_setup_corners(corners, ncorners, p->tile_size);
  TileGeo &g = R.g;
  g.scx = ss.cx; g.scy = ss.cy; g.spacing = ss.spacing; g.r = ss.radius;
  g.lo = ss.lo; g.hi = ss.hi;
  g.ntiles = (uint32_t)((int64_t)ss.hi - ss.lo + 1);
  for (int k = 0; k < 8; k++) R.ev[k] = wb_event_get(c);
  hipEvent_t *ev = R.ev;
  WB_CHECK(hipEventRecord(ev[0], st));
  const wb_ctx::TileGeoCache &geo = tile_geometry(c, g);
  int32_t *tex = R.tex = geo.tex;
  int32_t *tey = R.tey = geo.tey;
  uint32_t *tile_cnt = R.tile_cnt = (uint32_t *)wb_alloc(c, 4ull * g.ntiles + 4);
  uint32_t *tile_fill = R.tile_fill = (uint32_t *)wb_alloc(c, 4ull * g.ntiles + 4);
  uint8_t *state = R.state = (uint8_t *)wb_alloc(c, (size_t)g.ntiles + 4);
  TileRec *rec = R.rec = (TileRec *)wb_alloc(c, sizeof(TileRec) * (size_t)g.ntiles);
  int32_t *memb = R.memb = (int32_t *)wb_alloc(c, 4ull * MAX_MEMB * n + 16);
  uint32_t *nmemb = R.nmemb = (uint32_t *)wb_alloc(c, 4ull * n + 4);
  // err[0] error flags; then u64 counters: 0 sector borderline, 1 exact atan2i
  // steps, 2-4 class histogram, 5 non-empty tiles, 6 (two u32) exact gap
  // points and heavy points, 7 FP64 fit fallbacks; u32 18-19 work counters of
  // the heavy and resident ground kernels, 20-26 the scan's class list lengths;
  // past the words the host reads: 32-37 walk B's units of each class, records
  // and units taken, u64 at 38 its leaf list entries
  uint32_t *err = R.err = (uint32_t *)wb_alloc(c, 256);
  unsigned long long *ctr = R.ctr = (unsigned long long *)err + 1;
  uint32_t *nslow = R.nslow = (uint32_t *)(ctr + 6);
  R.heavy_next = err + 18;
  hipLaunchKernelGGL(k_pass_init, dim3(wb_blocks(std::max<uint64_t>(g.ntiles, 256), 1024)),
                     dim3(256), 0, st, g.ntiles, tile_cnt, tile_fill, (uint32_t *)state, err);
  TreeView T = view(t);
  g.gx0 = geo.gx0;
  g.gy0 = geo.gy0;
  g.gw = geo.gw;
  g.gh = geo.gh;
  g.grid = R.grid = geo.grid;
  LeafWin *lwin = (LeafWin *)wb_alloc(c, sizeof(LeafWin) * ((size_t)t->nleaves + 1));
  uint8_t *lflags = (uint8_t *)wb_alloc(c, (size_t)LEAF_WIN * t->nleaves + 16);
  if (t->nleaves)
    hipLaunchKernelGGL(k_leaf_tiles, dim3(t->nleaves), dim3(64), 0, st, T, g, lwin, lflags);
  if (n > 0)
    hipLaunchKernelGGL(k_membership, dim3(wb_blocks(n, 256)), dim3(256), 0, st, T, g, lwin,
                       lflags, memb, nmemb, tile_cnt, err);
  wb_free(c, lwin, sizeof(LeafWin) * ((size_t)t->nleaves + 1));
  wb_free(c, lflags, (size_t)LEAF_WIN * t->nleaves + 16);
  // tile lists in canonical order
  uint32_t *tile_off = R.tile_off = (uint32_t *)wb_alloc(c, 4ull * g.ntiles + 4);
  wb_exclusive_scan_u32_to(c, tile_cnt, tile_off, g.ntiles);
  // room for the most list entries there can be, so that the host need not
  // wait for their number (about 40 us); from 16M points, where the wait is
  // lost in the pass and the room is not, the number itself
  uint64_t total = MAX_MEMB * n;
  if (n > (16u << 20)) {
    WB_CHECK(hipStreamSynchronize(st));
    const uint32_t *h = c->hbox + WB_HBOX_SCAN;
    total = (uint64_t)h[0] | ((uint64_t)h[1] << 32);
  }
  R.total = total;
  uint32_t *lists = R.lists = (uint32_t *)wb_alloc(c, 4 * total + 4);
  if (n > 0)
    hipLaunchKernelGGL(k_tile_lists, dim3(wb_blocks(n, 256)), dim3(256), 0, st, n, memb, nmemb,
                       g.lo, t->crank, tile_off, tile_fill, lists);
  WB_CHECK(hipEventRecord(ev[1], st));
  {
    // the size classes' tile lists, then one wave per tile of each class,
    // grid-stride over its list
    uint32_t *la = tile_fill;  // free until the ground counts
    uint32_t *lb = (uint32_t *)wb_alloc(c, 4ull * g.ntiles + 4);
    uint32_t *lc = (uint32_t *)wb_alloc(c, 4ull * g.ntiles + 4);
    uint32_t *ld = (uint32_t *)wb_alloc(c, 4ull * g.ntiles + 4);
    uint32_t *ncls = err + 20;
    // a wave per step of a class's kernel: no more than there can be points
    // for, and no more than keep the chip busy
    auto nb = [&](uint64_t least, unsigned per) {
      const uint64_t tiles = std::min<uint64_t>(g.ntiles, MAX_MEMB * n / least + 1);
      return dim3((unsigned)std::min<uint64_t>((tiles + per - 1) / per, SCAN_GRID));
    };
    const int prec = p->fit_precision;
    const bool many = n >= SCAN_MANY && prec == WB_FIT_FP64;
    if (g.ntiles) {
      hipLaunchKernelGGL(k_scan_classes, dim3(wb_blocks(g.ntiles, 1024)), dim3(1024), 0, st,
                         g.ntiles, tile_cnt, la, lb, lc, ld, ncls, many ? 8u : 0u);
      const uint32_t e = g.ntiles - 1;
      const ClassList c8 = {la, 1, ncls}, c16 = {lb, 1, ncls + 1}, c32 = {lc, 1, ncls + 2};
      const ClassList c64 = {ld, 1, ncls + 3}, c128 = {lc + e, -1, ncls + 4};
      const ClassList c256 = {lb + e, -1, ncls + 5}, cbig = {la + e, -1, ncls + 6};
#define WB_SCAN_REG(K, F32, T, W, least, CL)                                                      \
  hipLaunchKernelGGL((k_scan_reg<K, F32, T, W>), nb(least, T), dim3(64), 0, st, T_, g, tex, tey,  \
                     tile_off, tile_cnt, lists, CL, p->min_hs, prec, rec, state, ctr)
      const TreeView &T_ = T;
      if (many) {
        hipLaunchKernelGGL(k_scan_lane, nb(1, WAVE), dim3(64), 0, st, T, g, tex, tey, tile_off,
                           tile_cnt, lists, c8, p->min_hs, rec, state, ctr);
#define WB_SCAN_ROW(GS, R, W, least, CL)                                                          \
  hipLaunchKernelGGL((k_scan_row<GS, R, W>), nb(least, WAVE / GS * R), dim3(64), 0, st, T, g, tex, \
                     tey, tile_off, tile_cnt, lists, CL, p->min_hs, rec, state, ctr)
        WB_SCAN_ROW(16, 4, 3, 9, c16);
        WB_SCAN_ROW(32, 4, 3, 17, c32);
        WB_SCAN_REG(1, false, 4, 4, 33, c64);
        WB_SCAN_REG(2, false, 2, 4, 65, c128);
#undef WB_SCAN_ROW
        WB_SCAN_REG(4, false, 1, 4, 129, c256);
      } else if (prec == WB_FIT_FP64) {
        hipLaunchKernelGGL(k_scan_mixed, nb(1, 1), dim3(64), 0, st, T, g, tex, tey, tile_off, tile_cnt,
                           lists, c16, c32, c64, c128, c256, p->min_hs, rec, state, ctr);
      } else {
        WB_SCAN_REG(1, true, 1, 4, 1, c16);
        WB_SCAN_REG(1, true, 1, 4, 17, c32);
        WB_SCAN_REG(1, true, 1, 4, 33, c64);
        WB_SCAN_REG(2, true, 1, 4, 65, c128);
        WB_SCAN_REG(4, true, 1, 4, 129, c256);
      }
#undef WB_SCAN_REG
      hipLaunchKernelGGL(k_scan, dim3(std::min(nb(257, 1).x, 4096u)), dim3(64), 0, st, T, g, tex,
                         tey, tile_off, tile_cnt, lists, cbig, p->min_hs, prec, rec, state, err, ctr);
    }
    wb_free(c, lb, 4ull * g.ntiles + 4);
    wb_free(c, lc, 4ull * g.ntiles + 4);
    wb_free(c, ld, 4ull * g.ntiles + 4);
  }
  hipLaunchKernelGGL(k_postscan, dim3(wb_blocks(g.ntiles, 256)), dim3(256), 0, st, g, tex, tey,
                     state, rec, (int32_t *)tile_fill, ctr + 5);
  WB_CHECK(hipEventRecord(ev[2], st));
  for (int k = 4; k < 8; k++) WB_CHECK(hipEventRecord(ev[k], st));
  if (scan_only) return;
  R.cls = (uint8_t *)wb_alloc(c, n + 16);
  ClassifyArgs &A = R.A;
  A.T = T; A.g = g; A.memb = memb; A.nmemb = nmemb; A.rec = rec;
  A.thickness = p->thickness; A.max_slope = p->max_slope;
  A.cube_wedges = t->outside_root ? 0 : 1;
  A.tab = c->d_tan; A.K = c->kconst; A.cls = R.cls; A.cls_in = d_class_out; A.nslow = nslow;
  A.edges = c->d_edges;
  A.atan_exact = ctr + 1;
  A.items = nullptr;
  A.n_items = 0;
  A.item_cls = nullptr;
  R.heavy = (HeavyRec *)wb_alloc(c, sizeof(HeavyRec) * (n + 1));
  A.heavy = R.heavy;
  open_buffers(c, A, n, nbatch, R.open);
  A.nopen = err + 32;
  A.open_next = err + 37;
  A.npool = (unsigned long long *)(err + 38);
  A.heavy_next = R.heavy_next;
  A.nheavy = nslow + 1;
}

// walk A, walk B and the heavy kernel over n work indices of A; ev (may be
// null): events around the first two and around the heavy kernel
static void launch_ground(wb_ctx *c, const ClassifyArgs &A, uint64_t n, uint32_t *resident_next,
                          hipEvent_t *ev)
{
  hipStream_t st = c->stream;
  const uint32_t ncu = (uint32_t)c->ncu;
  if (ev) WB_CHECK(hipEventRecord(ev[0], st));
  if (n > 0) {
    const uint32_t nb = wb_blocks(n, A.walk_per);
    const dim3 one(WAVE);
    // sharing: 16 of the 20 waves a CU holds: a wave slot and LDS stay free on
    // every SIMD for other contexts' kernels
    const bool res = c->sharing && resident_next;
    const dim3 rgrid(std::min<uint32_t>(nb, 16u * ncu));
    if (A.cube_wedges) {
      if (res)
        hipLaunchKernelGGL((k_ground_resident<true, WB_GROUND_MINW>), rgrid, one, 0, st, A,
                           resident_next);
      else
        hipLaunchKernelGGL((k_ground<true, WB_GROUND_MINW>), dim3(nb), one, 0, st, A);
    } else {
      if (res)
        hipLaunchKernelGGL((k_ground_resident<false, WB_GROUND_MINW>), rgrid, one, 0, st, A,
                           resident_next);
      else
        hipLaunchKernelGGL((k_ground<false, WB_GROUND_MINW>), dim3(nb), one, 0, st, A);
    }
    const bool cap = A.open_budget != INT32_MAX;
    if (c->sharing) {  // 12 of the 20 waves a CU holds
      const dim3 ogrid(std::min<uint32_t>(nb, 12u * ncu));
      if (!A.cube_wedges)
        hipLaunchKernelGGL((k_ground_open_resident<false, true>), ogrid, one, 0, st, A);
      else if (cap)
        hipLaunchKernelGGL((k_ground_open_resident<true, true>), ogrid, one, 0, st, A);
      else
        hipLaunchKernelGGL((k_ground_open_resident<true, false>), ogrid, one, 0, st, A);
    } else {
      const dim3 ogrid(nb * (A.walk_per / A.open_per));
      // with many units six waves per SIMD hide more than the registers they
      // give up cost (23.7M points, mostly ground: about 1 ms of 29 less than
      // with five); with few the longest unit is the kernel (1.17M: 1.95 ms
      // with five, 2.09 with six)
      if (!A.cube_wedges)
        hipLaunchKernelGGL((k_ground_open<false, true, WB_OPEN_MINW>), ogrid, one, 0, st, A);
      else if (cap && A.open_classes)
        hipLaunchKernelGGL((k_ground_open<true, true, WB_OPEN_MINW>), ogrid, one, 0, st, A);
      else if (cap)
        hipLaunchKernelGGL((k_ground_open<true, true, 6>), ogrid, one, 0, st, A);
      else if (A.open_classes)
        hipLaunchKernelGGL((k_ground_open<true, false, WB_OPEN_MINW>), ogrid, one, 0, st, A);
      else
        hipLaunchKernelGGL((k_ground_open<true, false, 6>), ogrid, one, 0, st, A);
    }
  }
  if (ev) {
    WB_CHECK(hipEventRecord(ev[1], st));
    WB_CHECK(hipEventRecord(ev[2], st));
  }
  if (n > 0) {
    // at most one block per handed-over point, and no more than fit on the
    // device at once; the count is read on the device
    // sharing: 8 blocks per CU, about half the LDS the kernel could hold
    const unsigned nb =
        (unsigned)std::min<uint64_t>(n, c->sharing ? 8ull * ncu : (uint64_t)HEAVY_GRID);
    hipLaunchKernelGGL(k_ground_heavy, dim3(nb), dim3(64), 0, st, A, A.heavy, A.nheavy,
                       A.heavy_next);
  }
  if (ev) WB_CHECK(hipEventRecord(ev[3], st));
}

// the ground test of one tree
static void classify_ground_single(ClassifyRun &R)
{
  launch_ground(R.c, R.A, R.n, R.err + 19, R.ev + 4);
}

static void classify_finish(ClassifyRun &R)
{
  wb_tree *t = R.t;
  wb_ctx *c = R.c;
  hipStream_t st = R.st;
  const uint64_t n = R.n;
  const TileGeo &g = R.g;
  hipEvent_t *ev = R.ev;
  ClassifyOut *out = R.out;
  const bool want_tiles = R.tiles_out != nullptr, scan_only = R.scan_only;
  int32_t *memb = R.memb;
  uint32_t *nmemb = R.nmemb, *nslow = R.nslow, *err = R.err;
  TileRec *rec = R.rec;
  unsigned long long *ctr = R.ctr;
  uint8_t *cls = R.cls, *d_class_out = R.d_class_out;
  const ClassifyArgs &A = R.A;
  int32_t *nground = (int32_t *)R.tile_fill;  // (k_postscan cleared it)
  if (!scan_only) {
    if (n > 0) {
      const unsigned nbk = wb_blocks(n, 256);
      uint32_t *partial = (uint32_t *)wb_alloc(c, 12ull * nbk);
      hipLaunchKernelGGL(k_count_ground, dim3(nbk), dim3(256), 0, st, n, cls, memb, nmemb, rec,
                         g.lo, nground, partial, want_tiles ? 1 : 0);
      hipLaunchKernelGGL(k_sum_hist, dim3(std::min(wb_blocks(nbk, 256), 64u)), dim3(256), 0, st,
                         partial, nbk, ctr + 2);
      wb_free(c, partial, 12ull * nbk);
      if (t->ndup)
        hipLaunchKernelGGL(k_dup_class, dim3(wb_blocks(t->ndup, 256)), dim3(256), 0, st, t->ndup,
                           t->dup_pairs, d_class_out);
    }
    if (want_tiles && n > 0) {
      // Tile::nGround of the tiles that do not decide a point they hold:
      // the ground test again with their hyperboloid size, for the
      // (point, tile) pairs whose size differs from the deciding tile's
      uint32_t *off = (uint32_t *)wb_alloc(c, 4 * n + 4);
      hipLaunchKernelGGL(k_overlap_items, dim3(wb_blocks(n, 256)), dim3(256), 0, st, n, memb,
                         nmemb, rec, g.lo, off, nullptr);
      const uint64_t nitems = wb_exclusive_scan_u32(c, off, n);
      if (nitems > 0xffffffffull) {
        wb_free(c, off, 4 * n + 4);
        throw std::string("more than 2^32-1 (point, tile) pairs to recount");
      }
      if (nitems) {
        uint2 *items = (uint2 *)wb_alloc(c, 8 * nitems);
        uint8_t *icls = (uint8_t *)wb_alloc(c, nitems + 16);
        HeavyRec *iheavy = (HeavyRec *)wb_alloc(c, sizeof(HeavyRec) * (nitems + 1));
        // the pass's own counters: exact gap points, handed-over items,
        // emulated atan2i steps (the statistics keep the main pass's)
        unsigned long long *ict = (unsigned long long *)wb_alloc(c, 64);
        WB_CHECK(hipMemsetAsync(ict, 0, 64, st));
        hipLaunchKernelGGL(k_overlap_items, dim3(wb_blocks(n, 256)), dim3(256), 0, st, n, memb,
                           nmemb, rec, g.lo, off, items);
        ClassifyArgs B = A;
        B.items = items;
        B.n_items = nitems;
        B.item_cls = icls;
        B.heavy = iheavy;
        B.nslow = (uint32_t *)ict;
        B.nheavy = (uint32_t *)ict + 1;
        B.atan_exact = ict + 1;
        B.heavy_next = (uint32_t *)ict + 4;
        B.nopen = (uint32_t *)ict + 5;
        B.open_next = (uint32_t *)ict + 10;
        B.npool = ict + 6;
        OpenBuffers ib;
        open_buffers(c, B, nitems, 0, ib);
        launch_ground(c, B, nitems, nullptr, nullptr);
        hipLaunchKernelGGL(k_item_ground, dim3(wb_blocks(nitems, 256)), dim3(256), 0, st, nitems,
                           items, icls, nground);
        WB_CHECK(hipStreamSynchronize(st));
        wb_free(c, items, 8 * nitems);
        wb_free(c, icls, nitems + 16);
        wb_free(c, iheavy, sizeof(HeavyRec) * (nitems + 1));
        wb_free(c, ict, 64);
        open_release(c, ib);
      }
      wb_free(c, off, 4 * n + 4);
    }
  }
  WB_CHECK(hipEventRecord(ev[3], st));
  uint32_t *herr = c->hbox + WB_HBOX_ERR;
  WB_CHECK(hipMemcpyAsync(herr, err, 128, hipMemcpyDeviceToHost, st));
  WB_CHECK(hipStreamSynchronize(st));
  uint32_t h_err[32];
  std::copy(herr, herr + 32, h_err);
  // the exact-gap and heavy point counts (nslow[0], nslow[1])
  R.h_nslow = h_err[14];
  R.h_nheavy = h_err[15];
  if (want_tiles && g.ntiles && !(h_err[0] & 3u)) {
    // the records as the caller holds them, in one copy
    wb_tile *tiles = (wb_tile *)wb_alloc(c, sizeof(wb_tile) * (size_t)g.ntiles);
    hipLaunchKernelGGL(k_tile_out, dim3(wb_blocks(g.ntiles, 256)), dim3(256), 0, st, g.ntiles,
                       R.tile_cnt, rec, R.tex, R.tey, scan_only ? nullptr : nground, tiles);
    WB_CHECK(hipMemcpyAsync(R.tiles_out, tiles, sizeof(wb_tile) * (size_t)g.ntiles,
                            hipMemcpyDeviceToHost, st));
    WB_CHECK(hipStreamSynchronize(st));
    wb_free(c, tiles, sizeof(wb_tile) * (size_t)g.ntiles);
  }
  float ms1 = 0, ms2 = 0, ms3 = 0;
  hipEventElapsedTime(&ms1, ev[0], ev[1]);
  hipEventElapsedTime(&ms2, ev[1], ev[2]);
  hipEventElapsedTime(&ms3, ev[2], ev[3]);
  float ms4 = 0;
  hipEventElapsedTime(&ms4, ev[4], ev[5]);
  out->ms_classify_kernel = ms4;
  float ms5 = 0;
  hipEventElapsedTime(&ms5, ev[6], ev[7]);
  out->ms_heavy_kernel = ms5;
  for (int k = 0; k < 8; k++) wb_event_put(c, ev[k]);
  unsigned long long *hc = (unsigned long long *)(h_err + 2);
  out->borderline = hc[0];
  out->atan_exact = hc[1];
  out->hist[0] = hc[2]; out->hist[1] = hc[3]; out->hist[2] = hc[4];
  out->nonempty = hc[5];
  out->fallbacks = hc[7];
  out->nslow = R.h_nslow;
  out->ms_tiles = ms1; out->ms_scan = ms2; out->ms_classify = ms3;
  wb_free(c, R.tile_cnt, 4ull * g.ntiles + 4);
  wb_free(c, R.tile_fill, 4ull * g.ntiles + 4);
  wb_free(c, rec, sizeof(TileRec) * (size_t)g.ntiles);
  wb_free(c, R.state, (size_t)g.ntiles + 4);
  wb_free(c, memb, 4ull * MAX_MEMB * n + 16);
  wb_free(c, nmemb, 4ull * n + 4);
  wb_free(c, R.tile_off, 4ull * g.ntiles + 4);
  wb_free(c, R.lists, 4 * R.total + 4);
  if (cls) wb_free(c, cls, n + 16);
  if (R.heavy) {
    wb_free(c, R.heavy, sizeof(HeavyRec) * (n + 1));
    open_release(c, R.open);
  }
  out->nheavy = R.h_nheavy;
  if (h_err[0] & 1u) { wb_free(c, err, 256); throw std::string("a point lies in more than 4 tile cylinders"); }
  if (h_err[0] & 2u) { wb_free(c, err, 256); throw std::string("a tile cylinder holds more than 1024 points"); }
  wb_free(c, err, 256);
}

void wb_run_classify(wb_tree *t, const double *corners, int ncorners,
                     const wb_classify_params *p, uint8_t *d_class_out, wb_tile *tiles_out,
                     bool scan_only, ClassifyOut *out)
{
  ClassifyRun R;
  classify_prepare(R, t, t->ctx, corners, ncorners, p, d_class_out, tiles_out, scan_only, 0, out);
  if (!scan_only) classify_ground_single(R);
  classify_finish(R);
}

void wb_run_classify_batch(wb_ctx *c, wb_tree *const *trees, int ntrees, const double *corners,
                           const wb_classify_params *p, uint8_t *const *d_class_out,
                           ClassifyOut *outs)
{
  hipStream_t st = c->stream;
  std::vector<ClassifyRun> R(ntrees);
  uint64_t nbatch = 0;
  for (int k = 0; k < ntrees; k++) nbatch += trees[k]->n;
  for (int k = 0; k < ntrees; k++)
    classify_prepare(R[k], trees[k], c, corners + 6 * k, 2, p, d_class_out[k], nullptr, false,
                     nbatch, &outs[k]);
  // one launch of walk A over every tree's points, one of walk B and one of
  // the heavy kernel over what the trees' walks left; the counts stay on the
  // device
  std::vector<ClassifyArgs> AA(ntrees);
  std::vector<uint32_t> boff(ntrees + 1, 0);
  bool inside = true;  // every tree's points lie in their leaves' cubes
  bool cap = false;    // a tree's units are cut short
  for (int k = 0; k < ntrees; k++) {
    AA[k] = R[k].A;
    inside = inside && AA[k].cube_wedges;
    cap = cap || AA[k].open_budget != INT32_MAX;
    const uint64_t nb = boff[k] + (uint64_t)wb_blocks(R[k].n, AA[k].walk_per);
    if (nb > 0xffffffffull) throw std::string("too many points in one batch");
    boff[k + 1] = (uint32_t)nb;
  }
  ClassifyArgs *dAA = (ClassifyArgs *)wb_alloc(c, sizeof(ClassifyArgs) * ntrees);
  uint32_t *doff = (uint32_t *)wb_alloc(c, 4 * (ntrees + 1));
  const size_t nsum = (size_t)ntrees * OPEN_CLASSES + 1;
  uint32_t *dsum = (uint32_t *)wb_alloc(c, 4 * nsum);
  WB_CHECK(hipMemcpyAsync(dAA, AA.data(), sizeof(ClassifyArgs) * ntrees, hipMemcpyHostToDevice, st));
  WB_CHECK(hipMemcpyAsync(doff, boff.data(), 4 * (ntrees + 1), hipMemcpyHostToDevice, st));
  for (int k = 0; k < ntrees; k++) WB_CHECK(hipEventRecord(R[k].ev[4], st));
  if (boff[ntrees]) {
    const dim3 one(WAVE), ogrid(boff[ntrees] * (AA[0].walk_per / AA[0].open_per));
    if (inside) {
      hipLaunchKernelGGL((k_ground_batch<true, WB_GROUND_MINW>), dim3(boff[ntrees]), one, 0, st, dAA,
                         doff, ntrees);
      hipLaunchKernelGGL(k_batch_sums, dim3(1), one, 0, st, dAA, ntrees, 1, dsum);
      if (cap) hipLaunchKernelGGL((k_ground_open_batch<true, true>), ogrid, one, 0, st, dAA, dsum, ntrees);
      else hipLaunchKernelGGL((k_ground_open_batch<true, false>), ogrid, one, 0, st, dAA, dsum, ntrees);
    } else {
      hipLaunchKernelGGL((k_ground_batch<false, WB_GROUND_MINW>), dim3(boff[ntrees]), one, 0, st,
                         dAA, doff, ntrees);
      hipLaunchKernelGGL(k_batch_sums, dim3(1), one, 0, st, dAA, ntrees, 1, dsum);
      hipLaunchKernelGGL((k_ground_open_batch<false, true>), ogrid, one, 0, st, dAA, dsum, ntrees);
    }
  }
  for (int k = 0; k < ntrees; k++) {
    WB_CHECK(hipEventRecord(R[k].ev[5], st));
    WB_CHECK(hipEventRecord(R[k].ev[6], st));
  }
  if (boff[ntrees]) {
    hipLaunchKernelGGL(k_batch_sums, dim3(1), dim3(WAVE), 0, st, dAA, ntrees, 0, dsum);
    hipLaunchKernelGGL(k_ground_heavy_batch,
                       dim3((uint32_t)std::min<uint64_t>((uint64_t)boff[ntrees] * WAVE, HEAVY_GRID)),
                       dim3(64), 0, st, dAA, dsum, ntrees);
  }
  for (int k = 0; k < ntrees; k++) WB_CHECK(hipEventRecord(R[k].ev[7], st));
  // (the arguments' host copy is read until here)
  WB_CHECK(hipStreamSynchronize(st));
  wb_free(c, dAA, sizeof(ClassifyArgs) * ntrees);
  wb_free(c, doff, 4 * (ntrees + 1));
  wb_free(c, dsum, 4 * nsum);
  for (int k = 0; k < ntrees; k++) classify_finish(R[k]);
}
