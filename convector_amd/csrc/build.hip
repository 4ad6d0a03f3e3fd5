// build.hip -- the reference BVH build (bvh.rs:91-545) on gfx950.
//
// The tree is the one InterimNode::split_recursive builds: per node and per
// axis 64 centroid bins, replaced by bins of the stably sorted triangles when
// the node has at most 32 triangles or one bin holds more than n/8 of n > 64
// triangles; the cheapest split by the TreeSurfaceAreaHeuristic, ties to the
// first axis and the first position; no split when n*120 is cheaper; the
// child with the smaller surface area first.  crystallize's depth-first
// layout of sibling pairs is reproduced exactly.  The build also runs with
// 16 or 32 bins (bins.len() changed: at most bins/2 triangles or more than
// n/8 of n > bins in one bin take the sorted bins, in chunks of
// ceil(n/bins)); below, "32" stands for bins/2 and "64" for bins.
//
// Level-synchronous down to nodes of kSub triangles:
//   k_level_plan resets the next level's counters and lists the chunks of the
//     wide nodes;
//   k_decide (one workgroup per node) bins the three axes in LDS and picks
//     the split;
//   k_sort sorts the axes that fall back to sorted binning (stable LSD radix
//     sort, one workgroup per node and axis);
//   k_partition reorders the node's triangle references as the reference
//     collects them (stable by bin) and creates the children.
// A node of more than kWide triangles is split over chunks of references:
// k_bin_chunks bins each chunk into a partial, k_sum_chunks adds the partials
// up (counts and ordered-integer min / max, so the bins are exact), and
// k_part_chunks scatters the chunks and bounds their children, so that the
// top levels, where one node holds most triangles, use the whole GPU.
// k_subtree splits each node of at most kSub triangles down to nodes of at
// most bins/2 within one workgroup, and k_small finishes those, two per wave,
// with the triangles in the lanes.  k_depth and k_depth_lists list the inner nodes
// by depth; k_bottom_up counts leaves and the area ratio statistic, deepest
// depth first, and k_place puts every node where crystallize puts it, from the
// root down.
//
// The TreeSAH cost uses powf/log2f; their values for every triangle count are
// tabulated on the host with the C library so that near-ties resolve as in the
// reference.
#include <math.h>

#include <algorithm>
#include <exception>
#include <thread>
#include <type_traits>
#include <vector>

#include "internal.hpp"

namespace cvk {
namespace bvh {

constexpr uint32_t kLeaf = 1, kParity = 2, kIsC1 = 4, kPending = 8, kSplit = 16;
// an id that a small subtree reserved and did not use (no node)
constexpr uint32_t kHole = 32;
constexpr uint32_t kBlock = 512;
constexpr uint32_t kWide = 4096;    // nodes above this many triangles are chunked
constexpr uint32_t kSub = 1024;     // nodes of at most this many triangles go to k_subtree
constexpr uint32_t kLevelBatch = 4;   // levels enqueued between the host's looks at the lists
constexpr uint32_t kDepthFew = 2048;  // nodes of a depth that shares a launch with others
constexpr uint32_t kBinWords = 3 * 64 * 7;  // counts, then outer bounds, of 3 x 64 bins

struct INode {
  float box[6];   // outer: min.xyz, max.xyz
  float cbox[6];  // barycenter bounds (large nodes only)
  uint32_t begin, count;
  int32_t parent;
  int32_t child[2];
  uint32_t flags;
  uint32_t leaves;
  float sar;
  uint32_t depth;
  uint32_t axis, split_bin, left_count, uniform_mask;
  // chunks of a wide node in the level's chunk list and its row of `tot`
  uint32_t chunk_base, nchunks, slot;
  // k_place: nodes.len() when the node is crystallised (bvh.rs:389-428) and
  // the position of its first triangle
  uint32_t pairs, first_tri;
};

struct Ctx {
  uint32_t node_count;
  uint32_t large[2];      // nodes in the lists of the even and the odd levels
  uint32_t small_count;
  uint32_t error;
  uint32_t next_wide;     // wide nodes in the next level's list
  uint32_t wide_count;    // wide nodes and chunks of the current level
  uint32_t total_chunks;
  uint32_t sub_count;     // nodes for k_subtree
  uint32_t sub_levels;    // most levels that a subtree of k_subtree took
  uint32_t max_depth;
  uint32_t max_leaf;
  uint32_t root_box[6];   // okeys
  uint32_t root_cbox[6];  // okeys
};

struct Args {
  const float4* A;  // bmin.xyz, c.x
  const float4* B;  // bmax.xyz, c.y
  const float* C;   // c.z
  uint32_t* buf[2];
  uint32_t* sorted[3];
  uint32_t* tmp[3];
  INode* nodes;
  Ctx* ctx;
  const uint32_t* list;
  uint32_t parity;  // of the level: list holds ctx->large[parity] nodes
  uint32_t* next_list;
  uint32_t* sub_list;
  uint32_t* small_list;
  const float* tpm;   // powf(0.8f, log2f(n))
  const float* tpm1;  // powf(0.8f, log2f(n) - 1.0f)
  uint32_t mode;
  uint32_t ntris;
  uint32_t nbins;      // centroid bins per axis: 64 (the reference), 32 or 16
  uint32_t small_max;  // nodes of at most nbins / 2 triangles go to k_small
  // chunked wide nodes: the level's, per node its bins (kBinWords), and per
  // chunk the node, the bins and the children's bounds (2 sides x 12 okeys)
  uint32_t chunk;
  uint32_t* wide_list;
  uint32_t* tot;
  uint32_t* chunk_node;
  uint32_t* part;
  uint32_t* side;
};

__device__ __forceinline__ uint32_t okey(float f) {
  uint32_t u = f2u(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float okey_dec(uint32_t k) {
  return u2f((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
// Total-order min/max (the reference's f32::min / f32::max except that the
// kept zero's sign is fixed).
__device__ __forceinline__ float tmin_f(float a, float b) { return okey(b) < okey(a) ? b : a; }
__device__ __forceinline__ float tmax_f(float a, float b) { return okey(b) > okey(a) ? b : a; }
// Aabb::area (aabb.rs:97-103)
__device__ __forceinline__ float area6(const float* b) {
  float sx = b[3] - b[0], sy = b[4] - b[1], sz = b[5] - b[2];
  float x = sy * sz;
  float y = sz * sx;
  float z = sx * sy;
  return 2.0f * ((x + y) + z);
}
// Sort key of a barycenter coordinate; -0.0 == +0.0 as in partial_cmp.
__device__ __forceinline__ uint32_t sort_key(float c) { return okey(c == 0.0f ? 0.0f : c); }

__device__ __forceinline__ float centroid(const Args& a, uint32_t r, uint32_t axis) {
  return axis == 0 ? a.A[r].w : axis == 1 ? a.B[r].w : a.C[r];
}

// TreeSurfaceAreaHeuristic::aabb_cost (bvh.rs:452-469), constants 40/120/0.8.
__device__ __forceinline__ float tree_sah(const Args& a, float parent_area, const float* b,
                                          uint32_t n) {
  const float p = 0.8f;
  float ac_ap = area6(b) / parent_area;
  float nf = (float)n;
  float aabb_term = 1.0f + (ac_ap * (2.0f * p - nf * a.tpm[n])) / (p - (2.0f * p) * p);
  float tri_term = (nf * a.tpm1[n]) * ac_ap;
  return aabb_term * 40.0f + tri_term * 120.0f;
}

// centroid bin of bin_triangles (bvh.rs:149-156) with nb bins; NaN and nb
// clamp to nb - 1.
__device__ __forceinline__ uint32_t centroid_bin(float c, float mn, float size, uint32_t nb) {
  const float fb = (float)nb;
  float f = floorf((fb * (c - mn)) / size);
  return (f >= 0.0f && f < fb) ? (uint32_t)f : nb - 1u;
}

__device__ __forceinline__ uint32_t load_coherent(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void k_trefs(const float* v9, uint32_t n, float4* A, float4* B,
                                               float* C, uint32_t* buf0, Ctx* ctx) {
  __shared__ uint32_t sbox[12];
  if (threadIdx.x < 12) sbox[threadIdx.x] = (threadIdx.x % 6) < 3 ? 0xffffffffu : 0u;
  __syncthreads();
  uint32_t lb[12];
  for (int k = 0; k < 12; k++) lb[k] = (k % 6) < 3 ? 0xffffffffu : 0u;
  const float third = 1.0f / 3.0f;  // 3.0f32.recip()
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float* t = v9 + 9 * (size_t)i;
    float mn[3], mx[3], c[3];
    bool nan = false;
    for (int k = 0; k < 3; k++) {
      float x = t[k], y = t[3 + k], z = t[6 + k];
      nan |= (x != x) || (y != y) || (z != z);
      mn[k] = tmin_f(tmin_f(x, y), z);  // Aabb::enclose_points (aabb.rs:56-71)
      mx[k] = tmax_f(tmax_f(x, y), z);
      c[k] = ((x + y) + z) * third;  // Triangle::barycenter (triangle.rs:55-57)
    }
    if (nan) atomicOr(&ctx->error, 1u);
    A[i] = make_float4(mn[0], mn[1], mn[2], c[0]);
    B[i] = make_float4(mx[0], mx[1], mx[2], c[1]);
    C[i] = c[2];
    buf0[i] = i;
    for (int k = 0; k < 3; k++) {
      lb[k] = min(lb[k], okey(mn[k]));
      lb[3 + k] = max(lb[3 + k], okey(mx[k]));
      lb[6 + k] = min(lb[6 + k], okey(c[k]));
      lb[9 + k] = max(lb[9 + k], okey(c[k]));
    }
  }
  // (a wave's bounds first: 256 LDS atomics per value follow each other)
  for (int k = 0; k < 12; k++) {
    uint32_t v = lb[k];
    for (int off = 32; off > 0; off >>= 1) {
      const uint32_t w = __shfl_xor(v, off);
      v = (k % 6) < 3 ? min(v, w) : max(v, w);
    }
    if ((threadIdx.x & 63u) == 0) {
      if ((k % 6) < 3)
        atomicMin(&sbox[k], v);
      else
        atomicMax(&sbox[k], v);
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    uint32_t k = threadIdx.x;
    if (k < 3) {
      atomicMin(&ctx->root_box[k], sbox[k]);
      atomicMin(&ctx->root_cbox[k], sbox[6 + k]);
    } else {
      atomicMax(&ctx->root_box[k], sbox[k]);
      atomicMax(&ctx->root_cbox[k], sbox[6 + k]);
    }
  }
}

__global__ void k_root(INode* nodes, Ctx* ctx, uint32_t n) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  INode r;
  for (int k = 0; k < 6; k++) {
    r.box[k] = okey_dec(ctx->root_box[k]);
    r.cbox[k] = okey_dec(ctx->root_cbox[k]);
  }
  r.begin = 0;
  r.count = n;
  r.parent = -1;
  r.child[0] = r.child[1] = -1;
  r.flags = 0;
  r.leaves = 0;
  r.sar = 0.0f;
  r.depth = 0;
  r.axis = r.split_bin = r.left_count = r.uniform_mask = 0;
  r.chunk_base = r.nchunks = r.slot = r.pairs = r.first_tri = 0;
  nodes[0] = r;
  ctx->node_count = 1;
}

// The helpers below run on a group of BS threads: a workgroup, or (BS == 64)
// one wave of a workgroup of any size.
template <uint32_t BS>
__device__ __forceinline__ uint32_t group_tid() {
  return BS == 64 ? threadIdx.x & 63u : threadIdx.x;
}
// Orders the group's memory accesses; a wave's lanes run in step, so it needs
// the waits only.
template <uint32_t BS>
__device__ __forceinline__ void group_sync() {
  if (BS == 64) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// Grows a bin's bounds (LDS).  Few triangles of a bin move its bounds, and
// the atomics of many lanes on one bin follow each other, so a bound is read
// first (the reads of one bin are a broadcast) and left alone when the
// triangle lies within: a stale value is only further in, never past the
// bound, so nothing is missed.
__device__ __forceinline__ void grow_bin(uint32_t* b, const uint32_t* kmn, const uint32_t* kmx) {
  volatile uint32_t* v = b;
  for (int j = 0; j < 3; j++) {
    if (kmn[j] < v[j]) atomicMin(&b[j], kmn[j]);
    if (kmx[j] > v[3 + j]) atomicMax(&b[3 + j], kmx[j]);
  }
}

// Centroid bins of refs[0, n) on the axes not in umask (bin_triangles,
// bvh.rs:149-156): counts and outer bounds as ordered integers in LDS.
template <uint32_t BS>
__device__ __forceinline__ void bin_centroids(const Args& a, const uint32_t* refs, uint32_t n,
                                              const float* cmn, const float* csz, uint32_t umask,
                                              uint32_t (*cnt)[64], uint32_t (*bx)[64][6]) {
  for (uint32_t e = group_tid<BS>(); e < n; e += BS) {
    uint32_t r = refs[e];
    float4 A = a.A[r], B = a.B[r];
    float cz = a.C[r];
    float c[3] = {A.w, B.w, cz};
    uint32_t kmn[3] = {okey(A.x), okey(A.y), okey(A.z)};
    uint32_t kmx[3] = {okey(B.x), okey(B.y), okey(B.z)};
    for (uint32_t axis = 0; axis < 3; axis++) {
      if ((umask >> axis) & 1u) continue;
      uint32_t b = centroid_bin(c[axis], cmn[axis], csz[axis], a.nbins);
      atomicAdd(&cnt[axis][b], 1u);
      grow_bin(bx[axis][b], kmn, kmx);
    }
  }
}

template <uint32_t BS>
__device__ __forceinline__ void clear_bins(uint32_t (*cnt)[64], uint32_t (*bx)[64][6]) {
  for (uint32_t k = group_tid<BS>(); k < 3 * 64; k += BS) {
    (&cnt[0][0])[k] = 0;
    for (int j = 0; j < 6; j++) (&bx[0][0][0])[k * 6 + j] = j < 3 ? 0xffffffffu : 0u;
  }
}

// The cheapest split position of each axis (find_cheapest_split,
// bvh.rs:218-261): a wave per axis, or one wave axis by axis; one lane per
// position.  Lane i holds bin i, and the boxes and counts left of position i
// (bins below i) and right of it are scans over the lanes (ordered min / max
// and sums: any order gives the same values).  Every lane walking all 64 bins
// by itself and one thread comparing the costs took 52 us a launch on the
// levels of a 20,506-triangle build, the scans 13 us.
struct AxisSplits {
  float cost[3];
  uint32_t pos[3];   // 64: none
  uint32_t left[3];  // triangles left of pos
};
template <uint32_t BS>
__device__ __forceinline__ void axis_splits(const Args& a, float parent_area, uint32_t n,
                                            const uint32_t (*cnt)[64],
                                            const uint32_t (*bx)[64][6], AxisSplits* out) {
  for (uint32_t axis = group_tid<BS>() >> 6; axis < 3; axis += BS / 64) {
    const uint32_t i = threadIdx.x & 63u;
    const uint32_t ci = cnt[axis][i];
    const uint64_t ne = __ballot(ci != 0);
    const uint32_t first = __ffsll((unsigned long long)ne);  // first non-empty + 1
    const uint32_t last = 64 - __clzll((long long)ne);        // last non-empty + 1
    float pre[6], suf[6];
    uint32_t below = ci;
    for (int k = 0; k < 6; k++)
      pre[k] = suf[k] = ci ? okey_dec(bx[axis][i][k]) : k < 3 ? INFINITY : -INFINITY;
    for (uint32_t d = 1; d < 64; d <<= 1) {
      const uint32_t cu = __shfl_up(below, d);
      if (i >= d) below += cu;
      for (int k = 0; k < 6; k++) {
        const float up = __shfl_up(pre[k], d), dn = __shfl_down(suf[k], d);
        if (i >= d) pre[k] = k < 3 ? tmin_f(pre[k], up) : tmax_f(pre[k], up);
        if (i + d < 64) suf[k] = k < 3 ? tmin_f(suf[k], dn) : tmax_f(suf[k], dn);
      }
    }
    float lb[6];
    for (int k = 0; k < 6; k++) lb[k] = __shfl_up(pre[k], 1);
    below -= ci;
    float cst = 0.0f;
    bool in = __popcll(ne) > 1 && i >= first && i < last;
    if (in) cst = tree_sah(a, parent_area, lb, below) + tree_sah(a, parent_area, suf, n - below);
    // the reference scans the positions upward and replaces its choice only
    // by a strictly smaller cost, so that a NaN is chosen at the first
    // position only, and then for good
    uint32_t pos = 64;
    if (in && (cst == cst || i == first)) pos = i;
    const bool nan_first = __any(in && i == first && cst != cst);
    for (uint32_t d = 32; d > 0; d >>= 1) {
      const float cd = __shfl_xor(cst, d);
      const uint32_t pd = __shfl_xor(pos, d);
      if (pd < 64 && (pos == 64 || cd < cst || (cd == cst && pd < pos))) {
        cst = cd;
        pos = pd;
      }
    }
    if (nan_first) {
      pos = first;
      cst = NAN;
    }
    if (i == 0) {
      out->pos[axis] = pos;
      out->cost[axis] = cst;
    }
    if (i == pos) out->left[axis] = below;
  }
}

// The choice between the axes: the reference's scan order X, Y, Z, replaced
// only by a strictly smaller cost (bvh.rs:265-322).  -1: no axis splits.
__device__ __forceinline__ int choose_axis(const AxisSplits& s, float* best) {
  int axis = -1;
  for (int k = 0; k < 3; k++) {
    if (s.pos[k] >= 64) continue;
    if (axis < 0 || s.cost[k] < *best) {
      *best = s.cost[k];
      axis = k;
    }
  }
  return axis;
}

// Axes whose centroid bins fall back to sorted bins (bvh.rs:159-169): some
// bin above n / 8 with n > bins.  One wave.
__device__ __forceinline__ uint32_t fallback_axes(const Args& a, uint32_t n,
                                                  const uint32_t (*cnt)[64]) {
  uint32_t fb = 0;
  for (uint32_t axis = 0; axis < 3; axis++) {
    const uint64_t over = __ballot(cnt[axis][threadIdx.x & 63u] > n / 8);
    if (over && n > a.nbins) fb |= 1u << axis;
  }
  return fb;
}

// bin_triangles_uniform (bvh.rs:176-201): chunks of ceil(n/bins) of the
// stably sorted references of one axis.
template <uint32_t BS>
__device__ __forceinline__ void bin_sorted(const Args& a, const uint32_t* srt, uint32_t n,
                                           uint32_t* cnt, uint32_t (*bx)[6]) {
  const uint32_t tpb = (n + a.nbins - 1) / a.nbins;
  for (uint32_t s = group_tid<BS>(); s < n; s += BS) {
    const uint32_t r = srt[s];
    const float4 A = a.A[r], B = a.B[r];
    const uint32_t b = s / tpb;
    const uint32_t kmn[3] = {okey(A.x), okey(A.y), okey(A.z)};
    const uint32_t kmx[3] = {okey(B.x), okey(B.y), okey(B.z)};
    atomicAdd(&cnt[b], 1u);
    grow_bin(bx[b], kmn, kmx);
  }
}

// Start of a level: the next level's counters back to zero and the chunk
// list of the level's wide nodes.  One workgroup: the list in tiles of 1024
// nodes, a prefix sum of the chunk counts per tile, and the tile's chunk
// entries written by all threads.
__global__ __launch_bounds__(1024) void k_level_plan(Args a) {
  __shared__ uint32_t wsum[16];
  __shared__ uint32_t s_base, s_wide;
  __shared__ uint32_t t_end[1024], t_id[1024];  // the tile's wide nodes: last chunk + 1, id
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t nlist = a.ctx->large[a.parity];
  if (threadIdx.x == 0) s_base = s_wide = 0;
  __syncthreads();
  for (uint32_t i0 = 0; i0 < nlist; i0 += 1024) {
    const uint32_t i = i0 + threadIdx.x;
    uint32_t id = 0, nc = 0;
    if (i < nlist) {
      id = a.list[i];
      const uint32_t n = a.nodes[id].count;
      nc = n > kWide ? (n + a.chunk - 1) / a.chunk : 0u;
    }
    uint32_t inc = nc;
    for (uint32_t off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off);
      if (lane >= off) inc += y;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    uint32_t prior = 0, tile = 0;
    for (uint32_t w = 0; w < 16; w++) {
      prior += w < wave ? wsum[w] : 0u;
      tile += wsum[w];
    }
    t_end[threadIdx.x] = prior + inc;
    t_id[threadIdx.x] = id;
    if (i < nlist) {
      uint32_t slot = 0;
      if (nc) {
        slot = atomicAdd(&s_wide, 1u);
        a.wide_list[slot] = id;
      }
      a.nodes[id].chunk_base = s_base + prior + inc - nc;
      a.nodes[id].nchunks = nc;
      a.nodes[id].slot = slot;
    }
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < tile; t += 1024) {
      uint32_t lo = 0, hi = 1023;  // the first node whose chunks end above t
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (t_end[mid] > t)
          hi = mid;
        else
          lo = mid + 1;
      }
      a.chunk_node[s_base + t] = t_id[lo];
    }
    __syncthreads();
    if (threadIdx.x == 0) s_base += tile;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    a.ctx->total_chunks = s_base;
    a.ctx->wide_count = s_wide;
    a.ctx->large[a.parity ^ 1u] = 0;
    a.ctx->next_wide = 0;
  }
}

// Centroid bins of one chunk of a wide node into its partial.
__global__ __launch_bounds__(kBlock) void k_bin_chunks(Args a) {
  const uint32_t c = blockIdx.x;
  if (c >= a.ctx->total_chunks) return;
  const INode* nd = &a.nodes[a.chunk_node[c]];
  const uint32_t lo = (c - nd->chunk_base) * a.chunk;
  const uint32_t n = min(nd->count, lo + a.chunk) - lo;
  const uint32_t* refs = a.buf[(nd->flags & kParity) ? 1 : 0] + nd->begin + lo;
  __shared__ uint32_t cnt[3][64];
  __shared__ uint32_t bx[3][64][6];
  clear_bins<kBlock>(cnt, bx);
  __syncthreads();
  float cmn[3], csz[3];
  for (int k = 0; k < 3; k++) {
    cmn[k] = nd->cbox[k];
    csz[k] = nd->cbox[3 + k] - cmn[k];
  }
  bin_centroids<kBlock>(a, refs, n, cmn, csz, 0u, cnt, bx);
  __syncthreads();
  uint32_t* out = a.part + (size_t)c * kBinWords;
  for (uint32_t k = threadIdx.x; k < 3 * 64; k += kBlock) out[k] = (&cnt[0][0])[k];
  for (uint32_t k = threadIdx.x; k < 3 * 64 * 6; k += kBlock) out[192 + k] = (&bx[0][0][0])[k];
}

// The bins of the wide nodes: their chunks' partials added up, 64 words of
// one node per workgroup, every fourth chunk by each of its waves (integer
// sums and ordered min / max: any order gives the same bins; 16 loads are
// issued before they are combined).  One workgroup per node reading all
// partials took 208 us on a 1.33 M-triangle node, this and the split 45.
__global__ __launch_bounds__(256) void k_sum_chunks(Args a) {
  if (blockIdx.x >= a.ctx->wide_count) return;
  const INode* nd = &a.nodes[a.wide_list[blockIdx.x]];
  __shared__ uint32_t red[4][64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t k = blockIdx.y * 64 + lane, nch = nd->nchunks;
  const uint32_t* q = a.part + (size_t)nd->chunk_base * kBinWords + k;
  const int op = k < 192 ? 0 : ((k - 192) % 6) < 3 ? 1 : 2;  // sum, min, max
  auto acc = [&](uint32_t v, uint32_t w) {
    return op == 0 ? v + w : op == 1 ? min(v, w) : max(v, w);
  };
  const uint32_t none = op == 1 ? 0xffffffffu : 0u;
  uint32_t v = none;
  for (uint32_t c0 = wave; c0 < nch; c0 += 64) {
    uint32_t w[16];
#pragma unroll
    for (uint32_t j = 0; j < 16; j++)
      w[j] = c0 + 4 * j < nch ? q[(size_t)(c0 + 4 * j) * kBinWords] : none;
#pragma unroll
    for (uint32_t j = 0; j < 16; j++) v = acc(v, w[j]);
  }
  red[wave][lane] = v;
  __syncthreads();
  if (wave == 0)
    a.tot[(size_t)nd->slot * kBinWords + k] =
        acc(acc(red[0][lane], red[1][lane]), acc(red[2][lane], red[3][lane]));
}

// ---------------------------------------------------------------------------
// k_decide: bins + split choice for nodes of more than 32 triangles
// (InterimNode::split, bvh.rs:265-322).
// mode 0: centroid bins for all axes; a node whose binning falls back to
//         sorted bins on some axis is marked pending.
// mode 1: pending nodes only; sorted (uniform) bins from k_sort's output.
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(kBlock) void k_decide(Args a) {
  constexpr uint32_t BS = kBlock;
  if (blockIdx.x >= a.ctx->large[a.parity]) return;
  const uint32_t id = a.list[blockIdx.x];
  INode* nd = &a.nodes[id];
  const uint32_t flags = nd->flags;
  if (a.mode == 1 && !(flags & kPending)) return;
  const uint32_t n = nd->count, begin = nd->begin;
  const uint32_t* refs = a.buf[(flags & kParity) ? 1 : 0] + begin;
  const uint32_t umask = a.mode == 1 ? nd->uniform_mask : 0u;
  __shared__ uint32_t cnt[3][64];
  __shared__ uint32_t bx[3][64][6];
  __shared__ AxisSplits splits;
  __shared__ bool deferred;
  const uint32_t tid = threadIdx.x;
  const uint32_t nch = nd->nchunks;
  clear_bins<BS>(cnt, bx);
  __syncthreads();
  float cmn[3], csz[3];
  for (int k = 0; k < 3; k++) {
    cmn[k] = nd->cbox[k];
    csz[k] = nd->cbox[3 + k] - cmn[k];
  }
  if (nch) {
    // a wide node: k_sum_chunks has its bins
    const uint32_t* tot = a.tot + (size_t)nd->slot * kBinWords;
    for (uint32_t k = tid; k < kBinWords; k += BS) {
      const uint32_t axis = k < 192 ? k / 64 : (k - 192) / 384;
      if ((umask >> axis) & 1u) continue;
      if (k < 192)
        (&cnt[0][0])[k] = tot[k];
      else
        (&bx[0][0][0])[k - 192] = tot[k];
    }
  } else {
    bin_centroids<BS>(a, refs, n, cmn, csz, umask, cnt, bx);
  }
  if (umask) {
    for (uint32_t axis = 0; axis < 3; axis++)
      if ((umask >> axis) & 1u)
        bin_sorted<BS>(a, a.sorted[axis] + begin, n, cnt[axis], bx[axis]);
  }
  __syncthreads();
  if (a.mode == 0 && tid < 64) {
    const uint32_t fb = fallback_axes(a, n, cnt);
    if (fb && tid == 0) {
      nd->uniform_mask = fb;
      nd->flags = flags | kPending;
    }
    if (tid == 0) deferred = fb != 0;
  }
  __syncthreads();
  if (a.mode == 0 && deferred) return;
  axis_splits<BS>(a, area6(nd->box), n, cnt, bx, &splits);
  __syncthreads();
  if (tid == 0) {
    float best = 0.0f;
    const int best_axis = choose_axis(splits, &best);
    uint32_t f = flags & ~kPending;
    if (best_axis < 0) {
      atomicOr(&a.ctx->error, 2u);  // assert!(!is_first), bvh.rs:303
      f |= kLeaf;
    } else if ((float)n * 120.0f < best) {
      f |= kLeaf;  // bvh.rs:311-314
    } else {
      nd->axis = (uint32_t)best_axis;
      nd->split_bin = splits.pos[best_axis];
      nd->left_count = splits.left[best_axis];
      if (a.mode == 0) nd->uniform_mask = 0;
      f |= kSplit;
    }
    nd->flags = f;
  }
}

// ---------------------------------------------------------------------------
// Stable counting-sort pass of a segment inside one workgroup: elements are
// taken in tiles of BS in order; within a tile a lane's rank among equal
// digits comes from ballots, across waves from LDS counts.  Digit d starts
// at start[d] when start is given (a chunk of a larger sort), else after
// the segment's smaller digits.
// ---------------------------------------------------------------------------

template <int BITS, uint32_t BS, typename DigitFn, typename LoadFn>
__device__ __forceinline__ void wg_stable_pass(uint32_t n, LoadFn load, DigitFn digit_of,
                                               uint32_t* dst, uint32_t* hist, uint32_t* wcount,
                                               const uint32_t* start = nullptr) {
  constexpr uint32_t R = 1u << BITS;
  constexpr uint32_t W = BS / 64;
  const uint32_t tid = group_tid<BS>(), lane = tid & 63, wave = tid >> 6;
  if (start) {
    for (uint32_t k = tid; k < R; k += BS) hist[k] = start[k];
  } else {
    for (uint32_t k = tid; k < R; k += BS) hist[k] = 0;
    group_sync<BS>();
    for (uint32_t e = tid; e < n; e += BS) atomicAdd(&hist[digit_of(load(e))], 1u);
    group_sync<BS>();
    if (tid < 64) {  // exclusive prefix sums, R / 64 digits a lane
      constexpr uint32_t E = R / 64;
      uint32_t c[E], own = 0;
      for (uint32_t k = 0; k < E; k++) {
        c[k] = own;
        own += hist[tid * E + k];
      }
      uint32_t inc = own;
      for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(inc, d);
        if (lane >= d) inc += y;
      }
      for (uint32_t k = 0; k < E; k++) hist[tid * E + k] = c[k] + inc - own;
    }
  }
  for (uint32_t k = tid; k < W * R; k += BS) wcount[k] = 0;
  group_sync<BS>();
  const uint64_t lt = (1ull << lane) - 1ull;
  for (uint32_t t0 = 0; t0 < n; t0 += BS) {
    uint32_t e = t0 + tid;
    bool valid = e < n;
    uint32_t v = valid ? load(e) : 0u;
    uint32_t d = valid ? digit_of(v) : 0u;
    uint64_t match = __ballot(valid);
    for (int b = 0; b < BITS; b++) {
      uint64_t m = __ballot((d >> b) & 1u);
      match &= ((d >> b) & 1u) ? m : ~m;
    }
    uint32_t rank = __popcll(match & lt);
    if (valid && rank == 0) wcount[wave * R + d] = __popcll(match);
    group_sync<BS>();
    if (valid) {
      uint32_t prior = 0;
      for (uint32_t w = 0; w < wave; w++) prior += wcount[w * R + d];
      dst[hist[d] + prior + rank] = v;
    }
    group_sync<BS>();
    for (uint32_t k = tid; k < R; k += BS) {
      uint32_t s = 0;
      for (uint32_t w = 0; w < W; w++) {
        s += wcount[w * R + k];
        wcount[w * R + k] = 0;
      }
      hist[k] += s;
    }
    group_sync<BS>();
  }
}

// Sorted binning input: a stable sort of the segment by barycenter
// coordinate (bvh.rs:176-190), as 4 stable 8-bit LSD passes.
__global__ __launch_bounds__(kBlock) void k_sort(Args a) {
  if (blockIdx.x / 3 >= a.ctx->large[a.parity]) return;
  const uint32_t id = a.list[blockIdx.x / 3];
  const uint32_t axis = blockIdx.x % 3;
  const INode* nd = &a.nodes[id];
  if (!(nd->flags & kPending) || !((nd->uniform_mask >> axis) & 1u)) return;
  const uint32_t n = nd->count, begin = nd->begin;
  const uint32_t* refs = a.buf[(nd->flags & kParity) ? 1 : 0] + begin;
  uint32_t* X = a.tmp[axis] + begin;
  uint32_t* Y = a.sorted[axis] + begin;
  __shared__ uint32_t hist[256];
  __shared__ uint32_t wcount[(kBlock / 64) * 256];
  for (int pass = 0; pass < 4; pass++) {
    const uint32_t* src = pass == 0 ? refs : (pass & 1) ? X : Y;
    uint32_t* dst = (pass & 1) ? Y : X;
    const uint32_t shift = 8 * pass;
    auto load = [&](uint32_t e) { return pass == 0 ? src[e] : load_coherent(src + e); };
    auto digit = [&](uint32_t r) { return (sort_key(centroid(a, r, axis)) >> shift) & 255u; };
    wg_stable_pass<8, kBlock>(n, load, digit, dst, hist, wcount);
    __threadfence();
    __syncthreads();
  }
}

// Outer and barycenter bounds of the two children over order[lo, hi) (side
// 0: position below L when uniform, else bin below split), reduced into
// cb (LDS, initialised by the caller) with one atomic per wave and value.
template <uint32_t BS, typename BinFn>
__device__ __forceinline__ void side_bounds(const Args& a, const uint32_t* order, uint32_t lo,
                                            uint32_t hi, bool uniform, uint32_t L, uint32_t split,
                                            BinFn bin_of, uint32_t (*cb)[12]) {
  uint32_t lk[2][12];
  for (int s = 0; s < 2; s++)
    for (int k = 0; k < 12; k++) lk[s][k] = (k % 6) < 3 ? 0xffffffffu : 0u;
  for (uint32_t e = lo + group_tid<BS>(); e < hi; e += BS) {
    uint32_t r = order[e];
    int side = uniform ? (e < L ? 0 : 1) : (bin_of(r) < split ? 0 : 1);
    float4 A = a.A[r], B = a.B[r];
    float cz = a.C[r];
    uint32_t* l = lk[side];
    l[0] = min(l[0], okey(A.x));
    l[1] = min(l[1], okey(A.y));
    l[2] = min(l[2], okey(A.z));
    l[3] = max(l[3], okey(B.x));
    l[4] = max(l[4], okey(B.y));
    l[5] = max(l[5], okey(B.z));
    l[6] = min(l[6], okey(A.w));
    l[7] = min(l[7], okey(B.w));
    l[8] = min(l[8], okey(cz));
    l[9] = max(l[9], okey(A.w));
    l[10] = max(l[10], okey(B.w));
    l[11] = max(l[11], okey(cz));
  }
  for (int s = 0; s < 2; s++)
    for (int k = 0; k < 12; k++) {
      uint32_t v = lk[s][k];
      // wave reduction first to cut LDS atomics
      for (int off = 32; off > 0; off >>= 1) {
        uint32_t o = __shfl_xor(v, off);
        v = (k % 6) < 3 ? min(v, o) : max(v, o);
      }
      if ((threadIdx.x & 63u) == 0) {
        if ((k % 6) < 3)
          atomicMin(&cb[s][k], v);
        else
          atomicMax(&cb[s][k], v);
      }
    }
  group_sync<BS>();
}

// One chunk of a wide node that splits: its references go behind those of
// smaller bins and of earlier chunks' same bin (a stable sort by bin, or the
// sorted order's copy for a uniform axis), and its part of the children's
// bounds to its side partial.  Every chunk adds up the counts of the chunks
// before it, 8 waves sharing them: reading on average half of a node's counts
// per chunk costs less than a scan of its own (60 us in one workgroup at
// 1.33 M triangles).  The reads grow with the square of the chunks: about 35 GB
// of a 24 M-triangle build, which takes 107 ms on the device (286 when a scan
// placed the chunks and the levels were launched node by node).
__global__ __launch_bounds__(kBlock) void k_part_chunks(Args a) {
  const uint32_t c = blockIdx.x;
  if (c >= a.ctx->total_chunks) return;
  const INode* nd = &a.nodes[a.chunk_node[c]];
  if (!(nd->flags & kSplit)) return;
  const uint32_t n = nd->count, begin = nd->begin;
  const uint32_t lo = (c - nd->chunk_base) * a.chunk, hi = min(n, lo + a.chunk);
  const uint32_t par = (nd->flags & kParity) ? 1u : 0u;
  const uint32_t* src = a.buf[par] + begin;
  uint32_t* dst = a.buf[par ^ 1u] + begin;
  const uint32_t axis = nd->axis, split = nd->split_bin, L = nd->left_count;
  const bool uniform = (nd->uniform_mask >> axis) & 1u;
  __shared__ uint32_t hist[64];
  __shared__ uint32_t wcount[(kBlock / 64) * 64];
  __shared__ uint32_t cb[2][12];
  const uint32_t tid = threadIdx.x;
  if (tid < 24) (&cb[0][0])[tid] = ((tid % 12) % 6) < 3 ? 0xffffffffu : 0u;
  __syncthreads();
  const float mn = nd->cbox[axis], size = nd->cbox[3 + axis] - mn;
  auto bin_of = [&](uint32_t r) {
    return centroid_bin(centroid(a, r, axis), mn, size, a.nbins);
  };
  if (uniform) {
    const uint32_t* srt = a.sorted[axis] + begin;
    for (uint32_t s = lo + tid; s < hi; s += kBlock) dst[s] = srt[s];
  } else {
    __shared__ uint32_t start[64];
    __shared__ uint32_t before[kBlock / 64][64];
    const uint32_t lane = tid & 63u, wave = tid >> 6, prior = c - nd->chunk_base;
    const uint32_t* q = a.part + (size_t)nd->chunk_base * kBinWords + axis * 64 + lane;
    uint32_t sum = 0;
    for (uint32_t c0 = wave; c0 < prior; c0 += 8 * (kBlock / 64)) {
      uint32_t v[8];
#pragma unroll
      for (uint32_t j = 0; j < 8; j++) {
        const uint32_t k = c0 + j * (kBlock / 64);
        v[j] = k < prior ? q[(size_t)k * kBinWords] : 0u;
      }
#pragma unroll
      for (uint32_t j = 0; j < 8; j++) sum += v[j];
    }
    before[wave][lane] = sum;
    __syncthreads();
    if (wave == 0) {
      const uint32_t own = a.tot[(size_t)nd->slot * kBinWords + axis * 64 + lane];
      uint32_t inc = own;
      for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(inc, d);
        if (lane >= d) inc += y;
      }
      inc -= own;
      for (uint32_t w = 0; w < kBlock / 64; w++) inc += before[w][lane];
      start[lane] = inc;
    }
    __syncthreads();
    auto load = [&](uint32_t e) { return src[lo + e]; };
    wg_stable_pass<6, kBlock>(hi - lo, load, bin_of, dst, hist, wcount, start);
  }
  side_bounds<kBlock>(a, uniform ? a.sorted[axis] + begin : src, lo, hi, uniform, L, split, bin_of,
                     cb);
  if (tid < 24) a.side[(size_t)c * 24 + tid] = (&cb[0][0])[tid];
}

// The two children of a node split at left_count, with their bounds from cb
// (per side: outer min.xyz max.xyz, barycenter min.xyz max.xyz as okeys).
// Returns the first child's id.  One thread.
__device__ __forceinline__ uint32_t make_children(const Args& a, INode* nd, uint32_t id,
                                                  const uint32_t (*cb)[12]) {
  const uint32_t c = atomicAdd(&a.ctx->node_count, 2u);
  const uint32_t L = nd->left_count, n = nd->count;
  const uint32_t par = (nd->flags & kParity) ? 1u : 0u;
  INode ch[2];
  for (int s = 0; s < 2; s++) {
    for (int k = 0; k < 6; k++) {
      ch[s].box[k] = okey_dec(cb[s][k]);
      ch[s].cbox[k] = okey_dec(cb[s][6 + k]);
    }
    ch[s].begin = nd->begin + (s == 0 ? 0 : L);
    ch[s].count = s == 0 ? L : n - L;
    ch[s].parent = (int32_t)id;
    ch[s].child[0] = ch[s].child[1] = -1;
    ch[s].flags = (par ^ 1u) ? kParity : 0u;
    ch[s].leaves = 0;
    ch[s].sar = 0.0f;
    ch[s].depth = nd->depth + 1;
    ch[s].axis = ch[s].split_bin = ch[s].left_count = ch[s].uniform_mask = 0;
    ch[s].chunk_base = ch[s].nchunks = ch[s].slot = ch[s].pairs = ch[s].first_tri = 0;
  }
  // smaller area first (bvh.rs:337-345)
  const bool swap = area6(ch[0].box) > area6(ch[1].box);
  ch[swap ? 0 : 1].flags |= kIsC1;
  for (int s = 0; s < 2; s++) {
    if (ch[s].count == 1) ch[s].flags |= kLeaf;
    a.nodes[c + s] = ch[s];
  }
  nd->child[0] = (int32_t)(swap ? c + 1 : c);
  nd->child[1] = (int32_t)(swap ? c : c + 1);
  return c;
}

// Reorders the segment as split() collects the children (bins in order,
// references in push order) and creates the children.
__global__ __launch_bounds__(kBlock) void k_partition(Args a) {
  constexpr uint32_t BS = kBlock;
  if (blockIdx.x >= a.ctx->large[a.parity]) return;
  const uint32_t id = a.list[blockIdx.x];
  INode* nd = &a.nodes[id];
  const uint32_t flags = nd->flags;
  if (!(flags & kSplit)) return;
  const uint32_t n = nd->count, begin = nd->begin;
  const uint32_t par = (flags & kParity) ? 1u : 0u;
  const uint32_t* src = a.buf[par] + begin;
  uint32_t* dst = a.buf[par ^ 1u] + begin;
  const uint32_t axis = nd->axis, split = nd->split_bin, L = nd->left_count;
  const bool uniform = (nd->uniform_mask >> axis) & 1u;
  __shared__ uint32_t hist[64];
  __shared__ uint32_t wcount[(BS / 64) * 64];
  __shared__ uint32_t cb[2][12];  // per side: outer min.xyz max.xyz, barycenter min.xyz max.xyz
  const uint32_t tid = threadIdx.x;
  if (tid < 24) (&cb[0][0])[tid] = ((tid % 12) % 6) < 3 ? 0xffffffffu : 0u;
  __syncthreads();
  const float mn = nd->cbox[axis], size = nd->cbox[3 + axis] - mn;
  auto bin_of = [&](uint32_t r) {
    return centroid_bin(centroid(a, r, axis), mn, size, a.nbins);
  };
  if (nd->nchunks) {
    // a wide node: k_part_chunks reordered it; its chunks' bounds are added
    // up here
    // (ordered min / max: any order gives the same bounds; BS / 32 groups of
    // 24 lanes take every (BS / 32)-th chunk, then 24 lanes combine them)
    const uint32_t* sp = a.side + (size_t)nd->chunk_base * 24;
    __shared__ uint32_t red[BS / 32][24];
    const uint32_t k = tid % 24, g = tid / 24;  // 21 groups of 24 lanes
    const bool lo = ((k % 12) % 6) < 3;
    if (g < BS / 32) {
      uint32_t v = lo ? 0xffffffffu : 0u;
      for (uint32_t c = g; c < nd->nchunks; c += BS / 32) {
        const uint32_t w = sp[(size_t)c * 24 + k];
        v = lo ? min(v, w) : max(v, w);
      }
      red[g][k] = v;
    }
    __syncthreads();
    if (tid < 24) {
      uint32_t v = lo ? 0xffffffffu : 0u;
      for (uint32_t j = 0; j < BS / 32; j++) v = lo ? min(v, red[j][tid]) : max(v, red[j][tid]);
      (&cb[0][0])[tid] = v;
    }
    __syncthreads();
  } else {
    if (uniform) {
      const uint32_t* srt = a.sorted[axis] + begin;
      for (uint32_t s = tid; s < n; s += BS) dst[s] = srt[s];
    } else {
      auto load = [&](uint32_t e) { return src[e]; };
      wg_stable_pass<6, BS>(n, load, bin_of, dst, hist, wcount);
    }
    side_bounds<BS>(a, uniform ? a.sorted[axis] + begin : src, 0, n, uniform, L, split, bin_of, cb);
  }
  if (tid == 0) {
    const uint32_t c = make_children(a, nd, id, cb);
    for (uint32_t s = 0; s < 2; s++) {
      const uint32_t count = s == 0 ? L : n - L;
      if (count > kSub) {
        a.next_list[atomicAdd(&a.ctx->large[a.parity ^ 1u], 1u)] = c + s;
        if (count > kWide) atomicAdd(&a.ctx->next_wide, 1u);
      } else if (count > a.small_max) {
        a.sub_list[atomicAdd(&a.ctx->sub_count, 1u)] = c + s;
      } else if (count >= 2) {
        a.small_list[atomicAdd(&a.ctx->small_count, 1u)] = c + s;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// k_subtree: one workgroup of kSubWaves waves splits a node of at most kSub
// triangles down to nodes of at most bins/2, level by level within the workgroup:
// the whole workgroup per node of more than kSubWide triangles, then a wave
// per node for the rest; a node's bins, the sorts of axes that fall back to
// sorted bins, its split and its partition follow each other.  Bound by the
// latency of the passes over a node's references; a launch per pass and level
// for the whole tree, with 512-thread workgroups for nodes of a few hundred
// triangles, took 4.5 ms for 1.33 M triangles, this 1.6 ms.
// ---------------------------------------------------------------------------
constexpr uint32_t kSubWaves = 8;
constexpr uint32_t kSubWide = 256;
constexpr uint32_t kSubList = kSub / 9 + 1;  // nodes of more than 8 triangles (16 bins)

struct SubWork {
  uint32_t cnt[3][64];
  uint32_t bx[3][64][6];
  uint32_t hist[256];
  uint32_t cb[2][12];
  AxisSplits splits;
};

// Splits node id with BS threads; children of more than small_max triangles
// join `next`.
template <uint32_t BS>
__device__ __forceinline__ void split_node(const Args& a, uint32_t id, SubWork& w,
                                           uint32_t* wcount, uint32_t* next, uint32_t* nnext) {
  const uint32_t tid = group_tid<BS>();
  INode* nd = &a.nodes[id];
  const uint32_t n = __builtin_amdgcn_readfirstlane(nd->count);
  const uint32_t begin = __builtin_amdgcn_readfirstlane(nd->begin);
  const uint32_t flags = __builtin_amdgcn_readfirstlane(nd->flags);
  const uint32_t par = (flags & kParity) ? 1u : 0u;
  const uint32_t* src = a.buf[par] + begin;
  uint32_t* dst = a.buf[par ^ 1u] + begin;
  float cmn[3], csz[3];
  for (int j = 0; j < 3; j++) {
    cmn[j] = nd->cbox[j];
    csz[j] = nd->cbox[3 + j] - cmn[j];
  }
  const float area = area6(nd->box);
  clear_bins<BS>(w.cnt, w.bx);
  if (tid < 24) (&w.cb[0][0])[tid] = ((tid % 12) % 6) < 3 ? 0xffffffffu : 0u;
  group_sync<BS>();
  bin_centroids<BS>(a, src, n, cmn, csz, 0u, w.cnt, w.bx);
  group_sync<BS>();
  const uint32_t umask = fallback_axes(a, n, w.cnt);
  for (uint32_t axis = 0; axis < 3; axis++) {
    if (!((umask >> axis) & 1u)) continue;
    uint32_t* X = a.tmp[axis] + begin;
    uint32_t* Y = a.sorted[axis] + begin;
    for (uint32_t pass = 0; pass < 4; pass++) {
      const uint32_t* from = pass == 0 ? src : (pass & 1) ? X : Y;
      uint32_t* to = (pass & 1) ? Y : X;
      auto load = [&](uint32_t e) { return from[e]; };
      auto digit = [&](uint32_t r) {
        return (sort_key(centroid(a, r, axis)) >> (8 * pass)) & 255u;
      };
      wg_stable_pass<8, BS>(n, load, digit, to, w.hist, wcount);
      group_sync<BS>();
    }
    for (uint32_t k = tid; k < 64; k += BS) {
      w.cnt[axis][k] = 0;
      for (int j = 0; j < 6; j++) w.bx[axis][k][j] = j < 3 ? 0xffffffffu : 0u;
    }
    group_sync<BS>();
    bin_sorted<BS>(a, Y, n, w.cnt[axis], w.bx[axis]);
    group_sync<BS>();
  }
  axis_splits<BS>(a, area, n, w.cnt, w.bx, &w.splits);
  group_sync<BS>();
  float best = 0.0f;
  const int axis = choose_axis(w.splits, &best);
  if (axis < 0 || (float)n * 120.0f < best) {
    if (tid == 0) {
      if (axis < 0) atomicOr(&a.ctx->error, 2u);  // assert!(!is_first), bvh.rs:303
      nd->flags = flags | kLeaf;                  // bvh.rs:311-314
    }
    return;
  }
  const uint32_t L = __builtin_amdgcn_readfirstlane(w.splits.left[axis]);
  const float mn = nd->cbox[axis], size = nd->cbox[3 + axis] - mn;
  auto bin_of = [&](uint32_t r) {
    return centroid_bin(centroid(a, r, (uint32_t)axis), mn, size, a.nbins);
  };
  if ((umask >> axis) & 1u) {
    const uint32_t* srt = a.sorted[axis] + begin;
    for (uint32_t e = tid; e < n; e += BS) dst[e] = srt[e];
  } else {
    auto load = [&](uint32_t e) { return src[e]; };
    wg_stable_pass<6, BS>(n, load, bin_of, dst, w.hist, wcount);
  }
  group_sync<BS>();
  side_bounds<BS>(a, dst, 0, n, true, L, 0u, bin_of, w.cb);
  if (tid == 0) {
    nd->left_count = L;
    nd->flags = flags | kSplit;
    const uint32_t c = make_children(a, nd, id, w.cb);
    for (uint32_t s = 0; s < 2; s++) {
      const uint32_t cn = s == 0 ? L : n - L;
      if (cn > a.small_max)
        next[atomicAdd(nnext, 1u)] = c + s;
      else if (cn >= 2)
        a.small_list[atomicAdd(&a.ctx->small_count, 1u)] = c + s;
    }
  }
}

__global__ __launch_bounds__(64 * kSubWaves) void k_subtree(Args a) {
  __shared__ SubWork work[kSubWaves];
  __shared__ uint32_t wcount[kSubWaves * 256];
  __shared__ uint32_t list[2][kSubList];
  __shared__ uint32_t count[2];
  if (blockIdx.x >= a.ctx->sub_count || (a.ctx->error & 1u)) return;
  const uint32_t wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) {
    list[0][0] = a.sub_list[blockIdx.x];
    count[0] = 1;
    count[1] = 0;
  }
  __syncthreads();
  uint32_t levels = 0;
  for (uint32_t cur = 0;; cur ^= 1u, levels++) {
    const uint32_t nodes = count[cur];
    if (nodes == 0) break;
    uint32_t* next = list[cur ^ 1u];
    for (uint32_t k = 0; k < nodes; k++) {
      const uint32_t id = __builtin_amdgcn_readfirstlane(list[cur][k]);
      if (__builtin_amdgcn_readfirstlane(a.nodes[id].count) <= kSubWide) continue;
      split_node<64 * kSubWaves>(a, id, work[0], wcount, next, &count[cur ^ 1u]);
      __syncthreads();
    }
    for (uint32_t k = wave; k < nodes; k += kSubWaves) {
      const uint32_t id = __builtin_amdgcn_readfirstlane(list[cur][k]);
      if (__builtin_amdgcn_readfirstlane(a.nodes[id].count) > kSubWide) continue;
      split_node<64>(a, id, work[wave], wcount + wave * 256, next, &count[cur ^ 1u]);
      group_sync<64>();
    }
    __syncthreads();
    if (threadIdx.x == 0) count[cur] = 0;
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicMax(&a.ctx->sub_levels, levels);
}

// ---------------------------------------------------------------------------
// k_small: finishes the subtrees of nodes of 2..32 triangles, two per wave (32
// lanes each), breadth first: the lanes hold the triangles of all nodes of one
// depth, each node a segment [off, off + cnt) of consecutive lanes, and every
// sort and scan runs over all segments at once.  With at most 32 triangles
// every split uses sorted single-triangle bins (bvh.rs:145-147), so a depth is
// three sorts of the lanes and two scans.  A sort ranks each lane within its
// segment by its key (ties by lane: the stable order), and one ds_permute
// sends every lane to its rank; lanes of finished nodes keep their place.
// Bound by the latency of the lane exchanges: node after node in depth-first
// order, one subtree a wave, took 7.06 ms for 1.33 M triangles and 490 us for
// 20,506, now 0.65 ms and 128 us.
// ---------------------------------------------------------------------------

// tree_sah with the power terms of counts up to 32 from LDS
__device__ __forceinline__ float tree_sah_small(const float (*tp)[33], float parent_area,
                                                const float* b, uint32_t n) {
  const float p = 0.8f;
  float ac_ap = area6(b) / parent_area;
  float nf = (float)n;
  float aabb_term = 1.0f + (ac_ap * (2.0f * p - nf * tp[0][n])) / (p - (2.0f * p) * p);
  float tri_term = (nf * tp[1][n]) * ac_ap;
  return aabb_term * 40.0f + tri_term * 120.0f;
}

__global__ __launch_bounds__(256) void k_small(Args a) {
  const uint32_t lane = threadIdx.x & 63, half = lane >> 5;
  __shared__ float tp[2][33];
  if (blockIdx.x * 8 >= a.ctx->small_count || a.ctx->error) return;
  if (threadIdx.x < 66) {
    const uint32_t k = threadIdx.x % 33;
    tp[threadIdx.x / 33][k] = k <= a.ntris ? (threadIdx.x < 33 ? a.tpm[k] : a.tpm1[k]) : 0.0f;
  }
  __syncthreads();
  const uint32_t si = blockIdx.x * 8 + (threadIdx.x >> 5);
  const bool here = si < a.ctx->small_count;
  uint32_t root = 0, n = 0, sbegin = 0, rflags = 0, depth = 0;
  int32_t parent = -1;
  float box[6] = {0, 0, 0, 0, 0, 0};
  if (here) {
    root = a.small_list[si];
    const INode& R = a.nodes[root];
    n = R.count;
    sbegin = R.begin;
    rflags = R.flags;
    parent = R.parent;
    depth = R.depth;
    for (int k = 0; k < 6; k++) box[k] = R.box[k];
  }
  const uint32_t par = rflags & kParity;
  uint32_t* seg = a.buf[par ? 1 : 0] + sbegin;
  const uint32_t pos = lane & 31u;
  uint32_t ref = 0;
  float bmn[3] = {0, 0, 0}, bmx[3] = {0, 0, 0}, c[3] = {0, 0, 0};
  bool open = here && pos < n;
  if (open) {
    ref = seg[pos];
    float4 A = a.A[ref], B = a.B[ref];
    bmn[0] = A.x; bmn[1] = A.y; bmn[2] = A.z;
    bmx[0] = B.x; bmx[1] = B.y; bmx[2] = B.z;
    c[0] = A.w; c[1] = B.w; c[2] = a.C[ref];
  }
  // The subtree has at most n - 1 inner nodes, so its nodes take ids from
  // 2 (n - 1) reserved with one atomic (one counter for every node would
  // serialise them); ids left over are written as holes at the end.
  uint32_t ids = 0;
  if (here && pos == 0) ids = atomicAdd(&a.ctx->node_count, 2u * (n - 1u));
  ids = __shfl(ids, (int)(half << 5));
  const uint32_t ids_end = here ? ids + 2u * (n - 1u) : ids;
  // the lane's node
  uint32_t off = open ? half << 5 : lane, cnt = open ? n : 0u, id = root, flags = rflags;
  auto write_node = [&](uint32_t f, int32_t c0, int32_t c1) {
    INode& w = a.nodes[id];
    for (int k = 0; k < 6; k++) w.box[k] = box[k];
    w.begin = sbegin + (off & 31u);
    w.count = cnt;
    w.parent = parent;
    w.child[0] = c0;
    w.child[1] = c1;
    w.flags = f;
    w.depth = depth;
  };
  for (; __any(open); depth++) {
    if (open && cnt == 1) {
      write_node(flags | kLeaf, -1, -1);
      open = false;
    }
    uint32_t most = open ? cnt : 0u;
    for (int o = 32; o > 0; o >>= 1) most = max(most, (uint32_t)__shfl_xor(most, o));
    most = __builtin_amdgcn_readfirstlane(most);
    if (most == 0) break;
    const uint32_t at = lane - off;  // position in the segment
    const float parent_area = area6(box);
    int best_axis = -1;
    uint32_t best_i = 0, best_src = lane;
    float best = 0.0f;
    float lb[6], rb[6];  // the best axis' prefix and suffix boxes at this lane
    for (int k = 0; k < 6; k++) lb[k] = rb[k] = 0.0f;
    for (uint32_t axis = 0; axis < 3; axis++) {
      const uint32_t key = sort_key(axis == 0 ? c[0] : axis == 1 ? c[1] : c[2]);
      uint32_t rank = 0;
      for (uint32_t j = 0; j < most; j++) {
        const uint32_t kj = __shfl(key, (int)(off + j));  // wraps beyond the wave: not used
        rank += j < cnt && (kj < key || (kj == key && j < at)) ? 1u : 0u;
      }
      // lane off + rank receives this lane's index: the source of each
      // sorted position
      const uint32_t src = (uint32_t)__builtin_amdgcn_ds_permute(
          (int)((open ? off + rank : lane) * 4), (int)lane);
      float pre[6], suf[6];
      for (int k = 0; k < 3; k++) {
        pre[k] = suf[k] = __shfl(bmn[k], (int)src);
        pre[3 + k] = suf[3 + k] = __shfl(bmx[k], (int)src);
      }
      for (uint32_t d = 1; d < most; d <<= 1)
        for (int k = 0; k < 6; k++) {
          const float up = __shfl_up(pre[k], d), dn = __shfl_down(suf[k], d);
          if (at >= d) pre[k] = k < 3 ? tmin_f(pre[k], up) : tmax_f(pre[k], up);
          if (at + d < cnt) suf[k] = k < 3 ? tmin_f(suf[k], dn) : tmax_f(suf[k], dn);
        }
      float rsuf[6];
      for (int k = 0; k < 6; k++) rsuf[k] = __shfl_down(suf[k], 1);
      // the cost of splitting after this lane, and its position (0: none);
      // the reference scans the positions upward and replaces its choice only
      // by a strictly smaller cost, so that a NaN is chosen at the first
      // position only
      float cst = 0.0f;
      uint32_t pick = 0;
      if (open && at + 1 < cnt) {
        cst = tree_sah_small(tp, parent_area, pre, at + 1) +
              tree_sah_small(tp, parent_area, rsuf, cnt - at - 1);
        pick = at == 0 || cst == cst ? at + 1 : 0u;
      }
      for (uint32_t d = 1; d < most; d <<= 1) {
        const float cd = __shfl_down(cst, d);
        const uint32_t pd = __shfl_down(pick, d);
        if (at + d < cnt && pd && (!pick || cd < cst)) {
          cst = cd;
          pick = pd;
        }
      }
      const float acost = __shfl(cst, (int)off);
      const uint32_t apick = __shfl(pick, (int)off);
      if (open && (best_axis < 0 || acost < best)) {
        best = acost;
        best_axis = (int)axis;
        best_i = apick;
        best_src = src;
        for (int k = 0; k < 6; k++) {
          lb[k] = pre[k];
          rb[k] = suf[k];
        }
      }
    }
    if (open && (float)cnt * 120.0f < best) {
      if (at == 0) write_node(flags | kLeaf, -1, -1);
      open = false;
      best_src = lane;
    }
    // the triangles in the order of the chosen axis, the two children's
    // boxes, ids and segments
    ref = __shfl(ref, (int)best_src);
    for (int k = 0; k < 3; k++) {
      bmn[k] = __shfl(bmn[k], (int)best_src);
      bmx[k] = __shfl(bmx[k], (int)best_src);
      c[k] = __shfl(c[k], (int)best_src);
    }
    float cl[6], cr[6];
    for (int k = 0; k < 6; k++) {
      cl[k] = __shfl(lb[k], (int)(off + best_i - 1u));
      cr[k] = __shfl(rb[k], (int)(off + best_i));
    }
    const uint32_t heads = (uint32_t)(__ballot(open && at == 0) >> (half << 5));
    const uint32_t cid = ids + 2u * __popc(heads & ((1u << (off & 31u)) - 1u));
    ids += 2u * __popc(heads);
    if (open) {
      // smaller area first (bvh.rs:337-345)
      const bool swap = area6(cl) > area6(cr);
      if (at == 0)
        write_node((flags & ~kLeaf) | kSplit, (int32_t)(swap ? cid + 1 : cid),
                   (int32_t)(swap ? cid : cid + 1));
      const uint32_t side = at >= best_i ? 1u : 0u;
      parent = (int32_t)id;
      id = cid + side;
      flags = par | (((side == 1) != swap) ? kIsC1 : 0u);
      off += side ? best_i : 0u;
      cnt = side ? cnt - best_i : best_i;
      for (int k = 0; k < 6; k++) box[k] = side ? cr[k] : cl[k];
    }
  }
  if (here && pos < n) seg[pos] = ref;
  for (uint32_t h = ids + pos; h < ids_end; h += 32) {
    INode w{};
    w.flags = kHole;
    w.parent = -1;
    w.child[0] = w.child[1] = -1;
    a.nodes[h] = w;
  }
}

// ---------------------------------------------------------------------------
// Statistics and layout
// ---------------------------------------------------------------------------

// The tree's depth, the largest leaf and the leaves' statistics (one leaf,
// summed_area_ratio 0 + 0); inner nodes are counted per depth (dcount holds
// dcap >= max depth + 1 words), in LDS per workgroup first (one global atomic
// per workgroup and value: a global counter shared by all nodes serialises).
constexpr uint32_t kDepthLds = 512;
__global__ __launch_bounds__(256) void k_depth(Args a, uint32_t ninodes, uint32_t* dcount,
                                               uint32_t dcap) {
  __shared__ uint32_t cnt[kDepthLds];
  __shared__ uint32_t deepest, largest;
  const bool local = dcap <= kDepthLds;
  if (local)
    for (uint32_t k = threadIdx.x; k < dcap; k += 256) cnt[k] = 0;
  if (threadIdx.x == 0) deepest = largest = 0;
  __syncthreads();
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  INode* nodes = a.nodes;
  if (x < ninodes && !(nodes[x].flags & kHole)) {
    const uint32_t d = nodes[x].depth;
    if (nodes[x].flags & kLeaf) {
      nodes[x].leaves = 1;
      nodes[x].sar = 0.0f + 0.0f;
      atomicMax(&deepest, d);
      atomicMax(&largest, nodes[x].count);
    } else if (d < dcap) {
      atomicAdd(local ? &cnt[d] : &dcount[d], 1u);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicMax(&a.ctx->max_depth, deepest);
    atomicMax(&a.ctx->max_leaf, largest);
  }
  if (local)
    for (uint32_t k = threadIdx.x; k < dcap; k += 256)
      if (cnt[k]) atomicAdd(&dcount[k], cnt[k]);
}

// The inner nodes listed by depth: cursor[d] starts at depth d's offset;
// a workgroup reserves one range per depth and ranks its nodes in LDS.
__global__ __launch_bounds__(256) void k_depth_lists(Args a, uint32_t ninodes, uint32_t* cursor,
                                                     uint32_t dcap, uint32_t* list) {
  __shared__ uint32_t cnt[kDepthLds];
  const bool local = dcap <= kDepthLds;
  if (local)
    for (uint32_t k = threadIdx.x; k < dcap; k += 256) cnt[k] = 0;
  __syncthreads();
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  bool inner = false;
  uint32_t d = 0, rank = 0;
  if (x < ninodes) {
    const INode& n = a.nodes[x];
    inner = !(n.flags & (kLeaf | kHole)) && n.depth < dcap;
    d = n.depth;
  }
  if (inner && local) rank = atomicAdd(&cnt[d], 1u);
  __syncthreads();
  if (local)
    for (uint32_t k = threadIdx.x; k < dcap; k += 256)
      if (cnt[k]) cnt[k] = atomicAdd(&cursor[k], cnt[k]);
  __syncthreads();
  if (inner) list[local ? cnt[d] + rank : atomicAdd(&cursor[d], 1u)] = x;
}

// Runs visit(x) for the inner nodes x of the depths lo .. hi (listed by
// k_depth_lists; ends[d] is the end of depth d's part of the list), one depth
// after the other, deepest first (UP) or last.  One depth takes any number of
// workgroups; several, a launch each of which would mostly be its overhead,
// one workgroup.
template <bool UP, typename Visit>
__device__ __forceinline__ void by_depth(const uint32_t* list, const uint32_t* ends, uint32_t lo,
                                         uint32_t hi, Visit visit) {
  for (uint32_t q = 0; q <= hi - lo; q++) {
    const uint32_t d = UP ? hi - q : lo + q;
    const uint32_t end = ends[d];
    for (uint32_t k = (d ? ends[d - 1] : 0u) + blockIdx.x * blockDim.x + threadIdx.x; k < end;
         k += gridDim.x * blockDim.x)
      visit(list[k]);
    if (lo != hi) __syncthreads();
  }
}

// Leaf counts and summed_area_ratio (bvh.rs:380-386) of inner nodes from
// their children.
__global__ __launch_bounds__(1024) void k_bottom_up(Args a, const uint32_t* list,
                                                    const uint32_t* ends, uint32_t lo,
                                                    uint32_t hi) {
  INode* nodes = a.nodes;
  by_depth<true>(list, ends, lo, hi, [&](uint32_t x) {
    const int32_t c0 = nodes[x].child[0], c1 = nodes[x].child[1];
    const float s0 = nodes[c0].sar, s1 = nodes[c1].sar;
    const float A = area6(nodes[x].box);
    const float cc = (0.0f + s0) + s1;
    const float cs = (0.0f + area6(nodes[c0].box) / A) + area6(nodes[c1].box) / A;
    nodes[x].leaves = nodes[c0].leaves + nodes[c1].leaves;
    nodes[x].sar = cs + cc;
  });
}

// crystallize (bvh.rs:389-428), from the root down: an inner node's two
// children are written at nodes.len() at its turn, L(x).  The first child's
// own children follow at L(x) + 2, the second's behind all pairs of the
// first's subtree, and triangles follow their leaves' order.  (Every node
// walking up to the root for these sums took 0.98 ms for 1.33 M triangles.)
__global__ __launch_bounds__(1024) void k_place(Args a, const uint32_t* list, const uint32_t* ends,
                                                uint32_t lo, uint32_t hi, DevNode* out,
                                                uint32_t* order) {
  INode* nodes = a.nodes;
  by_depth<false>(list, ends, lo, hi, [&](uint32_t x) {
    const uint32_t at = nodes[x].pairs;
    uint32_t L = at + 2, T = nodes[x].first_tri;
    for (uint32_t s = 0; s < 2; s++) {
      INode& c = nodes[nodes[x].child[s]];
      const bool leaf = c.flags & kLeaf;
      DevNode d;
      d.a = make_float4(c.box[0], c.box[1], c.box[2], c.box[3]);
      d.b = make_float4(c.box[4], c.box[5], u2f(leaf ? T : L), u2f(leaf ? c.count : 0u));
      out[at + s] = d;
      if (leaf) {
        const uint32_t* src = a.buf[(c.flags & kParity) ? 1 : 0] + c.begin;
        for (uint32_t k = 0; k < c.count; k++) order[T + k] = src[k];
      } else {
        c.pairs = L;
        c.first_tri = T;
      }
      T += c.count;
      L += 2 * (c.leaves - 1);
    }
  });
}

}  // namespace bvh

// ---------------------------------------------------------------------------
// Host driver
// ---------------------------------------------------------------------------

#define BVH_CHECK(x)                \
  do {                              \
    hipError_t e_ = (x);            \
    if (e_ != hipSuccess) {         \
      cleanup();                    \
      return e_;                    \
    }                               \
  } while (0)

hipError_t build_reference_bvh(const float* d_v9, uint32_t ntris, DevNode* nodes_out,
                               uint32_t* order_out, BuildResult* res, hipStream_t s,
                               uint32_t nbins) {
  using namespace bvh;
  res->error = 0;
  if (nbins != 16 && nbins != 32 && nbins != 64) return hipErrorInvalidValue;
  // One allocation for all scratch: every hipMalloc / hipFree of the build's
  // 26 buffers waits for the device.  The first pass over the requests (base
  // null) adds up the sizes.
  char* arena = nullptr;
  size_t arena_bytes = 0;
  auto cleanup = [&]() {
    if (arena) (void)hipFree(arena);
    arena = nullptr;
  };
  auto take = [&](auto** p, size_t count) {
    *p = reinterpret_cast<std::remove_reference_t<decltype(*p)>>(arena + arena_bytes);
    arena_bytes += (count * sizeof(**p) + 255) / 256 * 256;
  };
  const size_t N = ntris;
  Args a{};
  a.ntris = ntris;
  a.nbins = nbins;
  a.small_max = nbins / 2;
  float4 *A, *B;
  float* C;
  // Node ids: the levels take 1 + 2 S for S splits of nodes of more than 32
  // triangles, and each small subtree of n triangles reserves 2 (n - 1).
  // Those S splits form a full binary tree whose leaves are the small
  // subtrees, the single triangles and the unsplit large nodes, so S is
  // their number - 1 and all ids together are 2 (singles + unsplit large
  // nodes + triangles of small subtrees) - 1 <= 2 N - 1.
  const size_t ninodes_cap = 2 * N + 2;
  Ctx* ctx;
  const size_t list_cap = N / (kSub + 1) + 2, sub_cap = N / (a.small_max + 1) + 2;
  uint32_t *listA, *listB, *sub, *small, *dcount, *dlist;
  // references per chunk of a wide node: enough chunks for the 256 CUs, but
  // not more partials than they are worth (device ms with 512 / 1024 / 2048 /
  // 4096: 20,506 triangles 0.90 / 0.91 / 0.96 / 1.01, 131,072 1.41 / 1.42 / 1.49 /
  // 1.61, 300,000 2.04 / 2.02 / 2.02 / 2.19, 524,288 2.88 / 2.81 / 2.85 / 2.88,
  // 1.33 M 6.22 / 6.12 / 6.03 / 6.05)
  a.chunk = N <= 131072 ? 512u : N <= 524288 ? 1024u : 2048u;
  // chunks of the wide nodes of one level: their triangles are disjoint, so
  // at most N / chunk + (number of wide nodes) chunks
  const size_t max_wide = N / (kWide + 1) + 1, max_chunks = N / a.chunk + max_wide + 1;
  // depths: at most one level per triangle
  const size_t dcount_cap = 2 * N + 64;
  float *d_tpm, *d_tpm1;
  for (int pass = 0; pass < 2; pass++) {
    arena_bytes = 0;
    take(&A, N);
    take(&B, N);
    take(&C, N);
    for (int k = 0; k < 2; k++) take(&a.buf[k], N);
    for (int k = 0; k < 3; k++) {
      take(&a.sorted[k], N);
      take(&a.tmp[k], N);
    }
    take(&a.nodes, ninodes_cap);
    take(&ctx, 1);
    take(&listA, list_cap);
    take(&listB, list_cap);
    take(&sub, sub_cap);
    take(&small, N / 2 + 2);
    take(&a.wide_list, max_wide);
    take(&a.tot, max_wide * kBinWords);
    take(&a.chunk_node, max_chunks);
    take(&a.part, max_chunks * kBinWords);
    take(&a.side, max_chunks * 24);
    take(&d_tpm, N + 1);
    take(&d_tpm1, N + 1);
    take(&dcount, dcount_cap);
    take(&dlist, ninodes_cap);
    if (pass == 0) BVH_CHECK(hipMalloc((void**)&arena, arena_bytes));
  }
  a.A = A;
  a.B = B;
  a.C = C;
  a.ctx = ctx;
  a.sub_list = sub;
  a.small_list = small;
  // TreeSAH power tables with the C library (same values as the CPU build)
  // (two powf and a log2f per triangle count: 33 ms for 1.33 M counts on one
  // thread, so large tables are filled by up to 8)
  std::vector<float> tpm(N + 1), tpm1(N + 1);
  auto fill = [&](size_t lo, size_t hi) {
    for (size_t n = lo; n < hi; n++) {
      float m = log2f((float)n);
      tpm[n] = powf(0.8f, m);
      tpm1[n] = powf(0.8f, m - 1.0f);
    }
  };
  tpm[0] = tpm1[0] = 0.0f;
  const size_t parts = std::min<size_t>(8, N / 16384 + 1), per = N / parts + 1;
  std::vector<std::thread> workers;
  size_t first = 1;
  try {
    for (size_t k = 1; k < parts; k++, first += per)
      workers.emplace_back(fill, first, std::min(first + per, N + 1));
  } catch (const std::exception&) {
    // no thread to be had: the rest of the table is filled here
  }
  fill(first, N + 1);
  for (std::thread& w : workers) w.join();
  BVH_CHECK(hipMemcpyAsync(d_tpm, tpm.data(), (N + 1) * 4, hipMemcpyHostToDevice, s));
  BVH_CHECK(hipMemcpyAsync(d_tpm1, tpm1.data(), (N + 1) * 4, hipMemcpyHostToDevice, s));
  a.tpm = d_tpm;
  a.tpm1 = d_tpm1;

  hipEvent_t ev0, ev1;
  BVH_CHECK(hipEventCreate(&ev0));
  BVH_CHECK(hipEventCreate(&ev1));
  BVH_CHECK(hipEventRecord(ev0, s));

  Ctx init{};
  for (int k = 0; k < 6; k++) {
    init.root_box[k] = k < 3 ? 0xffffffffu : 0u;
    init.root_cbox[k] = k < 3 ? 0xffffffffu : 0u;
  }
  BVH_CHECK(hipMemcpyAsync(ctx, &init, sizeof(Ctx), hipMemcpyHostToDevice, s));
  {
    uint32_t blocks = (ntris + 255) / 256;
    if (blocks > 1024) blocks = 1024;  // each ends with 12 atomics on the same 12 words
    hipLaunchKernelGGL(k_trefs, dim3(blocks), dim3(256), 0, s, d_v9, ntris, A, B, C, a.buf[0],
                       ctx);
    BVH_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_root, dim3(1), dim3(64), 0, s, a.nodes, ctx, ntris);
    BVH_CHECK(hipGetLastError());
  }
  uint32_t zero = 0, one = 1;
  uint32_t nlist = 0;
  if (ntris > kSub) {
    BVH_CHECK(hipMemcpyAsync(listA, &zero, 4, hipMemcpyHostToDevice, s));
    BVH_CHECK(hipMemcpyAsync(&ctx->large[0], &one, 4, hipMemcpyHostToDevice, s));
    nlist = 1;
  } else if (ntris > a.small_max) {
    BVH_CHECK(hipMemcpyAsync(sub, &zero, 4, hipMemcpyHostToDevice, s));
    BVH_CHECK(hipMemcpyAsync(&ctx->sub_count, &one, 4, hipMemcpyHostToDevice, s));
  } else if (ntris >= 2) {
    BVH_CHECK(hipMemcpyAsync(small, &zero, 4, hipMemcpyHostToDevice, s));
    BVH_CHECK(hipMemcpyAsync(&ctx->small_count, &one, 4, hipMemcpyHostToDevice, s));
  }
  uint32_t* lists[2] = {listA, listB};
  bool wide = ntris > kWide;
  uint32_t nsub = ntris > a.small_max ? 1u : 0u;  // nodes for k_subtree so far
  uint32_t levels = 0;                            // iterations of the level phase
  // The lists' lengths stay on the device and the grids are their bounds (a
  // level has at most twice the nodes of the one before), so that the host
  // waits once in kLevelBatch levels; the levels enqueued past the last one
  // find empty lists.
  while (nlist > 0) {
    for (uint32_t q = 0; q < kLevelBatch; q++, levels++) {
      const uint32_t most = (uint32_t)std::min<size_t>((size_t)nlist << q, list_cap);
      const uint32_t most_wide = (uint32_t)std::min<size_t>(most, max_wide);
      a.parity = levels & 1u;
      a.list = lists[a.parity];
      a.next_list = lists[a.parity ^ 1u];
      hipLaunchKernelGGL(k_level_plan, dim3(1), dim3(1024), 0, s, a);
      BVH_CHECK(hipGetLastError());
      if (wide) {
        hipLaunchKernelGGL(k_bin_chunks, dim3((uint32_t)max_chunks), dim3(kBlock), 0, s, a);
        BVH_CHECK(hipGetLastError());
        hipLaunchKernelGGL(k_sum_chunks, dim3(most_wide, kBinWords / 64), dim3(256), 0, s, a);
        BVH_CHECK(hipGetLastError());
      }
      a.mode = 0;
      hipLaunchKernelGGL(k_decide, dim3(most), dim3(kBlock), 0, s, a);
      BVH_CHECK(hipGetLastError());
      hipLaunchKernelGGL(k_sort, dim3(most * 3), dim3(kBlock), 0, s, a);
      BVH_CHECK(hipGetLastError());
      a.mode = 1;
      hipLaunchKernelGGL(k_decide, dim3(most), dim3(kBlock), 0, s, a);
      BVH_CHECK(hipGetLastError());
      if (wide) {
        hipLaunchKernelGGL(k_part_chunks, dim3((uint32_t)max_chunks), dim3(kBlock), 0, s, a);
        BVH_CHECK(hipGetLastError());
      }
      hipLaunchKernelGGL(k_partition, dim3(most), dim3(kBlock), 0, s, a);
      BVH_CHECK(hipGetLastError());
    }
    Ctx hl;
    BVH_CHECK(hipMemcpyAsync(&hl, ctx, sizeof(Ctx), hipMemcpyDeviceToHost, s));
    BVH_CHECK(hipStreamSynchronize(s));
    if (hl.error) break;
    nlist = hl.large[levels & 1u];
    wide = hl.next_wide > 0;
    nsub = hl.sub_count;
  }
  // (both exit at once after an error, and k_small beyond the nodes listed,
  // so neither waits for the host to read the counters)
  if (nsub) {
    hipLaunchKernelGGL(k_subtree, dim3(nsub), dim3(64 * kSubWaves), 0, s, a);
    BVH_CHECK(hipGetLastError());
  }
  hipLaunchKernelGGL(k_small, dim3((ntris / 2 + 7) / 8 + 1), dim3(256), 0, s, a);
  BVH_CHECK(hipGetLastError());
  Ctx hc;
  BVH_CHECK(hipMemcpyAsync(&hc, ctx, sizeof(Ctx), hipMemcpyDeviceToHost, s));
  BVH_CHECK(hipStreamSynchronize(s));
  uint32_t ninodes = hc.node_count;
  INode root_h;
  if (hc.error == 0) {
    BVH_CHECK(hipMemcpyAsync(&root_h, a.nodes, sizeof(INode), hipMemcpyDeviceToHost, s));
    BVH_CHECK(hipStreamSynchronize(s));
  }
  if (hc.error & 1u) {
    res->error = 9;  // CV_ERR_NAN
  } else if (hc.error & 2u) {
    res->error = 8;  // CV_ERR_BVH_NO_SPLIT
  } else if (root_h.child[0] < 0) {
    res->error = 8;  // the root must split (bvh.rs:512)
  }
  if (res->error) {
    (void)hipEventDestroy(ev0);
    (void)hipEventDestroy(ev1);
    cleanup();
    return hipSuccess;
  }
  uint32_t blocks = (ninodes + 255) / 256;
  // depths: the level phase's nodes lie at most `levels` deep, k_subtree adds
  // at most sub_levels and a small subtree of at most 32 triangles 31
  const uint32_t dcap = levels + hc.sub_levels + 34;
  BVH_CHECK(hipMemsetAsync(dcount, 0, (size_t)dcap * 4, s));
  hipLaunchKernelGGL(k_depth, dim3(blocks), dim3(256), 0, s, a, ninodes, dcount, dcap);
  BVH_CHECK(hipGetLastError());
  std::vector<uint32_t> hcount(dcap), hoff(dcap);
  BVH_CHECK(hipMemcpyAsync(hcount.data(), dcount, (size_t)dcap * 4, hipMemcpyDeviceToHost, s));
  BVH_CHECK(hipMemcpyAsync(&hc, ctx, sizeof(Ctx), hipMemcpyDeviceToHost, s));
  BVH_CHECK(hipStreamSynchronize(s));
  if (hc.max_depth >= dcap) {
    cleanup();
    return hipErrorInvalidValue;
  }
  uint32_t run = 0;
  for (uint32_t d = 0; d < dcap; d++) {
    hoff[d] = run;
    run += hcount[d];
  }
  // (k_depth_lists moves every depth's offset to the depth's end)
  BVH_CHECK(hipMemcpyAsync(dcount, hoff.data(), (size_t)dcap * 4, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_depth_lists, dim3(blocks), dim3(256), 0, s, a, ninodes, dcount, dcap,
                     dlist);
  BVH_CHECK(hipGetLastError());
  // consecutive depths of few nodes share a launch of one workgroup
  struct Depths {
    uint32_t lo, hi, blocks;
  };
  std::vector<Depths> groups;
  for (uint32_t d = 0; d < hc.max_depth; d++) {
    const bool few = hcount[d] <= kDepthFew;
    if (few && !groups.empty() && groups.back().blocks == 1)
      groups.back().hi = d;
    else
      groups.push_back(Depths{d, d, few ? 1u : (hcount[d] + 255) / 256});
  }
  for (size_t k = groups.size(); k-- > 0;) {
    const Depths& g = groups[k];
    hipLaunchKernelGGL(k_bottom_up, dim3(g.blocks), dim3(g.blocks == 1 ? 1024 : 256), 0, s, a,
                       dlist, dcount, g.lo, g.hi);
    BVH_CHECK(hipGetLastError());
  }
  for (const Depths& g : groups) {
    hipLaunchKernelGGL(k_place, dim3(g.blocks), dim3(g.blocks == 1 ? 1024 : 256), 0, s, a, dlist,
                       dcount, g.lo, g.hi, nodes_out, order_out);
    BVH_CHECK(hipGetLastError());
  }
  BVH_CHECK(hipEventRecord(ev1, s));
  BVH_CHECK(hipMemcpyAsync(&hc, ctx, sizeof(Ctx), hipMemcpyDeviceToHost, s));
  BVH_CHECK(hipMemcpyAsync(&root_h, a.nodes, sizeof(INode), hipMemcpyDeviceToHost, s));
  BVH_CHECK(hipStreamSynchronize(s));
  float ms = 0.0f;
  (void)hipEventElapsedTime(&ms, ev0, ev1);
  (void)hipEventDestroy(ev0);
  (void)hipEventDestroy(ev1);
  res->leaves = root_h.leaves;
  res->num_nodes = 2 * (root_h.leaves - 1);
  res->depth = hc.max_depth;
  res->max_leaf = hc.max_leaf;
  res->avg_area_ratio = root_h.sar / (float)(2 * root_h.leaves - 1);
  res->avg_tris_per_leaf = (float)ntris / (float)root_h.leaves;
  res->build_ms = ms;
  cleanup();
  return hipSuccess;
}

}  // namespace cvk
