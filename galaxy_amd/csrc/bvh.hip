// bvh.hip — BVH construction on the GPU for the model commit (the place of
// Embree's SAH build at ospCommit(ospModel), Visualization.cpp:219-277).
//
// 1. centroid bounds (wave reduction + ordered-int atomics) and 63-bit Morton
//    codes of the primitive centroids (21 bits per axis);
// 2. LSD radix sort of (code, primitive) pairs, 8 bits per pass: per-tile
//    digit histograms in LDS, one device-wide exclusive scan of the
//    digit-major histogram, and a stable scatter whose in-tile ranks come from
//    wave ballots over the digit bits;
// 3. Karras topology (HPG 2012): one work-item per inner node finds its key
//    range and split with the delta() prefix length (equal codes broken by
//    index);
// 4. treelet restructuring (Karras and Aila, "Fast Parallel Construction of
//    High-Quality Bounding Volume Hierarchies", HPG 2013): every node with at
//    least gamma primitives below it roots a treelet of 7 leaves, grown from its
//    two children by opening the inner leaf of largest surface area; the
//    SAH-optimal binary tree over those 7 leaves (dynamic programming over the
//    127 subsets, leaf option included) replaces the treelet when it is
//    cheaper, reusing its inner nodes.  Nodes are processed by depth, deepest
//    first (one launch per depth; treelets of one depth are disjoint, and a
//    treelet needs the ones below it only, so the tree is that of any bottom-up
//    order), three rounds with gamma = 7, 14, 28.  The launches refresh primitive
//    counts and SAH costs as they go and form the boxes in the first round.
//    Depths come from pointer jumping over the parent links and a counting sort
//    of the inner nodes by depth.  Kernel boundaries order the levels, so no
//    work-item waits on another's stores;
// 5. bottom-up refit, one launch per depth: child boxes, primitive counts, and
//    the SAH cost with the cheaper of leaf or node at each subtree that fits a
//    leaf;
// 6. layout, top-down in breadth-first frontiers: a subtree whose SAH cost is
//    lower as one leaf (at most GXY_BVH_LEAF primitives) becomes a leaf, inner
//    nodes are renumbered (root 0, the inner children of a node adjacent) and
//    the primitives reordered so that every leaf covers a contiguous range.  The
//    frontiers' sizes stay on the device: one launch per depth of the tree, no
//    wait in between;
// 7. 4-wide collapse, top-down in frontiers: a node takes its two children and
//    opens the inner child of largest surface area until it holds four.
// Node layout: BVHNode (both child boxes, 64 B) and BVH4Node (128 B); child
// codes are inner indices >= 0 or leaf codes ~(first << 4 | count - 1).
#include <cstring>
#include <vector>

#include "gxy_device.h"
#include "gxy_internal.h"

namespace gxy {

// SAH cost of visiting a node (per unit of surface area): a node visit fetches
// 64 B and tests two boxes.  The cost of testing one primitive is the build's
// prim_cost argument (a triangle test, 36 B and about 50 flops, is about 1).
#define BVH_CI 1.2f

__device__ __forceinline__ unsigned int okey(float f) {
  unsigned int u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ounkey(unsigned int k) {
  unsigned int u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
  return __uint_as_float(u);
}

__host__ __device__ __forceinline__ int leaf_code(int k) { return ~(k << 4); }
__host__ __device__ __forceinline__ int leaf_code_n(int first, int count) { return ~((first << 4) | (count - 1)); }

__device__ __forceinline__ float half_area(const float lo[3], const float hi[3]) {
  const float dx = fmaxf(hi[0] - lo[0], 0.f), dy = fmaxf(hi[1] - lo[1], 0.f), dz = fmaxf(hi[2] - lo[2], 0.f);
  return dx * dy + dy * dz + dz * dx;
}

__device__ __forceinline__ void slot_box(const BVHNode *nd, int slot, float lo[3], float hi[3]) {
  const float *l = slot ? nd->lo1 : nd->lo0, *h = slot ? nd->hi1 : nd->hi0;
  for (int a = 0; a < 3; a++) { lo[a] = l[a]; hi[a] = h[a]; }
}

// ------------------------------------------------------------------ Morton codes
__global__ void k_bounds_init(unsigned int *b) {
  for (int k = 0; k < 3; k++) { b[k] = 0xffffffffu; b[3 + k] = 0u; }
}

// Six atomics on one cache line per workgroup at the end: they run one after
// the other (11 ns each), so the launch has few, large workgroups and one
// wave adds what the workgroup found.  1M boxes: 1066 us with six atomics from every
// wave of 3907 workgroups, 11 us now (the boxes alone, 24 MB, take 5 us).
#define CB_BLOCK 1024
#define CB_GRID 256
__global__ __launch_bounds__(CB_BLOCK) void k_centroid_bounds(const float *boxes, int n, unsigned int *b) {
  __shared__ unsigned int s_lo[CB_BLOCK / 64][3], s_hi[CB_BLOCK / 64][3];
  unsigned int lo[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, hi[3] = {0u, 0u, 0u};
  for (int64_t i = (int64_t)blockIdx.x * CB_BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * CB_BLOCK) {
    const float *p = boxes + 6 * i;
    for (int k = 0; k < 3; k++) {
      unsigned int c = okey(0.5f * (p[k] + p[3 + k]));
      lo[k] = min(lo[k], c);
      hi[k] = max(hi[k], c);
    }
  }
  for (int k = 0; k < 3; k++) {
    for (int o = 32; o > 0; o >>= 1) {
      lo[k] = min(lo[k], (unsigned int)__shfl_xor((int)lo[k], o, 64));
      hi[k] = max(hi[k], (unsigned int)__shfl_xor((int)hi[k], o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
      s_lo[threadIdx.x >> 6][k] = lo[k];
      s_hi[threadIdx.x >> 6][k] = hi[k];
    }
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    unsigned int l = 0xffffffffu, h = 0u;
    for (int w = 0; w < CB_BLOCK / 64; w++) {
      l = min(l, s_lo[w][threadIdx.x]);
      h = max(h, s_hi[w][threadIdx.x]);
    }
    atomicMin(b + threadIdx.x, l);
    atomicMax(b + 3 + threadIdx.x, h);
  }
}

__device__ __forceinline__ uint64_t spread21(uint64_t x) {
  x &= 0x1fffff;
  x = (x | x << 32) & 0x1f00000000ffffull;
  x = (x | x << 16) & 0x1f0000ff0000ffull;
  x = (x | x << 8) & 0x100f00f00f00f00full;
  x = (x | x << 4) & 0x10c30c30c30c30c3ull;
  x = (x | x << 2) & 0x1249249249249249ull;
  return x;
}

__global__ __launch_bounds__(GXY_BLOCK) void k_morton(const float *boxes, int n, const unsigned int *b,
                                                      uint64_t *keys, int *vals) {
  int i = blockIdx.x * GXY_BLOCK + threadIdx.x;
  if (i >= n) return;
  const float *p = boxes + 6 * (int64_t)i;
  uint64_t code = 0;
  for (int k = 0; k < 3; k++) {
    float lo = ounkey(b[k]), hi = ounkey(b[3 + k]);
    float c = 0.5f * (p[k] + p[3 + k]);
    float e = hi - lo;
    float u = e > 0.f ? (c - lo) / e : 0.5f;
    u = u < 0.f ? 0.f : (u > 1.f ? 1.f : u);
    uint64_t q = (uint64_t)(u * 2097151.0f);
    code |= spread21(q) << (2 - k);
  }
  keys[i] = code;
  vals[i] = i;
}

// ------------------------------------------------------------------ radix sort
#define RS_ITEMS 16
#define RS_TILE (GXY_BLOCK * RS_ITEMS)

// digit histogram of one tile, written digit-major (hist[d * ntiles + tile])
__global__ __launch_bounds__(GXY_BLOCK) void k_rs_hist(const uint64_t *keys, int n, int shift, int ntiles, int *hist) {
  __shared__ int h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * RS_TILE;
  for (int k = 0; k < RS_ITEMS; k++) {
    const int64_t i = base + (int64_t)k * GXY_BLOCK + threadIdx.x;
    if (i < n) atomicAdd(&h[(int)(keys[i] >> shift) & 255], 1);
  }
  __syncthreads();
  hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

__device__ __forceinline__ unsigned long long rs_lanemask_lt() {
  const int lane = threadIdx.x & 63;
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// Stable scatter of one tile: keys are taken in index order (slot by slot,
// wave by wave, lane by lane); a key's destination is its digit's global base
// for this tile + the keys of the same digit before it in the tile.
__global__ __launch_bounds__(GXY_BLOCK) void k_rs_scatter(const uint64_t *kin, const int *vin, int n, int shift,
                                                          int ntiles, const int *off, uint64_t *kout, int *vout) {
  __shared__ int run[256];
  __shared__ int wc[GXY_BLOCK / 64][256];
  const int t = threadIdx.x, w = t >> 6;
  run[t] = off[(int64_t)t * ntiles + blockIdx.x];
  const int64_t base = (int64_t)blockIdx.x * RS_TILE;
  for (int k = 0; k < RS_ITEMS; k++) {
    const int64_t i = base + (int64_t)k * GXY_BLOCK + t;
    const bool valid = i < n;
    uint64_t key = 0;
    int val = 0, d = 0;
    if (valid) {
      key = kin[i];
      val = vin[i];
      d = (int)(key >> shift) & 255;
    }
    for (int q = 0; q < GXY_BLOCK / 64; q++) wc[q][t] = 0;
    unsigned long long m = __ballot(valid);
    for (int b = 0; b < 8; b++) {
      const unsigned long long bb = __ballot((d >> b) & 1);
      m &= ((d >> b) & 1) ? bb : ~bb;
    }
    const int rk = __popcll(m & rs_lanemask_lt());
    __syncthreads();
    if (valid && rk == 0) wc[w][d] = __popcll(m);
    __syncthreads();
    if (valid) {
      int pos = run[d] + rk;
      for (int q = 0; q < w; q++) pos += wc[q][d];
      kout[pos] = key;
      vout[pos] = val;
    }
    __syncthreads();
    int add = 0;
    for (int q = 0; q < GXY_BLOCK / 64; q++) add += wc[q][t];
    run[t] += add;
    __syncthreads();
  }
}

// Sorts n (key, value) pairs by the low `bits` bits of the keys (stable);
// the result ends in (k0, v0) or (k1, v1): the return value says which (0/1).
static int radix_sort_pairs(uint64_t *k0, int *v0, uint64_t *k1, int *v1, int n, int bits, int *hist, int *off,
                            void *scan_tmp, hipStream_t s, hipError_t *err) {
  const int ntiles = (n + RS_TILE - 1) / RS_TILE;
  int cur = 0;
  for (int shift = 0; shift < bits; shift += 8) {
    uint64_t *ki = cur ? k1 : k0, *ko = cur ? k0 : k1;
    int *vi = cur ? v1 : v0, *vo = cur ? v0 : v1;
    hipLaunchKernelGGL(k_rs_hist, dim3(ntiles), dim3(GXY_BLOCK), 0, s, (const uint64_t *)ki, n, shift, ntiles, hist);
    hipError_t e = launch_exclusive_sum(hist, off, (long long)256 * ntiles, scan_tmp, s);
    if (e != hipSuccess) { *err = e; return cur; }
    hipLaunchKernelGGL(k_rs_scatter, dim3(ntiles), dim3(GXY_BLOCK), 0, s, (const uint64_t *)ki, (const int *)vi, n,
                       shift, ntiles, (const int *)off, ko, vo);
    cur ^= 1;
  }
  *err = hipGetLastError();
  return cur;
}

// ------------------------------------------------------------------ Karras topology
__device__ __forceinline__ int delta(const uint64_t *keys, int n, int i, int j) {
  if (j < 0 || j > n - 1) return -1;
  uint64_t a = keys[i], b = keys[j];
  if (a == b) return 64 + __clz((unsigned int)(i ^ j));
  return __clzll(a ^ b);
}

// parent[i] of inner node i, parent[ni + k] of leaf k (ni = n - 1; root -1)
__global__ __launch_bounds__(GXY_BLOCK) void k_karras(const uint64_t *keys, int n, BVHNode *nodes, int *parent) {
  int i = blockIdx.x * GXY_BLOCK + threadIdx.x;
  if (i >= n - 1) return;
  const int ni = n - 1;
  int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
  int dmin = delta(keys, n, i, i - d);
  int lmax = 2;
  while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
  int l = 0;
  for (int t = lmax >> 1; t >= 1; t >>= 1)
    if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
  int j = i + l * d;
  int dnode = delta(keys, n, i, j);
  int s = 0, t = l;
  do {
    t = (t + 1) >> 1;
    if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
  } while (t > 1);
  int g = i + s * d + (d < 0 ? -1 : 0);
  int lo = i < j ? i : j, hi = i < j ? j : i;
  int c0, c1;
  if (lo == g) { c0 = leaf_code(g); parent[ni + g] = i; }
  else { c0 = g; parent[g] = i; }
  if (hi == g + 1) { c1 = leaf_code(g + 1); parent[ni + g + 1] = i; }
  else { c1 = g + 1; parent[g + 1] = i; }
  nodes[i].c0 = c0;
  nodes[i].c1 = c1;
  nodes[i].pad_[0] = nodes[i].pad_[1] = 0;
  if (i == 0) parent[0] = -1;
}

// ------------------------------------------------------------------ refit
// Per inner node: cnt (primitives below), costc (SAH cost with each subtree of
// <= GXY_BVH_LEAF primitives made a leaf where that is cheaper), leaf (1: costc
// chose a leaf here).  Costs are in units of half surface area.
struct BuildArrays {
  int *cnt;
  float *costc;
  int *leaf;
  float ct;   // SAH cost of one primitive test
};

__device__ __forceinline__ void child_totals(const BuildArrays &A, int code, const float lo[3], const float hi[3],
                                             int &c, float &costc) {
  if (code >= 0) {
    c = A.cnt[code];
    costc = A.costc[code];
  } else {
    c = 1;
    costc = A.ct * half_area(lo, hi);
  }
}

// Depth of every inner node by pointer jumping over the parent links: after
// round r, anc is the ancestor 2^r levels up (-1 past the root) and dep the
// distance to it (the full depth once anc is -1).  Eight rounds give exact
// depths below 256; deeper nodes keep a depth >= 256.
__global__ __launch_bounds__(GXY_BLOCK) void k_depth_init(const int *parent, int ni, int *anc, int *dep) {
  const int i = blockIdx.x * GXY_BLOCK + threadIdx.x;
  if (i >= ni) return;
  const int a = parent[i];
  anc[i] = a;
  dep[i] = a >= 0 ? 1 : 0;
}
__global__ __launch_bounds__(GXY_BLOCK) void k_depth_jump(const int *anc, const int *dep, int ni, int *anc2,
                                                          int *dep2) {
  const int i = blockIdx.x * GXY_BLOCK + threadIdx.x;
  if (i >= ni) return;
  const int a = anc[i];
  dep2[i] = a >= 0 ? dep[i] + dep[a] : dep[i];
  anc2[i] = a >= 0 ? anc[a] : -1;
}

// Counting sort of node indices by a small key (depth or height, clamped to
// GXY_BVH_MAXH - 1).  Equal keys are common within a wave (neighbouring nodes
// sit at the same height), so a wave adds each distinct key once: the lowest
// active lane's key, all lanes holding it, one atomic.  k_level_hist counts;
// k_level_scatter reserves each key's range for its LEVEL_TILE nodes with one
// global atomic per key and places them (order within a key is arbitrary).
#define LEVEL_TILE (GXY_BLOCK * 8)
__device__ __forceinline__ int level_key(const int *key, int64_t i, int n) {
  return i < n ? min(max(key[i], 0), GXY_BVH_MAXH - 1) : -1;
}
__global__ __launch_bounds__(GXY_BLOCK) void k_level_hist(const int *key, int n, int *hist) {
  __shared__ int h[GXY_BVH_MAXH];
  for (int t = threadIdx.x; t < GXY_BVH_MAXH; t += GXY_BLOCK) h[t] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * LEVEL_TILE;
  for (int r = 0; r < LEVEL_TILE / GXY_BLOCK; r++) {
    const int k = level_key(key, base + (int64_t)r * GXY_BLOCK + threadIdx.x, n);
    unsigned long long act = __ballot(k >= 0);
    while (act) {
      const int kk = __shfl(k, __ffsll((long long)act) - 1, 64);
      const unsigned long long same = __ballot(k == kk) & act;
      if (k == kk && __popcll(same & rs_lanemask_lt()) == 0) atomicAdd(&h[kk], __popcll(same));
      act &= ~same;
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < GXY_BVH_MAXH; t += GXY_BLOCK)
    if (h[t]) atomicAdd(hist + t, h[t]);
}
__global__ __launch_bounds__(GXY_BLOCK) void k_level_scatter(const int *key, int n, int *cursor, int *list) {
  __shared__ int h[GXY_BVH_MAXH];
  for (int t = threadIdx.x; t < GXY_BVH_MAXH; t += GXY_BLOCK) h[t] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * LEVEL_TILE;
  for (int r = 0; r < LEVEL_TILE / GXY_BLOCK; r++) {
    const int k = level_key(key, base + (int64_t)r * GXY_BLOCK + threadIdx.x, n);
    unsigned long long act = __ballot(k >= 0);
    while (act) {
      const int kk = __shfl(k, __ffsll((long long)act) - 1, 64);
      const unsigned long long same = __ballot(k == kk) & act;
      if (k == kk && __popcll(same & rs_lanemask_lt()) == 0) atomicAdd(&h[kk], __popcll(same));
      act &= ~same;
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < GXY_BVH_MAXH; t += GXY_BLOCK)
    if (h[t]) h[t] = atomicAdd(cursor + t, h[t]);   // this tile's first position for key t
  __syncthreads();
  for (int r = 0; r < LEVEL_TILE / GXY_BLOCK; r++) {
    const int64_t i = base + (int64_t)r * GXY_BLOCK + threadIdx.x;
    const int k = level_key(key, i, n);
    unsigned long long act = __ballot(k >= 0);
    while (act) {
      const int kk = __shfl(k, __ffsll((long long)act) - 1, 64);
      const unsigned long long same = __ballot(k == kk) & act;
      int first = 0;
      if (k == kk && __popcll(same & rs_lanemask_lt()) == 0) first = atomicAdd(&h[kk], __popcll(same));
      first = __shfl(first, __ffsll((long long)same) - 1, 64);
      if (k == kk) list[first + __popcll(same & rs_lanemask_lt())] = (int)i;
      act &= ~same;
    }
  }
}

// The box of node p's slot `slot` from what is below it: an inner child's own
// two boxes, or the primitive's.
__device__ __forceinline__ void child_box(const float *boxes, const int *order, const BVHNode *nodes, int code,
                                          float lo[3], float hi[3]) {
  if (code >= 0) {
    const BVHNode *ch = nodes + code;
    for (int a = 0; a < 3; a++) {
      lo[a] = fminf(ch->lo0[a], ch->lo1[a]);
      hi[a] = fmaxf(ch->hi0[a], ch->hi1[a]);
    }
  } else {
    const float *pb = boxes + 6 * (int64_t)order[(~code) >> 4];
    for (int a = 0; a < 3; a++) { lo[a] = pb[a]; hi[a] = pb[3 + a]; }
  }
}

// Refit of the inner nodes of one depth (every deeper node done by earlier
// launches): the children's boxes go into this node's slots, and the totals
// of its subtree are formed from the children's.
__global__ __launch_bounds__(GXY_BLOCK) void k_refit_level(const float *boxes, const int *order, BVHNode *nodes,
                                                           const int *list, int count, BuildArrays A) {
  const int i = blockIdx.x * GXY_BLOCK + threadIdx.x;
  if (i >= count) return;
  const int p = list[i];
  BVHNode *nd = nodes + p;
  float l[2][3], h[2][3], q[2];
  int c[2];
  for (int slot = 0; slot < 2; slot++) {
    const int code = slot ? nd->c1 : nd->c0;
    child_box(boxes, order, nodes, code, l[slot], h[slot]);
    child_totals(A, code, l[slot], h[slot], c[slot], q[slot]);
  }
  float lo[3], hi[3];
  for (int a = 0; a < 3; a++) {
    nd->lo0[a] = l[0][a]; nd->hi0[a] = h[0][a];
    nd->lo1[a] = l[1][a]; nd->hi1[a] = h[1][a];
    lo[a] = fminf(l[0][a], l[1][a]);
    hi[a] = fmaxf(h[0][a], h[1][a]);
  }
  const float ar = half_area(lo, hi);
  const int cc = c[0] + c[1];
  const float inner = BVH_CI * ar + q[0] + q[1], asleaf = A.ct * ar * (float)cc;
  const bool lf = p != 0 && cc <= GXY_BVH_LEAF && asleaf <= inner;
  A.cnt[p] = cc;
  A.costc[p] = lf ? asleaf : inner;
  A.leaf[p] = lf ? 1 : 0;
}

// ------------------------------------------------------------------ treelets
#define TL 7                 // treelet leaves
#define TLS (1 << TL)        // subsets
#define TWAVES 4             // waves per workgroup of the treelet kernel

__device__ __forceinline__ float rl_f(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ int rl_i(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ void tl_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// a subset's split so far: the cost of its two parts and the part that holds
// the subset's lowest leaf; of equal costs the part of the largest number wins
struct Split {
  float v;
  int part;
  __device__ __forceinline__ void take(float ov, int op) {
    if (ov < v || (ov == v && op > part)) { v = ov; part = op; }
  }
};

// The best split of every subset of K leaves, one subset per lane (s, or 0 for
// a lane that has none): all 2^(K-1) - 1 parts in descending order.
template <int K>
__device__ __forceinline__ Split best_split(const float *sc, int s) {
  const int low = s & -s, rest = s ^ low;
  Split b = {3e38f, low};
  int q = rest;
#pragma unroll
  for (int k = 0; k < (1 << (K - 1)) - 1; k++) {
    q = (q - 1) & rest;
    const int part = q | low;
    const float v = sc[part] + sc[s ^ part];
    if (v < b.v) { b.v = v; b.part = part; }
  }
  return b;
}

// Restructures the treelet rooted at p (the costs below it final) with the 64
// lanes of a wave: lane j < 7 holds leaf j, and lane s the boxes of the subsets
// s and s + 64 of the leaves.  sc and sp: cost and best split of every subset in
// LDS.  Returns the treelet root's cost as restructured (or as it was).
__device__ __forceinline__ float treelet(BVHNode *nodes, int *parent, const BuildArrays &A, int ni, int p, float cur,
                                         float *sc, unsigned char *sp) {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));   // keeps the subsets' numbers out of the caller's loop (216 VGPRs hoisted)
  float l[3] = {0.f, 0.f, 0.f}, h[3] = {0.f, 0.f, 0.f};
  int code = -1, inner = p;   // lane k < 6: the treelet's inner node k
  if (lane < 2) {
    slot_box(nodes + p, lane, l, h);
    code = lane ? nodes[p].c1 : nodes[p].c0;
  }
  // grow the treelet: open the inner leaf of largest area until there are 7
  int nl = 2;
  for (; nl < TL; nl++) {
    const float a = lane < nl && code >= 0 ? half_area(l, h) : -1.f;
    float m = fmaxf(a, __shfl_xor(a, 1, 8));
    m = fmaxf(m, __shfl_xor(m, 2, 8));
    m = fmaxf(m, __shfl_xor(m, 4, 8));
    m = rl_f(m, 0);
    const unsigned long long eq = __ballot(a == m) & 127;
    if (!(m > -1.f) || eq == 0) return cur;   // no inner leaf left: fewer than 7 leaves
    const int best = __ffsll((long long)eq) - 1, q = rl_i(code, best);
    if (lane == nl - 1) inner = q;
    if (lane == best || lane == nl) {
      const int slot = lane == nl;
      slot_box(nodes + q, slot, l, h);
      code = slot ? nodes[q].c1 : nodes[q].c0;
    }
  }
  int cnt = 1;
  float cst = 0.f;
  if (lane < TL) {
    if (code >= 0) {
      cnt = A.cnt[code];
      cst = A.costc[code];
    } else {
      cst = A.ct * half_area(l, h);
    }
    sc[1 << lane] = cst;
  }
  // box and primitive count of subsets lane and lane + 64
  float l0[3] = {3e38f, 3e38f, 3e38f}, h0[3] = {-3e38f, -3e38f, -3e38f}, l1[3], h1[3];
  int c0 = 0;
#pragma unroll
  for (int j = 0; j < TL - 1; j++) {
    const bool in = (lane >> j) & 1;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      l0[a] = fminf(l0[a], in ? rl_f(l[a], j) : 3e38f);
      h0[a] = fmaxf(h0[a], in ? rl_f(h[a], j) : -3e38f);
    }
    c0 += in ? rl_i(cnt, j) : 0;
  }
#pragma unroll
  for (int a = 0; a < 3; a++) {
    l1[a] = fminf(l0[a], rl_f(l[a], TL - 1));
    h1[a] = fmaxf(h0[a], rl_f(h[a], TL - 1));
  }
  const int c1 = c0 + rl_i(cnt, TL - 1);
  const float ar0 = half_area(l0, h0), ar1 = half_area(l1, h1);
  const int pop = __popc((unsigned)lane);
  tl_sync();
  // optimal split of every subset by its size, smallest first; at size k a lane
  // has subset lane, subset lane + 64 or none
  auto finish = [&](int s, const Split &b) {
    const bool up = s >= 64;
    const int c = up ? c1 : c0;
    const float ar = up ? ar1 : ar0;
    float v = BVH_CI * ar + b.v;
    if (c <= GXY_BVH_LEAF) v = fminf(v, A.ct * ar * (float)c);
    sc[s] = v;
    sp[s] = (unsigned char)b.part;
  };
  auto own = [&](int k) { return pop == k ? lane : pop == k - 1 ? lane | 64 : 0; };
#define TL_SIZE(K)                              \
  {                                             \
    const int s = own(K);                       \
    if (s) finish(s, best_split<K>(sc, s));     \
    tl_sync();                                  \
  }
  TL_SIZE(2)
  TL_SIZE(3)
  TL_SIZE(4)
  TL_SIZE(5)
#undef TL_SIZE
  {
    // size 6, the leaves without leaf g: eight lanes per subset, four parts each
    const int g = lane >> 3, s = (TLS - 1) ^ (1 << g);
    Split b = {3e38f, 0};
    if (g < TL) {
      const int keep = (1 << g) - 1;
#pragma unroll
      for (int k = 3; k >= 0; k--) {
        const int six = ((((lane & 7) << 2) | k) << 1) | 1;   // part as a subset of six leaves
        const int part = ((six & ~keep) << 1) | (six & keep);
        if (part != s) b.take(sc[part] + sc[s ^ part], part);
      }
    }
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) b.take(__shfl_xor(b.v, o, 64), __shfl_xor(b.part, o, 64));
    // the winner goes to the lane that holds the subset's box
    const int mine = own(6), from = mine ? (__ffs((TLS - 1) ^ mine) - 1) * 8 : 0;
    b.v = __shfl(b.v, from, 64);
    b.part = __shfl(b.part, from, 64);
    if (mine) {
      if (!(b.v < 3e38f)) b = {3e38f, mine & -mine};
      finish(mine, b);
    }
    tl_sync();
  }
  {
    // all seven: one part per lane
    const int part = (lane << 1) | 1;
    Split b = {3e38f, 0};
    if (part != TLS - 1) b.take(sc[part] + sc[(TLS - 1) ^ part], part);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) b.take(__shfl_xor(b.v, o, 64), __shfl_xor(b.part, o, 64));
    if (!(b.v < 3e38f)) b = {3e38f, 1};
    if (lane == 63) finish(TLS - 1, b);
    tl_sync();
  }
  const float best = rl_f(sc[TLS - 1], 0);
  if (!(best < cur * 0.99999f)) return cur;
  // rebuild: subsets in a queue (a byte each), inner node k of the treelet for
  // entry k; the lane that holds a subset's box stores it
  unsigned long long qs = TLS - 1;
  int nq = 1;
#pragma unroll 1
  for (int k = 0; k < TL - 1; k++) {
    const int s = (int)(qs >> (8 * k)) & 255, node = rl_i(inner, k);
    const int left = __builtin_amdgcn_readfirstlane((int)sp[s]);
#pragma unroll 1
    for (int side = 0; side < 2; side++) {
      const int sub = side ? s ^ left : left;
      int ccode;
      if ((sub & (sub - 1)) == 0) {
        ccode = rl_i(code, __ffs(sub) - 1);
      } else {
        ccode = rl_i(inner, nq);
        qs |= (unsigned long long)sub << (8 * nq);
        nq++;
      }
      if (lane == (sub & 63)) {
        const bool up = sub >= 64;
        BVHNode *nd = nodes + node;
        float *pl = side ? nd->lo1 : nd->lo0, *ph = side ? nd->hi1 : nd->hi0;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          pl[a] = up ? l1[a] : l0[a];
          ph[a] = up ? h1[a] : h0[a];
        }
        *(side ? &nd->c1 : &nd->c0) = ccode;
        parent[ccode >= 0 ? ccode : ni + ((~ccode) >> 4)] = node;
      }
    }
    if (lane == (s & 63)) {
      const float v = sc[s];
      A.cnt[node] = s >= 64 ? c1 : c0;
      A.costc[node] = v;
    }
  }
  return best;
}

// The inner nodes of one depth: refresh each node's totals from its children
// (final: deeper nodes ran before), and restructure its treelet when it has at
// least gamma primitives below it.  What a node reads lies below it and no other
// node of its depth writes there.  A wave takes `per` nodes: a lane each for the
// totals, then all lanes together for one treelet after the other.  FIT (the
// first round): the nodes' boxes are not there yet and come from the children.
//
// The search over the 127 subsets (966 pairs of LDS reads) and the treelet's
// growth (five dependent node reads) are a serial chain: with one work-item per
// treelet a launch took its 124 us however few nodes it had, 110 launches
// 13.7 ms of a build over 1M triangles.  With a wave per treelet: 33 us a launch of the
// first round (boxes included), 18 us of the others, 2.5 ms (64 VGPRs, 8 waves per SIMD).
template <bool FIT>
__global__ __launch_bounds__(64 * TWAVES) __attribute__((amdgpu_waves_per_eu(8, 8)))
void k_treelet_level(const float *boxes, const int *order, const int *list, int count, int per, BVHNode *nodes,
                     int *parent, int ni, BuildArrays A, int gamma) {
  __shared__ float s_cost[TWAVES][TLS];
  __shared__ unsigned char s_split[TWAVES][TLS];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t i = ((int64_t)blockIdx.x * TWAVES + w) * per + lane;
  const bool have = lane < per && i < count;
  int p = 0, c = 0;
  float cost = 0.f;
  if (have) {
    p = list[i];
    BVHNode *nd = nodes + p;
    const int k0 = nd->c0, k1 = nd->c1;
    float l0[3], h0[3], l1[3], h1[3];
    if (FIT) {
      child_box(boxes, order, nodes, k0, l0, h0);
      child_box(boxes, order, nodes, k1, l1, h1);
      for (int a = 0; a < 3; a++) {
        nd->lo0[a] = l0[a]; nd->hi0[a] = h0[a];
        nd->lo1[a] = l1[a]; nd->hi1[a] = h1[a];
      }
    } else {
      slot_box(nd, 0, l0, h0);
      slot_box(nd, 1, l1, h1);
    }
    int n0, n1;
    float q0, q1;
    child_totals(A, k0, l0, h0, n0, q0);
    child_totals(A, k1, l1, h1, n1, q1);
    float lo[3], hi[3];
    for (int a = 0; a < 3; a++) { lo[a] = fminf(l0[a], l1[a]); hi[a] = fmaxf(h0[a], h1[a]); }
    const float ar = half_area(lo, hi);
    c = n0 + n1;
    cost = BVH_CI * ar + q0 + q1;
    if (c <= GXY_BVH_LEAF && p != 0) cost = fminf(cost, A.ct * ar * (float)c);
  }
  if (FIT) tl_sync();   // the boxes a lane has just stored are read by the lanes that grow the treelet
  unsigned long long todo = __ballot(have && c >= gamma);
  while (todo) {
    const int t = __ffsll((long long)todo) - 1;
    todo &= todo - 1;
    const float v = treelet(nodes, parent, A, ni, rl_i(p, t), rl_f(cost, t), s_cost[w], s_split[w]);
    if (lane == t) cost = v;
  }
  if (have) {
    A.cnt[p] = c;
    A.costc[p] = cost;
  }
}

// ------------------------------------------------------------------ layout
// A frontier entry: old inner node, first primitive.  Entry k of level L has the
// node index base[L] + k.  Levels[0 .. GXY_BVH_MAXH] holds the levels' entry
// counts, Levels[GXY_BVH_MAXH + 1 ...] their bases: a launch reads its own count
// and adds up the next one's, so no level waits for the host.
struct LayEnt {
  int old, first;
};
#define LEVELS (GXY_BVH_MAXH + 1)
#define LV_BLOCK 1024

// Positions for `want` (0 .. 4) entries per work-item at the end of the next
// level: one atomic per workgroup (a level's counter is one address; an atomic
// on it per wave took as long as the level's work).
__device__ __forceinline__ int level_reserve(int want, int *next_count) {
  __shared__ int s_w[LV_BLOCK / 64], s_base;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int at = 0, sum = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const unsigned long long m = __ballot(want > k);
    at += __popcll(m & rs_lanemask_lt());
    sum += __popcll(m);
  }
  if (lane == 0) s_w[w] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int q = 0; q < LV_BLOCK / 64; q++) {
      const int v = s_w[q];
      s_w[q] = t;
      t += v;
    }
    s_base = t ? atomicAdd(next_count, t) : 0;
  }
  __syncthreads();
  return s_base + s_w[w] + at;
}

// Primitives of the subtree under code in depth-first order (at most
// GXY_BVH_LEAF of them, so at most GXY_BVH_LEAF - 1 inner nodes).
__device__ int subtree_prims(const BVHNode *nodes, int code, int *out) {
  int st[GXY_BVH_LEAF];
  int sp = 0, n = 0;
  st[sp++] = code;
  while (sp > 0) {
    const int c = st[--sp];
    if (c < 0) {
      if (n < GXY_BVH_LEAF) out[n] = (~c) >> 4;
      n++;
    } else if (sp + 2 <= GXY_BVH_LEAF) {
      st[sp++] = nodes[c].c1;
      st[sp++] = nodes[c].c0;
    } else {
      return GXY_BVH_LEAF + 1;   // malformed: more than a leaf holds
    }
  }
  return n;
}

__global__ __launch_bounds__(LV_BLOCK) void k_layout(const LayEnt *fr, int level, int *lv, const BVHNode *nodes, int n,
                                                     const int *cnt, const int *leaf, const int *order, BVHNode *out,
                                                     int *neworder, LayEnt *next, int *bad, int cap) {
  const int count = lv[level], base = lv[LEVELS + level], nbase = base + count;
  if ((int64_t)blockIdx.x * LV_BLOCK >= count) return;   // (blocks of a level smaller than its bound)
  const int i = blockIdx.x * LV_BLOCK + threadIdx.x;
  if (i == 0) lv[LEVELS + level + 1] = nbase;
  const bool have = i < count && nbase <= cap;
  LayEnt e = {0, 0};
  BVHNode nd;
  int cc[2] = {-1, -1}, ninner = 0;
  bool in[2] = {false, false};
  if (have) {
    e = fr[i];
    nd = nodes[e.old];
    cc[0] = nd.c0;
    cc[1] = nd.c1;
    for (int s = 0; s < 2; s++) {
      in[s] = cc[s] >= 0 && !leaf[cc[s]];
      ninner += in[s];
    }
  }
  const int nslot = level_reserve(ninner, lv + level + 1);
  if (i < count && (!have || nbase + nslot + ninner > cap)) {   // more inner nodes than the tree has: malformed
    atomicAdd(bad, 1);
    return;
  }
  if (!have) return;
  int first = e.first, k = 0;
  for (int s = 0; s < 2; s++) {
    const int c = cc[s];
    int code;
    if (c < 0) {
      if (first < n) neworder[first] = order[(~c) >> 4];
      else atomicAdd(bad, 1);
      code = leaf_code_n(first, 1);
      first += 1;
    } else if (!in[s]) {
      int prims[GXY_BVH_LEAF];
      const int m = subtree_prims(nodes, c, prims);
      if (m < 1 || m > GXY_BVH_LEAF || first + m > n) {
        atomicAdd(bad, 1);
        code = leaf_code_n(first, 1);
      } else {
        for (int j = 0; j < m; j++) neworder[first + j] = order[prims[j]];
        code = leaf_code_n(first, m);
        first += m;
      }
    } else {
      next[nslot + k] = {c, first};
      code = nbase + nslot + k;
      k++;
      first += cnt[c];
    }
    if (s == 0) nd.c0 = code;
    else nd.c1 = code;
  }
  nd.pad_[0] = nd.pad_[1] = 0;
  out[base + i] = nd;
}

// ------------------------------------------------------------------ 4-wide collapse
// level 0: one entry (ints zeros), index 0
__global__ __launch_bounds__(LV_BLOCK) void k_levels_init(int *lv, int *bad, int *entry, int ints) {
  for (int k = threadIdx.x; k < 2 * LEVELS; k += LV_BLOCK) lv[k] = k == 0 ? 1 : 0;
  if ((int)threadIdx.x < ints) entry[threadIdx.x] = 0;
  if (threadIdx.x == 0) *bad = 0;
}

// (frontier entries: binary nodes)
__global__ __launch_bounds__(LV_BLOCK) void k_wide(const int *fr, int level, int *lv, const BVHNode *nodes,
                                                   BVH4Node *out, int *next, int cap, int *bad) {
  const int count = lv[level], base = lv[LEVELS + level], nbase = base + count;
  if ((int64_t)blockIdx.x * LV_BLOCK >= count) return;
  const int i = blockIdx.x * LV_BLOCK + threadIdx.x;
  if (i == 0) lv[LEVELS + level + 1] = nbase;
  const int bin = i < count && nbase <= cap ? fr[i] : -1;
  const bool have = bin >= 0 && bin < cap;
  int code[4];
  float lo[4][3], hi[4][3];
  const BVHNode b = nodes[have ? bin : 0];
  code[0] = b.c0;
  code[1] = b.c1;
  for (int a = 0; a < 3; a++) { lo[0][a] = b.lo0[a]; hi[0][a] = b.hi0[a]; lo[1][a] = b.lo1[a]; hi[1][a] = b.hi1[a]; }
  int m = 2;
#pragma unroll
  for (int grow = 2; grow < 4; grow++) {
    int best = -1;
    float ba = -1.f;
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (j < m && code[j] >= 0) {
        const float a = half_area(lo[j], hi[j]);
        if (a > ba) { ba = a; best = j; }
      }
    if (best < 0) break;
    int q = 0;
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (j == best) q = code[j];
    const BVHNode c = nodes[q];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (j == best) {
        code[j] = c.c0;
        for (int a = 0; a < 3; a++) { lo[j][a] = c.lo0[a]; hi[j][a] = c.hi0[a]; }
      }
      if (j == m) {
        code[j] = c.c1;
        for (int a = 0; a < 3; a++) { lo[j][a] = c.lo1[a]; hi[j][a] = c.hi1[a]; }
      }
    }
    m++;
  }
  int ninner = 0;
#pragma unroll
  for (int j = 0; j < 4; j++)
    if (j < m && code[j] >= 0) ninner++;
  const int nslot = level_reserve(have ? ninner : 0, lv + level + 1);
  if (i < count && (!have || nbase + nslot + ninner > cap)) {
    atomicAdd(bad, 1);
    return;
  }
  if (!have) return;
  BVH4Node o;
  int k = 0;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (j < m) {
      o.lox[j] = lo[j][0]; o.loy[j] = lo[j][1]; o.loz[j] = lo[j][2];
      o.hix[j] = hi[j][0]; o.hiy[j] = hi[j][1]; o.hiz[j] = hi[j][2];
      if (code[j] >= 0) {
        next[nslot + k] = code[j];
        o.child[j] = nbase + nslot + k;
        k++;
      } else {
        o.child[j] = code[j];
      }
    } else {
      o.lox[j] = o.loy[j] = o.loz[j] = __builtin_inff();
      o.hix[j] = o.hiy[j] = o.hiz[j] = -__builtin_inff();
      o.child[j] = leaf_code(0);   // (a ray that skips every axis enters this slot too)
    }
    o.pad_[j] = 0;
  }
  out[base + i] = o;
}

// ------------------------------------------------------------------ SAH of the final tree
__global__ __launch_bounds__(GXY_BLOCK) void k_sah(const BVHNode *nodes, int nn, float ct, double *acc) {
  __shared__ double red[GXY_BLOCK / 64];
  const int i = blockIdx.x * GXY_BLOCK + threadIdx.x;
  double v = 0.0;
  if (i < nn) {
    const BVHNode b = nodes[i];
    float lo[3], hi[3];
    for (int a = 0; a < 3; a++) { lo[a] = fminf(b.lo0[a], b.lo1[a]); hi[a] = fmaxf(b.hi0[a], b.hi1[a]); }
    v = BVH_CI * (double)half_area(lo, hi);
    const int cc[2] = {b.c0, b.c1};
    for (int s = 0; s < 2; s++)
      if (cc[s] < 0)
        v += ct * (double)((((~cc[s]) & 15) + 1)) * (double)half_area(s ? b.lo1 : b.lo0, s ? b.hi1 : b.hi0);
  }
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < GXY_BLOCK / 64; w++) s += red[w];
    atomicAdd(acc, s);
  }
}

// ------------------------------------------------------------------ structural check
// One mark per child reference: marks[0 .. nn) of the nodes, then nprim of the
// primitives.  A child's index has to be larger than its parent's, as both the
// layout and the collapse number them: with every node but the root marked
// exactly once, the parent links then descend to node 0, so no node is out of
// reach of the root.
__device__ __forceinline__ bool mark_child(int i, int c, int nn, int nprim, int *marks) {
  if (c >= 0) {
    if (c <= i || c >= nn) return false;
    atomicAdd(marks + c, 1);
    return true;
  }
  const int code = ~c, first = code >> 4, cnt = (code & 15) + 1;
  if (first < 0 || first > nprim - cnt) return false;
  for (int q = first; q < first + cnt; q++) atomicAdd(marks + nn + q, 1);
  return true;
}
__global__ __launch_bounds__(GXY_BLOCK) void k_mark_binary(const BVHNode *nodes, int nn, int nprim, int *marks,
                                                           int *bad) {
  const int i = blockIdx.x * GXY_BLOCK + threadIdx.x;
  if (i >= nn) return;
  const int c0 = nodes[i].c0, c1 = nodes[i].c1;
  bool ok = mark_child(i, c0, nn, nprim, marks);
  if (!(nn == 1 && c1 == c0)) ok = mark_child(i, c1, nn, nprim, marks) && ok;   // (one primitive: both children are it)
  if (!ok) atomicOr(bad, 1);
}
__global__ __launch_bounds__(GXY_BLOCK) void k_mark_wide(const BVH4Node *nodes, int nn, int nprim, int *marks,
                                                         int *bad) {
  const int64_t t = (int64_t)blockIdx.x * GXY_BLOCK + threadIdx.x;
  const int i = (int)(t >> 2), k = (int)t & 3;
  if (i >= nn) return;
  if (!(nodes[i].lox[k] <= nodes[i].hix[k])) return;   // empty slot
  if (!mark_child(i, nodes[i].child[k], nn, nprim, marks)) atomicOr(bad, 1);
}
__global__ __launch_bounds__(GXY_BLOCK) void k_check_marks(const int *marks, int n, int *bad) {
  const int i = blockIdx.x * GXY_BLOCK + threadIdx.x;
  if (i < n && marks[i] != (i == 0 ? 0 : 1)) atomicOr(bad, 1);
}

// ------------------------------------------------------------------ driver
namespace {
struct Pool {
  alloc_fn_t alloc;
  free_fn_t dfree;
  std::vector<void *> held;
  void *get(size_t bytes) {
    void *p = alloc(bytes ? bytes : 1);
    if (p) held.push_back(p);
    return p;
  }
  void release(void *p) {
    for (auto &q : held)
      if (q == p) { dfree(p); q = nullptr; }
  }
  ~Pool() {
    for (void *p : held)
      if (p) dfree(p);
  }
};
}  // namespace

#define BVH_CHK(x)                      \
  do {                                  \
    const hipError_t e_ = (x);          \
    if (e_ != hipSuccess) return e_;    \
  } while (0)

static hipError_t read_ints(const int *dev, int *host, int n, hipStream_t s) {
  BVH_CHK(hipMemcpyAsync(host, dev, sizeof(int) * n, hipMemcpyDeviceToHost, s));
  return hipStreamSynchronize(s);
}

// Node indices sorted by key (see k_level_hist): cnt[k] and start[k] of each
// key on the host, the list on the device.  hh holds 2 * GXY_BVH_MAXH ints.
static hipError_t sort_by_level(const int *key, int n, int *hh, int *cnt, int *start, int *list, hipStream_t s) {
  const dim3 grid((n + LEVEL_TILE - 1) / LEVEL_TILE);
  BVH_CHK(hipMemsetAsync(hh, 0, sizeof(int) * GXY_BVH_MAXH, s));
  hipLaunchKernelGGL(k_level_hist, grid, dim3(GXY_BLOCK), 0, s, key, n, hh);
  BVH_CHK(read_ints(hh, cnt, GXY_BVH_MAXH, s));
  start[0] = 0;
  for (int k = 0; k < GXY_BVH_MAXH; k++) start[k + 1] = start[k] + cnt[k];
  if (cnt[GXY_BVH_MAXH - 1] > 0) return hipErrorInvalidValue;   // deeper than the level table
  BVH_CHK(hipMemcpyAsync(hh + GXY_BVH_MAXH, start, sizeof(int) * GXY_BVH_MAXH, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_level_scatter, grid, dim3(GXY_BLOCK), 0, s, key, n, hh + GXY_BVH_MAXH, list);
  return hipGetLastError();
}

// The ni inner nodes sorted by depth (cnt and start of each depth on the host,
// the list on the device) and the number of depths; t0..t3 are ni ints each of
// scratch.
static hipError_t sort_by_depth(int ni, const int *parent, int *t0, int *t1, int *t2, int *t3, int *hh, int *cnt,
                                int *start, int *list, int *depths, hipStream_t s) {
  const dim3 grid((ni + GXY_BLOCK - 1) / GXY_BLOCK);
  hipLaunchKernelGGL(k_depth_init, grid, dim3(GXY_BLOCK), 0, s, parent, ni, t0, t1);
  int *anc = t0, *dep = t1, *anc2 = t2, *dep2 = t3;
  for (int r = 0; r < 8; r++) {
    hipLaunchKernelGGL(k_depth_jump, grid, dim3(GXY_BLOCK), 0, s, (const int *)anc, (const int *)dep, ni, anc2, dep2);
    int *t = anc; anc = anc2; anc2 = t;
    t = dep; dep = dep2; dep2 = t;
  }
  BVH_CHK(sort_by_level(dep, ni, hh, cnt, start, list, s));
  *depths = 0;
  for (int d = 0; d < GXY_BVH_MAXH; d++)
    if (cnt[d] > 0) *depths = d + 1;
  return hipSuccess;
}

hipError_t build_lbvh(const float *boxes_dev, int n, float prim_cost, alloc_fn_t alloc, free_fn_t dfree,
                      BVHBuildResult *out, hipStream_t s) {
  memset(out, 0, sizeof *out);
  if (n <= 0) return hipSuccess;
  Pool P{alloc, dfree, {}};
  if (n == 1) {
    BVHNode h;
    float b[6];
    BVH_CHK(hipMemcpyAsync(b, boxes_dev, 6 * sizeof(float), hipMemcpyDeviceToHost, s));
    BVH_CHK(hipStreamSynchronize(s));
    for (int a = 0; a < 3; a++) {
      h.lo0[a] = b[a]; h.hi0[a] = b[3 + a];
      h.lo1[a] = 3.0e38f; h.hi1[a] = -3.0e38f;
    }
    h.c0 = leaf_code(0);
    h.c1 = leaf_code(0);
    h.pad_[0] = h.pad_[1] = 0;
    BVH4Node w;
    for (int j = 0; j < 4; j++) {
      w.lox[j] = j ? INFINITY : b[0]; w.loy[j] = j ? INFINITY : b[1]; w.loz[j] = j ? INFINITY : b[2];
      w.hix[j] = j ? -INFINITY : b[3]; w.hiy[j] = j ? -INFINITY : b[4]; w.hiz[j] = j ? -INFINITY : b[5];
      w.child[j] = leaf_code(0);
      w.pad_[j] = 0;
    }
    out->nodes = (BVHNode *)alloc(sizeof(BVHNode));
    out->order = (int *)alloc(sizeof(int));
    out->nodes4 = (BVH4Node *)alloc(sizeof(BVH4Node));
    if (!out->nodes || !out->order || !out->nodes4) return hipErrorOutOfMemory;
    int zero = 0;
    BVH_CHK(hipMemcpyAsync(out->nodes, &h, sizeof h, hipMemcpyHostToDevice, s));
    BVH_CHK(hipMemcpyAsync(out->order, &zero, sizeof zero, hipMemcpyHostToDevice, s));
    BVH_CHK(hipMemcpyAsync(out->nodes4, &w, sizeof w, hipMemcpyHostToDevice, s));
    BVH_CHK(hipStreamSynchronize(s));
    out->nnodes = 1;
    out->depth = 1;
    out->nnodes4 = 1;
    out->depth4 = 1;
    out->leaves = 1;
    out->sah = BVH_CI + prim_cost;   // the root, then its one primitive, over the same surface
    return hipGetLastError();
  }
  const int nb = (n + GXY_BLOCK - 1) / GXY_BLOCK, ni = n - 1;
  const int ntiles = (n + RS_TILE - 1) / RS_TILE;
  unsigned int *bnd = (unsigned int *)P.get(8 * sizeof(unsigned int));
  uint64_t *k0 = (uint64_t *)P.get(sizeof(uint64_t) * n), *k1 = (uint64_t *)P.get(sizeof(uint64_t) * n);
  int *v0 = (int *)P.get(sizeof(int) * n), *v1 = (int *)P.get(sizeof(int) * n);
  int *hist = (int *)P.get(sizeof(int) * 256 * (size_t)ntiles);
  int *hoff = (int *)P.get(sizeof(int) * 256 * (size_t)ntiles);
  void *stmp = P.get(scan_temp_bytes((long long)256 * ntiles));
  if (!bnd || !k0 || !k1 || !v0 || !v1 || !hist || !hoff || !stmp) return hipErrorOutOfMemory;
  // 1-2: Morton codes, sorted
  hipLaunchKernelGGL(k_bounds_init, dim3(1), dim3(1), 0, s, bnd);
  const int nc = (n + CB_BLOCK - 1) / CB_BLOCK;
  hipLaunchKernelGGL(k_centroid_bounds, dim3(nc < CB_GRID ? nc : CB_GRID), dim3(CB_BLOCK), 0, s, boxes_dev, n, bnd);
  hipLaunchKernelGGL(k_morton, dim3(nb), dim3(GXY_BLOCK), 0, s, boxes_dev, n, (const unsigned int *)bnd, k0, v0);
  hipError_t e = hipSuccess;
  const int res = radix_sort_pairs(k0, v0, k1, v1, n, 63, hist, hoff, stmp, s, &e);
  BVH_CHK(e);
  uint64_t *keys = res ? k1 : k0;
  int *order = res ? v1 : v0;
  P.release(hist);
  P.release(hoff);
  P.release(stmp);
  // 3: topology
  BVHNode *nodes = (BVHNode *)P.get(sizeof(BVHNode) * (size_t)ni);
  int *parent = (int *)P.get(sizeof(int) * (size_t)(ni + n));
  int *t0 = (int *)P.get(sizeof(int) * (size_t)ni), *t1 = (int *)P.get(sizeof(int) * (size_t)ni);
  int *t2 = (int *)P.get(sizeof(int) * (size_t)ni), *t3 = (int *)P.get(sizeof(int) * (size_t)ni);
  BuildArrays A;
  A.ct = prim_cost;
  A.cnt = (int *)P.get(sizeof(int) * (size_t)ni);
  A.costc = (float *)P.get(sizeof(float) * (size_t)ni);
  A.leaf = (int *)P.get(sizeof(int) * (size_t)ni);
  int *hh = (int *)P.get(sizeof(int) * 2 * GXY_BVH_MAXH);
  int *hlist = (int *)P.get(sizeof(int) * (size_t)ni);
  if (!nodes || !parent || !t0 || !t1 || !t2 || !t3 || !A.cnt || !A.costc || !A.leaf || !hh || !hlist)
    return hipErrorOutOfMemory;
  hipLaunchKernelGGL(k_karras, dim3((ni + GXY_BLOCK - 1) / GXY_BLOCK), dim3(GXY_BLOCK), 0, s, (const uint64_t *)keys,
                     n, nodes, parent);
  P.release(k0);
  P.release(k1);
  // 4-5: treelet rounds, then the refit
  int dcount[GXY_BVH_MAXH], dstart[GXY_BVH_MAXH + 1], depths = 0;
  for (int round = 0; round < 3 && ni >= TL; round++) {
    BVH_CHK(sort_by_depth(ni, parent, t0, t1, t2, t3, hh, dcount, dstart, hlist, &depths, s));
    if (depths > GXY_BVH_MAXH - 2) return hipErrorInvalidValue;
    const int gamma = TL << round;
    for (int d = depths - 1; d >= 0; d--) {
      if (dcount[d] == 0) continue;
      // One node per wave up to 65536 nodes, else an equal share: which nodes of a
      // depth have a treelet is uneven, so far more waves than run at a time (8192)
      // even it out.  Commit of 1M triangles with 8192 / 16384 / 32768 / 65536 / any
      // number of waves: 6.58 / 5.48 / 4.99 / 4.81 / 4.94 ms.
      int per = (dcount[d] + 65535) / 65536;
      per = per < 64 ? per : 64;
      const int waves = (dcount[d] + per - 1) / per;
      const dim3 grid((waves + TWAVES - 1) / TWAVES), block(64 * TWAVES);
      if (round == 0)
        hipLaunchKernelGGL(k_treelet_level<true>, grid, block, 0, s, boxes_dev, (const int *)order,
                           (const int *)(hlist + dstart[d]), dcount[d], per, nodes, parent, ni, A, gamma);
      else
        hipLaunchKernelGGL(k_treelet_level<false>, grid, block, 0, s, boxes_dev, (const int *)order,
                           (const int *)(hlist + dstart[d]), dcount[d], per, nodes, parent, ni, A, gamma);
    }
    BVH_CHK(hipGetLastError());
  }
  BVH_CHK(sort_by_depth(ni, parent, t0, t1, t2, t3, hh, dcount, dstart, hlist, &depths, s));
  for (int d = depths - 1; d >= 0; d--)
    if (dcount[d] > 0)
      hipLaunchKernelGGL(k_refit_level, dim3((dcount[d] + GXY_BLOCK - 1) / GXY_BLOCK), dim3(GXY_BLOCK), 0, s, boxes_dev,
                         (const int *)order, nodes, (const int *)(hlist + dstart[d]), dcount[d], A);
  // 6: layout (leaf collapse, renumbering, primitive order)
  BVHNode *fin = (BVHNode *)P.get(sizeof(BVHNode) * (size_t)ni);
  int *neworder = (int *)P.get(sizeof(int) * (size_t)n);
  LayEnt *fa = (LayEnt *)P.get(sizeof(LayEnt) * (size_t)ni), *fb = (LayEnt *)P.get(sizeof(LayEnt) * (size_t)ni);
  int *lv = (int *)P.get(sizeof(int) * 2 * LEVELS), *bad = (int *)P.get(sizeof(int));
  if (!fin || !neworder || !fa || !fb || !lv || !bad) return hipErrorOutOfMemory;
  hipLaunchKernelGGL(k_levels_init, dim3(1), dim3(LV_BLOCK), 0, s, lv, bad, (int *)fa, (int)(sizeof(LayEnt) / 4));
  // (a level has at most the nodes of its depth)
  for (int d = 0; d < depths; d++) {
    hipLaunchKernelGGL(k_layout, dim3((dcount[d] + LV_BLOCK - 1) / LV_BLOCK), dim3(LV_BLOCK), 0, s, (const LayEnt *)fa,
                       d, lv, (const BVHNode *)nodes, n, (const int *)A.cnt, (const int *)A.leaf, (const int *)order,
                       fin, neworder, fb, bad, ni);
    LayEnt *t = fa;
    fa = fb;
    fb = t;
  }
  int hlv[LEVELS], hbad = 0, nn = 0, levels = 0;
  BVH_CHK(hipMemcpyAsync(&hbad, bad, sizeof hbad, hipMemcpyDeviceToHost, s));
  BVH_CHK(read_ints(lv, hlv, depths + 1, s));
  if (hbad != 0 || hlv[depths] != 0) return hipErrorInvalidValue;
  for (; levels < depths && hlv[levels] > 0; levels++) nn += hlv[levels];
  P.release(nodes);
  P.release(parent);
  P.release(t0);
  P.release(t1);
  P.release(t2);
  P.release(t3);
  // 7: 4-wide collapse
  BVH4Node *w4 = (BVH4Node *)P.get(sizeof(BVH4Node) * (size_t)nn);
  int *wa = (int *)P.get(sizeof(int) * (size_t)nn), *wb = (int *)P.get(sizeof(int) * (size_t)nn);
  if (!w4 || !wa || !wb) return hipErrorOutOfMemory;
  hipLaunchKernelGGL(k_levels_init, dim3(1), dim3(LV_BLOCK), 0, s, lv, bad, wa, 1);
  // (a level has at most four times the nodes of the one above, the tree at most the
  // binary one's levels; how many is known once a level is empty: looked up every 8)
  int nn4 = 0, wlevels = 0;
  int64_t bound = 1;
  for (int d = 0; d <= levels; d++) {
    if (d == levels || (d > 0 && d % 8 == 0)) {
      BVH_CHK(hipMemcpyAsync(&hbad, bad, sizeof hbad, hipMemcpyDeviceToHost, s));
      BVH_CHK(read_ints(lv, hlv, d + 1, s));
      if (hbad != 0) return hipErrorInvalidValue;
      if (hlv[d] == 0) break;
      if (d == levels) return hipErrorInvalidValue;
      bound = hlv[d];
    }
    hipLaunchKernelGGL(k_wide, dim3((unsigned)((bound + LV_BLOCK - 1) / LV_BLOCK)), dim3(LV_BLOCK), 0, s,
                       (const int *)wa, d, lv, (const BVHNode *)fin, w4, wb, nn, bad);
    bound = bound * 4 < nn ? bound * 4 : nn;
    int *t = wa;
    wa = wb;
    wb = t;
  }
  for (; wlevels < levels && hlv[wlevels] > 0; wlevels++) nn4 += hlv[wlevels];
  // SAH cost of the final binary tree, relative to the root's surface
  double *acc = (double *)P.get(sizeof(double));
  if (!acc) return hipErrorOutOfMemory;
  BVH_CHK(hipMemsetAsync(acc, 0, sizeof(double), s));
  hipLaunchKernelGGL(k_sah, dim3((nn + GXY_BLOCK - 1) / GXY_BLOCK), dim3(GXY_BLOCK), 0, s, (const BVHNode *)fin, nn,
                     prim_cost, acc);
  double sah = 0.0;
  BVHNode root;
  BVH_CHK(hipMemcpyAsync(&sah, acc, sizeof sah, hipMemcpyDeviceToHost, s));
  BVH_CHK(hipMemcpyAsync(&root, fin, sizeof root, hipMemcpyDeviceToHost, s));
  BVH_CHK(hipStreamSynchronize(s));
  float rl[3], rh[3];
  for (int a = 0; a < 3; a++) { rl[a] = fminf(root.lo0[a], root.lo1[a]); rh[a] = fmaxf(root.hi0[a], root.hi1[a]); }
  const float rx = rh[0] - rl[0], ry = rh[1] - rl[1], rz = rh[2] - rl[2];
  const double ra = (double)rx * ry + (double)ry * rz + (double)rz * rx;
  // hand the results over (the pool frees everything else)
  for (auto &q : P.held)
    if (q == fin || q == neworder || q == w4) q = nullptr;
  out->nodes = fin;
  out->order = neworder;
  out->nnodes = nn;
  out->depth = levels + 1;
  out->nodes4 = w4;
  out->nnodes4 = nn4;
  out->depth4 = wlevels;
  out->sah = ra > 0.0 ? (float)(sah / ra) : 0.f;
  out->leaves = 0;
  return hipGetLastError();
}

// Every child index in range, every node of both trees and every primitive
// reached exactly once from the root?  *ok = 0 when not (or when the marks'
// memory is not there).  Trees without nodes are not looked at.
hipError_t check_trees(const BVHNode *nodes, int nn, const BVH4Node *nodes4, int nn4, int nprim, alloc_fn_t alloc,
                       free_fn_t dfree, int *ok, hipStream_t s) {
  *ok = 0;
  Pool P{alloc, dfree, {}};
  const size_t n2 = nn > 0 ? (size_t)nn + nprim : 0, n4 = nn4 > 0 ? (size_t)nn4 + nprim : 0;
  if (n2 > INT32_MAX || n4 > INT32_MAX) return hipSuccess;
  int *marks = (int *)P.get(sizeof(int) * (1 + n2 + n4));   // the verdict, then the marks
  if (!marks) return hipSuccess;
  BVH_CHK(hipMemsetAsync(marks, 0, sizeof(int) * (1 + n2 + n4), s));
  int *m2 = marks + 1, *m4 = m2 + n2;
  auto grid = [](size_t n) { return dim3((unsigned)((n + GXY_BLOCK - 1) / GXY_BLOCK)); };
  if (n2) {
    hipLaunchKernelGGL(k_mark_binary, grid(nn), dim3(GXY_BLOCK), 0, s, nodes, nn, nprim, m2, marks);
    hipLaunchKernelGGL(k_check_marks, grid(n2), dim3(GXY_BLOCK), 0, s, (const int *)m2, (int)n2, marks);
  }
  if (n4) {
    hipLaunchKernelGGL(k_mark_wide, grid(4 * (size_t)nn4), dim3(GXY_BLOCK), 0, s, nodes4, nn4, nprim, m4, marks);
    hipLaunchKernelGGL(k_check_marks, grid(n4), dim3(GXY_BLOCK), 0, s, (const int *)m4, (int)n4, marks);
  }
  BVH_CHK(hipGetLastError());
  int bad = 1;
  BVH_CHK(read_ints(marks, &bad, 1, s));
  *ok = bad == 0;
  return hipSuccess;
}

}  // namespace gxy
