// batch.hip — batched passes: many uneven ray lists over many resident
// datasets, traced by one persistent launch per pass.
//
// A pass reads a device chunk table (list, source, start, count; at most CH
// rays per chunk, every ray of a chunk belongs to one list and one dataset)
// whose length lives in device memory.  The trace kernel is persistent: each
// wave pops the next chunk from a device work queue (one atomic per chunk),
// stages the dataset's transfer-function tables in its own LDS slice when the
// dataset changes, and runs the per-ray trace (TraceRays_TraceRays,
// SamplerTraceRays) on up to CH rays with its 64 lanes.  The post-pass then
// applies, per chunk, the reference's lighting sequence and spawns secondary
// rays (TraceRays.cpp:68-146), classifies (Renderer.cpp:304-454, with no
// neighbouring partition), accumulates terminated rays into the list's
// framebuffer (Renderer.cpp:456-502) or appends sampler particles
// (Sampler.cpp:51-89), and compacts spawned and kept rays into the next pass's
// ray pool with wave ballots; chunk offsets come from a device-count scan, so
// no pass needs the host, and a fixed sequence of passes can be captured in a
// HIP graph.  All kernels here are launched with fixed grids and read their
// work counts from device memory.
#include "light_dev.h"
#include "route_dev.h"
#include "march_dev.h"

namespace gxy {

#define BWAVES (GXY_BLOCK / 64)
// isovalue crossings a sampler ray follows within one pass before it is
// re-queued as a KEEP_HERE ray

__device__ __forceinline__ unsigned long long bl_lanemask_lt() {
  const int lane = threadIdx.x & 63;
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

__device__ __forceinline__ int first_lane_i(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Reads of tables that no kernel of the pass writes while it runs, through the
// constant address space: a wave-uniform address then becomes a scalar load
// into SGPRs instead of a vector load into every lane's VGPRs.
// (The address goes through readfirstlane and an integer so that the cast is
// not folded back into the generic pointer it came from.)
template <class T>
__device__ __forceinline__ const T &kconst(const T *p) {
  const unsigned long long a = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
  const __attribute__((address_space(4))) T *q =
      (const __attribute__((address_space(4))) T *)(((unsigned long long)hi << 32) | lo);
  return *(const T *)q;
}

// a RayList whose 25 array pointers are known to be global
__device__ __forceinline__ RayList_ispc rl_global(const RayList_ispc &S) {
  RayList_ispc R;
  R.ox = gptr(S.ox); R.oy = gptr(S.oy); R.oz = gptr(S.oz);
  R.dx = gptr(S.dx); R.dy = gptr(S.dy); R.dz = gptr(S.dz);
  R.nx = gptr(S.nx); R.ny = gptr(S.ny); R.nz = gptr(S.nz);
  R.sample = gptr(S.sample);
  R.r = gptr(S.r); R.g = gptr(S.g); R.b = gptr(S.b); R.o = gptr(S.o);
  R.sr = gptr(S.sr); R.sg = gptr(S.sg); R.sb = gptr(S.sb); R.so = gptr(S.so);
  R.t = gptr(S.t); R.tMax = gptr(S.tMax);
  R.x = gptr(S.x); R.y = gptr(S.y);
  R.type = gptr(S.type); R.term = gptr(S.term); R.classification = gptr(S.classification);
  return R;
}

__device__ __forceinline__ RayList_ispc chunk_rays(const BatchArgs &A, const BatchChunk &ch) {
  return rl_global(kconst(A.rls + ch.src));
}

// per-workgroup totals of the BS_* statistics, one slot per workgroup
__device__ __forceinline__ void block_partials(unsigned long long *v, int k0, int k1, unsigned long long *part,
                                               int nblocks, int q = 0) {
  __shared__ unsigned long long ws[BWAVES][BS_COUNT];
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0)
    for (int k = k0; k < k1; k++) ws[w][k] = v[k];
  __syncthreads();
  if (threadIdx.x < k1 - k0) {
    const int k = k0 + threadIdx.x;
    unsigned long long t = 0;
    for (int q = 0; q < BWAVES; q++) t += ws[q][k];
    part[(size_t)k * 4 * nblocks + (size_t)q * nblocks + blockIdx.x] = t;
  }
}

// voxel addressing of a dataset's volume (the SM codes of the trace kernels):
// bricked (8 or 4) with 32-bit offsets when the bricked copy allows them
// (DVolume::bsmall), else with 64-bit addresses (16 or 12), small linear (1),
// large linear (0)
__device__ __forceinline__ int chunk_layout(const TraceParams &P) { return sm_of(P.vv[0].vol); }

// Lanes per ray of the batched marches (march_dev.h): sampler lists hold random
// rays, and so may render lists.
#define BG_RENDER 4
#define BG_SAMPLE 8

// Whether a render chunk is marched with one lane per ray rather than BG_RENDER.
// Four lanes cost about 1.3 times the VALU work and pay by fetching fewer lines:
// the lanes of a ray share them, while 64 random rays touch 64 places per load.
// Rays that lie close together, as a camera's do, share lines without that, and
// so does everything in a volume that the L2 holds.  So the chunk's first rays are
// looked at: the mean distance, in voxels, of a ray to the next one in the list,
// halfway along primary rays and at the origins of shadow and AO rays (a parent's
// follow each other).  P.near (batch_near, runtime.cpp) has the distances, of
// primary and other rays, at which both forms take the same time.  A chunk of up
// to 64 / BG_RENDER rays is one round either way.
__device__ __forceinline__ bool one_lane_chunk(const TraceParams &P, const RayList_ispc &R, const BatchChunk &ch) {
  if (!P.vv[0].tf.bounded) return true;   // tables with infinities or NaN, as in launch_march
  if (ch.count <= 64 / BG_RENDER) return false;
  const bool primary = first_lane_i(gptr(R.type + ch.start)[0]) == RAY_PRIMARY;
  const float near = P.near[primary ? 0 : 1];
  if (near > 1e30f || near <= 0.f) return near > 0.f;
  const int lane = threadIdx.x & 63;
  float x = 0.f, y = 0.f, z = 0.f;
  int in = 0;
  if (lane < ch.count) {
    const unsigned k = (unsigned)lane;
    const f3 org = ray_org(R, ch.start, k), dir = ray_dir(R, ch.start, k);
    float t0, t1;
    box_clip(org, dir, P.blo, P.bhi, t0, t1);
    t0 = mxf(t0, gptr(R.t + ch.start)[k]);
    t1 = mnf(t1, gptr(R.tMax + ch.start)[k]);
    in = t0 <= t1;
    const float t = primary ? 0.5f * (t0 + t1) : t0;
    const VoxRay v = vox_ray(P.vv[0].vol, org, dir);
    x = __builtin_fmaf(t, v.b0, v.a0);
    y = __builtin_fmaf(t, v.b1, v.a1);
    z = __builtin_fmaf(t, v.b2, v.a2);
  }
  const float dx = fabsf(x - __shfl_down(x, 1, 64)), dy = fabsf(y - __shfl_down(y, 1, 64)),
              dz = fabsf(z - __shfl_down(z, 1, 64));
  const bool pair = lane < 63 && in && __shfl_down(in, 1, 64);
  float sum = pair ? mxf(dx, mxf(dy, dz)) : 0.f;
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  const int n = __popcll(__builtin_amdgcn_ballot_w64(pair));
  return __builtin_amdgcn_ballot_w64(sum < near * (float)n) != 0;
}

// The render rays of one volume chunk (MI = 1: the volume has at most one
// isovalue), with one lane per ray (a wave with primary and other rays runs the
// march of each kind) ...
template <int SM, int MI>
__device__ __forceinline__ unsigned long long render_chunk_one(const TraceParams &P, const RayList_ispc &R,
                                                               const BatchChunk &ch, const float (*col)[3 * GXY_TF_MAX],
                                                               const float (*op)[GXY_TF_MAX]) {
  unsigned long long n = 0;
  const int start = ch.start;
  NoStack stack;
  for (int k = threadIdx.x & 63; k < ch.count; k += 64) {
    if (gptr(R.type + start)[k] == RAY_PRIMARY) n += trace_one<1, false, SM, MI, 1>(P, R, start + k, col, op, stack);
    else n += trace_one<1, false, SM, MI, 2>(P, R, start + k, col, op, stack);
  }
  return n;
}
// ... and with BG_RENDER lanes per ray
template <int SM, int MI>
__device__ __forceinline__ unsigned long long render_chunk_group(const TraceParams &P, const RayList_ispc &R,
                                                                 const BatchChunk &ch,
                                                                 const float (*col)[3 * GXY_TF_MAX],
                                                                 const float (*op)[GXY_TF_MAX]) {
  unsigned long long n = 0;
  const int start = ch.start;
  for (int k = (threadIdx.x & 63) / BG_RENDER; k < ch.count; k += 64 / BG_RENDER) {
    if (gptr(R.type + start)[k] == RAY_PRIMARY)
      n += trace_group<BG_RENDER, SM, MI, true>(P, R, start, (unsigned)k, col[0], op[0]);
    else n += trace_group<BG_RENDER, SM, MI, false>(P, R, start, (unsigned)k, col[0], op[0]);
  }
  return n;
}
// by the chunk's layout (bricked volumes with more than one isovalue take the
// 64-bit variants, which serve any bricked copy)
#define GXY_BY_LAYOUT(F)                                                      \
  const int lay = chunk_layout(P);                                            \
  const bool one = P.vv[0].nIso <= 1;                                         \
  if (one && lay == 4) return F<4, 1>(P, R, ch, col, op);                     \
  if (one && lay == 12) return F<12, 1>(P, R, ch, col, op);                   \
  if (one && lay == 8) return F<8, 1>(P, R, ch, col, op);                     \
  if (one && lay == 16) return F<16, 1>(P, R, ch, col, op);                   \
  if (lay == 8 || lay == 16) return F<16, GXY_MAX_ISO>(P, R, ch, col, op);    \
  if (lay == 4 || lay == 12) return F<12, GXY_MAX_ISO>(P, R, ch, col, op);    \
  if (lay == 1) return F<1, GXY_MAX_ISO>(P, R, ch, col, op);                  \
  return F<0, GXY_MAX_ISO>(P, R, ch, col, op);
__device__ __forceinline__ unsigned long long render_chunk_one_any(const TraceParams &P, const RayList_ispc &R,
                                                                   const BatchChunk &ch,
                                                                   const float (*col)[3 * GXY_TF_MAX],
                                                                   const float (*op)[GXY_TF_MAX]) {
  GXY_BY_LAYOUT(render_chunk_one)
}
__device__ __forceinline__ unsigned long long render_chunk_group_any(const TraceParams &P, const RayList_ispc &R,
                                                                     const BatchChunk &ch,
                                                                     const float (*col)[3 * GXY_TF_MAX],
                                                                     const float (*op)[GXY_TF_MAX]) {
  GXY_BY_LAYOUT(render_chunk_group)
}
#undef GXY_BY_LAYOUT

// The sampler rays of one chunk, every crossing of each in this launch: samples
// and segments (counted as ray passes).
typedef unsigned long long SampleCounts __attribute__((ext_vector_type(2)));   // (returned in registers)
__device__ __forceinline__ SampleCounts sample_chunk(const TraceParams &P, const RayList_ispc &R, const BatchList &Ls,
                                                     int start, int count, int ms, float *buf) {
  float *xyz = gptr(Ls.xyz);
  int *pc = Ls.pcount;
  const int cap = Ls.pcap, lay = chunk_layout(P);
  ParticleBuffer B = {buf, 0};
  unsigned long long ns = 0, np = 0;
  if (lay == 4) sample_range<BG_SAMPLE, 4>(P, R, start, count, B, xyz, pc, cap, ms, ns, np);
  else if (lay == 8) sample_range<BG_SAMPLE, 8>(P, R, start, count, B, xyz, pc, cap, ms, ns, np);
  else if (lay == 16) sample_range<BG_SAMPLE, 16>(P, R, start, count, B, xyz, pc, cap, ms, ns, np);
  else if (lay == 12) sample_range<BG_SAMPLE, 12>(P, R, start, count, B, xyz, pc, cap, ms, ns, np);
  else if (lay == 1) sample_range<BG_SAMPLE, 1>(P, R, start, count, B, xyz, pc, cap, ms, ns, np);
  else sample_range<BG_SAMPLE, 0>(P, R, start, count, B, xyz, pc, cap, ms, ns, np);
  B.flush(xyz, pc, cap);
  return SampleCounts{ns, np};
}

// A wave's transfer-function tables: an LDS slice that the kernels fill and the
// called march below reads.
typedef float ChunkCol[3 * GXY_TF_MAX];
typedef float ChunkOp[GXY_TF_MAX];
__device__ __forceinline__ ChunkCol *wave_col() {
  __shared__ ChunkCol s_col[BWAVES];
  return s_col + (threadIdx.x >> 6);
}
__device__ __forceinline__ ChunkOp *wave_op() {
  __shared__ ChunkOp s_op[BWAVES];
  return s_op + (threadIdx.x >> 6);
}

// The kernel that takes chunks of every kind calls these three (one call a chunk)
// and has the one-lane march inlined.  With everything inlined it had 128 VGPRs
// and 187 spilled SGPRs (140 so), and the march of a long ray took 5 %
// longer.  The arguments arrive in VGPRs: uniform ones are read from the first lane.
#define GXY_CALLED __attribute__((noinline))
__device__ GXY_CALLED SampleCounts sample_chunk_call(const TraceParams *P, const RayList_ispc *R, const BatchList *Ls,
                                                     int start, int count, int ms) {
  __shared__ float s_part[BWAVES][3 * 64];
  return sample_chunk(kconst(P), rl_global(kconst(R)), kconst(Ls), first_lane_i(start), first_lane_i(count),
                      first_lane_i(ms), s_part[threadIdx.x >> 6]);
}
template <int STK>
__device__ __forceinline__ void geom_chunk(const TraceParams &P, const RayList_ispc &R, int start, int count) {
  constexpr int NL = STK > 0 ? STK : GXY_LDS_STACK;
  __shared__ int s_stack[NL][GXY_BLOCK];
  GXY_LDS int *base = (GXY_LDS int *)&s_stack[0][threadIdx.x];
  const int lane = threadIdx.x & 63;
  if (STK > 0 && P.model.wide != 1 && P.model.depth + 2 <= STK) {
    LdsStack<NL, GXY_BLOCK> stack;
    stack.base = base;
    for (int k = lane; k < count; k += 64) trace_geom_one<decltype(stack), 2>(P, R, start, k, stack);
    return;
  }
  HybStack<NL, GXY_BLOCK> stack;
  stack.base = base;
  const bool wide = P.model.wide == 1 || (P.model.wide == 2 && STK == 0);
  for (int k = lane; k < count; k += 64) {
    if (wide) trace_geom_one<decltype(stack), 4>(P, R, start, k, stack);
    else trace_geom_one<decltype(stack), 2>(P, R, start, k, stack);
  }
}
template <int STK>
__device__ GXY_CALLED void geom_chunk_call(const TraceParams *P, const RayList_ispc *R, int start, int count) {
  geom_chunk<STK>(kconst(P), rl_global(kconst(R)), first_lane_i(start), first_lane_i(count));
}
__device__ GXY_CALLED unsigned long long render_chunk_group_call(const TraceParams *P, const RayList_ispc *R, int start,
                                                                 int count) {
  BatchChunk ch;
  ch.start = first_lane_i(start);
  ch.count = first_lane_i(count);
  return render_chunk_group_any(kconst(P), rl_global(kconst(R)), ch, wave_col(), wave_op());
}

// ------------------------------------------------------------------ pass set-up
// work-queue head, per-list pending counts and the output count cleared
// (kernels, not memsets, so that the pass can be captured in a graph)
__global__ __launch_bounds__(1024) void k_bbegin(BatchArgs A) {
  if (threadIdx.x == 0) {
    *A.head = 0;
    *A.nout = 0;
    *A.nrays_out = 0;
  }
  if (threadIdx.x < 3) {
    A.kcount[threadIdx.x] = 0;
    A.khead[threadIdx.x] = 0;
  }
  for (int l = threadIdx.x; l < A.nlists; l += 1024) A.lpend[l] = 0;
  for (long long k = threadIdx.x; k < (long long)BS_COUNT * 4 * A.nblocks; k += 1024) A.part[k] = 0;
}

// kind of a chunk: 0 volume render, 1 geometry render, 2 sampler
__device__ __forceinline__ int chunk_kind(const BatchArgs &A, const BatchChunk &ch) {
  const BatchList &Ls = A.lists[ch.list];
  if (Ls.mode == BM_SAMPLE) return 2;
  return A.ds[Ls.ds].has_model ? 1 : 0;
}

// per-kind lists of the input chunks (order within a list is irrelevant)
__global__ __launch_bounds__(GXY_BLOCK) void k_bsplit(BatchArgs A) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int nin = *A.nin;
  for (int base = (blockIdx.x * BWAVES + w) * 64; base < nin; base += gridDim.x * BWAVES * 64) {
    const int c = base + lane;
    const int kind = c < nin ? chunk_kind(A, A.tin[c]) : -1;
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const unsigned long long m = __ballot(kind == q);
      if (!m) continue;
      int b0 = 0;
      if (lane == 0) b0 = atomicAdd(A.kcount + q, __popcll(m));
      b0 = first_lane_i(b0);
      if (kind == q) A.kidx[(size_t)q * A.kcap + b0 + __popcll(m & bl_lanemask_lt())] = c;
    }
  }
}

// appends n host-built chunks (already on the device) to the input table
__global__ __launch_bounds__(256) void k_bappend(BatchChunk *tab, int *ntab, int cap, const BatchChunk *add, int n,
                                                 int *overflow) {
  const int base = *ntab;
  for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += gridDim.x * 256) {
    if (base + k < cap) tab[base + k] = add[k];
  }
  __syncthreads();
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (base + n > cap) *overflow |= 2;
  }
}

__global__ void k_bappend_count(int *ntab, int cap, int n) {
  int v = *ntab + n;
  *ntab = v < cap ? v : cap;
}

__global__ void k_bset_count(int *ntab, int v) { *ntab = v; }

// ------------------------------------------------------------------ trace
// At least 4 waves per SIMD (128 VGPRs): with all kinds inlined the compiler takes
// 153 (3 waves) by itself, and 64 lists of 16K rays run 13.7 instead of 12.6 ms per
// flush.  More do not fit: the LDS of a workgroup (36 KB: transfer-function tables,
// particles, traversal stack) lets four onto a CU.
template <int STK>
__global__ __launch_bounds__(GXY_BLOCK) __attribute__((amdgpu_waves_per_eu(4, 8)))
void k_btrace(BatchArgs A) {
  const int lane = threadIdx.x & 63;
  const int nc = *A.nin;
  unsigned long long acc[BS_COUNT];
#pragma unroll
  for (int k = 0; k < BS_COUNT; k++) acc[k] = 0;
  int cur_tf = -1;
  for (;;) {
    int c = 0;
    if (lane == 0) c = atomicAdd(A.head, 1);
    c = first_lane_i(c);
    if (c >= nc) break;
    const BatchChunk ch = kconst(A.tin + c);
    const BatchList &Ls = kconst(A.lists + ch.list);
    const int ds = Ls.ds, mode = Ls.mode;
    const TraceParams &P = kconst(A.ds + ds);
    if (mode == BM_SAMPLE) {
      const SampleCounts n = sample_chunk_call(A.ds + ds, A.rls + ch.src, A.lists + ch.list, ch.start, ch.count,
                                               A.max_segments);
      acc[BS_SAMPLES] += n.x;
      acc[BS_RAYS] += n.y;
      continue;
    }
    acc[BS_RAYS] += lane < ch.count ? (ch.count - 1 - lane) / 64 + 1 : 0;
    if (P.has_model) {
      geom_chunk_call<STK>(A.ds + ds, A.rls + ch.src, ch.start, ch.count);
      continue;
    }
    if (ds != cur_tf) {
      const DTF &T = P.vv[0].tf;
      for (int k = lane; k < 3 * T.nc; k += 64) wave_col()[0][k] = T.col[k];
      for (int k = lane; k < T.no; k += 64) wave_op()[0][k] = T.op[k];
      wave_lds_sync();
      cur_tf = ds;
    }
    const RayList_ispc R = chunk_rays(A, ch);
    acc[BS_SAMPLES] += one_lane_chunk(P, R, ch)
                           ? render_chunk_one_any(P, R, ch, wave_col(), wave_op())
                           : render_chunk_group_call(A.ds + ds, A.rls + ch.src, ch.start, ch.count);
  }
  // lane sums of the sample and ray-pass counts
  acc[BS_SAMPLES] = wave_sum_u64(acc[BS_SAMPLES]);
  acc[BS_RAYS] = wave_sum_u64(acc[BS_RAYS]);
  block_partials(acc, BS_RAYS, BS_SAMPLES + 1, A.part, A.nblocks);
}

// ------------------------------------------------------------------ trace, one kernel per kind
// The same per-chunk work as k_btrace for the chunks of one kind (the list
// k_bsplit built), so that each kind gets its own register allocation and
// occupancy; the three kernels of a pass run concurrently on three streams.
template <int KIND, int STK, int WPE>
__global__ __launch_bounds__(GXY_BLOCK) __attribute__((amdgpu_waves_per_eu(WPE > 0 ? WPE : 1, 8)))
void k_btrace_kind(BatchArgs A) {
  __shared__ float s_part[BWAVES][KIND == 2 ? 3 * 64 : 1];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nk = A.kcount[KIND];
  const int *idx = A.kidx + (size_t)KIND * A.kcap;
  unsigned long long acc[BS_COUNT];
#pragma unroll
  for (int k = 0; k < BS_COUNT; k++) acc[k] = 0;
  int cur_tf = -1;
  for (;;) {
    int q = 0;
    if (lane == 0) q = atomicAdd(A.khead + KIND, 1);
    q = first_lane_i(q);
    if (q >= nk) break;
    const int c = first_lane_i(idx[q]);
    const BatchChunk ch = kconst(A.tin + c);
    const BatchList &Ls = kconst(A.lists + ch.list);
    const int ds = Ls.ds;
    const TraceParams &P = kconst(A.ds + ds);
    const RayList_ispc R = chunk_rays(A, ch);
    if (KIND == 2) {
      const SampleCounts n = sample_chunk(P, R, Ls, ch.start, ch.count, A.max_segments, s_part[w]);
      acc[BS_SAMPLES] += n.x;
      acc[BS_RAYS] += n.y;
      continue;
    }
    acc[BS_RAYS] += lane < ch.count ? (ch.count - 1 - lane) / 64 + 1 : 0;
    if (KIND == 1) {
      geom_chunk<STK>(P, R, ch.start, ch.count);
      continue;
    }
    if (ds != cur_tf) {
      const DTF &T = P.vv[0].tf;
      for (int k = lane; k < 3 * T.nc; k += 64) wave_col()[0][k] = T.col[k];
      for (int k = lane; k < T.no; k += 64) wave_op()[0][k] = T.op[k];
      wave_lds_sync();
      cur_tf = ds;
    }
    acc[BS_SAMPLES] += one_lane_chunk(P, R, ch) ? render_chunk_one_any(P, R, ch, wave_col(), wave_op())
                                                : render_chunk_group_any(P, R, ch, wave_col(), wave_op());
  }
  acc[BS_SAMPLES] = wave_sum_u64(acc[BS_SAMPLES]);
  acc[BS_RAYS] = wave_sum_u64(acc[BS_RAYS]);
  block_partials(acc, BS_RAYS, BS_SAMPLES + 1, A.part, A.nblocks, 1 + KIND);
}

// ------------------------------------------------------------------ post-pass: counts
struct ChunkFlags {
  bool valid, par, keep, term, drop, surf;
  int cls;
};

__device__ __forceinline__ ChunkFlags chunk_flags(const BatchArgs &A, const RayList_ispc &R, int mode, int i,
                                                  bool valid) {
  ChunkFlags f;
  f.valid = valid;
  f.par = f.keep = f.term = f.drop = f.surf = false;
  f.cls = 0;
  if (!valid) return f;
  const int typ = R.type[i], term = R.term[i];
  int c = classify_ray(typ, term, R.classification[i], A.L.reverse);
  // AssignDestinations with no neighbouring partition (Renderer.cpp:423-454)
  if (c == RAY_BOUNDARY)
    c = ((typ == RAY_SHADOW || typ == RAY_AO) && A.L.reverse) ? GXY_DROP_ON_FLOOR : GXY_TERMINATED;
  f.cls = c;
  f.par = mode == BM_RENDER && typ == RAY_PRIMARY && (term & RAY_SURFACE);
  f.keep = c == GXY_KEEP_HERE;
  f.term = c == GXY_TERMINATED;
  f.drop = c == GXY_DROP_ON_FLOOR;
  f.surf = (term & RAY_SURFACE) != 0;
  return f;
}

__global__ __launch_bounds__(GXY_BLOCK) void k_bcount(BatchArgs A) {
  const int lane = threadIdx.x & 63;
  const int nc = *A.nin;
  const int gw = blockIdx.x * BWAVES + (threadIdx.x >> 6), nw = gridDim.x * BWAVES;
  const int nsp = A.L.nAO + (A.L.doShadows ? A.L.nLights : 0);
  for (int c = gw; c < nc; c += nw) {
    const BatchChunk ch = A.tin[c];
    const int mode = A.lists[ch.list].mode;
    const RayList_ispc R = chunk_rays(A, ch);
    int npar = 0, nkeep = 0;
    for (int k0 = 0; k0 < ch.count; k0 += 64) {
      const int k = k0 + lane;
      ChunkFlags f = chunk_flags(A, R, mode, ch.start + k, k < ch.count);
      npar += __popcll(__ballot(f.par));
      nkeep += __popcll(__ballot(f.keep));
    }
    if (lane == 0) {
      const int out = npar * nsp + nkeep;
      A.cpar[c] = npar;
      A.cout[c] = out;
      A.cchk[c] = (out + A.chunk - 1) / A.chunk;
      if (out) atomicAdd(A.lpend + ch.list, out);
    }
  }
}

// ------------------------------------------------------------------ device-count scan
// Exclusive scan of (cout, cchk) over the nin input chunks: NSEG workgroups,
// each owning one contiguous segment.
#define BSCAN_SEG 256

__global__ __launch_bounds__(256) void k_bscan_a(BatchArgs A) {
  __shared__ long long sr[4], sc[4];
  const int n = *A.nin;
  const int seg = (n + BSCAN_SEG - 1) / BSCAN_SEG;
  const int s0 = min(n, blockIdx.x * seg), s1 = min(n, s0 + seg);
  long long r = 0, c = 0;
  for (int k = s0 + threadIdx.x; k < s1; k += 256) {
    r += A.cout[k];
    c += A.cchk[k];
  }
  for (int o = 32; o > 0; o >>= 1) {
    r += __shfl_xor(r, o);
    c += __shfl_xor(c, o);
  }
  if ((threadIdx.x & 63) == 0) {
    sr[threadIdx.x >> 6] = r;
    sc[threadIdx.x >> 6] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    A.segr[blockIdx.x] = sr[0] + sr[1] + sr[2] + sr[3];
    A.segc[blockIdx.x] = sc[0] + sc[1] + sc[2] + sc[3];
  }
}

__global__ __launch_bounds__(BSCAN_SEG) void k_bscan_b(BatchArgs A) {
  __shared__ long long pr[BSCAN_SEG], pc[BSCAN_SEG];
  const int t = threadIdx.x;
  pr[t] = A.segr[t];
  pc[t] = A.segc[t];
  __syncthreads();
  for (int o = 1; o < BSCAN_SEG; o <<= 1) {
    long long vr = t >= o ? pr[t - o] : 0, vc = t >= o ? pc[t - o] : 0;
    __syncthreads();
    pr[t] += vr;
    pc[t] += vc;
    __syncthreads();
  }
  A.segr[t] = t > 0 ? pr[t - 1] : 0;
  A.segc[t] = t > 0 ? pc[t - 1] : 0;
  if (t == BSCAN_SEG - 1) {
    const long long rays = pr[t], chunks = pc[t];
    bool over = rays > A.pool_cap || chunks > A.tcap;
    if (over) *A.overflow |= 1;
    *A.nrays_out = over ? 0 : (int)rays;
    *A.nout = over ? 0 : (int)chunks;
  }
}

__global__ __launch_bounds__(256) void k_bscan_c(BatchArgs A) {
  __shared__ long long wr[4], wc[4];
  __shared__ long long carry_r, carry_c;
  const int n = *A.nin;
  const int seg = (n + BSCAN_SEG - 1) / BSCAN_SEG;
  const int s0 = min(n, blockIdx.x * seg), s1 = min(n, s0 + seg);
  if (threadIdx.x == 0) {
    carry_r = A.segr[blockIdx.x];
    carry_c = A.segc[blockIdx.x];
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int b = s0; b < s1; b += 256) {
    const int k = b + threadIdx.x;
    long long r = k < s1 ? A.cout[k] : 0, c = k < s1 ? A.cchk[k] : 0;
    // inclusive wave scan
    long long ir = r, ic = c;
    for (int o = 1; o < 64; o <<= 1) {
      long long vr = __shfl_up(ir, o), vc = __shfl_up(ic, o);
      if (lane >= o) {
        ir += vr;
        ic += vc;
      }
    }
    if (lane == 63) {
      wr[w] = ir;
      wc[w] = ic;
    }
    __syncthreads();
    long long br = carry_r, bc = carry_c;
    for (int q = 0; q < w; q++) {
      br += wr[q];
      bc += wc[q];
    }
    if (k < s1) {
      A.coff[k] = (int)(br + ir - r);
      A.cchkoff[k] = (int)(bc + ic - c);
    }
    __syncthreads();
    if (threadIdx.x == 255) {
      carry_r = br + ir;
      carry_c = bc + ic;
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ post-pass: writes
__device__ __forceinline__ void copy_ray(const RayList_ispc &S, int i, const RayList_ispc &D, int j) {
  D.ox[j] = S.ox[i]; D.oy[j] = S.oy[i]; D.oz[j] = S.oz[i];
  D.dx[j] = S.dx[i]; D.dy[j] = S.dy[i]; D.dz[j] = S.dz[i];
  D.nx[j] = S.nx[i]; D.ny[j] = S.ny[i]; D.nz[j] = S.nz[i];
  D.sample[j] = S.sample[i];
  D.r[j] = S.r[i]; D.g[j] = S.g[i]; D.b[j] = S.b[i]; D.o[j] = S.o[i];
  D.sr[j] = S.sr[i]; D.sg[j] = S.sg[i]; D.sb[j] = S.sb[i]; D.so[j] = S.so[i];
  D.t[j] = S.t[i]; D.tMax[j] = S.tMax[i];
  D.x[j] = S.x[i]; D.y[j] = S.y[i];
  D.type[j] = S.type[i]; D.term[j] = S.term[i]; D.classification[j] = S.classification[i];
}

#define BATCH_MAX_CHUNK 1024

// Per chunk (one wave): (1) rank the parents and keep their ray offsets in
// the wave's LDS slice; (2) write every child, one lane per child at
// base + p * (nAO + nLights) + j (AO children first, then shadow children of
// the p-th parent), from the parents' unmodified fields, so that consecutive
// lanes store consecutive children; (3) per ray: the parent's ambient and
// diffuse update, framebuffer accumulation of terminated rays (after that
// update), keepers copied after the children, sampler particles.
__global__ __launch_bounds__(GXY_BLOCK) void k_bwrite(BatchArgs A) {
  __shared__ int s_pl[BWAVES][BATCH_MAX_CHUNK];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int nc = *A.nin;
  const bool over = *A.overflow != 0;
  const int gw = blockIdx.x * BWAVES + w, nw = gridDim.x * BWAVES;
  const int nLs = A.L.doShadows ? A.L.nLights : 0;
  const int nAO = A.L.nAO;
  const int nsp = nAO + nLs;
  const RayList_ispc O = rl_global(kconst(A.rls + A.out_pool));
  unsigned long long acc[BS_COUNT];
#pragma unroll
  for (int k = 0; k < BS_COUNT; k++) acc[k] = 0;
  for (int c = gw; c < nc; c += nw) {
    const BatchChunk ch = A.tin[c];
    const BatchList &Ls = A.lists[ch.list];
    const int mode = Ls.mode;
    const RayList_ispc R = chunk_rays(A, ch);
    const int base = A.coff[c], npar = A.cpar[c];
    const int keep_base = base + npar * nsp;
    // (1) parents in rank order
    int par_run = 0;
    if (mode == BM_RENDER && nsp > 0) {
      for (int k0 = 0; k0 < ch.count; k0 += 64) {
        const int k = k0 + lane;
        ChunkFlags f = chunk_flags(A, R, mode, ch.start + k, k < ch.count);
        const unsigned long long mp = __ballot(f.par);
        if (f.par) s_pl[w][par_run + __popcll(mp & bl_lanemask_lt())] = k;
        par_run += __popcll(mp);
      }
      wave_lds_sync();
      // (2) children
      if (!over) {
        for (int q = lane; q < npar * nsp; q += 64) {
          const int p = q / nsp, j = q - p * nsp;
          const ParentRay P = parent_load(R, ch.start + s_pl[w][p]);
          if (j < nAO) light_ao_child(A.L, P, j, O, base + q);
          else light_shadow_child(A.L, P, A.L.reverse ? light_diffused_alpha(A.L, P.o) : P.o, j - nAO, O, base + q);
        }
      }
      wave_lds_sync();   // the slice is rewritten by the next chunk
    }
    // (3) parents' colours, accumulation, keepers, particles
    int keep_run = 0;
    for (int k0 = 0; k0 < ch.count; k0 += 64) {
      const int k = k0 + lane, i = ch.start + k;
      ChunkFlags f = chunk_flags(A, R, mode, i, k < ch.count);
      const unsigned long long mp = __ballot(f.par), mk = __ballot(f.keep);
      const unsigned long long mt = __ballot(f.term), md = __ballot(f.drop);
      const int krank = keep_run + __popcll(mk & bl_lanemask_lt());
      if (!over) {
        if (mode == BM_RENDER) {
          int x = 0, y = 0;
          float cr = 0.f, cg = 0.f, cb = 0.f, co = 0.f;
          if (f.par) {
            // ambientLighting + diffuseLighting (TraceRays.cpp:124-131); without
            // reverse lighting only those whose rays are not cast (:133-141)
            ParentRay P = parent_load(R, i);
            if (A.L.reverse || A.L.nAO <= 0) light_ambient(A.L, P);
            if (A.L.reverse || !(A.L.doShadows && A.L.nLights > 0)) light_diffuse(A.L, P);
            R.r[i] = P.r; R.g[i] = P.g; R.b[i] = P.b; R.o[i] = P.o;
            if (f.term) {
              x = P.px; y = P.py;
              cr = P.r; cg = P.g; cb = P.b; co = P.o;
            }
          } else if (f.term) {
            x = R.x[i];
            y = R.y[i];
            cr = R.r[i];
            cg = R.g[i];
            cb = R.b[i];
            co = R.o[i];
          }
          fb_accumulate_wave(Ls.fb, Ls.width, Ls.height, f.term, x, y, cr, cg, cb, co);
        }
        if (f.keep) copy_ray(R, i, O, keep_base + krank);
        if (mode == BM_SAMPLE) {
          // Sampler::HandleTerminatedRays (Sampler.cpp:71-84): a particle at o + t*d
          const unsigned long long ms = __ballot(f.surf);
          int pbase = 0;
          if (lane == 0 && ms) pbase = atomicAdd(Ls.pcount, __popcll(ms));
          pbase = first_lane_i(pbase);
          if (f.surf) {
            const int off = pbase + __popcll(ms & bl_lanemask_lt());
            if (off < Ls.pcap) {
              const float t = R.t[i];
              Ls.xyz[3 * (int64_t)off + 0] = R.ox[i] + t * R.dx[i];
              Ls.xyz[3 * (int64_t)off + 1] = R.oy[i] + t * R.dy[i];
              Ls.xyz[3 * (int64_t)off + 2] = R.oz[i] + t * R.dz[i];
            }
          }
        }
      }
      acc[BS_SPAWNED] += (unsigned long long)__popcll(mp) * nsp;
      acc[BS_TERMINATED] += __popcll(mt);
      acc[BS_DROPPED] += __popcll(md);
      acc[BS_KEPT] += __popcll(mk);
      keep_run += __popcll(mk);
    }
    if (!over) {
      const int total = npar * nsp + keep_run;
      const int nch = A.cchk[c], cb = A.cchkoff[c];
      for (int q = lane; q < nch; q += 64) {
        BatchChunk o;
        o.src = A.out_pool;
        o.start = base + q * A.chunk;
        o.count = min(A.chunk, total - q * A.chunk);
        o.list = ch.list;
        A.tout[cb + q] = o;
      }
    }
  }
  block_partials(acc, BS_SPAWNED, BS_COUNT, A.part, A.nblocks);
}

// adds the per-workgroup partials of every statistic into A.stats
__global__ __launch_bounds__(1024) void k_breduce(BatchArgs A, int k0, int k1) {
  __shared__ unsigned long long ws[16];
  for (int k = k0; k < k1; k++) {
    unsigned long long v = 0;
    for (int b = threadIdx.x; b < 4 * A.nblocks; b += 1024) v += A.part[(size_t)k * 4 * A.nblocks + b];
    v = wave_sum_u64(v);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned long long t = 0;
      for (int q = 0; q < 16; q++) t += ws[q];
      A.stats[k] += t;
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ synthetic ray lists
// Random rays of one list: origins uniform in [lo, hi], isotropic directions
// (z = 1 - 2u, phi = 2 pi u'), t = 0, tMax = inf, pixel x = index % width,
// y = index / width; a PCG hash of (seed, ray index, draw) gives the uniforms.
__device__ __forceinline__ unsigned pcg_hash(unsigned v) {
  unsigned s = v * 747796405u + 2891336453u;
  unsigned w = ((s >> ((s >> 28u) + 4u)) ^ s) * 277803737u;
  return (w >> 22u) ^ w;
}

__device__ __forceinline__ float u01(unsigned seed, unsigned i, unsigned k) {
  unsigned h = pcg_hash(seed ^ pcg_hash(i * 8u + k + 0x9e3779b9u * (seed + 1u)));
  return (float)(h >> 8) * (1.0f / 16777216.0f);
}

__global__ __launch_bounds__(GXY_BLOCK) void k_random_rays(RayList_ispc R, int n, unsigned seed, int width, int type,
                                                           float lx, float ly, float lz, float hx, float hy,
                                                           float hz) {
  const int i = blockIdx.x * GXY_BLOCK + threadIdx.x;
  if (i >= n) return;
  float ux = u01(seed, i, 0), uy = u01(seed, i, 1), uz = u01(seed, i, 2);
  float zc = 1.0f - 2.0f * u01(seed, i, 3), ph = 6.2831855f * u01(seed, i, 4);
  float rr = sqrtf(fmaxf(0.f, 1.0f - zc * zc));
  R.ox[i] = lx + ux * (hx - lx);
  R.oy[i] = ly + uy * (hy - ly);
  R.oz[i] = lz + uz * (hz - lz);
  R.dx[i] = rr * cosf(ph);
  R.dy[i] = rr * sinf(ph);
  R.dz[i] = zc;
  R.nx[i] = 0.f; R.ny[i] = 0.f; R.nz[i] = 0.f;
  R.sample[i] = 0.f;
  R.r[i] = 0.f; R.g[i] = 0.f; R.b[i] = 0.f; R.o[i] = 0.f;
  R.sr[i] = 0.f; R.sg[i] = 0.f; R.sb[i] = 0.f; R.so[i] = 0.f;
  R.t[i] = 0.f;
  R.tMax[i] = __builtin_inff();
  R.x[i] = width > 0 ? i % width : i;
  R.y[i] = width > 0 ? i / width : 0;
  R.type[i] = type;
  R.term[i] = 0;
  R.classification[i] = 0;
}

__global__ __launch_bounds__(256) void k_fill_f32(float *p, long long n, float v) {
  for (long long k = (long long)blockIdx.x * 256 + threadIdx.x; k < n; k += (long long)gridDim.x * 256) p[k] = v;
}
__global__ void k_fill_i32_one(int *p, int v) { *p = v; }

// ------------------------------------------------------------------ launchers
template <int STK>
static void btrace_as(const BatchArgs &A, int blocks, hipStream_t s) {
  hipLaunchKernelGGL((k_btrace<STK>), dim3(blocks), dim3(GXY_BLOCK), 0, s, A);
}

template <int KIND, int STK, int WPE>
static void bkind_as(const BatchArgs &A, int blocks, hipStream_t s) {
  hipLaunchKernelGGL((k_btrace_kind<KIND, STK, WPE>), dim3(blocks), dim3(GXY_BLOCK), 0, s, A);
}

static void launch_split_trace(const BatchArgs &A, const BatchLaunch &K, hipStream_t s, const hipStream_t *ks,
                               const hipEvent_t *ev) {
  const int tb = K.trace_blocks;
  hipLaunchKernelGGL(k_bsplit, dim3(K.post_blocks), dim3(GXY_BLOCK), 0, s, A);
  (void)hipEventRecord(ev[0], s);
  for (int q = 0; q < 3; q++) (void)hipStreamWaitEvent(ks[q], ev[0], 0);
  // volume render: occupancy request 5 or 6 waves per SIMD when asked (LDS TF slices only)
  if (K.wpe == 6) bkind_as<0, 0, 6>(A, tb, ks[0]);
  else if (K.wpe == 5) bkind_as<0, 0, 5>(A, tb, ks[0]);
  else if (K.wpe == 4) bkind_as<0, 0, 4>(A, tb, ks[0]);
  else bkind_as<0, 0, 0>(A, tb, ks[0]);
  if (K.stack == 16) bkind_as<1, 16, 0>(A, tb, ks[1]);
  else if (K.stack == 24) bkind_as<1, 24, 0>(A, tb, ks[1]);
  else if (K.stack == 32) bkind_as<1, 32, 0>(A, tb, ks[1]);
  else bkind_as<1, 0, 0>(A, tb, ks[1]);
  bkind_as<2, 0, 8>(A, tb, ks[2]);
  for (int q = 0; q < 3; q++) {
    (void)hipEventRecord(ev[1 + q], ks[q]);
    (void)hipStreamWaitEvent(s, ev[1 + q], 0);
  }
}

hipError_t launch_batch_pass(const BatchArgs &A, const BatchLaunch &K, hipStream_t s, const hipStream_t *ks,
                             const hipEvent_t *ev) {
  hipLaunchKernelGGL(k_bbegin, dim3(1), dim3(1024), 0, s, A);
  const int tb = K.trace_blocks;
  if (K.split && ks && ev) {
    launch_split_trace(A, K, s, ks, ev);
  } else if (K.stack == 16) btrace_as<16>(A, tb, s);
  else if (K.stack == 24) btrace_as<24>(A, tb, s);
  else if (K.stack == 32) btrace_as<32>(A, tb, s);
  else btrace_as<0>(A, tb, s);
  hipLaunchKernelGGL(k_bcount, dim3(K.post_blocks), dim3(GXY_BLOCK), 0, s, A);
  hipLaunchKernelGGL(k_bscan_a, dim3(BSCAN_SEG), dim3(256), 0, s, A);
  hipLaunchKernelGGL(k_bscan_b, dim3(1), dim3(BSCAN_SEG), 0, s, A);
  hipLaunchKernelGGL(k_bscan_c, dim3(BSCAN_SEG), dim3(256), 0, s, A);
  hipLaunchKernelGGL(k_bwrite, dim3(K.post_blocks), dim3(GXY_BLOCK), 0, s, A);
  return hipGetLastError();
}

hipError_t launch_batch_reduce(const BatchArgs &A, hipStream_t s) {
  hipLaunchKernelGGL(k_breduce, dim3(1), dim3(1024), 0, s, A, 0, (int)BS_COUNT);
  return hipGetLastError();
}

hipError_t launch_batch_append(BatchChunk *tab, int *ntab, int cap, const BatchChunk *add, int n, int *overflow,
                               hipStream_t s) {
  if (n <= 0) return hipSuccess;
  int g = (n + 255) / 256;
  if (g > 1024) g = 1024;
  hipLaunchKernelGGL(k_bappend, dim3(g), dim3(256), 0, s, tab, ntab, cap, add, n, overflow);
  hipLaunchKernelGGL(k_bappend_count, dim3(1), dim3(1), 0, s, ntab, cap, n);
  return hipGetLastError();
}

hipError_t launch_set_count(int *p, int v, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_i32_one, dim3(1), dim3(1), 0, s, p, v);
  return hipGetLastError();
}

hipError_t launch_fill_f32(float *p, long long n, float v, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  long long g = (n + 255) / 256;
  if (g > 8192) g = 8192;
  hipLaunchKernelGGL(k_fill_f32, dim3((unsigned)g), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

hipError_t launch_random_rays(const RayList_ispc &R, int n, unsigned seed, int width, int type, const float *lo,
                              const float *hi, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_random_rays, dim3((n + GXY_BLOCK - 1) / GXY_BLOCK), dim3(GXY_BLOCK), 0, s, R, n, seed, width,
                     type, lo[0], lo[1], lo[2], hi[0], hi[1], hi[2]);
  return hipGetLastError();
}

}  // namespace gxy
