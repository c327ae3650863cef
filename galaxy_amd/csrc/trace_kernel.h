// trace_kernel.h — the one-ray-per-work-item trace kernel of scenes with volumes
// (trace.hip instantiates it).
#pragma once

#include "trace_dev.h"

namespace gxy {

// A per-item count added to the counters at ctr: the wave's total, one 64-bit
// atomic per wave to the workgroup's slot (every lane of the wave calls it).
// With one counter for all, a 1 M-ray sampler loop at 8 lanes per ray (440 K
// waves) took 6.8 ms, with the slots 3.5.
__device__ __forceinline__ void wave_add_count(unsigned long long v, unsigned long long *ctr) {
  v = wave_sum_u64(v);
  if ((threadIdx.x & 63) == 0 && v) atomicAdd(ctr + (blockIdx.x % GXY_COUNT_SLOTS) * GXY_COUNT_STRIDE, v);
}

// WPE > 0 asks the compiler for at least WPE waves per SIMD (fewer VGPRs);
// the autotuner picks the variant.
// SM = 1 when every volume is small (32-bit voxel offsets), -1 otherwise.
// MI: isovalues per volume the iso test is unrolled for (1 when no volume
// has more than one, fewer scalar branches per sample).
// BS: work-items per workgroup (64, 128 or 256).  A workgroup's slots are
// refilled only as a whole, so smaller workgroups let a SIMD take new rays as
// soon as one wave's rays are done, at the price of staging the transfer
// function tables once per wave.
// Workgroups reach the eight XCDs (one L2 each) round robin; this renumbering
// hands each XCD runs of C consecutive workgroups' rays instead (neighbouring
// camera tiles read the same bricks), the runs still dealt round robin so the
// XCDs' shares of the image stay alike.  C = 1 is the dispatch order itself;
// the workgroups past the last whole round of 8*C keep their own numbers.
template <int C>
__device__ __forceinline__ int xcd_block() {
  const int b = blockIdx.x;
  if (C <= 1) return b;
  const int full = (int)gridDim.x / (8 * C) * (8 * C);
  if (b >= full) return b;
  const int x = b & 7, j = b >> 3;
  return ((j / C) * 8 + x) * C + j % C;
}

template <int NV, bool GEOM, int WPE, int SM, int MI = GXY_MAX_ISO, int BS = GXY_BLOCK>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(WPE > 0 ? WPE : 1, 8)))
void k_trace(TraceParams P, RayList_ispc R, int n) {
  constexpr int NVS = NV > 0 ? NV : 1;
  __shared__ float s_col[NVS][3 * GXY_TF_MAX];
  __shared__ float s_op[NVS][GXY_TF_MAX];
  // a launch queued before its list's size was known covers the capacity:
  // workgroups past the size leave at once (before staging the TF tables)
  const int blk = xcd_block<(NV > 0 && !GEOM) ? 8 : 1>();
  if (P.dn) {
    n = min(n, *P.dn * P.dn_mul);
    if (blk * BS >= n) return;
  }
#pragma unroll
  for (int v = 0; v < NV; v++) {
    for (int k = threadIdx.x; k < 3 * P.vv[v].tf.nc; k += BS) s_col[v][k] = P.vv[v].tf.col[k];
    for (int k = threadIdx.x; k < P.vv[v].tf.no; k += BS) s_op[v][k] = P.vv[v].tf.op[k];
  }
  if (NV > 0) __syncthreads();

  const int i = blk * BS + threadIdx.x;
  unsigned long long nsamp = 0;
  if constexpr (GEOM) {
    __shared__ int s_stack[GXY_LDS_STACK][BS];
    HybStack<GXY_LDS_STACK, BS> stack;
    stack.base = (GXY_LDS int *)&s_stack[0][threadIdx.x];
    if (i < n) nsamp = trace_one<NV, true, SM, MI>(P, R, i, s_col, s_op, stack);
  } else if (i < n) {
    NoStack stack;
    if (NV == 0) {
      nsamp = trace_one<NV, false, SM, MI>(P, R, i, s_col, s_op, stack);
    } else {
      // a wave whose rays are all primary, or all not, takes the march
      // compiled for that kind (lists of one kind are the usual case)
      const unsigned long long pm = __builtin_amdgcn_ballot_w64(gptr(R.type)[i] == RAY_PRIMARY);
      const unsigned long long am = __builtin_amdgcn_ballot_w64(true);
      if (pm == am) nsamp = trace_one<NV, false, SM, MI, 1>(P, R, i, s_col, s_op, stack);
      else if (pm == 0) nsamp = trace_one<NV, false, SM, MI, 2>(P, R, i, s_col, s_op, stack);
      else nsamp = trace_one<NV, false, SM, MI>(P, R, i, s_col, s_op, stack);
    }
  }
  if (P.sample_count) wave_add_count(nsamp, P.sample_count);
}

}  // namespace gxy
