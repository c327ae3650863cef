// trace_geom.hip — TraceRays_TraceRays over geometry without volumes: one
// work-item per ray, BVH walk, shading of primary rays' hits.
#include <type_traits>

#include "trace_dev.h"

namespace gxy {

// W: the walk (trace_dev.h); NL: stack entries in LDS; WPE: waves per SIMD asked
// for; BS: work-items per workgroup; LDS: the stack has no other entries.
//
// Bound by VALU issue (about 0.7 of it on the nine-icosphere AO pass, a wave's
// lanes being at different nodes: lane utilisation 0.41), then by the latency of
// the node loads.  So the walk is the 4-wide one with few instructions per node
// (1.6 against 2.7 K VALU instructions per launched wave for the binary walk
// with a private stack), its live registers are kept to 78 (6 waves per SIMD
// without spills; 8 waves spill and lose 2x), and a workgroup is one wave, so
// that a SIMD takes new rays as soon as a wave's longest walk ends.
// Trace time per frame, binary walk with a private stack before -> this kernel:
// nine icospheres 11.8 M triangles 3840x2160 with 16 AO rays 8.36 -> 5.45 ms,
// 200 K spheres 1024^2 with 4 AO rays 1.57 -> 1.06 ms, 4000 path lines 1024^2
// 2.08 -> 1.50 ms, 20 K triangles 512^2 0.25 -> 0.16 ms.  With 256-item
// workgroups: 5.60, 1.11, 1.61 and 0.16 ms; 12 or 24 stack entries in LDS are
// within 1 % of 16.
template <int W, int NL, int WPE, int BS, bool LDS>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(WPE > 0 ? WPE : 1, 8)))
void k_geom(TraceParams P, RayList_ispc R, int n) {
  __shared__ int s_stack[NL][BS];
  // a launch queued before its list's size was known covers the capacity
  if (P.dn) n = min(n, *P.dn * P.dn_mul);
  const int first = blockIdx.x * BS;
  if (first >= n || (int)threadIdx.x >= n - first) return;
  typename std::conditional<LDS, LdsStack<NL, BS>, HybStack<NL, BS>>::type stack;
  stack.base = (GXY_LDS int *)&s_stack[0][threadIdx.x];
  trace_geom_one<decltype(stack), W>(P, R, first, threadIdx.x, stack);
}

template <int W, int NL, int WPE, int BS, bool LDS = false>
static void launch_geom(const TraceParams &P, const RayList_ispc &R, int n, hipStream_t s) {
  const unsigned nb = (unsigned)(((long long)n + BS - 1) / BS);
  hipLaunchKernelGGL((k_geom<W, NL, WPE, BS, LDS>), dim3(nb), dim3(BS), 0, s, P, R, n);
}

// The 4-wide walk wherever the model's trees allow it (make_trace_params); the
// binary one for trees too deep or too large for it, or when one of its
// settings asks for it.  An LDS stack setting that holds the tree's depth + 2 needs
// no private entries and takes one-wave workgroups (32 entries, frames: nine
// icospheres of 20 K triangles 1024^2 with 4 AO rays 1005 -> 863 us, 985 with
// 256-item workgroups; 20 K triangles 512x512 301 -> 298).  Path-line models
// take the variants that trace curve pieces (W = 16 + width).
hipError_t launch_trace_geom(const TraceParams &P, const RayList_ispc &R, int n, int stack, int gwaves,
                             hipStream_t s) {
  const bool curves = P.model.ncurve > 0;
  if (P.model.wide == 1 || (P.model.wide == 2 && stack == 0 && gwaves == 0)) {
    if (curves) launch_geom<20, GXY_LDS_STACK, 6, 64>(P, R, n, s);
    else launch_geom<4, GXY_LDS_STACK, 6, 64>(P, R, n, s);
  } else if (curves) {
    if (gwaves == 8) launch_geom<18, GXY_LDS_STACK, 8, GXY_BLOCK>(P, R, n, s);
    else launch_geom<18, GXY_LDS_STACK, 0, GXY_BLOCK>(P, R, n, s);
  } else if (P.model.depth + 2 <= stack) {
    if (stack == 16) launch_geom<2, 16, 0, 64, true>(P, R, n, s);
    else if (stack == 24) launch_geom<2, 24, 0, 64, true>(P, R, n, s);
    else launch_geom<2, 32, 0, 64, true>(P, R, n, s);
  } else {
    if (stack == 24) launch_geom<2, 24, 0, GXY_BLOCK>(P, R, n, s);
    else if (stack == 32) launch_geom<2, 32, 0, GXY_BLOCK>(P, R, n, s);
    else if (gwaves == 8 && stack == 0) launch_geom<2, GXY_LDS_STACK, 8, GXY_BLOCK>(P, R, n, s);
    else launch_geom<2, GXY_LDS_STACK, 0, GXY_BLOCK>(P, R, n, s);
  }
  return hipGetLastError();
}

}  // namespace gxy
