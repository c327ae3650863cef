// sampler.hip — SamplerTraceRays_SamplerTraceRays on gfx950.
#include "march_dev.h"
#include "trace_kernel.h"

namespace gxy {

// several volumes: one ray per lane (the crossings of all of them compete for
// the same positions)
template <int NV, int SM>
__global__ __launch_bounds__(GXY_BLOCK) void k_sampler(TraceParams P, RayList_ispc R, int n) {
  const int i = blockIdx.x * GXY_BLOCK + threadIdx.x;
  unsigned long long nsamp = 0;
  if (i < n) nsamp = sample_one<NV, SM>(P, R, i);
  if (P.sample_count) wave_add_count(nsamp, P.sample_count);
}

// One volume, G lanes per ray.  The sampler's rays are random: 64 of them per
// wave read 64 places of the volume per load, march as long as the longest of
// 64 and fetch each line again and again (the one-lane march was bound by line
// fetches and by its longest rays).  With G = 8 a wave holds eight rays whose
// lanes read neighbouring cells: 1 M rays through 256^3 6.2 -> 3.5 ms per
// gxy_sample_raylist (4^3 bricks) and 12.4 -> 5.5 ms (linear), 2 M rays through
// 400^3 18.4 -> 8.7 ms, 2 M through 48^3 3.1 -> 2.3 ms.  Lanes past the crossing
// sample in vain (G / 2 samples per segment of about 60), and positions cost G
// adds per lane: G = 16 takes 3.6, 5.8, 8.7 and 2.5 ms there, G = 4 3.6, 5.8,
// 9.8 and 2.4 ms.  Below 2^16 rays the waves of G = 8 leave SIMDs idle and the
// longest ray is all that counts: 20 K rays through 256^3 take 2.53 ms with one
// lane, 1.05 with eight, 0.97 with sixteen.
template <int G, int SM>
__global__ __launch_bounds__(GXY_BLOCK) void k_sampler_group(TraceParams P, RayList_ispc R, int n) {
  const int first = (int)(blockIdx.x * (GXY_BLOCK / G));
  const unsigned k = threadIdx.x / G;
  unsigned long long nsamp = 0;
  if ((int)k < n - first) nsamp = sample_group<G, SM>(P, R, first, k);
  if (P.sample_count) wave_add_count(nsamp, P.sample_count);
}

template <int G>
static void launch_sampler_group(const TraceParams &P, const RayList_ispc &R, int n, hipStream_t s) {
  dim3 g((unsigned)(((long long)n * G + GXY_BLOCK - 1) / GXY_BLOCK)), b(GXY_BLOCK);
  switch (sm_of(P.vv[0].vol)) {
    case 4: hipLaunchKernelGGL((k_sampler_group<G, 4>), g, b, 0, s, P, R, n); break;
    case 8: hipLaunchKernelGGL((k_sampler_group<G, 8>), g, b, 0, s, P, R, n); break;
    case 12: hipLaunchKernelGGL((k_sampler_group<G, 12>), g, b, 0, s, P, R, n); break;
    case 16: hipLaunchKernelGGL((k_sampler_group<G, 16>), g, b, 0, s, P, R, n); break;
    case 1: hipLaunchKernelGGL((k_sampler_group<G, 1>), g, b, 0, s, P, R, n); break;
    default: hipLaunchKernelGGL((k_sampler_group<G, 0>), g, b, 0, s, P, R, n); break;
  }
}

hipError_t launch_sampler(const TraceParams &P, const RayList_ispc &R, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (P.nvv == 1) {
    if (n <= (1 << 16)) launch_sampler_group<16>(P, R, n, s);
    else launch_sampler_group<8>(P, R, n, s);
    return hipGetLastError();
  }
  dim3 g((n + GXY_BLOCK - 1) / GXY_BLOCK), b(GXY_BLOCK);
  bool small = P.nvv > 0;
  for (int v = 0; v < P.nvv && v < GXY_MAX_VOLVIS; v++) small = small && P.vv[v].vol.small;
  switch (P.nvv * 2 + (small ? 1 : 0)) {
    case 4: hipLaunchKernelGGL((k_sampler<2, -1>), g, b, 0, s, P, R, n); break;
    case 5: hipLaunchKernelGGL((k_sampler<2, 1>), g, b, 0, s, P, R, n); break;
    case 6: hipLaunchKernelGGL((k_sampler<3, -1>), g, b, 0, s, P, R, n); break;
    case 7: hipLaunchKernelGGL((k_sampler<3, 1>), g, b, 0, s, P, R, n); break;
    case 8: hipLaunchKernelGGL((k_sampler<4, -1>), g, b, 0, s, P, R, n); break;
    case 9: hipLaunchKernelGGL((k_sampler<4, 1>), g, b, 0, s, P, R, n); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace gxy
