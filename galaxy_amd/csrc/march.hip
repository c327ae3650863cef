// march.hip — TraceRays_TraceRays over one volume without geometry, several lanes
// per ray.
#include "march_dev.h"
#include "trace_kernel.h"

namespace gxy {

// What bounds a march of one ray per lane (k_trace) is the serial chain of each
// ray once the queue of waves is empty, and lanes that wait for the longest of
// 64 rays before; small lists are nothing but that chain.  G lanes per ray cut
// the chain to a G-th and the divergence to 64 / G rays per wave, at about 1.7
// times the VALU work per sample (G = 4): positions cost G adds, compositing is
// done by every lane of the group, and a wave sets up fewer rays at once.
// 76 VGPRs, six waves per SIMD.  Trace per frame, one lane -> this kernel:
// 128x128 through 64^3 0.148 -> 0.039 ms (G = 16), 256x256 through 128^3 0.226 ->
// 0.078 (16), 512x512 through 256^3 0.37 -> 0.20 (4), 1920x1080 through 512^3
// 0.90 -> 0.67 (4; G = 2 0.74, 8 0.98), 800x600 with 8 AO rays per hit 0.67 ->
// 0.58 (4).
template <int G, int SM, int MI>
__global__ __launch_bounds__(GXY_BLOCK) __attribute__((amdgpu_waves_per_eu(6, 8)))
void k_march(TraceParams P, RayList_ispc R, int n) {
  __shared__ float s_col[3 * GXY_TF_MAX];
  __shared__ float s_op[GXY_TF_MAX];
  constexpr int RAYS = GXY_BLOCK / G;
  const int blk = xcd_block<8>();
  // a launch queued before its list's size was known covers the capacity
  if (P.dn) n = min(n, *P.dn * P.dn_mul);
  if (blk >= (n + RAYS - 1) / RAYS) return;
  for (int k = threadIdx.x; k < 3 * P.vv[0].tf.nc; k += GXY_BLOCK) s_col[k] = P.vv[0].tf.col[k];
  for (int k = threadIdx.x; k < P.vv[0].tf.no; k += GXY_BLOCK) s_op[k] = P.vv[0].tf.op[k];
  __syncthreads();
  const int first = blk * RAYS;
  const unsigned i = threadIdx.x / G;
  unsigned long long nsamp = 0;
  if ((int)i < n - first) {
    if (gptr(R.type + first)[i] == RAY_PRIMARY) nsamp = trace_group<G, SM, MI, true>(P, R, first, i, s_col, s_op);
    else nsamp = trace_group<G, SM, MI, false>(P, R, first, i, s_col, s_op);
  }
  if (P.sample_count) wave_add_count(nsamp, P.sample_count);
}

template <int G>
static void launch_march_lanes(const TraceParams &P, const RayList_ispc &R, int n, hipStream_t s) {
  const dim3 g((unsigned)(((long long)n * G + GXY_BLOCK - 1) / GXY_BLOCK)), b(GXY_BLOCK);
  const int sm = sm_of(P.vv[0].vol);
  if (P.vv[0].nIso <= 1 && sm != 0) {
    switch (sm) {
      case 1: hipLaunchKernelGGL((k_march<G, 1, 1>), g, b, 0, s, P, R, n); break;
      case 4: hipLaunchKernelGGL((k_march<G, 4, 1>), g, b, 0, s, P, R, n); break;
      case 8: hipLaunchKernelGGL((k_march<G, 8, 1>), g, b, 0, s, P, R, n); break;
      case 12: hipLaunchKernelGGL((k_march<G, 12, 1>), g, b, 0, s, P, R, n); break;
      default: hipLaunchKernelGGL((k_march<G, 16, 1>), g, b, 0, s, P, R, n); break;
    }
    return;
  }
  // (several isovalues: the 64-bit brick variants serve any bricked copy)
  switch (sm) {
    case 0: hipLaunchKernelGGL((k_march<G, 0, GXY_MAX_ISO>), g, b, 0, s, P, R, n); break;
    case 1: hipLaunchKernelGGL((k_march<G, 1, GXY_MAX_ISO>), g, b, 0, s, P, R, n); break;
    case 4:
    case 12: hipLaunchKernelGGL((k_march<G, 12, GXY_MAX_ISO>), g, b, 0, s, P, R, n); break;
    default: hipLaunchKernelGGL((k_march<G, 16, GXY_MAX_ISO>), g, b, 0, s, P, R, n); break;
  }
}

// Lanes per ray for a list of at most n rays, dn_mul of them per parent, whose
// box is `steps` march steps long.  A large list of short rays keeps the chip's
// VALUs busy with one lane per ray; the fewer rays there are for the length of
// their chains, the more lanes each gets.  The lines lie where the two sides
// measure alike (512x288 to 1440x1080 pixels through 48^3 to 512^3, trace per
// frame): at 2750 rays per step G = 4 against 2 0.207 / 0.271 ms below
// (960x540, 192^3) and 0.204 / 0.188 above (1280x720, 96^3); at 5000 G = 2
// against one lane 0.482 / 0.558 below (1440x1080, 192^3) and 0.256 / 0.239
// above (96^3).  Up to 2^16 rays leave SIMDs idle even so: G = 16.  AO lists hold
// incoherent rays, one lane's divergence costs them more, and their capacity is
// several times their size: a quarter of it counts (8 AO rays per hit, 800x600
// through 201x157x120: 0.63 ms with four or two lanes, 0.67 with one).
int march_lanes(int n, int dn_mul, float steps) {
  if (n <= (1 << 16)) return 16;
  const float rays = dn_mul > 1 ? 0.25f * (float)n : (float)n;
  if (rays <= 2750.f * steps) return 4;
  return rays <= 5000.f * steps ? 2 : 1;
}

bool launch_march(const TraceParams &P, const RayList_ispc &R, int n, hipStream_t s) {
  // (weights of 0 stand for samples that do not count, so the tables must be
  // finite; the one-lane march branches around such samples)
  if (P.nvv != 1 || P.has_model || !P.vv[0].tf.bounded || !P.integrate) return false;
  float edge = 0.f;
  for (int a = 0; a < 3; a++) edge = std::max(edge, P.bhi[a] - P.blo[a]);
  const float steps = P.step > 0.f ? edge / P.step : 0.f;
  switch (march_lanes(n, P.dn ? P.dn_mul : 1, steps)) {
    case 2: launch_march_lanes<2>(P, R, n, s); return true;
    case 4: launch_march_lanes<4>(P, R, n, s); return true;
    case 16: launch_march_lanes<16>(P, R, n, s); return true;
  }
  return false;
}

}  // namespace gxy
