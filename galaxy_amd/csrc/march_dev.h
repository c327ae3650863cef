// march_dev.h — volume marches with several lanes per ray.
//
// One lane per ray leaves a march with a serial chain per sample (gathers, the
// interpolation, the test) and 64 rays' samples spread over 64 places of the
// volume in every load.  The samples of a ray do not depend on each other, only
// on its positions t, and those are a chain of two cheap instructions per step.
// So G adjacent lanes share a ray here: lane j takes every G-th position,
// starting at the j-th, and what depends on the order (the first crossing) is
// settled between the lanes each round.  The positions are the ones that the
// one-lane march reaches, added up step by step in the same order, so results
// are bit-identical for every G.
#pragma once

#include "trace_dev.h"

namespace gxy {

// Lane j of its group of G (G = 2, 4, 8 or 16 adjacent lanes).
template <int G>
__device__ __forceinline__ int group_lane() { return threadIdx.x & (G - 1); }
// the value of the lane before this one (lane 0 of a row of 16 keeps its own)
__device__ __forceinline__ float dpp_prev(float v) {
  const int i = __float_as_int(v);
  return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x111, 0xf, 0xf, false));
}
// the value of the group's last lane, in lane 0 (other lanes: some lane's value)
template <int G>
__device__ __forceinline__ float dpp_last_to_first(float v) {
  constexpr int ctrl = G == 2 ? 0xB1 : G == 4 ? 0x1B : G == 8 ? 0x141 : 0x140;   // quad, half-row and row mirrors
  const int i = __float_as_int(v);
  return __int_as_float(__builtin_amdgcn_update_dpp(i, i, ctrl, 0xf, 0xf, false));
}
// the group's bits of a wave mask, bit 0 its first lane
template <int G>
__device__ __forceinline__ unsigned group_bits(unsigned long long m) {
  return (unsigned)(m >> ((threadIdx.x & 63) & ~(G - 1))) & ((1u << G) - 1u);
}

// The next round's positions of a lane: G steps on from t, added one by one, and
// the one before.  Positions past the limit are cut to it once, after the adds
// (the chain never comes back from beyond it).
template <int G>
__device__ __forceinline__ void group_advance(float t, float first_step, float step, float lim, float &tn, float &tpn) {
  tn = t;
#pragma unroll
  for (int k = 0; k < G; k++) {
    tpn = tn;
    tn += k == 0 ? first_step : step;
  }
  tn = __builtin_fminf(tn, lim);
  tpn = __builtin_fminf(tpn, lim);
}

// sample_one of one volume with G lanes per ray (every lane of the group calls
// it with the same i).  Position T_0 is the entry point and T_k+1 = min(T_k +
// step, tExit); the march ends where that no longer advances.
template <int G, int SM>
__device__ __forceinline__ unsigned sample_group(const TraceParams &P, const RayList_ispc &R, const int i) {
  const int j = group_lane<G>();
  const DVolume &V = P.vv[0].vol;
  f3 org = mk3(gptr(R.ox)[i], gptr(R.oy)[i], gptr(R.oz)[i]);
  f3 dir = mk3(gptr(R.dx)[i], gptr(R.dy)[i], gptr(R.dz)[i]);
  const float rt = gptr(R.t)[i];
  if (dir.x == 0.f) dir.x = 1e-6f;
  if (dir.y == 0.f) dir.y = 1e-6f;
  if (dir.z == 0.f) dir.z = 1e-6f;
  float tEntry, tExit;
  box_clip(org, dir, P.blo, P.bhi, tEntry, tExit);
  if (tEntry < rt) tEntry = rt;
  const float step = P.step, iso = P.vv[0].iso[0];
  const VoxRay VR = vox_ray(V, org, dir);
  // the first step is not cut at the exit: a ray whose first step leaves takes
  // no step at all (its chain stays at the entry)
  const bool go0 = tEntry + step <= tExit;
  const float lim = go0 ? tExit : tEntry;
  float t = tEntry, tp = tEntry;
#pragma unroll
  for (int k = 1; k < G; k++)
    if (k <= j) {
      tp = t;
      t += step;
    }
  t = __builtin_fminf(t, lim);
  tp = __builtin_fminf(tp, lim);
  VFetch F = vox_fetch<SM>(V, VR, t);
  float sEnd = 0.f;   // lane 0: the last lane's sample of the round before
  unsigned nsamp = j == 0 ? 1u : 0u;
  // (round `iter` holds positions iter .. iter + G - 1; at most GXY_MAX_MARCH
  // samples after the first, a multiple of G)
  for (int iter = 0;; iter += G) {
    // the next round's positions, and its gathers before this round's samples are used
    float tn, tpn;
    group_advance<G>(t, step, step, lim, tn, tpn);
    const float s = vol_finish_fma(F);
    F = vox_fetch<SM>(V, VR, tn);
    const float sl0 = dpp_prev(s);
    const float sl = j == 0 ? sEnd : sl0;
    sEnd = dpp_last_to_first<G>(s);
    const bool live = t > tp && (iter < GXY_MAX_MARCH || j == 0);   // (T_0 ends no interval: tp = t)
    const bool cross = live && ((sl < iso && s >= iso) || (sl > iso && s <= iso));
    const unsigned cm = group_bits<G>(__builtin_amdgcn_ballot_w64(cross));
    const int hit = cm ? __builtin_ctz(cm) : G;
    nsamp += (live && j <= hit) ? 1u : 0u;
    if (cm) {
      if (j == hit) {
        const float tHit = tp + (((iso - sl) / (s - sl)) * (t - tp));
        gptr(R.t)[i] = tHit + 0.001f;
        gptr(R.term)[i] = RAY_SURFACE;
      }
      break;
    }
    // lane 0's next position is the one after this round's last
    if (!(group_bits<G>(__builtin_amdgcn_ballot_w64(tn > tpn)) & 1u)) {
      if (j == G - 1) {
        gptr(R.t)[i] = go0 ? t : tEntry + step;
        gptr(R.term)[i] = RAY_BOUNDARY;
      }
      break;
    }
    if (iter >= GXY_MAX_MARCH) {
      if (j == 1) {
        gptr(R.t)[i] = t;
        gptr(R.term)[i] = RAY_BOUNDARY;
      }
      break;
    }
    t = tn;
    tp = tpn;
  }
  return nsamp;
}

}  // namespace gxy
