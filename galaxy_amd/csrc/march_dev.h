// march_dev.h — volume marches with several lanes per ray, shared by the
// one-list kernels (sampler.hip, march.hip) and the batched kernels (batch.hip).
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

// LDS writes of one wave become visible to its other lanes
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

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

// the value of lane k of the group, in all its lanes
template <int G>
__device__ __forceinline__ float dpp_bcast(float v, int k) {
  const int i = __float_as_int(v);
  int r = i;
  // (k is a constant once the loops around the calls are unrolled)
#define GXY_BC(K)                                                                            \
  if (k == K) {                                                                              \
    if (G == 2) r = __builtin_amdgcn_mov_dpp(i, (K & 1) ? 0xF5 : 0xA0, 0xf, 0xf, false);     \
    else if (G == 4) r = __builtin_amdgcn_mov_dpp(i, (K & 3) * 0x55, 0xf, 0xf, false);       \
    else if (G == 16) r = __builtin_amdgcn_mov_dpp(i, 0x150 + (K & 15), 0xf, 0xf, false);    \
    else {                                                                                   \
      r = __builtin_amdgcn_update_dpp(i, i, 0x150 + (K & 7), 0xf, 0x3, false);               \
      r = __builtin_amdgcn_update_dpp(r, i, 0x158 + (K & 7), 0xf, 0xc, false);               \
    }                                                                                        \
  }
  GXY_BC(0) GXY_BC(1) GXY_BC(2) GXY_BC(3) GXY_BC(4) GXY_BC(5) GXY_BC(6) GXY_BC(7)
  GXY_BC(8) GXY_BC(9) GXY_BC(10) GXY_BC(11) GXY_BC(12) GXY_BC(13) GXY_BC(14) GXY_BC(15)
#undef GXY_BC
  return __int_as_float(r);
}

// One march of SamplerTraceRays through one volume with G lanes per ray: from t
// = rt (or the box's entry) to the next crossing of the first isovalue, or out.
// Position T_0 is the entry point and T_k+1 = min(T_k + step, tExit); the march
// ends where that no longer advances.  tBox, tExit: the box clip of the ray; rt:
// its t before and after (the crossing + 0.001, or where it left), in all lanes
// of the group, as is the returned flag of a crossing.  nsamp: this lane's
// samples.
template <int G, int SM>
__device__ __forceinline__ bool sample_segment(const TraceParams &P, const VoxRay &VR, float tBox, float tExit,
                                               float &rt, unsigned &nsamp) {
  const int j = group_lane<G>();
  const DVolume &V = P.vv[0].vol;
  float tEntry = tBox;
  if (tEntry < rt) tEntry = rt;
  const float step = P.step, iso = P.vv[0].iso[0];
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
  nsamp += j == 0 ? 1u : 0u;
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
      const float tHit = tp + (((iso - sl) / (s - sl)) * (t - tp));
      rt = __shfl(tHit, ((threadIdx.x & 63) & ~(G - 1)) + hit, 64) + 0.001f;
      return true;
    }
    // (the last round's position is lane 0's: the march stops at the one after it)
    if (iter >= GXY_MAX_MARCH) {
      rt = dpp_bcast<G>(t, 1);
      return false;
    }
    // lane 0's next position is the one after this round's last
    if (!(group_bits<G>(__builtin_amdgcn_ballot_w64(tn > tpn)) & 1u)) {
      rt = go0 ? dpp_bcast<G>(t, G - 1) : tEntry + step;
      return false;
    }
    t = tn;
    tp = tpn;
  }
}

// sample_one of one volume with G lanes per ray (every lane of the group calls
// it for the same ray, the k-th after the uniform `first`).
template <int G, int SM>
__device__ __forceinline__ unsigned sample_group(const TraceParams &P, const RayList_ispc &R, const int first,
                                                 const unsigned k) {
  const f3 org = ray_org(R, first, k), dir = ray_dir(R, first, k);
  float rt = gptr(R.t + first)[k];
  float tBox, tExit;
  box_clip(org, dir, P.blo, P.bhi, tBox, tExit);
  unsigned nsamp = 0;
  const bool hit = sample_segment<G, SM>(P, vox_ray(P.vv[0].vol, org, dir), tBox, tExit, rt, nsamp);
  if (group_lane<G>() == 0) {
    gptr(R.t + first)[k] = rt;
    gptr(R.term + first)[k] = hit ? RAY_SURFACE : RAY_BOUNDARY;
  }
  return nsamp;
}

// The particles of one wave on their way to a list's array: kept in LDS (buf,
// 64 of them) and appended 64 at a time, so that the waves of a list do not queue
// on its counter for every crossing.  Every lane of the wave makes each call.
struct ParticleBuffer {
  float *buf;   // 3 x 64 floats of the wave
  int count;    // uniform
  __device__ __forceinline__ void flush(float *xyz, int *pcount, int pcap) {
    if (count == 0) return;
    const int lane = threadIdx.x & 63;
    int off = 0;
    if (lane == 0) off = atomicAdd(pcount, count);
    off = __builtin_amdgcn_readfirstlane(off);
    if (lane < count && off + lane < pcap) {
      float *p = xyz + 3 * (int64_t)(off + lane);
      for (int a = 0; a < 3; a++) p[a] = buf[64 * a + lane];
    }
    count = 0;
    wave_lds_sync();
  }
  __device__ __forceinline__ void add(bool f, f3 p, float *xyz, int *pcount, int pcap) {
    const unsigned long long m = __builtin_amdgcn_ballot_w64(f);
    const int n = __popcll(m);
    if (n == 0) return;
    if (count + n > 64) flush(xyz, pcount, pcap);
    if (f) {
      const int lane = threadIdx.x & 63;
      const int k = count + __popcll(m & ((1ull << lane) - 1ull));
      buf[k] = p.x;
      buf[64 + k] = p.y;
      buf[128 + k] = p.z;
    }
    count += n;
    wave_lds_sync();
  }
};

// The sampler loop without re-queueing for `count` rays after `first` (uniform),
// by one wave: SamplerTraceRays marches to the next isovalue crossing,
// Sampler::HandleTerminatedRays appends the particle at o + t*d (t = crossing +
// 0.001, Sampler.cpp:71-84), and the ray continues from there (the KEEP_HERE
// re-trace of Renderer.cpp:659-691) until it leaves the volume.  Every segment is
// one ray pass with the samples of sample_one, so counts and particles equal
// those of the per-list loop (the particles' order differs).  After max_segments
// segments a ray is left as a SURFACE ray for the caller to re-queue (its
// particle not yet emitted).  A group whose ray is done takes the next ray of the
// range, while the others go on.
template <int G, int SM>
__device__ __forceinline__ void sample_range(const TraceParams &P, const RayList_ispc &R, const int first,
                                             const int count, ParticleBuffer &B, float *xyz, int *pcount, int pcap,
                                             int max_segments, unsigned long long &samples,
                                             unsigned long long &passes) {
  const int lane = threadIdx.x & 63, j = group_lane<G>();
  const unsigned long long heads = G == 2 ? 0x5555555555555555ull : G == 4 ? 0x1111111111111111ull
                                   : G == 8 ? 0x0101010101010101ull : 0x0001000100010001ull;
  int next = 0;            // uniform: rays handed out
  bool busy = false;
  unsigned k = 0, nsamp = 0;
  int segs = 0;
  f3 org = mk3(0.f, 0.f, 0.f), dir = org;   // dir as stored (the particle's), not the march's
  VoxRay VR = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float rt = 0.f, tBox = 0.f, tExit = 0.f;
  for (;;) {
    const unsigned long long idle = __builtin_amdgcn_ballot_w64(!busy) & heads;
    if (idle && next < count) {
      const int q = next + __popcll(idle & ((1ull << (lane & ~(G - 1))) - 1ull));
      if (!busy && q < count) {
        busy = true;
        k = (unsigned)q;
        segs = 0;
        org = ray_org(R, first, k);
        const f3 d = ray_dir(R, first, k);
        dir = mk3(gptr(R.dx + first)[k], gptr(R.dy + first)[k], gptr(R.dz + first)[k]);
        rt = gptr(R.t + first)[k];
        box_clip(org, d, P.blo, P.bhi, tBox, tExit);
        VR = vox_ray(P.vv[0].vol, org, d);
      }
      next += __popcll(idle);
    }
    if (!__builtin_amdgcn_ballot_w64(busy)) break;
    bool emit = false;
    f3 p = org;
    if (busy) {
      const bool hit = sample_segment<G, SM>(P, VR, tBox, tExit, rt, nsamp);
      segs++;
      passes += j == 0 ? 1u : 0u;
      if (hit && segs < max_segments) {
        emit = j == 0;
        p = mk3(org.x + rt * dir.x, org.y + rt * dir.y, org.z + rt * dir.z);
      } else {
        busy = false;
        if (j == 0) {
          gptr(R.t + first)[k] = rt;
          gptr(R.term + first)[k] = hit ? RAY_SURFACE : RAY_BOUNDARY;
        }
      }
    }
    B.add(emit, p, xyz, pcount, pcap);
  }
  samples += nsamp;
}

// trace_one of one volume without geometry, with G lanes per ray (every lane of
// the group calls it for the same ray, the k-th after ray `first`, which is
// uniform over the wave).  Position T_0 is the entry point, T_1 = T_0 + epsilon,
// T_k+1 = min(T_k + step, tTermination); the samples at T_k are taken side by
// side, and their colours are composited in order: each round every lane applies
// the samples of its group's lanes up to its own, one after another, to the
// colour at the round's start, so that lane j holds the colour after its sample.
// The first lane whose sample crosses an isovalue or makes the ray opaque ends
// the march and writes the ray.  (A lane past it, or one whose sample has no
// opacity, applies weight 0, which changes nothing as long as the tables and
// the ray's alpha are finite: the launcher checks the tables, `odd` the rays.)
// shade: the rays are primary (a wave with both kinds runs this once for each).
template <int G, int SM, int MI, bool shade>
__device__ __forceinline__ unsigned trace_group(const TraceParams &P, const RayList_ispc &R, const int first,
                                                const unsigned i, const float *s_col, const float *s_op) {
  const int j = group_lane<G>();
  const DVolVis &VV = P.vv[0];
  const DVolume &V = VV.vol;
  const DTF &T = VV.tf;
  unsigned nsamp = 0;
  float ray_t0 = gptr(R.t + first)[i];
  float ray_t = gptr(R.tMax + first)[i];
  float cr = gptr(R.r + first)[i], cg = gptr(R.g + first)[i], cb = gptr(R.b + first)[i], ca = gptr(R.o + first)[i];
  // Only what the march needs stays in registers through it (six waves per
  // SIMD): the ray's origin and direction, its slice's normal and colour are
  // read or formed again afterwards.
  VoxRay VR;
  float tEntry, tExitVolume;
  int slice = -1;
  {
    const f3 org = ray_org(R, first, i), dir = ray_dir(R, first, i);
    box_clip(org, dir, P.blo, P.bhi, tEntry, tExitVolume);
    if (tEntry < ray_t0) tEntry = ray_t0;
    else if (tEntry > ray_t0) ray_t0 = tEntry;
    ray_t = mnf(ray_t, tExitVolume);
    // LookForSliceHit (TraceRays.ispc:143-250)
    for (int m = 0; m < VV.nSlices; m++) {
      const f3 pn = mk3(VV.slices[4 * m], VV.slices[4 * m + 1], VV.slices[4 * m + 2]);
      const float denom = dot3(dir, pn);
      if (fabsf(denom) > 0.0001f) {
        const float t = (VV.slices[4 * m + 3] - dot3(org, pn)) / denom;
        if (t >= ray_t0 && t <= ray_t) {
          ray_t = t;
          slice = m;
        }
      }
    }
    VR = vox_ray(V, org, dir);
  }

  float tTermination = ray_t;
  bool owner = j == G - 1, hit_iso = false;
  float hit_sample = 0.f;
  if (P.integrate && tEntry <= tTermination && !opaque_of(cr, cg, cb, ca, P.opaque_alpha)) {
    const float step = P.step, eps = P.eps;
    const bool odd = __builtin_amdgcn_ballot_w64(!(fabsf(ca) < 1e30f)) != 0;
    const float T1 = tEntry + eps;
    const float lim = (T1 > tEntry && T1 <= tTermination) ? tTermination : tEntry;
    float t = j == 0 ? tEntry : T1, tp = tEntry;
#pragma unroll
    for (int k = 2; k < G; k++)
      if (k <= j) {
        tp = t;
        t += step;
      }
    t = __builtin_fminf(t, lim);
    tp = __builtin_fminf(tp, lim);
    VFetch F = vox_fetch<SM>(V, VR, t);
    float sEnd = 0.f, tThis;
    float fstep = j == 0 ? eps : step;   // (the step after T_0 is epsilon)
    nsamp = j == 0 ? 1u : 0u;
    int iter = 0, hI, end;
    bool go;
    do {
      if (VV.dvr) {
        // the colour after the last round
        cr = dpp_bcast<G>(cr, G - 1);
        cg = dpp_bcast<G>(cg, G - 1);
        cb = dpp_bcast<G>(cb, G - 1);
        ca = dpp_bcast<G>(ca, G - 1);
      }
      // this round's samples; the next round's gathers before they are used
      float tn, tpn;
      group_advance<G>(t, fstep, step, lim, tn, tpn);
      fstep = step;
      float s = vol_finish_fma(F);
      F = vox_fetch<SM>(V, VR, tn);
      const float sl0 = dpp_prev(s);
      const float sl = j == 0 ? sEnd : sl0;
      sEnd = dpp_last_to_first<G>(s);
      const bool step_ok = t > tp;
      const bool live = step_ok && tp >= eps;
      // LookForIsoHit: the last matching isovalue in list order wins
      bool ih = false;
#pragma unroll
      for (int m = 0; m < MI; m++)
        if (m < VV.nIso) {
          const float iso = VV.iso[m];
          if (((iso >= sl) && (iso < s)) || ((iso <= sl) && (iso > s))) {
            ih = live;
            hit_sample = iso;
          }
        }
      tThis = t;
      hI = G;
      const unsigned long long im = __builtin_amdgcn_ballot_w64(ih);
      if (im) {
        const unsigned b = group_bits<G>(im);
        hI = b ? __builtin_ctz(b) : G;
        if (j == hI) {
          tThis = tp + ((hit_sample - sl) / (s - sl)) * (t - tp);
          s = vox_sample<SM>(V, VR, tThis);
        }
      }
      end = hI;
      if (VV.dvr) {
        const float d = (sl + s) - T.lo2;
        float w = tf_opacity_d2(s_op, T, d);
        w = live && j <= hI && w > 0.f ? clamp01f(w * V.irate) : 0.f;
        const bool some = w != 0.f;
        if (__builtin_amdgcn_ballot_w64(some)) {
          if (shade) {
            const f3 sc = tf_color_num_d2(s_col, T, d);
            if (!odd) {
#pragma unroll
              for (int k = 0; k < G; k++) {
                const float wk0 = dpp_bcast<G>(w, k);
                const float wk = k <= j ? wk0 : 0.f;
                const float a = 1.0f - ca, aw = a * wk;
                cr = __builtin_fmaf(aw, dpp_bcast<G>(sc.x, k), cr);
                cg = __builtin_fmaf(aw, dpp_bcast<G>(sc.y, k), cg);
                cb = __builtin_fmaf(aw, dpp_bcast<G>(sc.z, k), cb);
                ca = __builtin_fmaf(a, wk, ca);
              }
            } else {
#pragma unroll
              for (int k = 0; k < G; k++) {
                const float wk = dpp_bcast<G>(w, k);
                const f3 sk = mk3(dpp_bcast<G>(sc.x, k), dpp_bcast<G>(sc.y, k), dpp_bcast<G>(sc.z, k));
                if (k <= j && wk != 0.f) composite(cr, cg, cb, ca, sk, wk);
              }
            }
          } else {
            const float f = some ? 1.0f - ((tThis - tp) * P.istep) * w : 1.0f;
#pragma unroll
            for (int k = 0; k < G; k++) {
              const float fk0 = dpp_bcast<G>(f, k);
              const float fk = k <= j ? fk0 : 1.f;
              cr *= fk; cg *= fk; cb *= fk; ca *= fk;
            }
          }
          const unsigned long long om =
              __builtin_amdgcn_ballot_w64(step_ok && opaque_of(cr, cg, cb, ca, P.opaque_alpha));
          if (om) {
            const unsigned b = group_bits<G>(om);
            end = b ? min(hI, (int)__builtin_ctz(b)) : hI;
          }
        }
      }
      nsamp += (step_ok && j <= end) ? 1u : 0u;
      // on, unless an event ended the march or the position after this round's
      // last (lane 0's next) no longer advances
      iter += G;
      const float tl = dpp_bcast<G>(t, G - 1);
      go = end == G && __builtin_fminf(tl + step, lim) > tl && iter < GXY_MAX_MARCH;
      t = tn;
      tp = tpn;
    } while (go);
    if (end < G) {
      // lane `end` ended the march: by an isovalue when it is hI
      owner = j == end;
      hit_iso = end == hI;
      tTermination = tThis;
      nsamp += owner && hit_iso ? 1u : 0u;
    }
  }
  asm volatile("" ::: "memory");   // the fields are read again, not kept
  f3 nrm = mk3(0.f, 0.f, 0.f), col = nrm;
  bool surface_opaque = slice >= 0;
  if (slice >= 0) {
    const f3 org = ray_org(R, first, i), dir = ray_dir(R, first, i);
    const f3 pn = mk3(VV.slices[4 * slice], VV.slices[4 * slice + 1], VV.slices[4 * slice + 2]);
    nrm = dot3(dir, pn) > 0 ? neg3(pn) : pn;
    if (shade && !hit_iso) col = tf_color(s_col, T, vol_sample_t<SM>(V, add3(org, scl3(ray_t, dir))));
  }
  if (shade && hit_iso) {
    // LookForIsoHit shading (TraceRays.ispc:284-307): the four samples of the
    // forward-difference gradient side by side in the group's lanes
    surface_opaque = true;
    const f3 org = ray_org(R, first, i), dir = ray_dir(R, first, i);
    const unsigned ob = group_bits<G>(__builtin_amdgcn_ballot_w64(owner));
    const float ht = __shfl(tTermination, ((threadIdx.x & 63) & ~(G - 1)) + __builtin_ctz(ob), 64);
    const f3 p = add3(org, scl3(ht, dir));
    float g[4];
#pragma unroll
    for (int q = 0; q < 4; q += G) {
      const int a = q + j;
      const float v = vol_sample_t<SM>(
          V, add3(p, mk3(a == 1 ? V.sp[0] : 0.f, a == 2 ? V.sp[1] : 0.f, a == 3 ? V.sp[2] : 0.f)));
#pragma unroll
      for (int k = 0; k < G && q + k < 4; k++) g[q + k] = dpp_bcast<G>(v, k);
    }
    nrm = safe_normalize3(mk3((g[1] - g[0]) / V.sp[0], (g[2] - g[0]) / V.sp[1], (g[3] - g[0]) / V.sp[2]));
    if (dot3(dir, nrm) > 0) nrm = neg3(nrm);
    col = tf_color(s_col, T, hit_sample);
  }
  if (!owner) return nsamp;
  gptr(R.r + first)[i] = cr; gptr(R.g + first)[i] = cg; gptr(R.b + first)[i] = cb; gptr(R.o + first)[i] = ca;
  int term = opaque_of(cr, cg, cb, ca, P.opaque_alpha) ? RAY_OPAQUE : 0;
  if (slice >= 0 || hit_iso) {
    term |= RAY_SURFACE;
    if (surface_opaque) term |= RAY_OPAQUE;
    gptr(R.sr + first)[i] = col.x; gptr(R.sg + first)[i] = col.y; gptr(R.sb + first)[i] = col.z;
    gptr(R.so + first)[i] = 1.0f;
    gptr(R.nx + first)[i] = nrm.x; gptr(R.ny + first)[i] = nrm.y; gptr(R.nz + first)[i] = nrm.z;
  } else if (tTermination == tExitVolume) {
    term |= RAY_BOUNDARY;
  } else if (tTermination == gptr(R.tMax + first)[i]) {
    term |= RAY_TIMEOUT;
  }
  gptr(R.t + first)[i] = tTermination;
  gptr(R.term + first)[i] = term;
  return nsamp;
}

}  // namespace gxy
