// The carry of the one-launch forward kernels: a workgroup of kOnePassW waves
// holds the maps of one segment (kOnePassW consecutive chunks of a head group),
// publishes their composition, and folds the state entering the segment from
// the maps of the earlier ones (the look-back of the one-pass forward, described
// with fused_fwd_onepass_kernel).
#pragma once

#include "common.hpp"

namespace cdssm {

// Look-back flag bits of the one-pass forward (below the epoch, flag = epoch << 3 | bits).
constexpr unsigned long long kFlagMap = 1ull;    // segment map published
constexpr unsigned long long kFlagLeave = 2ull;  // state leaving the segment published (anchor ends)
constexpr unsigned long long kFlagGroup = 4ull;  // group map published (group ends)

// Wave-wide wait: lane i watches the flag of segment js (>= 0; -1: nothing)
// of the head group's flags f0 (stride H per segment) until it carries this
// call's epoch and the bits `need`.  True once every lane's flag does; false
// when the wait bound passes first.  Wave-uniform.
__device__ __forceinline__ bool watch_flags(const unsigned long long* f0, int H, unsigned long long epoch, int js,
                                            unsigned long long need) {
  const uint64_t t_start = __builtin_amdgcn_s_memrealtime();
  for (;;) {
    bool ready = true;
    if (js >= 0) {
      const unsigned long long fv = __hip_atomic_load(const_cast<unsigned long long*>(f0 + int64_t(js) * H),
                                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      ready = (fv >> 3) == epoch && (fv & need) == need;
    }
    if (__builtin_amdgcn_ballot_w64(!ready) == 0ull) return true;
    if (__builtin_amdgcn_s_memrealtime() - t_start > kSpinTicks) return false;
    __builtin_amdgcn_s_sleep(2);
  }
}

// G s + F, the state s after the map (G, F).  Its roundings are spelled out: where the compiler forms the
// multiply-adds, which of two products keeps its own rounding changes with the code around them, and with it
// the bits of every later output (24 bf16 layers make 1e-2 of one such change).  IM_RE: the imaginary part's
// fma takes the state's real part, else its imaginary part.
template <bool IM_RE>
__device__ __forceinline__ float2 map_apply(float2 G, float2 s, float2 F) {
#pragma clang fp contract(off)
  const float re = fmaf(G.x, s.x, -(G.y * s.y));
  const float im = IM_RE ? fmaf(G.y, s.x, G.x * s.y) : fmaf(G.x, s.y, G.y * s.x);
  return make_float2(re + F.x, im + F.y);
}

// Phase stamps of cdssm_fused_scan_fwd_stamped: segment entry, staging done,
// local pass done, segment map published, look-back wait done, carry folded,
// correction pass done, segment end.
constexpr int kStampPoints = 8;

// In: the chunk maps of the segment's n_live chunks in LDS, Fx (per chunk the
// HPW heads' states at its end from zero) and GF (per chunk and head the
// rotation product in x, y).  Out: Sx, the state entering the segment.
// `calls` and `status` are the calling unit's epoch counter and sticky status
// word, `tag` its epoch tag; `arrive`: this is the workgroup's first segment.
// stamp(i) records phase i.  Ends with a workgroup barrier; wv is this wave's
// index (wave-uniform), ctrl one int of LDS.
template <int D, int HPW, typename Stamp>
__device__ __forceinline__ void segment_carry(const OnePassBufs& ob, const float* __restrict__ h0,
                                              float* __restrict__ h_final, int H, int NSEG, int bi, int seg, int hbase,
                                              int n_live, int wv, const float2* Fx, const float4* GF, float2* Sx,
                                              int* ctrl, unsigned long long epoch, bool arrive,
                                              unsigned long long* calls, unsigned* status, unsigned tag,
                                              Stamp&& stamp) {
  constexpr int SEGN = HPW * D;                  // complex elements of a head group's state
  constexpr int EPT = SEGN / (kWave * kOnePassW);  // of which each thread composes EPT
  static_assert(EPT >= 1 && EPT * kWave * kOnePassW == SEGN, "segment state tiles the workgroup");
  constexpr bool RE = EPT > 1;                   // map_apply's order in the folds across segments
  const int lane = int(threadIdx.x) % kWave;
  // 2. segment map over the live chunks; thread x composes elements
  // e = x * EPT + i of the head group's state (head e / D, element e % D)
  const int e0 = int(threadIdx.x) * EPT;
  const int ej = e0 / D;
  const int ed = e0 % D;
  const int eh = hbase + ej;
  const bool ehok = eh < H;
  float2 segF[EPT];
  float2 segG = make_float2(1.0f, 0.0f);
#pragma unroll
  for (int i = 0; i < EPT; ++i) segF[i] = make_float2(0.0f, 0.0f);
  for (int u = 0; u < n_live; ++u) {
    const float4 g = GF[u * HPW + ej];
    const float2 gu = make_float2(g.x, g.y);
#pragma unroll
    for (int i = 0; i < EPT; ++i) segF[i] = map_apply<false>(gu, segF[i], Fx[u * SEGN + e0 + i]);
    segG = rotate(gu, segG);
  }
  const int64_t sb0 = (int64_t(bi) * NSEG + seg) * H;  // (b, seg, head 0)
  unsigned long long* flag = ob.flag + sb0 + hbase;

  // publish the segment map (every segment: later ones fold it in).  Flag
  // words are epoch << 3 | bits: kFlagMap the segment map, kFlagLeave the
  // state leaving the segment (anchor ends), kFlagGroup its group's map
  // (group ends); thread 0 stores the word with every bit published so far.
  // A group end whose group map some later segment reads flags its own map
  // together with the group map (one store acknowledgement, one flag): it
  // waits only on lower segments' maps, which never wait on it.
  if (ehok) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) st_agent(ob.seg_f + (sb0 + eh) * D + ed + i, segF[i]);
    if (ed == 0) st_agent(ob.seg_g + sb0 + eh, segG);
  }
  const bool gend = seg % kFwdGroup == kFwdGroup - 1 && fwd_group_read(seg / kFwdGroup, NSEG);
  unsigned long long bits = kFlagMap;
  if (!gend) {
    wait_stores_acked();
    __syncthreads();
    if (threadIdx.x == 0) {
      __hip_atomic_store(flag, (epoch << 3) | bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (arrive) leave_next_epoch(ob, calls, tag);
    }
  }

  stamp(3);
  const unsigned long long* f0 = ob.flag + (int64_t(bi) * NSEG) * H + hbase;  // (b, segment 0, head group)
  const int64_t lb = int64_t(bi) * NSEG * H + eh;                            // (b, segment 0, head eh)
  const int ngrp_all = fwd_groups(NSEG);
  // a group end (the last segment of a group some later segment folds)
  // composes its group's map, oldest first: the maps its group's other
  // segments published, then its own
  if (gend) {
    const int s0 = seg - (kFwdGroup - 1);
    if (wv == 0) {
      const bool got = watch_flags(f0, H, epoch, lane < kFwdGroup - 1 ? s0 + lane : -1, kFlagMap);
      if (lane == 0) {
        ctrl[0] = got;
        if (!got) __hip_atomic_fetch_or(status, kTimeoutFwd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
    const int okg = ctrl[0];
    if (ehok) {
      float2 G[kFwdGroup - 1], F[kFwdGroup - 1][EPT];
#pragma unroll
      for (int u = 0; u < kFwdGroup - 1; ++u) {
        G[u] = ld_agent(ob.seg_g + lb + int64_t(s0 + u) * H);
#pragma unroll
        for (int i = 0; i < EPT; ++i) F[u][i] = ld_agent(ob.seg_f + (lb + int64_t(s0 + u) * H) * D + ed + i);
      }
      float2 Gg = make_float2(1.0f, 0.0f), Fg[EPT];
#pragma unroll
      for (int i = 0; i < EPT; ++i) Fg[i] = make_float2(0.0f, 0.0f);
#pragma unroll
      for (int u = 0; u < kFwdGroup; ++u) {
        const float2 gu = u < kFwdGroup - 1 ? G[u] : segG;
#pragma unroll
        for (int i = 0; i < EPT; ++i) Fg[i] = map_apply<RE>(gu, Fg[i], u < kFwdGroup - 1 ? F[u][i] : segF[i]);
        Gg = rotate(gu, Gg);
      }
      if (!okg) {
#pragma unroll
        for (int i = 0; i < EPT; ++i) Fg[i] = make_float2(__builtin_nanf(""), __builtin_nanf(""));
      }
      const int64_t gb = (int64_t(bi) * ngrp_all + seg / kFwdGroup) * H + eh;
#pragma unroll
      for (int i = 0; i < EPT; ++i) st_agent(ob.grp_f + gb * D + ed + i, Fg[i]);
      if (ed == 0) st_agent(ob.grp_g + gb, Gg);
    }
    wait_stores_acked();  // the segment map and the group map
    __syncthreads();
    bits |= kFlagGroup;
    if (threadIdx.x == 0) {
      __hip_atomic_store(flag, (epoch << 3) | bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (arrive) leave_next_epoch(ob, calls, tag);
    }
  }

  // state entering the segment, in a fixed order (so results do not depend on
  // timing): from the anchor a = kFwdAnchor * floor((seg - 1) / kFwdAnchor)
  // -- h0 for a = 0, else the published state leaving segment a - 1 -- fold
  // the maps of the segments a .. seg - 1 where there are at most kFwdDirect
  // of them, else the maps of the whole groups in [a, seg) and then those of
  // the segments of seg's own group before it; oldest first.  Wave 0 waits
  // until they are published (lanes 0 .. ngrp-1: group maps; then the segment
  // maps; lane 63: the anchor state).
  const int anc = seg == 0 ? 0 : kFwdAnchor * ((seg - 1) / kFwdAnchor);
  const bool direct = seg - anc <= kFwdDirect;
  const int g0 = anc / kFwdGroup, g1 = direct ? g0 : seg / kFwdGroup;
  const int ngrp = g1 - g0;                  // <= kFwdAnchor / kFwdGroup
  const int sg0 = g1 * kFwdGroup;            // first segment folded one by one
  const int nmap = seg - sg0;                // <= kFwdDirect
  int ok = 1;
  if (seg > 0) {
    if (wv == 0) {
      int js = -1;
      unsigned long long need = 0ull;
      if (lane < ngrp) {
        js = (g0 + lane) * kFwdGroup + kFwdGroup - 1;
        need = kFlagGroup;
      } else if (lane < ngrp + nmap) {
        js = sg0 + lane - ngrp;
        need = kFlagMap;
      } else if (lane == kWave - 1 && anc > 0) {
        js = anc - 1;
        need = kFlagLeave;
      }
      const bool got = watch_flags(f0, H, epoch, js, need);
      if (lane == 0) {
        ctrl[0] = got;
        if (!got) __hip_atomic_fetch_or(status, kTimeoutFwd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
    ok = ctrl[0];
  }
  stamp(4);
  float2 Sin[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) Sin[i] = make_float2(0.0f, 0.0f);
  if (ehok) {
    if (anc == 0) {
      if (h0) {
        const int64_t hb = (int64_t(bi) * H + eh) * 2 * D;
#pragma unroll
        for (int i = 0; i < EPT; ++i) Sin[i] = make_float2(h0[hb + ed + i], h0[hb + D + ed + i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < EPT; ++i) Sin[i] = ld_agent(ob.seg_s + (lb + int64_t(anc - 1) * H) * D + ed + i);
    }
    // at most max(kFwdDirect, kFwdAnchor / kFwdGroup + kFwdGroup - 1) maps, all requested at once
    constexpr int kMaps = kFwdDirect > kFwdAnchor / kFwdGroup + kFwdGroup - 1 ? kFwdDirect
                                                                            : kFwdAnchor / kFwdGroup + kFwdGroup - 1;
    float2 G[kMaps], F[kMaps][EPT];
#pragma unroll
    for (int u = 0; u < kMaps; ++u) {
      if (u < ngrp) {
        const int64_t gb = (int64_t(bi) * ngrp_all + g0 + u) * H + eh;
        G[u] = ld_agent(ob.grp_g + gb);
#pragma unroll
        for (int i = 0; i < EPT; ++i) F[u][i] = ld_agent(ob.grp_f + gb * D + ed + i);
      } else if (u < ngrp + nmap) {
        const int64_t sb = lb + int64_t(sg0 + u - ngrp) * H;
        G[u] = ld_agent(ob.seg_g + sb);
#pragma unroll
        for (int i = 0; i < EPT; ++i) F[u][i] = ld_agent(ob.seg_f + sb * D + ed + i);
      }
    }
#pragma unroll
    for (int u = 0; u < kMaps; ++u) {
      if (u < ngrp + nmap) {
#pragma unroll
        for (int i = 0; i < EPT; ++i)
          Sin[i] = u == 0 ? map_apply<false>(G[u], Sin[i], F[u][i]) : map_apply<RE>(G[u], Sin[i], F[u][i]);
      }
    }
    if (!ok) {
#pragma unroll
      for (int i = 0; i < EPT; ++i) Sin[i] = make_float2(__builtin_nanf(""), __builtin_nanf(""));
    }
  }
  // the state leaving the segment: h_final for the last segment; published
  // for the segments that start from it (anchor ends, (seg + 1) % kFwdAnchor == 0)
  const bool anchor_end = seg + 1 < NSEG && (seg + 1) % kFwdAnchor == 0;
#pragma unroll
  for (int i = 0; i < EPT; ++i) Sx[e0 + i] = Sin[i];
  if (ehok && (anchor_end || seg + 1 == NSEG)) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const float2 so = map_apply<RE>(segG, Sin[i], segF[i]);
      if (anchor_end) {
        st_agent(ob.seg_s + (sb0 + eh) * D + ed + i, so);
      } else {
        const int64_t hb = (int64_t(bi) * H + eh) * 2 * D;
        h_final[hb + ed + i] = so.x;
        h_final[hb + D + ed + i] = so.y;
      }
    }
  }
  if (anchor_end) wait_stores_acked();
  __syncthreads();
  if (anchor_end && threadIdx.x == 0)
    __hip_atomic_store(flag, (epoch << 3) | bits | kFlagLeave, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

}

}  // namespace cdssm
