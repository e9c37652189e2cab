// Device helpers shared by the block's fused elementwise kernels (lm_fused.hip)
// and the decode step's fused tail (decode.hip).
#pragma once

#include "common.hpp"

namespace cdssm {
namespace lm {

// Round to the element type (identity for fp32).
template <typename T>
__device__ __forceinline__ float rnd(float x) {
  if constexpr (T::bytes == 2)
    return bf16_to_f32(f32_to_bf16(x));
  else
    return x;
}

// Round a pair to the element type with one packed conversion (identity for fp32).
template <typename T>
__device__ __forceinline__ void rnd2(float& a, float& b) {
  if constexpr (T::bytes == 2) {
    const uint32_t p = pack_bf16x2(a, b);
    a = bf16_lo(p);
    b = bf16_hi(p);
  }
}

// silu(u) = u sigmoid(u) with the hardware reciprocal (about 1 ulp)
__device__ __forceinline__ float silu_fast(float u) { return u * __builtin_amdgcn_rcpf(1.0f + __expf(-u)); }

// ---------------------------------------------------------------------------
// GroupNorm + gate for one decode token of batch row b, with running
// statistics: gsum (B, G, 4) fp32 = (shift K, sum (x - K), sum (x - K)^2,
// count) over every position so far (block.py:215-225).  The row's y is read
// from `y`, or, with `rs` (the row's kr retrieved values in LDS, rounded to the
// element type), formed by the readout projection y_c = rnd(sum_j rs_j W[c][j])
// (block.py:213).  The new token's group sums are added in a fixed order (one
// thread per group), the statistics formed from the totals, and the token
// normalised, gated and skipped as gn_gate_kernel does: with the prefix's sums
// this equals the GroupNorm of a forward over the prefix plus the token, for
// that token.  Threads of the workgroup that take no part pass as many barriers
// (one, with rs two).  gst (G float2) and ys (ys_at(C, ys_shift(C, G)) floats) are the caller's LDS.
// ---------------------------------------------------------------------------
// What the step reads and writes, beside its row of y: with wr, the readout weight (C, kr).
template <typename T, typename P>
struct RowArgs {
  const typename T::raw* wr;
  int kr;
  float4* gsum;  // (B, G) shifted running sums
  const typename P::raw *gamma, *beta;
  const typename T::raw* z;
  int64_t z_bs;
  const typename T::raw *xc, *Dp;
  typename T::raw* out;
  int C, G;
  float eps;
  // two channels per thread with 4-byte accesses where the bf16 rows allow
  __device__ __forceinline__ bool pairs(int b) const {
    const auto a4 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0; };
    return T::bytes == 2 && P::bytes == 2 && C / G % 2 == 0 && a4(z + int64_t(b) * z_bs) &&
           a4(xc + int64_t(b) * C) && a4(out + int64_t(b) * C) && a4(Dp) && a4(gamma) && a4(beta);
  }
};

// Two channels of z, xc, D, gamma and beta as they lie in memory.
template <typename T, typename P>
struct RowPair {
  uint32_t z, x, d, g, b;
  __device__ __forceinline__ void load(int bi, const RowArgs<T, P>& a, int c) {
    z = *reinterpret_cast<const uint32_t*>(a.z + int64_t(bi) * a.z_bs + c);
    x = *reinterpret_cast<const uint32_t*>(a.xc + int64_t(bi) * a.C + c);
    d = *reinterpret_cast<const uint32_t*>(a.Dp + c);
    g = *reinterpret_cast<const uint32_t*>(a.gamma + c);
    b = *reinterpret_cast<const uint32_t*>(a.beta + c);
  }
};

// The first of everything a thread (tid of nthr) reads in the step, requested before y or the retrieved
// values are there: up to kVecs 16-byte vectors of readout weight (all of its channels or, with n = 0, none),
// its first group's sums, its first two channels' rows.  Read one after the other behind the token step, these
// were 6.9 of the decode tail's 12 us (B 64, C 1024, kr 32).  Held in registers: 3.1.
template <typename T, typename P>
struct RowPrefetch {
  static constexpr int kVecs = 8, E = 16 / T::bytes;
  uint4 w[kVecs];
  float4 gs;
  RowPair<T, P> rows;
  int n = 0;            // vectors per channel, 0: the weights are not held
  __device__ __forceinline__ void load(int bi, const RowArgs<T, P>& a, int tid, int nthr) {
    if (tid < a.G) gs = a.gsum[int64_t(bi) * a.G + tid];
    if constexpr (T::bytes == 2 && P::bytes == 2)
      if (2 * tid < a.C && a.pairs(bi)) rows.load(bi, a, 2 * tid);
    const int nv = a.kr / E, slots = (a.C + nthr - 1) / nthr;
    if (a.wr && a.kr % E == 0 && nv * slots <= kVecs && (reinterpret_cast<uintptr_t>(a.wr) & 15u) == 0) {
      n = nv;
      int c = tid, j = 0;
#pragma unroll
      for (int i = 0; i < kVecs; ++i) {
        w[i] = *reinterpret_cast<const uint4*>(a.wr + int64_t(min(c, a.C - 1)) * a.kr + j * E);
        if (++j == nv) j = 0, c += nthr;
      }
    }
  }
};

// Channel c of y lies at ys_at(c, ys_shift(C, G)) in LDS, and y takes ys_at(C, ...) floats: a word of padding
// per 32 where the groups' first channels would all fall on one bank, within the 64 KB that a launch may ask
// for (C <= 8192: 33 KB, the groups' statistics 2 KB, the retrieved values 16 KB at the most).
__host__ __device__ __forceinline__ int ys_shift(int C, int G) { return C <= 8192 && C / G % 32 == 0 ? 5 : 31; }
__host__ __device__ __forceinline__ int ys_at(int c, int shift) { return c + (c >> shift); }

// Threads tid = 0 .. nthr - 1; PF: they have loaded pf.
template <typename T, typename P, bool PF>
__device__ __forceinline__ void gn_row_step(int b, const typename T::raw* __restrict__ y, const float* rs,
                                            const RowArgs<T, P>& a, float2* gst, float* ys, int tid, int nthr,
                                            const RowPrefetch<T, P>& pf) {
  using raw = typename T::raw;
  const int C = a.C, G = a.G, kr = a.kr, Cg = C / G, sh = ys_shift(C, G);
  const raw* yr = y ? y + int64_t(b) * C : nullptr;
  if (rs) {
    constexpr int E = RowPrefetch<T, P>::E;  // elements per 16-byte load
    // W rows as 16-byte loads when every row starts on a 16-byte boundary
    const bool vec = kr % E == 0 && (reinterpret_cast<uintptr_t>(a.wr) & 15u) == 0;
    if (PF && pf.n > 0) {
      float s = 0.0f;
      int c = tid, j = 0;
#pragma unroll
      for (int i = 0; i < RowPrefetch<T, P>::kVecs; ++i) {
        if (c < C) {
          const uint32_t wd[4] = {pf.w[i].x, pf.w[i].y, pf.w[i].z, pf.w[i].w};
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if constexpr (T::bytes == 2) {
              s = fmaf(rs[j * E + 2 * u], bf16_lo(wd[u]), s);
              s = fmaf(rs[j * E + 2 * u + 1], bf16_hi(wd[u]), s);
            } else {
              s = fmaf(rs[j * E + u], __uint_as_float(wd[u]), s);
            }
          }
          if (j == pf.n - 1) ys[ys_at(c, sh)] = rnd<T>(s);
        }
        if (++j == pf.n) j = 0, c += nthr, s = 0.0f;
      }
    } else {
      for (int c = tid; c < C; c += nthr) {
        const raw* wc = a.wr + int64_t(c) * kr;
        float s = 0.0f;
        if (vec) {
          for (int j = 0; j < kr; j += E) {
            const uint4 v = *reinterpret_cast<const uint4*>(wc + j);
            const raw* e = reinterpret_cast<const raw*>(&v);
#pragma unroll
            for (int u = 0; u < E; ++u) s = fmaf(rs[j + u], T::load(e + u), s);
          }
        } else {
          for (int j = 0; j < kr; ++j) s = fmaf(rs[j], T::load(wc + j), s);
        }
        ys[ys_at(c, sh)] = rnd<T>(s);
      }
    }
    __syncthreads();
  }
  auto yv = [&](int c) -> float { return rs ? ys[ys_at(c, sh)] : T::load(yr + c); };
  for (int g = tid; g < G; g += nthr) {
    float4 s;
    if (PF && g == tid)
      s = pf.gs;
    else
      s = a.gsum[int64_t(b) * G + g];
    float s1 = 0.0f, s2 = 0.0f;
    int c = 0;
    for (; c + 8 <= Cg; c += 8) {  // eight values in flight, added in order
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = yv(g * Cg + c + u);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float d = v[u] - s.x;
        s1 += d;
        s2 = fmaf(d, d, s2);
      }
    }
    for (; c < Cg; ++c) {
      const float d = yv(g * Cg + c) - s.x;
      s1 += d;
      s2 = fmaf(d, d, s2);
    }
    s.y += s1;
    s.z += s2;
    s.w += float(Cg);
    a.gsum[int64_t(b) * G + g] = s;
    const float m = s.y / s.w;
    gst[g] = make_float2(s.x + m, rsqrtf(fmaxf(s.z / s.w - m * m, 0.0f) + a.eps));
  }
  __syncthreads();
  // the token normalised, gated and skipped: two channels per thread (8 took 1.9 us of a row's chain, on a quarter of the
  // threads), else one
  const raw* zr = a.z + int64_t(b) * a.z_bs;
  const raw* xr = a.xc + int64_t(b) * C;
  raw* orow = a.out + int64_t(b) * C;
  if constexpr (T::bytes == 2 && P::bytes == 2) {
    if (a.pairs(b)) {
      for (int c0 = 2 * tid; c0 < C; c0 += 2 * nthr) {
        RowPair<T, P> r;
        if (PF && c0 == 2 * tid)
          r = pf.rows;
        else
          r.load(b, a, c0);
        const float2 st = gst[c0 / Cg];
        float r2[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float zz = h ? bf16_hi(r.z) : bf16_lo(r.z), xx = h ? bf16_hi(r.x) : bf16_lo(r.x);
          const float dd = h ? bf16_hi(r.d) : bf16_lo(r.d), ga = h ? bf16_hi(r.g) : bf16_lo(r.g);
          const float be = h ? bf16_hi(r.b) : bf16_lo(r.b);
          const float gn = rnd<T>(fmaf((yv(c0 + h) - st.x) * st.y, ga, be));
          const float sv = rnd<T>(silu_fast(zz));
          r2[h] = rnd<T>(gn * sv) + rnd<T>(dd * xx);
        }
        *reinterpret_cast<uint32_t*>(orow + c0) = pack_bf16x2(r2[0], r2[1]);
      }
      return;
    }
  }
  for (int c = tid; c < C; c += nthr) {
    const float2 st = gst[c / Cg];
    const float gn = rnd<T>(fmaf((yv(c) - st.x) * st.y, P::load(a.gamma + c), P::load(a.beta + c)));
    const float s = rnd<T>(silu_fast(T::load(zr + c)));
    const float p = rnd<T>(gn * s);
    const float d = rnd<T>(T::load(a.Dp + c) * T::load(xr + c));
    T::store(orow + c, p + d);
  }
}

}  // namespace lm
}  // namespace cdssm
