// The one-launch inference forward on the matrix cores: scan-level bf16
// inputs, state_dim 2 (one complex value per head), fp32 states, R-mode
// semantics and look-back carry of fused_fwd_onepass_kernel.
//
// The sequential form runs every token's dot products and updates over D on
// the VALU, one dependent step per token.  Here a chunk goes in blocks of 16
// tokens, and everything that is a contraction over D or over the block's
// tokens runs on MFMA; what is left is a 16-step triangular solve on scalars,
// 4 heads at once.  For one head, with H the local state (true units) and c
// the decay-free correction state entering the block (complex D-vectors),
// f_t = prod_{u<=t} a_u within the block and g_{t-1} the chunk's product before t:
//   x^_t = w_t / f_t - beta_t (k_t.H) - beta_t sum_{s<t} (k_t.k_s) x^_s    (update coefficients, z_t = f_t (H + sum_{s<=t} x^_s k_s))
//   x_t  =             beta_t (k_t.c) - beta_t sum_{s<t} (k_t.k_s) x_s     (c_{t+1} = c - sum_{s<=t} x_s k_s)
//   y_t  = sel_t (f_t (q_t.H + sum_{s<=t} (q_t.k_s) x^_s) + g_{t-1} (q_t.c - sum_{s<t} (q_t.k_s) x_s))
//   H'   = f_15 H + sum_s (f_15 x^_s) k_s,   c' = c - sum_s x_s k_s
// A head whose quotients w_t / f_t would leave fp32's range (f_t near its limits,
// or a large w_t) runs its block in true units: the same solve with the products
// of a carried forward one step at a time, which never divides.  That is decided
// per head, and nothing else crosses heads, so a head's bits do not depend on the
// others of its wave.  With |f| down to 2^-112 in the quotients one block in 20 of
// a drawn call at B 8, H 16, L 4096 is such a one for some head of its wave (one
// in 5 at 2^-76); if all are, the call takes 48.7 in place of 42.2 us.
//
// A wave holds 4 heads of one chunk; a workgroup the 4 chunks of a segment.
// Lane (g, i) = (lane / 16, lane % 16) owns token i of head g in the solve.
// MFMA operands (16x16x32: A row / B column lane % 16, k = 8 (lane / 16) ..+8;
// 16x16x16: k = 4 (lane / 16) ..+4; result column lane % 16, rows 4 (lane / 16) ..+4):
//  * K and Q fragments are loaded straight from HBM in operand layout (one
//    16-byte load per lane, 32 dims of 16 tokens).
//  * Gram tiles K K^T, K Q^T per head; the 4 heads' tiles are transposed
//    against the 4 lane groups with permlane swaps (4 for 4 registers), which
//    leaves lane (g, i) with row i of its own head: no LDS round trip.
//  * k.H, k.c, q.H, q.c: the state as the A operand, rows 4 h + part of head
//    h only (lanes of the other heads read zeros), so the 4 heads accumulate
//    into one tile whose rows land in the head's own lane group.
//  * sum_s x_s k_s: A = the coefficients (rows 4 h + part), B = K^T, which an
//    MFMA against a selection matrix produces from the K fragments: its result
//    layout, rounded back to bf16 (exact), is the B layout of 16x16x16.
//  * sum_s (q_t.k_s) x_s, both fp32: 4 x 1 by 1 x 4 fp32 products (4x4x1, 16 blocks), block = (head, 4
//    tokens), whose results are the 4 sums of the lane's own token and head.
// fp32 operands against K and Q (states, coefficients) enter as three bf16 terms,
// hi + mid + lo = x to 2^-24 relative, so every sum keeps fp32 accuracy, the
// readouts' too: y is the difference of a state's part and the part that erased
// it, and where the two nearly cancel, operands of two terms (2^-16) leave
// errors in its bf16 digits (D 64, a state 100 times the values written over it:
// above 1e-3 of y's rounding in a quarter of the outputs, now in 1 in 300).
// us per call with two terms / now: B 8, H 16, L 4096, D 64 45.2 / 44.9, L 2048
// 29.9 / 29.4, B 1, H 4, L 512 22.8 / 23.4; D 128, B 4, H 16, L 2048 71.3 / 69.6.
// The third term cost 0.4 to 3 us of it; scaling the state and the coefficients
// ahead of the update, not the sum after it, gave that back.
// Zeros times a non-finite value are not zero, so non-finite inputs are kept to their head and to the
// tokens from theirs on: a block whose Gram sums are not finite zeroes the affected k slices, the tokens
// with a non-finite k, write or beta enter the block with zero coefficients, and the head's state after the
// block and its outputs from the token on are made NaN, as the recurrence would leave them.
#include "onepass_mfma.hpp"

#include "chunk_sweep.hpp"
#include "fwd_lookback.hpp"

namespace cdssm {

namespace {

__device__ unsigned long long g_mf_calls;   // one-launch calls of this unit (source of the look-back epochs)
__device__ unsigned int g_mf_status;        // kTimeoutFwd once a look-back wait gave up
constexpr unsigned kMfTag = 3u;             // epoch tag (the other one-launch passes use 1 and 2)

__global__ __launch_bounds__(64) void mf_epoch_kernel(unsigned long long* ctl) {
  if (threadIdx.x == 0) {
    const unsigned long long n =
        __hip_atomic_fetch_add(&g_mf_calls, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1ull;
    __hip_atomic_store(ctl + 1, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(ctl, epoch_word(kMfTag, n), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

constexpr int kMfHeads = 4;            // heads per wave
// A head's block runs in true units where some |2^60 f|^2 is below kMfTiny (|f| < 2^-112) or infinite, or some
// quotient w / f not below kMfLarge (2^12 are left for the block's sums).
constexpr float kMfTiny = 0x1p-104f;
constexpr float kMfScale = 0x1p60f;
constexpr float kMfLarge = 0x1p115f;

typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

template <int D>
struct MfCfg {
  static constexpr int KS = D / 32;              // 32-dim steps of the contractions over D
  static constexpr int SROW = 3 * D / 2 + 16;    // operand row, dwords: H | c | lo parts of D/2 each, and a pad
  static constexpr int OP = 16 * SROW + 64;      // 16 rows, 16 dwords apart per head (conflict-free writes)
  static constexpr int EB = 16 * 24;             // coefficient rows: 3 terms x 16 tokens bf16
  static constexpr int ZERO = 16 * (KS - 1) + 20;  // zeros, read in place of rows that do not take part
  static constexpr int NB(int Q) { return (Q + 15) / 16; }
  static constexpr int wave_dwords(int Q) { return NB(Q) * 64 * 8 + OP + EB; }
  static size_t lds_bytes(int Q) {
    return size_t(kOnePassW) * wave_dwords(Q) * 4 + ZERO * 4 + size_t(kOnePassW) * kMfHeads * D * 8 +
           size_t(kOnePassW) * kMfHeads * 16 + size_t(kMfHeads) * D * 8 + 16;
  }
};

struct MfArgs {
  const uint16_t *q, *k, *v, *beta, *sel, *dt, *r;
  const float *alpha, *omega;
  float c;
  const float* h0;
  uint16_t* y;
  float* h_final;
  OnePassBufs ob;
  int L, H, Q, NC, NSEG, B, n_hg;
  bool wide;  // 8-byte loads of the per-token scalars
  unsigned long long* stamps;
  int stamp_heads;  // heads to a stamp record's item
};

// LDS handed between lanes of one wave: the wave's LDS accesses complete in
// order, so only the compiler has to keep them in order.
__device__ __forceinline__ void wave_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

// x through an opaque copy: comparisons with it are formed where they stand (rare branches) instead of
// being hoisted out of the block loops, where 16 lane masks would spill.
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// x0, x1 as three bf16 terms each, packed in pairs: hi and mid truncated, lo rounded; their sum is x to 2^-24.
__device__ __forceinline__ void split3(float x0, float x1, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  const uint32_t u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
  hi = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
  const float r0 = x0 - __uint_as_float(u0 & 0xffff0000u), r1 = x1 - __uint_as_float(u1 & 0xffff0000u);
  const uint32_t v0 = __float_as_uint(r0), v1 = __float_as_uint(r1);
  mid = __builtin_amdgcn_perm(v1, v0, 0x07060302u);
  lo = pack_bf16x2(r0 - __uint_as_float(v0 & 0xffff0000u), r1 - __uint_as_float(v1 & 0xffff0000u));
}

// The K or Q fragments of one block: head h, dims 32 ks + 8 (lane / 16) ..+8 of token lane % 16.
template <int KS>
struct MfFrags {
  bf16x8_t f[kMfHeads][KS];
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, int voff, const int (&hoff)[kMfHeads]) {
#pragma unroll
    for (int h = 0; h < kMfHeads; ++h)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        f[h][ks] = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, hoff[h] + 64 * ks, 0));
  }
};

// 16 x 16 tiles a_h b_h^T of the 4 heads: lane (g, i) gets a_{4g+r} . b_i in tile h, register r.
template <int KS>
__device__ __forceinline__ void mf_gram(const MfFrags<KS>& a, const MfFrags<KS>& b, f32x4_t (&t)[kMfHeads]) {
#pragma unroll
  for (int h = 0; h < kMfHeads; ++h) t[h] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int h = 0; h < kMfHeads; ++h) t[h] = mfma16(a.f[h][ks], b.f[h][ks], t[h]);
}

__device__ __forceinline__ bool mf_finite(const f32x4_t (&t)[kMfHeads]) {
  float s = 0.0f;
#pragma unroll
  for (int h = 0; h < kMfHeads; ++h) s += (t[h][0] + t[h][1]) + (t[h][2] + t[h][3]);
  return __builtin_amdgcn_ballot_w64(!(fabsf(s) < __builtin_inff())) == 0ull;
}

// Zero the slices of f that hold a non-finite element; whether this lane's own token (lane % 16 of head
// lane / 16) has one.
template <int KS>
__device__ __forceinline__ bool mf_sanitize(MfFrags<KS>& f, int g, int i) {
  bool own = false;
#pragma unroll
  for (int h = 0; h < kMfHeads; ++h) {
    u16x2_t top = {0, 0};  // the largest magnitude pattern of the slice, per half
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const uint4 u = __builtin_bit_cast(uint4, f.f[h][ks]);
      const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2_t, w[e] & 0x7fff7fffu));
    }
    const bool bad = max(uint32_t(top[0]), uint32_t(top[1])) >= 0x7f80u;
    const unsigned long long m = __builtin_amdgcn_ballot_w64(bad);
    const uint32_t tok = uint32_t(m | (m >> 16) | (m >> 32) | (m >> 48)) & 0xffffu;
    if (opaque(g) == h) own = (tok >> i) & 1u;
    const bf16x8_t zero8 = {};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) f.f[h][ks] = bad ? zero8 : f.f[h][ks];
  }
  return own;
}

__device__ __forceinline__ void swap32(float& a, float& b) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(s[0]);
  b = __uint_as_float(s[1]);
}
__device__ __forceinline__ void swap16(float& a, float& b) {
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(s[0]);
  b = __uint_as_float(s[1]);
}

// x[h] of lane group g' <-> x[g'] of lane group h
__device__ __forceinline__ void mf_exchange(float (&x)[kMfHeads]) {
  swap32(x[0], x[2]);
  swap32(x[1], x[3]);
  swap16(x[0], x[1]);
  swap16(x[2], x[3]);
}

// Tiles of 4 heads -> rows: lane (g, i) gets row[s] = tile_g[s][i] (s = 4 g' + r held by lane group g') for
// s < i, else zero.
__device__ __forceinline__ void mf_rows(const f32x4_t (&t)[kMfHeads], int g, int i, float (&row)[16]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float x[kMfHeads];
#pragma unroll
    for (int h = 0; h < kMfHeads; ++h) x[h] = 4 * g + r < i ? t[h][r] : 0.0f;
    mf_exchange(x);
#pragma unroll
    for (int gp = 0; gp < 4; ++gp) row[4 * gp + r] = x[gp];
  }
}

// tile_g[i][i] for lane (g, i)
__device__ __forceinline__ float mf_diag(const f32x4_t (&t)[kMfHeads], int g, int i) {
  float x[kMfHeads];
#pragma unroll
  for (int h = 0; h < kMfHeads; ++h) {
    x[h] = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[h] = 4 * g + r == i ? t[h][r] : x[h];
  }
  mf_exchange(x);
  return (x[0] + x[1]) + (x[2] + x[3]);  // three zeros
}

// (I - L) x = x in place over the lane's 16-lane row, L strictly lower (row of this lane's token).
__device__ __forceinline__ void mf_solve(const float (&L)[16], float& xr, float& xi) {
#pragma unroll
  for (int s = 0; s < 15; ++s) {
    const float br = row_bcast_dyn(xr, s), bi = row_bcast_dyn(xi, s);
    xr = fmaf(L[s], br, xr);
    xi = fmaf(L[s], bi, xi);
  }
}

// One segment of 4 chunks of a head group; idx enumerates (unit = segment of a batch row, head group) so
// that the head groups of a unit, which share the lines of the per-token scalars, lie 8 apart (one XCD
// under the round-robin placement of workgroups) and lower segments come first.
template <int D>
__device__ __forceinline__ void mf_segment(const MfArgs& a, int idx, unsigned long long epoch) {
  using Cfg = MfCfg<D>;
  constexpr int KS = Cfg::KS, SROW = Cfg::SROW, W = kOnePassW, SEGN = kMfHeads * D;
  extern __shared__ __align__(16) uint32_t mf_lds[];
  unsigned long long ts[kStampPoints] = {};
  const bool stamping = a.stamps != nullptr;
  auto clock = [&](int n) {
    if (stamping) ts[n] = __builtin_amdgcn_s_memrealtime();
  };
  clock(0);

  const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
  const int lane = int(threadIdx.x) % kWave, g = lane / 16, i = lane % 16;
  const int n_unit = a.NSEG * a.B, grp = idx / (8 * a.n_hg), loc = idx - grp * 8 * a.n_hg;
  const int width = min(8, n_unit - 8 * grp);
  const int hg = loc / width, unit = 8 * grp + (loc - hg * width);
  const int seg = unit / a.B, bi = unit - seg * a.B;
  const int hbase = hg * kMfHeads;
  const int H = a.H, L = a.L, Q = a.Q;
  const int n_live = min(W, a.NC - seg * W);
  const bool live = wv < n_live;
  const int chunk = min(seg * W + wv, a.NC - 1);
  const int t0 = chunk * Q, nt = min(Q, L - t0), nb = (nt + 15) / 16, tlast = nt - 1;
  const int64_t row0 = int64_t(bi) * L + t0;
  const int hv = hbase + g;
  const bool hok = hv < H;
  const int hl = hok ? hv : H - 1;

  // LDS: per wave the token slots (A: coefficient re, im, beta, sel, and in the correction pass a block's fp32
  // coefficient rows; B: f re, im, a re, im), the operand rows and the coefficient rows; then the zeros, the chunk maps and the carry's buffers
  uint32_t* wl = mf_lds + wv * Cfg::wave_dwords(Q);
  float4* tokA = reinterpret_cast<float4*>(wl);
  float4* tokB = tokA + Cfg::NB(Q) * 64;
  uint32_t* op = reinterpret_cast<uint32_t*>(tokB + Cfg::NB(Q) * 64);
  uint32_t* eb = op + Cfg::OP;
  uint32_t* zero = mf_lds + W * Cfg::wave_dwords(Q);
  float2* Fx = reinterpret_cast<float2*>(zero + Cfg::ZERO);
  float4* GF = reinterpret_cast<float4*>(Fx + W * SEGN);
  float2* Sx = reinterpret_cast<float2*>(GF + W * kMfHeads);
  int* ctrl = reinterpret_cast<int*>(Sx + SEGN);
  if (threadIdx.x < Cfg::ZERO) zero[threadIdx.x] = 0u;

  const int rowb = H * D * 2;  // bytes from token to token
  int hoff[kMfHeads];
#pragma unroll
  for (int h = 0; h < kMfHeads; ++h) hoff[h] = min(hbase + h, H - 1) * D * 2;
  const int64_t rest = int64_t(L - t0) * H * D * 2;
  const uint32_t nrec = uint32_t(rest > 0xffffffffll ? 0xffffffffll : rest);
  const auto krs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.k + row0 * H * D), short(0), int(nrec),
                                                     0x00020000);
  const auto qrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.q + row0 * H * D), short(0), int(nrec),
                                                     0x00020000);
  auto voff = [&](int b) { return min(16 * b + i, tlast) * rowb + 16 * g; };

  // operand row of this lane's state (head g) when writing, and per head h the address this lane reads as
  // row lane % 16 of head h's operand (the zeros where the row is another head's)
  uint32_t* opw = op + 4 * g * SROW + 16 * g + i;
  const uint32_t* opr = op + i * SROW + 16 * (i / 4) + 4 * g;
  const uint32_t* oprc = (i & 2) ? zero + 4 * g : opr + D;  // the lo part of c alone (rows 2, 3 hold H's there)
  const uint32_t* ebr = eb + i * 24 + 2 * g;
  uint16_t* ebw = reinterpret_cast<uint16_t*>(eb) + 4 * g * 48 + i;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) opw[2 * SROW + D + 16 * ks] = opw[3 * SROW + D + 16 * ks] = 0u;  // none in the local pass
  // selection operands: column n picks dim 2 n + u of a 32-dim step
  bf16x8_t sel2[2];
  {
    const int w = i - 4 * g;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint32_t one = u ? 0x3f800000u : 0x3f80u;
      sel2[u] = __builtin_bit_cast(bf16x8_t, make_uint4(w == 0 ? one : 0u, w == 1 ? one : 0u, w == 2 ? one : 0u,
                                                       w == 3 ? one : 0u));
    }
  }

  MfFrags<KS> fk, fq;  // the current block's K and Q fragments

  // ---- staging: lane (g, i) computes token i of each block for its head ----
  // bit 4 b + h: block b of head h runs in true units (at most 8 blocks); bit b: block b holds a non-finite
  // coefficient, beta or k
  uint32_t exact = 0, marked = 0;
  float Gr = 1.0f, Gi = 0.0f;
  if (live) {
    const float al = a.alpha[hl], om = a.omega[hl];
#pragma unroll 1
    for (int b0 = 0; b0 < nb; b0 += 4) {
      float sb[4], ss[4], sd[4], sr4[4], sv0[4], sv1[4];
      if (a.wide) {
        // one 8-byte row (4 heads) of array g (beta, sel, dt, r) per lane and token, and the
        // token's v pair of the lane's own head; the 4 x 4 exchange between lane groups and heads
        // leaves each lane with its head's four scalars
        uint2 w4[4];
        uint32_t pv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int64_t tk = (row0 + min(16 * (b0 + u) + i, tlast)) * H;
          const uint16_t* src = g == 0 ? a.beta : g == 1 ? a.sel : g == 2 ? a.dt : a.r;
          w4[u] = *reinterpret_cast<const uint2*>(src + tk + hbase);
          pv[u] = *reinterpret_cast<const uint32_t*>(a.v + 2 * (tk + hl));
        }
        if (b0 == 0) fk.load(krs, voff(0), hoff);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          float x[4] = {bf16_lo(w4[u].x), bf16_hi(w4[u].x), bf16_lo(w4[u].y), bf16_hi(w4[u].y)};
          swap32(x[0], x[2]);
          swap32(x[1], x[3]);
          swap16(x[0], x[1]);
          swap16(x[2], x[3]);
          sb[u] = x[0];
          ss[u] = x[1];
          sd[u] = x[2];
          sr4[u] = x[3];
          sv0[u] = bf16_lo(pv[u]);
          sv1[u] = bf16_hi(pv[u]);
        }
      } else {
      uint16_t rb[4], rs[4], rd[4], rr[4], rv0[4], rv1[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = min(16 * (b0 + u) + i, tlast);
        const int64_t e = (row0 + t) * H + hl;
        rb[u] = a.beta[e];
        rs[u] = a.sel[e];
        rd[u] = a.dt[e];
        rr[u] = a.r[e];
        rv0[u] = a.v[2 * e];
        rv1[u] = a.v[2 * e + 1];
      }
      // the rows go out after the first scalars, so waiting for those does not wait for the rows
      if (b0 == 0) fk.load(krs, voff(0), hoff);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        sb[u] = bf16_to_f32(rb[u]);
        ss[u] = bf16_to_f32(rs[u]);
        sd[u] = bf16_to_f32(rd[u]);
        sr4[u] = bf16_to_f32(rr[u]);
        sv0[u] = bf16_to_f32(rv0[u]);
        sv1[u] = bf16_to_f32(rv1[u]);
      }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int b = b0 + u;
        if (b < nb) {
          const bool real = hok && 16 * b + i < nt;
          const Transition tr = cayley_gated(sd[u], sr4[u], al, om, a.c);
          const float bt = real ? sb[u] : 0.0f;
          const float fw = bt * tr.vp;
          const float wr = real ? fw * sv0[u] : 0.0f, wi = real ? fw * sv1[u] : 0.0f;
          const float ar = real ? tr.ar : 1.0f, ai = real ? tr.ai : 0.0f;
          float fr = ar, fi = ai;
          row_cumprod(fr, fi);
          const float sr = fr * kMfScale, si = fi * kMfScale;
          const float m2 = sr * sr + si * si;
          const float inv = __builtin_amdgcn_rcpf(m2);
          float er = (wr * sr + wi * si) * inv * kMfScale, ei = (wi * sr - wr * si) * inv * kMfScale;
          const bool out = !(m2 >= kMfTiny && m2 < __builtin_inff()) || !(fabsf(er) + fabsf(ei) < kMfLarge);
          const unsigned long long m = __builtin_amdgcn_ballot_w64(out);
          if (m) {
            uint32_t heads = 0;
#pragma unroll
            for (int h = 0; h < kMfHeads; ++h) heads |= ((m >> (16 * h)) & 0xffffull) ? 1u << h : 0u;
            exact |= heads << (kMfHeads * b);
            if ((heads >> opaque(g)) & 1u) {
              er = wr;
              ei = wi;
            }
          }
          marked |= __builtin_amdgcn_ballot_w64(!((fabsf(er) + fabsf(ei)) + bt < __builtin_inff())) != 0ull ? 1u << b : 0u;
          tokA[b * 64 + lane] = make_float4(er, ei, bt, real ? ss[u] : 0.0f);
          tokB[b * 64 + lane] = make_float4(fr, fi, ar, ai);
          cmul_acc(Gr, Gi, row_bcast<15>(fr), row_bcast<15>(fi));
        }
      }
    }
    if (i == 0) GF[wv * kMfHeads + g] = make_float4(Gr, Gi, 0.0f, 0.0f);
  }
  clock(1);
  __syncthreads();  // the zeros

  f32x4_t st[KS][2];  // dims 32 ks + 2 i + u of head g: (H re, H im, c re, c im)

  // the state into the operand rows, hi in rows 0, 1 (re, im) and mid in rows 2, 3; the lo part of H in rows
  // 0, 1 in the local pass, in rows 2, 3 in the correction pass, where rows 0, 1 hold c's
  auto put_state = [&](bool corr) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint32_t hi, mid, lo;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        split3(st[ks][0][p], st[ks][1][p], hi, mid, lo);
        opw[p * SROW + 16 * ks] = hi;
        opw[(2 + p) * SROW + 16 * ks] = mid;
        opw[(corr ? 2 + p : p) * SROW + D + 16 * ks] = lo;
      }
      if (corr) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          split3(st[ks][0][2 + p], st[ks][1][2 + p], hi, mid, lo);
          opw[p * SROW + D / 2 + 16 * ks] = hi;
          opw[(2 + p) * SROW + D / 2 + 16 * ks] = mid;
          opw[p * SROW + D + 16 * ks] = lo;
        }
      }
    }
  };
  // the operand rows (lane: row lane % 16, 8 dims of each step) at dword offset off
  auto load_op = [&](int off, bf16x8_t (&s)[KS]) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      s[ks] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(opr + off + 16 * ks));
  };
  // acc[h] += (operand rows) . f of head h; rows 4 h + part of acc[h] are head h's, in lane group h
  auto project = [&](const bf16x8_t (&s)[KS], const MfFrags<KS>& f, f32x4_t (&acc)[kMfHeads]) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int h = 0; h < kMfHeads; ++h) acc[h] = mfma16(s[ks], f.f[h][ks], acc[h]);
  };
  // the lane group's own head's register of four heads' tiles
  const bool g1 = (g & 1) != 0, g2 = (g & 2) != 0;
  auto own = [&](float x0, float x1, float x2, float x3) {
    const float a0 = g1 ? x1 : x0, a1 = g1 ? x3 : x2;
    return g2 ? a1 : a0;
  };
#define MF_OWN(T, R) own(T[0][R], T[1][R], T[2][R], T[3][R])
  // K^T of the block in the B layout, two heads to an operand: kt[p][ks][u] = tokens 4 g ..+4 of dim
  // 32 ks + 2 i + u of head 2 p, then of head 2 p + 1
  auto transpose_k = [&](const MfFrags<KS>& f, bf16x8_t (&kt)[kMfHeads / 2][KS][2]) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      f32x4_t x[kMfHeads][2];
#pragma unroll
      for (int h = 0; h < kMfHeads; ++h)
#pragma unroll
        for (int u = 0; u < 2; ++u) x[h][u] = mfma16(f.f[h][ks], sel2[u], f32x4_t{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
      for (int p = 0; p < kMfHeads / 2; ++p)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          uint32_t w[4];
#pragma unroll
          for (int n = 0; n < 4; ++n) {
            const f32x4_t& y = x[2 * p + n / 2][u];
            w[n] = __builtin_amdgcn_perm(__float_as_uint(y[2 * (n % 2) + 1]), __float_as_uint(y[2 * (n % 2)]), 0x07060302u);
          }
          // packed here, not at the use: the unpacked tiles would hold twice the registers until then
          asm("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
          kt[p][ks][u] = __builtin_bit_cast(bf16x8_t, make_uint4(w[0], w[1], w[2], w[3]));
        }
    }
  };
  // the coefficient rows as A operands: e[p][m], term m (hi, mid, lo) of heads 2 p (k first half) and 2 p + 1
  auto load_coef = [&](bf16x8_t (&e)[kMfHeads / 2][3]) {
    const int hi = opaque(i) / 4;
#pragma unroll
    for (int p = 0; p < kMfHeads / 2; ++p)
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        const uint2 x = *reinterpret_cast<const uint2*>((hi == 2 * p ? ebr : zero) + 8 * m);
        const uint2 y = *reinterpret_cast<const uint2*>((hi == 2 * p + 1 ? ebr : zero) + 8 * m);
        e[p][m] = __builtin_bit_cast(bf16x8_t, make_uint4(x.x, x.y, y.x, y.y));
      }
  };
  // state += sum over the block's tokens of (coefficient row) k_s
  auto update_state = [&](const bf16x8_t (&e)[kMfHeads / 2][3], const bf16x8_t (&kt)[kMfHeads / 2][KS][2]) {
#pragma unroll
    for (int p = 0; p < kMfHeads / 2; ++p)
#pragma unroll
      for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int u = 0; u < 2; ++u) st[ks][u] = mfma16(e[p][m], kt[p][ks][u], st[ks][u]);
  };
  auto put_coef = [&](int part, float x0, float x1) {
    uint32_t hi, mid, lo;
    split3(x0, x1, hi, mid, lo);
    uint16_t* w = ebw + part * 48;
    w[0] = uint16_t(hi & 0xffffu);
    w[48] = uint16_t(hi >> 16);
    w[16] = uint16_t(mid & 0xffffu);
    w[64] = uint16_t(mid >> 16);
    w[32] = uint16_t(lo & 0xffffu);
    w[80] = uint16_t(lo >> 16);
  };
  auto scale_local = [&](float sr, float si) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float xr = st[ks][u][0], xi = st[ks][u][1];
        cmul_acc(xr, xi, sr, si);
        st[ks][u][0] = xr;
        st[ks][u][1] = xi;
      }
  };
  // prod_{s<u<=15} a_u over the block (true units' weight of token s in the state after the block)
  auto suffix = [&](float ar, float ai, float& xr, float& xi) {
    for_shifts<16>([&](auto sh) {
      constexpr int N = decltype(sh)::value;
      const float yr = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(1.0f), __float_as_int(ar), 0x100 + N,
                                                                  0xF, 0xF, false));
      const float yi = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ai), 0x100 + N, 0xF, 0xF, false));
      cmul_acc(ar, ai, yr, yi);
    });
    xr = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(1.0f), __float_as_int(ar), 0x101, 0xF, 0xF, false));
    xi = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ai), 0x101, 0xF, 0xF, false));
  };
  const float qnan = __builtin_nanf("");
  auto mine = [&](int b) { return ((exact >> (kMfHeads * b)) >> opaque(g)) & 1u; };  // this lane's head in true units
  // Tokens of a marked block (bit t) whose coefficient or beta is not finite in this lane's head; their
  // coefficient and beta are replaced by zeros.
  auto poison = [&](float4& ta) {
    const unsigned long long m =
        __builtin_amdgcn_ballot_w64(!((fabsf(ta.x) + fabsf(ta.y)) + fabsf(ta.z) < __builtin_inff()));
    const uint32_t row = uint32_t(m >> (16 * opaque(g))) & 0xffffu;
    if ((row >> i) & 1u) ta.x = ta.y = ta.z = 0.0f;
    return row;
  };

  // ---- local pass: update coefficients and the state at the chunk's end, from zero ----
  auto local_block = [&](int b) {
    f32x4_t gt[kMfHeads], ka[kMfHeads];
    bf16x8_t kt[kMfHeads / 2][KS][2];
    bf16x8_t s1[KS], s2[KS];
    load_op(0, s1);
    load_op(D, s2);
    float4 ta = tokA[b * 64 + lane];
    const float4 tb = tokB[b * 64 + lane];
    for (int pass = 0;; ++pass) {
      mf_gram<KS>(fk, fk, gt);
      transpose_k(fk, kt);
#pragma unroll
      for (int h = 0; h < kMfHeads; ++h) ka[h] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      project(s1, fk, ka);
      project(s2, fk, ka);
      if (pass || mf_finite(gt)) break;
      if (mf_sanitize<KS>(fk, g, i)) ta.x = qnan;
      marked |= 1u << b;
    }
    fk.load(krs, voff(b + 1), hoff);
    uint32_t bad = 0;
    if ((marked >> b) & 1u) bad = poison(ta);
    const float khr = MF_OWN(ka, 0) + MF_OWN(ka, 2), khi = MF_OWN(ka, 1) + MF_OWN(ka, 3);
    float Lr[16];
    mf_rows(gt, g, i, Lr);
#pragma unroll
    for (int s = 0; s < 16; ++s) Lr[s] *= -ta.z;
    const bool ex = (exact >> (kMfHeads * b)) & 15u;
    float f15r = row_bcast<15>(tb.x);
    const float f15i = row_bcast<15>(tb.y);
    if (bad) f15r = qnan;  // the state after the block
    scale_local(f15r, f15i);
    float xr = fmaf(-ta.z, khr, ta.x), xi = fmaf(-ta.z, khi, ta.y);
    mf_solve(Lr, xr, xi);
    float cr = f15r, ci = f15i;  // to the block's end
    if (ex) {
      asm volatile("");  // a branch, not selects
      // e_t = w_t - beta_t f_t (k_t.H) + a_t A_t, A_t = sum_{s<t} prod_{s<u<t} a_u L_ts e_s
      const float br = ta.x - ta.z * (tb.x * khr - tb.y * khi), bi2 = ta.y - ta.z * (tb.x * khi + tb.y * khr);
      float Ar = 0.0f, Ai = 0.0f, tr = 0.0f, ti = 0.0f;
      const int ii = opaque(i);
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        const float er = br + (tb.z * Ar - tb.w * Ai), ei = bi2 + (tb.z * Ai + tb.w * Ar);
        tr = s == ii ? er : tr;
        ti = s == ii ? ei : ti;
        const float sr = row_bcast_dyn(tb.z, s), si = row_bcast_dyn(tb.w, s);
        cmul_acc(Ar, Ai, sr, si);
        Ar = fmaf(Lr[s], row_bcast_dyn(er, s), Ar);
        Ai = fmaf(Lr[s], row_bcast_dyn(ei, s), Ai);
      }
      float ur, ui;
      suffix(tb.z, tb.w, ur, ui);
      const bool m = mine(b);
      xr = m ? tr : xr;
      xi = m ? ti : xi;
      cr = m ? ur : cr;
      ci = m ? ui : ci;
    }
    cmul_acc(cr, ci, xr, xi);
    tokA[b * 64 + lane] = make_float4((bad >> i) & 1u ? qnan : xr, xi, ta.z, ta.w);
    put_coef(0, cr, ci);
    wave_fence();
    bf16x8_t e[kMfHeads / 2][3];
    load_coef(e);
    update_state(e, kt);
    if (b + 1 < nb) put_state(false);
    wave_fence();
  };
  if (live) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) st[ks][0] = st[ks][1] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    put_state(false);
    wave_fence();
#pragma unroll 1
    for (int b = 0; b < nb; ++b) local_block(b);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      *reinterpret_cast<float4*>(&Fx[wv * SEGN + g * D + 32 * ks + 2 * i]) =
          make_float4(st[ks][0][0], st[ks][0][1], st[ks][1][0], st[ks][1][1]);
  }
  __syncthreads();
  clock(2);

  // ---- carry; the correction's first rows are requested once the segment map is out ----
  segment_carry<D, kMfHeads>(a.ob, a.h0, a.h_final, H, a.NSEG, bi, seg, hbase, n_live, wv, Fx, GF, Sx, ctrl, epoch,
                             true, &g_mf_calls, &g_mf_status, kMfTag, [&](int n) {
                               if (n == 3 && live) {
                                 fk.load(krs, voff(0), hoff);
                                 fq.load(qrs, voff(0), hoff);
                               }
                               clock(n);
                             });
  clock(5);

  // ---- correction pass ----
  char* yblk = reinterpret_cast<char*>(a.y) + (row0 * H + hbase) * 4;  // the block's rows
  auto corr_block = [&](int b) {
    f32x4_t gt[kMfHeads], pt[kMfHeads], ka[kMfHeads], qh[kMfHeads], qc[kMfHeads], ql[kMfHeads];
    bf16x8_t kt[kMfHeads / 2][KS][2];
    bf16x8_t s1[KS], s2[KS], s3[KS];
    load_op(0, s1);
    load_op(D / 2, s2);
    load_op(D, s3);
    const bool ex = (exact >> (kMfHeads * b)) & 15u;
    // the three phases (q, k, the rest) are kept apart: interleaved, their tiles would not fit the registers
#pragma unroll
    for (int h = 0; h < kMfHeads; ++h) qh[h] = qc[h] = ql[h] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    mf_gram<KS>(fk, fq, pt);
    project(s3, fq, ql);
    project(s1, fq, qh);
    const float qhr = MF_OWN(qh, 0) + (MF_OWN(qh, 2) + MF_OWN(ql, 2));
    const float qhi = MF_OWN(qh, 1) + (MF_OWN(qh, 3) + MF_OWN(ql, 3));
    __builtin_amdgcn_sched_barrier(0);
    project(s2, fq, qc);
    float qcr = MF_OWN(qc, 0) + (MF_OWN(qc, 2) + MF_OWN(ql, 0)), qci = MF_OWN(qc, 1) + (MF_OWN(qc, 3) + MF_OWN(ql, 1));
    fq.load(qrs, voff(b + 1), hoff);
    __builtin_amdgcn_sched_barrier(0);
    for (int pass = 0;; ++pass) {
      mf_gram<KS>(fk, fk, gt);
      transpose_k(fk, kt);
#pragma unroll
      for (int h = 0; h < kMfHeads; ++h) ka[h] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s3[ks] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(oprc + 16 * ks));
      project(s2, fk, ka);
      project(s3, fk, ka);
      if (pass || mf_finite(gt)) break;
      mf_sanitize<KS>(fk, g, i);  // the local pass has marked the token
    }
    float4 ta = tokA[b * 64 + lane];
    const float4 tb = tokB[b * 64 + lane];
    fk.load(krs, voff(b + 1), hoff);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t bad = 0;
    if ((marked >> b) & 1u) {
      bad = poison(ta);
      if (bad & ((2u << i) - 1u)) ta.w = qnan;  // outputs from the first such token on
    }
    float cxr = ta.z * (MF_OWN(ka, 0) + MF_OWN(ka, 2)), cxi = ta.z * (MF_OWN(ka, 1) + MF_OWN(ka, 3));
    {
      float Lr[16];
      mf_rows(gt, g, i, Lr);
#pragma unroll
      for (int s = 0; s < 16; ++s) Lr[s] *= -ta.z;
      mf_solve(Lr, cxr, cxi);
    }
    float f15r = row_bcast<15>(tb.x);
    const float f15i = row_bcast<15>(tb.y);
    if (bad) f15r = qnan;  // the local state, and through the product of a every later output of the chunk
    float cr = f15r, ci = f15i;
    if (ex) {
      asm volatile("");  // a branch, not selects
      float ur, ui;
      suffix(tb.z, tb.w, ur, ui);
      const bool m = mine(b);
      cr = m ? ur : cr;
      ci = m ? ui : ci;
    }
    cmul_acc(cr, ci, ta.x, ta.y);
    put_coef(0, cr, ci);
    put_coef(2, -cxr, -cxi);
    wave_fence();
    // sum_{s<t} P_ts (coefficient rows of s), in fp32: 16 products of 4 x 1 by 1 x 4 per step s, of which lane
    // (g, i) gets the 4 sums of its own token and head; the coefficient rows pass through the block's slots
    float* cf = reinterpret_cast<float*>(tokA + b * 64);
    cf[64 * g + i] = ta.x;
    cf[64 * g + 16 + i] = ta.y;
    cf[64 * g + 32 + i] = -cxr;
    cf[64 * g + 48 + i] = -cxi;
    wave_fence();
    float P[16];
    mf_rows(pt, g, i, P);
    const float pd = mf_diag(pt, g, i);
    f32x4_t ps = {0.0f, 0.0f, 0.0f, 0.0f}, ps2 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 16; s += 4) {
      const float4 x = *reinterpret_cast<const float4*>(cf + 64 * g + 16 * (i % 4) + s);
      ps = __builtin_amdgcn_mfma_f32_4x4x1f32(x.x, P[s], ps, 0, 0, 0);
      ps2 = __builtin_amdgcn_mfma_f32_4x4x1f32(x.y, P[s + 1], ps2, 0, 0, 0);
      ps = __builtin_amdgcn_mfma_f32_4x4x1f32(x.z, P[s + 2], ps, 0, 0, 0);
      ps2 = __builtin_amdgcn_mfma_f32_4x4x1f32(x.w, P[s + 3], ps2, 0, 0, 0);
    }
    ps += ps2;
    qcr += ps[2];
    qci += ps[3];
    const float vr = qhr + fmaf(pd, ta.x, ps[0]), vi = qhi + fmaf(pd, ta.y, ps[1]);
    float lr = tb.x * vr - tb.y * vi, li = tb.x * vi + tb.y * vr;
    if (ex) {
      asm volatile("");
      float er = 0.0f, ei = 0.0f;
      const int ii = opaque(i);
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        float nr = er, ni = ei;
        cmul_acc(nr, ni, row_bcast_dyn(tb.z, s), row_bcast_dyn(tb.w, s));
        const float p = s == ii ? pd : P[s];
        nr = fmaf(p, row_bcast_dyn(ta.x, s), nr);
        ni = fmaf(p, row_bcast_dyn(ta.y, s), ni);
        er = s <= ii ? nr : er;
        ei = s <= ii ? ni : ei;
      }
      if (mine(b)) {
        lr = fmaf(tb.x, qhr, fmaf(-tb.y, qhi, er));
        li = fmaf(tb.x, qhi, fmaf(tb.y, qhr, ei));
      }
    }
    bf16x8_t e[kMfHeads / 2][3];
    load_coef(e);
    // g_{t-1} of the chunk
    float gr = row_shr<1>(tb.x, 1.0f), gi = row_shr<1>(tb.y, 0.0f);
    cmul_acc(gr, gi, Gr, Gi);
    const float yr = ta.w * fmaf(gr, qcr, fmaf(-gi, qci, lr)), yi = ta.w * fmaf(gr, qci, fmaf(gi, qcr, li));
    if (hok && 16 * b + i < nt) *reinterpret_cast<uint32_t*>(yblk + uint32_t(i * H + g) * 4u) = pack_bf16x2(yr, yi);
    if (b + 1 < nb) {
      scale_local(f15r, f15i);
      update_state(e, kt);
      put_state(true);
      wave_fence();
      cmul_acc(Gr, Gi, f15r, f15i);
    }
  };
  if (live) {
    // state entering this wave's chunk
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int e0 = g * D + 32 * ks + 2 * i;
      float4 s = *reinterpret_cast<const float4*>(&Sx[e0]);
      for (int u = 0; u < wv; ++u) {
        const float4 G = GF[u * kMfHeads + g];
        const float4 F = *reinterpret_cast<const float4*>(&Fx[u * SEGN + e0]);
        const float2 n0 = map_apply<false>(make_float2(G.x, G.y), make_float2(s.x, s.y), make_float2(F.x, F.y));
        const float2 n1 = map_apply<false>(make_float2(G.x, G.y), make_float2(s.z, s.w), make_float2(F.z, F.w));
        s = make_float4(n0.x, n0.y, n1.x, n1.y);
      }
      if (!hok) s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      st[ks][0] = f32x4_t{0.0f, 0.0f, s.x, s.y};
      st[ks][1] = f32x4_t{0.0f, 0.0f, s.z, s.w};
    }
    put_state(true);
    wave_fence();
    Gr = 1.0f;
    Gi = 0.0f;
#pragma unroll 1
    for (int b = 0; b < nb; ++b) {
      corr_block(b);
      yblk += 64 * H;
    }
  }
  clock(6);
  if (stamping && lane == 0) {
    clock(7);
    const int n_hg = (H + a.stamp_heads - 1) / a.stamp_heads, sg = hbase / a.stamp_heads;
    unsigned long long* o = a.stamps + (((int64_t(seg) * a.B + bi) * n_hg + sg) * W + wv) * kStampPoints;
    if (sg * a.stamp_heads == hbase)
#pragma unroll
      for (int n = 0; n < kStampPoints; ++n) o[n] = ts[n];
  }
}

// One workgroup per segment, all resident at once (a workgroup may wait on any earlier segment).  Shapes
// with more segments than that run the persistent fused_fwd_onepass_kernel: a loop over segments here
// keeps the staging's pointers live through the passes (46 to 190 scalar registers spilled), and measured
// slower than that kernel from two rounds on (B1 H32 L65536 D64: 196-206 against 177 us).
template <int D>
__global__ __launch_bounds__(kWave* kOnePassW, D == 64 ? 2 : 1) void mf_onepass_kernel(MfArgs a) {
  mf_segment<D>(a, int(blockIdx.x), call_epoch(a.ob));
}

template <int D>
int mf_capacity(int Q) {
  return cdssm_host::resident_capacity(reinterpret_cast<const void*>(&mf_onepass_kernel<D>), kWave * kOnePassW,
                                       MfCfg<D>::lds_bytes(Q));
}

template <int D>
int mf_launch(const MfmaForward& p, hipStream_t stream, hipEvent_t* ev) {
  const FwdLayout w = fwd_layout(p.B, p.L, p.H, D, p.Q);
  MfArgs a;
  a.q = static_cast<const uint16_t*>(p.q);
  a.k = static_cast<const uint16_t*>(p.k);
  a.v = static_cast<const uint16_t*>(p.v);
  a.beta = static_cast<const uint16_t*>(p.beta);
  a.sel = static_cast<const uint16_t*>(p.sel_c);
  a.dt = static_cast<const uint16_t*>(p.dt);
  a.r = static_cast<const uint16_t*>(p.r);
  a.alpha = p.alpha;
  a.omega = p.omega;
  a.c = p.c;
  a.h0 = p.h0;
  a.y = static_cast<uint16_t*>(p.y);
  a.h_final = p.h_final;
  const int64_t nsd = int64_t(p.B) * w.NSEG * p.H * D, nsh = int64_t(p.B) * w.NSEG * p.H;
  float2* base = p.lookback;
  unsigned long long* flags = reinterpret_cast<unsigned long long*>(base + 2 * nsd + nsh);
  a.ob = OnePassBufs{base, base + nsd, base + 2 * nsd, flags, flags + nsh};
  a.ob.grp_f = reinterpret_cast<float2*>(flags + nsh + kCtlWords);
  a.ob.grp_g = a.ob.grp_f + int64_t(p.B) * fwd_groups(w.NSEG) * p.H * D;
  a.L = p.L;
  a.H = p.H;
  a.Q = p.Q;
  a.NC = w.NC;
  a.NSEG = w.NSEG;
  a.B = p.B;
  a.n_hg = (p.H + kMfHeads - 1) / kMfHeads;
  auto on = [](const void* x, uintptr_t n) { return (reinterpret_cast<uintptr_t>(x) & (n - 1)) == 0; };
  a.wide = p.H % kMfHeads == 0 && on(p.beta, 8) && on(p.sel_c, 8) && on(p.dt, 8) && on(p.r, 8) && on(p.v, 4);
  const int64_t items = int64_t(w.NSEG) * p.B * a.n_hg;
  a.stamps = nullptr;
  a.stamp_heads = kMfHeads;
  if (p.stamps) {
    // a buffer for items of 8 heads (the sequential kernel's) takes the records of each one's first 4
    if (p.stamps_len < items * kOnePassW * kStampPoints && D == 64) a.stamp_heads = 2 * kMfHeads;
    const int64_t words = int64_t(w.NSEG) * p.B * ((p.H + a.stamp_heads - 1) / a.stamp_heads) * kOnePassW * kStampPoints;
    if (p.stamps_len < words) {
      cdssm_host::set_error("cdssm_fused_scan_fwd_stamped: %lld stamp words needed (%lld given)", (long long)words,
                            (long long)p.stamps_len);
      return CDSSM_EINVAL;
    }
    a.stamps = p.stamps;
  }
  if (!p.cont) a.ob.epoch = cdssm_host::draw_call_epoch(kMfTag, stream);
  if (!p.cont && !a.ob.epoch) {
    hipLaunchKernelGGL(mf_epoch_kernel, dim3(1), dim3(64), 0, stream, a.ob.ctl);
    const int st = cdssm_host::check_launch("cdssm_fused_scan_fwd/epoch");
    if (st) return st;
  }
  if (ev)
    for (int n = 0; n < 4; ++n) (void)hipEventRecord(ev[n], stream);
  hipLaunchKernelGGL((mf_onepass_kernel<D>), dim3(unsigned(items)), dim3(kWave * kOnePassW),
                     MfCfg<D>::lds_bytes(p.Q), stream, a);
  const int st = cdssm_host::check_launch("cdssm_fused_scan_fwd/mfma");
  if (ev) (void)hipEventRecord(ev[4], stream);
  return st;
}

}  // namespace

bool mfma_forward_fits(int64_t B, int64_t L, int64_t H, int D, int Q) {
  const int64_t nc = (L + Q - 1) / Q, nseg = (nc + kOnePassW - 1) / kOnePassW;
  return nseg * B * ((H + kMfHeads - 1) / kMfHeads) <= (D == 64 ? mf_capacity<64>(Q) : mf_capacity<128>(Q));
}

int launch_mfma_forward(const MfmaForward& p, hipStream_t stream, hipEvent_t* ev) {
  return p.D == 64 ? mf_launch<64>(p, stream, ev) : mf_launch<128>(p, stream, ev);
}

int mfma_forward_status(bool clear, unsigned* out) {
  unsigned v = 0;
  if (hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_mf_status), sizeof(v), 0, hipMemcpyDeviceToHost) != hipSuccess) {
    cdssm_host::set_error("cdssm_lookback_status: reading the forward status word failed: %s",
                          hipGetErrorString(hipGetLastError()));
    return CDSSM_EHIP;
  }
  if (clear && v) {
    const unsigned zero = 0;
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_mf_status), &zero, sizeof(zero), 0, hipMemcpyHostToDevice) != hipSuccess) {
      cdssm_host::set_error("cdssm_lookback_status: clearing the forward status word failed: %s",
                            hipGetErrorString(hipGetLastError()));
      return CDSSM_EHIP;
    }
  }
  *out = v;
  return CDSSM_OK;
}

}  // namespace cdssm
