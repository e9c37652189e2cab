// Skinny GEMM for decode batches: Y (M x N) = X (M x K) W^T (+ bias) (+ R),
// M <= 64, bf16 operands, fp32 accumulation, bf16 out.  With a norm weight
// the rows of X are RMS-normalised first (the model's RMSNorm ahead of
// in_proj and of the LM head, modules.py:49-53):
//   Y = rs ⊙ ((X ⊙ w_norm) W^T),  rs[m] = rsqrt(mean_k X[m,k]^2 + eps),
// with X ⊙ w_norm rounded to bf16 on the way into the matrix cores and rs
// applied to the fp32 result.
//
// These products (decode: in_proj 1024 -> 3104, the stacked gate/Q
// projection 1024 -> 1136 and out_proj 1024 -> 1024 at M = 64) read a weight
// once and a 128 KB activation many times; the library GEMMs tile them for
// large M.  (At N = 32000, the tied head, the activation's re-reads dominate:
// 46 us here against 18 us for the library GEMM.)  Here a workgroup owns 16
// output columns and 16, 32 or 64 rows: its waves split K (8 waves when K is a
// multiple of 256, so that at K = 1024 each wave issues all of its loads in
// one batch; 4 otherwise), each running v_mfma_f32_16x16x32_bf16 on operands
// loaded straight from global memory in the instruction's layout (a 16-byte
// load per lane per fragment: rows of X, rows of W), and the waves' partial
// tiles are summed in a fixed order through LDS.  The order of every sum is
// the same for any number of rows per workgroup.
//
// A call is one latency chain: its weight rows, its activation rows, the sum.
// What bounds it is how many loads one CU has to issue and return, so the rows
// are split over the CUs as far as one round of workgroups takes them
// (one per CU).  Measured on MI355X at M = 64, K = 1024, us per call back to
// back, for 16 / 32 / 64 rows per workgroup: N = 1024 4.5 / 5.2 / 7.0,
// N = 1552 6.2 / 5.3 / 6.9, N = 2048 6.2 / 5.5 / 7.3, N = 3104 9.7 / 8.6 / 7.9;
// with the norm at N = 1024 5.2 / 6.0 / 8.0, N = 3104 10.9 / 8.9 / 8.9.  At
// M = 16, K = 2048, N = 4096 7.5 / 7.7 / 9.0.  (Always 64 rows before.)  Where the
// line lies, 256 CUs, M = 64, K = 1024, in a graph over 8 weights, 16 / 32 / 64
// rows: N = 1024 (256 workgroups of 16 rows) 4.1 / - / 6.8, N = 1040 (260) 5.7 / 5.0
// / 6.8, N = 1136 (284) 5.8 / 5.0 / 6.8, N = 1440 (360) 6.0 / 5.3 / 7.1.
//
// Fragment layouts of v_mfma_f32_16x16x32_bf16 (checked on MI355X):
//   A (16 x 32): lane l holds row l % 16, k = 8 (l / 16) .. + 8
//   B (32 x 16): lane l holds column l % 16, k = 8 (l / 16) .. + 8
//   C (16 x 16): lane l holds column l % 16, rows 4 (l / 16) .. + 4
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "lm_common.hpp"

namespace cdssm {
namespace sg {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kCols = 16;   // output columns per workgroup
constexpr int kMaxRows = 64;
constexpr int kUnroll = 4;  // k-steps (of 32) whose loads are issued together

__device__ __forceinline__ uint4 ld16(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }

// a 16-byte fragment times 8 bf16 weights, rounded back to bf16
__device__ __forceinline__ uint4 scale_frag(uint4 a, uint4 w) {
  uint4 o;
  o.x = pack_bf16x2(bf16_lo(a.x) * bf16_lo(w.x), bf16_hi(a.x) * bf16_hi(w.x));
  o.y = pack_bf16x2(bf16_lo(a.y) * bf16_lo(w.y), bf16_hi(a.y) * bf16_hi(w.y));
  o.z = pack_bf16x2(bf16_lo(a.z) * bf16_lo(w.z), bf16_hi(a.z) * bf16_hi(w.z));
  o.w = pack_bf16x2(bf16_lo(a.w) * bf16_lo(w.w), bf16_hi(a.w) * bf16_hi(w.w));
  return o;
}

__device__ __forceinline__ float sumsq_frag(uint4 a, float s) {
  const uint32_t u[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    s = fmaf(bf16_lo(u[i]), bf16_lo(u[i]), s);
    s = fmaf(bf16_hi(u[i]), bf16_hi(u[i]), s);
  }
  return s;
}

// A causal conv step on C of the product's columns, from column col0 (conv1d_silu_step_kernel's arithmetic on
// the rounded result): window (M, taps - 1, C) is read and shifted, y (M, C) written.
constexpr int kMaxTaps = 8;
struct ConvStep {
  uint16_t* window;
  const uint16_t *w, *bias;  // (C, taps), (C)
  uint16_t* y;
  int col0, C, taps;
};

// 16 * MT rows by 16 columns per workgroup.  CONV: with a conv step on the tile as rounded, spread over all
// threads, which request its windows and weights ahead of the product's loads.  It saves a launch and the wait
// for those loads: M 64, K 1024, N 3104, C 1024, 4 taps on MI355X 11.6 us in place of 9.5 and 4.7 (13.2 with
// the step on the MT finishing waves alone).
template <bool NORM, int kWaves, int MT, bool CONV>
__global__ __launch_bounds__(kWave * kWaves) void skinny_gemm_kernel(
    const uint16_t* __restrict__ X, int64_t ldx, const uint16_t* __restrict__ W, int64_t ldw,
    const uint16_t* __restrict__ bias, const uint16_t* __restrict__ R, int64_t ldr,
    const uint16_t* __restrict__ wnorm, float eps, uint16_t* __restrict__ Y, int64_t ldy, int M, int N, int K, ConvStep cv) {
  __shared__ f32x4_t part[kWaves][MT][kWave];  // 1 KB per wave and row tile: its partial tiles
  __shared__ float ssq[kWaves][16 * MT];       // each wave's partial row sums of squares
  __shared__ uint16_t ytile[CONV ? 16 * MT * kCols : 1];  // the tile as rounded, for the conv step
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
  const int lane = int(threadIdx.x) % kWave;
  const int col = lane % 16, kq = lane / 16;
  // the row groups of a column tile lie 8 workgroups apart (one XCD under the round-robin placement), so the
  // tile's weight rows come from HBM once and from that XCD's L2 for the others
  const int n_nt = (N + kCols - 1) / kCols, n_mg = (M + 16 * MT - 1) / (16 * MT);
  const int grp = int(blockIdx.x) / (8 * n_mg), loc = int(blockIdx.x) - grp * 8 * n_mg;
  const int width = min(8, n_nt - 8 * grp);
  const int mg = loc / width;
  const int n0 = (8 * grp + loc - mg * width) * kCols, m0 = mg * 16 * MT;
  const int n = min(n0 + col, N - 1);  // loads clamped into the matrix; stores masked
  const int kw = K / kWaves;
  const int kb = wave * kw;
  const uint16_t* wrow = W + int64_t(n) * ldw + kb + 8 * kq;
  const uint16_t* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) xrow[mt] = X + int64_t(min(m0 + mt * 16 + col, M - 1)) * ldx + kb + 8 * kq;
  const uint16_t* nrow = NORM ? wnorm + kb + 8 * kq : nullptr;

  // the conv step, spread over all threads: thread t has channel t % 16 of the tile in kItems rows
  constexpr int kRowsApart = kWave * kWaves / kCols, kItems = CONV ? (16 * MT + kRowsApart - 1) / kRowsApart : 1;
  const int ch = CONV ? n0 + col - cv.col0 : -1, cr0 = int(threadIdx.x) / kCols;
  const bool conv = CONV && ch >= 0 && ch < cv.C;
  uint16_t cw[kMaxTaps], cb = 0, win[kItems][kMaxTaps];
  if constexpr (CONV) {
    if (conv) {
#pragma unroll
      for (int i = 0; i < kItems; ++i)
#pragma unroll
        for (int j = 0; j + 1 < kMaxTaps; ++j)
          if (j + 1 < cv.taps)
            win[i][j] =
                cv.window[(int64_t(min(m0 + cr0 + i * kRowsApart, M - 1)) * (cv.taps - 1) + j) * cv.C + ch];
      cb = cv.bias[ch];
#pragma unroll
      for (int j = 0; j < kMaxTaps; ++j)
        if (j < cv.taps) cw[j] = cv.w[int64_t(ch) * cv.taps + j];
    }
  }

  f32x4_t acc[MT];
  float sq[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    acc[mt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    sq[mt] = 0.0f;
  }
  // U k-steps of 32 from k: every load first, then the products
  const auto steps = [&](int k, auto uc) {
    constexpr int U = decltype(uc)::value;
    uint4 b[U], a[U][MT], g[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      b[u] = ld16(wrow + k + 32 * u);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[u][mt] = ld16(xrow[mt] + k + 32 * u);
      if constexpr (NORM) g[u] = ld16(nrow + k + 32 * u);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bf16x8_t bv = __builtin_bit_cast(bf16x8_t, b[u]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        uint4 av = a[u][mt];
        if constexpr (NORM) {
          sq[mt] = sumsq_frag(av, sq[mt]);
          av = scale_frag(av, g[u]);
        }
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av), bv, acc[mt], 0, 0, 0);
      }
    }
  };
  // the wave's quarter of K (a multiple of 32): groups of kUnroll steps, then single steps
  int k = 0;
  for (; k + 32 * kUnroll <= kw; k += 32 * kUnroll) steps(k, std::integral_constant<int, kUnroll>{});
  for (; k < kw; k += 32) steps(k, std::integral_constant<int, 1>{});
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) part[wave][mt][lane] = acc[mt];
  if constexpr (NORM) {
    // the lanes of a row (col) over kq: lanes col, col + 16, col + 32, col + 48
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float s = sq[mt];
      s += __shfl_xor(s, 16, kWave);
      s += __shfl_xor(s, 32, kWave);
      if (kq == 0) ssq[wave][mt * 16 + col] = s;
    }
  }
  __syncthreads();

  // wave w < MT finishes row tile w: the partials in wave order, then the epilogue
  if (wave < MT) {
    const int mt = wave;
    f32x4_t c = part[0][mt][lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) {
      const f32x4_t p = part[w][mt][lane];
      c[0] += p[0];
      c[1] += p[1];
      c[2] += p[2];
      c[3] += p[3];
    }
    const int nn = n0 + col;
    const float bv = bias && nn < N ? bf16_to_f32(bias[nn]) : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ml = mt * 16 + 4 * kq + i, m = m0 + ml;
      if (m < M && nn < N) {
        float y = c[i];
        if constexpr (NORM) {
          float s = 0.0f;
#pragma unroll
          for (int w = 0; w < kWaves; ++w) s += ssq[w][ml];
          s /= float(K);
          y *= __builtin_amdgcn_rsqf(s + eps);
        }
        y += bv;
        if (R) y += bf16_to_f32(R[int64_t(m) * ldr + nn]);
        const uint16_t yb = f32_to_bf16(y);
        Y[int64_t(m) * ldy + nn] = yb;
        if constexpr (CONV) ytile[ml * kCols + col] = yb;
      }
    }
  }
  if constexpr (CONV) {
    __syncthreads();
    if (!conv) return;
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const int ml = cr0 + i * kRowsApart, m = m0 + ml;
      if (ml < 16 * MT && m < M) {
        float u = bf16_to_f32(cb);
        uint16_t* wr = cv.window + int64_t(m) * (cv.taps - 1) * cv.C + ch;
#pragma unroll
        for (int j = 0; j < kMaxTaps; ++j) {
          if (j < cv.taps) {
            const uint16_t in = j + 1 == cv.taps ? ytile[ml * kCols + col] : win[i][j];
            u = fmaf(bf16_to_f32(cw[j]), bf16_to_f32(in), u);
            if (j > 0) wr[int64_t(j - 1) * cv.C] = in;
          }
        }
        cv.y[int64_t(m) * cv.C + ch] = f32_to_bf16(lm::silu_fast(u));
      }
    }
  }
}

}  // namespace sg
}  // namespace cdssm

using namespace cdssm;

static int skinny_gemm(const char* op, int dtype, const void* X, int64_t ldx, const void* W, int64_t ldw,
                       const void* bias, const void* R, int64_t ldr, const void* wnorm, float eps, void* Y,
                       int64_t ldy, int64_t M, int64_t N, int64_t K, const sg::ConvStep* cv, hipStream_t stream) {
  if (dtype != 1) {
    cdssm_host::set_error("%s: bf16 only (dtype 1), got %d", op, dtype);
    return CDSSM_EINVAL;
  }
  if (!X || !W || !Y) {
    cdssm_host::set_error("%s: X, W and Y must not be null", op);
    return CDSSM_EINVAL;
  }
  if (M < 1 || M > sg::kMaxRows || N < 1 || K < 128 || K % 128 != 0 || N > 0x7fffffffLL / sg::kCols) {
    cdssm_host::set_error("%s: needs 1 <= M <= 64, K a positive multiple of 128, N >= 1 "
                          "(M %lld, N %lld, K %lld)", op, (long long)M, (long long)N, (long long)K);
    return CDSSM_EINVAL;
  }
  if (ldx < K || ldw < K || ldy < N || (R && ldr < N) || ldx % 8 || ldw % 8 ||
      (reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(W) |
       reinterpret_cast<uintptr_t>(wnorm)) % 16) {
    cdssm_host::set_error("%s: rows of X and W (and wnorm) must be 16-byte aligned and the "
                          "leading dimensions cover the rows", op);
    return CDSSM_EINVAL;
  }
  const auto* x = static_cast<const uint16_t*>(X);
  const auto* w = static_cast<const uint16_t*>(W);
  const auto* b = static_cast<const uint16_t*>(bias);
  const auto* r = static_cast<const uint16_t*>(R);
  const auto* g = static_cast<const uint16_t*>(wnorm);
  auto* y = static_cast<uint16_t*>(Y);
  auto go = [&](auto norm, auto waves, auto mt) {
    constexpr int kW = decltype(waves)::value, MT = decltype(mt)::value;
    const dim3 grid(unsigned((N + sg::kCols - 1) / sg::kCols * ((M + 16 * MT - 1) / (16 * MT)))), block(kWave * kW);
    constexpr bool kNorm = decltype(norm)::value;
    if (cv)
      hipLaunchKernelGGL((sg::skinny_gemm_kernel<kNorm, kW, MT, true>), grid, block, 0, stream, x, ldx, w, ldw, b, r,
                         ldr, g, eps, y, ldy, int(M), int(N), int(K), *cv);
    else
      hipLaunchKernelGGL((sg::skinny_gemm_kernel<kNorm, kW, MT, false>), grid, block, 0, stream, x, ldx, w, ldw, b, r,
                         ldr, g, eps, y, ldy, int(M), int(N), int(K), sg::ConvStep{});
  };
  using W8 = std::integral_constant<int, 8>;  // K a multiple of 256: K / 8 (a multiple of 32) per wave
  using W4 = std::integral_constant<int, 4>;
  auto rows = [&](auto norm, auto waves) {
    const int64_t nt = (N + sg::kCols - 1) / sg::kCols, mt = (M + 15) / 16;
    const int64_t cap = cdssm_host::device_cus();  // one round: a workgroup per CU
    if (nt * mt <= cap) return go(norm, waves, std::integral_constant<int, 1>{});
    if (nt * ((mt + 1) / 2) <= cap) return go(norm, waves, std::integral_constant<int, 2>{});
    go(norm, waves, std::integral_constant<int, sg::kMaxRows / 16>{});
  };
  if (K % 256 == 0)
    wnorm ? rows(std::true_type{}, W8{}) : rows(std::false_type{}, W8{});
  else
    wnorm ? rows(std::true_type{}, W4{}) : rows(std::false_type{}, W4{});
  return cdssm_host::check_launch(op);
}

// Y (M x N, row stride ldy) = X (M x K, row stride ldx) W^T (W: N x K, row
// stride ldw) + bias (N, or null) + R (M x N, row stride ldr, or null); with
// wnorm (K, or null) the rows of X are RMS-normalised first (eps), as
// described above.  bf16 only (dtype 1); M in 1..64, K a multiple of 128,
// rows 16-byte aligned.  No counterpart in the reference (its decode
// re-forwards the whole sequence through torch's GEMMs).
extern "C" int cdssm_skinny_gemm(int dtype, const void* X, int64_t ldx, const void* W, int64_t ldw,
                                 const void* bias, const void* R, int64_t ldr, const void* wnorm, float eps,
                                 void* Y, int64_t ldy, int64_t M, int64_t N, int64_t K, hipStream_t stream) {
  return skinny_gemm("cdssm_skinny_gemm", dtype, X, ldx, W, ldw, bias, R, ldr, wnorm, eps, Y, ldy, M, N, K, nullptr,
                     stream);
}

// The same, then cdssm_conv1d_silu_step on the rounded columns conv_col .. conv_col + C.
extern "C" int cdssm_skinny_gemm_conv_step(int dtype, const void* X, int64_t ldx, const void* W, int64_t ldw,
                                           const void* bias, const void* wnorm, float eps, void* Y, int64_t ldy,
                                           int64_t M, int64_t N, int64_t K, int64_t conv_col, void* window,
                                           const void* conv_weight, const void* conv_bias, void* conv_y, int64_t C,
                                           int64_t taps, hipStream_t stream) {
  const char* op = "cdssm_skinny_gemm_conv_step";
  if (!conv_weight || !conv_bias || !conv_y || (taps > 1 && !window)) {
    cdssm_host::set_error("%s: null pointer argument", op);
    return CDSSM_EINVAL;
  }
  if (taps < 1 || taps > sg::kMaxTaps || C < 1 || conv_col < 0 || C > N || conv_col > N - C) {
    cdssm_host::set_error("%s: needs 1 <= kernel_size <= 8 and the conv's columns inside the product's "
                          "(column %lld, C %lld, N %lld, kernel_size %lld)", op, (long long)conv_col, (long long)C,
                          (long long)N, (long long)taps);
    return CDSSM_EINVAL;
  }
  const sg::ConvStep cv{static_cast<uint16_t*>(window), static_cast<const uint16_t*>(conv_weight),
                        static_cast<const uint16_t*>(conv_bias), static_cast<uint16_t*>(conv_y), int(conv_col), int(C),
                        int(taps)};
  return skinny_gemm(op, dtype, X, ldx, W, ldw, bias, nullptr, 0, wnorm, eps, Y, ldy, M, N, K, &cv, stream);
}
