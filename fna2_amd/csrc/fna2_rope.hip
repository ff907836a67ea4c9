// fna2_rope.hip — varlen rotary position embedding for gfx950.
//
// Replaces NaylisAttention._apply_rope_varlen, which loops over the packed
// sequences on the host (a .tolist() synchronisation per call) and applies
// RotaryPositionalEmbedding.forward to each (FNA2/attention_fna2.py:620-647,
// :143-170).  Here one launch covers every token: token t of sequence b
// (cu[b] <= t < cu[b+1]) sits at position p = t - cu[b], found on the
// device, and for i < D/2
//     angle_i   = p * inv_freq[i]
//     y_i       = x_i cos(angle_i) - x_{i+D/2} sin(angle_i)
//     y_{i+D/2} = x_{i+D/2} cos(angle_i) + x_i sin(angle_i)
// (rotate_half, :158-161; the cos/sin table repeats the D/2 angles,
// :150-154).  The reference builds the table in the tensor's dtype, so for
// bf16/fp16 the position, inv_freq, the angle, cos and sin are each rounded
// to that dtype, and the products and their sum are rounded as separate
// elementwise ops (:169-170); the kernel rounds at the same points (no
// contraction into fused multiply-adds).  sign = -1 rotates by -angle: the
// gradient of the rotation, with the same rounding as autograd's
// g cos + rotate_half^T(g sin).
//
// HBM-bound: each (token, head) row is read once and written once.  A lane
// owns 16 bytes of the row's first half and the matching 16 bytes of its
// second half; the lanes of a wave cover 64 / LPR rows at a time, and the
// lane keeps the cos/sin of its 16-byte column range for all the token's
// heads (computed once per token).  A workgroup covers 4 to 16 consecutive
// tokens; the sequence of a wave's first token comes from a
// binary search of cu_seqlens, later ones by stepping.
#include "fna2_kernels.h"

namespace fna2 {

namespace {

constexpr int kRopeWaves = 4;
constexpr int kRopePasses = 4;  // row passes whose loads are in flight together
// The norm backward reads two tensors and is bound by how many loads the CU
// has in flight: its rows stay raw words until used and the norm weights
// stay in LDS, so that four waves share a SIMD (two with fp32 rows and the
// weights in registers).  Passes in flight per wave, 16-bit and fp32: with
// 16-bit rows a second one no longer fits four waves' registers (c3 pack: 90.6
// us; two passes at three waves 98, four at two 109; before, 104.  fp32, 6000
// tokens: two passes 66, one 73; before, 84.  fp16, c3 pack: 90; before, 108).
constexpr int kBwdOcc = 4;
template <int DT>
constexpr int kBwdPasses = DT == kRopeF32 ? 2 : 1;

// Products and sums that are never fused into a multiply-add (the
// reference evaluates them as separate elementwise ops).
__device__ __forceinline__ float mul_rn(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}
__device__ __forceinline__ float add_rn(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

// Rounding to the element type, as a float.
template <int DT>
__device__ __forceinline__ float rnd(float x) {
  if constexpr (DT == kRopeBF16) {
    return bf16_lo(pack_bf16(x, 0.f));
  } else if constexpr (DT == kRopeF16) {
    return (float)(_Float16)x;
  } else {
    return x;
  }
}

// 16 bytes <-> EPL floats.
template <int DT>
struct Chunk {
  static constexpr int EPL = DT == kRopeF32 ? 4 : 8;
  float v[EPL];
  __device__ __forceinline__ void load(const void* p) {
    const u32x4 w = *(const u32x4*)p;
    if constexpr (DT == kRopeF32) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t u = w[i];  // (a vector element is copied out first)
        v[i] = __builtin_bit_cast(float, u);
      }
    } else if constexpr (DT == kRopeBF16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[2 * i] = bf16_lo(w[i]), v[2 * i + 1] = bf16_hi(w[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const _Float16 lo = __builtin_bit_cast(_Float16, (uint16_t)(w[i] & 0xffffu));
        const _Float16 hi = __builtin_bit_cast(_Float16, (uint16_t)(w[i] >> 16));
        v[2 * i] = (float)lo, v[2 * i + 1] = (float)hi;
      }
    }
  }
  __device__ __forceinline__ void store(void* p) const {
    u32x4 w;
    if constexpr (DT == kRopeF32) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float f = v[i];
        w[i] = __builtin_bit_cast(uint32_t, f);
      }
    } else if constexpr (DT == kRopeBF16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = pack_bf16(v[2 * i], v[2 * i + 1]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        w[i] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[2 * i]) |
               ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[2 * i + 1]) << 16);
    }
    *(u32x4*)p = w;
  }
};

// 16 bytes as loaded (EPL elements), unpacked on use: rows in flight cost
// half the registers of their fp32 values.
template <int DT>
struct Raw {
  static constexpr int EPL = Chunk<DT>::EPL;
  u32x4 w;
  __device__ __forceinline__ void load(const void* p) { w = *(const u32x4*)p; }
  __device__ __forceinline__ void store(void* p) const { *(u32x4*)p = w; }
  __device__ __forceinline__ float get(int e) const {
    if constexpr (DT == kRopeF32) {
      return __builtin_bit_cast(float, (uint32_t)w[e]);
    } else if constexpr (DT == kRopeBF16) {
      return (e & 1) ? bf16_hi(w[e >> 1]) : bf16_lo(w[e >> 1]);
    } else {
      const uint32_t u = w[e >> 1];
      return (float)__builtin_bit_cast(_Float16, (uint16_t)((e & 1) ? (u >> 16) : (u & 0xffffu)));
    }
  }
};

// Lane layout and the token -> sequence walk shared by the kernels: lane
// owns columns [col, col + EPL) of both halves of row lrow + j * rpw of a
// token; a wave covers P.tpw consecutive tokens from t0.
template <int DT>
struct RopeLanes {
  static constexpr int EPL = Chunk<DT>::EPL;
  int lane, half, lpr, rpw, col, lrow, nrows, t0, b;
  __device__ __forceinline__ RopeLanes(const RopeParams& P, int wave_id) {
    lane = threadIdx.x & 63;
    half = P.D / 2;
    lpr = half / EPL;  // lanes per row (divides 64)
    rpw = 64 / lpr;    // rows per wave pass
    col = (lane % lpr) * EPL;
    lrow = lane / lpr;
    nrows = P.Hq + P.Hk;
    t0 = wave_id * P.tpw;
    // Largest b with cu[b] <= t0 (b = -1: before the first sequence).
    const auto cu = const_space(P.cu);
    const int n = P.nseq;
    int lo = -1, hi = n;  // cu[lo] <= t0 < cu[hi]
    if (t0 < P.T) {
      if (uni(cu[n]) <= t0) lo = n;
      else
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (uni(cu[mid]) <= t0) lo = mid;
          else hi = mid;
        }
    }
    b = lo;
  }
  // Step to token t; returns its position, or -1 outside every sequence.
  __device__ __forceinline__ int position(const RopeParams& P, int t) {
    const auto cu = const_space(P.cu);
    while (b < P.nseq && uni(cu[b + 1]) <= t) ++b;
    return (b >= 0 && b < P.nseq) ? t - uni(cu[b]) : -1;
  }
  // Row pointers (q rows first, then k rows).
  __device__ __forceinline__ const char* in_row(const RopeParams& P, const void* q, const void* k,
                                                int64_t qs, int64_t qh, int64_t ks, int64_t kh,
                                                int t, int r) const {
    constexpr int ES = DT == kRopeF32 ? 4 : 2;
    const bool isq = r < P.Hq;
    const int h = isq ? r : r - P.Hq;
    return (const char*)(isq ? q : k) +
           ((int64_t)t * (isq ? qs : ks) + (int64_t)h * (isq ? qh : kh)) * ES;
  }
};

// cos and sin of a token's D / 2 angles, each formed by one lane of the wave
// and handed to the others through LDS: the 64 / lpr rows of a wave pass
// share their columns, so forming them where they are used repeats every
// sincosf 64 / lpr times (8 at d = 128 in bf16).  TD: the type the table is
// rounded to.  (c3 pack, 16384 tokens x 32 heads of 128, bf16: norm backward
// 108 -> 104 us; the forward, bound by its stores, unchanged at 50.)
constexpr int kMaxHalf = 256;
template <int TD, int EPL>
struct RopeTable {
  float* cos;  // this wave's [kMaxHalf], then sin
  float invf[kMaxHalf / 64];
  __device__ __forceinline__ RopeTable(const RopeParams& P, float* lds, int lane, int half)
      : cos(lds) {
#pragma unroll
    for (int k = 0; k < kMaxHalf / 64; ++k)
      invf[k] = lane + 64 * k < half ? rnd<TD>(P.inv_freq[lane + 64 * k]) : 0.f;
  }
  // Position p's cos and sin (times `sign`) of columns col .. col + EPL - 1.
  __device__ __forceinline__ void at(int p, int sign, int lane, int half, int col,
                                     float (&c)[EPL], float (&s)[EPL]) const {
    const float pos = rnd<TD>((float)p);
    float* sin = cos + kMaxHalf;
#pragma unroll
    for (int k = 0; k < kMaxHalf / 64; ++k) {
      if (lane + 64 * k < half) {
        float sv, cv;
        sincosf(rnd<TD>(mul_rn(pos, invf[k])), &sv, &cv);  // the accurate library routine
        cos[lane + 64 * k] = rnd<TD>(cv);
        sin[lane + 64 * k] = sign * rnd<TD>(sv);
      }
    }
    // (one wave's own LDS: its reads follow its writes in order)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int e = 0; e < EPL; ++e) c[e] = cos[col + e], s[e] = sin[col + e];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
};

// Sum over the lpr lanes of a row (lanes lrow * lpr .. + lpr - 1); every
// lane of the wave takes part.
__device__ __forceinline__ float row_sum(float v, int lpr) {
  for (int m = 1; m < lpr; m <<= 1) v += __shfl_xor(v, m);
  return v;
}

// Forward.  NORM: q and / or k rows are RMS-normalised first (weights wq /
// wk; a null weight leaves those rows unnormalised), and the chain then runs
// in fp32 with one rounding at the store.
template <int DT, bool NORM>
__global__ __launch_bounds__(64 * kRopeWaves) void rope_kernel(const RopeParams P) {
  using Ch = Chunk<DT>;
  constexpr int EPL = Ch::EPL;
  constexpr int ES = DT == kRopeF32 ? 4 : 2;
  constexpr int TD = NORM ? kRopeF32 : DT;  // type of the table and of the rotation
  const int wv = uni(threadIdx.x >> 6);
  RopeLanes<DT> L(P, blockIdx.x * kRopeWaves + wv);
  // (no early return before the weights' barrier: a wave past the last
  // token runs no token iteration below)
  const int col = L.col, half = L.half;

  __shared__ __attribute__((aligned(16))) float table[kRopeWaves][2 * kMaxHalf];
  const RopeTable<TD, EPL> tab(P, table[wv], L.lane, half);
  // the norm weights (q, k), in LDS rather than in every lane's registers
  __shared__ float wsh[NORM ? 2 : 1][NORM ? 512 : 1];
  if constexpr (NORM) {
    for (int d = threadIdx.x; d < P.D; d += 64 * kRopeWaves) {
      wsh[0][d] = P.wq ? P.wq[d] : 1.f;
      wsh[1][d] = P.wk ? P.wk[d] : 1.f;
    }
    __syncthreads();
  }
  const float inv_d = 1.f / (float)P.D;

  for (int i = 0; i < P.tpw; ++i) {
    const int t = L.t0 + i;
    if (t >= P.T) break;
    const int p = L.position(P, t);
    const bool inside = p >= 0;
    float c[EPL], s[EPL];
    if (inside) tab.at(p, P.sign, L.lane, half, col, c, s);
    // Four row passes at a time: every load first, then the arithmetic and
    // the stores.  (With the norm every lane makes the same passes: the row
    // sums cross lanes.)
    for (int r0 = L.lrow; (NORM ? r0 - L.lrow : r0) < L.nrows; r0 += kRopePasses * L.rpw) {
      Raw<DT> x1[kRopePasses], x2[kRopePasses];
      float rs[kRopePasses];  // the row's RMS factor (0: no norm)
      char* dst[kRopePasses];
      bool copy[kRopePasses], isq[kRopePasses];
#pragma unroll
      for (int j = 0; j < kRopePasses; ++j) {
        const int r = r0 + j * L.rpw;
        dst[j] = nullptr;
        isq[j] = r < P.Hq;
        if (r < L.nrows) {
          const char* src = L.in_row(P, P.q, P.k, P.q_ss, P.q_sh, P.k_ss, P.k_sh, t, r);
          dst[j] = (char*)L.in_row(P, P.q_out, P.k_out, P.qo_ss, P.qo_sh, P.ko_ss, P.ko_sh, t, r);
          copy[j] = dst[j] != src;
          x1[j].load(src + col * ES);
          x2[j].load(src + (half + col) * ES);
        }
      }
#pragma unroll
      for (int j = 0; j < kRopePasses; ++j) rs[j] = 0.f;
      if constexpr (NORM) {
        if (inside) {
          // RMS of each row (every lane joins the cross-lane sums)
#pragma unroll
          for (int j = 0; j < kRopePasses; ++j) {
            float ss = 0.f;
            if (dst[j]) {
#pragma unroll
              for (int e = 0; e < EPL; ++e) {
                const float a = x1[j].get(e), b2 = x2[j].get(e);
                ss += a * a + b2 * b2;
              }
            }
            ss = row_sum(ss, L.lpr);
            const bool has_w = isq[j] ? P.wq != nullptr : P.wk != nullptr;
            if (dst[j] && has_w) rs[j] = rsqrtf(ss * inv_d + P.eps);
          }
        }
      }
#pragma unroll
      for (int j = 0; j < kRopePasses; ++j) {
        if (!dst[j]) continue;
        if (inside) {
          Ch y1, y2;
#pragma unroll
          for (int e = 0; e < EPL; ++e) {
            float a = x1[j].get(e), b2 = x2[j].get(e);
            if (NORM && rs[j] != 0.f) {  // x r w, as (x r) w
              const float* w = wsh[isq[j] ? 0 : 1];
              a = a * rs[j] * w[col + e];
              b2 = b2 * rs[j] * w[half + col + e];
            }
            y1.v[e] = rnd<TD>(add_rn(rnd<TD>(mul_rn(a, c[e])), rnd<TD>(mul_rn(-b2, s[e]))));
            y2.v[e] = rnd<TD>(add_rn(rnd<TD>(mul_rn(b2, c[e])), rnd<TD>(mul_rn(a, s[e]))));
          }
          y1.store(dst[j] + col * ES);
          y2.store(dst[j] + (half + col) * ES);
        } else if (copy[j]) {  // outside every sequence: unchanged
          x1[j].store(dst[j] + col * ES);
          x2[j].store(dst[j] + (half + col) * ES);
        }
      }
    }
  }
}

// Backward of the normalised rotation (fp32 chain, as the forward with a
// norm): g' = R(-angle) dy, then for rows with a weight
//     dx = r (w g') - x r^3 <x, w g'> / D,     dw += x r g'
// (r = rsqrt(mean(x^2) + eps)); rows without one get dx = g'; tokens
// outside every sequence pass dy through.  Each workgroup writes its dw
// partial sums (fixed order) to part[2][gridDim.x][D].
template <int DT>
__global__ __launch_bounds__(64 * kRopeWaves, kBwdOcc) void rope_norm_bwd_kernel(const RopeParams P) {
  using Ch = Chunk<DT>;
  constexpr int EPL = Ch::EPL;
  constexpr int ES = DT == kRopeF32 ? 4 : 2;
  constexpr int NP = kBwdPasses<DT>;
  __shared__ __attribute__((aligned(16))) float red[2][kRopeWaves][512];
  __shared__ __attribute__((aligned(16))) float table[kRopeWaves][2 * kMaxHalf];
  __shared__ __attribute__((aligned(16))) float wsh[2][512];
  const int wv = uni(threadIdx.x >> 6);
  RopeLanes<DT> L(P, blockIdx.x * kRopeWaves + wv);
  const int col = L.col, half = L.half, lane = L.lane;
  const RopeTable<kRopeF32, EPL> tab(P, table[wv], lane, half);
  for (int d = threadIdx.x; d < P.D; d += 64 * kRopeWaves) {
    wsh[0][d] = P.wq ? P.wq[d] : 1.f;
    wsh[1][d] = P.wk ? P.wk[d] : 1.f;
  }
  __syncthreads();
  float dw1[2][EPL], dw2[2][EPL];  // dw partials of this lane's columns (q, k)
#pragma unroll
  for (int e = 0; e < EPL; ++e) dw1[0][e] = dw2[0][e] = dw1[1][e] = dw2[1][e] = 0.f;
  const float inv_d = 1.f / (float)P.D;

  for (int i = 0; i < P.tpw && L.t0 < P.T; ++i) {
    const int t = L.t0 + i;
    if (t >= P.T) break;
    const int p = L.position(P, t);
    const bool inside = p >= 0;
    float c[EPL], s[EPL];
    if (inside) tab.at(p, P.sign, lane, half, col, c, s);
    // Up to two row passes at once: slot j takes row `r` of side `side`
    // (0: q, 1: k), a compile-time one: its weights and pointers.
    auto passes = [&](auto n_, auto side0_, auto side1_, int row0, int row1) {
      constexpr int N = decltype(n_)::value;
      // every load first, as raw words
      Raw<DT> x1[N], x2[N], g1[N], g2[N];
      static_for<N>([&](auto j_) {
        constexpr int j = decltype(j_)::value;
        constexpr int side = j ? decltype(side1_)::value : decltype(side0_)::value;
        const int r = j ? row1 : row0;
        x1[j].w = x2[j].w = g1[j].w = g2[j].w = u32x4{0u, 0u, 0u, 0u};
        if (r < (side ? P.Hk : P.Hq)) {
          const char* xs = (const char*)(side ? P.k : P.q) + (int64_t)t * (side ? P.k_ss : P.q_ss) * ES;
          const char* gs = (const char*)(side ? P.gk : P.gq) + (int64_t)t * (side ? P.gk_ss : P.gq_ss) * ES;
          const char* x = xs + r * ((side ? P.k_sh : P.q_sh) * ES);
          const char* g = gs + r * ((side ? P.gk_sh : P.gq_sh) * ES);
          x1[j].load(x + col * ES);
          x2[j].load(x + (half + col) * ES);
          g1[j].load(g + col * ES);
          g2[j].load(g + (half + col) * ES);
        }
      });
      static_for<N>([&](auto j_) {
        constexpr int j = decltype(j_)::value;
        constexpr int side = j ? decltype(side1_)::value : decltype(side0_)::value;
        const int r = j ? row1 : row0;
        const bool live = r < (side ? P.Hk : P.Hq);
        char* os = (char*)(side ? P.k_out : P.q_out) + (int64_t)t * (side ? P.ko_ss : P.qo_ss) * ES;
        const int64_t oh = (side ? P.ko_sh : P.qo_sh) * ES;
        if (!inside) {  // (the same for every lane)
          if (live) {
            g1[j].store(os + r * oh + col * ES);
            g2[j].store(os + r * oh + (half + col) * ES);
          }
          return;
        }
        // g' = R(-angle) dy (the transpose of the forward rotation)
        Ch y1, y2;
        float ss = 0.f, tw = 0.f;
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
          const float a = g1[j].get(e), b = g2[j].get(e);
          const float u = x1[j].get(e), v = x2[j].get(e);
          y1.v[e] = add_rn(mul_rn(a, c[e]), mul_rn(b, s[e]));
          y2.v[e] = add_rn(mul_rn(b, c[e]), mul_rn(-a, s[e]));
          ss += u * u + v * v;
          tw += u * wsh[side][col + e] * y1.v[e] + v * wsh[side][half + col + e] * y2.v[e];
        }
        // (a lane past the rows holds zeros; every lane joins the sums)
        ss = row_sum(ss, L.lpr);
        tw = row_sum(tw, L.lpr);
        // (fp16: the products below stay behind the sums.  Begun ahead of
        // them, they spilled 9 registers: 16384 tokens, d128 91.0 -> 90.1
        // us, 6000 35.2 -> 34.5, 3000 26.5 -> 26.8.  In bf16 the order
        // costs 1 to 3%.)
        if constexpr (DT == kRopeF16) asm volatile("" : "+v"(ss));
        if ((side ? P.wk : P.wq) != nullptr) {
          const float rr = rsqrtf(ss * inv_d + P.eps);
          const float k3 = rr * rr * rr * tw * inv_d;
          if (live) {
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
              const float u = x1[j].get(e), v = x2[j].get(e);
              dw1[side][e] += u * rr * y1.v[e];
              dw2[side][e] += v * rr * y2.v[e];
              y1.v[e] = rr * wsh[side][col + e] * y1.v[e] - u * k3;
              y2.v[e] = rr * wsh[side][half + col + e] * y2.v[e] - v * k3;
            }
          }
        }
        if (live) {
          y1.store(os + r * oh + col * ES);
          y2.store(os + r * oh + (half + col) * ES);
        }
      });
    };
    constexpr std::integral_constant<int, NP> np{};
    constexpr std::integral_constant<int, 0> q_{};
    constexpr std::integral_constant<int, 1> k_{};
    const int q0 = L.lrow;
    bool together = false;
    if constexpr (NP == 2) together = max(P.Hq, P.Hk) <= L.rpw;
    if (together) {
      // A pass has room for all of a side's rows: both sides' together, so
      // that the token waits for its loads once (fp32, 40000 tokens: d64 1/1
      // heads 55 us, one after the other 70; d128 4/2 89, 105).  Not with
      // more rows: d64 16/4 at 15000 tokens 49.9, one after the other 48.4.
      if constexpr (NP == 2) passes(np, q_, k_, q0, q0);
    } else {
      for (int r = q0; r - q0 < P.Hq; r += NP * L.rpw) passes(np, q_, q_, r, r + L.rpw);
      for (int r = q0; r - q0 < P.Hk; r += NP * L.rpw) passes(np, k_, k_, r, r + L.rpw);
    }
  }

  // dw partials: lanes sharing columns (lane % lpr), then the waves, in a
  // fixed order.
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    for (int m = L.lpr; m < 64; m <<= 1) {
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        dw1[side][e] += __shfl_xor(dw1[side][e], m);
        dw2[side][e] += __shfl_xor(dw2[side][e], m);
      }
    }
  }
  if (lane < L.lpr) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        red[side][wv][col + e] = dw1[side][e];
        red[side][wv][half + col + e] = dw2[side][e];
      }
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < 2 * P.D; d += 64 * kRopeWaves) {
    const int which = d / P.D, dd = d - which * P.D;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < kRopeWaves; ++w) v += red[which][w][dd];
    P.part[((int64_t)which * gridDim.x + blockIdx.x) * P.D + dd] = v;
  }
}

// dw = sum over the workgroups' partials, in a fixed order: workgroup x
// takes 64 of the 2 D columns (lane = column); its 16 waves sum interleaved
// rows of partials (coalesced 256-byte rows), then wave 0 adds the 16 sums.
__global__ __launch_bounds__(1024) void rope_dw_reduce_kernel(const RopeParams P, int nblocks) {
  __shared__ float acc[16][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int d = blockIdx.x * 64 + lane;  // in [0, 2 D)
  const bool ok = d < 2 * P.D;
  const int which = ok ? d / P.D : 0, dd = ok ? d - which * P.D : 0;
  const float* src = P.part + (int64_t)which * nblocks * P.D + dd;
  float v = 0.f;
  if (ok) {
    int b = wv;
    for (; b + 7 * 16 < nblocks; b += 8 * 16) {  // eight loads in flight
      float t[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) t[u] = src[(int64_t)(b + 16 * u) * P.D];
#pragma unroll
      for (int u = 0; u < 8; ++u) v += t[u];
    }
    for (; b < nblocks; b += 16) v += src[(int64_t)b * P.D];
  }
  acc[wv][lane] = v;
  __syncthreads();
  if (wv == 0 && ok) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < 16; ++w) s += acc[w][lane];
    float* out = which == 0 ? P.dwq : P.dwk;
    if (out) out[dd] = s;
  }
}

}  // namespace

// Consecutive tokens per wave.  A wave's tokens are one chain of latencies
// and share its start (and, in the norm backward, its dw partials): few of
// them while the waves leave the chip with room, four once they fill it.
// us with 1 / 2 / 4 tokens (bf16, d = 128, 32 heads), norm + RoPE forward: 400
// tokens x 16 heads 7.5 / 9.1 / 15.3, 4000 tokens 15.7 / 19.6 / 26.3, 16384
// 53.8 / 52.9 / 49.5; norm backward 12.3 / 13.6 / 18.9, 28.9 / 26.8 / 34.5,
// 94.7 / 91.9 / 89.0 (fp32, 6000 tokens: forward 37 / 35 / 46, backward 59 /
// 57 / 66).
static int fwd_tokens_per_wave(int T) { return T <= 4096 ? 1 : T <= 12288 ? 2 : 4; }
static int bwd_tokens_per_wave(int T) { return T <= 1024 ? 1 : T <= 12288 ? 2 : 4; }
static int blocks_of(int T, int tpw) {
  return (int)(((int64_t)T + kRopeWaves * tpw - 1) / (kRopeWaves * tpw));
}

int rope_bwd_blocks(int T) { return blocks_of(T, bwd_tokens_per_wave(T)); }

namespace {
template <int DT>
void launch_rope_dt(const RopeParams& P, dim3 grid, dim3 block, hipStream_t s) {
  if (P.wq || P.wk)
    hipLaunchKernelGGL((rope_kernel<DT, true>), grid, block, 0, s, P);
  else
    hipLaunchKernelGGL((rope_kernel<DT, false>), grid, block, 0, s, P);
}
}  // namespace

hipError_t launch_rope(const RopeParams& args, hipStream_t s) {
  RopeParams P = args;
  if (P.T <= 0 || P.Hq + P.Hk <= 0) return hipSuccess;
  P.tpw = fwd_tokens_per_wave(P.T);
  const dim3 grid(blocks_of(P.T, P.tpw)), block(64 * kRopeWaves);
  switch (P.dtype) {
    case kRopeBF16: launch_rope_dt<kRopeBF16>(P, grid, block, s); break;
    case kRopeF16: launch_rope_dt<kRopeF16>(P, grid, block, s); break;
    case kRopeF32: launch_rope_dt<kRopeF32>(P, grid, block, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_rope_norm_bwd(const RopeParams& args, hipStream_t s) {
  RopeParams P = args;
  if (P.T <= 0 || P.Hq + P.Hk <= 0) return hipSuccess;
  P.tpw = bwd_tokens_per_wave(P.T);
  const int nb = rope_bwd_blocks(P.T);
  const dim3 grid(nb), block(64 * kRopeWaves);
  switch (P.dtype) {
    case kRopeBF16: hipLaunchKernelGGL(rope_norm_bwd_kernel<kRopeBF16>, grid, block, 0, s, P); break;
    case kRopeF16: hipLaunchKernelGGL(rope_norm_bwd_kernel<kRopeF16>, grid, block, 0, s, P); break;
    case kRopeF32: hipLaunchKernelGGL(rope_norm_bwd_kernel<kRopeF32>, grid, block, 0, s, P); break;
    default: return hipErrorInvalidValue;
  }
  if (hipGetLastError() != hipSuccess) return hipErrorLaunchFailure;
  hipLaunchKernelGGL(rope_dw_reduce_kernel, dim3((2 * P.D + 63) / 64), dim3(1024), 0, s, P, nb);
  return hipGetLastError();
}

}  // namespace fna2
