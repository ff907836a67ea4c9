// fna2_bwd.hip — FlashNaylisAttention-2 backward for gfx950.
//
// This file holds the backward's small kernels; dQ/dRq (which also forms
// delta = sum_d O dO, the reference's _fna2_bwd_preprocess[_varlen]_kernel,
// FNA2/flash_naylis_attn.py:356-382, :900-921) and dK/dV/dRk are in
// fna2_bwd_dq.hip and fna2_bwd_dkdv.hip.
//   zero rows: varlen tokens outside [cu[0], cu[N]) get zero gradients;
//   d_gs:      fixed-order sum of the dQ kernel's per-wave partials;
//   dK/dV:     fixed-order sum of the fp32 partials of items in chunks.
// Together: no atomics anywhere, bitwise deterministic, no pre-zeroing.
//
// Math, per head, with Qa = [a Q | b Rq], Ka = [K | Rk], S = c Qa Ka^T:
//   P = exp(S - LSE),  dP = dO V^T,  dS = P (dP - delta),  dA = c dS
//   dV = P^T dO,  [dK | dRk] = dA^T Qa,  [dQ/a | dRq/b] = dA Ka,
//   d_gs = sum_i <Rq_i, (dS Rk)_i> = (1/c) sum_i <Rq_i, (dA Rk)_i>.
#include "fna2_kernels.h"

namespace fna2 {

namespace {

// d_gs when the dK/dV kernel does not run (no keys): one wave per head.
__global__ __launch_bounds__(64) void dgs_reduce_kernel(const BwdParams P) {
  reduce_dgs_waves(P, blockIdx.x, gridDim.x, threadIdx.x);
}

// dK, dV and dRk of the key tiles whose items ran in chunks: one wave per
// 32 x 32 tile of a key slice sums the chunks' fp32 tiles in chunk order (the
// registers' own layout, 16 bytes per lane: every access is a whole line),
// scales and rounds once, and stores 8 consecutive features per lane.
template <bool F16>
__global__ __launch_bounds__(256) void kv_reduce_kernel(const BwdParams P, int bn, int nrb) {
  const Problem& p = P.p;
  const int lane = threadIdx.x & 63;
  const int l32 = lane & 31, hl = lane >> 5;
  const int ndb = p.D / 32, slices = bn / 32;
  const int per_kv = 2 * ndb, per_item = per_kv + p.group * nrb;  // tiles per slice
  int u = uni((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  const int t = u % per_item;
  u /= per_item;
  const int sl = u % slices;
  u /= slices;
  const int item = u, tix = item / p.H_KV, kvh = item - tix * p.H_KV;
  const int n_tiles =
      P.tiles_k ? min(uni(*const_space(P.n_tiles_k)), P.k_tiles) : p.nseq * cdiv(p.sk, bn);
  if (tix >= min(n_tiles, P.split_tiles)) return;
  int b, kt;
  SeqExt e;
  if (P.tiles_k) {
    tile_decode(P.tiles_k, tix, b, kt, e);
  } else {
    b = tix % p.nseq;
    kt = tix / p.nseq;
    e = seq_ext_uniform(p, b);
  }
  const int nqb = max(cdiv(e.lq, kKvBM) - (p.causal ? kt * bn / kKvBM : 0), 0);
  const KvChunks k = kv_chunks(p.group * nqb, P.split_log2);
  if (k.n <= 1) return;  // written by the dK/dV kernel
  int c0 = 0, c1 = k.n;  // chunks to sum
  int64_t step, at;      // floats between chunks' tiles; the first one
  float scale = 1.f;
  TView out;
  int head, feat;
  if (t < per_kv) {
    step = (int64_t)slices * per_kv * 1024;
    at = ((int64_t)item << P.split_log2) * step + ((int64_t)sl * per_kv + t) * 1024;
    const bool dk = t < ndb;
    if (dk) scale = p.qa * p.c;
    out = dk ? P.dk : P.dv;
    head = kvh;
    feat = 32 * (dk ? t : t - ndb);
  } else {
    const int hi = (t - per_kv) / nrb, f = (t - per_kv) - hi * nrb;
    head = kvh * p.group + hi;
    if (head >= p.H_G || nqb <= 0) return;
    c0 = hi * nqb / k.len;
    c1 = ((hi + 1) * nqb - 1) / k.len + 1;
    if (c1 - c0 <= 1) return;  // a whole head: written by the dK/dV kernel
    step = (int64_t)slices * nrb * 1024;
    at = ((int64_t)item * drk_slots(p.group, P.split_log2) + hi + c0) * step +
         ((int64_t)sl * nrb + f) * 1024;
    scale = *const_space(P.gs + head);
    out = P.drk;
    feat = 32 * f;
  }
  const float* src = (t < per_kv ? P.kv_part : P.drk_part) + at + lane * 4;
  f32x4_t acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = *(const f32x4_t*)(src + i * 256);
#pragma unroll 4
  for (int c = c0 + 1; c < c1; ++c) {
    src += step;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] += *(const f32x4_t*)(src + i * 256);
  }
  // register v of the 32 x 32 tile is feature 8 (v / 4) + 4 hl + v % 4 of
  // key l32: one exchange between the lane halves per pair of groups
  const int key = kt * bn + sl * 32 + l32;
  const int width = t < per_kv ? p.D : p.R;
  uint16_t* row = seq_base<uint16_t>(out, p, b, e.k0, head) + (int64_t)key * out.ss + feat + 8 * hl;
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    auto pk = [&](int g, int j) {
      const float x = scale * acc[g][j], y = scale * acc[g][j + 1];
      return (F16 && t < per_kv) ? pack_e<F16>(x, y) : pack_bf16(x, y);
    };
    const auto lo = __builtin_amdgcn_permlane32_swap(pk(2 * w, 0), pk(2 * w + 1, 0), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(pk(2 * w, 2), pk(2 * w + 1, 2), false, false);
    if (key < e.lk && feat + 16 * w + 8 * hl < width)
      st16(row + 16 * w, u32x4{lo[0], hi[0], lo[1], hi[1]});
  }
}

}  // namespace

hipError_t launch_bwd_kv_reduce(const BwdParams& P, int rpl, hipStream_t s) {
  const int bn = kv_bn(P.p.D, rpl), nrb = rpl / 32;
  const int64_t waves = (int64_t)P.split_tiles * P.p.H_KV * (bn / 32) *
                        (2 * (P.p.D / 32) + P.p.group * nrb);
  if (waves <= 0) return hipSuccess;
  if ((waves + 3) / 4 > INT32_MAX / 4) return hipErrorInvalidValue;
  const dim3 grid((uint32_t)((waves + 3) / 4));
  if (P.p.f16)
    hipLaunchKernelGGL(kv_reduce_kernel<true>, grid, dim3(256), 0, s, P, bn, nrb);
  else
    hipLaunchKernelGGL(kv_reduce_kernel<false>, grid, dim3(256), 0, s, P, bn, nrb);
  return hipGetLastError();
}

hipError_t launch_bwd_dgs(const BwdParams& P, hipStream_t s) {
  if (P.p.H_G <= 0) return hipSuccess;
  hipLaunchKernelGGL(dgs_reduce_kernel, dim3(P.p.H_G), dim3(64), 0, s, P);
  return hipGetLastError();
}

}  // namespace fna2
