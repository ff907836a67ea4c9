// fna2_capi.cpp — the extern "C" boundary: validation, workspace layout and
// kernel dispatch.  Host code only; every GPU launch goes through the
// launch_* wrappers of the .hip files.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>

#include "fna2.h"
#include "fna2_kernels.h"
#include "fna2_sched.h"

namespace {

using fna2::kDqBM;
using fna2::kDqBN;
using fna2::kFwdBM;
using fna2::kFwdBN;
using fna2::kKvBM;

constexpr size_t kAlign = 256;
constexpr int64_t kMaxGrid = (int64_t)1 << 24;  // workgroups per launch

size_t align_up(size_t x) { return (x + kAlign - 1) / kAlign * kAlign; }

int64_t cdiv64(int64_t a, int64_t b) { return (a + b - 1) / b; }

bool aligned(const void* p, size_t a) { return ((uintptr_t)p % a) == 0; }

// Rows of the query / key side (dense: B * S, varlen: tokens).
int64_t rows_q(const fna2_problem& p) {
  return p.varlen ? (int64_t)p.total_q : (int64_t)p.batch * p.seqlen_q;
}
int64_t rows_k(const fna2_problem& p) {
  return p.varlen ? (int64_t)p.total_k : (int64_t)p.batch * p.seqlen_k;
}

int check_problem(const fna2_problem& p) {
  if (p.dtype != FNA2_BF16 && p.dtype != FNA2_F16) return FNA2_E_DTYPE;
  if (p.head_dim != 64 && p.head_dim != 128) return FNA2_E_HEAD_DIM;
  if (p.heads <= 0 || p.heads_kv <= 0 || p.heads % p.heads_kv != 0) return FNA2_E_HEADS;
  if (p.heads_graph < 0 || p.heads_graph > p.heads) return FNA2_E_HEADS;
  if (p.heads_graph > 0 && (p.rank < 8 || p.rank > 64 || p.rank % 8 != 0)) return FNA2_E_RANK;
  if (p.batch < 0) return FNA2_E_SHAPE;
  if (p.varlen) {
    if (p.total_q < 0 || p.total_k < 0) return FNA2_E_SHAPE;
    if (p.batch > 0 && (!p.cu_seqlens_q || !p.cu_seqlens_k)) return FNA2_E_SEQLENS;
  } else {
    if (p.seqlen_q < 0 || p.seqlen_k < 0) return FNA2_E_SHAPE;
  }
  if (!std::isfinite(p.softmax_scale)) return FNA2_E_SCALE;
  return FNA2_OK;
}

// feat: elements per row (16-byte vectors) or 0 for an fp32 scalar view.
int check_view(const fna2_tensor& t, const fna2_problem& p, bool required, bool vec,
               size_t esize) {
  if (!required) return FNA2_OK;
  if (!t.ptr) return FNA2_E_NULL;
  const size_t a = vec ? 16 : esize;
  if (!aligned(t.ptr, a)) return FNA2_E_STRIDE;
  const int64_t ss = t.stride_s, sh = t.stride_h, sb = p.varlen ? 0 : t.stride_b;
  const int64_t unit = vec ? (int64_t)(16 / esize) : 1;
  if (ss % unit || sh % unit || sb % unit) return FNA2_E_STRIDE;
  return FNA2_OK;
}

#define FNA2_TRY(x)              \
  do {                           \
    int _s = (x);                \
    if (_s != FNA2_OK) return _s; \
  } while (0)

struct Grids {
  int64_t fwd_bound = 0;  // varlen tile-list capacity
  int64_t fwd_grid = 0;
  int64_t dq_bound = 0, dq_grid = 0;
  int64_t kv_bound = 0, kv_grid = 0;
  int64_t kv_tiles = 0;   // key tiles (varlen: bound)
  int64_t q_tiles = 0;    // dQ query tiles (varlen: bound)
};

// Keys per dK/dV item of the problem.
int kv_tile(const fna2_problem& p) {
  return fna2::kv_bn(p.head_dim, fna2::padded_rank32(p.heads_graph, p.rank));
}

Grids grids(const fna2_problem& p) {
  Grids g;
  if (p.batch <= 0) return g;
  const int kbn = kv_tile(p);
  if (p.varlen) {
    g.fwd_bound = fna2::tile_bound(p.total_q, p.batch, kFwdBM);
    g.fwd_grid = g.fwd_bound * p.heads;
    g.dq_bound = fna2::tile_bound(p.total_q, p.batch, kDqBM);
    g.dq_grid = g.dq_bound * p.heads;
    g.kv_bound = fna2::tile_bound(p.total_k, p.batch, kbn);
    g.kv_grid = g.kv_bound * p.heads_kv;
    g.kv_tiles = g.kv_bound;
    g.q_tiles = g.dq_bound;
  } else {
    g.fwd_grid = (int64_t)p.batch * cdiv64(p.seqlen_q, kFwdBM) * p.heads;
    g.dq_grid = (int64_t)p.batch * cdiv64(p.seqlen_q, kDqBM) * p.heads;
    g.kv_grid = (int64_t)p.batch * cdiv64(p.seqlen_k, kbn) * p.heads_kv;
    g.kv_tiles = (int64_t)p.batch * cdiv64(p.seqlen_k, kbn);
    g.q_tiles = (int64_t)p.batch * cdiv64(p.seqlen_q, kDqBM);
  }
  return g;
}

int check_grids(const fna2_problem& p) {
  const Grids g = grids(p);
  if (g.fwd_grid > kMaxGrid || g.dq_grid > kMaxGrid || g.kv_grid > kMaxGrid) return FNA2_E_SHAPE;
  if (rows_q(p) > INT32_MAX || rows_k(p) > INT32_MAX) return FNA2_E_SHAPE;
  return FNA2_OK;
}

// Workspace layouts (byte offsets), all 256-byte aligned.
struct FwdWs {
  size_t tiles = 0, count = 0, bytes = 0;
};
FwdWs fwd_ws(const fna2_problem& p) {
  FwdWs w;
  const Grids g = grids(p);
  if (p.varlen && g.fwd_bound > 0) {
    w.tiles = 0;
    w.count = align_up(sizeof(fna2::TileRec) * g.fwd_bound);
    w.bytes = w.count + kAlign;
  }
  return w;
}

struct BwdWs {
  size_t tiles_q = 0, count_q = 0, tiles_k = 0, count_k = 0, partial = 0, nlse = 0;
  size_t bytes = 0;
};
BwdWs bwd_ws(const fna2_problem& p) {
  BwdWs w;
  const Grids g = grids(p);
  size_t off = 0;
  if (p.varlen && g.dq_bound > 0) {
    w.tiles_q = off;
    off += align_up(sizeof(fna2::TileRec) * g.dq_bound);
    w.count_q = off;
    off += kAlign;
    w.tiles_k = off;
    off += align_up(sizeof(fna2::TileRec) * g.kv_bound);
    w.count_k = off;
    off += kAlign;
  }
  w.partial = off;
  // d_gs partials: [query tiles][4 waves][H_G]
  off += align_up(sizeof(float) * 4u * (size_t)(g.q_tiles > 0 ? g.q_tiles : 1) *
                  (size_t)(p.heads_graph > 0 ? p.heads_graph : 1));
  // -LSE log2(e), fp32 [H][rows_q] (per batch)
  w.nlse = off;
  off += align_up((size_t)rows_q(p) * (size_t)p.heads * 4u);
  w.bytes = off;
  return w;
}

// Key groups of the forward's and dQ's kernels: with few query tiles, several
// groups of four waves share a tile's keys (one workgroup of 8 to 16 waves per
// tile and CU).  The tiles' longest key loop is then the kernel's time, and
// the groups cut it, for some 3 us of combining: `min_keys` keys at least in
// the longest tile.  Up to 256 tiles each has a CU to itself.  Up to 512 under
// the causal mask, whose short tiles make a second round: it pays as long as
// the long ones are few, `pairs` (sequence, head) pairs, each with one longest
// tile.  Measured in bf16 (fp16 within 2%), us without -> with key groups, H
// heads x S causal, nc: not:
//   forward d64 r16   5x8x768 15.8 -> 15.3, 16x2048 32 -> 25, 32x1531 27 -> 26,
//     32x2048 36 -> 35, 40x1024 19.8 -> 21.4, 10x8x768 17.9 -> 24.0; nc 5x8x768
//     15.3 -> 15.6, 32x1024 19.3 -> 17.6.  r0 32x2048 30.9 -> 31.9, 24x2048 29.2
//     -> 27.2; r64 32x2048 42 -> 40
//   forward d128 r32  8x512 17.5 -> 16.3, 32x1531 43 -> 36.5, 32x2048 58 -> 52,
//     37x1531 45.4 -> 45.5, 64x1024 34 -> 36; nc 5x8x768 23.8 -> 22.4, 16x2048
//     53 -> 45.  r0 and r64 the same within 3%
//   dQ d64 r16   32x1280 39 -> 33, 32x2048 58 -> 54, 48x1024 34 -> 36; nc 32x1024
//     32 -> 29
//   dQ d128 r32  34x1024 40 -> 38, 32x1531 55 -> 53.6, 32x2048 77.7 -> 78, 64x1024
//     47 -> 54; nc 16x1024 36.8 -> 36.6, 8x2048 62 -> 57.5, 32x1024 39.7 -> 41,
//     16x2048 67.8 -> 67.6; 768 keys: 0.7 to 2.5 us slower
// A varlen call counts its tiles by the tokens and half a tile per sequence.
// Its keys are what some sequence must have, the mean: max_seqlen_k is only a
// bound, often a loose one, and short packs in these kernels lose a half (10
// x 400, 8 heads: forward 20 -> 29 us).
constexpr int kSplitCUs = 256;  // (a fixed figure: the answer depends on the arguments alone)

// Tokens of a varlen pack's sequences, if they were of one length.
int64_t mean_len(int64_t total, int64_t hint, int64_t batch) {
  const int64_t mean = cdiv64(total, std::max<int64_t>(batch, 1));
  return hint > 0 ? std::min(hint, mean) : mean;
}

bool few_tiles(const fna2_problem& p, int64_t min_keys, int64_t pairs) {
  int64_t tiles, keys;
  if (p.varlen) {
    tiles = cdiv64(p.total_q, kFwdBM) + p.batch / 2;
    keys = mean_len(p.total_k, p.seqlen_k, p.batch);
  } else {
    tiles = (int64_t)p.batch * cdiv64(p.seqlen_q, kFwdBM);
    keys = p.causal ? std::min(p.seqlen_q, p.seqlen_k) : p.seqlen_k;
  }
  tiles *= p.heads;
  if (keys < min_keys) return false;
  return tiles <= kSplitCUs ||
         (p.causal && tiles <= 2 * kSplitCUs && tiles <= pairs * cdiv64(keys, kFwdBM));
}

int fwd_groups(const fna2_problem& p) {
  const bool wide = p.head_dim == 128;
  const int64_t min_keys = p.causal ? (wide ? 512 : 768) : (wide ? 768 : 1024);
  if (!few_tiles(p, min_keys, wide || p.heads_graph > 0 ? 32 : 24)) return 1;
  return fna2::fwd_key_groups(p.head_dim, fna2::padded_rank32(p.heads_graph, p.rank));
}

int dq_groups(const fna2_problem& p) {
  const bool wide = p.head_dim == 128;
  bool few = few_tiles(p, wide ? 1024 : 768, 32);
  if (wide && !p.causal && few) {  // (every tile is a longest one)
    const int64_t tiles =
        p.heads * (p.varlen ? cdiv64(p.total_q, kDqBM) + p.batch / 2
                            : (int64_t)p.batch * cdiv64(p.seqlen_q, kDqBM));
    few = tiles <= kSplitCUs / 2 || few_tiles(p, 2048, 32);
  }
  return few ? fna2::dq_key_groups(p.head_dim, fna2::padded_rank32(p.heads_graph, p.rank)) : 1;
}

// dK/dV items in chunks.  The persistent dK/dV kernel deals (key tile, KV
// head) items to the CUs; where these are fewer than the CUs, or one item is
// longer than a CU's share of the work, the time is the longest item's.
// Then the items of the first `tiles` tiles of the list (longest first) run
// in up to 2^log2 chunks of their (query head, query block) sequence, which
// write fp32 partials to the workspace for a reduction kernel.  The rule
// compares, in blocks (32 queries against a key tile), the longest chunk and
// a CU's share with what entering a chunk costs (kEnter) and the reduction
// (its launch and the partials written and read); without the causal mask all
// chunks are alike, so the CUs also go through them in whole rounds.  In
// varlen mode the host does not know the lengths, and max_seqlen is only a
// bound, often a loose one: chunks that the real items do not need cost up to
// their own time (32 x 128, 8/4 heads, d 64, max_seqlen 4096: backward 39 ->
// 75 us).  So the best split is taken for a pack of max_seqlen's sequences,
// of those that cost a pack of its mean length nothing: up to 1.1 times the
// whole items by this estimate, in 2 to 8 chunks (of 33 such packs measured
// none was slower; of 27 between 1.2 and 1.4, 12 were, and 16 chunks at 1.1).
// A max_seqlen that is the token count names no length, so whole items of it
// make no rounds that chunks would shorten ([8000, 900, 700, 617], H32/8 d128
// r64, not causal: 4.81 ms whole, 5.09 in halves; of 20 such packs 18 were 1
// to 13% slower in chunks; with a true or no max_seqlen 3 of 11).
//
// Measured (dK/dV and its reduction, us, whole items -> the rule's chunks):
// B2 H16/4 L1531 d128 fp16 238 -> 88 (chunks of 1/2: 138, 1/4: 86, 1/8: 96,
// 1/16: 120), B1 H8/4 L512 d64 51 -> 24, B1 H32/8 L1024 d128 158 -> 60, B1
// H8/4 L8192 d128 580 -> 355; packs of one long sequence, max_seqlen exact or
// not, the backward: [1191, 6 x ~117] H16/4 d128 233 -> 110, [7083, 3 x ~1150]
// H12/4 d64 not causal 1142 -> 833.  Where the rule keeps them whole: B1 H16
// L2048 d128 (256 items) 85 whole, 82 in halves, 104 in quarters; B1 H8 L128
// 15 against 18; B3 L3209 H12/4 d64 not causal (156 items) 350 whole, 408 in
// halves.
struct KvSplit {
  int log2 = 0;
  int64_t tiles = 0;
  size_t kv_part = 0, drk_part = 0, bytes = 0;  // offsets in the split's own region
};
constexpr int64_t kSplitMaxBytes = (int64_t)512 << 20;

KvSplit kv_split(const fna2_problem& p) {
  KvSplit best;
  const Grids g = grids(p);
  if (p.batch <= 0 || g.kv_grid <= 0) return best;
  const int bn = kv_tile(p);
  const int group = p.heads / p.heads_kv;
  const int64_t rpl = fna2::padded_rank32(p.heads_graph, p.rank);
  // The work as nseq sequences of lq x lk: items, blocks in all and of the
  // longest item.
  struct Work {
    int64_t kt = 0, items = 0, total = 0, longest = 0;
  };
  auto work = [&](int64_t lq, int64_t lk, int64_t nseq) {
    Work w;
    const int64_t qb = cdiv64(lq, kKvBM), lo = p.causal ? bn / kKvBM : 0;
    w.kt = cdiv64(lk, bn);
    // blocks of one sequence and head: sum over its key tiles of qb - lo t
    const int64_t seen = lo > 0 ? std::min<int64_t>(w.kt, cdiv64(qb, lo)) : w.kt;
    w.items = nseq * w.kt * p.heads_kv;
    w.total = nseq * p.heads * (seen * qb - lo * (seen * (seen - 1) / 2));
    w.longest = (int64_t)group * qb;
    return w;
  };
  constexpr double kEnter = 4, kLaunch = 5, kBytesPerBlock = 4e6;
  auto cost = [&](const Work& w, int log2, bool rounds) {
    const int64_t n = (int64_t)1 << log2;
    const int64_t len = std::max<int64_t>(cdiv64(w.longest, n), log2 ? fna2::kKvMinChunk : 1);
    const double chunks = std::min((double)w.items * n,
                                   std::max((double)w.total / fna2::kKvMinChunk, (double)w.items));
    double t = std::max(len + kEnter, (w.total + kEnter * chunks) / kSplitCUs);
    if (rounds)
      t = std::max(t, cdiv64(w.items * cdiv64(w.longest, len), kSplitCUs) * (len + kEnter));
    if (log2 > 0) t += kLaunch + chunks * bn * (2 * p.head_dim + rpl) * 8.0 / kBytesPerBlock;
    return t;
  };
  const int64_t lq = p.varlen ? mean_len(p.total_q, p.seqlen_q, p.batch) : p.seqlen_q;
  const int64_t lk = p.varlen ? mean_len(p.total_k, p.seqlen_k, p.batch) : p.seqlen_k;
  const Work even = work(lq, lk, p.batch);
  Work hinted = even;
  if (p.varlen && p.seqlen_q > lq && p.seqlen_k > lk) {
    const int64_t hk = std::min(p.seqlen_k, p.total_k);
    hinted = work(std::min(p.seqlen_q, p.total_q), hk, std::max<int64_t>(p.total_k / hk, 1));
  }
  if (even.total <= 0) return best;
  // (a whole item after the chunks is the last to end: in a pack of equal
  // lengths every tile is cut, in others the shortest may stay whole)
  const int64_t cut =
      std::min(g.kv_tiles, std::max(p.batch * even.kt, p.varlen ? cdiv64(p.total_k, bn) + 8 : 0));
  const bool alike = !p.causal;  // (`rounds`: see above)
  const bool told = alike && !(p.varlen && p.batch > 1 && p.seqlen_k >= p.total_k);
  double least = 0.9 * cost(hinted, 0, told);
  const double whole = cost(even, 0, alike);
  for (int log2 = 1; log2 <= 4; ++log2) {
    KvSplit s;
    s.log2 = log2;
    s.tiles = cut;
    const int64_t kv = (int64_t)p.heads_kv * ((int64_t)1 << log2) * bn * 2 * p.head_dim * 4;
    const int64_t dr = p.heads_graph > 0
                           ? (int64_t)p.heads_kv * fna2::drk_slots(group, log2) * bn * rpl * 4
                           : 0;
    s.tiles = std::min<int64_t>(s.tiles, kSplitMaxBytes / (kv + dr));
    if (s.tiles <= 0 || (s.tiles * p.heads_kv) << log2 > kMaxGrid) continue;
    s.drk_part = align_up((size_t)(s.tiles * kv));
    s.bytes = s.drk_part + align_up((size_t)(s.tiles * dr));
    if (cost(even, log2, alike) > (log2 < 4 && hinted.longest > even.longest ? 1.1 : 0.9) * whole) continue;
    const double t = cost(hinted, log2, alike);
    if (t < least) {
      least = t;
      best = s;
    }
  }
  return best;
}

// Plan (varlen): the query-tile list the forward and the dQ kernel share
// (the same tile shape) and the dK/dV key-tile list.
static_assert(kFwdBM == kDqBM && kFwdBN == kDqBN, "the forward and dQ share their tile list");
struct PlanLayout {
  size_t tiles_q = 0, count_q = 0, tiles_k = 0, count_k = 0, bytes = 0;
};
PlanLayout plan_layout(const fna2_problem& p) {
  PlanLayout L;
  if (!p.varlen || p.batch <= 0) return L;
  const Grids g = grids(p);
  size_t off = 0;
  L.tiles_q = off;
  off += align_up(sizeof(fna2::TileRec) * (size_t)g.fwd_bound);
  L.count_q = off;
  off += kAlign;
  L.tiles_k = off;
  off += align_up(sizeof(fna2::TileRec) * (size_t)g.kv_bound);
  L.count_k = off;
  off += kAlign;
  L.bytes = off;
  return L;
}

bool use_plan(const void* plan, const fna2_problem& p) { return plan && p.varlen && p.batch > 0; }

// Plans that fna2_fwd filled, by address, with the problem each was built
// for.  The tile records carry extents clamped to that problem's token
// counts and lists sized by its sequence count, so a backward may only read
// a plan built for the same sequences: fna2_bwd uses a plan found here with
// a matching key, and otherwise builds its own lists (as without a plan).
// A small ring: an address reused by a later forward is re-registered.  The
// key-tile size (head_dim and padded rank pick it) shapes the key list, so
// it is part of the key: a plan built for another tile size is not used.
uint64_t plan_key(const fna2_problem& p) {
  const uint64_t f[] = {(uint64_t)p.batch,          (uint64_t)p.total_q,
                        (uint64_t)p.total_k,        (uint64_t)p.causal,
                        (uint64_t)(uintptr_t)p.cu_seqlens_q,
                        (uint64_t)(uintptr_t)p.cu_seqlens_k,
                        (uint64_t)kv_tile(p)};
  uint64_t h = 1469598103934665603ull;  // FNV-1a over the words
  for (uint64_t w : f) {
    for (int i = 0; i < 8; ++i) {
      h ^= (w >> (8 * i)) & 0xffu;
      h *= 1099511628211ull;
    }
  }
  return h;
}
struct PlanEntry {
  const void* plan;
  uint64_t key;
};
constexpr int kPlanSlots = 256;
std::mutex g_plan_mu;
PlanEntry g_plans[kPlanSlots];
int g_plan_next = 0;

void plan_register(const void* plan, const fna2_problem& p) {
  std::lock_guard<std::mutex> lk(g_plan_mu);
  const uint64_t key = plan_key(p);
  for (PlanEntry& e : g_plans) {
    if (e.plan == plan) {
      e.key = key;
      return;
    }
  }
  g_plans[g_plan_next] = PlanEntry{plan, key};
  g_plan_next = (g_plan_next + 1) % kPlanSlots;
}

bool plan_filled_for(const void* plan, const fna2_problem& p) {
  std::lock_guard<std::mutex> lk(g_plan_mu);
  const uint64_t key = plan_key(p);
  for (const PlanEntry& e : g_plans)
    if (e.plan == plan) return e.key == key;
  return false;
}

fna2::Problem make_problem(const fna2_problem& p) {
  fna2::Problem P;
  std::memset(&P, 0, sizeof(P));
  P.varlen = p.varlen;
  P.nseq = p.batch;
  P.sq = p.varlen ? 0 : p.seqlen_q;
  P.sk = p.varlen ? 0 : p.seqlen_k;
  P.total_q = p.varlen ? p.total_q : 0;
  P.total_k = p.varlen ? p.total_k : 0;
  P.H = p.heads;
  P.H_KV = p.heads_kv;
  P.H_G = p.heads_graph;
  P.D = p.head_dim;
  P.R = p.heads_graph > 0 ? p.rank : 0;
  P.causal = p.causal ? 1 : 0;
  P.f16 = p.dtype == FNA2_F16 ? 1 : 0;
  P.group = p.heads / p.heads_kv;
  const float s = p.softmax_scale;
  if (s > 0.f) {
    P.c = s;
    P.qa = 1.f;
  } else if (s < 0.f) {
    P.c = -s;
    P.qa = -1.f;
  } else {
    P.c = 1.f;
    P.qa = 0.f;
  }
  P.c2 = P.c * fna2::kLog2e;
  P.cu_q = p.cu_seqlens_q;
  P.cu_k = p.cu_seqlens_k;
  return P;
}

// Records caller-owned event i on the stream when events are requested.
bool mark(void* const* events, int i, hipStream_t stream) {
  if (!events || !events[i]) return true;
  return hipEventRecord((hipEvent_t)events[i], stream) == hipSuccess;
}

fna2::TView view(const fna2_tensor& t) {
  fna2::TView v;
  v.ptr = t.ptr;
  v.sb = t.stride_b;
  v.ss = t.stride_s;
  v.sh = t.stride_h;
  return v;
}

// Kernels exist for gfx950 only; cache the answer (and the CU count, which
// sizes the persistent grids) per device.
int check_device(int* num_cus = nullptr) {
  static std::mutex mu;
  static int state[64] = {0};  // 0 unknown, 1 ok, -1 wrong arch
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return FNA2_E_DEVICE;
  if (dev < 0 || dev >= 64) return FNA2_E_DEVICE;
  std::lock_guard<std::mutex> lk(mu);
  if (state[dev] == 0) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return FNA2_E_DEVICE;
    state[dev] = std::strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : -1;
    cus[dev] = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 1;
  }
  if (num_cus) *num_cus = cus[dev];
  return state[dev] == 1 ? FNA2_OK : FNA2_E_DEVICE;
}

}  // namespace

extern "C" {

int fna2_version(void) { return FNA2_ABI_VERSION; }

const char* fna2_status_string(int s) {
  switch (s) {
    case FNA2_OK: return "ok";
    case FNA2_E_NULL: return "a required pointer is NULL";
    case FNA2_E_DTYPE: return "unsupported dtype (attention: bf16 or fp16)";
    case FNA2_E_HEAD_DIM: return "head_dim must be 64 or 128";
    case FNA2_E_RANK: return "rank must be a multiple of 8 in [8, 64]";
    case FNA2_E_HEADS: return "heads must be a multiple of heads_kv and heads_graph <= heads";
    case FNA2_E_SHAPE: return "negative extent or problem too large";
    case FNA2_E_STRIDE: return "pointer or stride breaks 16-byte row alignment";
    case FNA2_E_SEQLENS: return "varlen mode needs cu_seqlens_q and cu_seqlens_k";
    case FNA2_E_WORKSPACE: return "workspace missing or too small";
    case FNA2_E_LAUNCH: return "kernel launch failed";
    case FNA2_E_DEVICE: return "current device is not gfx950";
    case FNA2_E_SCALE: return "softmax_scale must be finite";
    case FNA2_E_ALIAS: return "an output overlaps its input without being equal to it";
    case FNA2_E_SCRATCH:
      return "the problem needs more than the allocation-free entry point's static scratch "
             "(fna2_fwd_noalloc_max_bytes); use fna2_fwd with a workspace";
  }
  return "unknown status";
}

int fna2_check_fwd(const fna2_fwd_args* a) {
  if (!a) return FNA2_E_NULL;
  const fna2_problem& p = a->p;
  FNA2_TRY(check_problem(p));
  FNA2_TRY(check_grids(p));
  const bool qw = rows_q(p) > 0, kw = rows_k(p) > 0;
  const bool g = p.heads_graph > 0;
  FNA2_TRY(check_view(a->q, p, qw, true, 2));
  FNA2_TRY(check_view(a->out, p, qw, true, 2));
  FNA2_TRY(check_view(a->lse, p, qw, false, 4));
  FNA2_TRY(check_view(a->k, p, qw && kw, true, 2));
  FNA2_TRY(check_view(a->v, p, qw && kw, true, 2));
  FNA2_TRY(check_view(a->r_q, p, qw && g, true, 2));
  FNA2_TRY(check_view(a->r_k, p, qw && kw && g, true, 2));
  if (qw && g && !a->graph_scale) return FNA2_E_NULL;
  if (use_plan(a->plan, p)) {
    if (a->plan_bytes < plan_layout(p).bytes || !aligned(a->plan, 32)) return FNA2_E_WORKSPACE;
  } else if (a->workspace_bytes < fwd_ws(p).bytes || (fwd_ws(p).bytes && !a->workspace)) {
    return FNA2_E_WORKSPACE;
  }
  return FNA2_OK;
}

int fna2_check_bwd(const fna2_bwd_args* a) {
  if (!a) return FNA2_E_NULL;
  const fna2_problem& p = a->p;
  FNA2_TRY(check_problem(p));
  FNA2_TRY(check_grids(p));
  const bool qw = rows_q(p) > 0, kw = rows_k(p) > 0;
  const bool g = p.heads_graph > 0;
  FNA2_TRY(check_view(a->q, p, qw, true, 2));
  FNA2_TRY(check_view(a->out, p, qw, true, 2));
  FNA2_TRY(check_view(a->dout, p, qw, true, 2));
  FNA2_TRY(check_view(a->dq, p, qw, true, 2));
  FNA2_TRY(check_view(a->lse, p, qw, false, 4));
  FNA2_TRY(check_view(a->delta, p, qw, false, 4));
  FNA2_TRY(check_view(a->k, p, kw, true, 2));
  FNA2_TRY(check_view(a->v, p, kw, true, 2));
  FNA2_TRY(check_view(a->dk, p, kw, true, 2));
  FNA2_TRY(check_view(a->dv, p, kw, true, 2));
  FNA2_TRY(check_view(a->r_q, p, qw && g, true, 2));
  FNA2_TRY(check_view(a->dr_q, p, qw && g, true, 2));
  FNA2_TRY(check_view(a->r_k, p, kw && g, true, 2));
  FNA2_TRY(check_view(a->dr_k, p, kw && g, true, 2));
  if (g && (!a->graph_scale || !a->d_graph_scale)) return FNA2_E_NULL;
  // The dK/dV kernel addresses one sequence's query rows of a head with
  // 32-bit byte offsets.  In varlen mode seqlen_q is only a scheduling hint:
  // total_q bounds every sequence's length.
  const uint64_t span_rows =
      (uint64_t)(p.varlen ? std::max(p.total_q, p.seqlen_q) : p.seqlen_q);
  auto span_ok = [&](const fna2_tensor& t, uint64_t esize) {
    const uint64_t ss = (uint64_t)(t.stride_s < 0 ? -t.stride_s : t.stride_s);
    return span_rows * ss * esize < (1ull << 31);
  };
  if (qw && !(span_ok(a->q, 2) && span_ok(a->dout, 2) && span_ok(a->delta, 4)))
    return FNA2_E_SHAPE;
  // (the workspace copy of bf16(b Rq), one padded-rank row per query row)
  if (qw && g && span_rows * (uint64_t)fna2::padded_rank32(p.heads_graph, p.rank) * 2u >=
                     (1ull << 31))
    return FNA2_E_SHAPE;
  const BwdWs w = bwd_ws(p);
  if (a->workspace_bytes < w.bytes || !a->workspace) return FNA2_E_WORKSPACE;
  if (use_plan(a->plan, p) && (a->plan_bytes < plan_layout(p).bytes || !aligned(a->plan, 32)))
    return FNA2_E_WORKSPACE;
  return FNA2_OK;
}

size_t fna2_fwd_workspace_bytes(const fna2_problem* p) {
  if (!p || check_problem(*p) != FNA2_OK) return 0;
  return fwd_ws(*p).bytes;
}

size_t fna2_bwd_workspace_bytes(const fna2_problem* p) {
  if (!p || check_problem(*p) != FNA2_OK) return 0;
  return bwd_ws(*p).bytes;
}

size_t fna2_bwd_split_bytes(const fna2_problem* p) {
  if (!p || check_problem(*p) != FNA2_OK) return 0;
  return kv_split(*p).bytes;
}

int fna2_key_groups(const fna2_problem* p, int backward) {
  if (!p) return FNA2_E_NULL;
  FNA2_TRY(check_problem(*p));
  return backward ? dq_groups(*p) : fwd_groups(*p);
}

size_t fna2_plan_bytes(const fna2_problem* p) {
  if (!p || check_problem(*p) != FNA2_OK) return 0;
  return plan_layout(*p).bytes;
}

}  // extern "C"

namespace {

// The forward, with its varlen tile list in `ws` (at least fwd_ws(p).bytes;
// unused with a plan or in dense mode).  `a` has been checked.
int fwd_launch(const fna2_fwd_args* a, void* ws, hipStream_t stream) {
  const fna2_problem& p = a->p;
  // A plan is filled even without query rows: the backward relies on it.
  if (p.batch == 0 || (rows_q(p) == 0 && !use_plan(a->plan, p))) return FNA2_OK;
  FNA2_TRY(check_device());
  fna2::FwdParams K;
  std::memset(&K, 0, sizeof(K));
  K.p = make_problem(p);
  K.q = view(a->q);
  K.k = view(a->k);
  K.v = view(a->v);
  K.rq = view(a->r_q);
  K.rk = view(a->r_k);
  K.o = view(a->out);
  K.lse = view(a->lse);
  K.gs = a->graph_scale;
  const Grids g = grids(p);
  if (p.varlen && use_plan(a->plan, p)) {
    // One launch builds this call's list and the backward's key-tile list,
    // unless the caller vouches that an earlier forward of this problem
    // filled the plan (and our record of it agrees).
    const PlanLayout L = plan_layout(p);
    char* pl = (char*)a->plan;
    fna2::TileRec* tiles = (fna2::TileRec*)(pl + L.tiles_q);
    int* count = (int*)(pl + L.count_q);
    if (!(a->plan_filled && plan_filled_for(a->plan, p))) {
      const fna2::TileList lq{{0, kFwdBM, kFwdBN, 1}, tiles, count, (int)g.fwd_bound};
      const fna2::TileList lk{{1, kv_tile(p), kKvBM, 0}, (fna2::TileRec*)(pl + L.tiles_k),
                              (int*)(pl + L.count_k), (int)g.kv_bound};
      if (fna2::launch_build_tiles(K.p, lq, &lk, nullptr, stream) != hipSuccess)
        return FNA2_E_LAUNCH;
      plan_register(a->plan, p);
    }
    if (rows_q(p) == 0) return FNA2_OK;
    K.tiles = tiles;
    K.n_tiles = count;
  } else if (p.varlen) {
    const FwdWs w = fwd_ws(p);
    fna2::TileRec* tiles = (fna2::TileRec*)((char*)ws + w.tiles);
    int* count = (int*)((char*)ws + w.count);
    const fna2::TileList list{{0, kFwdBM, kFwdBN, 1}, tiles, count, (int)g.fwd_bound};
    if (fna2::launch_build_tiles(K.p, list, nullptr, nullptr, stream) != hipSuccess)
      return FNA2_E_LAUNCH;
    K.tiles = tiles;
    K.n_tiles = count;
  }
  const int rpl = fna2::padded_rank32(K.p.H_G, K.p.R);
  if (!mark(a->events, 0, stream)) return FNA2_E_LAUNCH;
  K.key_groups = fwd_groups(p);
  if (fna2::launch_fwd(K, rpl, (int)g.fwd_grid, stream) != hipSuccess) return FNA2_E_LAUNCH;
  if (!mark(a->events, 1, stream)) return FNA2_E_LAUNCH;
  return FNA2_OK;
}

// Device memory of the allocation-free forward: the varlen tile list (and
// its count) that fna2_fwd keeps in the caller's workspace.  Every GPU the
// library runs on holds its own copy until the process ends.  In host code
// `scratch` names a host-side stand-in, never its device address: that is
// resolved per device (hipGetSymbolAddress, with the device current) and
// only the resolved pointer is handed to kernels.
constexpr size_t kScratchBytes = (size_t)1 << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

int scratch_ptr(void** out) {
  static std::mutex mu;
  static void* ptrs[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return FNA2_E_DEVICE;
  std::lock_guard<std::mutex> lk(mu);
  if (!ptrs[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr)
      return FNA2_E_DEVICE;
    ptrs[dev] = ptr;
  }
  *out = ptrs[dev];
  return FNA2_OK;
}

}  // namespace

extern "C" {

int fna2_fwd(const fna2_fwd_args* a, void* stream_ptr) {
  FNA2_TRY(fna2_check_fwd(a));
  return fwd_launch(a, a->workspace, (hipStream_t)stream_ptr);
}

size_t fna2_fwd_noalloc_max_bytes(void) { return kScratchBytes; }

int fna2_fwd_noalloc(const fna2_fwd_args* a, void* stream_ptr) {
  if (!a) return FNA2_E_NULL;
  // Validate as fna2_fwd would with a workspace of the scratch's size (the
  // caller's workspace fields are ignored).
  fna2_fwd_args b = *a;
  b.workspace = nullptr;
  b.workspace_bytes = 0;
  FNA2_TRY(check_problem(b.p));
  if (!use_plan(b.plan, b.p) && fwd_ws(b.p).bytes > kScratchBytes) return FNA2_E_SCRATCH;
  void* ws = nullptr;
  if (!use_plan(b.plan, b.p) && fwd_ws(b.p).bytes > 0) {
    FNA2_TRY(scratch_ptr(&ws));
    b.workspace = ws;
    b.workspace_bytes = kScratchBytes;
  }
  FNA2_TRY(fna2_check_fwd(&b));
  return fwd_launch(&b, ws, (hipStream_t)stream_ptr);
}

int fna2_bwd(const fna2_bwd_args* a, void* stream_ptr) {
  FNA2_TRY(fna2_check_bwd(a));
  const fna2_problem& p = a->p;
  int n_cu = 1;
  FNA2_TRY(check_device(&n_cu));
  hipStream_t stream = (hipStream_t)stream_ptr;
  fna2::BwdParams K;
  std::memset(&K, 0, sizeof(K));
  K.p = make_problem(p);
  K.q = view(a->q);
  K.k = view(a->k);
  K.v = view(a->v);
  K.rq = view(a->r_q);
  K.rk = view(a->r_k);
  K.o = view(a->out);
  K.lse = view(a->lse);
  K.dout = view(a->dout);
  K.delta = view(a->delta);
  K.dq = view(a->dq);
  K.dk = view(a->dk);
  K.dv = view(a->dv);
  K.drq = view(a->dr_q);
  K.drk = view(a->dr_k);
  K.gs = a->graph_scale;
  K.dgs = a->d_graph_scale;
  const BwdWs w = bwd_ws(p);
  const Grids g = grids(p);
  K.dgs_partial = (float*)((char*)a->workspace + w.partial);
  K.q_tiles = (int)g.q_tiles;
  K.k_tiles = (int)g.kv_tiles;
  const int rpl = fna2::padded_rank32(K.p.H_G, K.p.R);
  // Head-major (a head's rows are contiguous): the dK/dV kernel reads it per
  // head, 32 rows at a time.
  const int64_t seq_rows = p.varlen ? (int64_t)p.total_q : (int64_t)p.seqlen_q;
  K.nlse.ptr = (char*)a->workspace + w.nlse;
  K.nlse.ss = 1;
  K.nlse.sh = seq_rows;
  K.nlse.sb = p.varlen ? 0 : (int64_t)p.heads * seq_rows;

  if (p.batch > 0 && (rows_q(p) > 0 || rows_k(p) > 0)) {
    if (p.varlen && use_plan(a->plan, p) && rows_q(p) > 0 && plan_filled_for(a->plan, p)) {
      // The forward built both lists; the dQ kernel's spare workgroups zero
      // the rows no sequence covers.  (Without query rows no dQ kernel runs:
      // the lists are then built, and the rows zeroed, below.)
      const PlanLayout L = plan_layout(p);
      const char* pl = (const char*)a->plan;
      K.tiles_q = (const fna2::TileRec*)(pl + L.tiles_q);
      K.n_tiles_q = (const int*)(pl + L.count_q);
      K.tiles_k = (const fna2::TileRec*)(pl + L.tiles_k);
      K.n_tiles_k = (const int*)(pl + L.count_k);
      K.zero_uncovered = 1;
    } else if (p.varlen) {
      fna2::TileRec* tq = (fna2::TileRec*)((char*)a->workspace + w.tiles_q);
      int* cq = (int*)((char*)a->workspace + w.count_q);
      fna2::TileRec* tk = (fna2::TileRec*)((char*)a->workspace + w.tiles_k);
      int* ck = (int*)((char*)a->workspace + w.count_k);
      const fna2::TileList lq{{0, kDqBM, kDqBN, 1}, tq, cq, (int)g.dq_bound};
      const fna2::TileList lk{{1, kv_tile(p), kKvBM, 0}, tk, ck, (int)g.kv_bound};
      const fna2::ZeroRows zero{K.dq, K.drq, K.dk, K.dv, K.drk,
                                (int)std::max(p.total_q, p.total_k)};
      if (fna2::launch_build_tiles(K.p, lq, &lk, &zero, stream) != hipSuccess)
        return FNA2_E_LAUNCH;
      K.tiles_q = tq;
      K.n_tiles_q = cq;
      K.tiles_k = tk;
      K.n_tiles_k = ck;
    }
    // dQ first: it also stores delta, which the dK/dV kernel reads.
    if (!mark(a->events, 0, stream)) return FNA2_E_LAUNCH;
    // (with a plan, one more row of workgroups than tiles can fill, so that
    // spare workgroups exist for the zeroing whatever the lengths)
    const int dq_grid = (int)g.dq_grid + (K.zero_uncovered ? p.heads : 0);
    K.key_groups = dq_groups(p);
    if (rows_q(p) > 0 && fna2::launch_bwd_dq(K, rpl, dq_grid, stream) != hipSuccess)
      return FNA2_E_LAUNCH;
    if (!mark(a->events, 1, stream) || !mark(a->events, 2, stream)) return FNA2_E_LAUNCH;
    // Items in chunks, where the rule asks for it and the caller's workspace
    // has the room (bwd_ws and fna2_bwd_split_bytes).
    const KvSplit sp = kv_split(p);
    int64_t items = g.kv_grid;
    if (sp.bytes > 0 && rows_q(p) > 0 && a->workspace_bytes >= w.bytes + sp.bytes &&
        aligned(a->workspace, 16)) {
      char* base = (char*)a->workspace + w.bytes;
      K.split_tiles = (int)sp.tiles;
      K.split_log2 = sp.log2;
      K.kv_part = (float*)(base + sp.kv_part);
      K.drk_part = (float*)(base + sp.drk_part);
      items += ((sp.tiles * p.heads_kv) << sp.log2) - sp.tiles * p.heads_kv;
    }
    // persistent: one workgroup per CU walks the (key tile, KV head) items
    const int kv_grid = (int)std::min<int64_t>(items, n_cu);
    if (rows_k(p) > 0 && fna2::launch_bwd_dkdv(K, rpl, kv_grid, stream) != hipSuccess)
      return FNA2_E_LAUNCH;
    if (K.split_tiles > 0 && rows_k(p) > 0 &&
        fna2::launch_bwd_kv_reduce(K, rpl, stream) != hipSuccess)
      return FNA2_E_LAUNCH;
    if (!mark(a->events, 3, stream)) return FNA2_E_LAUNCH;
  } else if (p.varlen && p.batch == 0 && (rows_q(p) > 0 || rows_k(p) > 0)) {
    // No sequences: every token lies outside them and gets zero gradients.
    const fna2::ZeroRows zero{K.dq, K.drq, K.dk, K.dv, K.drk,
                              (int)std::max(p.total_q, p.total_k)};
    if (fna2::launch_zero_rows(K.p, zero, stream) != hipSuccess) return FNA2_E_LAUNCH;
  }
  // The dK/dV kernel reduces d_gs when it runs.
  const bool dkdv_ran = p.batch > 0 && rows_k(p) > 0 && g.kv_grid > 0;
  if (!dkdv_ran && fna2::launch_bwd_dgs(K, stream) != hipSuccess) return FNA2_E_LAUNCH;
  return FNA2_OK;
}

}  // extern "C"

namespace {

// Byte range [lo, hi) a [T, heads, D] view covers.
void rope_extent(const fna2_tensor& t, int T, int heads, int D, size_t es, uintptr_t& lo,
                 uintptr_t& hi) {
  int64_t a = 0, b = D;
  const int64_t ds = (int64_t)(T - 1) * t.stride_s, dh = (int64_t)(heads - 1) * t.stride_h;
  (ds < 0 ? a : b) += ds;
  (dh < 0 ? a : b) += dh;
  lo = (uintptr_t)t.ptr + (uintptr_t)(a * (int64_t)es);
  hi = (uintptr_t)t.ptr + (uintptr_t)(b * (int64_t)es);
}

int rope_pair(const fna2_tensor& in, const fna2_tensor& out, int T, int heads, int D,
              size_t es) {
  if (!in.ptr || !out.ptr) return FNA2_E_NULL;
  for (const fna2_tensor* t : {&in, &out}) {
    if ((uintptr_t)t->ptr % 16 || (t->stride_s * (int64_t)es) % 16 ||
        (t->stride_h * (int64_t)es) % 16)
      return FNA2_E_STRIDE;
  }
  if (in.ptr == out.ptr)
    return in.stride_s == out.stride_s && in.stride_h == out.stride_h ? FNA2_OK : FNA2_E_ALIAS;
  uintptr_t l0, h0, l1, h1;
  rope_extent(in, T, heads, D, es, l0, h0);
  rope_extent(out, T, heads, D, es, l1, h1);
  return (l0 < h1 && l1 < h0) ? FNA2_E_ALIAS : FNA2_OK;
}

// Checks shared by the forward and the backward (no tensors).
int rope_common(const fna2_rope_args* a) {
  if (!a) return FNA2_E_NULL;
  if (a->dtype != FNA2_BF16 && a->dtype != FNA2_F16 && a->dtype != FNA2_F32) return FNA2_E_DTYPE;
  const int D = a->head_dim;
  if (D < 16 || D > 512 || (D & (D - 1)) != 0) return FNA2_E_HEAD_DIM;
  if (a->total_tokens < 0 || a->heads_q < 0 || a->heads_k < 0 || a->nseq < 0 ||
      (a->sign != 1 && a->sign != -1))
    return FNA2_E_SHAPE;
  if ((a->norm_q || a->norm_k) && !(std::isfinite(a->norm_eps) && a->norm_eps >= 0.f))
    return FNA2_E_SCALE;
  if (a->total_tokens == 0 || a->heads_q + a->heads_k == 0) return FNA2_OK;
  if (!a->cu_seqlens) return FNA2_E_SEQLENS;
  if (!a->inv_freq) return FNA2_E_NULL;
  return FNA2_OK;
}

bool rope_empty(const fna2_rope_args* a) {
  return a->total_tokens == 0 || a->heads_q + a->heads_k == 0;
}

size_t rope_esize(const fna2_rope_args* a) { return a->dtype == FNA2_F32 ? 4 : 2; }

fna2::RopeParams rope_params(const fna2_rope_args* a) {
  fna2::RopeParams P;
  std::memset(&P, 0, sizeof(P));
  P.dtype = a->dtype == FNA2_BF16 ? fna2::kRopeBF16
            : a->dtype == FNA2_F16 ? fna2::kRopeF16
                                   : fna2::kRopeF32;
  P.T = a->total_tokens;
  P.Hq = a->heads_q;
  P.Hk = a->heads_k;
  P.D = a->head_dim;
  P.nseq = a->nseq;
  P.sign = a->sign;
  P.cu = a->cu_seqlens;
  P.inv_freq = a->inv_freq;
  P.q = a->q.ptr;
  P.k = a->k.ptr;
  P.q_ss = a->q.stride_s;
  P.q_sh = a->q.stride_h;
  P.k_ss = a->k.stride_s;
  P.k_sh = a->k.stride_h;
  P.wq = a->heads_q > 0 ? a->norm_q : nullptr;
  P.wk = a->heads_k > 0 ? a->norm_k : nullptr;
  P.eps = a->norm_eps;
  return P;
}

void rope_out(fna2::RopeParams& P, const fna2_tensor& qo, const fna2_tensor& ko) {
  P.q_out = qo.ptr;
  P.k_out = ko.ptr;
  P.qo_ss = qo.stride_s;
  P.qo_sh = qo.stride_h;
  P.ko_ss = ko.stride_s;
  P.ko_sh = ko.stride_h;
}

size_t rope_ws(const fna2_rope_args* a) {
  if (!(a->norm_q || a->norm_k) || rope_empty(a)) return 0;
  return align_up(sizeof(float) * 2u * (size_t)fna2::rope_bwd_blocks(a->total_tokens) *
                  (size_t)a->head_dim);
}

}  // namespace

extern "C" {

int fna2_check_rope(const fna2_rope_args* a) {
  FNA2_TRY(rope_common(a));
  if (rope_empty(a)) return FNA2_OK;
  const int T = a->total_tokens, D = a->head_dim;
  const size_t es = rope_esize(a);
  if (a->heads_q > 0) FNA2_TRY(rope_pair(a->q, a->q_out, T, a->heads_q, D, es));
  if (a->heads_k > 0) FNA2_TRY(rope_pair(a->k, a->k_out, T, a->heads_k, D, es));
  return FNA2_OK;
}

int fna2_rope_varlen(const fna2_rope_args* a, void* stream) {
  FNA2_TRY(fna2_check_rope(a));
  if (rope_empty(a)) return FNA2_OK;
  FNA2_TRY(check_device());
  fna2::RopeParams P = rope_params(a);
  rope_out(P, a->q_out, a->k_out);
  if (fna2::launch_rope(P, (hipStream_t)stream) != hipSuccess) return FNA2_E_LAUNCH;
  return FNA2_OK;
}

size_t fna2_rope_bwd_workspace_bytes(const fna2_rope_args* a) {
  if (!a || rope_common(a) != FNA2_OK) return 0;
  return rope_ws(a);
}

int fna2_check_rope_bwd(const fna2_rope_bwd_args* b) {
  if (!b) return FNA2_E_NULL;
  const fna2_rope_args* a = &b->fwd;
  FNA2_TRY(rope_common(a));
  if (rope_empty(a)) return FNA2_OK;
  const int T = a->total_tokens, D = a->head_dim;
  const size_t es = rope_esize(a);
  const bool norm = a->norm_q || a->norm_k;
  if (a->heads_q > 0) {
    FNA2_TRY(rope_pair(b->dq_out, b->dq, T, a->heads_q, D, es));
    if (norm) FNA2_TRY(rope_pair(a->q, b->dq, T, a->heads_q, D, es));
    if (a->norm_q && !b->dnorm_q) return FNA2_E_NULL;
  }
  if (a->heads_k > 0) {
    FNA2_TRY(rope_pair(b->dk_out, b->dk, T, a->heads_k, D, es));
    if (norm) FNA2_TRY(rope_pair(a->k, b->dk, T, a->heads_k, D, es));
    if (a->norm_k && !b->dnorm_k) return FNA2_E_NULL;
  }
  const size_t need = rope_ws(a);
  if (need && (!b->workspace || b->workspace_bytes < need)) return FNA2_E_WORKSPACE;
  return FNA2_OK;
}

int fna2_rope_bwd(const fna2_rope_bwd_args* b, void* stream) {
  FNA2_TRY(fna2_check_rope_bwd(b));
  const fna2_rope_args* a = &b->fwd;
  if (rope_empty(a)) return FNA2_OK;
  FNA2_TRY(check_device());
  fna2::RopeParams P = rope_params(a);
  rope_out(P, b->dq, b->dk);
  if (!(P.wq || P.wk)) {  // the inverse rotation of the gradients
    P.q = b->dq_out.ptr;
    P.k = b->dk_out.ptr;
    P.q_ss = b->dq_out.stride_s;
    P.q_sh = b->dq_out.stride_h;
    P.k_ss = b->dk_out.stride_s;
    P.k_sh = b->dk_out.stride_h;
    P.sign = -a->sign;
    if (fna2::launch_rope(P, (hipStream_t)stream) != hipSuccess) return FNA2_E_LAUNCH;
    return FNA2_OK;
  }
  P.gq = b->dq_out.ptr;
  P.gk = b->dk_out.ptr;
  P.gq_ss = b->dq_out.stride_s;
  P.gq_sh = b->dq_out.stride_h;
  P.gk_ss = b->dk_out.stride_s;
  P.gk_sh = b->dk_out.stride_h;
  P.part = (float*)b->workspace;
  P.dwq = P.wq ? b->dnorm_q : nullptr;
  P.dwk = P.wk ? b->dnorm_k : nullptr;
  if (fna2::launch_rope_norm_bwd(P, (hipStream_t)stream) != hipSuccess) return FNA2_E_LAUNCH;
  return FNA2_OK;
}

}  // extern "C"

namespace {

// Work units of a decode launch are sized for MI355X's 256 compute units
// (a fixed figure, so that the split count and the workspace size are a
// function of the arguments alone).
constexpr int kDecodeCUs = 256;
constexpr int64_t kOff31 = ((int64_t)1 << 31) - 16;  // buffer-offset bound

int dec_group(const fna2_decode_args& a) { return a.heads / a.heads_kv; }

// Graph heads of the widest KV-head group and their rank chunks.
int dec_graph_heads(const fna2_decode_args& a) {
  return a.heads_graph > 0 ? std::min(dec_group(a), a.heads_graph) : 0;
}
int dec_rc(const fna2_decode_args& a) {
  return fna2::decode_rank_chunks(dec_graph_heads(a) * (a.heads_graph > 0 ? a.rank / 8 : 0));
}

int check_bf16_rows(const fna2_tensor& t) {
  if (!t.ptr) return FNA2_E_NULL;
  if (!aligned(t.ptr, 16)) return FNA2_E_STRIDE;
  if (t.stride_b < 0 || t.stride_s < 0 || t.stride_h < 0) return FNA2_E_STRIDE;
  if (t.stride_b % 8 || t.stride_s % 8 || t.stride_h % 8) return FNA2_E_STRIDE;
  return FNA2_OK;
}

struct DecSplit {
  int n = 1, keys = 32;
};

// The library's split count.
//
// Small caches: the least estimated time over the counts that differ.  A
// wave walks its split's 32-key steps, each a chain of latencies (`step`,
// longer with the rank tile and with more waves on the CU), behind its own
// start (`kStart`).  As many waves run at once as the ring's LDS leaves room
// for, so they come in rounds, the last partly filled, each as long as its
// chain or as reading its share of the cache takes.  More than one split adds
// the merge (`kMerge` and its partials).  Where the lengths differ (the host
// does not know them) the last round holds a longest split; the others, and
// the bytes, count two thirds.
// Large ones (kDecodeLarge): the rate follows the waves in flight, up to four
// per CU, so one round of them as full as whole splits make it, of at least
// four steps; with differing lengths (kDecodeRagged) up to eight rounds, which
// level them, of eight steps, while the partials are few.
//
// Fitted to 388 calls of 1 to 128 sequences, 4 to 32 heads and 33 to 40,000
// rows, timed behind a full queue at up to 20 counts each (us).  Against the
// best count of each, mean and most: small caches 1.006 and 1.14, large ones
// 1.02 and 1.10, ragged 1.03 and 1.13.  (One round of waves and one-step
// splits for few units, at any size: 1.056 and 1.9 for the small, 1.05 and
// 1.18 for the large and ragged; two rounds: 1.16 and 1.9, 1.07 and 1.3.)
// What those missed:
//   up to four to six steps a second launch costs more than it saves: B4 H4/1
//     d64 L84 5.2 whole, 7.4 in three; B2 H8/2 d128 r16 L73 8.0, 9.9
//   waves just past a round: B3 H32 d128 L7267 9 splits 65, 12 80; B118 H4/2
//     d128 r8 L305 4 splits 15.1, 5 19.2
//   ragged lengths in full rounds anyway: B97 H32 d128 L304 59 whole, 76 in
//     three
//   large and ragged: B26 H8 d128 r32 L23182 4 splits 388, 32 341
// The lines: equal lengths, 300 to 600 MB, the estimate's counts 1.04 times
// the best, one round 1.01 (B20 H32/8 L6000, 491 MB: 104, 90); below the 256
// MB that the last cache level holds 1.011 and 1.016.  Differing lengths, 350
// to 600 MB: the estimate 1.03, the rounds 1.10; above, 1.055 and 1.03.
constexpr double kDecodeLarge = 256e6, kDecodeRagged = 600e6;
DecSplit dec_split(const fna2_decode_args& a, bool ragged) {
  DecSplit s;
  const int64_t L = a.max_seqlen_k;
  if (L <= 0) return s;
  const int64_t steps = cdiv64(L, 32);
  int64_t n = a.num_splits;
  if (n <= 0) {
    const int rc = std::max(dec_rc(a), 0);
    // (one byte less: the full 160 KB do not all go to workgroups)
    const int per_cu = std::max(
        1, (160 * 1024 - 1) / (fna2::kDecodeStages * fna2::decode_stage_bytes(a.head_dim, rc)));
    const int64_t units = std::max<int64_t>((int64_t)a.batch * a.heads_kv, 1);
    const double bytes = 2. * L * a.batch * (2. * a.heads_kv * a.head_dim +
                                             (double)a.heads_graph * a.rank);
    n = 1;
    const double partials = 4. * a.batch * a.heads * a.head_dim;  // bytes a split
    if (bytes >= (ragged ? kDecodeRagged : kDecodeLarge)) {
      const int64_t fill = (int64_t)kDecodeCUs * std::min(per_cu, 4);
      if (ragged) {
        n = std::min(cdiv64(8 * fill, units), (int64_t)(0.006 * bytes / partials));
        n = std::min(std::max<int64_t>(std::max(n, cdiv64(fill, units)), 4), cdiv64(steps, 8));
      } else {
        n = std::min(fill / units, cdiv64(steps, 4));
      }
      n = std::max<int64_t>(std::min<int64_t>(n, 64), 1);
    } else {
      // us; us a byte of the cache and of the partials
      constexpr double kStart = 3.2, kMerge = 3.4, kRead = 0.16e-6, kPart = 0.8e-6;
      const double step = 0.32 + 0.034 * rc + 0.38 * a.head_dim / 64;
      const double cap = (double)kDecodeCUs * per_cu;
      const double part = ragged ? 2. / 3 : 1.;  // of the longest
      const double read = kRead * part * bytes;
      double least = 0;
      for (int64_t i = 1, last = 0; i <= std::min<int64_t>(steps, 64); ++i) {
        const int64_t len = cdiv64(steps, i);  // steps a split
        const int64_t count = cdiv64(steps, len);
        if (count == last) continue;
        last = count;
        const double waves = (double)units * count;
        auto round = [&](double w, double of) {
          return std::max(kStart + of * len * step * (1 + 0.155 * std::max(w / kDecodeCUs - 1, 0.)),
                          read * w / waves);
        };
        const double full = std::floor(waves / cap), rest = waves - full * cap;
        double t = full > 0 ? full * round(cap, part) : 0;
        if (rest > 0) t += round(rest, 1);
        if (count > 1) t += kMerge + kPart * partials * count;
        if (i == 1 || t < 0.98 * least) {
          least = t;
          n = count;
        }
      }
    }
  }
  n = std::min<int64_t>(n, steps);
  s.keys = (int)(cdiv64(cdiv64(L, n), 32) * 32);
  s.n = (int)cdiv64(L, s.keys);
  return s;
}
DecSplit dec_split(const fna2_decode_args& a) { return dec_split(a, a.seqlens_k != nullptr); }

size_t dec_workspace(const fna2_decode_args& a, const DecSplit& s) {
  if (s.n <= 1) return 0;
  const size_t rows = (size_t)s.n * (size_t)a.batch * (size_t)a.heads;
  return align_up(rows * (size_t)a.head_dim * 4u) + align_up(rows * 8u);
}

}  // namespace

extern "C" {

int fna2_check_decode(const fna2_decode_args* a) {
  if (!a) return FNA2_E_NULL;
  if (a->head_dim != 64 && a->head_dim != 128) return FNA2_E_HEAD_DIM;
  if (a->heads <= 0 || a->heads_kv <= 0 || a->heads % a->heads_kv != 0) return FNA2_E_HEADS;
  if (dec_group(*a) > 32) return FNA2_E_HEADS;
  if (a->heads_graph < 0 || a->heads_graph > a->heads) return FNA2_E_HEADS;
  const bool graph = a->heads_graph > 0;
  if (graph && (a->rank < 8 || a->rank > 64 || a->rank % 8 != 0)) return FNA2_E_RANK;
  if (graph && dec_rc(*a) < 0) return FNA2_E_RANK;
  if (a->batch < 0 || a->max_seqlen_k < 0) return FNA2_E_SHAPE;
  if (a->num_splits < 0 || a->num_splits > 64) return FNA2_E_SHAPE;
  if (!std::isfinite(a->softmax_scale)) return FNA2_E_SCALE;
  if (a->batch == 0) return FNA2_OK;
  FNA2_TRY(check_bf16_rows(a->q));
  FNA2_TRY(check_bf16_rows(a->out));
  const bool rows = a->max_seqlen_k > 0;  // an empty cache is never read
  if (rows) {
    FNA2_TRY(check_bf16_rows(a->k_cache));
    FNA2_TRY(check_bf16_rows(a->v_cache));
  }
  if (graph) {
    FNA2_TRY(check_bf16_rows(a->r_q));
    if (rows) FNA2_TRY(check_bf16_rows(a->rk_cache));
    if (!a->graph_scale) return FNA2_E_NULL;
  }
  if (a->lse.ptr) {
    if (!aligned(a->lse.ptr, 4) || a->lse.stride_b < 0 || a->lse.stride_h < 0)
      return FNA2_E_STRIDE;
  }
  const int64_t g = dec_group(*a), D = a->head_dim;
  if ((g - 1) * a->q.stride_h * 2 + D * 2 > kOff31) return FNA2_E_SHAPE;
  if (32 * a->k_cache.stride_s * 2 > kOff31 || 32 * a->v_cache.stride_s * 2 > kOff31)
    return FNA2_E_SHAPE;
  if (graph) {
    const int64_t gg = dec_graph_heads(*a), R = a->rank;
    if ((gg - 1) * a->r_q.stride_h * 2 + R * 2 > kOff31) return FNA2_E_SHAPE;
    if ((gg - 1) * a->rk_cache.stride_h * 2 + 31 * a->rk_cache.stride_s * 2 + R * 2 > kOff31)
      return FNA2_E_SHAPE;
  }
  const int64_t units = (int64_t)a->batch * a->heads_kv;  // (at most 64 splits)
  if (units > kMaxGrid / 64 && units * dec_split(*a).n > kMaxGrid) return FNA2_E_SHAPE;
  return FNA2_OK;
}

int fna2_decode_num_splits(const fna2_decode_args* a) {
  FNA2_TRY(fna2_check_decode(a));
  return dec_split(*a).n;
}

size_t fna2_decode_workspace_bytes(const fna2_decode_args* a) {
  if (fna2_check_decode(a) != FNA2_OK) return 0;
  return dec_workspace(*a, dec_split(*a));
}

int fna2_decode(const fna2_decode_args* a, void* stream_ptr) {
  FNA2_TRY(fna2_check_decode(a));
  if (a->batch == 0) return FNA2_OK;
  FNA2_TRY(check_device());
  // (a workspace sized without the lengths has the room of the even split)
  DecSplit s = dec_split(*a);
  if (dec_workspace(*a, s) > a->workspace_bytes) s = dec_split(*a, false);
  const size_t need = dec_workspace(*a, s);
  if (need > 0 && (!a->workspace || a->workspace_bytes < need || !aligned(a->workspace, 16)))
    return FNA2_E_WORKSPACE;
  hipStream_t stream = (hipStream_t)stream_ptr;
  fna2::DecodeParams K;
  std::memset(&K, 0, sizeof(K));
  K.B = a->batch;
  K.H = a->heads;
  K.H_KV = a->heads_kv;
  K.H_G = a->heads_graph;
  K.D = a->head_dim;
  K.R = a->heads_graph > 0 ? a->rank : 0;
  K.group = dec_group(*a);
  K.nsplit = s.n;
  K.split_keys = s.keys;
  K.max_len = a->max_seqlen_k;
  const float sc = a->softmax_scale;
  K.c = sc > 0.f ? sc : sc < 0.f ? -sc : 1.f;
  K.qa = sc > 0.f ? 1.f : sc < 0.f ? -1.f : 0.f;
  K.c2 = K.c * fna2::kLog2e;
  K.seqlens = a->seqlens_k;
  K.q = view(a->q);
  K.rq = view(a->r_q);
  K.k = view(a->k_cache);
  K.v = view(a->v_cache);
  K.rk = view(a->rk_cache);
  K.o = view(a->out);
  K.lse = view(a->lse);
  K.gs = a->graph_scale;
  if (s.n > 1) {
    const size_t rows = (size_t)s.n * (size_t)a->batch * (size_t)a->heads;
    K.acc = (float*)a->workspace;
    K.ml = (float*)((char*)a->workspace + align_up(rows * (size_t)a->head_dim * 4u));
  }
  const int rc = a->heads_graph > 0 ? dec_rc(*a) : 0;
  if (!mark(a->events, 0, stream)) return FNA2_E_LAUNCH;
  if (fna2::launch_decode(K, rc, stream) != hipSuccess) return FNA2_E_LAUNCH;
  if (!mark(a->events, 1, stream)) return FNA2_E_LAUNCH;
  if (fna2::launch_decode_merge(K, stream) != hipSuccess) return FNA2_E_LAUNCH;
  return FNA2_OK;
}

int fna2_check_decode_rows(const fna2_decode_rows_args* a) {
  if (!a) return FNA2_E_NULL;
  if (a->head_dim != 64 && a->head_dim != 128) return FNA2_E_HEAD_DIM;
  if (a->heads <= 0 || a->heads_kv <= 0 || a->heads_graph < 0) return FNA2_E_HEADS;
  if (a->heads_graph > 0 && (a->rank < 8 || a->rank > 64 || a->rank % 8 != 0))
    return FNA2_E_RANK;
  if (a->batch < 0) return FNA2_E_SHAPE;
  if ((int64_t)a->batch * ((int64_t)a->heads + 2 * (int64_t)a->heads_kv + a->heads_graph) >
      kMaxGrid)
    return FNA2_E_SHAPE;
  if ((a->norm_q && !std::isfinite(a->eps_q)) || (a->norm_k && !std::isfinite(a->eps_k)))
    return FNA2_E_SCALE;
  if (!a->cos != !a->sin) return FNA2_E_NULL;
  for (const void* w : {a->norm_q, a->norm_k, a->cos, a->sin})
    if (!aligned(w, 16)) return FNA2_E_STRIDE;
  if (a->batch == 0) return FNA2_OK;
  for (const fna2_tensor* t : {&a->q, &a->k, &a->v, &a->q_out, &a->k_out, &a->v_out})
    FNA2_TRY(check_bf16_rows(*t));
  if (a->heads_graph > 0) {
    FNA2_TRY(check_bf16_rows(a->r_k));
    FNA2_TRY(check_bf16_rows(a->rk_out));
  }
  return FNA2_OK;
}

int fna2_decode_rows(const fna2_decode_rows_args* a, void* stream) {
  FNA2_TRY(fna2_check_decode_rows(a));
  if (a->batch == 0) return FNA2_OK;
  FNA2_TRY(check_device());
  fna2::DecodeRowsParams K;
  std::memset(&K, 0, sizeof(K));
  K.B = a->batch;
  K.H = a->heads;
  K.H_KV = a->heads_kv;
  K.H_G = a->heads_graph;
  K.D = a->head_dim;
  K.R = a->heads_graph > 0 ? a->rank : 0;
  K.q = view(a->q);
  K.k = view(a->k);
  K.v = view(a->v);
  K.rk = view(a->r_k);
  K.qo = view(a->q_out);
  K.ko = view(a->k_out);
  K.vo = view(a->v_out);
  K.rko = view(a->rk_out);
  K.wq = (const uint16_t*)a->norm_q;
  K.wk = (const uint16_t*)a->norm_k;
  K.eps_q = a->eps_q;
  K.eps_k = a->eps_k;
  K.cos = (const uint16_t*)a->cos;
  K.sin = (const uint16_t*)a->sin;
  if (fna2::launch_decode_rows(K, (hipStream_t)stream) != hipSuccess) return FNA2_E_LAUNCH;
  return FNA2_OK;
}

}  // extern "C"
