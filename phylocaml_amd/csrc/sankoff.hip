// Sankoff (1975) parsimony under an integer transformation cost matrix, the
// whole tree in one launch.
//
// The reference has the cost-matrix type (PTcm.X, lib/pTcm.ml:5-50) and the
// median search over it (lib/costMatrix.ml:52-65, child state j under
// median k costs tcm[j][k]) but no tree-level Sankoff pass; this is the
// standard dynamic programme over that cost convention:
//   C_leaf[k] = 0 for k in the leaf's state set, else infinite
//   C_v[k]    = sum over children c of min_j (C_c[j] + tcm[j][k])
//   site cost = min_k C_root[k].
//
// Layout: lane = site (one byte per leaf and site holds the state set, K <= 8
// states).  A wave walks a post-order program (Sethi-Ullman order, accumulator
// plus LDS stack); the K x K matrix is wave-uniform (SGPRs), so an interior
// operand costs K^2 adds and K^2 - K mins on the lane's own K-vector.  A leaf
// operand is one LDS read of a table built once per block: tab[code][k] = min
// over j in code of tcm[j][k].  Leaf bytes stream in batches of 8 leaves, issued
// 16-24 leaves ahead.  All arithmetic is int32 (the host bounds the costs so no
// sum can overflow) and exact.
//
// With few sites the chain of the tree's nodes is the bound, and with a few
// waves per SIMD it is the SIMDs that have one more than the others.  The split
// form gives 64 sites to a block, whose waves take the parts of the tree
// (about sqrt(N)) off a counter, leave the parts' roots in LDS, and one of them
// walks the top.  512 taxa x 20,000 sites, K = 5: 175 -> 70 us; 301 x 200,003:
// 176 -> 154 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>

#include "common.hpp"
#include "stream.hpp"

namespace {

constexpr int32_t kInf = 1 << 28;  // larger than any finite cost of a site

// One byte per leaf for this lane's site: a window of 16 leaves, the next 8 in
// flight.  `rows` (uniform) is the wave's first site in the first leaf's row.
template <bool TOP>
struct TipBytes {
  const uint8_t* rows;
  int64_t stride;
  uint32_t off;
  const int32_t* ids;
  int n_leaves;
  uint32_t cur0, cur1, nxt0, nxt1;
  uint32_t pre[8];
  int pos, next_start;

  __device__ __forceinline__ void issue(int start, uint32_t* to) const {
    const int4* iv = reinterpret_cast<const int4*>(ids + start);
    const int4 a = iv[0], b = iv[1];
    const int id[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // a cut node of a top program has no tip row
      const int i = TOP && id[j] >= n_leaves ? 0 : id[j];
      to[j] = (rows + (int64_t)i * stride)[off];
    }
  }
  static __device__ __forceinline__ uint32_t pack(const uint32_t* b) {
    return b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
  }
  __device__ __forceinline__ void init(const uint8_t* r, int64_t s, uint32_t o, const int32_t* id, int n) {
    rows = r;
    stride = s;
    off = o;
    ids = id;
    n_leaves = n;
    uint32_t b0[8], b1[8];
    issue(0, b0);
    issue(8, b1);
    issue(16, pre);
    cur0 = pack(b0), cur1 = pack(b0 + 4), nxt0 = pack(b1), nxt1 = pack(b1 + 4);
    next_start = 16;
    pos = 0;
  }
  __device__ __forceinline__ uint32_t get() {
    const uint32_t v = ((pos < 4 ? cur0 : cur1) >> (8 * (pos & 3))) & 255u;
    if (++pos == 8) {
      cur0 = nxt0;
      cur1 = nxt1;
      nxt0 = pack(pre);
      nxt1 = pack(pre + 4);
      next_start += 8;
      issue(next_start, pre);
      pos = 0;
    }
    return v;
  }
};
static_assert(24 + 8 <= (int)kFifoSlack, "leaf stream look-ahead vs id padding");

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

constexpr int kSplitWaves = 8;
constexpr size_t kLdsMax = 64 * 1024;   // per block
constexpr size_t kLdsCu = 160 * 1024;

template <int K>
struct Cost {
  int32_t v[K];
};

// m[k] = min_j x[j] + T[j][k]
template <int K>
__device__ __forceinline__ void through(const int32_t (&T)[K][K], const int32_t* x, int32_t* m) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    int32_t v = x[0] + T[0][k];
#pragma unroll
    for (int j = 1; j < K; ++j) v = min(v, x[j] + T[j][k]);
    m[k] = v;
  }
}

// One program's walk, to its last node's vector.  stk is the lane's column of
// the wave's stack [depth][K][64], cut that of the parts' results [P][K][64],
// which are through the matrix already.
template <int K, bool TOP>
__device__ __forceinline__ Cost<K> walk(const int4* __restrict__ prog, int n_ops, TipBytes<TOP>& ts,
                                        const int32_t (&T)[K][K], const int32_t* tab, const int32_t* cut,
                                        int32_t* stk) {
  constexpr int NC = 1 << K;
  int32_t acc[K];
#pragma unroll
  for (int k = 0; k < K; ++k) acc[k] = 0;
  int sp = 0;
  auto leaf = [&](int32_t* m, int part) {
    const int c = (int)(ts.get() & (NC - 1));
    const int32_t* p = TOP && part ? cut + (part - 1) * K * 64 : tab + c * K;
    const int step = TOP && part ? 64 : 1;
#pragma unroll
    for (int k = 0; k < K; ++k) m[k] = p[k * step];
  };
  for_each_entry(prog, n_ops, [&](int, const int4 op) {
    const int fl = op.w;
    if (fl & DOWN_SPILL) {
#pragma unroll
      for (int k = 0; k < K; ++k) stk[(sp * K + k) * 64] = acc[k];
      ++sp;
    }
    int32_t ma[K], mb[K];
    const int sa = fl & 3, sb = (fl >> 2) & 3;
    if (sa == SRC_LEAF) {
      leaf(ma, (fl >> 8) & 255);
    } else if (sa == SRC_ACC) {
      through(T, acc, ma);
    } else {
      --sp;
      int32_t x[K];
#pragma unroll
      for (int k = 0; k < K; ++k) x[k] = stk[(sp * K + k) * 64];
      through(T, x, ma);
    }
    if (sb == SRC_LEAF)
      leaf(mb, (fl >> 16) & 255);
    else
      through(T, acc, mb);
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = ma[k] + mb[k];
  });
  Cost<K> c;
#pragma unroll
  for (int k = 0; k < K; ++k) c.v[k] = acc[k];
  return c;
}

template <int K, bool SPLIT>
__global__ __launch_bounds__(512) void k_sankoff_down(
    const int4* __restrict__ prog, int n_ops, const int32_t* __restrict__ fifo,
    const int32_t* __restrict__ meta, int P, int n_leaves, int depth, const int32_t* __restrict__ tcm,
    const uint8_t* __restrict__ tips, int64_t stride, int64_t n_sites, const uint32_t* __restrict__ wt,
    uint32_t* __restrict__ site_cost, unsigned long long* __restrict__ total) {
  constexpr int NC = 1 << K;
  extern __shared__ int32_t lds[];
  __shared__ int next_part;
  const int tid = threadIdx.x, bd = blockDim.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int32_t* tab = lds;                                       // [NC][K]
  int32_t* cut = tab + NC * K + lane;                       // [P][K][64]
  int32_t* stk = cut + (P + wave * depth) * K * 64;         // [wave][depth][K][64]
  for (int e = tid; e < NC * K; e += bd) {
    const int c = e / K ? e / K : NC - 1, k = e % K;  // code 0: every state
    int32_t m = kInf;
    for (int j = 0; j < K; ++j)
      if ((c >> j) & 1) m = min(m, tcm[j * K + k]);
    tab[e] = m;
  }
  if (SPLIT && tid == 0) next_part = bd >> 6;
  int32_t T[K][K];
#pragma unroll
  for (int j = 0; j < K; ++j)
#pragma unroll
    for (int k = 0; k < K; ++k) T[j][k] = tcm[j * K + k];
  __syncthreads();

  const int64_t s0 = SPLIT ? (int64_t)blockIdx.x * 64 : (int64_t)blockIdx.x * bd + wave * 64;
  const int64_t s = s0 + lane;
  const bool act = s < n_sites;
  const uint8_t* rows = tips + (s0 < n_sites ? s0 : 0);
  const uint32_t off = act ? lane : 0;
  TipBytes<false> ts;
  ts.init(rows, stride, off, fifo + (SPLIT ? meta[2 * (P + 1) + wave] : 0), n_leaves);
  Cost<K> root;
  if constexpr (SPLIT) {
    for (int p = wave;;) {  // wave < P
      const Cost<K> c = walk<K, false>(prog + meta[p], meta[P + 1 + p], ts, T, tab, cut, stk);
      int32_t m[K];
      through(T, c.v, m);
#pragma unroll
      for (int k = 0; k < K; ++k) cut[(p * K + k) * 64] = m[k];
      int q = 0;
      if (lane == 0) q = atomicAdd(&next_part, 1);
      p = __builtin_amdgcn_readfirstlane(q);
      if (p >= P) break;
      ts.init(rows, stride, off, fifo + meta[2 * (P + 1) + p], n_leaves);
    }
    TipBytes<true> tt;
    if (wave == 0) tt.init(rows, stride, off, fifo + meta[2 * (P + 1) + P], n_leaves);
    __syncthreads();
    if (wave != 0) return;
    root = walk<K, true>(prog + meta[P], meta[P + 1 + P], tt, T, tab, cut, stk);
  } else {
    root = walk<K, false>(prog, n_ops, ts, T, tab, cut, stk);
  }

  int32_t best = root.v[0];
#pragma unroll
  for (int k = 1; k < K; ++k) best = min(best, root.v[k]);
  uint64_t contrib = 0;
  if (act) {
    site_cost[s] = (uint32_t)best;
    contrib = (uint64_t)(wt ? wt[s] : 1u) * (uint64_t)best;
  }
  contrib = wave_sum_u64(contrib);
  if (lane == 0 && contrib) atomicAdd(total, (unsigned long long)contrib);
}

template <int K>
int sankoff_launch(phy_ctx* ctx, const phy_topo* topo, const int32_t* tcm, const uint8_t* tips,
                   int64_t stride, int64_t n_sites, const uint32_t* wt, uint32_t* site_cost,
                   unsigned long long* total) {
  const size_t tables = (size_t)(1 << K) * K * 4;
  const size_t wave_row = (size_t)K * 64 * 4;
  const int64_t groups = (n_sites + 63) / 64;
  KernelSpan span(ctx, "sankoff_down");
  // The split form pays while it holds more waves on a SIMD than the whole form
  // has for it (64 sites each): 512 taxa, K = 5, 200,003 sites 250 us against
  // 276 with 4.5 waves to 3, 1,024 taxa 538 against 508 with 3.  From K = 7 on
  // its matrix no longer stays in SGPRs and it has to hold two and three times as
  // many: 301 taxa, K = 7, 100,003 sites 179 us against 175, 5,000 sites 61
  // against 136; 128 taxa, K = 8, 100,003 sites 123 against 118, 50,000 sites 84
  // against 97.  At K = 6 half as many again: 300,000 sites, 64 taxa 104 against 110,
  // 100 taxa 134 against 130, 150 taxa 158 against 147.  Below 48 taxa, whose parts
  // are a few leaves, from K = 7 on twice that: 40 taxa, K = 7, 200,000 sites 90
  // against 86, K = 8, 100,000 sites 74 against 72, 50,000 sites 55 against 60.
  // Under three waves a block it does not pay at all.  Of the
  // numbers of waves the largest serves where every CU has at most one block, the
  // one with the most waves on a CU elsewhere.  PHY_SANKOFF_SPLIT=0: the whole form.
  const FitchSplit& f = topo->fine;
  const char* env = getenv("PHY_SANKOFF_SPLIT");
  const int P = env && env[0] == '0' ? 0 : (int)f.parts.size();
  int waves = 0, held = 0;
  size_t lds = 0;
  for (int w = std::min(kSplitWaves, P); w >= 3; --w) {
    const size_t need = 16 + tables + (size_t)(P + w * f.down.depth) * wave_row;
    const int h = std::min(32, w * (int)(kLdsCu / need));
    if (need > kLdsMax || h <= held || (waves && groups <= 256)) continue;
    waves = w, held = h, lds = need;
  }
  const int twice = K <= 5 ? 2 : K == 6 ? 3 : 2 * (K - 5) * (topo->n_leaves < 48 ? 2 : 1);  // 2 x the factor
  if ((int64_t)held * 512 > groups * twice) {
    hipLaunchKernelGGL((k_sankoff_down<K, true>), dim3((unsigned)groups), dim3(64 * waves), lds, ctx->stream,
                       f.down.d_prog, 0, f.down.d_fifo, f.down.d_meta, P, topo->n_leaves, f.down.depth, tcm, tips,
                       stride, n_sites, wt, site_cost, total);
    PHY_LAUNCHED(ctx);
    return PHY_OK;
  }
  int bs = 256;
  const auto whole_lds = [&] { return tables + (size_t)(bs / 64) * topo->down_depth * wave_row; };
  while (bs > 64 && whole_lds() > kLdsMax) bs /= 2;
  if (whole_lds() > kLdsMax) return set_err(ctx, PHY_ERANGE, "sankoff: LDS stack too deep");
  const int64_t nb = (n_sites + bs - 1) / bs;
  hipLaunchKernelGGL((k_sankoff_down<K, false>), dim3((unsigned)nb), dim3(bs), whole_lds(), ctx->stream,
                     topo->d_down_prog, topo->n_leaves - 1, topo->d_down_fifo, nullptr, 0, topo->n_leaves,
                     topo->down_depth, tcm, tips, stride, n_sites, wt, site_cost, total);
  PHY_LAUNCHED(ctx);
  return PHY_OK;
}

}  // namespace

extern "C" {

int phy_sankoff_downpass(phy_ctx* ctx, const phy_topo* topo, int32_t n_states,
                         const int32_t* d_tcm, const uint8_t* d_leaves, int64_t stride,
                         int64_t n_sites, const uint32_t* d_weights, uint32_t* d_site_cost,
                         uint64_t* d_total) {
  if (!ctx) return PHY_EINVAL;
  if (!topo || !topo->d_down_prog) return set_err(ctx, PHY_EINVAL, "sankoff: topology not on a device");
  if (n_states < 2 || n_states > 8) return set_err(ctx, PHY_EINVAL, "sankoff: n_states must be 2..8");
  if (n_sites < 0 || stride < n_sites) return set_err(ctx, PHY_EINVAL, "sankoff: stride < n_sites");
  if (!d_tcm || !d_site_cost || !d_total || (n_sites > 0 && !d_leaves))
    return set_err(ctx, PHY_EINVAL, "sankoff: null buffer");
  int rc;
  if ((rc = phy_zero_u64(ctx, d_total, 1))) return rc;
  if (n_sites == 0) return PHY_OK;
  auto* tt = reinterpret_cast<unsigned long long*>(d_total);
  switch (n_states) {
    case 2: return sankoff_launch<2>(ctx, topo, d_tcm, d_leaves, stride, n_sites, d_weights, d_site_cost, tt);
    case 3: return sankoff_launch<3>(ctx, topo, d_tcm, d_leaves, stride, n_sites, d_weights, d_site_cost, tt);
    case 4: return sankoff_launch<4>(ctx, topo, d_tcm, d_leaves, stride, n_sites, d_weights, d_site_cost, tt);
    case 5: return sankoff_launch<5>(ctx, topo, d_tcm, d_leaves, stride, n_sites, d_weights, d_site_cost, tt);
    case 6: return sankoff_launch<6>(ctx, topo, d_tcm, d_leaves, stride, n_sites, d_weights, d_site_cost, tt);
    case 7: return sankoff_launch<7>(ctx, topo, d_tcm, d_leaves, stride, n_sites, d_weights, d_site_cost, tt);
    default: return sankoff_launch<8>(ctx, topo, d_tcm, d_leaves, stride, n_sites, d_weights, d_site_cost, tt);
  }
}

}  // extern "C"
