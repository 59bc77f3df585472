// Batched 20-state (amino-acid) Felsenstein pruning on BF16 MFMA.
//
// Many independent trees of uneven taxon and pattern counts, each with its own
// GTR-20 model and Gamma rates, are evaluated in one persistent launch:
// workgroups take (tree, pattern tile) items from atomic queues until they are
// empty (every workgroup reaches the exit).  A workgroup of WAVES waves owns
// 16*WAVES patterns of one tree and walks that tree's post-order program
// (phy_topo_create's Sethi-Ullman order); the waves stay in lock step, so the
// transition-matrix operands of the node being computed are staged once into
// LDS and shared.
//
// Per node, child partial x (16 patterns x 20 states, R rates) times P^T with
// v_mfma_f32_16x16x32_bf16, A = P, B = x (columns = patterns).  The 20 states
// of a rate split into 16 + 4: R main tiles of 16 output states, and one tile
// whose 16 output rows are the last 4 states of up to 4 rates (row 4 rho + v =
// rate rho, state 16 + v).  Lane l (pattern l % 16, quarter q = l / 16) then
// holds states 4q .. 4q+3 of every rate and states 16 .. 19 of rate q: 4R + 4
// values with no padding at R = 4.  The k index of a product is free, so its
// slots are laid out as the lanes hold them -- slots 8q .. 8q+7 of the main
// product of rate r are the lane's 4 states of rate r and its 4 extra states
// (A is zero there unless q = r) -- and partials never move between lanes.
// The extra tile takes R products over the same operands (A holds the rows of
// rate r only), so a child is 2R products of R operands.
// (Padding each rate to 32 states gave 8R values a lane, 12 of every 32 of
// them zero: 196 VGPRs and two waves per SIMD against 146 to 158 and three at 4
// groups per tile here.  With the rest of the node loop below, 256 trees of 16-256
// taxa and 1,000-20,000 patterns take 9.1 ms against 17.1 at 8 groups per tile and
// 9.8 against 16.2 at 4.  Bound: the node's LDS reads and barrier, with the VALU
// held 59% and the matrix cores 29% of the time.  The pairs of figures at the rules
// below compare forms of one earlier state of the code on one card, 8.0 and 8.3 ms there.)
// Combining the two children, per-pattern power-of-two rescaling and the root
// sum are FP32 / FP64 VALU work on 4R + 4 values per lane.  A wave may own G
// groups of 16 patterns, which share each P operand it reads from LDS.
// Spilled partials are stored as the BF16 operand they will be used as (no
// extra rounding).
//
// Precision: MFMA inputs are BF16 (8-bit mantissa), accumulation, partials and
// exponents FP32 / int32, the root log-sum FP64.  P(t) = U diag(exp(lambda t))
// Ui is formed in FP64 from the host eigen-decomposition of each tree's Q.
#include <algorithm>
#include <cstdlib>
#include <cmath>
#include <numeric>

#include "common.hpp"
#include "model_host.hpp"
#include "stream.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int KAA = 20;
constexpr int OPB = 64;  // uint4 (16 B) per lane-ordered operand block (1 KiB)

// Work queues, one per XCD (workgroups are dealt round-robin to the 8 XCDs, so
// blockIdx % 8 names a workgroup's XCD).  The tiles of a tree share its P
// operands (7 KiB a branch at R = 4, ~2 MB for 128 taxa), which one XCD's 4 MB
// L2 holds and eight would each fetch: with one queue for all, the 256 trees
// above took 22.7 ms at 4 groups per tile, with these 9.4 (98% L2 hits).
// A workgroup whose queue is empty takes from the next one, so the placement
// is only a preference.
constexpr int kQueues = 8;
constexpr int kCounterPitch = 32;  // uint32: a 128-byte line per counter

struct AADev {
  const int4* prog;
  const int64_t* prog_off;  // entries
  const int32_t* n_leaves;
  const uint8_t* tips;
  const int64_t* tips_off;  // bytes
  const int64_t* pitch;     // padded patterns of each tree
  const uint32_t* wts;
  const int64_t* w_off;
  const uint4* pops;
  const int64_t* pop_off;   // uint4 units
  const double* pi;         // [T][20]
  const double* probs;      // [T][R]
  const int2* items;        // (tree, tile), queue by queue
  int q_off[kQueues + 1];   // first item of each queue
  double* part;
  const int64_t* part_off;
  unsigned* counter;        // items taken from each queue
  int depth;                // LDS stack entries per wave
};

// operand blocks (1 KiB) of one branch: R main products, R of the extra tile
constexpr int aa_blocks(int R) { return 2 * R; }

// --- P operands: a block of R waves takes `per` consecutive branches,
// wave r forming P(rate_r t) in FP64 from U and Ui staged in LDS (a 2 x 4
// tile of entries per lane), then the waves write the branch's operand blocks.
// (One wave per (branch, rate) reading U and Ui from memory for every entry:
// 425 us for 64 trees of 16-256 taxa, here 93.) ---
// Branches per block: up to 8 share a tree's staged U and Ui, fewer when that
// would leave CUs without a block.
constexpr int kPopsPerBlock = 8;

template <int R>
__global__ __launch_bounds__(64 * R) void k_aa_pops(
    const double* __restrict__ eig,  // [T][U 400|lam 20|Ui 400]
    const double* __restrict__ rates,  // [T][R]
    const double* __restrict__ blen,   // flat
    const int64_t* __restrict__ blen_off,
    const int32_t* __restrict__ br_tree,  // flat branch -> tree
    int64_t n_branches, int per, const int64_t* __restrict__ pop_off, uint4* __restrict__ pops) {
  constexpr int NB = aa_blocks(R), KK = KAA * KAA;
  const int r = threadIdx.x >> 6, l = threadIdx.x & 63;
  __shared__ double U[KK], Ui[KK], ex[R][KAA], P[R][KK];
  int staged = -1;
  const int64_t b0 = (int64_t)blockIdx.x * per;
  const int64_t b1 = b0 + per < n_branches ? b0 + per : n_branches;
  for (int64_t gb = b0; gb < b1; ++gb) {  // flat branch index (block-uniform)
    const int t = br_tree[gb];
    const int64_t b = gb - blen_off[t];
    const double* E = eig + (size_t)t * (2 * KK + KAA);
    const double rt = rates[(size_t)t * R + r] * blen[gb];
    if (t != staged) {  // the previous branch's reads ended before its last barrier
      for (int e = threadIdx.x; e < KK; e += 64 * R) {
        U[e] = E[e];
        Ui[e] = E[KK + KAA + e];
      }
      staged = t;
    }
    if (l < KAA) ex[r][l] = exp(E[KK + l] * rt);
    __syncthreads();
    if (l < 50) {  // rows i0, i0 + 1, columns j0 .. j0 + 3
      const int i0 = 2 * (l / 5), j0 = 4 * (l % 5);
      double s[2][4] = {};
      for (int m = 0; m < KAA; ++m) {
        const double e = ex[r][m], u0 = U[i0 * KAA + m] * e, u1 = U[(i0 + 1) * KAA + m] * e;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const double v = Ui[m * KAA + j0 + j];
          s[0][j] += u0 * v;
          s[1][j] += u1 * v;
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          double v = s[i][j];
          if (!(rt >= 1e-10)) v = (i0 + i == j0 + j) ? 1.0 : 0.0;  // compose rule, lib/mlmodel.c:339-341
          P[r][(i0 + i) * KAA + j0 + j] = v;
        }
    }
    __syncthreads();
    uint4* dst = pops + pop_off[t] + b * (NB * OPB);
    const int row = l & 15, q = l >> 4;
    for (int blk = r; blk < NB; blk += R) {
      bf16x8 a;
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        // main: state `row` of rate `br`; extra tile: state 16 + row % 4 of
        // rate row / 4, zero unless that is `br`
        const int br = blk % R;
        const int st = blk < R ? row : (row >> 2) == br ? 16 + (row & 3) : -1;
        double val = 0.0;
        if (st >= 0) {
          if (v < 4) val = P[br][st * KAA + 4 * q + v];
          else if (q == br) val = P[br][st * KAA + 16 + v - 4];
        }
        a[v] = (__bf16)(float)val;
      }
      dst[blk * OPB + l] = *reinterpret_cast<uint4*>(&a);
    }
  }
}

// four values as packed BF16
__device__ __forceinline__ uint2 pack4(const float* x) {
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  bf16x4 r;
#pragma unroll
  for (int v = 0; v < 4; ++v) r[v] = (__bf16)x[v];
  return *reinterpret_cast<const uint2*>(&r);
}
__device__ __forceinline__ bf16x8 operand(const uint2 lo, const uint2 hi) {
  const uint4 u = make_uint4(lo.x, lo.y, hi.x, hi.y);
  return *reinterpret_cast<const bf16x8*>(&u);
}

// a lane's slots of a tip: states 4q .. 4q+3, then 16 .. 19
__device__ __forceinline__ bf16x8 tip_operand(uint32_t code, int q) {
  bf16x8 r;
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    const int s = v < 4 ? 4 * q + v : 12 + v;
    r[v] = (__bf16)((code >= (uint32_t)KAA || s == (int)code) ? 1.0f : 0.0f);
  }
  return r;
}

// 16-byte units of one LDS stack level of a 16-pattern group: R + 1 packed
// quadruples a lane, and 16 exponents
constexpr int aa_level(int R) { return (R + 1) * 32 + 4; }

// a partial as BF16 operands, with its exponent
template <int R>
struct AAVec {
  uint2 own[R], ext;
  int e;
};

// TW: 16-pattern groups of a tile; G: groups of a wave
template <int TW, int G, int R, int LV>
__global__ __launch_bounds__(64 * (TW / G)) void k_aa_prune(AADev a) {
  static_assert(TW % G == 0, "whole groups per wave");
  constexpr int NW = TW / G, NT = 64 * NW;
  constexpr int NB = aa_blocks(R);
  constexpr int NBLK = 2 * NB;              // 1 KiB operand blocks per node
  __shared__ uint4 stage[2][NBLK * OPB];    // double buffer: node i and node i+1
  __shared__ uint4 tipop[(KAA + 1) * 4];    // B operand of a tip: [code 0..20][quarter]
  __shared__ int s_item;
  extern __shared__ uint4 dyn[];
  // the wave index is uniform: readfirstlane keeps the operand DMA loop scalar
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63,
            q = l >> 4, pl = l & 15;
  // per-group stack: the bottom LV levels in registers (selected by the
  // uniform stack pointer with value selects), the rest in LDS
  const int rows = a.depth > LV ? a.depth - LV : 0;
  uint4* stk = dyn + (size_t)wave * G * rows * aa_level(R);
  AAVec<R> rs[LV > 0 ? LV : 1][G];
  // the 21 tip operands (a state 0..19, or missing = all 20 states) for each
  // quarter of the lanes, built once; a tip child is then one LDS read
  for (int e = tid; e < (KAA + 1) * 4; e += NT) {
    const bf16x8 b = tip_operand((uint32_t)(e >> 2), e & 3);
    tipop[e] = *reinterpret_cast<const uint4*>(&b);
  }

  bool own_empty = false;
  for (;;) {
    __syncthreads();
    if (tid < 64) {
      const int own = (int)(blockIdx.x % kQueues);
      auto take = [&](int xq) {
        int k = 0;
        if (l == 0) k = (int)atomicAdd(a.counter + xq * kCounterPitch, 1u);
        k = a.q_off[xq] + __builtin_amdgcn_readfirstlane(k);
        return k < a.q_off[xq + 1] ? k : -1;
      };
      int item = own_empty ? -1 : take(own);
      own_empty = item < 0;
      // one parallel look at every queue before each attempt: counters only
      // grow, so an attempt that fails leaves one queue less
      while (item < 0) {
        const int x = l < kQueues ? l : 0;
        const unsigned taken = __hip_atomic_load(a.counter + x * kCounterPitch, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
        const bool left = l < kQueues && (int)taken < a.q_off[x + 1] - a.q_off[x];
        const unsigned m = (unsigned)__ballot(left);
        if (!m) break;
        const unsigned after = m & ~((2u << own) - 1u);  // the next queue that has items, cyclically
        item = take(__builtin_ctz(after ? after : m));
      }
      if (l == 0) s_item = item;
    }
    __syncthreads();
    // uniform in fact; readfirstlane tells the compiler, so everything
    // derived from the item (tree offsets, operand addresses) is
    // scalar
    const int item = __builtin_amdgcn_readfirstlane(s_item);
    if (item < 0) break;
    const int2 it = a.items[item];
    const int t = __builtin_amdgcn_readfirstlane(it.x), tile = __builtin_amdgcn_readfirstlane(it.y);
    const int64_t pitch = a.pitch[t];
    // pattern of group 0; group g is 16 g further, all < pitch by construction
    const int64_t p = (int64_t)tile * (16 * TW) + wave * (16 * G) + pl;
    const int N = a.n_leaves[t];
    const int4* prog = a.prog + a.prog_off[t];
    const uint8_t* tips = a.tips + a.tips_off[t];
    const uint4* pops = a.pops + a.pop_off[t];
    int sp = 0;
    float acc[G][R + 1][4];  // [r]: states 4q+v of rate r; [R]: states 16+v of rate q
    int acc_e[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      acc_e[g] = 0;
#pragma unroll
      for (int r = 0; r <= R; ++r)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[g][r][v] = 0.f;
    }

    // Every global load issued while node i computes (the operand DMA of node
    // i+1, the tip codes of node i+1) is consumed at node i+1
    // or later, after the node's closing vmcnt(0) and barrier.  Nothing loaded
    // from global memory is waited on in the middle of a node, so the DMA
    // latency overlaps a whole node of MFMA and VALU work.
    //
    // operands of a node's two children straight into LDS (global_load_lds,
    // 16 B per lane: one 1 KiB block per wave instruction), no registers
    // a wave copies consecutive blocks of one child (of both if it is alone),
    // four to an address
    auto dma_stage = [&](const int4 o, int buf) {
      constexpr int HW = NW > 1 ? NW / 2 : 1;     // waves per child
      constexpr int CH = (NB + HW - 1) / HW;      // blocks per wave and child
      const int first = (wave % HW) * CH;
#pragma unroll
      for (int cc = 0; cc < (NW > 1 ? 1 : 2); ++cc) {
        const int c = NW > 1 ? wave / HW : cc;
        const uint32_t child = (uint32_t)(c ? o.z : o.y) * (NB * OPB);
#pragma unroll
        for (int k = 0; k < CH; k += 4) {
          if (NB % CH != 0 || HW * CH > NB)
            if (first + k >= NB) break;
          const uint4* src = pops + child + (first + k) * OPB + l;
          uint4* dst = &stage[buf][(c * NB + first + k) * OPB];
          static_for<0, (CH < 4 ? CH : 4)>([&](auto j) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                             (__attribute__((address_space(3))) void*)dst, 16,
                                             decltype(j)::value * 1024, 0);
          });
        }
      }
    };
    // tip codes of a node's leaf children (row 0 for a child that is no leaf)
    auto leaf_codes = [&](const int4 o, uint32_t* ca, uint32_t* cb) {
      const uint8_t* ta = tips + (int64_t)((o.w & 3) == SRC_LEAF ? o.y : 0) * pitch;
      const uint8_t* tb = tips + (int64_t)(((o.w >> 2) & 3) == SRC_LEAF ? o.z : 0) * pitch;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        ca[g] = ta[p + 16 * g];
        cb[g] = tb[p + 16 * g];
      }
    };
    uint32_t code_a[G], code_b[G];
    {
      const int4 o0 = prog[0];
      leaf_codes(o0, code_a, code_b);
      dma_stage(o0, 0);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the DMA has landed
    __syncthreads();

    auto packed = [&](int g) {
      AAVec<R> u;
#pragma unroll
      for (int r = 0; r < R; ++r) u.own[r] = pack4(acc[g][r]);
      u.ext = pack4(acc[g][R]);
      u.e = acc_e[g];
      return u;
    };
    auto select = [&](bool hit, AAVec<R>& d, const AAVec<R>& x) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        d.own[r].x = hit ? x.own[r].x : d.own[r].x;
        d.own[r].y = hit ? x.own[r].y : d.own[r].y;
      }
      d.ext.x = hit ? x.ext.x : d.ext.x;
      d.ext.y = hit ? x.ext.y : d.ext.y;
      d.e = hit ? x.e : d.e;
    };

    for_each_entry_ahead(prog, N - 1, [&](int i, const int4 op, const int4 on) {
      const int buf = i & 1;
      const bool more = i + 1 < N - 1;
      const int fl = op.w;
      if (more) dma_stage(on, buf ^ 1);  // in flight while node i computes
      uint32_t ca[G], cb[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        ca[g] = code_a[g];
        cb[g] = code_b[g];
      }
      leaf_codes(on, code_a, code_b);  // node i+1's tips, used there
      auto pop = [&](int c, int blk) {
        const uint4 u = stage[buf][(c * NB + blk) * OPB + l];
        return *reinterpret_cast<const bf16x8*>(&u);
      };
      if (fl & DOWN_SPILL) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const AAVec<R> u = packed(g);
          if (sp < LV) {
            static_for<0, LV>([&](auto lv) { select(sp == lv, rs[lv][g], u); });
          } else {
            uint2* s = reinterpret_cast<uint2*>(stk + (size_t)((sp - LV) * G + g) * aa_level(R));
#pragma unroll
            for (int r = 0; r < R; ++r) s[r * 64 + l] = u.own[r];
            s[R * 64 + l] = u.ext;
            if (q == 0) reinterpret_cast<int*>(s + (R + 1) * 64)[pl] = u.e;
          }
        }
        ++sp;
      }
      float xa[G][R + 1][4];
      int ea[G];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int src = c ? ((fl >> 2) & 3) : (fl & 3);
        AAVec<R> x[G];
        if (src == SRC_LEAF) {
#pragma unroll
          for (int g = 0; g < G; ++g) {
            const uint4 tu = tipop[min(c ? cb[g] : ca[g], (uint32_t)KAA) * 4 + q];
#pragma unroll
            for (int r = 0; r < R; ++r) x[g].own[r] = make_uint2(tu.x, tu.y);
            x[g].ext = make_uint2(tu.z, tu.w);
            x[g].e = 0;
          }
        } else if (src == SRC_ACC) {
#pragma unroll
          for (int g = 0; g < G; ++g) x[g] = packed(g);
        } else {
          --sp;
#pragma unroll
          for (int g = 0; g < G; ++g) {
            if (sp < LV) {
              x[g] = rs[0][g];
              static_for<1, LV>([&](auto lv) { select(sp == lv, x[g], rs[lv][g]); });
            } else {
              const uint2* s = reinterpret_cast<const uint2*>(stk + (size_t)((sp - LV) * G + g) * aa_level(R));
#pragma unroll
              for (int r = 0; r < R; ++r) x[g].own[r] = s[r * 64 + l];
              x[g].ext = s[R * 64 + l];
              x[g].e = reinterpret_cast<const int*>(s + (R + 1) * 64)[pl];
            }
          }
        }
        auto combine = [&](int g, int r, const f32x4 d) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            if (c == 0) xa[g][r][v] = d[v];
            else acc[g][r][v] = xa[g][r][v] * d[v];
          }
        };
        f32x4 d[G];
#pragma unroll
        for (int g = 0; g < G; ++g) d[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const bf16x8 Am = pop(c, r), Ax = pop(c, R + r);
#pragma unroll
          for (int g = 0; g < G; ++g) {
            const bf16x8 b = operand(x[g].own[r], x[g].ext);
            combine(g, r, __builtin_amdgcn_mfma_f32_16x16x32_bf16(Am, b, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0));
            d[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Ax, b, d[g], 0, 0, 0);
          }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          combine(g, R, d[g]);
          if (c == 0) ea[g] = x[g].e;
          else acc_e[g] = ea[g] + x[g].e;
        }
      }
      // Every node is rescaled, one of two leaves too: two such sisters of ~1e-17
      // each (short branches, states without direct exchange) leave FP32's range
      // at their parent.
#pragma unroll
      for (int g = 0; g < G; ++g) {
        // per-pattern rescale: lanes l, l^16, l^32, l^48 share pattern pl
        float mx = 0.f;
#pragma unroll
        for (int r = 0; r <= R; ++r)
#pragma unroll
          for (int v = 0; v < 4; ++v) mx = fmaxf(mx, acc[g][r][v]);
        // with lanes l ^ 16 and l ^ 32 (v_permlane16/32_swap: no LDS round trip);
        // the values are not negative, so their bits compare as integers
        {
          unsigned u = __float_as_uint(mx);
          const auto s16 = __builtin_amdgcn_permlane16_swap(u, u, false, false);
          u = s16[0] > s16[1] ? s16[0] : s16[1];
          const auto s32 = __builtin_amdgcn_permlane32_swap(u, u, false, false);
          mx = __uint_as_float(s32[0] > s32[1] ? s32[0] : s32[1]);
        }
        if (mx < 0x1p-24f && mx > 0.f) {
          int ex;
          (void)frexpf(mx, &ex);
#pragma unroll
          for (int r = 0; r <= R; ++r)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[g][r][v] = ldexpf(acc[g][r][v], -ex);
          acc_e[g] += ex;
        }
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): node i+1 operands and tips landed
      __syncthreads();
    });
    // root: L_p = sum_r prob_r sum_i pi_i L[r][i]
    const double* pi = a.pi + (size_t)t * KAA;
    const double* pr = a.probs + (size_t)t * R;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      double s = 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        double sr = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) sr += pi[4 * q + v] * (double)acc[g][r][v];
        s += pr[r] * sr;
      }
      if (q < R) {
        double sr = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) sr += pi[16 + v] * (double)acc[g][R][v];
        s += pr[q] * sr;
      }
      s += __shfl_xor(s, 16, 64);
      s += __shfl_xor(s, 32, 64);
      const uint32_t w = a.wts[a.w_off[t] + p + 16 * g];
      double contrib = (q == 0 && w) ? (double)w * (log(s) + (double)acc_e[g] * 0.6931471805599453) : 0.0;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) contrib += __shfl_xor(contrib, off, 64);
      if (l == 0) a.part[a.part_off[t] + (int64_t)tile * TW + wave * G + g] = contrib;
    }
  }
}

// one block per tree: Neumaier sum of its partials
__global__ void k_aa_reduce(const double* __restrict__ part, const int64_t* __restrict__ off,
                            double* __restrict__ out) {
  const int t = blockIdx.x;
  const int64_t b = off[t], e = off[t + 1];
  __shared__ double ss[256], cc[256];
  double s = 0.0, c = 0.0;
  for (int64_t i = b + threadIdx.x; i < e; i += blockDim.x) {
    const double v = part[i], y = s + v;
    if (fabs(s) >= fabs(v)) c += (s - y) + v; else c += (v - y) + s;
    s = y;
  }
  ss[threadIdx.x] = s;
  cc[threadIdx.x] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    double S = 0.0, C = 0.0;
    for (int k = 0; k < (int)blockDim.x; ++k) {
      const double v = ss[k], y = S + v;
      if (fabs(S) >= fabs(v)) C += (S - y) + v; else C += (v - y) + S;
      S = y;
      C += cc[k];
    }
    out[t] = S + C;
  }
}

__global__ void k_zero_u32(unsigned* p) { p[threadIdx.x * kCounterPitch] = 0u; }

}  // namespace

// ---------------------------------------------------------------------------
struct phy_aa_batch {
  phy_ctx* ctx = nullptr;
  int32_t T = 0, R = 4, waves = 4, depth = 0;
  std::vector<int32_t> n_leaves;
  std::vector<int64_t> n_pat, pitch;
  int64_t n_items = 0;
  int32_t q_off[kQueues + 1] = {};
  int64_t n_branches = 0, pattern_nodes = 0;
  std::vector<void*> bufs;  // owned device allocations
  // device arrays
  int4* prog = nullptr;
  int64_t *prog_off = nullptr, *tips_off = nullptr, *pitch_d = nullptr,
          *w_off = nullptr, *pop_off = nullptr, *part_off = nullptr, *blen_off = nullptr;
  int32_t *nl = nullptr, *br_tree = nullptr;
  uint8_t* tips = nullptr;
  uint32_t* wts = nullptr;
  uint4* pops = nullptr;
  double *pi = nullptr, *probs = nullptr, *rates = nullptr, *eig = nullptr, *blen = nullptr,
         *part = nullptr;
  int2* items = nullptr;
  unsigned* counter = nullptr;
};

namespace {

template <class T>
int upload(phy_aa_batch* b, T** dst, const std::vector<T>& src) {
  const size_t bytes = std::max<size_t>(src.size() * sizeof(T), 16);
  if (hipMalloc((void**)dst, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return set_err(b->ctx, PHY_ENOMEM, "aa_batch: device allocation failed");
  }
  b->bufs.push_back(*dst);
  if (!src.empty()) PHY_HIP(b->ctx, hipMemcpy(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice));
  return PHY_OK;
}

// Order the items (given tree by tree) into the queues: trees by decreasing
// taxa, so that every queue runs its longest items first, each to the queue
// with the least work so far (a tile costs its tree's taxa).  A tree of more
// than 1/32 of the whole work is dealt in runs of tiles that small, so that
// few or uneven trees still spread over the chip.
void deal_items(const std::vector<int32_t>& n_leaves, std::vector<int2>& items, int32_t* q_off) {
  const size_t T = n_leaves.size();
  std::vector<int64_t> first(T + 1, 0);
  int64_t total = 0;
  for (const int2& it : items) {
    ++first[it.x + 1];
    total += n_leaves[it.x];
  }
  for (size_t t = 0; t < T; ++t) first[t + 1] += first[t];
  std::vector<int32_t> order(T);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int32_t x, int32_t y) { return n_leaves[x] > n_leaves[y]; });
  std::vector<int2> q[kQueues];
  int64_t load[kQueues] = {};
  for (const int32_t t : order) {
    const int64_t run = std::max<int64_t>(1, total / 32 / n_leaves[t]);
    for (int64_t k = first[t]; k < first[t + 1]; k += run) {
      const int x = (int)(std::min_element(load, load + kQueues) - load);
      const int64_t end = std::min(k + run, first[t + 1]);
      q[x].insert(q[x].end(), items.begin() + k, items.begin() + end);
      load[x] += (end - k) * n_leaves[t];
    }
  }
  items.clear();
  for (int x = 0; x < kQueues; ++x) {
    q_off[x] = (int32_t)items.size();
    items.insert(items.end(), q[x].begin(), q[x].end());
  }
  q_off[kQueues] = (int32_t)items.size();
}

size_t lds_bytes(int waves, int R, int depth, int lv) {
  return (size_t)waves * (depth > lv ? depth - lv : 0) * aa_level(R) * sizeof(uint4);
}

// Groups of 16 patterns per wave: two where a tile has 8 (the waves of a
// workgroup then share its operand copies less often but read each operand
// from LDS once for 32 patterns: 8.0 against 12.1 ms for the 256 trees above),
// else one (at 4 groups per tile two waves would copy the 16 KiB of a node:
// 15.1 against 8.3 ms).  One too where every CU has at most one workgroup, whose
// chain of nodes is then the bound (one tree of 200 taxa x 2,000 patterns, R = 4:
// 258 against 285 us; 12 trees of 64 x 3,000, 259 tiles: 158 against 127), and with
// two rate classes (64 trees of 200 x 9,000: 1,647 against 1,728; R = 1 1,237
// against 1,007).
int aa_groups(int waves, int R, int64_t n_items, int n_cu) {
  return waves == 8 && R != 2 && n_items > n_cu ? 2 : 1;
}

// Stack levels kept in registers: none for stacks of 1 or 2 levels (fewer
// VGPRs), else 3, or 4 with one group per wave for stacks of 5 or more (at 5
// levels three workgroups of 4 waves then fit a CU's LDS instead of two, and
// the registers still allow three waves per SIMD: 8.3 against 10.9 ms).
// PHY_AA_REG=0|3 overrides.
int aa_register_levels(int depth, int groups) {
  const char* s = getenv("PHY_AA_REG");
  if (s && (s[0] == '0' || s[0] == '3') && s[1] == 0) return s[0] - '0';
  return depth >= 5 && groups == 1 ? 4 : depth >= 3 ? 3 : 0;
}

template <int TW, int G, int R, int LV>
int launch(phy_ctx* ctx, phy_aa_batch* b) {
  AADev a;
  a.prog = b->prog;
  a.prog_off = b->prog_off;
  a.n_leaves = b->nl;
  a.tips = b->tips;
  a.tips_off = b->tips_off;
  a.pitch = b->pitch_d;
  a.wts = b->wts;
  a.w_off = b->w_off;
  a.pops = b->pops;
  a.pop_off = b->pop_off;
  a.pi = b->pi;
  a.probs = b->probs;
  a.items = b->items;
  for (int k = 0; k <= kQueues; ++k) a.q_off[k] = b->q_off[k];
  a.part = b->part;
  a.part_off = b->part_off;
  a.counter = b->counter;
  a.depth = std::max(1, b->depth);
  const size_t lds = lds_bytes(TW, R, a.depth, LV);
  constexpr int NT = 64 * (TW / G);
  int dev = 0, n_cu = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (k_aa_prune<TW, G, R, LV>), NT, lds) != hipSuccess || per_cu < 1)
    per_cu = 1;
  const int64_t grid = std::min<int64_t>((int64_t)n_cu * per_cu, b->n_items);
  KernelSpan span(ctx, "aa_prune");
  hipLaunchKernelGGL((k_aa_prune<TW, G, R, LV>), dim3((unsigned)std::max<int64_t>(grid, 1)), dim3(NT), lds,
                     ctx->stream, a);
  PHY_LAUNCHED(ctx);
  return PHY_OK;
}

template <int TW, int G, int R>
int launch_g(phy_ctx* ctx, phy_aa_batch* b) {
  switch (aa_register_levels(std::max(1, b->depth), G)) {
    case 0: return launch<TW, G, R, 0>(ctx, b);
    case 3: return launch<TW, G, R, 3>(ctx, b);
    default: return launch<TW, G, R, G == 1 ? 4 : 3>(ctx, b);
  }
}

template <int TW, int R>
int launch_l(phy_ctx* ctx, phy_aa_batch* b) {
  int n_cu = 256;
  (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, ctx->device);
  if constexpr (TW == 8 && R != 2)
    if (aa_groups(TW, R, b->n_items, n_cu) == 2) return launch_g<TW, 2, R>(ctx, b);
  return launch_g<TW, 1, R>(ctx, b);
}

template <int R>
int launch_w(phy_ctx* ctx, phy_aa_batch* b) {
  switch (b->waves) {
    case 1: return launch_l<1, R>(ctx, b);
    case 2: return launch_l<2, R>(ctx, b);
    case 4: return launch_l<4, R>(ctx, b);
    case 8: return launch_l<8, R>(ctx, b);
    default: return set_err(ctx, PHY_ERANGE, "aa_batch: waves per workgroup must be 1, 2, 4 or 8");
  }
}

}  // namespace

extern "C" {

int phy_aa_batch_create(phy_ctx* ctx, int32_t T, const int32_t* n_leaves, const int64_t* n_patterns,
                        const int32_t* children, const int32_t* roots, const double* blen,
                        const double* pi, const double* Q, int32_t R, const double* rates,
                        const double* probs, const uint8_t* tips, const uint32_t* weights,
                        int32_t waves, phy_aa_batch** out) {
  if (!ctx || !out) return PHY_EINVAL;
  *out = nullptr;
  if (T < 1 || !n_leaves || !n_patterns || !children || !roots || !blen || !pi || !Q || !rates ||
      !probs || !tips || !weights)
    return set_err(ctx, PHY_EINVAL, "aa_batch: null argument");
  if (!(R == 1 || R == 2 || R == 4)) return set_err(ctx, PHY_ERANGE, "aa_batch: n_rates must be 1, 2 or 4");
  if (!(waves == 1 || waves == 2 || waves == 4 || waves == 8))
    return set_err(ctx, PHY_ERANGE, "aa_batch: waves must be 1, 2, 4 or 8");
  phy_aa_batch* b = new phy_aa_batch();
  b->ctx = ctx;
  b->T = T;
  b->R = R;
  b->waves = waves;
  const int tile = 16 * waves;
  std::vector<int4> prog;
  std::vector<int64_t> prog_off, tips_off, pitch, w_off, pop_off, part_off, blen_off;
  std::vector<int32_t> nl, br_tree;
  std::vector<uint8_t> tipv;
  std::vector<uint32_t> wv;
  std::vector<double> eig, blv;
  std::vector<int2> items;
  int64_t ch_pos = 0, tip_pos = 0, pat_pos = 0, pop_pos = 0, part_pos = 0;
  for (int32_t t = 0; t < T; ++t) {
    const int32_t N = n_leaves[t];
    const int64_t P = n_patterns[t];
    if (N < 2 || P < 1) {
      delete b;
      return set_err(ctx, PHY_EINVAL, "aa_batch: every tree needs N >= 2 and P >= 1");
    }
    phy_topo* topo = nullptr;
    if (phy_topo_create(nullptr, N, children + ch_pos, roots[t], &topo) != PHY_OK) {
      delete b;
      return set_err(ctx, PHY_EINVAL, "aa_batch: malformed tree " + std::to_string(t));
    }
    b->depth = std::max(b->depth, topo->down_depth);
    prog_off.push_back((int64_t)prog.size());
    for (size_t k = 0; k < topo->down_prog.size(); k += 4)
      prog.push_back(make_int4(topo->down_prog[k], topo->down_prog[k + 1], topo->down_prog[k + 2],
                               topo->down_prog[k + 3]));
    phy_topo_destroy(topo);
    nl.push_back(N);
    const int64_t pp = (P + tile - 1) / tile * tile;
    pitch.push_back(pp);
    tips_off.push_back((int64_t)tipv.size());
    for (int32_t leaf = 0; leaf < N; ++leaf) {
      const uint8_t* row = tips + tip_pos + (size_t)leaf * P;
      tipv.insert(tipv.end(), row, row + P);
      tipv.insert(tipv.end(), (size_t)(pp - P), (uint8_t)255);  // padding: missing data
    }
    tip_pos += (int64_t)N * P;
    w_off.push_back((int64_t)wv.size());
    wv.insert(wv.end(), weights + pat_pos, weights + pat_pos + P);
    wv.insert(wv.end(), (size_t)(pp - P), 0u);
    pat_pos += P;
    // eigen-decomposition of Q_t on the host
    std::vector<double> U(KAA * KAA), lam(KAA), Ui(KAA * KAA);
    std::string err;
    if (!phy::eigen_reversible(KAA, Q + (size_t)t * KAA * KAA, U.data(), lam.data(), Ui.data(), &err)) {
      delete b;
      return set_err(ctx, PHY_ENUMERIC, "aa_batch: tree " + std::to_string(t) + ": " + err);
    }
    eig.insert(eig.end(), U.begin(), U.end());
    eig.insert(eig.end(), lam.begin(), lam.end());
    eig.insert(eig.end(), Ui.begin(), Ui.end());
    const int32_t M = 2 * N - 1;
    blen_off.push_back((int64_t)blv.size());
    blv.insert(blv.end(), blen + b->n_branches, blen + b->n_branches + M);
    for (int32_t v = 0; v < M; ++v) br_tree.push_back(t);
    b->n_branches += M;
    pop_off.push_back(pop_pos);
    pop_pos += (int64_t)M * aa_blocks(R) * OPB;
    part_off.push_back(part_pos);
    const int64_t tiles = pp / tile;
    part_pos += tiles * waves;
    for (int64_t k = 0; k < tiles; ++k) items.push_back(make_int2(t, (int)k));
    ch_pos += 2 * (int64_t)(N - 1);
    b->n_leaves.push_back(N);
    b->n_pat.push_back(P);
    b->pitch.push_back(pp);
    b->pattern_nodes += P * (N - 1);
  }
  part_off.push_back(part_pos);
  b->n_items = (int64_t)items.size();
  if (b->n_items > 0x7fffffff) {
    delete b;
    return set_err(ctx, PHY_ERANGE, "aa_batch: too many work items");
  }
  deal_items(nl, items, b->q_off);
  // static operand double buffer (2 nodes x 2 children) plus the dynamic
  // stack, within the device's LDS per workgroup
  int lds_max = 64 * 1024, dev = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
  const int lv = aa_register_levels(std::max(1, b->depth), waves == 8 ? 2 : 1);  // the larger stack of the two forms
  if (lds_bytes(waves, R, std::max(1, b->depth), lv) + (size_t)2 * 2 * aa_blocks(R) * OPB * sizeof(uint4) > (size_t)lds_max) {
    delete b;
    return set_err(ctx, PHY_ERANGE, "aa_batch: LDS stack too deep for this many waves per workgroup");
  }
  std::vector<double> pis(pi, pi + (size_t)T * KAA), prv(probs, probs + (size_t)T * R),
      rtv(rates, rates + (size_t)T * R);
  int rc = PHY_OK;
  if (!rc) rc = upload(b, &b->prog, prog);
  if (!rc) rc = upload(b, &b->prog_off, prog_off);
  if (!rc) rc = upload(b, &b->nl, nl);
  if (!rc) rc = upload(b, &b->tips, tipv);
  if (!rc) rc = upload(b, &b->tips_off, tips_off);
  if (!rc) rc = upload(b, &b->pitch_d, pitch);
  if (!rc) rc = upload(b, &b->wts, wv);
  if (!rc) rc = upload(b, &b->w_off, w_off);
  if (!rc) rc = upload(b, &b->pop_off, pop_off);
  if (!rc) rc = upload(b, &b->part_off, part_off);
  if (!rc) rc = upload(b, &b->pi, pis);
  if (!rc) rc = upload(b, &b->probs, prv);
  if (!rc) rc = upload(b, &b->rates, rtv);
  if (!rc) rc = upload(b, &b->eig, eig);
  if (!rc) rc = upload(b, &b->blen, blv);
  if (!rc) rc = upload(b, &b->blen_off, blen_off);
  if (!rc) rc = upload(b, &b->br_tree, br_tree);
  if (!rc) rc = upload(b, &b->items, items);
  if (!rc) rc = upload(b, &b->pops, std::vector<uint4>((size_t)pop_pos));
  if (!rc) rc = upload(b, &b->part, std::vector<double>((size_t)part_pos));
  if (!rc) rc = upload(b, &b->counter, std::vector<unsigned>(kQueues * kCounterPitch, 0u));
  if (rc) {
    phy_aa_batch_destroy(b);
    return rc;
  }
  *out = b;
  return PHY_OK;
}

void phy_aa_batch_destroy(phy_aa_batch* b) {
  if (!b) return;
  for (void* p : b->bufs) (void)hipFree(p);
  delete b;
}

int phy_aa_batch_info(const phy_aa_batch* b, int64_t* pattern_nodes, int64_t* n_items,
                      int32_t* stack_depth) {
  if (!b) return PHY_EINVAL;
  if (pattern_nodes) *pattern_nodes = b->pattern_nodes;
  if (n_items) *n_items = b->n_items;
  if (stack_depth) *stack_depth = b->depth;
  return PHY_OK;
}

int phy_aa_batch_run(phy_ctx* ctx, phy_aa_batch* b, double* d_lnl) {
  if (!ctx || !b || !d_lnl) return PHY_EINVAL;
  if (b->ctx != ctx) return set_err(ctx, PHY_EINVAL, "aa_batch: built on another context");
  // 1. P operands for every (tree, branch, rate)
  int n_cu = 256;
  (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, ctx->device);
  const int per = (int)std::min<int64_t>(kPopsPerBlock, 1 + b->n_branches / (4 * n_cu));
  const unsigned nwg = (unsigned)((b->n_branches + per - 1) / per);
  auto pops = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(nwg), dim3(64 * b->R), 0, ctx->stream, b->eig, b->rates, b->blen, b->blen_off,
                       b->br_tree, b->n_branches, per, b->pop_off, b->pops);
  };
  switch (b->R) {
    case 1: pops(k_aa_pops<1>); break;
    case 2: pops(k_aa_pops<2>); break;
    default: pops(k_aa_pops<4>); break;
  }
  PHY_LAUNCHED(ctx);
  // 2. the persistent pruning launch
  hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(kQueues), 0, ctx->stream, b->counter);
  PHY_LAUNCHED(ctx);
  int rc;
  switch (b->R) {
    case 1: rc = launch_w<1>(ctx, b); break;
    case 2: rc = launch_w<2>(ctx, b); break;
    default: rc = launch_w<4>(ctx, b); break;
  }
  if (rc) return rc;
  // 3. per-tree compensated sums
  hipLaunchKernelGGL(k_aa_reduce, dim3((unsigned)b->T), dim3(256), 0, ctx->stream, b->part, b->part_off, d_lnl);
  PHY_LAUNCHED(ctx);
  return PHY_OK;
}

}  // extern "C"
