// Grouped DeepSeek-V3 FP8 MoE for gfx950 (deepseek_v2_fp8_moe): router, grouped top-k, expert sort,
// per-token input quantization, two grouped 128x128-block-scaled FP8 GEMMs and a deterministic
// weighted combine, all on the caller's stream, scratch from the caller's workspace.
//
// Data flow for T tokens, S slots per token (topk routed + the shared expert), R = T * S rows:
//   router_kernel    fp32 partials over K ranges of x @ router^T                 (bf16 MFMA)
//   route_kernel     logits[T, Er] = bf16(sum of the partials); ids[T, S], weights[T, S]: sigmoid, grouped
//                    top-k, shared slot last
//   align_quant_kernel, two halves side by side:
//     sort           one workgroup: per-expert counts, the rows sorted by expert (stable only per
//                    expert, which nothing depends on), each row's position, and the tables of
//                    256-, 128- and 64-row blocks (expert, first row, rows) the GEMMs walk
//     quantization   x -> e4m3 per 1 x 128 at scale max(amax / 448, tiny) (a true division, as the
//                    checkpoint's FP8 scheme quantizes the linears' inputs), scales [D/128, T]
//   moe_gemm<GATEUP> per block class, per (block, 128 columns of the intermediate): rows gathered by token, gate and up
//                    weight rows interleaved per 16 so each lane holds both for the same columns;
//                    epilogue silu(gate) * up -> bf16 -> e4m3 per 1 x 128 (same division) into h
//   moe_gemm<DOWN>   per (block, 256 output columns): h rows in sorted order -> y (bf16, sorted)
//   combine_kernel   out[t] = bf16(sum over slots, in slot order, of weight * y[row of (t, slot)])
// The GEMMs are persistent (one 512-thread workgroup per CU walks the work items) and read the block
// count from device memory, so the whole pipeline runs without a host synchronization.
#include "common.h"

AKLR_SCALAR_FP32_BEGIN

namespace aklr {
namespace moe {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Row-block classes: an expert's rows split into full 256-row blocks and one last block for the
// remainder, of the smallest class that holds it (64, 128 or 256 rows). Every block streams the
// expert's weight tile once, so an expert costs ceil(rows / 256) weight reads -- the fewest for tiles
// of at most 256 rows -- at the price of some padded MFMA rows in the last block.
constexpr int kClasses = 3;
constexpr int kMinTM = 64;
__host__ __device__ constexpr int class_rows(int k) { return k == 0 ? 256 : (k == 1 ? 128 : 64); }
constexpr int kTN = 256;   // weight rows per GEMM tile
constexpr int kItemSteps = 16;  // K steps of a DOWN item of several tiles (its b_scale rows: 2 values a step)
constexpr int kMaxExperts = 2048;  // expert slots the align kernel's LDS holds
constexpr float kFp32Tiny = 1.17549435e-38f;

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// ---------------------------------------------------------------------------------------------
// router: fp32 partial logits part[ks][T][E] of x @ router^T over K ranges, V_MFMA_F32_16X16X32_BF16 with
// operands straight from global memory: lane (li, g) loads the 8 bf16 at k0 + 8g of its row. The MFMA
// pairs A's and B's lane groups the same way, so this assignment of k only has to match between them.
// A workgroup of 4 waves owns 16 * MT tokens x 16 * NT * (4 / KW) experts of one K range; with KW = 4 its
// waves take a quarter of the range each and meet in LDS, in wave order. route_kernel adds the ranges.
//
// Bound by load latency: a wave that walks all of K in one chain of 224 load-to-MFMA round trips took
// 94 us at 4 tokens x 256 experts x 7168 (3.7 MB), and 89 at 128. Splitting K over waves and workgroups
// (plan_router) leaves each wave a few batches of UK steps, the next batch's loads in flight under the
// current one's MFMAs: 4.9 us and 9.4.
template <int MT, int NT, int KW, int UK>
__global__ __launch_bounds__(256) void router_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ wr,
                                                     float* __restrict__ part, int T, int E, int D, int ks_count,
                                                     int steps_per_wave) {
  constexpr int EW = 4 / KW;
  __shared__ f32x4 red[KW > 1 ? KW - 1 : 1][MT * NT][64];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kw = KW > 1 ? w : 0, ew = KW > 1 ? 0 : w;
  const int tiles_e = (E + 16 * NT * EW - 1) / (16 * NT * EW);
  const int ks = blockIdx.x % ks_count, tile = blockIdx.x / ks_count;
  const int t0 = (tile / tiles_e) * 16 * MT, e0 = ((tile % tiles_e) * EW + ew) * 16 * NT;
  const int li = lane & 15, g = lane >> 4;
  const int s_begin = (ks * KW + kw) * steps_per_wave, s_end = min(D / 32, s_begin + steps_per_wave);
  // rows past T and experts past E read the out-of-range offset (zeros)
  const rsrc_t xr = make_rsrc(x + (int64_t)t0 * D, (uint32_t)((int64_t)min(16 * MT, T - t0) * D * 2));
  const rsrc_t br = make_rsrc(wr + (int64_t)min(e0, E - 1) * D, (uint32_t)((int64_t)max(0, min(16 * NT, E - e0)) * D * 2));
  uint32_t x_off[MT], b_off[NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    x_off[mt] = t0 + mt * 16 + li < T ? (uint32_t)(((mt * 16 + li) * D + 8 * g) * 2) : kOobOffset;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    b_off[nt] = e0 + nt * 16 + li < E ? (uint32_t)(((nt * 16 + li) * D + 8 * g) * 2) : kOobOffset;
  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 xa[2][UK][MT], xb[2][UK][NT];
  auto load = [&](int buf, int s0) {
#pragma unroll
    for (int u = 0; u < UK; ++u) {
      const bool on = s0 + u < s_end;
      const uint32_t kb = (uint32_t)(s0 + u) * 64;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xa[buf][u][mt] = buf_ld16(xr, on ? x_off[mt] + kb : kOobOffset);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) xb[buf][u][nt] = buf_ld16(br, on ? b_off[nt] + kb : kOobOffset);
    }
  };
  auto fma = [&](int buf) {
#pragma unroll
    for (int u = 0; u < UK; ++u)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xa[buf][u][mt]),
                                                                __builtin_bit_cast(bf16x8, xb[buf][u][nt]),
                                                                acc[mt][nt], 0, 0, 0);
  };
  load(0, s_begin);
  for (int s0 = s_begin; s0 < s_end; s0 += 2 * UK) {
    load(1, s0 + UK);
    fma(0);
    load(0, s0 + 2 * UK);
    fma(1);
  }
  if constexpr (KW > 1) {
    if (w > 0) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) red[w - 1][mt * NT + nt][lane] = acc[mt][nt];
    }
    __syncthreads();
    if (w > 0) return;
#pragma unroll
    for (int v = 0; v < KW - 1; ++v)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] += red[v][mt * NT + nt][lane];
  }
  // lane holds tokens 4g + r, expert li of each tile
  float* const out = part + (int64_t)ks * T * E;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int e = e0 + nt * 16 + li;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = t0 + mt * 16 + 4 * g + r;
        if (t < T && e < E) out[(int64_t)t * E + e] = acc[mt][nt][r];
      }
    }
}

// Router plan. One 16 x 16 tile a workgroup up to 16 tokens (all waves on K); 32 x 32 tiles, which halve the
// operand reads per product, up to 1023 tokens or where the experts do not fill four waves; 64 x 256 tiles
// (a wave per 64 experts) from 1024 tokens, where re-reading the weights per token tile is what counts.
// K is cut until about 512 workgroups run, into at most 16 ranges (route_kernel reads one partial of each).
struct RouterPlan {
  int shape;  // 0: 16 x 16, 1: 32 x 32, 2: 64 x 256
  int ranges, steps_per_wave;
  int64_t groups;
};

static RouterPlan plan_router(int64_t T, int64_t E, int64_t D) {
  RouterPlan p;
  p.shape = T <= 16 ? 0 : ((T < 1024 || E <= 64) ? 1 : 2);
  const int64_t tm = p.shape == 0 ? 16 : (p.shape == 1 ? 32 : 64), tn = p.shape == 0 ? 16 : (p.shape == 1 ? 32 : 256);
  const int64_t tiles = ((T + tm - 1) / tm) * ((E + tn - 1) / tn);
  const int64_t waves = p.shape == 2 ? 1 : 4, steps = D / 32;
  int64_t r = 512 / tiles;
  r = r < 1 ? 1 : (r > 16 ? 16 : r);
  p.steps_per_wave = (int)((steps + r * waves - 1) / (r * waves));
  p.ranges = (int)((steps + p.steps_per_wave * waves - 1) / (p.steps_per_wave * waves));
  p.groups = tiles * p.ranges;
  return p;
}

// fp32 partials the scratch of a T-token call holds: at least ranges * T * E of every plan for up to T tokens,
// so that the size never falls as T grows (ranges does) and a buffer made for the largest batch serves the
// smaller ones. A plan has one range, T * E partials, or at most 16 with at most 512 workgroups, each a tile.
static int64_t router_partials(int64_t T, int64_t E) {
  const auto cut = [E](int64_t t, int64_t tm, int64_t tn) {
    const int64_t most = 16 * ((t + tm - 1) / tm * tm) * E;
    return most < 512 * tm * tn ? most : 512 * tm * tn;
  };
  int64_t n = T * E;
  const auto cover = [&n](int64_t v) { n = v > n ? v : n; };
  const bool wide = T >= 1024 && E > 64;
  cover(cut(T < 16 ? T : 16, 16, 16));
  if (T > 16) cover(cut(wide ? 1023 : T, 32, 32));
  if (wide) cover(cut(T, 64, 256));
  return n;
}

// ---------------------------------------------------------------------------------------------
// route: one wave per token. (value, index) pairs compare by value, then the lower index first; a NaN is
// never picked. As one 64-bit key: the value's bits in an unsigned order, then the inverted index; 0 marks
// no candidate. The wave's maximum takes four DPP moves and two lane swaps, no LDS permutes (with 12
// maxima a token in 12 permutes each, the kernel took 15.5 us at 4 tokens of 256 experts in 8 groups and 47
// at 4096 ungrouped; now 6.9, the router's partials included, and 10.2).
constexpr int kNoIndex = 1 << 30;

__device__ __forceinline__ uint64_t rank_key(float v, int i) {
  if (!(v == v)) return 0;
  const uint32_t u = __float_as_uint(v + 0.0f);  // -0 counts as 0
  return ((uint64_t)(u ^ ((u & 0x80000000u) ? 0xFFFFFFFFu : 0x80000000u)) << 32) | (uint32_t)~i;
}
__device__ __forceinline__ int key_index(uint64_t k) { return k == 0 ? kNoIndex : (int)~(uint32_t)k; }

template <int CTRL>
__device__ __forceinline__ uint64_t dpp_max(uint64_t k) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)k, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(k >> 32), CTRL, 0xF, 0xF, false);
  const uint64_t o = ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
  return o > k ? o : k;
}

__device__ __forceinline__ uint64_t wave_max(uint64_t k) {
  k = dpp_max<0xB1>(k);   // quad_perm [1,0,3,2]
  k = dpp_max<0x4E>(k);   // quad_perm [2,3,0,1]
  k = dpp_max<0x141>(k);  // row_half_mirror: the other quad of the 8
  k = dpp_max<0x140>(k);  // row_mirror: the other 8 of the 16
  {
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)k, (uint32_t)k, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(k >> 32), (uint32_t)(k >> 32), false, false);
    const uint64_t a = ((uint64_t)hi[0] << 32) | lo[0], b = ((uint64_t)hi[1] << 32) | lo[1];
    k = a > b ? a : b;
  }
  const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)k, (uint32_t)k, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)(k >> 32), (uint32_t)(k >> 32), false, false);
  const uint64_t a = ((uint64_t)hi[0] << 32) | lo[0], b = ((uint64_t)hi[1] << 32) | lo[1];
  return a > b ? a : b;
}

// Logits: bf16 [T, E], or fp32 partials [ranges][T, E] whose sum, in range order, is rounded to bf16.
// PER_LANE * 64 experts at most (4: up to 256, 16: up to 1024); lane l holds experts l, l + 64, ...
template <bool PART, int PER_LANE>
__global__ __launch_bounds__(64) void route_kernel(const uint16_t* __restrict__ logits, const float* __restrict__ part,
                                                   int ranges, const uint16_t* __restrict__ bias, int T, int E, int G,
                                                   int topk, int topk_group, int renormalize, float scale, int shared,
                                                   int32_t* __restrict__ ids, float* __restrict__ weights) {
  __shared__ float sv[64 * PER_LANE];  // unbiased scores
  __shared__ float sb[64 * PER_LANE];  // biased scores
  const int t = blockIdx.x;
  const int lane = threadIdx.x;
  const int per = E / G;
  float x[PER_LANE], bs[PER_LANE];
#pragma unroll
  for (int j = 0; j < PER_LANE; ++j) {
    const int i = min(lane + 64 * j, E - 1);
    x[j] = PART ? part[(int64_t)t * E + i] : bf16_to_f32(logits[(int64_t)t * E + i]);
    bs[j] = bf16_to_f32(bias[i]);
  }
  if constexpr (PART) {
    // the partials come from other XCDs' writes, a long way off: kRouteBatch ranges' loads at a time
    constexpr int kRouteBatch = PER_LANE == 4 ? 15 : 5;
    for (int k0 = 1; k0 < ranges; k0 += kRouteBatch) {
      float v[kRouteBatch][PER_LANE];
#pragma unroll
      for (int k = 0; k < kRouteBatch; ++k)
#pragma unroll
        for (int j = 0; j < PER_LANE; ++j)
          v[k][j] = part[((int64_t)min(k0 + k, ranges - 1) * T + t) * E + min(lane + 64 * j, E - 1)];
#pragma unroll
      for (int k = 0; k < kRouteBatch; ++k)
#pragma unroll
        for (int j = 0; j < PER_LANE; ++j) x[j] += k0 + k < ranges ? v[k][j] : 0.0f;
    }
  }
  // straight through: lanes past E rank expert E - 1 again and drop it. With a branch a slot, the compiler kept a
  // copy of every array per branch at 16 slots (494 VGPRs, one wave a SIMD): 4096 tokens x 512 experts took 55 us,
  // now 24, 16384 200, now 72.
  uint64_t key[PER_LANE];
#pragma unroll
  for (int j = 0; j < PER_LANE; ++j) {
    const int i = lane + 64 * j;
    const float lx = PART ? __uint_as_float(f32_to_bf16_bits(x[j]) << 16) : x[j];
    const float v = 1.0f / (1.0f + expf(-lx));
    const float b = v + bs[j];
    const uint64_t k = rank_key(b, i);
    key[j] = i < E ? k : 0;
    sv[i] = v;
    sb[i] = b;
  }
  __syncthreads();
  uint64_t kept = ~0ull;
  if (G > 1 || topk_group != 1) {
    // group score: the sum of its two best biased scores, found by nsub lanes a group (a power of two)
    int nsub = 64;
    while (nsub * G > 64) nsub >>= 1;
    const int gi = lane / nsub, sub = lane % nsub;
    float m1 = -INFINITY, m2 = -INFINITY;
    if (gi < G)
      for (int i = gi * per + sub; i < gi * per + per; i += nsub) {
        const float v = sb[i];
        if (v > m1) {
          m2 = m1;
          m1 = v;
        } else if (v > m2) {
          m2 = v;
        }
      }
    for (int off = nsub >> 1; off >= 1; off >>= 1) {
      const float o1 = __shfl_xor(m1, off), o2 = __shfl_xor(m2, off);
      m2 = fmaxf(fminf(m1, o1), fmaxf(m2, o2));
      m1 = fmaxf(m1, o1);
    }
    // keep the topk_group best groups (G <= 64); sub-lane 0 speaks for its group
    uint64_t gk = (gi < G && sub == 0) ? rank_key(m1 + m2, gi) : 0;
    kept = 0;
    for (int r = 0; r < topk_group; ++r) {
      const int i = key_index(wave_max(gk));
      if (gk != 0 && i == gi) gk = 0;
      kept |= 1ull << (i & 63);
    }
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
      const int e = min(lane + 64 * j, E - 1);
      if (!(kept >> (e / per) & 1ull)) key[j] = 0;
    }
  }
  // the topk best biased scores among the kept groups' experts
  float wsum = 0.0f;
  int my_id = 0;
  float my_v = 0.0f;
  for (int r = 0; r < topk; ++r) {
    uint64_t best = key[0];
#pragma unroll
    for (int j = 1; j < PER_LANE; ++j) best = key[j] > best ? key[j] : best;
    best = wave_max(best);
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) key[j] = key[j] == best ? 0 : key[j];
    const int i = key_index(best);
    const float sc = i == kNoIndex ? 0.0f : sv[i];
    wsum += sc;
    if (lane == r) {
      my_id = i;
      my_v = sc;
    }
  }
  const int S = topk + (shared ? 1 : 0);
  if (lane < topk) {
    const float w = renormalize ? my_v / wsum : my_v;
    ids[(int64_t)t * S + lane] = my_id;
    weights[(int64_t)t * S + lane] = w * scale;
  }
  if (shared && lane == 0) {
    ids[(int64_t)t * S + topk] = E;
    weights[(int64_t)t * S + topk] = 1.0f;
  }
}

// ---------------------------------------------------------------------------------------------
// align (the sort): one 1024-thread workgroup. Entries whose expert is out of [0, E) get row -1 (ignored).
__device__ int block_exclusive_scan(int v, int* wsum, int* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(incl, off);
    if (lane >= off) incl += y;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    int acc = 0;
    for (int i = 0; i < 16; ++i) {
      const int s = wsum[i];
      wsum[i] = acc;
      acc += s;
    }
    *total = acc;
  }
  __syncthreads();
  const int r = wsum[w] + incl - v;
  __syncthreads();
  return r;
}

// Block table: for each class k, expert[k][i], first row[k][i] and rows[k][i] of its blocks, cap
// entries per class, and count[k].
struct BlockTable {
  int32_t* expert;
  int32_t* row;
  int32_t* rows;
  int32_t* count;
  int cap;
};

__device__ __forceinline__ int class_blocks(int c, int k) {
  const int full = c / 256, rem = c - 256 * full;
  const int last = rem == 0 ? -1 : (rem > 128 ? 0 : (rem > 64 ? 1 : 2));  // class of the remainder block
  return (k == 0 ? full : 0) + (k == last ? 1 : 0);
}

struct AlignSmem {
  int cnt[kMaxExperts];
  int off[kMaxExperts];
  int boff[kClasses][kMaxExperts];
  int wsum[16];
  int total;
};

// kAlignBatch ids a thread are loaded before the first is used: the two walks over the R slots are chains
// of load, LDS atomic and store, and one id at a time they took 54 us at 36864 slots (46 now, with the
// quantization of 4096 rows in the same launch).
constexpr int kAlignBatch = 8;

__device__ void align_block(AlignSmem& sm, const int32_t* __restrict__ ids, int R, int S, int E,
                            int32_t* __restrict__ row_of, int32_t* __restrict__ sorted_tok, const BlockTable& bt,
                            int* __restrict__ tickets) {
  const int tid = threadIdx.x;
  if (tid < 2) tickets[tid] = 0;  // the grouped GEMMs' work-item counters (gate-up, down)
  for (int e = tid; e < kMaxExperts; e += 1024) sm.cnt[e] = 0;
  __syncthreads();
  for (int i0 = tid; i0 < R; i0 += 1024 * kAlignBatch) {
    int e[kAlignBatch], r[kAlignBatch];
#pragma unroll
    for (int j = 0; j < kAlignBatch; ++j) e[j] = i0 + 1024 * j < R ? ids[i0 + 1024 * j] : -1;
#pragma unroll
    for (int j = 0; j < kAlignBatch; ++j) r[j] = (e[j] >= 0 && e[j] < E) ? atomicAdd(&sm.cnt[e[j]], 1) : -1;
#pragma unroll
    for (int j = 0; j < kAlignBatch; ++j)
      if (i0 + 1024 * j < R) row_of[i0 + 1024 * j] = r[j];
  }
  __syncthreads();
  // two experts per thread: exclusive prefix of rows, then of each class's blocks
  const int e0 = 2 * tid, e1 = 2 * tid + 1;
  const int c0 = e0 < E ? sm.cnt[e0] : 0, c1 = e1 < E ? sm.cnt[e1] : 0;
  const int o = block_exclusive_scan(c0 + c1, sm.wsum, &sm.total);
  if (e0 < kMaxExperts) sm.off[e0] = o;
  if (e1 < kMaxExperts) sm.off[e1] = o + c0;
#pragma unroll
  for (int k = 0; k < kClasses; ++k) {
    const int b0 = class_blocks(c0, k), b1 = class_blocks(c1, k);
    const int bo = block_exclusive_scan(b0 + b1, sm.wsum, &sm.total);
    if (e0 < kMaxExperts) sm.boff[k][e0] = bo;
    if (e1 < kMaxExperts) sm.boff[k][e1] = bo + b0;
    if (tid == 0) bt.count[k] = sm.total;
  }
  __syncthreads();
  for (int i0 = tid; i0 < R; i0 += 1024 * kAlignBatch) {
    int e[kAlignBatch], r[kAlignBatch];
#pragma unroll
    for (int j = 0; j < kAlignBatch; ++j) {
      const int i = i0 + 1024 * j;
      e[j] = i < R ? ids[i] : -1;
      r[j] = i < R ? row_of[i] : -1;  // this thread's own store
    }
#pragma unroll
    for (int j = 0; j < kAlignBatch; ++j) {
      const int i = i0 + 1024 * j;
      if (e[j] < 0 || e[j] >= E) continue;
      const int pos = sm.off[e[j]] + r[j];
      row_of[i] = pos;
      sorted_tok[pos] = i / S;
    }
  }
  for (int e = tid; e < E; e += 1024) {
    const int c = sm.cnt[e];
    int row = sm.off[e], left = c;
#pragma unroll
    for (int k = 0; k < kClasses; ++k) {
      const int nb = class_blocks(c, k);
      for (int j = 0; j < nb; ++j) {
        const int idx = k * bt.cap + sm.boff[k][e] + j;
        const int n = min(class_rows(k), left);
        bt.expert[idx] = e;
        bt.row[idx] = row;
        bt.rows[idx] = n;
        row += n;
        left -= n;
      }
    }
  }
}

// quant: 16 lanes per 1 x 128 group, 8 values each. scale = max(amax / 448, tiny); code =
// e4m3(x / scale), both true IEEE divisions.
__device__ void quant_div_block(int block, const uint16_t* __restrict__ x, int T, int D, uint8_t* __restrict__ q,
                                float* __restrict__ s) {
  const int groups = D / 128;
  const int gid = block * 64 + (threadIdx.x >> 4);
  if (gid >= T * groups) return;
  const int t = gid / groups, grp = gid - t * groups;
  const int sub = threadIdx.x & 15;
  const int64_t base = (int64_t)t * D + grp * 128 + sub * 8;
  const u32x4 v = ld16(x + base);
  float f[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = bf16_lo(v[i]);
    f[2 * i + 1] = bf16_hi(v[i]);
  }
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(f[i]));
  amax = fmaxf(amax, dpp_f32<0xB1>(amax));   // the group's 16 lanes are one DPP row: quad_perm [1,0,3,2]
  amax = fmaxf(amax, dpp_f32<0x4E>(amax));   // quad_perm [2,3,0,1]
  amax = fmaxf(amax, dpp_f32<0x141>(amax));  // row_half_mirror
  amax = fmaxf(amax, dpp_f32<0x140>(amax));  // row_mirror
  const float sc = fmaxf(__fdiv_rn(amax, 448.0f), kFp32Tiny);
  float c[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) c[i] = fminf(fmaxf(__fdiv_rn(f[i], sc), -448.0f), 448.0f);
  u32x2 out;
  out[0] = pack4_e4m3(c[0], c[1], c[2], c[3]);
  out[1] = pack4_e4m3(c[4], c[5], c[6], c[7]);
  *reinterpret_cast<u32x2*>(q + base) = out;
  if (sub == 0) s[(int64_t)grp * T + t] = sc;
}

// One launch for the expert sort (workgroup 0) and the input quantization (the others): neither needs the
// other, so the sort's single workgroup runs beside the quantization instead of before it (5.4 + 5.2 us
// apart at 4 tokens, 53.8 + 26.0 at 4096; 6.3 and 45.9 together).
__global__ __launch_bounds__(1024) void align_quant_kernel(const int32_t* __restrict__ ids, int R, int S, int E,
                                                           int32_t* __restrict__ row_of,
                                                           int32_t* __restrict__ sorted_tok, BlockTable bt,
                                                           int* __restrict__ tickets, const uint16_t* __restrict__ x,
                                                           int T, int D, uint8_t* __restrict__ q,
                                                           float* __restrict__ s) {
  __shared__ AlignSmem sm;
  if (blockIdx.x == 0)
    align_block(sm, ids, R, S, E, row_of, sorted_tok, bt, tickets);
  else
    quant_div_block((int)blockIdx.x - 1, x, T, D, q, s);
}

// ---------------------------------------------------------------------------------------------
// grouped GEMM
enum { kGateUp = 0, kDown = 1 };

struct MoeGemmArgs {
  const uint8_t* a;          // GATEUP: x codes [T, K]; DOWN: h codes [R, K]
  const float* sa;           // a scales, [K/128, sa_ld]
  int64_t sa_ld;             // T (GATEUP) or R (DOWN)
  const int32_t* sorted_tok; // GATEUP: sorted row -> token
  const uint8_t* b;          // expert weights, [experts, N, K] row-major or 16x16-preshuffled per expert
  int64_t b_stride;          // bytes per expert
  const float* sb;           // [experts, ceil(N/128), K/128]
  int64_t sb_stride;         // floats per expert
  const int32_t* blk_expert;  // block table of class 0; class k at + k * blk_cap
  const int32_t* blk_row;
  const int32_t* blk_rows;
  const int32_t* nblk;        // blocks per class
  int blk_cap;
  int* tickets;               // work-item counter, zero at launch (align_block clears it)
  int K, N, I;               // reduction length, weight rows, intermediate size
  int tiles_n;               // GATEUP: I / 128; DOWN: ceil(N / 256)
  uint8_t* hq;               // GATEUP out: [R, I] codes
  float* hs;                 // GATEUP out: [I/128, R] scales
  int64_t R;
  uint16_t* y;               // DOWN out: [R, N] bf16
};

__device__ __forceinline__ float silu(float g) { return g / (1.0f + expf(-g)); }

__device__ __forceinline__ float round_bf16(float v) { return __uint_as_float(f32_to_bf16_bits(v) << 16); }

// One work item: a TM-row block (class TM of the block table) x 256 weight rows; 8 waves in 2 (m) x 4
// (n), each TM/2 rows x 64 weight rows (MT = TM/32, NT = 4 tiles of 16x16); K steps of 128 through a
// direct-to-LDS ring of as many stages as LDS holds (3 for TM <= 128, 2 for 256), with the swizzled
// LDS tiles, load schedule and fold of the dense LDS kernel. GATEUP orders the tile's 256 weight rows
// as (gate 16, up 16) pairs over 128 intermediate columns, so tiles nt = 2q and 2q + 1 of a wave are
// the gate and the up of the same 16 columns. LDS comes from the caller's buffer, as MoeSmem lays it out.
//
// DOWN items of the 64- and 128-row classes take `tiles` consecutive weight tiles from pn on, in one stream of
// tiles * KB steps through the ring (the 256-row class, whose accumulators leave no registers for it, one): a
// tile's results are stored between two steps while the next tile's stages are in flight. On short K an item of
// one tile is mostly its own start (a ticket, the block's entry, the b_scale rows and the first stages, one after
// the other): 128 tokens on 256 experts of 7168 x 256 (2 K blocks, 28 tiles) took 100 us for 460 MB of weights,
// and 75 in items of 6 tiles. From 16 K blocks on items keep one tile (32 steps an item instead of 16: 4096
// tokens at 2048, 3420 -> 3470 us a call, the last items end too far apart).
template <int TM>
struct MoeSmem {
  static constexpr int S = TM == 256 ? 2 : 3, MT = TM / 32;
  static constexpr int kStageA = TM * 128, kStageB = kTN * 128;
  static constexpr int kA = 0, kB = kA + S * kStageA, kS = kB + S * kStageB, kDummy = kS + S * TM * 4,
                       kSB = kDummy + 8 * 64 * 4, kAmax = kSB + 2 * 512 * 4, kBytes = kAmax + 2 * MT * 16 * 4 * 4;
};
constexpr int kMoeSmemBytes =
    MoeSmem<256>::kBytes > MoeSmem<128>::kBytes
        ? (MoeSmem<256>::kBytes > MoeSmem<64>::kBytes ? MoeSmem<256>::kBytes : MoeSmem<64>::kBytes)
        : (MoeSmem<128>::kBytes > MoeSmem<64>::kBytes ? MoeSmem<128>::kBytes : MoeSmem<64>::kBytes);
static_assert(kMoeSmemBytes <= 160 * 1024, "LDS");

template <int MODE, bool PRE, int TM>
__device__ __forceinline__ void moe_item(const MoeGemmArgs& p, uint8_t* smem, int cls, int blk, int pn, int tiles) {
  using L = MoeSmem<TM>;
  constexpr int TN = kTN, S = L::S;
  constexpr int MT = TM / 32, NT = TN / 64;
  constexpr int AI = TM / 64, BI = TN / 64;
  constexpr int kLoads = AI + BI + 1;
  constexpr int kScaleWaves = TM / 64;
  constexpr int kStageA = L::kStageA, kStageB = L::kStageB;
  constexpr bool kMany = MODE == kDown && TM < 256;  // several tiles an item
  uint8_t* sA = smem + L::kA;
  uint8_t* sB = smem + L::kB;
  float* sS = reinterpret_cast<float*>(smem + L::kS);
  float* sDummy = reinterpret_cast<float*>(smem + L::kDummy);
  float* sSB = reinterpret_cast<float*>(smem + L::kSB);
  float (*sAmax)[MT][16][4] = reinterpret_cast<float (*)[MT][16][4]>(smem + L::kAmax);

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int wm = w >> 2, wn = w & 3;
  const int lr = lane >> 3, lp = lane & 7;
  const int c = lp ^ lr;
  const int KB = p.K >> 7;
  const int64_t kt32 = p.K >> 5;
  {
    const int bi = cls * p.blk_cap + blk;
    // in SGPRs: the loads' descriptors are made from them
    const int e = __builtin_amdgcn_readfirstlane(p.blk_expert[bi]), row0 = __builtin_amdgcn_readfirstlane(p.blk_row[bi]),
              rows = __builtin_amdgcn_readfirstlane(p.blk_rows[bi]);

    // A: wave w moves tile rows [w*TM/8, (w+1)*TM/8) in slabs of 8; waves below kScaleWaves also move
    // a_scale rows [64w, 64w + 64), the others an empty load (same count per wave).
    const i32x4 ars = make_rsrc_words(p.a, (uint32_t)(p.sa_ld * p.K));  // A has sa_ld rows of K codes
    uint32_t a_off[AI];
#pragma unroll
    for (int j = 0; j < AI; ++j) {
      const int ar = w * (TM / 8) + j * 8 + lr;
      int64_t arow = 0;
      if (ar < rows) arow = MODE == kGateUp ? p.sorted_tok[row0 + ar] : row0 + ar;
      a_off[j] = ar < rows ? (uint32_t)(arow * p.K + c * 16) : kOobOffset;
    }
    const bool scale_wave = w < kScaleWaves;
    const int sr = w * 64 + lane;
    int64_t srow = 0;
    if (scale_wave && sr < rows) srow = MODE == kGateUp ? p.sorted_tok[row0 + sr] : row0 + sr;
    const i32x4 sars = make_rsrc_words(p.sa, (uint32_t)((int64_t)KB * p.sa_ld * 4));
    const uint32_t sa_off = (scale_wave && sr < rows) ? (uint32_t)(srow * 4) : kOobOffset;
    const uint32_t sa_kstep = (uint32_t)(p.sa_ld * 4);
    // B: this expert's weight; wave w moves tile rows [32w, 32w + 32) in 4 slabs of 8.
    const i32x4 brs = make_rsrc_words(p.b + (int64_t)e * p.b_stride, (uint32_t)p.b_stride);
    uint32_t b_off[BI];
#pragma unroll
    for (int j = 0; j < BI; ++j) {
      const int rr = w * 32 + j * 8 + lr;
      int wrow;
      if (MODE == kGateUp) {
        const int blk16 = rr >> 4;
        wrow = ((blk16 & 1) ? p.I : 0) + pn * 128 + (blk16 >> 1) * 16 + (rr & 15);
      } else {
        wrow = pn * TN + rr;
      }
      if (wrow >= p.N)
        b_off[j] = kOobOffset;
      else if (PRE)
        b_off[j] = (uint32_t)(((int64_t)(wrow >> 4) * kt32 + (c >> 1)) * 512 + (c & 1) * 256 + (wrow & 15) * 16);
      else
        b_off[j] = (uint32_t)((int64_t)wrow * p.K + c * 16);
    }
    const uint32_t lds_a = lds_addr(&sA[w * (TM / 8) * 128]), lds_b = lds_addr(&sB[w * 32 * 128]);
    const uint32_t lds_s = scale_wave ? lds_addr(&sS[w * 64]) : lds_addr(&sDummy[w * 64]);
    const uint32_t lds_s_step = scale_wave ? TM * 4 : 0;
    // the next stage to load: K block ikb of the item's tile itile (rows past N lie past the descriptor)
    int ikb = 0, itile = 0;
    const int n_tiles = kMany ? tiles : 1;
    auto issue = [&](int st) {
      const int kb = ikb;
      const bool on = itile < n_tiles;
      const uint32_t ak = (uint32_t)kb * 128u;
      const uint32_t bk = (PRE ? (uint32_t)kb * 2048u : (uint32_t)kb * 128u) + (kMany ? (uint32_t)itile * (uint32_t)(TN * p.K) : 0u);
#pragma unroll
      for (int j = 0; j < AI; ++j)
        lds_dma16(ars, lds_a + st * kStageA + j * 1024, on && a_off[j] != kOobOffset ? a_off[j] + ak : kOobOffset);
#pragma unroll
      for (int j = 0; j < BI; ++j)
        lds_dma16(brs, lds_b + st * kStageB + j * 1024, on && b_off[j] != kOobOffset ? b_off[j] + bk : kOobOffset);
      lds_dma4(sars, lds_s + st * lds_s_step, on && sa_off != kOobOffset ? sa_off + (uint32_t)kb * sa_kstep : kOobOffset);
      if (++ikb == KB) {
        ikb = 0;
        ++itile;
      }
    };

    // b_scale rows of the tile over K: GATEUP gate block pn and up block I/128 + pn; DOWN the
    // tiles' two 128-row blocks each, tile after tile (they are consecutive rows).
    {
      const float* sbe = p.sb + (int64_t)e * p.sb_stride;
      if (MODE == kGateUp) {
        for (int i = threadIdx.x; i < 2 * KB; i += 512)
          sSB[i] = sbe[(int64_t)(i >= KB ? (p.I >> 7) + pn : pn) * KB + (i >= KB ? i - KB : i)];
      } else {
        const int last = ((p.N - 1) >> 7) * KB + KB - 1 - 2 * pn * KB;  // the expert's last value, from the first row
        for (int i = threadIdx.x; i < 2 * KB * n_tiles; i += 512) sSB[i] = sbe[(int64_t)2 * pn * KB + min(i, last)];
      }
    }

    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int swz_lo = (g ^ (li & 7)) << 4, swz_hi = ((4 + g) ^ (li & 7)) << 4;
    const int a_row = (wm * (TM / 2) + li) * 128, b_row = (wn * 64 + li) * 128;
    // The dense LDS kernel's step (gemm_a8w8.hip): the smaller fragment set held, the other streamed
    // one tile ahead, and each MFMA's fold kLag MFMAs after it (bitwise the same sums).
    constexpr int kLag = 3, kT = MT * NT;
    constexpr bool kHoldA = MT <= NT;
    constexpr int kHeld = kHoldA ? MT : NT, kStreamed = kHoldA ? NT : MT;
    auto tmt = [](int t) { return kHoldA ? t % MT : t / NT; };
    auto tnt = [](int t) { return kHoldA ? t / MT : t % NT; };
    f32x4 pend[kLag];
    float pend_s[kLag];
#pragma unroll
    for (int j = 0; j < kLag; ++j) {
      pend[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      pend_s[j] = 0.f;
    }
    auto compute = [&](int kb, int tile, int st) {
      const uint8_t* A = sA + st * kStageA;
      const uint8_t* B = sB + st * kStageB;
      const float* SA = sS + st * TM + wm * (TM / 2) + li;
      float sbv[2];
      if (MODE == kGateUp) {
        sbv[0] = sSB[kb];
        sbv[1] = sSB[KB + kb];
      } else {
        sbv[0] = sbv[1] = sSB[(kMany ? 2 * tile + (wn >> 1) : wn >> 1) * KB + kb];
      }
      auto read_a = [&](int mt) {
        return cat(*reinterpret_cast<const u32x4*>(A + a_row + swz_lo + mt * 2048),
                   *reinterpret_cast<const u32x4*>(A + a_row + swz_hi + mt * 2048));
      };
      auto read_b = [&](int nt) {
        return cat(*reinterpret_cast<const u32x4*>(B + b_row + swz_lo + nt * 2048),
                   *reinterpret_cast<const u32x4*>(B + b_row + swz_hi + nt * 2048));
      };
      i32x8 held[kHeld];
#pragma unroll
      for (int i = 0; i < kHeld; ++i) held[i] = kHoldA ? read_a(i) : read_b(i);
      float s0[MT], s1[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const float sa = SA[mt * 16];
        s0[mt] = sa * sbv[0];
        s1[mt] = sa * sbv[1];
      }
      i32x8 cur, nxt = kHoldA ? read_b(0) : read_a(0);
      f32x4 part[kT];
      float sc[kT];
#pragma unroll
      for (int t = 0; t < kT; ++t) {
        const int mt = tmt(t), nt = tnt(t);
        const int si = t / kHeld, hi = t % kHeld;
        if (hi == 0) {
          cur = nxt;
          if (si + 1 < kStreamed) nxt = kHoldA ? read_b(si + 1) : read_a(si + 1);
        }
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
        // lane: row li, columns 4g..4g+3 (the weight is the first operand)
        part[t] = kHoldA ? mfma16x128<0>(cur, held[hi], z) : mfma16x128<0>(held[hi], cur, z);
        sc[t] = (nt & 1) ? s1[mt] : s0[mt];
        if (t >= kLag) {
          const int u = t - kLag;
          asm volatile("" : "+v"(part[u]) : "v"(part[t]));
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[tmt(u)][tnt(u)][r] = fmaf(part[u][r], sc[u], acc[tmt(u)][tnt(u)][r]);
        } else {
          const int u = kT - kLag + t;
          asm volatile("" : "+v"(pend[t]) : "v"(part[t]));
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[tmt(u)][tnt(u)][r] = fmaf(pend[t][r], pend_s[t], acc[tmt(u)][tnt(u)][r]);
        }
      }
#pragma unroll
      for (int j = 0; j < kLag; ++j) {
        pend[j] = part[kT - kLag + j];
        pend_s[j] = sc[kT - kLag + j];
      }
    };

    // the last folds of a tile, then (DOWN) y rows in sorted order, bf16; lane pairs swap halves for 16-byte
    // stores (see the dense kernel)
    auto finish_folds = [&]() {
#pragma unroll
      for (int j = 0; j < kLag; ++j) {
        const int u = kT - kLag + j;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[tmt(u)][tnt(u)][r] = fmaf(pend[j][r], pend_s[j], acc[tmt(u)][tnt(u)][r]);
      }
    };
    auto store_y = [&](int tile) {
      const int col_s = (pn + tile) * TN + wn * 64 + (g & 1) * 16 + (g >> 1) * 8;
#pragma unroll
      for (int nt = 0; nt < NT; nt += 2)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const f32x4 xv = acc[mt][nt], yv = acc[mt][nt + 1];
          const uint32_t x0 = pack_bf16x2(xv[0], xv[1]), x1 = pack_bf16x2(xv[2], xv[3]);
          const uint32_t y0 = pack_bf16x2(yv[0], yv[1]), y1 = pack_bf16x2(yv[2], yv[3]);
          const auto s0 = __builtin_amdgcn_permlane16_swap(x0, y0, false, false);
          const auto s1 = __builtin_amdgcn_permlane16_swap(x1, y1, false, false);
          const u32x4 v = {s0[0], s1[0], s0[1], s1[1]};
          const int tr = wm * (TM / 2) + mt * 16 + li, col = col_s + nt * 16;
          if (tr < rows && col < p.N) *reinterpret_cast<u32x4*>(p.y + (int64_t)(row0 + tr) * p.N + col) = v;
        }
    };

#pragma unroll
    for (int s = 0; s < S - 1; ++s) issue(s);
    int st = 0, st_fill = S - 1;
    for (int tile = 0; tile < n_tiles; ++tile) {
      if (kMany && tile > 0) {
        // the tile before this one; its stores are younger than the stages in flight, so the next waits
        // cover those stages and some of the stores
        finish_folds();
        store_y(tile - 1);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        // both: the next tile folds 0 * pend_s first, and a scale of this tile may be infinite or NaN
#pragma unroll
        for (int j = 0; j < kLag; ++j) {
          pend[j] = f32x4{0.f, 0.f, 0.f, 0.f};
          pend_s[j] = 0.f;
        }
      }
      for (int kb = 0; kb < KB; ++kb) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * kLoads) : "memory");
        __syncthreads();
        issue(st_fill);
        compute(kb, tile, st);
        st = st + 1 == S ? 0 : st + 1;
        st_fill = st_fill + 1 == S ? 0 : st_fill + 1;
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    finish_folds();

    if (MODE == kGateUp) {
      // h = bf16(silu(gate) * up), kept in the gate tiles' registers; per row, e4m3 at scale
      // max(amax / 448, tiny) over the tile's 128 columns (the wave's 32 here, the other 3 waves'
      // through LDS).
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        float m = 0.0f;
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = round_bf16(silu(acc[mt][2 * q][r]) * acc[mt][2 * q + 1][r]);
            acc[mt][2 * q][r] = v;
            m = fmaxf(m, fabsf(v));
          }
        m = fmaxf(m, __shfl_xor(m, 16));
        m = fmaxf(m, __shfl_xor(m, 32));
        if (g == 0) sAmax[wm][mt][li][wn] = m;
      }
      __syncthreads();
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const float m = fmaxf(fmaxf(sAmax[wm][mt][li][0], sAmax[wm][mt][li][1]),
                              fmaxf(sAmax[wm][mt][li][2], sAmax[wm][mt][li][3]));
        const float sc = fmaxf(__fdiv_rn(m, 448.0f), kFp32Tiny);
        const int tr = wm * (TM / 2) + mt * 16 + li;
        if (tr < rows) {
          const int64_t row = row0 + tr;
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            float cv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) cv[r] = fminf(fmaxf(__fdiv_rn(acc[mt][2 * q][r], sc), -448.0f), 448.0f);
            const int col = pn * 128 + wn * 32 + q * 16 + 4 * g;
            *reinterpret_cast<uint32_t*>(p.hq + row * p.I + col) = pack4_e4m3(cv[0], cv[1], cv[2], cv[3]);
          }
          if (wn == 0 && g == 0) p.hs[(int64_t)pn * p.R + row] = sc;
        }
      }
    } else {
      store_y(n_tiles - 1);
    }
  }
}

// Grouped GEMM over all three block classes in one persistent launch. Workgroups claim work items from
// a ticket counter; the claim order spreads the 256-row items (large experts, MFMA-bound) evenly
// among the 128- and 64-row items (small experts, bound by their weight stream), so at any time some
// CUs run each kind and the two overlap instead of running one after the other. Within a class the
// items run block by block (a block's weight tiles on consecutive tickets), so the re-reads of a
// block's A rows, and of a weight tile by the next block of the same expert, follow within a few
// microseconds, while the memory-side cache still holds them (the tile-major order put a block's
// tiles a whole class apart: T=4096 on Zipf(1.1) routing 3.226 -> 3.110 ms, T=1024 2.207 -> 2.146,
// T=64 1.125 -> 1.106, bitwise the same outputs; one queue per XCD measured 3.370 ms at T=4096). A
// workgroup leaves once its ticket is past the last item.
template <int MODE, bool PRE>
__global__ __launch_bounds__(512) void moe_gemm_kernel(MoeGemmArgs p) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kMoeSmemBytes];
  __shared__ int ticket;
  const int n0 = p.nblk[0], n1 = p.nblk[1], n2 = p.nblk[2];
  // weight tiles per item (DOWN): up to kItemSteps K steps, while four items a CU are left
  int per = 1;
  if (MODE == kDown) {
    per = min(kItemSteps / (p.K >> 7), (int)((int64_t)(n0 + n1 + n2) * p.tiles_n / (4 * (int)gridDim.x)));
    per = per < 1 ? 1 : per;
    const int groups = (p.tiles_n + per - 1) / per;
    per = (p.tiles_n + groups - 1) / groups;  // the same number of items, evenly filled
  }
  const int tn = (p.tiles_n + per - 1) / per;  // items of a 64- or 128-row block
  const int heavy = n0 * p.tiles_n, c1 = n1 * tn, items = heavy + c1 + n2 * tn;
  for (;;) {
    __syncthreads();  // every wave is done with the previous item's LDS and has read the ticket
    if (threadIdx.x == 0) ticket = atomicAdd(p.tickets, 1);
    __syncthreads();
    const int t = ticket;
    if (t >= items) break;
    const int hk = (int)((int64_t)t * heavy / items);  // 256-row items before ticket t
    if ((int64_t)(t + 1) * heavy / items > hk) {
      moe_item<MODE, PRE, 256>(p, smem, 0, hk / p.tiles_n, hk % p.tiles_n, 1);
    } else {
      const int i = t - hk, pn = i % tn * per, tiles = min(per, p.tiles_n - pn);  // c1 is a multiple of tn
      if (i < c1)
        moe_item<MODE, PRE, 128>(p, smem, 1, i / tn, pn, tiles);
      else
        moe_item<MODE, PRE, 64>(p, smem, 2, (i - c1) / tn, pn, tiles);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// combine: out[t] = bf16(sum over slots in slot order of weight * y[row]); 8 columns per thread. The rows
// of kCombineBatch slots load together: one row at a time (an index load, then the row it names) the
// kernel took 15.6 us at 4 tokens x 9 slots of 7168, whose bytes take a microsecond; together 4.8. At 4096
// tokens the rows' 590 MB bound it (119.7 -> 117.6 us).
constexpr int kCombineBatch = 9, kCombineThreads = 128;
__global__ __launch_bounds__(kCombineThreads) void combine_kernel(const uint16_t* __restrict__ y,
                                                                  const int32_t* __restrict__ row_of,
                                                                  const float* __restrict__ weights, int S, int D,
                                                                  uint16_t* __restrict__ out) {
  const int t = blockIdx.x;
  const int c0 = (blockIdx.y * kCombineThreads + threadIdx.x) * 8;
  if (c0 >= D) return;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < S; s0 += kCombineBatch) {
    int row[kCombineBatch];
    float wt[kCombineBatch];
    u32x4 v[kCombineBatch];
#pragma unroll
    for (int j = 0; j < kCombineBatch; ++j) {
      const int64_t i = (int64_t)t * S + min(s0 + j, S - 1);
      row[j] = s0 + j < S ? row_of[i] : -1;
      wt[j] = weights[i];
    }
#pragma unroll
    for (int j = 0; j < kCombineBatch; ++j) v[j] = ld16(y + (int64_t)max(row[j], 0) * D + c0);
#pragma unroll
    for (int j = 0; j < kCombineBatch; ++j) {
      if (row[j] < 0) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] = fmaf(wt[j], bf16_lo(v[j][i]), acc[2 * i]);
        acc[2 * i + 1] = fmaf(wt[j], bf16_hi(v[j][i]), acc[2 * i + 1]);
      }
    }
  }
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = pack_bf16x2(acc[2 * i], acc[2 * i + 1]);
  *reinterpret_cast<u32x4*>(out + (int64_t)t * D + c0) = o;
}

// ---------------------------------------------------------------------------------------------
// host side
struct Workspace {
  size_t part, ids, weights, row_of, sorted_tok, blk_expert, blk_row, blk_rows, nblk, tickets, xq, xs, hq, hs, y,
      total;
  int blk_cap;  // block-table entries per class
};

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// Scratch layout for T tokens, S slots, model dim D, intermediate I, E expert slots, Er router rows
// (0: no router scratch).
static Workspace layout(int64_t T, int64_t S, int64_t D, int64_t I, int64_t E, int64_t Er) {
  Workspace w{};
  const int64_t R = T * S;
  const int64_t cap = R / kMinTM + E + 1;
  const int64_t maxblk = cap * kClasses;
  w.blk_cap = (int)cap;
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o = align256(o + bytes);
    return at;
  };
  w.part = take((size_t)(Er ? router_partials(T, Er) * 4 : 0));
  w.ids = take((size_t)(Er ? R * 4 : 0));
  w.weights = take((size_t)(Er ? R * 4 : 0));
  w.row_of = take((size_t)R * 4);
  w.sorted_tok = take((size_t)R * 4);
  w.blk_expert = take((size_t)maxblk * 4);
  w.blk_row = take((size_t)maxblk * 4);
  w.blk_rows = take((size_t)maxblk * 4);
  w.nblk = take(4 * kClasses);
  w.tickets = take(4 * 2);
  w.xq = take((size_t)(T * D));
  w.xs = take((size_t)(D / 128 * T * 4));
  w.hq = take((size_t)(R * I));
  w.hs = take((size_t)(I / 128 * R * 4));
  w.y = take((size_t)(R * D * 2));
  w.total = o;
  return w;
}

// The persistent grid: one workgroup per CU of the current device (the runtime answers from its
// device table; nothing is kept between calls).
static int num_cus() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 256;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
  return n;
}

static bool dims_ok(int64_t T, int64_t D, int64_t I, int64_t E, int64_t S) {
  if (T <= 0 || T > 65536 || D < 128 || D > 16384 || D % 128 || I < 128 || I > 16384 || I % 128) return false;
  if (E < 1 || E > kMaxExperts || S < 1 || S > 64) return false;
  const int64_t R = T * S;
  // 32-bit offsets: activations, h, y and a row's scales stay below 2 GiB
  return R * D * 2 < 0x7FFFFFFFll && R * I < 0x7FFFFFFFll && T * D < 0x7FFFFFFFll;
}

template <bool PRE>
static void launch_gemms(const MoeGemmArgs& gu, const MoeGemmArgs& dn, hipStream_t stream) {
  const dim3 grid((unsigned)num_cus());
  hipLaunchKernelGGL((moe_gemm_kernel<kGateUp, PRE>), grid, dim3(512), 0, stream, gu);
  hipLaunchKernelGGL((moe_gemm_kernel<kDown, PRE>), grid, dim3(512), 0, stream, dn);
}

// Grouped top-k on bf16 logits, or (part) on the router's fp32 partials.
static void launch_route(const uint16_t* logits, const float* part, int ranges, const uint16_t* bias, int64_t T,
                         int64_t E, int G, int topk, int topk_group, int renormalize, float scale, int shared,
                         int32_t* ids, float* weights, hipStream_t stream) {
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)T), dim3(64), 0, stream, logits, part, ranges, bias, (int)T, (int)E, G,
                       topk, topk_group, renormalize ? 1 : 0, scale, shared ? 1 : 0, ids, weights);
  };
  if (part)
    E <= 256 ? go(route_kernel<true, 4>) : go(route_kernel<true, 16>);
  else
    E <= 256 ? go(route_kernel<false, 4>) : go(route_kernel<false, 16>);
}

// The arguments the grouped top-k takes.
static bool route_ok(int64_t tokens, int64_t n_routed, int topk, int num_expert_group, int topk_group) {
  if (tokens <= 0 || tokens > 65536 || n_routed < 2 || n_routed > 1024) return false;
  if (num_expert_group < 1 || num_expert_group > 64 || n_routed % num_expert_group) return false;
  if (n_routed / num_expert_group < 2 || topk_group < 1 || topk_group > num_expert_group) return false;
  return topk >= 1 && topk <= 63 && topk <= topk_group * (n_routed / num_expert_group);
}

// Experts on a routing already in ids/weights ([T, S], slots in [0, E); others are skipped).
static int run_experts(const uint16_t* hidden, int64_t T, int64_t D, int64_t I, int64_t E, const int32_t* ids,
                       const float* weights, int64_t S, const uint8_t* w1, const float* w1s, const uint8_t* w2,
                       const float* w2s, int w_layout, uint16_t* out, uint8_t* ws, const Workspace& L,
                       hipStream_t stream) {
  const int64_t R = T * S;
  int32_t* row_of = reinterpret_cast<int32_t*>(ws + L.row_of);
  int32_t* sorted_tok = reinterpret_cast<int32_t*>(ws + L.sorted_tok);
  BlockTable bt;
  bt.expert = reinterpret_cast<int32_t*>(ws + L.blk_expert);
  bt.row = reinterpret_cast<int32_t*>(ws + L.blk_row);
  bt.rows = reinterpret_cast<int32_t*>(ws + L.blk_rows);
  bt.count = reinterpret_cast<int32_t*>(ws + L.nblk);
  bt.cap = L.blk_cap;
  uint8_t* xq = ws + L.xq;
  float* xs = reinterpret_cast<float*>(ws + L.xs);
  uint8_t* hq = ws + L.hq;
  float* hs = reinterpret_cast<float*>(ws + L.hs);
  uint16_t* y = reinterpret_cast<uint16_t*>(ws + L.y);
  int* tickets = reinterpret_cast<int*>(ws + L.tickets);

  const int64_t qgroups = T * (D / 128);
  hipLaunchKernelGGL(align_quant_kernel, dim3((unsigned)(1 + (qgroups + 63) / 64)), dim3(1024), 0, stream, ids, (int)R,
                     (int)S, (int)E, row_of, sorted_tok, bt, tickets, hidden, (int)T, (int)D, xq, xs);
  MoeGemmArgs gu{};
  gu.a = xq;
  gu.sa = xs;
  gu.sa_ld = T;
  gu.sorted_tok = sorted_tok;
  gu.b = w1;
  gu.b_stride = 2 * I * D;
  gu.sb = w1s;
  gu.sb_stride = (2 * I / 128) * (D / 128);
  gu.K = (int)D;
  gu.N = (int)(2 * I);
  gu.I = (int)I;
  gu.tiles_n = (int)(I / 128);
  gu.hq = hq;
  gu.hs = hs;
  gu.R = R;
  gu.blk_expert = bt.expert;
  gu.blk_row = bt.row;
  gu.blk_rows = bt.rows;
  gu.nblk = bt.count;
  gu.blk_cap = bt.cap;
  gu.tickets = tickets;
  MoeGemmArgs dn = gu;
  dn.a = hq;
  dn.sa = hs;
  dn.sa_ld = R;
  dn.sorted_tok = nullptr;
  dn.b = w2;
  dn.b_stride = D * I;
  dn.sb = w2s;
  dn.sb_stride = ((D + 127) / 128) * (I / 128);
  dn.K = (int)I;
  dn.N = (int)D;
  dn.tiles_n = (int)((D + kTN - 1) / kTN);
  dn.y = y;
  dn.tickets = tickets + 1;
  if (w_layout == AKLR_B_PRESHUFFLE_16x16)
    launch_gemms<true>(gu, dn, stream);
  else
    launch_gemms<false>(gu, dn, stream);
  hipLaunchKernelGGL(combine_kernel, dim3((unsigned)T, (unsigned)((D / 8 + kCombineThreads - 1) / kCombineThreads)),
                     dim3(kCombineThreads), 0, stream, y, row_of, weights, (int)S, (int)D, out);
  AKLR_LAUNCH_CHECK();
  return AKLR_OK;
}

}  // namespace moe
}  // namespace aklr

using namespace aklr;
using namespace aklr::moe;

extern "C" size_t aklr_moe_fp8_workspace_bytes(int64_t tokens, int64_t model_dim, int64_t inter_dim, int64_t n_experts,
                                               int64_t slots, int64_t n_router_rows) {
  if (!dims_ok(tokens, model_dim, inter_dim, n_experts, slots) || n_router_rows < 0) return 0;
  return layout(tokens, slots, model_dim, inter_dim, n_experts, n_router_rows).total;
}

extern "C" int aklr_moe_fp8_route(const void* logits, const void* bias, int64_t tokens, int64_t n_routed, int topk,
                                  int num_expert_group, int topk_group, int renormalize, float routed_scaling_factor,
                                  int append_shared, int32_t* ids, float* weights, hipStream_t stream) {
  if (!logits || !bias || !ids || !weights) return AKLR_ERR_INVALID_ARGUMENT;
  if (!route_ok(tokens, n_routed, topk, num_expert_group, topk_group)) return AKLR_ERR_INVALID_ARGUMENT;
  launch_route(static_cast<const uint16_t*>(logits), nullptr, 0, static_cast<const uint16_t*>(bias), tokens, n_routed,
               num_expert_group, topk, topk_group, renormalize, routed_scaling_factor, append_shared, ids, weights,
               stream);
  AKLR_LAUNCH_CHECK();
  return AKLR_OK;
}

extern "C" int aklr_moe_fp8_experts(const void* hidden, int64_t tokens, int64_t model_dim, int64_t inter_dim,
                                    int64_t n_experts, const int32_t* ids, const float* weights, int64_t slots,
                                    const void* w1, const float* w1_scale, const void* w2, const float* w2_scale,
                                    int w_layout, void* out, void* workspace, size_t workspace_bytes,
                                    hipStream_t stream) {
  if (!hidden || !ids || !weights || !w1 || !w1_scale || !w2 || !w2_scale || !out) return AKLR_ERR_INVALID_ARGUMENT;
  if (!dims_ok(tokens, model_dim, inter_dim, n_experts, slots)) return AKLR_ERR_INVALID_ARGUMENT;
  if (w_layout != AKLR_B_ROW_MAJOR && w_layout != AKLR_B_PRESHUFFLE_16x16) return AKLR_ERR_UNSUPPORTED;
  if (!aklr_aligned16(hidden) || !aklr_aligned16(w1) || !aklr_aligned16(w2) || !aklr_aligned16(out))
    return AKLR_ERR_INVALID_ARGUMENT;
  const Workspace L = layout(tokens, slots, model_dim, inter_dim, n_experts, 0);
  if (!workspace || workspace_bytes < L.total || !aklr_aligned16(workspace)) return AKLR_ERR_WORKSPACE;
  return run_experts(static_cast<const uint16_t*>(hidden), tokens, model_dim, inter_dim, n_experts, ids, weights, slots,
                     static_cast<const uint8_t*>(w1), w1_scale, static_cast<const uint8_t*>(w2), w2_scale, w_layout,
                     static_cast<uint16_t*>(out), static_cast<uint8_t*>(workspace), L, stream);
}

extern "C" int aklr_deepseek_v2_fp8_moe(const void* hidden, const void* router_weight, const void* correction_bias,
                                        const void* w1, const float* w1_scale, const void* w2, const float* w2_scale,
                                        int64_t tokens, int64_t model_dim, int64_t inter_dim, int64_t n_routed,
                                        int topk, int num_expert_group, int topk_group, int renormalize,
                                        float routed_scaling_factor, int w_layout, void* out, void* workspace,
                                        size_t workspace_bytes, hipStream_t stream) {
  if (!hidden || !router_weight || !correction_bias || !w1 || !w1_scale || !w2 || !w2_scale || !out)
    return AKLR_ERR_INVALID_ARGUMENT;
  if (!route_ok(tokens, n_routed, topk, num_expert_group, topk_group)) return AKLR_ERR_INVALID_ARGUMENT;
  const int64_t S = topk + 1, E = n_routed + 1;
  if (!dims_ok(tokens, model_dim, inter_dim, E, S)) return AKLR_ERR_INVALID_ARGUMENT;
  if (w_layout != AKLR_B_ROW_MAJOR && w_layout != AKLR_B_PRESHUFFLE_16x16) return AKLR_ERR_UNSUPPORTED;
  if (!aklr_aligned16(hidden) || !aklr_aligned16(router_weight) || !aklr_aligned16(w1) || !aklr_aligned16(w2) ||
      !aklr_aligned16(out))
    return AKLR_ERR_INVALID_ARGUMENT;
  const Workspace L = layout(tokens, S, model_dim, inter_dim, E, n_routed);
  if (!workspace || workspace_bytes < L.total || !aklr_aligned16(workspace)) return AKLR_ERR_WORKSPACE;
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  float* part = reinterpret_cast<float*>(ws + L.part);
  int32_t* ids = reinterpret_cast<int32_t*>(ws + L.ids);
  float* weights = reinterpret_cast<float*>(ws + L.weights);
  const RouterPlan rp = plan_router(tokens, n_routed, model_dim);
  const auto router = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)rp.groups), dim3(256), 0, stream, static_cast<const uint16_t*>(hidden),
                       static_cast<const uint16_t*>(router_weight), part, (int)tokens, (int)n_routed, (int)model_dim,
                       rp.ranges, rp.steps_per_wave);
  };
  if (rp.shape == 0)
    router(router_kernel<1, 1, 4, 4>);
  else if (rp.shape == 1)
    router(router_kernel<2, 2, 4, 4>);
  else
    router(router_kernel<4, 4, 1, 1>);
  launch_route(nullptr, part, rp.ranges, static_cast<const uint16_t*>(correction_bias), tokens, n_routed,
               num_expert_group, topk, topk_group, renormalize, routed_scaling_factor, 1, ids, weights, stream);
  return run_experts(static_cast<const uint16_t*>(hidden), tokens, model_dim, inter_dim, E, ids, weights, S,
                     static_cast<const uint8_t*>(w1), w1_scale, static_cast<const uint8_t*>(w2), w2_scale, w_layout,
                     static_cast<uint16_t*>(out), ws, L, stream);
}

AKLR_SCALAR_FP32_END
