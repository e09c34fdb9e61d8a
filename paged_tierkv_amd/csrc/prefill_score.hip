// Prefill block scores on gfx950 without materialising the attention
// probabilities.
//
// Replaces compute_block_scores on the prefill attention weights
// (tierkv_policy.py:1380-1389, called from modeling_llama.py:282-292): for one
// sequence, the mean causal-softmax probability of each key block over every
// query head and every query,
//
//   mass[blk] = sum_{h, q} sum_{t in blk} p[h, q, t] / (H * T) / len(blk),
//   p[h, q, t] = exp(s * q_h . k_t - lse[h, q])  for t <= q, 0 otherwise.
//
// The reference needs the eager attention's [B, H, T, T] probabilities; with
// SDPA it falls back to a sink + recency proxy (modeling_llama.py:294-302).
// Here they are recomputed on MFMA and never leave the workgroup.
//
// Workgroup = (sequence, kv head, 64 (head, query) rows): four slots of 16
// queries, each one head of the GQA group.  Its waves all hold the 64 rows
// as B-operands and split the keys: wave w takes the 16-key tiles w, w + NW,
// ... up to the diagonal.  Per tile and row a wave forms
//   s = sum_t 2^(x_t - m),  m the row's reference (its first tile's maximum;
//   raised only when a sum passes 2^64, so the loop carries no maximum),
// and keeps s in LDS.  When the tiles are done the waves combine their
// (m, sum of s) per row into M and L, so each row's weight 2^(m - M) / L is
// known and the stored sums are weighted, added over the 64 rows and
// written: every q . k and every exponential is computed once.  Prompts
// whose sums do not fit the LDS (above 4096 tokens) make a second pass over
// K with the log-sum-exps instead.  Partial tile masses go to a workspace
// [B, H_kv, row blocks, tiles] and a second kernel reduces them in a fixed
// order, so results are deterministic.
//
// What bounds it: issue.  Per tile and wave 16 MFMAs (D = 128; 16 cycles
// each, of which about 8 block the VALU, measured with independent streams),
// 16 exponentials and about 60 other VALU instructions.  Measured against a
// two-pass kernel whose four waves took 16 queries each and walked all of K
// together (B x tokens, 32 / 8 heads, D = 128, fp16): 16 x 2048 700 -> 370 us,
// 16 x 700 134 -> 55, 2 x 300 41 -> 12, 2 x 4096 453 -> 202, 1 x 8192 (two
// passes) 746 -> 560; 3 x 1001, 32 / 4 heads, D = 64, bf16 163 -> 18.8 (that
// kernel ran 192 workgroups there, each a chain of 63 tiles, twice, for 8
// heads).  Splitting the keys needs no barrier per tile and gives every wave
// the same number of tiles; eight waves per workgroup at 2048 tokens took
// 614 us, as each wave pays its operands and its merge for half the tiles.
//
// MFMA 16x16x32 (gfx950): A = K tile (lane l: key l%16), B = Q^T (lane l:
// query l%16), both with the head dimension visited in the same order
// d = 32*s + 8*(l/16) + i (16-byte chunks); the accumulator holds
// S^T[key = 4*(l/16) + j][query = l%16], so a lane's four logits belong to
// one query and the per-query sums need no shuffles within a slot.  An
// operand load touches 16 rows per instruction, which the vector cache
// serves one 16-byte lane at a time (631 us at 16 x 2048): K tiles and Q go
// through LDS, filled by whole-row loads that write it directly.

#include "tierkv_common.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace tierkv {

constexpr int PS_MAX_TILES = 2048;         // 16-key tiles: T <= 32768
constexpr int PS_MAX_GROUP = 8;            // GQA group

constexpr float PS_FLOOR = -1e30f;         // reference of a row that has seen no key (finite)

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template <typename T>
__device__ __forceinline__ f32x4 mfma32(const uint4& a, const uint4& b, f32x4 c);

template <>
__device__ __forceinline__ f32x4 mfma32<__half>(const uint4& a, const uint4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                0);
}

template <>
__device__ __forceinline__ f32x4 mfma32<__hip_bfloat16>(const uint4& a, const uint4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}

struct PrefillParams {
  const void* q;
  const void* k;
  int64_t qs_b, qs_h, qs_t;      // element strides of q [B, H, T, D]
  int64_t ks_b, ks_h, ks_t;      // element strides of k [B, H_kv, T, D]
  float* partial;                // [B, H_kv, rows, ntiles], rows = nqb * sets
  int32_t heads, kv_heads, tokens, nqb, ntiles, batch, run, sets;
  float scale_log2;
};

// One pass up to 4096 tokens: 64 rows x 256 tiles x 4 B of LDS beside eight
// waves' K tiles.  At 8192 tokens one workgroup of four waves would have the
// CU to itself; two passes with four waves per workgroup keep three there.
constexpr int PL_ONE_PASS_TILES = 256;
constexpr int PL_FOUR_WAVES = 128;         // four waves per workgroup up to 2048 tokens
constexpr int TWO_SETS_ROWS = 2048;
constexpr float PL_BIG = 0x1p64f;          // a tile sum above it re-bases the row's reference

// Value of lane 16 * (lane / 16) + (lane + N) % 16 (DPP row rotate).
template <int N>
__device__ __forceinline__ float row_ror_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, false));
}

// Sum over the four 16-lane rows of each of four values: lane (n, g) of the
// result holds the sum of v[g] over lanes n, n + 16, n + 32, n + 48, in a
// fixed order.
__device__ __forceinline__ float fold_rows4(const float* v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[2]), false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[1]), __float_as_uint(v[3]), false, false);
  const float y02 = __uint_as_float(a[0]) + __uint_as_float(a[1]);   // rows 0, 1: v[0]; rows 2, 3: v[2]
  const float y13 = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  const auto c = __builtin_amdgcn_permlane16_swap(__float_as_uint(y02), __float_as_uint(y13), false, false);
  return __uint_as_float(c[0]) + __uint_as_float(c[1]);
}

typedef const void __attribute__((address_space(1)))* gptr_t;
typedef void __attribute__((address_space(3)))* lptr_t;

// GP heads of a kv head's group share a workgroup's rows: slot s is head
// h0 + s % GP of the group and query block s / GP of the workgroup's 4 / GP
// blocks of 16 queries.  A group of more than GP heads has two head sets: a
// workgroup each (sets = 2), or one after the other in the same workgroup.
template <int D, typename T, int GP, int NW, bool ONE_PASS>
__global__ __launch_bounds__(64 * NW, 3) void prefill_block_mass_kernel(PrefillParams p) {
  constexpr int KS = D / 32;                 // MFMA k-steps (one 16-byte chunk per lane each)
  constexpr int RC = D / 8;                  // 16-byte chunks per K row
  constexpr int LD = 16 * RC / 64;           // 1 KB loads per K tile
  constexpr int QS = 4 / GP;
  extern __shared__ __align__(16) char s_dyn[];
  __shared__ float s_m[NW][64], s_l[NW][64];
  uint4* const s_k = reinterpret_cast<uint4*>(s_dyn);                           // [NW][16 * RC]
  uint4* const s_q = s_k + NW * 16 * RC;                                        // [64 * RC], then
  float* const s_sum = reinterpret_cast<float*>(s_q);                           // [tiles][64 rows] (ONE_PASS)
  const int wg = int(blockIdx.x);
  const int npairs = p.kv_heads * p.batch;
  // Consecutive workgroups go to the 8 XCDs in turn: with a multiple of 8
  // pairs, each XCD serves its own.  Its pairs are taken p.run at a time, the
  // long rows of all of them first.
  const int rows = p.nqb * p.sets;
  const bool by_xcd = (npairs & 7) == 0;
  const int slot = by_xcd ? wg >> 3 : wg;
  const int mine = by_xcd ? npairs >> 3 : npairs;
  const int batch0 = slot / (rows * p.run) * p.run;
  const int width = min(p.run, mine - batch0);
  const int in = slot - rows * batch0;
  const int local = batch0 + in % width;
  const int pair = by_xcd ? local * 8 + (wg & 7) : local;
  const int row = rows - 1 - in / width;
  const int first_head = p.sets == 2 ? (row & 1) * GP : 0;
  const int qb = p.sets == 2 ? row >> 1 : row;
  const int kvh = pair % p.kv_heads, b = pair / p.kv_heads;
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int n = lane & 15, g = lane >> 4;
  const int G = p.heads / p.kv_heads;
  const int Tn = p.tokens;
  const int q0 = qb * 16 * QS;
  const float sl = p.scale_log2;
  const int diag0 = q0 >> 4;                                // the first query block's diagonal tile
  const int last = min(diag0 + QS - 1, (Tn - 1) >> 4);      // the workgroup's last tile
  float* out = p.partial + (int64_t(pair) * rows + row) * p.ntiles;

  // K tiles: this wave's own 16 rows in LDS, filled by loads that go straight
  // there (1 KB each, whole rows).  Chunk c of row r lies at position
  // c ^ swz(r) of the row, so the operand reads (one chunk of 16 rows per
  // quarter wave) touch every bank once.
  uint4* const k_tile = s_k + w * 16 * RC;
  auto swz = [](int r) -> int { return (RC == 16) ? r : (r >> 1) & (RC - 1); };
  const T* kbase = reinterpret_cast<const T*>(p.k) + b * p.ks_b + int64_t(kvh) * p.ks_h;
  // Each lane's source of the tile to load next, advanced by NW tiles per
  // load (a tile that ends past the prompt re-reads its last row).
  const int64_t kstep = int64_t(NW) * 16 * p.ks_t;
  const T* src[LD];
  int src_tile = 0;
  auto start_k = [&]() {
    src_tile = w;
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      const int r = (i * 64 + lane) / RC;
      src[i] = kbase + int64_t(w * 16 + r) * p.ks_t + 8 * (((i * 64 + lane) % RC) ^ swz(r));
    }
  };
  auto load_k = [&]() {
    if (src_tile > last) return;
    if (src_tile * 16 + 16 > Tn) {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
        const int r = (i * 64 + lane) / RC;
        src[i] -= int64_t(max(src_tile * 16 + r - (Tn - 1), 0)) * p.ks_t;
      }
    }
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      __builtin_amdgcn_global_load_lds((gptr_t)src[i], (lptr_t)(k_tile + i * 64), 16, 0, 0);
      src[i] += kstep;
    }
    src_tile += NW;
  };

  for (int h0 = first_head; h0 < G; h0 += GP * p.sets) {
    // Q: slot s's 16 rows are staged by wave s like a K tile, in the LDS that
    // holds the tile sums later, and every wave reads its B-operands from
    // there (queries and heads clamped; rows outside the prompt or the group
    // get weight 0 at the end).  Operand-wise loads from memory would have
    // every wave of the workgroup fetch the 64 rows in 64-byte pieces.
    if (h0 > first_head) __syncthreads();          // the previous head set's sums have been read
#pragma unroll
    for (int s = w; s < 4; s += NW) {
      const int head = kvh * G + min(h0 + s % GP, G - 1);
      const T* base = reinterpret_cast<const T*>(p.q) + b * p.qs_b + head * p.qs_h;
#pragma unroll
      for (int i = 0; i < LD; ++i) {
        const int r = (i * 64 + lane) / RC;
        const int c = ((i * 64 + lane) % RC) ^ swz(r);
        const T* qsrc = base + min(q0 + 16 * (s / GP) + r, Tn - 1) * p.qs_t + 8 * c;
        __builtin_amdgcn_global_load_lds((gptr_t)qsrc, (lptr_t)(s_q + s * 16 * RC + i * 64), 16, 0, 0);
      }
    }
    start_k();
    load_k();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    uint4 qv[4][KS];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int k = 0; k < KS; ++k) qv[s][k] = s_q[(s * 16 + n) * RC + ((4 * k + g) ^ swz(n))];
    __syncthreads();

    float m[4];                                    // reference of row (slot, n), log2 units
#pragma unroll
    for (int s = 0; s < 4; ++s) m[s] = PS_FLOOR;
    float l = 0.f;                                 // this wave's sum of row (slot g, n)

    // The tile's raw logits; the next tile's loads leave once this one has
    // been read.
    auto products = [&](f32x4* acc) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      uint4 kv[KS];
#pragma unroll
      for (int k = 0; k < KS; ++k) kv[k] = k_tile[n * RC + ((4 * k + g) ^ swz(n))];
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      load_k();
#pragma unroll
      for (int s = 0; s < 4; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[s] = mfma32<T>(kv[k], qv[s][k], acc[s]);
      // Keep the four slots' chains interleaved: an MFMA that follows the one
      // it depends on waits for its whole latency.
      __builtin_amdgcn_sched_barrier(0);
    };
    // Logit of key 4g + j (log2 units) less c; -inf past the query.
    auto logit = [&](auto MASK, int kt, const f32x4* acc, int s, int j, float c) -> float {
      float a = fmaf(acc[s][j], sl, -c);
      if constexpr (decltype(MASK)::value) {
        const int d = kt - (diag0 + s / GP);
        a = (d < 0 || (d == 0 && 4 * g + j <= n)) ? a : -INFINITY;
      }
      return a;
    };
    auto sums = [&](auto MASK, int kt, const f32x4* acc, float* v) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        float e[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) e[j] = __builtin_amdgcn_exp2f(logit(MASK, kt, acc, s, j, m[s]));
        v[s] = (e[0] + e[1]) + (e[2] + e[3]);
      }
    };
    auto tile = [&](auto FIRST, auto MASK, int kt) {
      constexpr bool first = decltype(FIRST)::value;
      f32x4 acc[4];
      products(acc);
      float v[4];
      if constexpr (!first) sums(MASK, kt, acc, v);
      if (first || __builtin_expect(__any(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])) > PL_BIG), 0)) {
        // Rows whose sum leaves the headroom take the tile's maximum as
        // their reference and their earlier sums are rescaled; the wave's
        // first tile sets the references.
        float fown = 1.f;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          float mx = -INFINITY;
#pragma unroll
          for (int j = 0; j < 4; ++j) mx = fmaxf(mx, logit(MASK, kt, acc, s, j, 0.f));
          mx = fmaxf(mx, xor16_f(mx));
          mx = fmaxf(mx, xor32_f(mx));
          if constexpr (first) {
            m[s] = fmaxf(PS_FLOOR, mx);
          } else {
            float big = fmaxf(v[s], xor16_f(v[s]));
            big = fmaxf(big, xor32_f(big));
            const float mn = (big > PL_BIG) ? fmaxf(m[s], mx) : m[s];
            const float f = __builtin_amdgcn_exp2f(m[s] - mn);
            m[s] = mn;
            fown = (g == s) ? f : fown;
          }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) asm volatile("" : "+v"(m[s]));
        if constexpr (!first) {
          l *= fown;
          if constexpr (ONE_PASS)
            for (int t = w; t < kt; t += NW) s_sum[t * 64 + lane] *= fown;
        }
        sums(MASK, kt, acc, v);
      }
      const float r = fold_rows4(v);
      l += r;
      if constexpr (ONE_PASS) s_sum[kt * 64 + lane] = r;
    };
    using No = std::integral_constant<bool, false>;
    using Yes = std::integral_constant<bool, true>;
    if (w <= last) tile(Yes{}, Yes{}, w);
    int kt = w + NW;
    for (; kt < min(diag0, last + 1); kt += NW) tile(No{}, No{}, kt);
    for (; kt <= last; kt += NW) tile(No{}, Yes{}, kt);

    // Combine the waves' (m, l) per row.
    const float mo = (g == 0) ? m[0] : (g == 1) ? m[1] : (g == 2) ? m[2] : m[3];
    s_m[w][lane] = mo;
    s_l[w][lane] = l;
    if constexpr (!ONE_PASS) {
      start_k();
      load_k();
    }
    __syncthreads();
    float M = PS_FLOOR, L = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) M = fmaxf(M, s_m[i][lane]);
#pragma unroll
    for (int i = 0; i < NW; ++i) L += s_l[i][lane] * __builtin_amdgcn_exp2f(s_m[i][lane] - M);
    const bool row_ok = q0 + 16 * (g / GP) + n < Tn && h0 + g % GP < G;

    // The masses of four tiles t0, t0 + NW, ... from each lane's share of
    // them: folded over the 64 lanes (the tiles' sums end in the four
    // 16-lane rows) and written.
    auto write4 = [&](int t0, const float* v) {
      float r = fold_rows4(v);
      r += row_ror_f<8>(r);
      r += row_ror_f<4>(r);
      r += row_ror_f<2>(r);
      r += row_ror_f<1>(r);
      const int t = t0 + g * NW;
      if (n == 0 && t <= last) out[t] = (h0 > first_head) ? out[t] + r : r;
    };
    if constexpr (ONE_PASS) {
      // Weight of the row in this wave, and this wave's tiles four at a time.
      const float wt = (L == 0.f) ? 0.f : __builtin_amdgcn_exp2f(mo - M) / L;
      for (int t0 = w; t0 <= last; t0 += 4 * NW) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = t0 + i * NW;
          const float x = s_sum[min(t, last) * 64 + lane] * wt;
          v[i] = (row_ok && t <= last) ? x : 0.f;
        }
        write4(t0, v);
      }
    } else {
      // Second pass over the tiles with the rows' log-sum-exps.
      const float lse = (L == 0.f || !row_ok) ? INFINITY : M + log2f(L);
      __syncthreads();                             // every wave has read the maxima
      s_m[w][lane] = lse;                          // own wave's copy: [slot][query]
#pragma unroll
      for (int s = 0; s < 4; ++s) m[s] = s_m[w][16 * s + n];
      for (int t0 = w; t0 <= last; t0 += 4 * NW) {
        float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = t0 + i * NW;
          if (t > last) continue;
          f32x4 acc[4];
          products(acc);
          float u[4];
          if (t < diag0) sums(No{}, t, acc, u);
          else sums(Yes{}, t, acc, u);
          v[i] = (u[0] + u[1]) + (u[2] + u[3]);
        }
        write4(t0, v);
      }
    }
  }
}

// mass[b, blk] = sum over the partial rows (kv head, 16 * QS queries, head set)
// and the block's tiles, in a fixed order, / (H * T) / len(blk).  Row r of a kv
// head holds tiles up to its last query's, QS * (r / sets) + QS - 1.  One workgroup per (sequence, RED_COLS
// blocks): RED_COLS neighbouring blocks per row (whole 64-byte segments) and
// RED_ROWS rows at a time, from the first row that reaches the blocks on, the
// kv heads' loads four at a time.  Walking all (kv head, row) pairs, half of
// them above the diagonal, with a division each, took 11.9 us at 16 x 2048
// (8 kv heads) and 5.0 at 3 x 1001 (4); now 5.1 and 3.9.
constexpr int RED_COLS = 16;
constexpr int RED_ROWS = 64;
__global__ __launch_bounds__(RED_COLS * RED_ROWS) void prefill_mass_reduce_kernel(const float* partial, float* mass,
                                                                                   int kv_heads, int rows, int sets,
                                                                                   int qs, int ntiles, int heads,
                                                                                   int tokens, int block_size,
                                                                                   int nblk) {
  __shared__ float s_part[RED_COLS * RED_ROWS / 64][RED_COLS];
  const int b = blockIdx.y;
  const int col = threadIdx.x % RED_COLS;
  const int blk = int(blockIdx.x) * RED_COLS + col;
  const int tpb = block_size / 16;
  const int t0 = min(blk, nblk - 1) * tpb;
  const int tn = min(tpb, ntiles - t0);
  const float* base = partial + int64_t(b) * kv_heads * rows * ntiles;
  float acc = 0.f;
  const int first = int(blockIdx.x) * RED_COLS * tpb / qs * sets;
  for (int r = first + int(threadIdx.x) / RED_COLS; r < rows; r += RED_ROWS) {
    const int end = min(t0 + tn, qs * (r >> (sets - 1)) + qs);
    for (int t = t0; t < end; ++t) {
      const float* x = base + int64_t(r) * ntiles + t;
      int h = 0;
      for (; h + 4 <= kv_heads; h += 4) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = x[int64_t(h + i) * rows * ntiles];
        acc += (v[0] + v[1]) + (v[2] + v[3]);
      }
      for (; h < kv_heads; ++h) acc += x[int64_t(h) * rows * ntiles];
    }
  }
  acc += shfl_xor_f(acc, 16);
  acc += shfl_xor_f(acc, 32);
  if ((threadIdx.x & 63) < RED_COLS) s_part[threadIdx.x >> 6][col] = acc;
  __syncthreads();
  if (threadIdx.x < RED_COLS && blk < nblk) {
    float sum = 0.f;
    for (int i = 0; i < RED_COLS * RED_ROWS / 64; ++i) sum += s_part[i][col];
    const int len = min(block_size, tokens - blk * block_size);
    mass[int64_t(b) * nblk + blk] = sum / (float(heads) * float(tokens)) / float(max(len, 1));
  }
}

// The two head sets of a group above four heads run side by side, each
// workgroup half as long, when the launch has no more than eight rows per CU
// (and the workspace holds a partial row for each): 1 x 1000 (8 / 1 heads,
// D = 128) 22.1 -> 14.4 us, 3 x 1001 (32 / 4, D = 64) 21.6 -> 18.8,
// 4 x 2048 (32 / 4, D = 128) 99.7 -> 97.7, 1 x 8192 626 -> 585.  Longer
// launches are full either way and read twice the partials: 16 x 700
// (32 / 4, D = 64, 2816 rows) 41.7 -> 42.8, 2 x 4096 (64 / 8, D = 128, 4096
// rows) 409 -> 421.
static bool head_sets_side_by_side(int groups, int64_t pairs, int64_t ntiles) {
  return groups > 4 && pairs * ntiles <= TWO_SETS_ROWS;
}

template <int D, typename T, int GP>
static hipError_t launch_prefill(const PrefillParams& p, hipStream_t stream) {
  const dim3 grid(unsigned(int64_t(p.nqb) * p.sets * p.kv_heads * p.batch));
  const size_t tile = 16 * D * 2;
  const size_t q = 64 * D * 2;   // the tile sums take its place
  const size_t sums = std::max(q, size_t(p.ntiles) * 64 * sizeof(float));
  // Four waves per workgroup while three workgroups fit a CU's LDS (up to 2048
  // tokens); above, the sums leave room for one or two, so eight waves.
  if (p.ntiles <= PL_FOUR_WAVES)
    hipLaunchKernelGGL((prefill_block_mass_kernel<D, T, GP, 4, true>), grid, dim3(64 * 4), 4 * tile + sums, stream, p);
  else if (p.ntiles <= PL_ONE_PASS_TILES)
    hipLaunchKernelGGL((prefill_block_mass_kernel<D, T, GP, 8, true>), grid, dim3(64 * 8), 8 * tile + sums, stream, p);
  else
    hipLaunchKernelGGL((prefill_block_mass_kernel<D, T, GP, 4, false>), grid, dim3(64 * 4), 4 * tile + q, stream, p);
  return hipGetLastError();
}

template <int D, typename T>
static hipError_t launch_prefill_group(const PrefillParams& p, hipStream_t stream) {
  const int G = p.heads / p.kv_heads;
  if (G == 1) return launch_prefill<D, T, 1>(p, stream);
  if (G == 2) return launch_prefill<D, T, 2>(p, stream);
  return launch_prefill<D, T, 4>(p, stream);
}

}  // namespace tierkv

using namespace tierkv;

extern "C" int64_t tierkv_prefill_block_mass_workspace_bytes(int32_t batch, int32_t num_kv_heads, int32_t tokens) {
  if (batch <= 0 || num_kv_heads <= 0 || tokens <= 0) return -1;
  // A row of tiles per 16 queries (fewer rows are used when the GQA group is
  // below three heads), in whole groups of 64 queries.
  const int64_t rows = (tokens + 63) / 64 * 4;
  const int64_t ntiles = (tokens + 15) / 16;
  return int64_t(batch) * num_kv_heads * rows * ntiles * 4;
}

extern "C" int64_t tierkv_prefill_block_mass_full_workspace_bytes(int32_t batch, int32_t num_heads,
                                                                  int32_t num_kv_heads, int32_t tokens) {
  const int64_t need = tierkv_prefill_block_mass_workspace_bytes(batch, num_kv_heads, tokens);
  if (need < 0 || num_heads <= 0) return -1;
  const bool two = head_sets_side_by_side(num_heads / num_kv_heads, int64_t(batch) * num_kv_heads, (tokens + 15) / 16);
  return two ? 2 * need : need;
}

extern "C" int32_t tierkv_prefill_block_mass(
    const void* q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t,
    const void* k, int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_t, int32_t dtype,
    float* mass, int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t tokens, int32_t head_dim,
    int32_t block_size, float scaling, void* workspace, int64_t workspace_bytes, void* stream_) {
  clear_error();
  if (!q || !k || !mass || !workspace) return fail(TIERKV_ERR_INVALID, "null pointer");
  if (batch <= 0 || num_heads <= 0 || num_kv_heads <= 0 || tokens <= 0)
    return fail(TIERKV_ERR_INVALID, "empty prefill");
  if (batch > 65535) return fail(TIERKV_ERR_UNSUPPORTED, "batch too large");
  if (num_heads % num_kv_heads != 0) return fail(TIERKV_ERR_INVALID, "num_heads must be a multiple of num_kv_heads");
  const int G = num_heads / num_kv_heads;
  if (G > PS_MAX_GROUP) return fail(TIERKV_ERR_UNSUPPORTED, "GQA group above 8");
  if (head_dim != 64 && head_dim != 128) return fail(TIERKV_ERR_UNSUPPORTED, "head_dim must be 64 or 128");
  if (block_size <= 0 || block_size % 16 != 0) return fail(TIERKV_ERR_UNSUPPORTED, "block_size must be a multiple of 16");
  if ((tokens + 15) / 16 > PS_MAX_TILES) return fail(TIERKV_ERR_UNSUPPORTED, "prompts above 32768 tokens");
  if (dtype != TIERKV_DTYPE_F16 && dtype != TIERKV_DTYPE_BF16) return fail(TIERKV_ERR_INVALID, "unknown dtype");
  // Every row load is 16 bytes at element offsets that are multiples of 8.
  const int64_t strides[6] = {q_stride_b, q_stride_h, q_stride_t, k_stride_b, k_stride_h, k_stride_t};
  for (int64_t s : strides)
    if (s % 8 != 0) return fail(TIERKV_ERR_INVALID, "q/k strides must be multiples of 8 elements");
  if (!aligned16(q) || !aligned16(k)) return fail(TIERKV_ERR_INVALID, "q and k must be 16-byte aligned");
  const int64_t need = tierkv_prefill_block_mass_workspace_bytes(batch, num_kv_heads, tokens);
  if (workspace_bytes < need) return fail(TIERKV_ERR_INVALID, "workspace too small");
  PrefillParams p{};
  p.q = q;
  p.k = k;
  p.qs_b = q_stride_b;
  p.qs_h = q_stride_h;
  p.qs_t = q_stride_t;
  p.ks_b = k_stride_b;
  p.ks_h = k_stride_h;
  p.ks_t = k_stride_t;
  p.partial = reinterpret_cast<float*>(workspace);
  p.heads = num_heads;
  p.kv_heads = num_kv_heads;
  p.tokens = tokens;
  p.ntiles = (tokens + 15) / 16;
  p.batch = batch;
  const int qs = G == 1 ? 4 : G == 2 ? 2 : 1;    // 16-query blocks per workgroup and partial row
  p.nqb = (p.ntiles + qs - 1) / qs;
  const int64_t grid = int64_t(p.nqb) * num_kv_heads * batch;
  if (grid > 0x7fffffff) return fail(TIERKV_ERR_UNSUPPORTED, "prefill grid too large");
  const int64_t pairs = int64_t(num_kv_heads) * batch;
  p.sets = (head_sets_side_by_side(G, pairs, p.ntiles) && workspace_bytes >= 2 * need) ? 2 : 1;
  // Pairs whose rows are dealt together: as many as keep their K within half
  // of an XCD's L2, so that the short rows come last and fill the end of the
  // launch.  One pair after the other left its last pair's long rows to the
  // end: 3 x 1001 (32 / 4 heads, D = 64, 12 pairs) 28.8 us against 21.5,
  // 4 x 2048 (32 / 8, D = 128) 99 against 91, 16 x 2048 382 against 374.
  // Above 2048 tokens a workgroup has its CU to itself or makes two passes,
  // and rows of one length running in step are slower (2 x 4096: 204 us pair
  // by pair, 213 with two pairs dealt together).
  const int64_t pair_bytes = int64_t(tokens) * head_dim * 2;
  p.run = p.ntiles > PL_FOUR_WAVES
              ? 1
              : int32_t(std::max<int64_t>(1, std::min<int64_t>((int64_t(2) << 20) / pair_bytes,
                                                               pairs % 8 == 0 ? pairs / 8 : pairs)));
  p.scale_log2 = scaling * 1.4426950408889634f;
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  hipError_t e;
  if (dtype == TIERKV_DTYPE_F16)
    e = head_dim == 128 ? launch_prefill_group<128, __half>(p, stream) : launch_prefill_group<64, __half>(p, stream);
  else
    e = head_dim == 128 ? launch_prefill_group<128, __hip_bfloat16>(p, stream)
                        : launch_prefill_group<64, __hip_bfloat16>(p, stream);
  if (e != hipSuccess) return fail(TIERKV_ERR_HIP, std::string("prefill_block_mass_kernel: ") + hipGetErrorString(e));
  const int nblk = (tokens + block_size - 1) / block_size;
  hipLaunchKernelGGL(prefill_mass_reduce_kernel, dim3((nblk + RED_COLS - 1) / RED_COLS, batch),
                     dim3(RED_COLS * RED_ROWS), 0, stream, p.partial, mass, num_kv_heads,
                     p.nqb * p.sets, p.sets, qs, p.ntiles, num_heads, tokens, block_size, nblk);
  return check_launch("prefill_mass_reduce_kernel");
}
