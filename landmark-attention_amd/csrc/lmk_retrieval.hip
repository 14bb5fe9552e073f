// Mem-cache retrieval for gfx950: landmark scoring, top-k block selection, gather + attend.
//
// Replaces the inline retrieval of LlamaAttention.forward (llama/llama_mem.py:344-412) and
// the attend step over retrieved blocks (:447-477) for the per-head, per-token branch.
//
// Selection must be reproducible bit for bit, so the score of (query, landmark) is defined
// as: fp32 dot product accumulated sequentially over the head dim with one fma per element,
// rounded to the model dtype, divided in fp32 by sqrt(hd), rounded again (the two roundings of
// `matmul(...) / math.sqrt(head_dim)`, :367).  Every pair is evaluated that way up to 64 blocks (a block per
// lane), up to 256 where at most 16 are picked (matrix-core tiles of the same chain), and for few rows (slices); elsewhere
// that would dominate the step, so the work is split:
//   lk      rotate every cached landmark key at its slot position (:359-366), exactly as the
//           model dtype would round it, into a dense side array, with its 2-norm
//   score   MFMA product q . lk^T -> approximate fp32 scores
//   select  per query: bracket every score by the accumulation-error bound
//           eps = 2^-14 |q| |k|, push both ends through the (monotone) rounding contract, find
//           the k-th best lower end, and re-evaluate in the defined order only the "contenders"
//           whose upper end reaches it; then pick the k best under (score desc, index asc)
//           and write them in ascending order as int64 (:384).
//   gather  per query: stream the k selected K/V blocks straight from the cache, rotate keys at
//           their gather positions (:386-388, :408-410), local softmax per block gated by its
//           landmark, and merge with the attention over the local chunk (computed by the fused
//           forward kernel) through the shared global softmax bucket.
#include <algorithm>
#include "lmk_common.hpp"
#include "lmk_landmark_keys.hpp"
#include "lmk_launch.hpp"
#include "lmk_topk_slice.hpp"

namespace lmk {

__device__ __forceinline__ u32x4_t shfl_xor4(u32x4_t v, int mask) {
  u32x4_t r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = (uint32_t)__shfl_xor((int)v[i], mask, 64);
  return r;
}

// ---------------------------------------------------------------------------
// lk: rotated landmark keys (dense) and their norms
// ---------------------------------------------------------------------------
template <class T, int D>
__global__ __launch_bounds__(256) void lmk_landmark_keys_kernel(RetrParams p) {
  landmark_keys_body<T, D, 256>(p, (int)blockIdx.x);
}

// ---------------------------------------------------------------------------
// one selection per head (llama_mem.py:373-384 with aggregate == "max_over_tokens"): every query's
// scores go through an fp32 softmax over the cached blocks, are rounded to the model dtype and
// reduced with a maximum over the queries; the head's k best blocks serve all its queries.
// The softmax needs every score exactly as the contract defines it, so there is no bracketing
// here: a lane evaluates the sequential dot product for its blocks.
// ---------------------------------------------------------------------------

// 2^t for t <= 0 with every rounding fixed, so that a CPU can reproduce it bit for bit:
// n = rint(t), f = t - n (exact), degree-6 Horner polynomial with one rounding after each product
// and each sum (the empty asm keeps the compiler from fusing them), times 2^n (exact).
__device__ __forceinline__ float exp2_contract(float t) {
  if (t < -126.f) return 0.f;
  const float n = __builtin_rintf(t);
  const float f = t - n;
  float pl = 1.5403530393381608e-4f;
  const float c[6] = {1.3333558146428443e-3f, 9.618129107628477e-3f, 5.550410866482158e-2f,
                      2.402265069591007e-1f,  6.931471805599453e-1f, 1.0f};
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    float m = pl * f;
    asm volatile("" : "+v"(m));
    pl = m + c[i];
  }
  return __builtin_ldexpf(pl, (int)n);
}

// Sum over the wave, folded by halves (lanes 32 apart, 16 apart, ... 1 apart), every lane gets it.  Behind the fold by 8 a lane's
// value depends on its low three bits alone, so that a rotation by 4 within the row is the exchange of lanes 4 apart.
__device__ __forceinline__ float wave_sum_halves(float v) {
  v = v + __shfl_xor(v, 32, 64);
  v = v + __shfl_xor(v, 16, 64);
  v = v + dpp_f<0x128>(v);                                        // row_ror 8
  v = v + dpp_f<0x124>(v);                                        // row_ror 4
  v = v + dpp_f<0x4E>(v);                                         // quad_perm [2,3,0,1]
  return v + dpp_f<0xB1>(v);                                      // quad_perm [1,0,3,2]
}

template <class T>
__device__ __forceinline__ uint32_t prob_bits(float x);   // non-negative fp32 -> 16-bit pattern (RNE); monotone
template <>
__device__ __forceinline__ uint32_t prob_bits<bf16_t>(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;           // integer rounding: also right for subnormal x
}
template <>
__device__ __forceinline__ uint32_t prob_bits<f16_t>(float x) { return pack2<f16_t>(x, 0.f) & 0xffffu; }

// Scores of every query against every landmark key, in the contract's order, into p.approx (B*H*T, num_mems).
// The contract's dot product is a chain of fp32 fmas over d ascending, and v_mfma_f32_32x32x1_2b_f32 is 2 x 32 x 32 of
// exactly that step: C[i][j] = fma(A[i], B[j], C[i][j]).  A wave takes 64 query rows (a lane holds its row, packed) and 32
// keys (both halves of the wave hold them); per dimension one unpack each and one MFMA of 64 cycles.  (On the vector unit a
// score is 128 fmas plus whatever brings the key's value to every lane -- an unpack per
// fma with a key per lane, scalar loads of 8 bytes per score with the key in scalar registers, 16 times the LDS
// traffic with every lane reading the value, fmas that take the value from the lane that holds it (row_newbcast) --
// and every such kernel took 50-60 us at the shapes below.)
// A workgroup's four waves are QW groups of query rows x 4 / QW groups of keys; it rotates its keys itself, into LDS.
// A chain of 128 dependent MFMAs is 4 us, and what lies around it -- first loads, rotation, 32 quotients, stores -- 6 more: with
// tiles of 64 keys and the rotation in a launch of its own, 32 heads, 256 queries, 256 blocks took 3.9 + 19.6 us (D64 3.5 + 16.4),
// as it is 13.8 (11.0); 64 heads, 512 queries, 1024 blocks 12.1 + 103.8 and 106 (7.3 + 67.1 and 61).
constexpr int kScoreRows = 64, kScoreKeys = 32;                   // per wave
constexpr int kProbMems = 64 * 32;                                // vectors of more blocks take their maxima in memory, from zero

template <class T, int D, int QW>
__global__ __launch_bounds__(256) void lmk_block_score_kernel(RetrParams p, int n_qs, int n_kc, int64_t agg_words, int agg_per_wg) {
  constexpr int CPR = D / 8;                                      // 16-byte chunks per row of 16-bit values
  constexpr int KEYS = kScoreKeys * 4 / QW;                       // of the workgroup
  constexpr int ROWB = 2 * D + 16;                                // 16 lanes reading 16 B of 16 rows hit every bank once
  constexpr int NI = KEYS * CPR / 256;
  static_assert(KEYS * CPR % 256 == 0, "whole chunks per thread");
  constexpr int QROWB = 80;                                       // a row's four chunks in the query tile: likewise
  __shared__ __align__(16) unsigned char keys[KEYS * ROWB], rows[4][64 * QROWB];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NM = p.num_mems;
  // workgroup -> (queries, keys, head), queries first: the workgroups that run side by side read the same keys
  const uint32_t at = blockIdx.x / (uint32_t)n_qs;
  const int qg = (int)(blockIdx.x - at * n_qs) * QW + wave % QW;
  const int bh = (int)(at / (uint32_t)n_kc), m0 = (int)(at - (uint32_t)bh * n_kc) * KEYS;
  const int b = bh / p.H, hh = bh % p.H;
  // the keys of this thread, two at a time: four would cost head dim 128 its third wave per SIMD
  constexpr int NB = NI < 2 ? NI : 2;
  LandmarkChunk raw[NB];
  auto load_raw = [&](int first) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int it = tid + 256 * (first + i);
      raw[i] = load_landmark_chunk<D>(p, b, hh, min(m0 + it / CPR, NM - 1), it % CPR);   // keys behind the last one: a re-read, never stored
    }
  };
  load_raw(0);
  // the wave's 64 query rows, 64 bytes of 16 rows per load; they change lanes through LDS
  u32x4_t qp[CPR];                                                // this lane's query row, packed
#pragma unroll
  for (int c = 0; c < CPR; ++c) {
    const int t = min(qg * kScoreRows + 16 * (c & 3) + (lane >> 2), p.T - 1);   // rows behind the last one: likewise
    qp[c] = *(const u32x4_t*)((const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h + (int64_t)t * p.qs_r) + 64 * (c >> 2) + 16 * (lane & 3));
  }
  // the vectors the next kernel may take its maxima into start at zero: every workgroup of this one clears its share
  for (int i = tid; i < agg_per_wg; i += 256) {
    const int64_t w = (int64_t)blockIdx.x * agg_per_wg + i;
    if (w < agg_words) p.agg[w] = 0u;
  }
#pragma unroll
  for (int first = 0; first < NI; first += NB) {
    if (first > 0) load_raw(first);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int it = tid + 256 * (first + i), j = it % CPR;
      float r[8];
      rotate_chunk<T>(raw[i].x, raw[i].other, raw[i].c, raw[i].s, j >= CPR / 2, r);
      *(u32x4_t*)(keys + it / CPR * ROWB + 16 * j) = u32x4_t{pack2<T>(r[0], r[1]), pack2<T>(r[2], r[3]), pack2<T>(r[4], r[5]), pack2<T>(r[6], r[7])};
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int c = 0; c < CPR; c += 4) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();                              // the chunks before have been read
#pragma unroll
    for (int i = 0; i < 4; ++i) *(u32x4_t*)(rows[wave] + (16 * i + (lane >> 2)) * QROWB + 16 * (lane & 3)) = qp[c + i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 4; ++i) qp[c + i] = *(const u32x4_t*)(rows[wave] + lane * QROWB + 16 * i);
  }
  __syncthreads();
  const int k0 = wave / QW * kScoreKeys, key = lane & 31;
  if (qg * kScoreRows >= p.T || m0 + k0 >= NM) return;            // no barrier below
  // its key, two chunks at a time: as a whole it would cost a third of the waves a SIMD takes
  u32x4_t kp[2];
  auto load_key = [&](int c) __attribute__((always_inline)) { kp[c & 1] = *(const u32x4_t*)(keys + (k0 + key) * ROWB + 16 * c); };
  load_key(0);
  load_key(1);
  f32x32_t acc;
#pragma unroll
  for (int r = 0; r < 32; ++r) acc[r] = 0.f;
  // dimensions 8 c + i.  A chunk's operands are unpacked together, under the MFMAs of the chunk before: an unpack that writes
  // the operand of an MFMA in flight waits for its end
  float qv[2][8], kv[2][8];
  auto unpack = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      qv[c & 1][i] = (i & 1) ? unpack_hi<T>(qp[c][i >> 1]) : unpack_lo<T>(qp[c][i >> 1]);
      kv[c & 1][i] = (i & 1) ? unpack_hi<T>(kp[c & 1][i >> 1]) : unpack_lo<T>(kp[c & 1][i >> 1]);
      asm volatile("" : "+v"(qv[c & 1][i]), "+v"(kv[c & 1][i]));
    }
    if (c + 2 < CPR) load_key(c + 2);
  };
  unpack(0);
#pragma unroll
  for (int c = 0; c < CPR; ++c) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      acc = __builtin_amdgcn_mfma_f32_32x32x1f32(qv[c & 1][i], kv[c & 1][i], acc, 0, 0, 0);
      if (i == 3 && c + 1 < CPR) unpack(c + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int r = 0; r < 32; ++r) acc[r] = contract<T>(acc[r], p.sqrt_hd);
  // register 16 blk + r of lane l: row 32 blk + 8 (r / 4) + 4 (l / 32) + r % 4, key l % 32
  if (m0 + k0 + key >= NM) return;
  const int t0 = qg * kScoreRows + 4 * (lane >> 5);
  float* dst = p.approx + ((int64_t)bh * p.T + t0) * NM + m0 + k0 + key;
  const bool whole = (qg + 1) * kScoreRows <= p.T;                // uniform
#pragma unroll
  for (int r = 0; r < 32; ++r) {
    const int t = 32 * (r >> 4) + 8 * ((r & 15) >> 2) + (r & 3);
    if (whole || t0 + t < p.T) dst[(int64_t)t * NM] = acc[r];
  }
}

template <class T, int D>
static int launch_scores(const RetrParams& p, hipStream_t stream) {
  // A workgroup's waves share its keys as far as there are query rows for them and at most a quarter of the waves is left
  // without (5 groups of rows, 24 heads of 512 blocks, D128: a step takes 73.6 us with four waves along the rows, 72.9 with two)
  const int groups = (p.T + kScoreRows - 1) / kScoreRows;
  int qw = 4;
  while (qw > 1 && 3 * ((groups + qw - 1) / qw * qw) > 4 * groups) qw >>= 1;
  const int keys = kScoreKeys * 4 / qw, n_qs = (groups + qw - 1) / qw, n_kc = (p.num_mems + keys - 1) / keys;
  const int64_t wgs = (int64_t)p.B * p.H * n_qs * n_kc, words = p.num_mems <= kProbMems ? 0 : (int64_t)(p.agg_over_heads ? p.B * p.T : p.B * p.H) * p.num_mems;
  const int per_wg = (int)((words + wgs - 1) / wgs);
  const dim3 grid((unsigned)wgs);
  if (qw == 4) hipLaunchKernelGGL((lmk_block_score_kernel<T, D, 4>), grid, dim3(256), 0, stream, p, n_qs, n_kc, words, per_wg);
  else if (qw == 2) hipLaunchKernelGGL((lmk_block_score_kernel<T, D, 2>), grid, dim3(256), 0, stream, p, n_qs, n_kc, words, per_wg);
  else hipLaunchKernelGGL((lmk_block_score_kernel<T, D, 1>), grid, dim3(256), 0, stream, p, n_qs, n_kc, words, per_wg);
  return (int)hipGetLastError();
}

// The rows' scores (p.approx) -> softmax -> 16-bit probabilities -> maximum per block into agg, which holds zeros on
// entry: one vector per (batch, head), maxima over the queries -- or per (batch, query), maxima over the heads.
// A lane owns the blocks m = lane, lane + 64, ...; a row's sum is each lane's running sum in that order, folded
// across lanes by halves.  A wave takes rows that share a vector one after the other with the row in registers (NPL values
// per lane: num_mems <= 64 NPL), the next one on its way, and the running maxima too; a workgroup's four waves fold theirs in
// LDS.  Where the vector's rows fit one workgroup (n_parts == 1) its first wave picks from it there and then; otherwise every
// workgroup leaves its part of the maxima, and lmk_block_select_kernel folds and picks.  32 heads, 256 queries, 256 blocks, top 5:
// 5.4 + 4.0 us; with an atomic maximum in memory per block and wave, and picks by a wave over the vector in LDS, 7.4 + 7.5.
// Probabilities are not negative, so their bit patterns order like the values.

// maximum over the 16 lanes of a DPP row, every lane of the row gets it
__device__ __forceinline__ uint32_t row_max_u32(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, false));
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, false));
}

// The k best of a vector of 64 NPL words, lane l holding words l, l + 64, ...: 0 = no block, larger = better, equal words in
// ascending order.  Lane j gets the j-th.  One wave.
template <int NPL>
__device__ __forceinline__ int pick_blocks(uint32_t (&x)[NPL], int k, int lane) {
  int mine = 0x7fffffff;
  for (int j = 0; j < k; ++j) {
    uint32_t bv = 0;
    int bi = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < NPL; ++i)
      if (x[i] > bv) {                                            // ascending i = ascending index: strict > keeps the first
        bv = x[i];
        bi = 64 * i + lane;
      }
    uint32_t best = row_max_u32(bv);
    best = max(max((uint32_t)__builtin_amdgcn_readlane((int)best, 0), (uint32_t)__builtin_amdgcn_readlane((int)best, 16)),
               max((uint32_t)__builtin_amdgcn_readlane((int)best, 32), (uint32_t)__builtin_amdgcn_readlane((int)best, 48)));
    if (best == 0) break;                                         // nothing left (wave-uniform)
    const uint64_t eq = __ballot(bv == best);
    int win;
    if (__popcll(eq) == 1) win = __builtin_amdgcn_readlane(bi, __builtin_ctzll(eq));
    else win = wave_min(bv == best ? bi : 0x7fffffff);
#pragma unroll
    for (int i = 0; i < NPL; ++i) x[i] = (64 * i + lane == win) ? 0u : x[i];
    if (lane == j) mine = win;
  }
  return mine;
}

// The words of a finished vector -> picks, and the copy the caller may have asked for.  One wave.
template <int NPL>
__device__ __forceinline__ void select_blocks(const RetrParams& p, int vec, uint32_t (&x)[NPL], int lane) {
  const int NM = p.num_mems;
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const int m = 64 * i + lane;
    if (m < NM && p.agg_out != nullptr) p.agg_out[(int64_t)vec * NM + m] = (uint16_t)x[i];   // the vector itself, in the model dtype
    // a zero probability is a block still; an fp32 NaN is never picked, a 16-bit one first
    x[i] = (m < NM && !(p.prob32 && x[i] > 0x7f800000u)) ? x[i] + 1 : 0u;
  }
  write_ascending(p.idx + (int64_t)vec * p.k, pick_blocks<NPL>(x, p.k, lane), lane, p.k, NM, p.ring_start);
}

template <int NPL>
__global__ __launch_bounds__(256) void lmk_block_prob_kernel(RetrParams p, int model_is_bf16, int rows_per_wave, int n_parts) {
  __shared__ uint32_t part[3][64 * NPL];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int NM = p.num_mems;
  // rows that share a vector: the T queries of a (batch, head), or the H heads of a (batch, query)
  const int group = p.agg_over_heads ? p.H : p.T;
  const uint32_t vec = blockIdx.x / (uint32_t)n_parts;            // (batch, query) or (batch, head)
  const int first = ((int)(blockIdx.x - vec * n_parts) * 4 + wave) * rows_per_wave, last = min(first + rows_per_wave, group);
  const uint32_t vec_b = vec / (uint32_t)p.T, vec_t = vec - vec_b * p.T;   // (with agg_over_heads)
  uint32_t best[NPL];
#pragma unroll
  for (int i = 0; i < NPL; ++i) best[i] = 0u;
  float next[NPL];
  auto load = [&](int g) __attribute__((always_inline)) {
    // over heads: vec = b T + t, row (b H + g) T + t; over queries: vec = b H + h, row vec T + g
    const int64_t row = p.agg_over_heads ? ((int64_t)vec_b * p.H + g) * p.T + vec_t : (int64_t)vec * p.T + g;
    const float* sc = p.approx + row * NM;
#pragma unroll
    for (int i = 0; i < NPL; ++i) next[i] = (lane + 64 * i < NM) ? sc[lane + 64 * i] : -INFINITY;
  };
  if (first < last) load(first);
  for (int g = first; g < last; ++g) {
    float x[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) x[i] = next[i];
    if (g + 1 < last) load(g + 1);
    float mx = x[0];
#pragma unroll
    for (int i = 1; i < NPL; ++i) mx = fmaxf(mx, x[i]);
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      if (lane + 64 * i < NM) {
        float d = x[i] - mx;
        asm volatile("" : "+v"(d));                               // the product below stays a product
        x[i] = exp2_contract(d * kLog2e);
        sum += x[i];
      }
    }
    sum = wave_sum_halves(sum);
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      if (lane + 64 * i < NM) {
        const float pr = __fdiv_rn(x[i], sum);
        const uint32_t bits = p.prob32 ? __float_as_uint(pr) : (model_is_bf16 ? prob_bits<bf16_t>(pr) : prob_bits<f16_t>(pr));
        best[i] = max(best[i], bits);
      }
    }
  }
  if (wave > 0)
#pragma unroll
    for (int i = 0; i < NPL; ++i) part[wave - 1][64 * i + lane] = best[i];
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int i = 0; i < NPL; ++i)
    best[i] = max(max(best[i], part[0][64 * i + lane]), max(part[1][64 * i + lane], part[2][64 * i + lane]));
  if (n_parts == 1) {
    select_blocks<NPL>(p, (int)vec, best, lane);
    return;
  }
#pragma unroll
  for (int i = 0; i < NPL; ++i)
    if (lane + 64 * i < NM) p.agg[(int64_t)blockIdx.x * NM + lane + 64 * i] = best[i];
}

// A vector's parts, split over four waves -> its picks.
template <int NPL>
__global__ __launch_bounds__(256) void lmk_block_select_kernel(RetrParams p, int n_parts) {
  __shared__ uint32_t part[3][64 * NPL];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), NM = p.num_mems;
  uint32_t best[NPL];
#pragma unroll
  for (int i = 0; i < NPL; ++i) best[i] = 0u;
  constexpr int U = NPL <= 4 ? 8 : (NPL <= 16 ? 2 : 1);           // parts in flight
  for (int s = wave; s < n_parts; s += 4 * U) {
    uint32_t v[U][NPL];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t* src = p.agg + ((int64_t)blockIdx.x * n_parts + min(s + 4 * u, n_parts - 1)) * NM;   // past the end: the last again
#pragma unroll
      for (int i = 0; i < NPL; ++i) v[u][i] = (lane + 64 * i < NM) ? src[lane + 64 * i] : 0u;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < NPL; ++i) best[i] = max(best[i], v[u][i]);
  }
  if (wave > 0)
#pragma unroll
    for (int i = 0; i < NPL; ++i) part[wave - 1][64 * i + lane] = best[i];
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int i = 0; i < NPL; ++i)
    best[i] = max(max(best[i], part[0][64 * i + lane]), max(part[1][64 * i + lane], part[2][64 * i + lane]));
  select_blocks<NPL>(p, (int)blockIdx.x, best, lane);
}

// Scores, probabilities and maxima in one launch, for one selection per head over at most 256 blocks: the scores of 16 (8 / TW)
// query rows never leave the compute unit.  The scores are tiles of 16 rows x 64 landmarks by v_mfma_f32_16x16x1_4b_f32, the step
// of the contract's chain that lmk_block_score_kernel takes 32 x 32 at a time: half as long a chain, twice as many waves to
// overlap.  A workgroup rotates the head's landmark keys itself; TW of its eight waves share them out, the others' rows reuse them.
// LDS: the rotated keys, then the scores and the waves' maxima in their place; the query rows.  What bounds it is a workgroup's
// own chain (load, rotation, products, quotients, softmax, each behind a barrier); it saves the score plane's way to memory and
// back and a launch -- with one part, two: there the picks are made here too.
template <int D, int TW>
struct ScoreProb {
  static constexpr int G = 8 / TW, ROWS = G * 16;                 // 128 / TW rows
  static constexpr int ROWB = 2 * D + 16;                         // 16 lanes reading 16 B of 16 rows hit every bank once
  static constexpr int KEYB = 40;                                 // a landmark's 16 scores, 8 bytes apart from a multiple of 32
  static constexpr int SC = G * TW * 64 * KEYB, PART = 8 * TW * 64 * 4;
  static constexpr int KEYS = TW * 64 * ROWB > SC + PART ? TW * 64 * ROWB : SC + PART;
  static constexpr int LDS = KEYS + ROWS * ROWB;
};

template <class T, int D, int TW>
__global__ __launch_bounds__(512) void lmk_block_score_prob_kernel(RetrParams p, int model_is_bf16, int n_parts) {
  using C = ScoreProb<D, TW>;
  constexpr int CPR = D / 8, ROWB = C::ROWB, KEYB = C::KEYB;
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned char *keys = smem, *sc = smem, *q_lds = smem + C::KEYS;
  uint32_t* part = (uint32_t*)(smem + C::SC);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NM = p.num_mems;
  const int bh = (int)(blockIdx.x / (uint32_t)n_parts), t0 = (int)(blockIdx.x - (uint32_t)bh * n_parts) * C::ROWS;
  const int b = bh / p.H, hh = bh - b * p.H;
  const int tile = wave % TW, group = wave / TW;
  {
    constexpr int NQ = (C::ROWS * CPR + 511) / 512, NI = TW * 64 * CPR / 512, NB = NI < 4 ? NI : 4;
    LandmarkChunk raw[NB];
    auto load_raw = [&](int i) __attribute__((always_inline)) {   // keys behind the last one: a re-read
      const int it = tid + 512 * i;
      raw[i % NB] = load_landmark_chunk<D>(p, b, hh, min(it / CPR, NM - 1), it % CPR);
    };
    u32x4_t rows[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {                                // rows behind the last one: likewise
      const int c = min(tid + 512 * i, C::ROWS * CPR - 1), t = min(t0 + c / CPR, p.T - 1);
      rows[i] = *(const u32x4_t*)((const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h + (int64_t)t * p.qs_r + 8 * (c % CPR)));
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) load_raw(i);
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int c = min(tid + 512 * i, C::ROWS * CPR - 1);
      *(u32x4_t*)(q_lds + c / CPR * ROWB + 16 * (c % CPR)) = rows[i];
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int it = tid + 512 * i, j = it % CPR;
      const LandmarkChunk& k = raw[i % NB];
      float r[8];
      rotate_chunk<T>(k.x, k.other, k.c, k.s, j >= CPR / 2, r);
      *(u32x4_t*)(keys + it / CPR * ROWB + 16 * j) = u32x4_t{pack2<T>(r[0], r[1]), pack2<T>(r[2], r[3]), pack2<T>(r[4], r[5]), pack2<T>(r[6], r[7])};
      if (i + NB < NI) load_raw(i + NB);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();
  f32x16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  const bool busy = 64 * tile < NM && t0 + 16 * group < p.T;      // wave-uniform
  if (busy) {
    const unsigned char* qr = q_lds + (16 * group + (lane & 15)) * ROWB;
    const unsigned char* key = keys + (64 * tile + lane) * ROWB;
    // a chunk's operands are unpacked together, under the MFMAs of the chunk before: an unpack that writes the operand of an
    // MFMA in flight waits for its end
    float qv[2][8], kv[2][8];
    u32x4_t qc = *(const u32x4_t*)qr, kc = *(const u32x4_t*)key;
    auto unpack = [&](int c) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        qv[c & 1][i] = (i & 1) ? unpack_hi<T>(qc[i >> 1]) : unpack_lo<T>(qc[i >> 1]);
        kv[c & 1][i] = (i & 1) ? unpack_hi<T>(kc[i >> 1]) : unpack_lo<T>(kc[i >> 1]);
        asm volatile("" : "+v"(qv[c & 1][i]), "+v"(kv[c & 1][i]));
      }
      if (c + 1 < CPR) {
        qc = *(const u32x4_t*)(qr + 16 * (c + 1));
        kc = *(const u32x4_t*)(key + 16 * (c + 1));
      }
    };
    unpack(0);
#pragma unroll
    for (int c = 0; c < CPR; ++c) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        acc = __builtin_amdgcn_mfma_f32_16x16x1f32(qv[c & 1][i], kv[c & 1][i], acc, 0, 0, 0);
        if (i == 3 && c + 1 < CPR) unpack(c + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  __syncthreads();                                                // the keys have been read
  if (busy) {
    // register 4 blk + r of lane l: row 4 (l / 16) + r, landmark 16 blk + l % 16 of the tile
    unsigned char* dst = sc + ((group * TW + tile) * 64 + (lane & 15)) * KEYB + 8 * (lane >> 4);
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = contract<T>(acc[4 * blk + i], p.sqrt_hd);
      *(u32x2_t*)(dst + 16 * blk * KEYB) = u32x2_t{pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3])};   // exact: rounded already
    }
  }
  __syncthreads();
  // softmax and maxima as in lmk_block_prob_kernel, the rows from LDS
  uint32_t best[TW];
#pragma unroll
  for (int i = 0; i < TW; ++i) best[i] = 0u;
  constexpr int RU = 4;                                           // rows side by side: a row is a chain of reductions
  for (int r0 = wave; r0 < C::ROWS && t0 + r0 < p.T; r0 += 8 * RU) {
    float x[RU][TW], mx[RU], sum[RU];
#pragma unroll
    for (int u = 0; u < RU; ++u) {
      const int r = min(r0 + 8 * u, p.T - 1 - t0);                // rows behind the last one: that one again
      const unsigned char* src = sc + (r / 16 * TW * 64 + lane) * KEYB + 2 * (r % 16);
#pragma unroll
      for (int i = 0; i < TW; ++i)
        x[u][i] = (lane + 64 * i < NM) ? unpack_lo<T>((uint32_t)*(const uint16_t*)(src + 64 * i * KEYB)) : -INFINITY;
    }
#pragma unroll
    for (int u = 0; u < RU; ++u) {
      mx[u] = x[u][0];
#pragma unroll
      for (int i = 1; i < TW; ++i) mx[u] = fmaxf(mx[u], x[u][i]);
      mx[u] = wave_max(mx[u]);
    }
#pragma unroll
    for (int u = 0; u < RU; ++u) {
      sum[u] = 0.f;
#pragma unroll
      for (int i = 0; i < TW; ++i) {
        float d = x[u][i] - mx[u];
        asm volatile("" : "+v"(d));                               // the product below stays a product
        x[u][i] = exp2_contract(d * kLog2e);
        sum[u] += lane + 64 * i < NM ? x[u][i] : 0.f;             // + 0 changes nothing
      }
    }
#pragma unroll
    for (int u = 0; u < RU; ++u) sum[u] = wave_sum_halves(sum[u]);
#pragma unroll
    for (int u = 0; u < RU; ++u)
#pragma unroll
      for (int i = 0; i < TW; ++i) {
        const float pr = __fdiv_rn(x[u][i], sum[u]);
        const uint32_t bits = p.prob32 ? __float_as_uint(pr) : (model_is_bf16 ? prob_bits<bf16_t>(pr) : prob_bits<f16_t>(pr));
        best[i] = max(best[i], bits);
      }
  }
  if (wave > 0)
#pragma unroll
    for (int i = 0; i < TW; ++i) part[(wave * TW + i) * 64 + lane] = best[i];
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 1; w < 8; ++w)
#pragma unroll
    for (int i = 0; i < TW; ++i) best[i] = max(best[i], part[(w * TW + i) * 64 + lane]);
  if (n_parts == 1) {
    select_blocks<TW>(p, bh, best, lane);
    return;
  }
#pragma unroll
  for (int i = 0; i < TW; ++i)
    if (lane + 64 * i < NM) p.agg[(int64_t)blockIdx.x * NM + lane + 64 * i] = best[i];
}

// The same for vectors of any length: one wave per row, the row's exponentials written back over its scores.
__global__ __launch_bounds__(256) void lmk_block_prob_long_kernel(RetrParams p, int model_is_bf16) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= (int64_t)p.B * p.H * p.T) return;
  const int bh = (int)(row / p.T), t = (int)(row % p.T), b = bh / p.H;
  const int NM = p.num_mems;
  float* sc = p.approx + row * NM;                                // this row's scores, then its exponentials
  float mx = -INFINITY;
  for (int m = lane; m < NM; m += 64) mx = fmaxf(mx, sc[m]);
#pragma unroll
  for (int msk = 32; msk >= 1; msk >>= 1) mx = fmaxf(mx, __shfl_xor(mx, msk, 64));
  float sum = 0.f;
  for (int m = lane; m < NM; m += 64) {
    float d = sc[m] - mx;
    asm volatile("" : "+v"(d));                                   // the product below stays a product
    const float e = exp2_contract(d * kLog2e);
    sc[m] = e;
    sum += e;
  }
  sum = wave_sum_halves(sum);
  uint32_t* agg = p.agg + (int64_t)(p.agg_over_heads ? b * p.T + t : bh) * NM;
  for (int m = lane; m < NM; m += 64) {
    const float pr = __fdiv_rn(sc[m], sum);
    const uint32_t bits = p.prob32 ? __float_as_uint(pr) : (model_is_bf16 ? prob_bits<bf16_t>(pr) : prob_bits<f16_t>(pr));
    atomicMax(agg + m, bits);
  }
}

// Behind it, one workgroup per vector: the k best blocks of agg under (value desc, index asc), ascending.
// Four waves bring the head's vector into LDS (and write the copy the caller may have asked for); the
// first wave then picks k times over it.  Vectors too long for the LDS buffer are read in place.
constexpr int kSelectLds = 8192;                                  // words of the LDS copy

__global__ __launch_bounds__(256) void lmk_block_select_long_kernel(RetrParams p) {
  __shared__ uint32_t cached[kSelectLds];
  const int tid = threadIdx.x, lane = tid & 63, bh = blockIdx.x, NM = p.num_mems;
  const uint32_t* agg = p.agg + (int64_t)bh * NM;
  const bool in_lds = NM <= kSelectLds;                           // uniform
  for (int m = tid; m < NM; m += 256) {
    const uint32_t v = agg[m];
    if (in_lds) cached[m] = v;
    if (p.agg_out != nullptr) p.agg_out[(int64_t)bh * NM + m] = (uint16_t)v;   // the head's vector itself, in the model dtype
  }
  __syncthreads();
  if (tid >= 64) return;
  int mine = -1;
  float pv = INFINITY;
  int pi = -1;
  for (int j = 0; j < p.k; ++j) {
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for (int m = lane; m < NM; m += 64) {
      const uint32_t u = in_lds ? cached[m] : agg[m];
      const float x = p.prob32 ? __uint_as_float(u) : (float)u;   // 16-bit patterns as numbers: exact, order-preserving
      const bool after = (x < pv) || (x == pv && m > pi);
      if (after && (x > bv || (x == bv && m < bi))) {
        bv = x;
        bi = m;
      }
    }
    wave_best(bv, bi);
    pv = bv;
    pi = bi;
    if (lane == j) mine = bi;
  }
  write_ascending(p.idx + (int64_t)bh * p.k, mine, lane, p.k, p.num_mems, p.ring_start);
}

// ---------------------------------------------------------------------------
// score + select where a lane can hold a block: caches of at most 64 blocks
// ---------------------------------------------------------------------------
// The bracket of the fused kernel below saves exact dot products where a row has a thousand scores to rank; a row with 64
// pays for its steps (score tile, bracket, list, evaluation, each behind a barrier or an LDS round trip) and gets little.  Here
// lane m keeps block m's rotated key in registers, every score is the contract's dot product, and a wave takes kDirectRows rows
// at a time, whose chains of dependent fmas fill each other's latency.  A row's values reach the fmas as scalar operands.
// What bounds it is latency: one round trip for the keys, D * kDirectRows fmas, k picks.  40 blocks, 6120 rows, D64: 14.4 us
// and 3.3 us of key rotation before, 8.5 us with OWN_KEYS; 136 rows over 16 blocks of 128, D128, which went by slices and their
// merge, 9.1 -> 6.9 us.  (Left to itself the compiler sinks each row's fmas into the branch of the lanes that hold a block, one
// row behind the other, with the loads of its values in front: 10.7 us.)
// OWN_KEYS: the keys are rotated here, by the workgroup into LDS, once for its 4 * kDirectRows rows -- for a caller that keeps
// no rotated keys (the ring cache).  Otherwise they are read from p.lk_rot.
constexpr int kDirectRows = 4;

template <class T, int D, bool OWN_KEYS>
__global__ __launch_bounds__(256) void lmk_topk_direct_kernel(RetrParams p) {
  constexpr int CH = D / 8;                                       // 16-byte chunks of a key
  constexpr int KEYB = 2 * D + 16;                                // 16 lanes reading 16 B of 16 keys hit every bank once
  __shared__ __align__(16) unsigned char keys[OWN_KEYS ? 64 * KEYB : 16];
  const int tid = threadIdx.x, lane = tid & 63, NM = p.num_mems;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t groups = (uint32_t)(p.T + 4 * kDirectRows - 1) / (4 * kDirectRows);
  const uint32_t bh = blockIdx.x / groups;
  const int b = (int)(bh / (uint32_t)p.H), hh = (int)bh - b * p.H;
  const int t0 = (int)(blockIdx.x - bh * groups) * 4 * kDirectRows + kDirectRows * wave;
  // The rows come through the scalar cache (nothing in this launch writes them), 16 dims of each at a time; the next 16 are
  // asked for when these are here, since scalar loads return in any order.  Rows past the end: the last one again.
  typedef uint32_t u32x8_t __attribute__((ext_vector_type(8), aligned(16)));
  typedef const __attribute__((address_space(4))) char* scalar_row_t;
  const int rows = min(p.T - t0, kDirectRows);                    // wave-uniform; below 1: the wave only rotates keys
  scalar_row_t q[kDirectRows];
  u32x8_t now[kDirectRows];
#pragma unroll
  for (int r = 0; r < kDirectRows; ++r) {
    q[r] = (scalar_row_t)(uintptr_t)((const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h + (int64_t)min(t0 + r, p.T - 1) * p.qs_r));
    now[r] = *(const __attribute__((address_space(4))) u32x8_t*)q[r];
  }
  u32x4_t kk[CH];
  if constexpr (OWN_KEYS) {
    constexpr int N = 64 * CH / 256;                              // chunks per thread, all requested together
    LandmarkChunk c[N];
#pragma unroll
    for (int i = 0; i < N; ++i) c[i] = load_landmark_chunk<D>(p, b, hh, min(tid / CH + 256 / CH * i, NM - 1), tid % CH);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      float r[8];
      rotate_chunk<T>(c[i].x, c[i].other, c[i].c, c[i].s, tid % CH >= CH / 2, r);
      const u32x4_t o = {pack2<T>(r[0], r[1]), pack2<T>(r[2], r[3]), pack2<T>(r[4], r[5]), pack2<T>(r[6], r[7])};
      *(u32x4_t*)(keys + (tid / CH + 256 / CH * i) * KEYB + 16 * (tid % CH)) = o;
    }
    __syncthreads();
#pragma unroll
    for (int c8 = 0; c8 < CH; ++c8) kk[c8] = *(const u32x4_t*)(keys + lane * KEYB + 16 * c8);
  } else {
    const char* lk = (const char*)p.lk_rot + (int64_t)bh * lk_tiles(NM) * lk_tile_bytes(D) + lk_key_offset(min(lane, NM - 1), D);
#pragma unroll
    for (int c8 = 0; c8 < CH; ++c8) kk[c8] = *(const u32x4_t*)(lk + 512 * c8);
  }
  if (rows < 1) return;                                           // behind the only barrier
  float v[kDirectRows];
#pragma unroll
  for (int r = 0; r < kDirectRows; ++r) v[r] = 0.f;
  static_assert(kDirectRows == 4, "the operands of the two empty statements below");
#pragma unroll
  for (int st = 0; st < D / 16; ++st) {
    u32x8_t next[kDirectRows];
    if (st + 1 < D / 16) {
      int off = 32 * (st + 1);
      asm volatile("" : "+s"(off) : "s"(now[0][0]), "s"(now[1][0]), "s"(now[2][0]), "s"(now[3][0]));
#pragma unroll
      for (int r = 0; r < kDirectRows; ++r) next[r] = *(const __attribute__((address_space(4))) u32x8_t*)(q[r] + off);
      __builtin_amdgcn_sched_barrier(0);                          // left alone they sink below the fmas they are to hide behind
    }
#pragma unroll
    for (int w = 0; w < 8; ++w) {                                 // the sequential dot product of the contract, d ascending
      const uint32_t ku = kk[2 * st + w / 4][w % 4];
      const float k0 = unpack_lo<T>(ku), k1 = unpack_hi<T>(ku);
#pragma unroll
      for (int r = 0; r < kDirectRows; ++r) v[r] = __builtin_fmaf(unpack_lo<T>(now[r][w]), k0, v[r]);
#pragma unroll
      for (int r = 0; r < kDirectRows; ++r) v[r] = __builtin_fmaf(unpack_hi<T>(now[r][w]), k1, v[r]);
    }
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));   // by all lanes and all rows, step by step
#pragma unroll
    for (int r = 0; r < kDirectRows; ++r) now[r] = next[r];
  }
  // k best of every row: the lowest lane among those that hold the maximum is the lowest block among the best.  No lane holds
  // it (NaN in all that are left): the slot keeps an index past the end, clamped below.
  uint64_t open[kDirectRows];                                     // blocks not picked yet
  int age[kDirectRows], mine[kDirectRows], rank[kDirectRows];     // lane j: the j-th pick, and its place in the order of age
#pragma unroll
  for (int r = 0; r < kDirectRows; ++r) {
    const float x = contract<T>(v[r], p.sqrt_hd);
    v[r] = lane < NM ? x : -INFINITY;
    open[r] = ~0ull >> (64 - NM);
    mine[r] = 0x7fffffff;
  }
  for (int j = 0; j < p.k; ++j)
#pragma unroll
    for (int r = 0; r < kDirectRows; ++r) {
      const float best = wave_max(v[r]);
      const uint64_t eq = __ballot(v[r] == best) & open[r];
      const int win = eq ? __builtin_ctzll(eq) : 0x7fffffff;
      open[r] &= ~(eq & (0 - eq));
      v[r] = lane == win ? -INFINITY : v[r];
      mine[r] = lane == j ? win : mine[r];
    }
#pragma unroll
  for (int r = 0; r < kDirectRows; ++r) {                         // as rank_ascending does, the rows side by side
    mine[r] = min(mine[r], NM - 1);
    age[r] = mine[r] - p.ring_start;
    age[r] += age[r] < 0 ? NM : 0;
    rank[r] = 0;
  }
  for (int j = 0; j < p.k; ++j)
#pragma unroll
    for (int r = 0; r < kDirectRows; ++r) {
      const int o = __builtin_amdgcn_readlane(age[r], j);
      rank[r] += (o < age[r] || (o == age[r] && j < lane)) ? 1 : 0;
    }
  int64_t* out = p.idx + ((int64_t)bh * p.T + t0) * p.k;
#pragma unroll
  for (int r = 0; r < kDirectRows; ++r)
    if (r < rows && lane < p.k) out[r * p.k + rank[r]] = (int64_t)mine[r];
}

// ---------------------------------------------------------------------------
// score + select, every score exact, for caches of 65 to 256 blocks
// ---------------------------------------------------------------------------
// v_mfma_f32_16x16x1_4b_f32 is 4 x 16 x 16 steps of the contract's chain of fmas (see lmk_block_score_kernel): a wave takes 16
// rows and 64 landmarks, one per lane, and per dimension unpacks one value of each and multiplies for 32 cycles.  A workgroup of
// eight waves is TW waves along the landmarks times 8 / TW groups of 16 rows:
//   score    the rows' values come from LDS, the keys from L2 four chunks ahead; a score, rounded, divided and rounded again, is
//            a 16-bit pattern, and LDS keeps it as a number in the scores' order
//   select   a wave takes four rows at a time, 16 lanes each: a lane holds the scores of landmarks l, l + 16, ... above
//            65535 - landmark, so that one unsigned maximum finds the best score at the lowest landmark, and the next pick is the
//            largest number below it
// What bounds it is the chain of a tile (64 or 128 dependent steps, 1 or 2 us) and the select step's vector instructions; the
// bracket's kernel also keeps a whole compute unit per 32 rows, so that its time goes in steps of 256 of them.  Selection in us,
// bracket / exact: 96 blocks, 8192 rows, D64 12.7 / 7.6, D128 14.5 / 9.6; 128 blocks, 32000 rows 46.0 / 12.2, 54.0 / 18.2, 1600
// rows 12.3 / 7.5, 14.4 / 10.0; a chunk's whole step over 256 blocks, 8320 rows 117.9 / 106.4, 189.5 / 177.7.  1024 blocks, 8192 rows, D128, by this design
// with eight waves along the landmarks: 22 / 31, the quotients and the select step as long as the 13.7 us of matrix cores.
constexpr int kExactMems = 256;                                   // landmarks, at most
constexpr int kExactRows = 16;                                    // per wave
constexpr int kExactTopK = 16;                                    // a lane per pick

template <class T>
struct ScoreOrder;                                                // 16-bit patterns with the sign bit flipped, or all bits of a
template <>                                                       // negative value: [-inf, +inf] in order, NaN outside
struct ScoreOrder<bf16_t> {
  static constexpr uint32_t lo = 0x007f, hi = 0xff80;
};
template <>
struct ScoreOrder<f16_t> {
  static constexpr uint32_t lo = 0x03ff, hi = 0xfc00;
};

// TW: waves along the landmarks, one tile of 64 each
template <class T, int D, int TW>
__global__ __launch_bounds__(512, 4) void lmk_topk_exact_kernel(RetrParams p) {
  constexpr int CPR = D / 8;                                      // 16-byte chunks per row of 16-bit values
  constexpr int QROWB = 2 * D + 16;                               // 16 lanes reading 16 B of 16 rows hit every bank once
  constexpr int G = 8 / TW, ROWS = G * kExactRows;                // row groups and rows of the workgroup
  constexpr int KEYB = 2 * kExactRows + 8;                        // a landmark's 16 scores: 16 lanes reading 4 rows hit no bank twice
  constexpr int PW = ROWS / 4 / 8;                                // passes of four rows per wave
  constexpr int NS = 4 * TW;                                      // landmarks per lane of a pass
  __shared__ __align__(16) unsigned char q_lds[ROWS * QROWB];
  __shared__ __align__(16) unsigned char sc[G * TW * 64 * KEYB];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NM = p.num_mems;
  const int n_qt = (p.T + ROWS - 1) / ROWS;
  // Workgroups go to the eight XCDs in turn; the ones that read the same head's landmark keys are put on
  // one XCD, so the keys come out of HBM once rather than once per L2.
  const uint32_t wg = (gridDim.x & 7) ? blockIdx.x : (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int bh = (int)(wg / (uint32_t)n_qt), t0 = (int)(wg - (uint32_t)bh * n_qt) * ROWS;
  const int b = bh / p.H, hh = bh - b * p.H;
  const char* qp = (const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h);
  const char* lk = (const char*)p.lk_rot + (int64_t)bh * lk_tiles(NM) * lk_tile_bytes(D);

  const int tile = wave % TW, group = wave / TW;
  constexpr int NQ = (ROWS * CPR + 511) / 512;
  u32x4_t rows[NQ], kc[4];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {                                  // rows past the end: the last one again, never picked for
    const int c = min(tid + 512 * i, ROWS * CPR - 1), t = min(t0 + c / CPR, p.T - 1);
    rows[i] = *(const u32x4_t*)(qp + 2 * ((int64_t)t * p.qs_r + 8 * (c % CPR)));
  }
  const char* key = lk + lk_key_offset(min(64 * tile + lane, NM - 1), D);   // past the end: a re-read, never picked
#pragma unroll
  for (int c = 0; c < 4; ++c) kc[c] = *(const u32x4_t*)(key + 512 * c);
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int c = min(tid + 512 * i, ROWS * CPR - 1);             // past the last chunk: that one again
    *(u32x4_t*)(q_lds + c / CPR * QROWB + 16 * (c % CPR)) = rows[i];
  }
  __syncthreads();
  if (64 * tile < NM) {                                           // wave-uniform
    const unsigned char* qr = q_lds + (group * kExactRows + (lane & 15)) * QROWB;
    u32x4_t qc = *(const u32x4_t*)qr;
    // a chunk's operands are unpacked together, under the MFMAs of the chunk before: an unpack that writes the operand of an
    // MFMA in flight waits for its end
    float qv[2][8], kv[2][8];
    f32x16_t acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    auto unpack = [&](int c) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        qv[c & 1][i] = (i & 1) ? unpack_hi<T>(qc[i >> 1]) : unpack_lo<T>(qc[i >> 1]);
        kv[c & 1][i] = (i & 1) ? unpack_hi<T>(kc[c & 3][i >> 1]) : unpack_lo<T>(kc[c & 3][i >> 1]);
        asm volatile("" : "+v"(qv[c & 1][i]), "+v"(kv[c & 1][i]));
      }
      if (c + 1 < CPR) qc = *(const u32x4_t*)(qr + 16 * (c + 1));
      if (c + 4 < CPR) kc[c & 3] = *(const u32x4_t*)(key + 512 * (c + 4));
    };
    unpack(0);
#pragma unroll
    for (int c = 0; c < CPR; ++c) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        acc = __builtin_amdgcn_mfma_f32_16x16x1f32(qv[c & 1][i], kv[c & 1][i], acc, 0, 0, 0);
        if (i == 3 && c + 1 < CPR) unpack(c + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // register 4 blk + r of lane l: row 4 (l / 16) + r, landmark 16 blk + l % 16 of the tile
    unsigned char* dst = sc + ((group * TW + tile) * 64 + (lane & 15)) * KEYB + 8 * (lane >> 4);
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      uint32_t o[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {                               // + 0.0: -0 equals +0, and goes to the lower landmark
        typedef short s16x2_t __attribute__((ext_vector_type(2)));
        const uint32_t u = pack2<T>(contract<T>(acc[4 * blk + 2 * i], p.sqrt_hd) + 0.0f,
                                    contract<T>(acc[4 * blk + 2 * i + 1], p.sqrt_hd) + 0.0f);
        const s16x2_t sign = __builtin_bit_cast(s16x2_t, u) >> 15;
        o[i] = u ^ (__builtin_bit_cast(uint32_t, sign) | 0x80008000u);
      }
      *(u32x2_t*)(dst + 16 * blk * KEYB) = u32x2_t{o[0], o[1]};
    }
  }
  __syncthreads();

  const int l16 = lane & 15;
  uint32_t x[PW][NS], best[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int row = 4 * (PW * wave + i) + (lane >> 4);            // of the workgroup
    const unsigned char* src = sc + (row / kExactRows * TW * 64 + l16) * KEYB + 2 * (row % kExactRows);
    best[i] = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const uint32_t v = *(const uint16_t*)(src + 16 * s * KEYB), m = 16 * s + l16;
      x[i][s] = ((int)m < NM && v - ScoreOrder<T>::lo <= ScoreOrder<T>::hi - ScoreOrder<T>::lo) ? v << 16 | (0xffffu - m) : 0u;
      best[i] = max(best[i], x[i][s]);
    }
  }
  int mine[PW], age[PW], rank[PW];                                // lane l: pick l of its row, then its place in the order of age
#pragma unroll
  for (int i = 0; i < PW; ++i) mine[i] = 0;
  for (int j = 0; j < p.k; ++j)
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const uint32_t win = row_max_u32(best[i]);                  // 0: nothing left (NaN)
      mine[i] = l16 == j ? (int)win : mine[i];
      uint32_t below = 0u - win;                                  // the largest below `win`, seen from there: 0 stands for none
#pragma unroll
      for (int s = 0; s < NS; ++s) below = max(below, x[i][s] - win);
      best[i] = win ? below + win : 0u;
    }
#pragma unroll
  for (int i = 0; i < PW; ++i) {                                  // as rank_ascending does
    mine[i] = mine[i] ? 0xffff - (mine[i] & 0xffff) : NM - 1;
    age[i] = mine[i] - p.ring_start;
    age[i] += age[i] < 0 ? NM : 0;
    rank[i] = 0;
  }
  for (int j = 0; j < p.k; ++j)
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int o = __shfl(age[i], (lane & 48) + j, 64);
      rank[i] += (o < age[i] || (o == age[i] && j < l16)) ? 1 : 0;
    }
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int t = t0 + 4 * (PW * wave + i) + (lane >> 4);
    if (t < p.T && l16 < p.k) p.idx[((int64_t)bh * p.T + t) * p.k + rank[i]] = (int64_t)mine[i];
  }
}

// ---------------------------------------------------------------------------
// fused score + select: the approximate scores of 32 query rows never leave the CU
// ---------------------------------------------------------------------------
// A workgroup (16 waves) owns 32 consecutive query rows of one (batch, head) and walks the cached blocks
// in segments of at most kFusedMaxMems:
//   score   the waves split the segment's landmarks; S = Q LK^T by MFMA with the landmark in the lane,
//           so a register (= one query row) lands in 32 consecutive LDS words
//   select  each wave takes 2 of the rows in turn; a lane holds the 16 scores m = 64 j + lane of the
//           row in registers: bracket, k-th best lower end, exact re-evaluation of the contenders
//           (written back over their approximate score), k best
//   merge   (more than one segment) a row's k best are the k best of the segments' k best: lane j of the
//           row's wave keeps the j-th best (score, index) so far and every segment's picks are inserted
//           in order; ascending index order at the end
// The bracket uses a cheap monotone over-/under-estimate of the rounding contract: round_T(x) / sqrt(hd)
// is replaced by a multiplication by the rounded reciprocal, pushed outwards by 2^-21 relative (the
// product is within 2^-22 of the correctly rounded quotient) before the final rounding.  That only
// adds contenders; the ranking itself uses the exact contract.
constexpr int kFusedMaxMems = 1024;
constexpr int kFusedRows = 32;
constexpr int kFusedWaves = 16;
constexpr int kFusedList = 64;                                    // a row's contender list: what one pass of the exact evaluation takes

template <class T, int D, bool SEGMENTS>
__global__ __launch_bounds__(64 * kFusedWaves) void lmk_topk_fused_kernel(RetrParams p) {
  constexpr int KS = D / 16;
  constexpr int NJ = kFusedMaxMems / 64;                          // scores per lane and row
  extern __shared__ __align__(16) unsigned char smem[];
  const int NMall = p.num_mems;
  constexpr int NMp = kFusedMaxMems + 8;                          // row stride (words): the two half-waves of a store (rows 4
                                                                  // apart) then hit different banks; a constant, so that the
                                                                  // sixteen stores of a tile share their address registers
  float* sc = (float*)smem;                                       // [32][NMp]
  float* q_lds = sc + kFusedRows * NMp;                           // [32][D]: the query rows in fp32
  unsigned short* cand = (unsigned short*)(q_lds + kFusedRows * D);   // [32][kFusedList]: a row's contenders (index in the segment)
  unsigned char* q_raw = (unsigned char*)(cand + kFusedRows * kFusedList);    // [32][D] in the model dtype, rows of QROWB bytes
  constexpr int QROWB = 2 * D + 16;                               // 16 lanes reading 16 B of 16 rows hit every bank once
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);      // in a scalar register: what depends on it alone is scalar too
  const int ql = lane & 31, h = lane >> 5;
  const int n_qt = (p.T + kFusedRows - 1) / kFusedRows;
  // Workgroups go to the eight XCDs in turn; the ones that read the same head's landmark keys are put on
  // one XCD, so the keys come out of HBM once rather than once per L2.
  const int wg = (gridDim.x & 7) ? (int)blockIdx.x : (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3));
  const int bh = wg / n_qt, t0 = (wg % n_qt) * kFusedRows;
  const int b = bh / p.H, hh = bh % p.H;
  const char* qp = (const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h);
  const char* lk_all = (const char*)p.lk_rot + (int64_t)bh * lk_tiles(NMall) * lk_tile_bytes(D);
  const float* lkn_all = p.lk_norm + (int64_t)bh * NMall;

  // ---- the 32 query rows -> LDS (MFMA operand of the score phase; the select phase reads them from there too):
  // requested behind the first segment's landmark keys, so that one memory round trip lies in front of the first MFMA
  static_assert(kFusedRows * (D / 8) <= 64 * kFusedWaves && kFusedRows * (D / 8) % 64 == 0, "one chunk of the query rows per thread, whole waves");
  // running k best of every row this wave owns (rows wave, wave + 16): lane j holds the j-th best so far
  float run_v[kFusedRows / kFusedWaves];
  int run_i[kFusedRows / kFusedWaves];
#pragma unroll
  for (int i = 0; i < kFusedRows / kFusedWaves; ++i) {
    run_v[i] = -INFINITY;
    run_i[i] = 0x7fffffff;
  }
  // ---- the cached blocks in segments of at most kFusedMaxMems: a row's k best are the k best of the
  // segments' k best, merged under the same order
  for (int seg = 0; seg < NMall; seg += kFusedMaxMems) {
    const int NM = min(NMall - seg, kFusedMaxMems);                 // landmarks of this segment
    const int NMr = (NM + 63) & ~63;                                // columns read by the select phase
    const char* lk = lk_all + lk_key_offset(seg, D);                // a segment starts a tile
    const float* lkn = lkn_all + seg;
    float nrm[NJ];                                                  // |k_m| of this lane's landmarks, for the select phase:
#pragma unroll                                                     // requested with the keys
    for (int j = 0; j < NJ; ++j) {
      const int m = 64 * j + lane;
      nrm[j] = (m < NM) ? lkn[m] : 0.f;
    }
    // ---- score: A = query rows (lane -> row, from LDS), B = landmark keys (lane -> landmark).  A wave's tiles are
    // 32 * kFusedWaves landmarks apart, at most two per segment, and both are requested before the first is used.
    // MFMA step ks takes chunks 2 ks, 2 ks + 1 of the landmark in the lane: one load instruction reads 1 KB in a row.
    {
      constexpr int NT = kFusedMaxMems / (32 * kFusedWaves);
      u32x4_t kf[NT][KS];
#pragma unroll
      for (int it = 0; it < NT; ++it) {
        const int m0 = 32 * wave + 32 * kFusedWaves * it;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          u32x4_t z = {0, 0, 0, 0};
          kf[it][ks] = z;
          if (m0 < NM) kf[it][ks] = *(const u32x4_t*)(lk + lk_key_offset(m0 + ql, D) + 512 * (2 * ks + h));
        }
      }
      if (seg == 0) {
        if (wave < kFusedRows * (D / 8) / 64) {                     // wave-uniform
          u32x4_t q_chunk = {0, 0, 0, 0};
          if (t0 + tid / (D / 8) < p.T)
            q_chunk = *(const u32x4_t*)(qp + 2 * ((int64_t)(t0 + tid / (D / 8)) * p.qs_r + 8 * (tid % (D / 8))));
          *(u32x4_t*)(q_raw + (tid / (D / 8)) * QROWB + 16 * (tid % (D / 8))) = q_chunk;
        }
        __syncthreads();
      }
#pragma unroll
      for (int it = 0; it < NT; ++it) {
        const int m0 = 32 * wave + 32 * kFusedWaves * it;
        if (m0 < NMr) {                                             // wave-uniform
          const int m = m0 + ql;
          f32x16_t s;
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
            s = mfma32<T>(*(const u32x4_t*)(q_raw + ql * QROWB + 32 * ks + 16 * h), kf[it][ks], s);
          // register r belongs to query row 8 (r / 4) + 4 h + r % 4: four address registers, made here and not kept,
          // and the row within the four as the store's immediate offset (the score tile starts the LDS, at byte 0)
          int base0 = (4 * h * NMp + m) * 4;
          asm volatile("" : "+v"(base0));                           // opaque: what follows is computed here, each time
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const int base = base0 + 8 * a * NMp * 4;
#pragma unroll
            for (int b = 0; b < 4; ++b) lds_st32(base + b * NMp * 4, (m < NM) ? s[4 * a + b] : -INFINITY);
          }
        }
      }
    }
    __syncthreads();

    // ---- select.  A wave owns the rows wave and wave + 16: bracket, threshold and contender list of each, then
    // ONE exact evaluation for the contenders of both (a lane per contender: the two short lists share a pass),
    // then the k best of each.
    const float sq = p.sqrt_hd, inv_sq = 1.0f / sq;
    const int nj = NMr >> 6;                                        // slices in use (wave-uniform)
    constexpr int RPW = kFusedRows / kFusedWaves;
    static_assert(RPW == 2, "two rows per wave");
    auto row_of = [&](int ri) { return wave + kFusedWaves * ri; };

    // wave-wide arg-best of v[] under (value desc, index asc); the winner's slot is set to -inf
    auto take_best = [&](float* v, float& bv_out, int& bi_out) {
      float bv = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (j < nj && v[j] > bv) {                                  // ascending j = ascending index: strict > keeps the first
          bv = v[j];
          bi = 64 * j + lane;
        }
      wave_best(bv, bi);
      const int win = __builtin_amdgcn_readfirstlane(bi);
      const bool owner = lane == (win & 63);
#pragma unroll
      for (int j = 0; j < NJ; ++j) v[j] = (owner && j == (win >> 6)) ? -INFINITY : v[j];
      bv_out = bv;
      bi_out = win;
    };

    // the same with one candidate (value v, index id, unique in the wave) per lane
    auto take_one = [&](float& v, int id, float& bv_out, int& bi_out) {
      wave_best_one(v, id, bv_out, bi_out);
      if (bi_out == id) v = -INFINITY;
    };

    // exact scores of the first cA contenders of row riA and the first cB of row riB, one lane per contender,
    // written over their approximate scores
    auto evaluate = [&](int cA, int riA, int cB, int riB) {
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_s_waitcnt(0xc07f);                           // this wave's LDS writes (q rows, lists) are visible
      for (int c0 = 0; c0 < cA + cB; c0 += 64) {
        const int c = c0 + lane;
        if (c < cA + cB) {
          const bool second = c >= cA;
          const int qi = row_of(second ? riB : riA);
          const int m = cand[qi * kFusedList + (second ? c - cA : c)];
          const float* qrow = q_lds + qi * D;
          const char* kr = lk + lk_key_offset(m, D);
          float acc = 0.f;
#pragma unroll
          for (int g = 0; g < D / 64; ++g) {                        // 8 loads in flight, then their 64 dependent fmas
            u32x4_t kv[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) kv[i] = *(const u32x4_t*)(kr + 512 * (8 * g + i));
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const u32x4_t kk = kv[i];
              const float4 qa = *(const float4*)&qrow[8 * (8 * g + i)];
              const float4 qb = *(const float4*)&qrow[8 * (8 * g + i) + 4];
              acc = __builtin_fmaf(qa.x, unpack_lo<T>(kk[0]), acc);
              acc = __builtin_fmaf(qa.y, unpack_hi<T>(kk[0]), acc);
              acc = __builtin_fmaf(qa.z, unpack_lo<T>(kk[1]), acc);
              acc = __builtin_fmaf(qa.w, unpack_hi<T>(kk[1]), acc);
              acc = __builtin_fmaf(qb.x, unpack_lo<T>(kk[2]), acc);
              acc = __builtin_fmaf(qb.y, unpack_hi<T>(kk[2]), acc);
              acc = __builtin_fmaf(qb.z, unpack_lo<T>(kk[3]), acc);
              acc = __builtin_fmaf(qb.w, unpack_hi<T>(kk[3]), acc);
            }
          }
          sc[qi * NMp + m] = contract<T>(acc, sq);
        }
      }
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_s_waitcnt(0xc07f);
    };

    // what a row leaves for the steps behind its list: entries still in the list, whether the list was emptied
    // on the way, the slices of this lane that hold a contender
    int left[RPW] = {0, 0};
    bool flushed[RPW] = {false, false};
    uint32_t is_c[RPW] = {0u, 0u};
#pragma unroll 1
    for (int ri = 0; ri < RPW; ++ri) {
      const int qi = row_of(ri);
      if (t0 + qi >= p.T) break;                                    // wave-uniform
      // q row -> fp32 in LDS (read back by the evaluation), and its norm
      const unsigned char* qr = q_raw + qi * QROWB;
      float* qrow_lds = q_lds + qi * D;
      float qn = 0.f;
      for (int d = 2 * lane; d < D; d += 128) {
        const uint32_t u = *(const uint32_t*)(qr + 2 * d);
        const float x0 = unpack_lo<T>(u), x1 = unpack_hi<T>(u);
        qrow_lds[d] = x0;
        qrow_lds[d + 1] = x1;
        qn += x0 * x0 + x1 * x1;
      }
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1) qn += __shfl_xor(qn, m, 64);
      const float eps_q = sqrtf(qn) * 1.000001f * (1.0f / 16384.0f);

      const float* srow = sc + qi * NMp;
      // raw bracket of the fp32 dot product: [a - e, a + e] around the MFMA score a.  The contract (round, divide,
      // round) is monotone, and so are the outward-rounded estimates T_lo / T_hi of it below, so the order
      // statistics are taken on the raw ends and only the few values that matter go through T_lo / T_hi.
      float up[NJ];
      float lm = -INFINITY;                                         // this lane's best raw lower end
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        up[j] = -INFINITY;
        if (j < nj) {
          const float a = srow[64 * j + lane];
          const float e = eps_q * nrm[j];
          up[j] = a + e;                                            // -inf (no landmark) stays -inf
          lm = fmaxf(lm, a - e);
        }
      }
      auto t_lo = [&](float x) {
        const float cl = round_to<T>(x) * inv_sq;
        return round_to<T>(cl - fabsf(cl) * 4.76837158203125e-7f);
      };
      auto t_hi = [&](float x) {
        const float ch = round_to<T>(x) * inv_sq;
        return round_to<T>(ch + fabsf(ch) * 4.76837158203125e-7f);
      };
      // tau = T_lo of the k-th best of the lanes' best lower ends: k different blocks reach it, so the k-th best
      // exact score does too (a little below the k-th best lower end itself, and k times cheaper to find)
      float tau_raw = -INFINITY;
      for (int j = 0; j < p.k; ++j) {
        int bi;
        take_one(lm, lane, tau_raw, bi);
      }
      const float tau = t_lo(tau_raw);
      // T_hi(x) >= tau needs x >= tau_raw up to the roundings of both estimates (two roundings to 8 or 11 bits
      // each, 3 % covers them; 1e-5 covers the subnormal range): everything below theta is out without being rounded
      const float theta = tau_raw - (fabsf(tau_raw) * 0.03f + 1e-5f);
      // contenders: upper end reaches tau.  They go into the row's list, which holds what one pass of the exact
      // evaluation takes; the seldom row with more is evaluated here, a list at a time.
      unsigned short* cnd = cand + qi * kFusedList;
      uint32_t mine_c = 0;
      int count = 0;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        if (j < nj && __any(up[j] >= theta && up[j] > -INFINITY)) {   // wave-uniform: most slices hold no contender
          const bool c = up[j] >= theta && up[j] > -INFINITY && t_hi(up[j]) >= tau;
          const uint64_t bal = __ballot(c);
          const int at = count + __popcll(bal & ((1ull << lane) - 1));
          if (c) {
            if (at < kFusedList) cnd[at] = (unsigned short)(64 * j + lane);
            mine_c |= 1u << j;
          }
          count += __popcll(bal);
        }
      }
      bool emptied = false;                                         // wave-uniform
      if (count > kFusedList) {
        const int total = count;
#pragma unroll 1
        for (int first = 0; first < total; first += kFusedList) {   // contenders first .. first + 63, in the order of above
          __builtin_amdgcn_wave_barrier();                          // the list has been read
          int seen = 0;
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            const bool c = (mine_c >> j) & 1;
            const uint64_t bal = __ballot(c);
            const int at = seen + __popcll(bal & ((1ull << lane) - 1)) - first;
            if (c && at >= 0 && at < kFusedList) cnd[at] = (unsigned short)(64 * j + lane);
            seen += __popcll(bal);
          }
          evaluate(min(total - first, kFusedList), ri, 0, ri);
        }
        count = 0;
        emptied = true;
      }
      if (ri == 0) {
        left[0] = count;
        flushed[0] = emptied;
        is_c[0] = mine_c;
      } else {
        left[1] = count;
        flushed[1] = emptied;
        is_c[1] = mine_c;
      }
    }
    if (left[0] + left[1] > 0) evaluate(left[0], 0, left[1], 1);

#pragma unroll 1
    for (int ri = 0; ri < RPW; ++ri) {
      const int qi = row_of(ri);
      const int t = t0 + qi;
      if (t >= p.T) break;                                          // wave-uniform
      const float* srow = sc + qi * NMp;
      const int count = ri == 0 ? left[0] : left[1];
      const bool emptied = ri == 0 ? flushed[0] : flushed[1];
      const uint32_t mine_c = ri == 0 ? is_c[0] : is_c[1];
      // k best exact scores, best first, handed to `use`: in a single segment they are the row's (written
      // in ascending index order), otherwise each is inserted into the row's running list
      auto consume = [&](auto&& pick) {
        if constexpr (!SEGMENTS) {
          int mine = -1;                                           // lane j keeps the j-th pick
          for (int j = 0; j < p.k; ++j) {
            float bv;
            int bi;
            pick(bv, bi);
            if (lane == j) mine = bi;
          }
          write_ascending(p.idx + ((int64_t)bh * p.T + t) * p.k, mine, lane, p.k, p.num_mems, p.ring_start);
        } else {
          float rv = ri == 0 ? run_v[0] : run_v[1];
          int rx = ri == 0 ? run_i[0] : run_i[1];
          for (int j = 0; j < p.k; ++j) {
            float bv;
            int bi;
            pick(bv, bi);
            if (!(bv > -INFINITY)) break;                           // fewer than k landmarks in this segment (wave-uniform)
            bi += seg;
            const bool better = lane < p.k && (rv > bv || (rv == bv && rx < bi));   // a prefix of the sorted list
            const int pos = __popcll(__ballot(better));
            if (pos >= p.k) break;                                  // worse than the k kept: so are the rest
            const float up_v = __shfl_up(rv, 1, 64);
            const int up_i = __shfl_up(rx, 1, 64);
            if (lane > pos) {
              rv = up_v;
              rx = up_i;
            } else if (lane == pos) {
              rv = bv;
              rx = bi;
            }
          }
          if (ri == 0) {
            run_v[0] = rv;
            run_i[0] = rx;
          } else {
            run_v[1] = rv;
            run_i[1] = rx;
          }
        }
      };
      if (!emptied) {                                               // the usual case: few contenders, still in the list
        float cv = -INFINITY;
        int ci = 0x7fffffff;
        if (lane < count) {
          ci = cand[qi * kFusedList + lane];
          cv = srow[ci];
        }
        consume([&](float& bv, int& bi) { take_one(cv, ci, bv, bi); });
      } else {                                                      // exact scores picked up from the row, 16 per lane
        float x[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) x[j] = (j < nj && ((mine_c >> j) & 1)) ? srow[64 * j + lane] : -INFINITY;
        consume([&](float& bv, int& bi) { take_best(x, bv, bi); });
      }
    }
    __syncthreads();                                                // the next segment overwrites the score tile
  }

  // ---- ascending order of the k kept blocks
  if constexpr (!SEGMENTS) return;
  for (int qi = wave, ri = 0; qi < kFusedRows; qi += kFusedWaves, ++ri) {
    const int t = t0 + qi;
    if (t >= p.T) break;
    int mine = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < kFusedRows / kFusedWaves; ++i)
      if (i == ri) mine = run_i[i];
    write_ascending(p.idx + ((int64_t)bh * p.T + t) * p.k, mine, lane, p.k, p.num_mems, p.ring_start);
  }
}

// ---------------------------------------------------------------------------
// select without the bracket, for a handful of query rows (decoding): see lmk_topk_slice.hpp
// ---------------------------------------------------------------------------
template <class T, int D>
__global__ __launch_bounds__(64 * kSliceWaves) void lmk_topk_slice_kernel(RetrParams p, int n_slices) {
  __shared__ __align__(16) unsigned char lds[kSliceLdsBytes];
  topk_slice_body<T, D>(p, n_slices, (int)blockIdx.x, lds);
}

// One wave per query row: the k best of the row's n_slices * k candidates, written in ascending index order.
__global__ __launch_bounds__(256) void lmk_topk_slice_merge_kernel(RetrParams p, int n_slices) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= (int64_t)p.B * p.H * p.T) return;                      // wave-uniform
  const int mine = merge_slices_row(p, n_slices, row, lane);
  write_ascending(p.idx + row * p.k, mine, lane, p.k, p.num_mems, p.ring_start);
}

// ---------------------------------------------------------------------------
// gather + attend over the selected blocks, merged with the local-chunk attention
// ---------------------------------------------------------------------------
__device__ __forceinline__ float sum8(float d) {                  // sum over the 8 lanes of a key group (lane & 7)
  d += dpp_f<0xB1>(d);                                            // quad_perm [1,0,3,2]
  d += dpp_f<0x4E>(d);                                            // quad_perm [2,3,0,1]
  d += dpp_f<0x141>(d);                                           // row_half_mirror
  return d;
}

// One wave per query row.  Eight lanes share a key: lane j of the group holds head dims 8j..8j+7 and
// 64+8j..64+8j+7 (head dim 128; 4j..4j+3 and 32+4j..32+4j+3 at head dim 64), i.e. both partners of the rotary pair, so the rotation needs no exchange between
// lanes; the eight key groups of the wave take keys g, g+8, .. of a block.  Rotation and scores are
// evaluated in fp32 from the 16-bit cache and table values (the reference rounds the rotated key to
// the model dtype first; the difference is far inside the 2e-2 bound of this step, and selection --
// where bits matter -- does not go through here).
// A block passes through the registers in chunks of at most 64 keys -- first the keys of every chunk
// (scores of the whole block, which the block's softmax needs before any weight is final), then the
// values, so keys and values are never live together and the kernel keeps several waves per SIMD.  The
// loads of the next chunk are issued before the arithmetic on the current one.
// PADDED: the cache's blocks hold p.block < BS tokens (the benchmark models' 51).  A block is then worked on in BS
// slots: slot s < p.block - 1 is normal key s, the last slot is the landmark (token p.block - 1), the slots in
// between re-read a normal key and get the score -inf, i.e. weight 0 in the block's softmax and in the output.
// The picked blocks of a row are read at p.idx[b * idx_sb + h * idx_sh + t * idx_st + 0 .. k-1] (selections shared
// by the heads or by the queries have a zero stride there); a block counts among the k newest, whose keys sit one
// block further on, by its age in the ring (p.ring_start = slot of the oldest block, 0 for a flat cache).
// Keys per chunk: with the window inside, chunks of 32 leave room for three waves per SIMD at blocks of 64 and head dim
// 128; without it two run whichever is taken, and 64 keys keep more loads in flight (a chunk step at block 64: 256 queries of
// 32 heads, top 4, 186.5 -> 184.0 us; 64 queries, top 5, 86.6 -> 83.5).
constexpr int gather_chunk(int BS, int D, bool LOCAL) { return BS == 32 || (LOCAL && BS == 64 && D == 128) ? 32 : 64; }
template <int E> struct PieceVec;
template <> struct PieceVec<8> { using type = u32x4_t; };
template <> struct PieceVec<4> { using type = u32x2_t; };

// MERGE: the row's blocks are picked from the slices' candidates first (p.merge_slices > 0); a template parameter
// because the four registers it holds on to would cost the plain kernel its third wave per SIMD (172 against 168).
// LOCAL: the row's local window -- the tokens of the cache behind its last complete block and the new tokens up to
// the row's own, at most one block together -- is attended to here as well, as one more item of the row's online
// softmax, instead of coming in as (o_loc, L_loc, M_loc) from a forward launch over a window another launch built:
// a decode step is then the selection and this kernel.  Its keys join the global bucket directly (own-block rule:
// causal, the landmark token does not see itself; flash_landmark_attention.py:78-100).
// (Decode steps of more rows than lmk_gather_decode_kernel is the better one for.)
template <class T, int D, int BS, bool SPLIT, bool PADDED, bool MERGE = false, bool LOCAL = false,
          int CK = gather_chunk(BS, D, LOCAL)>
__global__ __launch_bounds__(256) void lmk_gather_attend_kernel(RetrParams p) {
  constexpr int NWV = SPLIT ? 4 : 1;                              // waves that share the row's blocks out
  static_assert((D == 128 || D == 64) && (BS == 32 || BS % 64 == 0), "8 lanes x 2 pieces per row; whole chunks of keys");
  static_assert(!LOCAL || (!PADDED && !SPLIT), "the local window sits in a block of BS tokens; a wave per row");
  constexpr int E = D / 16;                                       // head dims per lane and rotary half: 8 or 4
  constexpr int PB = 2 * E;                                       // bytes of one piece
  using vec_t = typename PieceVec<E>::type;                       // one piece: E 16-bit values
  constexpr int KPG = CK / 8;                                     // keys per 8-lane group and chunk
  constexpr int NC = BS / CK;                                     // chunks per block
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = SPLIT || LOCAL ? tid >> 6 : __builtin_amdgcn_readfirstlane(tid >> 6);   // (what they make of it overflows the scalar registers)
  const int j = lane & 7, g = lane >> 3;                           // head-dim chunk pair, key group
  // (bh, t): a wave's own row, or -- SPLIT, for launches with few rows -- the workgroup's row, whose
  // selected blocks its waves share out (block js goes to wave js % 4) and merge at the end
  const uint32_t row = SPLIT ? blockIdx.x : blockIdx.x * 4 + wave;   // scalar, and 32-bit as every launch's waves are
  if (row >= (uint32_t)(p.B * p.H) * (uint32_t)p.T) return;       // SPLIT: the whole workgroup leaves
  const int js0 = SPLIT ? wave : 0, jstep = NWV;
  const int bh = (int)(row / (uint32_t)p.T), t = (int)(row - (uint32_t)bh * p.T);
  const int b = (int)((uint32_t)bh / (uint32_t)p.H), hh = bh - b * p.H;

  auto unpack8 = [](const vec_t u, float* o) {
#pragma unroll
    for (int i = 0; i < E / 2; ++i) {
      o[2 * i] = unpack_lo<T>(u[i]);
      o[2 * i + 1] = unpack_hi<T>(u[i]);
    }
  };
  float qlo[E], qhi[E];
  {
    const char* qp = (const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h + (int64_t)t * p.qs_r);
    unpack8(*(const vec_t*)(qp + PB * j), qlo);
    unpack8(*(const vec_t*)(qp + D + PB * j), qhi);
  }
  // The row's own key (without rotary) and value on their way into the cache: fetched here
  // (lanes 0 .. D/8-1 the key, 32 .. the value), stored at the end, so that nothing waits for them.  Nobody reads the
  // destination in this launch: it lies behind the cached rows.
  const bool appends = LOCAL && p.ap_k != nullptr && (lane & 31) < D / 8;
  u32x4_t ap = {0, 0, 0, 0};
  if (LOCAL && appends)
    ap = *(const u32x4_t*)((lane < 32 ? (const char*)p.ap_k + 2 * (b * p.aks_b + hh * p.aks_h + (int64_t)t * p.aks_r)
                                      : (const char*)p.ap_v + 2 * (b * p.avs_b + hh * p.avs_h + (int64_t)t * p.avs_r)) +
                           16 * (lane & 31));
  const char* kc = (const char*)p.kcache + 2 * (b * p.kcs_b + hh * p.kcs_h);
  const char* vc = (const char*)p.vcache + 2 * (b * p.vcs_b + hh * p.vcs_h);
  const float c2 = p.scale_log2;
  const int nreal = PADDED ? p.block : BS;                        // tokens of a block in the cache
  auto token_of = [&](int slot) {                                 // slot of the block's BS -> token of the block it reads
    if (!PADDED) return slot;
    return slot == BS - 1 ? nreal - 1 : min(slot, nreal - 2);
  };
  const int64_t* idx_row = p.idx + (b * p.idx_sb + hh * p.idx_sh + (int64_t)t * p.idx_st);
  // The decode-time selection leaves a row's candidates (k per slice of the cache) rather than its indices: the wave
  // picks the k best first -- lane r of `sorted` gets the r-th block in the order of the output -- and one wave per
  // row writes them where the caller expects the indices.
  constexpr bool merged = MERGE;
  int sorted = 0;
  if constexpr (MERGE) {
    int mine = merge_slices_row(p, p.merge_slices, row, lane);
    const int rank = rank_ascending(mine, lane, p.k, p.num_mems, p.ring_start);
    sorted = __builtin_amdgcn_ds_permute(4 * (lane < p.k ? rank : lane), mine);
    if (lane < p.k && (!SPLIT || wave == 0)) p.idx[b * p.idx_sb + hh * p.idx_sh + (int64_t)t * p.idx_st + rank] = (int64_t)mine;
  }
  auto picked = [&](int js) {                                      // idx is a caller's array: never read outside the cache
    return merged ? __shfl(sorted, js, 64) : min(max((int)idx_row[js], 0), p.num_mems - 1);
  };
  auto newest = [&](int blk) {                                    // one of the k newest blocks: its keys sit one block further on
    int age = blk - p.ring_start;
    age += age < 0 ? p.num_mems : 0;
    return age >= p.num_mems - p.k;
  };

  float Mrun = kNoScore, lrun = 0.f;
  float alo[E], ahi[E];
#pragma unroll
  for (int i = 0; i < E; ++i) {
    alo[i] = 0.f;
    ahi[i] = 0.f;
  }

  // one chunk = CK rows of K or of V: this lane's KPG rows (g, g+8, ..) x its two 16-byte pieces
  vec_t clo[KPG], chi[KPG], nlo[KPG], nhi[KPG];
  auto fetch = [&](const char* base, int64_t row_stride, int64_t key0, int slot0) {
#pragma unroll
    for (int i = 0; i < KPG; ++i) {
      const char* r = base + 2 * ((key0 + token_of(slot0 + g + 8 * i)) * row_stride) + PB * j;
      nlo[i] = *(const vec_t*)(r);
      nhi[i] = *(const vec_t*)(r + D);
    }
  };
  auto take = [&]() {
#pragma unroll
    for (int i = 0; i < KPG; ++i) {
      clo[i] = nlo[i];
      chi[i] = nhi[i];
    }
  };
  if constexpr (LOCAL) {
    const int inc = p.local_inc, own = inc + t;                 // window rows: inc of the cache, then the new tokens
    const char* kn = (const char*)p.k_new + 2 * (b * p.kns_b + hh * p.kns_h);
    const char* vn = (const char*)p.v_new + 2 * (b * p.vns_b + hh * p.vns_h);
    float s_loc[KPG * NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (CK * c > own) {                                       // a chunk behind the row's own token (wave-uniform)
#pragma unroll
        for (int i = 0; i < KPG; ++i) s_loc[KPG * c + i] = -INFINITY;
        continue;
      }
#pragma unroll
      for (int i = 0; i < KPG; ++i) {
        const int r = CK * c + g + 8 * i;
        const bool visible = r <= own && !(r == BS - 1 && own == BS - 1);
        const int rc = min(r, own);                             // rows behind the row's own are never read
        const bool cached = rc < inc;
        const char* kr = (cached ? kc + 2 * ((p.local_row0 + rc) * p.kcs_r) : kn + 2 * ((int64_t)(rc - inc) * p.kns_r)) + PB * j;
        const int64_t pos = inc > 0 ? p.local_pos0 + min(rc, inc - 1) : 0;   // a position the tables hold, used by cached rows only
        const char* cr = (const char*)p.cos + 2 * (pos * p.cs_r) + PB * j;
        const char* sr = (const char*)p.sin + 2 * (pos * p.cs_r) + PB * j;
        float kl[E], kh[E], cl[E], ch[E], sl[E], sh[E];
        unpack8(*(const vec_t*)(kr), kl);
        unpack8(*(const vec_t*)(kr + D), kh);
        unpack8(*(const vec_t*)(cr), cl);
        unpack8(*(const vec_t*)(cr + D), ch);
        unpack8(*(const vec_t*)(sr), sl);
        unpack8(*(const vec_t*)(sr + D), sh);
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {                           // cached keys are rotated in the model dtype, as the cache's
          const float rl = cached ? round_to<T>(__builtin_fmaf(kl[e], cl[e], -kh[e] * sl[e])) : kl[e];   // window is (llama_mem.py:336-338)
          const float rh = cached ? round_to<T>(__builtin_fmaf(kh[e], ch[e], kl[e] * sh[e])) : kh[e];
          d = __builtin_fmaf(qlo[e], rl, d);
          d = __builtin_fmaf(qhi[e], rh, d);
        }
        s_loc[KPG * c + i] = visible ? sum8(d) * c2 : -INFINITY;
      }
    }
    float mx = s_loc[0];                                        // row 0 is always visible
#pragma unroll
    for (int i = 1; i < KPG * NC; ++i) mx = fmaxf(mx, s_loc[i]);
    mx = fmaxf(mx, dpp_f<0x128>(mx));
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    float den = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (CK * c > own) continue;
#pragma unroll
      for (int i = 0; i < KPG; ++i) {
        const int rc = min(CK * c + g + 8 * i, own);
        const bool cached = rc < inc;
        const char* vr = (cached ? vc + 2 * ((p.local_row0 + rc) * p.vcs_r) : vn + 2 * ((int64_t)(rc - inc) * p.vns_r)) + PB * j;
        const vec_t vlo = *(const vec_t*)(vr), vhi = *(const vec_t*)(vr + D);
        const float e = fast_exp2(s_loc[KPG * c + i] - mx);
        den += e;
        const float w = round_to<T>(e);                         // weights enter PV in the model dtype
#pragma unroll
        for (int e2 = 0; e2 < E / 2; ++e2) {
          alo[2 * e2] = __builtin_fmaf(w, unpack_lo<T>(vlo[e2]), alo[2 * e2]);
          alo[2 * e2 + 1] = __builtin_fmaf(w, unpack_hi<T>(vlo[e2]), alo[2 * e2 + 1]);
          ahi[2 * e2] = __builtin_fmaf(w, unpack_lo<T>(vhi[e2]), ahi[2 * e2]);
          ahi[2 * e2 + 1] = __builtin_fmaf(w, unpack_hi<T>(vhi[e2]), ahi[2 * e2 + 1]);
        }
      }
    }
    den += dpp_f<0x128>(den);
    den += __shfl_xor(den, 16, 64);
    den += __shfl_xor(den, 32, 64);
    Mrun = mx;
    lrun = den;
  }
  int blk = 0;
  if (js0 < p.k) {
    blk = picked(js0);
    fetch(kc, p.kcs_r, (int64_t)blk * nreal, 0);
  }
  for (int js = js0; js < p.k; js += jstep) {
    const int64_t key0 = (int64_t)blk * nreal;
    const int64_t pos0 = (int64_t)js * nreal + (newest(blk) ? nreal : 0) + p.prefix_len;
    float sc[KPG * NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      take();
      if (c + 1 < NC) fetch(kc, p.kcs_r, key0, CK * (c + 1));
      else fetch(vc, p.vcs_r, key0, 0);
#pragma unroll
      for (int i = 0; i < KPG; ++i) {
        const int slot = CK * c + g + 8 * i;
        const int kk = token_of(slot);
        const char* cr = (const char*)p.cos + 2 * ((pos0 + kk) * p.cs_r) + PB * j;
        const char* sr = (const char*)p.sin + 2 * ((pos0 + kk) * p.cs_r) + PB * j;
        float kl[E], kh[E], cl[E], ch[E], sl[E], sh[E];
        unpack8(clo[i], kl);
        unpack8(chi[i], kh);
        unpack8(*(const vec_t*)(cr), cl);
        unpack8(*(const vec_t*)(cr + D), ch);
        unpack8(*(const vec_t*)(sr), sl);
        unpack8(*(const vec_t*)(sr + D), sh);
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float rl = __builtin_fmaf(kl[e], cl[e], -kh[e] * sl[e]);
          const float rh = __builtin_fmaf(kh[e], ch[e], kl[e] * sh[e]);
          d = __builtin_fmaf(qlo[e], rl, d);
          d = __builtin_fmaf(qhi[e], rh, d);
        }
        sc[KPG * c + i] = sum8(d) * c2;                           // log2 domain
        if (PADDED && slot >= nreal - 1 && slot != BS - 1) sc[KPG * c + i] = -INFINITY;   // a slot without a token
      }
    }
    // landmark = key BS-1 = last chunk, group 7, last of the group's keys
    const float t_lm = __shfl(sc[KPG * NC - 1], 56, 64);
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < KPG * NC; ++i)
      if (!(i == KPG * NC - 1 && g == 7)) mx = fmaxf(mx, sc[i]);
    mx = fmaxf(mx, dpp_f<0x128>(mx));                             // row_ror 8: the other key group of the row
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    float den = 0.f;
#pragma unroll
    for (int i = 0; i < KPG * NC; ++i) {
      float e = fast_exp2(sc[i] - mx);
      if (i == KPG * NC - 1 && g == 7) e = 0.f;
      sc[i] = e;
      den += e;
    }
    den += dpp_f<0x128>(den);
    den += __shfl_xor(den, 16, 64);
    den += __shfl_xor(den, 32, 64);
    const float Mnew = fmaxf(Mrun, t_lm);
    const float alpha = fast_exp2(Mrun - Mnew);
    const float gate = fast_exp2(t_lm - Mnew);
    lrun = lrun * alpha + gate;
    Mrun = Mnew;
    const float f = gate / den;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      alo[e] *= alpha;
      ahi[e] *= alpha;
    }
    int blk_next = blk;
    if (js + jstep < p.k) blk_next = picked(js + jstep);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      take();
      if (c + 1 < NC) fetch(vc, p.vcs_r, key0, CK * (c + 1));
      else if (js + jstep < p.k) fetch(kc, p.kcs_r, (int64_t)blk_next * nreal, 0);
#pragma unroll
      for (int i = 0; i < KPG; ++i) {
        const float w = round_to<T>(sc[KPG * c + i] * f);         // weights enter PV in the model dtype
#pragma unroll
        for (int e = 0; e < E / 2; ++e) {
          alo[2 * e] = __builtin_fmaf(w, unpack_lo<T>(clo[i][e]), alo[2 * e]);
          alo[2 * e + 1] = __builtin_fmaf(w, unpack_hi<T>(clo[i][e]), alo[2 * e + 1]);
          ahi[2 * e] = __builtin_fmaf(w, unpack_lo<T>(chi[i][e]), ahi[2 * e]);
          ahi[2 * e + 1] = __builtin_fmaf(w, unpack_hi<T>(chi[i][e]), ahi[2 * e + 1]);
        }
      }
    }
    blk = blk_next;
  }
  if (LOCAL && appends)
    *(u32x4_t*)((lane < 32 ? (char*)p.ap_kd + 2 * (b * p.akd_b + hh * p.akd_h + (int64_t)t * p.akd_r)
                           : (char*)p.ap_vd + 2 * (b * p.avd_b + hh * p.avd_h + (int64_t)t * p.avd_r)) +
                16 * (lane & 31)) = ap;
#pragma unroll
  for (int e = 0; e < E; ++e) {                                   // sum over the eight key groups
    alo[e] += dpp_f<0x128>(alo[e]);
    ahi[e] += dpp_f<0x128>(ahi[e]);
    alo[e] += __shfl_xor(alo[e], 16, 64);
    ahi[e] += __shfl_xor(ahi[e], 16, 64);
    alo[e] += __shfl_xor(alo[e], 32, 64);
    ahi[e] += __shfl_xor(ahi[e], 32, 64);
  }
  if constexpr (SPLIT) {                                          // the waves' partial (M, l, acc) -> wave 0
    __shared__ float part_acc[NWV][D];
    __shared__ float part_ml[NWV][2];
    if (g == 0) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        part_acc[wave][E * j + e] = alo[e];
        part_acc[wave][D / 2 + E * j + e] = ahi[e];
      }
      if (j == 0) {
        part_ml[wave][0] = Mrun;
        part_ml[wave][1] = lrun;
      }
    }
    __syncthreads();
    if (wave != 0) return;
    float mw[NWV], Mall = part_ml[0][0];                          // wave 0 always has a block (k >= 1)
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      mw[w] = part_ml[w][0];
      Mall = fmaxf(Mall, mw[w]);
    }
    lrun = 0.f;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      alo[e] = 0.f;
      ahi[e] = 0.f;
    }
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      const float sw = fast_exp2(mw[w] - Mall);                   // 0 for a wave without blocks, or times nothing
      lrun = __builtin_fmaf(part_ml[w][1], sw, lrun);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        alo[e] = __builtin_fmaf(part_acc[w][E * j + e], sw, alo[e]);
        ahi[e] = __builtin_fmaf(part_acc[w][D / 2 + E * j + e], sw, ahi[e]);
      }
    }
    Mrun = Mall;
  }
  if constexpr (LOCAL) {                                          // the local window is in the sums already
    const float inv = 1.0f / lrun;
    if (g == 0) {
      char* outp = (char*)p.out + 2 * (b * p.outs_b + hh * p.outs_h + (int64_t)t * p.outs_r) + PB * j;
      vec_t ov;
#pragma unroll
      for (int i = 0; i < E / 2; ++i) ov[i] = pack2<T>(alo[2 * i] * inv, alo[2 * i + 1] * inv);
      *(vec_t*)(outp) = ov;
#pragma unroll
      for (int i = 0; i < E / 2; ++i) ov[i] = pack2<T>(ahi[2 * i] * inv, ahi[2 * i + 1] * inv);
      *(vec_t*)(outp + D) = ov;
    }
    return;
  }
  // merge with the local chunk: out_loc (normalised), L_loc, M_loc (natural-log units)
  const int64_t srow = (int64_t)bh * p.stat_stride + t;
  const float Ml = p.M_loc[srow] * kLog2e, Ll = p.L_loc[srow];
  const float Mt = fmaxf(Mrun, Ml);
  const float wr = fast_exp2(Mrun - Mt), wl = fast_exp2(Ml - Mt) * Ll;
  const float inv = 1.0f / (lrun * wr + wl);
  if (g == 0) {
    const char* olp = (const char*)p.o_loc + 2 * (b * p.ols_b + hh * p.ols_h + (int64_t)t * p.ols_r) + PB * j;
    char* outp = (char*)p.out + 2 * (b * p.outs_b + hh * p.outs_h + (int64_t)t * p.outs_r) + PB * j;
    float ol[E], o[E];
    vec_t ov;
    unpack8(*(const vec_t*)(olp), ol);
#pragma unroll
    for (int i = 0; i < E; ++i) o[i] = (alo[i] * wr + ol[i] * wl) * inv;
#pragma unroll
    for (int i = 0; i < E / 2; ++i) ov[i] = pack2<T>(o[2 * i], o[2 * i + 1]);
    *(vec_t*)(outp) = ov;
    unpack8(*(const vec_t*)(olp + D), ol);
#pragma unroll
    for (int i = 0; i < E; ++i) o[i] = (ahi[i] * wr + ol[i] * wl) * inv;
#pragma unroll
    for (int i = 0; i < E / 2; ++i) ov[i] = pack2<T>(o[2 * i], o[2 * i + 1]);
    *(vec_t*)(outp + D) = ov;
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
int launch_topk_slice_merge(const RetrParams& p, hipStream_t stream) {
  const int64_t rows = (int64_t)p.B * p.H * p.T;
  hipLaunchKernelGGL(lmk_topk_slice_merge_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, p, topk_slices(p));
  return (int)hipGetLastError();
}

template <class T, int D>
static int launch_topk_t(const RetrParams& p, LandmarkKeys keys, hipStream_t stream) {
  constexpr int RPW = 256 / (D / 8);
  const int64_t lkrows = (int64_t)p.B * p.H * p.num_mems;
  const bool direct = p.num_mems <= 64;                             // a lane per block
  const dim3 direct_grid((unsigned)p.B * p.H * (unsigned)((p.T + 4 * kDirectRows - 1) / (4 * kDirectRows)));
  int rc;
  if (direct && keys == LandmarkKeys::kTransient) {
    hipLaunchKernelGGL((lmk_topk_direct_kernel<T, D, true>), direct_grid, dim3(256), 0, stream, p);
    return (int)hipGetLastError();
  }
  if (keys != LandmarkKeys::kRotated) {
    hipLaunchKernelGGL((lmk_landmark_keys_kernel<T, D>), dim3((unsigned)((lkrows + RPW - 1) / RPW)), dim3(256), 0, stream, p);
    if ((rc = (int)hipGetLastError())) return rc;
  }
  if (direct) {
    hipLaunchKernelGGL((lmk_topk_direct_kernel<T, D, false>), direct_grid, dim3(256), 0, stream, p);
    return (int)hipGetLastError();
  }
  const int64_t rows = (int64_t)p.B * p.H * p.T;
  const int n_slices = topk_slices(p);
  if (n_slices > 0) {                                               // a handful of rows: every score exact, slices over the chip
    hipLaunchKernelGGL((lmk_topk_slice_kernel<T, D>), dim3((unsigned)(rows * n_slices)), dim3(64 * kSliceWaves), 0, stream, p, n_slices);
    if ((rc = (int)hipGetLastError())) return rc;
    return launch_topk_slice_merge(p, stream);
  }
  if (p.num_mems <= kExactMems && p.k <= kExactTopK) {
    auto launch = [&](auto kern, int rows_per_wg) {
      const int64_t wgs = (int64_t)p.B * p.H * ((p.T + rows_per_wg - 1) / rows_per_wg);
      hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(512), 0, stream, p);
    };
    if (p.num_mems <= 128) launch(lmk_topk_exact_kernel<T, D, 2>, 4 * kExactRows);
    else launch(lmk_topk_exact_kernel<T, D, 4>, 2 * kExactRows);
    return (int)hipGetLastError();
  }
  constexpr int lds_max = (kFusedRows * (kFusedMaxMems + 8) + kFusedRows * D) * 4 + kFusedRows * kFusedList * 2 + kFusedRows * (2 * D + 16);
  static_assert(lds_max <= 160 * 1024, "the score tile, the query rows and the lists fill the LDS of a compute unit");
  constexpr int lds = lds_max;                                    // one workgroup of 16 waves per compute unit whatever it takes
  const int n_rt = (p.T + kFusedRows - 1) / kFusedRows;
  const dim3 grid(p.B * p.H * n_rt), block(64 * kFusedWaves);
  if (p.num_mems <= kFusedMaxMems) {
    auto kern = lmk_topk_fused_kernel<T, D, false>;
    static std::atomic<uint64_t> lds_ok{0};
    if ((rc = allow_dynamic_lds(kern, lds_max, lds_ok))) return rc;
    hipLaunchKernelGGL(kern, grid, block, lds, stream, p);
  } else {
    auto kern = lmk_topk_fused_kernel<T, D, true>;
    static std::atomic<uint64_t> lds_ok{0};
    if ((rc = allow_dynamic_lds(kern, lds_max, lds_ok))) return rc;
    hipLaunchKernelGGL(kern, grid, block, lds, stream, p);
  }
  return (int)hipGetLastError();
}

template <class T, int D>
static int launch_topk_shared_t(const RetrParams& p, hipStream_t stream) {
  int rc;
  const int64_t sel_rows = p.agg_over_heads ? (int64_t)p.B * p.T : (int64_t)p.B * p.H;   // vectors to pick from
  const int is_bf16 = std::is_same<T, bf16_t>::value ? 1 : 0;
  // Scores and maxima in one launch, but for more than 128 blocks at head dim 128 where a head's rows take several workgroups:
  // each rotates 64 KB of keys.  Steps in us, two launches / one: 256 queries, 256 blocks, D64 35.2 / 28.9; 2 x 512 queries, 128
  // blocks, D64 46.0 / 39.9, D128 59.8 / 54.7; 64 blocks, 512 queries, D128 43.4 / 41.0; 16 queries over 8 blocks 25.0 / 17.6.
  // 256 blocks, D128: 16 queries 33.6 / 29.6, 256 queries 38.2 / 37.7, 512 queries 52.3 / 53.8, 2 x 400 queries 68.7 / 75.8.
  const int tw = p.num_mems <= 64 ? 1 : (p.num_mems <= 128 ? 2 : 4), prob_parts = (p.T + 128 / tw - 1) / (128 / tw);
  if (!p.agg_over_heads && p.num_mems <= 256 && (D == 64 || tw < 4 || prob_parts == 1)) {
    static std::atomic<uint64_t> lds_ok[3];
    auto launch = [&](auto kern, int lds, std::atomic<uint64_t>& ok, auto select) {
      if (int e = allow_dynamic_lds(kern, lds, ok)) return e;
      hipLaunchKernelGGL(kern, dim3((unsigned)(sel_rows * prob_parts)), dim3(512), lds, stream, p, is_bf16, prob_parts);
      if (prob_parts > 1) hipLaunchKernelGGL(select, dim3((unsigned)sel_rows), dim3(256), 0, stream, p, prob_parts);
      return (int)hipGetLastError();
    };
    if (tw == 1) return launch(lmk_block_score_prob_kernel<T, D, 1>, ScoreProb<D, 1>::LDS, lds_ok[0], lmk_block_select_kernel<1>);
    if (tw == 2) return launch(lmk_block_score_prob_kernel<T, D, 2>, ScoreProb<D, 2>::LDS, lds_ok[1], lmk_block_select_kernel<2>);
    return launch(lmk_block_score_prob_kernel<T, D, 4>, ScoreProb<D, 4>::LDS, lds_ok[2], lmk_block_select_kernel<4>);
  }
  if ((rc = launch_scores<T, D>(p, stream))) return rc;
  const int64_t rows = (int64_t)p.B * p.H * p.T;
  if (p.num_mems <= kProbMems) {
    // rows per wave: a vector's rows in one workgroup where that is at most 8 each (the launch saved outweighs the rows in a
    // row: 255 tokens over 40 blocks, maxima over 12 heads, 44.6 -> 42.1 us a step); over more than 256 blocks, where a row is 16 or
    // 32 values a lane, at most 3 each or with other vectors to fill the chip; else as many as leave the chip a few thousand
    // waves.  A selection of 8 heads, D128, 16 queries over 516 blocks: one row each 21.3 us, four 24.7; 32 queries 21.7, eight 33.1;
    // over 2048 blocks 30.6 and 61.9.  Maxima over 12 heads, 500 blocks: one 26.6, three 26.1; over 32, 1000 blocks, 2 x 16 queries
    // 31.4, eight 45.5, 2 x 500 150.7 and 137.6.
    const int group = p.agg_over_heads ? p.H : p.T;
    const bool whole = group <= (p.num_mems <= 256 || rows >= 16384 ? 32 : 12);
    const int rpw = whole ? (group + 3) / 4 : (int)std::max<int64_t>(1, std::min<int64_t>(8, rows / 4096));
    const int n_parts = (group + 4 * rpw - 1) / (4 * rpw);
    const dim3 grid((unsigned)(sel_rows * n_parts));
    auto launch = [&](auto prob, auto select) {
      hipLaunchKernelGGL(prob, grid, dim3(256), 0, stream, p, is_bf16, rpw, n_parts);
      if (n_parts > 1) hipLaunchKernelGGL(select, dim3((unsigned)sel_rows), dim3(256), 0, stream, p, n_parts);
    };
    if (p.num_mems <= 64) launch(lmk_block_prob_kernel<1>, lmk_block_select_kernel<1>);
    else if (p.num_mems <= 64 * 4) launch(lmk_block_prob_kernel<4>, lmk_block_select_kernel<4>);
    else if (p.num_mems <= 64 * 16) launch(lmk_block_prob_kernel<16>, lmk_block_select_kernel<16>);
    else launch(lmk_block_prob_kernel<32>, lmk_block_select_kernel<32>);
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(lmk_block_prob_long_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, p, is_bf16);
  if ((rc = (int)hipGetLastError())) return rc;
  hipLaunchKernelGGL(lmk_block_select_long_kernel, dim3((unsigned)sel_rows), dim3(256), 0, stream, p);
  return (int)hipGetLastError();
}

int launch_retrieve_topk_shared(const RetrParams& p, int D, int dtype, hipStream_t stream) {
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_topk_shared_t<bf16_t, 128>(p, stream);
    if (D == 64) return launch_topk_shared_t<bf16_t, 64>(p, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_topk_shared_t<f16_t, 128>(p, stream);
    if (D == 64) return launch_topk_shared_t<f16_t, 64>(p, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

template <class T, int D>
static int launch_lk_t(const RetrParams& p, hipStream_t stream) {
  constexpr int RPW = 256 / (D / 8);
  const int64_t lkrows = (int64_t)p.B * p.H * p.num_mems;
  hipLaunchKernelGGL((lmk_landmark_keys_kernel<T, D>), dim3((unsigned)((lkrows + RPW - 1) / RPW)), dim3(256), 0, stream, p);
  return (int)hipGetLastError();
}

// The slice step of the selection alone (topk_slices(p) > 0): a row's candidates stay in p.approx / p.exact for a
// gather step that merges them (RetrParams::merge_slices).
template <class T, int D>
static int launch_slices_t(const RetrParams& p, hipStream_t stream) {
  const int n_slices = topk_slices(p);
  if (n_slices <= 0) return LMK_ERR_UNSUPPORTED;
  const int64_t rows = (int64_t)p.B * p.H * p.T;
  hipLaunchKernelGGL((lmk_topk_slice_kernel<T, D>), dim3((unsigned)(rows * n_slices)), dim3(64 * kSliceWaves), 0, stream, p, n_slices);
  return (int)hipGetLastError();
}

int launch_topk_slices(const RetrParams& p, int D, int dtype, hipStream_t stream) {
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_slices_t<bf16_t, 128>(p, stream);
    if (D == 64) return launch_slices_t<bf16_t, 64>(p, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_slices_t<f16_t, 128>(p, stream);
    if (D == 64) return launch_slices_t<f16_t, 64>(p, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

int launch_landmark_keys(const RetrParams& p, int D, int dtype, hipStream_t stream) {
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_lk_t<bf16_t, 128>(p, stream);
    if (D == 64) return launch_lk_t<bf16_t, 64>(p, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_lk_t<f16_t, 128>(p, stream);
    if (D == 64) return launch_lk_t<f16_t, 64>(p, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

int launch_retrieve_topk(const RetrParams& p, int D, int dtype, LandmarkKeys keys, hipStream_t stream) {
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_topk_t<bf16_t, 128>(p, keys, stream);
    if (D == 64) return launch_topk_t<bf16_t, 64>(p, keys, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_topk_t<f16_t, 128>(p, keys, stream);
    if (D == 64) return launch_topk_t<f16_t, 64>(p, keys, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

template <class T, int D, int BS, bool PADDED>
static int launch_gather_b(const RetrParams& p, hipStream_t stream) {
  const int64_t rows = (int64_t)p.B * p.H * p.T;
  if (p.local) {                          // with the row's local window: blocks as they are only
    if constexpr (!PADDED && D == 128 && BS <= 64) {
      const dim3 grid((unsigned)((rows + 3) / 4));
      if (p.merge_slices > 0) hipLaunchKernelGGL((lmk_gather_attend_kernel<T, D, BS, false, PADDED, true, true>), grid, dim3(256), 0, stream, p);
      else hipLaunchKernelGGL((lmk_gather_attend_kernel<T, D, BS, false, PADDED, false, true>), grid, dim3(256), 0, stream, p);
      return (int)hipGetLastError();
    } else {
      return LMK_ERR_UNSUPPORTED;
    }
  }
  if (p.merge_slices > 0) {               // the selection stopped after its slice step: blocks of 32 as they are only
    if constexpr (BS == 32 && !PADDED) {
      if (rows <= 1024 && p.k > 1)
        hipLaunchKernelGGL((lmk_gather_attend_kernel<T, D, BS, true, PADDED, true>), dim3((unsigned)rows), dim3(256), 0, stream, p);
      else
        hipLaunchKernelGGL((lmk_gather_attend_kernel<T, D, BS, false, PADDED, true>), dim3((unsigned)((rows + 3) / 4)), dim3(256),
                           0, stream, p);
      return (int)hipGetLastError();
    } else {
      return LMK_ERR_UNSUPPORTED;
    }
  }
  if (rows <= 1024 && p.k > 1) {          // fewer rows than SIMDs: one workgroup per row, its waves share the blocks out
    hipLaunchKernelGGL((lmk_gather_attend_kernel<T, D, BS, true, PADDED>), dim3((unsigned)rows), dim3(256), 0, stream, p);
  } else {
    hipLaunchKernelGGL((lmk_gather_attend_kernel<T, D, BS, false, PADDED>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0,
                       stream, p);
  }
  return (int)hipGetLastError();
}

// BS: slots a block is worked on in (32, 64, 128); p.block: tokens of a block in the cache (<= BS)
template <class T, int D>
static int launch_gather_t(const RetrParams& p, int BS, hipStream_t stream) {
  if (p.block > BS || p.block < 2) return LMK_ERR_UNSUPPORTED;
  if (p.block == BS) {
    if (BS == 32) return launch_gather_b<T, D, 32, false>(p, stream);
    if (BS == 64) return launch_gather_b<T, D, 64, false>(p, stream);
    if (BS == 128) return launch_gather_b<T, D, 128, false>(p, stream);
  } else {
    if (BS == 64) return launch_gather_b<T, D, 64, true>(p, stream);
    if (BS == 128) return launch_gather_b<T, D, 128, true>(p, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

// ---------------------------------------------------------------------------
// local window: [cached tail | new chunk] when the cache ends in an incomplete block
// (llama_mem.py:321-342), optionally behind the k blocks one per-head selection picked
// (:386-388, :400-406).  One 16-byte chunk per thread:
//   k_win = [rot(selected keys, slot positions) ; rot(tail keys, positions full_len ..) ; k_loc]
//   v_win = [selected values ; tail values ; v_loc]
//   q_win = [zero rows for the tail ; q]   -- rows in front of the queries so that the fused forward
//           kernel, run with the selected blocks as history, yields the new tokens' attention in its
//           last T rows
// ---------------------------------------------------------------------------
template <class T, int D>
__global__ __launch_bounds__(256) void lmk_local_window_kernel(WindowParams p) {
  constexpr int LPR = D / 8;
  constexpr int RPW = 256 / LPR;
  const int tid = threadIdx.x, j = tid % LPR;
  const int W = p.n_sel + p.inc + p.T;
  const uint32_t row = blockIdx.x * RPW + tid / LPR;              // (bh, r); 32-bit as every launch's threads are
  const int bh = (int)(row / (uint32_t)W), r = (int)(row - (uint32_t)bh * W);
  if (bh >= p.B * p.H) return;
  const int b = (int)((uint32_t)bh / (uint32_t)p.H), hh = bh - b * p.H;
  u32x4_t qo = {0, 0, 0, 0}, ko, vo;
  if (r < p.n_sel + p.inc) {
    int64_t src_row, pos;
    if (r < p.n_sel) {
      const int slot = (int)((uint32_t)r / (uint32_t)p.block), tok = r - slot * p.block;
      int64_t blk = p.idx[(int64_t)bh * p.k + slot];
      blk = blk < 0 ? 0 : (blk >= p.num_mems ? p.num_mems - 1 : blk);   // never read outside the cache
      src_row = blk * p.block + tok;
      pos = (int64_t)r + (blk >= p.num_mems - p.k ? p.block : 0) + p.prefix_len;   // llama_mem.py:386-388
    } else {
      src_row = p.full_len + (r - p.n_sel);
      pos = p.tail_pos + (r - p.n_sel);
    }
    const char* src = (const char*)p.kcache + 2 * (b * p.kcs_b + hh * p.kcs_h + src_row * p.kcs_r);
    const u32x4_t x = *(const u32x4_t*)(src + 16 * j);
    const u32x4_t other = *(const u32x4_t*)(src + 16 * (j ^ (LPR / 2)));
    const u32x4_t c = *(const u32x4_t*)((const char*)p.cos + 2 * (pos * p.cs_r) + 16 * j);
    const u32x4_t s = *(const u32x4_t*)((const char*)p.sin + 2 * (pos * p.cs_r) + 16 * j);
    float o[8];
    rotate_chunk<T>(x, other, c, s, j >= LPR / 2, o);
    ko = u32x4_t{pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]), pack2<T>(o[4], o[5]), pack2<T>(o[6], o[7])};
    vo = *(const u32x4_t*)((const char*)p.vcache + 2 * (b * p.vcs_b + hh * p.vcs_h + src_row * p.vcs_r) + 16 * j);
  } else {
    const int t = r - p.n_sel - p.inc;
    qo = *(const u32x4_t*)((const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h + t * p.qs_r) + 16 * j);
    ko = *(const u32x4_t*)((const char*)p.k_loc + 2 * (b * p.kls_b + hh * p.kls_h + t * p.kls_r) + 16 * j);
    vo = *(const u32x4_t*)((const char*)p.v_loc + 2 * (b * p.vls_b + hh * p.vls_h + t * p.vls_r) + 16 * j);
  }
  if (r >= p.n_sel && p.q_win != nullptr)
    *(u32x4_t*)((char*)p.q_win + 2 * (b * p.qws_b + hh * p.qws_h + (int64_t)(r - p.n_sel) * p.qws_r) + 16 * j) = qo;
  *(u32x4_t*)((char*)p.k_win + 2 * (b * p.kws_b + hh * p.kws_h + (int64_t)r * p.kws_r) + 16 * j) = ko;
  *(u32x4_t*)((char*)p.v_win + 2 * (b * p.vws_b + hh * p.vws_h + (int64_t)r * p.vws_r) + 16 * j) = vo;
}

template <class T, int D>
static int launch_window_t(const WindowParams& p, hipStream_t stream) {
  constexpr int RPW = 256 / (D / 8);
  const int64_t rows = (int64_t)p.B * p.H * (p.n_sel + p.inc + p.T);
  hipLaunchKernelGGL((lmk_local_window_kernel<T, D>), dim3((unsigned)((rows + RPW - 1) / RPW)), dim3(256), 0, stream, p);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// rotary embedding of a whole (B, H, L, D) tensor at per-(batch, token) positions
// (apply_rotary_pos_emb, llama_mem.py:134-149): x*cos + rotate_half(x)*sin with the model dtype's
// rounding after each of the three elementwise operations.  A thread takes the 16-byte chunk j of a row's first half and
// its partner of the second, so that every value is read once, and reads both before it stores either: out may be x itself.
// PAIR: a second tensor of the same shape (the layer's q and k, :298) is rotated by the same thread with the
// same table rows, in the same launch.
// Rows that lie side by side in memory -- the heads of a token in (B, L, H, D)-backed views -- are taken side by side, and
// workgroups over the ends of batches: with one token of one head of 64 in each of 8192 batches, workgroups of one batch take
// 11.9 us, these 5.2; 8 heads 12.7 and 8.4.
// Bound by memory: 2 x 128 heads of 512 rows of 128 (67 MB) take 13.2 us, 5.1 TB/s; with 64-bit row indices, 73 wide multiplies
// a thread, and every row read twice 14.7.
// ---------------------------------------------------------------------------
template <class T, int D, bool PAIR>
__global__ __launch_bounds__(256) void lmk_rotary_kernel(RotaryParams p, int heads_inner) {
  constexpr int LPR = D / 16;
  constexpr int RPW = 256 / LPR;
  const int tid = threadIdx.x, j = tid % LPR;
  const uint32_t n = blockIdx.x * RPW + tid / LPR;                // row of the launch's batches, 32-bit as its threads are
  const uint32_t inner = heads_inner ? p.H : p.L, outer = heads_inner ? p.L : p.H;
  const uint32_t qb = n / inner, bl = qb / outer;
  const int q = (int)(qb - bl * outer), r = (int)(n - qb * inner);
  const int l = heads_inner ? q : r, hh = heads_inner ? r : q, b = p.b0 + (int)bl;
  if (b >= p.B) return;                                           // p.B: the end of the launch's batches
  int64_t pos = p.pos[(int64_t)b * p.pos_stride_b + l];
  pos = pos < 0 ? 0 : (pos >= p.n_pos ? p.n_pos - 1 : pos);      // never read outside the tables
  const char* src = (const char*)p.x + 2 * (b * p.xs_b + hh * p.xs_h + (int64_t)l * p.xs_r) + 16 * j;
  const u32x4_t lo = *(const u32x4_t*)src, hi = *(const u32x4_t*)(src + D);
  u32x4_t lo2 = {0, 0, 0, 0}, hi2 = {0, 0, 0, 0};
  if (PAIR) {                                                     // the second tensor's row at the same (b, h, l)
    const char* src2 = (const char*)p.x2 + 2 * (b * p.x2s_b + hh * p.x2s_h + (int64_t)l * p.x2s_r) + 16 * j;
    lo2 = *(const u32x4_t*)src2;
    hi2 = *(const u32x4_t*)(src2 + D);
  }
  const char *cr = (const char*)p.cos + 2 * (pos * p.cs_r) + 16 * j, *sr = (const char*)p.sin + 2 * (pos * p.cs_r) + 16 * j;
  const u32x4_t cl = *(const u32x4_t*)cr, ch = *(const u32x4_t*)(cr + D);
  u32x4_t sl = *(const u32x4_t*)(sr + (p.transposed ? D : 0)), sh = *(const u32x4_t*)(sr + (p.transposed ? 0 : D));
  const uint32_t flip = p.transposed ? 0x80008000u : 0u;         // sign bits of two 16-bit values
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    sl[i] ^= flip;
    sh[i] ^= flip;
  }
  auto rotate = [&](const u32x4_t& a, const u32x4_t& z, char* dst) __attribute__((always_inline)) {
    float o[8];
    rotate_chunk<T>(a, z, cl, sl, false, o);
    const u32x4_t x = {pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]), pack2<T>(o[4], o[5]), pack2<T>(o[6], o[7])};
    rotate_chunk<T>(z, a, ch, sh, true, o);
    const u32x4_t y = {pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]), pack2<T>(o[4], o[5]), pack2<T>(o[6], o[7])};
    *(u32x4_t*)dst = x;
    *(u32x4_t*)(dst + D) = y;
  };
  rotate(lo, hi, (char*)p.out + 2 * (b * p.os_b + hh * p.os_h + (int64_t)l * p.os_r) + 16 * j);
  if (PAIR) rotate(lo2, hi2, (char*)p.out2 + 2 * (b * p.o2s_b + hh * p.o2s_h + (int64_t)l * p.o2s_r) + 16 * j);
}

template <class T, int D>
static int launch_rotary_t(const RotaryParams& p, hipStream_t stream) {
  constexpr int RPW = 256 / (D / 16);
  const int64_t rows = (int64_t)p.H * p.L;                        // of a batch
  const int heads_inner = p.xs_h < p.xs_r ? 1 : 0;
  const int per = (int)std::max<int64_t>(1, std::min<int64_t>(p.B, (((int64_t)1 << 31) / (D / 16)) / rows));   // batches of a launch: 2^31 threads
  RotaryParams c = p;
  for (c.b0 = 0; c.b0 < p.B; c.b0 += per) {
    c.B = std::min(p.B - c.b0, per) + c.b0;
    const dim3 grid((unsigned)(((c.B - c.b0) * rows + RPW - 1) / RPW));
    if (p.x2 != nullptr) hipLaunchKernelGGL((lmk_rotary_kernel<T, D, true>), grid, dim3(256), 0, stream, c, heads_inner);
    else hipLaunchKernelGGL((lmk_rotary_kernel<T, D, false>), grid, dim3(256), 0, stream, c, heads_inner);
  }
  return (int)hipGetLastError();
}

// New rows of a cache's keys (blockIdx.y 0) and values (1), one 16-byte chunk per thread.
__global__ __launch_bounds__(256) void lmk_copy_rows_kernel(CopyRowsParams p) {
  const int w = blockIdx.y;
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;              // 32-bit as every launch's threads are
  const uint32_t row = i / (uint32_t)p.chunks;
  const int c = (int)(i - row * p.chunks);
  const int bh = (int)(row / (uint32_t)p.T), t = (int)(row - (uint32_t)bh * p.T);
  if (bh >= p.B * p.H) return;
  const int b = (int)((uint32_t)bh / (uint32_t)p.H), h = bh - b * p.H;
  const char* s = (const char*)p.src[w] + 2 * (b * p.ss_b[w] + h * p.ss_h[w] + t * p.ss_r[w]) + 16 * c;
  char* d = (char*)p.dst[w] + 2 * (b * p.ds_b[w] + h * p.ds_h[w] + t * p.ds_r[w]) + 16 * c;
  *(u32x4_t*)d = *(const u32x4_t*)s;
}

// One 16-byte chunk per thread of the rows [tail ; new tokens] of keys (blockIdx.y 0) and values (1); blockIdx.y 2: the
// new tail's marks, a byte per thread.  A tail row is read and overwritten in the same launch, so its thread does both:
// row i < n_tail goes to the ring and then, if the new tail has a row i, fetches that row too.
__global__ __launch_bounds__(256) void lmk_ring_store_kernel(RingStoreParams p) {
  const int w = blockIdx.y, rows = p.n_tail + p.T, rest = rows - p.full;
  const uint32_t n = blockIdx.x * 256 + threadIdx.x;              // 32-bit as every launch's threads are
  if (w == 2) {
    const int b = (int)(n / (uint32_t)p.block), j = (int)(n - (uint32_t)b * p.block);
    const int src = p.full + j - p.n_tail;                        // token of the chunk behind row j of the tail; < 0: row j stays
    if (b < p.B && j < rest && src >= 0) p.tail_is_mem[b * p.tims_b + j] = p.is_mem[b * p.ims_b + src];
    return;
  }
  const uint32_t bhi = n / (uint32_t)p.chunks;
  const int c = (int)(n - bhi * p.chunks);
  const int bh = (int)(bhi / (uint32_t)rows), i = (int)(bhi - (uint32_t)bh * rows);
  if (bh >= p.B * p.H) return;
  const int b = (int)((uint32_t)bh / (uint32_t)p.H), h = bh - b * p.H;
  const char* src = (const char*)p.src[w] + 2 * (b * p.ss_b[w] + h * p.ss_h[w]) + 16 * c;
  char* tail = (char*)p.tail[w] + 2 * (b * p.ts_b[w] + h * p.ts_h[w]) + 16 * c;
  auto chunk_row = [&](int t) { return *(const u32x4_t*)(src + 2 * t * p.ss_r[w]); };
  auto tail_row = [&](int j) { return (u32x4_t*)(tail + 2 * j * p.ts_r[w]); };
  if (i < p.full) {
    const u32x4_t x = i < p.n_tail ? *tail_row(i) : chunk_row(i - p.n_tail);
    const int whole = (int)((uint32_t)i / (uint32_t)p.block), blk = whole - p.dropped;
    if (blk >= 0) {
      const int slot = (int)((uint32_t)(p.first_slot + blk) % (uint32_t)p.n_slots);
      *(u32x4_t*)((char*)p.ring[w] + 2 * (b * p.rs_b + slot * p.rs_slot + (i - whole * p.block) * p.rs_tok + h * p.rs_h) + 16 * c) = x;
    }
    if (i < p.n_tail && i < rest) *tail_row(i) = chunk_row(p.full + i - p.n_tail);   // full > n_tail: a token of the chunk
  } else {
    const int j = i - p.full;                                     // row of the new tail
    if (p.full > 0 ? j >= p.n_tail : i >= p.n_tail) *tail_row(j) = chunk_row(i - p.n_tail);
  }
}

int launch_ring_store(const RingStoreParams& p, hipStream_t stream) {
  const int64_t n = (int64_t)p.B * p.H * (p.n_tail + p.T) * p.chunks, marks = (int64_t)p.B * p.block;
  hipLaunchKernelGGL(lmk_ring_store_kernel, dim3((unsigned)((std::max(n, marks) + 255) / 256), 3), dim3(256), 0, stream, p);
  return (int)hipGetLastError();
}

int launch_copy_rows(const CopyRowsParams& p, hipStream_t stream) {
  const int64_t n = (int64_t)p.B * p.H * p.T * p.chunks;
  hipLaunchKernelGGL(lmk_copy_rows_kernel, dim3((unsigned)((n + 255) / 256), 2), dim3(256), 0, stream, p);
  return (int)hipGetLastError();
}

int launch_rotary(const RotaryParams& p, int D, int dtype, hipStream_t stream) {
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_rotary_t<bf16_t, 128>(p, stream);
    if (D == 64) return launch_rotary_t<bf16_t, 64>(p, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_rotary_t<f16_t, 128>(p, stream);
    if (D == 64) return launch_rotary_t<f16_t, 64>(p, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

int launch_local_window(const WindowParams& p, int D, int dtype, hipStream_t stream) {
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_window_t<bf16_t, 128>(p, stream);
    if (D == 64) return launch_window_t<bf16_t, 64>(p, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_window_t<f16_t, 128>(p, stream);
    if (D == 64) return launch_window_t<f16_t, 64>(p, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

int launch_gather_attend(const RetrParams& p, int D, int BS, int dtype, hipStream_t stream) {
  // A decode step of so many rows that waves of 16 KB each fill the chip whichever way: a wave per row is as fast and has no
  // waves for windows (2048 rows, block 64, top 6, D128: 92.2 us against 94.5; 1024 rows: 80.7 against 57.6)
  if (p.local && !(D == 128 && BS <= 64 && (int64_t)p.B * p.H * p.T > 4 * cu_count())) return launch_gather_decode(p, D, dtype, stream);
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_gather_t<bf16_t, 128>(p, BS, stream);
    if (D == 64) return launch_gather_t<bf16_t, 64>(p, BS, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_gather_t<f16_t, 128>(p, BS, stream);
    if (D == 64) return launch_gather_t<f16_t, 64>(p, BS, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

}  // namespace lmk
