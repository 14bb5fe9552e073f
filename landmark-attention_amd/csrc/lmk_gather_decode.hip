// Gather + attend of a decode step: a row's picked cache blocks and its local window -- the tokens of the cache behind its
// last complete block and the new tokens up to the row's own, at most one block together -- in one launch, a workgroup per
// row: a wave for every picked block (up to eight), one for the window.
//
// The step reads 16 KB of keys and 16 KB of values per block and row once, from memory, and has to have them on their way
// early: a block's keys go straight into LDS, all of them requested at once; its values into registers, requested while
// the scores are formed.  The memory counter of a wave counts in order, so what is waited for first is requested first:
// keys, then the table rows of the first two groups of 16 keys, then a group's table rows while the group two in front of
// it is worked on, and the values only behind the last of them -- requested earlier, every wait for a table row from the L2
// would be one for values from memory (which is what the kernel that fetched a chunk of keys or values ahead and then the
// table rows did: four trips to memory one after the other, 64 us for the 177 MB of 1024 rows of five blocks of 64).
// 1024 rows over 4096 tokens, five blocks of 64, D128: 63.4 -> 41.5 us, the step 74 -> 52; four blocks of 128: 1.3 times as fast.
//
// Eight lanes share a key: lane j of the group holds head dims 8j .. and 64 + 8j .. (head dim 64: 4j .. and 32 + 4j ..), i.e. both
// partners of the rotary pair; the eight groups of the wave take keys g, g + 8 of 16.  Rotation and scores are fp32 from the
// 16-bit cache and tables.
#include <algorithm>

#include "lmk_common.hpp"
#include "lmk_launch.hpp"
#include "lmk_split.hpp"
#include "lmk_topk_slice.hpp"

namespace lmk {

constexpr int kDecodeWaves = 8;                         // waves for the blocks, at most

template <int D, int BS>
struct DecodeCfg {
  static constexpr int E = D / 16;                      // head dims per lane and rotary half: 8 or 4
  static constexpr int PB = 2 * E;                      // bytes of one piece
  static constexpr int ROWB = 2 * D;
  static constexpr int CH = D / 8;                      // 16-byte chunks per row
  static constexpr int NG = BS / 16;                    // groups of 16 keys
  static constexpr int REGION = BS * ROWB;              // LDS of a wave: its block's keys, at the end its partial sums
  static constexpr int REQ = REGION / 1024;             // requests of 1 KB
  static constexpr int RPD = 1024 / ROWB;               // rows per request
};
template <int E> struct DecodePiece;
template <> struct DecodePiece<8> { using type = u32x4_t; };
template <> struct DecodePiece<4> { using type = u32x2_t; };

// Eight groups of eight lanes read the first (or second) halves of eight rows at a time: the halves of a row change places
// where that spreads the rows over the banks' 256 bytes.
template <int D>
__device__ __forceinline__ int decode_swizzle(int row) { return D == 128 ? (row & 1) << 3 : (row & 2) << 1; }

__device__ __forceinline__ float sum_of_8(float d) {    // over the lanes of a key
  d += dpp_f<0xB1>(d);                                  // quad_perm [1,0,3,2]
  d += dpp_f<0x4E>(d);                                  // quad_perm [2,3,0,1]
  d += dpp_f<0x141>(d);                                 // row_half_mirror
  return d;
}
__device__ __forceinline__ float max_over_groups(float x) {
  x = fmaxf(x, dpp_f<0x128>(x));                        // row_ror 8: the other key group of the 16 lanes
  x = fmaxf(x, __shfl_xor(x, 16, 64));
  return fmaxf(x, __shfl_xor(x, 32, 64));
}
__device__ __forceinline__ float sum_over_groups(float x) {
  x += dpp_f<0x128>(x);
  x += __shfl_xor(x, 16, 64);
  return x + __shfl_xor(x, 32, 64);
}

// MERGE: the selection stopped after its slice step (p.merge_slices > 0); the row's blocks are picked from the slices'
// candidates first.
template <class T, int D, int BS, bool MERGE>
__global__ __launch_bounds__(64 * (kDecodeWaves + 1), 3) void lmk_gather_decode_kernel(RetrParams p) {
  using C = DecodeCfg<D, BS>;
  constexpr int E = C::E, PB = C::PB, NG = C::NG;
  using vec_t = typename DecodePiece<E>::type;          // one piece: E 16-bit values
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 7, g = lane >> 3;
  const uint32_t row = blockIdx.x;
  const int bh = (int)(row / (uint32_t)p.T), t = (int)(row - (uint32_t)bh * p.T);
  const int b = (int)((uint32_t)bh / (uint32_t)p.H), hh = bh - b * p.H;
  const char* kc = (const char*)p.kcache + 2 * (b * p.kcs_b + hh * p.kcs_h);
  const char* vc = (const char*)p.vcache + 2 * (b * p.vcs_b + hh * p.vcs_h);
  const float c2 = p.scale_log2;
  auto unpack = [](const vec_t u, float* o) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < E / 2; ++i) {
      o[2 * i] = unpack_lo<T>(u[i]);
      o[2 * i + 1] = unpack_hi<T>(u[i]);
    }
  };
  float qlo[E], qhi[E];
  {
    const char* qp = (const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h + (int64_t)t * p.qs_r) + PB * j;
    unpack(*(const vec_t*)qp, qlo);
    unpack(*(const vec_t*)(qp + D), qhi);
  }
  float Mrun = kNoScore, lrun = 0.f;                    // global bucket: maximum (log2 domain), sum
  float alo[E], ahi[E];
#pragma unroll
  for (int i = 0; i < E; ++i) alo[i] = ahi[i] = 0.f;
  auto accumulate = [&](float w, const vec_t lo, const vec_t hi) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < E / 2; ++e) {
      alo[2 * e] = __builtin_fmaf(w, unpack_lo<T>(lo[e]), alo[2 * e]);
      alo[2 * e + 1] = __builtin_fmaf(w, unpack_hi<T>(lo[e]), alo[2 * e + 1]);
      ahi[2 * e] = __builtin_fmaf(w, unpack_lo<T>(hi[e]), ahi[2 * e]);
      ahi[2 * e + 1] = __builtin_fmaf(w, unpack_hi<T>(hi[e]), ahi[2 * e + 1]);
    }
  };
  auto over_groups = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      alo[e] = sum_over_groups(alo[e]);
      ahi[e] = sum_over_groups(ahi[e]);
    }
  };

  if (wave < p.block_waves) {
    // ---- the row's blocks js = wave, wave + block_waves, ..
    const int64_t* idx_row = p.idx + (b * p.idx_sb + hh * p.idx_sh + (int64_t)t * p.idx_st);
    int sorted = 0;                                     // lane r: the r-th block in the order of the output
    if constexpr (MERGE) {
      int mine = merge_slices_row(p, p.merge_slices, row, lane);
      const int rank = rank_ascending(mine, lane, p.k, p.num_mems, p.ring_start);
      sorted = __builtin_amdgcn_ds_permute(4 * (lane < p.k ? rank : lane), mine);
      if (lane < p.k && wave == 0) p.idx[b * p.idx_sb + hh * p.idx_sh + (int64_t)t * p.idx_st + rank] = (int64_t)mine;
    }
    const int region = wave * C::REGION;
    for (int js = wave; js < p.k; js += p.block_waves) {
      const int blk = MERGE ? __builtin_amdgcn_readlane(sorted, js)   // idx is a caller's array: never read outside the cache
                            : __builtin_amdgcn_readfirstlane(min(max((int)idx_row[js], 0), p.num_mems - 1));
      int age = blk - p.ring_start;                     // one of the k newest blocks: its keys sit one block further on
      age += age < 0 ? p.num_mems : 0;
      const int64_t pos0 = (int64_t)js * BS + (age >= p.num_mems - p.k ? BS : 0) + p.prefix_len;
      const char* kb = kc + 2 * ((int64_t)blk * BS * p.kcs_r);
      const char* vb = vc + 2 * ((int64_t)blk * BS * p.vcs_r);
      const char *cb = (const char*)p.cos + 2 * (pos0 * p.cs_r), *sb = (const char*)p.sin + 2 * (pos0 * p.cs_r);
      __builtin_amdgcn_s_waitcnt(0xc07f);               // the block before: its keys have been read
      // What the addresses have in common per lane, in 32 bits (gather_takes_local_window); formed here, or the loop would keep
      // forty sums of it.
      int ln = lane;
      asm volatile("" : "+v"(ln));
      {
        const int r0 = ln / C::CH;                      // (the swizzle of row RPD i + r0 is that of r0)
        const uint32_t off = (uint32_t)r0 * (uint32_t)(2 * p.kcs_r) + 16 * ((ln % C::CH) ^ decode_swizzle<D>(r0));
#pragma unroll
        for (int i = 0; i < C::REQ; ++i) {
          split_dma16(kb, off, region + 1024 * i);
          kb += (int64_t)C::RPD * (2 * p.kcs_r);
          asm volatile("" : "+s"(kb));                  // one pointer, not one per request
        }
      }
      const uint32_t off_t = (uint32_t)(ln >> 3) * (uint32_t)(2 * p.cs_r) + PB * (ln & 7);
      const uint32_t off_v = (uint32_t)(ln >> 3) * (uint32_t)(2 * p.vcs_r) + PB * (ln & 7);
      const int at = region + (ln >> 3) * C::ROWB + ((16 * decode_swizzle<D>(ln >> 3)) ^ (PB * (ln & 7)));   // PB j < D: the swizzle turns the half's bit
      vec_t tab[2][2][4];                               // a group's table rows: cos, sin of this lane's two keys, both halves
      auto fetch_tables = [&](int x) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          vec_t* o = tab[x & 1][i];
          o[0] = *(const vec_t*)(cb + off_t);
          o[1] = *(const vec_t*)(cb + off_t + D);
          o[2] = *(const vec_t*)(sb + off_t);
          o[3] = *(const vec_t*)(sb + off_t + D);
          cb += 8 * (2 * p.cs_r);                       // groups come in order
          sb += 8 * (2 * p.cs_r);
          asm volatile("" : "+s"(cb), "+s"(sb));
        }
      };
      vec_t val[4][2][2];                               // values of four groups on their way
      auto fetch_values = [&](int x) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          val[x & 3][i][0] = *(const vec_t*)(vb + off_v);
          val[x & 3][i][1] = *(const vec_t*)(vb + off_v + D);
          vb += 8 * (2 * p.vcs_r);
          asm volatile("" : "+s"(vb));
        }
      };
      fetch_tables(0);
      fetch_tables(1);
      if (NG == 2) fetch_values(0);
      // the keys are older than everything else: with that still on its way they have landed
      constexpr int YOUNGER = 16 + (NG == 2 ? 4 : 0);
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"(YOUNGER) : "memory");
      float sc[2 * NG];
#pragma unroll
      for (int x = 0; x < NG; ++x) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int r = at + (16 * x + 8 * i) * C::ROWB;
          float kl[E], kh[E], cl[E], ch[E], sl[E], sh[E];
          unpack(*(const vec_t*)(smem + r), kl);
          unpack(*(const vec_t*)(smem + (r ^ D)), kh);
          unpack(tab[x & 1][i][0], cl);
          unpack(tab[x & 1][i][1], ch);
          unpack(tab[x & 1][i][2], sl);
          unpack(tab[x & 1][i][3], sh);
          float d = 0.f;
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const float rl = __builtin_fmaf(kl[e], cl[e], -kh[e] * sl[e]);
            const float rh = __builtin_fmaf(kh[e], ch[e], kl[e] * sh[e]);
            d = __builtin_fmaf(qlo[e], rl, d);
            d = __builtin_fmaf(qhi[e], rh, d);
          }
          sc[2 * x + i] = sum_of_8(d) * c2;             // log2 domain
          __builtin_amdgcn_sched_barrier(0);            // one key's 48 numbers at a time
        }
        if (x + 2 < NG) fetch_tables(x + 2);
        // the last table rows are requested: now the values, as registers get free
        if (NG == 2 && x == 0) fetch_values(1);
        if (NG == 4 && x == 1) fetch_values(0);
        if (NG > 2 && x + 2 == NG) {
          if (NG > 4) fetch_values(0);
          fetch_values(1);
          if (NG == 4) fetch_values(2);
        }
        if (NG > 2 && x + 1 == NG) {
          if (NG > 4) fetch_values(2);
          fetch_values(3);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // landmark = key BS - 1: last group, i = 1, g = 7
      const float t_lm = __shfl(sc[2 * NG - 1], 56, 64);
      if (g == 7) sc[2 * NG - 1] = -INFINITY;
      float mx = sc[0];
#pragma unroll
      for (int i = 1; i < 2 * NG; ++i) mx = fmaxf(mx, sc[i]);
      mx = max_over_groups(mx);
      float den = 0.f;
#pragma unroll
      for (int i = 0; i < 2 * NG; ++i) {
        float e = fast_exp2(sc[i] - mx);
        if (i == 2 * NG - 1 && g == 7) e = 0.f;
        sc[i] = e;
        den += e;
      }
      den = sum_over_groups(den);
      const float Mnew = fmaxf(Mrun, t_lm);
      const float alpha = fast_exp2(Mrun - Mnew), gate = fast_exp2(t_lm - Mnew);
      lrun = lrun * alpha + gate;
      Mrun = Mnew;
      const float f = gate / den;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        alo[e] *= alpha;
        ahi[e] *= alpha;
      }
#pragma unroll
      for (int x = 0; x < NG; ++x) {
#pragma unroll
        for (int i = 0; i < 2; ++i) accumulate(round_to<T>(sc[2 * x + i] * f), val[x & 3][i][0], val[x & 3][i][1]);   // weights enter PV in the model dtype
        if (x + 4 < NG) fetch_values(x + 4);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    over_groups();
    // partial (M, l, acc) for the window's wave, over the keys, which nobody reads any more
    __builtin_amdgcn_s_waitcnt(0xc07f);
    float* part = (float*)(smem + region);
    if (g == 0) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        part[E * j + e] = alo[e];
        part[D / 2 + E * j + e] = ahi[e];
      }
      if (j == 0) {
        part[D] = Mrun;
        part[D + 1] = lrun;
      }
    }
    __syncthreads();
    return;
  }

  // ---- the window: inc rows of the cache, then the new tokens; keys join the global bucket directly (own-block rule:
  // causal, the landmark token does not see itself; flash_landmark_attention.py:78-100)
  // The row's own key (without rotary) and value on their way into the cache (lanes 0 .. D/8-1 the key, 32 .. the value).
  // Nobody reads the destination in this launch: it lies behind the cached rows.
  const bool appends = p.ap_k != nullptr && (lane & 31) < D / 8;
  u32x4_t ap = {0, 0, 0, 0};
  if (appends)
    ap = *(const u32x4_t*)((lane < 32 ? (const char*)p.ap_k + 2 * (b * p.aks_b + hh * p.aks_h + (int64_t)t * p.aks_r)
                                      : (const char*)p.ap_v + 2 * (b * p.avs_b + hh * p.avs_h + (int64_t)t * p.avs_r)) +
                           16 * (lane & 31));
  {
    const int inc = p.local_inc, own = inc + t;
    const char* kn = (const char*)p.k_new + 2 * (b * p.kns_b + hh * p.kns_h);
    const char* vn = (const char*)p.v_new + 2 * (b * p.vns_b + hh * p.vns_h);
    const int last = own >> 4;                          // the row's own token's group of 16: the groups behind it are skipped
    float sc[2 * NG];
    vec_t key[2][2][2], tab[2][2][4], val[4][2][2];
    auto fetch_keys = [&](int x) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int rc = min(16 * x + 8 * i + g, own);    // rows behind the row's own are never read
        const bool cached = rc < inc;
        const char* kr = (cached ? kc + 2 * ((p.local_row0 + rc) * p.kcs_r) : kn + 2 * ((int64_t)(rc - inc) * p.kns_r)) + PB * j;
        const int64_t pos = inc > 0 ? p.local_pos0 + min(rc, inc - 1) : 0;   // a position the tables hold, used by cached rows only
        const char *cr = (const char*)p.cos + 2 * (pos * p.cs_r) + PB * j, *sr = (const char*)p.sin + 2 * (pos * p.cs_r) + PB * j;
        key[x & 1][i][0] = *(const vec_t*)kr;
        key[x & 1][i][1] = *(const vec_t*)(kr + D);
        tab[x & 1][i][0] = *(const vec_t*)cr;
        tab[x & 1][i][1] = *(const vec_t*)(cr + D);
        tab[x & 1][i][2] = *(const vec_t*)sr;
        tab[x & 1][i][3] = *(const vec_t*)(sr + D);
      }
    };
    auto fetch_values = [&](int x) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int rc = min(16 * x + 8 * i + g, own);
        const char* vr = (rc < inc ? vc + 2 * ((p.local_row0 + rc) * p.vcs_r) : vn + 2 * ((int64_t)(rc - inc) * p.vns_r)) + PB * j;
        val[x & 3][i][0] = *(const vec_t*)vr;
        val[x & 3][i][1] = *(const vec_t*)(vr + D);
      }
    };
    fetch_keys(0);                                      // (a group behind the last is a re-read of the own row)
    fetch_keys(1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < NG; ++x) {
      if (x > last) {                                   // wave-uniform
        sc[2 * x] = sc[2 * x + 1] = -INFINITY;
        continue;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 16 * x + 8 * i + g;
        const bool visible = r <= own && !(r == BS - 1 && own == BS - 1), cached = min(r, own) < inc;
        float kl[E], kh[E], cl[E], ch[E], sl[E], sh[E];
        unpack(key[x & 1][i][0], kl);
        unpack(key[x & 1][i][1], kh);
        unpack(tab[x & 1][i][0], cl);
        unpack(tab[x & 1][i][1], ch);
        unpack(tab[x & 1][i][2], sl);
        unpack(tab[x & 1][i][3], sh);
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {                   // cached keys are rotated in the model dtype, as the cache's window is (llama_mem.py:336-338)
          const float rl = cached ? round_to<T>(__builtin_fmaf(kl[e], cl[e], -kh[e] * sl[e])) : kl[e];
          const float rh = cached ? round_to<T>(__builtin_fmaf(kh[e], ch[e], kl[e] * sh[e])) : kh[e];
          d = __builtin_fmaf(qlo[e], rl, d);
          d = __builtin_fmaf(qhi[e], rh, d);
        }
        sc[2 * x + i] = visible ? sum_of_8(d) * c2 : -INFINITY;
        __builtin_amdgcn_sched_barrier(0);
      }
      if (x + 2 < NG && x + 2 <= last) fetch_keys(x + 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    fetch_values(0);
#pragma unroll
    for (int x = 1; x < 4 && x < NG; ++x)
      if (x <= last) fetch_values(x);
    __builtin_amdgcn_sched_barrier(0);
    float mx = sc[0];                                   // row 0 is always visible
#pragma unroll
    for (int i = 1; i < 2 * NG; ++i) mx = fmaxf(mx, sc[i]);
    mx = max_over_groups(mx);
    float den = 0.f;
#pragma unroll
    for (int x = 0; x < NG; ++x) {
      if (x > last) continue;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float e = fast_exp2(sc[2 * x + i] - mx);
        den += e;
        accumulate(round_to<T>(e), val[x & 3][i][0], val[x & 3][i][1]);   // weights enter PV in the model dtype
      }
      if (x + 4 < NG && x + 4 <= last) fetch_values(x + 4);
      __builtin_amdgcn_sched_barrier(0);
    }
    Mrun = mx;
    lrun = sum_over_groups(den);
  }
  if (appends)
    *(u32x4_t*)((lane < 32 ? (char*)p.ap_kd + 2 * (b * p.akd_b + hh * p.akd_h + (int64_t)t * p.akd_r)
                           : (char*)p.ap_vd + 2 * (b * p.avd_b + hh * p.avd_h + (int64_t)t * p.avd_r)) +
                16 * (lane & 31)) = ap;
  over_groups();
  __syncthreads();                                      // the blocks' partial sums are there
  const int nw = p.block_waves;
  float mw[kDecodeWaves], Mall = Mrun;
#pragma unroll
  for (int w = 0; w < kDecodeWaves; ++w) {
    mw[w] = ((const float*)(smem + min(w, nw - 1) * C::REGION))[D];
    mw[w] = w < nw ? mw[w] : -INFINITY;
    Mall = fmaxf(Mall, mw[w]);
  }
  const float sw0 = fast_exp2(Mrun - Mall);
  lrun *= sw0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    alo[e] *= sw0;
    ahi[e] *= sw0;
  }
#pragma unroll
  for (int w = 0; w < kDecodeWaves; ++w) {
    if (w < nw) {                                       // wave-uniform
      const float* part = (const float*)(smem + w * C::REGION);
      const float sw = fast_exp2(mw[w] - Mall);
      lrun = __builtin_fmaf(part[D + 1], sw, lrun);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        alo[e] = __builtin_fmaf(part[E * j + e], sw, alo[e]);
        ahi[e] = __builtin_fmaf(part[D / 2 + E * j + e], sw, ahi[e]);
      }
    }
  }
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
}

template <class T, int D, int BS>
static int launch_decode_t(RetrParams p, hipStream_t stream) {
  using C = DecodeCfg<D, BS>;
  // Waves for the blocks.  Up to a row per compute unit: a wave per block.  With more rows a compute unit should hold several
  // workgroups, one's first loads under another's arithmetic, and it holds those whose waves go around its SIMDs evenly: three
  // (head dim 64: four) of four waves, but one of five to eight where a SIMD takes three waves.  us a step by waves for the
  // blocks, D128: 512 rows, block 64, top 8: 8 46.8, 4 48.1, 3 43.1, 2 44.2; 1024 rows, top 5: 5 58.3, 3 55.6, 2 51.7 (with two, four
  // workgroups: all rows at once); block 128: 1024 rows, top 5: 5 110.6, 2 94.3, 1 85.3, 512 rows, top 4: 4 48.0, 2 43.5, 1 51.6;
  // D64, 512 rows, block 64, top 8: 8 30.0, 4 27.3, 3 28.5, 1024 rows, top 5: 5 39.7, 4 33.2, 3 32.8.  Over 300 to 1024 rows and top 1,
  // 2, 3, 4, 5 and 8 the lines below are within 1.3 % (geometric mean) of the best of one to four waves in every band, block and
  // head dim, but for 3 % at D64, block 128, above 768 rows; against the kernels of longer chunks 0.83 of the time, 1.04 at worst
  // (block 128, D128, top 6, 8 rows: 25.8 for 24.8; top 5 takes five waves, all of a compute unit's LDS: 20.7, with three 24.8).
  constexpr int most = std::min(kDecodeWaves, 163840 / C::REGION);
  const int64_t rows = (int64_t)p.B * p.H * p.T, cus = cu_count();
  int cap = most;
  if (rows > cus) {
    if (C::REGION > 16384) cap = rows > 2 * cus ? 1 : 2;
    else if (D == 64) cap = rows > 2 * cus ? 3 : std::min(7, 81920 / C::REGION);
    else cap = rows > 3 * cus && rows <= 4 * cus ? 2 : 3;
  }
  const int per = (p.k + cap - 1) / cap;                // blocks a wave walks one after the other
  p.block_waves = (p.k + per - 1) / per;
  const dim3 grid((unsigned)rows), wg(64 * (p.block_waves + 1));
  const int lds = p.block_waves * C::REGION;
  static std::atomic<uint64_t> lds_ok[2] = {{0}, {0}};
  auto kern = p.merge_slices > 0 ? lmk_gather_decode_kernel<T, D, BS, true> : lmk_gather_decode_kernel<T, D, BS, false>;
  if (int rc = allow_dynamic_lds(kern, most * C::REGION, lds_ok[p.merge_slices > 0])) return rc;
  hipLaunchKernelGGL(kern, grid, wg, lds, stream, p);
  return (int)hipGetLastError();
}

template <class T, int D>
static int launch_decode_d(const RetrParams& p, hipStream_t stream) {
  if (p.block == 32) return launch_decode_t<T, D, 32>(p, stream);
  if (p.block == 64) return launch_decode_t<T, D, 64>(p, stream);
  if (p.block == 128) return launch_decode_t<T, D, 128>(p, stream);
  return LMK_ERR_UNSUPPORTED;
}

int launch_gather_decode(const RetrParams& p, int D, int dtype, hipStream_t stream) {
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_decode_d<bf16_t, 128>(p, stream);
    if (D == 64) return launch_decode_d<bf16_t, 64>(p, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_decode_d<f16_t, 128>(p, stream);
    if (D == 64) return launch_decode_d<f16_t, 64>(p, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

}  // namespace lmk
