// Backward kernels of fused landmark attention for gfx950.
//
// Replace `_bwd_preprocess` and `_bwd_kernel` of the reference
// (llama/ltriton/flash_landmark_attention.py:125-149, :152-305).  The reference runs one
// program per (batch, head) and read-modify-writes dQ in global memory; here the work is
// split so that every accumulator stays in registers and no atomics are needed:
//
//   pre    delta = rowsum(O * dO),  mhat = M*log2(e) + log2(L)          (per query row; the dQ kernels do
//          this in their prologue, the separate kernel exists for timing the phases one by one)
//   dq     query-stationary, S^T layout (lane = query): recomputes the local softmax of
//          every earlier block, the gate, nD = rowsum(P * dP), forms dS and accumulates
//          dQ^T = K^T dS^T.  It also writes, per (query, earlier block), the three numbers
//          the third kernel needs:  a  with  gate*P = exp2(s*c - a),  nD,  and dS at the
//          block's landmark key.
//   dkdv   key-stationary, S layout (lane = key): purely elementwise between its four
//          products S = Q K^T, dP = dO V^T, dV^T += dO^T W, dK^T += Q^T dS
//          (lmk_bwd_dkdv_split.hip with 64 keys a workgroup, lmk_bwd_dkdv32.hip with 128).
// This file holds the pre kernel, the dQ kernel for many query rows of whole blocks of 64 keys (block 32 has its own in
// lmk_bwd_dq32.hip, everything else is lmk_bwd_dq_split.hip's) and the dispatch.
//
// All probabilities are used normalised (exp2(s*c - mhat) already divides by L), so dO is
// consumed as is; the reference's rescaled copy dO/L (:147) is not needed.
#include <cstdlib>
#include <type_traits>

#include "lmk_common.hpp"
#include "lmk_launch.hpp"

namespace lmk {

// ---------------------------------------------------------------------------
// pre: delta and mhat
// ---------------------------------------------------------------------------
template <class T, int D>
__global__ __launch_bounds__(256) void lmk_bwd_pre_kernel(BwdParams p, int block_slots) {
  constexpr int LPR = D / 8;          // lanes per row (16 bytes each)
  constexpr int RPW = 256 / LPR;      // rows per workgroup
  const int tid = threadIdx.x;
  const int64_t row = (int64_t)blockIdx.x * RPW + tid / LPR;
  const int64_t total = (int64_t)p.B * p.H * p.Lq;
  float sum = 0.f;
  int64_t li = row;                                         // index of the row in L and M; -1: a slot without a token
  if (row < total) {
    const int bh = (int)(row / p.Lq);
    int qi = (int)(row % p.Lq);
    if (p.Lq_real > 0) {                                    // token layout: the workspace rows are slots
      const int* seg_q = p.seg != nullptr ? p.seg + p.n_prefix : nullptr;   // the queries' first block
      qi = block_slots == 64 ? slot_to_token_row<64>(qi, p.n_real, p.n_full_q, seg_q)
                             : slot_to_token_row<128>(qi, p.n_real, p.n_full_q, seg_q);
      li = qi < 0 ? -1 : (int64_t)bh * p.Lq_real + qi;
    }
    if (qi >= 0) {
      const int b = bh / p.H, hh = bh % p.H;
      const int d0 = 8 * (tid % LPR);
      const u32x4_t o4 = *(const u32x4_t*)((const char*)p.o + 2 * (b * p.os_b + hh * p.os_h + (int64_t)qi * p.os_r + d0));
      const u32x4_t g4 = *(const u32x4_t*)((const char*)p.dout + 2 * (b * p.dos_b + hh * p.dos_h + (int64_t)qi * p.dos_r + d0));
#pragma unroll
      for (int i = 0; i < 4; ++i)
        sum += unpack_lo<T>(o4[i]) * unpack_lo<T>(g4[i]) + unpack_hi<T>(o4[i]) * unpack_hi<T>(g4[i]);
    }
  }
#pragma unroll
  for (int m = LPR / 2; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, 64);
  if (row < total && (tid % LPR) == 0) {
    p.delta[row] = sum;
    p.mhat[row] = li < 0 ? 1e30f : p.M[li] * kLog2e + fast_log2(p.L[li]);
  }
}

// ---------------------------------------------------------------------------
// dq (+ per-block statistics), landmark blocks of 64 keys, many query rows
// ---------------------------------------------------------------------------
// A workgroup is 8 waves = 256 query rows, two waves per SIMD; a wave keeps the fragments of its 32
// rows of Q and dO and its dQ^T accumulator in registers.  One stage is one landmark block: its K and
// V rows come into one of two LDS buffers by direct global->LDS loads (no staging registers: the kernel
// has to stay inside 256 registers for two waves to share a SIMD), requested one stage ahead, each wave
// fetching its share; one barrier per stage.  The block's local softmax needs all its scores before any
// weight is final, so the S^T tiles of the whole block stay in registers.
template <class T, int D>
struct DqCfg {
  static constexpr int BS = 64;
  static constexpr int NT = BS / 32;                       // MFMA tiles per landmark block
  static constexpr int NW = 8;
  static constexpr int CH = D / 8;
  static constexpr int KS = D / 16;
  static constexpr int DC = D / 32;
  static constexpr int ROWB = 2 * D;
  static constexpr int TILE_BYTES = BS * ROWB;             // K (or V) of one block
  static constexpr int STAGE_BYTES = 2 * TILE_BYTES;       // K, then V
  static constexpr int LDS_BYTES = 2 * STAGE_BYTES;
  static constexpr int RPD = 1024 / ROWB;                  // rows covered by one 1 KB request
  static constexpr int NREQ = 2 * BS / RPD;                // requests per stage
  static constexpr int PER_WAVE = NREQ / NW;
  static_assert(NREQ % NW == 0, "every wave issues the same number of requests");
};

// One 1 KB direct global->LDS request of a wave: lane i's 16 bytes land at lds_off + 16*i.
// lds_off must be wave-uniform (it travels in M0).
__device__ __forceinline__ void dq_dma16(const void* base_uniform, uint32_t voff, uint32_t lds_off) {
  const uint64_t b = (uint64_t)base_uniform;
  const uint64_t base = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32) |
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(voff), "s"(base), "s"(__builtin_amdgcn_readfirstlane(lds_off)) : "memory");
}

template <class T, int D>
__global__ __launch_bounds__(512, 2) void lmk_bwd_dq_kernel(BwdParams p) {
  using C = DqCfg<T, D>;
  constexpr int BS = C::BS;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ql = lane & 31, h = lane >> 5;

  const int nq256 = (p.Lq + 255) >> 8;
  int bh, qt;                                              // (batch*head, 256-row query tile); most work first
  {
    const int bid = blockIdx.x, BH = p.B * p.H;
    if ((BH & 7) == 0) {
      const int xcd = bid & 7, j = bid >> 3, ngrp = BH >> 3;
      qt = nq256 - 1 - j / ngrp;
      bh = (j % ngrp) * 8 + xcd;
    } else {
      qt = nq256 - 1 - bid / BH;
      bh = bid % BH;
    }
  }
  const int b = bh / p.H, hh = bh % p.H;
  const char* qp = (const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h);
  const char* kp = (const char*)p.k + 2 * (b * p.ks_b + hh * p.ks_h);
  const char* vp = (const char*)p.v + 2 * (b * p.vs_b + hh * p.vs_h);
  const char* gp = (const char*)p.dout + 2 * (b * p.dos_b + hh * p.dos_h);
  char* dqp = (char*)p.dq + 2 * (b * p.dqs_b + hh * p.dqs_h);

  const int q0 = qt * 256 + wave * 32;
  const int dt = p.n_prefix * C::NT + (q0 >> 5);
  const int cblk = dt / C::NT, tsub = dt % C::NT;          // the wave's own block and its tile inside it
  const bool active = q0 < p.Lq;                           // Lq is a multiple of the block: whole tiles only
  const int qrow = q0 + ql;

  u32x4_t qf[C::KS], gf[C::KS];
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) {
    u32x4_t z = {0, 0, 0, 0};
    qf[ks] = z;
    gf[ks] = z;
    if (active) {
      qf[ks] = *(const u32x4_t*)(qp + 2 * ((int64_t)qrow * p.qs_r + 16 * ks + 8 * h));
      gf[ks] = *(const u32x4_t*)(gp + 2 * ((int64_t)qrow * p.dos_r + 16 * ks + 8 * h));
    }
  }
  // row terms (the reference's _bwd_preprocess, flash_landmark_attention.py:125-149): delta = rowsum(O * dO)
  // from the dO fragments already in registers, mhat = M*log2(e) + log2(L); left in the workspace for the
  // dK/dV kernel as well
  float mhat = 0.f, delta = 0.f;
  if (active) {
    float sum = 0.f;
    const char* orow = (const char*)p.o + 2 * (b * p.os_b + hh * p.os_h + (int64_t)qrow * p.os_r);
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) {
      const u32x4_t o4 = *(const u32x4_t*)(orow + 2 * (16 * ks + 8 * h));
#pragma unroll
      for (int i = 0; i < 4; ++i)
        sum += unpack_lo<T>(o4[i]) * unpack_lo<T>(gf[ks][i]) + unpack_hi<T>(o4[i]) * unpack_hi<T>(gf[ks][i]);
    }
    delta = pair_sum(sum);
    const int64_t ri = (int64_t)bh * p.Lq + qrow;
    mhat = p.M[ri] * kLog2e + fast_log2(p.L[ri]);
    if (h == 0) {
      p.delta[ri] = delta;
      p.mhat[ri] = mhat;
    }
  }

  // stages = blocks up to the own block of the workgroup's last query tile
  const int last_q0 = min(qt * 256 + 224, p.Lq - 32);
  const int n_stages = min(p.n_blocks, (p.n_prefix * C::NT + (last_q0 >> 5)) / C::NT + 1);

  // this wave's requests of a stage: request r covers rows RPD*(r % (BS/RPD)) .. of K (r < BS/RPD) or V.
  // The LDS swizzle is applied on the source side: lane i lands at +16*i, i.e. row i/CH, chunk position
  // i%CH, so it fetches the chunk tile_off() stores there.
  uint32_t src[C::PER_WAVE];                               // per-lane byte offset inside the (batch, head) slice of K or V
  const int n_k = BS / C::RPD;                             // requests that fetch K rows; the rest fetch V rows
#pragma unroll
  for (int i = 0; i < C::PER_WAVE; ++i) {
    const int r = wave * C::PER_WAVE + i;
    const bool is_v = r >= n_k;
    const int row = C::RPD * (r % n_k) + lane / C::CH, cp = lane % C::CH;
    const int f = tile_swizzle<D>(row);
    src[i] = (uint32_t)(2 * ((int64_t)row * (is_v ? p.vs_r : p.ks_r) + 8 * (cp ^ f)));
  }
  const uint32_t step_k = (uint32_t)(2 * (int64_t)BS * p.ks_r), step_v = (uint32_t)(2 * (int64_t)BS * p.vs_r);
  auto request = [&](int buf) __attribute__((always_inline)) {   // next block in key order -> buffer buf
#pragma unroll
    for (int i = 0; i < C::PER_WAVE; ++i) {
      const int r = wave * C::PER_WAVE + i;
      const bool is_v = r >= n_k;                          // wave-uniform
      const int dst = buf * C::STAGE_BYTES + (is_v ? C::TILE_BYTES : 0) + C::RPD * (r % n_k) * C::ROWB;
      dq_dma16(is_v ? vp : kp, src[i], dst);
      src[i] += is_v ? step_v : step_k;
    }
  };

  f32x16_t acc[C::DC];
#pragma unroll
  for (int dc = 0; dc < C::DC; ++dc)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[dc][r] = 0.f;
  const float c2 = p.scale_log2;

  // LDS byte offsets of this lane's operand fragments inside a 32-row tile: the swizzle repeats every 16
  // rows, so a tile at row 32u is the same offsets plus 32u rows -- an immediate of the LDS instruction
  int koff[C::KS];
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) {
    koff[ks] = tile_off<D>(ql, 2 * ks + h);
    // the compiler must not know the value's range: it would turn "offset + constant" into an OR computed by a
    // vector instruction per read; as a plain sum the constant stays the read's immediate offset
    asm volatile("" : "+v"(koff[ks]));
  }
  int voff[C::DC][2];
  {
    const int i = lane & 15, g2 = (lane >> 4) & 1;
#pragma unroll
    for (int dc = 0; dc < C::DC; ++dc) {
      const int col = 32 * dc + 16 * g2 + 4 * (i & 3);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        voff[dc][hf] = tile_off<D>(4 * h + (i >> 2) + 8 * hf, col >> 3) + ((col >> 2) & 1) * 8;
        asm volatile("" : "+v"(voff[dc][hf]));             // as for koff
      }
    }
  }
  // The wave issues in order, so in the earlier blocks' code the instruction stream is the schedule: every LDS
  // operand is asked for two MFMAs ahead of its use and the order is pinned.
  // (32 rows each of NTL consecutive LDS tiles) x (this wave's 32 queries)
  auto row_tiles = [&](int tile_bytes, const u32x4_t* bf, f32x16_t* out, auto ntl_c) __attribute__((always_inline)) {
    constexpr int NX = decltype(ntl_c)::value * C::KS, PFX = 2;
    u32x4_t fk[NX];
#pragma unroll
    for (int n = 0; n < PFX; ++n) fk[n] = lds_ld128(tile_bytes + 32 * (n / C::KS) * C::ROWB + koff[n % C::KS]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < NX; ++n) {
      if (n + PFX < NX) fk[n + PFX] = lds_ld128(tile_bytes + 32 * ((n + PFX) / C::KS) * C::ROWB + koff[(n + PFX) % C::KS]);
      const int u = n / C::KS, ks = n % C::KS;
      if (ks == 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) out[u][r] = 0.f;
      }
      out[u] = mfma32<T>(fk[n], bf[ks], out[u]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // dQ^T += (K tiles)^T dS^T for NTL consecutive tiles, dS = e f (dP - nD) in slices of 16 keys: a slice is formed
  // and packed under the MFMAs of the one before.  u0: first tile's index in the block (the landmark is the last
  // tile's last key); dP of tile u0 + i is d[d_stride * i].
  auto dq_tiles = [&](int tile_bytes, int u0, const f32x16_t* e, const f32x16_t* d, int d_stride, float f, float nD,
                      float dslm, auto ntl_c) __attribute__((always_inline)) {
    constexpr int NTL = decltype(ntl_c)::value, NZ = NTL * 2 * C::DC, PFZ = 2;
    auto zload = [&](int n) __attribute__((always_inline)) {
      const int sl = n / C::DC, dc = n % C::DC;
      const int base = tile_bytes + 16 * sl * C::ROWB;
      const u32x2_t a0 = lds_ld_tr(base + voff[dc][0]), a1 = lds_ld_tr(base + voff[dc][1]);
      const u32x4_t a = {a0[0], a0[1], a1[0], a1[1]};
      return a;
    };
    auto slice = [&](int sl) __attribute__((always_inline)) {
      const int i = sl >> 1, j = sl & 1;
      float ds[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) ds[r] = e[i][8 * j + r] * f * (d[d_stride * i][8 * j + r] - nD);
      if (j == 1 && u0 + i == C::NT - 1 && h == 1) ds[7] = dslm;
      const u32x4_t wf = {pack2<T>(ds[0], ds[1]), pack2<T>(ds[2], ds[3]), pack2<T>(ds[4], ds[5]), pack2<T>(ds[6], ds[7])};
      return wf;
    };
    u32x4_t zf[NZ], wf[2];
#pragma unroll
    for (int n = 0; n < PFZ; ++n) zf[n] = zload(n);
    wf[0] = slice(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < NZ; ++n) {
      if (n + PFZ < NZ) zf[n + PFZ] = zload(n + PFZ);
      const int sl = n / C::DC, dc = n % C::DC;
      acc[dc] = mfma32<T>(zf[n], wf[sl & 1], acc[dc]);
      if (dc == 0 && sl + 1 < 2 * NTL) wf[(sl + 1) & 1] = slice(sl + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto row_tile = [&](int tile_bytes, const u32x4_t* bf) __attribute__((always_inline)) {   // one tile, the compiler's order
    f32x16_t s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) s = mfma32<T>(lds_ld128(tile_bytes + koff[ks]), bf[ks], s);
    return s;
  };
  auto dq_tile = [&](int tile_bytes, const float* ds) __attribute__((always_inline)) {   // dQ^T += (K tile)^T dS^T
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      u32x4_t wf = {pack2<T>(ds[8 * j + 0], ds[8 * j + 1]), pack2<T>(ds[8 * j + 2], ds[8 * j + 3]),
                    pack2<T>(ds[8 * j + 4], ds[8 * j + 5]), pack2<T>(ds[8 * j + 6], ds[8 * j + 7])};
#pragma unroll
      for (int dc = 0; dc < C::DC; ++dc) {
        const int base = tile_bytes + 16 * j * C::ROWB;
        const u32x2_t a0 = lds_ld_tr(base + voff[dc][0]), a1 = lds_ld_tr(base + voff[dc][1]);
        const u32x4_t a = {a0[0], a0[1], a1[0], a1[1]};
        acc[dc] = mfma32<T>(a, wf, acc[dc]);
      }
    }
  };

  const uint32_t stat_row = 4u * (uint32_t)qrow;
  // ---------------- earlier block s at LDS byte addresses kb (K rows) / vb (V rows)
  auto earlier_block = [&](const int kb, const int vb, const int s) __attribute__((always_inline)) {
    f32x16_t sc[C::NT], dp[C::NT];
    row_tiles(kb, qf, sc, std::integral_constant<int, C::NT>{});
    const float s_last = sc[C::NT - 1][15];
    float mx = (h == 0) ? s_last : -INFINITY;
    float t_lm = 0.f, mloc = 0.f, den = 0.f, spd = 0.f;
    {
      // dP^T does not depend on S^T: at head dim 64 its MFMAs carry the local softmax of the scores, a slice behind
      // each -- first the maximum (one slice per tile), then the exponentials and their sum.  (At head dim 128 the
      // same placement measured 7 % slower than the softmax behind the MFMAs, in the compiler's order.)
      constexpr bool UNDER = D == 64;
      constexpr int NX = C::NT * C::KS, PFX = 2, NEXP = NX - C::NT, PER = (16 * C::NT + NEXP - 1) / NEXP;
      auto ywork = [&](int n) __attribute__((always_inline)) {
        if (n < C::NT) {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (!(n == C::NT - 1 && r == 15)) mx = fmaxf(mx, sc[n][r]);
          if (n == C::NT - 1) {
            mx = pair_max(mx);
            t_lm = pair_hi(s_last) * c2;
            mloc = mx * c2;
          }
        } else {
#pragma unroll
          for (int i = (n - C::NT) * PER; i < (n - C::NT + 1) * PER && i < 16 * C::NT; ++i) {
            const int u = i >> 4, r = i & 15;
            float e = fast_exp2(__builtin_fmaf(sc[u][r], c2, -mloc));
            if (u == C::NT - 1 && r == 15) e = (h == 0) ? e : 0.f;
            sc[u][r] = e;
            den += e;
          }
        }
      };
      u32x4_t fk[NX];
#pragma unroll
      for (int n = 0; n < PFX; ++n) fk[n] = lds_ld128(vb + 32 * (n / C::KS) * C::ROWB + koff[n % C::KS]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < NX; ++n) {
        if (n + PFX < NX) fk[n + PFX] = lds_ld128(vb + 32 * ((n + PFX) / C::KS) * C::ROWB + koff[(n + PFX) % C::KS]);
        const int u = n / C::KS, ks = n % C::KS;
        if (ks == 0) {
#pragma unroll
          for (int r = 0; r < 16; ++r) dp[u][r] = 0.f;
        }
        dp[u] = mfma32<T>(fk[n], gf[ks], dp[u]);
        if constexpr (UNDER) ywork(n);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (!UNDER) {
#pragma unroll
        for (int n = 0; n < NX; ++n) ywork(n);
      }
#pragma unroll
      for (int u = 0; u < C::NT; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) spd = __builtin_fmaf(sc[u][r], dp[u][r], spd);
    }
    den = pair_sum(den);
    spd = pair_sum(spd);
    const float invden = fast_rcp(den);
    const float nD = spd * invden;
    const float glog = t_lm - mhat;                        // log2 of the normalised gate
    const float g = fast_exp2(glog);
    const float f = g * invden;
    const float dslm = g * (nD - delta);                   // dS at the block's landmark key
    if (h == 0) {                                          // a scalar base per (head, block) plus the row's 32-bit offset
      const int64_t sb = 4 * ((int64_t)bh * p.n_blocks + s) * p.Lq;
      *(float*)((char*)p.stat_a + sb + stat_row) = mloc + fast_log2(den) - glog;
      *(float*)((char*)p.stat_n + sb + stat_row) = nD;
      *(float*)((char*)p.stat_l + sb + stat_row) = dslm;
    }
    dq_tiles(kb, 0, sc, dp, 1, f, nD, dslm, std::integral_constant<int, C::NT>{});
  };

  // Stages in front of the workgroup's first query block are earlier blocks for every wave: they run two at a
  // time without a branch, the LDS addresses of both buffers as immediates of the instructions.
  const int first_cblk = (p.n_prefix * C::NT + qt * 8) / C::NT;   // wave 0's own block: the least of the workgroup's
  const int s_uniform = min(first_cblk, n_stages - 1);
  auto uniform_stage = [&](auto buf_c, int s) __attribute__((always_inline)) {
    constexpr int buf = decltype(buf_c)::value;
    __builtin_amdgcn_s_waitcnt(0x0f70);                    // vmcnt(0): this wave's share of stage s has landed
    __syncthreads();                                       // ... and everyone's; stage s-1 has been consumed
    request(buf ^ 1);
    if (active) earlier_block(buf * C::STAGE_BYTES, buf * C::STAGE_BYTES + C::TILE_BYTES, s);
  };

  request(0);
  int s = 0;
  for (; s + 2 <= s_uniform; s += 2) {
    uniform_stage(std::integral_constant<int, 0>{}, s);
    uniform_stage(std::integral_constant<int, 1>{}, s + 1);
  }
  for (; s < n_stages; ++s) {
    const int buf = s & 1;
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (s + 1 < n_stages) request(buf ^ 1);
    const int kb = buf * C::STAGE_BYTES, vb = kb + C::TILE_BYTES;   // LDS byte addresses (the dynamic array starts at 0)
    if (!active) continue;
    if (s < cblk) {
      earlier_block(kb, vb, s);
    } else if (s == cblk) {
      const int lim = ql - ((tsub == C::NT - 1 && ql == 31) ? 1 : 0);
#pragma unroll
      for (int u = 0; u < C::NT; ++u) {
        if (u <= tsub) {
          f32x16_t sc = row_tile(kb + 32 * u * C::ROWB, qf);
          f32x16_t d = row_tile(vb + 32 * u * C::ROWB, gf);
          float ds[16];
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = 8 * (r >> 2) + 4 * h + (r & 3);
            const float pr = (u < tsub || key <= lim) ? fast_exp2(__builtin_fmaf(sc[r], c2, -mhat)) : 0.f;
            ds[r] = pr * (d[r] - delta);
          }
          dq_tile(kb + 32 * u * C::ROWB, ds);
        }
      }
    }
  }

  // dQ leaves as row segments through the wave's share of the stage buffer the last stage did not use: every wave
  // is past the barrier in front of the last stage, so nobody reads that buffer and no request targets it
  if (active) {
    static_assert(C::STAGE_BYTES / C::NW >= 2048, "32 rows x 32 columns of 16 bits per wave");
    const int free_buf = (n_stages & 1) * C::STAGE_BYTES;  // the last stage sits in buffer (n_stages - 1) & 1
    store_tile_rows<T, C::DC, false>(acc, p.scale, free_buf + wave * (C::STAGE_BYTES / C::NW),
                              [&](int r) __attribute__((always_inline)) -> char* {
      return dqp + 2 * ((int64_t)(q0 + r) * p.dqs_r);
    });
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// Whether workgroups of 256 rows (lmk_bwd_dq_kernel) are faster than those of 64 rows whose waves split the keys
// (lmk_bwd_dq_split.hip): only with whole blocks of 64 keys and more long rows than fill the chip twice.  Measured (us, 256
// rows -> 64 rows, D128, at n = workgroups of 256 rows / compute unit): n 0.5 79 -> 30 (L2048), n 1 34.2 -> 29.6 (L512),
// n 1.5 141 -> 134 (L3072), n 2 125.5 -> 124.5 (L2048), n 3 121 -> 117 (L960), n 4 134 -> 127 (L512) but 449 -> 469 (L4096),
// n 8 551 -> 661 (L2048); D64 n 4 286 -> 293 (L4096), 72 -> 69 (L512).  With tokens in slots or blocks of 128 the 64-row
// kernel was 1 % behind at worst and 30-60 % ahead at block 128 (no room for a block's dP tiles in the other).
static bool many_query_rows(const BwdParams& p) {
  const int64_t n = (int64_t)p.B * p.H * ((p.Lq + 255) / 256);
  return p.Lq_real <= 0 && p.n_real == 64 && p.Lk > 1024 && n > 2 * cu_count();
}

// Whether the dK/dV kernel with 128 keys per workgroup and roles (lmk_bwd_dkdv32.hip) is faster than the one with 64 keys
// (lmk_bwd_dkdv_split.hip).  At head dim 128 it is when its workgroups come in whole rounds of the compute units, from two
// 64-key workgroups per compute unit on.  Measured (us, 128 keys -> 64 keys): filled, B4 H32 L512 32.6 -> 38.6, B2 H32 L2048
// 142 -> 155, B32 H32 L512 272 -> 299; not filled, B3 H32 L1024 (288 workgroups) 93 -> 72, B16 H12 L448 (384) 49 -> 44, B2 H32
// L2040 block 51 (320) all of the backward 516 -> 415; few workgroups, B2 H8 L1024 32.4 -> 22.7, B1 H8 L4096 108 -> 82.  At
// head dim 64 three 64-key workgroups share a compute unit, and they lose only where long walks meet few workgroups:
// B3 H32 L1024 65 -> 44, B2 H32 L2048 93 -> 93, B32 H32 L512 161 -> 149, but B1 H12 L4096 81 -> 86, B1 H8 L16384 618 -> 649.
static bool dkdv_fills_the_chip(const BwdParams& p, int D) {
  const int64_t heads = (int64_t)p.B * p.H, cus = cu_count(), n64 = heads * ((p.Lk + 63) / 64);
  if (n64 <= 2 * cus) return false;
  const int64_t wgs = heads * dkdv32_groups(p), rounds = (wgs + cus - 1) / cus;
  const bool filled = 10 * wgs >= 9 * rounds * cus;
  return D == 128 ? filled : p.Lk >= 2048 && (n64 <= 3 * cus || (filled && p.Lk > 8192));
}

template <class T, int D, int BS>
static int launch_bwd_t(const BwdParams& p, int phases, hipStream_t stream) {
  int rc;
  // the dQ kernels compute delta and mhat themselves, so the separate pass only runs when asked for alone
  if ((phases & 1) && !(phases & 2)) {
    constexpr int RPW = 256 / (D / 8);
    const int64_t rows = (int64_t)p.B * p.H * p.Lq;
    hipLaunchKernelGGL((lmk_bwd_pre_kernel<T, D>), dim3((unsigned)((rows + RPW - 1) / RPW)), dim3(256), 0, stream, p, BS);
    if ((rc = (int)hipGetLastError())) return rc;
  }
  if (phases & 2) {
    if constexpr (BS == 32) {
      if ((rc = launch_bwd_dq32(p, D, std::is_same<T, bf16_t>::value ? LMK_DTYPE_BF16 : LMK_DTYPE_F16, stream))) return rc;
    } else if (BS == 128 || !many_query_rows(p)) {
      if ((rc = launch_bwd_dq_split(p, D, BS, std::is_same<T, bf16_t>::value ? LMK_DTYPE_BF16 : LMK_DTYPE_F16, stream))) return rc;
    } else {
      using C = DqCfg<T, D>;
      auto kern = lmk_bwd_dq_kernel<T, D>;
      static std::atomic<uint64_t> lds_ok{0};
      if ((rc = allow_dynamic_lds(kern, C::LDS_BYTES, lds_ok))) return rc;
      hipLaunchKernelGGL(kern, dim3(((p.Lq + 255) / 256) * p.B * p.H), dim3(64 * C::NW), C::LDS_BYTES, stream, p);
      if ((rc = (int)hipGetLastError())) return rc;
    }
  }
  if (phases & 4) {
    if (p.ds_tiles != nullptr) {
      if (BS != 32) return LMK_ERR_UNSUPPORTED;
      return launch_bwd_dkdv32_handover(p, D, std::is_same<T, bf16_t>::value ? LMK_DTYPE_BF16 : LMK_DTYPE_F16, stream);
    }
    if (BS != 32 && !dkdv_fills_the_chip(p, D))
      return launch_bwd_dkdv_split(p, D, BS, std::is_same<T, bf16_t>::value ? LMK_DTYPE_BF16 : LMK_DTYPE_F16, stream);
    return launch_bwd_dkdv32(p, D, BS, std::is_same<T, bf16_t>::value ? LMK_DTYPE_BF16 : LMK_DTYPE_F16, stream);
  }
  return 0;
}

template <class T>
static int launch_bwd_d(const BwdParams& p, int D, int BS, int phases, hipStream_t stream) {
  if (D == 128) {
    if (BS == 32) return launch_bwd_t<T, 128, 32>(p, phases, stream);
    if (BS == 64) return launch_bwd_t<T, 128, 64>(p, phases, stream);
    if (BS == 128) return launch_bwd_t<T, 128, 128>(p, phases, stream);
  } else if (D == 64) {
    if (BS == 32) return launch_bwd_t<T, 64, 32>(p, phases, stream);
    if (BS == 64) return launch_bwd_t<T, 64, 64>(p, phases, stream);
    if (BS == 128) return launch_bwd_t<T, 64, 128>(p, phases, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

int launch_bwd(const BwdParams& p, int D, int BS, int dtype, int phases, hipStream_t stream) {
  if (dtype == LMK_DTYPE_BF16) return launch_bwd_d<bf16_t>(p, D, BS, phases, stream);
  if (dtype == LMK_DTYPE_F16) return launch_bwd_d<f16_t>(p, D, BS, phases, stream);
  return LMK_ERR_UNSUPPORTED;
}

}  // namespace lmk
