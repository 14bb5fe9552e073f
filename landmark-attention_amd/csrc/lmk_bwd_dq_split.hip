// dQ kernel of the backward pass for launches whose query rows do not fill the chip: landmark blocks of 64 and 128
// slots, the keys of a row split over several waves.  The same mathematics as lmk_bwd_dq_kernel (lmk_bwd.hip: row terms,
// local softmax, nD, gate, dS, dQ^T = K^T dS^T, and the three terms per row and earlier block for the dK/dV kernel),
// the same split as lmk_fwd_split.hip: a workgroup has 64 query rows and 2 KP waves, wave (tq, part) the 32 rows of tile tq
// and the 64 keys of chunk `part` of every stage of 64 KP keys; a block of 128 is two parts, which exchange their maximum,
// sum and rowsum(e dP) through LDS.  The parts' dQ accumulators add up at the end.
//
// K and V of a stage have one LDS buffer each and travel under each other's products: dP^T = V dO^T is formed while K is
// on its way, the scores, the softmax and dQ^T += K^T dS^T while the next stage's V is.  Two barriers per stage; with two
// parts two workgroups share a compute unit.
#include <type_traits>

#include "lmk_common.hpp"
#include "lmk_launch.hpp"
#include "lmk_split.hpp"

namespace lmk {

template <class T, int D, int BS, int KP>
struct DqSplitCfg {
  static constexpr int NT = BS / 32;                    // 32-key tiles per block
  static constexpr int NH = BS / 64;                    // parts per block
  static constexpr int QT = 2;                          // query tiles per workgroup
  static constexpr int NW = QT * KP;
  static constexpr int ROWB = 2 * D;
  static constexpr int CH = D / 8;                      // 16-byte chunks per row
  static constexpr int KS = D / 16;                     // MFMA k-steps over the head dim
  static constexpr int DC = D / 32;                     // 32-wide output chunks of the head dim
  static constexpr int V_BASE = 64 * KP * ROWB;         // K of the stage, then V
  static constexpr int E_BASE = 2 * V_BASE;             // O rows at first; then the exchange and the factors; then the output tiles
  static constexpr int Q_ROWS = 64 * ROWB;              // Q and dO rows come in through the K buffer
  static constexpr int E_BYTES = Q_ROWS > NW * 2048 ? Q_ROWS : NW * 2048;
  static constexpr int X_PART = 512;                    // per (query tile, part): maximum, sum, rowsum(e dP), landmark score
  static constexpr int GS_BASE = E_BASE + QT * KP * X_PART;   // per wave the 64 lanes' group factors
  static constexpr int LDS_BYTES = E_BASE + E_BYTES;    // 80 KB at KP 2, D128
  static constexpr int RPD = 1024 / ROWB;               // rows covered by one 1 KB request
  static constexpr int PER_WAVE = 32 / RPD;             // requests per wave for a stage's K (or V): 32 rows
  static constexpr int Q_PER_WAVE = 64 / RPD / NW;
  static_assert(64 * KP % BS == 0, "a stage is whole blocks");
  static_assert(Q_PER_WAVE * NW * RPD == 64, "every wave issues the same number of requests");
  static_assert(2 * Q_ROWS <= V_BASE, "the Q and dO rows fit the K buffer");
  static_assert(GS_BASE + NW * 256 <= LDS_BYTES, "the exchange fits the O rows' area");
  static_assert(QT * DC * (KP - 1) * 4096 <= E_BASE, "the parts' accumulators fit the stage");
};

template <class T, int D, int BS, int KP, int LAYOUT>
__global__ __launch_bounds__(128 * KP, 2) void lmk_bwd_dq_split_kernel(BwdParams p) {
  constexpr bool plain = LAYOUT == PLAIN, GS = LAYOUT == FACTORS, SEG = LAYOUT == TABLE;
  using C = DqSplitCfg<T, D, BS, KP>;
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int part = wave % KP, tq = wave / KP;
  const int ql = lane & 31, h = lane >> 5;

  // workgroup -> head, batch, 64-row query tile (launch_rows64)
  const int hh = blockIdx.x, b = p.b0 + blockIdx.y, qt = p.qt_top - blockIdx.z;
  const int bh = b * p.H + hh;
  const char* qp = (const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h);
  const char* kp = (const char*)p.k + 2 * (b * p.ks_b + hh * p.ks_h);
  const char* vp = (const char*)p.v + 2 * (b * p.vs_b + hh * p.vs_h);
  const char* gp = (const char*)p.dout + 2 * (b * p.dos_b + hh * p.dos_h);
  const char* op = (const char*)p.o + 2 * (b * p.os_b + hh * p.os_h);
  char* dqp = (char*)p.dq + 2 * (b * p.dqs_b + hh * p.dqs_h);

  const int q0 = qt * 64 + tq * 32;                     // first query row of this wave; Lq is whole blocks
  const int cblk = p.n_prefix + qt * 64 / BS;           // the workgroup's landmark block
  const int tsub = (q0 % BS) >> 5;                      // the wave's tile in it
  const int qrow = q0 + ql;
  const bool tokens = !plain && p.Lq_real > 0;          // rows are tokens; otherwise rows are slots
  const int n_tok = tokens ? p.n_real : BS;             // rows per block
  const int n_complete = tokens ? p.n_full_k : p.Lk / BS;
  const int* const seg_q = SEG ? p.seg + p.n_prefix : nullptr;
  auto q_token = [&](int row) __attribute__((always_inline)) {   // row of the tensors, or -1
    return plain ? row : slot_to_token_row<BS>(row, n_tok, tokens ? p.n_full_q : p.Lq / BS, seg_q);
  };
  // a slot without a token is a query row of zeros with mhat = 1e30: every term it leaves for the dK/dV kernel is an exact zero
  const int qtok = q_token(qrow);
  float l_row = 1.f, m_row = 0.f;
  if (qtok >= 0) {
    const int64_t li = (int64_t)bh * (tokens ? p.Lq_real : p.Lq) + qtok;   // L, M follow the tensors' layout
    l_row = p.L[li];
    m_row = p.M[li];
  }

  // ---- direct loads, as in lmk_fwd_split.hip
  const int r_lane = lane / C::CH, cp = lane % C::CH;
  auto swz = [&](int row) __attribute__((always_inline)) {
    const int f = tile_swizzle<D>(row);
    return 16 * (cp ^ f);
  };
  auto first_row = [&](int blk) __attribute__((always_inline)) { return SEG ? p.seg[blk] : blk * n_tok; };
  auto slot_row = [&](int slot, int n) __attribute__((always_inline)) {
    return plain ? slot : (slot == BS - 1 ? n - 1 : (slot < n - 1 ? slot : 0));
  };
  // a wave fetches rows 32*wave .. +31 of every stage: slots row0 .. of block (stage's first block + blk0).  What the
  // requests of a stage have in common per lane: PLAIN, the first one's byte offset without its swizzle; TOKENS, the
  // rows of the eight (of head dim 64: four) requests inside the block, a byte each.
  const int row0 = wave * 32 % BS, blk0 = wave * 32 / BS;
  const int swz0 = swz(row0 + r_lane);
  const uint32_t plain_k = (uint32_t)(row0 + r_lane) * (uint32_t)(2 * p.ks_r), plain_v = (uint32_t)(row0 + r_lane) * (uint32_t)(2 * p.vs_r);
  uint32_t rows[2] = {0, 0};
  if constexpr (!plain) {
#pragma unroll
    for (int i = 0; i < C::PER_WAVE; ++i) rows[i >> 2] |= (uint32_t)slot_row(row0 + C::RPD * i + r_lane, n_tok) << (8 * (i & 3));
  }
  auto request = [&](bool is_v, int st) __attribute__((always_inline)) {   // this wave's rows of K or V of stage st
    const int blk = st * (KP / C::NH) + blk0;
    if (blk > cblk) return;                             // no query here sees it, and there may be none
    const char* src = is_v ? vp : kp;
    const int row_b = first_row(blk);
    const uint32_t rs = (uint32_t)(2 * (is_v ? p.vs_r : p.ks_r)), first = (uint32_t)row_b * rs;
    const int dst = (is_v ? C::V_BASE : 0) + 32 * wave * C::ROWB;
    const int n = SEG ? p.seg[blk + 1] - row_b : 0;
#pragma unroll
    for (int i = 0; i < C::PER_WAVE; ++i) {
      constexpr int STEP = C::RPD;                      // rows between requests: 4 or 8, which turn the swizzle's low bits
      const int sw = swz0 ^ (16 * ((STEP * i >> 2) & 3));
      uint32_t off;
      if (plain) {
        off = (is_v ? plain_v : plain_k) + (first + (uint32_t)(STEP * i) * rs) + sw;
      } else {
        const uint32_t t = SEG ? (uint32_t)slot_row(row0 + STEP * i + r_lane, n) : (rows[i >> 2] >> (8 * (i & 3))) & 255;
        off = t * rs + first + sw;
      }
      split_dma16(src, off, dst + 1024 * i);
    }
  };

  // ---- LDS byte addresses of this lane's operand fragments in the first tile of the part's chunk of K; at() is what
  // another row of the buffer adds to them, V_BASE leads to V
  const int krow = 64 * part;
  auto at = [&](int row) __attribute__((always_inline)) { return (row - krow) * C::ROWB; };
  // The swizzle makes an operand's other chunks XORs of the first one's address; they are formed where they are used,
  // because nine registers more than that are nine too many here (koff, voff; a plain sum with a value the compiler
  // knows nothing of keeps a constant the read's immediate offset).
  const int koff0 = krow * C::ROWB + tile_off<D>(ql, h);
  int voff0;
  {
    const int i = lane & 15, g2 = (lane >> 4) & 1, col = 16 * g2 + 4 * (i & 3);
    voff0 = krow * C::ROWB + tile_off<D>(4 * h + (i >> 2), col >> 3) + ((col >> 2) & 1) * 8;
  }
  auto k_offsets = [&](int* koff) __attribute__((always_inline)) {      // chunk 2 ks + h of row ql
    int k0 = koff0;
    asm volatile("" : "+v"(k0));
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) {
      koff[ks] = k0 ^ (32 * ks);
      asm volatile("" : "+v"(koff[ks]));
    }
  };
  auto v_offsets = [&](int* voff) __attribute__((always_inline)) {      // columns 32 dc ..; 8 rows on: bit 5 turned (and 8 rows added)
    int v0 = voff0;
    asm volatile("" : "+v"(v0));
#pragma unroll
    for (int n = 0; n < 2 * C::DC; ++n) {
      voff[n] = v0 ^ (64 * (n >> 1) + 32 * (n & 1));
      asm volatile("" : "+v"(voff[n]));
    }
  };

  // ---- Q, dO and O rows through LDS, the first stage's V behind them; delta = rowsum(O * dO)
  u32x4_t qf[C::KS], gf[C::KS];                         // fragments (B operands): row qrow, head dims 16*ks + 8h .. +7
  float delta = 0.f;
  {
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const char* src = x == 0 ? qp : x == 1 ? gp : op;
      const uint32_t rs = (uint32_t)(2 * (x == 0 ? p.qs_r : x == 1 ? p.dos_r : p.os_r));
#pragma unroll
      for (int i = 0; i < C::Q_PER_WAVE; ++i) {
        const int r = wave * C::Q_PER_WAVE + i;
        const int row = C::RPD * r + r_lane, t = q_token(qt * 64 + row);
        const int tok = t >= 0 ? t : q_token((qt * 64 + row) / BS * BS);
        split_dma16(src, (uint32_t)tok * rs + swz(row), (x == 2 ? C::E_BASE : x * C::Q_ROWS) + 1024 * r);
      }
    }
    request(true, 0);
    if (blk0 <= cblk) __builtin_amdgcn_s_waitcnt(0x0f70 | C::PER_WAVE);
    else wait_vm0();
    __syncthreads();
    int koff[C::KS];
    k_offsets(koff);
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) {
      const int a = at(32 * tq) + koff[ks];
      qf[ks] = lds_ld128(a);
      gf[ks] = lds_ld128(C::Q_ROWS + a);
      const u32x4_t o4 = lds_ld128(C::E_BASE + a);
      if (!plain && qtok < 0) {
        const u32x4_t z = {0, 0, 0, 0};
        qf[ks] = z;
        gf[ks] = z;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        delta += unpack_lo<T>(o4[i]) * unpack_lo<T>(gf[ks][i]) + unpack_hi<T>(o4[i]) * unpack_hi<T>(gf[ks][i]);
    }
    delta = pair_sum(delta);
  }

  f32x16_t acc[C::DC];
#pragma unroll
  for (int dc = 0; dc < C::DC; ++dc) zero16(acc[dc]);
  f32x16_t sc[2], dp[2];                                // scores, then exponentials; dP -- of the wave's two tiles
  const float c2 = p.scale_log2;
  const int half = part % C::NH;                        // BS 128: the part's half of its block

  // (rows of one or two LDS tiles, t0 and t1 from the chunk's first row) x (this wave's queries), as in lmk_fwd_split.hip
  auto row_tiles = [&](int t0, int t1, const u32x4_t* bf, f32x16_t* out, auto n_c, auto under) __attribute__((always_inline)) {
    constexpr int NX = decltype(n_c)::value * C::KS, PF = 3;
    int koff[C::KS];
    k_offsets(koff);
    auto ld = [&](int n) __attribute__((always_inline)) { return lds_ld128((n / C::KS ? t1 : t0) + koff[n % C::KS]); };
    u32x4_t fk[NX];
#pragma unroll
    for (int n = 0; n < PF; ++n) fk[n] = ld(n);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < NX; ++n) {
      if (n + PF < NX) fk[n + PF] = ld(n + PF);
      if (n % C::KS == 0) zero16(out[n / C::KS]);
      out[n / C::KS] = mfma32<T>(fk[n], bf[n % C::KS], out[n / C::KS]);
      under(n);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // dQ^T += K^T dS^T of one or two tiles; ds(u, r) is formed and packed in slices of 16 keys under the MFMAs before
  auto product = [&](int t0, int t1, auto n_c, auto ds) __attribute__((always_inline)) {
    constexpr int NZ = decltype(n_c)::value * 2 * C::DC, PF = 3;
    int voff[2 * C::DC];
    v_offsets(voff);
    auto ld = [&](int n) __attribute__((always_inline)) {
      const int sl = n / C::DC, dc = n % C::DC;
      const int base = (sl >> 1 ? t1 : t0) + 16 * (sl & 1) * C::ROWB;
      const u32x2_t a0 = lds_ld_tr(base + voff[2 * dc]), a1 = lds_ld_tr(base + 8 * C::ROWB + voff[2 * dc + 1]);
      const u32x4_t a = {a0[0], a0[1], a1[0], a1[1]};
      return a;
    };
    auto slice = [&](int sl) __attribute__((always_inline)) {
      u32x4_t wf;
#pragma unroll
      for (int i = 0; i < 4; ++i) wf[i] = pack2<T>(ds(sl >> 1, 8 * (sl & 1) + 2 * i), ds(sl >> 1, 8 * (sl & 1) + 2 * i + 1));
      return wf;
    };
    u32x4_t zf[NZ], wf[2];
#pragma unroll
    for (int n = 0; n < PF; ++n) zf[n] = ld(n);
    wf[0] = slice(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < NZ; ++n) {
      if (n + PF < NZ) zf[n + PF] = ld(n + PF);
      const int sl = n / C::DC, dc = n % C::DC;
      acc[dc] = mfma32<T>(zf[n], wf[sl & 1], acc[dc]);
      if (dc == 0 && (sl + 1) * C::DC < NZ) wf[(sl + 1) & 1] = slice(sl + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  auto nothing = [](int) {};
  auto normal_keys = [&](int blk) __attribute__((always_inline)) {   // slots behind them, up to the landmark's, hold no key
    return SEG ? block_normal_keys<BS>(blk, p.n_real, n_complete, p.seg) : p.n_real - 1;
  };
  auto mask_padding = [&](f32x16_t& x, int u, int n_norm) __attribute__((always_inline)) {   // of tile u of a block
    if (plain || n_norm >= BS - 1 || n_norm >= 32 * u + 32) return;
    const int h4 = 4 * (lane_id() >> 5);                // formed here: kept, the 16 masks fill the scalar registers
    const int first = n_norm - 32 * u - h4, last = BS - 1 - 32 * u - h4;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int kl = 8 * (r >> 2) + (r & 3);
      if (kl >= first && kl < last) x[r] = -INFINITY;
    }
  };

  // ---- an earlier block's 64 keys (or half of its 128), dP there: scores and the part's maximum (log2 domain), sum and
  // rowsum(e dP)
  float mhat = 0.f, mpart = 0.f, den = 0.f, spd = 0.f, t_lm = 0.f;
  auto earlier_scores = [&](int st) __attribute__((always_inline)) {
    const int n_norm = normal_keys(st * (KP / C::NH) + part / C::NH);
    float m0 = -INFINITY, m1 = -INFINITY;
    row_tiles(0, 32 * C::ROWB, qf, sc, Two{}, [&](int n) __attribute__((always_inline)) {   // tile 0's maximum under tile 1's MFMAs
      if (n == C::KS + 1) mask_padding(sc[0], 2 * half, n_norm);
      if (n > C::KS + 1) {
        constexpr int PER = (16 + C::KS - 3) / (C::KS - 2);
#pragma unroll
        for (int r = (n - C::KS - 2) * PER; r < (n - C::KS - 1) * PER && r < 16; ++r) {
          if (r & 1) m1 = fmaxf(m1, sc[0][r]);
          else m0 = fmaxf(m0, sc[0][r]);
        }
      }
    });
    mask_padding(sc[1], 2 * half + 1, n_norm);
    const int ln = lane_id(), xrow = C::E_BASE + tq * KP * C::X_PART + 4 * (ln & 31), h = ln >> 5;
    const bool lm = half == C::NH - 1 && h == 1;        // the landmark: last tile, r = 15, h = 1
    const float s_last = sc[1][15];
    m1 = fmaxf(m1, lm ? -INFINITY : s_last);
#pragma unroll
    for (int r = 0; r < 15; ++r) {
      if (r & 1) m1 = fmaxf(m1, sc[1][r]);
      else m0 = fmaxf(m0, sc[1][r]);
    }
    const float mx = pair_max(fmaxf(m0, m1));
    t_lm = pair_hi(s_last) * c2;
    float mloc = mx * c2;
    mpart = mloc;
    if (!plain && C::NH > 1) mloc = mx == -INFINITY ? 0.f : mloc;   // a half without a normal key
    float d0 = 0.f, d1 = 0.f, s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const int u = i >> 4, r = i & 15;
      float x = fast_exp2(__builtin_fmaf(sc[u][r], c2, -mloc));
      if (i == 31) x = lm ? 0.f : x;
      sc[u][r] = x;
      if (i & 1) {
        d1 += x;
        s1 = __builtin_fmaf(x, dp[u][r], s1);
      } else {
        d0 += x;
        s0 = __builtin_fmaf(x, dp[u][r], s0);
      }
    }
    den = pair_sum(d0 + d1);
    spd = pair_sum(s0 + s1);
    if constexpr (C::NH > 1) {
      lds_st32(xrow + part * C::X_PART + 128 * h, h == 0 ? mpart : den);
      lds_st32(xrow + part * C::X_PART + 256 + 128 * h, h == 0 ? spd : t_lm);
    }
  };
  // the block's terms, for the dK/dV kernel as well, and the product
  auto earlier_product = [&](int st) __attribute__((always_inline)) {
    const int blk = st * (KP / C::NH) + part / C::NH;
    float m = mpart, fp = 1.f;
    if constexpr (C::NH > 1) {
      const int other = C::E_BASE + (tq * KP + (part ^ 1)) * C::X_PART + 4 * (lane_id() & 31);
      const float mo = lds_ld32(other), dn = lds_ld32(other + 128), sp = lds_ld32(other + 256);
      if (half == 0) t_lm = lds_ld32(other + 384);
      m = fmaxf(mpart, mo);
      fp = fast_exp2(mpart - m);
      const float fo = fast_exp2(mo - m);
      den = __builtin_fmaf(den, fp, dn * fo);
      spd = __builtin_fmaf(spd, fp, sp * fo);
    }
    float gscale = 1.f;                                 // group dropout: this block's factor for this query row
    if constexpr (GS) gscale = qtok >= 0 ? lds_ld32(C::GS_BASE + wave * 256 + 4 * lane_id()) : 1.f;
    const float invden = fast_rcp(den);
    const float nD = spd * invden;
    const float glog = t_lm - mhat;                     // log2 of the normalised gate
    const float g = fast_exp2(glog);
    // out_i = .. + gscale * g * (P V): the weights carry the factor, the landmark's dS sees it through nD
    const float f = g * invden * gscale * fp;
    const float dslm = g * (gscale * nD - delta);       // dS at the block's landmark key
    const int ln = lane_id();
    if (half == C::NH - 1 && ln < 32) {                 // a scalar base per (head, block) plus the row's 32-bit offset
      const int64_t sb = 4 * ((int64_t)bh * p.n_blocks + blk) * p.Lq;
      const uint32_t sr = 4u * (uint32_t)(q0 + ln);
      *(float*)((char*)p.stat_a + sb + sr) = gscale > 0.f ? m + fast_log2(den) - glog - fast_log2(gscale) : 1e30f;
      *(float*)((char*)p.stat_n + sb + sr) = nD;
      *(float*)((char*)p.stat_l + sb + sr) = dslm;
    }
    const float nf = -nD * f;
    const bool lm = half == C::NH - 1 && ln >= 32;
    product(0, 32 * C::ROWB, Two{}, [&](int u, int r) __attribute__((always_inline)) {   // dS = e f (dP - nD)
      const float x = sc[u][r] * __builtin_fmaf(dp[u][r], f, nf);
      return u == 1 && r == 15 && lm ? dslm : x;
    });
  };
  auto request_k = [&](int st) __attribute__((always_inline)) {
    request(false, st);
    if constexpr (GS) {                                 // this lane's row's factor of the part's block
      const int blk = min(st * (KP / C::NH) + part / C::NH, cblk - 1);
      if (blk >= 0) split_dma4(p.group_scale + (int64_t)bh * p.gs_bh + (int64_t)blk * p.gs_blk + max(qtok, 0), C::GS_BASE + wave * 256);
    }
  };
  auto meet = [&]() __attribute__((always_inline)) {       // everyone's requests have landed
    wait_vm0();
    __syncthreads();
  };

  meet();                                               // V of the first stage; the Q, dO and O rows are in registers
  mhat = qtok >= 0 ? m_row * kLog2e + fast_log2(l_row) : 1e30f;
  if (part == 0 && h == 0) {                            // left in the workspace for the dK/dV kernel as well
    p.delta[(int64_t)bh * p.Lq + qrow] = delta;
    p.mhat[(int64_t)bh * p.Lq + qrow] = mhat;
  }
  // ---- stages of earlier blocks only
  const int last = cblk * C::NH / KP, own = cblk * C::NH % KP;   // the stage of the own block, and the own block's first part
  for (int st = 0; st < last; ++st) {
    request_k(st);
    row_tiles(C::V_BASE, C::V_BASE + 32 * C::ROWB, gf, dp, Two{}, nothing);
    meet();                                             // K is there; V has been read
    request(true, st + 1);
    earlier_scores(st);
    if constexpr (C::NH > 1) __syncthreads();           // the halves' numbers
    earlier_product(st);
    meet();                                             // the next V is there; K has been read
  }
  // ---- the own block's stage: parts in front of it have an earlier block, the others take its causal tiles
  {
    const int np = KP - own;                            // tile u of the own block goes to part own + u % np
    const int u0 = part - own, u1 = u0 + np;            // at most two per part
    const bool earlier = part < own, has0 = !earlier && u0 <= tsub, has1 = !earlier && u1 <= tsub;
    const int t0 = earlier ? 0 : at(64 * own + 32 * u0), t1 = earlier ? 32 * C::ROWB : at(64 * own + 32 * u1);
    request_k(last);
    if (earlier || has1) row_tiles(C::V_BASE + t0, C::V_BASE + t1, gf, dp, Two{}, nothing);
    else if (has0) row_tiles(C::V_BASE + t0, 0, gf, dp, One{}, nothing);
    meet();
    if (earlier) {
      earlier_scores(last);
    } else if (has0) {
      if (has1) row_tiles(t0, t1, qf, sc, Two{}, nothing);
      else row_tiles(t0, 0, qf, sc, One{}, nothing);
      const int n_norm = normal_keys(cblk);
      auto weigh = [&](int i, int u) __attribute__((always_inline)) {
        mask_padding(sc[i], u, n_norm);                 // only the landmark query could reach such a slot
        const int ln = lane_id(), row = ln & 31;
        const int lim = u < tsub ? 32 : row - ((tsub == C::NT - 1 && row == 31) ? 1 : 0) - 4 * (ln >> 5);   // landmark query looks one left
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float x = fast_exp2(__builtin_fmaf(sc[i][r], c2, -mhat));
          sc[i][r] = (8 * (r >> 2) + (r & 3) <= lim ? x : 0.f) * (dp[i][r] - delta);
        }
      };
      weigh(0, u0);
      if (has1) weigh(1, u1);
    }
    if constexpr (C::NH > 1) __syncthreads();
    auto ds = [&](int u, int r) __attribute__((always_inline)) { return sc[u][r]; };
    if (earlier) earlier_product(last);
    else if (has1) product(t0, t1, Two{}, ds);
    else if (has0) product(t0, 0, One{}, ds);
  }

  // ---- the parts meet: every part leaves its accumulator, except for the output chunks dc = part, part + KP, .. which
  // it collects
  __syncthreads();                                      // nobody reads the stage any more
  const int l16 = 16 * lane_id();
#pragma unroll
  for (int dc = 0; dc < C::DC; ++dc) {
    if (dc % KP == part) continue;
    const int to = ((tq * C::DC + dc) * (KP - 1) + part - (part > dc % KP ? 1 : 0)) * 4096 + l16;   // in part order
#pragma unroll
    for (int g = 0; g < 4; ++g)
      lds_st128(to + 1024 * g, u32x4_t{__float_as_uint(acc[dc][4 * g]), __float_as_uint(acc[dc][4 * g + 1]),
                                       __float_as_uint(acc[dc][4 * g + 2]), __float_as_uint(acc[dc][4 * g + 3])});
  }
  __syncthreads();
#pragma unroll
  for (int dc = 0; dc < C::DC; ++dc) {
    if (dc % KP == part) {
#pragma unroll
      for (int from = 0; from < KP - 1; ++from) {
        const int to = ((tq * C::DC + dc) * (KP - 1) + from) * 4096 + l16;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const u32x4_t v = lds_ld128(to + 1024 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[dc][4 * g + i] += __uint_as_float(v[i]);
        }
      }
      store_tile_rows<T, 1>(&acc[dc], p.scale, C::E_BASE + wave * 2048, [&](int r) __attribute__((always_inline)) -> char* {
        const int tok = q_token(q0 + r);
        return tok < 0 ? nullptr : dqp + 2 * ((int64_t)tok * p.dqs_r) + 64 * dc;
      });
    }
  }
}

template <class T, int D, int BS, int KP, int LAYOUT>
static int launch_dq_split_t(const BwdParams& p, hipStream_t stream) {
  using C = DqSplitCfg<T, D, BS, KP>;
  auto kern = lmk_bwd_dq_split_kernel<T, D, BS, KP, LAYOUT>;
  static std::atomic<uint64_t> lds_ok{0};
  return launch_rows64(kern, p, 64 * C::NW, C::LDS_BYTES, lds_ok, stream);
}

template <class T, int D, int BS, int KP>
static int launch_dq_split_v(const BwdParams& p, hipStream_t stream) {
  if (p.seg != nullptr) return launch_dq_split_t<T, D, BS, KP, TABLE>(p, stream);
  if (p.group_scale != nullptr) return launch_dq_split_t<T, D, BS, KP, FACTORS>(p, stream);
  if (p.Lq_real <= 0 && p.n_real == BS) return launch_dq_split_t<T, D, BS, KP, PLAIN>(p, stream);
  return launch_dq_split_t<T, D, BS, KP, TOKENS>(p, stream);
}

template <class T, int D>
static int launch_dq_split_d(const BwdParams& p, int BS, int kparts, hipStream_t stream) {
  if (BS == 64) return kparts == 4 ? launch_dq_split_v<T, D, 64, 4>(p, stream) : launch_dq_split_v<T, D, 64, 2>(p, stream);
  if (BS == 128) return kparts == 4 ? launch_dq_split_v<T, D, 128, 4>(p, stream) : launch_dq_split_v<T, D, 128, 2>(p, stream);
  return LMK_ERR_UNSUPPORTED;
}

int launch_bwd_dq_split(const BwdParams& p, int D, int BS, int dtype, hipStream_t stream) {
  if (p.seg != nullptr && p.group_scale != nullptr) return LMK_ERR_UNSUPPORTED;
  const int kparts = key_parts(p.B, p.H, p.Lq, p.Lk);
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_dq_split_d<bf16_t, 128>(p, BS, kparts, stream);
    if (D == 64) return launch_dq_split_d<bf16_t, 64>(p, BS, kparts, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_dq_split_d<f16_t, 128>(p, BS, kparts, stream);
    if (D == 64) return launch_dq_split_d<f16_t, 64>(p, BS, kparts, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

}  // namespace lmk
