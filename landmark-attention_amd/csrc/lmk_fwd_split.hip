// Forward kernel of fused landmark attention for launches whose query rows do not fill the chip: landmark blocks of
// 64 and 128 slots, the keys of a row split over several waves.
//
// lmk_fwd_kernel (lmk_fwd.hip) gives a workgroup 256 query rows; B2 H8 L1024 is 64 workgroups on 256 compute units,
// and the longest walks 16 blocks one after the other.  Here a workgroup has 64 query rows and 2 KP waves: wave
// (tq, part) owns the 32 queries of tile tq and, of every stage of 64 KP keys, the 64 keys of chunk `part` (a block, or
// half of a block of 128, whose two waves exchange the maximum and the sum of the local softmax through LDS).
// The first pass over the landmark keys fixes the maximum R the earlier blocks are summed against (as in
// lmk_fwd.hip), so the parts' accumulators add up without a running maximum; only the own block's causal tiles, which
// go to the parts that have no earlier block in the last stage, can raise a part's maximum.  The parts meet once, at
// the end, through LDS.
// A stage's K and V have one LDS buffer each: V travels under the scores and the softmax, the next stage's K under the
// second product.
#include <type_traits>

#include "lmk_common.hpp"
#include "lmk_launch.hpp"
#include "lmk_split.hpp"

namespace lmk {

template <class T, int D, int BS, int KP>
struct FwdSplitCfg {
  static constexpr int NT = BS / 32;                    // 32-key tiles per block
  static constexpr int NH = BS / 64;                    // parts per block
  static constexpr int QT = 2;                          // query tiles per workgroup
  static constexpr int NW = QT * KP;
  static constexpr int ROWB = 2 * D;
  static constexpr int CH = D / 8;                      // 16-byte chunks per row
  static constexpr int KS = D / 16;                     // MFMA k-steps over the head dim
  static constexpr int DC = D / 32;                     // 32-wide output chunks of the head dim
  static constexpr int V_BASE = 64 * KP * ROWB;         // K of the stage, then V
  static constexpr int LM_BASE = 2 * V_BASE;            // first pass: 64 landmark keys; at the end the output tiles
  static constexpr int LM_ROWS = 64;
  static constexpr int LM_BYTES = LM_ROWS * ROWB > NW * 2048 ? LM_ROWS * ROWB : NW * 2048;
  static constexpr int X_BASE = LM_BASE;                // behind the first pass: per (query tile, part) maximum, sum, landmark score ..
  static constexpr int X_PART = 384;
  static constexpr int GS_BASE = X_BASE + QT * KP * X_PART;   // .. and per wave the 64 lanes' group factors
  static constexpr int LDS_BYTES = LM_BASE + LM_BYTES;  // 80 KB at KP 2, D128: two workgroups per compute unit
  static constexpr int RPD = 1024 / ROWB;               // rows covered by one 1 KB request
  static constexpr int PER_WAVE = 32 / RPD;             // requests per wave for a stage's K (or V): 32 rows
  static constexpr int LM_PER_WAVE = LM_ROWS / RPD / NW;
  static constexpr int Q_PER_WAVE = 32 * QT / RPD / NW;
  static_assert(64 * KP % BS == 0, "a stage is whole blocks");
  static_assert(LM_PER_WAVE * NW * RPD == LM_ROWS && Q_PER_WAVE * NW * RPD == 32 * QT, "every wave issues the same number of requests");
  static_assert(GS_BASE + NW * 256 <= LDS_BYTES, "the exchange fits the landmark keys' area");
  static constexpr int STORE_BASE = QT * DC * (KP - 1) * 4096 + NW * 2048 <= LM_BASE ? LM_BASE - NW * 2048 : LM_BASE;
  static_assert(QT * DC * (KP - 1) * 4096 <= (KP > 2 ? LM_BASE : V_BASE), "the parts' accumulators fit the stage");
};

template <class T, int D, int BS, int KP, int LAYOUT>
__global__ __launch_bounds__(128 * KP, 2) void lmk_fwd_split_kernel(FwdParams p) {
  constexpr bool plain = LAYOUT == PLAIN, GS = LAYOUT == FACTORS, SEG = LAYOUT == TABLE;
  using C = FwdSplitCfg<T, D, BS, KP>;
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int part = wave % KP, tq = wave / KP;
  const int ql = lane & 31, h = lane >> 5;

  // ---- workgroup -> head, batch, 64-row query tile (launch_rows64)
  const int hh = blockIdx.x, b = p.b0 + blockIdx.y, qt = p.qt_top - blockIdx.z;
  const int bh = b * p.H + hh;
  const char* qp = (const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h);
  const char* kp = (const char*)p.k + 2 * (b * p.ks_b + hh * p.ks_h);
  const char* vp = (const char*)p.v + 2 * (b * p.vs_b + hh * p.vs_h);
  char* op = (char*)p.o + 2 * (b * p.os_b + hh * p.os_h);

  const int q0 = qt * 64 + tq * 32;                     // first query row of this wave
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
  const int qtok = qrow >= p.Lq ? -1 : q_token(qrow);

  // ---- direct loads.  The LDS swizzle is applied on the source side: lane i lands at +16*i, i.e. row i/CH, chunk
  // position i%CH, so it fetches the chunk tile_off() stores there.
  const int r_lane = lane / C::CH, cp = lane % C::CH;
  auto swz = [&](int row) __attribute__((always_inline)) {
    const int f = tile_swizzle<D>(row);
    return 16 * (cp ^ f);
  };
  // A block of n tokens holds them in its first slots, the last one (of a complete block: its landmark) in slot BS-1;
  // the slots in between read the block's first token.
  const int lk_rows = tokens ? p.Lk_real : p.Lk;
  auto first_row = [&](int blk) __attribute__((always_inline)) { return SEG ? p.seg[blk] : blk * n_tok; };
  auto slot_row = [&](int slot, int n) __attribute__((always_inline)) {
    return plain ? slot : (slot == BS - 1 ? n - 1 : (slot < n - 1 ? slot : 0));
  };
  // a wave fetches rows 32*wave .. +31 of every stage: slots row0 .. of block (stage's first block + blk0)
  const int row0 = wave * 32 % BS, blk0 = wave * 32 / BS;
  uint32_t off_k[C::PER_WAVE], off_v[C::PER_WAVE];      // this lane's byte offsets inside a block at its first token
#pragma unroll
  for (int i = 0; i < C::PER_WAVE; ++i) {
    const int row = row0 + C::RPD * i + r_lane;
    off_k[i] = (uint32_t)slot_row(row, n_tok) * (uint32_t)(2 * p.ks_r) + swz(row);
    off_v[i] = (uint32_t)slot_row(row, n_tok) * (uint32_t)(2 * p.vs_r) + swz(row);
  }
  auto request = [&](bool is_v, int st) __attribute__((always_inline)) {   // this wave's rows of K or V of stage st
    const int blk = st * (KP / C::NH) + blk0;
    const char* src = is_v ? vp : kp;
    if (blk > cblk) return;                             // no query here sees it, and there may be none
    const int row_b = first_row(blk);
    const uint32_t rs = (uint32_t)(2 * (is_v ? p.vs_r : p.ks_r)), first = (uint32_t)row_b * rs;
    const int dst = (is_v ? C::V_BASE : 0) + 32 * wave * C::ROWB;
    if (!SEG && blk < n_complete) {
#pragma unroll
      for (int i = 0; i < C::PER_WAVE; ++i) split_dma16(src, (is_v ? off_v[i] : off_k[i]) + first, dst + 1024 * i);
    } else {                                            // an incomplete last block holds its tokens in the first slots
      const int n = SEG ? p.seg[blk + 1] - row_b : lk_rows - row_b;
      int rl = r_lane;
      asm volatile("" : "+v"(rl));
#pragma unroll
      for (int i = 0; i < C::PER_WAVE; ++i) {
        const int row = row0 + C::RPD * i + rl;
        const int t = SEG && blk < n_complete ? slot_row(row, n) : min(row, n - 1);
        split_dma16(src, (uint32_t)t * rs + swz(row) + first, dst + 1024 * i);
      }
    }
  };

  u32x4_t qf[C::KS];                                    // Q fragments (B operand): query qrow, head dims 16*ks + 8h .. +7
  const float c2 = p.scale_log2;
  auto normal_keys = [&](int blk) __attribute__((always_inline)) {   // slots behind them, up to the landmark's, hold no key
    return SEG ? block_normal_keys<BS>(blk, p.n_real, n_complete, p.seg) : p.n_real - 1;
  };

  // LDS byte addresses of this lane's operand fragments in the first tile of the part's chunk of K and of V (see
  // lmk_fwd.hip); at() is what another row of the buffer adds to them
  const int krow = 64 * part;
  auto at = [&](int row) __attribute__((always_inline)) { return (row - krow) * C::ROWB; };
  int koff[C::KS];
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) {
    koff[ks] = krow * C::ROWB + tile_off<D>(ql, 2 * ks + h);
    asm volatile("" : "+v"(koff[ks]));                  // a plain sum keeps a constant the read's immediate offset
  }
  int voff[C::DC][2];
  {
    const int i = lane & 15, g2 = (lane >> 4) & 1;
#pragma unroll
    for (int dc = 0; dc < C::DC; ++dc) {
      const int col = 32 * dc + 16 * g2 + 4 * (i & 3);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        voff[dc][hf] = C::V_BASE + krow * C::ROWB + tile_off<D>(4 * h + (i >> 2) + 8 * hf, col >> 3) + ((col >> 2) & 1) * 8;
        asm volatile("" : "+v"(voff[dc][hf]));
      }
    }
  }
  f32x16_t acc[C::DC];
#pragma unroll
  for (int dc = 0; dc < C::DC; ++dc) zero16(acc[dc]);

  // ---- Q rows through LDS (the V buffer), and the first pass: R = the maximum over the earlier blocks' landmark
  // scores, 64 landmarks at a time.  The first stage's K travels behind them.
  float R;
  {
#pragma unroll
    for (int i = 0; i < C::Q_PER_WAVE; ++i) {
      const int r = wave * C::Q_PER_WAVE + i;
      const int row = C::RPD * r + r_lane;
      const int slot = min(qt * 64 + row, p.Lq - 1), t = q_token(slot);
      const int tok = t >= 0 ? t : q_token(slot / BS * BS);   // a slot without a token reads its block's first
      split_dma16(qp, (uint32_t)tok * (uint32_t)(2 * p.qs_r) + swz(row), C::V_BASE + 1024 * r);
    }
    float mx = -INFINITY;
    for (int base = 0; base == 0 || base < cblk; base += C::LM_ROWS) {
      if (cblk > 0) {
#pragma unroll
        for (int i = 0; i < C::LM_PER_WAVE; ++i) {
          const int r = wave * C::LM_PER_WAVE + i;
          const int row = C::RPD * r + r_lane;
          const int tok = first_row(min(base + row, cblk - 1) + 1) - 1;    // an earlier block: complete
          split_dma16(kp, (uint32_t)tok * (uint32_t)(2 * p.ks_r) + swz(row), C::LM_BASE + 1024 * r);
        }
      }
      if (base == 0 && blk0 < n_complete && blk0 <= cblk) {
        request(false, 0);
        __builtin_amdgcn_s_waitcnt(0x0f70 | C::PER_WAVE);
      } else {
        if (base == 0) request(false, 0);
        wait_vm0();
      }
      __syncthreads();
      if (base == 0) {
#pragma unroll
        for (int ks = 0; ks < C::KS; ++ks) qf[ks] = lds_ld128(C::V_BASE + at(32 * tq) + koff[ks]);
        if (p.rope_cos != nullptr && qtok >= 0) {       // q without rotary: rotate the fragments at the row's position
          int64_t pos = p.rope_pos[(int64_t)b * p.rope_pos_stride_b + qtok];
          pos = pos < 0 ? 0 : (pos >= p.rope_n_pos ? p.rope_n_pos - 1 : pos);
          rotate_fragments<T, C::KS>(qf, (const char*)p.rope_cos + 2 * pos * p.rope_cs_r, (const char*)p.rope_sin + 2 * pos * p.rope_cs_r, h);
        }
      }
#pragma unroll
      for (int u = 0; u < C::LM_ROWS / 32; ++u) {
        if (base + 32 * u < cblk) {
          f32x16_t sl;
          zero16(sl);
#pragma unroll
          for (int ks = 0; ks < C::KS; ++ks) sl = mfma32<T>(lds_ld128(C::LM_BASE + at(32 * u) + koff[ks]), qf[ks], sl);
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = (base + 32 * u + 8 * (r >> 2) + 4 * h + (r & 3) < cblk) ? fmaxf(mx, sl[r]) : mx;
        }
      }
      if (base + C::LM_ROWS < cblk) __syncthreads();    // the area is written again
    }
    R = pair_max(mx) * c2;
  }

  float lrun = 0.f;                                     // this part's share of the global bucket's sum
  f32x16_t sc[2];                                       // scores, then exponentials, of the wave's two tiles
  const int half = part % C::NH;                        // BS 128: the part's half of its block
  const int xrow = C::X_BASE + tq * KP * C::X_PART + 4 * ql;

  // S^T of one or two tiles, t0 and t1 from the chunk's first row: the wave issues in order, so the instruction stream
  // is the schedule -- every operand is asked for PF MFMAs ahead of its use (a wave alone on its SIMD waits for LDS
  // otherwise), the order is pinned, and under(n) is vector work for the slot behind MFMA n
  auto scores = [&](int t0, int t1, auto n_c, auto under) __attribute__((always_inline)) {
    constexpr int NX = decltype(n_c)::value * C::KS, PF = 5 < NX ? 5 : NX;
    auto ld = [&](int n) __attribute__((always_inline)) { return lds_ld128((n / C::KS ? t1 : t0) + koff[n % C::KS]); };
    u32x4_t fk[NX];
#pragma unroll
    for (int n = 0; n < PF; ++n) fk[n] = ld(n);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < NX; ++n) {
      if (n + PF < NX) fk[n + PF] = ld(n + PF);
      if (n % C::KS == 0) zero16(sc[n / C::KS]);
      sc[n / C::KS] = mfma32<T>(fk[n], qf[n % C::KS], sc[n / C::KS]);
      under(n);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // O^T += V^T W of one or two tiles, W = f * sc: a slice of 16 keys is scaled and packed under the MFMAs of
  // the slice before
  auto product = [&](int t0, int t1, float f, auto n_c) __attribute__((always_inline)) {
    constexpr int NZ = decltype(n_c)::value * 2 * C::DC, PF = 4;
    auto ld = [&](int n) __attribute__((always_inline)) {
      const int sl = n / C::DC, dc = n % C::DC;
      const int base = (sl >> 1 ? t1 : t0) + 16 * (sl & 1) * C::ROWB;
      const u32x2_t a0 = lds_ld_tr(base + voff[dc][0]), a1 = lds_ld_tr(base + voff[dc][1]);
      const u32x4_t a = {a0[0], a0[1], a1[0], a1[1]};
      return a;
    };
    auto slice = [&](int sl) __attribute__((always_inline)) {
      const int u = sl >> 1, j = sl & 1;
      u32x4_t wf;
#pragma unroll
      for (int i = 0; i < 4; ++i) wf[i] = pack2<T>(sc[u][8 * j + 2 * i] * f, sc[u][8 * j + 2 * i + 1] * f);
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
  // slots of tile u of a block (rows 32u .. of it) that hold no key leave the softmax
  auto mask_padding = [&](f32x16_t& x, int u, int n_norm) __attribute__((always_inline)) {
    if (plain || n_norm >= BS - 1 || n_norm >= 32 * u + 32) return;
    int first = n_norm - 32 * u - 4 * h, last = BS - 1 - 32 * u - 4 * h;
    asm volatile("" : "+v"(first), "+v"(last));         // formed here: kept, the 16 masks fill the scalar registers
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int kl = 8 * (r >> 2) + (r & 3);
      if (kl >= first && kl < last) x[r] = -INFINITY;
    }
  };

  // ---- earlier block, first half: local softmax of the part's 64 keys.  mpart, den: maximum (log2 domain) and sum
  float mpart = 0.f, den = 0.f, t_lm = 0.f;
  auto earlier_scores = [&](int st) __attribute__((always_inline)) {
    const int n_norm = normal_keys(st * (KP / C::NH) + part / C::NH);
    float m0 = -INFINITY, m1 = -INFINITY;
    scores(0, 32 * C::ROWB, Two{}, [&](int n) __attribute__((always_inline)) {   // tile 0's maximum under tile 1's MFMAs
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
    float d0 = 0.f, d1 = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const int u = i >> 4, r = i & 15;
      float x = fast_exp2(__builtin_fmaf(sc[u][r], c2, -mloc));
      if (i == 31) x = lm ? 0.f : x;
      sc[u][r] = x;
      if (i & 1) d1 += x;
      else d0 += x;
    }
    den = pair_sum(d0 + d1);
    if constexpr (C::NH > 1) {
      lds_st32(xrow + part * C::X_PART + 128 * h, h == 0 ? mpart : den);
      if (half == C::NH - 1 && h == 0) lds_st32(xrow + part * C::X_PART + 256, t_lm);
    }
  };
  // second half, with the other half's numbers there: the weights' factor, and the product
  auto earlier_product = [&]() __attribute__((always_inline)) {
    float f;
    if constexpr (C::NH > 1) {
      const int other = xrow + (part ^ 1) * C::X_PART;
      const float mo = lds_ld32(other), dn = lds_ld32(other + 128);
      if (half == 0) t_lm = lds_ld32(other + 256);
      const float m = fmaxf(mpart, mo);
      const float a = fast_exp2(mpart - m);
      f = a * fast_rcp(__builtin_fmaf(den, a, dn * fast_exp2(mo - m)));
    } else {
      f = fast_rcp(den);
    }
    const float gate = fast_exp2(t_lm - R);             // R is the first pass's maximum: no greater landmark comes
    if (half == C::NH - 1) lrun += gate;
    f *= gate;
    if constexpr (GS) f *= lds_ld32(C::GS_BASE + wave * 256 + 4 * lane);
    product(0, 32 * C::ROWB, f, Two{});
  };
  auto request_v = [&](int st) __attribute__((always_inline)) {
    request(true, st);
    if constexpr (GS) {                                 // this lane's row's factor of the part's block
      const int blk = min(st * (KP / C::NH) + part / C::NH, cblk - 1);
      if (blk >= 0) {
        const float* src = p.group_scale + (int64_t)bh * p.gs_bh + (int64_t)blk * p.gs_blk + max(qtok, 0);
        split_dma4(src, C::GS_BASE + wave * 256);
      }
    }
  };

  // ---- stages of earlier blocks only
  const int last = cblk * C::NH / KP, own = cblk * C::NH % KP;   // the stage of the own block, and the own block's first part
  for (int st = 0; st < last; ++st) {
    wait_vm0();
    __syncthreads();                                    // K of the stage is there; V of the one before has been read
    request_v(st);
    earlier_scores(st);
    wait_vm0();
    __syncthreads();                                    // V is there; K has been read
    request(false, st + 1);
    earlier_product();
  }
  // ---- the own block's stage: parts in front of it have an earlier block, the others take its causal tiles
  float Mrun = R;
  {
    wait_vm0();
    __syncthreads();
    request_v(last);
    const int np = KP - own;                            // tile u of the own block goes to part own + u % np
    const int u0 = part - own, u1 = u0 + np;            // at most two per part
    const int otile = 64 * own;                         // the own block's first row in the stage
    const bool earlier = part < own, has0 = !earlier && u0 <= tsub, has1 = !earlier && u1 <= tsub;
    if (earlier) {
      earlier_scores(last);
    } else if (has0) {
      auto nothing = [](int) {};
      if (has1) scores(at(otile + 32 * u0), at(otile + 32 * u1), Two{}, nothing);
      else scores(at(otile + 32 * u0), 0, One{}, nothing);
      float mt = -INFINITY;
      const int n_norm = normal_keys(cblk);
      auto visible = [&](f32x16_t& x, int u) __attribute__((always_inline)) {
        mask_padding(x, u, n_norm);                         // only the landmark query could reach such a slot
        int lim = u < tsub ? 32 : ql - ((tsub == C::NT - 1 && ql == 31) ? 1 : 0) - 4 * h;   // landmark query looks one left
        asm volatile("" : "+v"(lim));
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          x[r] = 8 * (r >> 2) + (r & 3) <= lim ? x[r] * c2 : -INFINITY;
          mt = fmaxf(mt, x[r]);
        }
      };
      visible(sc[0], u0);
      if (has1) visible(sc[1], u1);
      Mrun = fmaxf(R, pair_max(mt));
      const float Msafe = Mrun == -INFINITY ? 0.f : Mrun;   // nothing for this part in the whole row
      const float alpha = fast_exp2(R - Msafe);
      float sum = 0.f;
      auto weigh = [&](f32x16_t& x) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          x[r] = fast_exp2(x[r] - Msafe);
          sum += x[r];
        }
      };
      weigh(sc[0]);
      if (has1) weigh(sc[1]);
      lrun = lrun * alpha + pair_sum(sum);
      if (__any(alpha != 1.0f)) {
#pragma unroll
        for (int dc = 0; dc < C::DC; ++dc)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[dc][r] *= alpha;
      }
    }
    wait_vm0();
    __syncthreads();
    if (earlier) {
      earlier_product();
    } else if (has0) {
      if (has1) product(at(otile + 32 * u0), at(otile + 32 * u1), 1.f, Two{});
      else product(at(otile + 32 * u0), 0, 1.f, One{});
    }
  }

  // ---- the parts meet: every part leaves its maximum, sum and accumulator, except for the output chunks dc = part,
  // part + KP, .. which it collects.  With two parts they fit the K buffer, which nobody reads any more.
  if constexpr (KP > 2 || C::NH > 1) __syncthreads();
  lds_st32(xrow + part * C::X_PART + 128 * h, h == 0 ? Mrun : lrun);
#pragma unroll
  for (int dc = 0; dc < C::DC; ++dc) {
    if (dc % KP == part) continue;
    const int to = ((tq * C::DC + dc) * (KP - 1) + part - (part > dc % KP ? 1 : 0)) * 4096 + 16 * lane;   // in part order
#pragma unroll
    for (int g = 0; g < 4; ++g)
      lds_st128(to + 1024 * g, u32x4_t{__float_as_uint(acc[dc][4 * g]), __float_as_uint(acc[dc][4 * g + 1]),
                                       __float_as_uint(acc[dc][4 * g + 2]), __float_as_uint(acc[dc][4 * g + 3])});
  }
  __syncthreads();
  float M = -INFINITY, l = 0.f, a[KP];                  // a: what a part's accumulator counts
#pragma unroll
  for (int q = 0; q < KP; ++q) {
    a[q] = lds_ld32(xrow + q * C::X_PART);
    M = fmaxf(M, a[q]);
  }
#pragma unroll
  for (int q = 0; q < KP; ++q) {
    a[q] = fast_exp2(a[q] - M);
    l = __builtin_fmaf(lds_ld32(xrow + q * C::X_PART + 128), a[q], l);
  }
  const float linv = 1.0f / l;
  const float own_scl = fast_exp2(Mrun - M);
#pragma unroll
  for (int dc = 0; dc < C::DC; ++dc) {
    if (dc % KP == part) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[dc][r] *= own_scl;
#pragma unroll
      for (int from = 0; from < KP - 1; ++from) {
        const int to = ((tq * C::DC + dc) * (KP - 1) + from) * 4096 + 16 * lane;
        const float w = a[from + (from >= dc % KP ? 1 : 0)];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const u32x4_t v = lds_ld128(to + 1024 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[dc][4 * g + i] = __builtin_fmaf(__uint_as_float(v[i]), w, acc[dc][4 * g + i]);
        }
      }
      store_tile_rows<T, 1>(&acc[dc], linv, C::STORE_BASE + wave * 2048, [&](int r) __attribute__((always_inline)) -> char* {
        const int qr = q0 + r;
        if (qr >= p.Lq) return nullptr;
        const int tok = q_token(qr);
        return tok < 0 ? nullptr : op + 2 * ((int64_t)tok * p.os_r) + 64 * dc;
      });
    }
  }
  if (part == 0 && qtok >= 0 && h == 0) {               // statistics follow the tensors' layout
    const int64_t si = (int64_t)bh * (tokens ? p.Lq_real : p.Lq) + qtok;
    p.L[si] = l;
    p.M[si] = M * kLn2;
  }
}

template <class T, int D, int BS, int KP, int LAYOUT>
static int launch_fwd_split_t(const FwdParams& p, hipStream_t stream) {
  using C = FwdSplitCfg<T, D, BS, KP>;
  auto kern = lmk_fwd_split_kernel<T, D, BS, KP, LAYOUT>;
  static std::atomic<uint64_t> lds_ok{0};
  return launch_rows64(kern, p, 64 * C::NW, C::LDS_BYTES, lds_ok, stream);
}

template <class T, int D, int BS, int KP>
static int launch_fwd_split_v(const FwdParams& p, hipStream_t stream) {
  if (p.seg != nullptr) return launch_fwd_split_t<T, D, BS, KP, TABLE>(p, stream);
  if (p.group_scale != nullptr) return launch_fwd_split_t<T, D, BS, KP, FACTORS>(p, stream);
  if (p.Lq_real <= 0 && p.n_real == BS) return launch_fwd_split_t<T, D, BS, KP, PLAIN>(p, stream);
  return launch_fwd_split_t<T, D, BS, KP, TOKENS>(p, stream);
}

template <class T, int D>
static int launch_fwd_split_d(const FwdParams& p, int BS, int kparts, hipStream_t stream) {
  if (BS == 64) return kparts == 4 ? launch_fwd_split_v<T, D, 64, 4>(p, stream) : launch_fwd_split_v<T, D, 64, 2>(p, stream);
  if (BS == 128) return kparts == 4 ? launch_fwd_split_v<T, D, 128, 4>(p, stream) : launch_fwd_split_v<T, D, 128, 2>(p, stream);
  return LMK_ERR_UNSUPPORTED;
}

int launch_fwd_split(const FwdParams& p, int D, int BS, int dtype, hipStream_t stream) {
  if (p.seg != nullptr && p.group_scale != nullptr) return LMK_ERR_UNSUPPORTED;
  const int kparts = key_parts(p.B, p.H, p.Lq, p.Lk);
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_fwd_split_d<bf16_t, 128>(p, BS, kparts, stream);
    if (D == 64) return launch_fwd_split_d<bf16_t, 64>(p, BS, kparts, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_fwd_split_d<f16_t, 128>(p, BS, kparts, stream);
    if (D == 64) return launch_fwd_split_d<f16_t, 64>(p, BS, kparts, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

}  // namespace lmk
