// dK/dV kernel of the backward pass for landmark blocks of 64 and 128 slots, 64 keys per workgroup.  The mathematics is
// lmk_bwd_dkdv32.hip's:
//     S = Q K^T,  W = exp2(S c - x) (the attention weights),  dP = dO V^T,  dS = W (dP - y) + z,
//     dV^T += dO^T W,  dK^T += Q^T dS
//     own block:      x = mhat, y = delta, z = 0, keys behind the query masked
//     earlier block:  x = a, y = nD, z = 0; at the block's landmark key W = 0 and z = dS as the dQ kernel left it
// That kernel gives a workgroup 128 keys, walks the queries 32 at a time and splits the work by role, one wave the weights
// and dV, the other dS and dK; B2 H8 L1024 is 128 workgroups of up to 32 steps.  Here a workgroup has 64 keys and 4 QP waves
// (2 key tiles x 2 query tiles x QP query parts), a stage is 64 queries per part, and both waves of a key tile do the same
// amount of everything: each forms S, dP, W and dS of one query tile of the unit, then one adds both tiles to dV^T, the
// other to dK^T.  W of the second tile and dS of the first change hands through LDS in between.  Two barriers per
// stage; Q, dO and the row terms of the next stage travel under the whole of the stage at hand (two LDS buffers).  The
// query parts' accumulators add up at the end.
#include <type_traits>

#include "lmk_common.hpp"
#include "lmk_launch.hpp"
#include "lmk_split.hpp"

namespace lmk {

template <class T, int D, int BS, int QP>
struct DkvSplitCfg {
  static constexpr int NW = 4 * QP;
  static constexpr int UPB = BS / 64;                   // units of 64 rows per block
  static constexpr int ROWB = 2 * D;
  static constexpr int CH = D / 8;                      // 16-byte chunks per row
  static constexpr int KS = D / 16;                     // MFMA k-steps over the head dim
  static constexpr int DC = D / 32;                     // 32-wide output chunks of the head dim
  static constexpr int HALF = 64 * ROWB;                // Q rows of a unit, then dO rows
  static constexpr int UNIT = 2 * HALF;
  static constexpr int BUF = QP * UNIT;                 // one stage: a unit per query part
  static constexpr int T_BASE = 2 * BUF;                // row terms: [buffer][part] a, nD, dS at the landmark, mhat, delta: 64 floats each
  static constexpr int T_PART = 2048;
  static constexpr int W_BASE = T_BASE + 2 * QP * T_PART;   // [part][key tile] W of query tile 1, dS of tile 0: [slice of 16 rows][lane] 16 bytes
  static constexpr int C_BASE = W_BASE + QP * 2 * 4096;     // 32 x 1e30f
  static constexpr int LDS_BYTES = C_BASE + 256;        // 76 KB at QP 1, D128: two workgroups per compute unit
  static constexpr int RPD = 1024 / ROWB;               // rows covered by one 1 KB request
  static constexpr int PER_WAVE = 64 / RPD / 4;         // requests per wave for a unit's Q (or dO): 16 rows
  static_assert(4 * (QP - 1) * DC * 4096 <= 2 * BUF, "the parts' accumulators fit the buffers");
  static_assert(NW * 2048 <= QP * 2 * 4096, "a wave's output tile goes through the W area");
};

template <class T, int D, int BS, int QP, int LAYOUT>
__global__ __launch_bounds__(256 * QP, 2) void lmk_bwd_dkdv_split_kernel(BwdParams p) {
  constexpr bool plain = LAYOUT == PLAIN, SEG = LAYOUT == TABLE;
  using C = DkvSplitCfg<T, D, BS, QP>;
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int part = wave >> 2, tile = wave & 1;          // query part, key tile
  const int qt = (wave >> 1) & 1;                       // the wave's query tile in a unit; 0: collects dV, 1: dK
  const bool role_k = qt != 0;
  const int ql = lane & 31, h = lane >> 5;

  const int hh = blockIdx.x, b = p.b0 + blockIdx.y, ku = p.kt0 + blockIdx.z;   // ku: unit of 64 keys; the first sees the most queries
  const int bh = b * p.H + hh;
  const char* qp = (const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h);
  const char* gp = (const char*)p.dout + 2 * (b * p.dos_b + hh * p.dos_h);
  const char* kp = (const char*)p.k + 2 * (b * p.ks_b + hh * p.ks_h);
  const char* vp = (const char*)p.v + 2 * (b * p.vs_b + hh * p.vs_h);

  const bool tokens = !plain && p.Lq_real > 0;          // rows are tokens; otherwise rows are slots
  const int n_tok = tokens ? p.n_real : BS;             // rows per block
  auto slot_row = [&](int slot, int n) __attribute__((always_inline)) {   // slots without a token read their block's first
    return plain ? slot : (slot == BS - 1 ? n - 1 : (slot < n - 1 ? slot : 0));
  };
  const int kblk = ku / C::UPB;                         // the keys' block
  const int p_units = p.n_prefix * C::UPB, n_units = p.Lq >> 6;   // units of history, of queries
  const int j0 = max(0, ku - p_units);                  // first unit of queries that sees any of the keys
  const int n_stages = (n_units - j0 + QP - 1) / QP;

  // ---- direct loads: a wave fetches 16 rows of each tensor's 64; the LDS swizzle is applied on the source side
  const int r_lane = lane / C::CH, cp = lane % C::CH;
  auto swz = [&](int row) __attribute__((always_inline)) {
    const int f = tile_swizzle<D>(row);
    return 16 * (cp ^ f);
  };
  const int w4 = wave & 3;
  // request i of this wave's share of a unit's 64 rows of a tensor
  auto fetch = [&](const char* src, int64_t stride, int unit, const int* seg, int dst, int i) __attribute__((always_inline)) {
    const int blk = unit / C::UPB;
    const int row_b = SEG ? seg[blk] - seg[0] : blk * n_tok, n = SEG ? seg[blk + 1] - seg[blk] : n_tok;
    const uint32_t rs = (uint32_t)(2 * stride);
    const int row = 16 * w4 + r_lane + C::RPD * i;      // of the unit
    const uint32_t t = (uint32_t)(row_b + slot_row((unit % C::UPB) * 64 + row, n));
    split_dma16(src, t * rs + swz(row), dst + 1024 * (w4 * C::PER_WAVE + i));
  };
  const float* const plane_a = p.stat_a + ((int64_t)bh * p.n_blocks + kblk) * p.Lq;
  const float* const plane_n = p.stat_n + ((int64_t)bh * p.n_blocks + kblk) * p.Lq;
  const float* const plane_l = p.stat_l + ((int64_t)bh * p.n_blocks + kblk) * p.Lq;
  // Piece i of this wave's share of its part's unit of stage st.  A stage's pieces go out one behind every second MFMA of the
  // stage before: a compute unit takes in 64 bytes per cycle, four waves' requests of 1 KB are 64 cycles, and a wave stands
  // still while its request waits for the others' (asked for together, 1200-1700 of a stage's 5000 cycles).
  constexpr int PIECES = 2 * C::PER_WAVE + 1;           // C::KS of rows and one of terms
  static_assert(PIECES == C::KS + 1, "one per two MFMAs of S and dP");
  const int* const seg_q = SEG ? p.seg + p.n_prefix : nullptr;
  auto request_piece = [&](int st, int i) __attribute__((always_inline)) {
    const int j = j0 + st * QP + part, buf = st & 1;
    const int u = buf * C::BUF + part * C::UNIT;
    if (i < C::PER_WAVE) {
      fetch(qp, p.qs_r, j, seg_q, u, i);
    } else if (i < 2 * C::PER_WAVE) {
      fetch(gp, p.dos_r, j, seg_q, u + C::HALF, i - C::PER_WAVE);
    } else if (w4 < 2) {                                // 64 floats of a term are 16 lanes' 16 bytes
      const int arr = 4 * w4 + (lane >> 4);             // 0 .. 3, then delta (four times)
      const float* src = arr == 0 ? plane_a : arr == 1 ? plane_n : arr == 2 ? plane_l : (arr == 3 ? p.mhat : p.delta) + (int64_t)bh * p.Lq;
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                   :: "v"(src + 64 * j + 4 * (lane & 15)),
                      "s"(__builtin_amdgcn_readfirstlane(C::T_BASE + (buf * QP + part) * C::T_PART + 1024 * w4)) : "memory");
    }
  };

  // ---- LDS byte addresses of this lane's operand fragments: the wave's query tile in the part's unit, as rows (of Q;
  // HALF leads to dO) and transposed (of dO for dV, of Q for dK).  Kept for the buffer at hand: a stage turns their buffer bit instead of adding it to every read.
  static_assert((C::BUF & (C::BUF - 1)) == 0, "a buffer is one bit of the address");
  const int ubase = part * C::UNIT;
  int koff[C::KS];
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) {
    koff[ks] = ubase + 32 * qt * C::ROWB + tile_off<D>(ql, 2 * ks + h);
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
        voff[dc][hf] = ubase + (role_k ? 0 : C::HALF) + 32 * qt * C::ROWB + tile_off<D>(4 * h + (i >> 2) + 8 * hf, col >> 3) + ((col >> 2) & 1) * 8;
        asm volatile("" : "+v"(voff[dc][hf]));
      }
    }
  }

  // ---- the keys' rows through LDS (the second buffer; every part brings and reads its own), the first stage's unit beside them
  u32x4_t kf[C::KS], vf[C::KS];                         // stationary operands, lane = key
#pragma unroll
  for (int i = 0; i < C::PER_WAVE; ++i) {
    fetch(kp, p.ks_r, ku, SEG ? p.seg : nullptr, C::BUF + ubase, i);
    fetch(vp, p.vs_r, ku, SEG ? p.seg : nullptr, C::BUF + ubase + C::HALF, i);
  }
  if (j0 + part < n_units) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) request_piece(0, i);
  }
  if (tid < 32) lds_st32(C::C_BASE + 4 * tid, 1e30f);
  wait_vm0();
  __syncthreads();
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) {
    kf[ks] = lds_ld128(C::BUF + 32 * (tile - qt) * C::ROWB + koff[ks]);
    vf[ks] = lds_ld128(C::BUF + C::HALF + 32 * (tile - qt) * C::ROWB + koff[ks]);
  }
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) asm volatile("" : "+v"(kf[ks]), "+v"(vf[ks]));   // read before the barrier below

  f32x16_t acc[C::DC], sc, dp;
#pragma unroll
  for (int dc = 0; dc < C::DC; ++dc) zero16(acc[dc]);
  const float c2 = p.scale_log2;
  const bool lm_tile = tile == 1 && ku % C::UPB == C::UPB - 1;   // this key tile ends in its block's landmark
  const bool lm_lane = lm_tile && ql == 31;

  // the wave's 32 rows at `base` from its Q rows x its key tile: operands asked for PF MFMAs ahead, order pinned, under(n) behind MFMA n
  auto row_tile = [&](int base, const u32x4_t* bf, f32x16_t& out, auto under) __attribute__((always_inline)) {
    constexpr int PF = 4;
    u32x4_t fk[C::KS];
#pragma unroll
    for (int n = 0; n < PF; ++n) fk[n] = lds_ld128(base + koff[n]);
    __builtin_amdgcn_sched_barrier(0);
    zero16(out);
#pragma unroll
    for (int n = 0; n < C::KS; ++n) {
      if (n + PF < C::KS) fk[n + PF] = lds_ld128(base + koff[n + PF]);
      out = mfma32<T>(fk[n], bf[n], out);
      under(n);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // acc += (the unit's two tiles)^T x packed operands: the wave's own tile first, the other's
  // operand is still on its way
  auto product = [&](const u32x4_t* own, const u32x4_t* other) __attribute__((always_inline)) {
    constexpr int NZ = 4 * C::DC, PF = 4;
    int vo[C::DC][2];
#pragma unroll
    for (int dc = 0; dc < C::DC; ++dc)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        vo[dc][hf] = voff[dc][hf] ^ (32 * C::ROWB);
        asm volatile("" : "+v"(vo[dc][hf]));
      }
    auto ld = [&](int n) __attribute__((always_inline)) {
      const int dc = n % C::DC, sl = n / C::DC, at = 16 * (sl & 1) * C::ROWB;
      const u32x2_t a0 = lds_ld_tr(at + (sl < 2 ? voff : vo)[dc][0]), a1 = lds_ld_tr(at + (sl < 2 ? voff : vo)[dc][1]);
      const u32x4_t a = {a0[0], a0[1], a1[0], a1[1]};
      return a;
    };
    u32x4_t zf[NZ];
#pragma unroll
    for (int n = 0; n < PF; ++n) zf[n] = ld(n);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < NZ; ++n) {
      if (n + PF < NZ) zf[n + PF] = ld(n + PF);
      const int sl = n / C::DC;
      acc[n % C::DC] = mfma32<T>(zf[n], sl < 2 ? own[sl] : other[sl - 2], acc[n % C::DC]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
  auto ldf4 = [&](int addr) __attribute__((always_inline)) { return __builtin_bit_cast(f32x4, lds_ld128(addr)); };
  const int w_at = C::W_BASE + (part * 2 + tile) * 4096 + 16 * lane;   // W of query tile 1; dS of tile 0 behind it
  auto begin = [&]() __attribute__((always_inline)) {      // the stage's rows are there; the other buffer has been read
    wait_vm0();
    __syncthreads();
  };
  // The part's units: first those in the keys' own block (masked), then those behind it; each kind has a loop of its own,
  // so that the accumulators stay where they are.  A part without a unit in the last stage only meets the others.
  const int n_mine = (n_units - j0 - part + QP - 1) / QP;   // n_stages or one less
  const int own_end = (kblk + 1) * C::UPB - p_units;    // first unit of queries behind the own block
  const int n_own = ku < p_units ? 0 : min(n_mine, (max(own_end - j0 - part, 0) + QP - 1) / QP);
  auto stage = [&](auto own_c, int st) __attribute__((always_inline)) {
    constexpr bool OWN = decltype(own_c)::value;
    const int j = j0 + st * QP + part;
    begin();
    const bool more = j + QP < n_units;
    const int ta = C::T_BASE + ((st & 1) * QP + part) * C::T_PART + 128 * qt + 16 * h;   // this lane's rows 8g + 4h .. of tile qt
    const int xa = OWN ? ta + 768 : (lm_lane ? C::C_BASE + 16 * h : ta), ya = ta + (OWN ? 1024 : 256), za = ta + 512;
    u32x4_t wf[2], df[2];                               // W and dS of the wave's query tile, packed: slices of 16 rows
    float w[16];
    auto weigh = [&](int g) __attribute__((always_inline)) {   // registers 4g .. 4g+3: rows 8g + 4h .. of the tile
      const f32x4 x = ldf4(xa + 32 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = fast_exp2(__builtin_fmaf(sc[4 * g + e], c2, -x[e]));
        if (OWN) {                                      // key visible to this query row?  the landmark row of a block looks one position to the left
          const int qloc = 8 * g + 4 * h + e;
          const int krel = 32 * (2 * (ku - p_units - j) + tile - qt) + ql;   // key relative to the tile's first row
          const bool lmq = qloc == 31 && qt == 1 && j % C::UPB == C::UPB - 1;
          v = krel <= qloc - (lmq ? 1 : 0) ? v : 0.f;
        }
        w[4 * g + e] = v;
      }
      wf[g >> 1][2 * (g & 1)] = pack2<T>(w[4 * g], w[4 * g + 1]);
      wf[g >> 1][2 * (g & 1) + 1] = pack2<T>(w[4 * g + 2], w[4 * g + 3]);
    };
    row_tile(0, kf, sc, [&](int n) __attribute__((always_inline)) {
      if (more && n % 2 == 0) request_piece(st + 1, n / 2);
    });
    f32x4 y[4];
    row_tile(C::HALF, vf, dp, [&](int n) __attribute__((always_inline)) {   // W under dP's MFMAs
      constexpr int G0 = C::KS > 4 ? 2 : 0;
      if (n >= G0 && n - G0 < 4) weigh(n - G0);
      if (more && n % 2 == 0) request_piece(st + 1, (C::KS + n) / 2);
      if (more && n == 1) request_piece(st + 1, PIECES - 1);
      if (n == C::KS - 1) {
#pragma unroll
        for (int g = 0; g < 4; ++g) y[g] = ldf4(ya + 32 * g);
      }
    });
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float d[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) d[e] = w[4 * g + e] * (dp[4 * g + e] - y[g][e]);
      if (!OWN && lm_tile) {                            // wave-uniform; the landmark's W is zero
        const f32x4 z = ldf4(za + 32 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = lm_lane ? z[e] : d[e];
      }
      df[g >> 1][2 * (g & 1)] = pack2<T>(d[0], d[1]);
      df[g >> 1][2 * (g & 1) + 1] = pack2<T>(d[2], d[3]);
    }
#pragma unroll
    for (int n = 0; n < 2; ++n) lds_st128(w_at + (role_k ? 0 : 2048) + 1024 * n, role_k ? wf[n] : df[n]);
    __syncthreads();                                    // they change hands
    u32x4_t own[2], other[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      other[n] = lds_ld128(w_at + (role_k ? 2048 : 0) + 1024 * n);
      own[n] = role_k ? df[n] : wf[n];
    }
    product(own, other);
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) koff[ks] ^= C::BUF;
#pragma unroll
    for (int dc = 0; dc < C::DC; ++dc) voff[dc][0] ^= C::BUF, voff[dc][1] ^= C::BUF;
  };
  {
    int st = 0;
    for (; st < n_own; ++st) stage(std::true_type{}, st);
    for (; st < n_mine; ++st) stage(std::false_type{}, st);
  }
  if (n_mine < n_stages) {
    begin();
    __syncthreads();
  }

  // ---- the query parts meet: each leaves the output chunks dc with dc % QP != part for the other and collects its own
  char* const out = role_k ? (char*)p.dk + 2 * (b * p.dks_b + hh * p.dks_h) : (char*)p.dv + 2 * (b * p.dvs_b + hh * p.dvs_h);
  const int64_t out_r = role_k ? p.dks_r : p.dvs_r;
  const float scl = role_k ? p.scale : 1.f;
  auto row_ptr = [&](int r) __attribute__((always_inline)) -> char* {
    const int slot = ku * 64 + 32 * tile + r;
    const int row = plain ? slot : slot_to_token_row<BS>(slot, n_tok, tokens ? p.n_full_k : p.Lk / BS, SEG ? p.seg : nullptr);
    return row < 0 ? nullptr : out + 2 * ((int64_t)row * out_r);
  };
  __syncthreads();                                      // nobody reads the buffers or the hand-over any more
  if constexpr (QP == 1) {
    store_tile_rows<T, C::DC>(acc, scl, C::W_BASE + wave * 2048, row_ptr);
  } else {
    const int l16 = 16 * lane_id();
#pragma unroll
    for (int dc = 0; dc < C::DC; ++dc) {
      if (dc % QP == part) continue;
      const int to = ((wave & 3) * C::DC + dc) * 4096 + l16;
#pragma unroll
      for (int g = 0; g < 4; ++g)
        lds_st128(to + 1024 * g, u32x4_t{__float_as_uint(acc[dc][4 * g]), __float_as_uint(acc[dc][4 * g + 1]),
                                         __float_as_uint(acc[dc][4 * g + 2]), __float_as_uint(acc[dc][4 * g + 3])});
    }
    __syncthreads();
#pragma unroll
    for (int dc = 0; dc < C::DC; ++dc) {
      if (dc % QP != part) continue;
      const int to = ((wave & 3) * C::DC + dc) * 4096 + l16;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const u32x4_t v = lds_ld128(to + 1024 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[dc][4 * g + i] += __uint_as_float(v[i]);
      }
      store_tile_rows<T, 1>(&acc[dc], scl, C::W_BASE + wave * 2048, [&](int r) __attribute__((always_inline)) -> char* {
        char* const at = row_ptr(r);
        return at == nullptr ? nullptr : at + 64 * dc;
      });
    }
  }
}

template <class T, int D, int BS, int QP, int LAYOUT>
static int launch_dkdv_split_t(const BwdParams& p, hipStream_t stream) {
  using C = DkvSplitCfg<T, D, BS, QP>;
  auto kern = lmk_bwd_dkdv_split_kernel<T, D, BS, QP, LAYOUT>;
  static std::atomic<uint64_t> lds_ok{0};
  if (int rc = allow_dynamic_lds(kern, C::LDS_BYTES, lds_ok)) return rc;
  constexpr int kMax = 65535;
  const int n = p.Lk / 64;
  BwdParams c = p;
  for (c.b0 = 0; c.b0 < p.B; c.b0 += kMax)
    for (c.kt0 = 0; c.kt0 < n; c.kt0 += kMax)
      hipLaunchKernelGGL(kern, dim3(p.H, std::min(p.B - c.b0, kMax), std::min(n - c.kt0, kMax)), dim3(64 * C::NW), C::LDS_BYTES, stream, c);
  return (int)hipGetLastError();
}

template <class T, int D, int BS, int QP>
static int launch_dkdv_split_v(const BwdParams& p, hipStream_t stream) {
  if (p.seg != nullptr) return launch_dkdv_split_t<T, D, BS, QP, TABLE>(p, stream);
  if (p.Lq_real <= 0) return launch_dkdv_split_t<T, D, BS, QP, PLAIN>(p, stream);   // (padding slots are rows like others here)
  return launch_dkdv_split_t<T, D, BS, QP, TOKENS>(p, stream);
}

template <class T, int D>
static int launch_dkdv_split_d(const BwdParams& p, int BS, int parts, hipStream_t stream) {
  if (BS == 64) return parts == 2 ? launch_dkdv_split_v<T, D, 64, 2>(p, stream) : launch_dkdv_split_v<T, D, 64, 1>(p, stream);
  if (BS == 128) return parts == 2 ? launch_dkdv_split_v<T, D, 128, 2>(p, stream) : launch_dkdv_split_v<T, D, 128, 1>(p, stream);
  return LMK_ERR_UNSUPPORTED;
}

int launch_bwd_dkdv_split(const BwdParams& p, int D, int BS, int dtype, hipStream_t stream) {
  // two query parts put two waves on every SIMD where each compute unit has one workgroup (B2 H8 L1024: 28.9 -> 22.7 us), and
  // pay with two if the walk is long enough (B1 H32 L1024: 32.3 -> 30.2; at B4 H12 L640 they lose, 22.8 -> 23.4)
  const int64_t n = (int64_t)p.B * p.H * (p.Lk / 64), cus = cu_count();
  const int parts = n <= cus || (n <= 2 * cus && p.Lk >= 1024) ? 2 : 1;
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_dkdv_split_d<bf16_t, 128>(p, BS, parts, stream);
    if (D == 64) return launch_dkdv_split_d<bf16_t, 64>(p, BS, parts, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_dkdv_split_d<f16_t, 128>(p, BS, parts, stream);
    if (D == 64) return launch_dkdv_split_d<f16_t, 64>(p, BS, parts, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

}  // namespace lmk
