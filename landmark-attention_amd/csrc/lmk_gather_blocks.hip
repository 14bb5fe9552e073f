// Gather + attend by block: the same attention over picked cache blocks as lmk_gather_attend_kernel (lmk_retrieval.hip),
// for steps in which a block is picked by several query rows (a chunk of new tokens over a cache of few blocks, the
// benchmark models' ring cache).
//
// Row by row, a block that 25 rows picked is read, rotated and multiplied 25 times, on the vector unit: 255 queries of 24
// heads of 64 over a ring of 40 blocks of 51, top 4, took 54.7 us for 12 MB of cache; the two kernels here take 15.0 + 4.0.
// A workgroup owns up to four blocks of one (batch, head): it collects the rows that picked them, and attends for up to 32 of
// them at a time on the matrix cores.
// A pick is (row, rank), and a block's keys sit at positions that depend on the pick's rank in its row: a wave takes up to 32
// picks of one rank, rotates the keys for that rank, once for them, as it reads them -- fragment ks of a lane holds its key's head dims
// 16 ks + 8 h .. + 7, whose rotary partners are fragment ks + KS / 2 of the same lane -- and multiplies the rotated key as
// the sum of three 16-bit numbers, which keeps every bit of the fp32 rotation (KeyParts; with two, scores in the thousands
// came out up to 1.6 times as far from float64 as row by row; the third costs the step 1 to 3 %).  The local softmax and the
// sum over the values are those of the forward kernels (a lane owns a row).  (Rotating by the whole workgroup into LDS, with picks
// of all ranks side by side in one product, has two barriers and a round trip to the tables per rank: block 128, head dim 128,
// 32 heads, 256 queries, top 4 of 64 blocks 194 us a step against 123.)  What bounds it is the vector work of a rotation, ~12
// instructions per key and head dim, and the chain of loads in front of it: picks, queries, table rows.
// What a pick contributes -- the landmark's score and the normalised sum over the block, fp32 -- goes to a workspace, and
// lmk_gather_combine_kernel puts each row's picks and its local window together.
#include <algorithm>

#include "lmk_common.hpp"
#include "lmk_launch.hpp"
#include "lmk_split.hpp"

namespace lmk {

constexpr int kPickSegment = 2048;                      // picks of a (batch, head) looked through at a time

template <int D, int BS>
struct GatherBlocksCfg {
  static constexpr int NT = BS / 32;                    // 32-key tiles
  static constexpr int ROWB = 2 * D;
  static constexpr int CH = D / 8;                      // 16-byte chunks per row
  static constexpr int KS = D / 16;
  static constexpr int DC = D / 32;
  static constexpr int TILE = BS * ROWB;                // a block's keys, or its values
  static constexpr int MAX_OWN = 2 * TILE * 4 <= 65536 ? 4 : 65536 / (2 * TILE);   // blocks a workgroup owns at most: 64 KB
  // behind them: the segment's picks, 16 bits each; 256 counts; the groups, and four partial sums
  static constexpr int COUNT = 2 * kPickSegment, UNITS = COUNT + 4 * 256, MAX_UNITS = kPickSegment / 32 + 256;
  static constexpr int LIST_BYTES = UNITS + 4 * (MAX_UNITS + 4);
  static constexpr int RPD = 1024 / ROWB;               // rows covered by one 1 KB request
  static constexpr int PER_WAVE = BS / RPD / 4;         // requests per wave for the keys, and for the values
  static_assert(PER_WAVE * RPD * 4 == BS, "every wave issues the same number of requests");
};

// Rotated keys a, b (fp32) -> the operands hi, mid, lo of 16 bits each whose sum they are:
//   key = up (hi + step (mid + lo)),  score = up (q . hi + step (q . mid + q . lo))
// bf16: up = step = 1, three times eight bits by truncation: exact.  fp16: eleven bits and eleven of the rest, scaled by 1 / step
// to lie in fp16's range whatever the key, and what is left; up keeps rotated keys of fp16's largest values in range.
// The rest is formed from the clamped key, so that it stays finite where the key is infinite or NaN, which hi alone carries.
template <class T>
struct KeyParts;
template <>
struct KeyParts<bf16_t> {
  static constexpr float up = 1.f, step = 1.f;
  static __device__ __forceinline__ void split(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    constexpr float most = 3.4028234663852886e38f;
    auto top = [](float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); };
    auto tops = [](float x, float y) { return __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u); };
    const float ca = __builtin_amdgcn_fmed3f(a, -most, most), cb = __builtin_amdgcn_fmed3f(b, -most, most);
    const float ma = ca - top(ca), mb = cb - top(cb);
    hi = tops(a, b);
    mid = tops(ma, mb);
    lo = tops(ma - top(ma), mb - top(mb));
  }
};
template <>
struct KeyParts<f16_t> {
  static constexpr float up = 16.f, step = 1.f / 2048.f;
  static __device__ __forceinline__ uint32_t trunc2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
  }
  static __device__ __forceinline__ void split(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    constexpr float most = 65504.f;
    const float xa = a * (1.f / up), xb = b * (1.f / up);
    const float ca = __builtin_amdgcn_fmed3f(xa, -most, most), cb = __builtin_amdgcn_fmed3f(xb, -most, most);
    const uint32_t h = trunc2(ca, cb);
    const float ma = (ca - unpack_lo<f16_t>(h)) * (1.f / step), mb = (cb - unpack_hi<f16_t>(h)) * (1.f / step);
    hi = trunc2(xa, xb);
    mid = trunc2(ma, mb);
    lo = trunc2(ma - unpack_lo<f16_t>(mid), mb - unpack_hi<f16_t>(mid));
  }
};

// Rows t_first .. t_first + t_rows - 1 of every (batch, head); the workspace holds these rows' picks.
template <class T, int D, int BS, bool PADDED>
__global__ __launch_bounds__(256, 2) void lmk_gather_blocks_kernel(RetrParams p, int t_first, int t_rows, int n_own) {
  using C = GatherBlocksCfg<D, BS>;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ql = lane & 31, h = lane >> 5;
  // heads vary fastest: with a multiple of 8 of them a head's queries and picks are read through one XCD's L2
  const int bh = blockIdx.x, blk0 = blockIdx.y * n_own, b = bh / p.H, hh = bh % p.H;
  const int nreal = PADDED ? p.block : BS;
  auto token_of = [&](int slot) __attribute__((always_inline)) {   // slot of the block's BS -> token of the block it reads
    if (!PADDED) return slot;
    return slot == BS - 1 ? nreal - 1 : min(slot, nreal - 2);
  };
  const int k = p.k, picks = t_rows * k;                // of this (batch, head); at most 2^30 (gather_blocks_rows)
  const int64_t* idx = p.idx + (b * p.idx_sb + hh * p.idx_sh);
  const char* qp = (const char*)p.q + 2 * (b * p.qs_b + hh * p.qs_h);
  const char* kp = (const char*)p.kcache + 2 * (b * p.kcs_b + hh * p.kcs_h);
  const char* vp = (const char*)p.vcache + 2 * (b * p.vcs_b + hh * p.vcs_h);
  const int lists = 2 * C::TILE * n_own;                // LDS: per block its keys, then its values; then
  unsigned short* const list = (unsigned short*)(smem + lists);                    // the segment's picks by block and rank,
  int* const count = (int*)(smem + lists + C::COUNT);                              // how many (64 block + rank),
  uint32_t* const units = (uint32_t*)(smem + lists + C::UNITS);                    // and groups of at most 32 of one block and rank

  // ---- requests: the first segment's picks, the blocks' keys and values
  int64_t pick[kPickSegment / 256];
  auto fetch_picks = [&](int seg) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kPickSegment / 256; ++i) {
      const int e = seg + tid + 256 * i;
      pick[i] = -1;
      if (e < picks) {
        const int t = e / k;
        pick[i] = idx[(int64_t)(t_first + t) * p.idx_st + (e - t * k)];
      }
    }
  };
  fetch_picks(0);
  {
    const int row = C::RPD * C::PER_WAVE * wave + lane / C::CH;
    for (int g = 0; g < n_own; ++g) {
      const int64_t first = (int64_t)min(blk0 + g, p.num_mems - 1) * nreal;
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const char* src = v ? vp + 2 * (first * p.vcs_r) : kp + 2 * (first * p.kcs_r);
        const uint32_t stride = (uint32_t)(2 * (v ? p.vcs_r : p.kcs_r));
#pragma unroll
        for (int i = 0; i < C::PER_WAVE; ++i) {
          const int r = row + C::RPD * i, f = tile_swizzle<D>(r);
          split_dma16(src, (uint32_t)token_of(r) * stride + 16 * ((lane % C::CH) ^ f), (2 * g + v) * C::TILE + 1024 * (wave * C::PER_WAVE + i));
        }
      }
    }
  }

  int koff[C::KS];                                      // the operands' places in the first tile
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) koff[ks] = tile_off<D>(ql, 2 * ks + h);
  using P = KeyParts<T>;
  const float c2 = p.scale_log2 * P::up;

  for (int seg = 0; seg < picks; seg += kPickSegment) {
    if (seg > 0) {
      fetch_picks(seg);
      __syncthreads();                                  // the lists have been read
    }
    count[tid] = 0;
    __syncthreads();
    // ---- the list: a counting sort by block and rank.  The order within a rank is the order the threads came in; a
    // row's result does not depend on its place
    int place[kPickSegment / 256];                      // among the picks of its block and rank, and these; -1: not ours
#pragma unroll
    for (int i = 0; i < kPickSegment / 256; ++i) {
      const int e = seg + tid + 256 * i;
      place[i] = -1;
      if (e < picks) {
        const int g = min(max((int)pick[i], 0), p.num_mems - 1) - blk0;   // a caller's array
        if (g >= 0 && g < n_own) {
          const int key = 64 * g + e % k;
          place[i] = key + 256 * atomicAdd(count + key, 1);
        }
      }
    }
    __syncthreads();
    // thread: one (block, rank); a wave's four sums of 16 bits: picks in front of it and groups in front of it
    const int n_key = count[tid];
    uint32_t sum = (uint32_t)n_key | ((uint32_t)((n_key + 31) >> 5) << 16);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)sum, d, 64);
      sum += lane >= d ? y : 0;
    }
    if (lane == 63) units[C::MAX_UNITS + wave] = sum;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t x = units[C::MAX_UNITS + w];
      before += w < wave ? x : 0;
      all += x;
    }
    sum += before;
    const int at_key = (int)(sum & 0xffff) - n_key;
    count[tid] = at_key;                                // now where its picks start
    for (int i = 0, u = (int)(sum >> 16) - ((n_key + 31) >> 5); 32 * i < n_key; ++i, ++u)
      units[u] = (uint32_t)tid | ((uint32_t)(at_key + 32 * i) << 8) | ((uint32_t)min(n_key - 32 * i, 32) << 20);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPickSegment / 256; ++i)
      if (place[i] >= 0) list[count[place[i] & 255] + (place[i] >> 8)] = (unsigned short)(tid + 256 * i);
    wait_vm0();                                         // the keys and values
    __syncthreads();
    const int n_units = __builtin_amdgcn_readfirstlane((int)(all >> 16));
    for (int unit = wave; unit < n_units; unit += 4) {  // a wave's own: no barrier below
      const uint32_t ud = (uint32_t)__builtin_amdgcn_readfirstlane((int)units[unit]);
      const int g = (ud >> 6) & 3, r = ud & 63, ng = ud >> 20, blk = blk0 + g, ktile = 2 * g * C::TILE;
      int age = blk - p.ring_start;                     // one of the k newest blocks: its keys sit one block further on
      age += age < 0 ? p.num_mems : 0;
      const int64_t pos0 = p.prefix_len + (age >= p.num_mems - k ? nreal : 0);
      const int e = seg + list[((ud >> 8) & 0xfff) + min(ql, ng - 1)];
      const int t = e / k;
      u32x4_t qf[C::KS];
      const char* qr = qp + 2 * ((int64_t)(t_first + t) * p.qs_r) + 16 * h;
#pragma unroll
      for (int ks = 0; ks < C::KS; ++ks) qf[ks] = *(const u32x4_t*)(qr + 32 * ks);
      // ---- S^T, a pair of fragments at a time: their table rows are on their way PF pairs ahead
      constexpr int NX = C::NT * C::KS / 2, PF = C::KS / 2 < 4 || BS == 128 ? 2 : 4;
      const int64_t pos = 2 * (pos0 + (int64_t)r * nreal) * p.cs_r;
      const char *cb = (const char*)p.cos + pos, *sb = (const char*)p.sin + pos;
      u32x4_t tab[PF][4];
      auto fetch_tables = [&](int n) __attribute__((always_inline)) {
        const uint32_t off = (uint32_t)token_of(32 * (n / (C::KS / 2)) + ql) * (uint32_t)(2 * p.cs_r) + 16 * h;
        u32x4_t* x = tab[n % PF];
        x[0] = *(const u32x4_t*)(cb + off + 32 * (n % (C::KS / 2)));
        x[1] = *(const u32x4_t*)(cb + off + 32 * (n % (C::KS / 2)) + D);
        x[2] = *(const u32x4_t*)(sb + off + 32 * (n % (C::KS / 2)));
        x[3] = *(const u32x4_t*)(sb + off + 32 * (n % (C::KS / 2)) + D);
      };
#pragma unroll
      for (int n = 0; n < PF; ++n) fetch_tables(n);
      f32x16_t s[C::NT], rest;
#pragma unroll
      for (int n = 0; n < NX; ++n) {
        const int nt = n / (C::KS / 2), ks = n % (C::KS / 2);
        const u32x4_t klo = lds_ld128(ktile + 32 * nt * C::ROWB + koff[ks]), khi = lds_ld128(ktile + 32 * nt * C::ROWB + koff[ks + C::KS / 2]);
        const u32x4_t *x = tab[n % PF];
        u32x4_t hi[2], mid[2], lo[2];                   // of both halves
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          float y[2][2];                                // half, element
          auto rot = [&](float kl, float kh, float cl, float ch, float sl, float sh, int i) __attribute__((always_inline)) {
            y[0][i] = __builtin_fmaf(kl, cl, -kh * sl);
            y[1][i] = __builtin_fmaf(kh, ch, kl * sh);
          };
          rot(unpack_lo<T>(klo[d]), unpack_lo<T>(khi[d]), unpack_lo<T>(x[0][d]), unpack_lo<T>(x[1][d]), unpack_lo<T>(x[2][d]),
              unpack_lo<T>(x[3][d]), 0);
          rot(unpack_hi<T>(klo[d]), unpack_hi<T>(khi[d]), unpack_hi<T>(x[0][d]), unpack_hi<T>(x[1][d]), unpack_hi<T>(x[2][d]),
              unpack_hi<T>(x[3][d]), 1);
#pragma unroll
          for (int hf = 0; hf < 2; ++hf) {
            uint32_t a, b, c;
            P::split(y[hf][0], y[hf][1], a, b, c);
            hi[hf][d] = a;
            mid[hf][d] = b;
            lo[hf][d] = c;
          }
        }
        if (n + PF < NX) fetch_tables(n + PF);
        if (ks == 0) {
          zero16(s[nt]);
          if (P::step != 1.f) zero16(rest);
        }
        f32x16_t& low = P::step == 1.f ? s[nt] : rest;
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          s[nt] = mfma32<T>(hi[hf], qf[ks + hf * (C::KS / 2)], s[nt]);
          low = mfma32<T>(mid[hf], qf[ks + hf * (C::KS / 2)], low);
          low = mfma32<T>(lo[hf], qf[ks + hf * (C::KS / 2)], low);
        }
        if (P::step != 1.f && ks + 1 == C::KS / 2)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[nt][i] = __builtin_fmaf(rest[i], P::step, s[nt][i]);
        __builtin_amdgcn_sched_barrier(0);
      }
      // ---- softmax over the block's normal keys, the landmark's score as it is (last slot: last tile, register 15, h = 1)
      const float t_lm = pair_hi(s[C::NT - 1][15]) * c2;
      if (PADDED) {
        int first = nreal - 1 - 4 * h;                  // slots from here on hold no normal key
        asm volatile("" : "+v"(first));                 // formed here: kept, the masks fill the scalar registers
#pragma unroll
        for (int nt = 0; nt < C::NT; ++nt)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (32 * nt + 8 * (i >> 2) + (i & 3) >= first) s[nt][i] = -INFINITY;
      }
      if (h == 1) s[C::NT - 1][15] = -INFINITY;         // the landmark
      float mx = -INFINITY;
#pragma unroll
      for (int nt = 0; nt < C::NT; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[nt][i]);
      const float m2 = pair_max(mx) * c2;
      float den = 0.f;
#pragma unroll
      for (int nt = 0; nt < C::NT; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[nt][i] = fast_exp2(__builtin_fmaf(s[nt][i], c2, -m2));
          den += s[nt][i];
        }
      const float f = 1.0f / pair_sum(den);
      // ---- O^T = V^T W
      f32x16_t acc[C::DC];
#pragma unroll
      for (int dc = 0; dc < C::DC; ++dc) zero16(acc[dc]);
#pragma unroll
      for (int nt = 0; nt < C::NT; ++nt)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          u32x4_t wf;
#pragma unroll
          for (int i = 0; i < 4; ++i) wf[i] = pack2<T>(s[nt][8 * j + 2 * i] * f, s[nt][8 * j + 2 * i + 1] * f);
#pragma unroll
          for (int dc = 0; dc < C::DC; ++dc) acc[dc] = mfma32<T>(load_tr_frag<D>(smem + ktile + C::TILE, 32 * nt, j, dc, lane), wf, acc[dc]);
        }
      if (ql < ng) {
        const int64_t at = ((int64_t)bh * t_rows + t) * k + r;
        if (h == 0) p.part_score[at] = t_lm;
        float* dst = p.part + at * D + 4 * h;
#pragma unroll
        for (int dc = 0; dc < C::DC; ++dc)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            *(float4*)(dst + 32 * dc + 8 * i) = make_float4(acc[dc][4 * i], acc[dc][4 * i + 1], acc[dc][4 * i + 2], acc[dc][4 * i + 3]);
      }
    }
  }
}

// A row's picks and its local window: D / 4 lanes a row.
template <class T, int D>
__global__ __launch_bounds__(256) void lmk_gather_combine_kernel(RetrParams p, int t_first, int t_rows) {
  constexpr int LPR = D / 4;
  const uint32_t row = blockIdx.x * (256 / LPR) + threadIdx.x / LPR;   // 32-bit as every launch's threads are
  const int j = threadIdx.x % LPR, k = p.k;
  const int bh = (int)(row / (uint32_t)t_rows), t = t_first + (int)(row - (uint32_t)bh * t_rows);
  if (bh >= p.B * p.H) return;
  const int b = (int)((uint32_t)bh / (uint32_t)p.H), hh = bh - b * p.H;
  const float* sc = p.part_score + (int64_t)row * k;
  const float* part = p.part + (int64_t)row * k * D + 4 * j;
  const int64_t srow = (int64_t)bh * p.stat_stride + t;
  const float Ml = p.M_loc[srow] * kLog2e, Ll = p.L_loc[srow];
  const u32x2_t ol = *(const u32x2_t*)((const char*)p.o_loc + 2 * (b * p.ols_b + hh * p.ols_h + (int64_t)t * p.ols_r) + 8 * j);
  float M = Ml, l = 0.f, a[4] = {0.f, 0.f, 0.f, 0.f};
  for (int js = 0; js < k; ++js) M = fmaxf(M, sc[js]);
  constexpr int U = 4;                                  // loads in flight
  for (int j0 = 0; j0 < k; j0 += U) {
    float4 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = *(const float4*)(part + min(j0 + u, k - 1) * D);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (j0 + u >= k) break;
      const float w = fast_exp2(sc[j0 + u] - M);
      l += w;
      a[0] = __builtin_fmaf(x[u].x, w, a[0]);
      a[1] = __builtin_fmaf(x[u].y, w, a[1]);
      a[2] = __builtin_fmaf(x[u].z, w, a[2]);
      a[3] = __builtin_fmaf(x[u].w, w, a[3]);
    }
  }
  const float wl = fast_exp2(Ml - M) * Ll, inv = 1.0f / (l + wl);
  const u32x2_t o = {pack2<T>(__builtin_fmaf(unpack_lo<T>(ol[0]), wl, a[0]) * inv, __builtin_fmaf(unpack_hi<T>(ol[0]), wl, a[1]) * inv),
                     pack2<T>(__builtin_fmaf(unpack_lo<T>(ol[1]), wl, a[2]) * inv, __builtin_fmaf(unpack_hi<T>(ol[1]), wl, a[3]) * inv)};
  *(u32x2_t*)((char*)p.out + 2 * (b * p.outs_b + hh * p.outs_h + (int64_t)t * p.outs_r) + 8 * j) = o;
}

template <class T, int D, int BS, bool PADDED>
static int launch_blocks_t(const RetrParams& p, int rows, hipStream_t stream) {
  using C = GatherBlocksCfg<D, BS>;
  auto kern = lmk_gather_blocks_kernel<T, D, BS, PADDED>;
  static std::atomic<uint64_t> lds_ok{0};
  if (int rc = allow_dynamic_lds(kern, 2 * C::TILE * C::MAX_OWN + C::LIST_BYTES, lds_ok)) return rc;
  // Blocks per workgroup: its search of the picks and its first loads serve them all, and its waves even them out, as long
  // as every compute unit has two workgroups (256 queries of 32 heads of 128, top 4: 64 blocks of 32 take 63.4 us a step with one
  // block, 59.9 with two, 58.1 with four, 128 blocks of 64 118.9 and 107.9; 512 queries of 12 heads of 64, 128 blocks of 64: 47.3,
  // 45.1 and 48.7)
  int own = C::MAX_OWN;
  while (own > 1 && (int64_t)p.B * p.H * ((p.num_mems + own - 1) / own) < 2 * cu_count()) own >>= 1;
  for (int t = 0; t < p.T; t += rows) {                 // as many rows as the workspace holds the picks of
    const int n = std::min(rows, p.T - t);
    hipLaunchKernelGGL(kern, dim3((unsigned)(p.B * p.H), (unsigned)((p.num_mems + own - 1) / own)), dim3(256),
                       2 * C::TILE * own + C::LIST_BYTES, stream, p, t, n, own);
    if (int rc = (int)hipGetLastError()) return rc;
    constexpr int RPW = 256 / (D / 4);
    const int64_t all = (int64_t)p.B * p.H * n;
    hipLaunchKernelGGL((lmk_gather_combine_kernel<T, D>), dim3((unsigned)((all + RPW - 1) / RPW)), dim3(256), 0, stream, p, t, n);
    if (int rc = (int)hipGetLastError()) return rc;
  }
  return 0;
}

template <class T, int D>
static int launch_blocks_d(const RetrParams& p, int BS, int rows, hipStream_t stream) {
  if (p.block > BS || p.block < 2) return LMK_ERR_UNSUPPORTED;
  if (p.block == BS) {
    if (BS == 32) return launch_blocks_t<T, D, 32, false>(p, rows, stream);
    if (BS == 64) return launch_blocks_t<T, D, 64, false>(p, rows, stream);
    if (BS == 128) return launch_blocks_t<T, D, 128, false>(p, rows, stream);
  } else {
    if (BS == 64) return launch_blocks_t<T, D, 64, true>(p, rows, stream);
    if (BS == 128) return launch_blocks_t<T, D, 128, true>(p, rows, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

int launch_gather_blocks(const RetrParams& p, int D, int BS, int rows, int dtype, hipStream_t stream) {
  if (dtype == LMK_DTYPE_BF16) {
    if (D == 128) return launch_blocks_d<bf16_t, 128>(p, BS, rows, stream);
    if (D == 64) return launch_blocks_d<bf16_t, 64>(p, BS, rows, stream);
  } else if (dtype == LMK_DTYPE_F16) {
    if (D == 128) return launch_blocks_d<f16_t, 128>(p, BS, rows, stream);
    if (D == 64) return launch_blocks_d<f16_t, 64>(p, BS, rows, stream);
  }
  return LMK_ERR_UNSUPPORTED;
}

}  // namespace lmk
