// Rotated landmark keys and their norms (llama/llama_mem.py:357-366): the body shared by the kernel that does
// only this and by the one that runs it beside the forward over the local window.
#pragma once

#include "lmk_common.hpp"
#include "lmk_launch.hpp"

namespace lmk {

// Chunk j (8 head dims) of the landmark key of block m, what its rotation takes: the chunk, the one D / 2 away, the table rows.
struct LandmarkChunk {
  u32x4_t x, other, c, s;
};
template <int D>
__device__ __forceinline__ LandmarkChunk load_landmark_chunk(const RetrParams& p, int b, int hh, int m, int j) {
  int age = m - p.ring_start;                              // ring caches: slot ring_start holds the oldest block
  age += age < 0 ? p.num_mems : 0;
  const int slot = (age < p.num_mems - p.k) ? 0 : age - (p.num_mems - p.k) + 1;
  const int64_t pos = (int64_t)slot * p.block + (p.block - 1) + p.prefix_len;
  // the landmark is the last row of block m of the cache -- or row m of an array that holds the landmark keys alone
  const int64_t lm_row = p.lm_dense ? (int64_t)m : (int64_t)m * p.block + p.block - 1;
  const char* src = (const char*)p.kcache + 2 * (b * p.kcs_b + hh * p.kcs_h + lm_row * p.kcs_r);
  return {*(const u32x4_t*)(src + 16 * j), *(const u32x4_t*)(src + 16 * (j ^ (D / 16))),
          *(const u32x4_t*)((const char*)p.cos + 2 * (pos * p.cs_r) + 16 * j),
          *(const u32x4_t*)((const char*)p.sin + 2 * (pos * p.cs_r) + 16 * j)};
}

// One workgroup of NTHR threads rotates R * NTHR / (D / 8) landmark keys, R per thread with the loads of all R in
// flight together; `wg` is its index among the workgroups that do so (the kernel of lmk_retrieval.hip runs nothing
// else; the one of lmk_fwd32.hip runs them beside a forward, whose registers and LDS leave room for few workgroups
// per compute unit, hence R > 1 there).
template <class T, int D, int NTHR, int R = 1>
__device__ __forceinline__ void landmark_keys_body(const RetrParams& p, int wg) {
  constexpr int LPR = D / 8;
  constexpr int RPW = NTHR / LPR;
  const int tid = threadIdx.x, j = tid % LPR;
  // indices of threads and of what they work on stay below 2^32, the launch's own limit: a 64-bit division is 100 instructions
  const uint32_t total = (uint32_t)(p.B * p.H) * (uint32_t)p.num_mems;
  uint32_t row[R];
  int bh[R], m[R];
  LandmarkChunk k[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    row[i] = ((uint32_t)wg * R + i) * RPW + tid / LPR;     // (bh, m)
    const uint32_t rr = min(row[i], total - 1);            // past the end: a re-read that is never stored
    bh[i] = (int)(rr / (uint32_t)p.num_mems);
    m[i] = (int)(rr - (uint32_t)bh[i] * p.num_mems);
    const int b = (int)((uint32_t)bh[i] / (uint32_t)p.H);
    k[i] = load_landmark_chunk<D>(p, b, bh[i] - b * p.H, m[i], j);
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    float r[8];
    rotate_chunk<T>(k[i].x, k[i].other, k[i].c, k[i].s, j >= LPR / 2, r);
    const bool ok = row[i] < total;
    u32x4_t o = {pack2<T>(r[0], r[1]), pack2<T>(r[2], r[3]), pack2<T>(r[4], r[5]), pack2<T>(r[6], r[7])};
    if (ok) *(u32x4_t*)((char*)p.lk_rot + bh[i] * lk_tiles(p.num_mems) * lk_tile_bytes(D) + lk_key_offset(m[i], D) + 512 * j) = o;
    float nrm = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) nrm += r[e] * r[e];
#pragma unroll
    for (int msk = LPR / 2; msk >= 1; msk >>= 1) nrm += __shfl_xor(nrm, msk, 64);
    if (ok && j == 0) p.lk_norm[row[i]] = sqrtf(nrm) * 1.000001f;
  }
}

}  // namespace lmk
