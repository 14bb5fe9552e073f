// What the kernels whose waves split the keys of 64 query rows have in common (lmk_fwd_split.hip, lmk_bwd_dq_split.hip).
#pragma once

#include <algorithm>

#include "lmk_common.hpp"
#include "lmk_launch.hpp"

namespace lmk {

// How the tensors' rows make up the kernel's slots: PLAIN: every block has BS tokens in BS slots; TOKENS: blocks of
// n_real tokens, rows = tokens or rows = slots (FwdParams::Lq_real); FACTORS: the same with group dropout factors;
// TABLE: blocks of unequal length, looked up in FwdParams::seg.
enum { PLAIN, TOKENS, FACTORS, TABLE };

// One 1 KB direct global->LDS request of a wave: lane i's 16 bytes land at lds_off + 16*i (lds_off wave-uniform, in M0).
__device__ __forceinline__ void split_dma16(const void* base_uniform, uint32_t voff, uint32_t lds_off) {
  const uint64_t b = (uint64_t)base_uniform;
  const uint64_t base = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32) |
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(voff), "s"(base), "s"(__builtin_amdgcn_readfirstlane(lds_off)) : "memory");
}
// The same with 4 bytes per lane, each from its own address.
__device__ __forceinline__ void split_dma4(const float* src, uint32_t lds_off) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
               :: "v"(src), "s"(__builtin_amdgcn_readfirstlane(lds_off)) : "memory");
}

__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0f70); }   // vmcnt(0)

// The lane id where it is used: kept across a loop, what is derived from it takes registers and may be spilled.
__device__ __forceinline__ int lane_id() {
  int ln;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
  return ln;
}

__device__ __forceinline__ void zero16(f32x16_t& x) {
#pragma unroll
  for (int r = 0; r < 16; ++r) x[r] = 0.f;
}

// A workgroup per head (x), batch (y) and 64 query rows (z, the last rows first): heads vary fastest, so with a multiple of
// 8 heads all of a head's workgroups land on one XCD, and a kernel has nothing to divide.  y and z are 16-bit: what is
// beyond that goes into further launches.
template <class P, class K>
inline int launch_rows64(K kern, const P& p, int threads, int lds_bytes, std::atomic<uint64_t>& lds_ok, hipStream_t stream) {
  constexpr int kMax = 65535;
  if (int rc = allow_dynamic_lds(kern, lds_bytes, lds_ok)) return rc;
  P c = p;
  for (c.b0 = 0; c.b0 < p.B; c.b0 += kMax)
    for (c.qt_top = (p.Lq + 63) / 64 - 1; c.qt_top >= 0; c.qt_top -= kMax)
      hipLaunchKernelGGL(kern, dim3(p.H, std::min(p.B - c.b0, kMax), std::min(c.qt_top + 1, kMax)), dim3(threads), lds_bytes, stream, c);
  return (int)hipGetLastError();
}

}  // namespace lmk
