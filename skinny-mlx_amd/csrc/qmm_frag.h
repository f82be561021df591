// The packed W4 g64 block and the MFMA operands built from it, shared by the 1..16-token kernels
// (qmm.hip) and the many-row kernel (qmm_rows.hip). Internal to libskinny_hip.so.
#pragma once

#include "common.h"

namespace {

// Packed fragment block of (tile t, group pair p): 288 u32 at word (t*GP + p)*288.
//   words [0, 256):   lane l, word 2j + h at 4l + 2j + h — row 16t + l%16, columns
//                     64(2p+j) + 32h + 8(l/16) + 0..7 (nibble order of mlx_to_frag_word);
//   words [256, 288): row r at 256 + 2r: scales of groups 2p, 2p+1 (low, high half),
//                     then biases of the same two groups.
constexpr int kBlockWords = 288;
constexpr int kBlockBytes = kBlockWords * 4;
constexpr int kSbOffsetBytes = 1024;

// Eight codes of one fragment word -> the B operand: bf16 pairs (128 + e_2v, 128 + e_2v+1),
// built by v_perm_b32 from one code per byte and a 0x43 byte (bf16 128.0 = 0x4300, and
// 0x4300 | q = 128 + q exactly for q < 128).
__device__ __forceinline__ bf16x8_t unpack_nibbles(uint32_t w) {
  const uint32_t lo = w & 0x0F0F0F0Fu;         // e0 e1 e2 e3
  const uint32_t hi = (w >> 4) & 0x0F0F0F0Fu;  // e4 e5 e6 e7
  u32x4_t p;
  p.x = __builtin_amdgcn_perm(0x43434343u, lo, 0x04010400u);
  p.y = __builtin_amdgcn_perm(0x43434343u, lo, 0x04030402u);
  p.z = __builtin_amdgcn_perm(0x43434343u, hi, 0x04010400u);
  p.w = __builtin_amdgcn_perm(0x43434343u, hi, 0x04030402u);
  return __builtin_bit_cast(bf16x8_t, p);
}

// Weight side of one group pair for RF row tiles.
template <int RF>
struct WStage {
  u32x4_t w[RF];   // fragment words: (g0 h0, g0 h1, g1 h0, g1 h1)
  u32x2_t sb[RF];  // (scales of g0|g1, biases of g0|g1) for the lane's row
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  // gfx9 raw buffer: stride 0, byte-granular range check, word 3 = 0x00020000
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

template <int RF>
__device__ __forceinline__ void load_w(WStage<RF>& ws, __amdgpu_buffer_rsrc_t rw, uint32_t woff, uint32_t sboff,
                                       int gp, int GP) {
#pragma unroll
  for (int r = 0; r < RF; ++r) {
    const int blk = (r * GP + gp) * kBlockBytes;
    ws.w[r] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, woff, blk, 0));
    ws.sb[r] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rw, sboff, blk, 0));
  }
}

__device__ __forceinline__ bf16x8_t ones_operand() {
  return __builtin_bit_cast(bf16x8_t, u32x4_t{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
}

}  // namespace
