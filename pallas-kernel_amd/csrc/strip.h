// Shared pieces of the strip-specialised sweeps (gla_strip.hip, gla_strip_s.hip).
#pragma once
#include "tops_common.h"

namespace tops {

// The LDS planes are row-major, KP channels per row, without padding.  The 16-byte piece c of
// row r lies at piece c ^ swz(r) of that row, so that the three ways a plane is used spread over
// the banks: staging writes (8 or 16 bytes of adjacent pieces of a few rows), row reads
// (ds_read_b128, one piece of 16 rows) and transposed reads (ds_read_b64_tr_b16, four rows at
// four adjacent pieces).
template <int KP>
__device__ __forceinline__ constexpr int swz(int r) {
  const int b0 = r & 1, b1 = (r >> 1) & 1, b2 = (r >> 2) & 1, b3 = (r >> 3) & 1;
  return KP == 128 ? (((b1 ^ b3) << 3) | (b0 << 2) | (b3 << 1) | b2)
                   : (KP == 64 ? ((b1 << 2) | (b3 << 1) | b2) : ((b3 << 1) | b2));
}

__device__ __forceinline__ bf16x8 lds8(const uint16_t* p) {
  return __builtin_bit_cast(bf16x8, *(const uint4*)p);
}
// transposed read: this lane's address of a 4-row block (tr_read8's lane layout), two blocks
__device__ __forceinline__ bf16x8 tr2(const uint16_t* pa, const uint16_t* pb) {
  typedef __attribute__((address_space(3))) v4i16 lds_v4;
  const v4i16 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)pa);
  const v4i16 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)pb);
  const uint2 ua = __builtin_bit_cast(uint2, a), ub = __builtin_bit_cast(uint2, b);
  return __builtin_bit_cast(bf16x8, make_uint4(ua.x, ua.y, ub.x, ub.y));
}

// Factor of an fp16 checkpoint tile from the wave maxima of |S| (fp32 bits): 2^(14 - e), e the
// largest exponent.
__device__ __forceinline__ float ckpt_tile_scale(const uint32_t* smx) {
  const uint32_t m = max(max(smx[0], smx[1]), max(smx[2], smx[3]));
  int ex = (int)((m >> 23) & 0xffu) - 127;
  ex = ex < -100 ? -100 : ex;
  return __uint_as_float((uint32_t)(141 - ex) << 23);
}

}  // namespace tops
