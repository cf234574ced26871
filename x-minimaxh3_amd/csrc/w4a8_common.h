// Shared pieces of the group-scaled W4A8 kernels (w4a8.hip, w4a8_g128.hip).
#pragma once

#include "mxq_common.h"

namespace mxq {

constexpr int kW4BK = 128;

struct W4Args {
  const int8_t* a;
  const float* xs;
  const uint8_t* w;       // [N, K/2]
  const uint16_t* gs;     // [K/G, N] fp16
  const void* bias;
  void* d;
  int64_t M, N, K, ldd;
  int group_tiles;        // K-stages per group (G / 128)
  int tiles_m, tiles_n;
};

// 4 packed bytes (8 codes, even k low nibble) -> 8 int8 holding 16 (c - 8), natural k order.
MXQ_DEVICE void unpack8(uint32_t w, uint32_t& o0, uint32_t& o1) {
  const uint32_t x = w ^ 0x88888888u;
  const uint32_t xs = x << 4;
  o0 = __builtin_amdgcn_perm(x, xs, 0x05010400u) & 0xF0F0F0F0u;
  o1 = __builtin_amdgcn_perm(x, xs, 0x07030602u) & 0xF0F0F0F0u;
}

// The prepared layout (mxq_w4a8_prepare_grouped): each 32-bit word of a weight row still holds
// the 8 codes of k = 8w .. 8w + 7, but byte j holds (c[8w + j] ^ 8) in its low nibble and
// (c[8w + 4 + j] ^ 8) in its high nibble -- the offset-8 code as a 4-bit two's complement value
// c - 8. Unpacking to 16 (c - 8) per int8 in natural k order is then a shift and two masks.
MXQ_DEVICE void unpack8_prepared(uint32_t w, uint32_t& o0, uint32_t& o1) {
  o0 = (w << 4) & 0xF0F0F0F0u;
  o1 = w & 0xF0F0F0F0u;
}

// ---- the reference's grouped format: 16 levels per scale ----
// A weight's int8 value depends only on its group's scale and its code, so a group's 16 values are
// formed once, as 16 bytes in four words (level c in byte c % 4 of word c / 4), and its weights are byte
// selections from them: 15 VALU instructions per 8 weights, where forming each value from the
// code's float took about 12 per weight.

MXQ_DEVICE float e4m3fn_to_f32(uint32_t b) {
  const uint32_t s = b & 0x80u, e = (b >> 3) & 0xFu, m = b & 7u;
  float v;
  if ((b & 0x7Fu) == 0x7Fu) return __uint_as_float(0x7FC00000u);
  if (e == 0)
    v = (float)m * 0.001953125f;  // m / 8 * 2^-6
  else
    v = __uint_as_float(((e + 120u) << 23) | (m << 20));  // (1 + m/8) 2^(e-7)
  return s ? -v : v;
}

// The codebook's 16 floats (c - 8 without one); finite: none of them is an infinity or a NaN.
struct Levels {
  float v[16];
  bool finite;
};

MXQ_DEVICE Levels load_levels(const float* codebook) {
  Levels l;
  l.finite = true;
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    l.v[c] = codebook ? codebook[c] : (float)(c - 8);
    l.finite = l.finite && (__float_as_uint(l.v[c]) & 0x7F800000u) != 0x7F800000u;
  }
  return l;
}

// clamp(rne(v[c] * s), -127, 127) of the 16 levels (0 for a NaN product). Adding 1.5 * 2^23 to the clamped
// product rounds it to nearest even and leaves the integer in the low byte.
MXQ_DEVICE v4u level_values(const Levels& l, float s) {
  uint32_t q[16];
#pragma unroll
  for (int c = 0; c < 16; ++c)
    q[c] = __float_as_uint(__builtin_amdgcn_fmed3f(l.v[c] * s, -127.0f, 127.0f) + 12582912.0f);
  const bool finite = l.finite && (__float_as_uint(s) & 0x7F800000u) != 0x7F800000u;
  if (__builtin_amdgcn_ballot_w64(!finite)) {
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const float p = l.v[c] * s;
      if (p != p) q[c] = 0;
    }
  }
  v4u t;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t lo = __builtin_amdgcn_perm(q[4 * j + 1], q[4 * j], 0x0C0C0400u);
    const uint32_t hi = __builtin_amdgcn_perm(q[4 * j + 3], q[4 * j + 2], 0x04000C0Cu);
    t[j] = lo | hi;
  }
  return t;
}

// Four codes (bits 0-2 of each byte of c7, bit 3 of each byte of c8) to their bytes of t.
MXQ_DEVICE uint32_t select_levels(uint32_t c7, uint32_t c8, v4u t) {
  const uint32_t lo = __builtin_amdgcn_perm(t[1], t[0], c7);
  const uint32_t hi = __builtin_amdgcn_perm(t[3], t[2], c7);
  const uint32_t mask = __builtin_amdgcn_perm(0u, 0x0000FF00u, c8);  // selector 8: the sign of byte 1, i.e. 0xFF
  return (hi & mask) | (lo & ~mask);
}

// 4 packed bytes (8 codes, even k low nibble) -> 8 int8 in k order.
MXQ_DEVICE void decode8(uint32_t w, v4u t, uint32_t& o0, uint32_t& o1) {
  const uint32_t x = w >> 4;
  const uint32_t even = select_levels(w & 0x07070707u, w & 0x08080808u, t);
  const uint32_t odd = select_levels(x & 0x07070707u, x & 0x08080808u, t);
  o0 = __builtin_amdgcn_perm(odd, even, 0x05010400u);
  o1 = __builtin_amdgcn_perm(odd, even, 0x07030602u);
}

// The few-row GEMM on weights decoded in registers (w4a8_ref.hip) and its plan: whether it takes the problem, given
// room for its partial sums.
struct W4RefArgs {
  const int8_t* a;      // [M, K] int8
  const uint8_t* w;     // [N, K / 2]
  const void* s_rel;    // [N, K / G]
  const float* codebook;
  int64_t M, N, K;
  int e4m3, group;
};
struct W4RefPlan {
  int rows;        // 32-row blocks per tile; 0: not this kernel's problem
  int tiles_m, tiles_n, splits, stages;  // stages of 256 K per slice
  int64_t ldp, bytes;                    // int32 per row of the partial sums, bytes of them all
};
W4RefPlan plan_w4_ref(const W4RefArgs& p, int64_t room);
int launch_w4_ref(const W4RefArgs& p, const W4RefPlan& plan, int32_t* part, hipStream_t st);

// The INT8 GEMMs' limits (gemm_i8.hip): the largest K whose int32 sums cannot wrap (128 * 128 * K < 2^31), and the
// check of a tile-queue workspace (NULL or 256-byte aligned, no negative size).
constexpr int64_t kGemmMaxK = 131056;
int check_gemm_workspace(const void* workspace, int64_t workspace_bytes);

// Sums `splits` slices of partial results [M, ldp] and applies the dequant epilogue (gemm_i8.hip).
int launch_split_dequant(const int32_t* part, int splits, int64_t ldp, const float* xs, const float* ws, const void* bias,
                         void* d, int64_t M, int64_t N, int64_t ldd, int out_dtype, hipStream_t st);

// The group-128 pipelined kernel (w4a8_g128.hip): needs group size 128, N % 8 == 0 and 16-byte
// aligned scale rows; `prepared` selects the weight layout. Returns MXQ_ERR_UNSUPPORTED without
// launching (and without setting an error) when the operands are too large for its 32-bit
// offsets.
int launch_w4_g128(W4Args p, int out_dtype, bool prepared, hipStream_t st);

}  // namespace mxq
