// Pieces shared by the trellis kernels: the codebook, the 128-group Hadamard butterfly held in
// registers, and four-element activation loads.
#pragma once

#include "ttq_device.h"
#include "ttq_internal.h"

namespace ttq {

typedef __attribute__((ext_vector_type(2))) _Float16 half2_t;

// The codebook: a pure function of the 16-bit trellis state (bits 16..31 of `state` are ignored).
// The 32-bit multiply is not what limits the decode here: splitting it into two 16-bit
// multiply-adds was measured slower.
template <int CB>
struct Codebook {
  static constexpr uint32_t kMul = (CB == 0) ? 89226354u : 0xCBAC1FEDu;
  __device__ __forceinline__ void init() {}
  __device__ __forceinline__ _Float16 code(uint32_t state) const {
    uint32_t u = (state & 0xFFFFu) * kMul;
    if (CB == 0) u += 64248484u;
    u = (u & 0x8FFF8FFFu) ^ 0x3B603B60u;
    half2_t h;
    __builtin_memcpy(&h, &u, 4);
    return h[0] + h[1];  // fp16 add, round-to-nearest-even
  }
};

// Unnormalized FWHT of a 128-group held as 4 consecutive values in each of 32 consecutive lanes
// (value index = 4*lane + i): stages 1 and 2 inside the lane, stages 4..64 against the lane
// 1, 2, 4, 8, 16 away.  Same stage order and operand order as the textbook loop
// (lower index gets a+b, upper a-b), so the results do not depend on how it is laid out.
template <int D, int N>
__device__ __forceinline__ void fwht_lane_stage(float (&v)[N], int lane) {
  const float sign = (lane & D) != 0 ? -1.f : 1.f;      // (the sum and the difference by one instruction, rounded once as they are)
#pragma unroll
  for (int i = 0; i < N; i++) v[i] = fmaf_(sign, v[i], lane_xor<D>(v[i], lane));
}
__device__ __forceinline__ void fwht128_quad(float (&v)[4], int lane) {
  float t;
  t = v[0]; v[0] = t + v[1]; v[1] = t - v[1];
  t = v[2]; v[2] = t + v[3]; v[3] = t - v[3];
  t = v[0]; v[0] = t + v[2]; v[2] = t - v[2];
  t = v[1]; v[1] = t + v[3]; v[3] = t - v[3];
  fwht_lane_stage<1>(v, lane);
  fwht_lane_stage<2>(v, lane);
  fwht_lane_stage<4>(v, lane);
  fwht_lane_stage<8>(v, lane);
  fwht_lane_stage<16>(v, lane);
}

// Four consecutive activations (a multiple of four elements from the row start) as floats.
__device__ __forceinline__ void load_x4(const float* p, float (&v)[4]) {
  const float4 t = *reinterpret_cast<const float4*>(__builtin_assume_aligned(p, 16));
  v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
}
__device__ __forceinline__ void load_x4(const f16_tag* p, float (&v)[4]) {
  uint2 r;
  __builtin_memcpy(&r, __builtin_assume_aligned(p, 8), 8);
  v[0] = f16_bits_to_f32((uint16_t)r.x); v[1] = f16_bits_to_f32((uint16_t)(r.x >> 16));
  v[2] = f16_bits_to_f32((uint16_t)r.y); v[3] = f16_bits_to_f32((uint16_t)(r.y >> 16));
}
__device__ __forceinline__ void load_x4(const bf16_tag* p, float (&v)[4]) {
  uint2 r;
  __builtin_memcpy(&r, __builtin_assume_aligned(p, 8), 8);
  v[0] = bf16_bits_to_f32((uint16_t)r.x); v[1] = bf16_bits_to_f32((uint16_t)(r.x >> 16));
  v[2] = bf16_bits_to_f32((uint16_t)r.y); v[3] = bf16_bits_to_f32((uint16_t)(r.y >> 16));
}

// ------------------------------------------------------------------------------------------------
// Shared by the matrix-core trellis kernels (decode GEMV and prefill GEMM): workgroup shape, the
// decode of a lane's four weights of a tile into an A fragment, and the LDS layout of a pass of tiles.
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

// Codebook value of a 16-bit trellis state, written as an fp16 number into half HALF of `dst` (the other half is kept
// when HALF is 1): the sum of the two fp16 numbers that the masked hash holds, added by one instruction that picks both
// halves of its operand itself.
template <int CB, int HALF, bool LAST = false>
__device__ __forceinline__ void xm_code(uint32_t state, uint32_t& dst) {
  uint32_t u = state * Codebook<CB>::kMul;
  if constexpr (CB == 0) u += 64248484u;
  u = (u & 0x8FFF8FFFu) ^ 0x3B603B60u;
  if constexpr (HALF == 0)
    asm("v_add_f16_sdwa %0, %1, %1 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1" : "=v"(dst) : "v"(u));
  else if constexpr (!LAST)
    asm("v_add_f16_sdwa %0, %1, %1 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 src1_sel:WORD_1"
        : "+v"(dst) : "v"(u));
  else
    // (the wait states keep the matrix-core read that follows clear of the partial register write, which
    // the compiler cannot see inside the statement)
    asm("v_add_f16_sdwa %0, %1, %1 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 src1_sel:WORD_1\n\ts_nop 3"
        : "+v"(dst) : "v"(u));
}

// Four consecutive outputs (idx a multiple of four) in the output buffer's element type.
__device__ __forceinline__ void xm_store4(void* y, int y_dtype, int64_t idx, const float (&o)[4]) {
  if (y_dtype == kF32) {
    *reinterpret_cast<float4*>(static_cast<float*>(y) + idx) = make_float4(o[0], o[1], o[2], o[3]);
  } else {
    uint2 v;
    if (y_dtype == kF16) {
      v.x = (uint32_t)f32_to_f16_bits(o[0]) | ((uint32_t)f32_to_f16_bits(o[1]) << 16);
      v.y = (uint32_t)f32_to_f16_bits(o[2]) | ((uint32_t)f32_to_f16_bits(o[3]) << 16);
    } else {
      v.x = pack_bf16x2(o[0], o[1]);
      v.y = pack_bf16x2(o[2], o[3]);
    }
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(y) + idx) = v;
  }
}

// Four consecutive activations as loaded (converted when they are used, so that the load can stay in flight).
template <typename XT> struct XmRaw;
template <> struct XmRaw<float> {
  float4 r;
  __device__ __forceinline__ void load(const float* p) { r = *reinterpret_cast<const float4*>(__builtin_assume_aligned(p, 16)); }
  __device__ __forceinline__ void get(float (&v)[4]) const { v[0] = r.x; v[1] = r.y; v[2] = r.z; v[3] = r.w; }
};
template <> struct XmRaw<f16_tag> {
  uint2 r;
  __device__ __forceinline__ void load(const f16_tag* p) { __builtin_memcpy(&r, __builtin_assume_aligned(p, 8), 8); }
  __device__ __forceinline__ void get(float (&v)[4]) const {
    v[0] = f16_bits_to_f32((uint16_t)r.x); v[1] = f16_bits_to_f32((uint16_t)(r.x >> 16));
    v[2] = f16_bits_to_f32((uint16_t)r.y); v[3] = f16_bits_to_f32((uint16_t)(r.y >> 16));
  }
};
template <> struct XmRaw<bf16_tag> {
  uint2 r;
  __device__ __forceinline__ void load(const bf16_tag* p) { __builtin_memcpy(&r, __builtin_assume_aligned(p, 8), 8); }
  __device__ __forceinline__ void get(float (&v)[4]) const {
    v[0] = bf16_bits_to_f32((uint16_t)r.x); v[1] = bf16_bits_to_f32((uint16_t)(r.x >> 16));
    v[2] = bf16_bits_to_f32((uint16_t)r.y); v[3] = bf16_bits_to_f32((uint16_t)(r.y >> 16));
  }
};

// Where a lane's windows lie inside a packed tile, as it is in memory: a cyclic string of 16-bit words, most significant bit
// first.  The four bytes that a window starts in lie in two consecutive dwords; one byte permutation brings them into
// string order (byte s of the string is byte s ^ 1 in memory), and a weight's state is a bit field of the result: the
// first starts 0..7 bits below the top, which depends on the lane only where the number of bits per weight is odd.
// (Two funnel-shift operands with their halves swapped first take two more instructions per window.)  With five bits, four
// weights are 31 bits, more than what is left of 32 from the byte they start in, but not from the bit: there one funnel shift, and
// one window, against two permutations, two windows and twice the reads: 4096 x 4096 one row 10.2 -> 9.7 us, 512 rows 50.7 -> 46.6.
template <int BITS>
struct XmLane {
  static constexpr bool kFunnel = BITS == 5;
  static constexpr int kWin = BITS <= 5 ? 1 : 2;     // windows per four weights
  uint32_t at[kWin][2];                              // byte offsets of the two dwords in the tile
  uint32_t sel[kWin];                                // byte selector (funnel: shift)
  uint32_t down;                                     // 4 if the lane's windows start four bits lower, else 0
  __device__ __forceinline__ void init(int lane) {
    const int j = lane & 15, q = lane >> 4;
    down = (BITS & 1) ? 4u * (q & 1) : 0u;
    if constexpr (kFunnel) {
      // (a window that starts on a dword boundary takes the pair one dword earlier and shifts by nothing)
      const int bit = (16 * j + 4 * q) * BITS, o = bit & 31, d = (bit >> 5) - (o == 0);
      at[0][0] = 4u * ((d + 8 * BITS) % (8 * BITS));
      at[0][1] = 4u * ((d + 1) % (8 * BITS));
      sel[0] = (32 - o) & 31;
      return;
    }
#pragma unroll
    for (int w = 0; w < kWin; w++) {
      const int bit = (16 * j + 4 * q + 2 * w) * BITS;
      const int b = bit >> 3, d = b >> 2;
      at[w][0] = 4u * d;
      at[w][1] = 4u * ((d + 1) % (8 * BITS));
      sel[w] = 0;
#pragma unroll
      for (int i = 0; i < 4; i++) sel[w] |= (uint32_t)((b + 3 - i - 4 * d) ^ 1) << (8 * i);
    }
  }
  // The four weights as half of an A fragment (two registers of two fp16 each).  (The bits that a window of two weights
  // starts below its byte: 2 w BITS + 4 q BITS modulo 8; the first part is a constant, the second is `down`, and
  // where the sum passes 8 it starts in the byte after.)
  template <int CB, int W, int E, int HALF, bool LAST = false>
  __device__ __forceinline__ void code(uint32_t w, uint32_t& dst) const {
    constexpr int kTop = (2 * W * BITS) & 7;
    if constexpr ((BITS & 1) && !kFunnel) xm_code<CB, HALF, LAST>(__builtin_amdgcn_ubfe(w, field(W, E), 16), dst);
    else xm_code<CB, HALF, LAST>(__builtin_amdgcn_ubfe(w, 16 - kTop - E * BITS, 16), dst);
  }
  __device__ __forceinline__ uint32_t field(int w, int e) const { return 16u - (((uint32_t)(2 * w * BITS) + down) & 7u) - (uint32_t)(e * BITS); }
  template <int CB>
  __device__ __forceinline__ void decode(const uint32_t (&c)[kWin][2], uint32_t (&r)[2]) const {
    uint32_t w0;
    if constexpr (kFunnel)
      w0 = __builtin_amdgcn_alignbit(__builtin_amdgcn_alignbit(c[0][0], c[0][0], 16), __builtin_amdgcn_alignbit(c[0][1], c[0][1], 16), sel[0]);
    else
      w0 = __builtin_amdgcn_perm(c[0][1], c[0][0], sel[0]);
    if constexpr (kWin == 1) {
      code<CB, 0, 0, 0>(w0, r[0]);
      code<CB, 0, 1, 1>(w0, r[0]);
      code<CB, 0, 2, 0>(w0, r[1]);
      code<CB, 0, 3, 1, true>(w0, r[1]);
    } else {
      const uint32_t w1 = __builtin_amdgcn_perm(c[kWin - 1][1], c[kWin - 1][0], sel[kWin - 1]);
      code<CB, 0, 0, 0>(w0, r[0]);
      code<CB, 0, 1, 1>(w0, r[0]);
      code<CB, 1, 0, 0>(w1, r[1]);
      code<CB, 1, 1, 1, true>(w1, r[1]);
    }
  }
};

}  // namespace ttq
