// Tiles of packed weight blocks in LDS, shared by the kernels that stream them through rings of their wavefronts' own
// (ttq_gemv_tile.hip, ttq_gemm_rows.hip): requests, operand reads and unpacking.
#pragma once

#include <type_traits>

#include "ttq_stream_common.h"

namespace ttq {

// four bytes -> two dwords of 16-bit halves (byte | hi << 8)
__device__ __forceinline__ void spread_bytes(uint32_t u, uint32_t hi, uint32_t& a, uint32_t& b) {
  a = __builtin_amdgcn_perm(hi, u, 0x04010400u);
  b = __builtin_amdgcn_perm(hi, u, 0x04030402u);
}
template <class XT>
__device__ __forceinline__ f32x4_t tile_mfma(const uint4& x, const uint32_t (&w)[4], f32x4_t c) {
  if constexpr (std::is_same<XT, f16_tag>::value) {
    f16x8_t a, b;
    __builtin_memcpy(&a, &x, 16);
    __builtin_memcpy(&b, w, 16);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  } else {
    bf16x8_t a, b;
    __builtin_memcpy(&a, &x, 16);
    __builtin_memcpy(&b, w, 16);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
}

// One request: 64 lanes fetch 16 bytes each from base + off into 1 KiB of LDS.  In assembly, so that the compiler, which
// cannot tell these asynchronous writes from its own LDS accesses, does not wait for every one of them.  STREAM: lines that
// no other request shares leave the caches early.
template <bool STREAM>
__device__ __forceinline__ void tile_request(uint32_t lds, const uint8_t* base, uint32_t off) {
  if constexpr (STREAM)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds), "v"(off), "s"(base) : "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}

// 16 blocks of Q6_K -- { u8 ql[128]; u8 qh[64]; i8 scales[16]; f16 d }, 256 weights, w = d * scale[e / 16] * (q6[e] - 32) --
// of 16 / KQ weight rows by KQ blocks along K.  A block is cut into 14 pieces of 16 bytes, the last one ending with it, from its
// first byte rounded down to a dword; piece c of block n lies at place (c + n) % 14 of the block's slot, which puts the
// blocks of an operand read on different banks.
struct TlQ6K {
  static constexpr int kSub = 16;            // weights per scale
  static constexpr int kChains = 4;          // matrix products per tile, each over four sub-blocks of every block
  static constexpr int kSteps = kSub / 8;
  static constexpr int kChunks = 14;         // 16-byte pieces of a block in LDS
  static constexpr int kSlot = 16 * kChunks * 16;
  static constexpr int kRequests = 4;
  // chain 2h + p: sub-blocks 8h + 4p + g, g = lane / 16
  static __device__ __forceinline__ constexpr int lane_k(int g) { return 16 * g; }
  static __device__ __forceinline__ constexpr int chain_k(int c) { return 64 * c; }
  static __device__ __forceinline__ void sub_of(int sub, int& c, int& g) { c = sub >> 2; g = sub & 3; }

  struct Lane {
    uint32_t src[kRequests], odd2[kRequests];                   // request addresses
    uint32_t over, fix;                                          // bit i: request i is past the row's end / reads the last block
    uint32_t ql[2], qlx[2], qh[2], qhx[2], sc, dd;              // operand addresses in a slot
    uint32_t qh_shift, sc_shift, odd, d_mask, d_fix;
    // rows: of a group; kq_last: the last block of a row's last tile
    template <int KQ> __device__ __forceinline__ void init(int lane, int nsb, int rows, int kq_last, bool odd_total) {
      const int n = lane & 15, g = lane >> 4;
      over = fix = 0;
#pragma unroll
      for (int i = 0; i < kRequests; i++) {
        const int p = min(64 * i + lane, 16 * kChunks - 1);
        const int pb = p / kChunks, pos = p - pb * kChunks, c = (pos + 2 * kChunks - pb) % kChunks;
        const int r = min(pb / KQ, rows - 1), kq = pb % KQ;
        const uint32_t blk = (uint32_t)(r * nsb + kq);
        src[i] = blk * 210u + (c < 13 ? 16u * c : 196u);
        odd2[i] = 2u * (blk & 1u);
        if (kq > kq_last) over |= 1u << i;
        if (odd_total && r == rows - 1 && kq == kq_last && c == 13) fix |= 1u << i;
      }
      auto at = [&](int c) { return (uint32_t)(16 * (n * kChunks + (c + n) % kChunks)); };
#pragma unroll
      for (int h = 0; h < 2; h++) {
        ql[h] = at(4 * h + g);
        qlx[h] = at(4 * h + g + 1);
        qh[h] = at(8 + 2 * h + (g & 1));
        qhx[h] = at(8 + 2 * h + (g & 1) + 1);
      }
      sc = at(12);
      dd = at(13) + 12;
      qh_shift = 2u * (g >> 1);
      sc_shift = 8u * g;
      const int r = min(n / KQ, rows - 1), kq = n % KQ;
      odd = (uint32_t)(r * nsb + kq) & 1u;
      d_mask = kq > kq_last ? 0u : 0xFFFFu;
      d_fix = (odd_total && r == rows - 1 && kq == kq_last) ? 16u : 0u;
    }
  };
  // block: index of the tile's first block in the matrix; tail: a row's last tile; last: the matrix's last tile
  template <bool STREAM>
  static __device__ __forceinline__ void request(const Lane& L, int lane, uint32_t lds, const uint8_t* w, int64_t block, bool tail, bool last) {
    const bool odd = block & 1;
    const uint8_t* base = w + block * 210 - (odd ? 2 : 0);
    uint32_t off[kRequests];
#pragma unroll
    for (int i = 0; i < kRequests; i++) off[i] = L.src[i] + (odd ? L.odd2[i] : 0u - L.odd2[i]);
    if (tail) {
#pragma unroll
      for (int i = 0; i < kRequests; i++) {
        if ((L.over >> i) & 1u) off[i] = 0u;
        if (last && ((L.fix >> i) & 1u)) off[i] -= 2u;
      }
    }
#pragma unroll
    for (int i = 0; i < kRequests; i++)
      if (i < kRequests - 1 || lane < 32) tile_request<STREAM>(lds + 1024 * i, base, off[i]);
  }
  struct Raw { uint32_t ql[2][4], qh[2][4], sc[4], d; };
  static __device__ __forceinline__ void read(Raw& r, const uint8_t* slot, const Lane& L, int64_t block, bool tail, bool last) {
    const uint32_t sh = (((uint32_t)block + L.odd) & 1u) * 16u;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const uint4 a = *reinterpret_cast<const uint4*>(slot + L.ql[h]);
      const uint32_t ax = *reinterpret_cast<const uint32_t*>(slot + L.qlx[h]);
      const uint4 b = *reinterpret_cast<const uint4*>(slot + L.qh[h]);
      const uint32_t bx = *reinterpret_cast<const uint32_t*>(slot + L.qhx[h]);
      r.ql[h][0] = __builtin_amdgcn_alignbit(a.y, a.x, sh);
      r.ql[h][1] = __builtin_amdgcn_alignbit(a.z, a.y, sh);
      r.ql[h][2] = __builtin_amdgcn_alignbit(a.w, a.z, sh);
      r.ql[h][3] = __builtin_amdgcn_alignbit(ax, a.w, sh);
      r.qh[h][0] = __builtin_amdgcn_alignbit(b.y, b.x, sh + L.qh_shift);
      r.qh[h][1] = __builtin_amdgcn_alignbit(b.z, b.y, sh + L.qh_shift);
      r.qh[h][2] = __builtin_amdgcn_alignbit(b.w, b.z, sh + L.qh_shift);
      r.qh[h][3] = __builtin_amdgcn_alignbit(bx, b.w, sh + L.qh_shift);
    }
    const uint4 s = *reinterpret_cast<const uint4*>(slot + L.sc);
    const uint32_t e = *reinterpret_cast<const uint32_t*>(slot + L.dd);
    r.sc[0] = __builtin_amdgcn_alignbit(s.y, s.x, sh);
    r.sc[1] = __builtin_amdgcn_alignbit(s.z, s.y, sh);
    r.sc[2] = __builtin_amdgcn_alignbit(s.w, s.z, sh);
    r.sc[3] = __builtin_amdgcn_alignbit(e, s.w, sh);
    // (the last block of the matrix, at an even place: its last piece was fetched two bytes early; blocks past the end of
    // the row: no scale)
    r.d = (e >> (last ? (sh | L.d_fix) : sh)) & (tail ? L.d_mask : 0xFFFFu);
  }
  struct Prep { float s[4]; };
  static __device__ __forceinline__ void prepare(const Raw& r, const Lane& L, Prep& P) {
    const float d = f16_bits_to_f32((uint16_t)r.d);
#pragma unroll
    for (int c = 0; c < 4; c++) P.s[c] = d * (float)(int)__builtin_amdgcn_sbfe((int)r.sc[c], L.sc_shift, 8);
  }
  // q - 32 itself as bf16, for fp32 activations in three terms: with an offset in the sums, activations whose mean is not zero
  // leave a rounding that the fp32 kernel does not have (1.5e-7 to 2.0e-7 from the float64 product instead of 1.1e-7), and an
  // infinite one makes a NaN of every output.  4 q with its top bit turned is the signed byte 4 (q - 32), one conversion to
  // fp32 each, whose upper half is exact: times 4, which the caller takes out of the activations.
  static __device__ __forceinline__ void signed_weights(const Raw& r, int c, int t, uint32_t (&w)[4]) {
    const int h = c >> 1, p = c & 1;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const uint32_t l = r.ql[h][2 * t + k], q = r.qh[h][2 * t + k];
      const uint32_t u = (((p ? l >> 2 : l << 2) & 0x3C3C3C3Cu) | ((p ? q << 2 : q << 6) & 0xC0C0C0C0u)) ^ 0x80808080u;
      uint32_t f[4];
#pragma unroll
      for (int i = 0; i < 4; i++) f[i] = __float_as_uint((float)(int)(int8_t)(u >> (8 * i)));
      w[2 * k] = __builtin_amdgcn_perm(f[1], f[0], 0x07060302u);
      w[2 * k + 1] = __builtin_amdgcn_perm(f[3], f[2], 0x07060302u);
    }
  }
  // The integer q (0 .. 63) as a 16-bit float with an offset that costs no instruction: bf16 0x3D00 | q = (128 + q) / 4096, fp16
  // 0x5C00 | q << 2 = 256 + q.  The sums are started at -(offset + 32) * sum(x).  (The 4096, taken out of the finished sum by
  // kUnscale, keeps the sums of a sub-block finite for every finite bf16 activation.)
  template <class XT> static constexpr float kStart = std::is_same<XT, f16_tag>::value ? -288.f : -160.f / 4096.f;
  template <class XT> static constexpr float kUnscale = std::is_same<XT, f16_tag>::value ? 1.f : 4096.f;
  template <class XT>
  static __device__ __forceinline__ void weights(const Raw& r, int c, int t, uint32_t (&w)[4]) {
    constexpr bool H = std::is_same<XT, f16_tag>::value;
    constexpr uint32_t N = H ? 0x3C3C3C3Cu : 0x0F0F0F0Fu, Q = H ? 0xC0C0C0C0u : 0x30303030u;
    const int h = c >> 1, p = c & 1;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const uint32_t l = r.ql[h][2 * t + k], q = r.qh[h][2 * t + k];
      // (the bit pairs of the low nibbles are bits 0-1 of the bytes of q, those of the high nibbles bits 4-5)
      const uint32_t lo = H ? (p ? l >> 2 : l << 2) : (p ? l >> 4 : l), hi = H ? (p ? q << 2 : q << 6) : (p ? q : q << 4);
      const uint32_t u = (lo & N) | (hi & Q);
      spread_bytes(u, H ? 0x5C5C5C5Cu : 0x3D3D3D3Du, w[2 * k], w[2 * k + 1]);
    }
  }
};


// 16 blocks of Q4_K -- { f16 d, dmin; u8 scales[12]; u8 qs[128] }, 144 bytes for 256 weights, w = d * sc * q - dmin * mn -- of 16
// weight rows.  Nine 16-byte pieces of a block as they are: row strides of 144 bytes put an operand read on all banks.
struct TlQ4K {
  static constexpr int kSlot = 16 * 144;
  static constexpr int kRequests = 3;
  struct Lane {
    uint32_t src[kRequests], hdr, qs;
    bool upper;
    uint32_t sh;
    template <int KQ> __device__ __forceinline__ void init(int lane, int nsb, int rows, int, bool) {
      static_assert(KQ == 1, "one block of a row");
      const int n = lane & 15, g = lane >> 4;
#pragma unroll
      for (int i = 0; i < kRequests; i++) {
        const int p = min(64 * i + lane, 16 * 9 - 1);
        src[i] = (uint32_t)(min(p / 9, rows - 1) * nsb) * 144u + 16u * (uint32_t)(p % 9);
      }
      hdr = 144u * n;
      qs = hdr + 16u + 32u * g;
      upper = g >= 2;
      sh = 16u * (g & 1);
    }
  };
  template <bool STREAM>
  static __device__ __forceinline__ void request(const Lane& L, int lane, uint32_t lds, const uint8_t* w, int64_t block, bool, bool) {
    const uint8_t* base = w + block * 144;
#pragma unroll
    for (int i = 0; i < kRequests; i++)
      if (i < kRequests - 1 || lane < 16) tile_request<STREAM>(lds + 1024 * i, base, L.src[i]);
  }
  struct Raw { uint4 hdr, q[2]; };
  static __device__ __forceinline__ void read(Raw& r, const uint8_t* slot, const Lane& L, int64_t, bool, bool) {
    r.hdr = *reinterpret_cast<const uint4*>(slot + L.hdr);
    r.q[0] = *reinterpret_cast<const uint4*>(slot + L.qs);
    r.q[1] = *reinterpret_cast<const uint4*>(slot + L.qs + 16);
  }
};

}  // namespace ttq
