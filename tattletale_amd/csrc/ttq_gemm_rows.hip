// Q4_K / Q6_K linear layer for up to 64 activation rows over many weight rows, any number of them (the LM head and the gate||up
// projection of a batch of sequences): the few-row kernel's form that streams the weights through LDS.
//
// Same operator as ttq_gemm_skinny.hip (F.linear with seq_len > 1, workspace/libtorch/src/abi/neural_nets.nim:64-81).
//
// A wavefront owns a block of 16 weight rows at a time and walks K in steps of one weight block (256 values).  Its packed weights
// arrive in its own LDS ring as in ttq_gemv_tile.hip -- sixteen runs of 210 or 144 contiguous bytes -- two steps ahead, the step's
// activations once for the workgroup, by the same kind of request, one step ahead; one barrier a step hands the activations
// over.  They are requested before the step's weights are, so that waiting for them leaves the newest tile of weights in
// flight across the barrier.
//
// The kernel it stands in for reads weights and activations into registers, 16 rows to a load: such a load takes the memory
// pipeline 55 to 110 clocks whatever it carries, and the loads alone were its time (Q6_K 152064 x 3584 at 43 rows 190 us for
// 3 vector instructions a weight).  Here sixteen wavefronts of one block each, four to a SIMD, because a wavefront alone issues a
// vector instruction every eight clocks and waits for LDS in between (eight wavefronts of two blocks, which read every
// activation operand half as often: 158 us against 127).  What bounds it now: at 16 rows the requests (93 us for runs of
// 210 bytes), beyond that vector and LDS instructions, which wait for each other within a step.
//
// Weights.  Q4_K, and Q6_K for bf16 activations: canonical arithmetic in fp32 and one rounding to the activation type, as in the
// register kernel.  Q6_K for fp16 activations: (q - 32) * scale as one packed fp16 multiply-add on 256 + q (exact up to 2048, one
// rounding beyond), the block's d in fp32 on the sums: 1.4e-4 from the float64 product where rounded weights are at 2.0e-4,
// and one instruction for two weights instead of five.
//
// Measured (before: the register kernel; on odd numbers of outputs the tiled GEMM), us: Q6_K fp16 152064 x 3584 at 16 / 43 / 64 rows
// 179 / 194 / 224 -> 99 / 125 / 153, 128256 x 4096 at 16 / 43 158 / 170 -> 92 / 117, bf16 157 / 167 -> 96 / 122; Q4_K fp16 37888 x 3584 at
// 43 / 64 50 / 64 -> 33 / 36; bf16 32003 x 5120 at 16 rows 100 -> 35.  Exact, 128257 x 4096 fp16 at 43 rows 2412 -> 161 (passes of four
// rows in packed dots).
#include "ttq_internal.h"
#include "ttq_tile_common.h"

namespace ttq {
namespace {

constexpr int kRwDepth = 2;                // tiles in a wavefront's ring

// eight bytes u -> fp32 scale * u + offset
__device__ __forceinline__ void rows_fma_bytes(uint32_t q0, uint32_t q1, float scale, float offset, float (&f)[8]) {
  asm volatile("" : "+v"(q0), "+v"(q1));      // (keeps the words opaque: byte k converts with one v_cvt_f32_ubyte<k>)
#pragma unroll
  for (int k = 0; k < 4; k++) {
    f[k] = fmaf_(scale, (float)((q0 >> (8 * k)) & 0xFFu), offset);
    f[4 + k] = fmaf_(scale, (float)((q1 >> (8 * k)) & 0xFFu), offset);
  }
}
__device__ __forceinline__ uint32_t pk_fma_f16(uint32_t a, uint32_t b, uint32_t c) {
  f16x2_t x, y, z;
  __builtin_memcpy(&x, &a, 4);
  __builtin_memcpy(&y, &b, 4);
  __builtin_memcpy(&z, &c, 4);
  const f16x2_t r = __builtin_elementwise_fma(x, y, z);
  uint32_t u;
  __builtin_memcpy(&u, &r, 4);
  return u;
}

// EXACT (Q6_K and fp16 activations): (q - 32) * scale has up to 13 bits; with scale = 4 s1 + s0 it is the sum of two products that fit
// fp16, and two matrix products take the place of one.
template <class F, class XT, bool EXACT> struct RowsOps;

template <class XT, bool EXACT> struct RowsOps<TlQ6K, XT, EXACT> {
  static constexpr bool kF16 = std::is_same<XT, f16_tag>::value;
  static constexpr int kParts = EXACT ? 2 : 1;
  static constexpr bool kScaled = kF16;        // the block's d multiplies the sums
  // step i of lane group g: activations 64 (i / 2) + 16 g + 8 (i % 2) .. + 7, 16-byte piece 8 x_high + (x_lane ^ x_low)
  static __device__ __forceinline__ constexpr uint32_t x_lane(int g) { return 2u * g; }
  static __device__ __forceinline__ constexpr uint32_t x_low(int i) { return (uint32_t)i & 1u; }
  static __device__ __forceinline__ constexpr uint32_t x_high(int i) { return (uint32_t)i >> 1; }
  struct Prep { float d, s[4], o[4]; uint32_t s2[kParts][4], o2[kParts][4]; };
  static __device__ __forceinline__ void prepare(const TlQ6K::Raw& r, const TlQ6K::Lane& L, Prep& P) {
    P.d = f16_bits_to_f32((uint16_t)r.d);
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int si = (int)__builtin_amdgcn_sbfe((int)r.sc[c], L.sc_shift, 8);
      const float sc = (float)si;
      if constexpr (kF16) {
#pragma unroll
        for (int e = 0; e < kParts; e++) {
          const float s = !EXACT ? sc : (float)(e == 0 ? si & ~3 : si & 3);
          P.s2[e][c] = pack_f16x2(s, s);
          P.o2[e][c] = pack_f16x2(-288.f * s, -288.f * s);      // exact: 9 * s * 2^5, 11 bits
        }
      } else {
        P.s[c] = P.d * sc;
        P.o[c] = -32.f * P.s[c];
      }
    }
  }
  static __device__ __forceinline__ void weights(const TlQ6K::Raw& r, const Prep& P, int i, uint32_t (&wp)[kParts][4]) {
    const int c = i >> 1, t = i & 1;
    uint32_t (&w)[4] = wp[0];
    if constexpr (kF16) {
      TlQ6K::weights<XT>(r, c, t, w);                        // 256 + q
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const uint32_t u = w[k];
#pragma unroll
        for (int e = 0; e < kParts; e++) wp[e][k] = pk_fma_f16(u, P.s2[e][c], P.o2[e][c]);
      }
    } else {
      const int h = c >> 1, p = c & 1;
      uint32_t u[2];
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const uint32_t l = r.ql[h][2 * t + k], q = r.qh[h][2 * t + k];
        u[k] = ((p ? l >> 4 : l) & 0x0F0F0F0Fu) | ((p ? q : q << 4) & 0x30303030u);
      }
      float f[8];
      rows_fma_bytes(u[0], u[1], P.s[c], P.o[c], f);
#pragma unroll
      for (int k = 0; k < 4; k++) w[k] = pack_x2<XT>(f[2 * k], f[2 * k + 1]);
    }
  }
};

template <class XT> struct RowsOps<TlQ4K, XT, false> {
  static constexpr int kParts = 1;
  static constexpr bool kScaled = false;
  // step i of lane group g: activations 64 g + 8 i .. + 7
  static __device__ __forceinline__ constexpr uint32_t x_lane(int g) { return 8u * g; }
  static __device__ __forceinline__ constexpr uint32_t x_low(int i) { return (uint32_t)i; }
  static __device__ __forceinline__ constexpr uint32_t x_high(int) { return 0u; }
  struct Prep { float d, s[2], o[2]; };
  static __device__ __forceinline__ void prepare(const TlQ4K::Raw& r, const TlQ4K::Lane& L, Prep& P) {
    // sub-blocks 2g and 2g + 1: two bytes each of the three scale words
    const uint32_t a = r.hdr.y >> L.sh, b = r.hdr.z >> L.sh, c = r.hdr.w >> L.sh;
    const uint32_t sc = L.upper ? (c & 0x0F0Fu) | ((a >> 2) & 0x3030u) : a & 0x3F3Fu;
    const uint32_t mn = L.upper ? ((c >> 4) & 0x0F0Fu) | ((b >> 2) & 0x3030u) : b & 0x3F3Fu;
    const float step = __builtin_amdgcn_cvt_pk_f32_fp8(1, false)[0];
    const float d = f16_bits_to_f32((uint16_t)(r.hdr.x & 0xFFFFu)) * (1.f / step), dmin = f16_bits_to_f32((uint16_t)(r.hdr.x >> 16));
    P.d = 1.f;
    P.s[0] = d * (float)(sc & 0xFFu);
    P.s[1] = d * (float)((sc >> 8) & 0xFFu);
    P.o[0] = -(dmin * (float)(mn & 0xFFu));
    P.o[1] = -(dmin * (float)((mn >> 8) & 0xFFu));
  }
  // nibbles read as 8-bit floats are 0 .. 15 times one power of two (subnormals and the first binade), two to a conversion
  static __device__ __forceinline__ void weights(const TlQ4K::Raw& r, const Prep& P, int i, uint32_t (&wp)[1][4]) {
    uint32_t (&w)[4] = wp[0];
    const int p = i >> 2, t = i & 3;
    const uint32_t* q = reinterpret_cast<const uint32_t*>(&r.q[t >> 1]) + 2 * (t & 1);
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const uint32_t u = (p ? q[k] >> 4 : q[k]) & 0x0F0F0F0Fu;
      const f32x2_t a = __builtin_amdgcn_cvt_pk_f32_fp8((int)u, false), b = __builtin_amdgcn_cvt_pk_f32_fp8((int)u, true);
      w[2 * k] = pack_x2<XT>(fmaf_(P.s[p], a[0], P.o[p]), fmaf_(P.s[p], a[1], P.o[p]));
      w[2 * k + 1] = pack_x2<XT>(fmaf_(P.s[p], b[0], P.o[p]), fmaf_(P.s[p], b[1], P.o[p]));
    }
  }
};

// TB: blocks of 16 tokens; W: wavefronts
template <class F, class XT, int TB, int W, bool EXACT>
__global__ void __launch_bounds__(64 * W)
gemm_rows_kernel(const uint8_t* __restrict__ w, const uint16_t* __restrict__ x, int n_out, int n_in, int m, int y_dtype,
                 void* __restrict__ y, const void* __restrict__ bias, int bias_dtype, const float* __restrict__ row_scale) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t rw_lds[];
  using Ops = RowsOps<F, XT, EXACT>;
  constexpr int kXBuf = 16 * TB * 512;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int nsb = n_in >> 8;
  const int blocks = (n_out + 15) >> 4;
  const int b0 = (int)(((int64_t)blocks * (int)blockIdx.x) / (int)gridDim.x);
  const int nb = (int)(((int64_t)blocks * ((int)blockIdx.x + 1)) / (int)gridDim.x) - b0;
  const int passes = (nb + W - 1) / W;
  auto pass_start = [&](int p) { return (nb * p) / passes; };
  // a block of 16 weight rows to a wavefront, as far as the pass has them
  auto mine = [&](int p) { return wave < pass_start(p + 1) - pass_start(p); };
  const int last_row0 = max(0, n_out - 16);
  auto first_row = [&](int p) { return min(16 * (b0 + pass_start(p) + wave), last_row0); };

  uint8_t* ring = rw_lds + wave * kRwDepth * F::kSlot;
  uint8_t* xbuf = rw_lds + W * kRwDepth * F::kSlot;
  const uint32_t ring_lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)sm_lds(ring));
  const uint32_t x_lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)sm_lds(xbuf));

  typename F::Lane L;
  L.template init<1>(lane, nsb, min(16, n_out), 0, ((int64_t)n_out * nsb) & 1);

  // tiles are requested in order: pass by pass, along K
  int r_p = 0, r_k = 0, r_slot = 0;
  auto skip = [&]() { while (r_p < passes && !mine(r_p)) r_p++; };
  skip();
  auto request_next = [&]() {
    if (r_p == passes) return 0;
    const int row = first_row(r_p);
    const bool tail = r_k == nsb - 1;
    F::template request<false>(L, lane, ring_lds + r_slot * F::kSlot, w, (int64_t)row * nsb + r_k, tail, tail && row == last_row0);
    r_slot ^= 1;
    if (++r_k == nsb) {
      r_k = 0;
      r_p++;
      skip();
    }
    return 1;
  };
  // activations 256 k .. of all tokens, two tokens to a request; piece c of a token lies at place c ^ (token % 8), which puts
  // the sixteen tokens of an operand read on all banks (tokens past the last one repeat it)
  auto request_x = [&](int k, int buf) {
    for (int i = wave; i < 8 * TB; i += W) {
      const uint32_t tok = 2u * (uint32_t)i + ((uint32_t)lane >> 5);
      const uint32_t off = (uint32_t)min((int)tok, m - 1) * (uint32_t)n_in * 2u + 16u * (((uint32_t)lane & 31u) ^ (tok & 7u));
      tile_request<false>(x_lds + (uint32_t)(buf * kXBuf + 1024 * i), reinterpret_cast<const uint8_t*>(x) + 512 * (int64_t)k, off);
    }
  };
  request_x(0, 0);
  for (int d = 0; d < kRwDepth; d++) request_next();
  sm_wait_vmcnt<0>();
  sm_barrier();

  const uint32_t x_at = 512u * n + 16u * (Ops::x_lane(g) ^ ((uint32_t)n & 7u));
  int slot = 0, buf = 0;
  for (int p = 0; p < passes; p++) {
    const bool active = mine(p);
    const int row = first_row(p);
    f32x4_t acc[TB];
#pragma unroll
    for (int tb = 0; tb < TB; tb++) acc[tb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < nsb; k++) {
      const bool more = k < nsb - 1 || p < passes - 1;
      if (more) request_x(k < nsb - 1 ? k + 1 : 0, buf ^ 1);
      int sent = 0;
      if (active) {
        // (this tile was requested before the activations of this step were, and those have landed)
        typename F::Raw raw;
        F::read(raw, ring + slot * F::kSlot, L, (int64_t)row * nsb + k, k == nsb - 1, k == nsb - 1 && row == last_row0);
        slot ^= 1;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        sent = request_next();
        typename Ops::Prep P;
        Ops::prepare(raw, L, P);
        f32x4_t d[TB];
#pragma unroll
        for (int tb = 0; tb < TB; tb++) d[tb] = Ops::kScaled ? f32x4_t{0.f, 0.f, 0.f, 0.f} : acc[tb];
        const uint8_t* xb = xbuf + buf * kXBuf;
#pragma unroll
        for (int i = 0; i < 8; i++) {
          uint4 xf[TB];
#pragma unroll
          for (int tb = 0; tb < TB; tb++)
            xf[tb] = *reinterpret_cast<const uint4*>(xb + (x_at ^ (16u * Ops::x_low(i))) + 128 * Ops::x_high(i) + 8192 * tb);
          uint32_t wv[Ops::kParts][4];
          Ops::weights(raw, P, i, wv);
#pragma unroll
          for (int e = 0; e < Ops::kParts; e++)
#pragma unroll
            for (int tb = 0; tb < TB; tb++) d[tb] = tile_mfma<XT>(xf[tb], wv[e], d[tb]);
        }
#pragma unroll
        for (int tb = 0; tb < TB; tb++) {
          if constexpr (Ops::kScaled) {
#pragma unroll
            for (int i = 0; i < 4; i++) acc[tb][i] = fmaf_(P.d, d[tb][i], acc[tb][i]);
          } else {
            acc[tb] = d[tb];
          }
        }
      }
      // the next step's activations have landed (behind them only this step's tile was requested), in every wavefront
      if (sent) sm_wait_vmcnt<F::kRequests>();
      else sm_wait_vmcnt<0>();
      sm_barrier();
      buf ^= 1;
    }
    // accumulator lane (n, g): weight row n, tokens 4 g .. 4 g + 3 of each block
    const int col = row + n;
    if (active && col >= 16 * (b0 + pass_start(p) + wave) && col < n_out) {
      const float bv = load_bias(bias, bias_dtype, col);
#pragma unroll
      for (int tb = 0; tb < TB; tb++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int tok = 16 * tb + 4 * g + i;
          if (tok >= m) continue;
          float v = acc[tb][i];
          if (row_scale) v *= row_scale[tok];
          v += bv;
          const int64_t o = (int64_t)tok * n_out + col;
          if (y_dtype == kF32) YElem<float>::store(static_cast<float*>(y), o, v);
          else if (y_dtype == kF16) YElem<f16_tag>::store(static_cast<f16_tag*>(y), o, v);
          else YElem<bf16_tag>::store(static_cast<bf16_tag*>(y), o, v);
        }
    }
  }
}

template <class F, class XT, int TB, bool EXACT>
hipError_t launch_rows_tb(const uint8_t* w, const uint16_t* x, void* y, int y_dtype, const void* bias, int bias_dtype, int64_t m,
                          int64_t n_out, int64_t n_in, hipStream_t s, const float* row_scale) {
  // (exact: twelve wavefronts from three token blocks on, for their registers)
  constexpr int W = 16 * kRwDepth * F::kSlot + 2 * 16 * TB * 512 <= 160 * 1024 && !(EXACT && TB > 2) ? 16 : 12;
  constexpr size_t lds = (size_t)W * kRwDepth * F::kSlot + (size_t)2 * 16 * TB * 512;
  static_assert(lds <= 160 * 1024, "fits the compute unit");
  auto kernel = gemm_rows_kernel<F, XT, TB, W, EXACT>;
  static LargeLds configured;
  if (lds > 64 * 1024) {
    const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kernel), configured);
    if (e != hipSuccess) return e;
  }
  const int64_t blocks = (n_out + 15) / 16, cus = device_num_cus();
  hipLaunchKernelGGL(kernel, dim3((unsigned)(blocks < cus ? blocks : cus)), dim3(64 * W), lds, s, w, x, (int)n_out, (int)n_in,
                     (int)m, y_dtype, y, bias, bias_dtype, row_scale);
  return hipGetLastError();
}

template <class F, class XT, bool EXACT = false>
hipError_t launch_rows_f(const uint8_t* w, const uint16_t* x, void* y, int y_dtype, const void* bias, int bias_dtype, int64_t m,
                         int64_t n_out, int64_t n_in, hipStream_t s, const float* row_scale) {
  switch ((m + 15) / 16) {
    case 1: return launch_rows_tb<F, XT, 1, EXACT>(w, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, row_scale);
    case 2: return launch_rows_tb<F, XT, 2, EXACT>(w, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, row_scale);
    case 3: return launch_rows_tb<F, XT, 3, EXACT>(w, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, row_scale);
    case 4: return launch_rows_tb<F, XT, 4, EXACT>(w, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, row_scale);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

bool gemm_rows_supported(int format, int64_t m, int64_t n_out, int64_t n_in) {
  static const int disabled = dev_knob("TTQ_NO_ROWS", 0);
  return !disabled && (format == kQ4_K || format == kQ6_K) && m >= 1 && m <= 64 && n_out > 0 && n_out <= 0x3FFFFFFF && n_in > 0 &&
         n_in % 256 == 0 && n_in <= (1 << 22);
}

// From five blocks of 16 weight rows for every compute unit: a workgroup's wavefronts share one step of activations, and fewer
// blocks leave wavefronts idle.  Measured at 16 rows, us, here / the register kernel, which splits K over its wavefronts: Q4_K
// 28672 x 4096 (seven blocks) 22.7 / 26.2, 14336 x 4096 (three and a half) 16.6 / 14.4; Q6_K fp16 28672 x 8192 48 / 67,
// 13824 x 5120 23.2 / 23.4, 5120 x 13824 48 / 30.
bool gemm_rows_preferred(int64_t n_out) {
  const int64_t blocks = (n_out + 15) / 16;
  return blocks >= 5 && blocks >= 5 * (int64_t)device_num_cus();      // (asked per device, as everywhere)
}

// A launch + passes x steps along K x (a step's chain of waits and reads + its tiles) + the outputs, fitted to 95 shapes of 31 to
// 152064 rows by 256 to 15360 values at 16 to 64 activation rows: 5 percent off on the average, 15 in the square mean.
float gemm_rows_estimate_us(int format, int64_t m, int64_t n_out, int64_t n_in) {
  static const float kStep[4] = {0.58f, 0.65f, 0.8f, 0.9f}, kTile[4] = {0.1f, 0.12f, 0.135f, 0.155f};
  const bool q6 = format == kQ6_K;
  const int t = (int)((m + 15) / 16) - 1;
  const int64_t blocks = (n_out + 15) / 16, cus = device_num_cus(), most = (blocks + cus - 1) / cus;
  const int64_t waves = q6 && t == 3 ? 12 : 16, passes = (most + waves - 1) / waves;
  return (q6 ? 5.f : 4.2f) + (float)(n_in >> 8) * ((float)passes * kStep[t] + (float)most * kTile[t] * (q6 ? 1.2f : 1.f)) * (q6 ? 1.f : 0.94f) +
         (float)(m * n_out) * 0.7e-6f;
}

hipError_t launch_gemm_rows_exact(const void* w, const uint16_t* x_f16, void* y, int y_dtype, const void* bias, int bias_dtype, int64_t m,
                                  int64_t n_out, int64_t n_in, hipStream_t s) {
  return launch_rows_f<TlQ6K, f16_tag, true>(static_cast<const uint8_t*>(w), x_f16, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, nullptr);
}

hipError_t launch_gemm_rows(int format, const void* w, const uint16_t* x, int x_dtype, void* y, int y_dtype, const void* bias,
                            int bias_dtype, int64_t m, int64_t n_out, int64_t n_in, hipStream_t s, const float* row_scale) {
  const uint8_t* wb = static_cast<const uint8_t*>(w);
  const bool h = x_dtype == kF16;
  if (format == kQ4_K)
    return h ? launch_rows_f<TlQ4K, f16_tag>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, row_scale)
             : launch_rows_f<TlQ4K, bf16_tag>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, row_scale);
  if (format == kQ6_K)
    return h ? launch_rows_f<TlQ6K, f16_tag>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, row_scale)
             : launch_rows_f<TlQ6K, bf16_tag>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, row_scale);
  return hipErrorInvalidValue;
}

}  // namespace ttq
