// Decode GEMV for matrices of a few MB (Q8_0 / Q4_K / Q6_K, up to eight activation rows of any type) on gfx950: everything
// that a workgroup reads is asked for at once, straight into registers.
//
// Operator: F.linear with a few activation rows (workspace/libtorch/src/abi/neural_nets.nim:64-81) over the block formats.
//
// What bounds it: latency.  A matrix of 1 to 10 MB is 0.2 to 1.5 us of the memory's time; the rest is the launch (1.6 us), one trip
// to memory, the arithmetic of a wavefront and the way to the sums.  The kernels that stage activations in LDS and then
// walk rows pay for two trips, barriers and lanes that a short row leaves idle (a row of 1024 values is 16 units of 64 weights).
// Here a wavefront takes 1024 values of K, 16 or 32 weights to a lane, of two or four weight rows; it asks for all of their blocks,
// then for its activations, and multiplies once both are there.  Wavefronts of a workgroup share K and meet in LDS once
// (rows of up to 1024 values: not at all).  Nothing is staged, nothing is looped over, so rows far beyond the card's
// wavefronts make it slower than the streams; the rule at gemv_short_preferred has the measured limits.
//
// Arithmetic: fp32 as in gemv_generic_kernel (sums of q * x over a sub-block, scales afterwards); the sums of lanes and wavefronts are
// added in fp64, which costs a dozen instructions and keeps the result at 0.6e-7 to 1.1e-7 from the float64 product although
// a row is cut into more pieces (generic kernel 0.7e-7 to 1.3e-7, packed dots 0.7e-7 to 5e-7, 15-bit block fixed point 1e-5 to 1e-4).
//
// Measured, us, before / now: one row Q8_0 fp32 2048 x 1024 4.6 / 2.8, 1024 x 4096 4.1 / 3.3; Q4_K bf16 1024 x 1024 4.1 / 2.7,
// 1024 x 4096 4.1 / 3.4; Q6_K bf16 1024 x 1024 4.6 / 2.7, 10240 x 1280 10.2 / 6.4, fp32 6144 x 1024 9.3 / 3.7; four rows Q6_K bf16
// 4096 x 1024 8.1 / 4.2, Q8_0 fp32 2048 x 2048 10.5 / 5.0.
#include "ttq_device.h"
#include "ttq_internal.h"

namespace ttq {
namespace {

constexpr int kShMaxWaves = 16;

// N consecutive activations (a multiple of eight, 16-byte aligned) as floats
template <class XT, int N>
__device__ __forceinline__ void short_x(const XT* p, float* f) {
  constexpr int kVec = 16 / (int)sizeof(XT);
#pragma unroll
  for (int i = 0; i < N; i += kVec) {
    XT raw[kVec];
    const uint4 v = *reinterpret_cast<const uint4*>(__builtin_assume_aligned(p + i, 16));
    __builtin_memcpy(raw, &v, 16);
#pragma unroll
    for (int k = 0; k < kVec; k++) f[i + k] = XElem<XT>::load(raw, k);
  }
}

// A format: kW weights to a lane, kG lanes to 1024 values of a row.  Raw: a lane's bytes; Weights: its quants as floats and
// their scales; dot: its share of the row's sum, sx being what sums() makes of the activations.
struct ShQ8 {                       // piece p: quants 16 (p & 1) .. of block p / 2
  static constexpr int kW = 16, kG = 64, kSums = 1;
  static __device__ __forceinline__ uint32_t row_bytes(int n_in) { return (uint32_t)(n_in >> 5) * 34u; }
  struct Raw { uint4 q; uint32_t d; };
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* row, int p) {
    const uint8_t* b = row + 34u * (uint32_t)(p >> 1);
    r.q = load16_a2(b + 2 + 16 * (p & 1));
    r.d = load2(b);
  }
  template <class XT> static __device__ __forceinline__ void x(const XT* xp, int p, float (&f)[kW]) { short_x<XT, 16>(xp + 16 * p, f); }
  struct Weights { float q[kW], d; };
  static __device__ __forceinline__ void weights(const Raw& r, int, Weights& W) {
    const uint32_t dw[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
#pragma unroll
    for (int i = 0; i < kW; i++) W.q[i] = (float)(int)(int8_t)(dw[i >> 2] >> (8 * (i & 3)));
    W.d = f16_bits_to_f32((uint16_t)r.d);
  }
  static __device__ __forceinline__ void sums(const float (&)[kW], float (&)[kSums]) {}
  // (the product with the block's scale is exact in fp64)
  static __device__ __forceinline__ double dot(const Weights& W, const float (&x)[kW], const float (&)[kSums]) {
    float s[2] = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kW; i++) s[i >> 3] = fmaf_(W.q[i], x[i], s[i >> 3]);
    return (double)W.d * (double)(s[0] + s[1]);
  }
};

struct ShQ4 {                       // piece 8 b + t: 16 bytes of quants, the low halves of sub-block t / 2 * 2 of block b, the high ones of the next
  static constexpr int kW = 32, kG = 32, kSums = 2;
  static __device__ __forceinline__ uint32_t row_bytes(int n_in) { return (uint32_t)(n_in >> 8) * 144u; }
  struct Raw { uint4 hdr, q; };
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* row, int p) {
    const uint8_t* b = row + 144u * (uint32_t)(p >> 3);
    r.q = load16_a16(b + 16 + 16 * (p & 7));
    r.hdr = load16_a16(b);
  }
  template <class XT> static __device__ __forceinline__ void x(const XT* xp, int p, float (&f)[kW]) {
    const XT* k = xp + 256 * (p >> 3) + 64 * ((p >> 1) & 3) + 16 * (p & 1);
    short_x<XT, 16>(k, f);
    short_x<XT, 16>(k + 32, f + 16);
  }
  struct Weights { float q[kW], s[2], m[2]; };
  static __device__ __forceinline__ void weights(const Raw& r, int p, Weights& W) {
    const uint32_t dw[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t lo = dw[i] & 0x0F0F0F0Fu, hi = (dw[i] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        W.q[4 * i + k] = (float)((lo >> (8 * k)) & 0xFFu);
        W.q[16 + 4 * i + k] = (float)((hi >> (8 * k)) & 0xFFu);
      }
    }
    // both sub-blocks' scales and minima, a byte each: six bits of sub-blocks 0 to 3, four and two of the others
    const float d = f16_bits_to_f32((uint16_t)(r.hdr.x & 0xFFFFu)), dmin = f16_bits_to_f32((uint16_t)(r.hdr.x >> 16));
    const uint32_t sh = 8u * (p & 2);
    const uint32_t s = r.hdr.y >> sh, m = r.hdr.z >> sh, t = r.hdr.w >> sh;
    const bool upper = p & 4;
    const uint32_t sc = upper ? (t & 0x0F0Fu) | ((s >> 2) & 0x3030u) : s & 0x3F3Fu;
    const uint32_t mn = upper ? ((t >> 4) & 0x0F0Fu) | ((m >> 2) & 0x3030u) : m & 0x3F3Fu;
    W.s[0] = d * (float)(sc & 0xFFu);
    W.s[1] = d * (float)((sc >> 8) & 0xFFu);
    W.m[0] = dmin * (float)(mn & 0xFFu);
    W.m[1] = dmin * (float)((mn >> 8) & 0xFFu);
  }
  static __device__ __forceinline__ void sums(const float (&x)[kW], float (&sx)[kSums]) {
    sx[0] = sx[1] = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) { sx[0] += x[i]; sx[1] += x[16 + i]; }
  }
  static __device__ __forceinline__ double dot(const Weights& W, const float (&x)[kW], const float (&sx)[kSums]) {
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      a = fmaf_(W.q[i], x[i], a);
      b = fmaf_(W.q[16 + i], x[16 + i], b);
    }
    return (W.s[0] * a - W.m[0] * sx[0]) + (W.s[1] * b - W.m[1] * sx[1]);
  }
};

struct ShQ6 {                       // piece 8 b + 4 h + t: weights 128 h + 32 j + 8 t + i of block b, j = 0..3, i = 0..7
  static constexpr int kW = 32, kG = 32, kSums = 1;
  static __device__ __forceinline__ uint32_t row_bytes(int n_in) { return (uint32_t)(n_in >> 8) * 210u; }
  struct Raw { uint2 a, b, h, sc; uint32_t d; };
  static __device__ __forceinline__ uint2 load8(const uint8_t* p) {
    uint2 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 8);
    return v;
  }
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* row, int p) {
    const uint8_t* b = row + 210u * (uint32_t)(p >> 3);
    const int h = (p >> 2) & 1, t = p & 3;
    r.a = load8(b + 64 * h + 8 * t);
    r.b = load8(b + 64 * h + 32 + 8 * t);
    r.h = load8(b + 128 + 32 * h + 8 * t);
    r.sc = load8(b + 192 + 8 * h);
    r.d = load2(b + 208);
  }
  template <class XT> static __device__ __forceinline__ void x(const XT* xp, int p, float (&f)[kW]) {
    const XT* k = xp + 256 * (p >> 3) + 128 * ((p >> 2) & 1) + 8 * (p & 3);
#pragma unroll
    for (int j = 0; j < 4; j++) short_x<XT, 8>(k + 32 * j, f + 8 * j);
    // a quarter of them: the weights are four times themselves
#pragma unroll
    for (int i = 0; i < kW; i++) f[i] *= 0.25f;
  }
  struct Weights { float q[kW], s[4]; };
  static __device__ __forceinline__ void weights(const Raw& r, int p, Weights& W) {
    const uint32_t A[2] = {r.a.x, r.a.y}, B[2] = {r.b.x, r.b.y}, H[2] = {r.h.x, r.h.y};
    constexpr uint32_t N = 0x3C3C3C3Cu, Q = 0xC0C0C0C0u, T = 0x80808080u;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      // 4 q with its top bit turned is the signed byte 4 (q - 32): one conversion a weight
      const uint32_t q[4] = {(((A[i] << 2) & N) | ((H[i] << 6) & Q)) ^ T, (((B[i] << 2) & N) | ((H[i] << 4) & Q)) ^ T,
                             (((A[i] >> 2) & N) | ((H[i] << 2) & Q)) ^ T, (((B[i] >> 2) & N) | (H[i] & Q)) ^ T};
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int k = 0; k < 4; k++) W.q[8 * j + 4 * i + k] = (float)(int)(int8_t)(q[j] >> (8 * k));
    }
    const float d = f16_bits_to_f32((uint16_t)r.d);
    const uint32_t lo = r.sc.x >> (4 * (p & 2)), hi = r.sc.y >> (4 * (p & 2));
    W.s[0] = d * (float)(int)(int8_t)(lo & 0xFFu);
    W.s[1] = d * (float)(int)(int8_t)((lo >> 16) & 0xFFu);
    W.s[2] = d * (float)(int)(int8_t)(hi & 0xFFu);
    W.s[3] = d * (float)(int)(int8_t)((hi >> 16) & 0xFFu);
  }
  static __device__ __forceinline__ void sums(const float (&)[kW], float (&)[kSums]) {}
  static __device__ __forceinline__ double dot(const Weights& W, const float (&x)[kW], const float (&)[kSums]) {
    float t = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++) s = fmaf_(W.q[8 * j + i], x[8 * j + i], s);
      t = j ? fmaf_(W.s[j], s, t) : W.s[j] * s;
    }
    return t;
  }
};

struct Halves { uint32_t lo, hi; };
__device__ __forceinline__ Halves halves(double v) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  return {(uint32_t)u, (uint32_t)(u >> 32)};
}
__device__ __forceinline__ double whole(uint32_t lo, uint32_t hi) { return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo)); }
template <int D> __device__ __forceinline__ double lane_xor_f64(double v, int lane) {
  const Halves h = halves(v);
  return whole(__float_as_uint(lane_xor<D>(__uint_as_float(h.lo), lane)), __float_as_uint(lane_xor<D>(__uint_as_float(h.hi), lane)));
}
// lanes with bit BIT clear get a[i] + a[i ^ BIT], the others b[i] + b[i ^ BIT]
template <int BIT> __device__ __forceinline__ double fold(double a, double b, int lane) {
  if constexpr (BIT >= 16) {
    const Halves ha = halves(a), hb = halves(b);
    if constexpr (BIT == 32) {
      const auto l = __builtin_amdgcn_permlane32_swap(ha.lo, hb.lo, false, false), h = __builtin_amdgcn_permlane32_swap(ha.hi, hb.hi, false, false);
      return whole(l[0], h[0]) + whole(l[1], h[1]);
    } else {
      const auto l = __builtin_amdgcn_permlane16_swap(ha.lo, hb.lo, false, false), h = __builtin_amdgcn_permlane16_swap(ha.hi, hb.hi, false, false);
      return whole(l[0], h[0]) + whole(l[1], h[1]);
    }
  } else {
    const double keep = (lane & BIT) ? b : a, give = (lane & BIT) ? a : b;
    return keep + lane_xor_f64<BIT>(give, lane);
  }
}
// N sums over 2 BIT lanes at once: every fold leaves half of the values, the others in the other half of the lanes.  index: which
// value a lane has got.
template <int BIT, int N>
__device__ __forceinline__ double fold_all(const double (&v)[N], int lane, int& index, int step) {
  if constexpr (N > 1) {
    double h[N / 2];
#pragma unroll
    for (int i = 0; i < N / 2; i++) h[i] = fold<BIT>(v[2 * i], v[2 * i + 1], lane);
    index += (lane & BIT) ? step : 0;
    return fold_all<BIT / 2, N / 2>(h, lane, index, 2 * step);
  } else {
    double t = v[0];
    if constexpr (BIT >= 32) t = fold<32>(t, t, lane);
    if constexpr (BIT >= 16) t = fold<16>(t, t, lane);
    if constexpr (BIT >= 8) t += lane_xor_f64<8>(t, lane);
    if constexpr (BIT >= 4) t += lane_xor_f64<4>(t, lane);
    if constexpr (BIT >= 2) t += lane_xor_f64<2>(t, lane);
    return t + lane_xor_f64<1>(t, lane);
  }
}

struct ShArgs {
  const void* w;
  const void* x;
  void* y;
  const void* bias;
  int m, n_out, n_in, y_dtype, bias_dtype;
};

// RW weight rows and M activation rows to a lane.  ks wavefronts share a row's K, rg groups of rows are in a workgroup.
template <class F, class XT, int RW, int M>
__global__ void __launch_bounds__(M > 1 ? 512 : 1024)
gemv_short_kernel(const uint8_t* __restrict__ w, const XT* __restrict__ x, int n_out, int n_in, int m, int ks, int rg, int y_dtype,
                  void* __restrict__ y, const void* __restrict__ bias, int bias_dtype) {
  constexpr int G = F::kG, P = 64 / G, R = P * RW;          // rows of a wavefront
  __shared__ double part[kShMaxWaves * R * M];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int group = 0, kw = wave;
  while (kw >= ks) { kw -= ks; group++; }
  const int p0 = lane & (G - 1), sub = lane / G;
  const int row0 = ((int)blockIdx.x * rg + group) * R, m0 = (int)blockIdx.y * M;
  const int pieces = n_in / F::kW, p = kw * G + p0, at = p < pieces ? p : 0;     // (past the row's end: the first piece, its sums left out)
  const uint32_t rb = F::row_bytes(n_in);
  typename F::Raw raw[RW];
#pragma unroll
  for (int r = 0; r < RW; r++) F::load(raw[r], w + (size_t)rb * (uint32_t)min(row0 + P * r + sub, n_out - 1), at);
  float xv[F::kW];
  F::template x<XT>(x + (int64_t)min(m0, m - 1) * n_in, at, xv);
  typename F::Weights W[RW];
  double acc[M * RW];
#pragma unroll
  for (int j = 0; j < M; j++) {
    float next[F::kW];
    if (j + 1 < M) F::template x<XT>(x + (int64_t)min(m0 + j + 1, m - 1) * n_in, at, next);
    if (j == 0) {
#pragma unroll
      for (int r = 0; r < RW; r++) F::weights(raw[r], p, W[r]);
    }
    float sx[F::kSums];
    F::sums(xv, sx);
#pragma unroll
    for (int r = 0; r < RW; r++) {
      const double t = F::dot(W[r], xv, sx);
      acc[j * RW + r] = p < pieces ? t : 0.0;      // (not by zeros among the activations: that block's scale may be an infinity)
    }
    if (j + 1 < M) {
#pragma unroll
      for (int i = 0; i < F::kW; i++) xv[i] = next[i];
    }
  }
  int index = 0;
  const double v = fold_all<G / 2, M * RW>(acc, lane, index, 1);
  constexpr int kSame = G / (M * RW);                        // lanes with the same sum
  const bool first = (lane & (kSame - 1)) == 0;
  const int j = index / RW, o = P * (index % RW) + sub;
  auto put = [&](int row, int col, float t) {
    t += load_bias(bias, bias_dtype, col);
    const int64_t at_y = (int64_t)row * n_out + col;
    if (y_dtype == kF32) YElem<float>::store_through(static_cast<float*>(y), at_y, t);
    else if (y_dtype == kF16) YElem<f16_tag>::store(static_cast<f16_tag*>(y), at_y, t);
    else YElem<bf16_tag>::store(static_cast<bf16_tag*>(y), at_y, t);
  };
  if (ks == 1) {
    if (first && m0 + j < m && row0 + o < n_out) put(m0 + j, row0 + o, (float)v);
    return;
  }
  if (first) part[(wave * M + j) * R + o] = v;
  __syncthreads();
  for (int e = tid; e < rg * R * M; e += (int)blockDim.x) {
    const int jj = e / (rg * R), c = e - jj * (rg * R), g = c / R;
    const int col = (int)blockIdx.x * rg * R + c;
    if (m0 + jj >= m || col >= n_out) continue;
    const double* sums = part + g * ks * M * R + jj * R + c % R;      // of the wavefronts of a row, in their order
    double t = sums[0];
    for (int k = 1; k < ks; k++) t += sums[k * M * R];
    put(m0 + jj, col, (float)t);
  }
}

template <class F, class XT, int RW, int M>
hipError_t launch_short_t(const ShArgs& a, hipStream_t s) {
  const int ks = (a.n_in + 1023) / 1024;
  if (ks > (M > 1 ? kShMaxWaves / 2 : kShMaxWaves)) return hipErrorInvalidValue;
  const int rg = ks == 1 ? 4 : (ks == 2 ? 2 : 1);            // four wavefronts at least
  const int per = 64 / F::kG * RW * rg;
  hipLaunchKernelGGL((gemv_short_kernel<F, XT, RW, M>), dim3((unsigned)((a.n_out + per - 1) / per), (unsigned)((a.m + M - 1) / M)),
                     dim3(64 * ks * rg), 0, s, static_cast<const uint8_t*>(a.w), static_cast<const XT*>(a.x), a.n_out, a.n_in, a.m, ks, rg,
                     a.y_dtype, a.y, a.bias, a.bias_dtype);
  return hipGetLastError();
}

// Rows to a lane.  Few wavefronts: as many of them as there is work for; more wavefronts than some three to a SIMD: four rows
// to each, which read the activations once.  us, two / four rows to a wavefront: Q4_K 1024 x 1024 2.7 / 3.0, 6144 x 1024 3.5 / 3.7,
// 4096 x 2048 4.0 / 3.8, 1024 x 14336 5.9 / 5.2; Q8_0 1024 x 2048 2.9 / 3.1, 1024 x 3072 3.2 / 3.0, 1024 x 14336 7.1 / 6.5.
template <class F, class XT>
hipError_t launch_short_x(const ShArgs& a, hipStream_t s) {
  const int64_t waves = (int64_t)((a.n_in + 1023) / 1024) * ((a.n_out + 1) / 2);        // of two rows
  const int cus = device_num_cus();
  if constexpr (F::kG == 64) {
    if (a.m >= 3) return launch_short_t<F, XT, 2, 4>(a, s);
    if (a.m == 2) return launch_short_t<F, XT, 2, 2>(a, s);
    return waves <= 4 * cus ? launch_short_t<F, XT, 2, 1>(a, s) : launch_short_t<F, XT, 4, 1>(a, s);
  } else {
    // (several rows in pairs; small matrices and odd numbers one by one: Q4_K 1024 x 1024 at four rows 2.9 / 3.6, 2560 x 2560 7.9 / 7.0)
    if (a.m % 2 == 0 && waves > 2 * cus) return launch_short_t<F, XT, 2, 2>(a, s);
    return waves * a.m <= 12 * cus ? launch_short_t<F, XT, 1, 1>(a, s) : launch_short_t<F, XT, 2, 1>(a, s);
  }
}
template <class F>
hipError_t launch_short_f(const ShArgs& a, int x_dtype, hipStream_t s) {
  if (x_dtype == kF32) return launch_short_x<F, float>(a, s);
  if (x_dtype == kF16) return launch_short_x<F, f16_tag>(a, s);
  return launch_short_x<F, bf16_tag>(a, s);
}

// millions of weights as wavefronts see them
float short_mega(int64_t n_out, int64_t n_in) { return (float)(n_out * ((n_in + 1023) / 1024)) * 1.024e-3f; }

}  // namespace

bool gemv_short_supported(int format, int64_t m, int64_t n_out, int64_t n_in) {
  if (format != kQ8_0 && format != kQ4_K && format != kQ6_K) return false;
  return m >= 1 && m <= 8 && n_in <= (m > 1 ? 8192 : 16384) && n_out <= (1 << 20);
}

// The time of a call, us.  Of 15981 timed calls 0.74 to 1.19 of it in nine of ten, 0.66 to 1.31 in 49 of 50: too low for small matrices, whose
// launch is most of it, for Q8_0 with 16-bit rows and for rows of many wavefronts (Q4_K 1152 x 10240 5.2 for 7.1, Q6_K 1712 x 5120 at four
// rows 7.9 for 10.8), too high for 8 million weights and more of the K formats.  It decides between this kernel and the few-row kernel for fp32
// calls of two to eight rows: of 545 timed calls that this took from the few-row kernel one got more than 3 percent slower (1712 x 5376 Q6_K at
// four rows 10.6 / 11.1), 17 of them between 8 and 12 million weights.
float gemv_short_estimate_us(int format, int x_dtype, int64_t m, int64_t n_out, int64_t n_in) {
  const float row = format == kQ8_0 && x_dtype != kF32 ? 0.08f : (x_dtype == kF32 ? 0.15f : 0.13f);
  return 2.6f + short_mega(n_out, n_in) * (0.09f + row * (float)m * (m > 1 && m % 2 ? 1.1f : 1.f));
}

// Whether it is the faster one; the kernels that would run otherwise are asked for in the order of launch_gemv.  E: millions of
// weights, rows rounded up to 1024 values.  us, the other kernel / this one, 16-bit rows with 16-bit outputs unless it says otherwise:
//   one row.  Q8_0, the stream (16 rows to a compute unit, whole rounds): 4096 x 2048 4.5 / 4.6, so not there; the windows, from 2048 rows
//     of weights on, 3072 x 2304 (E = 9.4) 6.4 / 4.9, 9504 x 256 (9.7) 4.1 / 4.3, 5520 x 2048 (11) 5.8 / 6.2; else 1024 x 14336 (15) 10.6 / 6.5.
//     Q4_K, the stream: 4096 x 2048 3.1 / 3.8; the int8 kernel, from 2048 rows of weights on, 16-bit 5120 x 1280 (10) 4.4 / 4.0,
//     2048 x 4096 (8.4) 3.8 / 3.9, 10240 x 1280 4.9 / 5.4, fp32 4096 x 1024 3.8 / 3.4, 2048 x 2048 3.5 / 3.4, 2560 x 2560 4.1 / 4.1;
//     packed dots, 1024 x 14336 6.4 / 5.2, a wave of workgroups; 1152 x 10240 (12) 5.6 / 7.1, two; the generic kernel 1536 x 6912 8.1 / 5.4.
//     Q6_K, the stream: 4096 x 2048 4.0 / 4.4; packed dots 10240 x 1280 10.2 / 6.4, 1536 x 6912 6.5 / 5.5, 1152 x 14848 8.9 / 9.4; generic
//     kernel 3072 x 2304 6.7 / 4.7.
//     fp32 outputs of 16-bit rows cost the packed dots 0.8 less than 16-bit ones and this kernel nothing: Q4_K bf16 1536 x 4096 (6.3) 3.5 / 3.7,
//     1024 x 4096 3.4 / 3.4, so from E = 3.3 on, rows of 2049 to 4096 values, they keep the dots.  fp16 rows do not, although 1 to 11 percent
//     slower: their sums with the quants as 1024 + q are 5e-6 to 9e-6 from 64 bits, here 0.5e-7; nor Q8_0 8300 x 256 and more (4.1 / 4.3): the windows
//     read 16-bit rows as fixed point (2e-5).
//   two to four rows.  Q4_K 16-bit, the four-row int8 kernel: 2560 x 2560 (7.9) at two / four rows 6.5 / 5.0, 6.5 / 7.0; packed dots
//     624 x 3584 (2.5) at two 3.8 / 4.0, 1024 x 4096 at four 5.0 / 5.0, 1145 x 2816 (3.5) with 16-bit outputs 5.2 / 5.4.  Q6_K: packed dots
//     1216 x 4096 (5) at two 4.7 / 4.9, 1312 x 2560 (4) 4.3 / 4.6 (1025 to 2048 rows of 2049 to 4096 values), 1712 x 5120 (8.8) at four 9.0 / 10.8; tiles 2560 x 2560 at two 6.1 / 5.0, 7008 x 1024 (7.2) at four 5.7 / 6.2.  fp32 Q4_K 2048 x 2048
//     at two rows 3.8 / 4.2, 2560 x 2560 6.7 / 5.1.  Q8_0: 1536 x 6912 (11) at two / four 11.6 / 8.9, 13.9 / 12.8.
//   five to eight: Q8_0 2560 x 2560 fp32 19.9 / 11.5, 1536 x 6912 14.1 / 20; the windows on long fp32 rows, 1289 x 5632 (E = 7.9) at eight
//     12.6 / 13.6, 1536 x 4608 (7.9) at seven 12.0 / 12.9; E of 6.5 to 7 0.93 of their time in the mean, 7 to 7.5 0.96, 7.5 to 8 0.99.
bool gemv_short_preferred(int format, int x_dtype, int y_dtype, int64_t m, int64_t n_out, int64_t n_in) {
  static const int disabled = dev_knob("TTQ_NO_SHORT", 0);
  if (n_out * n_in > 22000000 || disabled || !gemv_short_supported(format, m, n_out, n_in)) return false;
  const float e = short_mega(n_out, n_in);
  const bool f32 = x_dtype == kF32;
  const auto one_wave = [n_out] { return n_out <= 4 * device_num_cus(); };      // a workgroup of four rows to a compute unit
  if (format == kQ8_0) {
    if (m == 1) return e <= (n_out <= 2048 ? 16.f : 9.5f) && !gemv_q8_stream_supported(format, x_dtype, n_out, n_in);
    if (m <= 4) return e <= 12.f;
    return e <= (f32 && n_in > 3072 && gemv_q8_win_supported(format, n_out, n_in) ? 7.2f : 8.f);
  }
  if (format == kQ6_K) {
    if (m > 4) return f32 && e <= 8.f && n_in <= 4096;
    if (m == 1) return (n_in <= 14336 || one_wave()) && !gemv_q6k_stream_supported(format, x_dtype, n_out, n_in);
    if (f32) return e <= 12.f;
    if (m == 2 && n_out > 1024 && n_out <= 2048 && n_in > 2048 && n_in <= 4096) return false;
    return e <= (m > 2 ? 6.f : (n_out <= 2048 ? 4.5f : 8.f)) && !gemv_q6k_stream4_supported(format, x_dtype, m, n_out, n_in);
  }
  if (m == 1) {
    // (sizes first: what asks for the device costs a launch on the host 0.1 us)
    const bool mfma = gemv_mfma_supported(format, x_dtype, n_out, n_in);
    if (mfma && !(f32 ? e <= 4.2f && n_in <= 1024 : e <= 8.f)) return false;
    if (gemv_q4k_stream_supported(format, x_dtype, n_out, n_in) || gemv_q4k_slice_supported(format, x_dtype, n_out, n_in)) return false;
    if (!mfma && x_dtype == kBF16 && y_dtype == kF32 && n_in > 2048 && n_in <= 4096 && e > 3.3f) return false;
    return mfma || f32 || e <= 7.2f || one_wave();
  }
  if (m > 4) return f32 && e <= 6.f && n_in <= 4096;
  if (f32) return e <= 8.f && (m > 2 || n_in % 2048 != 0 || !gemv_mfma_supported(format, x_dtype, n_out, n_in));
  if (gemv_q4k_stream4_supported(format, x_dtype, m, n_out, n_in)) return false;
  if (gemv_q4k_batch4_supported(format, x_dtype, m, n_out, n_in)) return e <= (m == 2 ? 8.f : 5.f);
  return e <= (m == 2 ? 2.f : (m == 4 && y_dtype != kF32 && n_in > 2048 && n_in <= 3072 ? 3.1f : 4.f));
}

hipError_t launch_gemv_short(int format, const void* w, const void* x, int x_dtype, void* y, int y_dtype, const void* bias,
                             int bias_dtype, int64_t m, int64_t n_out, int64_t n_in, hipStream_t s) {
  const ShArgs a{w, x, y, bias, (int)m, (int)n_out, (int)n_in, y_dtype, bias_dtype};
  if (format == kQ8_0) return launch_short_f<ShQ8>(a, x_dtype, s);
  if (format == kQ4_K) return launch_short_f<ShQ4>(a, x_dtype, s);
  return launch_short_f<ShQ6>(a, x_dtype, s);
}

}  // namespace ttq
