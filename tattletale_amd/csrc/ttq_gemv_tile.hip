// Decode GEMV for Q6_K weights and one to eight activation rows (one or two of fp32) on gfx950, any number of weight rows: the
// quants as small integers on the 16-bit matrix cores.  All activations of a pass are in LDS, which bounds the rows' length:
// 45056 values for one 16-bit row, 22528 for two, 11008 for three and four, 5120 for five to eight; 16384 for one fp32 row (the
// decode kernels' own bound), 7936 for two.
//
// Operator: F.linear with a few activation rows (workspace/libtorch/src/abi/neural_nets.nim:64-81) over GGUF Q6_K blocks
// { u8 ql[128]; u8 qh[64]; i8 scales[16]; f16 d } of 256 weights, w = d * scale[e / 16] * (q6[e] - 32).
//
// Arithmetic.  A quant of six bits is exact in 16-bit floating point, and so is its product with a bf16 or fp16 activation in
// the fp32 sums of v_mfma_f32_16x16x32: nothing is rounded before the block scales meet the sum over a sub-block.  Two bytes
// become two 16-bit floats with one v_perm: 0x3D over q is the bf16 number (128 + q) / 4096, 0x5C over 4 q the fp16 number 256 + q.  The
// offset is not subtracted (one instruction for two weights) but summed with the activations beforehand: every sum starts at
// -(offset + 32) * sum(x).  An fp32 activation is three bf16 terms that add up to it, taken as three rows, and meets q - 32 itself
// (five instructions for four weights more, 128256 x 4096 91 -> 105 us).  From the float64 product, activations of mean zero /
// of mean one and deviation one: fp32 0.8e-7 to 1.0e-7 either way (the generic kernel 1.1e-7), bf16 0.9e-7 to 1.3e-7 / 1.3e-7 to
// 2.0e-7 (packed dots 1.3e-7 to 1.7e-7 / 3.4e-7 to 3.9e-7), fp16 2.8e-7 to 3.5e-7 / 6e-7 to 9e-7 (packed dots 3e-6 / 8e-6 to
// 9e-6); the int8 kernels that read activations as 15-bit block fixed point are at 1e-5 to 3e-5.
//
// Matrix layout.  Weights are the operand with one weight per column, and lane (n, g), n = lane % 16, g = lane / 16, holds
// sub-blocks 4 c + g of its block, eight weights of a different sub-block in every lane group.  The other operand is
// block-diagonal: row 4 b + i holds activations for the k-slots of lane group b only and zeros elsewhere, so that one product
// yields the sums of four sub-blocks apart, and accumulator lane (n, g) gets those of the very sub-block whose scale byte
// it has at hand: four scales a lane and tile, one multiply-add each.  i counts activation rows, and where there are fewer than
// four of them, blocks along K as well (KQ): a tile is then 16 / KQ weight rows by KQ blocks, and a lane keeps the sums of its
// own block.  KQ = 4 for one row lets work be dealt out four weight rows at a time, in runs of 840 contiguous bytes.
//
// Stream.  A wavefront owns a run of tiles, in order along K and then along the rows; runs differ by one tile at most, within a
// workgroup, and workgroups by one group of rows.  Tiles arrive in the wavefront's own LDS ring by global_load_lds requests,
// without registers and without barriers; rows are cut at 16-byte boundaries of the block, rounded down to a dword (blocks are
// 210 bytes), and the operands of a block at an odd place are shifted by 16 bits in registers.  A row of blocks that several
// wavefronts share is added up in LDS in a fixed order.
//
// What bounds it: the requests.  They alone take 69 us for 128256 x 4096 (431 MB) in runs of 840 bytes and 80 in runs of 210
// (KQ = 1), the arithmetic alone 52 to 61, both together 81 (5.3 TB/s); whole-line requests would take 64, but operands then
// start at any dword of LDS, where pairs of dwords take three times as long as 16 bytes on their own boundary: 85.  (Parts switched
// off in forms that are not kept.  Counters at eight rows: LDS busy 76 % of the time, 42 % in conflicts, vector units 56 %, matrix cores 17 %.)  A third
// ring slot, sixteen wavefronts, operands of four tiles in registers: no gain.  Measured (before: packed-dot or generic
// kernel, passes of the several-row int8 kernel), us: 32003 x 5120 fp16 one row 45.3 -> 27.5, two 56.9 -> 28.4, four 101.8 -> 29.3,
// eight 188 -> 32.1; fp32 one row 56.9 -> 34.1; 5120 x 5120 fp16 12.0 -> 8.8, four rows 19.5 -> 11.2; 5120 x 13824 19.6 -> 16.3;
// 128256 x 4096 bf16 at eight rows 152 -> 96, fp32 one row 120 -> 102; 1024 x 41472 bf16 18.2 -> 12.3.
#include "ttq_internal.h"
#include "ttq_tile_common.h"

namespace ttq {
namespace {

constexpr int kTlWaves = 8, kTlThreads = 64 * kTlWaves;
constexpr int kTlDepth = 2;                // tiles in a wavefront's ring: one multiplied, one in flight (56 KiB a compute unit)

static_assert(kTlDepth == 2, "slots and waits alternate");

constexpr int kTlXBlock = 528;             // 256 activations in LDS: the four lanes of a product's k-set on different banks
constexpr int kTlZeroBytes = 512;          // what the lanes off the block diagonal read

// sum + k * both halves of v
template <class XT> __device__ __forceinline__ float add_halves(float k, uint32_t v, float sum) {
  if constexpr (std::is_same<XT, f16_tag>::value) return fmaf_(k, f16_bits_to_f32((uint16_t)(v & 0xFFFFu)), fmaf_(k, f16_bits_to_f32((uint16_t)(v >> 16)), sum));
  else return fmaf_(k, __uint_as_float(v << 16), fmaf_(k, __uint_as_float(v & 0xFFFF0000u), sum));
}
// J: activation rows as the matrix cores see them, PARTS to an activation row (three for fp32).  KQ: blocks along K of a tile, of
// 16 / KQ weight rows.
template <class XT, int J, int KQ, int PARTS>
__global__ void __launch_bounds__(kTlThreads)
gemv_tile_kernel(const uint8_t* __restrict__ w, const void* __restrict__ x, int n_out, int n_in, int m, int y_dtype,
                 void* __restrict__ y, const void* __restrict__ bias, int bias_dtype) {
  using F = TlQ6K;
  extern __shared__ __attribute__((aligned(1024))) uint8_t tl_lds[];
  constexpr int JB = (J * KQ + 3) / 4, JI = J * KQ < 4 ? J * KQ : 4, R = 16 / KQ;
  constexpr int SB = F::kSub, M = J / PARTS;                    // activation rows at most
  constexpr bool kSigned = PARTS > 1;                           // weights without an offset: the sums start at zero
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int nsb = n_in >> 8, tpr = (nsb + KQ - 1) / KQ;       // blocks and tiles of a row
  const int groups = (n_out + R - 1) / R;                      // of R rows

  uint8_t* ring = tl_lds + wave * kTlDepth * F::kSlot;
  uint8_t* zero = tl_lds + kTlWaves * kTlDepth * F::kSlot;
  float* sums = reinterpret_cast<float*>(zero + kTlZeroBytes);                  // [tile][chain][jb][4 g + pseudo row % 4]
  uint8_t* xs = reinterpret_cast<uint8_t*>(sums + (kSigned ? 0 : tpr * F::kChains * JB * 16));
  const uint32_t kpad = (uint32_t)tpr * KQ * 256u, xstride = (uint32_t)tpr * KQ * kTlXBlock;
  float* part = reinterpret_cast<float*>(xs + J * xstride);                     // [wave][first, last][M][R]
  const uint32_t ring_lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)sm_lds(ring)), xs_lds = sm_lds(xs);

  // ---- 16-bit activations: requests straight to their place
  if constexpr (PARTS == 1) {
    for (int row = 0; row < m; row++)
      for (int b = wave; b < nsb; b += kTlWaves)
        if (lane < 32)
          tile_request<false>((uint32_t)__builtin_amdgcn_readfirstlane((int)(xs_lds + row * xstride + kTlXBlock * b)),
                            static_cast<const uint8_t*>(x) + ((int64_t)row * n_in + 256 * b) * 2, 16u * (uint32_t)lane);
  } else {
    for (int e = tid; e < m * (n_in / 8); e += kTlThreads) {
      const int row = e / (n_in / 8), v8 = e - row * (n_in / 8);
      // three bf16 terms that add up to the fp32 value: every term is the rest cut to its upper 16 bits, and what is left of an
      // infinite value is nothing.  A quarter of it: the weights are four times themselves.
      const float4* src = reinterpret_cast<const float4*>(static_cast<const float*>(x) + (int64_t)row * n_in + 8 * v8);
      const float4 f0 = src[0], f1 = src[1];
      float f[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
#pragma unroll
      for (int i = 0; i < 8; i++) f[i] *= 0.25f;
#pragma unroll
      for (int p = 0; p < 3; p++) {
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const uint32_t lo = __float_as_uint(f[2 * i]) & 0xFFFF0000u, hi = __float_as_uint(f[2 * i + 1]) & 0xFFFF0000u;
          o[i] = (lo >> 16) | hi;
          f[2 * i] = f[2 * i] == __uint_as_float(lo) ? 0.f : f[2 * i] - __uint_as_float(lo);
          f[2 * i + 1] = f[2 * i + 1] == __uint_as_float(hi) ? 0.f : f[2 * i + 1] - __uint_as_float(hi);
        }
        *reinterpret_cast<uint4*>(xs + (3 * row + p) * xstride + kTlXBlock * (v8 >> 5) + 16 * (v8 & 31)) = make_uint4(o[0], o[1], o[2], o[3]);
      }
    }
  }

  // ---- the workgroup's groups, and the wavefront's run of their tiles (row by row of groups, along K)
  const int g0 = (int)(((int64_t)groups * (int)blockIdx.x) / (int)gridDim.x);
  const int tiles = ((int)(((int64_t)groups * ((int)blockIdx.x + 1)) / (int)gridDim.x) - g0) * tpr;
  auto run_start = [&](int v) { return (int)(((uint32_t)tiles * (uint32_t)v) / kTlWaves); };
  const int t0 = run_start(wave), t1 = run_start(wave + 1);
  const int qa = t0 / tpr;

  typename F::Lane L;
  L.template init<KQ>(lane, nsb, min(R, n_out), nsb - 1 - (tpr - 1) * KQ, ((int64_t)n_out * nsb) & 1);
  const int last_row0 = max(0, n_out - R);
  auto first_row = [&](int q) { return min(R * (g0 + q), last_row0); };
  int r_left = t1 - t0, r_k = t0 - qa * tpr, r_q = qa, r_slot = 0;       // next request
  int r_row = first_row(qa);
  auto request_next = [&]() {
    if (r_left <= 0) return;
    r_left--;
    const bool tail = r_k == tpr - 1;
    F::template request<KQ == 4>(L, lane, ring_lds + r_slot * F::kSlot, w, (int64_t)r_row * nsb + r_k * KQ, tail, tail && r_row == last_row0);
    r_slot ^= 1;
    r_k++;
    if (tail) {
      r_k = 0;
      r_row = first_row(++r_q);
    }
  };
  for (int d = 0; d < kTlDepth; d++) request_next();

  // ---- zeros: for the lanes off the block diagonal, and behind the rows
  if (tid < kTlZeroBytes / 16) reinterpret_cast<uint4*>(zero)[tid] = make_uint4(0, 0, 0, 0);
  if (KQ > 1 && tpr * KQ > nsb) for (int e = tid; e < J * (KQ - 1) * 32; e += kTlThreads) {
    const int blk = e >> 5, row = blk / (KQ > 1 ? KQ - 1 : 1), b = nsb + blk % (KQ > 1 ? KQ - 1 : 1);
    if (row < J && b < tpr * KQ) *reinterpret_cast<uint4*>(xs + row * xstride + kTlXBlock * b + 16 * (e & 31)) = make_uint4(0, 0, 0, 0);
  }
  // (requests complete in order)
  if constexpr (PARTS == 1) {                                   // the activations have landed: all but the first tiles
    if (t1 - t0 >= 2) sm_wait_vmcnt<2 * F::kRequests>();
    else if (t1 - t0 == 1) sm_wait_vmcnt<F::kRequests>();
    else sm_wait_vmcnt<0>();
  }
  sm_barrier();
  // ---- sums of the activations over sub-blocks, times what the sums of products start at
  if constexpr (!kSigned) {
    const int subs = (int)kpad / SB;
    for (int row = 0; row < J; row++)
      for (int sub = tid; sub < subs; sub += kTlThreads) {
        int c, gg;
        F::sub_of(sub & (256 / SB - 1), c, gg);
        const int blk = sub / (256 / SB), t = blk / KQ, P = row * KQ + blk % KQ;
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < SB / 8; k++) {
          const uint4 q = reinterpret_cast<const uint4*>(xs + row * xstride + kTlXBlock * blk + 2 * SB * (sub & (256 / SB - 1)))[k];
          const uint32_t d4[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
          for (int i = 0; i < 4; i++) v = add_halves<XT>(F::template kStart<XT>, d4[i], v);
        }
        sums[((t * F::kChains + c) * JB + (P >> 2)) * 16 + 4 * gg + (P & 3)] = v;
      }
    sm_barrier();
  }

  // operand lane (i = n, g): pseudo row i % 4 of the block diagonal i / 4 == g; pseudo row P = KQ * row + block
  uint32_t xbase[JB], xmask[JB];
#pragma unroll
  for (int jb = 0; jb < JB; jb++) {
    const int P = 4 * jb + (n & 3), j = P / KQ;
    const bool on = (n >> 2) == g && j < J;
    xmask[jb] = on ? ~0u : 0u;
    xbase[jb] = on ? (uint32_t)(xs - tl_lds) + j * xstride + kTlXBlock * (P % KQ) + 2u * F::lane_k(g) : (uint32_t)(zero - tl_lds);
  }

  f32x4_t acc[JB];
  auto clear = [&]() {
#pragma unroll
    for (int jb = 0; jb < JB; jb++) acc[jb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  // a tile's activations and the values its sums start at
  struct Acts { uint4 x[JB][F::kChains][F::kSteps]; f32x4_t s[kSigned ? 1 : F::kChains][JB]; };
  auto load_acts = [&](Acts& t, int k) {
#pragma unroll
    for (int c = 0; c < F::kChains; c++)
#pragma unroll
      for (int jb = 0; jb < JB; jb++) {
        const uint32_t xa = xbase[jb] + (xmask[jb] & (uint32_t)(kTlXBlock * KQ * k));
        if constexpr (!kSigned) t.s[c][jb] = *reinterpret_cast<const f32x4_t*>(sums + ((k * F::kChains + c) * JB + jb) * 16 + 4 * g);
#pragma unroll
        for (int i = 0; i < F::kSteps; i++) t.x[jb][c][i] = *reinterpret_cast<const uint4*>(tl_lds + xa + 2 * F::chain_k(c) + 16 * i);
      }
  };
  auto multiply = [&](const typename F::Raw& r, const Acts& a) {
    typename F::Prep P;
    F::prepare(r, L, P);
    f32x4_t d[F::kChains][JB];
#pragma unroll
    for (int c = 0; c < F::kChains; c++) {
#pragma unroll
      for (int jb = 0; jb < JB; jb++) d[c][jb] = kSigned ? f32x4_t{0.f, 0.f, 0.f, 0.f} : a.s[kSigned ? 0 : c][jb];
#pragma unroll
      for (int i = 0; i < F::kSteps; i++) {
        uint32_t wv[4];
        if constexpr (kSigned) F::signed_weights(r, c, i, wv);
        else F::template weights<XT>(r, c, i, wv);
#pragma unroll
        for (int jb = 0; jb < JB; jb++) d[c][jb] = tile_mfma<XT>(a.x[jb][c][i], wv, d[c][jb]);
      }
    }
    // (a tile's four products among themselves first: the running sum, the largest of them, is rounded once a tile)
#pragma unroll
    for (int jb = 0; jb < JB; jb++)
#pragma unroll
      for (int i = 0; i < JI; i++) {
        float t = P.s[0] * d[0][jb][i];
#pragma unroll
        for (int c = 1; c < F::kChains; c++) t = fmaf_(P.s[c], d[c][jb][i], t);
        acc[jb][i] += t;
      }
  };

  auto put = [&](int row, int col, float v) {
    v += load_bias(bias, bias_dtype, col);
    const int64_t o = (int64_t)row * n_out + col;
    if (y_dtype == kF32) YElem<float>::store(static_cast<float*>(y), o, v);
    else if (y_dtype == kF16) YElem<f16_tag>::store(static_cast<f16_tag*>(y), o, v);
    else YElem<bf16_tag>::store(static_cast<bf16_tag*>(y), o, v);
  };
  // the wavefront has done its tiles of group q: whole rows are outputs, else the sums wait for the other wavefronts'
  auto finish = [&](int q, bool whole, int which) {
    const int kq = n % KQ, r = n / KQ, col = first_row(q) + r;
    float tot[(M + 3) / 4 * 4];
#pragma unroll
    for (int j = 0; j < (M + 3) / 4 * 4; j++) tot[j] = 0.f;
#pragma unroll
    for (int j = J - 1; j >= 0; j--) {        // (an fp32 row's small terms first)
      // the lane's own block among the pseudo rows of row j
      float v = acc[(j * KQ) >> 2][(j * KQ) & 3];
#pragma unroll
      for (int k = 1; k < KQ; k++) v = kq == k ? acc[(j * KQ + k) >> 2][(j * KQ + k) & 3] : v;
      v = add_xor32(add_xor16(v));
      if constexpr (KQ >= 2) v += lane_xor<1>(v, lane);
      if constexpr (KQ >= 4) v += lane_xor<2>(v, lane);
      tot[j / PARTS] += v;
    }
    if constexpr (!kSigned) {
#pragma unroll
      for (int j = 0; j < M; j++) tot[j] *= F::template kUnscale<XT>;
    }
#pragma unroll
    for (int jb = 0; jb < (M + 3) / 4; jb++) {
      const int j = 4 * jb + g;
      const float v = g == 0 ? tot[4 * jb] : (g == 1 ? tot[4 * jb + 1] : (g == 2 ? tot[4 * jb + 2] : tot[4 * jb + 3]));
      if (kq == 0 && j < m) {
        if (!whole) part[((wave * 2 + which) * M + j) * R + r] = v;
        else if (col >= R * (g0 + q) && col < n_out) put(j, col, v);
      }
    }
    clear();
  };

  int q = qa, k = t0 - qa * tpr, slot = 0, begun = k, row = first_row(qa);
  for (int t = t0; t < t1; t++) {
    Acts acts;
    load_acts(acts, k);
    const bool tail = k == tpr - 1;
    if (t < t1 - 1) sm_wait_vmcnt<F::kRequests>();                // all but the next tile
    else sm_wait_vmcnt<0>();
    typename F::Raw r;
    F::read(r, ring + slot * F::kSlot, L, (int64_t)row * nsb + k * KQ, tail, tail && row == last_row0);
    // (the slot is free for a later tile once the reads have returned)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    request_next();
    multiply(r, acts);
    slot ^= 1;
    k++;
    if (tail || t == t1 - 1) {
      finish(q, tail && begun == 0, q == qa ? 0 : 1);
      k = begun = 0;
      row = first_row(++q);
    }
  }
  // ---- groups that several wavefronts shared: wavefront v adds up the group in which its run starts, if no earlier
  // wavefront's run starts inside of it
  sm_barrier();
  if (wave > 0 && t0 > qa * tpr && t0 < tiles) {
    if (run_start(wave - 1) <= qa * tpr) {
      for (int e = lane; e < m * R; e += 64) {
        const int r = e % R, j = e / R;
        float v = part[((2 * (wave - 1) + (run_start(wave - 1) == qa * tpr ? 0 : 1)) * M + j) * R + r];
        for (int u = wave; u < kTlWaves && run_start(u) < (qa + 1) * tpr; u++)
          if (run_start(u + 1) > run_start(u)) v += part[(2 * u * M + j) * R + r];
        const int col = first_row(qa) + r;
        if (col >= R * (g0 + qa) && col < n_out) put(j, col, v);
      }
    }
  }
}

struct TlArgs {
  const uint8_t* w;
  const void* x;
  void* y;
  const void* bias;
  int m, n_out, n_in, y_dtype, bias_dtype;
};

constexpr size_t kTlLds = 160 * 1024;
size_t tile_lds_bytes(int j, int kq, int parts, int64_t n_in) {
  using F = TlQ6K;
  const size_t jb = (j * kq + 3) / 4, tpr = ((n_in >> 8) + kq - 1) / kq;
  return (size_t)kTlWaves * kTlDepth * F::kSlot + kTlZeroBytes + (parts > 1 ? 0 : tpr * F::kChains * jb * 64) + (size_t)j * (kTlXBlock * kq * tpr) +
         (size_t)2 * kTlWaves * j * (16 / kq) * 4;
}

template <class XT, int J, int KQ, int PARTS = 1>
hipError_t launch_tile_j(const TlArgs& a, hipStream_t s) {
  const size_t lds = tile_lds_bytes(J, KQ, PARTS, a.n_in);
  if (lds > kTlLds) return hipErrorInvalidValue;
  if (route_probe(kRouteGemvTile)) return hipSuccess;      // (here, so that the query answers for the form that would run)
  auto kernel = gemv_tile_kernel<XT, J, KQ, PARTS>;
  static LargeLds configured;
  if (lds > 64 * 1024) {
    const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kernel), configured);
    if (e != hipSuccess) return e;
  }
  const int64_t groups = ((int64_t)a.n_out + 16 / KQ - 1) / (16 / KQ), cus = device_num_cus();
  hipLaunchKernelGGL(kernel, dim3((unsigned)(groups < cus ? groups : cus)), dim3(kTlThreads), lds, s, a.w, a.x, a.n_out, a.n_in,
                     a.m, a.y_dtype, a.y, a.bias, a.bias_dtype);
  return hipGetLastError();
}

// The form of a call: activation rows as the matrix cores see them, blocks along K of a tile.
struct TlForm { int j, kq; };
TlForm tile_form(int x_dtype, int64_t m, int64_t n_out, int64_t n_in) {
  if (x_dtype == kF32) return m == 1 ? TlForm{3, 2} : TlForm{6, 1};
  if (m > 1) return m == 2 ? TlForm{2, 2} : TlForm{m <= 4 ? 4 : 8, 1};
  // One row: four blocks to a tile, except where the last tile of long matrices' rows would be half empty (32003 x 2560 21.3 us
  // with four, 17.9 with two; 7168 x 3584 9.7 / 9.9).  Two take more LDS, and end at rows of 41216 values.
  const bool wide = (n_in >> 8) % 4 == 0 || n_out * (n_in >> 8) * 210 < (24 << 20);
  return TlForm{1, wide || tile_lds_bytes(1, 2, 1, n_in) > kTlLds ? 4 : 2};
}

template <class XT>
hipError_t launch_tile_x(const TlArgs& a, const TlForm& f, hipStream_t s) {
  if (f.j == 1) return f.kq == 4 ? launch_tile_j<XT, 1, 4>(a, s) : launch_tile_j<XT, 1, 2>(a, s);
  if (f.j == 2) return launch_tile_j<XT, 2, 2>(a, s);
  if (f.j == 4) return launch_tile_j<XT, 4, 1>(a, s);
  return launch_tile_j<XT, 8, 1>(a, s);
}

}  // namespace

int gemv_tile_rows(int x_dtype) { return x_dtype == kF32 ? 2 : 8; }

// Whether the kernel takes the shape: all activations of a pass are in LDS at once, beside the ring.
bool gemv_tile_supported(int format, int x_dtype, int64_t m, int64_t n_out, int64_t n_in) {
  static const int disabled = dev_knob("TTQ_NO_TILE", 0);
  if (disabled || format != kQ6_K || n_in % 256 != 0 || m < 1 || m > 8 || n_out > 0x3FFFFFFF || n_in > (1 << 22)) return false;
  if (m > gemv_tile_rows(x_dtype)) return false;
  const TlForm f = tile_form(x_dtype, m, n_out, n_in);
  return tile_lds_bytes(f.j, f.kq, x_dtype == kF32 ? 3 : 1, n_in) <= kTlLds;
}

// Whether it competes with the other decode kernels at all: startup (the activations' sums, a barrier, one tile's chain) is some
// 4 us, so small matrices stay where they are, and 16-bit calls that the int8 stream takes stay there (8192 x 8192 one row 14.7 us
// here, 13.4 there), except for more rows than that kernel takes at once: it computes what the single-row stream computes, to
// 2e-6, and up to 100 MB, where a second pass costs little, that agreement is kept (128256 x 4096 at eight rows 95 / 152.7,
// 151936 x 1024 35.7 / 55.3; four rows of 128256 x 4096 84.7 / 78).
bool gemv_tile_competes(int format, int x_dtype, int64_t m, int64_t n_out, int64_t n_in) {
  const float mb = (float)(n_out * (n_in >> 8) * 210) * 1e-6f;
  if (format != kQ6_K || mb < 5.f) return false;      // (first: small calls are where the host's time counts)
  if (!gemv_tile_supported(format, x_dtype, m, n_out, n_in)) return false;
  if (x_dtype == kF32) return true;
  return m == 1 ? !gemv_q6k_stream_supported(format, x_dtype, n_out, n_in)
                : !gemv_q6k_stream4_supported(format, x_dtype, m, n_out, n_in) || (m > 4 && mb >= 100.f);
}

// Whether it is the faster one, for as many rows as a pass takes.  A workgroup has 4, 8 or 16 weight rows at least and all of K: where
// that leaves compute units idle, the kernels that give a wavefront a row of its own win as long as they hold a row's activations
// in registers (up to 4096 values) or their rounds are whole.  Measured, us, this kernel / the other:
//   one row, 16-bit, against packed dots: rows of more than 4096 values from 12 MB on, 2560 x 6912 8.2 / 9.7, 1000 x 16128 8.0 / 8.7,
//     but for 1025 to 2048 of them, a whole round there: 2048 x 8192 7.3 / 7.1, 1536 x 11008 8.5 / 7.9, 2048 x 16128 10.5 / 10.1
//     (2048 x 22528 12.6 / 13.8); rows of up to 4096 values 7168 x 3584 (21 MB) 9.7 / 8.4, 13824 x 2560 (29 MB) 10.7 / 11.0,
//     32003 x 2560 17.9 / 21.1
//   one fp32 row, against the generic kernel: up to 4096 values 3072 x 4096 8.3 / 7.3, 3328 x 3328 7.5 / 8.5, 4096 x 4096 8.6 / 9.1;
//     longer 1024 x 9216 9.3 / 8.4, 1152 x 9216 9.6 / 12.7, 768 x 15104 11.2 / 10.5,
//     896 x 14336 11.0 / 10.7, 1024 x 14336 11.2 / 11.8; 2560 x 2560 6.8 / 6.8
//   two rows, against packed dots: 2048 x 4096 6.1 / 4.8, 2560 x 4096 7.4 / 7.5, 2048 x 8192 8.4 / 7.8, 2048 x 14336 11.0 / 11.9,
//     768 x 22528 12.3 / 13.9
//   three and four: 2048 x 11008 12.8 / 12.2, 2560 x 4096 8.0 / 9.1, 32003 x 5120 30 / 101
//   five to eight: 1536 x 4096 10.1 / 9.7, 2048 x 3072 9.4 / 10.0, 1536 x 5120 11.4 / 14.8
//   two fp32 rows, against the generic kernel: 1536 x 4096 7.9 / 6.5, 2048 x 4096 8.1 / 8.1, 1024 x 7936 11.0 / 8.6, 1536 x 6912 11.1 / 11.6
bool gemv_tile_preferred(int format, int x_dtype, int64_t m, int64_t n_out, int64_t n_in) {
  static const int always = dev_knob("TTQ_TILE_FIRST", 0);
  if (!gemv_tile_competes(format, x_dtype, m, n_out, n_in)) return false;
  if (always) return true;
  const float mb = (float)(n_out * (n_in >> 8) * 210) * 1e-6f;
  const bool shorter = n_in <= 4096;
  if (x_dtype == kF32) {
    if (m > 1) return n_out > (shorter ? 1536 : 1024);
    return mb >= 7.f && (shorter ? n_out > 3072 : n_out >= (n_in >= 14336 ? 1024 : 1025));
  }
  if (m == 1) return shorter ? mb >= 27.f : mb >= 12.f && !(n_out > 1024 && n_out <= 2048 && n_in <= 16384);
  if (m == 2) return n_out > 2048 || mb >= 18.f || n_in > 16384;
  return m <= 4 ? n_out > 2048 : !shorter || n_out > 1792;
}

// Several rows, us: 21.5 / 134 / 431 MB 10.2 / 28.9 / 84 for two rows, 11.8 / 30 / 87 for four, 15.1 / 33.4 / 98 for eight.  fp32 rows,
// which are three each: small matrices by the tiles that a wavefront has one after the other, one row 2048 x 4096 (one) 6.1,
// 512 x 16128 (four) 11.5, two rows 4096 x 4096 (two) 7.9, 1024 x 6144 (three) 9.7.  The signed weights add a tenth to large ones, which
// is left out: where the few-row kernel over rounded weights is faster by no more than that, the call keeps its precision.
float gemv_tile_estimate_us(int x_dtype, int64_t m, int64_t n_out, int64_t n_in) {
  const float mb = (float)(n_out * (n_in >> 8) * 210) * 1e-6f;
  const float us = (x_dtype == kF32 ? 3 * m : m) <= 4 ? 5.f + mb / 5.2f : 8.3f + mb / 4.8f;
  if (x_dtype != kF32) return us;
  const int rows = m == 1 ? 2048 : 4096;             // a group of them for every compute unit
  const float steps = (float)(n_in >> 8) * (m == 1 ? 1.f / 16 : 1.f / 8) * (float)((n_out + rows - 1) / rows);
  return us < 4.2f + 1.9f * steps ? us : 4.2f + 1.9f * steps;
}

hipError_t launch_gemv_tile(int format, const void* w, const void* x, int x_dtype, void* y, int y_dtype, const void* bias,
                            int bias_dtype, int64_t m, int64_t n_out, int64_t n_in, hipStream_t s) {
  if (m == 0 || n_out == 0) return hipSuccess;
  if (format != kQ6_K) return hipErrorInvalidValue;
  const TlArgs a{static_cast<const uint8_t*>(w), x, y, bias, (int)m, (int)n_out, (int)n_in, y_dtype, bias_dtype};
  const TlForm f = tile_form(x_dtype, m, n_out, n_in);
  if (x_dtype == kF32) return f.j == 3 ? launch_tile_j<bf16_tag, 3, 2, 3>(a, s) : launch_tile_j<bf16_tag, 6, 1, 3>(a, s);
  if (x_dtype == kF16) return launch_tile_x<f16_tag>(a, f, s);
  return launch_tile_x<bf16_tag>(a, f, s);
}

}  // namespace ttq
