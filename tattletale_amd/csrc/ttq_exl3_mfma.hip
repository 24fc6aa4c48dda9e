// Trellis-coded (EXL3-style) decode GEMV on the fp16 matrix cores, one launch:
//
//   y = svh o H( T * H(suh o x) ) + bias
//
// Work split.  A workgroup owns one Hadamard group of 128 output channels (8 tiles across) and one
// slice of the reduction dimension; two of its 16 wavefronts take a 16-channel tile column, half of every
// group's eight k-tiles each.  The
// slices of a group hand their sums to the group's last slice through tagged words in a workspace (one
// store and one load each); the last slice adds them in a fixed order, rotates the 128 sums of
// each row and writes y.  With one slice there is no workspace traffic.
//
// Activations.  They are rotated into LDS before the wavefronts part, as much of the slice as fits (all of it for a
// few rows): x o suh, the 128-group butterfly in registers, then a power-of-two scale per (row, group) that brings the
// group's largest magnitude to 2^14, and a split into two fp16 terms (value and remainder), which together carry 22
// bits.  The B operand holds up to 8 activation rows as 16 columns (term 0, term 1 of each); the two columns are added
// at the end, and each group's matrix-core sum is scaled back in fp32 before it joins the running sum.
//
// Weights.  A wavefront copies the tiles that it decodes into a ring of its own by LDS DMA, packed as they are in
// memory, 16 tiles to a stage, and waits for nobody: there is no barrier until its tiles are done.  (With passes of 32 k-tiles
// that all wavefronts staged together, every pass waited twice for the slowest one, and for the two that rotated its
// activations.  us, one row, passes / rings: 28672 x 4096 3 bits 30.7 / 24.9, 5 bits 35.8 / 27.3, 7 bits 43.9 / 30.5; 4096 x 14336 3 bits
// 18.9 / 16.8, 6 bits 26.6 / 19.1; 4096 x 4096 1 .. 8 bits 8.0 / 8.65 / 8.5 / 9.7 / 9.7 / 12.1 / 11.2 / 12.6 and 8.2 / 8.0 / 8.5 / 8.7 / 9.7 /
// 10.5 / 10.7 / 11.1; 2048 x 1024, where a slice is one group, 2 bits 5.86 / 6.09, 4 bits 6.04 / 6.26, 6 bits 6.7 / 6.5: there the passes
// were 0.2 faster up to five bits, and the launch, the rotation and the hand-off are most of it.)
//
// Decode.  The matrix cores want from lane (j = lane % 16, q = lane / 16) the four weights k = 4q .. 4q+3 of channel j
// of a tile: the windows that start at bit (16j + 4q + e) * bits, e = 0..3.  The lane reads the two dwords that hold
// them, a byte permutation lines them up, and per weight there are a bit-field extract, a 32-bit multiply, one
// three-input bit operation and one fp16 add that writes its half of the A fragment directly, 17 instructions of
// the 19 that a tile costs a wavefront (the vector units are busy 81 % of the time at 28672 x 4096, one row; 224 of 256 compute units).
#include "ttq_exl3_common.h"
#include "ttq_stream_common.h"

#include <mutex>
#include <unordered_map>

namespace ttq {

constexpr int kXmThreads = 1024;                      // 16 wavefronts: the decode is a chain of instructions, which four to a SIMD hide
constexpr int kXmTok = 8;                             // activation rows per workgroup (two B columns each)
constexpr int kXmKSplit = kXmThreads / kWave / 8;     // wavefronts per tile column; each takes 8 / kXmKSplit k-tiles of a group
constexpr int kXmTilesPerWave = 8 / kXmKSplit;
constexpr int kXmStageGroups = 4;                     // Hadamard groups (128 k) to a stage of the ring
constexpr int kXmLds = 160 * 1024;

// A stage is kXmStageGroups * kXmTilesPerWave packed tiles of 32 * BITS bytes.  Two stages in flight behind the one that is
// decoded are 6 KiB * BITS a workgroup for up to 4 bits; above that one is as much.
template <int BITS>
struct XmGeom {
  static constexpr int kTileBytes = 32 * BITS;
  static constexpr int kTiles = kXmStageGroups * kXmTilesPerWave;
  static constexpr int kPieces = kTiles * 2 * BITS;                       // of 16 bytes
  static constexpr int kReq = (kPieces + 63) / 64;                        // requests per stage
  static constexpr int kSlotBytes = kReq * 1024;
  static constexpr int kDepth = BITS <= 4 ? 3 : 2;
  static constexpr int kRingBytes = (kXmThreads / kWave) * kDepth * kSlotBytes;
};
template <typename T>
__device__ __forceinline__ T lds_at(uint32_t a) {
  return *(const __attribute__((address_space(3))) T*)(size_t)a;
}
constexpr int kXmColPad = 8;                          // halfs: the 16 columns of a B read fall on different banks
// LDS for `groups` Hadamard groups of activations of `cols` columns: the terms and their scales
constexpr int xm_x_bytes(int cols, int groups) { return cols * (groups * 128 + kXmColPad) * 2 + cols * groups * 4; }

// The first activations (16 bytes a lane in fp32, else 8) and their signs, then the N requests of a stage at lds and the 1 KiB
// places after it, and a wait for the activations alone.  In one statement: the compiler, which knows nothing of the
// requests, would wait for them too.
#define TTQ_XM_REQUEST(I) "s_add_u32 m0, %[lds], " #I "*1024\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %[a" #I "], off\n\t"
#define TTQ_XM_FIRST(X, REQUESTS, N, ...)                                                                                  \
  asm volatile("global_load_dwordx2 %[s], %[sp], off\n\tglobal_load_" X " %[x], %[xp], off\n\t" REQUESTS "s_waitcnt vmcnt(" #N ")" \
               : [s] "=&v"(s), [x] "=&v"(v)                                                                                \
               : [sp] "v"(sp), [xp] "v"(xp), [lds] "s"(lds), __VA_ARGS__                                                  \
               : "memory", "scc")
#define TTQ_XM_FIRST_N(X)                                                                                                  \
  if constexpr (N == 1) TTQ_XM_FIRST(X, TTQ_XM_REQUEST(0), 1, [a0] "v"(a[0]));                                            \
  else if constexpr (N == 2) TTQ_XM_FIRST(X, TTQ_XM_REQUEST(0) TTQ_XM_REQUEST(1), 2, [a0] "v"(a[0]), [a1] "v"(a[1]));      \
  else if constexpr (N == 3)                                                                                               \
    TTQ_XM_FIRST(X, TTQ_XM_REQUEST(0) TTQ_XM_REQUEST(1) TTQ_XM_REQUEST(2), 3, [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2])); \
  else                                                                                                                     \
    TTQ_XM_FIRST(X, TTQ_XM_REQUEST(0) TTQ_XM_REQUEST(1) TTQ_XM_REQUEST(2) TTQ_XM_REQUEST(3), 4, [a0] "v"(a[0]),            \
                 [a1] "v"(a[1]), [a2] "v"(a[2]), [a3] "v"(a[3]))
typedef uint32_t xm_u32x2 __attribute__((ext_vector_type(2)));
template <int N, typename XT>
__device__ __forceinline__ void xm_first_loads(XmRaw<XT>& xv, uint2& sv, const XT* xp, const uint16_t* sp, uint32_t lds,
                                               const uint8_t* const (&a)[N]) {
  static_assert(N >= 1 && N <= 4);
  xm_u32x2 s;
  if constexpr (sizeof(xv) == 16) {
    sm_u32x4 v;
    TTQ_XM_FIRST_N("dwordx4");
    __builtin_memcpy(&xv, &v, 16);
  } else {
    xm_u32x2 v;
    TTQ_XM_FIRST_N("dwordx2");
    __builtin_memcpy(&xv, &v, 8);
  }
  __builtin_memcpy(&sv, &s, 8);
}
#undef TTQ_XM_FIRST_N
#undef TTQ_XM_FIRST
#undef TTQ_XM_REQUEST

template <int BITS, int CB, typename XT>
__global__ void __launch_bounds__(kXmThreads)
gemv_exl3_mfma_kernel(const uint16_t* __restrict__ trellis, const uint16_t* __restrict__ suh,
                      const uint16_t* __restrict__ svh, const XT* __restrict__ x, void* __restrict__ y, int y_dtype,
                      const void* __restrict__ bias, int bias_dtype, int m, int n_out, int n_in, int slice_groups,
                      int chunk_groups, unsigned long long* __restrict__ accum, int poll_limit) {
  using G = XmGeom<BITS>;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  _Float16* xs = reinterpret_cast<_Float16*>(lds + G::kRingBytes);
  float* yp = reinterpret_cast<float*>(lds);                      // (after the last tile: the rings are done with)
  float* yq = yp + kXmTok * 128;                                  // the other wavefronts of a tile column

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = blockIdx.x, slice = blockIdx.y, nslices = gridDim.y;
  const int t0 = blockIdx.z * kXmTok;
  const int ntok = min(kXmTok, m - t0), cols = 2 * ntok;
  const int nt_n = n_out >> 4;
  // Hadamard groups of this slice: slice_groups, and one more in as many of the last slices as are left over (worked out here:
  // with one argument more the grid's size is read in a second round trip, 0.06 to 0.4 us)
  const int longer = slice + (n_in >> 7) - (slice_groups + 1) * nslices;
  const int kt_begin = 8 * (slice * slice_groups + max(longer, 0));
  const int groups = slice_groups + (longer >= 0 ? 1 : 0);
  const int col = lane & 15, q = lane >> 4;
  const int xstride = chunk_groups * 128 + kXmColPad;
  float* inv_s = reinterpret_cast<float*>(xs + cols * xstride);                  // [group of the chunk][column]
  const int tcol = wave & 7, kpart = wave >> 3;          // tile column, and which k-tiles of every group

  XmLane<BITS> ln;
  ln.init(lane);

  // The tag of this launch's hand-off words: the workspace's generation count + 1 (read now, needed at the end).
  // accum[0] holds the generation, accum[1] the number of groups that have finished, the words start at accum + 8.
  // (Without a branch around the load, which would be waited for where the branch ends; a launch that is not sliced reads
  // any dword.)
  const uint32_t generation =
      __hip_atomic_load(nslices > 1 ? reinterpret_cast<const uint32_t*>(accum) : reinterpret_cast<const uint32_t*>(trellis),
                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  // ---- weights: stage s holds this wavefront's tiles of the groups 4s .. 4s+3 of the slice (past its end what it has, again)
  const int64_t row_bytes = (int64_t)nt_n * G::kTileBytes;
  const uint8_t* wbase = reinterpret_cast<const uint8_t*>(trellis) + ((int64_t)grp * 8 + tcol) * G::kTileBytes +
                         (int64_t)(kt_begin + kpart * kXmTilesPerWave) * row_bytes;
  const uint32_t ring = sm_lds(lds) + (uint32_t)(wave * G::kDepth * G::kSlotBytes);
  const int stages = (groups + kXmStageGroups - 1) / kXmStageGroups;
  int64_t src[G::kReq];
  auto place = [&](int left) {                           // left: groups from the stage's first on
    // (where the lanes past the last piece are more than none, they and those of absent groups repeat the last one: 2304 x 768, seven
    // bits, 8.7 -> 7.0 us; whole requests repeat the last group: 3072 x 1024, eight bits, 6.7 against 7.0)
    constexpr bool kWhole = G::kPieces % 64 == 0;
    const uint32_t last = kWhole ? G::kPieces - 1 : (uint32_t)min(left, kXmStageGroups) * (kXmTilesPerWave * 2 * BITS) - 1;
#pragma unroll
    for (int r = 0; r < G::kReq; r++) {
      const uint32_t p = min(64u * r + (uint32_t)lane, last), t = p / (2u * BITS), c = p - t * (2u * BITS);
      const uint32_t gl = kWhole ? min(t / kXmTilesPerWave, (uint32_t)left - 1u) : t / kXmTilesPerWave;
      src[r] = (int64_t)((uint64_t)(gl * 8 + t % kXmTilesPerWave) * (uint64_t)row_bytes) + 16u * c;
    }
  };
  place(groups);
  int asked = 0, ask_slot = 0;
  auto request = [&]() {
    const int left = groups - asked * kXmStageGroups;
    if (left < kXmStageGroups) place(left);
    const uint8_t* base = wbase + (int64_t)asked * (kXmStageGroups * 8) * row_bytes;
    const uint32_t dst = ring + (uint32_t)(ask_slot * G::kSlotBytes);
#pragma unroll
    for (int r = 0; r < G::kReq; r++) {
      const uint8_t* a = base + src[r];
      // (in assembly: the compiler would wait for all of them before any LDS read that follows)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst + r * 1024), "v"(a) : "memory");
    }
    asked++;
    ask_slot = ask_slot == G::kDepth - 1 ? 0 : ask_slot + 1;
  };

  // ---- activations of a chunk: (row, group) items of 32 lanes, four values each; the next item's are requested before
  // one is rotated (and the first one's before the weights')
  const int hw = tid >> 5, l32 = tid & 31;
  XmRaw<XT> xv;
  uint2 sv;
  const uint16_t* sp;
  const XT* xp;
  // (item / ng by a reciprocal, an integer division being 0.15 to 0.3 us of a launch of several rows: a quotient below 8 is off by
  // 8 * 2^-22 at most and 0.5 / ng from the next whole number, with ng below 320 for what LDS holds)
  auto row_of = [&](int item, int ng) { return (int)(((float)item + 0.5f) * __builtin_amdgcn_rcpf((float)ng)); };
  auto x_place = [&](int g0, int ng, int item) {
    const int it = min(item, ntok * ng - 1), t = row_of(it, ng), gl = it - t * ng;
    const int64_t k = (int64_t)kt_begin * 16 + (int64_t)(g0 + gl) * 128 + 4 * l32;
    sp = suh + k;
    xp = x + (int64_t)(t0 + t) * n_in + k;
  };
  auto x_request = [&](int g0, int ng, int item) {
    x_place(g0, ng, item);
    __builtin_memcpy(&sv, __builtin_assume_aligned(sp, 8), 8);
    xv.load(xp);
  };
  auto x_stage = [&](int g0, int ng) {
    for (int item = hw; item < ntok * ng; item += kXmThreads / 32) {
      const int t = row_of(item, ng), gl = item - t * ng;
      float v[4];
      xv.get(v);
      v[0] *= f16_bits_to_f32((uint16_t)sv.x);
      v[1] *= f16_bits_to_f32((uint16_t)(sv.x >> 16));
      v[2] *= f16_bits_to_f32((uint16_t)sv.y);
      v[3] *= f16_bits_to_f32((uint16_t)(sv.y >> 16));
      if (item + kXmThreads / 32 < ntok * ng) x_request(g0, ng, item + kXmThreads / 32);
      fwht128_quad(v, lane);
      float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
      amax = fmaxf(amax, lane_xor<1>(amax, lane));
      amax = fmaxf(amax, lane_xor<2>(amax, lane));
      amax = fmaxf(amax, lane_xor<4>(amax, lane));
      amax = fmaxf(amax, lane_xor<8>(amax, lane));
      amax = fmaxf(amax, lane_xor<16>(amax, lane));
      // scale 2^(14 - exponent of amax); all-zero groups get the largest scale, which changes nothing
      int se = 268 - (int)((__float_as_uint(amax) >> 23) & 0xFF);
      se = se > 254 ? 254 : se;
      const float sc = __uint_as_float((uint32_t)se << 23);
      f16x4_t hi, lo;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float s = v[i] * sc;
        hi[i] = (_Float16)s;
        lo[i] = (_Float16)(s - (float)hi[i]);
      }
      // (a B operand of 32 k is 16 consecutive bytes: four k of one k-tile, the same four of the next)
      const int kl = gl * 128 + (l32 >> 3) * 32 + (l32 & 3) * 8 + (l32 >> 2 & 1) * 4;
      *reinterpret_cast<f16x4_t*>(xs + (2 * t) * xstride + kl) = hi;
      *reinterpret_cast<f16x4_t*>(xs + (2 * t + 1) * xstride + kl) = lo;
      if (l32 == 0) {
        // 1/sqrt(128) of the input rotation over the scale
        const float inv = 0.08838834764831845f * __uint_as_float((uint32_t)(254 - se) << 23);
        inv_s[gl * cols + 2 * t] = inv;
        inv_s[gl * cols + 2 * t + 1] = inv;
      }
    }
  };

  // (half-wavefronts split unevenly over the items: the lanes of one wavefront may leave x_stage's loop at different times, which
  // lane_xor within 32 lanes does not mind)
  {
    x_place(0, min(chunk_groups, groups), hw);
    const uint8_t* first[G::kReq];
#pragma unroll
    for (int r = 0; r < G::kReq; r++) first[r] = wbase + src[r];
    xm_first_loads<G::kReq>(xv, sv, xp, sp, ring, first);
    asked = ask_slot = 1;
  }

  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  const int xcol = col < cols ? col : 0;                 // (columns past the last row's: their sums are not looked at)
  int slot = 0, done = 0;
  for (int g0 = 0; g0 < groups; g0 += chunk_groups) {    // a chunk is a whole number of stages, or the slice
    const int ng = min(chunk_groups, groups - g0);
    if (g0 > 0) {
      sm_barrier();                                      // the chunk before has been read
      x_request(g0, ng, hw);
    }
    x_stage(g0, ng);
    while (asked < min(stages, done + G::kDepth)) request();
    sm_barrier();
    // LDS addresses in registers, so that the reads of a stage differ in their constant offsets only
    uint32_t xa = sm_lds(xs + xcol * xstride + kpart * kXmTilesPerWave * 16 + 8 * q), ia = sm_lds(inv_s + xcol);
    for (int left = ng; left > 0; left -= kXmStageGroups) {
      // requests complete in order: all but those of the stages after this one have landed
      switch (asked - done - 1) {
        case 0: sm_wait_vmcnt<0>(); break;
        case 1: sm_wait_vmcnt<G::kReq>(); break;
        default: sm_wait_vmcnt<2 * G::kReq>(); break;
      }
      constexpr int kWin = XmLane<BITS>::kWin;
      uint32_t cw[2][kXmTilesPerWave][kWin][2];
      f16x8_t bx[2][kXmTilesPerWave / 2];
      float inv[2];
      uint32_t wa[kWin][2];
#pragma unroll
      for (int w = 0; w < kWin; w++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          wa[w][h] = ring + (uint32_t)(slot * G::kSlotBytes) + ln.at[w][h];
          asm("" : "+v"(wa[w][h]));
        }
      asm("" : "+v"(xa), "+v"(ia));
      auto fetch_group = [&](int gl, int buf) {
#pragma unroll
        for (int i = 0; i < kXmTilesPerWave; i++) {
#pragma unroll
          for (int w = 0; w < kWin; w++)
#pragma unroll
            for (int h = 0; h < 2; h++)
              cw[buf][i][w][h] = lds_at<uint32_t>(wa[w][h] + (gl * kXmTilesPerWave + i) * G::kTileBytes);
          if (i % 2 == 0) bx[buf][i / 2] = lds_at<f16x8_t>(xa + (gl * 128 + i * 16) * 2);
        }
        inv[buf] = lds_at<float>(ia + gl * 4 * cols);
      };
      auto compute_group = [&](int buf) {
        f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kXmTilesPerWave; i += 2) {
          uint32_t r[4];
          ln.template decode<CB>(cw[buf][i], reinterpret_cast<uint32_t(&)[2]>(r[0]));
          ln.template decode<CB>(cw[buf][i + 1], reinterpret_cast<uint32_t(&)[2]>(r[2]));
          f16x8_t a;
          __builtin_memcpy(&a, r, 16);
          d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bx[buf][i / 2], d, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) acc[r] = fmaf_(d[r], inv[buf], acc[r]);
      };
      // the LDS reads of a group are issued while the group before it is decoded
      fetch_group(0, 0);
#pragma unroll
      for (int gl = 0; gl < kXmStageGroups; gl++) {
        if (gl < left) {
          if (gl + 1 < kXmStageGroups && gl + 1 < left) fetch_group(gl + 1, (gl + 1) & 1);
          compute_group(gl & 1);
        }
      }
      // (the slot is free for a later stage: its reads have returned)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      done++;
      slot = slot == G::kDepth - 1 ? 0 : slot + 1;
      if (asked < stages) request();
      xa += kXmStageGroups * 256;
      ia += kXmStageGroups * 4 * cols;
    }
  }
  // ---- the two terms of each row.  Then, in a sliced launch, every slice but the last hands its sums
  // to the last one straight from the registers, through tagged 64-bit words (the launch's tag in the high
  // half, the float in the low half) written and read with agent-scope accesses, which are coherent across
  // the chip without cache maintenance.  The last slice polls each word until this launch's tag is there
  // (a bounded number of times: rows it gave up on come out as NaN) and adds everything in a fixed order.
  // Nothing is cleared: the tag is the workspace's generation count + 1, and the group that finishes last
  // advances the count, so the words of this launch -- also those of a slice that arrives after its group
  // gave up on it -- can never pass for words of a later one.  The count lives in the workspace and not in
  // a kernel argument because a captured graph replays its arguments.  What remains: a slice that has not
  // even begun when its group gives up reads the advanced count and tags its words like the next launch
  // will; that takes a wavefront dispatch held back for poll_limit polls (tens of milliseconds by default).
#pragma unroll
  for (int r = 0; r < 4; r++) acc[r] += lane_xor<1>(acc[r], lane);
  const bool owner = (col & 1) == 0 && (col >> 1) < ntok;      // this lane holds 4 channel sums of row col / 2
  constexpr int kPartWords = kXmTok * 128;                        // words per (slice, k part)
  const uint32_t tag = generation + 1u;
  unsigned long long* words = nullptr;
  if (nslices > 1) {
    words = accum + 8 + (((int64_t)blockIdx.z * gridDim.x + grp) * nslices) * (kXmKSplit * kPartWords);
    if (slice != nslices - 1) {
      if (owner) {
        unsigned long long* dst = words + ((int64_t)slice * kXmKSplit + kpart) * kPartWords + (col >> 1) * 128 + tcol * 16 + 4 * q;
#pragma unroll
        for (int r = 0; r < 4; r++)
          __hip_atomic_store(dst + r, ((unsigned long long)tag << 32) | __float_as_uint(acc[r]), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      }
      return;
    }
  }
  sm_barrier();                                          // all tiles have been read: the rings' place is free
  {
    float* dst = kpart == 0 ? yp : yq + (kpart - 1) * kPartWords;
    if (owner) *reinterpret_cast<float4*>(dst + (col >> 1) * 128 + tcol * 16 + 4 * q) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  }
  __syncthreads();
  // The other slices' words, sixteen loads in flight before the first is looked at, and dealt out over several threads to a sum
  // where there are more: a round trip to the memory side is most of what this costs, and with one thread to a sum the 62
  // words of 32 slices took four of them (1024 x 4096, one row: 8.95 -> 7.4 us).  Sixteen words are a batch, batch b is
  // added to part b % 8, the parts to each other: the same order for any number of rows.
  constexpr int kHandoffBatch = 16, kHandoffParts = 8;
  float* red = yq + (kXmKSplit - 1) * kPartWords;              // [part][sum]
  const int nwords = (nslices - 1) * kXmKSplit, sums = ntok * 128;
  const int batches = (nwords + kHandoffBatch - 1) / kHandoffBatch, parts = min(batches, kHandoffParts);
  int deal = 1;                                                // threads to a sum (scalar shifts and compares: an integer division here is 0.4 us)
  while (deal < parts && sums * deal * 2 <= kXmThreads) deal *= 2;
  float handed = 0.f;
  if (nwords > 0) {
    // The slices of a group finish their decode within a fraction of a microsecond of each other, and a word asked for
    // before it has reached the memory side costs a second round trip (about 0.9 us): 256 clocks of patience before
    // the first look make it the only one.  64 are enough for slices of a few groups with a look at sixteen words, and up to three
    // bits, where the decode is short.  us with 64 / 256 clocks: 2048 x 1024 two bits 6.05 / 6.19, four 6.22 / 6.35, 4096 x 4096 three
    // 8.46 / 8.65, four 8.99 / 8.83, six 11.2 / 11.0, 1536 x 1536 (22 words) four 6.87 / 6.68.
    if (BITS <= 3 || (groups < kXmStageGroups && nwords <= kHandoffBatch)) __builtin_amdgcn_s_sleep(1);
    else __builtin_amdgcn_s_sleep(4);
    int d = 0;
    for (int r = wave >> 1; r >= ntok; r -= ntok) d++;
    const int e = tid - d * sums;
    if (d < deal) {
      for (int part = d; part < parts; part += deal) {
        float c = 0.f;
        bool late = false;
        for (int b = part; b < batches; b += kHandoffParts) {
          const int p0 = b * kHandoffBatch;
          unsigned long long w[kHandoffBatch];
#pragma unroll
          for (int i = 0; i < kHandoffBatch; i++)
            w[i] = __hip_atomic_load(words + (int64_t)min(p0 + i, nwords - 1) * kPartWords + e, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
          for (int i = 0; i < kHandoffBatch; i++) {
            if (p0 + i < nwords) {
              unsigned long long* wp = words + (int64_t)(p0 + i) * kPartWords + e;
              for (int polls = 0; (uint32_t)(w[i] >> 32) != tag && polls < poll_limit; polls++) {
                __builtin_amdgcn_s_sleep(2);
                w[i] = __hip_atomic_load(wp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              }
              late |= (uint32_t)(w[i] >> 32) != tag;
              c += __uint_as_float((uint32_t)w[i]);
            }
          }
        }
        if (late) c = __uint_as_float(0x7FC00000u);
        if (deal > 1) red[part * sums + e] = c;
        else handed += c;
      }
    }
    if (deal > 1) __syncthreads();
  }
  if (tid < sums) {
    if (deal > 1)
      for (int part = 0; part < parts; part++) handed += red[part * sums + tid];
    float s = handed;
    s += yp[tid];
#pragma unroll
    for (int k = 1; k < kXmKSplit; k++) s += yq[(k - 1) * kPartWords + tid];
    yp[tid] = s;
  }
  // The workgroup has now seen (or given up on) a word of every other slice of its group, so each of them has read
  // the generation count.  Thread 0 counts its group in here and looks at the answer after the output phase: the group
  // that is counted last advances the generation.
  uint32_t counted = 0;
  if (nslices > 1 && tid == 0)
    counted = __hip_atomic_fetch_add(reinterpret_cast<uint32_t*>(accum) + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();

  // ---- output side: rotate the 128 sums of each row, svh, bias
  if (hw < ntok) {
    float v[4];
    const float4 t = *reinterpret_cast<const float4*>(yp + hw * 128 + 4 * l32);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    fwht128_quad(v, lane);
    const int n = grp * 128 + 4 * l32;
    uint2 sraw;
    __builtin_memcpy(&sraw, __builtin_assume_aligned(svh + n, 8), 8);
    const float svf[4] = {f16_bits_to_f32((uint16_t)sraw.x), f16_bits_to_f32((uint16_t)(sraw.x >> 16)),
                          f16_bits_to_f32((uint16_t)sraw.y), f16_bits_to_f32((uint16_t)(sraw.y >> 16))};
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      o[i] = v[i] * 0.08838834764831845f * svf[i];
      if (bias) o[i] += load_bias(bias, bias_dtype, n + i);
    }
    xm_store4(y, y_dtype, (int64_t)(t0 + hw) * n_out + n, o);
  }
  if (nslices > 1 && tid == 0 && counted == gridDim.x * gridDim.z - 1) {
    uint32_t* ctl = reinterpret_cast<uint32_t*>(accum);
    __hip_atomic_store(ctl + 2, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(ctl, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ------------------------------------------------------------------------------ launch
Exl3Plan exl3_mfma_plan(int64_t m, int64_t n_out, int64_t n_in) {
  Exl3Plan p;
  p.groups = (int)(n_out / 128);
  p.row_groups = (int)((m + kXmTok - 1) / kXmTok);
  const int64_t units = (int64_t)p.groups * p.row_groups;
  const int cus = device_num_cus();
  // Enough slices to put a workgroup on every compute unit, each a whole number of Hadamard groups, as few as leave the longest as
  // long as it is, and no two more than one group apart.  The longest are the last ones: a last slice that is done before the
  // others asks again and again for words that they have yet to write, which holds up the writers (us, all but the last slice
  // equally long and the last what is left / the extra groups in the first slices / in the last ones: 7168 x 1792, 14 groups in
  // four slices, one row of six bits 14.0 / 10.1 / 10.0, eight rows 22.4 / 14.2 / 12.1; 5120 x 5120 eight rows of two bits
  // 18.7 / 15.4 / 13.2; the one shape of 30 that loses, 9984 x 2816 with 22 groups in three, 13.4 / 13.3 / 14.1).
  int64_t want = units >= cus ? 1 : cus / units;
  const int k_groups = (int)(n_in / 128);
  if (want > k_groups) want = k_groups;
  const int longest = (int)((k_groups + want - 1) / want);
  p.slices = (k_groups + longest - 1) / longest;
  p.slice_groups = k_groups / p.slices;
  p.accum_words = p.slices > 1 ? 8 + units * p.slices * kXmKSplit * kXmTok * 128 : 0;   // 8 control words in front
  return p;
}

// How often the last slice of a group looks at a word that has not arrived before it gives the row up (NaN).
// A host-side setting so that the give-up path can be exercised without any kernel misbehaving.
static std::atomic<int> g_exl3_poll_limit{1 << 16};
int exl3_set_poll_limit(int limit) { return g_exl3_poll_limit.exchange(limit < 0 ? 0 : limit); }

template <int BITS, int CB, typename XT>
static hipError_t xm_launch(const Exl3Plan& p, const uint16_t* trellis, const uint16_t* suh, const uint16_t* svh,
                            const void* x, void* y, int y_dtype, const void* bias, int bias_dtype, int64_t m,
                            int64_t n_out, int64_t n_in, unsigned long long* accum, hipStream_t s) {
  const dim3 grid((unsigned)p.groups, (unsigned)p.slices, (unsigned)p.row_groups), block(kXmThreads);
  // activations in LDS: the whole slice, or as many whole stages of the ring as fit
  const int cols = 2 * (int)(m < kXmTok ? m : kXmTok), room = kXmLds - XmGeom<BITS>::kRingBytes;
  int chunk = (int)((n_in / 128 + p.slices - 1) / p.slices);
  if (xm_x_bytes(cols, chunk) > room) {
    chunk = (room - xm_x_bytes(cols, 0)) / (xm_x_bytes(cols, 1) - xm_x_bytes(cols, 0));
    chunk = chunk / kXmStageGroups * kXmStageGroups;
  }
  const size_t lds = (size_t)XmGeom<BITS>::kRingBytes + xm_x_bytes(cols, chunk);
  auto kernel = gemv_exl3_mfma_kernel<BITS, CB, XT>;
  static LargeLds configured;
  const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kernel), configured);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, grid, block, lds, s, trellis, suh, svh,
                     static_cast<const XT*>(x), y, y_dtype, bias, bias_dtype, (int)m, (int)n_out, (int)n_in, p.slice_groups,
                     chunk, accum, g_exl3_poll_limit.load(std::memory_order_relaxed));
  return hipGetLastError();
}

template <int BITS, int CB>
static hipError_t xm_launch_x(const Exl3Plan& p, const uint16_t* trellis, const uint16_t* suh, const uint16_t* svh,
                              const void* x, int x_dtype, void* y, int y_dtype, const void* bias, int bias_dtype, int64_t m,
                              int64_t n_out, int64_t n_in, unsigned long long* accum, hipStream_t s) {
  switch (x_dtype) {
    case kF32: return xm_launch<BITS, CB, float>(p, trellis, suh, svh, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, accum, s);
    case kF16: return xm_launch<BITS, CB, f16_tag>(p, trellis, suh, svh, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, accum, s);
    case kBF16: return xm_launch<BITS, CB, bf16_tag>(p, trellis, suh, svh, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, accum, s);
    default: return hipErrorInvalidValue;
  }
}

template <int BITS>
static hipError_t xm_launch_cb(const Exl3Plan& p, const uint16_t* trellis, const uint16_t* suh, const uint16_t* svh,
                               const void* x, int x_dtype, void* y, int y_dtype, const void* bias, int bias_dtype, int64_t m,
                               int64_t n_out, int64_t n_in, int cb, unsigned long long* accum, hipStream_t s) {
  return cb == 0 ? xm_launch_x<BITS, 0>(p, trellis, suh, svh, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, accum, s)
                 : xm_launch_x<BITS, 1>(p, trellis, suh, svh, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, accum, s);
}

hipError_t launch_gemv_exl3_mfma(const Exl3Plan& p, const uint16_t* trellis, const uint16_t* suh,
                                 const uint16_t* svh, const void* x, int x_dtype, void* y, int y_dtype, const void* bias,
                                 int bias_dtype, int64_t m, int64_t n_out, int64_t n_in, int bits, int cb,
                                 unsigned long long* accum, hipStream_t s) {
  if (m == 0 || n_out == 0) return hipSuccess;
  if (p.slices > 1 && !accum) return hipErrorInvalidValue;
  switch (bits) {
    case 1: return xm_launch_cb<1>(p, trellis, suh, svh, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, cb, accum, s);
    case 2: return xm_launch_cb<2>(p, trellis, suh, svh, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, cb, accum, s);
    case 3: return xm_launch_cb<3>(p, trellis, suh, svh, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, cb, accum, s);
    case 4: return xm_launch_cb<4>(p, trellis, suh, svh, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, cb, accum, s);
    case 5: return xm_launch_cb<5>(p, trellis, suh, svh, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, cb, accum, s);
    case 6: return xm_launch_cb<6>(p, trellis, suh, svh, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, cb, accum, s);
    case 7: return xm_launch_cb<7>(p, trellis, suh, svh, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, cb, accum, s);
    case 8: return xm_launch_cb<8>(p, trellis, suh, svh, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, cb, accum, s);
    default: return hipErrorInvalidValue;
  }
}

// ------------------------------------------------------------------------------ workspace
// Sliced launches exchange their sums through tagged 64-bit words behind eight control words (generation count,
// groups finished), all zero before the first launch.  A caller-owned workspace (ttq_workspace.hip) supplies them
// when one is bound; otherwise the library keeps one array per (device, stream): launches on one stream run in
// order and can share it, launches on different streams may overlap and get their own.  Sized for the largest
// plan: launches are sliced only while there are fewer (group, row group) units than compute units.
namespace {
std::mutex g_ws_mutex;
std::unordered_map<uint64_t, unsigned long long*> g_ws;
}  // namespace

// units * slices <= compute units
int64_t exl3_workspace_words() { return 8 + (int64_t)device_num_cus() * kXmKSplit * kXmTok * 128; }

hipError_t exl3_workspace(hipStream_t s, unsigned long long** accum) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  void* bound = nullptr;
  if (caller_workspace_region(kCwExl3Words, (size_t)exl3_workspace_words() * sizeof(unsigned long long), &bound, &e)) {
    *accum = static_cast<unsigned long long*>(bound);
    return e;
  }
  const uint64_t key = ((uint64_t)(uint32_t)dev << 48) ^ (uint64_t)reinterpret_cast<uintptr_t>(s);
  std::lock_guard<std::mutex> lock(g_ws_mutex);
  auto it = g_ws.find(key);
  if (it == g_ws.end()) {
    const size_t bytes = (size_t)exl3_workspace_words() * sizeof(unsigned long long);
    void* p = nullptr;
    e = hipMalloc(&p, bytes);
    if (e != hipSuccess) return e;
    e = hipMemsetAsync(p, 0, bytes, s);     // ordered before the launches that use it: they are all on this stream
    if (e != hipSuccess) {
      (void)hipFree(p);
      return e;
    }
    it = g_ws.emplace(key, static_cast<unsigned long long*>(p)).first;
  }
  *accum = it->second;
  return hipSuccess;
}

// ------------------------------------------------------------------------------ resident workspace
// The same words as a file-scope array in device memory, for the entry point that must not allocate:
// every GPU the library runs on holds its own copy from the moment the code object is loaded there
// until the process ends, zero-initialised; the launches only ever advance its generation count.
// The array's name is only a handle in host code; the address on a device comes from
// hipGetSymbolAddress, asked once per device with that device current.
constexpr int64_t kXmResidentWords = 8 + (int64_t)256 * kXmKSplit * kXmTok * 128;      // 4 MiB
static __device__ __align__(256) unsigned long long scratch[kXmResidentWords];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_resident_mutex;
unsigned long long* g_resident[kMaxDevices] = {};
}  // namespace

int64_t exl3_resident_words() { return kXmResidentWords; }

hipError_t exl3_resident_workspace(unsigned long long** accum) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_resident_mutex);
  if (!g_resident[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_resident[dev] = static_cast<unsigned long long*>(p);
  }
  *accum = g_resident[dev];
  return hipSuccess;
}

// Frees the library-owned arrays (ttq_release_workspaces: nothing that uses them may be in flight or captured).
hipError_t exl3_release_workspaces() {
  std::lock_guard<std::mutex> lock(g_ws_mutex);
  hipError_t first = hipSuccess;
  for (auto& kv : g_ws) {
    const hipError_t e = hipFree(kv.second);
    if (e != hipSuccess && first == hipSuccess) first = e;
  }
  g_ws.clear();
  return first;
}

}  // namespace ttq
