// Prefill GEMM for Q4_K, Q6_K and Q8_0 weights on gfx950, producer/consumer form (kernel: ttq_gemm_pc.h):
// tile choice, split along K and its workspace, and the launchers behind ttq_gemm_* / ttq_linear_forward.
#include "ttq_gemm_pc.h"

#include <stdio.h>

namespace ttq {

// x: the activations, or (tile_if_packed >= 0) their packed copy and the tile's index for launch_gemm_packed
template <int FMT, int MB, int NJ, bool FUSE>
static hipError_t launch_pc_tile(const uint8_t* wb, const uint16_t* x, void* y, int y_dtype, const void* bias,
                                 int bias_dtype, int64_t m, int64_t n_out, int64_t n_in, int splits, int tile_if_packed,
                                 hipStream_t s, bool x_f16 = false, const float* row_scale = nullptr) {
  PcSplit sp{1, 0, nullptr, nullptr};
  if (!FUSE && splits > 1) {
    // (the chooser has checked that the blocks of a row divide evenly and that the counters suffice)
    constexpr int BO = NJ * 16, BM = pc_bm(MB);
    const size_t units = (size_t)((n_out + BO - 1) / BO) * (size_t)((m + BM - 1) / BM) * 4;
    void* part = nullptr;
    void* cnt = nullptr;
    hipError_t e = stream_workspace(kWsGemmPartials, s, units * splits * (size_t)(MB * NJ * 1024), &part);
    if (e == hipSuccess) e = stream_workspace(kWsGemmCounters, s, (size_t)kPcMaxCounters * 4, &cnt, true);
    if (e != hipSuccess) return e;
    sp.splits = splits;
    sp.partials = static_cast<float*>(part);
    sp.counters = static_cast<uint32_t*>(cnt);
  }
  if (tile_if_packed >= 0)
    return launch_gemm_packed(FMT, FUSE, tile_if_packed, wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, sp, s, x_f16, row_scale);
  return launch_pc_grid<FMT, MB, NJ, FUSE>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, sp, s);
}

// Tile choice.  A workgroup owns 64 * mb rows x 16 * nj columns (8 * nj outputs when fused).
struct PcTile { int mb, nj; };
static const PcTile kPcTiles[] = {{4, 7}, {4, 4}, {2, 7}, {2, 4}, {1, 7}, {1, 4}};
constexpr int kPcTileCount = 6;
static const int kPcSplits[] = {1, 2, 4, 7, 8};

// Whether a call comes here at all: rounds of workgroups x (64-k steps x time per step of the tile + a fixed cost per workgroup).
// The kernels that compete (few rows, decode) were weighed against these figures, and which calls may have their weights
// rounded follows from them, so they stay when the kernels behind them get faster.
struct PcRouteTile { int mb, nj; float step_us; };
static const PcRouteTile kPcRouteTiles[] = {{4, 7, 0.87f}, {4, 4, 0.68f}, {2, 7, 0.585f}, {2, 4, 0.55f}, {1, 7, 0.46f}, {1, 4, 0.52f}};
struct PcRoute { int tile, splits; float cost_us; };
static PcRoute pc_route(int64_t m, int64_t n_out, int64_t n_in) {
  const int cus = device_num_cus();
  const int64_t blocks = n_in / 256;
  PcRoute best{0, 1, 1e30f};
  for (int i = 0; i < kPcTileCount; i++) {
    const PcRouteTile& t = kPcRouteTiles[i];
    const int64_t bm = pc_bm(t.mb), nt = (n_out + t.nj * 16 - 1) / (t.nj * 16), mt = (m + bm - 1) / bm, tiles = nt * mt;
    for (int sp : kPcSplits) {
      if (sp > 1 && (blocks % sp != 0 || blocks / sp < 2 || tiles * sp > cus || tiles * 4 > kPcMaxCounters)) continue;
      const int64_t rounds = (tiles * sp + cus - 1) / cus;
      float cost = (float)rounds * ((float)(n_in / 64 / sp) * t.step_us + 6.f);
      if (sp > 1) {      // 2 + copies trips to the memory side (3 for two copies), the partial sums twice at 4 TB/s
        const float trip = 0.9f + 0.06f * (float)(t.mb * t.nj);
        cost += (sp == 2 ? 3.f : 2.f + (float)sp) * trip + 2.f * (float)sp * (float)(mt * bm) * (float)(nt * t.nj * 16) * 4.f / 4.0e6f;
      }
      if (cost < best.cost_us * 0.999f) best = PcRoute{i, sp, cost};
    }
  }
  return best;
}

// What a launch takes, us, by format, by where the activations are read (row-major through LDS, or a packed copy) and by tile:
//   rounds of workgroups * (64-k steps * (step + full * share of the compute units at work) + round) + launch
//   + (split along K) trips0 + trips1 * copies + bytes of the partial sums, written and read, * traffic / 4 TB/s,
// fitted to 150000 timed launches of 19000 layers: 768 .. 8192 wide models at 65 .. 4096 rows, and any 256 .. 120000 x 256 .. 14336 at 20 and
// more, every tile, one to eight copies, both ways to the activations, 256 compute units; standard deviation 6 to 12 percent for tiles
// of 128 and 64 rows, 9 to 17 for 256 (profiles/gemm_tile_times.md has the fit and what it leaves over).  What these estimates choose is
// 1 to 4 percent above the fastest launch of all (geometric means, per format and type) and 5 to 10 percent below what the model above
// chooses, which has one time per step for all formats; its choice is kept where the two are within five percent (slower than it by more
// than that: 0.1 to 1.6 percent of the layers).  A short grid is split along K while all copies fit one round: the length of a short round is
// the latency of its K loop.  The fused gate||up form goes by the row-major times of Q4_K, although its tiles have half the outputs and an
// epilogue of their own: over 1384 random layers its choice is 0.6 to 1.5 percent above the fastest tile, the model above 2.7 to 4.2.
struct PcCost { float step, full, round, launch, trips0, trips1, traffic; };
static const PcCost kPcCosts[3][2][kPcTileCount] = {      // [format: Q8_0, Q4_K, Q6_K][packed][tile]
    {  // Q8_0
        {{0.663f, 0.201f, 6.98f, 4.21f, 3.17f, 7.70f, 0.57f}, {0.569f, 0.098f, 2.69f, 6.17f, 2.17f, 4.28f, 0.57f}, {0.497f, 0.111f, 4.56f, 4.79f, 1.97f, 1.14f, 0.58f},
         {0.410f, 0.065f, 1.85f, 6.01f, 1.46f, 0.82f, 0.69f}, {0.474f, 0.056f, 3.26f, 4.88f, 0.95f, 0.80f, 0.89f}, {0.352f, 0.039f, 1.52f, 5.63f, 0.89f, 0.66f, 1.12f}},
        {{0.617f, 0.184f, 11.29f, 2.55f, 2.79f, 1.84f, 0.51f}, {0.461f, 0.103f, 6.65f, 3.50f, 2.20f, 1.31f, 0.52f}, {0.511f, 0.105f, 3.53f, 6.88f, 1.85f, 1.08f, 0.48f},
         {0.380f, 0.012f, 1.85f, 6.43f, 1.44f, 0.78f, 0.76f}, {0.473f, 0.055f, 2.42f, 6.14f, 1.16f, 0.74f, 0.72f}, {0.319f, 0.f, 1.29f, 6.32f, 1.02f, 0.57f, 1.45f}},
    },
    {  // Q4_K
        {{0.567f, 0.200f, 6.74f, 4.18f, 2.38f, 7.64f, 0.59f}, {0.449f, 0.112f, 2.65f, 5.65f, 1.48f, 4.21f, 0.60f}, {0.400f, 0.110f, 2.59f, 6.27f, 1.22f, 0.98f, 0.75f},
         {0.295f, 0.071f, 1.83f, 5.58f, 0.77f, 0.67f, 0.80f}, {0.356f, 0.061f, 1.99f, 5.80f, 0.74f, 0.69f, 0.85f}, {0.230f, 0.052f, 1.41f, 5.52f, 0.52f, 0.56f, 0.77f}},
        {{0.461f, 0.222f, 10.20f, 3.11f, 1.49f, 1.95f, 0.66f}, {0.333f, 0.115f, 5.74f, 3.75f, 1.75f, 1.25f, 0.55f}, {0.374f, 0.060f, 2.44f, 7.43f, 1.14f, 1.03f, 0.75f},
         {0.245f, 0.037f, 1.42f, 6.46f, 1.00f, 0.67f, 0.83f}, {0.343f, 0.f, 1.62f, 6.79f, 0.53f, 0.59f, 1.33f}, {0.205f, 0.f, 1.03f, 6.02f, 0.82f, 0.50f, 1.22f}},
    },
    {  // Q6_K
        {{0.735f, 0.164f, 8.38f, 3.99f, 1.96f, 7.68f, 0.57f}, {0.567f, 0.091f, 3.53f, 6.07f, 0.99f, 4.18f, 0.54f}, {0.541f, 0.097f, 3.80f, 6.34f, 0.91f, 0.99f, 0.66f},
         {0.400f, 0.068f, 2.53f, 5.76f, 0.68f, 0.62f, 0.74f}, {0.503f, 0.049f, 3.11f, 5.72f, 0.39f, 0.68f, 0.84f}, {0.336f, 0.047f, 2.06f, 5.55f, 0.20f, 0.51f, 1.00f}},
        {{0.631f, 0.168f, 8.51f, 4.39f, 2.39f, 1.80f, 0.55f}, {0.440f, 0.095f, 5.06f, 4.67f, 1.75f, 1.12f, 0.56f}, {0.528f, 0.017f, 3.16f, 7.74f, 0.76f, 0.95f, 0.79f},
         {0.357f, 0.012f, 2.07f, 6.59f, 0.79f, 0.64f, 0.85f}, {0.460f, 0.f, 2.25f, 7.47f, 0.67f, 0.64f, 0.94f}, {0.295f, 0.f, 1.71f, 6.32f, 0.47f, 0.50f, 1.21f}},
    },
};

struct PcChoice { int tile, splits; bool packed; float cost_us; };

// The pass that makes the packed copy: 2.5 us and its bytes, fp32 rows (a factor per row first) 5.5.
static float pc_pack_us(int x_dtype, int64_t m, int64_t n_in) {
  return x_dtype == kF32 ? 5.5f + (float)(m * n_in * 10) / 5.0e6f : 2.5f + (float)(m * n_in * 4) / 5.0e6f;
}

// The tile, the copies along K and the way to the activations of a launch.  Only bf16 activations can be read as they are, and the
// fused gate||up form must (its epilogue does not fit beside the packed kernel's three steps of A fragments).  copied: the packed copy is
// there already (a block of rows of a longer launch), so it is read and costs nothing.
static PcChoice pc_choose(int format, int x_dtype, int64_t m, int64_t n_out, int64_t n_in, bool fuse, bool copied = false) {
  static const int forced = dev_knob("TTQ_GEMM_TILE", -1);
  static const int forced_splits = dev_knob("TTQ_GEMM_SPLITS", 0);   // A/B: 1 = never split, n = n ways where possible
  static const int forced_packed = dev_knob("TTQ_GEMM_PACKED", -1);  // A/B: 0 never, 1 always
  const int cus = device_num_cus();
  const int64_t blocks = n_in / 256;
  PcChoice best{0, 1, false, 1e30f}, before = best;
  const PcRoute route = fuse ? PcRoute{-1, 1, 0.f} : pc_route(m, n_out, n_in);
  const bool route_packed = copied || x_dtype != kBF16 || (kPcTiles[route.tile < 0 ? 0 : route.tile].mb == 4 && route.cost_us >= 45.f);
  for (int packed = fuse || (x_dtype == kBF16 && !copied) ? 0 : 1; packed <= (fuse ? 0 : 1); packed++) {
    if (!fuse && !copied && x_dtype == kBF16 && forced_packed >= 0 && forced_packed != packed) continue;
    const float pack = packed && !copied ? pc_pack_us(x_dtype, m, n_in) : 0.f;
    for (int i = 0; i < kPcTileCount; i++) {
      if (forced >= 0 && forced < kPcTileCount && i != forced) continue;
      const PcTile& t = kPcTiles[i];
      const PcCost& c = kPcCosts[format][packed][i];
      const int64_t bo = fuse ? t.nj * 8 : t.nj * 16, bm = pc_bm(t.mb);
      const int64_t nt = (n_out + bo - 1) / bo, mt = (m + bm - 1) / bm, tiles = nt * mt;
      for (int sp : kPcSplits) {
        if (forced_splits > 0 && sp != 1 && sp != forced_splits) continue;
        if (sp > 1 && (fuse || blocks % sp != 0 || blocks / sp < 2 || tiles * sp > cus || tiles * 4 > kPcMaxCounters)) continue;
        // (beyond four rounds the last one overlaps the others)
        const float full = (float)(tiles * sp) / (float)cus;
        const float rounds = full > 4.f ? full + 0.5f : (float)((tiles * sp + cus - 1) / cus);
        const float step = c.step + c.full * (full < rounds ? full / rounds : 1.f);
        float cost = pack + rounds * ((float)(n_in / 64 / sp) * step + c.round) + c.launch;
        if (sp > 1)
          cost += c.trips0 + c.trips1 * (float)(sp > 2 ? sp : 1) + c.traffic * 2.f * (float)sp * (float)(mt * bm) * (float)(nt * bo) / 1.0e6f;
        if (i == route.tile && sp == route.splits && (packed != 0) == route_packed) before = PcChoice{i, sp, packed != 0, cost};
        // (long launches of the K formats read a packed copy: the estimates are least sure of short rows, 20112 x 1024 Q4_K at 4079 rows
        // 222 us without it and 208; and of Q8_0 beyond 4096 rows, but for few columns, where a packed block of 8192 rows leaves compute
        // units idle: 5184 x 512 at 16871 rows 269 / 174, 9136 x 256 at 5868 102 / 90, but 512 x 4096 at 20000 0.6 to 0.9 of the time)
        if (!fuse && !packed && forced_packed < 0 && cost >= 45.f && (format != kQ8_0 || (m > 4096 && n_out > 1024))) continue;
        if (cost < best.cost_us * 0.999f || (forced_splits > 0 && sp == forced_splits && best.splits != sp))
          best = PcChoice{i, sp, packed != 0, cost};
      }
    }
  }
  // (short rows of very many weight rows: the estimates' other weak place, Q8_0 108544 x 256 at 712 rows 116 -> 165 us, Q6_K
  // 43392 x 256 at 104 fp16 rows 15.4 -> 18.2, Q4_K 39552 x 512 at 92 16.6 -> 18.4: the model above decides)
  // (long launches one after the other run at the clock that the power limit leaves, where tiles that dequantize a weight for fewer
  // products lose what they win alone: a block of 4096 / 14336 at 4096 rows with 64-column tiles in three of its layers 1860 us
  // against 1830, each of those layers alone 2 to 5 percent faster)
  // (beyond 4096 rows, which the fit has not seen, and for 256x112 tiles of Q4_K and Q8_0 from 2048 on, whose time it puts too high,
  // 16-bit rows change over where the new choice is a fifth ahead: of 8200 such calls 11 percent were more than 5 percent slower than the
  // earlier choice, by up to half, and 0.7 are; Q4_K 34944 x 1024 at 5993 rows 615 / 513 us, fp16 12288 x 1024 at 3905 161 / 133, Q8_0
  // fp16 512 x 4096 at 6338 82 / 68)
  float margin = n_in <= (format == kQ8_0 ? 1024 : 512) && n_out > 16384 ? 0.f : (before.cost_us >= 100.f ? 0.9f : 0.95f);
  const bool unsure = m > 4096 || (m > 2048 && format != kQ6_K && before.tile == 0 && best.tile != 0);
  if (unsure && x_dtype != kF32 && margin > 0.8f) margin = 0.8f;
  // (up to 64 rows, few of which the fit has seen, one copy of smaller tiles instead of two: Q4_K 14048 x 8192 at 62 rows 44 / 39, 49 of 55
  // such calls that were within a tenth 2 to 13 percent slower)
  if (m <= 64 && before.splits > 1 && best.splits == 1 && margin > 0.9f) margin = 0.9f;
  return before.cost_us < 1e29f && forced < 0 && forced_splits == 0 && best.cost_us > margin * before.cost_us ? before : best;
}

constexpr int64_t kPackRows = 8192;         // rows packed (and multiplied) at a time

// the launch of `rows` of the m rows of a call that goes through the packed copy
static PcChoice pc_choose_block(const PcChoice& whole, int64_t rows, int format, int x_dtype, int64_t m, int64_t n_out, int64_t n_in) {
  return rows == m ? whole : pc_choose(format, x_dtype, rows, n_out, n_in, false, true);
}

static size_t pc_partials_bytes(const PcChoice& c, int64_t m, int64_t n_out) {
  if (c.splits <= 1) return 0;
  const PcTile& t = kPcTiles[c.tile];
  const int64_t nt = (n_out + t.nj * 16 - 1) / (t.nj * 16), mt = (m + pc_bm(t.mb) - 1) / pc_bm(t.mb);
  return (size_t)(nt * mt * 4) * (size_t)c.splits * (size_t)(t.mb * t.nj * 1024);
}

// bytes of partial sums that a call of this shape keeps in the workspace at a time (0: not split along K)
size_t gemm_pc_partials_bytes(int format, int x_dtype, int64_t m, int64_t n_out, int64_t n_in) {
  if (m <= 0 || n_out <= 0 || n_in < 256) return 0;
  const PcChoice whole = pc_choose(format, x_dtype, m, n_out, n_in, false);
  if (!whole.packed || m <= kPackRows) return pc_partials_bytes(whole, m, n_out);
  size_t most = 0;
  for (int64_t rows : {kPackRows, m % kPackRows}) {
    const size_t bytes = rows ? pc_partials_bytes(pc_choose_block(whole, rows, format, x_dtype, m, n_out, n_in), rows, n_out) : 0;
    most = bytes > most ? bytes : most;
  }
  return most;
}

// Rough time of the GEMM for this shape (microseconds), for callers that can also run the
// operator as a few GEMV passes.  The Q6_K and Q8_0 producers are slower than the Q4_K one.
float gemm_pc_estimate_us(int format, int64_t m, int64_t n_out, int64_t n_in) {
  return pc_route(m, n_out, n_in).cost_us * (format == kQ8_0 ? 1.9f : (format == kQ6_K ? 1.4f : 1.f)) + 2.f;
}

// The fitted time, for the choice against chunks of the few-row kernel.  It errs most for one or two short row tiles, so up to 128 rows
// the tiles have to be a tenth ahead, Q8_0 a quarter, and long rows of weights go by the model above alone.  Where it still sent calls to tiles
// that were more than 3 percent slower there than in chunks (of 10600 timed calls that it had moved), the model above decides too:
//   Q6_K, 65 to 128 rows, more than 4096 outputs and values: two thirds of them (fp16 5440 x 6400 at 68 rows 39 us in chunks, 55 in tiles)
//   Q6_K, 129 to 184 rows, a full tile and the rest of the next: over rows of more than 6144 values, up to 144 rows of 4096, a fifth to a
//     half (bf16 192 x 6400 at 141 39 / 50)
//   Q8_0, 97 to 128 rows, 1025 to 4096 outputs, more than 2048 values, if not a third ahead: a sixth to a half (fp16 2608 x 6400 at 122 35 / 43)
// (altogether 9.0 percent were slower, 0.7 are; the mean over all of them is 0.848 of the time in chunks, 0.844 before.)
float gemm_pc_cost_us(int format, int x_dtype, int64_t m, int64_t n_out, int64_t n_in) {
  if (m <= 128 && n_in > 8192) return 1e30f;
  if (format == kQ6_K && (m <= 128 ? n_out > 4096 && n_in > 4096 : m <= 184 && n_in > (m <= 144 ? 4096 : 6144))) return 1e30f;
  const bool q8_gap = format == kQ8_0 && m > 96 && n_out > 1024 && n_out <= 4096 && n_in > 2048;
  const float margin = m > 128 ? 1.f : (q8_gap ? 1.35f : (format == kQ8_0 ? 1.25f : 1.1f));
  return pc_choose(format, x_dtype, m, n_out, n_in, false).cost_us * margin;
}

// Whether that model would divide a launch along K.
bool gemm_pc_splits_k(int64_t m, int64_t n_out, int64_t n_in) { return pc_route(m, n_out, n_in).splits > 1; }

template <int FMT, bool FUSE>
static hipError_t launch_pc_rows(const PcChoice& c, int tile_if_packed, const uint8_t* wb, const uint16_t* x, void* y,
                                 int y_dtype, const void* bias, int bias_dtype, int64_t m, int64_t n_out, int64_t n_in,
                                 hipStream_t s, bool x_f16 = false, const float* row_scale = nullptr) {
  const int p = tile_if_packed;
  switch (c.tile) {
    case 0: return launch_pc_tile<FMT, 4, 7, FUSE>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, c.splits, p, s, x_f16, row_scale);
    case 1: return launch_pc_tile<FMT, 4, 4, FUSE>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, c.splits, p, s, x_f16, row_scale);
    case 2: return launch_pc_tile<FMT, 2, 7, FUSE>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, c.splits, p, s, x_f16, row_scale);
    case 3: return launch_pc_tile<FMT, 2, 4, FUSE>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, c.splits, p, s, x_f16, row_scale);
    case 4: return launch_pc_tile<FMT, 1, 7, FUSE>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, c.splits, p, s, x_f16, row_scale);
    default: return launch_pc_tile<FMT, 1, 4, FUSE>(wb, x, y, y_dtype, bias, bias_dtype, m, n_out, n_in, c.splits, p, s, x_f16, row_scale);
  }
}

static void say_pc(const char* kernel, const PcChoice& c) {
  const PcTile& t = kPcTiles[c.tile];
  char copies[16] = "";
  if (c.splits > 1) snprintf(copies, sizeof copies, " k/%d", c.splits);
  route_say("%s %dx%d%s%s", kernel, pc_bm(t.mb), t.nj * 16, copies, c.packed ? " packed" : "");
}

// x in x_dtype: any type when the launch goes through the packed copy (the packing pass
// rounds to bf16, or -- keep_f16 -- leaves fp16 activations as they are for the fp16 form of the kernel).
template <int FMT, bool FUSE>
static hipError_t launch_pc_fmt(const uint8_t* wb, const void* x, int x_dtype, void* y, int y_dtype, const void* bias,
                                int bias_dtype, int64_t m, int64_t n_out, int64_t n_in, hipStream_t s,
                                int f16_mode = 0) {      // 1: fp16 activations stay fp16; 2: fp32 activations as scaled fp16
  const PcChoice whole = pc_choose(FMT, x_dtype, m, n_out, n_in, FUSE);
  if (!whole.packed)
    return launch_pc_rows<FMT, FUSE>(whole, -1, wb, static_cast<const uint16_t*>(x), y, y_dtype, bias, bias_dtype, m, n_out,
                                     n_in, s);
  const int64_t block_rows = m < kPackRows ? m : kPackRows;
  void* ws = nullptr;
  // (fp32 activations as scaled fp16: the rows' inverse factors follow the packed copy)
  const size_t copy_bytes = (gemm_packed_activation_bytes(block_rows, n_in) + 255) & ~(size_t)255;
  hipError_t e = stream_workspace(kWsPackedActivations, s, copy_bytes + (f16_mode == 2 ? (size_t)block_rows * 4 : 0), &ws);
  if (e != hipSuccess) return e;
  float* row_scale = f16_mode == 2 ? reinterpret_cast<float*>(static_cast<char*>(ws) + copy_bytes) : nullptr;
  const int64_t xsize = x_dtype == kF32 ? 4 : 2, ysize = y_dtype == kF32 ? 4 : 2;
  for (int64_t r0 = 0; r0 < m; r0 += kPackRows) {
    const int64_t rows = m - r0 < kPackRows ? m - r0 : kPackRows;
    if (f16_mode == 2)
      e = launch_gemm_pack_activations_scaled(static_cast<const float*>(x) + r0 * n_in, static_cast<uint16_t*>(ws), row_scale,
                                              rows, n_in, s);
    else
      e = launch_gemm_pack_activations(static_cast<const char*>(x) + r0 * n_in * xsize, x_dtype, static_cast<uint16_t*>(ws),
                                       rows, n_in, s, f16_mode == 1);
    if (e != hipSuccess) return e;
    const PcChoice c = pc_choose_block(whole, rows, FMT, x_dtype, m, n_out, n_in);
    e = launch_pc_rows<FMT, FUSE>(c, c.tile, wb, static_cast<const uint16_t*>(ws), static_cast<char*>(y) + r0 * n_out * ysize,
                                  y_dtype, bias, bias_dtype, rows, n_out, n_in, s, f16_mode != 0, row_scale);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// 112- and 64-column tiles are built in this form: with 128 columns the consumers' 128
// accumulator registers plus the fragment rings do not fit the 168 registers a wavefront gets
// when twelve of them share a CU.
bool gemm_pc_supported(int format, int64_t m, int64_t n_out, int64_t n_in, int bn) {
  static const int disabled = dev_knob("TTQ_GEMM_NO_PC", 0);
  // activation byte offsets are 32-bit in the kernel; a step loop iteration is 256 k
  return !disabled && (format == kQ4_K || format == kQ6_K || format == kQ8_0) && bn == 112 &&
         m * n_in * 2 < ((int64_t)1 << 32) && n_out > 0 && n_in > 0 && n_in % 256 == 0;
}

// x: bf16 activations; or (x_dtype fp16 / fp32) activations that may be rounded to bf16: those always go through the
// packed copy, whose packing pass does the rounding; or (f16_native) the fp16 form of the kernel, which rounds the
// weights to fp16 and multiplies on the fp16 matrix cores: fp16 activations stay as they are in the packed copy, fp32
// activations become fp16 there after every row has been scaled by a power of two (undone in the epilogue).
hipError_t launch_gemm_pc_x(int format, const void* w, const void* x, int x_dtype, void* y, int y_dtype,
                            const void* bias, int bias_dtype, int64_t m, int64_t n_out, int64_t n_in, hipStream_t s,
                            bool f16_native) {
  if (m == 0 || n_out == 0) return hipSuccess;
  if (y_dtype != kBF16 && y_dtype != kF32 && y_dtype != kF16) return hipErrorInvalidValue;
  if (f16_native && x_dtype != kF16 && x_dtype != kF32) return hipErrorInvalidValue;
  const PcChoice c = pc_choose(format, x_dtype, m, n_out, n_in, false);
  const bool packed = c.packed;
  if (route_probe(f16_native ? (x_dtype == kF32 ? kRouteGemmPcF32ScaledF16 : kRouteGemmPcF16)
                             : (x_dtype != kBF16 ? kRouteGemmPcBf16Copy
                                                 : (c.splits > 1 ? (packed ? kRouteGemmPcPackedSplitK : kRouteGemmPcSplitK)
                                                                 : (packed ? kRouteGemmPcPacked : kRouteGemmPc))))) {
    say_pc("gemm_pc", packed ? pc_choose_block(c, m < kPackRows ? m : kPackRows, format, x_dtype, m, n_out, n_in) : c);
    if (packed && m > kPackRows && m % kPackRows) say_pc("gemm_pc", pc_choose_block(c, m % kPackRows, format, x_dtype, m, n_out, n_in));
    return hipSuccess;
  }
  const uint8_t* wb = static_cast<const uint8_t*>(w);
  switch (format) {
    case kQ4_K: return launch_pc_fmt<kQ4_K, false>(wb, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, f16_native ? (x_dtype == kF32 ? 2 : 1) : 0);
    case kQ6_K: return launch_pc_fmt<kQ6_K, false>(wb, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, f16_native ? (x_dtype == kF32 ? 2 : 1) : 0);
    case kQ8_0: return launch_pc_fmt<kQ8_0, false>(wb, x, x_dtype, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s, f16_native ? (x_dtype == kF32 ? 2 : 1) : 0);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_gemm_pc(int format, const void* w, const uint16_t* x_bf16, void* y, int y_dtype,
                          const void* bias, int bias_dtype, int64_t m, int64_t n_out, int64_t n_in,
                          hipStream_t s) {
  return launch_gemm_pc_x(format, w, x_bf16, kBF16, y, y_dtype, bias, bias_dtype, m, n_out, n_in, s);
}

// bytes of the packed copy a launch of this shape takes from the workspace (0: it reads X itself)
size_t gemm_pc_packed_bytes(int format, int64_t m, int64_t n_out, int64_t n_in, int x_dtype) {
  if (m <= 0 || n_out <= 0 || n_in < 256) return 0;
  if (!pc_choose(format, x_dtype, m, n_out, n_in, false).packed) return 0;
  const int64_t rows = m < kPackRows ? m : kPackRows;
  // (fp32 activations: room for a factor per row behind the copy, whichever way they are narrowed)
  return ((gemm_packed_activation_bytes(rows, n_in) + 255) & ~(size_t)255) + (x_dtype == kF32 ? (size_t)rows * 4 : 0);
}


// gate||up projection + silu_and_mul in the GEMM epilogue: w holds 2*n_ff rows (gate rows first),
// y is (m, n_ff).  Q4_K weights.
hipError_t launch_gemm_pc_silu_mul(const void* w, const uint16_t* x_bf16, void* y, int y_dtype, const void* bias,
                                   int bias_dtype, int64_t m, int64_t n_ff, int64_t n_in, hipStream_t s) {
  if (m == 0 || n_ff == 0) return hipSuccess;
  if (y_dtype != kBF16 && y_dtype != kF32) return hipErrorInvalidValue;
  if (route_probe(kRouteGemmPc)) {
    say_pc("gemm_pc_silu_mul", pc_choose(kQ4_K, kBF16, m, n_ff, n_in, true));
    return hipSuccess;
  }
  return launch_pc_fmt<kQ4_K, true>(static_cast<const uint8_t*>(w), x_bf16, kBF16, y, y_dtype, bias, bias_dtype, m, n_ff,
                                    n_in, s);
}

}  // namespace ttq
