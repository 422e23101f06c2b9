// Choice of the GEMM kernel for a projection, and its launches: the MFMA tiles (gemm_tile.hpp), the
// narrow tiles for few tokens (gemm_narrow.hpp), and for widths that are no multiple of 64 the
// ragged forms of both (gemm_ragged.hip).
#include "gemm_narrow.hpp"
#include "gemm_tile.hpp"

namespace tt {

// ---- host-side tile selection ----
struct TileCfg {
  int bm, bn;
};
static int run_narrow(int mode, const half* x, const half* w, int m, int n, int k,
                      const EpiArgs& ep, hipStream_t stream) {
  switch (mode) {
    case TT_EPI_BIAS: return launch_narrow_mode<TT_EPI_BIAS, false>(x, w, m, n, k, ep, stream);
    case TT_EPI_BIAS_GELU: return launch_narrow_mode<TT_EPI_BIAS_GELU, false>(x, w, m, n, k, ep, stream);
    case TT_EPI_RESID_MASKED: return launch_narrow_mode<TT_EPI_RESID_MASKED, false>(x, w, m, n, k, ep, stream);
    case TT_EPI_MASKED_RESID: return launch_narrow_mode<TT_EPI_MASKED_RESID, false>(x, w, m, n, k, ep, stream);
    default: return launch_narrow_mode<TT_EPI_QKV, false>(x, w, m, n, k, ep, stream);
  }
}

template <int MODE>
static int run_mode(int tile, const half* x, const half* w, int m, int n, int k, const EpiArgs& ep,
                    hipStream_t stream) {
  switch (tile) {
    case 0: return run_tile<256, 256, MODE, 0, 8>(x, w, m, n, k, ep, stream);
    case 1: return run_tile<256, 128, MODE, 0>(x, w, m, n, k, ep, stream);
    case 2: return run_tile<128, 128, MODE, 0>(x, w, m, n, k, ep, stream);
    case 3: return run_tile<128, 64, MODE, 0>(x, w, m, n, k, ep, stream);
    case 6: return run_tile<128, 256, MODE, 1>(x, w, m, n, k, ep, stream);
    case 7: return run_tile<128, 128, MODE, 1>(x, w, m, n, k, ep, stream);
    case 8: return run_tile<128, 64, MODE, 1>(x, w, m, n, k, ep, stream);
    case 9: return run_tile<256, 128, MODE, 1>(x, w, m, n, k, ep, stream);
    case 10: return run_tile<256, 128, MODE, 0, 8>(x, w, m, n, k, ep, stream);
    case 11: return run_tile<64, 64, MODE, 1>(x, w, m, n, k, ep, stream);
    default: return run_tile<64, 64, MODE, 0>(x, w, m, n, k, ep, stream);
  }
}

// index 0: 256 x 256 on 8 waves; index 5: 32 x 32 narrow tiles (gemm_narrow_kernel), chosen for
// grids that leave most CUs idle; indices 6-9: 128 x 256, 128 x 128, 128 x 64, 256 x 128 on the
// register path; index 10: 256 x 128 on 8 waves with a three-stage ring; index 11: 64 x 64 on the
// register path
static const TileCfg kTiles[] = {{256, 256}, {256, 128}, {128, 128}, {128, 64}, {64, 64},
                                 {32, 32},   {128, 256}, {128, 128}, {128, 64}, {256, 128},
                                 {256, 128}, {64, 64}};
constexpr int kNumTiles = (int)(sizeof(kTiles) / sizeof(kTiles[0]));

static int g_tile_override = -1;  // test hook: force one tile configuration

// Tile choice, from measurements on MI355X (M = 8192, N in {1024, 3072, 4096}, K in {1024,
// 4096}; round-robin medians of interleaved runs in one process): the 8-wave 256 x 256 block
// (two waves per SIMD, half the operand traffic per FLOP of 128 x 128) wins when its tiles fill
// whole rounds of the chip, at least two (ffn_in, 8192 x 4096 x 1024: 85 against 87 us with
// GELU, 71 against 76 us with bias only); with 1.5 rounds (QKV, N = 3072) or half a round (N =
// 1024) two 128 x 128 blocks per CU are faster (QKV 57 against 63 us, ffn_out 65 against 95 us).
// Narrower tiles are used when a wider one would leave CUs idle, down to the 32x32 narrow kernel
// for few-token grids.  Exactly one round of 8-wave 256 x 128 tiles with the three-stage ring
// (N = 1024 at M = 8192) beats two 128 x 128 blocks per CU inside the forward, with or without a
// row mask (same-process A/B of whole forwards: C5 -2.5%, C4 with 20% padded rows -3.4%), although
// a GEMM repeated on its own favours the 128-row tiles for out_proj and for padded rows.  The QKV
// projection takes the same tile for whole rounds of it (C5, 8192 x 3072 x 1024: three rounds;
// forward -2.0%) unless its live row count is read on the device (packed rows, whose live tiles
// end inside a round: C4 +0.4 / +0.8% with it).
static int pick_tile(int m, int n, int k, int mode, int cus, bool packed = false) {
  if (g_tile_override >= 0 && g_tile_override < kNumTiles && n % kTiles[g_tile_override].bn == 0)
    return g_tile_override;
  auto tiles = [&](int i) { return (long)((m + kTiles[i].bm - 1) / kTiles[i].bm) * (n / kTiles[i].bn); };
  if (n % 256 == 0 && tiles(0) >= 2 * cus && tiles(0) % cus == 0) return 0;
  // One round of it that leaves at most a fifth of the CUs without a tile, against two 128 x 128 blocks per CU
  // (measured on MI355X: 16384 x 1024 x 1024 with residual 46.3 -> 40.3 us, K 4096 135.5 -> 122, 8192 x 2048 x 1024 with
  // GELU 45.6 -> 43.5, K 512 30.5 -> 30.2; 0.81 of a round with GELU 41.7 -> 40.3, with 0.75 of one 38.6 -> 39.9).
  // Not for packed rows, whose live tiles are fewer, nor for the QKV projection (not measured).
  if (n % 256 == 0 && !packed && mode != TT_EPI_QKV && k >= 512 && tiles(0) <= cus && 5 * tiles(0) >= 4L * cus)
    return 0;
  if (n % 128 == 0 && k >= 1024 &&
      (tiles(10) == cus || (mode == TT_EPI_QKV && !packed && tiles(10) % cus == 0)))
    return 10;
  // One round of 128 x 64 tiles streaming a long K is latency-bound: each CU moves only the bytes
  // it keeps in flight, and the register path keeps two more K stages in flight than the direct
  // copies (measured on MI355X, 4096 x 512 x 2048: 22.3 -> 15.8 us).  On grids of several tiles
  // per CU the direct path is as fast or faster (M = 8192 projections), so it stays there.
  for (int i = 2; i < 4; ++i)
    if (n % kTiles[i].bn == 0 && tiles(i) >= cus) return (i == 3 && k >= 1024) ? 8 : i;
  // Few tokens: 64 x 64 tiles that would fill at most half the CUs become 32 x 32 narrow tiles
  // (measured on MI355X: C1 77 -> 68 us, C2 138 -> 106 us; C1 / C2 ffn_out has 32 / 4 tiles of
  // K = 1024 at 64 x 64, 10-11 us, each CU limited by the bytes it keeps in flight).
  if (2 * tiles(4) <= cus) return 5;
  // 64x64: every N that is a multiple of 64.  About one tile per CU, so as above a long K wants the stages the
  // register path keeps in flight (measured on MI355X, direct copies -> registers: 1000 x 1024 x 4096 32.3 -> 19.2 us,
  // 700 x 1024 x 2048 16.5 -> 9.7, 1500 x 768 x 1536 14.3 -> 12.0, 768 x 1024 x 768 6.4 -> 6.0; K = 512 equal, and
  // at K = 768 with more tiles than CUs 396 x 3072 x 768 7.5 -> 7.7).
  return k >= 1024 || (k >= 768 && tiles(4) <= cus) ? 11 : 4;
}

int device_cus() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
      cus = 256;
  }
  return cus;
}

static bool is_ragged(int n, int k) { return k % kBK != 0 || n % 64 != 0; }

// Tile choice for ragged widths (no width of these models divides a tile, so the partial last tile of
// each row counts as whole): 128 x 128 once its tiles reach every CU (measured on MI355X against
// 64 x 64: 6000 x 1000 x 1000 35.8 -> 29.0 us, 4096 x 1000 x 1000 24.3 -> 18.6; one of ten shapes loses,
// 10000 x 480 x 480 15.7 -> 16.8), 32 x 32 narrow tiles where 64 x 64 would fill at most half the CUs (the
// rule of the aligned widths), else 64 x 64.  Against the vector-ALU kernel these replaced: 1600 x 480 x 160
// (QKV) 58 -> 5 us, 1600 x 640 x 160 91 -> 6 us.
// Rows of 2^22 values and more stay on the narrow tiles, which address each row by a pointer: the others mark
// loads past K by a buffer offset just below 2^31, which has to lie past the tile's 128 rows.
static RaggedTile pick_ragged(int m, int n, int k, int mode, int cus) {
  if (k >= 1 << 22) return RaggedTile::kNarrow;
  auto tiles = [&](int bm, int bn) {
    const long cols = mode == TT_EPI_QKV ? 3 * ((n / 3 + bn - 1) / bn) : (n + bn - 1) / bn;
    return (long)((m + bm - 1) / bm) * cols;
  };
  if (tiles(128, 128) >= cus) return RaggedTile::k128x128;
  if (2 * tiles(64, 64) <= cus) return RaggedTile::kNarrow;
  return RaggedTile::k64x64;
}

bool linear_is_narrow(int m, int n, int k, int mode) {
  if (is_ragged(n, k)) return pick_ragged(m, n, k, mode, device_cus()) == RaggedTile::kNarrow;
  return pick_tile(m, n, k, mode, device_cus()) == 5;
}

int linear_stats_width(int m, int n, int k, int mode) {
  // the narrow ragged kernel (epilogue4); the wider ragged tiles write none (launch_linear)
  if (is_ragged(n, k)) return n % kNarrow == 0 ? kNarrow : 8;
  const int tile = pick_tile(m, n, k, mode, device_cus());
  if (tile == 5) return kNarrow;               // gemm_narrow_kernel: 8 threads per 32 columns
  return kTiles[tile].bn / 2;                  // MFMA tiles: the column range of one wave
}

int launch_linear(const half* x, const half* w, int m, int n, int k, const EpiArgs& ep,
                  hipStream_t stream) {
  TT_REQUIRE(m >= 0 && n > 0 && k > 0, "linear: bad shape m=%d n=%d k=%d", m, n, k);
  TT_REQUIRE(k % 8 == 0 && n % 8 == 0, "linear: N=%d and K=%d must be multiples of 8", n, k);
  TT_REQUIRE((int64_t)n * k < (1LL << 31), "linear: weight of more than 2^31 elements (n=%d k=%d)",
             n, k);
  if (ep.mode == TT_EPI_RESID_MASKED || ep.mode == TT_EPI_MASKED_RESID || ep.mode == TT_EPI_BIAS ||
      ep.mode == TT_EPI_BIAS_GELU)
    TT_REQUIRE(ep.ldy >= n && ep.ldy % 8 == 0, "linear: ldy=%d must be >= N=%d and a multiple of 8",
               ep.ldy, n);
  TT_REQUIRE(ep.mode >= TT_EPI_BIAS && ep.mode <= TT_EPI_QKV, "linear: bad epilogue %d", ep.mode);
  TT_REQUIRE(ep.bias != nullptr && ep.y != nullptr, "linear: null bias/output");
  if (ep.mode == TT_EPI_RESID_MASKED || ep.mode == TT_EPI_MASKED_RESID)
    TT_REQUIRE(ep.resid != nullptr, "linear: residual epilogue needs a residual");
  if (ep.mode == TT_EPI_QKV) {
    TT_REQUIRE(ep.heads > 0 && ep.head_dim > 0 && ep.head_dim % 4 == 0 &&
                   ep.heads * ep.head_dim == ep.d_model && n == 3 * ep.d_model &&
                   (long)ep.batch * ep.seq == m,
               "linear(qkv): inconsistent shape m=%d n=%d batch=%d seq=%d heads=%d hd=%d", m, n,
               ep.batch, ep.seq, ep.heads, ep.head_dim);
  }
  // Heads of 4, 12, 20, ... features run on the narrow tiles at every size: their epilogue stores 4 features
  // at a time, that of the wider tiles 8 of one head.
  // Ragged shapes with an operand that is not 16-byte aligned run on the narrow tiles too, in their staged form.
  const bool unaligned = (((uintptr_t)x | (uintptr_t)w) & 15) != 0;
  const bool narrow = (ep.mode == TT_EPI_QKV && ep.head_dim % 8 != 0) ||
                      (unaligned && is_ragged(n, k) && ep.m_dev == nullptr) || linear_is_narrow(m, n, k, ep.mode);
  if (ep.ln_part != nullptr) {
    TT_REQUIRE(ep.mode == TT_EPI_QKV || ep.mode == TT_EPI_BIAS_GELU || ep.mode == TT_EPI_BIAS,
               "linear: a folded LayerNorm needs a bias / GELU / QKV epilogue");
    TT_REQUIRE(narrow,
               "linear: a folded LayerNorm runs on the narrow kernels only (m=%d n=%d)", m, n);
    TT_REQUIRE(ep.ln_colsum != nullptr && ep.ln_bias != nullptr && ep.ln_slots > 0 &&
                   k % ep.ln_slots == 0 && ep.ln_stride >= ep.ln_slots,
               "linear: bad folded-LayerNorm arguments (slots %d, stride %d, K %d)", ep.ln_slots,
               ep.ln_stride, k);
  }
  if (ep.part_out != nullptr) {
    TT_REQUIRE(ep.mode == TT_EPI_RESID_MASKED || ep.mode == TT_EPI_MASKED_RESID,
               "linear: row statistics are written by the residual epilogues only");
    TT_REQUIRE(ep.ln_stride >= n / linear_stats_width(m, n, k, ep.mode),
               "linear: statistics row stride %d < %d slots", ep.ln_stride,
               n / linear_stats_width(m, n, k, ep.mode));
    TT_REQUIRE(!is_ragged(n, k) || (narrow && ep.ldy == n),
               "linear: row statistics of a ragged shape need the narrow kernel (m=%d n=%d k=%d)", m, n, k);
  }
  if (ep.m_dev != nullptr || ep.rowmap != nullptr) {
    TT_REQUIRE(!narrow,
               "linear: packed variable-length rows run on the MFMA tiles only (m=%d n=%d k=%d)", m,
               n, k);
    TT_REQUIRE(ep.ln_part == nullptr && ep.part_out == nullptr,
               "linear: packed rows take no folded LayerNorm");
    TT_REQUIRE(ep.mode != TT_EPI_QKV || (ep.m_dev != nullptr && ep.rowmap != nullptr),
               "linear(qkv): packed rows need both the row count and the row map");
  }
  if (m == 0) return TT_OK;
  if (narrow && unaligned) return run_ragged(RaggedTile::kNarrowStaged, x, w, m, n, k, ep, stream);
  if (is_ragged(n, k))
    return run_ragged(narrow ? RaggedTile::kNarrow : pick_ragged(m, n, k, ep.mode, device_cus()), x, w, m, n, k, ep,
                      stream);
  if (narrow) return run_narrow(ep.mode, x, w, m, n, k, ep, stream);
  const int tile = pick_tile(m, n, k, ep.mode, device_cus(), ep.m_dev != nullptr);
  switch (ep.mode) {
    case TT_EPI_BIAS: return run_mode<TT_EPI_BIAS>(tile, x, w, m, n, k, ep, stream);
    case TT_EPI_BIAS_GELU: return run_mode<TT_EPI_BIAS_GELU>(tile, x, w, m, n, k, ep, stream);
    case TT_EPI_RESID_MASKED: return run_mode<TT_EPI_RESID_MASKED>(tile, x, w, m, n, k, ep, stream);
    case TT_EPI_MASKED_RESID: return run_mode<TT_EPI_MASKED_RESID>(tile, x, w, m, n, k, ep, stream);
    default: return run_mode<TT_EPI_QKV>(tile, x, w, m, n, k, ep, stream);
  }
}

}  // namespace tt

extern "C" int tt_gemm_tile_override(int index) {
  TT_REQUIRE(index >= -1 && index < tt::kNumTiles, "gemm_tile_override: index %d out of [-1, %d)",
             index, tt::kNumTiles);
  tt::g_tile_override = index;
  return TT_OK;
}

extern "C" int tt_linear_fwd(const void* x, const void* w, const void* bias, const void* residual,
                             const uint8_t* valid, void* y, int m, int n, int k, int epilogue,
                             int batch, int seq, int heads, void* stream) {
  TT_REQUIRE(x && w && bias && y, "linear: null pointer");
  tt::EpiArgs ep{};
  ep.bias = (const tt::half*)bias;
  ep.resid = (const tt::half*)residual;
  ep.valid = valid;
  ep.y = (tt::half*)y;
  ep.ldy = n;
  ep.mode = epilogue;
  ep.batch = batch;
  ep.seq = seq;
  ep.heads = heads;
  ep.d_model = n / 3;
  ep.head_dim = heads > 0 ? (n / 3) / heads : 0;
  return tt::launch_linear((const tt::half*)x, (const tt::half*)w, m, n, k, ep,
                           (hipStream_t)stream);
}
