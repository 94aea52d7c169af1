// variants.cpp -- the variant table and the calibrated cost model
// (declarations and the role of each in variants.h).
#include "variants.h"

#include <algorithm>
#include <cmath>

#include "wtc/wtc_hip.h"

namespace wtc {

namespace {

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

int in_bytes(int dt) { return dt == WTC_DTYPE_F32 ? 4 : (dt == WTC_DTYPE_FP8_E4M3 ? 1 : 2); }
int out_bytes(int dt) { return dt == WTC_DTYPE_F32 ? 4 : 2; }
bool valid_in(int dt) { return dt >= WTC_DTYPE_F32 && dt <= WTC_DTYPE_FP8_E4M3; }

constexpr unsigned bit(int path) { return 1u << path; }
constexpr unsigned kTilePaths = bit(WTC_PATH_EXCHANGE) | bit(WTC_PATH_SPLIT) | bit(WTC_PATH_UNFUSED);
constexpr unsigned kSplitPaths = bit(WTC_PATH_SPLIT) | bit(WTC_PATH_UNFUSED);

// ---- calibration -------------------------------------------------------------
// The model: a call costs its kernels' back-to-back launch time, plus the
// tile kernel's waves times one tile's cycles at the clock the chip holds
// under that load, plus the passes that stream the output (split: the
// rescale; unfused: four f32 row passes), plus the row exchange (a fixed
// part and a part per column tile of a row block).  The full waves (every
// CU busy) and the last, partial one are priced separately.  One tile's
// cycles are a fixed part (first loads and epilogue) and, per 128 bytes of
// K, the variant's own cycles plus the cycles its A and B bytes add as they
// stream in (bytes of every active tile over a chip-wide rate).
//
// The constants were fitted (least squares on the log of the time) to
// back-to-back timings of every variant on every path over the 60 shapes
// of calibrate.py on MI355X.  Fitted on three of its four shape sets and
// scored on the fourth, in turn, the fused ranking lost 0.78 % on average
// against the measured fastest choice (the hand-written rules it replaces:
// 5.3 %).
struct TileCal {
  double kt_cyc;        // own cycles per k-tile
  double fixed_cyc[3];  // per tile: exchange, split, logits epilogues
};
// [tile variant][0: 16-bit, 1: fp8, 2: f32, 3: f32 64 x 64]; fixed parts shared
// across 16-bit and fp8 inputs.  Rows: kVarTile128, kVarTile128Loaders, kVarTile256, kVarTile256x256.
const TileCal kTileCal[4][4] = {
    /* kVarTile128 */ {{629.84, {3269.7, 4715.4, 0}}, {632.56, {3269.7, 4715.4, 0}}, {2169.61, {2450.2, 2450.2, 0}}, {755.79, {4185.3, 0, 0}}},
    /* kVarTile128Loaders */ {{560.75, {3641.3, 5208.9, 254}}, {550.35, {3641.3, 5208.9, 254}}, {0, {0, 0, 0}}},
    /* kVarTile256 */ {{1153.19, {0, 9714.1, 0}}, {1272.56, {0, 9714.1, 0}}, {0, {0, 0, 0}}},
    /* kVarTile256x256 */ {{2026.70, {0, 18521.3, 6164}}, {1694.63, {0, 18521.3, 6164}}, {0, {0, 0, 0}}},
};
int cal_row(int id) { return id == kVarTile256x256 ? 3 : id; }
// Rows kernel, cycles per row block: a fixed part, and one per 128-column tile
// (both passes) with 8 k-steps and with 4 (k <= 64), and what the stores of
// 128 rows of f32 outputs add (14 shapes of 12 to 84 row blocks took 15 to 50 % more
// than modelled without it: 37 x 152 x 1952 x 128 f16 58.6 us, 43.8 with 256-row
// tiles; 296 x 4 x 5192 x 96, 4 rows stored, does not: 166, split 236).
constexpr double kRowsBlockCyc = 2100.0, kRowsTileCyc = 4520.9, kRowsTile4Cyc = 3223.4, kRowsTileF32Cyc = 1500.0;
// Few-row kernel: a workgroup's first loads and its softmax (us), one 16 KiB unit
// of B (us), and the rate at which all workgroups together read B (GB/s): read
// off 36 timings of 4 to 512 batches x 1 to 16 rows x 256 to 7936 columns (not
// in the table above, whose shapes have more rows).  For so few rows the model
// prices the 128-row tiles up to 30 % too high, so the few-row kernel is priced
// as much too high: it is then taken where it loses by 3 % at the most (split in
// place of it: 16 x 1 x 2304 x 128 11.7 us against 13.8, 19 x 1 x 4752 x 64 15.2
// against 17.7; taken: 32 x 2 x 1312 x 128 10.5 us, split 12.1, and 24 x 2 x 5368 x
// 64 19.4, 18.8).
constexpr double kFewFixedUs = 1.5, kFewUnitUs = 0.245, kFewHbmGBs = 6000.0, kFewMargin = 1.3;
// Back-to-back launch cost of one kernel (us); the row exchange after the
// last tile of a row block: fixed (us) and per column tile (us); the HBM
// rate of the fused paths' streaming passes and the chip-wide rate that
// prices k-tile bytes (GB/s).
constexpr double kLaunchUs = 3.9154, kExchangeUs = 0.2854, kExchangePerTileUs = 0.09870;
constexpr double kHbmGBs = 6776.6, kFeedGBs = 117314.0;
// The parts below are not in the fit (the table has few f32 outputs and few B
// rows that do not start on a cache line): read off the timings of 6000 drawn
// calls, every choice of each (16-bit and fp8 general products, attention, logits),
// so that few calls lose to the choice before the fit (16 by more than 3 %, 3 by
// more than 10 %; without them 29 and 14) and the picks lose 1.6 % on average
// against the fastest (2.0).
// k-rows of B that do not start on a cache line: lines fetched beyond the row's
// own (bf16 1303 x 4616 x 1536, 407 tiles of 128 x 128: 44.5 us, priced 36.0 without
// this, 37.7 with; 222 of 256 x 128 37.5, priced 37.1.  Tiles of 256 columns pay half as much per column).
constexpr double kUnalignedLines = 2.5;
// A 256 x 256 tile of f32 outputs: its second staging round and stores (fp8 4 x
// 1015 x 4488 x 400: 79.7 us, 60.1 with 128 x 128 tiles; f16 943 x 17592 x 1984,
// 276 tiles: 160, 128 with 128 x 128).
constexpr double kManyWaves = 1.1, kWideF32Cyc = 7000.0;
// A 256 x 128 tile's fixed part on the exchange path (its k-tiles cost what the split
// path's do), and what f32 outputs add (twice the entries and stores): modelled and
// measured us: 1536 x 4096 x 1024 bf16 25.3, 24.8; 4096 x 2048 x 512 f16 20.5, 19.8,
// to f32 22.0, 23.7; 12 x 1754 x 248 x 128 bf16 to f32 13.0, 14.8 (rows kernel 12.1).
constexpr double kTallFixedCyc = 11500.0, kTallF32Cyc = 2300.0;
// f32 inputs: two 64 x 64 tiles on a CU at once take this part of one after the
// other; the split path's tile pass takes this much longer (us) than the exchange
// path's on the same tiles (602 x 2296 x 64: 11.7 us, split 16.7).
constexpr double kF32PairShare = 0.75, kF32SplitUs = 2.6;
// Unfused row passes (one 256-thread workgroup per row, eight per CU): HBM
// rate, and the rate one workgroup streams its row at (GB/s).
constexpr double kRowPassHbmGBs = 5293.0, kRowPassWgGBs = 5.573;

// Core clock under load, from the share of busy CUs: 1.5 GHz
// with every CU busy throughout, ~2.1 with half of them or fewer (the chip's
// power limit, not the workload, sets it).
double clock_ghz(double busy) {
  busy = std::min(1.0, std::max(0.0, busy));
  return busy <= 0.5 ? 2.1 : 2.1 - 1.2 * (busy - 0.5);
}

int in_class(int in_dt) {
  return in_dt == WTC_DTYPE_FP8_E4M3 ? 1 : (in_dt == WTC_DTYPE_F32 ? 2 : 0);
}

}  // namespace

static std::vector<VariantDesc> make_variants(int in_dt) {
  std::vector<VariantDesc> v;
  if (!valid_in(in_dt)) return v;
  const int64_t tk = 128 / in_bytes(in_dt);
  if (in_dt == WTC_DTYPE_F32) {
    v.push_back({kVarTile128, "tile128x128_wave64x64", 128, 128, tk, 2, 32, 128, 0, kTilePaths});
    return v;
  }
  v.push_back({kVarTile128, "tile128x128_wave64x32", 128, 128, tk, 2, 16, 128, 0, kTilePaths});
  v.push_back({kVarTile128Loaders, "tile128x128_wave64x64_loaders", 128, 128, tk, 2, 32, 128, 1,
               kTilePaths});
  v.push_back({kVarTile256, "tile256x128_wave64x64", 256, 128, tk, 2, 32, 256, 0, kSplitPaths});
  if (in_dt == WTC_DTYPE_F16 || in_dt == WTC_DTYPE_BF16)
    v.push_back({kVarRows, "rows128_wave64x32_k128", 128, 128, kRowsMaxK, 2, 16, 128, 0,
                 bit(WTC_PATH_ROWS)});
  // tile_k: one 64-byte k-slab per ring stage
  v.push_back({kVarTile256x256, "tile256x256_wave128x128", 256, 256, tk / 2, 4, 64, 256, 0,
               kSplitPaths});
  return v;
}

const std::vector<VariantDesc>& variants_for(int in_dt) {
  static const std::vector<VariantDesc> tables[5] = {
      make_variants(WTC_DTYPE_F32), make_variants(WTC_DTYPE_F16), make_variants(WTC_DTYPE_BF16),
      make_variants(WTC_DTYPE_FP8_E4M3), {}};
  return tables[valid_in(in_dt) ? in_dt : 4];
}

bool find_variant(int in_dt, int64_t tm, int64_t tn, int64_t tk, int64_t ttm, int64_t ttn,
                  VariantDesc* out) {
  for (const VariantDesc& v : variants_for(in_dt))
    if (v.tile_m == tm && v.tile_n == tn && v.tile_k == tk && v.thread_tile_m == ttm &&
        v.thread_tile_n == ttn) {
      if (out) *out = v;
      return true;
    }
  return false;
}

bool variant_by_id(int in_dt, int id, VariantDesc* out) {
  for (const VariantDesc& v : variants_for(in_dt))
    if (v.id == id) {
      if (out) *out = v;
      return true;
    }
  return false;
}

// Whether tile_shape's 256-row tiles carry the exchange path: 128-row tiles do
// not fit on the CUs, 256-row tiles do.
static bool tall_exchange(const VariantDesc& v, const Problem& p) {
  if (v.id != kVarTile128Loaders) return false;
  const int64_t nT = cdiv(p.n, 128), tiles = p.batch * cdiv(p.m, 256) * nT;
  return p.batch * cdiv(p.m, 128) * nT > (int64_t)p.cu_count * std::max(1, p.xch_per_cu) && tiles <= p.cu_count &&
         nT <= kTallMaxColTiles && tall_slots(p.out_dt) * tiles <= kExchangeMaxTiles;
}

bool feasible(const VariantDesc& v, int path, const Problem& p) {
  if (path < WTC_PATH_EXCHANGE || path > WTC_PATH_ROWS || !(v.paths & bit(path))) return false;
  const int64_t nT = cdiv(p.n, v.tile_n);
  switch (path) {
    case WTC_PATH_EXCHANGE: {
      const int64_t tiles = p.batch * cdiv(p.m, v.tile_rows) * nT;
      return (tiles <= (int64_t)p.cu_count * std::max(1, p.xch_per_cu) &&
              nT <= kExchangeMaxColTiles && tiles <= kExchangeMaxTiles) ||
             tall_exchange(v, p);
    }
    case WTC_PATH_SPLIT:
      return nT <= kSplitMaxColTiles;
    case WTC_PATH_ROWS:
      return p.k <= kRowsMaxK;
    default:
      return true;
  }
}

TileShape tile_shape(const VariantDesc& v, int path, const Problem& p) {
  if (path == WTC_PATH_ROWS) {
    const int64_t logits = p.m * (cdiv(p.n, 128) * 128 + 4);
    if (p.m > kFewRows || logits > kFewRowsLogits) return {128, 128, 0, 1};
    return {(int)kFewRows, 128, 0, logits <= kFewRowsLogitsPair && p.batch > p.cu_count ? 2 : 1};
  }
  if (path == WTC_PATH_EXCHANGE && tall_exchange(v, p)) return {256, 128, 0, 1};
  if (p.in_dt != WTC_DTYPE_F32)
    return {v.tile_rows, (int)v.tile_n, v.loaders, path == WTC_PATH_EXCHANGE ? std::max(1, p.xch_per_cu) : 1};
  if (path == WTC_PATH_EXCHANGE) {
    const int64_t nT = cdiv(p.n, 64), tiles = p.batch * cdiv(p.m, 64) * nT;
    if (tiles <= (int64_t)kF32SmallTilesPerCu * p.cu_count && tiles <= kExchangeMaxTiles &&
        nT <= kExchangeMaxColTiles)
      return {64, 64, p.k > kF32OneGroupK ? 1 : 0, kF32SmallTilesPerCu};
  }
  return {128, 128, 1, 1};
}

std::string infeasible_reason(const VariantDesc& v, int path, const Problem& p) {
  static const char* const kPathNames[] = {"auto", "exchange", "split", "unfused", "rows"};
  if (path < WTC_PATH_EXCHANGE || path > WTC_PATH_ROWS) return "unknown path";
  if (!(v.paths & bit(path)))
    return path == WTC_PATH_ROWS ? "rows path needs 16-bit inputs and k <= 128"
                                 : std::string("variant ") + v.name + " does not run the " +
                                       kPathNames[path] + " path";
  const int64_t nT = cdiv(p.n, v.tile_n);
  switch (path) {
    case WTC_PATH_EXCHANGE: {
      const int64_t tiles = p.batch * cdiv(p.m, v.tile_rows) * nT;
      const int64_t resident = (int64_t)p.cu_count * std::max(1, p.xch_per_cu);
      if (tiles > resident)
        return "exchange path needs every tile co-resident: " + std::to_string(tiles) + " tiles > " +
               std::to_string(resident) + " resident workgroups";
      if (nT > kExchangeMaxColTiles || tiles > kExchangeMaxTiles)
        return "exchange path supports n <= 8192 and <= " + std::to_string(kExchangeMaxTiles) +
               " tiles";
      return "";
    }
    case WTC_PATH_SPLIT:
      return nT > kSplitMaxColTiles
                 ? "split path supports n <= " + std::to_string(kSplitMaxColTiles * v.tile_n) +
                       " with " + std::to_string(v.tile_n) + "-column tiles"
                 : "";
    case WTC_PATH_ROWS:
      return p.k > kRowsMaxK ? "rows path needs 16-bit inputs and k <= 128" : "";
    default:
      return "";
  }
}

int64_t variant_grid(const VariantDesc& v, int path, const Problem& p) {
  const TileShape ts = tile_shape(v, path, p);
  const int64_t row_blocks = p.batch * cdiv(p.m, ts.rows);
  return path == WTC_PATH_ROWS ? row_blocks : row_blocks * cdiv(p.n, ts.cols);  // rows: all of n per workgroup
}

double estimate_us(const VariantDesc& v, int path, const Problem& p) {
  const double cu = std::max(1, p.cu_count);
  const double isz = in_bytes(p.in_dt), osz = out_bytes(p.out_dt);
  const double elems = (double)p.batch * (double)p.m * (double)p.n;
  const double ab_bytes = (double)p.batch * ((double)p.m * p.k + (double)p.k * p.n) * isz;
  const double us_per_byte = 1e6 / (kHbmGBs * 1e9);
  const TileShape ts = tile_shape(v, path, p);
  const double nT = (double)cdiv(p.n, ts.cols);
  if (path == WTC_PATH_ROWS) {
    const double blocks = (double)variant_grid(v, path, p);
    if (ts.rows == kFewRows) {
      // one stream of B per batch: 16 KiB units at what a CU's loads in flight
      // bring, or at the HBM rate shared with the other workgroups
      const double units = nT * (p.k > 64 ? 2 : 1);
      auto round_us = [&](double active) {
        return kFewFixedUs / ts.per_cu + std::max(units * kFewUnitUs, ab_bytes / blocks * active * 1e6 / (kFewHbmGBs * 1e9));
      };
      const double full = std::floor(blocks / cu), rem = blocks - full * cu;
      return kFewMargin * (kLaunchUs + full * round_us(cu) + (rem > 0 ? round_us(rem) : 0.0));
    }
    const double waves = std::ceil(blocks / cu);
    const double f = clock_ghz(blocks / (waves * cu));
    const double f32_cyc = osz == 4 ? kRowsTileF32Cyc * (double)std::min<int64_t>(p.m, 128) / 128 : 0.0;
    const double cyc = kRowsBlockCyc + nT * ((p.k <= 64 ? kRowsTile4Cyc : kRowsTileCyc) + f32_cyc);
    const double t_blocks = waves * cyc / (f * 1e3);
    const double t_hbm = (ab_bytes + elems * osz) * us_per_byte;
    return kLaunchUs + std::max(t_blocks, t_hbm);
  }
  const bool tall = path == WTC_PATH_EXCHANGE && ts.rows == 256;
  const TileCal& cal = kTileCal[tall ? 2 : cal_row(v.id)][in_class(p.in_dt) + (ts.rows == 64 ? 1 : 0)];
  const int epi = path == WTC_PATH_EXCHANGE ? 0 : (path == WTC_PATH_SPLIT ? 1 : 2);
  const double tiles = (double)variant_grid(v, path, p);
  const double nk = (double)cdiv(p.k * in_bytes(p.in_dt), 128);
  // A and B per 128 bytes of K
  const bool unaligned = p.n * in_bytes(p.in_dt) % 128 != 0;
  const double kt_bytes = (ts.rows + ts.cols + (unaligned ? kUnalignedLines * 128.0 / isz : 0.0)) * 128.0;
  auto wave_us = [&](double active) {
    // One full wave and a part of another: each at its own clock (fp8 1000 x 4104
    // x 2064, 264 tiles of 128 x 128: 35.2 us, where the mean clock gave 26 and
    // the 256 x 128 tiles take 31.2).  With more waves, whose tiles run side by
    // side, and with 256 x 256 tiles the mean clock ranked better.
    const bool own = tiles <= 2 * cu && v.id != kVarTile256x256;
    const double f = clock_ghz(own ? active / cu : tiles / (std::ceil(tiles / cu) * cu));
    const double kt = cal.kt_cyc + kt_bytes * active * f / kFeedGBs;
    const double wide_f32 = v.id == kVarTile256x256 && epi == 1 && osz == 4 ? kWideF32Cyc : 0.0;
    const double fixed = tall ? kTallFixedCyc + (osz == 4 ? kTallF32Cyc : 0.0) : cal.fixed_cyc[epi];
    return (fixed + wide_f32 + nk * kt) / (f * 1e3);
  };
  const double full = std::floor(tiles / cu), rem = tiles - full * cu;
  // 128-column tiles of more than two waves re-read A and B more than the rates
  // above say: without this part a row of 145 of them was put before 73 tiles of
  // 256 x 256 (bf16 607 x 18520 x 2240: 101 us, 70 with the latter).
  const double many = tiles > 2 * cu && v.id != kVarTile256x256 ? kManyWaves : 1.0;
  const double pair = ts.rows == 64 && tiles > cu ? kF32PairShare : 1.0;
  const double t_tiles = many * pair * (full * wave_us(cu) + (rem > 0 ? wave_us(rem) : 0.0));
  if (path == WTC_PATH_EXCHANGE) {
    const double t_hbm = (ab_bytes + elems * osz) * us_per_byte;
    const double t_xch = p.n > ts.cols ? kExchangeUs + kExchangePerTileUs * nT : 0.0;
    return kLaunchUs + std::max(t_tiles, t_hbm) + t_xch;
  }
  if (path == WTC_PATH_SPLIT) {
    // the tile pass writes the output and the row statistics; the rescale
    // pass reads and rewrites the output
    const double stats = (double)p.batch * (double)p.m * nT * 8.0;
    const double t_hbm = (ab_bytes + elems * osz + stats) * us_per_byte;
    const double t_rescale = (2.0 * elems * osz + stats) * us_per_byte;
    const double f32 = p.in_dt == WTC_DTYPE_F32 ? kF32SplitUs : 0.0;
    return 2 * kLaunchUs + std::max(t_tiles, t_hbm) + t_rescale + f32;
  }
  // unfused: f32 logits, then max, exp, sum and divide passes over them,
  // each at the HBM rate or, with few rows, at the rate of its workgroups
  const double row_us_per_byte = 1e6 / (kRowPassHbmGBs * 1e9);
  double t = 5 * kLaunchUs + std::max(t_tiles, (ab_bytes + elems * 4.0) * row_us_per_byte);
  const double row_waves = std::ceil((double)p.batch * (double)p.m / (cu * 8));
  for (const double bpe : {4.0, 8.0, 4.0, 4.0 + osz})
    t += std::max(elems * bpe * row_us_per_byte,
                  row_waves * (double)p.n * bpe * 1e6 / (kRowPassWgGBs * 1e9));
  return t;
}

std::vector<Choice> rank_choices(const Problem& p, int path, int variant) {
  std::vector<Choice> out;
  for (const VariantDesc& v : variants_for(p.in_dt)) {
    if (variant >= 0 && v.id != variant) continue;
    for (int q = WTC_PATH_EXCHANGE; q <= WTC_PATH_ROWS; ++q) {
      if (path == WTC_PATH_AUTO ? q == WTC_PATH_UNFUSED : q != path) continue;
      if (!feasible(v, q, p)) continue;
      out.push_back({v, q, estimate_us(v, q, p)});
    }
  }
  std::stable_sort(out.begin(), out.end(),
                   [](const Choice& a, const Choice& b) { return a.est_us < b.est_us; });
  return out;
}

bool best_choice(const Problem& p, int path, int variant, Choice* out) {
  bool found = false;
  for (const VariantDesc& v : variants_for(p.in_dt)) {
    if (variant >= 0 && v.id != variant) continue;
    for (int q = WTC_PATH_EXCHANGE; q <= WTC_PATH_ROWS; ++q) {
      if (path == WTC_PATH_AUTO ? q == WTC_PATH_UNFUSED : q != path) continue;
      if (!feasible(v, q, p)) continue;
      const double est = estimate_us(v, q, p);
      if (!found || est < out->est_us) {  // ties keep the earlier pair, as the stable sort does
        *out = Choice{v, q, est};
        found = true;
      }
    }
  }
  return found;
}

}  // namespace wtc
