// C-ABI layer: argument validation, kernel selection (tune table, then heuristic) and launch.
// Mirrors the reference's host launchers: no allocation, no synchronisation, work enqueued on
// the caller's stream (src/mm/fp16/mm.cu:6-42, examples/005.fp8.mm.cu:2466-2500).
#include "../../include/llmmm.h"
#include "../../include/llmmm_probe.h"
#include "kernels.h"
#include "tune_table.h"

#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <mutex>
#include <vector>

namespace {

thread_local char g_last_error[256] = "";

int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int fail(int code, const char* fmt, ...)
{
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
  return code;
}

}  // namespace

int llmmm::num_cus()
{
  static const int n = [] {
    int            dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0) return prop.multiProcessorCount;
    (void)hipGetLastError();  // no device: not an error of the call that asked
    return 256;
  }();
  return n;
}

// The same for the other files of the library (declared in kernels.h).
int llmmm::report_error(int code, const char* fmt, ...)
{
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
  return code;
}

namespace {

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

constexpr int    MAX_SPLIT_K     = 32;
// Compute units of the current device (llmmm::num_cus: read from the runtime once; 256, the MI355X, where no device
// can be asked -- the size queries also work without one).
#define NUM_CUS (llmmm::num_cus())

constexpr int SKINNY_MAX_M = 128;  // rows the weight-streaming kernel takes

int max_split_for(int K) { return (K / 128) < MAX_SPLIT_K ? (K / 128) : MAX_SPLIT_K; }

// Split count for the weight-streaming kernel when the tune table has no entry: about one
// workgroup (one 128-column group x one split) per CU -- what the measured
// Qwen3-4B shapes settle on -- every split at least two 128-K slices long, but short enough
// that the activation rows of a split can be staged in LDS (64 KB: 32 slices of 16 rows).
int heuristic_split(int M, int N, int K)
{
  const int groups = N / 128, kb = K / 128;
  // whole workgroups per CU, never more workgroups than CUs (96 column groups in three splits are 288 workgroups, a
  // second round: 16 x 12288 x 4096 took 18.6 us so, 13.1 us in two splits), and no more than eight splits: beyond that
  // the planes and the reduce kernel cost more than the shorter streams give (3072 x 8192 at M = 16: 9.8 us in ten, 8.5 in eight)
  int s = NUM_CUS / groups;
  if (s > 8) s = 8;
  if (s > kb / 2) s = kb / 2;
  const int mblk = M <= 16 ? 1 : M <= 32 ? 2 : M <= 64 ? 4 : 8;
  const int cap  = 32 / mblk;  // slices whose rows fit the staging area
  if (s < (kb + cap - 1) / cap) s = (kb + cap - 1) / cap;
  if (s > MAX_SPLIT_K) s = MAX_SPLIT_K;
  if (s > kb) s = kb;
  if (s < 1) s = 1;
  return s;
}

constexpr int MAX_TILE_SPLIT = 8;

// The FP8 tile kernels' time in microseconds: a CU holds `per_cu` tiles side by side and works a 128-wide slice of them all in `all` and of
// a lone one in `one`; every round of tiles starts and ends in `setup`.  Launches of at most one workgroup per CU (and a single tile row)
// run in the deep rings and have constants of their own.  S > 1 shares of K add a second kernel (`launch`) and S fp32 planes on their way
// through memory (per MB of a plane; 0.1 on top of what was fitted, for what the planes displace in the caches).  Fitted to every (tile, S) of 644 shapes on the MI355X -- 128 .. 4096 rows, N 1024 .. 57344, K 1024 .. 28672,
// half of them the tuned families' projections at other M -- each on weights from the caches and from HBM (geometric mean of the two).  The
// choice (best_fp8_tile) takes 0.939 of the time of the rules before it on the 600 with more
// than 128 rows; the smallest estimate by itself 0.936, within 0.6 % of the best (tile, S), but on weights that just fit the caches it loses by
// its planes (384 x 3584 x 18944, three sets of weights in turn: 39.0 us in three shares of 128 x 128 tiles, 40.3 in six of 128 x 256).  (Rounds weighted by tile area, and a split
// only where the tiles leave most of the chip idle, were 6.9 % off, 31 % at worst: 1408 x 26624 x 9216 468 us in 128 x 256 tiles for 381 in 128 x 128;
// 1024 x 2688 x 22016 103 unsplit for 70 in three shares; 896 x 10240 x 8192 126 for 83 in 128 x 160 tiles; 128 x 10496 x 1536
// 16.7 streaming for 11.4 in 128 x 128 tiles.)
double fp8_tile_estimate(int tile, int M, int N, int K, int S)
{
  static const struct {
    int    id, bm, bn, per_cu;
    double setup, one, all, deep_setup, deep_slice, launch, per_share, per_mb;
  } form[] = {{LLMMM_TILE_256x256, 256, 256, 1, 5.85, 1.393, 1.393, 5.85, 1.393, 4.05, 0.253, 0.052},
              {LLMMM_TILE_128x256, 128, 256, 1, 2.81, 1.100, 1.100, 4.05, 0.804, 3.59, 0.306, 0.042},
              {LLMMM_TILE_256x128, 256, 128, 1, 3.59, 1.032, 1.032, 4.23, 0.768, 2.78, 0.285, 0.228},
              {LLMMM_TILE_128x128, 128, 128, 2, 2.55, 0.677, 1.045, 4.41, 0.538, 2.21, 0.425, 0.056},
              {LLMMM_TILE_128x160, 128, 160, 2, 2.41, 0.743, 1.302, 4.40, 0.679, 2.21, 0.425, 0.056}};
  for (const auto& f : form) {
    if (f.id != tile) continue;
    const long   tiles_m = (M + f.bm - 1) / f.bm, groups = tiles_m * (N / f.bn) * S;
    const int    slices = (K / 128 + S - 1) / S;
    const bool   deep   = groups <= NUM_CUS || tiles_m == 1;
    const long   per = (groups + NUM_CUS - 1) / NUM_CUS, side = deep ? 1 : f.per_cu, full = per / side, left = per % side ? 1 : 0;
    const double us  = (full + left) * (deep ? f.deep_setup : f.setup) + slices * (full * (deep ? f.deep_slice : f.all) + left * f.one);
    return S > 1 ? us + f.launch + (double)M * N * 4e-6 * ((f.per_share + 0.1) * S + f.per_mb) : us;
  }
  return 1e30;
}
bool tile_dims(int tile, int& bm, int& bn);
bool fp16_only(int tile) { return tile == LLMMM_TILE_64x128 || tile == LLMMM_TILE_64x64; }

// The choice among `tiles` (the largest first), with at most one workgroup per CU in a split and shares of two slices or more; returns the
// tile, -1 if none divides the shape (fewer than 128 rows count as a row tail of a 128-row tile).  Each tile with the split it is fastest
// in; of tiles within 3 % of the fastest the one with the fewest shares, and of unsplit ones beyond one workgroup per CU the largest (it
// reads the least: 1024 x 18176 x 18560 takes 420 us in 256 x 256 tiles, 444 in 128 x 128 ones, 2 % below them by estimate).
int best_fp8_tile(const int* tiles, int n, int M, int N, int K, int* split)
{
  constexpr double NEAR = 1.03;
  constexpr int    MAX_TILES = 8;
  struct {
    double us;
    int    split, area;  // area: of an unsplit launch beyond one workgroup per CU, otherwise 0
  } of[MAX_TILES];
  double smallest = 1e30;
  if (n > MAX_TILES) n = MAX_TILES;
  for (int i = 0; i < n; ++i) {
    int bm, bn;
    of[i] = {1e30, 1, 0};
    if (!tile_dims(tiles[i], bm, bn) || (M % bm && !(M < 128 && bm == 128)) || N % bn) continue;
    const long count = (long)((M + bm - 1) / bm) * (N / bn);
    for (int s = 1; s == 1 || (s <= MAX_TILE_SPLIT && count * s <= NUM_CUS && s <= K / 256); ++s) {
      const double us = fp8_tile_estimate(tiles[i], M, N, K, s);
      if (us < of[i].us) of[i] = {us, s, s == 1 && count > NUM_CUS ? bm * bn : 0};
    }
    if (of[i].us < smallest) smallest = of[i].us;
  }
  int best = -1;
  for (int i = 0; i < n; ++i) {
    if (of[i].us >= 1e30 || of[i].us > smallest * NEAR) continue;
    if (best < 0 || of[i].split < of[best].split || (of[i].split == of[best].split && of[i].us < of[best].us && of[i].area >= of[best].area)) best = i;
  }
  if (best < 0) return -1;
  *split = of[best].split;
  return tiles[best];
}
// Split-K factor for a given tile.
int heuristic_tile_split(int tile, int M, int N, int K)
{
  int split = 1;
  best_fp8_tile(&tile, 1, M, N, K, &split);
  return split;
}
// Tile and split for a shape the table does not list.  (The 128 x 160 tile serves some outputs only: prefer_wide_tile.)
int heuristic_tile(int M, int N, int K, int* split)
{
  static const int cand[] = {LLMMM_TILE_256x256, LLMMM_TILE_128x256, LLMMM_TILE_256x128, LLMMM_TILE_128x128};
  return best_fp8_tile(cand, 4, M, N, K, split);
}

// The FP16 / BF16 kernels' tile for shapes the table does not list.  A launch takes about
//   fixed + rounds * setup + K / 64 * (full rounds * all + (a round is left over) * one)   microseconds,
// where a CU holds `per_cu` tiles side by side, works K = 64 of them all in `all` and of a lone one in `one`, every round starts and
// ends in `setup`, and the busiest CU gets ceil(tiles / CUs) tiles.  The constants are fitted to the measured times of every tile on
// 1170 shapes x both B layouts on the MI355X (M, N log-uniform in 128 .. 8192, K in 16 .. 8192, half of them below 512): the choice
// is within 0.2 % of the best tile on average and 24 % at worst (256 x 384 x 6832), and a fit to 70 % of them is within 0.2 %
// on the rest.  (Without the term in the rounds, and fitted from K = 256 up only, it took the largest tiles at short K: 17 % off on
// average, 1408 x 256 x 160 5.7 us in 128 x 256 tiles for 3.3 in 64 x 64.)
int heuristic_tile_fp16(int M, int N, int K, double* estimate = nullptr)
{
  static const struct {
    int    id, bm, bn, per_cu;
    double fixed, setup, one, all;
    int    form;  // 128 x 128: 1 = the shallow rings, 2 = the deep ones (llmmm::fp16_deep)
  } cand[] = {{LLMMM_TILE_256x256, 256, 256, 1, 0.00, 9.14, 1.048, 1.048, 0}, {LLMMM_TILE_128x256, 128, 256, 1, 0.00, 5.14, 0.707, 0.707, 0},
              {LLMMM_TILE_256x128, 256, 128, 1, 0.10, 4.60, 0.684, 0.684, 0}, {LLMMM_TILE_128x128, 128, 128, 2, 0.42, 3.05, 0.398, 0.999, 1},
              {LLMMM_TILE_128x128, 128, 128, 1, 0.00, 3.92, 0.380, 0.380, 2}, {LLMMM_TILE_64x128, 64, 128, 2, 0.64, 2.28, 0.303, 0.673, 0},
              {LLMMM_TILE_64x64, 64, 64, 2, 1.06, 1.71, 0.182, 0.397, 0}};
  int    best    = -1;
  double best_us = 0.;
  for (const auto& c : cand) {
    if (M % c.bm || N % c.bn || (c.form && (c.form == 2) != llmmm::fp16_deep(M, N, K))) continue;
    const long tiles = (long)(M / c.bm) * (N / c.bn);
    const long per   = (tiles + NUM_CUS - 1) / NUM_CUS;  // tiles of the busiest CU
    const long full  = per / c.per_cu, left = per % c.per_cu ? 1 : 0;
    double     round = 1.;  // of the last round, what it takes of a whole one
    if (c.id == LLMMM_TILE_256x256) {  // a partly filled last round runs in half-size tiles where launch_fp16 can arrange it
      const long tm = M / 256, tn = N / 256, whole = tiles / NUM_CUS * NUM_CUS;
      if (tiles > NUM_CUS && tm > 1 && whole % tm == 0 && tn - whole / tm > 0 && (tn - whole / tm) * tm * 2 <= NUM_CUS) round = 0.6;
    }
    const double us = c.fixed + (full + left - 1 + round) * c.setup + K / 64. * ((full - 1 + round) * c.all + left * c.one);
    if (best < 0 || us < best_us) best = c.id, best_us = us;
  }
  if (estimate) *estimate = best_us;
  return best;
}
// Split-K of the FP16 / BF16 kernels: S shares of every tile, at most one workgroup per CU, their fp32 planes written and added by a
// second kernel.  What that adds to a share's own time is fitted to every (tile, S) of 550 shapes with at most 1.2 tiles of 128 x 128
// per CU (K 256 .. 8192); a split is taken where the estimate is 6 % ahead of the unsplit choice's (`unsplit`).  On those shapes it then never
// lost, 99 took it, and the mean time is 0.94 of the unsplit choice's, 1.7 % above the best (tile, S) of each (us, unsplit / split:
// 256 x 128 x 7504 20.6 / 9.4, 384 x 640 x 5264 24.6 / 12.7, 256 x 1408 x 7024 26.1 / 16.8, 512 x 128 x 2048 7.8 / 7.2).  The planes' way
// through memory bounds it: 1024^3 in two shares takes 9.9 for 6.1.  Returns S (1: no split) and, if S > 1, the tile.
int heuristic_split_fp16(int M, int N, int K, double unsplit, int* tile)
{
  static const struct {
    int    id, bm, bn;
    double start, stage, launch, per_share, per_mb;  // (the 128 x 128 tile in its deep rings)
  } cand[] = {{LLMMM_TILE_128x128, 128, 128, 3.92, 0.380, 3.54, 0.440, 0.147},
              {LLMMM_TILE_64x128, 64, 128, 2.92, 0.303, 2.50, 0.447, -0.490},
              {LLMMM_TILE_64x64, 64, 64, 2.77, 0.182, 2.78, 0.451, -0.501}};
  const double mb     = (double)M * N * 4e-6;
  const int    stages = (K + 63) / 64;
  double       limit  = unsplit * 0.94;
  int          split  = 1;
  for (const auto& c : cand) {
    const long tiles = (long)(M / c.bm) * (N / c.bn);
    for (int s = 2; s <= llmmm::FP16_MAX_SPLIT && s <= stages && (tiles + 7) / 8 * 8 * s <= NUM_CUS; ++s) {
      const double us = c.start + (stages + s - 1) / s * c.stage + c.launch + mb * (c.per_share * s + c.per_mb);
      if (us < limit) *tile = c.id, split = s, limit = us;
    }
  }
  return split;
}

bool tile_dims(int tile, int& bm, int& bn)
{
  switch (tile) {
    case LLMMM_TILE_256x256: bm = 256; bn = 256; return true;
    case LLMMM_TILE_128x256: bm = 128; bn = 256; return true;
    case LLMMM_TILE_256x128: bm = 256; bn = 128; return true;
    case LLMMM_TILE_128x128: bm = 128; bn = 128; return true;
    case LLMMM_TILE_64x128: bm = 64; bn = 128; return true;  // FP16/BF16 only
    case LLMMM_TILE_64x64: bm = 64; bn = 64; return true;    // FP16/BF16 only
    case LLMMM_TILE_128x160: bm = 128; bn = 160; return true;  // FP8 only, outputs without 1x128 groups
    default: return false;
  }
}

// ---- tune tables: entries read at run time from the file LLMMM_TUNE_FILE names (if any) come first, the compiled-in
// table (tune_table.h) second.  File format, one entry per line, '#' starts a comment:
//   skinny <m_max> <N> <K> <split_k>          FP8 weight-streaming kernel, applies to M <= m_max
//   tile   <M> <N> <K> <tile id> <split_k>    FP8 MFMA tile kernels (tile ids: LLMMM_TILE_*; split_k 0 = heuristic)
//   fp16   <M> <N> <K> <tile id>              FP16 / BF16 GEMM
// (`python -m llmmm_amd.tune --write-file PATH` writes it.)  The reference only hints at tuning: tune(N, K),
// src/mm/fp32/impl.h:20-23.
struct TuneOverride {
  std::vector<llmmm::SkinnyTune> skinny;
  std::vector<llmmm::TileTune>   tile, fp16;
};
const TuneOverride& tune_override()
{
  static const TuneOverride t = [] {
    TuneOverride o;
    const char*  path = getenv("LLMMM_TUNE_FILE");
    if (!path || !*path) return o;
    FILE* f = fopen(path, "r");
    if (!f) {
      fprintf(stderr, "llmmm: LLMMM_TUNE_FILE=%s cannot be read; using the built-in table\n", path);
      return o;
    }
    char line[256];
    int  lineno = 0;
    while (fgets(line, sizeof(line), f)) {
      ++lineno;
      if (!strchr(line, '\n') && !feof(f)) {
        // longer than the buffer: no entry is, so the whole line is dropped (its tail must not be read as a new entry)
        int ch;
        while ((ch = fgetc(f)) != EOF && ch != '\n') {}
        fprintf(stderr, "llmmm: %s:%d: line too long, ignored\n", path, lineno);
        continue;
      }
      if (char* h = strchr(line, '#')) *h = 0;
      char kind[16];
      int  a, b, c, d, e;
      const int n = sscanf(line, "%15s %d %d %d %d %d", kind, &a, &b, &c, &d, &e);
      if (n <= 0) continue;  // blank
      int bm, bn;
      if (n == 5 && !strcmp(kind, "skinny") && a >= 1 && a <= SKINNY_MAX_M && b > 0 && c > 0 && d >= 1 && d <= MAX_SPLIT_K)
        o.skinny.push_back({a, b, c, d});
      // (a tile must divide the shape it is entered for -- an entry that does not would turn a call the heuristic serves
      // into "not aligned"; the one exception is a row tail: fewer than 128 rows in 128 x 128 tiles)
      else if (n == 6 && !strcmp(kind, "tile") && a > 0 && b > 0 && c > 0 && tile_dims(d, bm, bn) && !fp16_only(d) && d != LLMMM_TILE_128x160 && e >= 0 &&
               e <= MAX_SPLIT_K && b % bn == 0 && (a % bm == 0 || (a < 128 && d == LLMMM_TILE_128x128)))
        o.tile.push_back({a, b, c, d, e});
      else if (n == 5 && !strcmp(kind, "fp16") && a > 0 && b > 0 && c > 0 && tile_dims(d, bm, bn) && d != LLMMM_TILE_128x160 && a % bm == 0 && b % bn == 0)
        o.fp16.push_back({a, b, c, d, 1});
      else
        fprintf(stderr, "llmmm: %s:%d: not a tune entry, ignored\n", path, lineno);
    }
    fclose(f);
    return o;
  }();
  return t;
}

// FP8 tile kernels: the entry of this exact shape; failing that, for an (N, K) the tables know at other M, the tile of the
// entry nearest in M (by ratio, less than a factor of two away) whose tile divides this M -- its split count does not carry over (it depends on how many
// tiles M makes), the heuristic decides that.  false: nothing known about (N, K).
template <typename Table>
bool lookup_tile_in(const Table& table, int M, int N, int K, int* tile, int* split, double* best_ratio)
{
  bool found = false;
  for (const auto& e : table) {
    if (e.N != N || e.K != K) continue;
    int bm, bn;
    if (!tile_dims(e.tile, bm, bn) || N % bn) continue;
    // (an entry for fewer than 128 rows is a row tail of 128 x 128 tiles and speaks for exactly its M)
    if (M % bm && !(M < 128 && e.M == M && e.tile == LLMMM_TILE_128x128)) continue;
    if (e.M < 128 && e.M != M) continue;
    const double ratio = e.M > M ? (double)e.M / M : (double)M / e.M;
    if (ratio < *best_ratio) {
      *best_ratio = ratio, *tile = e.tile, *split = e.M == M ? e.split_k : 0;
      found = true;
    }
  }
  return found;
}
bool lookup_tile(int M, int N, int K, int* tile, int* split, bool exact_only = false)
{
  // (beyond a factor of two in M the tile count changes too much for the tuned tile to say anything: M = 8192 on the
  // 2560-column projections runs 7 % faster in the heuristic's 256 x 256 tiles than in the 128 x 128 ones tuned at M = 2048)
  const double limit = exact_only ? 1.0 + 1e-9 : 2.0;
  double       best  = limit;
  if (lookup_tile_in(tune_override().tile, M, N, K, tile, split, &best) && best == 1.0) return true;  // an exact entry of the file wins
  double best2 = best;
  int    t2 = 0, s2 = 0;
  if (lookup_tile_in(llmmm::kTileTune, M, N, K, &t2, &s2, &best2) && best2 < best) *tile = t2, *split = s2, best = best2;
  return best < limit;
}
bool lookup_skinny(int M, int N, int K, int* split, int* m_max = nullptr)
{
  for (const auto& e : tune_override().skinny)
    if (e.N == N && e.K == K && M <= e.m_max) return *split = e.split_k, (m_max ? *m_max = e.m_max : 0), true;
  for (const auto& e : llmmm::kSkinnyTune)
    if (e.N == N && e.K == K && M <= e.m_max) return *split = e.split_k, (m_max ? *m_max = e.m_max : 0), true;
  return false;
}
bool lookup_fp16_tile(int M, int N, int K, int* tile)
{
  // (an entry whose tile does not divide the shape is no entry: the heuristic decides)
  auto fits = [&](int t) {
    int bm, bn;
    return tile_dims(t, bm, bn) && M % bm == 0 && N % bn == 0;
  };
  for (const auto& e : tune_override().fp16)
    if (e.M == M && e.N == N && e.K == K && fits(e.tile)) return *tile = e.tile, true;
  for (const auto& e : llmmm::kFp16TileTune)
    if (e.M == M && e.N == N && e.K == K && fits(e.tile)) return *tile = e.tile, true;
  return false;
}

int choose_fp8(int M, int N, int K, llmmm_gemm_cfg* cfg)
{
  if (M <= 0 || N <= 0 || K <= 0) return fail(LLMMM_ERR_INVALID_ARGUMENT, "M, N and K must be positive (got %d, %d, %d)", M, N, K);
  if (N % 128 || K % 128) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
  cfg->tile     = -1;
  cfg->split_k  = 0;
  cfg->b_layout = LLMMM_FP8_B_ROWS;
  cfg->a_layout = LLMMM_FP8_A_QUANTISED;
  {
    int t, sp;  // an entry for exactly this shape (one for fewer than 128 rows can only name the 128 x 128 tile: a row tail)
    if (lookup_tile(M, N, K, &t, &sp, true) && (M % 128 == 0 || (M < 128 && t == LLMMM_TILE_128x128))) cfg->tile = t, cfg->split_k = sp;
  }
  // 64 < M < 128 with a weight-streaming entry measured in that range (m_max < 128): it was timed against the row-tail
  // tiles below and won (2560 x 9728 up to 96 rows: 13.0 us in four splits of 32-row groups, 14.5 us in tiles)
  if (cfg->tile < 0 && M > 64 && M < 128) {
    int sp, mm;
    if (lookup_skinny(M, N, K, &sp, &mm) && mm < 128) cfg->tile = LLMMM_TILE_SKINNY, cfg->split_k = sp;
  }
  // 64 < M < 128: where the table gives M = 128 to 128 x 128 tiles, the same tiles take the shorter matrix too (the
  // rows of the tile beyond M are computed and not stored) -- 96 x 19456 x 2560: 20 us instead of 33 us in the
  // weight-streaming kernel, whose eight 16-row blocks per wave are bound by their LDS reads and fp32 planes
  // (where that entry is unsplit -- enough column groups to fill the chip, i.e. a large weight matrix -- already from 33
  // rows on: 19456 x 2560 at M = 48 / 64: 15.9 / 16.7 us in tiles, 18.0 / 19.5 us streaming in three splits; at 32: 15.3 / 15.5)
  if (cfg->tile < 0 && M > 32 && M < 128) {
    int t, sp;
    if (lookup_tile(128, N, K, &t, &sp, true) && t == LLMMM_TILE_128x128 && (M > 64 || sp <= 1)) cfg->tile = t, cfg->split_k = sp;
  }
  if (cfg->tile < 0 && M <= SKINNY_MAX_M) {
    int sp;
    if (lookup_skinny(M, N, K, &sp)) cfg->tile = LLMMM_TILE_SKINNY, cfg->split_k = sp;
    // untuned shapes: the weight-streaming kernel up to 32 rows; its 16-row blocks per wave and its fp32 planes grow with M, and
    // one row of 128-row tiles (128 x 128 as a row tail for M < 128) is the faster from 65 rows on at every size (167 shapes with 65 .. 128
    // rows, N 1024 .. 32768, K 1024 .. 28672: 0.59 of the streaming time on average, 1.02 at most; us: 128 x 10496 x 1536 16.7 / 11.4, 128 x 2304 x 7808
    // 21.7 / 14.7, 96 x 28672 x 4096 66.7 / 27.1).  Between, on large matrices and on medium ones with many columns (137 shapes: 0.865 of
    // streaming alone; 40 x 16512 x 1408 15.1 / 9.2, 64 x 12416 x 1152 12.1 / 8.3 -- but 64 x 1152 x 17920 12.5 / 14.9).
    const long nk = (long)N * K;
    if (cfg->tile < 0) {
      if (M <= 32 || (M <= 64 && nk < 40000000L && (N < 7000 || nk < 12000000L)))
        cfg->tile = LLMMM_TILE_SKINNY;
      else if (M == 128)
        cfg->tile = heuristic_tile(M, N, K, &cfg->split_k);
      else
        cfg->tile = LLMMM_TILE_128x128;
    }
  }
  if (cfg->tile < 0) {
    if (M % 128) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
    // an (N, K) that was tuned at other M: the tile of the nearest tuned M; otherwise the heuristic
    // -- unless the estimates are 15 % apart (1536 x 4608 x 3584: 41 us in the 256 x 256 tiles of M = 2048, 30 in 256 x 128 ones)
    int t, sp;
    cfg->tile = heuristic_tile(M, N, K, &cfg->split_k);
    if (lookup_tile(M, N, K, &t, &sp)) {
      if (sp <= 0) sp = heuristic_tile_split(t, M, N, K);
      if (fp8_tile_estimate(t, M, N, K, sp) * 0.85 <= fp8_tile_estimate(cfg->tile, M, N, K, cfg->split_k)) cfg->tile = t, cfg->split_k = sp;
    }
  }
  if (cfg->tile == LLMMM_TILE_SKINNY) {
    if (cfg->split_k <= 0) cfg->split_k = heuristic_split(M, N, K);
  }
  else if (cfg->split_k <= 0)
    cfg->split_k = heuristic_tile_split(cfg->tile, M < 128 ? 128 : M, N, K);
  return LLMMM_OK;
}

// The SwiGLU output.  In the tile kernels the activation is either fused into the epilogue of a 256-column tile
// (whose two halves are the gate and the up columns of the same outputs), or -- with a 128-column tile, or
// whenever K is split -- applied by the reduce kernel to fp32 planes in the workspace.  The second way costs a
// round trip of M * N floats, which only pays while that is small and the 256-column tiles would leave
// most of the chip idle (decode-sized M).
constexpr size_t SWIGLU_PLANE_LIMIT = 16u << 20;

// Outputs without 1x128 groups (fp32, bf16, residual add) may use the 160-column tile, unsplit, where its estimate is the smaller: 2560
// columns at M = 2048 are 256 such tiles, one per CU (O / down in 320 tiles of 128 x 128: 30.0 -> 26.9 us, 64.0 -> 55.8).
void prefer_wide_tile(llmmm_gemm_cfg* cfg, int M, int N, int K)
{
  int bm, bn;
  if (N % 640 || M % 128 || !tile_dims(cfg->tile, bm, bn)) return;
  if (fp8_tile_estimate(LLMMM_TILE_128x160, M, N, K, 1) < fp8_tile_estimate(cfg->tile, M, N, K, cfg->split_k < 1 ? 1 : cfg->split_k)) cfg->tile = LLMMM_TILE_128x160, cfg->split_k = 1;
}

// The weight-streaming kernel in column strips (one launch, the K split inside the workgroup) takes what the split-K
// form of that kernel would otherwise do in two launches, for the outputs it has: no 1x128 groups.
bool strip_fits(int M, int N, int K) { return M >= 1 && M <= llmmm::STRIP_MAX_M && N % 16 == 0 && K % 128 == 0 && K / 128 >= 8; }
// Where strips beat the split-K form with its second kernel (measured, pre-shuffled weights; `fused` = with the 1x128
// quantisation, whose exchange between the strips of a column group costs 1.4 - 1.6 us, about what the reduce launch did).
// Every strip reads all M activation rows over all of K, so the strips' cost grows with M while the split form's hardly does.
//  * at most one 16-column strip per CU (2560 and 4096 columns): plain outputs up to M = 8, up to 16 for K <= 4096; fused
//    while M * K <= 65536 (2560 x 4096, us, strips / split + reduce: 5.4 / 6.5 at M = 1, 6.6 / 7.0 at 16; 2560 x 9728: 8.0 / 8.4
//    at M = 1, 9.1 / 9.0 at 8);
//  * more, but 32-column strips fit one round and the matrix is small (llmmm::strip_fragments; 6144 x 2560, 6144 x 4096,
//    5120 x 5120): plain outputs as above (6144 x 4096 at M = 16: 7.5 / 8.8), fused up to M = 4 (6144 x 2560: 6.2 / 6.65 at M = 1,
//    7.0 / 6.7 at 8; 6144 x 4096: 7.2 / 8.65 and 7.8 / 8.7; 5120 x 5120: 7.9 / 8.4 and 8.7 / 8.55);
//  * two 16-column strips on (nearly) every CU -- between 1.75 and 2 per CU, which share it side by side (8192 x 8192, 512
//    strips: 13.2 / 15.1 fused at M = 1, 14.3 / 15.3 at 8, 16.5 / 15.3 at 16; 7168 x 5120, 448 strips: 10.3 / 11.7 at M = 1;
//    8192 x 28672: 39.9 / 39.5 at M = 1 and 40.7 / 37.6 at 4, hence the same M * K bound as above);
//  * otherwise not: 5120 x 13824 at M = 1 takes 19.5 us in 320 strips, a round and a quarter, and 14.8 us in six splits
//    (5120 x 17408: 21.4 / 17.5; 10240 x 8192, 640 strips: 17.9 / 18.1).
bool strips_pay(int M, int N, int K, bool fused)
{
  const long cus = NUM_CUS, s16 = N / 16;
  const bool plain_ok = M <= 8 || (M <= 16 && K <= 4096);
  if (s16 <= cus) return fused ? (long)M * K <= 65536 : plain_ok;
  if (llmmm::strip_fragments(N, K) == 2) return fused ? M <= 4 : plain_ok;
  if (s16 <= 2 * cus && s16 * 8 >= 2 * cus * 7) return (long)M * K <= (fused ? 65536 : 131072);  // (plain: 8192 x 8192 up to M = 16)
  return false;
}
// Plain outputs, one 16-column strip per CU, measured against the split form (bf16 out, us, strips / split + reduce):
// O 4.0 / 6.2 (M = 1), 4.9 / 6.5 (8), 5.6 / 6.8 (16), 7.7 / 7.3 (32); down 6.7 / 8.2, 7.7 / 8.9, 9.4 / 9.1, 13.7 / 9.7.
void prefer_strip(llmmm_gemm_cfg* cfg, int M, int N, int K)
{
  if (cfg->tile == LLMMM_TILE_SKINNY && cfg->split_k > 1 && strip_fits(M, N, K) && strips_pay(M, N, K, false)) cfg->tile = LLMMM_TILE_STRIP, cfg->split_k = 1;
}

// The fused 1x128 output in column strips (one launch; the strips of a column group exchange their row maxima through
// device memory, fp8_skinny.hip): M <= 16 and few enough column groups for the exchange area.
bool strip_fp8q_fits(int M, int N, int K) { return strip_fits(M, N, K) && M <= 16 && N % 128 == 0 && N / 128 <= llmmm::STRIP_XCH_MAX_GROUPS; }
void prefer_strip_fp8q(llmmm_gemm_cfg* cfg, int M, int N, int K)
{
  if (cfg->tile == LLMMM_TILE_SKINNY && cfg->split_k > 1 && strip_fp8q_fits(M, N, K) && strips_pay(M, N, K, true)) cfg->tile = LLMMM_TILE_STRIP, cfg->split_k = 1;
}

// The exchange area of a stream (0 .. STRIP_XCH_AREAS - 1): launches on one stream are ordered, so they may share an
// area; every stream the library meets gets one of its own, for the life of the process, and streams beyond the number
// of areas get -1 -- their calls keep the split-K form.  Host bookkeeping only: nothing here touches the device.
int strip_exchange_area(void* stream)
{
  static std::mutex mu;
  static void*      owner[llmmm::STRIP_XCH_AREAS];
  static int        used = 0;
  std::lock_guard<std::mutex> lock(mu);
  for (int i = 0; i < used; ++i)
    if (owner[i] == stream) return i;
  if (used == llmmm::STRIP_XCH_AREAS) return -1;
  owner[used] = stream;
  return used++;
}

// The QKV projection with per-head norm and rotary embedding (bf16) in column strips, one launch (ST_OUT_ROPE in fp8_skinny.hip): one
// strip of 32 columns per CU at most -- 10240 columns are 320, 5120 of K at M = 1: 12.8 split + second kernel / 14.3 so -- and few rows, every strip
// reading all of them (us, split + second kernel / so: 6144 x 2560 6.9 / 6.3 at M = 1, 7.4 / 7.1 at 8, 7.3 / 8.2 at 12; 4096 x 2048 5.9 / 5.4,
// 6.0 / 6.1, 6.2 / 6.0; 7168 x 5120 11.4 / 9.4, 11.8 / 10.0, 11.6 / 11.0 and 11.8 / 12.4 at 16; 6144 x 4096 9.2 / 8.1, 9.4 / 8.5, 9.3 / 8.8, 9.7 / 9.0).
bool rope_strips_pay(int M, int N, int K)
{
  return K / 128 >= 8 && N / 128 <= llmmm::STRIP_XCH_MAX_GROUPS && N / 32 <= NUM_CUS &&
         (M <= 8 || (M <= 16 && (long)M * K <= 65536 && (long)N * K >= 24000000L));
}

// The same beyond 16 rows: a workgroup holds whole heads of 16 or 32 rows over all of K and rotates them itself (0: planes and a second
// kernel).  Where the split form would not split, the launch is saved at the same sums; 16-row groups while they fit one round of the chip
// -- every group streams its heads' weights again, from the L2 -- and 32-row ones beyond (us, plane + second kernel / groups of 16 / 32:
// 4096 x 2048 9.9 / 7.5 / 8.2 at M = 80, 10.0 / 7.5 / 8.4 at 128; 6144 x 2560 12.1 / 9.2 / 10.2 at M = 80, 12.3 / 16.6 / 10.2 at 100).  Against a split
// run from 48 rows on, where its planes have grown (6144 x 2560 in five splits 8.0 / 9.3 / 10.6 at M = 32, 9.3 / 9.1 at 48, 10.0 / 9.2 at 64;
// 6144 x 4096 in four 11.8 / 12.5 at 64).
int rope_row_group(int M, int N, int K, int split)
{
  if (M <= 16 || M > SKINNY_MAX_M || K < 512 || (split > 1 && (M < 48 || K > 2560))) return 0;
  const int heads = N / 128;
  if ((M + 15) / 16 * heads <= NUM_CUS && K <= 5120) return 16;
  return split <= 1 && (M + 31) / 32 * heads <= NUM_CUS && K <= 2560 ? 32 : 0;
}

// A SwiGLU launch of exchanging workgroups that fills every CU (249 .. 256 of them, pair_place) loses at K = 4096, where the columns that an
// XCD reads side by side meet on the same channels (32768 columns pre-shuffled, us, with planes / so: 27.7 / 32.2 at M = 1, 29.3 / 31.1 at 16,
// 31.5 / 33.9 at 48 -- but 36.4 / 33.7 at 100, and K = 2048 15.7 / 14.8 at M = 1).
bool swiglu_pair_camps(int N, int K) { return N / 128 > NUM_CUS - 8 && N / 128 <= NUM_CUS && K % 4096 == 0; }

// The SwiGLU output of the weight-streaming kernel in one launch (64 gate + 64 up columns per workgroup, K unsplit; figures in
// fp8_skinny.hip).  Its N / 128 workgroups have to fill the chip or a good part of its last round: with fewer, splitting K pulls more
// (12288 x 2048, 96 workgroups, M = 24: 9.4 in two splits + reduce / 9.9 so), and 272 or 296 run a nearly empty second round
// (34816 x 5120 at M = 1: 36.8 / 43.6; 51200 x 5120, 400 of them: 48.9 / 47.9 at M = 1, 54.6 / 49.2 at 16). 
// Row-major weights, which stream less evenly, need more of them (12288 x 2048: 8.5 / 9.2 at M = 1, 9.3 / 10.6 at 16; 16384 x 3072 at M = 1
// 13.9 / 14.7; pre-shuffled 8.7 / 8.8, 9.3 / 9.5 and 13.2 / 13.4 for a launch less).
bool swiglu_pair_pays(int M, int N, int K, bool pre)
{
  const int groups = N / 128, last = groups % NUM_CUS;
  if (swiglu_pair_camps(N, K)) return false;
  return llmmm::fp8_skinny_swiglu_fits(M, N, K) && groups >= (!pre ? 144 : M <= 16 ? 96 : 128) && (groups <= NUM_CUS || last == 0 || last >= NUM_CUS / 2);
}

// The SwiGLU output of fewer than 128 rows in 256-column tiles (a row tail; each holds whole 1x128 groups, so nothing is exchanged): from
// 33 rows on where the 128-column ones would be more than one round of the chip, from 17 -- against the weight-streaming kernel -- where they
// fill three quarters of a round (us, pre-shuffled, before / so: 37888 x 3584 43.4 / 35.8 at M = 48, 49.2 / 38.3 at 100; 34816 x 5120 63.8 / 50.9 at 100;
// 57344 x 8192 115 / 83.7 at 100; 51200 x 5120, 200 tiles, 63.4 / 50.1 at 32, 59.0 / 48.9 at 20 -- but 148 tiles of 37888 x 3584 33.5 / 34.7 at 20).
// Up to 32 rows only with a long K: 65536 x 2048 30.4 / 32.5 at 24.
bool swiglu_wide_tail(int M, int N, int K)
{
  if (M >= 128 || N % 256) return false;
  return M > 32 ? N / 128 > NUM_CUS : M > 16 && K >= 4096 && N / 256 >= NUM_CUS * 3 / 4 && N / 256 <= NUM_CUS;
}

// The split the weight-streaming kernel runs this shape in when it is the split-K form after all (tune table, then heuristic).
int skinny_split_for(int M, int N, int K)
{
  int sp;
  return lookup_skinny(M, N, K, &sp) ? sp : heuristic_split(M, N, K);
}

// Planes a strip-capable shape needs when the call turns out not to run in strips after all: activations the kernel makes
// itself (cfg.a_layout) and explicit splits belong to the split-K form, and generated activations need a split whose K
// range fits the staging buffer.  The size queries cannot see the caller's cfg, so they answer for this case.
size_t strip_fallback_plane_bytes(int M, int N, int K)
{
  int s = skinny_split_for(M, N, K);
  const int kb = K / 128, min_split = (kb + 31) / 32;  // = agen_min_split(K)
  if (s < min_split) s = min_split;
  if (s > max_split_for(K)) s = max_split_for(K);
  return (size_t)(s < 1 ? 1 : s) * M * N * sizeof(float);
}

int choose_fp8_out(int out_kind, int M, int N, int K, llmmm_gemm_cfg* cfg)
{
  const int rc = choose_fp8(M, N, K, cfg);
  if (rc) return rc;
  if (out_kind == LLMMM_OUT_F32 || out_kind == LLMMM_OUT_BF16) prefer_wide_tile(cfg, M, N, K), prefer_strip(cfg, M, N, K);
  if (out_kind == LLMMM_OUT_FP8Q) prefer_strip_fp8q(cfg, M, N, K);
  if (out_kind == LLMMM_OUT_FP8Q_SWIGLU) {
    if (N % 256) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
    if (cfg->tile != LLMMM_TILE_SKINNY && cfg->split_k <= 1) {
      const bool narrow      = cfg->tile == LLMMM_TILE_256x128 || cfg->tile == LLMMM_TILE_128x128;
      const long wide_tiles  = (long)(M / 128) * (N / 256);
      const bool small_plane = (size_t)M * N * sizeof(float) <= SWIGLU_PLANE_LIMIT;
      if (small_plane && wide_tiles < NUM_CUS / 2) {
        if (!narrow) cfg->tile = LLMMM_TILE_128x128;  // through one fp32 plane, twice the workgroups
      }
      else if (narrow && M % 128 == 0)  // (a row tail stays with the 128 x 128 tiles and the plane)
        cfg->tile = M % 256 == 0 && fp8_tile_estimate(LLMMM_TILE_256x256, M, N, K, 1) < fp8_tile_estimate(LLMMM_TILE_128x256, M, N, K, 1) ? LLMMM_TILE_256x256
                                                                                                                                          : LLMMM_TILE_128x256;
    }
  }
  return LLMMM_OK;
}

}  // namespace

extern "C" {

const char* llmmm_error_string(int code)
{
  switch (code) {
    case LLMMM_OK: return "ok";
    case LLMMM_ERR_NOT_ALIGNED: return "M or N or K are not aligned.";
    case LLMMM_ERR_UNSUPPORTED_TYPE: return "T is not supported.";
    case LLMMM_ERR_INVALID_ARGUMENT: return "invalid argument";
    case LLMMM_ERR_WORKSPACE: return "workspace missing or too small";
    case LLMMM_ERR_RUNTIME: return "HIP runtime error";
    default: return "unknown error";
  }
}

const char* llmmm_last_error(void) { return g_last_error; }

int llmmm_version(void) { return 100; }

// Kernel choice of a call without (or with AUTO) cfg; split > 1 needs split * M * N floats.
static void choose_fp16(int M, int N, int K, bool may_split, int* tile, int* split)
{
  *split = 1;
  if (lookup_fp16_tile(M, N, K, tile)) return;
  double us;
  *tile = heuristic_tile_fp16(M, N, K, &us);
  if (may_split) *split = heuristic_split_fp16(M, N, K, us, tile);
}

size_t llmmm_fp16_gemm_workspace(int M, int N, int K)
{
  if (M <= 0 || N <= 0 || K <= 0 || M % 128 || N % 128 || K % 16) return 0;
  int tile, split;
  choose_fp16(M, N, K, true, &tile, &split);
  return split > 1 ? (size_t)split * M * N * sizeof(float) : 0;
}

int llmmm_fp16_gemm_ws(int dtype, const void* A, const void* B, void* C, int M, int N, int K, int b_layout, void* workspace, size_t workspace_bytes,
                       const llmmm_gemm_cfg* cfg, void* stream)
{
  if (dtype != LLMMM_DTYPE_F16 && dtype != LLMMM_DTYPE_BF16) return fail(LLMMM_ERR_UNSUPPORTED_TYPE, "T is not supported.");
  if (b_layout != LLMMM_B_ROW_MAJOR && b_layout != LLMMM_B_TRANSPOSED)
    return fail(LLMMM_ERR_INVALID_ARGUMENT, "unknown B layout %d", b_layout);
  if (M <= 0 || N <= 0 || K <= 0) return fail(LLMMM_ERR_INVALID_ARGUMENT, "M, N and K must be positive (got %d, %d, %d)", M, N, K);
  if (M % 128 || N % 128 || K % 16) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
  if (!A || !B || !C) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (!aligned16(A) || !aligned16(B) || !aligned16(C)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 16-byte aligned");
  if ((long)M * K >= (1L << 31) || (long)N * K >= (1L << 31) || (long)M * N >= (1L << 31))
    return fail(LLMMM_ERR_INVALID_ARGUMENT, "matrix has 2^31 or more elements");
  const size_t plane = (size_t)M * N * sizeof(float);
  int          tile = cfg ? cfg->tile : LLMMM_TILE_AUTO, split = 1;
  if (tile == LLMMM_TILE_AUTO) {
    choose_fp16(M, N, K, workspace != nullptr, &tile, &split);
    if (split > 1 && workspace_bytes < split * plane) choose_fp16(M, N, K, false, &tile, &split);  // (documented: no room, no split)
  }
  int bm, bn;
  if (!tile_dims(tile, bm, bn) || tile == LLMMM_TILE_128x160) return fail(LLMMM_ERR_INVALID_ARGUMENT, "unknown tile id %d", tile);
  if (M % bm || N % bn) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
  if (cfg && cfg->tile != LLMMM_TILE_AUTO && cfg->split_k > 1 && workspace) {  // (ignored without a workspace, as llmmm_fp16_gemm_ex ignores it)
    split = cfg->split_k;
    if (split > llmmm::FP16_MAX_SPLIT || split > (K + 63) / 64 || (tile != LLMMM_TILE_128x128 && !fp16_only(tile)))
      return fail(LLMMM_ERR_INVALID_ARGUMENT, "split-K %d: 128 x 128 and smaller tiles, at most %d shares and one per 64 of K", split, llmmm::FP16_MAX_SPLIT);
    if (workspace_bytes < split * plane) return fail(LLMMM_ERR_WORKSPACE, "workspace holds %zu bytes, split-K %d needs %zu", workspace_bytes, split, split * plane);
  }
  if (split > 1 && !aligned16(workspace)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "workspace must be 16-byte aligned");
  const hipError_t e = split > 1 ? llmmm::fp16_gemm_split_launch(dtype, b_layout, tile, A, B, C, M, N, K, split, (float*)workspace, (hipStream_t)stream)
                                 : llmmm::fp16_gemm_launch(dtype, b_layout, tile, A, B, C, M, N, K, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "fp16 gemm launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

int llmmm_fp16_gemm_ex(int dtype, const void* A, const void* B, void* C, int M, int N, int K, int b_layout, const llmmm_gemm_cfg* cfg, void* stream)
{
  return llmmm_fp16_gemm_ws(dtype, A, B, C, M, N, K, b_layout, nullptr, 0, cfg, stream);
}

int llmmm_fp16_gemm(int dtype, const void* A, const void* B, void* C, int M, int N, int K, int b_layout, void* stream)
{
  return llmmm_fp16_gemm_ex(dtype, A, B, C, M, N, K, b_layout, nullptr, stream);
}

int llmmm_fp8_gemm_query(int out_kind, int M, int N, int K, llmmm_gemm_cfg* cfg)
{
  if (out_kind < LLMMM_OUT_F32 || out_kind > LLMMM_OUT_FP8Q_SWIGLU) return fail(LLMMM_ERR_INVALID_ARGUMENT, "unknown output kind %d", out_kind);
  if (!cfg) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null cfg");
  return choose_fp8_out(out_kind, M, N, K, cfg);
}

size_t llmmm_fp8_gemm_workspace(int out_kind, int M, int N, int K)
{
  if (M <= 0 || N <= 0 || K <= 0 || N % 128 || K % 128) return 0;
  llmmm_gemm_cfg cfg;
  if (choose_fp8_out(out_kind, M, N, K, &cfg) != LLMMM_OK) return 0;
  if (cfg.tile == LLMMM_TILE_STRIP) return strip_fallback_plane_bytes(M, N, K);  // strips need none; a call with generated activations leaves them
  const int  s       = cfg.split_k;  // the split the library would pick (an explicit cfg->split_k = S needs S planes)
  const bool narrow  = cfg.tile == LLMMM_TILE_256x128 || cfg.tile == LLMMM_TILE_128x128;
  const bool a_plane = out_kind == LLMMM_OUT_FP8Q_SWIGLU && (cfg.tile == LLMMM_TILE_SKINNY || narrow);  // SwiGLU outside a 256-column tile
  if (s <= 1 && !a_plane) return 0;
  return (size_t)(s < 1 ? 1 : s) * M * N * sizeof(float);
}

// cfg.a_layout = LLMMM_FP8_A_SWIGLU_F32: the weight-streaming kernel makes the activations itself for M <= 4 when a
// split's K range fits its staging buffer (32 slices of 128); otherwise h is quantised into the front of the workspace.
// (Every column group's workgroup repeats the activation work of its K range, so its cost grows with M: measured on the
// Qwen3-4B down projection, +0.8 us at M = 1, +1.8 at M = 4, +2.5 at M = 8, +4.6 at M = 16, against the 2.4 us that the
// separate SwiGLU quantiser launch costs.  The kernel itself takes up to 16 rows.)
constexpr int AGEN_MAX_M = 4, AGEN_MAX_SLICES = 32;
static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
static size_t swiglu_a_bytes(int M, int K) { return align256((size_t)M * K) + align256((size_t)(K / 128) * M * sizeof(float)); }
static int agen_min_split(int K) { return ((K / 128) + AGEN_MAX_SLICES - 1) / AGEN_MAX_SLICES; }

size_t llmmm_fp8_swiglu_a_workspace(int M, int N, int K)
{
  llmmm_gemm_cfg cfg;
  if (choose_fp8(M, N, K, &cfg) != LLMMM_OK) return 0;
  if (cfg.tile == LLMMM_TILE_SKINNY && M <= AGEN_MAX_M) return 0;
  return swiglu_a_bytes(M, K);
}

// How a call gets its A operand: given quantised (agen 0), generated by the weight-streaming kernel from the fp32 gate_up
// result (1) or from a hidden state still in pieces (2, with what the kernel needs in `ag`).
struct APrep {
  int               agen         = 0;
  int               hidden_dtype = 0;
  llmmm::SkinnyGenA ag;
};
constexpr int AGEN2_MAX_M = 2, AGEN2_MAX_K = 3072;

size_t llmmm_fp8_planes_rmsnorm_a_workspace(int M, int N, int K)
{
  llmmm_gemm_cfg cfg;
  if (choose_fp8(M, N, K, &cfg) != LLMMM_OK) return 0;
  // (the generating kernel writes fp32 only: any other output kind goes through one fp32 plane and the reduce kernel, and
  // an unsplit call has no plane in llmmm_fp8_gemm_workspace's answer -- this one covers it)
  if (cfg.tile == LLMMM_TILE_SKINNY && M <= AGEN2_MAX_M && K <= AGEN2_MAX_K) return (size_t)M * N * sizeof(float);
  return swiglu_a_bytes(M, K);  // the same codes + scales block
}

// Resolves a_layout for a call whose kernel choice is `tile`: either the kernel generates A (prep->agen != 0; A is not
// used as an operand pointer any more), or the operand is quantised into the front of the workspace now and A / As /
// workspace are redirected to it.
static int prepare_a(const llmmm_gemm_cfg* user, int tile, const void*& A, const float*& As, int M, int K, void*& workspace, size_t& workspace_bytes,
                     void* stream, APrep* prep)
{
  *prep = APrep();
  if (!user || user->a_layout == LLMMM_FP8_A_QUANTISED) return LLMMM_OK;
  if (user->a_layout != LLMMM_FP8_A_SWIGLU_F32 && user->a_layout != LLMMM_FP8_A_PLANES_RMSNORM)
    return fail(LLMMM_ERR_INVALID_ARGUMENT, "unknown A layout %d", user->a_layout);
  if ((long)M * 2 * K >= (1L << 31)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "matrix has 2^31 or more elements");
  const llmmm_a_planes_rmsnorm* d = nullptr;
  if (user->a_layout == LLMMM_FP8_A_PLANES_RMSNORM) {
    d = (const llmmm_a_planes_rmsnorm*)A;  // a host structure
    if (!d->planes || !d->residual || !d->hidden_out || !d->norm_weight) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
    if (d->hidden_dtype != LLMMM_DTYPE_F16 && d->hidden_dtype != LLMMM_DTYPE_BF16 && d->hidden_dtype != LLMMM_DTYPE_F32)
      return fail(LLMMM_ERR_UNSUPPORTED_TYPE, "T is not supported.");
    if (d->splits < 1 || d->splits > MAX_SPLIT_K) return fail(LLMMM_ERR_INVALID_ARGUMENT, "splits must be 1..%d (got %d)", MAX_SPLIT_K, d->splits);
    if (!(d->eps >= 0.f)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "eps must be non-negative");
    if (K > 10240) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the fused norm handles rows of at most 10240 columns (got %d)", K);
    if (!aligned16(d->planes) || !aligned16(d->residual) || !aligned16(d->hidden_out) || !aligned16(d->norm_weight))
      return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 16-byte aligned");
    // (every generating workgroup reads the residual while one writes the hidden state: an in-place update takes the
    // quantise-first route below, where one workgroup owns each row)
    if (tile == LLMMM_TILE_SKINNY && M <= AGEN2_MAX_M && K <= AGEN2_MAX_K && d->splits <= llmmm::SKINNY_GEN_MAX_PLANES && d->hidden_out != d->residual) {
      prep->agen         = 2;
      prep->hidden_dtype = d->hidden_dtype;
      prep->ag.planes = d->planes, prep->ag.residual = d->residual, prep->ag.hidden = d->hidden_out, prep->ag.w = d->norm_weight;
      prep->ag.eps = d->eps, prep->ag.splits = d->splits;
      return LLMMM_OK;
    }
  }
  else if (tile == LLMMM_TILE_SKINNY && M <= AGEN_MAX_M) {
    prep->agen = 1;
    return LLMMM_OK;
  }
  const size_t need = swiglu_a_bytes(M, K);
  if (!workspace || workspace_bytes < need)
    return fail(LLMMM_ERR_WORKSPACE, "workspace holds %zu bytes, quantising the activations first needs %zu", workspace ? workspace_bytes : (size_t)0, need);
  if (!aligned16(workspace)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "workspace must be 16-byte aligned");
  uint8_t*   hq = (uint8_t*)workspace;
  float*     hs = (float*)(hq + align256((size_t)M * K));
  hipError_t e;
  if (d)
    e = llmmm::planes_add_rmsnorm_quant_launch(d->hidden_dtype, d->planes, d->splits, d->residual, d->hidden_out, d->norm_weight, d->eps, hq, hs, M, K,
                                               (hipStream_t)stream);
  else
    e = llmmm::fp8_splitk_reduce_launch(LLMMM_OUT_FP8Q_SWIGLU, (const float*)A, 1, hq, hs, M, 2 * K, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "activation quantiser launch: %s", hipGetErrorString(e));
  A               = hq;
  As              = hs;
  workspace       = hq + need;
  workspace_bytes = workspace_bytes - need;
  if (workspace_bytes == 0) workspace = nullptr;
  return LLMMM_OK;
}

int llmmm_fp8_gemm_ex(int out_kind, const void* A, const float* As, const void* Bt, const float* Bs, void* C, float* Cs, int M,
                      int N, int K, void* workspace, size_t workspace_bytes, const llmmm_gemm_cfg* user, void* stream)
{
  if (out_kind < LLMMM_OUT_F32 || out_kind > LLMMM_OUT_FP8Q_SWIGLU) return fail(LLMMM_ERR_INVALID_ARGUMENT, "unknown output kind %d", out_kind);
  const bool     swiglu = out_kind == LLMMM_OUT_FP8Q_SWIGLU;
  llmmm_gemm_cfg cfg;
  const int      rc = choose_fp8_out(out_kind, M, N, K, &cfg);
  if (rc) return rc;
  const bool a_swiglu = user && user->a_layout == LLMMM_FP8_A_SWIGLU_F32;
  const bool a_made   = user && user->a_layout != LLMMM_FP8_A_QUANTISED;  // A is not the quantised operand: As is not used
  if (!A || (!As && !a_made) || !Bt || !Bs || !C) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (a_swiglu && swiglu) return fail(LLMMM_ERR_INVALID_ARGUMENT, "SwiGLU on both the A operand and the output");
  if ((out_kind == LLMMM_OUT_FP8Q || swiglu) && !Cs) return fail(LLMMM_ERR_INVALID_ARGUMENT, "C_scale_transposed is required for fp8 output");
  // (with a_layout = PLANES_RMSNORM, A is a host structure: prepare_a checks the device pointers inside it)
  const bool a_host = user && user->a_layout == LLMMM_FP8_A_PLANES_RMSNORM;
  if ((!a_host && !aligned16(A)) || !aligned16(Bt) || !aligned16(C)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 16-byte aligned");
  if ((long)M * K >= (1L << 31) || (long)N * K >= (1L << 31) || (long)M * N >= (1L << 31))
    return fail(LLMMM_ERR_INVALID_ARGUMENT, "matrix has 2^31 or more elements");
  if (user) {
    // (a named weight-streaming kernel where the library would have taken tiles: the split is that kernel's own heuristic)
    if (user->tile == LLMMM_TILE_SKINNY && cfg.tile == LLMMM_TILE_STRIP)
      cfg.split_k = skinny_split_for(M, N, K);  // (the split-K form named where the library would have taken strips)
    else if (user->tile == LLMMM_TILE_SKINNY && cfg.tile != LLMMM_TILE_SKINNY && M <= SKINNY_MAX_M)
      cfg.split_k = heuristic_split(M, N, K);
    if (user->tile != LLMMM_TILE_AUTO) cfg.tile = user->tile;
    if (user->split_k > 0) cfg.split_k = user->split_k;
    if (user->b_layout != LLMMM_FP8_B_ROWS && user->b_layout != LLMMM_FP8_B_PRESHUFFLED)
      return fail(LLMMM_ERR_INVALID_ARGUMENT, "unknown B layout %d", user->b_layout);
    cfg.b_layout = user->b_layout;
  }
  hipError_t e;
  APrep      prep;
  if (cfg.tile == LLMMM_TILE_SKINNY && M > SKINNY_MAX_M) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the weight-streaming kernel handles M <= %d", SKINNY_MAX_M);
  const int rca = prepare_a(user, cfg.tile, A, As, M, K, workspace, workspace_bytes, stream, &prep);
  if (rca) return rca;
  const int agen = prep.agen;
  if (cfg.tile == LLMMM_TILE_STRIP && (agen || (user && user->split_k > 1))) {
    // generated activations and an explicit split are the split-K form's: a strip the library picked itself gives way, one asked for is refused
    if (user && user->tile == LLMMM_TILE_STRIP) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the column-strip kernel takes quantised activations and does not split K over workgroups");
    cfg.tile = LLMMM_TILE_SKINNY;
    if (!(user && user->split_k > 0)) cfg.split_k = skinny_split_for(M, N, K);
  }
  int xarea = -1;
  if (cfg.tile == LLMMM_TILE_STRIP && out_kind == LLMMM_OUT_FP8Q && strip_fp8q_fits(M, N, K) && (xarea = strip_exchange_area(stream)) < 0 &&
      !(user && user->tile == LLMMM_TILE_STRIP)) {
    // more streams than exchange areas: a strip the library picked itself gives way to the split-K form
    cfg.tile    = LLMMM_TILE_SKINNY;
    cfg.split_k = skinny_split_for(M, N, K);
  }
  if (cfg.tile == LLMMM_TILE_STRIP) {
    if (out_kind == LLMMM_OUT_FP8Q) {
      if (!strip_fp8q_fits(M, N, K))
        return fail(LLMMM_ERR_INVALID_ARGUMENT, "the column-strip kernel quantises C for M <= 16, K >= 1024 and at most %d column groups", llmmm::STRIP_XCH_MAX_GROUPS);
      if (xarea < 0) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the column-strip kernel's fp8 output serves %d streams per process", llmmm::STRIP_XCH_AREAS);
      e = llmmm::fp8_strip_fp8q_launch(cfg.b_layout, A, As, Bt, Bs, C, Cs, M, N, K, xarea, (hipStream_t)stream);
    }
    else {
      if (out_kind != LLMMM_OUT_F32 && out_kind != LLMMM_OUT_BF16) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the column-strip kernel has fp32, bf16 and fp8 (1x128) outputs only");
      if (!strip_fits(M, N, K)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the column-strip kernel handles M <= %d and K >= 1024", llmmm::STRIP_MAX_M);
      e = llmmm::fp8_strip_launch(out_kind, cfg.b_layout, A, As, Bt, Bs, C, M, N, K, (hipStream_t)stream);
    }
  }
  else if (cfg.tile == LLMMM_TILE_SKINNY) {
    int split = cfg.split_k;
    if (split > max_split_for(K)) split = max_split_for(K);
    if (split < 1) split = 1;
    if (!workspace) split = 1;  // documented: no workspace, no split
    const int min_split = agen ? agen_min_split(K) : 1;  // generated activations: a split's K range must fit the staging buffer
    if (split < min_split) {
      if ((user && user->split_k > 0) || !workspace)
        return fail(user && user->split_k > 0 ? LLMMM_ERR_INVALID_ARGUMENT : LLMMM_ERR_WORKSPACE,
                    "generated activations need split-K >= %d for K = %d (at most %d slices of 128 per split), and a workspace for it", min_split, K, AGEN_MAX_SLICES);
      split = min_split;
    }
    float* partial = nullptr;
    int    pair_area;
    if (swiglu && !workspace) return fail(LLMMM_ERR_WORKSPACE, "the SwiGLU output at M <= %d needs a workspace of at least M * N floats", SKINNY_MAX_M);
    if (split > 1 && !(user && user->split_k > 0)) {
      // a split the library chose itself shrinks to what the caller's workspace holds
      const size_t room = workspace_bytes / ((size_t)M * N * sizeof(float));
      if ((size_t)split > room) split = room < 2 ? 1 : (int)room;
      if (split < min_split) split = min_split;  // (fails the size check below)
    }
    // (the norm-generating kernel only writes fp32: any other output goes through one plane and the reduce kernel)
    if (split > 1 || swiglu || (agen == 2 && out_kind != LLMMM_OUT_F32)) {
      const size_t need = (size_t)split * M * N * sizeof(float);
      if (!workspace || workspace_bytes < need) return fail(LLMMM_ERR_WORKSPACE, "workspace holds %zu bytes, split-K %d needs %zu", workspace ? workspace_bytes : (size_t)0, split, need);
      if (!aligned16(workspace)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "workspace must be 16-byte aligned");
      partial = (float*)workspace;
    }
    const bool wide = swiglu && !agen && !(user && (user->split_k > 0 || user->tile != LLMMM_TILE_AUTO)) && swiglu_wide_tail(M, N, K);
    const bool pair = swiglu && !wide && !agen && !(user && user->split_k > 0) && swiglu_pair_pays(M, N, K, cfg.b_layout == LLMMM_FP8_B_PRESHUFFLED) && (pair_area = strip_exchange_area(stream)) >= 0;
    if (wide)
      e = llmmm::fp8_gemm_launch(out_kind, LLMMM_TILE_128x256, cfg.b_layout, A, As, Bt, Bs, C, Cs, M, N, K, 1, nullptr, (hipStream_t)stream), partial = nullptr;
    else if (pair)
      e = llmmm::fp8_skinny_swiglu_launch(cfg.b_layout, A, As, Bt, Bs, C, Cs, M, N, K, pair_area, (hipStream_t)stream), partial = nullptr;
    else if (agen == 2)
      e = llmmm::fp8_skinny_rmsnorm_a_launch(prep.hidden_dtype, cfg.b_layout, prep.ag, Bt, Bs, (float*)C, M, N, K, split, partial, (hipStream_t)stream);
    else if (agen)
      e = llmmm::fp8_skinny_swiglu_a_launch(partial ? LLMMM_OUT_F32 : out_kind, cfg.b_layout, (const float*)A, Bt, Bs, C, Cs, M, N, K, split, partial,
                                            (hipStream_t)stream);
    else
      e = llmmm::fp8_skinny_launch(partial ? LLMMM_OUT_F32 : out_kind, cfg.b_layout, A, As, Bt, Bs, C, Cs, M, N, K, split, partial, (hipStream_t)stream);
    if (e == hipSuccess && partial) e = llmmm::fp8_splitk_reduce_launch(out_kind, partial, split, C, Cs, M, N, (hipStream_t)stream);
  }
  else {
    int bm, bn;
    if (!tile_dims(cfg.tile, bm, bn) || fp16_only(cfg.tile)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "unknown tile id %d", cfg.tile);
    if (cfg.tile == LLMMM_TILE_128x160 && (out_kind == LLMMM_OUT_FP8Q || swiglu)) {
      // its waves straddle the 1x128 groups of the fused quantisation: a tile the library picked itself gives way, one asked for is refused
      if (user && user->tile == LLMMM_TILE_128x160) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the 128 x 160 tile has no fp8 output");
      cfg.tile = LLMMM_TILE_128x128;
      tile_dims(cfg.tile, bm, bn);
    }
    // (128 x 128 tiles also take a single tile row of fewer than 128 rows)
    if ((M % bm && !(cfg.tile == LLMMM_TILE_128x128 && M < 128)) || N % bn) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
    if (user && user->tile != LLMMM_TILE_AUTO && user->split_k <= 0) cfg.split_k = heuristic_tile_split(cfg.tile, M < bm ? bm : M, N, K);
    int split = cfg.split_k;
    if (split > K / 128) split = K / 128;
    if (split > MAX_SPLIT_K) split = MAX_SPLIT_K;
    if (split < 1 || !workspace) split = 1;  // documented: no workspace, no split
    float* planes = nullptr;
    if (split > 1 && !(user && user->split_k > 0)) {
      // a split the library chose itself shrinks to what the caller's workspace holds
      const size_t plane = (size_t)M * N * sizeof(float);
      const size_t room  = workspace_bytes / plane;
      if ((size_t)split > room) split = room < 2 ? 1 : (int)room;
    }
    if (swiglu && split <= 1 && bn != 256 && (!workspace || workspace_bytes < (size_t)M * N * sizeof(float))) {
      // no room for the fp32 plane a 128-column tile needs: the fused epilogue of a 256-column tile instead
      if ((user && user->tile != LLMMM_TILE_AUTO) || M % 128)
        return fail(LLMMM_ERR_WORKSPACE, "the SwiGLU output from a 128-column tile needs a workspace of M * N floats");
      cfg.tile = LLMMM_TILE_128x256;
      bn       = 256;
    }
    if (split > 1 || (swiglu && bn != 256)) {
      const size_t need = (size_t)split * M * N * sizeof(float);
      if (workspace_bytes < need) return fail(LLMMM_ERR_WORKSPACE, "workspace holds %zu bytes, split-K %d needs %zu", workspace_bytes, split, need);
      if (!aligned16(workspace)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "workspace must be 16-byte aligned");
      planes = (float*)workspace;
    }
    int pair_area;
    if (swiglu && cfg.tile == LLMMM_TILE_128x128 && split <= 1 && !(user && (user->split_k > 0 || user->tile != LLMMM_TILE_AUTO)) && swiglu_wide_tail(M, N, K))
      e = llmmm::fp8_gemm_launch(out_kind, LLMMM_TILE_128x256, cfg.b_layout, A, As, Bt, Bs, C, Cs, M, N, K, 1, nullptr, (hipStream_t)stream);
    else if (swiglu && cfg.tile == LLMMM_TILE_128x128 && split <= 1 && !(user && user->split_k > 0) && llmmm::fp8_gemm_swiglu_pair_fits(M, N, K) &&
             !(M <= 64 && cfg.b_layout == LLMMM_FP8_B_PRESHUFFLED && swiglu_pair_camps(N, K)) && (pair_area = strip_exchange_area(stream)) >= 0)
      e = llmmm::fp8_gemm_swiglu_pair_launch(cfg.b_layout, A, As, Bt, Bs, C, Cs, M, N, K, pair_area, (hipStream_t)stream);
    else
      e = llmmm::fp8_gemm_launch(out_kind, cfg.tile, cfg.b_layout, A, As, Bt, Bs, C, Cs, M, N, K, split, planes, (hipStream_t)stream);
  }
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "fp8 gemm launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

int llmmm_fp8_gemm(int out_kind, const void* A, const float* As, const void* Bt, const float* Bs, void* C, float* Cs, int M, int N,
                   int K, void* workspace, size_t workspace_bytes, void* stream)
{
  return llmmm_fp8_gemm_ex(out_kind, A, As, Bt, Bs, C, Cs, M, N, K, workspace, workspace_bytes, nullptr, stream);
}

int llmmm_quant_fp8(int kind, const float* x, void* q, float* scale, int M, int N, void* stream)
{
  if (kind < LLMMM_QUANT_1x128_T || kind > LLMMM_QUANT_128x128_T) return fail(LLMMM_ERR_INVALID_ARGUMENT, "unknown quantiser kind %d", kind);
  if (M <= 0 || N <= 0) return fail(LLMMM_ERR_INVALID_ARGUMENT, "M and N must be positive (got %d, %d)", M, N);
  if (N % 4) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
  if (!x || !q || !scale) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (!aligned16(x) || (reinterpret_cast<uintptr_t>(q) & 3u)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "x must be 16-byte and q 4-byte aligned");
  if ((long)M * N >= (1L << 31)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "matrix has 2^31 or more elements");
  const int quant_m   = (kind == LLMMM_QUANT_1x128_T || kind == LLMMM_QUANT_1x128) ? 1 : 128;
  const int transpose = (kind == LLMMM_QUANT_1x128_T || kind == LLMMM_QUANT_128x128_T) ? 1 : 0;
  const hipError_t e  = llmmm::quant_fp8_launch(quant_m, transpose, x, q, scale, M, N, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "quantiser launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

int llmmm_rmsnorm_quant_fp8(int in_dtype, const void* x, const float* weight, float eps, void* q, float* scale, int M, int K, void* stream)
{
  if (in_dtype != LLMMM_DTYPE_F16 && in_dtype != LLMMM_DTYPE_BF16 && in_dtype != LLMMM_DTYPE_F32) return fail(LLMMM_ERR_UNSUPPORTED_TYPE, "T is not supported.");
  if (M <= 0 || K <= 0) return fail(LLMMM_ERR_INVALID_ARGUMENT, "M and K must be positive (got %d, %d)", M, K);
  if (K % 128) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
  if (!x || !weight || !q || !scale) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (!(eps >= 0.f)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "eps must be non-negative");
  if (!aligned16(x) || !aligned16(weight) || !aligned16(q)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 16-byte aligned");
  if ((long)M * K >= (1L << 31)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "matrix has 2^31 or more elements");
  const hipError_t e = llmmm::rmsnorm_quant_launch(in_dtype, x, weight, eps, q, scale, M, K, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "rmsnorm + quantiser launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

int llmmm_probe_mfma(int kind, const void* operands, float* sink, int workgroups, int iters, void* stream)
{
  if (kind < 0 || kind > LLMMM_PROBE_FP8) return fail(LLMMM_ERR_UNSUPPORTED_TYPE, "T is not supported.");
  if (!operands || !sink) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (!aligned16(operands) || (reinterpret_cast<uintptr_t>(operands) & 31u)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "operands must be 32-byte aligned");
  if (workgroups <= 0 || workgroups > 65536 || iters <= 0) return fail(LLMMM_ERR_INVALID_ARGUMENT, "workgroups must be 1..65536 and iters positive");
  const hipError_t e = llmmm::probe_mfma_launch(kind, operands, sink, workgroups, iters, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "probe launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

double llmmm_probe_mfma_flops(int kind, int workgroups, int iters)
{
  if (kind < 0 || kind > LLMMM_PROBE_FP8 || workgroups <= 0 || iters <= 0) return 0.0;
  return llmmm::probe_mfma_flops(kind, workgroups, iters);
}

int llmmm_probe_hbm_read(const void* src, size_t bytes, float* sink, int workgroups, void* stream)
{
  if (!src || !sink) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (!aligned16(src) || bytes == 0 || bytes % 16) return fail(LLMMM_ERR_INVALID_ARGUMENT, "src must be 16-byte aligned and bytes a positive multiple of 16");
  if (workgroups <= 0 || workgroups > 65536) return fail(LLMMM_ERR_INVALID_ARGUMENT, "workgroups must be 1..65536");
  const hipError_t e = llmmm::probe_stream_read_launch(src, bytes, sink, workgroups, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "probe launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

// Workspace of the entry points whose epilogue runs either inside an unsplit tile kernel (no planes) or in a second
// kernel behind fp32 planes: the same decision as resolve_plane_cfg takes for a call without cfg.  A single tile row of
// fewer than 128 rows (64 < M < 128 in 128 x 128 tiles) has no epilogue of its own and always goes through one plane.
static size_t plane_route_workspace(int M, int N, int K, bool wide_ok)
{
  if (M <= 0 || N <= 0 || K <= 0 || N % 128 || K % 128) return 0;
  llmmm_gemm_cfg cfg;
  if (choose_fp8(M, N, K, &cfg) != LLMMM_OK) return 0;
  if (wide_ok) prefer_wide_tile(&cfg, M, N, K), prefer_strip(&cfg, M, N, K);
  if (cfg.tile == LLMMM_TILE_STRIP) return strip_fallback_plane_bytes(M, N, K);  // strips need none (epilogue inside the kernel); a call with generated activations leaves them
  int split = cfg.split_k < 1 ? 1 : cfg.split_k;
  if (split > max_split_for(K)) split = max_split_for(K);
  int bm = 0, bn = 0;
  if (cfg.tile != LLMMM_TILE_SKINNY && tile_dims(cfg.tile, bm, bn) && M % bm == 0 && split == 1) return 0;  // epilogue inside the tile kernel
  return (size_t)split * M * N * sizeof(float);
}

int llmmm_probe_strip_exchange_timeouts(unsigned* count)
{
  if (!count) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  const hipError_t e = llmmm::strip_exchange_timeouts(count);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "reading the exchange's time-out counter: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

size_t llmmm_probe_phases_bytes(int M, int N)
{
  if (M <= 0 || N <= 0 || M % 256 || N % 256) return 0;
  return (size_t)(M / 256) * (N / 256) * 8 * llmmm::PHASE_RECORD * sizeof(unsigned long long);
}

int llmmm_probe_fp8_gemm_phases(const void* A, const float* As, const void* Bt, const float* Bs, void* C, float* Cs, int M, int N, int K, void* stamps,
                                size_t stamps_bytes, void* stream)
{
  if (M <= 0 || N <= 0 || K <= 0) return fail(LLMMM_ERR_INVALID_ARGUMENT, "M, N and K must be positive (got %d, %d, %d)", M, N, K);
  if (M % 256 || N % 256 || K % 128) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
  if (!A || !As || !Bt || !Bs || !C || !Cs || !stamps) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (!aligned16(A) || !aligned16(Bt) || !aligned16(C) || !aligned16(stamps)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 16-byte aligned");
  if (stamps_bytes < llmmm_probe_phases_bytes(M, N)) return fail(LLMMM_ERR_WORKSPACE, "stamps holds %zu bytes, %zu needed", stamps_bytes, llmmm_probe_phases_bytes(M, N));
  const hipError_t e = llmmm::fp8_gemm_phases_launch(A, As, Bt, Bs, C, Cs, M, N, K, (unsigned long long*)stamps, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "probe launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

int llmmm_probe_fp16_gemm_phases(int dtype, const void* A, const void* B, void* C, int M, int N, int K, void* stamps, size_t stamps_bytes, void* stream)
{
  if (dtype != LLMMM_DTYPE_F16 && dtype != LLMMM_DTYPE_BF16) return fail(LLMMM_ERR_UNSUPPORTED_TYPE, "T is not supported.");
  if (M <= 0 || N <= 0 || K <= 0) return fail(LLMMM_ERR_INVALID_ARGUMENT, "M, N and K must be positive (got %d, %d, %d)", M, N, K);
  if (M % 256 || N % 256 || K % 32) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
  if (!A || !B || !C || !stamps) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (!aligned16(A) || !aligned16(B) || !aligned16(C) || !aligned16(stamps)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 16-byte aligned");
  if (stamps_bytes < llmmm_probe_phases_bytes(M, N)) return fail(LLMMM_ERR_WORKSPACE, "stamps holds %zu bytes, %zu needed", stamps_bytes, llmmm_probe_phases_bytes(M, N));
  const hipError_t e = llmmm::fp16_gemm_phases_launch(dtype, A, B, C, M, N, K, (unsigned long long*)stamps, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "probe launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

size_t llmmm_fp8_gemm_add_rmsnorm_quant_workspace(int M, int N, int K) { return plane_route_workspace(M, N, K, true); }

// Kernel and split for the entry points whose epilogue lives in a second kernel behind fp32 planes, chosen and
// validated as llmmm_fp8_gemm_ex does.  split == 0 on return: a tile kernel without split, which `allow_direct`
// callers run with the epilogue inside the kernel (no planes, no workspace); otherwise split >= 1 planes are needed
// and the workspace has been checked to hold them.
struct PlaneCfg {
  int  tile = 0, split = 0, b_layout = 0;
  bool  skinny = false;
  bool  strip  = false;  // the weight-streaming kernel in column strips: one launch, its fp32 result is the one "plane"
  APrep prep;
};
static int resolve_plane_cfg(const void*& A, const float*& As, const void* Bt, const float* Bs, int M, int N, int K, void*& workspace,
                             size_t& workspace_bytes, const llmmm_gemm_cfg* user, bool allow_direct, PlaneCfg* out, void* stream, bool wide_ok = true)
{
  llmmm_gemm_cfg cfg;
  const int      rc = choose_fp8(M, N, K, &cfg);
  if (rc) return rc;
  if (wide_ok) prefer_wide_tile(&cfg, M, N, K);
  // (wide_ok also stands for "no 1x128-grouped epilogue behind the GEMM": the callers that may take column strips.  Not with
  // activations the kernel has to make itself, nor against an explicit split.)
  if (wide_ok && !(user && (user->a_layout != LLMMM_FP8_A_QUANTISED || user->split_k > 0 || user->tile != LLMMM_TILE_AUTO))) prefer_strip(&cfg, M, N, K);
  const bool a_made = user && user->a_layout != LLMMM_FP8_A_QUANTISED;
  if (!A || (!As && !a_made) || !Bt || !Bs) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  const bool a_host = user && user->a_layout == LLMMM_FP8_A_PLANES_RMSNORM;  // a host structure, checked by prepare_a
  if ((!a_host && !aligned16(A)) || !aligned16(Bt)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 16-byte aligned");
  if ((long)M * K >= (1L << 31) || (long)N * K >= (1L << 31) || (long)M * N >= (1L << 31))
    return fail(LLMMM_ERR_INVALID_ARGUMENT, "matrix has 2^31 or more elements");
  if (user) {
    // (a named weight-streaming kernel where the library would have taken tiles: the split is that kernel's own heuristic)
    if (user->tile == LLMMM_TILE_SKINNY && cfg.tile != LLMMM_TILE_SKINNY && M <= SKINNY_MAX_M) cfg.split_k = heuristic_split(M, N, K);
    if (user->tile != LLMMM_TILE_AUTO) cfg.tile = user->tile;
    if (user->split_k > 0) cfg.split_k = user->split_k;
    if (user->b_layout != LLMMM_FP8_B_ROWS && user->b_layout != LLMMM_FP8_B_PRESHUFFLED)
      return fail(LLMMM_ERR_INVALID_ARGUMENT, "unknown B layout %d", user->b_layout);
    cfg.b_layout = user->b_layout;
  }
  int bm = 0, bn = 0;
  const bool skinny = cfg.tile == LLMMM_TILE_SKINNY;
  if (cfg.tile == LLMMM_TILE_STRIP) {
    if (!wide_ok) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the column-strip kernel cannot hold whole heads");
    if (a_made || (user && user->split_k > 1)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the column-strip kernel takes quantised activations and does not split K over workgroups");
    if (!strip_fits(M, N, K)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the column-strip kernel handles M <= %d and K >= 1024", llmmm::STRIP_MAX_M);
    out->prep = APrep();
    out->tile = cfg.tile, out->b_layout = cfg.b_layout, out->skinny = false, out->strip = true;
    if (allow_direct) {
      out->split = 0;  // the caller's epilogue is the strip kernel's own (residual add): no planes
      return LLMMM_OK;
    }
    const size_t plane1 = (size_t)M * N * sizeof(float);
    if (!workspace || workspace_bytes < plane1) return fail(LLMMM_ERR_WORKSPACE, "workspace holds %zu bytes, one fp32 plane needs %zu", workspace ? workspace_bytes : (size_t)0, plane1);
    if (!aligned16(workspace)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "workspace must be 16-byte aligned");
    out->split = 1;
    return LLMMM_OK;
  }
  if (skinny) {
    if (M > SKINNY_MAX_M) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the weight-streaming kernel handles M <= %d", SKINNY_MAX_M);
  }
  else {
    if (!tile_dims(cfg.tile, bm, bn) || fp16_only(cfg.tile)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "unknown tile id %d", cfg.tile);
    if ((M % bm && !(cfg.tile == LLMMM_TILE_128x128 && M < 128)) || N % bn) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N or K are not aligned.");
    if (user && user->tile != LLMMM_TILE_AUTO && user->split_k <= 0) cfg.split_k = heuristic_tile_split(cfg.tile, M < bm ? bm : M, N, K);
  }
  // the A operand given as the fp32 gate_up result: generated by the kernel, or quantised into the front of the workspace now
  const int rca = prepare_a(user, cfg.tile, A, As, M, K, workspace, workspace_bytes, stream, &out->prep);
  if (rca) return rca;
  int split = cfg.split_k < 1 ? 1 : cfg.split_k;
  if (split > max_split_for(K)) split = max_split_for(K);
  const size_t plane    = (size_t)M * N * sizeof(float);
  const bool   explicit_split = user && user->split_k > 0;
  const int    min_split = out->prep.agen ? agen_min_split(K) : 1;
  if (split < min_split) {
    if (explicit_split) return fail(LLMMM_ERR_INVALID_ARGUMENT, "generated activations need split-K >= %d for K = %d", min_split, K);
    split = min_split;
  }
  out->tile = cfg.tile, out->b_layout = cfg.b_layout, out->skinny = skinny;
  // (a row tail -- M < 128 in 128 x 128 tiles -- has no direct epilogues: always through planes)
  if (allow_direct && !skinny && M % bm == 0 && (split == 1 || (!explicit_split && (!workspace || workspace_bytes < 2 * plane)))) {
    out->split = 0;  // also when a split the library chose itself finds no room for two planes
    return LLMMM_OK;
  }
  if (!workspace || workspace_bytes < plane) return fail(LLMMM_ERR_WORKSPACE, "workspace holds %zu bytes, one fp32 plane needs %zu", workspace ? workspace_bytes : (size_t)0, plane);
  if (!aligned16(workspace)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "workspace must be 16-byte aligned");
  if ((size_t)split * plane > workspace_bytes) {
    if (explicit_split) return fail(LLMMM_ERR_WORKSPACE, "workspace holds %zu bytes, split-K %d needs %zu", workspace_bytes, split, (size_t)split * plane);
    split = (int)(workspace_bytes / plane);  // a split the library chose itself shrinks to the workspace (>= 1: checked above)
    if (split < min_split) return fail(LLMMM_ERR_WORKSPACE, "workspace holds %zu bytes, generated activations need split-K %d: %zu", workspace_bytes, min_split, (size_t)min_split * plane);
  }
  out->split = split;
  return LLMMM_OK;
}

static int launch_into_planes(const PlaneCfg& pc, const void* A, const float* As, const void* Bt, const float* Bs, int M, int N, int K,
                              void* workspace, void* stream)
{
  float*     planes = (float*)workspace;
  hipError_t e;
  if (pc.strip)
    e = llmmm::fp8_strip_launch(LLMMM_OUT_F32, pc.b_layout, A, As, Bt, Bs, planes, M, N, K, (hipStream_t)stream);
  else if (pc.skinny && pc.prep.agen == 2)
    e = llmmm::fp8_skinny_rmsnorm_a_launch(pc.prep.hidden_dtype, pc.b_layout, pc.prep.ag, Bt, Bs, nullptr, M, N, K, pc.split, planes, (hipStream_t)stream);
  else if (pc.skinny && pc.prep.agen == 1)
    e = llmmm::fp8_skinny_swiglu_a_launch(LLMMM_OUT_F32, pc.b_layout, (const float*)A, Bt, Bs, nullptr, nullptr, M, N, K, pc.split, planes, (hipStream_t)stream);
  else if (pc.skinny)
    e = llmmm::fp8_skinny_launch(LLMMM_OUT_F32, pc.b_layout, A, As, Bt, Bs, nullptr, nullptr, M, N, K, pc.split, planes, (hipStream_t)stream);
  else
    e = llmmm::fp8_gemm_launch(LLMMM_OUT_F32, pc.tile, pc.b_layout, A, As, Bt, Bs, nullptr, nullptr, M, N, K, pc.split, planes, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "fp8 gemm launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

size_t llmmm_fp8_gemm_planes_bytes(int M, int N, int K)
{
  if (M <= 0 || N <= 0 || K <= 0 || N % 128 || K % 128) return 0;
  llmmm_gemm_cfg cfg;
  if (choose_fp8(M, N, K, &cfg) != LLMMM_OK) return 0;
  const size_t own = (size_t)(cfg.split_k < 1 ? 1 : cfg.split_k) * M * N * sizeof(float);
  prefer_strip(&cfg, M, N, K);  // (strips write one plane; a call with generated activations leaves them for the split-K form)
  if (cfg.tile == LLMMM_TILE_STRIP) {
    const size_t fb = strip_fallback_plane_bytes(M, N, K);
    return fb > own ? fb : own;
  }
  return own;
}

int llmmm_fp8_gemm_planes(const void* A, const float* As, const void* Bt, const float* Bs, int M, int N, int K, float* planes, size_t planes_bytes,
                          int* splits, void* workspace, size_t workspace_bytes, const llmmm_gemm_cfg* user, void* stream)
{
  if (!splits || !planes) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  llmmm_gemm_cfg probe;
  int            rc = choose_fp8(M, N, K, &probe);
  if (rc) return rc;
  llmmm_gemm_cfg inner;
  inner.tile = LLMMM_TILE_AUTO, inner.split_k = 0, inner.b_layout = LLMMM_FP8_B_ROWS, inner.a_layout = LLMMM_FP8_A_QUANTISED;
  if (user) inner = *user;
  if (inner.a_layout != LLMMM_FP8_A_QUANTISED) {
    // an operand the library has to quantise first goes to `workspace` (the planes have a buffer of their own); one the
    // kernel generates is resolved a second time inside resolve_plane_cfg, which launches nothing for it
    if (!A) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
    const int tile = inner.tile != LLMMM_TILE_AUTO ? inner.tile : probe.tile;
    APrep     prep;
    rc = prepare_a(&inner, tile, A, As, M, K, workspace, workspace_bytes, stream, &prep);
    if (rc) return rc;
    if (prep.agen == 0) inner.a_layout = LLMMM_FP8_A_QUANTISED;
  }
  PlaneCfg pc;
  void*    pw = planes;
  size_t   pb = planes_bytes;
  rc = resolve_plane_cfg(A, As, Bt, Bs, M, N, K, pw, pb, &inner, false, &pc, stream);
  if (rc) return rc;
  rc = launch_into_planes(pc, A, As, Bt, Bs, M, N, K, pw, stream);
  if (rc) return rc;
  *splits = pc.split;
  return LLMMM_OK;
}

int llmmm_fp8_gemm_add_rmsnorm_quant(const void* A, const float* As, const void* Bt, const float* Bs, int hidden_dtype, const void* residual,
                                     void* hidden_out, const float* norm_weight, float eps, void* q, float* q_scale, int M, int N, int K,
                                     void* workspace, size_t workspace_bytes, const llmmm_gemm_cfg* user, void* stream)
{
  if (hidden_dtype != LLMMM_DTYPE_F16 && hidden_dtype != LLMMM_DTYPE_BF16 && hidden_dtype != LLMMM_DTYPE_F32)
    return fail(LLMMM_ERR_UNSUPPORTED_TYPE, "T is not supported.");
  llmmm_gemm_cfg probe;
  const int      rc0 = choose_fp8(M, N, K, &probe);  // shape checks first, with the reference's texts
  if (rc0) return rc0;
  if (N > 10240) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the fused norm handles rows of at most 10240 columns (got %d)", N);
  if (!residual || !hidden_out || !norm_weight || !q || !q_scale) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (!(eps >= 0.f)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "eps must be non-negative");
  if (!aligned16(residual) || !aligned16(hidden_out) || !aligned16(norm_weight) || !aligned16(q))
    return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 16-byte aligned");
  PlaneCfg pc;
  int      rc = resolve_plane_cfg(A, As, Bt, Bs, M, N, K, workspace, workspace_bytes, user, true, &pc, stream);
  if (rc) return rc;
  if (pc.split == 0) {
    // a tile kernel without split, or column strips: the residual is added in its epilogue, the norm + quantiser kernel follows on the
    // stored hidden state (the same two operations on the same values as behind planes, without the fp32 round trip)
    hipError_t e = pc.strip ? llmmm::fp8_strip_add_residual_launch(hidden_dtype, pc.b_layout, A, As, Bt, Bs, residual, hidden_out, M, N, K, (hipStream_t)stream)
                            : llmmm::fp8_gemm_add_residual_launch(hidden_dtype, pc.tile, pc.b_layout, A, As, Bt, Bs, residual, hidden_out, M, N, K, (hipStream_t)stream);
    if (e == hipSuccess) e = llmmm::rmsnorm_quant_launch(hidden_dtype, hidden_out, norm_weight, eps, q, q_scale, M, N, (hipStream_t)stream);
    if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "fp8 gemm + add, rmsnorm + quantiser launch: %s", hipGetErrorString(e));
    return LLMMM_OK;
  }
  rc = launch_into_planes(pc, A, As, Bt, Bs, M, N, K, workspace, stream);
  if (rc) return rc;
  const hipError_t e = llmmm::planes_add_rmsnorm_quant_launch(hidden_dtype, (const float*)workspace, pc.split, residual, hidden_out, norm_weight, eps, q,
                                                              q_scale, M, N, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "add + rmsnorm + quantiser launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

size_t llmmm_fp8_gemm_qkv_rope_workspace(int M, int N, int K) { return plane_route_workspace(M, N, K, false); }

int llmmm_fp8_gemm_qkv_rope(int out_kind, const void* A, const float* As, const void* Bt, const float* Bs, void* out, float* out_scale,
                            const float* q_norm_weight, const float* k_norm_weight, float eps, const float* cos_table, const float* sin_table,
                            int table_rows, const int* positions, int n_q_heads, int n_kv_heads, int M, int N, int K, void* workspace,
                            size_t workspace_bytes, const llmmm_gemm_cfg* user, void* stream)
{
  if (out_kind != LLMMM_OUT_BF16 && out_kind != LLMMM_OUT_FP8Q) return fail(LLMMM_ERR_INVALID_ARGUMENT, "output kind %d: bf16 or fp8 (1x128) only", out_kind);
  llmmm_gemm_cfg probe;
  const int      rc0 = choose_fp8(M, N, K, &probe);
  if (rc0) return rc0;
  if (n_q_heads < 1 || n_kv_heads < 1 || (long)(n_q_heads + 2L * n_kv_heads) * 128 != N)
    return fail(LLMMM_ERR_INVALID_ARGUMENT, "N = %d is not (n_q_heads + 2 n_kv_heads) * 128 with %d query and %d key/value heads", N, n_q_heads, n_kv_heads);
  if (!out || !cos_table || !sin_table || !positions) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (out_kind == LLMMM_OUT_FP8Q && !out_scale) return fail(LLMMM_ERR_INVALID_ARGUMENT, "out_scale is required for fp8 output");
  if (table_rows < 1) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the cos / sin tables need at least one row");
  if (!(eps >= 0.f)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "eps must be non-negative");
  if (!aligned16(out) || !aligned16(cos_table) || !aligned16(sin_table) || (q_norm_weight && !aligned16(q_norm_weight)) ||
      (k_norm_weight && !aligned16(k_norm_weight)) || (reinterpret_cast<uintptr_t>(positions) & 3u))
    return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 16-byte aligned (positions: 4-byte)");
  PlaneCfg pc;
  int      rc = resolve_plane_cfg(A, As, Bt, Bs, M, N, K, workspace, workspace_bytes, user, true, &pc, stream, false);
  if (rc) return rc;
  if (pc.skinny && !pc.prep.agen && !(user && (user->split_k > 0 || user->tile != LLMMM_TILE_AUTO))) {
    // one launch where it is the faster form: column strips, or whole heads per workgroup in row groups
    const int  group  = rope_row_group(M, N, K, pc.split);
    int        area   = -1;
    const bool strips = out_kind == LLMMM_OUT_BF16 && rope_strips_pay(M, N, K) && (area = strip_exchange_area(stream)) >= 0;
    if (strips || group) {
      llmmm::Fp8HeadOp op;
      op.qw = q_norm_weight, op.kw = k_norm_weight, op.cos_t = cos_table, op.sin_t = sin_table, op.pos = positions;
      op.eps = eps, op.table_rows = table_rows, op.n_q = n_q_heads, op.n_kv = n_kv_heads;
      const hipError_t e = strips ? llmmm::fp8_strip_rope_launch(pc.b_layout, A, As, Bt, Bs, out, M, N, K, op, area, (hipStream_t)stream)
                                  : llmmm::fp8_skinny_rope_launch(out_kind, group, pc.b_layout, A, As, Bt, Bs, out, out_scale, M, N, K, op, (hipStream_t)stream);
      if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "fp8 gemm + qk-norm + rope launch: %s", hipGetErrorString(e));
      return LLMMM_OK;
    }
  }
  if (pc.tile == LLMMM_TILE_128x160) return fail(LLMMM_ERR_INVALID_ARGUMENT, "the 128 x 160 tile cannot hold whole heads");
  if (pc.split == 0) {  // a tile kernel without split: norm and rope run on the accumulators, no planes
    llmmm::Fp8HeadOp op;
    op.qw = q_norm_weight, op.kw = k_norm_weight, op.cos_t = cos_table, op.sin_t = sin_table, op.pos = positions;
    op.eps = eps, op.table_rows = table_rows, op.n_q = n_q_heads, op.n_kv = n_kv_heads;
    const hipError_t e = llmmm::fp8_gemm_qk_rope_launch(out_kind, pc.tile, pc.b_layout, A, As, Bt, Bs, out, out_scale, M, N, K, op, (hipStream_t)stream);
    if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "fp8 gemm + qk-norm + rope launch: %s", hipGetErrorString(e));
    return LLMMM_OK;
  }
  rc = launch_into_planes(pc, A, As, Bt, Bs, M, N, K, workspace, stream);
  if (rc) return rc;
  const hipError_t e = llmmm::fp8_planes_qk_norm_rope_launch(out_kind, (const float*)workspace, pc.split, out, out_scale, q_norm_weight, k_norm_weight, eps,
                                                             cos_table, sin_table, table_rows, positions, n_q_heads, n_kv_heads, M, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "qk-norm + rope launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

static int preshuffle(int inverse, const void* src, void* dst, int N, int K, void* stream)
{
  if (N <= 0 || K <= 0) return fail(LLMMM_ERR_INVALID_ARGUMENT, "N and K must be positive (got %d, %d)", N, K);
  if (K % 128) return fail(LLMMM_ERR_NOT_ALIGNED, "K must be greater than 0 and divisible by 128.");
  if (N % 16) return fail(LLMMM_ERR_NOT_ALIGNED, "N must be divisible by 16.");
  if (!src || !dst) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if (!aligned16(src) || !aligned16(dst)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 16-byte aligned");
  if ((long)N * K >= (1L << 31)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "matrix has 2^31 or more elements");
  const char *a = (const char*)src, *b = (const char*)dst;
  if (a < b + (size_t)N * K && b < a + (size_t)N * K) return fail(LLMMM_ERR_INVALID_ARGUMENT, "source and destination overlap");
  const hipError_t e = llmmm::fp8_preshuffle_launch(inverse, src, dst, N, K, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "pre-shuffle launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

int llmmm_fp8_preshuffle_b(const void* Bt, void* Bp, int N, int K, void* stream) { return preshuffle(0, Bt, Bp, N, K, stream); }
int llmmm_fp8_unshuffle_b(const void* Bp, void* Bt, int N, int K, void* stream) { return preshuffle(1, Bp, Bt, N, K, stream); }

int llmmm_transpose(int elem_size, const void* src, void* dst, int M, int N, void* stream)
{
  if (elem_size != 1 && elem_size != 4) return fail(LLMMM_ERR_UNSUPPORTED_TYPE, "T is not supported.");
  if (M <= 0 || N <= 0) return fail(LLMMM_ERR_INVALID_ARGUMENT, "M and N must be positive (got %d, %d)", M, N);
  if (M % 128 || N % 128) return fail(LLMMM_ERR_NOT_ALIGNED, "M or N can't be divided 128.");
  if (!src || !dst) return fail(LLMMM_ERR_INVALID_ARGUMENT, "null pointer");
  if ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 3u) return fail(LLMMM_ERR_INVALID_ARGUMENT, "pointers must be 4-byte aligned");
  if ((long)M * N >= (1L << 31)) return fail(LLMMM_ERR_INVALID_ARGUMENT, "matrix has 2^31 or more elements");
  const size_t bytes = (size_t)M * N * elem_size;
  const char * a = (const char*)src, *b = (const char*)dst;
  if (a < b + bytes && b < a + bytes) return fail(LLMMM_ERR_INVALID_ARGUMENT, "source and destination overlap");
  const hipError_t e = llmmm::transpose_launch(elem_size, src, dst, M, N, (hipStream_t)stream);
  if (e != hipSuccess) return fail(LLMMM_ERR_RUNTIME, "transpose launch: %s", hipGetErrorString(e));
  return LLMMM_OK;
}

}  // extern "C"
