// sgemm_launch.hpp — host-side description of one tile-kernel launch.
//
// C (m x n, column-major, ldc) = alpha * op(A) * op(B) + beta * C, where
//   a_kcontig == false: A(i,p) = a[i + p*lda]   (op N on a column-major A)
//   a_kcontig == true : A(i,p) = a[p + i*lda]   (op T)
//   b_ncontig == false: B(p,j) = b[p + j*ldb]   (op N)
//   b_ncontig == true : B(p,j) = b[j + p*ldb]   (op T)
// beta == 0 means C is not read. Optional epilogue, applied after the beta
// term: + bias_row[i] (per row of C), + bias_col[j] (per column), then ReLU
// (negative values become 0; NaN is kept). The kernel requires 16-byte aligned bases,
// leading dimensions that are multiples of 4 floats and `padded` = true (every
// line may be read as whole 16-byte vectors up to its leading dimension), which
// frame-packed panels always satisfy; anything else returns hipErrorInvalidValue.
//
// Two K panels (optional): with a2 / b2 set, k rows [0, k_split) of op(A) and
// op(B) come from a / b and rows [k_split, k) from a2 / b2 (same leading
// dimensions): one launch over two separately stored panels. Only for m and n
// multiples of 256 with at least 256 tiles of 256 x 256, k a multiple of 4
// (N/T: a_kcontig false, b_ncontig true) or of 8 (the other forms), k_split a
// multiple of 32 inside (0, k), 16-byte aligned a2 / b2 and each operand panel
// spanning less than 2^31 bytes from its base (two_panel_valid below);
// anything else returns hipErrorInvalidValue.
//
// Fewer than 256 tiles of 256 x 256: smaller tiles whose K the waves of a
// workgroup share (kwave_plan_shape below), K split over workgroups too where
// that is faster and a workspace is set. What follows is for the launches that
// rule leaves: panels of 2^31 bytes and more (256 x 128 kernel) and deep
// interior ranges (ring kernels).
//
// Split K (optional, workspace set): a launch that would leave CUs idle may
// cut its K into ranges (split_k_shape below), one workgroup per tile and
// range; each stores the raw partial sums of its range to the workspace
// (`splits` column-major m x n matrices, leading dimension m rounded up to 4,
// split_partial_ld), and a second kernel adds them in range order and applies
// alpha, beta and the epilogue. Launches whose tiles are all interior 256 x
// 256 tiles (m and n multiples of 256, K a multiple of 4 for N/T and of 8 for
// the other forms) split on the ring kernels when they have fewer tiles than
// the chip has CUs; other launches with fewer than 256 tiles of 256 x 256
// split on the 256 x 128 kernel (two workgroups per CU) when a split runs
// faster by narrow_time. The order of the additions is fixed, so C
// is the same from run to run. Without a workspace large enough for two
// partials the launch runs unsplit. One K panel only. A launch of at least
// 256 interior tiles whose last round would leave CUs idle may run as a
// head and a split tail instead (tail_split_shape below).
//
// start_event / stop_event (hipEvent_t, optional) are recorded by the dispatch
// itself (hipExtLaunchKernelGGL): no separate marker packets run between
// kernels, and stop_event completes when the kernel does, so it can serve as
// the retire event of every panel the launch reads or writes. A start event
// costs the dispatch ~16 us of host time and ~5 us of device time; the
// executor passes none and derives starts from the events a launch follows.
#pragma once

#include <algorithm>
#include <cstdint>

namespace xvram::kernels {

// The most k values one accumulator may add in a row (0: as a launch's own rules
// have it): `inside` for the elements of rows [0, rows) and columns [0, cols),
// `edge` for the others.
struct ChainBound {
  int64_t inside = 0, edge = 0, rows = 0, cols = 0;
};

struct SgemmLaunch {
  const float* a = nullptr;
  const float* b = nullptr;
  float* c = nullptr;
  int64_t lda = 0, ldb = 0, ldc = 0;
  int m = 0, n = 0, k = 0;
  float alpha = 1.f, beta = 0.f;
  bool a_kcontig = false;
  bool b_ncontig = false;
  bool padded = false;
  const float* bias_row = nullptr;
  const float* bias_col = nullptr;
  bool relu = false;
  const float* a2 = nullptr;
  const float* b2 = nullptr;
  int k_split = 0;
  void* start_event = nullptr;
  void* stop_event = nullptr;
  float* workspace = nullptr; // split-K partials (16-byte aligned), nullptr = none
  uint64_t workspace_bytes = 0;
  ChainBound bound;   // of a part of another launch
  bool whole = false; // interior tiles that run unsplit on the ring kernels
};

// MI355X: 256 compute units; a launch with fewer tiles than this leaves CUs
// idle unless its K is split.
constexpr int64_t kComputeUnits = 256;
// K per workgroup of a split launch, at least (a shallower range spends more
// of its time on its first loads and on storing its partial than on MFMAs).
constexpr int64_t kSplitMinDepth = 64;
// K per workgroup of a split on the ring kernels, at least: shallower ranges
// of interior tiles run faster as the 256 x 128 kernel's split (1024^3, 64
// deep on the ring kernels: 44.4 against 55.0 us; 512 x 512 x 4096, 64:
// 46.7 against 63.9; 1024 x 1024 x 3072, 192: 76.1 against 82.0), deeper
// ones on the ring kernels (1536^3, 224: 91.3 against 94.1 us; 2048 x 2048 x
// 1024, 256: 99.8 against 102.6; 1024 x 1024 x 8192, 512: 151.2 against
// 159.6).
constexpr int64_t kRingSplitMinDepth = 224;
// Workgroups of one split launch on the 256 x 128 kernel, at most: two rounds
// of its two workgroups per CU. Its partials then hold at most this many
// 256 x 128 tiles (kSplitMaxPartialBytes).
constexpr int64_t kNarrowMaxGroups = 4 * kComputeUnits;
constexpr uint64_t kSplitMaxPartialBytes = uint64_t(kNarrowMaxGroups) * 256 * 128 * 4;

struct SplitK {
  int splits = 1;      // 1 = not split
  int depth = 0;       // K per range (multiple of 32); the last range holds the rest
  bool narrow = false; // the ranges run on the 256 x 128 kernel (else the ring kernels)
};

// Leading dimension of a split launch's partials: m rounded up to 4 floats,
// so every column starts 16-byte aligned.
inline int64_t split_partial_ld(int64_t m) { return (m + 3) / 4 * 4; }

// K ranges of `depth` (ceil(k / s) rounded up to 32) covering k.
inline SplitK split_ranges(int64_t k, int64_t s, bool narrow) {
  const int64_t depth = ((k + s - 1) / s + 31) / 32 * 32;
  return SplitK{static_cast<int>((k + depth - 1) / depth), static_cast<int>(depth), narrow};
}

// Time of an m x n x k launch on the 256 x 128 kernel as `groups` equal
// workgroups of K depth `depth` writing `splits` partials (1 = unsplit, no
// partials), in hundredths of the time a workgroup paired with another on its
// CU takes per unit of K. The dispatcher fills every CU's two slots round
// after round, so full rounds of 2 x CUs workgroups each take a pair's time,
// and so does a last round that pairs workgroups on some CUs; a last round of
// at most one workgroup per CU runs each alone, in 0.65 of a pair's time.
// Each workgroup pays a fixed cost worth 32 units of K, and each partial one
// 8e-6 units per element to write and read back. Fitted to sixteen launches
// of 4 to 384 tiles of 256 x 128 (config 2, seven other ragged shapes and
// eight of interior tiles, each at four to nine split counts from unsplit to
// three rounds): the rule's choice ran within 1.6 % of the fastest measured
// count on every one.
inline int64_t narrow_time(int64_t m, int64_t n, int64_t groups, int64_t depth, int64_t splits) {
  constexpr int64_t slots = 2 * kComputeUnits;
  const int64_t full = (groups - 1) / slots;
  const int64_t last = groups - full * slots;
  const int64_t partials = splits > 1 ? splits * m * n / 1250 : 0;
  return (depth + 32) * (100 * full + (last > kComputeUnits ? 100 : 65)) + partials;
}

// The split of an m x n x k launch of form `nt` (A op N, B op T) or not,
// given a workspace of `workspace_bytes` (see "Split K" above). Ranges are at
// least kSplitMinDepth deep and the workspace holds all their partials.
// `ring` = the ring kernels can address the operand panels (each spans less
// than 2^31 bytes).
//  - Interior tiles on the ring kernels (one workgroup per CU): as many
//    ranges as one round of the CUs takes (more rounds only add each
//    range's fixed costs), when those are at least kRingSplitMinDepth deep.
//  - Otherwise, on the 256 x 128 kernel, when the launch has fewer than
//    kComputeUnits tiles of 256 x 256: the number of ranges, within two rounds
//    of its workgroup slots (kNarrowMaxGroups), that narrow_time rates
//    fastest, the unsplit launch included (ties go to fewer ranges).
inline SplitK split_k_shape(int64_t m, int64_t n, int64_t k, bool nt, bool ring,
                            uint64_t workspace_bytes) {
  if (m <= 0 || n <= 0 || k <= 0) return {};
  const bool interior = ring && m % 256 == 0 && n % 256 == 0 && k % (nt ? 4 : 8) == 0;
  const int64_t partial = split_partial_ld(m) * n * 4;
  const int64_t deepest = k / kSplitMinDepth;
  const int64_t most =
      std::min(deepest, static_cast<int64_t>(std::min<uint64_t>(workspace_bytes / partial, 1 << 30)));
  if (most < 2) return {};
  if (interior) {
    // The kernel family follows from the shape alone, not from the
    // workspace: a launch given exactly the workspace its split wants
    // (launch_bytes_wanted) takes that same split.
    const int64_t tiles = (m / 256) * (n / 256);
    const int64_t one_round = std::min(deepest, kComputeUnits / tiles);
    if (one_round < 2) return {};
    if (split_ranges(k, one_round, false).depth >= kRingSplitMinDepth) {
      const SplitK sk = split_ranges(k, std::min(one_round, most), false);
      return sk.splits >= 2 ? sk : SplitK{};
    }
  }
  // At least one 256 x 256 tile per CU runs a 256 x 256 kernel unsplit.
  if (((m + 255) / 256) * ((n + 255) / 256) >= kComputeUnits) return {};
  const int64_t tiles = ((m + 255) / 256) * ((n + 127) / 128);
  SplitK best{};
  int64_t best_time = narrow_time(m, n, tiles, k, 1);
  for (int64_t s = 2; s <= most; ++s) {
    const SplitK sk = split_ranges(k, s, true);
    if (sk.splits < 2 || sk.splits == best.splits) continue;
    if (tiles * sk.splits > kNarrowMaxGroups) break;
    const int64_t t = narrow_time(m, n, tiles * sk.splits, sk.depth, sk.splits);
    if (t < best_time) {
      best = sk;
      best_time = t;
    }
  }
  return best;
}

// The split a launch takes given room for `workspace_bytes` of partials: none
// for a two-panel launch, else split_k_shape (on the ring kernels only when
// each operand panel spans less than 2^31 bytes, their 32-bit buffer offsets).
inline SplitK split_k_for(const SgemmLaunch& l, uint64_t workspace_bytes) {
  constexpr int64_t kLimit = int64_t(1) << 31;
  if (l.a2 != nullptr || l.b2 != nullptr) return {};
  const int64_t a_bytes = (l.a_kcontig ? int64_t{l.m} : int64_t{l.k}) * l.lda * 4;
  const int64_t b_bytes = (l.b_ncontig ? int64_t{l.k} : int64_t{l.n}) * l.ldb * 4;
  return split_k_shape(l.m, l.n, l.k, !l.a_kcontig && l.b_ncontig,
                       a_bytes < kLimit && b_bytes < kLimit, workspace_bytes);
}

// K below this runs on a plain kernel (each thread four rows of one column of
// C), not the MFMA tiles: a K remainder's last 1-7 rows, or any such launch.
constexpr int kThinK = 8;

// Launches over parts of K that one rectangle may run as (many_shape).
constexpr int64_t kMaxPasses = 4;

// Tiles whose K the waves share (sgemm_kwave.hip). A one-panel launch of K >= 8
// with fewer than kComputeUnits tiles of 256 x 256 runs on one of these,
// unsplit or with its K split over workgroups, whichever combination the model
// below rates fastest; except interior launches whose ring split fills at
// least 15/16 of the CUs with ranges at least 4096 deep, which stay on the
// ring kernels (16384 x 256 x 16384 T/N, 4 x 4096 deep: 995 against 1030 us;
// with 2048-deep ranges the two are level or these ahead: 4096 x 2048 x 4096 T/N
// 497 against 490, 2048 x 1024 x 16384 N/N 488 against 490).
//
// The model, in us: workgroups run in rounds of per_cu on each CU; a CU that
// holds x of them takes (depth + fixed) x max(alone, x * each); the operands
// take their bytes over 9.67 TB/s, and the shorter of the two adds 0.79 of
// itself to the longer; C costs 0.15 us per million elements, a launch 2 us, a
// split 3 us and 1.12 us per million partial elements; in a second to fourth
// round of two a CU a last round of more than a third counts as full. Fitted to 180 shapes
// (squares, boxes up to 16384, linear layers of 1 to 1024 columns up to 16384 x
// 16384, their input and weight gradients, Gram matrices up to K = 65536), each
// on every tile with one to 32 ranges: the rule's choice ran 3.4 % slower than
// the fastest measured one on average below 256 tiles of 256 x 256 (36 % at
// worst, on 6 us) and 0.1 % from there on.
struct KwaveTile {
  int mb, nb;    // 32 x 32 blocks of rows and of columns
  int per_cu;    // workgroups a CU holds
  int run;       // a fold's k values are a multiple of this; 0 = cannot fold
  double alone, each, fixed;
};
inline constexpr KwaveTile kKwaveTiles[] = {
    {1, 1, 4, 32, 0.00725, 0.0045, 108},  {2, 1, 3, 32, 0.00981, 0.00764, 117},
    {2, 2, 2, 32, 0.0145, 0.01308, 145},  {4, 1, 2, 32, 0.01462, 0.01376, 167},
    {1, 1, 1, 128, 0.0037, 0.00397, 583}, // slots of 32 k values, deep rings
    {4, 2, 2, 0, 0.0311, 0.0256, 104},    // N/T only
    {2, 2, 4, 0, 0.0173, 0.0136, 81},     // N/T only, slots of 8 k values
};
constexpr int kKwaveTileCount = 7;
constexpr int kKwaveNtTile = 5, kKwaveSkinnyTile = 3; // from kKwaveNtTile on: N/T only
constexpr uint64_t kKwaveMaxPartialBytes = uint64_t{64} << 20;

struct KwavePlan {
  int tile = -1;  // index in kKwaveTiles; -1 = not on these
  int splits = 1; // K ranges over workgroups
  int depth = 0;  // K per range
  int fold = 0;   // k values of one wave between folds of its accumulators, in tiles of
  int edge_fold = 0;          // rows [0, rows) x columns [0, cols) / that reach past them
  int64_t rows = 0, cols = 0;
};

// The fastest plan by the model of an m x n x k launch of form `nt` or not,
// given room for `workspace_bytes` of partials, and in *time its time. A
// launch of kComputeUnits tiles of 256 x 256 and more is not split over
// workgroups. The chains of a sum are no longer than the ranges of the split
// that split_k_shape takes for the launch (`old`; where those are 64 or 96 deep, 32, as
// measured against them), nor than `bound` says, nor than 1024. Folding costs 9 %
// at 32, 4.5 % at 64, 2 % at 128, 1 % at 256 and nothing measurable from 512 on
// (64 x 64 tiles, 4500 x 4300 x 4096 and five others), and as much where only the
// edge folds: its tiles are the last XCDs' (2975 x 7265 x 920 N/N, a tenth of the
// tiles at 32, 64, 128: 340, 327, 316 us against 314).
inline KwavePlan kwave_fastest(int64_t m, int64_t n, int64_t k, bool nt, uint64_t workspace_bytes,
                               double* time_out, const ChainBound& bound, const SplitK& old) {
  KwavePlan best;
  if (m <= 0 || n <= 0 || k < kThinK) return best;
  const bool many = ((m + 255) / 256) * ((n + 255) / 256) >= kComputeUnits;
  const int64_t own = std::min<int64_t>(old.splits > 1 ? old.depth : k, 1024);
  const int64_t chain = bound.inside > 0 ? std::min(own, bound.inside) : own;
  const int64_t edge = bound.edge > 0 ? std::min(chain, bound.edge) : chain;
  const double elements = 1e-6 * double(m) * double(n);
  const double memory = 4e-6 * (double(m) + double(n)) * double(k) / 9.67;
  const int64_t partial = split_partial_ld(m) * n * 4;
  double best_time = 0;
  for (int i = 0; i < kKwaveTileCount; ++i) {
    const KwaveTile& t = kKwaveTiles[i];
    // The tiles each shape was measured on: 128 x 64 for N/T, 128 x 32 up to
    // 128 columns (twice the operand traffic of 64 x 64 beyond), one column
    // block up to 32 columns.
    if ((i >= kKwaveNtTile && !nt) || (i == kKwaveSkinnyTile && n > 128) || (t.nb > 1 && n <= 32))
      continue;
    const int64_t tiles = ((m + 32 * t.mb - 1) / (32 * t.mb)) * ((n + 32 * t.nb - 1) / (32 * t.nb));
    if (tiles >= int64_t{1} << 24) continue; // a grid holds fewer than 2^32 threads
    for (const int s : {1, 2, 3, 4, 5, 6, 8, 11, 16, 24, 32}) {
      SplitK sk;
      sk.depth = static_cast<int>(k);
      if (s > 1) {
        if (many || tiles * s > 12 * kComputeUnits || k < 128 * s ||
            uint64_t(s) * uint64_t(partial) > std::min(workspace_bytes, kKwaveMaxPartialBytes))
          break;
        sk = split_ranges(k, s, false);
        if (sk.splits != s) continue;
      }
      const int64_t quarter = (sk.depth + 3) / 4;
      if (quarter > edge && (t.run == 0 || t.run > edge)) continue;
      const auto fold_at = [&](int64_t longest) {
        if (t.run == 0) return 0;
        if (quarter <= longest) return (1 << 28) / t.run * t.run;
        return static_cast<int>((longest == own && own <= 96 ? 32 : longest) / t.run * t.run);
      };
      const int64_t groups = tiles * s, slots = t.per_cu * kComputeUnits;
      const int64_t full = (groups - 1) / slots, last = groups - full * slots;
      // After a few rounds the freed places come in pairs.
      const bool pairs = t.per_cu == 2 && full >= 1 && full <= 3;
      const double held = double(std::min<int64_t>(
          t.per_cu, ((pairs ? 3 * last / 2 : last) + kComputeUnits - 1) / kComputeUnits));
      const double compute = (sk.depth + t.fixed) * (t.each * t.per_cu * double(full) +
                                                     std::max(t.alone, t.each * held));
      const double time = 2.0 + std::max(compute, memory) + 0.79 * std::min(compute, memory) +
                          0.15 * elements + (s > 1 ? 3.0 + 1.12 * s * elements : 0.0);
      if (best.tile < 0 || time < best_time) {
        best_time = time;
        best.tile = i;
        best.splits = s;
        best.depth = sk.depth;
        best.fold = fold_at(chain);
        best.edge_fold = fold_at(edge);
        best.rows = edge < chain ? bound.rows : m;
        best.cols = edge < chain ? bound.cols : n;
      }
    }
  }
  if (time_out != nullptr) *time_out = best_time;
  return best;
}

inline KwavePlan kwave_fastest(int64_t m, int64_t n, int64_t k, bool nt, uint64_t workspace_bytes,
                               double* time_out, const ChainBound& bound = {}) {
  return kwave_fastest(m, n, k, nt, workspace_bytes, time_out, bound,
                       split_k_shape(m, n, k, nt, true, ~uint64_t{0}));
}

// The plan of a launch of fewer than kComputeUnits tiles of 256 x 256, whose
// operand panels the kernels can address (each spans less than 2^31 bytes).
inline KwavePlan kwave_plan_shape(int64_t m, int64_t n, int64_t k, bool nt,
                                  uint64_t workspace_bytes, const ChainBound& bound = {}) {
  if (m <= 0 || n <= 0 || ((m + 255) / 256) * ((n + 255) / 256) >= kComputeUnits) return {};
  const SplitK old = split_k_shape(m, n, k, nt, true, ~uint64_t{0});
  if (old.splits > 1 && !old.narrow && old.depth >= 4096 &&
      uint64_t(old.splits) * uint64_t(m) * uint64_t(n) * 4 <= workspace_bytes &&
      16 * (m / 256) * (n / 256) * old.splits >= 15 * kComputeUnits &&
      (bound.inside == 0 || old.depth <= std::min(bound.inside, bound.edge)))
    return {};
  return kwave_fastest(m, n, k, nt, workspace_bytes, nullptr, bound, old);
}

// The plan a launch takes given room for `workspace_bytes` of partials.
inline KwavePlan kwave_plan_for(const SgemmLaunch& l, uint64_t workspace_bytes) {
  constexpr int64_t kLimit = int64_t(1) << 31;
  if (l.a2 != nullptr || l.b2 != nullptr) return {};
  const int64_t a_bytes = (l.a_kcontig ? int64_t{l.m} : int64_t{l.k}) * l.lda * 4;
  const int64_t b_bytes = (l.b_ncontig ? int64_t{l.k} : int64_t{l.n}) * l.ldb * 4;
  if (a_bytes >= kLimit || b_bytes >= kLimit) return {};
  return kwave_plan_shape(l.m, l.n, l.k, !l.a_kcontig && l.b_ncontig, workspace_bytes, l.bound);
}

// Tail split. A launch of at least kComputeUnits interior 256 x 256 tiles
// runs in rounds of one workgroup per CU, and a last round that fills few
// CUs costs as much as a full one (17 x 17 tiles: 2 rounds for 289 tiles).
// It may run instead as a head, tile rows [0, head_m) unsplit in whole
// rounds, followed by a tail, rows [head_m, m), whose K is split on the ring
// kernels (up to two rounds of ranges at least kRingSplitMinDepth deep, the
// partials in the workspace), when the model below rates that at most 0.9
// of the unsplit launch. Time is counted in units of K of one round: the head
// takes its rounds x K, the tail its rounds x (range depth + 48), plus 128 for
// its extra launch and the reduction.
struct TailSplit {
  int64_t head_m = 0; // rows of the head (a multiple of 256); 0 = no tail split
  SplitK tail;        // the split of the tail's m - head_m rows
};

// The rounds of one workgroup per CU that `groups` workgroups take.
inline int64_t cu_rounds(int64_t groups) { return (groups + kComputeUnits - 1) / kComputeUnits; }

// The tail split of an interior m x n x k launch (none: head_m 0) and, in
// *time, the model's time of the launch as it then runs (tail split or not).
inline TailSplit tail_split_timed(int64_t m, int64_t n, int64_t k, uint64_t workspace_bytes,
                                  int64_t* time) {
  const int64_t tiles_m = m / 256, tiles_n = n / 256;
  const int64_t unsplit = cu_rounds(tiles_m * tiles_n) * k;
  TailSplit best{};
  int64_t best_time = unsplit;
  for (int64_t t = 1; t < tiles_m && 2 * t * tiles_n <= 2 * kComputeUnits; ++t) {
    const int64_t tail_tiles = t * tiles_n;
    const uint64_t partial = uint64_t(t) * 256 * uint64_t(n) * 4;
    const int64_t head_time = cu_rounds((tiles_m - t) * tiles_n) * k;
    for (int64_t s = 2; s <= k / kSplitMinDepth; ++s) {
      const SplitK sk = split_ranges(k, s, false);
      if (sk.depth < kRingSplitMinDepth || tail_tiles * sk.splits > 2 * kComputeUnits ||
          uint64_t(sk.splits) * partial > workspace_bytes)
        break;
      const int64_t time = head_time + cu_rounds(tail_tiles * sk.splits) * (sk.depth + 48) + 128;
      if (time < best_time) {
        best_time = time;
        best = TailSplit{(tiles_m - t) * 256, sk};
      }
    }
  }
  if (10 * best_time > 9 * unsplit) {
    best = TailSplit{};
    best_time = unsplit;
  }
  if (time != nullptr) *time = best_time;
  return best;
}

inline TailSplit tail_split_shape(int64_t m, int64_t n, int64_t k, bool nt, bool ring,
                                  uint64_t workspace_bytes) {
  if (!ring || m <= 0 || n <= 0 || k <= 0 || m % 256 != 0 || n % 256 != 0 || k % (nt ? 4 : 8) != 0)
    return {};
  if ((m / 256) * (n / 256) < kComputeUnits) return {};
  return tail_split_timed(m, n, k, workspace_bytes, nullptr);
}

// The tail split a launch takes given room for `workspace_bytes` of
// partials: none for a two-panel launch or panels the ring kernels cannot
// address, else tail_split_shape.
inline TailSplit tail_split_for(const SgemmLaunch& l, uint64_t workspace_bytes) {
  constexpr int64_t kLimit = int64_t(1) << 31;
  if (l.a2 != nullptr || l.b2 != nullptr) return {};
  const int64_t a_bytes = (l.a_kcontig ? int64_t{l.m} : int64_t{l.k}) * l.lda * 4;
  const int64_t b_bytes = (l.b_ncontig ? int64_t{l.k} : int64_t{l.n}) * l.ldb * 4;
  return tail_split_shape(l.m, l.n, l.k, !l.a_kcontig && l.b_ncontig,
                          a_bytes < kLimit && b_bytes < kLimit, workspace_bytes);
}

// Edge split. A launch whose m or n is not a multiple of 256 and that has at
// least kComputeUnits tiles of 256 x 256 runs every tile on the ring kernels'
// edge instances (K a multiple of 4 for N/T, of 8 for the other forms), whose
// K loop is the interior one: rounds x (K x 26/25 + 50) in units of K of one
// round, within 4 % of 17 shapes measured. Its last round may fill few CUs. It
// may run instead as up to three launches of its own, one after another on
// its stream: the interior rows [0, mi) x columns [0, ni) (mi, ni = m, n
// rounded down to 256; ring kernels, or their tail split), the right strip
// rows [0, mi) x columns [ni, n) and the bottom strip rows [mi, m) x columns
// [0, n), each split by the rules above (the strips run on small tiles),
// sharing the workspace. Every element of C is computed by one of them. The
// split is modelled as the interior's time (tail_split_timed, one round for
// fewer than kComputeUnits tiles), plus the strips' 256 x 128 tiles x K x
// 2.7 over the 256 x 128 kernel's 512 slots (their split launches' first
// loads, partial stores and reductions, and mostly empty tiles: least squares
// over 20 shapes), plus 150 for the two extra launches, and taken when it
// models faster. On 22 shapes from 4100^2 x 240 to 11500 x 11000 x 1024 the
// model's split / whole ratio came within 7 % of the measured one and picked
// the faster plan every time (split 4100^2 x 4096 1.74x, 7000^3 1.31x, 5000^2
// x 2048 1.09x; whole 8191^2 x 8192 1.17x, 8100^2 x 4096 1.15x, 8000^3 1.07x).
// The 2.7 is of strips on the 256 x 128 kernel, which took longer than small tiles
// do now; the line it draws stands: of 21 shapes in two forms, timed again both
// ways, it picks the slower plan on 5280^3 only (which runs on small tiles), and of
// 65 in 100000 random launches where kwave_fastest rates the strips otherwise by
// 4 % and more, the 13 furthest ran up to 5 % faster the other way, 16121 x 1253 x
// 64 T/N 78 against 59 us.
// Only for one-panel launches with K a multiple of 4 (N/T) or 8 (the other
// forms), and panels below 2^31 bytes; when a part would split, only with a
// workspace (a strip unsplit would leave most CUs idle).
inline bool edge_split_rated_faster(int64_t m, int64_t n, int64_t k, bool nt) {
  if (m <= 0 || n <= 0 || k <= 0 || k % (nt ? 4 : 8) != 0) return false;
  const int64_t mi = m / 256 * 256, ni = n / 256 * 256;
  const int64_t whole_tiles = ((m + 255) / 256) * ((n + 255) / 256);
  if ((mi == m && ni == n) || whole_tiles < kComputeUnits || mi == 0 || ni == 0) return false;
  const int64_t whole = cu_rounds(whole_tiles) * (k * 26 / 25 + 50);
  const int64_t interior_tiles = (mi / 256) * (ni / 256);
  int64_t interior = cu_rounds(interior_tiles) * k;
  if (interior_tiles >= kComputeUnits) tail_split_timed(mi, ni, k, ~uint64_t{0}, &interior);
  // The strips' 256 x 128 tiles (the bottom strip's one row of them, the
  // right strip's column of them).
  const int64_t strip_tiles = (m > mi ? (n + 127) / 128 : 0) + (mi / 256) * ((n - ni + 127) / 128);
  const int64_t split = interior + 27 * k * strip_tiles / (20 * kComputeUnits) + 150;
  return split < whole;
}

struct EdgeParts {
  int count = 0; // 0 = no edge split
  SgemmLaunch part[3];
};

// Rows [r0, r0 + rows) x columns [c0, c0 + cols) of a launch as a launch of
// its own (no events).
inline SgemmLaunch sub_launch(const SgemmLaunch& l, int64_t r0, int rows, int64_t c0, int cols) {
  SgemmLaunch s = l;
  s.a = l.a_kcontig ? l.a + r0 * l.lda : l.a + r0;
  s.b = l.b_ncontig ? l.b + c0 : l.b + c0 * l.ldb;
  s.c = l.c + r0 + c0 * l.ldc;
  if (s.bias_row != nullptr) s.bias_row += r0;
  if (s.bias_col != nullptr) s.bias_col += c0;
  s.m = rows;
  s.n = cols;
  s.start_event = nullptr;
  s.stop_event = nullptr;
  return s;
}

// K rows [k0, k0 + depth) of a launch as a launch of its own (no events): alpha,
// on C as the caller left it from the first rows, onto the sum so far from the
// others; the epilogue with the last.
inline SgemmLaunch k_range(const SgemmLaunch& l, int64_t k0, int64_t depth) {
  SgemmLaunch s = l;
  s.k = static_cast<int>(depth);
  s.a = l.a_kcontig ? l.a + k0 : l.a + k0 * l.lda;
  s.b = l.b_ncontig ? l.b + k0 * l.ldb : l.b + k0;
  if (k0 > 0) s.beta = 1.f;
  if (k0 + depth < l.k) {
    s.bias_row = nullptr;
    s.bias_col = nullptr;
    s.relu = false;
  }
  s.start_event = nullptr;
  s.stop_event = nullptr;
  return s;
}

// The parts of a launch's edge split by shape alone (count 0: none).
inline EdgeParts edge_parts_shape(const SgemmLaunch& l) {
  constexpr int64_t kLimit = int64_t(1) << 31;
  EdgeParts e;
  if (l.a2 != nullptr || l.b2 != nullptr || l.m <= 0 || l.n <= 0 || l.k <= 0) return e;
  const bool nt = !l.a_kcontig && l.b_ncontig;
  const int64_t a_bytes = (l.a_kcontig ? int64_t{l.m} : int64_t{l.k}) * l.lda * 4;
  const int64_t b_bytes = (l.b_ncontig ? int64_t{l.k} : int64_t{l.n}) * l.ldb * 4;
  if (a_bytes >= kLimit || b_bytes >= kLimit || !edge_split_rated_faster(l.m, l.n, l.k, nt))
    return e;
  const int mi = l.m / 256 * 256, ni = l.n / 256 * 256;
  e.part[e.count++] = sub_launch(l, 0, mi, 0, ni);
  if (ni < l.n) e.part[e.count++] = sub_launch(l, 0, mi, ni, l.n - ni);
  if (mi < l.m) e.part[e.count++] = sub_launch(l, mi, l.m - mi, 0, l.n);
  e.part[0].start_event = l.start_event;
  e.part[e.count - 1].stop_event = l.stop_event;
  return e;
}

// K remainder. The ring kernels need K a multiple of 4 (N/T) or 8 (the other
// forms), and so do the tail and edge splits. A launch whose K is not, whose
// K rounded down to that multiple is at least 512, and which either has
// interior tiles and would take a tail split over the rounded K, or has
// ragged tiles, at least kComputeUnits of them (the rounded K then runs on
// the ring kernels' edge instances or takes an edge split, not the general
// kernel's predicated edge tiles), runs as two launches of its own: the first
// over the rounded K with alpha and beta and no epilogue, the second over the
// remaining 1 to 7 K rows with alpha and beta 1 onto the first's result, then
// the epilogue (one more read and write of C: 4500^3 N/N, 2.30 ms as one
// launch on the general kernel, gains far more from the split first part).
// Returns the rounded K (0: no K remainder).
inline int64_t k_remainder_shape(int64_t m, int64_t n, int64_t k, bool nt) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  const int64_t k1 = k - k % (nt ? 4 : 8);
  if (k1 == k || k1 < 512) return 0;
  const bool interior = m % 256 == 0 && n % 256 == 0;
  const bool gains = interior ? tail_split_shape(m, n, k1, nt, true, ~uint64_t{0}).head_m > 0
                              : ((m + 255) / 256) * ((n + 255) / 256) >= kComputeUnits;
  return gains ? k1 : 0;
}

// Many tiles on small ones. A launch of kComputeUnits tiles of 256 x 256 and
// more runs on the tiles of kKwaveTiles instead where they model at least 4 %
// faster than what the rules above make of it: shallow or odd K (no ring kernel
// takes a K that is not a multiple of its step below 512) and ragged shapes
// whose last round or strips cost much. The ring kernels are modelled, in us,
// at rounds x (0.2155 K + 14) + 2 (4 % more K and 16 for edge instances; 4096 x
// 4096 at K = 256 71 us, at 4096 907, 8192^3 7180, 8191^2 x 2048 1894), a
// split's partials at 1.2 us per million elements and 8, strips at what
// kwave_fastest says, a K remainder at 2.3 us per million elements of C and 4;
// the small tiles at 7 % over kwave_fastest's time from K = 1500 on (their
// operands no longer stay in the L2), proportionally less below. 3712 x 4590 x 503
// N/T 313 -> 139 us, 5994 x 3000 x 146 N/T 123 -> 61, 6379 x 2968 x 32 N/T 67 -> 34,
// 1504 x 15840 x 1728 N/T 782 -> 601, 5280^3 N/N 2331 -> 2095. Over 128 launches of
// 51 shapes, each timed on every plan, what this and the next rule choose is 5.4 %
// faster than the rules above and 1.5 % slower than the fastest (whose chains no
// rule bounds; 64 % at worst, 6379 x 2968 x 32 N/N, 69 us).
inline double ring_time(int64_t tiles, int64_t k) {
  return double(cu_rounds(tiles)) * (0.2155 * double(k) + 14.0);
}

// The same of the general kernel over interior tiles (an odd K): 4096 x 4096 at K
// = 1029, 2051, 4099 N/N 261, 490, 949 us, N/T 255, 478, 928 (T/N 3 % above N/N);
// 8192 x 8192 x 4099 N/N 3778.
inline double general_time(int64_t tiles, int64_t k, bool nt) {
  return double(cu_rounds(tiles)) * ((nt ? 0.2195 : 0.2241) * double(k) + 28.0);
}

// The same of many tiles on small ones.
inline double small_time(int64_t m, int64_t n, int64_t k, bool nt) {
  double time = 0;
  kwave_fastest(m, n, k, nt, 0, &time);
  return time * (1.0 + 0.07 * std::min(1.0, double(k) / 1500.0));
}

// The model's time of an interior launch with its tail split.
inline double interior_time(int64_t m, int64_t n, int64_t k) {
  const TailSplit ts = (m / 256) * (n / 256) >= kComputeUnits
                           ? tail_split_timed(m, n, k, ~uint64_t{0}, nullptr)
                           : TailSplit{};
  if (ts.head_m == 0) return ring_time((m / 256) * (n / 256), k) + 2.0;
  const int64_t tail_m = m - ts.head_m;
  return ring_time(ts.head_m / 256 * (n / 256), k) +
         ring_time(tail_m / 256 * (n / 256) * ts.tail.splits, ts.tail.depth) +
         1.2e-6 * double(ts.tail.splits) * double(tail_m) * double(n) + 8.0;
}

// The model's time of a launch of many tiles as the rules above run it (K a
// multiple of the ring kernels' step).
inline double ring_rules_time(int64_t m, int64_t n, int64_t k, bool nt) {
  if (m % 256 == 0 && n % 256 == 0) return interior_time(m, n, k);
  if (!edge_split_rated_faster(m, n, k, nt))
    return double(cu_rounds(((m + 255) / 256) * ((n + 255) / 256))) *
               (0.2241 * double(k) + 16.0) + 2.0;
  const int64_t mi = m / 256 * 256, ni = n / 256 * 256;
  double time = interior_time(mi, ni, k), strip = 0;
  if (ni < n && kwave_fastest(mi, n - ni, k, nt, ~uint64_t{0}, &strip).tile >= 0) time += strip + 3.0;
  if (mi < m && kwave_fastest(m - mi, n, k, nt, ~uint64_t{0}, &strip).tile >= 0) time += strip + 3.0;
  return time;
}

// Whole rounds. A launch of many tiles may also run as the rectangle of
// interior 256 x 256 tiles that fills whole rounds of the CUs best, on the ring
// kernels, and the rest of C, a right and a bottom strip, on small tiles: no
// round is mostly empty, no tile is padded to 256 and nothing is split and
// reduced. 5000^3 T/T, 16 x 16 tiles in two passes and strips 904 wide: 1832 -> 1794
// us; 4352 x 4096 x 1024 N/N 302 -> 258, 4500^3 N/N 1354 -> 1325, 11378 x 2374 x 7040
// T/T 2837 -> 2687. Modelled like the rest, the strips at 131 TFLOP/s and 8 us each,
// for K from 1024 on, and taken where that is 3 % faster than the rules above and
// than small tiles alone (4576^3, so rated, runs 1 % slower). Its tiles run
// unsplit on the ring kernels, as modelled, also where the chains (below)
// leave it a few less than a round. Where the best rectangle of all is one round
// of 244 to 255 tiles, so that the rules above leave most of a round idle too,
// the small tiles are taken up to 7 % above those rules' modelled time (none of
// 1086 such launches models above; their chains are at most 1024 instead of K):
// 1792 x 11520 x 4496 N/T 1309 us (those rules 1439, the rectangle with its 252 tiles
// on small ones 1335), 5586 x 3566 x 3344 N/N 1003 (986, 994).
struct ManyPlan {
  KwavePlan small;        // on small tiles (tile >= 0), or
  int64_t mi = 0, ni = 0; // the rectangle's rows and columns; neither: the rules above
  int64_t pass = 0;       // K of one pass of the rectangle (its K: one pass)
  ChainBound bound;       // of the strips' sums, by rows and columns of C
};

// The chains of a launch of many tiles under the rules above (K a multiple of
// the ring kernels' step): rows [0, rows) of its interior add all of K in one
// accumulator, a split tail's rows `tail` k values, and the shortest chain
// anywhere in C is `shortest`.
struct Chains {
  int64_t rows, tail, shortest;
};

inline Chains ring_rules_chains(int64_t m, int64_t n, int64_t k, bool nt) {
  constexpr uint64_t kAny = ~uint64_t{0};
  Chains c{m, k, k};
  const bool ragged = m % 256 != 0 || n % 256 != 0;
  if (ragged && !edge_split_rated_faster(m, n, k, nt)) return c;
  const int64_t mi = m / 256 * 256, ni = n / 256 * 256;
  const auto split_depth = [&](int64_t rows, int64_t cols) {
    const SplitK sk = split_k_shape(rows, cols, k, nt, true, kAny);
    return sk.splits > 1 ? int64_t{sk.depth} : k;
  };
  if (const TailSplit ts = tail_split_shape(mi, ni, k, nt, true, kAny); ts.head_m > 0) {
    c.rows = ts.head_m;
    c.tail = ts.tail.depth;
  } else if (split_depth(mi, ni) < k) { // an edge split's interior of few tiles
    c.rows = 0;
    c.tail = split_depth(mi, ni);
  }
  c.shortest = c.tail;
  if (ni < n) c.shortest = std::min(c.shortest, split_depth(mi, n - ni));
  if (mi < m) c.shortest = std::min(c.shortest, split_depth(m - mi, n));
  return c;
}

// No sum is added in longer chains than the rules above would add it in
// (ring_rules_chains): small tiles and the strips fold where a split tail's or
// an edge strip's sums lie, and a rectangle that reaches past the rows of whole
// sums runs its K in passes no deeper than the tail's ranges, each after the
// first adding to C (24 us a round: first loads, and C read back; 4096 x 4096 x
// 5000 in two passes 1139 against 1111 us). `bound` is that of a part of another
// launch: it goes to small tiles.
inline ManyPlan many_shape(int64_t m, int64_t n, int64_t k, bool nt, const ChainBound& bound = {}) {
  ManyPlan plan;
  if (m <= 0 || n <= 0 || k < kThinK ||
      ((m + 255) / 256) * ((n + 255) / 256) < kComputeUnits)
    return plan;
  const int64_t k1 = k - k % (nt ? 4 : 8);
  if (bound.inside > 0 || (k1 != k && k1 < 512)) { // or the general kernel's K
    plan.small = kwave_fastest(m, n, k, nt, 0, nullptr, bound);
    return plan;
  }
  // An odd K without a K remainder: the general kernel, on which no rectangle runs.
  const bool general = k1 != k && k_remainder_shape(m, n, k, nt) == 0;
  const Chains chains = general ? Chains{m, k, k} : ring_rules_chains(m, n, k1, nt);
  const ChainBound rules{chains.tail, chains.shortest, m / 256 * 256, n / 256 * 256};
  // Rated as if no chain were bounded: the folds cost little (kwave_fastest).
  const double small = small_time(m, n, k, nt);
  const KwavePlan kw = kwave_fastest(m, n, k, nt, 0, nullptr, rules);
  const double rest = k1 == k ? 0.0 : 2.3e-6 * double(m) * double(n) + 4.0;
  const double ring =
      general ? general_time(m / 256 * (n / 256), k, nt) : ring_rules_time(m, n, k1, nt) + rest;
  bool few = false; // the best rectangle, whatever its chains, is less than one round
  if (k >= 1024 && !general) {
    const int64_t tm = m / 256, tn = n / 256;
    struct {
      int64_t a = 0, b = 0, passes = 1;
      double time;
    } any, once, more; // the best one of all, in one pass, in more
    any.time = once.time = more.time = 0.97 * std::min(ring, small);
    // For each number of tile rows the most rounds that all columns fill, and the
    // three before: of fewer, none was ever the best (60000 random launches).
    for (int64_t a = 1; a <= tm; ++a) {
      const int64_t most = std::min(tm * tn / kComputeUnits, cu_rounds(a * tn));
      for (int64_t rounds = std::max<int64_t>(1, most - 3); rounds <= most; ++rounds) {
        const int64_t b = std::min(tn, rounds * kComputeUnits / a);
        if (20 * a * b < 19 * rounds * kComputeUnits || (a * 256 == m && b * 256 == n)) continue;
        const double area = double(m) * double(n) - 65536.0 * double(a * b);
        const double time = double(rounds) * (0.2155 * double(k1) + 14.0) + 2.0 +
                            2e-6 * double(k1) * area / 131.0 + (a * 256 < m ? 8.0 : 0.0) +
                            (b * 256 < n ? 8.0 : 0.0) + rest;
        if (time < any.time) any = {a, b, 1, time};
        const int64_t passes = a * 256 <= chains.rows ? 1 : (k1 + chains.tail - 1) / chains.tail;
        const double bounded = time + 24.0 * double(rounds) * double(passes - 1);
        auto& best = passes == 1 ? once : more;
        if (passes <= kMaxPasses && bounded < best.time) best = {a, b, passes, bounded};
      }
    }
    few = any.a > 0 && any.a * any.b < kComputeUnits;
    auto best = once.a > 0 ? once : more;
    if (once.a > 0 && more.a > 0) {
      // Close to each other as a rule: by the strips' own rounds then.
      const auto time = [&](const auto& r) {
        const int64_t mi = r.a * 256, ni = r.b * 256;
        double t = ring_time(r.a * r.b, k1) + 24.0 * double(cu_rounds(r.a * r.b) * (r.passes - 1));
        double strip = 0;
        if (ni < n && kwave_fastest(mi, n - ni, k1, nt, ~uint64_t{0}, &strip, rules).tile >= 0) t += strip;
        if (mi < m && kwave_fastest(m - mi, n, k1, nt, ~uint64_t{0}, &strip, rules).tile >= 0) t += strip;
        return t;
      };
      if (time(more) < time(once)) best = more;
    }
    if (best.a > 0 && !(few && small < 1.07 * ring)) {
      if (k1 == k) { // else the K remainder's first part comes here again
        plan.mi = best.a * 256;
        plan.ni = best.b * 256;
        plan.pass = best.passes == 1 ? k : split_ranges(k, best.passes, false).depth;
        if (chains.shortest < k) plan.bound = rules;
      }
      return plan;
    }
  }
  // Level with the general kernel the small tiles' shorter chains decide, to K = 1200
  // also where they are 3 % behind (4096 x 4096 x 1029 N/N 269 against 261 us).
  const double limit = general ? (k < 1200 ? 1.04 : 1.0) : few ? 1.07 : 0.96;
  if (small < limit * ring) plan.small = kw;
  return plan;
}

inline ManyPlan many_plan(const SgemmLaunch& l) {
  constexpr int64_t kLimit = int64_t(1) << 31;
  if (l.a2 != nullptr || l.b2 != nullptr) return {};
  const int64_t a_bytes = (l.a_kcontig ? int64_t{l.m} : int64_t{l.k}) * l.lda * 4;
  const int64_t b_bytes = (l.b_ncontig ? int64_t{l.k} : int64_t{l.n}) * l.ldb * 4;
  if (a_bytes >= kLimit || b_bytes >= kLimit) return {};
  return many_shape(l.m, l.n, l.k, !l.a_kcontig && l.b_ncontig, l.bound);
}

// The parts of a launch on the rectangle of `plan`, its passes first, and its
// strips.
struct ManyParts {
  int count = 0;
  SgemmLaunch part[kMaxPasses + 2];
};

inline ManyParts many_parts(const SgemmLaunch& l, const ManyPlan& plan) {
  const int mi = static_cast<int>(plan.mi), ni = static_cast<int>(plan.ni);
  ManyParts e;
  for (int64_t k0 = 0; k0 < l.k; k0 += plan.pass) {
    SgemmLaunch p = k_range(sub_launch(l, 0, mi, 0, ni), k0, std::min(l.k - k0, plan.pass));
    p.whole = true;
    e.part[e.count++] = p;
  }
  const auto strip = [&](int r0, int rows, int c0, int cols) {
    SgemmLaunch s = sub_launch(l, r0, rows, c0, cols);
    s.bound = plan.bound;
    s.bound.rows -= r0;
    s.bound.cols -= c0;
    e.part[e.count++] = s;
  };
  if (ni < l.n) strip(0, mi, ni, l.n - ni);
  if (mi < l.m) strip(mi, l.m - mi, 0, l.n);
  e.part[0].start_event = l.start_event;
  e.part[e.count - 1].stop_event = l.stop_event;
  return e;
}

struct KParts {
  int count = 0; // 0 = no K remainder
  SgemmLaunch part[2];
};

// The two launches of a K remainder by shape (count 0: none); one-panel
// launches whose panels the ring kernels can address only.
inline KParts k_remainder_parts_shape(const SgemmLaunch& l) {
  constexpr int64_t kLimit = int64_t(1) << 31;
  KParts r;
  if (l.a2 != nullptr || l.b2 != nullptr) return r;
  const int64_t a_bytes = (l.a_kcontig ? int64_t{l.m} : int64_t{l.k}) * l.lda * 4;
  const int64_t b_bytes = (l.b_ncontig ? int64_t{l.k} : int64_t{l.n}) * l.ldb * 4;
  if (a_bytes >= kLimit || b_bytes >= kLimit) return r;
  const int64_t k1 = k_remainder_shape(l.m, l.n, l.k, !l.a_kcontig && l.b_ncontig);
  if (k1 == 0) return r;
  r.part[0] = k_range(l, 0, k1);
  r.part[1] = k_range(l, k1, l.k - k1);
  r.part[0].start_event = l.start_event;
  r.part[1].stop_event = l.stop_event;
  r.count = 2;
  return r;
}

// How a launch runs: on one kernel, as head and tail, or as parts of its own.
enum class Run {
  kTwoPanel,   // ring kernels' two-panel instances
  kRectangle,  // parts: whole rounds of interior tiles, right strip, bottom strip (many_parts)
  kKRemainder, // parts: the rounded K, the rest (k_remainder_parts_shape)
  kEdgeSplit,  // parts: interior tiles, right strip, bottom strip (edge_parts_shape)
  kSmallTiles, // `small`
  kThinK,      // thin_k_kernel
  kRingSplit,  // `split` on the ring kernels
  kNarrowSplit, // `split` on the 256 x 128 kernel
  kTailSplit,  // `tail`
  kRing,       // ring kernels, interior or edge instances
  kGeneral,    // sgemm_wide_kernel
  kNarrow,     // 256 x 128 kernel
};
constexpr int kRunCount = static_cast<int>(Run::kNarrow) + 1;

struct Route {
  Run run = Run::kNarrow;
  KwavePlan small;
  SplitK split;
  TailSplit tail;
  int count = 0; // parts, run one after another
  SgemmLaunch part[kMaxPasses + 2];
};

inline uint64_t launch_bytes_wanted(const SgemmLaunch& l);

// The route of a launch whose operands and workspace are aligned, given room
// for `room` bytes of partials; `workspace` = it has any (without one a K
// remainder or edge split is taken only where its parts would not split).
inline Route route_with(const SgemmLaunch& l, bool workspace, uint64_t room) {
  constexpr int64_t kLimit = int64_t(1) << 31;
  Route r;
  const auto parts = [&](Run run, const SgemmLaunch* part, int count) {
    r.run = run;
    r.count = count;
    std::copy(part, part + count, r.part);
  };
  if (l.a2 != nullptr || l.b2 != nullptr) {
    r.run = Run::kTwoPanel;
    return r;
  }
  if (l.whole) {
    r.run = Run::kRing;
    return r;
  }
  if (const ManyPlan mp = many_plan(l); mp.small.tile >= 0) {
    r.run = Run::kSmallTiles;
    r.small = mp.small;
    return r;
  } else if (mp.mi > 0) {
    const ManyParts e = many_parts(l, mp);
    parts(Run::kRectangle, e.part, e.count);
    return r;
  }
  if (const KParts kp = k_remainder_parts_shape(l);
      kp.count > 0 && (workspace || launch_bytes_wanted(kp.part[0]) == 0)) {
    parts(Run::kKRemainder, kp.part, kp.count);
    return r;
  }
  if (const EdgeParts e = edge_parts_shape(l); e.count > 0) {
    // A part with parts of its own does without a workspace.
    bool alone = true;
    for (int i = 0; i < e.count && !workspace; ++i)
      alone = alone && (route_with(e.part[i], true, ~uint64_t{0}).count > 0 ||
                        launch_bytes_wanted(e.part[i]) == 0);
    if (alone) {
      parts(Run::kEdgeSplit, e.part, e.count);
      return r;
    }
  }
  if (l.k < kThinK) {
    r.run = Run::kThinK;
    return r;
  }
  if (r.small = kwave_plan_for(l, room); r.small.tile >= 0) {
    r.run = Run::kSmallTiles;
    return r;
  }
  if (r.split = split_k_for(l, room); r.split.splits > 1) {
    r.run = r.split.narrow ? Run::kNarrowSplit : Run::kRingSplit;
    return r;
  }
  if (r.tail = tail_split_for(l, room); r.tail.head_m > 0) {
    r.run = Run::kTailSplit;
    return r;
  }
  const int64_t tiles = ((int64_t{l.m} + 255) / 256) * ((int64_t{l.n} + 255) / 256);
  const int64_t a_bytes = (l.a_kcontig ? int64_t{l.m} : int64_t{l.k}) * l.lda * 4;
  const int64_t b_bytes = (l.b_ncontig ? int64_t{l.k} : int64_t{l.n}) * l.ldb * 4;
  if (tiles >= kComputeUnits && a_bytes < kLimit && b_bytes < kLimit)
    r.run = l.k % (!l.a_kcontig && l.b_ncontig ? 4 : 8) == 0 ? Run::kRing : Run::kGeneral;
  return r;
}

// The route of a launch with its own workspace (or none).
inline Route route(const SgemmLaunch& l) {
  const bool usable = l.workspace != nullptr && reinterpret_cast<uintptr_t>(l.workspace) % 16 == 0;
  return route_with(l, l.workspace != nullptr, usable ? l.workspace_bytes : 0);
}

// Bytes of partials one launch wants when the workspace is not the limit: its
// own, or the most that any of its parts wants (they share the workspace in
// turn).
inline uint64_t launch_bytes_wanted(const SgemmLaunch& l) {
  const Route r = route_with(l, true, ~uint64_t{0});
  const auto partials = [](int splits, int64_t m, int64_t n) {
    return uint64_t(splits) * uint64_t(split_partial_ld(m)) * uint64_t(n) * 4;
  };
  uint64_t bytes = 0;
  for (int i = 0; i < r.count; ++i) bytes = std::max(bytes, launch_bytes_wanted(r.part[i]));
  if (r.run == Run::kSmallTiles && r.small.splits > 1) bytes = partials(r.small.splits, l.m, l.n);
  if (r.run == Run::kRingSplit || r.run == Run::kNarrowSplit)
    bytes = partials(r.split.splits, l.m, l.n);
  if (r.run == Run::kTailSplit) bytes = partials(r.tail.tail.splits, l.m - r.tail.head_m, l.n);
  return bytes;
}

// Whether a launch given room for `room` bytes of partials, or a part of it,
// splits its K over workgroups.
inline bool uses_partials(const SgemmLaunch& l, uint64_t room) {
  const Route r = route_with(l, true, room);
  for (int i = 0; i < r.count; ++i)
    if (uses_partials(r.part[i], room)) return true;
  return r.small.splits > 1 || r.split.splits > 1 || r.tail.head_m > 0;
}

// Enqueues the launch on `stream` (a hipStream_t); returns a hipError_t.
int launch_sgemm(const SgemmLaunch& launch, void* stream);

// The two-panel part of the contract (a2 / b2 set); the one-panel part is
// checked separately.
inline bool two_panel_valid(const SgemmLaunch& l) {
  constexpr int64_t kLimit = int64_t(1) << 31;
  if (l.a2 == nullptr || l.b2 == nullptr || reinterpret_cast<uintptr_t>(l.a2) % 16 != 0 ||
      reinterpret_cast<uintptr_t>(l.b2) % 16 != 0)
    return false;
  const bool nt = !l.a_kcontig && l.b_ncontig;
  if (l.m % 256 != 0 || l.n % 256 != 0 || int64_t{l.m / 256} * (l.n / 256) < 256 ||
      l.k % (nt ? 4 : 8) != 0 || l.k_split % 32 != 0 || l.k_split <= 0 || l.k_split >= l.k)
    return false;
  for (const int64_t kk : {int64_t{l.k_split}, int64_t{l.k - l.k_split}}) {
    // Floats from a panel's base to the end of its last line.
    const int64_t a = l.a_kcontig ? (l.m - 1) * l.lda + kk : kk * l.lda;
    const int64_t b = l.b_ncontig ? kk * l.ldb : (l.n - 1) * l.ldb + kk;
    if (a * 4 >= kLimit || b * 4 >= kLimit) return false;
  }
  return true;
}

} // namespace xvram::kernels
