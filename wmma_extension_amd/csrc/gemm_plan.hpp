// What the host side of the GEMM driver decides with: policies, packed operand
// geometry, the fitted cost parameters, K-slice plans.  Shared by the C boundary
// (capi_gemm.hip) and the translation units that hold the kernels of one or two
// policies each (gemm_*.hip, through gemm_launch.hpp).
#pragma once
#include "capi_common.hpp"
#include <limits>
#include "tcec_gemm_fused_kernel.hpp"
#include "tcec_gemm_kernels.hpp"

namespace wmmae_driver {
using namespace wmmae_capi;
using wmmae_gemm::u32x4;

// ------------------------------------------------------------ policy table
struct PolicyInfo {
  int terms;       // stored terms per operand
  bool bf16;       // MFMA element type
  float inv_scale; // factor applied to the error accumulator
};
inline bool policy_info(const int policy, PolicyInfo &p) {
  switch (policy) {
  case WMMAE_POLICY_F16_EC:
    p = {2, false, 1.f / 2048.f};
    return true;
  case WMMAE_POLICY_F16_NOEC:
    p = {1, false, 1.f};
    return true;
  case WMMAE_POLICY_BF16X3_EC:
    p = {3, true, 1.f};
    return true;
  case WMMAE_POLICY_BF16X2_EC:
    p = {2, true, 1.f};
    return true;
  case WMMAE_POLICY_BF16_NOEC:
    p = {1, true, 1.f};
    return true;
  default:
    return false;
  }
}

// packed operand geometry: 16-row blocks, 32-wide k chunks
inline long long packed_row_blocks(const int rows) { return ceil_div(rows, 16); }
inline int packed_k_tiles(const int k) {
  return static_cast<int>(ceil_div(k, 32));
}
// u32x4 elements of one packed matrix
inline long long packed_elems(const int rows, const int k, const int terms) {
  return packed_row_blocks(rows) * packed_k_tiles(k) * terms * 64;
}

// ------------------------------------------------------------------ pack
// One operand of a split launch as the caller describes it.
struct PackSource {
  int rows;
  const float *X;
  const float *const *ptrs;
  long long row_stride, k_stride, batch_stride;
  void *packed;
};

inline wmmae_gemm::PackOperand pack_operand(const PackSource &src,
                                            const int KT) {
  wmmae_gemm::PackOperand o;
  o.X = src.X;
  o.ptrs = src.ptrs;
  o.row_stride = src.row_stride;
  o.k_stride = src.k_stride;
  o.batch_stride = src.batch_stride;
  o.rows = src.rows;
  o.chunks = packed_row_blocks(src.rows) * KT;
  o.out = static_cast<u32x4 *>(src.packed);
  return o;
}

// The batch index of the split, scale and fold kernels is the grid's y
// coordinate, which ends at 65535: longer batches take one launch per 65535
// entries.
constexpr int kMaxGridY = 65535;

// ------------------------------------------------------------------ gemm
struct GemmArgs {
  const u32x4 *a, *b;
  float *c;
  int m, n, k;
  long long ldc, stride_c;
  float alpha, beta, inv_scale;
  int batch, terms;
  float *const *c_ptrs; // device array of C pointers, or nullptr
  float *partial;  // split-K slices, or nullptr
  int splits;      // >= 1
  // room for the K slices of the tiles of a partly empty last round (used
  // only without split-K), or nullptr
  float *tail_ws;
  size_t tail_ws_bytes;
  hipStream_t stream;
  // fp32 operands for the kernel variant that splits them itself (a and b are
  // null then)
  bool is_direct = false;
  wmmae_gemm::DirectSource direct = {};
};

// ------------------------------------------------ fitted cost parameters
// Every number the path and tile choices below are made with, in one place.
// All are fits to measurements on MI355X (256 compute units, one box of the
// pool each; the boxes differ by 3 to 5 % in what they sustain under the power
// limit).  The estimates have one form: launch cost + rounds of tiles over the
// compute units x (k stages of 32 x time per stage + time per tile), bounded
// below by the bytes moved.
namespace fit {
// -- packed GEMM, time of one k stage of one tile, by stored terms (1, 2, 3).
//    Sweep: 216 products, m = n = 512 .. 2048, k = 512 .. 4096, each run with
//    1, 2, 3, 4, 6 and 8 K slices; the slice count chosen with them is within
//    0.7 % of the best measured one on average (1.9 % on 120 random products
//    with m, n = 64 .. 2900, k = 400 .. 32000, 1 .. 100 entries, 1 .. 32
//    slices forced).
constexpr double kStage256x128[3] = {0.8e-6, 1.0e-6, 1.82e-6};
constexpr double kStage128x128[3] = {0.45e-6, 0.6e-6, 0.99e-6};
constexpr double kStage64x64 = 0.25e-6;
constexpr double kTileOverhead = 7e-6;    // pipeline fill + epilogue of a tile
constexpr double kFoldLaunch = 6e-6;      // the pass that adds the K slices
constexpr double kFoldBytesPerS = 3e12;   // ... reads and writes its planes at
constexpr double kSplitMustBeat = 0.95;   // a split has to win by 5 %
// -- tile choice, cost of a tile in units of one 128x128 tile.  Sweep: both
//    tiles forced on 124 products, 1024^2 .. 8192^2, k = 256 .. 4096, some
//    batched: the choice is within 0.4 % of the faster tile on average.
constexpr double kUnits256x128 = 2.0;
constexpr double kUnits128x128 = 1.2;     // one and two terms
//    Three terms (sweep: both tiles forced on 36 products, 1024^2 .. 8192^2,
//    k = 1024 .. 5000, some batched or rectangular: a round of 256x128 tiles
//    costs 1.8 rounds of 128x128 tiles, so the large tile wins when it halves
//    the rounds, 8 to 14 %, and loses otherwise, 3 % at 7 -> 4 rounds, 17 to
//    20 % at 3 -> 2).
constexpr double kUnits256x128Terms3 = 1.8;
constexpr double kUnits128x128Terms3 = 1.0;
constexpr double kUnits64x64 = 0.4;
constexpr double units256x128(const int terms) {
  return terms == 3 ? kUnits256x128Terms3 : kUnits256x128;
}
constexpr double units128x128(const int terms) {
  return terms == 3 ? kUnits128x128Terms3 : kUnits128x128;
}
// -- K slices for a partly empty last round: slices, pipeline refills, fold.
//    Sweep: 126 products, 2304^2 .. 8192^2, k = 2048 .. 8192, two policies.
constexpr double kTailOverhead = 0.2;
// -- which path: the single kernel, split passes + GEMM on packed operands, or
//    the GEMM kernel that splits the fp32 operands itself.  Fit: 1860 random
//    products (m, n = 45 .. 5000, k = 32 .. 32768, 1 .. 1024 entries, half of
//    them with dimensions that are multiples of nothing, all five policies),
//    each run with every path forced; the constants below minimise the
//    squared log error of each path's estimate on 1060 of them and on 137
//    structured products (the reference harness's grid with 256 entries,
//    squares 1024 .. 8192, the baseline workloads; weighted four times).  On
//    the 800 held out the path chosen with them is 1.4 % slower than always
//    taking the fastest forced path on average (37 of 800 above 1.10 x, six
//    above 1.25 x), on the structured ones 0.5 % (two above 1.10 x); the
//    constants before (fits to the harness's grid and to square products)
//    were 3 to 6 % slower on the same 800, 3.1 x at worst.  Whole default
//    calls on 400 further random products: 1.1 % (worst 1.48 x).
//    Rows: one, two, three terms.
struct PathRates {
  double launch, stage, tile, bytes_per_s; // seconds, seconds, seconds, B/s
  double split_bytes_per_s;                // packed path only
  // A k stage takes longer the fuller the chip is (power limit, contention in
  // L2 and HBM): stage * (1 + busy * (compute units with a tile / all compute
  // units, averaged over the rounds))
  double busy;
};
constexpr PathRates kPacked[3] = {
    {8.35e-6, 0.131e-6, 3.07e-6, 3.65e12, 5.61e12, 0.359},
    {8.17e-6, 0.287e-6, 3.69e-6, 6.50e12, 5.57e12, 0.649},
    {7.10e-6, 0.652e-6, 4.65e-6, 6.50e12, 4.92e12, 0.361}};
// -- the packed path's GEMM kernel reading and splitting the fp32 operands
//    itself (256x128 tiles only; rows: one, two terms)
constexpr PathRates kDirect[2] = {
    {3.41e-6, 0.173e-6, 3.76e-6, 4.62e12, 0., 1.18},
    {5.00e-6, 0.355e-6, 3.65e-6, 4.92e12, 0., 0.750}};
// ... as the host sees it when it decides whether a launch of that kernel is
// bound by its bytes and should start its workgroups staggered (a fit of its
// own, to the reference harness's grid: 0.8 / 1.5 us per k stage of a 256x128
// tile and 6 us per tile, in units of half a tile)
constexpr PathRates kDirectStagger[2] = {
    {6.0e-6, 0.40e-6, 3.0e-6, 5.0e12, 0., 0.},
    {6.0e-6, 0.75e-6, 3.0e-6, 5.0e12, 0., 0.}};
// with K slices: the GEMM's time against the packed kernel's estimate for the
// same slices of 256x128 tiles (two terms: twelve K-sliced products, m, n =
// 64 .. 4096, k = 2048 .. 262144, each run on either path: with 1.4 the faster
// path is chosen for all of them, with 1.5 for eleven)
constexpr double kDirectSliceRatio[2] = {1.5, 1.4};
// Products that are cut into K slices (few output tiles): what the slice
// planner's time (split_time, whose constants are fitted for choosing the slice
// count) has to be scaled and shifted by to be the time of the whole call on
// each path; same fit as above.  Rows: scale, shift in seconds; by terms.
constexpr double kSlicedPacked[2][3] = {{0.724, 0.954, 0.955},
                                        {-0.65e-6, -6.0e-6, -6.0e-6}};
constexpr double kSlicedDirect[2][2] = {{0.759, 0.890}, {-6.0e-6, -6.0e-6}};
// Calls issued back to back cannot complete faster than the host issues their
// launches (250 products below 1.5e8 flop, called in a loop: 11, 14.5 and 12 us
// per call in the median): what decides among the paths for tiny products -
// one launch for the single kernel and the direct kernel, two or three for
// the packed path.  Order: single kernel, packed, direct.
constexpr double kCallFloor[3] = {11.0e-6, 14.3e-6, 11.5e-6};
// -- the single kernel (one launch, fp32 operands), by terms.  Its 64x64 tile
//    runs alone on a compute unit (stage64, tile64) or as one of two (pair64,
//    pair_tile64, for both), its 128x128 tile always alone; rows64 / rows128:
//    factor on a stage when an operand does not have k contiguous; busy64 (for
//    pairs) / busy128 as PathRates::busy.  Fit: 3000 random products (m, n =
//    32 .. 4096, k = 32 .. 8192, 1 .. 1024 entries, three transpose
//    combinations), each run with both tiles: 5 to 12 % rms, the tile chosen
//    with them 0.03 to 0.3 % slower than the faster one on average; stage64 is
//    that of operands that come from HBM (0.34, 0.40, 0.53 us; from L2 0.18,
//    0.32, 0.47), which one workgroup of a compute unit cannot hide.  The launch
//    is 0.8 us above the fit to those launches inside a graph, as the other
//    paths' are.
struct FusedRates {
  double launch, stage64, tile64, pair64, pair_tile64, busy64, rows64;
  double stage128, tile128, busy128, rows128, bytes_per_s;
};
constexpr FusedRates kFused[3] = {
    {4.1e-6, 0.330e-6, 1.18e-6, 0.242e-6, 2.06e-6, 0.811, 1.232,
     0.314e-6, 2.15e-6, 0.854, 1.114, 4.92e12},
    {4.7e-6, 0.360e-6, 0.97e-6, 0.341e-6, 1.90e-6, 0.748, 1.185,
     0.551e-6, 2.12e-6, 0.522, 1.157, 4.74e12},
    {5.2e-6, 0.500e-6, 0.41e-6, 0.601e-6, 1.70e-6, 0.465, 1.101,
     0.909e-6, 2.02e-6, 0.434, 1.084, 3.95e12}};
// ('T','N') products of at least 1024 x 1024 x 512, and fewer than 16 entries, take
// the single kernel only where it is well ahead: its time counts this much there.
// The path query answers for exactly these, and its answers for them are kept
// (1160x1544x1056, two terms: packed operands, though the single kernel takes 0.8
// of the time).  All others go by the times alone: on smaller outputs and shorter
// k the factor turned away products the single kernel takes 0.81 of the packed
// and 0.78 of the direct path's time for (medians of 63; 143 in all, where it is
// 0.65 to 1.18 of the path taken, above 1.03 for three), and made them need a
// workspace.
constexpr double kFusedTnMargin[3] = {1.25, 1.4, 1.25}; // by terms
constexpr bool fused_tn_margin(const int m, const int n, const int k,
                               const int batch) {
  return m >= 1024 && n >= 1024 && k >= 512 && batch < 16;
}
// An uncut product that would run in the direct kernel and moves more than the
// 256 MiB of the memory-side cache, with k above two stages and tiles of 256x128
// that lie within C for two thirds or more: the single kernel overlaps its stages
// with that traffic less well than its estimate says (1024^2 x 128, 256 entries:
// 403 us for 355 estimated, the direct kernel 347; 1024x768x224 x 256, one term,
// 393 against 287).  Of 119 products of the direct kernel that the times alone
// moved to the single kernel 17 became more than 5 % slower, up to 1.36 times,
// with this factor 4 stay so; none of 113 that had run in the single kernel before
// loses more than 4 %.
constexpr double kFusedStreamMargin = 1.4;
inline double fused_direct_margin(const int m, const int n, const int k,
                                  const int batch) {
  const double c = static_cast<double>(m) * n,
               bytes = 4.0 * batch * (c + (static_cast<double>(m) + n) * k),
               tiles = 32768.0 * static_cast<double>(ceil_div(m, 256) *
                                                     ceil_div(n, 128));
  return bytes > 256.0 * (1 << 20) && k > 64 && tiles < 1.5 * c
             ? kFusedStreamMargin
             : 1.0;
}
// An uncut product that the path query gives to another path runs in the single
// kernel where its own time is below this much of that path's estimate.  Of 500
// random ('T','N') products of those paths (m, n = 32 .. 8192, k up to 65536, 1 ..
// 1024 entries; each run both ways): packed operands with two or three terms, 214
// below 0.95, 0.66 of the time in the median, none above 1.03 (one term below 0.75:
// 425x1440x1450 x 3 at 0.8 is 1.2 times slower; the leading product outside the
// matrix core: 25 below 1.15, 0.55, none above 1.05; three terms of it in 128x128
// tiles, which are short of registers, below 1.03: of 78 more seven are 6 to 15 %
// slower between that and 1.15, 1862x1719x3244 x 24 3636 us for 3165, and one 3 %
// faster); the direct kernel below 0.75,
// 0.83, two above 1.03 (all of 20 that take it less than 20 us are faster), and
// below 0.6 where the batch exceeds the 256 MiB of the memory-side cache, 0.82
// (95x125x10978 x 172 at 0.64 is 1.3 times slower: the single kernel's estimate
// overlaps stages and traffic too well there).
constexpr double kSinglePacked = 0.95, kSinglePackedOneTerm = 0.75,
                 kSinglePackedRn = 1.15, kSinglePackedRnThreeTerms = 1.03,
                 kSingleDirect = 0.75,
                 kSingleDirectShort = 20e-6, kSingleDirectLarge = 0.6;
// Adding a K slice to the double-precision sums, for the workgroups of a compute
// unit at a time: 110 products run with the cut and uncut, 0.17 us in the median
// (one workgroup a unit), 0.10 (two), 3 % of a call.
constexpr double kFusedSliceFold = 0.15e-6;
// A product whose K is cut goes to the single kernel where this factor on its
// time still leaves it ahead.  In place of packed operands: of 120 products taken
// with it, 0.72 of their time in the median, none above 1.02.  In place of the
// direct kernel (by terms), whose one launch on 256x128 tiles loses least to long
// k: with 1.1 there too, 15 of 70 products that the larger factor turns away ran
// 1.03 to 1.74 times slower than the direct kernel, most of them with one term.
constexpr double kFusedSlicedMargin = 1.1;
constexpr double kFusedSlicedDirectMargin[2] = {1.25, 1.4};
// The single kernel with a workgroup for every K slice, by tile (64x64, 128x128)
// and terms: launch, a stage of a 64x64 tile with at most one workgroup on a
// compute unit, a stage with all resident ones (twice that for 64x64) and how
// much longer the fuller the chip is, pipeline fill and the slice's sums, the last
// workgroup's reading of one slice.  Fit: 1000 random products that are cut (m, n
// = 32 .. 8192, k up to 65536, 1 .. 1024 entries, all layouts), each with both
// tiles: 5 to 9 % rms (three terms), 9 to 12 (two), 15 to 17 (one).
struct SpreadRates {
  double launch, alone, stage, busy, tile, fold;
};
constexpr SpreadRates kSpread[2][3] = {
    {{4.9e-6, 0.184e-6, 0.300e-6, 1.03, 4.92e-6, 0.278e-6},
     {6.6e-6, 0.280e-6, 0.466e-6, 0.325, 3.94e-6, 0.263e-6},
     {6.1e-6, 0.496e-6, 0.782e-6, 0.093, 3.60e-6, 0.239e-6}},
    {{2.5e-6, 0., 0.216e-6, 2.03, 7.46e-6, 0.874e-6},
     {1.3e-6, 0., 0.469e-6, 0.772, 9.13e-6, 0.872e-6},
     {4.8e-6, 0., 0.675e-6, 0.812, 6.64e-6, 0.880e-6}}};
constexpr double kSpreadBytesPerS = 4.9e12;
// ... in place of the other kernels where their estimates are this many times its
// own.  1500 random products that are cut, each run without it and with both
// tiles, and 110 more for the direct kernel beyond a round of 128x128 tiles:
// * packed operands, 64x64 tiles that are all resident: 0.95 (both estimates are
//   too long for tiny outputs); more of them, and 128x128 tiles: 1.2.  Of 973
//   products 8 are more than 2 % slower than on packed operands, at most 10 %, all
//   of 973 take 0.73 of their time.  (1.2 everywhere, and packed operands taken
//   for no faster than 15 us and 0.4 a slice, which held before the fold read
//   its slices in groups: 17 more than 2 % slower, 256x288x6176 in 28 slices 30.2
//   us for 23.9.)
// * the direct kernel: 1.35 and 1.25 for one and two terms (1.25 for one term:
//   128x5376x7232 41.0 us for 37.7), 1.5 for 128x128 tiles of more than a round:
//   of those 110 products one is faster so, 3616x256x1696 x 3 56.7 us for 46.5.
// * the single kernel's slices one after the other, by tile and terms: of 244 such
//   products three are more than 3 % slower, at most 6 %, all take 0.87 of their
//   time.  (1.25 against an estimate that holds margins of its own: nine,
//   1248x96x1024 x 4 20.6 us for 16.0, 68x2738x891 14.4 for 11.5.)
constexpr double kSpreadPackedMargin[2] = {0.95, 1.2},
                 kSpreadDirectMargin[2] = {1.35, 1.25},
                 kSpreadDirectRounds = 1.5,
                 kSpreadSlicedMargin[2][3] = {{1.2, 1.14, 1.12},
                                              {1.1, 1.14, 1.12}};
// Its workgroups that are resident on a compute unit: 12 waves of up to 168
// registers (128x128), twice 8 waves of up to 128.
constexpr int fused_resident(const int bm) { return bm > 64 ? 1 : 2; }
// k % 32 != 0: the kernel variant that reads a shorter last stage (1024^2 x 1000
// against x 1024, batch 256: 301 against 336 TFLOPS, of which 2.4 % are the k)
constexpr double kDirectTailStage = 1.47;
} // namespace fit

// XCDs (chiplets with an L2 of their own) behind the current device.  HIP does
// not report them; a gfx950 XCD has 32 active compute units in every partition
// mode (SPX 256 = 8 x 32, DPX 128, QPX 64, CPX 32), so the count follows from
// the compute units.  Consecutive workgroup ids go round-robin over the XCDs;
// the kernels' XCD-aware item lists are written for eight of them and are used
// only then (other counts take the plain shared list: same results, tiles not
// grouped by L2).
inline int device_xcds() {
  const int cus = device_cus();
  return cus % 32 == 0 ? cus / 32 : 1;
}
constexpr int kKernelXcds = 8; // the constant XCDS of the kernels' item lists

// Number of K slices of every tile, when the 256x128 output tiles cannot fill
// half the chip.  For every candidate (at most 32 slices of at least 6 stages)
// the GEMM's time is estimated the way gemm_by_size will run it: the tile that
// the slice count leads to, rounds of those tiles over the compute units,
// stages per slice at that tile's time per stage, a fixed time per tile, and
// for more than one slice the fold (a launch plus the planes written and
// read).  The cheapest count is taken, any split having to beat the uncut run
// by 5 %.  Times per stage and tile: fits to measurements on MI355X (216
// products, m = n = 512 .. 2048, k = 512 .. 4096, one to three terms, each run
// with 1, 2, 3, 4, 6 and 8 slices: the choice is within 0.7 % of the best measured count on
// average; "as many slices as fill the chip with 256x128 tiles" was 7 % off,
// over-cutting outputs from 1280^2 up and not cutting short loops at all).
// Whether the 256x128 tile is a candidate at all: only where the 128x128 tiles
// need more than one round over the compute units (in a single round the
// smaller tile always finishes first), and not for the one-term kernels on
// loops of 32 stages or fewer, where the stores of C dominate and the smaller
// tile measured 8 to 12 % faster.  (Forced-tile runs of 124 products: the
// choice below is within 0.4 % of the faster tile on average; requiring a full
// round of 256x128 tiles instead had cost 2 %, up to 13 % at 2560^2 .. 2816^2.)
inline bool big_tile_candidate(const int terms, const long long mid,
                               const int kt) {
  return mid > device_cus() && !(terms == 1 && kt <= 32);
}
// `direct`: the kernel that splits the fp32 operands itself, which has the
// 256x128 tile only and takes kDirectSliceRatio times the packed kernel's time
// (its slice count must be planned with its own tiles: 4096 x 64 x 4096 cut
// for the 128x128 tiles of the packed path left half the compute units
// without a 256x128 item, 48 against 39 us).
inline double split_time(const int terms, const int m, const int n,
                         const int batch, const int kt, const int slices,
                         const bool direct = false) {
  const long long cus = device_cus();
  const int stages = static_cast<int>(ceil_div(kt, slices));
  const long long z = ceil_div(kt, stages);
  const long long big = ceil_div(m, 256) * ceil_div(n, 128) * batch * z;
  const long long mid = ceil_div(m, 128) * ceil_div(n, 128) * batch * z;
  double stage_time, rounds;
  const double r_big = static_cast<double>(ceil_div(big, cus));
  const double r_mid = static_cast<double>(ceil_div(mid, cus));
  if (direct ||
      (big_tile_candidate(terms, mid, stages) &&
       r_big * fit::units256x128(terms) <= r_mid * fit::units128x128(terms))) {
    stage_time = fit::kStage256x128[terms - 1];
    rounds = r_big;
  } else if (mid >= cus || (m > 64 && n > 64)) {
    stage_time = fit::kStage128x128[terms - 1];
    rounds = r_mid;
  } else {
    stage_time = fit::kStage64x64;
    rounds = static_cast<double>(
        ceil_div(ceil_div(m, 64) * ceil_div(n, 64) * batch * z, cus));
  }
  double t = rounds * (stages * stage_time + fit::kTileOverhead);
  if (z > 1)
    t += fit::kFoldLaunch + static_cast<double>(z + 1) * m * n * batch * 4.0 /
                                fit::kFoldBytesPerS;
  return direct ? t * fit::kDirectSliceRatio[terms - 1] : t;
}
// Test hook (wmmae_tcec_force_k_slices): a slice count for the calling thread's
// next calls instead of the estimates' choice, so that two kernels can be run on
// the same cut of K and compared bit by bit.  0: the estimates choose.
inline thread_local int t_forced_k_slices = 0;
// Measurement hook (wmmae_tcec_time_gemm_kernel): events this thread's calls
// record on their stream right before the MFMA GEMM kernel and right after it
// (after the fold of its K slices where there is one).
inline thread_local hipEvent_t t_gemm_begin = nullptr, t_gemm_end = nullptr;
constexpr int kMaxSplits = 32, kMinStagesPerSplit = 6;
inline int choose_splits(const int terms, const int m, const int n, const int k,
                         const int batch, const bool direct = false) {
  const long long tiles = ceil_div(m, 256) * ceil_div(n, 128) * batch;
  const int kt = static_cast<int>(ceil_div(k, 32));
  if (t_forced_k_slices > 0) {
    const int s = std::max(
        1, std::min({t_forced_k_slices, kMaxSplits, kt / kMinStagesPerSplit}));
    return static_cast<int>(ceil_div(kt, ceil_div(kt, s)));
  }
  if (tiles * 2 > device_cus())
    return 1;
  int best = 1;
  double t_best =
      fit::kSplitMustBeat * split_time(terms, m, n, batch, kt, 1, direct);
  for (int s = 2; s <= kMaxSplits && s * kMinStagesPerSplit <= kt; s++) {
    if (ceil_div(kt, ceil_div(kt, s)) != s)
      continue; // the same slices as a smaller count
    const double t = split_time(terms, m, n, batch, kt, s, direct);
    if (t < t_best) {
      t_best = t;
      best = s;
    }
  }
  return best;
}

// K slices for the tiles of the last round only.  `tiles` output tiles run in
// rounds of `resident` (one workgroup per item, long K loops); when the last
// round is less than half full its tiles are cut into `slices` K slices of at
// least 32 stages each, so that the round takes about 1/slices of a tile's
// time (plus the pass that folds the slices).  slices == 1: not worth it.
struct TailPlan {
  long long full = 0, tail = 0; // tiles in whole rounds, tiles in the last
  int slices = 1, stages = 0;   // K slices of a tail tile, stages per slice
};
inline TailPlan plan_tail(const long long tiles, const long long resident,
                          const int KT) {
  TailPlan t;
  t.full = tiles / resident * resident;
  t.tail = tiles - t.full;
  if (t.full == 0 || t.tail == 0 || t.tail * 2 > resident || KT < 64)
    return t;
  long long s = std::min<long long>({resident / t.tail, KT / 32, 16});
  if (s < 2)
    return t;
  t.stages = static_cast<int>(ceil_div(KT, s));
  t.slices = static_cast<int>(ceil_div(KT, t.stages));
  return t;
}
// Time of `tiles` tiles in units of one tile, with and without that plan.
inline double rounds_cost(const long long tiles, const long long resident,
                          const int KT, const bool tail_allowed) {
  const TailPlan t = plan_tail(tiles, resident, KT);
  const double full_rounds = static_cast<double>(t.full / resident);
  if (t.tail == 0)
    return full_rounds;
  if (!tail_allowed || t.slices < 2)
    return full_rounds + 1.0;
  return full_rounds + 1.0 / t.slices + fit::kTailOverhead;
}

// Deepest LDS ring (at most 4 stages) that fits the 160 KiB of a compute unit.
constexpr int ring_depth(const int bm, const int bn, const int terms) {
  const int stage_bytes = (bm / 16 + bn / 16) * terms * 1024;
  const int fit = (160 * 1024) / stage_bytes;
  return fit > 4 ? 4 : fit;
}

// ------------------------------------------------------ fused small GEMM
struct FusedArgs {
  wmmae_gemm::FusedSpreadParams p = {};
  // > 0: K slices made by a workgroup each, with tiles of this size
  int spread_tile = 0;
  hipStream_t stream;
};
// What those take of a workspace: a tile's sums for every slice, and a word a tile
inline size_t fused_spread_planes(const int m, const int n, const int batch,
                                  const int slices, const int tile) {
  return static_cast<size_t>(ceil_div(m, tile) * ceil_div(n, tile)) * batch *
         slices * tile * tile * 4u;
}
inline size_t fused_spread_bytes(const int m, const int n, const int batch,
                                 const int slices, const int tile) {
  return fused_spread_planes(m, n, batch, slices, tile) +
         static_cast<size_t>(ceil_div(m, tile) * ceil_div(n, tile)) * batch * 8u;
}

// Time of a call of the single kernel with its 64x64 or 128x128 tiles.  `rows`:
// an operand does not have k contiguous.  `slices`: K slices made in the kernel,
// more than one with 64x64 tiles only (the double-precision sums of a 128x128
// tile fit neither the registers nor LDS).
inline double fused_time(const int terms, const int m, const int n, const int k,
                         const int batch, const bool small, const bool rows,
                         const int slices = 1) {
  const fit::FusedRates &f = fit::kFused[terms - 1];
  const double kt = static_cast<double>(ceil_div(k, 32));
  const long long cus = device_cus();
  const int t = small ? 64 : 128;
  const long long tiles = ceil_div(m, t) * ceil_div(n, t) * batch;
  const long long rounds = ceil_div(tiles, cus);
  const double full = static_cast<double>(tiles) /
                      (static_cast<double>(rounds) * static_cast<double>(cus));
  double time;
  if (small) {
    const double factor = rows ? f.rows64 : 1.0;
    time = static_cast<double>(rounds / 2) *
               (kt * f.pair64 * factor * (1.0 + f.busy64 * full) +
                f.pair_tile64) +
           static_cast<double>(rounds % 2) * (kt * f.stage64 * factor + f.tile64) +
           (slices > 1 ? static_cast<double>(rounds) * slices *
                             fit::kFusedSliceFold
                       : 0.);
  } else {
    time = static_cast<double>(rounds) *
           (kt * f.stage128 * (rows ? f.rows128 : 1.0) *
                (1.0 + f.busy128 * full) +
            f.tile128);
  }
  const double bytes =
      4.0 * batch *
      (static_cast<double>(m) * n + (static_cast<double>(m) + n) * k);
  return f.launch + std::max(time, bytes / f.bytes_per_s);
}
// Time of a call whose K slices are made by a workgroup each.
inline double fused_spread_time(const int terms, const int m, const int n,
                                const int k, const int batch, const bool small,
                                const int slices) {
  const fit::SpreadRates &f = fit::kSpread[small ? 0 : 1][terms - 1];
  const double kt = static_cast<double>(ceil_div(ceil_div(k, 32), slices));
  const int t = small ? 64 : 128;
  const double items = static_cast<double>(ceil_div(m, t) * ceil_div(n, t)) *
                       batch * slices;
  const double x =
      items / (static_cast<double>(device_cus()) * fit::fused_resident(t));
  double time;
  if (small && x <= 0.5) {
    time = kt * f.alone + 0.5 * f.tile;
  } else {
    // (workgroups follow one another as they end, not in rounds)
    const double whole = std::ceil(x);
    const double rounds = x <= 1. ? 1. : 0.35 * whole + 0.65 * x;
    time = rounds * (kt * f.stage * (1. + f.busy * x / whole) + f.tile);
  }
  const double bytes =
      4.0 * batch *
      (static_cast<double>(m) * n + (static_cast<double>(m) + n) * k);
  return f.launch + std::max(time, bytes / fit::kSpreadBytesPerS) +
         slices * f.fold;
}
inline bool fused_small_tiles(const int terms, const int m, const int n,
                              const int k, const int batch, const bool rows) {
  return fused_time(terms, m, n, k, batch, true, rows) <=
         fused_time(terms, m, n, k, batch, false, rows);
}
// The kernels of one policy, as the driver calls them: one table per policy,
// filled in the gemm_*.hip translation units, which is what lets the kernels
// compile side by side.
struct PolicyKernels {
  // splits one operand (b == nullptr) or both of a product
  int (*pack)(int k, int batch, const PackSource &a, const PackSource *b,
              hipStream_t stream);
  int (*gemm)(const GemmArgs &g);
  int (*gemm_rn)(const GemmArgs &g); // nullptr: the policy has no such variant
  int (*fused)(const FusedArgs &f);
  int (*fused_rn)(const FusedArgs &f); // as gemm_rn
  // resident workgroups per compute unit of the packed kernel with tile shape
  // 0 (256x128), 1 (128x128) or 2 (64x64): the number the launch plans its
  // rounds with, for the workspace query
  int (*per_cu)(int shape);
};
const PolicyKernels &kernels_f16_ec();
const PolicyKernels &kernels_f16_noec();
const PolicyKernels &kernels_bf16x3_ec();
const PolicyKernels &kernels_bf16x2_ec();
const PolicyKernels &kernels_bf16_noec();
inline const PolicyKernels *policy_kernels(const int policy) {
  switch (policy) {
  case WMMAE_POLICY_F16_EC:
    return &kernels_f16_ec();
  case WMMAE_POLICY_F16_NOEC:
    return &kernels_f16_noec();
  case WMMAE_POLICY_BF16X3_EC:
    return &kernels_bf16x3_ec();
  case WMMAE_POLICY_BF16X2_EC:
    return &kernels_bf16x2_ec();
  case WMMAE_POLICY_BF16_NOEC:
    return &kernels_bf16_noec();
  default:
    return nullptr;
  }
}

} // namespace wmmae_driver
