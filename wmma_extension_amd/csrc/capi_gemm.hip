// extern "C" boundary of libwmmae_tcec.so, GEMM driver part: argument
// validation and path selection; the kernels live in the gemm_*.hip
// translation units, one per policy.  Declarations and per-entry documentation
// live in include/wmmae_tcec.h.
#include "gemm_plan.hpp"
#include <cmath>
#include <chrono>
#include <unistd.h>

namespace {
using namespace wmmae_driver;

// --------------------------------------------------------------------------
// scale_c_kernel: C = beta * C, the whole result when k == 0.
// --------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
    scale_c_kernel(float *__restrict__ C, const int M, const int N,
                   const long long ldc, const long long batch_stride_c,
                   float *const *__restrict__ c_ptrs, const float beta,
                   const unsigned entry0) {
  const long long e = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= static_cast<long long>(M) * N)
    return;
  const long long entry = entry0 + blockIdx.y;
  float *const cb =
      c_ptrs != nullptr ? c_ptrs[entry] : C + entry * batch_stride_c;
  float *const p = cb + (e % M) + (e / M) * ldc;
  *p = beta == 0.f ? 0.f : beta * *p;
}

// Which of the three paths?  The single ("fused") kernel reads the fp32 operands
// once per 64 or 128 rows or columns of C and takes one launch, in any layout;
// the packed path first writes and re-reads the split operands, which pays off
// when every operand element is used by many tiles, and can cut K where there
// are few; the "direct" path is the packed path's GEMM kernel (256x128 tiles)
// loading the fp32 operands itself and splitting them on their way into LDS - no
// packed copy and no split pass, at 1.2 to 1.9 times the time per k stage; it
// wins where an operand element is used by few tiles (batches of medium
// matrices, K-heavy products) and needs k contiguous in both operands, k at
// least 4 and at most two terms; same bits as the packed path.  All three times
// are estimated with the same shape, a launch cost plus rounds of tiles over the
// compute units times (k stages * time per stage + time per tile), bounded below
// by the bytes moved; products that are cut into K slices take the slice
// planner's time, rescaled.  The constants and what they were fitted to:
// namespace fit.
//   fused_ok : the single kernel is considered (fused_considered)
//   rows     : an operand does not have k contiguous
// The single kernel stands in for the faster of the other two, with that path's
// K slices (SLICED in its head comment): the choice never changes a bit, and no
// product is summed in a longer fp32 chain for being small.  (Taken by its time
// alone, over an uncut K, it left 1024^3 in two fp16 terms with a relative
// error of 2.2e-7 where the four slices give 1.3e-7, 8 x 320x321x12900 in three
// bf16 terms of one sign with 5.8e-7 for 0.8e-7.)
enum class Path { Fused, Packed, Direct };
// (see PathRates::busy)
inline double busy_factor(const fit::PathRates &r, const long long tiles) {
  const long long cus = device_cus();
  return 1.0 + r.busy * static_cast<double>(tiles) /
                   static_cast<double>(ceil_div(tiles, cus) * cus);
}
// the direct kernel's time without K slices: rounds of 256x128 tiles over the
// compute units, and the bytes it moves
struct DirectTimes {
  double tiles, bytes;
};
inline DirectTimes direct_times(const int m, const int n, const int k,
                                const int batch, const fit::PathRates &d) {
  const double kt = static_cast<double>(ceil_div(k, 32));
  const long long tiles256 = ceil_div(m, 256) * ceil_div(n, 128) * batch;
  const double ab = (static_cast<double>(m) + n) * k * batch;
  // (the variant for k % 32 != 0 spends one more instruction per load)
  const double stage = d.stage * busy_factor(d, tiles256) *
                       (k % 32 == 0 ? 1.0 : fit::kDirectTailStage);
  return {fit::kUnits256x128 *
              static_cast<double>(ceil_div(tiles256, device_cus())) *
              (kt * stage + d.tile),
          (4.0 * m * n * batch + 4.0 * ab) / d.bytes_per_s};
}
constexpr int kPathFlags =
    WMMAE_FLAG_PATH_PACKED | WMMAE_FLAG_PATH_FUSED | WMMAE_FLAG_PATH_DIRECT;
constexpr int kAllFlags = WMMAE_FLAG_RN_MAIN | kPathFlags;
inline bool one_path_at_most(const int flags) {
  const int f = flags & kPathFlags;
  return (f & (f - 1)) == 0;
}
// Estimated time of a call on each path, in seconds; a path that cannot run
// the product (or is not considered for it) has infinity.
struct PathEstimates {
  double packed, direct;
  Path base;          // the faster of the two ...
  int slices;         // ... the K slices it makes, 1: none ...
  double base_time;   // ... and its time, no less than issuing its launches takes
  double fused;       // the single kernel with that cut of K
};
inline PathEstimates estimate_paths(const int m, const int n, const int k,
                                    const int batch, const int terms,
                                    const bool fused_ok, const bool rows,
                                    const bool direct_ok) {
  constexpr double kNever = std::numeric_limits<double>::infinity();
  PathEstimates e{kNever, kNever, Path::Packed, 1, kNever, kNever};
  const auto finish = [&]() {
    e.base_time = std::max(e.packed, fit::kCallFloor[1]);
    const double direct = std::max(e.direct, fit::kCallFloor[2]);
    if (direct < e.base_time) {
      e.base = Path::Direct;
      e.base_time = direct;
    }
    e.slices = choose_splits(terms, m, n, k, batch, e.base == Path::Direct);
    if (!fused_ok)
      return e;
    if (e.slices > 1)
      e.fused = (e.base == Path::Direct
                     ? fit::kFusedSlicedDirectMargin[terms - 1]
                     : fit::kFusedSlicedMargin) *
                fused_time(terms, m, n, k, batch, true, rows, e.slices);
    else
      e.fused = (!rows && fit::fused_tn_margin(m, n, k, batch)
                     ? fit::kFusedTnMargin[terms - 1]
                     : 1.0) *
                (e.base == Path::Direct
                     ? fit::fused_direct_margin(m, n, k, batch)
                     : 1.0) *
                std::min(fused_time(terms, m, n, k, batch, true, rows),
                         fused_time(terms, m, n, k, batch, false, rows));
    return e;
  };
  const fit::PathRates &p = fit::kPacked[terms - 1];
  const long long cus = device_cus();
  const int kti = static_cast<int>(ceil_div(k, 32));
  const double kt = static_cast<double>(kti);
  const double c_bytes = 4.0 * m * n * batch;
  const double ab = (static_cast<double>(m) + n) * k * batch; // operand elements
  const long long tiles64 = ceil_div(m, 64) * ceil_div(n, 64) * batch;
  const long long tiles128 = ceil_div(m, 128) * ceil_div(n, 128) * batch;
  const long long tiles256 = ceil_div(m, 256) * ceil_div(n, 128) * batch;

  const double split_pass = (4.0 + 2.0 * terms) * ab / p.split_bytes_per_s;
  const int splits = choose_splits(terms, m, n, k, batch);
  if (splits != 1) {
    // K slices: the split pass and the packed kernel's slices against the
    // slower stages of the direct kernel (cut into the slices that suit its own
    // tile)
    e.packed = (p.launch + split_pass +
                split_time(terms, m, n, batch, kti, splits)) *
                   fit::kSlicedPacked[0][terms - 1] +
               fit::kSlicedPacked[1][terms - 1];
    if (direct_ok)
      e.direct =
          (fit::kDirect[terms - 1].launch +
           split_time(terms, m, n, batch, kti,
                      choose_splits(terms, m, n, k, batch, true), true)) *
              fit::kSlicedDirect[0][terms - 1] +
          fit::kSlicedDirect[1][terms - 1];
    return finish();
  }
  // packed path: rounds in units of one 128x128 tile as gemm_by_size counts
  // them (a 256x128 tile 2.0 and a 128x128 tile 1.2 for one and two terms,
  // 1.8 and 1.0 for three, a 64x64 tile 0.4)
  double units;
  long long p_tiles;
  const double r128 = static_cast<double>(ceil_div(tiles128, cus));
  if (big_tile_candidate(terms, tiles128, kti) &&
      fit::units256x128(terms) * static_cast<double>(ceil_div(tiles256, cus)) <=
          fit::units128x128(terms) * r128) {
    units = fit::units256x128(terms) *
            static_cast<double>(ceil_div(tiles256, cus));
    p_tiles = tiles256;
  } else if (tiles128 >= cus || (m > 64 && n > 64)) {
    units = r128 * fit::units128x128(terms);
    p_tiles = tiles128;
  } else {
    units = fit::kUnits64x64 * static_cast<double>(ceil_div(tiles64, cus));
    p_tiles = tiles64;
  }
  e.packed = p.launch + split_pass +
             std::max(units * (kt * p.stage * busy_factor(p, p_tiles) + p.tile),
                      c_bytes / p.bytes_per_s);
  if (direct_ok) {
    const DirectTimes d =
        direct_times(m, n, k, batch, fit::kDirect[terms - 1]);
    // (it cuts K for its own tile even where the packed path would not)
    const int own = choose_splits(terms, m, n, k, batch, true);
    e.direct =
        own > 1 ? (fit::kDirect[terms - 1].launch +
                   split_time(terms, m, n, batch, kti, own, true)) *
                          fit::kSlicedDirect[0][terms - 1] +
                      fit::kSlicedDirect[1][terms - 1]
                : fit::kDirect[terms - 1].launch + std::max(d.tiles, d.bytes);
  }
  return finish();
}
// How a product runs: the path whose bits it has, that path's K slices, and
// whether the single kernel makes them.
struct Choice {
  Path path; // Path::Fused: the single kernel over an uncut K
  int slices;
  bool single;
  double time = 0.; // estimated
};
inline Choice choose_path(const int m, const int n, const int k, const int batch,
                          const int flags, const int terms, const int policy,
                          const bool fused_ok, const bool rows,
                          const bool direct_ok) {
  // (the round-to-nearest flag with a policy that has no such variant is
  // turned down by the packed path's dispatch)
  const bool rn_unsupported =
      (flags & WMMAE_FLAG_RN_MAIN) != 0 && policy != WMMAE_POLICY_F16_EC &&
      policy != WMMAE_POLICY_BF16X3_EC;
  if (m <= 0 || n <= 0 || k <= 0 || batch <= 0)
    return {Path::Packed, 1, false};
  if (rn_unsupported)
    return {Path::Packed, choose_splits(terms, m, n, k, batch), false};
  const PathEstimates e =
      estimate_paths(m, n, k, batch, terms, fused_ok, rows, direct_ok);
  const double fused = std::max(e.fused, fit::kCallFloor[0]);
  const bool single = e.base == Path::Direct ? fused <= e.base_time
                                             : fused < e.base_time;
  return {single && e.slices == 1 ? Path::Fused : e.base, e.slices, single,
          single ? fused : e.base_time};
}
// what the direct kernel needs of a product (the operands' k strides are 1)
inline bool direct_possible(const int k, const int terms, const int flags,
                            const long long a_rs, const long long b_rs) {
  return k >= 4 && terms <= 2 &&
         (flags & WMMAE_FLAG_RN_MAIN) == 0 && a_rs < (1 << 24) &&
         b_rs < (1 << 24);
}

// Whether a workspace holds packed operands and `more` bytes behind them.
inline bool holds_packed(const int m, const int n, const int k, const int batch,
                         const int terms, const size_t workspace_bytes,
                         const size_t more) {
  const size_t operands = static_cast<size_t>(packed_elems(m, k, terms) +
                                              packed_elems(n, k, terms)) *
                          16u * static_cast<size_t>(batch);
  return workspace_bytes >= operands && workspace_bytes - operands >= more;
}
// A call that its path turns down for the workspace it is given stays with it.
inline bool refused_on_packed(const Choice &c, const int m, const int n,
                              const int k, const int batch, const int terms,
                              const void *const workspace,
                              const size_t workspace_bytes) {
  return !c.single && c.path == Path::Packed && workspace != nullptr &&
         (reinterpret_cast<uintptr_t>(workspace) % 16 != 0 ||
          !holds_packed(m, n, k, batch, terms, workspace_bytes, 0));
}
// Bytes for the K slices of the tiles of a partly empty last round: the largest
// need over the tile shapes and residencies the launch may choose; 0: no such
// tiles.
size_t tail_room(const int policy, const int m, const int n, const int k,
                 const int batch) {
  size_t need = 0;
  if (batch != 1 || m <= 0 || n <= 0)
    return need;
  const int shapes[3][2] = {{256, 128}, {128, 128}, {64, 64}};
  for (int i = 0; i < 3; i++) {
    const int *const sh = shapes[i];
    const TailPlan t =
        plan_tail(ceil_div(m, sh[0]) * ceil_div(n, sh[1]),
                  static_cast<long long>(device_cus()) *
                      policy_kernels(policy)->per_cu(i),
                  packed_k_tiles(k));
    if (t.slices >= 2)
      need = std::max<size_t>(need, static_cast<size_t>(t.slices) *
                                        static_cast<size_t>(t.tail) * sh[0] *
                                        sh[1] * 4u);
  }
  return need;
}
// Whether an uncut product that the path query gives to another path runs in the
// single kernel all the same: same bits, and by its time alone it is ahead
// (estimate_paths holds it back for the query's sake, ('T','N') products of k % 4
// != 0 or of large outputs).
inline bool single_is_ahead(const Choice &c, const int m, const int n,
                            const int k, const int batch, const int flags,
                            const int policy, const int terms, const bool rows,
                            const void *const workspace,
                            const size_t workspace_bytes) {
  // (it counts its tiles in 32 bits, more of them than the other kernels make)
  if (c.single || c.slices != 1 || c.time <= 0. || batch > (1 << 26) ||
      ceil_div(m, 64) * ceil_div(n, 64) * batch >= (1ll << 30) ||
      refused_on_packed(c, m, n, k, batch, terms, workspace, workspace_bytes))
    return false;
  const double bytes =
      4.0 * batch * (static_cast<double>(m) * n + (static_cast<double>(m) + n) * k);
  const double small = fused_time(terms, m, n, k, batch, true, rows),
               large = fused_time(terms, m, n, k, batch, false, rows);
  const double rn = terms == 3 && large < small ? fit::kSinglePackedRnThreeTerms
                                                : fit::kSinglePackedRn;
  const double ahead =
      c.path == Path::Packed
          ? ((flags & WMMAE_FLAG_RN_MAIN) != 0 ? rn
             : terms == 1                      ? fit::kSinglePackedOneTerm
                                               : fit::kSinglePacked)
      : bytes > 256.0 * (1 << 20)        ? fit::kSingleDirectLarge
      : c.time < fit::kSingleDirectShort ? fit::kSinglePacked
                                         : fit::kSingleDirect;
  const double time = std::max(fit::kCallFloor[0], std::min(small, large));
  // (the other kernels cut the tiles of a partly empty last round along K)
  return time < ahead * c.time && tail_room(policy, m, n, k, batch) == 0;
}
// Bytes for the K slices' sums of either GEMM kernel on packed operands or fp32
// ones (the one that splits the fp32 operands itself plans its slices for its own
// tile); 0: neither cuts K.
size_t slices_room(const int terms, const int m, const int n, const int k,
                   const int batch) {
  if (m == 0 || n == 0 || k == 0 || batch == 0)
    return 0;
  const int splits = std::max(choose_splits(terms, m, n, k, batch),
                              direct_possible(k, terms, 0, 1, 1)
                                  ? choose_splits(terms, m, n, k, batch, true)
                                  : 1);
  return splits > 1 ? static_cast<size_t>(splits) * batch * m * n * 4u : 0;
}
// Test hook (wmmae_tcec_force_spread_tile): 0 the estimates choose.
thread_local int t_forced_spread_tile = 0;
// Tile of the single kernel (64 or 128) that makes a cut product's slices with a
// workgroup each, 0: the slices are made as chosen.  The products that run on
// packed operands or in the direct kernel, or whose slices one workgroup of the
// single kernel would make one after the other: too few output tiles to fill the
// chip, and a split pass, a GEMM of at most a round and a fold launch for what is
// one launch here.  The same cut of K, so the same bits: where packed operands
// leave the workspace no room for the slices' sums, that path leaves K whole and
// so does the call.  Needs the caller's workspace to have the room; without one it
// allocates only where the path it stands in for would.
inline int choose_spread(const Choice &c, const int m, const int n, const int k,
                         const int batch, const int terms, const bool rows,
                         const void *const workspace,
                         const size_t workspace_bytes) {
  if (c.slices <= 1 || c.time <= 0. ||
      refused_on_packed(c, m, n, k, batch, terms, workspace, workspace_bytes))
    return 0;
  if (!c.single && c.path == Path::Packed && workspace != nullptr &&
      !holds_packed(m, n, k, batch, terms, workspace_bytes,
                    slices_room(terms, m, n, k, batch)))
    return 0;
  const auto fits = [&](const int tile) {
    return workspace == nullptr
               ? !c.single
               : reinterpret_cast<uintptr_t>(workspace) % 16 == 0 &&
                     workspace_bytes >=
                         fused_spread_bytes(m, n, batch, c.slices, tile);
  };
  if (t_forced_spread_tile != 0)
    return t_forced_spread_tile > 0 && fits(t_forced_spread_tile)
               ? t_forced_spread_tile
               : 0;
  // (its own time: c.time holds margins against the other paths)
  const double instead =
      c.single ? fused_time(terms, m, n, k, batch, true, rows, c.slices) : c.time;
  int chosen = 0;
  double best = std::numeric_limits<double>::infinity();
  for (const int tile : {64, 128}) {
    const double t =
        fused_spread_time(terms, m, n, k, batch, tile == 64, c.slices);
    const bool resident =
        ceil_div(m, tile) * ceil_div(n, tile) * batch * c.slices <=
        static_cast<long long>(device_cus()) * fit::fused_resident(tile);
    const double margin =
        c.single ? fit::kSpreadSlicedMargin[tile == 64 ? 0 : 1][terms - 1]
        : c.path == Path::Packed
            ? fit::kSpreadPackedMargin[tile == 64 && resident ? 0 : 1]
        : tile == 128 && !resident ? fit::kSpreadDirectRounds
                                   : fit::kSpreadDirectMargin[terms - 1];
    if (t < best && t * margin < instead && fits(tile)) {
      chosen = tile;
      best = t;
    }
  }
  return chosen;
}
// Tells a launch's arrival counts in a workspace from whatever else it may hold:
// 58 bits that no other launch of any process is likely to have used.
unsigned long long launch_number() {
  // (std::random_device may throw, which must not reach a C caller)
  static const unsigned long long seed =
      static_cast<unsigned long long>(
          std::chrono::system_clock::now().time_since_epoch().count()) ^
      (static_cast<unsigned long long>(getpid()) << 40) ^
      reinterpret_cast<uintptr_t>(&seed);
  static std::atomic<unsigned long long> count{0};
  unsigned long long z =
      seed + 0x9E3779B97F4A7C15ull * count.fetch_add(1, std::memory_order_relaxed);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z = (z ^ (z >> 31)) >> 6;
  return z != 0 ? z : 1;
}
// ('T','N') products with k % 4 != 0 and more than three stages stay with the
// other paths, as the path query has always answered.
inline bool fused_considered(const int k) { return k % 4 == 0 || k <= 96; }
// Which kernel runs a call without a path flag, and how K is cut.
struct Route {
  Path path;
  int slices;      // as chosen; what packed operands or the direct kernel make of
                   // them depends on the workspace too (plan_k_slices)
  int spread_tile; // > 0: made by a workgroup each, with tiles of this size
};
inline Route choose_route(const int m, const int n, const int k, const int batch,
                          const int rn, const int policy, const int terms,
                          const bool rows, const bool direct_ok,
                          const void *const workspace,
                          const size_t workspace_bytes) {
  const Choice c = choose_path(m, n, k, batch, rn, terms, policy,
                               rows || fused_considered(k), rows, direct_ok);
  Route r{c.single ? Path::Fused : c.path, c.slices, 0};
  if (single_is_ahead(c, m, n, k, batch, rn, policy, terms, rows, workspace,
                      workspace_bytes))
    r.path = Path::Fused;
  r.spread_tile =
      choose_spread(c, m, n, k, batch, terms, rows, workspace, workspace_bytes);
  if (r.spread_tile > 0)
    r.path = Path::Fused;
  return r;
}

// how the single kernel reads an operand (see its head comment)
inline int fused_source(const long long rs, const long long ks, const int k) {
  if (ks == 1 && k >= 4 && rs < (1 << 24))
    return wmmae_gemm::kFusedKRows;
  if (rs == 1 && ks < (1 << 24))
    return wmmae_gemm::kFusedRRows;
  return wmmae_gemm::kFusedAny;
}

inline bool is_n(const char t) { return t == 'N' || t == 'n'; }
inline bool is_t(const char t) {
  return t == 'T' || t == 't' || t == 'C' || t == 'c';
}

} // namespace

// ===========================================================================
extern "C" {

const char *wmmae_status_string(const int status) {
  switch (status) {
  case WMMAE_STATUS_SUCCESS:
    return "success";
  case WMMAE_STATUS_INVALID_VALUE:
    return "invalid value";
  case WMMAE_STATUS_NULL_POINTER:
    return "null pointer";
  case WMMAE_STATUS_BAD_LEADING_DIM:
    return "leading dimension too small";
  case WMMAE_STATUS_NOT_SUPPORTED:
    return "not supported";
  case WMMAE_STATUS_WORKSPACE_TOO_SMALL:
    return "workspace too small";
  case WMMAE_STATUS_RUNTIME_ERROR:
    return "HIP runtime error";
  case WMMAE_STATUS_MISALIGNED:
    return "buffer not 16-byte aligned";
  default:
    return "unknown status";
  }
}

int wmmae_query(const int what, long long *const out) {
  if (out == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if (what == 0) {
    *out = 100; // 0.1.0
    return WMMAE_STATUS_SUCCESS;
  }
  if (what == 3) {
    *out = 5;
    return WMMAE_STATUS_SUCCESS;
  }
  if (what == 1 || what == 2) {
    int dev = 0;
    hipDeviceProp_t prop;
    WMMAE_HIP_TRY(hipGetDevice(&dev));
    WMMAE_HIP_TRY(hipGetDeviceProperties(&prop, dev));
    *out = what == 1 ? prop.multiProcessorCount : prop.clockRate;
    return WMMAE_STATUS_SUCCESS;
  }
  return WMMAE_STATUS_INVALID_VALUE;
}

// ------------------------------------------------------------- pack / gemm
int wmmae_tcec_pack_bytes(const int rows, const int k, const int batch,
                          const int policy, size_t *const bytes) {
  PolicyInfo p;
  if (bytes == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if (!policy_info(policy, p) || rows < 0 || k < 0 || batch < 0)
    return WMMAE_STATUS_INVALID_VALUE;
  *bytes = static_cast<size_t>(packed_elems(rows, k, p.terms)) * 16u *
           static_cast<size_t>(batch);
  return WMMAE_STATUS_SUCCESS;
}

} // extern "C"

namespace {
// Shared implementations; X / C may be given as a base pointer with a batch
// stride or as a device array of per-matrix pointers.
// Argument checks of one operand of a split; WMMAE_STATUS_SUCCESS with
// `nothing` set when there is nothing to write.
int pack_check(const int policy, const int rows, const int k,
               const float *const X, const float *const *const ptrs,
               const long long row_stride, const long long k_stride,
               const int batch, void *const packed, const size_t packed_bytes,
               bool &nothing) {
  PolicyInfo p;
  nothing = false;
  if (!policy_info(policy, p) || rows < 0 || k < 0 || batch < 0)
    return WMMAE_STATUS_INVALID_VALUE;
  if (rows == 0 || k == 0 || batch == 0) {
    nothing = true;
    return WMMAE_STATUS_SUCCESS;
  }
  if ((X == nullptr && ptrs == nullptr) || packed == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if (row_stride < 1 || k_stride < 1 || (row_stride != 1 && k_stride != 1))
    return WMMAE_STATUS_BAD_LEADING_DIM;
  if (reinterpret_cast<uintptr_t>(packed) % 16 != 0)
    return WMMAE_STATUS_MISALIGNED;
  size_t need = 0;
  wmmae_tcec_pack_bytes(rows, k, batch, policy, &need);
  if (packed_bytes < need)
    return WMMAE_STATUS_WORKSPACE_TOO_SMALL;
  return WMMAE_STATUS_SUCCESS;
}

int pack_impl(const int policy, const int rows, const int k,
              const float *const X, const float *const *const ptrs,
              const long long row_stride, const long long k_stride,
              const long long batch_stride, const int batch, void *const packed,
              const size_t packed_bytes, void *const stream) {
  bool nothing = false;
  const int st = pack_check(policy, rows, k, X, ptrs, row_stride, k_stride,
                            batch, packed, packed_bytes, nothing);
  if (st != WMMAE_STATUS_SUCCESS || nothing)
    return st;
  const PackSource src{rows, X, ptrs, row_stride, k_stride, batch_stride, packed};
  return policy_kernels(policy)->pack(k, batch, src, nullptr,
                                      static_cast<hipStream_t>(stream));
}

// split-K, or K slices for a partly empty last round, only when the caller
// supplied room for the slices
void plan_k_slices(GemmArgs &g, void *const workspace,
                   const size_t workspace_bytes) {
  g.splits = choose_splits(g.terms, g.m, g.n, g.k, g.batch, g.is_direct);
  g.partial = nullptr;
  g.tail_ws = nullptr;
  g.tail_ws_bytes = 0;
  const bool ws_usable =
      workspace != nullptr && reinterpret_cast<uintptr_t>(workspace) % 16 == 0;
  if (g.splits > 1 && ws_usable &&
      workspace_bytes >=
          static_cast<size_t>(g.splits) * g.batch * g.m * g.n * 4u) {
    g.partial = static_cast<float *>(workspace);
  } else {
    g.splits = 1;
    if (ws_usable) {
      g.tail_ws = static_cast<float *>(workspace);
      g.tail_ws_bytes = workspace_bytes;
    }
  }
}

int gemm_packed_impl(const int policy, const int m, const int n, const int k,
                     const float *const alpha, const void *const packed_a,
                     const void *const packed_b, const float *const beta,
                     float *const C, float *const *const c_ptrs, const int ldc,
                     const long long stride_c, const int batch, const int flags,
                     void *const workspace, const size_t workspace_bytes,
                     void *const stream) {
  PolicyInfo p;
  if (!policy_info(policy, p) || m < 0 || n < 0 || k < 0 || batch < 0 ||
      (flags & ~WMMAE_FLAG_RN_MAIN) != 0)
    return WMMAE_STATUS_INVALID_VALUE;
  if (alpha == nullptr || beta == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if (m == 0 || n == 0 || batch == 0)
    return WMMAE_STATUS_SUCCESS;
  if ((C == nullptr && c_ptrs == nullptr) ||
      (k > 0 && (packed_a == nullptr || packed_b == nullptr)))
    return WMMAE_STATUS_NULL_POINTER;
  if (ldc < m)
    return WMMAE_STATUS_BAD_LEADING_DIM;
  if (k > 0 && (reinterpret_cast<uintptr_t>(packed_a) % 16 != 0 ||
                reinterpret_cast<uintptr_t>(packed_b) % 16 != 0))
    return WMMAE_STATUS_MISALIGNED;
  if (k == 0) {
    const long long blocks = ceil_div(static_cast<long long>(m) * n, 256);
    if (blocks > 0x7fffffffLL)
      return WMMAE_STATUS_NOT_SUPPORTED;
    for (int e0 = 0; e0 < batch; e0 += kMaxGridY)
      hipLaunchKernelGGL(scale_c_kernel,
                         dim3(static_cast<unsigned>(blocks),
                              std::min(batch - e0, kMaxGridY)),
                         dim3(256), 0, static_cast<hipStream_t>(stream), C, m, n,
                         static_cast<long long>(ldc), stride_c, c_ptrs, *beta,
                         static_cast<unsigned>(e0));
    return launch_status();
  }
  const OneDeviceCall one_device;
  GemmArgs g;
  g.a = static_cast<const u32x4 *>(packed_a);
  g.b = static_cast<const u32x4 *>(packed_b);
  g.c = C;
  g.c_ptrs = c_ptrs;
  g.m = m;
  g.n = n;
  g.k = k;
  g.ldc = ldc;
  g.stride_c = stride_c;
  g.alpha = *alpha;
  g.beta = *beta;
  g.inv_scale = p.inv_scale;
  g.batch = batch;
  g.terms = p.terms;
  g.stream = static_cast<hipStream_t>(stream);
  plan_k_slices(g, workspace, workspace_bytes);
  const PolicyKernels *const kernels = policy_kernels(policy);
  if ((flags & WMMAE_FLAG_RN_MAIN) == 0)
    return kernels->gemm(g);
  return kernels->gemm_rn != nullptr ? kernels->gemm_rn(g)
                                     : WMMAE_STATUS_NOT_SUPPORTED;
}

int sgemm_impl(const char transa, const char transb, const int m, const int n,
               const int k, const float *const alpha, const float *const A,
               const float *const *const a_ptrs, const int lda,
               const long long stride_a, const float *const B,
               const float *const *const b_ptrs, const int ldb,
               const long long stride_b, const float *const beta,
               float *const C, float *const *const c_ptrs, const int ldc,
               const long long stride_c, const int batch, const int policy,
               const int flags, void *workspace, const size_t workspace_bytes,
               void *const stream) {
  PolicyInfo p;
  if ((!is_n(transa) && !is_t(transa)) || (!is_n(transb) && !is_t(transb)) ||
      m < 0 || n < 0 || k < 0 || batch < 0 || !policy_info(policy, p) ||
      (flags & ~kAllFlags) != 0 || !one_path_at_most(flags))
    return WMMAE_STATUS_INVALID_VALUE;
  if (alpha == nullptr || beta == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if (m == 0 || n == 0 || batch == 0)
    return WMMAE_STATUS_SUCCESS;
  if ((C == nullptr && c_ptrs == nullptr) ||
      (k > 0 && ((A == nullptr && a_ptrs == nullptr) ||
                 (B == nullptr && b_ptrs == nullptr))))
    return WMMAE_STATUS_NULL_POINTER;
  const OneDeviceCall one_device;
  const int a_rows = is_n(transa) ? m : k; // rows of A as stored (column major)
  const int b_rows = is_n(transb) ? k : n;
  if (lda < (a_rows > 1 ? a_rows : 1) || ldb < (b_rows > 1 ? b_rows : 1) ||
      ldc < m)
    return WMMAE_STATUS_BAD_LEADING_DIM;

  const long long a_rs = is_n(transa) ? 1 : lda, a_ks = is_n(transa) ? lda : 1;
  const long long b_rs = is_n(transb) ? ldb : 1, b_ks = is_n(transb) ? 1 : ldb;
  const bool rows = a_ks != 1 || b_ks != 1;
  const bool direct_ok = a_ks == 1 && b_ks == 1 &&
                         direct_possible(k, p.terms, flags, a_rs, b_rs);
  const int rn = flags & WMMAE_FLAG_RN_MAIN;
  Path path = Path::Packed;
  int slices = 1; // of the single kernel; a forced one does not cut K
  int spread_tile = 0;
  if ((flags & WMMAE_FLAG_PATH_DIRECT) != 0) {
    if (!direct_ok)
      return WMMAE_STATUS_NOT_SUPPORTED;
    path = Path::Direct;
  } else if ((flags & WMMAE_FLAG_PATH_FUSED) != 0) {
    if (k <= 0 || (rn != 0 && policy != WMMAE_POLICY_F16_EC &&
                   policy != WMMAE_POLICY_BF16X3_EC))
      return WMMAE_STATUS_NOT_SUPPORTED;
    path = Path::Fused;
  } else if ((flags & WMMAE_FLAG_PATH_PACKED) == 0) {
    const Route r = choose_route(m, n, k, batch, rn, policy, p.terms, rows,
                                 direct_ok, workspace, workspace_bytes);
    path = r.path;
    slices = r.slices;
    spread_tile = r.spread_tile;
  }
  if (path == Path::Direct) {
    // the planes of the K slices are the only workspace this path uses
    size_t bytes_c = 0;
    wmmae_tcec_gemm_packed_workspace_bytes(policy, m, n, k, batch, &bytes_c);
    hipStream_t s = static_cast<hipStream_t>(stream);
    void *ws = workspace;
    size_t ws_bytes = workspace_bytes;
    bool own = false;
    // (a caller's workspace that is not 16-byte aligned is left alone by
    // plan_k_slices: this path can do without, as the single kernel does)
    if (ws == nullptr && bytes_c > 0) {
      WMMAE_HIP_TRY(hipMallocAsync(&ws, bytes_c, s));
      ws_bytes = bytes_c;
      own = true;
    }
    GemmArgs g;
    g.a = nullptr;
    g.b = nullptr;
    g.c = C;
    g.c_ptrs = c_ptrs;
    g.m = m;
    g.n = n;
    g.k = k;
    g.ldc = ldc;
    g.stride_c = stride_c;
    g.alpha = *alpha;
    g.beta = *beta;
    g.inv_scale = p.inv_scale;
    g.batch = batch;
    g.terms = p.terms;
    g.stream = s;
    g.is_direct = true;
    g.direct = wmmae_gemm::DirectSource{A,    B,    a_ptrs,   b_ptrs,
                                        a_rs, b_rs, stride_a, stride_b, 0, k};
    plan_k_slices(g, ws, ws_bytes);
    // staggered start for launches bound by their bytes (see the kernel)
    const DirectTimes dt =
        direct_times(m, n, k, batch, fit::kDirectStagger[p.terms - 1]);
    if (g.splits <= 1 && batch >= 8 && dt.bytes > dt.tiles)
      g.direct.stagger = 1;
    int st = policy_kernels(policy)->gemm(g);
    if (own && hipFreeAsync(ws, s) != hipSuccess && st == WMMAE_STATUS_SUCCESS)
      st = WMMAE_STATUS_RUNTIME_ERROR;
    return st;
  }
  if (path == Path::Fused) {
    if (batch > (1 << 26)) // tile indices are 32-bit
      return WMMAE_STATUS_NOT_SUPPORTED;
    FusedArgs f;
    wmmae_gemm::FusedSpreadParams &q = f.p;
    q.A = A;
    q.a_ptrs = a_ptrs;
    q.a_rs = a_rs;
    q.a_ks = a_ks;
    q.a_bs = stride_a;
    q.B = B;
    q.b_ptrs = b_ptrs;
    q.b_rs = b_rs;
    q.b_ks = b_ks;
    q.b_bs = stride_b;
    q.C = C;
    q.c_ptrs = c_ptrs;
    q.ldc = ldc;
    q.c_bs = stride_c;
    q.M = m;
    q.N = n;
    q.K = k;
    q.batch = batch;
    q.a_source = fused_source(a_rs, a_ks, k);
    q.b_source = fused_source(b_rs, b_ks, k);
    q.slice_stages =
        slices > 1 ? static_cast<int>(ceil_div(packed_k_tiles(k), slices)) : 0;
    q.alpha = *alpha;
    q.beta = *beta;
    q.inv_scale = p.inv_scale;
    f.stream = static_cast<hipStream_t>(stream);
    const PolicyKernels *const kernels = policy_kernels(policy);
    if (spread_tile == 0)
      return rn != 0 ? kernels->fused_rn(f) : kernels->fused(f);
    // the slices' sums and the tiles' arrival words in the caller's workspace or
    // in one allocated here
    const bool own = workspace == nullptr;
    if (own)
      WMMAE_HIP_TRY(hipMallocAsync(
          &workspace, fused_spread_bytes(m, n, batch, slices, spread_tile),
          f.stream));
    f.spread_tile = spread_tile;
    q.slices = slices;
    q.planes = static_cast<float *>(workspace);
    q.arrivals = reinterpret_cast<unsigned long long *>(
        static_cast<char *>(workspace) +
        fused_spread_planes(m, n, batch, slices, spread_tile));
    q.launch = launch_number();
    int st = rn != 0 ? kernels->fused_rn(f) : kernels->fused(f);
    if (own && hipFreeAsync(workspace, f.stream) != hipSuccess &&
        st == WMMAE_STATUS_SUCCESS)
      st = WMMAE_STATUS_RUNTIME_ERROR;
    return st;
  }

  size_t bytes_a = 0, bytes_b = 0, bytes_c = 0;
  wmmae_tcec_pack_bytes(m, k, batch, policy, &bytes_a);
  wmmae_tcec_pack_bytes(n, k, batch, policy, &bytes_b);
  wmmae_tcec_gemm_packed_workspace_bytes(policy, m, n, k, batch, &bytes_c);
  hipStream_t s = static_cast<hipStream_t>(stream);
  bool own = false;
  if (workspace == nullptr) {
    if (bytes_a + bytes_b + bytes_c > 0) {
      WMMAE_HIP_TRY(hipMallocAsync(&workspace, bytes_a + bytes_b + bytes_c, s));
      own = true;
    }
  } else {
    if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
      return WMMAE_STATUS_MISALIGNED;
    // the packed operands are required; the split-K slices are optional
    if (workspace_bytes < bytes_a + bytes_b)
      return WMMAE_STATUS_WORKSPACE_TOO_SMALL;
    if (workspace_bytes < bytes_a + bytes_b + bytes_c)
      bytes_c = 0;
  }
  void *const pa = workspace;
  void *const pb = static_cast<char *>(workspace) + bytes_a;
  void *const pc =
      bytes_c > 0 ? static_cast<char *>(workspace) + bytes_a + bytes_b : nullptr;

  int st = WMMAE_STATUS_SUCCESS;
  if (k > 0) {
    // op(A)(i,l): 'N' -> A[i + l*lda], 'T' -> A[l + i*lda]
    const PackSource sa{m, A, a_ptrs, is_n(transa) ? 1 : lda,
                        is_n(transa) ? lda : 1, stride_a, pa};
    // op(B)(l,j): 'N' -> B[l + j*ldb], 'T' -> B[j + l*ldb]; packed rows = j
    const PackSource sb{n, B, b_ptrs, is_n(transb) ? ldb : 1,
                        is_n(transb) ? 1 : ldb, stride_b, pb};
    bool none_a = false, none_b = false;
    st = pack_check(policy, sa.rows, k, sa.X, sa.ptrs, sa.row_stride,
                    sa.k_stride, batch, pa, bytes_a, none_a);
    if (st == WMMAE_STATUS_SUCCESS)
      st = pack_check(policy, sb.rows, k, sb.X, sb.ptrs, sb.row_stride,
                      sb.k_stride, batch, pb, bytes_b, none_b);
    // (m, n, k and batch are all positive here: both operands have work)
    if (st == WMMAE_STATUS_SUCCESS && !none_a && !none_b)
      st = policy_kernels(policy)->pack(k, batch, sa, &sb, s); // one launch
  }
  if (st == WMMAE_STATUS_SUCCESS)
    st = gemm_packed_impl(policy, m, n, k, alpha, pa, pb, beta, C, c_ptrs, ldc,
                          stride_c, batch, flags & WMMAE_FLAG_RN_MAIN, pc, bytes_c,
                          stream);
  if (own) {
    if (hipFreeAsync(workspace, s) != hipSuccess &&
        st == WMMAE_STATUS_SUCCESS)
      st = WMMAE_STATUS_RUNTIME_ERROR;
  }
  return st;
}
} // namespace

extern "C" {

int wmmae_tcec_pack(const int policy, const int rows, const int k,
                    const float *const X, const long long row_stride,
                    const long long k_stride, const long long batch_stride,
                    const int batch, void *const packed,
                    const size_t packed_bytes, void *const stream) {
  return pack_impl(policy, rows, k, X, nullptr, row_stride, k_stride,
                   batch_stride, batch, packed, packed_bytes, stream);
}

int wmmae_tcec_gemm_packed(const int policy, const int m, const int n,
                           const int k, const float *const alpha,
                           const void *const packed_a,
                           const void *const packed_b, const float *const beta,
                           float *const C, const int ldc,
                           const long long stride_c, const int batch,
                           const int flags, void *const workspace,
                           const size_t workspace_bytes, void *const stream) {
  return gemm_packed_impl(policy, m, n, k, alpha, packed_a, packed_b, beta, C,
                          nullptr, ldc, stride_c, batch, flags, workspace,
                          workspace_bytes, stream);
}

int wmmae_tcec_gemm_packed_workspace_bytes(const int policy, const int m,
                                           const int n, const int k,
                                           const int batch,
                                           size_t *const bytes) {
  PolicyInfo p;
  if (bytes == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if (!policy_info(policy, p) || m < 0 || n < 0 || k < 0 || batch < 0)
    return WMMAE_STATUS_INVALID_VALUE;
  *bytes = slices_room(p.terms, m, n, k, batch);
  if (*bytes == 0)
    *bytes = tail_room(policy, m, n, k, batch);
  return WMMAE_STATUS_SUCCESS;
}

int wmmae_tcec_sgemm_path(const int m, const int n, const int k,
                          const int batch, const int policy, const int flags,
                          int *const path) {
  PolicyInfo p;
  if (path == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if (m < 0 || n < 0 || k < 0 || batch < 0 || !policy_info(policy, p) ||
      (flags & ~WMMAE_FLAG_RN_MAIN) != 0)
    return WMMAE_STATUS_INVALID_VALUE;
  const Choice c = choose_path(m, n, k, batch, flags, p.terms, policy,
                               fused_considered(k), false,
                               direct_possible(k, p.terms, flags, 1, 1));
  *path = c.path == Path::Fused    ? 0
          : c.path == Path::Direct ? (c.slices > 1 ? 4 : 3)
                                   : (c.slices > 1 ? 2 : 1);
  return WMMAE_STATUS_SUCCESS;
}

int wmmae_tcec_sgemm_route(const char transa, const char transb, const int m,
                           const int n, const int k, const int lda,
                           const int ldb, const int batch, const int policy,
                           const int flags, const void *const workspace,
                           const size_t workspace_bytes, int *const route) {
  PolicyInfo p;
  if (route == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if ((!is_n(transa) && !is_t(transa)) || (!is_n(transb) && !is_t(transb)) ||
      m <= 0 || n <= 0 || k <= 0 || batch <= 0 || !policy_info(policy, p) ||
      (flags & ~WMMAE_FLAG_RN_MAIN) != 0)
    return WMMAE_STATUS_INVALID_VALUE;
  const OneDeviceCall one_device;
  const bool rows = is_n(transa) || !is_n(transb);
  const Route r = choose_route(
      m, n, k, batch, flags, policy, p.terms, rows,
      !rows && direct_possible(k, p.terms, flags, lda, ldb), workspace,
      workspace_bytes);
  // (the slices those two make where the workspace holds their sums)
  bool cut = true;
  if (workspace != nullptr && r.path != Path::Fused) {
    const size_t sums =
        r.path == Path::Packed
            ? slices_room(p.terms, m, n, k, batch)
            : static_cast<size_t>(r.slices) * batch * m * n * 4u;
    cut = reinterpret_cast<uintptr_t>(workspace) % 16 == 0 &&
          (r.path == Path::Packed
               ? holds_packed(m, n, k, batch, p.terms, workspace_bytes, sums)
               : workspace_bytes >= sums);
  }
  route[0] = r.path == Path::Fused ? 0 : r.path == Path::Packed ? 1 : 3;
  route[1] = cut ? r.slices : 1;
  route[2] = r.spread_tile;
  return WMMAE_STATUS_SUCCESS;
}

int wmmae_tcec_path_estimates(const int m, const int n, const int k,
                              const int batch, const int policy,
                              double *const seconds) {
  PolicyInfo p;
  if (seconds == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if (m <= 0 || n <= 0 || k <= 0 || batch <= 0 || !policy_info(policy, p))
    return WMMAE_STATUS_INVALID_VALUE;
  const PathEstimates e = estimate_paths(m, n, k, batch, p.terms,
                                         fused_considered(k), false,
                                         direct_possible(k, p.terms, 0, 1, 1));
  // (cut products: see the header)
  seconds[0] = e.slices == 1 || std::isinf(e.fused)
                   ? e.fused
                   : std::max(fused_time(p.terms, m, n, k, batch, true, false),
                              1.01 * e.base_time);
  seconds[1] = e.packed;
  seconds[2] = e.direct;
  return WMMAE_STATUS_SUCCESS;
}

int wmmae_tcec_time_gemm_kernel(void *const begin_event,
                                void *const end_event) {
  if ((begin_event == nullptr) != (end_event == nullptr))
    return WMMAE_STATUS_NULL_POINTER;
  t_gemm_begin = static_cast<hipEvent_t>(begin_event);
  t_gemm_end = static_cast<hipEvent_t>(end_event);
  return WMMAE_STATUS_SUCCESS;
}

int wmmae_tcec_force_k_slices(const int slices) {
  if (slices < 0)
    return WMMAE_STATUS_INVALID_VALUE;
  t_forced_k_slices = slices;
  return WMMAE_STATUS_SUCCESS;
}

int wmmae_tcec_force_spread_tile(const int tile) {
  if (tile != -1 && tile != 0 && tile != 64 && tile != 128)
    return WMMAE_STATUS_INVALID_VALUE;
  t_forced_spread_tile = tile;
  return WMMAE_STATUS_SUCCESS;
}

int wmmae_tcec_sgemm_k_slices(const int m, const int n, const int k,
                              const int batch, const int policy,
                              const int flags, int *const slices) {
  PolicyInfo p;
  if (slices == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  constexpr int kPathFlags = WMMAE_FLAG_PATH_PACKED | WMMAE_FLAG_PATH_FUSED |
                             WMMAE_FLAG_PATH_DIRECT;
  if (m < 0 || n < 0 || k < 0 || batch < 0 || !policy_info(policy, p) ||
      (flags & ~(WMMAE_FLAG_RN_MAIN | kPathFlags)) != 0)
    return WMMAE_STATUS_INVALID_VALUE;
  *slices = 1;
  if (m == 0 || n == 0 || k == 0 || batch == 0)
    return WMMAE_STATUS_SUCCESS;
  const bool direct_ok = direct_possible(k, p.terms, flags, 1, 1);
  if ((flags & WMMAE_FLAG_PATH_DIRECT) != 0) {
    if (!direct_ok)
      return WMMAE_STATUS_NOT_SUPPORTED;
    *slices = choose_splits(p.terms, m, n, k, batch, true);
  } else if ((flags & WMMAE_FLAG_PATH_PACKED) != 0) {
    *slices = choose_splits(p.terms, m, n, k, batch);
  } else if ((flags & WMMAE_FLAG_PATH_FUSED) == 0) {
    *slices = choose_path(m, n, k, batch, flags & WMMAE_FLAG_RN_MAIN, p.terms,
                          policy, fused_considered(k), false, direct_ok)
                  .slices;
  }
  return WMMAE_STATUS_SUCCESS;
}

int wmmae_tcec_sgemm_workspace_bytes(const int m, const int n, const int k,
                                     const int batch, const int policy,
                                     size_t *const bytes) {
  size_t a = 0, b = 0, c = 0;
  if (bytes == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if (m < 0 || n < 0)
    return WMMAE_STATUS_INVALID_VALUE;
  int s = wmmae_tcec_pack_bytes(m, k, batch, policy, &a);
  if (s != WMMAE_STATUS_SUCCESS)
    return s;
  s = wmmae_tcec_pack_bytes(n, k, batch, policy, &b);
  if (s != WMMAE_STATUS_SUCCESS)
    return s;
  s = wmmae_tcec_gemm_packed_workspace_bytes(policy, m, n, k, batch, &c);
  if (s != WMMAE_STATUS_SUCCESS)
    return s;
  *bytes = a + b + c;
  return WMMAE_STATUS_SUCCESS;
}

int wmmae_tcec_sgemm_strided_batched(
    const char transa, const char transb, const int m, const int n, const int k,
    const float *const alpha, const float *const A, const int lda,
    const long long stride_a, const float *const B, const int ldb,
    const long long stride_b, const float *const beta, float *const C,
    const int ldc, const long long stride_c, const int batch, const int policy,
    const int flags, void *const workspace, const size_t workspace_bytes,
    void *const stream) {
  return sgemm_impl(transa, transb, m, n, k, alpha, A, nullptr, lda, stride_a,
                    B, nullptr, ldb, stride_b, beta, C, nullptr, ldc, stride_c,
                    batch, policy, flags, workspace, workspace_bytes, stream);
}

int wmmae_tcec_sgemm_batched(const char transa, const char transb, const int m,
                             const int n, const int k, const float *const alpha,
                             const float *const *const A_array, const int lda,
                             const float *const *const B_array, const int ldb,
                             const float *const beta,
                             float *const *const C_array, const int ldc,
                             const int batch, const int policy, const int flags,
                             void *const workspace,
                             const size_t workspace_bytes,
                             void *const stream) {
  return sgemm_impl(transa, transb, m, n, k, alpha, nullptr, A_array, lda, 0,
                    nullptr, B_array, ldb, 0, beta, nullptr, C_array, ldc, 0,
                    batch, policy, flags, workspace, workspace_bytes, stream);
}

int wmmae_direct_read_first(const int tail, const int k, const int stage,
                            const int lane, long long *const first) {
  if (first == nullptr)
    return WMMAE_STATUS_NULL_POINTER;
  if (k < 4 || stage < 0 || stage >= ceil_div(k, 32) || lane < 0 || lane > 63 ||
      (tail == 0 && k % 32 != 0))
    return WMMAE_STATUS_INVALID_VALUE;
  *first = wmmae_gemm::direct_read_first(tail != 0, k, stage,
                                         static_cast<unsigned>(lane));
  return WMMAE_STATUS_SUCCESS;
}

// ---------------------------------------------- entry point that allocates
// nothing: the workspace is a device array that is part of the library image.
// Each GPU holds its own copy at its own address; in host code the array's
// name is only a handle for hipGetSymbolAddress, never a device address.
} // extern "C"

namespace {
constexpr size_t kStaticScratchBytes = WMMAE_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

// Device address of `scratch` on the current device, looked up once per
// device (with that device current) and kept.
int static_scratch(void **const out) {
  static std::atomic<void *> ptrs[64];
  int dev = 0;
  WMMAE_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64)
    return WMMAE_STATUS_NOT_SUPPORTED;
  void *p = ptrs[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    WMMAE_HIP_TRY(
        hipGetSymbolAddress(reinterpret_cast<void **>(&p), HIP_SYMBOL(scratch)));
    if (p == nullptr)
      return WMMAE_STATUS_RUNTIME_ERROR;
    ptrs[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return WMMAE_STATUS_SUCCESS;
}
} // namespace

extern "C" {

int wmmae_tcec_sgemm_static(const char transa, const char transb, const int m,
                            const int n, const int k, const float *const alpha,
                            const float *const A, const int lda,
                            const float *const B, const int ldb,
                            const float *const beta, float *const C,
                            const int ldc, const int policy, const int flags,
                            void *const stream) {
  void *ws = nullptr;
  const int st = static_scratch(&ws);
  if (st != WMMAE_STATUS_SUCCESS)
    return st;
  // sgemm_impl allocates only when it is handed no workspace; with one it
  // returns WMMAE_STATUS_WORKSPACE_TOO_SMALL when the split operands do not
  // fit, and makes K slices only if they fit as well
  return sgemm_impl(transa, transb, m, n, k, alpha, A, nullptr, lda, 0, B,
                    nullptr, ldb, 0, beta, C, nullptr, ldc, 0, 1, policy, flags,
                    ws, kStaticScratchBytes, stream);
}

int wmmae_tcec_sgemm(const char transa, const char transb, const int m,
                     const int n, const int k, const float *const alpha,
                     const float *const A, const int lda, const float *const B,
                     const int ldb, const float *const beta, float *const C,
                     const int ldc, const int policy, const int flags,
                     void *const workspace, const size_t workspace_bytes,
                     void *const stream) {
  return sgemm_impl(transa, transb, m, n, k, alpha, A, nullptr, lda, 0, B,
                    nullptr, ldb, 0, beta, C, nullptr, ldc, 0, 1, policy, flags,
                    workspace, workspace_bytes, stream);
}

} // extern "C"
