// Launches of the GEMM driver's kernels for one policy; instantiated by the
// gemm_*.hip translation units.
#pragma once
#include "gemm_plan.hpp"

namespace wmmae_driver {

// Splits one operand (b == nullptr) or both operands of a product in a single
// launch.
template <class T, int TERMS>
int launch_pack(const int k, const int batch, const PackSource &a,
                const PackSource *const b, hipStream_t stream) {
  const int KT = packed_k_tiles(k);
  const wmmae_gemm::PackOperand oa = pack_operand(a, KT);
  const long long blocks_a = ceil_div(oa.chunks * 64, 256);
  if (b == nullptr) {
    if (blocks_a > 0x7fffffffLL)
      return WMMAE_STATUS_NOT_SUPPORTED;
    for (int e0 = 0; e0 < batch; e0 += kMaxGridY)
      hipLaunchKernelGGL((wmmae_gemm::split_pack_kernel<T, TERMS>),
                         dim3(static_cast<unsigned>(blocks_a),
                              std::min(batch - e0, kMaxGridY)),
                         dim3(256), 0, stream, oa, k, KT,
                         static_cast<unsigned>(e0));
    return launch_status();
  }
  const wmmae_gemm::PackOperand ob = pack_operand(*b, KT);
  const long long blocks_b = ceil_div(ob.chunks * 64, 256);
  if (blocks_a + blocks_b > 0x7fffffffLL)
    return WMMAE_STATUS_NOT_SUPPORTED;
  for (int e0 = 0; e0 < batch; e0 += kMaxGridY)
    hipLaunchKernelGGL((wmmae_gemm::split_pack_pair_kernel<T, TERMS>),
                       dim3(static_cast<unsigned>(blocks_a + blocks_b),
                            std::min(batch - e0, kMaxGridY)),
                       dim3(256), 0, stream, oa, ob,
                       static_cast<unsigned>(blocks_a), k, KT,
                       static_cast<unsigned>(e0));
  return launch_status();
}

// Workgroups of one GEMM kernel that a compute unit holds at a time: what the
// runtime's occupancy query says (registers, LDS and wave slots together),
// looked up once per kernel and device; the LDS bound alone where the query
// gives nothing (no device visible).  The persistent work-item modes give
// every resident workgroup a fixed share of the items, so a count the
// registers do not allow would leave the extra workgroups' shares to run after
// everything else (the one-term direct kernel: 48 KiB of LDS, three by that
// bound, but 512 registers a lane).
template <class MT, int TERMS, int BM, int BN, int WGM, int WGN, bool RN,
          int DIRECT = 0>
int workgroups_per_cu() {
  constexpr int NSTAGE = DIRECT ? 2 : ring_depth(BM, BN, TERMS);
  using Cfg =
      wmmae_gemm::GemmConfig<MT, TERMS, BM, BN, WGM, WGN, NSTAGE, RN, DIRECT>;
  constexpr int by_lds =
      (160 * 1024) / Cfg::LDS_BYTES > 4 ? 4 : (160 * 1024) / Cfg::LDS_BYTES;
  static std::atomic<int> cached[64];
  static std::atomic<unsigned long long> lds_allowed{0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();
    return by_lds;
  }
  const int c = cached[dev].load(std::memory_order_relaxed);
  if (c > 0)
    return c;
  auto kernel = wmmae_gemm::tcec_gemm_kernel<MT, TERMS, BM, BN, WGM, WGN,
                                             NSTAGE, RN, DIRECT>;
  int n = 0;
  if (allow_dynamic_lds(reinterpret_cast<const void *>(kernel), Cfg::LDS_BYTES,
                        lds_allowed) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &n, reinterpret_cast<const void *>(kernel), Cfg::NTHREADS,
          Cfg::LDS_BYTES) != hipSuccess ||
      n <= 0) {
    (void)hipGetLastError();
    return by_lds;
  }
  n = n < by_lds ? n : by_lds;
  cached[dev].store(n, std::memory_order_relaxed);
  return n;
}

template <class MT, int TERMS, int BM, int BN, int WGM, int WGN, bool RN,
          int DIRECT = 0>
int launch_gemm(const GemmArgs &g) {
  constexpr int NSTAGE = DIRECT ? 2 : ring_depth(BM, BN, TERMS);
  using Cfg =
      wmmae_gemm::GemmConfig<MT, TERMS, BM, BN, WGM, WGN, NSTAGE, RN, DIRECT>;
  auto kernel = wmmae_gemm::tcec_gemm_kernel<MT, TERMS, BM, BN, WGM, WGN,
                                             NSTAGE, RN, DIRECT>;
  static std::atomic<unsigned long long> lds_allowed{0};
  WMMAE_HIP_TRY(allow_dynamic_lds(reinterpret_cast<const void *>(kernel),
                                  Cfg::LDS_BYTES, lds_allowed));
  const int tiles_m = static_cast<int>(ceil_div(g.m, BM));
  const int tiles_n = static_cast<int>(ceil_div(g.n, BN));
  const int KT = packed_k_tiles(g.k);
  const int rb_a = static_cast<int>(packed_row_blocks(g.m));
  const int rb_b = static_cast<int>(packed_row_blocks(g.n));
  const int splits = g.partial != nullptr ? g.splits : 1;
  const int split_stages = static_cast<int>(ceil_div(KT, splits));
  const int zdim = static_cast<int>(ceil_div(KT, split_stages));
  const long long items =
      static_cast<long long>(tiles_m) * tiles_n * g.batch * zdim;
  if (items >= (1ll << 31)) // the kernel counts items in 32 bits
    return WMMAE_STATUS_INVALID_VALUE;
  // Who takes which item (the large tiles take most of a compute unit's LDS,
  // so one workgroup per unit is resident):
  //  * 8 or more batch entries: an XCD owns whole entries, so that an entry's
  //    operands are read into one L2 only (batch 256 of 1024x1024x256:
  //    196 -> 256 effective TFLOPS), persistent workgroups when there are
  //    more items than resident workgroups;
  // and with more items than resident workgroups otherwise
  //  * short K loops: persistent workgroups walking one shared list, their
  //    requests running ahead into the next item;
  //  * long K loops (64 stages = 2048 of k or more per item) of few entries:
  //    one workgroup per item, handed out by the hardware as compute units
  //    become free, which evens out compute units of unequal speed over many
  //    rounds (a fixed share per workgroup measured 7 % slower at 16384^3).
  const int per_cu =
      workgroups_per_cu<MT, TERMS, BM, BN, WGM, WGN, RN, DIRECT>();
  const long long resident = static_cast<long long>(device_cus()) * per_cu;
  int grid = static_cast<int>(std::min(items, resident));
  int entry_per_xcd = 0;
  const bool eight_xcds = device_xcds() == kKernelXcds;
  if (zdim > 1 && eight_xcds && resident >= 8 && resident % 8 == 0) {
    // split-K: eight runs of the item list, one per XCD, so that an XCD holds
    // as few K slices as possible; the grid is padded to whole runs
    entry_per_xcd = 2;
    grid = static_cast<int>(std::min(8 * ceil_div(items, 8), resident));
  }
  unsigned tail_begin = 0xffffffffu; // no tail slices
  TailPlan tail;
  // (an XCD that owns one entry more than the others must not cost more
  // rounds than the shared list would take: 9 entries of 128 tiles are 8
  // rounds on the XCD with two entries, 5 on the shared list)
  const bool by_xcd = eight_xcds && resident >= 8 && resident % 8 == 0;
  const long long owned_rounds =
      by_xcd ? ceil_div(static_cast<long long>(tiles_m) * tiles_n *
                            ceil_div(g.batch, 8),
                        resident / 8)
             : 0;
  if (zdim == 1 && g.batch >= 8 && by_xcd &&
      owned_rounds * 100 <= ceil_div(items, resident) * 115) {
    // also when every item gets a workgroup of its own: a workgroup for every
    // item of the XCD that owns the most entries
    entry_per_xcd = 1;
    grid = static_cast<int>(std::min(
        8ll * tiles_m * tiles_n * ceil_div(g.batch, 8), resident));
  } else if (items > resident && entry_per_xcd == 0) {
    if (split_stages >= 64) {
      grid = static_cast<int>(items);
      // one entry, no split-K, room for the slices: the tiles of a partly
      // empty last round are cut along K
      if (g.batch == 1 && zdim == 1 && g.c_ptrs == nullptr &&
          g.tail_ws != nullptr) {
        tail = plan_tail(items, resident, KT);
        const size_t need =
            static_cast<size_t>(tail.slices) * tail.tail * BM * BN * 4u;
        if (tail.slices >= 2 && need <= g.tail_ws_bytes) {
          tail_begin = static_cast<unsigned>(tail.full);
          grid = static_cast<int>(tail.full + tail.tail * tail.slices);
        } else {
          tail.slices = 1;
        }
      }
    }
  }
  if (t_gemm_begin != nullptr)
    WMMAE_HIP_TRY(hipEventRecord(t_gemm_begin, g.stream));
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(Cfg::NTHREADS), Cfg::LDS_BYTES,
                     g.stream, g.a, g.b,
                     g.c, g.m, g.n, KT, rb_a, rb_b, g.ldc, g.alpha, g.beta,
                     g.inv_scale, tiles_m, tiles_n,
                     static_cast<long long>(rb_a) * KT * TERMS * 64,
                     static_cast<long long>(rb_b) * KT * TERMS * 64,
                     g.stride_c, split_stages,
                     zdim > 1 ? g.partial : static_cast<float *>(nullptr),
                     g.c_ptrs, g.batch, zdim, entry_per_xcd, tail_begin,
                     tail.stages, g.tail_ws, g.direct);
  int st = launch_status();
  if (st == WMMAE_STATUS_SUCCESS && tail_begin != 0xffffffffu) {
    hipLaunchKernelGGL((wmmae_gemm::reduce_tail_kernel<BM, BN>),
                       dim3(static_cast<unsigned>(tail.tail), BM * BN / 1024),
                       dim3(256), 0, g.stream, g.tail_ws, tail.slices,
                       tail_begin, static_cast<unsigned>(tiles_m * tiles_n),
                       tiles_m, tiles_n, g.c, g.m, g.n, g.ldc, g.alpha, g.beta);
    st = launch_status();
  }
  if (st == WMMAE_STATUS_SUCCESS && zdim > 1) {
    // 16 bytes per access where every slice column and every column of C starts
    // on a 16-byte boundary (entries of a pointer array: not known here)
    const bool vec = g.m % 4 == 0 && g.ldc % 4 == 0 && g.c_ptrs == nullptr &&
                     reinterpret_cast<uintptr_t>(g.c) % 16 == 0 &&
                     g.stride_c % 4 == 0 &&
                     reinterpret_cast<uintptr_t>(g.partial) % 16 == 0;
    const long long blocks =
        ceil_div(static_cast<long long>(g.m) * g.n, vec ? 1024 : 256);
    for (int e0 = 0; e0 < g.batch; e0 += kMaxGridY) {
      const dim3 grid(static_cast<unsigned>(blocks),
                      std::min(g.batch - e0, kMaxGridY));
      if (vec)
        hipLaunchKernelGGL(wmmae_gemm::reduce_splits_kernel<4>, grid, dim3(256),
                           0, g.stream, g.partial, zdim, g.c, g.m, g.n, g.ldc,
                           g.stride_c, g.c_ptrs, g.alpha, g.beta,
                           static_cast<long long>(g.batch),
                           static_cast<unsigned>(e0));
      else
        hipLaunchKernelGGL(wmmae_gemm::reduce_splits_kernel<1>, grid, dim3(256),
                           0, g.stream, g.partial, zdim, g.c, g.m, g.n, g.ldc,
                           g.stride_c, g.c_ptrs, g.alpha, g.beta,
                           static_cast<long long>(g.batch),
                           static_cast<unsigned>(e0));
    }
    st = launch_status();
  }
  if (st == WMMAE_STATUS_SUCCESS && t_gemm_end != nullptr)
    WMMAE_HIP_TRY(hipEventRecord(t_gemm_end, g.stream));
  return st;
}

// Tile choice: the 256x128 tile moves the fewest operand bytes per flop and is
// the choice whenever its rounds cost less; the tiles run in rounds
// of one per compute unit, so when the last round would be mostly empty the
// 128x128 tile (5 to 25 % slower per flop) can still finish sooner; 64x64
// tiles for problems too small to give the larger ones work.
template <class MT, int TERMS, bool RN> int gemm_by_size(const GemmArgs &g) {
  const int cus = device_cus();
  const long long z = g.partial != nullptr ? g.splits : 1;
  const long long big =
      ceil_div(g.m, 256) * ceil_div(g.n, 128) * g.batch * z;
  const long long mid =
      ceil_div(g.m, 128) * ceil_div(g.n, 128) * g.batch * z;
  if constexpr (TERMS <= 2 && !RN) {
    // (k a multiple of 32, or the variant with a shorter last stage)
    if (g.is_direct)
      return g.k % 32 == 0 ? launch_gemm<MT, TERMS, 256, 128, 2, 2, RN, 1>(g)
                           : launch_gemm<MT, TERMS, 256, 128, 2, 2, RN, 2>(g);
  }
  // (not with the separate fp32 adds of RN: their temporaries do not fit the
  // register file next to the large tile's accumulators)
  if constexpr (!RN) {
    const int KT = packed_k_tiles(g.k);
    if (big_tile_candidate(TERMS, mid, static_cast<int>(ceil_div(KT, z)))) {
      // time in units of one 128x128 tile: rounds * tile cost
      const bool tail_ok = g.batch == 1 && z == 1 && g.c_ptrs == nullptr &&
                           g.tail_ws != nullptr;
      const double t_big =
          rounds_cost(big, cus, KT, tail_ok) * fit::units256x128(TERMS);
      // (a 128x128 tile measured at 1.2 to 1.25 times half a 256x128 tile in
      // runs of two to eight rounds, 1.05 in long ones)
      const double t_mid =
          rounds_cost(mid, cus, KT, tail_ok) * fit::units128x128(TERMS);
      if (t_big <= t_mid)
        return launch_gemm<MT, TERMS, 256, 128, 2, 2, RN>(g);
    }
  }
  if (mid >= cus || (g.m > 64 && g.n > 64))
    return launch_gemm<MT, TERMS, 128, 128, 2, 2, RN>(g);
  return launch_gemm<MT, TERMS, 64, 64, 2, 2, RN>(g);
}

template <class MT, int TERMS> int per_cu_by_shape(const int shape) {
  switch (shape) {
  case 0:
    return workgroups_per_cu<MT, TERMS, 256, 128, 2, 2, false>();
  case 1:
    return workgroups_per_cu<MT, TERMS, 128, 128, 2, 2, false>();
  default:
    return workgroups_per_cu<MT, TERMS, 64, 64, 2, 2, false>();
  }
}
// the arguments that a kernel takes
template <int CUT>
wmmae_gemm::fused_params<CUT>
launch_params(const wmmae_gemm::FusedSpreadParams &p) {
  if constexpr (CUT == wmmae_gemm::kFusedSpread)
    return p;
  else
    return {p, p.alpha, p.beta, p.inv_scale};
}
template <class T, int TERMS, int BM, int BN, int CW, int PW, int DEPTH, bool RN,
          bool STREAM, int CUT>
int launch_fused_grid(const FusedArgs &f, const long long grid) {
  using Cfg = wmmae_gemm::FusedConfig<TERMS, BM, BN, CW, PW>;
  auto kernel = wmmae_gemm::tcec_gemm_fused_kernel<T, TERMS, BM, BN, CW, PW,
                                                   DEPTH, RN, STREAM, CUT>;
  static std::atomic<unsigned long long> lds_allowed{0};
  WMMAE_HIP_TRY(allow_dynamic_lds(reinterpret_cast<const void *>(kernel),
                                  Cfg::LDS_BYTES, lds_allowed));
  if (t_gemm_begin != nullptr)
    WMMAE_HIP_TRY(hipEventRecord(t_gemm_begin, f.stream));
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)),
                     dim3(Cfg::NTHREADS), Cfg::LDS_BYTES, f.stream,
                     launch_params<CUT>(f.p));
  const int st = launch_status();
  if (st == WMMAE_STATUS_SUCCESS && t_gemm_end != nullptr)
    WMMAE_HIP_TRY(hipEventRecord(t_gemm_end, f.stream));
  return st;
}

template <class T, int TERMS, int BM, int BN, int CW, int PW, int DEPTH, bool RN,
          int CUT>
int launch_fused(FusedArgs f) {
  wmmae_gemm::FusedSpreadParams &p = f.p;
  p.tiles_m = static_cast<int>(ceil_div(p.M, BM));
  p.tiles_n = static_cast<int>(ceil_div(p.N, BN));
  const long long tpb = static_cast<long long>(p.tiles_m) * p.tiles_n;
  const long long items = p.batch * tpb;
  if (items >= (1ll << 30)) // the kernel counts tiles in 32 bits
    return WMMAE_STATUS_NOT_SUPPORTED;
  if constexpr (CUT == wmmae_gemm::kFusedSpread) {
    const long long all = items * p.slices;
    if (all >= (1ll << 30))
      return WMMAE_STATUS_NOT_SUPPORTED;
    p.grouped = 0;
    return launch_fused_grid<T, TERMS, BM, BN, CW, PW, DEPTH, RN, false, CUT>(
        f, 8 * ceil_div(all, 8));
  } else {
  // with 8 or more batch entries an XCD (block index mod 8) owns whole entries
  // (not when the XCD that owns one entry more than the others would need over
  // 15 % more rounds of tiles than an even spread)
  const long long resident =
      static_cast<long long>(device_cus()) * fit::fused_resident(BM);
  const long long per_xcd = std::max(1ll, resident / 8);
  p.grouped = device_xcds() == kKernelXcds && p.batch >= 8 &&
              ceil_div(ceil_div(p.batch, 8) * tpb, per_xcd) * 100 <=
                  ceil_div(items, 8 * per_xcd) * 115;
  const long long spread = p.grouped ? 8 * ceil_div(p.batch, 8) * tpb : items;
  // one workgroup per tile when all of them are resident together, else
  // persistent workgroups
  if (spread <= resident)
    return launch_fused_grid<T, TERMS, BM, BN, CW, PW, DEPTH, RN, false, CUT>(
        f, spread);
  return launch_fused_grid<T, TERMS, BM, BN, CW, PW, DEPTH, RN, true, CUT>(
      f, p.grouped ? 8 * per_xcd : resident);
  }
}

// (RN has no rates of its own.  Three terms with RN are short of registers on the
// 128x128 tile, 48 to 80 bytes of scratch in the K loop, and even so no slower:
// 45 products for which it is chosen took 1.00 of its time with 64x64 tiles in
// the median, 0.86 to 1.21, and 0.61 of what they took on packed operands.)
template <class T, int TERMS, bool RN> int fused_by_size(const FusedArgs &f) {
  using namespace wmmae_gemm;
  if (f.spread_tile == 64)
    return launch_fused<T, TERMS, 64, 64, 4, 4, 4, RN, kFusedSpread>(f);
  if (f.spread_tile == 128)
    return launch_fused<T, TERMS, 128, 128, 8, 4, 2, RN, kFusedSpread>(f);
  if (f.p.slice_stages > 0) // (64x64 only: see fused_time)
    return launch_fused<T, TERMS, 64, 64, 4, 4, 4, RN, kFusedSliced>(f);
  if (fused_small_tiles(TERMS, f.p.M, f.p.N, f.p.K, f.p.batch,
                        f.p.a_source != wmmae_gemm::kFusedKRows ||
                            f.p.b_source != wmmae_gemm::kFusedKRows))
    return launch_fused<T, TERMS, 64, 64, 4, 4, 4, RN, kFusedWhole>(f);
  return launch_fused<T, TERMS, 128, 128, 8, 4, 2, RN, kFusedWhole>(f);
}

// The table of one policy: split tag T, MFMA element type MT, stored terms; RN:
// the policy has the variant that adds the leading product outside the matrix
// core.
template <class T, class MT, int TERMS, bool RN>
constexpr PolicyKernels make_policy_kernels() {
  PolicyKernels k{};
  k.pack = launch_pack<T, TERMS>;
  k.gemm = gemm_by_size<MT, TERMS, false>;
  if constexpr (RN) {
    k.gemm_rn = gemm_by_size<MT, TERMS, true>;
    k.fused_rn = fused_by_size<T, TERMS, true>;
  }
  k.fused = fused_by_size<T, TERMS, false>;
  k.per_cu = per_cu_by_shape<MT, TERMS>;
  return k;
}

} // namespace wmmae_driver
