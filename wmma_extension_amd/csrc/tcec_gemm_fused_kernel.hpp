// TCEC SGEMM for gfx950 in one launch, straight from the fp32 operands: for
// products that are over before a split pass (split_pack_kernel) and a second
// launch would pay, in any of the four transpose combinations, any leading
// dimension and any alignment.
//
//   HBM/L2 --global loads--> registers (fp32, DEPTH stages of 32 k in flight)
//       --split--> 16-bit terms in LDS, two stages, in the same fragment-major
//         chunk order the packed kernel uses (slots of a k group permuted,
//         direct_swizzle)
//       --ds_read_b128--> MFMA operands of the next stage
//
// The reference's tiled GEMM has the same shape of data flow (fp32 tiles in
// shared memory, split at fragment load: test/tcec/batch_gemm.cu:196-386,
// tcec/tcec.hpp:213-229) but splits every element once per warp that needs it;
// here every element of a tile is split once per workgroup.
//
// What bounds it: at these sizes a compute unit has one or two workgroups, and a
// k stage (32 of k) takes as long as its longest chain of instructions between
// two barriers, not what any unit could do: of the 0.39 us of a stage of a 64x64
// tile with two terms, done by four waves that load, split and multiply, the
// matrix cores need 0.08, LDS 0.16.  Hence
//   * two parts: PW producer waves load and split, CW consumer waves read
//     fragments and multiply, one of each on every SIMD, one barrier a stage
//     (0.39 -> 0.32 us; the kernel before, which took the fp32 values through an
//     LDS ring and read them back, 0.8);
//   * the fp32 values wait in the producers' registers, DEPTH stages in flight:
//     no second LDS round trip, and the memory latency is covered;
//   * the consumers read the fragments of stage s+1 while the MFMAs of stage s
//     run;
//   * few registers, so that two workgroups of the 64x64 tile share a compute
//     unit (0.45 us for a stage of both);
//   * with more tiles than resident workgroups the (tile, k stage) pairs of a
//     workgroup are one stream, so that the next tile's stages are loaded and
//     split while a tile is stored (STREAM).
// Whole launches, two terms, before -> now: 1024^3 30.5 -> 16.2 us (two kernels
// on packed operands 27.7), 512^3 16.7 -> 9.8, 7 x 777x1333x515 with rows
// contiguous 127 -> 58 (packed 61), 1024 entries of 100^3 35.2 -> 29.8; three
// terms: 1024^3 packed 27.3 -> 20.7.
//
// How an operand is read (chosen by the host for each operand; the two halves
// of a workgroup's waves load A and B, so a wave runs one of the three):
//   kFusedKRows  k contiguous, k >= 4: a row block (16 rows x 32 k) in two
//                16-byte loads per lane, load h covering rows 8h .. 8h+7, eight
//                lanes to a row's 128 bytes.  16-byte loads need only a
//                float's alignment.
//   kFusedRRows  rows contiguous: 64 rows x 8 k in eight 4-byte loads per
//                lane, lane = row, 256 contiguous bytes a load.
//   kFusedAny    64 rows x 8 k with 64-bit addresses: k < 4, or strides of
//                2^24 floats and more.
// Rows past the matrix are clamped to the last row (their results are never
// stored).  In a last stage of fewer than 32 k no lane reads past the end of k
// (load_tail_stage), and what lies there is zeroed before the split.
//
// Tiles: 128x128 (8 + 4 waves) reads an element half as often and takes 0.58 us
// for a stage, 64x64 (4 + 4) gives four times the workgroups; the host's estimate
// of either's time decides (fused_time).
//
// Operand element (r, l) of op(A) is A[r*a_rs + l*a_ks] (rows = m), of op(B) it
// is B[r*b_rs + l*b_ks] (rows = n); batch entry y is base + y*stride or ptrs[y].
// The products, their order and the epilogue are those of tcec_gemm_kernel, so
// both paths give the same bits.
#pragma once
#include "tcec_gemm_kernels.hpp"

namespace wmmae_gemm {

enum FusedSource { kFusedKRows = 0, kFusedRRows = 1, kFusedAny = 2 };
// K: whole, cut into slices that a workgroup makes one after the other, or cut
// into slices that a workgroup each makes
enum FusedCut { kFusedWhole = 0, kFusedSliced = 1, kFusedSpread = 2 };

struct FusedOperands {
  const float *A;
  const float *const *a_ptrs;
  long long a_rs, a_ks, a_bs;
  const float *B;
  const float *const *b_ptrs;
  long long b_rs, b_ks, b_bs;
  float *C;
  float *const *c_ptrs;
  long long ldc, c_bs;
  int M, N, K, batch;
  int tiles_m, tiles_n;
  // XCD x (block index mod 8) owns the batch entries x, x+8, ... (set by the
  // launcher for 8 or more entries that spread evenly enough)
  int grouped;
  int a_source, b_source; // FusedSource
  int slice_stages; // CUT: k stages of a slice
};
// What every workgroup reads of its launch, the number of workgroups behind it
// included, lies in three lines of 64 bytes: with the fields of the slices among
// them and a fourth line 1024^3 took 15.10 us for 14.92, calls of 9 us 0.1 more.
struct FusedParams : FusedOperands {
  float alpha, beta, inv_scale;
  // (FusedSpreadParams' names, for code that is never reached with these)
  static constexpr int slices = 1;
  static constexpr float *planes = nullptr;
  static constexpr unsigned long long *arrivals = nullptr, launch = 0;
};
static_assert(sizeof(FusedParams) + 4 <= 192, "three lines");
// kFusedSpread: K slices; room for the slices' sums, slice z of tile t (entry by
// entry) at planes + (t*slices + z)*BM*BN, and a word per tile (last_of_tile), with
// what tells this launch's counts from other contents
struct FusedSpreadParams : FusedOperands {
  int slices;
  float *planes;
  unsigned long long *arrivals, launch;
  float alpha, beta, inv_scale;
};
template <int CUT>
using fused_params =
    std::conditional_t<CUT == kFusedSpread, FusedSpreadParams, FusedParams>;

// CW consumer waves (2 x CW/2 over the tile), PW producer waves
template <int TERMS, int BM, int BN, int CW, int PW> struct FusedConfig {
  static constexpr int NTHREADS = 64 * (CW + PW);
  static constexpr int RBA = BM / 16, RBB = BN / 16, NRB = RBA + RBB;
  static constexpr int U = RBA / (PW / 2); // units of 512 floats per producer
  static constexpr int BUF_BYTES = NRB * TERMS * 1024;
  static constexpr int LDS_BYTES = 2 * BUF_BYTES;
  static_assert(BM == BN && BM % 64 == 0 && RBA % (PW / 2) == 0,
                "half the producers load A, half load B, in units of 64 x 8");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS of one compute unit");
};

// The word that counts the workgroups that have finished their slice of a tile
// holds the launch's number above six bits of count.  A workspace holds what its
// last user left there, so every workgroup, before it counts itself, replaces any
// other contents by a count of zero: whoever's exchange fails finds the word
// counting already.  The last one clears it, so that a captured launch, whose
// number stays, finds no count when it is replayed.  (Counting itself by an
// exchange that is tried until it succeeds takes 32 workgroups that finish
// together up to 32 round trips: 64x64x34272 34.5 us, now 24.2.)
__device__ __forceinline__ void
start_count(unsigned long long *const word, const unsigned long long launch) {
  unsigned long long seen = __hip_atomic_load(word, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
  if ((seen >> 6) != launch)
    __hip_atomic_compare_exchange_strong(word, &seen, launch << 6,
                                         __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
}
// Whether the calling workgroup is the last of the `count` (2 .. 32) of a tile.
// One lane, behind the barrier at which the workgroup's sums have reached memory.
__device__ __forceinline__ unsigned
last_of_tile(unsigned long long *const word, const unsigned count) {
  const unsigned long long before = __hip_atomic_fetch_add(
      word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const bool last = (before & 63u) + 1u >= count;
  if (last)
    __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return last ? 1u : 0u;
}

//   RN_MAIN : accumulate the leading product with fp32 adds outside the matrix
//             core (tcec_gemm_kernel's RN_MAIN; the reference's mma_rn_sync)
//   STREAM  : a workgroup walks several tiles; else one, the grid covers them all
//             (the cursor's step to the next tile costs a stage 5 to 10 %, a
//             pipeline refill per tile 2 to 3 us: 4096 tiles of 64x64 at k = 128
//             46.6 -> 30.3 us)
//   SLICED  : K is cut into slices of p.slice_stages stages.  A slice starts from
//             cleared accumulators, its sums are rounded to fp32 as the plane of
//             a slice in memory is, and the slices are added in double precision
//             in ascending order: the bits of the other kernels' K slices
//             (reduce_splits_kernel), without planes, fold launch or workspace.
//             1024^3 in four slices, whole calls: two fp16 terms 17.0 us (16.1
//             over an uncut K, 27.2 with packed operands, their GEMM and its
//             fold), three bf16 terms 22.9 (21.8, 27.2)
//   SPREAD  : a workgroup makes one slice of a tile; the slices' sums meet in
//             memory, and the last workgroup of a tile adds them in double
//             precision in ascending order: the same bits again.  For few output
//             tiles and long k, where a workgroup that makes all slices leaves the
//             chip idle and packed operands cost three launches.  Whole calls,
//             two fp16 terms, before -> now: 2005x64x23136 (rows contiguous) 148
//             -> 44 us, 64x3232x11712 60 -> 34, 32x480x7332 27 -> 18, 34x36x1874
//             18 -> 11; of 500 random products that are cut the 305 that it is
//             chosen for take 0.73 of their time without it, the slowest 1.09.  What
//             bounds it with many slices: the last workgroup's reading of them,
//             0.26 us each (128x128: 0.87), one compute unit's share of memory
//   DEPTH   : stages of fp32 values in flight in registers (even: the LDS
//             buffer and fragment set of a step are then compile-time choices)
template <class T, int TERMS, int BM, int BN, int CW, int PW, int DEPTH,
          bool RN_MAIN, bool STREAM, int CUT>
// (SLICED, and SPREAD's fold: the double-precision sums must not cost the second
// workgroup of a compute unit, four waves a SIMD; three bf16 terms with RN_MAIN
// took 130 registers of the 128 that leaves)
__global__ void __launch_bounds__(64 * (CW + PW), CUT == kFusedWhole ? 1
                                                  : BM > 64          ? 3
                                                                     : 4)
    tcec_gemm_fused_kernel(const fused_params<CUT> p) {
  using traits = mtk::wmma::tcec::detail::split_traits<T>;
  using S = typename traits::storage;
  typedef S ab_vec __attribute__((ext_vector_type(8)));
  typedef S s2_t __attribute__((ext_vector_type(2)));
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  using Cfg = FusedConfig<TERMS, BM, BN, CW, PW>;
  constexpr int RBA = Cfg::RBA, U = Cfg::U;
  constexpr int WGN = CW / 2;
  constexpr int WM = BM / 2, WN = BN / WGN;
  constexpr int MT_ = WM / 16, NT_ = WN / 16;
  static_assert(DEPTH % 2 == 0 && DEPTH >= 2, "even ring");
  constexpr bool SLICED = CUT == kFusedSliced, SPREAD = CUT == kFusedSpread;
  static_assert(!(STREAM && SPREAD), "a workgroup makes one slice");
  // Two sets of fragments where they fit the registers that two workgroups (64x64
  // tile) or three waves a SIMD (128x128) leave a wave; else one set, a term's
  // fragments refilled for the next stage once its last product has been issued.
  // (SLICED: the double-precision sums take the registers of the second set)
  constexpr bool RECYCLE = TERMS == 3 || BM > 64 || SLICED;

  extern __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[];

  const unsigned lane = threadIdx.x & 63u;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int M = p.M, N = p.N, K = p.K;
  const int all_k = (K + 31) / 32;

  // a producer's work: A or B, units unit0 .. unit0 + U-1 of it
  const bool loads_a = wave - CW < PW / 2;
  const int unit0 = (loads_a ? wave - CW : wave - CW - PW / 2) * U;
  const int source =
      __builtin_amdgcn_readfirstlane(loads_a ? p.a_source : p.b_source);

  // ---- this workgroup's tiles: v = first + i*stride while v < count
  const int tpb = p.tiles_m * p.tiles_n;
  // SPREAD: the (slice, tile) pairs, slice by slice, in eight runs, one per XCD:
  // what an XCD's tiles share is one slice of the operands
  const int spread_tiles = tpb * p.batch;
  int slice = 0, spread_tile = 0; // tile: entry by entry
  if constexpr (SPREAD) {
    const unsigned items = static_cast<unsigned>(spread_tiles * p.slices);
    const unsigned run = (items + 7) >> 3;
    const unsigned item = (blockIdx.x & 7u) * run + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= run || item >= items)
      return; // (before any barrier)
    slice = static_cast<int>(item / static_cast<unsigned>(spread_tiles));
    spread_tile = static_cast<int>(item) - slice * spread_tiles;
  }
  // the k stages this workgroup takes of a tile, stage0 the first
  const int stage0 = SPREAD ? slice * p.slice_stages : 0;
  const int num_k = SPREAD && all_k - stage0 > p.slice_stages ? p.slice_stages
                                                              : all_k - stage0;
  // k of the last stage, 1 .. 32
  const int k_left = stage0 + num_k == all_k ? K - 32 * (all_k - 1) : 32;
  const bool grouped = !SPREAD && p.grouped != 0;
  const int xcd = grouped ? static_cast<int>(blockIdx.x & 7u) : 0;
  const int first = grouped ? static_cast<int>(blockIdx.x >> 3)
                            : static_cast<int>(blockIdx.x);
  const int stride = grouped ? static_cast<int>(gridDim.x >> 3)
                             : static_cast<int>(gridDim.x);
  const int count = grouped ? ((p.batch - xcd + 7) >> 3) * tpb : p.batch * tpb;
  if (!SPREAD && first >= count)
    return; // nothing for this workgroup (before any barrier)
  const int n_my = STREAM ? (count - first + stride - 1) / stride : 1;
  auto decode = [&](const int i, int &entry, int &tm, int &tn) {
    const int v = SPREAD ? spread_tile : first + i * stride;
    const int bi = v / tpb;
    entry = grouped ? bi * 8 + xcd : bi;
    tile_of<8>(static_cast<unsigned>(v - bi * tpb), static_cast<unsigned>(tpb),
               static_cast<unsigned>(p.tiles_m),
               static_cast<unsigned>(p.tiles_n), !grouped && !SPREAD, tm, tn);
  };

  f32x4 acc_main[MT_][NT_], acc_err[MT_][NT_];
  auto clear_acc = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT_; i++)
#pragma unroll
      for (int j = 0; j < NT_; j++) {
        acc_main[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        acc_err[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  };
  // the accumulated value of tile (i, j), before alpha
  auto folded = [&](const int i, const int j) {
    f32x4 o = acc_main[i][j];
    if constexpr (TERMS >= 2)
      o = epilogue_fold(o, acc_err[i][j], p.inv_scale);
    return o;
  };
  struct Frags {
    ab_vec a[TERMS][MT_], b[TERMS][NT_];
  };
  // 16-byte slot of this lane's fragment inside a chunk
  const unsigned frag_off =
      16u * ((lane & 48u) + ((lane & 15u) ^ direct_swizzle(lane >> 4)));
  // the fragments of term TA of A and term TB of B (-1: none) of the stage in
  // the LDS buffer at `base`
  auto read_terms = [&](Frags &f, const unsigned base, auto TA, auto TB)
                        __attribute__((always_inline)) {
    constexpr int ta = decltype(TA)::value, tb = decltype(TB)::value;
    const unsigned char *const buf =
        lds_raw + base + frag_off;
    const unsigned char *const sa = buf + wm * MT_ * TERMS * 1024;
    const unsigned char *const sb = buf + (RBA + wn * NT_) * TERMS * 1024;
    if constexpr (tb >= 0) {
#pragma unroll
      for (int j = 0; j < NT_; j++)
        f.b[tb][j] =
            *reinterpret_cast<const ab_vec *>(sb + (j * TERMS + tb) * 1024);
    }
    if constexpr (ta >= 0) {
#pragma unroll
      for (int i = 0; i < MT_; i++)
        f.a[ta][i] =
            *reinterpret_cast<const ab_vec *>(sa + (i * TERMS + ta) * 1024);
    }
  };
  auto read_frags = [&](Frags &f, const unsigned base)
                        __attribute__((always_inline)) {
    static_for<0, TERMS>([&](auto T_) __attribute__((always_inline)) {
      read_terms(f, base, T_, T_);
    });
  };
  auto mfma = [](const ab_vec x, const ab_vec y, const f32x4 z) -> f32x4 {
    if constexpr (std::is_same<S, _Float16>::value)
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(x, y, z, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, z, 0, 0, 0);
  };
  // MFMA n of a step.  Same products and, per accumulator, the same order as
  // tcec_gemm_kernel, product by product over the wave's tiles (neighbouring
  // MFMAs never wait for each other's accumulator).
  constexpr int NPROD = TERMS == 1 ? 1 : (TERMS == 2 ? 3 : 6);
  constexpr int NTILE = MT_ * NT_;
  constexpr int NMFMA = NPROD * NTILE;
  auto multiply = [&](const Frags &f, auto N_) __attribute__((always_inline)) {
    constexpr int n = decltype(N_)::value, pr = n / NTILE;
    constexpr int i = (n % NTILE) / NT_, j = n % NT_;
    constexpr int first_product = TERMS == 1 ? 5 : (TERMS == 2 ? 3 : 0);
    // (term of A, term of B): smallest products first, the main product last
    constexpr int ta_of[6] = {2, 0, 1, 1, 0, 0}, tb_of[6] = {0, 2, 1, 0, 1, 0};
    constexpr int ta = ta_of[first_product + pr], tb = tb_of[first_product + pr];
    if constexpr (pr + 1 < NPROD)
      acc_err[i][j] = mfma(f.a[ta][i], f.b[tb][j], acc_err[i][j]);
    else if constexpr (RN_MAIN)
      acc_main[i][j] +=
          mfma(f.a[0][i], f.b[0][j], f32x4{0.f, 0.f, 0.f, 0.f});
    else
      acc_main[i][j] = mfma(f.a[0][i], f.b[0][j], acc_main[i][j]);
  };

  // A producer's part: the workgroup's (tile, k stage) pairs as one stream, so
  // that the next tile's first stages are on their way while the consumers store
  // a tile.  SRC: how this wave's operand is read.
  auto produce = [&](auto SRC) __attribute__((always_inline)) {
    constexpr int src_kind = decltype(SRC)::value;
    constexpr int NOFF = src_kind == kFusedKRows ? 2 : 8;
    // ---- source of this wave's operand
    typedef const float *const __attribute__((address_space(4))) *ptr_array_t;
    typedef const __attribute__((address_space(1))) char *gbytes_t;
    const float *const *const ptrs = loads_a ? p.a_ptrs : p.b_ptrs;
    const long long rs = loads_a ? p.a_rs : p.b_rs;
    const long long ks = loads_a ? p.a_ks : p.b_ks;
    const int last = (loads_a ? M : N) - 1;
    // src[u]: wave-uniform address at the load cursor's stage, voff[u][.]: the
    // lane's byte offsets from it
    unsigned long long src[U];
    unsigned voff[U][NOFF];
    // the load cursor: tile and stage, first row of the tile
    int ld_tile = 0, ld_stage = 0, tile_row = 0;
    // first row of unit u (KRows: a row block, else 64 rows), its k group
    auto unit_row = [&](const int u) {
      const int row = tile_row + (src_kind == kFusedKRows
                                      ? 16 * (unit0 + u)
                                      : 64 * ((unit0 + u) >> 2));
      return row < last ? row : last;
    };
    auto unit_k = [&](const int u) {
      return src_kind == kFusedKRows ? 0 : 8 * ((unit0 + u) & 3);
    };
    // sources of the cursor's stage when it is the last one and shorter than
    // 32: every lane reads inside the operand.  KRows: a lane whose four floats
    // would end past the row reads the row's last four instead (the uniform
    // address then starts four floats early where there are any, for the lanes
    // that read up to three floats before the stage); RRows: k clamped to the
    // last one.
    auto load_tail_stage = [&]() __attribute__((always_inline)) {
      const int k0 = 32 * (stage0 + ld_stage);
      int left = k_left;
      asm volatile("" : "+s"(left));
#pragma unroll
      for (int u = 0; u < U; u++) {
        if constexpr (src_kind == kFusedKRows) {
          const int bias = k0 > 0 ? kDirectBias : 0;
          const int back = direct_tail_shift(lane, left);
          src[u] -= 4ull * bias;
#pragma unroll
          for (int h = 0; h < 2; h++)
            voff[u][h] += 4u * static_cast<unsigned>(bias - back);
        } else if constexpr (src_kind == kFusedRRows) {
          const int behind = left - 1 - unit_k(u); // k of the unit after its first
          if (behind < 0)
            src[u] += static_cast<long long>(behind) * ks * 4;
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const int back = e - (behind < 0 ? 0 : behind);
            if (back > 0)
              voff[u][e] -= static_cast<unsigned>(back * ks) * 4u;
          }
        }
        asm volatile("" : "+s"(src[u]));
      }
    };
    // the cursor's tile: sources of its first stage
    auto set_tile = [&]() __attribute__((always_inline)) {
      int entry, tm, tn;
      decode(ld_tile, entry, tm, tn);
      tile_row = loads_a ? tm * BM : tn * BN;
      const float *const X =
          ptrs != nullptr
              ? ((ptr_array_t)ptrs)[entry]
              : (loads_a ? p.A + entry * p.a_bs : p.B + entry * p.b_bs);
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int row0 = unit_row(u);
        src[u] = reinterpret_cast<unsigned long long>(
            X + row0 * rs + (32ll * stage0 + unit_k(u)) * ks);
        asm volatile("" : "+s"(src[u]));
#pragma unroll
        for (int o = 0; o < NOFF; o++) {
          const int r = row0 + (src_kind == kFusedKRows
                                    ? 8 * o + static_cast<int>(lane >> 3)
                                    : static_cast<int>(lane));
          const int mine = (r < last ? r : last) - row0;
          voff[u][o] =
              src_kind == kFusedKRows
                  ? static_cast<unsigned>(mine * rs) * 4u + 16u * (lane & 7u)
              : src_kind == kFusedRRows
                  ? static_cast<unsigned>(mine) * 4u +
                        static_cast<unsigned>(o * ks) * 4u
                  : static_cast<unsigned>(mine);
        }
      }
      if (num_k == 1 && k_left < 32)
        load_tail_stage();
    };
    set_tile();
    auto advance = [&]() __attribute__((always_inline)) {
      if (ld_stage + 1 < num_k) {
        ld_stage++;
#pragma unroll
        for (int u = 0; u < U; u++) {
          src[u] += src_kind == kFusedKRows ? 128ull : 128ull * ks;
          asm volatile("" : "+s"(src[u]));
        }
        if (ld_stage + 1 == num_k && k_left < 32)
          load_tail_stage();
      } else if (STREAM && ld_tile + 1 < n_my) {
        ld_tile++;
        ld_stage = 0;
        set_tile();
      } // else: the last stage again, never used
    };
    // the tile stage that is split next
    int conv_k = 0;
    auto advance_conv = [&]() __attribute__((always_inline)) {
      conv_k = conv_k + 1 == num_k ? 0 : conv_k + 1;
    };
    float raw[DEPTH][U][8];
    auto load_unit = [&](auto SLOT, auto UN) __attribute__((always_inline)) {
      constexpr int slot = decltype(SLOT)::value, u = decltype(UN)::value;
      typedef f32x4 __attribute__((aligned(4))) f32x4_u;
      typedef const __attribute__((address_space(1))) f32x4_u *vec_ptr;
      typedef const __attribute__((address_space(1))) float *flt_ptr;
      const gbytes_t base = reinterpret_cast<gbytes_t>(src[u]);
      if constexpr (src_kind == kFusedAny) {
        const int k0 = 32 * (stage0 + ld_stage) + unit_k(u);
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const int k = k0 + e < K ? k0 + e : K - 1;
          raw[slot][u][e] = *reinterpret_cast<flt_ptr>(
              base + 4 * (static_cast<long long>(voff[u][e]) * rs +
                          (k - k0) * ks));
        }
      } else {
#pragma unroll
        for (int o = 0; o < NOFF; o++) {
          // (redefined in place so that the address is formed here, as the
          // instruction's scalar base + 32-bit lane offset)
          asm volatile("" : "+v"(voff[u][o]));
          if constexpr (src_kind == kFusedKRows) {
            const f32x4 x = *reinterpret_cast<vec_ptr>(base + voff[u][o]);
#pragma unroll
            for (int e = 0; e < 4; e++)
              raw[slot][u][4 * o + e] = x[e];
          } else {
            raw[slot][u][o] = *reinterpret_cast<flt_ptr>(base + voff[u][o]);
          }
        }
      }
    };
    // the values of a last, shorter stage waiting in `slot`: what lies past the
    // end of k becomes zero (`left` is redefined in place so that the masks are
    // worked out here and not kept through the loop)
    auto zero_tail = [&](auto SLOT) __attribute__((always_inline)) {
      constexpr int slot = decltype(SLOT)::value;
      int left = k_left;
      asm volatile("" : "+s"(left));
      if constexpr (src_kind == kFusedKRows) {
        const int shift = direct_tail_shift(lane, left);
        const bool by1 = (shift & 1) != 0, by2 = (shift & 2) != 0;
        const bool all = shift > 3;
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int h = 0; h < 2; h++) {
            float *const r = &raw[slot][u][4 * h];
            float v0 = r[0], v1 = r[1], v2 = r[2], v3 = r[3];
            v0 = by1 ? v1 : v0;
            v1 = by1 ? v2 : v1;
            v2 = by1 ? v3 : v2;
            v3 = by1 || by2 || all ? 0.f : v3;
            v0 = by2 ? v2 : v0;
            v1 = by2 ? (by1 ? 0.f : r[3]) : v1;
            v2 = by2 || all ? 0.f : v2;
            r[0] = all ? 0.f : v0;
            r[1] = all ? 0.f : v1;
            r[2] = v2;
            r[3] = v3;
          }
      } else {
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int mine = left - unit_k(u);
#pragma unroll
          for (int e = 0; e < 8; e++)
            raw[slot][u][e] = e < mine ? raw[slot][u][e] : 0.f;
        }
      }
    };
    // split the stage in `slot` into LDS buffer BUF and load the cursor's stage
    // into the slot, unit by unit
    auto convert = [&](auto SLOT, auto BUF) __attribute__((always_inline)) {
      constexpr int slot = decltype(SLOT)::value;
      unsigned char *const buf = lds_raw + decltype(BUF)::value * Cfg::BUF_BYTES +
                                 (loads_a ? 0 : RBA * TERMS * 1024);
      static_for<0, U>([&](auto UN) __attribute__((always_inline)) {
        constexpr int u = decltype(UN)::value;
        unsigned term[TERMS][4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
          s2_t h[3];
          mtk::wmma::tcec::detail::split2<T>(
              mtk::wmma::tcec::detail::f32x2_t{raw[slot][u][2 * q],
                                               raw[slot][u][2 * q + 1]},
              h[0], h[1], h[2]);
#pragma unroll
          for (int t = 0; t < TERMS; t++)
            term[t][q] = __builtin_bit_cast(unsigned, h[t]);
          if (src_kind == kFusedKRows && q % 2 == 1) {
            // the lane's four floats of load q/2: half of position (row, k group)
            unsigned char *const chunk = buf + (unit0 + u) * TERMS * 1024;
            const unsigned g = (lane & 7u) >> 1, r = 8u * (q / 2) + (lane >> 3);
            const unsigned off =
                256u * g + 16u * (r ^ direct_swizzle(g)) + 8u * (lane & 1u);
#pragma unroll
            for (int t = 0; t < TERMS; t++)
              *reinterpret_cast<u32x2 *>(chunk + t * 1024 + off) =
                  u32x2{term[t][q - 1], term[t][q]};
          }
        }
        if constexpr (src_kind != kFusedKRows) {
          const unsigned g = static_cast<unsigned>((unit0 + u) & 3);
          unsigned char *const chunk =
              buf + (4 * ((unit0 + u) >> 2) + static_cast<int>(lane >> 4)) *
                        (TERMS * 1024);
          const unsigned off =
              256u * g + 16u * ((lane & 15u) ^ direct_swizzle(g));
#pragma unroll
          for (int t = 0; t < TERMS; t++)
            *reinterpret_cast<u32x4 *>(chunk + t * 1024 + off) =
                u32x4{term[t][0], term[t][1], term[t][2], term[t][3]};
        }
        load_unit(SLOT, UN);
        __builtin_amdgcn_sched_barrier(0);
      });
    };

    // ---- prologue: stages 0 .. DEPTH-1 requested, 0 and 1 converted (their
    // slots take the stages DEPTH and DEPTH+1), stage 0's fragments read
    static_for<0, DEPTH>([&](auto SLOT) __attribute__((always_inline)) {
      static_for<0, U>([&](auto UN) __attribute__((always_inline)) {
        load_unit(SLOT, UN);
      });
      advance();
    });
    static_for<0, 2>([&](auto SLOT) __attribute__((always_inline)) {
      if (conv_k + 1 == num_k && k_left < 32)
        zero_tail(SLOT);
      convert(SLOT, SLOT);
      advance();
      advance_conv();
    });
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    asm volatile("s_barrier" ::: "memory"); // (the consumers hold stage 0)

    // step s of the stream: stage s+2 into the buffer stage s has left, stage
    // s+2+DEPTH requested
    int left = n_my * num_k;
    auto steps = [&](auto self, auto D_) __attribute__((always_inline)) {
      constexpr int d = decltype(D_)::value;
      if (conv_k + 1 == num_k && k_left < 32)
        zero_tail(ic<(d + 2) % DEPTH>{});
      convert(ic<(d + 2) % DEPTH>{}, ic<d & 1>{});
      advance();
      advance_conv();
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      left--;
      if constexpr (d + 1 < DEPTH)
        if (left > 0)
          self(self, ic<d + 1>{});
    };
    while (left > 0)
      steps(steps, ic<0>{});
  };

  // the matrix C of a batch entry
  auto c_of = [&](const int entry) {
    typedef float *const __attribute__((address_space(4))) *out_array_t;
    return p.c_ptrs != nullptr ? ((out_array_t)p.c_ptrs)[entry]
                               : p.C + static_cast<long long>(entry) * p.c_bs;
  };
  // SPREAD: the sums of slice z of this workgroup's tile: wave, tile of the wave,
  // halves of a lane's four rows, lane.  Written and read with the device's
  // scope, past the XCDs' own L2: with ordinary accesses between agent-scope
  // fences every wave writes its whole L2 back (0.5 us each, one after the other
  // on an XCD: 1024x1376x7016, 1760 slices of 64x64, took 536 us, now 93).
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  auto plane = [&](const int z) {
    return reinterpret_cast<unsigned long long *>(p.planes) +
           (static_cast<long long>(spread_tile) * p.slices + z) * (BM * BN / 2);
  };
  typedef double f64x2 __attribute__((ext_vector_type(2)));
  typedef double f64x4 __attribute__((ext_vector_type(4)));
  // SPREAD, every wave, after the consumers have written the slice's sums: the
  // workgroup that is the last of its tile's adds the slices in double precision
  // in ascending order (the bits of reduce_splits_kernel) and stores the tile.
  // No workgroup waits for another.
  auto fold_if_last = [&]() __attribute__((always_inline)) {
    // the wave's stores have reached memory
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    unsigned *const flag = reinterpret_cast<unsigned *>(lds_raw);
    if (wave == 0 && lane == 0)
      *flag = last_of_tile(p.arrivals + spread_tile,
                           static_cast<unsigned>(p.slices));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (__builtin_amdgcn_readfirstlane(*flag) == 0)
      return;
    int entry, tm, tn;
    decode(0, entry, tm, tn);
    float *const Cb = c_of(entry);
    // a unit: one column of a consumer wave's tiles
    for (int unit = wave; unit < CW * NT_; unit += CW + PW) {
      const int w = unit / NT_, j = unit - w * NT_;
      f64x2 sum[MT_][2];
#pragma unroll
      for (int i = 0; i < MT_; i++)
        sum[i][0] = sum[i][1] = f64x2{0., 0.};
      const unsigned long long *from = plane(0) + unit * (MT_ * 128) + lane;
      constexpr int AHEAD = 16 / MT_; // planes read at a time
      for (int z = 0; z < p.slices; z += AHEAD) {
        unsigned long long v[AHEAD][MT_][2];
#pragma unroll
        for (int a = 0; a < AHEAD; a++) {
          // (past the last plane the last one again, not added)
          const int zz = z + a < p.slices ? z + a : p.slices - 1;
          const unsigned long long *const src =
              from + static_cast<long long>(zz) * (BM * BN / 2);
#pragma unroll
          for (int i = 0; i < MT_; i++)
#pragma unroll
            for (int h = 0; h < 2; h++)
              v[a][i][h] =
                  __hip_atomic_load(src + (i * 2 + h) * 64, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int a = 0; a < AHEAD; a++)
          if (z + a < p.slices)
#pragma unroll
            for (int i = 0; i < MT_; i++)
#pragma unroll
              for (int h = 0; h < 2; h++)
                sum[i][h] += __builtin_convertvector(
                    __builtin_bit_cast(f32x2, v[a][i][h]), f64x2);
      }
      const auto value = [&](const int i, int) {
        const f32x2 lo = __builtin_convertvector(sum[i][0], f32x2),
                    hi = __builtin_convertvector(sum[i][1], f32x2);
        return f32x4{lo[0], lo[1], hi[0], hi[1]} * p.alpha;
      };
      store_piece<MT_, 1, MT_ % 2 == 0, MT_>(
          value, Cb, p.ldc, tm * BM + (w & 1) * WM,
          tn * BN + (w >> 1) * WN + 16 * j, M, N, p.beta, lane);
    }
  };

  // (the waves of a workgroup meet at the same number of barriers, two and one
  // a stage, whatever their part; the producers' vector instructions are the
  // longest part of a step: they go first where they share a SIMD with a
  // consumer: 128x128 tile, per k stage, 657 -> 580 ns, rows contiguous 757 ->
  // 660; 64x64 465 -> 437 with two workgroups on a compute unit)
  if (wave >= CW) {
    __builtin_amdgcn_s_setprio(2);
    if (source == kFusedKRows)
      produce(ic<kFusedKRows>{});
    else if (source == kFusedRRows)
      produce(ic<kFusedRRows>{});
    else
      produce(ic<kFusedAny>{});
    if constexpr (SPREAD) {
      __builtin_amdgcn_s_setprio(0);
      fold_if_last();
    }
    return;
  }

  // ---- consumer: step s of the stream, the MFMAs of stage s while the fragments
  // of stage s+1 (after a tile's last stage the next tile's first) are read
  if constexpr (SPREAD)
    if (wave == 0 && lane == 0) // (while the producers wait for their first loads)
      start_count(p.arrivals + spread_tile, p.launch);
  asm volatile("s_barrier" ::: "memory"); // stages 0 and 1 are there
  Frags f[RECYCLE ? 1 : 2];
  unsigned held = 0; // LDS offset of the buffer whose stage is in registers
  read_frags(f[0], 0u);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  // (LAST with RECYCLE: the fragments are read after the tile has been stored,
  // whose addresses and old values need their registers)
  auto step = [&](auto D_, auto LAST) __attribute__((always_inline)) {
    constexpr int d = decltype(D_)::value;
    const unsigned next = Cfg::BUF_BYTES - held; // buffer of stage s+1
    if constexpr (!RECYCLE) {
      read_frags(f[1 - d], next);
      __builtin_amdgcn_sched_barrier(0);
    }
    static_for<0, NMFMA>([&](auto N_) __attribute__((always_inline)) {
      constexpr int n = decltype(N_)::value;
      multiply(f[RECYCLE ? 0 : d], N_);
      if constexpr (RECYCLE && !decltype(LAST)::value &&
                    (n + 1) % NTILE == 0) {
        // the terms whose last product has just been issued
        constexpr int pr = n / NTILE + (6 - NPROD);
        constexpr int ta = TERMS == 1   ? 0
                           : TERMS == 2 ? (pr == 3 ? 1 : pr == 5 ? 0 : -1)
                                        : (pr == 0   ? 2
                                           : pr == 3 ? 1
                                           : pr == 5 ? 0
                                                     : -1);
        constexpr int tb = TERMS == 1   ? 0
                           : TERMS == 2 ? (pr == 4 ? 1 : pr == 5 ? 0 : -1)
                                        : (pr == 1   ? 2
                                           : pr == 4 ? 1
                                           : pr == 5 ? 0
                                                     : -1);
        __builtin_amdgcn_sched_barrier(0);
        read_terms(f[0], next, ic<ta>{}, ic<tb>{});
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    if constexpr (!(RECYCLE && decltype(LAST)::value)) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      held = next;
    }
  };
  for (int tile = 0; tile < n_my; tile++) {
    f64x4 sum[SLICED ? MT_ : 1][SLICED ? NT_ : 1]; // of the slices
    if constexpr (SLICED) {
#pragma unroll
      for (int i = 0; i < MT_; i++)
#pragma unroll
        for (int j = 0; j < NT_; j++)
          sum[i][j] = f64x4{0., 0., 0., 0.};
      int s = num_k; // stages left of the tile
      while (s > 0) {
        clear_acc();
        const bool last = s <= p.slice_stages;
        const int n = last ? s - 1 : p.slice_stages;
        for (int x = 0; x < n; x++)
          step(ic<0>{}, std::false_type{});
        if (last)
          step(ic<0>{}, std::true_type{});
        s -= p.slice_stages;
#pragma unroll
        for (int i = 0; i < MT_; i++)
#pragma unroll
          for (int j = 0; j < NT_; j++)
            sum[i][j] += __builtin_convertvector(folded(i, j), f64x4);
      }
    } else {
      clear_acc();
      int s = num_k;
      for (; s > (RECYCLE ? 2 : 1); s -= 2) {
        step(ic<0>{}, std::false_type{});
        step(ic<1>{}, std::false_type{});
      }
      if (RECYCLE && s == 2)
        step(ic<0>{}, std::false_type{});
      if (RECYCLE || s == 1) { // the next tile's first fragments arrive in the other set
        step(ic<0>{}, std::true_type{});
        if constexpr (!RECYCLE)
          f[0] = f[1];
      }
    }
    if constexpr (SPREAD) {
      if constexpr (RECYCLE) // (the producers' last barrier)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      unsigned long long *const to = plane(slice) + wave * (NTILE * 128) + lane;
#pragma unroll
      for (int j = 0; j < NT_; j++)
#pragma unroll
        for (int i = 0; i < MT_; i++) {
          const f32x4 v = folded(i, j);
#pragma unroll
          for (int h = 0; h < 2; h++)
            __hip_atomic_store(to + ((j * MT_ + i) * 2 + h) * 64,
                               __builtin_bit_cast(
                                   unsigned long long,
                                   f32x2{v[2 * h], v[2 * h + 1]}),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      fold_if_last();
      return;
    }
    int entry, tm, tn;
    decode(tile, entry, tm, tn);
    float *const Cb = c_of(entry);
    const float alpha = p.alpha;
    const auto out_value = [&](const int i, const int j) {
      if constexpr (SLICED)
        return __builtin_convertvector(sum[i][j], f32x4) * alpha;
      else
        return folded(i, j) * alpha;
    };
    store_piece<MT_, NT_, MT_ % 2 == 0, MT_>(
        out_value, Cb, p.ldc, tm * BM + wm * WM, tn * BN + wn * WN, M, N,
        p.beta, lane);
    if constexpr (RECYCLE) {
      held = Cfg::BUF_BYTES - held;
      if (STREAM)
        read_frags(f[0], held);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
  }
}

} // namespace wmmae_gemm
