// A tiled, batched SGEMM on the fragments of this library's device API, twice, in
// the shape of the reference's bgemm_kernel / mma_core / dmem2smem
// (test/tcec/batch_gemm.cu:74-116, 196-257, 261-386).
//
// tcec_api_gemm_kernel is written against the public functions alone
// (tcec::fragment, load_matrix_sync, mma_sync, store_matrix_sync,
// utils::cp_async), the way a user of the reference writes one.  (It runs fp32
// operands; most products of 16-bit terms take tcec_api_gemm_split_kernel below,
// which splits with tcec::detail::split4 and fills the fragments' registers
// itself.)
//   * fp32 tiles of A (row-major) and B (column-major) are staged in LDS by
//     utils::cp_async, two stages: the copies of stage s+1 are in flight while
//     stage s is multiplied;
//   * every wave splits the elements it needs while loading its fragments
//     (tcec::load_matrix_sync; k is contiguous in both tiles, so the loads
//     are 16 bytes wide) and multiplies with tcec::mma_sync;
//   * the operand fragments are double buffered over the k steps of a stage.
//
// Rows of a staged tile are exactly SK = 32 floats (128 bytes), unpadded, with
// the eight 16-byte pieces of row r stored at piece index p ^ ((r / 2) & 5)
// (tcec::row_major_swizzled / col_major_swizzled): a 16-byte LDS read is served
// sixteen lanes at a time - eight rows of one k group and eight rows of the
// next - and with this permutation they hit all 64 banks once.  No row padding
// does that (every padded stride costs a two-way conflict; the reference's
// skew of 8 floats, batch_gemm.cu:11, is made for 32 banks and 32 lanes).  The
// direct global->LDS copy of gfx950 writes lane-linear destinations, so the
// copy walks the tile image linearly, 16 bytes per lane
// (cp_async_lane_linear), and each lane fetches the logical piece that belongs
// at its place.
//
// Two workgroups of four waves share a compute unit (64 KiB of LDS and at
// most 256 registers each, WAVES_PER_SIMD = 2): while one waits at its
// barrier or for its copies, the other computes.  (One workgroup per compute
// unit with up to 512 registers measured slower for every policy, the
// three-term split included: 144 against 183 TFLOPS at 4096^3.)
//
// Three things the compiler has to be told for the stage loop to become one
// basic block whose MFMAs and conversions it can interleave: the wave index is
// wave-uniform (readfirstlane), the tile pointers handed to load_matrix_sync
// are 16-byte aligned (__builtin_assume_aligned: its 16-byte path is then
// chosen at compile time), and the wait for the copies stays where it is
// written (cp_async::wait_all is a scheduling barrier).
#pragma once
#include <wmma_extension/tcec/tcec.hpp>
#include <wmma_extension/utils.hpp>

namespace wmmae_harness {
namespace w = mtk::wmma;
namespace tcec = mtk::wmma::tcec;
namespace cpa = mtk::wmma::utils::cp_async;

struct ApiGemmShape {
  static constexpr int BM = 128, BN = 128; // block tile
  static constexpr int SK = 32;            // k per stage
  static constexpr int WM = 64, WN = 64;   // wave tile (2 x 2 waves)
  static constexpr int WK = 32;            // k per fragment
  static constexpr int LD = SK;            // unpadded rows, pieces swizzled
  static constexpr int STAGES = 2;
  static constexpr int THREADS = 256;
  static constexpr int STAGE_FLOATS = (BM + BN) * LD;
  static constexpr int LDS_BYTES = STAGES * STAGE_FLOATS * 4;
};

// Copy ROWS x SK floats (row r at src + r*ld) into a swizzled tile (see above).
// A pass of the workgroup moves THREADS / 8 whole rows: thread t writes
// physical piece t % 8 of row t / 8 and fetches the logical piece
// (t % 8) ^ swizzled_piece(row) for it; the rows of a pass are a multiple of
// 16, so a thread's logical piece and source offset are the same in every pass.
template <int ROWS, int SK, int THREADS>
__device__ __forceinline__ void stage_tile(float *const dst,
                                           const float *const src,
                                           const long long ld) {
  static_assert(SK == 32, "rows of 128 bytes");
  constexpr int RP = THREADS / 8; // rows per pass
  static_assert(RP % 16 == 0 && ROWS % RP == 0, "whole passes of whole rows");
  const int tid = static_cast<int>(threadIdx.x);
  const int r_in = tid / 8;
  const int c = (tid % 8) ^ static_cast<int>(tcec::swizzled_piece(r_in));
  const float *const from = src + r_in * ld + 4 * c;
#pragma unroll
  for (int r0 = 0; r0 < ROWS; r0 += RP)
    cpa::cp_async_lane_linear<16>(dst + 4 * (r0 * 8 + tid), from + r0 * ld);
}

// C tile = alpha * A tile * B tile + beta * C tile for one 128 x 128 tile of
// one batch entry.  A: m x k row-major (lda), B: k x n column-major (ldb), C:
// m x n column-major (ldc); m, n multiples of 128, k of 32; batch entry y at
// base + y*stride or, when the pointer arrays are set, at ptrs[y].
// ROUNDING: 0 tcec::mma_sync (the reference's default for the policy), 1
// mma_rn_sync, 2 mma_rz_sync.
template <class T, class Policy, int WAVES_PER_SIMD, int ROUNDING = 0>
__global__ void __launch_bounds__(ApiGemmShape::THREADS, WAVES_PER_SIMD)
    tcec_api_gemm_kernel(const int m, const int n, const int k,
                         const float alpha, const float *const A,
                         const float *const *const a_ptrs, const int lda,
                         const long long stride_a, const float *const B,
                         const float *const *const b_ptrs, const int ldb,
                         const long long stride_b, const float beta,
                         float *const C, float *const *const c_ptrs,
                         const int ldc, const long long stride_c) {
  using S = ApiGemmShape;
  extern __shared__ __attribute__((aligned(16))) float smem[];

  // tile of this workgroup: consecutive block ids run on different XCDs, so
  // ids are regrouped to give each XCD (id % 8) one contiguous run of tiles,
  // walked column by column through bands of eight tile rows
  const unsigned tiles_m = m / S::BM, tiles_n = n / S::BN;
  const unsigned tiles = tiles_m * tiles_n;
  const unsigned entry = blockIdx.x / tiles;
  unsigned t = blockIdx.x - entry * tiles;
  if (tiles % 8 == 0)
    t = (t % 8) * (tiles / 8) + t / 8;
  const unsigned band = t / (8 * tiles_n);
  const unsigned band_rows = tiles_m - 8 * band < 8 ? tiles_m - 8 * band : 8;
  const unsigned in_band = t - band * 8 * tiles_n;
  const unsigned tn = in_band / band_rows;
  const unsigned tm = 8 * band + in_band - tn * band_rows;

  const float *const a_base =
      (a_ptrs != nullptr ? a_ptrs[entry] : A + entry * stride_a) +
      static_cast<long long>(tm * S::BM) * lda;
  const float *const b_base =
      (b_ptrs != nullptr ? b_ptrs[entry] : B + entry * stride_b) +
      static_cast<long long>(tn * S::BN) * ldb;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wm = wave % 2, wn = wave / 2;

  using FragA =
      tcec::fragment<w::matrix_a, S::WM, S::WN, S::WK, T, w::row_major, Policy>;
  using FragB =
      tcec::fragment<w::matrix_b, S::WM, S::WN, S::WK, T, w::col_major, Policy>;
  using FragC =
      tcec::fragment<w::accumulator, S::WM, S::WN, S::WK, T, void, Policy>;
  FragC fc;
  tcec::fill_zero(fc);
  const auto mma = [](FragC &d, const FragA &a, const FragB &b) {
    if constexpr (ROUNDING == 1)
      tcec::mma_rn_sync(d, a, b, d);
    else if constexpr (ROUNDING == 2)
      tcec::mma_rz_sync(d, a, b, d);
    else
      tcec::mma_sync(d, a, b, d);
  };

  auto stage_in = [&](const int stage, const int k0) {
    float *const sa = smem + stage * S::STAGE_FLOATS;
    float *const sb = sa + S::BM * S::LD;
    stage_tile<S::BM, S::SK, S::THREADS>(sa, a_base + k0, lda);
    stage_tile<S::BN, S::SK, S::THREADS>(sb, b_base + k0, ldb);
    // (no cp_async::commit(): the loop waits with wait_all(), which needs no
    // groups, and commit() costs a round trip to its bookkeeping in LDS)
  };

  stage_in(0, 0);
  cpa::wait_all();
  __syncthreads();

  int stage = 0;
  for (int k0 = 0; k0 < k; k0 += S::SK) {
    if (k0 + S::SK < k)
      stage_in(1 - stage, k0 + S::SK);

    const float *const sa =
        static_cast<const float *>(__builtin_assume_aligned(
            smem + stage * S::STAGE_FLOATS + wm * S::WM * S::LD, 16));
    const float *const sb =
        static_cast<const float *>(__builtin_assume_aligned(
            smem + stage * S::STAGE_FLOATS + (S::BM + wn * S::WN) * S::LD, 16));
    // fragments double buffered over the k steps of the stage
    FragA fa[2];
    FragB fb[2];
    tcec::load_matrix_sync<tcec::row_major_swizzled>(fa[0], sa, S::LD, false);
    tcec::load_matrix_sync<tcec::col_major_swizzled>(fb[0], sb, S::LD, false);
#pragma unroll
    for (int kk = S::WK; kk < S::SK; kk += S::WK) {
      const int cur = (kk / S::WK) & 1;
      tcec::load_matrix_sync<tcec::row_major_swizzled>(fa[cur], sa + kk, S::LD,
                                                       false);
      tcec::load_matrix_sync<tcec::col_major_swizzled>(fb[cur], sb + kk, S::LD,
                                                       false);
      mma(fc, fa[1 - cur], fb[1 - cur]);
    }
    constexpr int last = ((S::SK / S::WK) - 1) & 1;
    mma(fc, fa[last], fb[last]);

    cpa::wait_all();
    __syncthreads();
    stage = 1 - stage;
  }

  float *const cw = (c_ptrs != nullptr ? c_ptrs[entry] : C + entry * stride_c) +
                    (tm * S::BM + wm * S::WM) +
                    static_cast<long long>(tn * S::BN + wn * S::WN) * ldc;
  if (beta == 0.f) {
    tcec::store_matrix_sync_with_mul<w::col_major>(cw, fc, ldc, alpha);
  } else {
    FragC fin;
    tcec::load_matrix_sync(fin, cw, ldc, w::mem_col_major);
    fc.integrate();
#pragma unroll
    for (unsigned i = 0; i < fc.num_elements; i++) // (the roundings written out)
      fc.x(i) = __builtin_fmaf(alpha, fc.x(i), beta * fin.x(i));
    tcec::store_matrix_sync(cw, fc, ldc, w::mem_col_major);
  }
}

// The same product for operands of 16-bit terms: every element is split once per
// workgroup, not once per wave that needs it, and no fp32 tile passes through LDS.
// A wave loads its share of a stage's row blocks (16 rows of op(A) or columns of
// op(B), 32 of k) into registers a stage ahead, splits them (split4, what
// load_matrix_sync splits with) and puts the terms into LDS where the lanes of a
// 16x16x32 fragment find theirs 16 bytes at a time; the waves fill the registers
// of their tcec:: fragments from there.  With a conversion per wave the kernel was
// bound by its instruction issue (1.66e8 vector instructions beside 2.5e7 matrix
// ones at 4096^3) and, on few tiles, by its own chain of copy, split and multiply.
// Two fp16 terms, before -> now, calls of both in turn: 4096^3 504 -> 439 us (a
// hundred of one in a row 505 -> 455 to 470), 1152x2816x7008 254 -> 180,
// 1920x1920x1024 43.8 -> 32.4, 256x256x8192 288 -> 133, 768x384x352 17.5 -> 7.7;
// three bf16 terms 4096^3 725 -> 691, 768x384x352 23.9 -> 10.0; one term
// 2944x3456x608 41.0 -> 30.8.  What bounds it now: conversions, the adds of
// mma_rn_sync and matrix instructions share a SIMD's one or two waves, and the
// terms' 8-byte writes conflict (28 % of the LDS cycles at 4096^3).  Loads of
// eight lanes to a row's 128 bytes: with a lane's eight k in two loads of its own
// the rows' requests ran at 9.5 TB/s, half the rate.
//   BM  : block tile (64 or 128), 2 x WGN waves
template <class T, class Policy, int BM_, int WGN> struct ApiSplitShape {
  static constexpr int BM = BM_, SK = 32, WM = BM / 2, WN = BM / WGN;
  static constexpr int NW = 2 * WGN, THREADS = 64 * NW;
  static constexpr int BLOCKS = 2 * BM / 16; // row blocks of a stage, A's first
  static constexpr int PER_WAVE = BLOCKS / NW;
  static constexpr int TERMS =
      tcec::fragment<w::matrix_a, 16, 16, SK, T, w::row_major, Policy>::num_terms;
  static constexpr int STAGE_BYTES = BLOCKS * TERMS * 1024;
  static constexpr int LDS_BYTES = 2 * STAGE_BYTES;
  static_assert(LDS_BYTES <= (NW > 4 ? 160 : 80) * 1024,
                "two stages, of two workgroups a compute unit with four waves");
};

template <class T, class Policy, class S, int ROUNDING>
__global__ void __launch_bounds__(S::THREADS, S::BM > 64 ? 2 : 3)
    tcec_api_gemm_split_kernel(const int m, const int n, const int k,
                               const float alpha, const float *const A,
                               const float *const *const a_ptrs, const int lda,
                               const long long stride_a, const float *const B,
                               const float *const *const b_ptrs, const int ldb,
                               const long long stride_b, const float beta,
                               float *const C, float *const *const c_ptrs,
                               const int ldc, const long long stride_c) {
  constexpr int BM = S::BM, WGN = S::NW / 2;
  extern __shared__ __attribute__((aligned(1024))) unsigned char terms_lds[];

  const unsigned tiles_m = m / BM, tiles_n = n / BM;
  const unsigned tiles = tiles_m * tiles_n;
  const unsigned entry = blockIdx.x / tiles;
  unsigned t = blockIdx.x - entry * tiles;
  if (tiles % 8 == 0)
    t = (t % 8) * (tiles / 8) + t / 8;
  const unsigned band = t / (8 * tiles_n);
  const unsigned band_rows = tiles_m - 8 * band < 8 ? tiles_m - 8 * band : 8;
  const unsigned in_band = t - band * 8 * tiles_n;
  const unsigned tn = in_band / band_rows;
  const unsigned tm = 8 * band + in_band - tn * band_rows;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wm = wave % 2, wn = wave / 2;
  const unsigned lane = threadIdx.x & 63u;

  using FragA =
      tcec::fragment<w::matrix_a, S::WM, S::WN, S::SK, T, w::row_major, Policy>;
  using FragB =
      tcec::fragment<w::matrix_b, S::WM, S::WN, S::SK, T, w::col_major, Policy>;
  using FragC =
      tcec::fragment<w::accumulator, S::WM, S::WN, S::SK, T, void, Policy>;
  FragC fc;
  tcec::fill_zero(fc);
  const auto mma = [](FragC &d, const FragA &a, const FragB &b) {
    if constexpr (ROUNDING == 1)
      tcec::mma_rn_sync(d, a, b, d);
    else if constexpr (ROUNDING == 2)
      tcec::mma_rz_sync(d, a, b, d);
    else
      tcec::mma_sync(d, a, b, d);
  };

  // this wave's row blocks: the first half of the waves takes A's, the others B's
  // (a lane's registers of a matrix_b fragment are those of a matrix_a fragment
  // with rows and columns exchanged)
  const bool is_a = wave < WGN;
  const int ld = is_a ? lda : ldb;
  const float *src =
      (is_a ? (a_ptrs != nullptr ? a_ptrs[entry] : A + entry * stride_a) +
                  static_cast<long long>(tm * BM) * lda
            : (b_ptrs != nullptr ? b_ptrs[entry] : B + entry * stride_b) +
                  static_cast<long long>(tn * BM) * ldb) +
      static_cast<long long>(wave % WGN) * (S::PER_WAVE * 16) * ld;

  // Load h of a row block takes its rows 8h .. 8h+7, eight lanes to a row's 128
  // bytes: four k, half of what a lane of a 16x16x32 operand holds.
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  f32x4 raw[S::PER_WAVE][2];
  src += static_cast<long long>(lane >> 3) * ld + 4 * (lane & 7u);
  const auto load_raw = [&]() {
#pragma unroll
    for (int p = 0; p < S::PER_WAVE; p++)
#pragma unroll
      for (int h = 0; h < 2; h++)
        raw[p][h] = *static_cast<const f32x4 *>(__builtin_assume_aligned(
            src + static_cast<long long>(16 * p + 8 * h) * ld, 16));
  };
  // 16-byte slot of (row r, k group q) in a chunk of 16 rows x 32 k of one term:
  // 16 q + (r ^ spread(q)), so that the lanes of a write that hold the same row do
  // not share their banks
  const auto spread = [](const unsigned q) { return 12u * (q & 1u) ^ 4u * (q >> 1); };
  const unsigned read_off =
      16u * ((lane & 48u) + ((lane & 15u) ^ spread(lane >> 4)));
  unsigned write_off[2];
#pragma unroll
  for (unsigned h = 0; h < 2; h++) {
    const unsigned q = (lane & 7u) >> 1, r = 8u * h + (lane >> 3);
    write_off[h] = 16u * (16u * q + (r ^ spread(q))) + 8u * (lane & 1u);
  }
  const auto chunk = [&](const int stage, const int block, const int term) {
    return terms_lds + stage * S::STAGE_BYTES +
           (block * S::TERMS + term) * 1024;
  };
  const auto get = [&](auto &sub, const unsigned char *const from) {
    static_assert(sizeof(sub.x) == 16, "eight 16-bit values a lane");
    __builtin_memcpy(sub.x, __builtin_assume_aligned(from + read_off, 16), 16);
  };
  const auto put_terms = [&](const int stage) {
    using E = typename tcec::detail::split_traits<T>::storage;
#pragma unroll
    for (int p = 0; p < S::PER_WAVE; p++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        E term[3][4];
        tcec::detail::split4<T>(raw[p][h], term[0], term[1], term[2]);
#pragma unroll
        for (int x = 0; x < S::TERMS; x++)
          __builtin_memcpy(__builtin_assume_aligned(
                               chunk(stage, wave * S::PER_WAVE + p, x) +
                                   write_off[h], 8),
                           term[x], 8);
      }
  };
  const auto get_frag = [&](auto &f, const int stage, const int block0) {
#pragma unroll
    for (int i = 0; i < std::remove_reference_t<decltype(f)>::num_sub_frags; i++) {
      get(f.sub_frag[i], chunk(stage, block0 + i, 0));
      if constexpr (S::TERMS >= 2)
        get(f.sub_d_frag[i], chunk(stage, block0 + i, 1));
      if constexpr (S::TERMS >= 3)
        get(f.sub_d2_frag[i], chunk(stage, block0 + i, 2));
    }
  };

  load_raw();
  put_terms(0);
  src += k > S::SK ? S::SK : 0;
  load_raw();
  __syncthreads();
  int stage = 0;
  for (int k0 = S::SK; k0 < k; k0 += S::SK) {
    FragA fa;
    FragB fb;
    get_frag(fa, stage, wm * (S::WM / 16));
    get_frag(fb, stage, S::BM / 16 + wn * (S::WN / 16));
    stage = 1 - stage;
    put_terms(stage);
    // (the last one again where there is no other, never used)
    src += k0 + S::SK < k ? S::SK : 0;
    load_raw();
    mma(fc, fa, fb);
    // a stage's vector instructions go between its matrix instructions, two after
    // each (three fp16 products, eight waves a tile: 1152x2816x7008 206 -> 180 us,
    // 4096^3 496 -> 465; three or more after each 1 to 13 % slower, and one
    // product is better left to the compiler)
    if constexpr (S::TERMS >= 2) {
#pragma unroll
      for (int i = 0; i < 48; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
      }
    }
    __syncthreads();
  }
  {
    FragA fa;
    FragB fb;
    get_frag(fa, stage, wm * (S::WM / 16));
    get_frag(fb, stage, S::BM / 16 + wn * (S::WN / 16));
    mma(fc, fa, fb);
  }

  float *const cw = (c_ptrs != nullptr ? c_ptrs[entry] : C + entry * stride_c) +
                    (tm * BM + wm * S::WM) +
                    static_cast<long long>(tn * BM + wn * S::WN) * ldc;
  if (beta == 0.f) {
    tcec::store_matrix_sync_with_mul<w::col_major>(cw, fc, ldc, alpha);
  } else {
    FragC fin;
    tcec::load_matrix_sync(fin, cw, ldc, w::mem_col_major);
    fc.integrate();
#pragma unroll
    for (unsigned i = 0; i < fc.num_elements; i++) // (the roundings written out)
      fc.x(i) = __builtin_fmaf(alpha, fc.x(i), beta * fin.x(i));
    tcec::store_matrix_sync(cw, fc, ldc, w::mem_col_major);
  }
}

} // namespace wmmae_harness
