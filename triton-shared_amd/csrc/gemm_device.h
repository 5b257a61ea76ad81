// Device code of the 16-bit and fp32 matrix-product kernels, in a header of its own because it is compiled twice: ahead of
// time into the library (kernels_gemm.hip, results stored as they are), and at run time with hipRTC when the Triton
// kernel applies elementwise ops to the accumulator before the store (a fused activation): the generated source
// defines TTS_GEMM_RTC (which kernel: 0 whole 256 x 256 x 32 tiles, 1 any shape in 128 x 128 x 64 tiles, 2 the sum of the K
// slices, 3 as 1 in 64 x 128 x 64 tiles, 4 ... 6 the other direct-to-LDS tiles, 7 ... 10 fp32 operands in four tilings), TTS_GEMM_BF16 and the functor TtsEp (a plain struct, passed as the kernel's last argument) that maps an accumulator value and its position to the value stored, then this file's text.  Nothing here may need a host header.
#pragma once
#ifdef __HIPCC_RTC__
typedef __INT64_TYPE__ int64_t;
typedef __UINT64_TYPE__ uint64_t;
typedef __UINT32_TYPE__ uint32_t;
typedef __UINT16_TYPE__ uint16_t;
typedef __UINTPTR_TYPE__ uintptr_t;
#else
#include <hip/hip_runtime.h>

#include <cstdint>
#endif

// C[M,N] = A[M,K] * B[K,N], 16-bit (or fp32) operands, fp32 accumulate; C is row-major, A and B row- or column-major
struct TtsGemmParams {
  const void *a, *b;
  void *c;
  int64_t M, N, K;
  int64_t lda, ldb, ldc;  // pitches in elements; the other stride of each matrix is 1
  int is_bf16;
  int a_trans, b_trans;   // A / B is column-major: element (m, k) of A is a[m + k * lda], (k, n) of B is b[k + n * ldb]
  // Gathered operands (null / 0 for a plain product): row m of A is row a_rows[m] of the matrix at `a` (row-major A only);
  // the rows of block m / b_block_rows multiply the matrix at b + b_block[m / b_block_rows] * b_block_stride elements,
  // or nothing at all when that id is negative (their part of C is not written).
  const int *a_rows;
  const int *b_block;
  int64_t b_block_stride;
  int b_block_rows;
  int gather_mul32;       // bit 0: a_rows[m] * lda, bit 1: id * b_block_stride is a 32-bit product that wraps, as the source computes it
  int is_f32;             // fp32 operands and result (kernels_gemm.hip: gemm_f32_kernel); is_bf16 is then 0
  // K in `split` slices, one workgroup per (tile, slice), for products with too few tiles to occupy the chip: slice s
  // leaves its fp32 sums at partial[s * M * N + m * N + n], and a second kernel adds the slices and narrows (1 = none)
  int split;
  float *partial;
  int meet;               // 1: slices may meet in the kernel (slices_meet), which counts their arrivals in
  int *counters;          // ... counters, 32 ints apart, zero between launches
  // A batch of products of one shape (grid.y of the launch = batches): batch b reads a + b * batch_a and b + b * batch_b
  // and writes c + b * batch_c (in elements); 1 / 0 for a single product
  int batches;
  int64_t batch_a, batch_b, batch_c;
};

namespace tts_gemm_device {
typedef TtsGemmParams GemmParams;

// the product of batch blockIdx.y of a launch (esize: bytes per element of the operands and of C)
__device__ __forceinline__ GemmParams of_batch(const GemmParams &p, int esize) {
  GemmParams q = p;
  const int64_t by = blockIdx.y;
  q.a = (const char *)p.a + by * p.batch_a * esize;
  q.b = (const char *)p.b + by * p.batch_b * esize;
  q.c = (char *)p.c + by * p.batch_c * esize;
  if (p.partial) q.partial = p.partial + by * (int64_t)p.split * p.M * p.N;
  return q;
}

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(2 * sizeof(_Float16)))) _Float16 f16x2;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

__device__ __forceinline__ uint16_t f32_to_bf16(float f) {  // round to nearest even
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ uint16_t f32_to_f16(float f) {
  _Float16 h = (_Float16)f;
  uint16_t r;
  __builtin_memcpy(&r, &h, 2);
  return r;
}

template <bool BF16>
__device__ __forceinline__ f32x16 mfma32(uint4 a, uint4 b, f32x16 c) {
  if (BF16) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// 8 consecutive 16-bit elements starting at p[0], zero beyond `valid`
__device__ __forceinline__ uint4 load8(const uint16_t *p, int valid, bool vec) {
  if (valid >= 8 && vec) return *reinterpret_cast<const uint4 *>(p);
  uint32_t w[4] = {0, 0, 0, 0};
  for (int i = 0; i < 8 && i < valid; i++) w[i >> 1] |= (uint32_t)p[i] << (16 * (i & 1));
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// eight elements without their first k (1 .. 7), moved to the front
__device__ __forceinline__ uint4 without_first(uint4 v, int k) {
  if (k & 4) v = make_uint4(v.z, v.w, 0, 0);
  if (k & 2) v = make_uint4(v.y, v.z, v.w, 0);
  if (k & 1) v = make_uint4(v.x >> 16 | v.y << 16, v.y >> 16 | v.z << 16, v.z >> 16 | v.w << 16, v.w >> 16);
  return v;
}

// ------------------------------------------------------------- 16-bit GEMM
// The kernel for any shape, any alignment, and operands that are row- or column-major.
// Workgroup: 256 threads = 2 x 2 wavefronts; each wavefront owns TM x TN MFMA tiles of 32 x 32.  An operand tile is
// R = BM or BN rows (rows of A, columns of B) by BK values of k and is staged through LDS (two buffers) in the form it
// has in memory, with 16-byte loads and stores:
//   k contiguous (A row-major, B column-major): LDS [r][k], pitch BK + 8 elements; a lane's MFMA operand (8 consecutive
//     k of row lane % 32) is one 16-byte read, and 32 consecutive rows hit distinct banks;
//   r contiguous (B row-major, A column-major): LDS [k][r], pitch R + 16 elements; `ds_read_b64_tr_b16` transposes on
//     the way out -- within 16 lanes, lane i receives element i % 4 of the 8-byte rows addressed by lanes i / 4,
//     i / 4 + 4, i / 4 + 8, i / 4 + 12, so lane j of a group addresses k row j / 4, elements 4 (j % 4) .. +3 of the
//     group's 16, and two reads (k 0-3, k 4-7) make one operand.
// What bounds it on ragged sizes is the way of the operands from memory: a chain of one load per K tile where a shape gives the
// chip less than one workgroup per CU, else the rate at which a CU takes 16-byte loads that are not 16-byte aligned.  Chunks are
// 16-byte loads at any alignment (global memory takes them at element addresses), untested, and two tiles are in flight.
// 1000 x 3001 x 1003 fp16 with a fused activation: 22 us, 26 from HBM (163 with two-byte loads, each behind a test, and 30 while only the last
// K tiles were loaded that way); TM, TN: 128 x 128 tiles or, for few of them, 64 x 128 (kernels_gemm.hip: any_rows).
// Rows of A may be taken through an index vector (p.a_rows) and the base of B may depend on the block of rows
// (p.b_block): a mixture-of-experts product is this kernel with both set.
// `ep(acc, row, col)` maps an accumulator value to the value that is stored at (row, col) of C (the identity for a plain
// product); it is only called for elements inside the problem.
template <bool V>
struct BoolConstant {
  static constexpr bool value = V;
};

template <int ROWS, int CHUNKS>  // an operand's tile: its rows, and how many 16-byte chunks of it a thread moves
struct TileOf {
  static constexpr int R = ROWS, N = CHUNKS;
};

template <int BM, int BN, int BK>
struct GemmStageLds {
  static constexpr int A_ELEMS = (BM * (BK + 8) > BK * (BM + 16)) ? BM * (BK + 8) : BK * (BM + 16);
  static constexpr int B_ELEMS = (BN * (BK + 8) > BK * (BN + 16)) ? BN * (BK + 8) : BK * (BN + 16);
  static constexpr int BUFFER_ELEMS = A_ELEMS + B_ELEMS;
  static constexpr int BYTES = 2 * BUFFER_ELEMS * 2;
};

//
// SK: the grid holds p.split workgroups per tile; workgroup (tile, s) walks the s-th share of the K tiles and leaves its fp32
// sums in p.partial (gemm_splitk_reduce_body adds them and applies the functor).
template <bool BF16, int TM, int TN, int BK, class Ep, bool SK = false>
__device__ __forceinline__ void gemm_mfma_body(const GemmParams &p, int tiles_m, int tiles_n, const Ep &ep) {
  constexpr int BM = 2 * TM * 32, BN = 2 * TN * 32;
  constexpr int PK = BK + 8;  // pitch of a k-contiguous tile (an r-contiguous one of R rows: R + 16)
  constexpr int CA = BM * BK / 8 / 256, CB = BN * BK / 8 / 256;  // 16-byte chunks of an operand tile per thread
  using Lds = GemmStageLds<BM, BN, BK>;
#ifdef TTS_GEMM_RTC
  __shared__ __align__(16) uint16_t smem[2 * Lds::BUFFER_ELEMS];
#else
  extern __shared__ __align__(16) uint16_t smem[];
#endif
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  // workgroup -> output tile: consecutive ids share an XCD's L2 (ids are dealt
  // round-robin to the 8 XCDs), and within an XCD walk 8-tile-tall column groups
  int bid = blockIdx.x;
  const int nwg = tiles_m * tiles_n;
  const int slice = SK ? bid / nwg : 0;
  if (SK) bid -= slice * nwg;
  if (nwg % 8 == 0) bid = (bid % 8) * (nwg / 8) + bid / 8;
  const int group = 8 * tiles_n;
  const int g0 = (bid / group) * 8;
  const int gh = min(tiles_m - g0, 8);
  const int tile_m = g0 + (bid % group) % gh, tile_n = (bid % group) / gh;
  const int64_t m0 = (int64_t)tile_m * BM, n0 = (int64_t)tile_n * BN;

  const uint16_t *__restrict__ A = (const uint16_t *)p.a;
  const uint16_t *__restrict__ B = (const uint16_t *)p.b;
  if (p.b_block) {  // the rows of this tile multiply a matrix of their own; a negative id: nothing to do for them
    const int which = p.b_block[m0 / p.b_block_rows];
    if (which < 0) return;
    B += (p.gather_mul32 & 2) ? (int64_t)(int)((uint32_t)which * (uint32_t)p.b_block_stride) : (int64_t)which * p.b_block_stride;
  }
  const bool a_vec = (p.lda % 8 == 0) && (((uintptr_t)A & 15) == 0);
  const bool b_vec = (p.ldb % 8 == 0) && (((uintptr_t)B & 15) == 0);
  const int K = (int)p.K;

  // where this thread's chunks of the tiles are: (row, k chunk) of a k-contiguous tile, (k, row chunk) of an
  // r-contiguous one; element offsets of the chunks' rows in memory (-1: outside the problem)
  int64_t a_at[CA], b_at[CB];
#pragma unroll
  for (int j = 0; j < CA; j++) {
    const int c = tid + 256 * j;
    if (p.a_trans) {
      a_at[j] = m0 + (c % (BM / 8)) * 8;  // first of 8 rows; the k row moves with the loop
    } else {
      const int64_t gr = m0 + c / (BK / 8);
      if (gr >= p.M) a_at[j] = -1;
      else if (!p.a_rows) a_at[j] = gr * p.lda;
      else a_at[j] = (p.gather_mul32 & 1) ? (int64_t)(int)((uint32_t)p.a_rows[gr] * (uint32_t)p.lda) : (int64_t)p.a_rows[gr] * p.lda;
    }
  }
#pragma unroll
  for (int j = 0; j < CB; j++) {
    const int c = tid + 256 * j;
    if (p.b_trans) {
      const int64_t gn = n0 + c / (BK / 8);
      b_at[j] = gn < p.N ? gn * p.ldb : -1;
    } else {
      b_at[j] = n0 + (c % (BN / 8)) * 8;
    }
  }
  auto load_operand = [&](auto of, auto &reg, const uint16_t *P, bool r_contiguous, const auto &at, int64_t ld, int64_t rows, bool vec, int k0) {
    constexpr int R = decltype(of)::R, N = decltype(of)::N;
#pragma unroll
    for (int j = 0; j < N; j++) {
      const int c = tid + 256 * j;
      if (r_contiguous) {
        const int gk = k0 + c / (R / 8);
        const int valid = (int)min((int64_t)8, rows - at[j]);
        reg[j] = (gk < K && valid > 0) ? load8(P + (int64_t)gk * ld + at[j], valid, vec) : make_uint4(0, 0, 0, 0);
      } else {
        const int gk = k0 + (c % (BK / 8)) * 8;
        reg[j] = at[j] >= 0 ? load8(P + at[j] + gk, K - gk, vec) : make_uint4(0, 0, 0, 0);
      }
    }
  };
  auto store_operand = [&](auto of, const auto &reg, uint16_t *S, bool r_contiguous) {
    constexpr int R = decltype(of)::R, N = decltype(of)::N;
#pragma unroll
    for (int j = 0; j < N; j++) {
      const int c = tid + 256 * j;
      if (r_contiguous) *reinterpret_cast<uint4 *>(S + (c / (R / 8)) * (R + 16) + (c % (R / 8)) * 8) = reg[j];
      else *reinterpret_cast<uint4 *>(S + (c / (BK / 8)) * PK + (c % (BK / 8)) * 8) = reg[j];
    }
  };
  // a lane's MFMA operand for the 32 rows starting at `row0` of a staged tile, k = ks * 16 + 8 (lane / 32) .. +7
  auto fragment = [&](auto of, const uint16_t *S, bool r_contiguous, int row0, int ks) -> uint4 {
    constexpr int R = decltype(of)::R;
    constexpr int PR = R + 16;
    if (!r_contiguous) return *reinterpret_cast<const uint4 *>(S + (row0 + (lane & 31)) * PK + ks * 16 + 8 * (lane >> 5));
    const int g = lane >> 4, j = lane & 15;
    const uint16_t *at = S + (ks * 16 + 8 * (g >> 1) + (j >> 2)) * PR + row0 + 16 * (g & 1) + 4 * (j & 3);
    typedef short s16x4_t __attribute__((ext_vector_type(4)));
    const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3))) *)((__attribute__((address_space(3))) void *)at));
    const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3))) *)((__attribute__((address_space(3))) void *)(at + 4 * PR)));
    const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
    return make_uint4(l2.x, l2.y, h2.x, h2.y);
  };
  const TileOf<BM, CA> of_a;
  const TileOf<BN, CB> of_b;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

  // The forms of the two operands are fixed for the launch: the loop is compiled once per combination, so that inside
  // it the loads, the LDS traffic and the MFMAs are straight-line code the compiler can overlap.
  const int nk_all = (K + BK - 1) / BK;
  const int k_begin = SK ? (int)((int64_t)slice * nk_all / p.split) : 0;
  const int nk = SK ? (int)((int64_t)(slice + 1) * nk_all / p.split) : nk_all;  // K tiles [k_begin, nk) are this workgroup's
  auto sweep_k = [&](auto a_form, auto b_form) {
    constexpr bool a_r = decltype(a_form)::value, b_r = decltype(b_form)::value;  // r-contiguous in memory and in LDS
    // Chunks are loaded without a test, at any alignment.  Rows (columns) beyond the problem are replaced by others, they only
    // reach results nobody stores; a chunk that starts inside a row of an r-contiguous operand and ends behind it reads into
    // the next row.  K tiles [0, nwide) have no chunk that reads past the operand that way.
    int nwide = K / BK;
    if (K % BK == 0 && ((a_r && m0 + BM > p.M) || (b_r && n0 + BN > p.N))) nwide = nk_all - 1;
    nwide = min(nwide, nk);
    // a row beyond the problem: the tile's first, or where rows are gathered the operand's first (store_tiles clears them)
    const int64_t a_first = a_r || p.a_rows ? 0 : m0 * p.lda, b_first = n0 * p.ldb;
    auto first_chunk = [&](auto of, auto &ptr, const uint16_t *P, bool r_contiguous, const auto &at, int64_t other, int64_t ld, int64_t rows) {
      constexpr int R = decltype(of)::R, N = decltype(of)::N;
#pragma unroll
      for (int j = 0; j < N; j++) {
        const int c = tid + 256 * j;
        ptr[j] = r_contiguous ? P + (c / (R / 8)) * ld + (at[j] < rows ? at[j] : 0) : P + (at[j] >= 0 ? at[j] : other) + (c % (BK / 8)) * 8;
      }
    };
    const uint16_t *a_ptr[CA], *b_ptr[CB];
    first_chunk(of_a, a_ptr, A, a_r, a_at, a_first, p.lda, p.M);
    first_chunk(of_b, b_ptr, B, b_r, b_at, b_first, p.ldb, p.N);
    struct Tiles { uint4 a[CA], b[CB]; };
    auto load_wide = [&](Tiles &t, int kt) {
      const int64_t a_k = a_r ? (int64_t)kt * BK * p.lda : (int64_t)kt * BK, b_k = b_r ? (int64_t)kt * BK * p.ldb : (int64_t)kt * BK;
#pragma unroll
      for (int j = 0; j < CA; j++) __builtin_memcpy(&t.a[j], a_ptr[j] + a_k, 16);
#pragma unroll
      for (int j = 0; j < CB; j++) __builtin_memcpy(&t.b[j], b_ptr[j] + b_k, 16);
    };
    // Any K tile, the one that ends the K loop included: there a chunk that sticks out of its row (k contiguous) or of the last k
    // row (r contiguous) is read from the last eight elements and put right when it is stored to LDS, chunks past K become
    // zeros.  Tiles past the last load it again, so that the loop's tail has no branch around a load either: at one, the
    // compiler waits for every load in flight.  (Element by element behind tests, and with branches, the last tiles took a
    // third of 1000 x 3001 x 1003 and of the slices of 600 x 601 x 3001.)
    auto load_tail = [&](auto of, auto &reg, const uint16_t *P, bool r_contiguous, const auto &at, int64_t other, int64_t ld, int64_t rows, int kt) {
      constexpr int R = decltype(of)::R, N = decltype(of)::N;
#pragma unroll
      for (int j = 0; j < N; j++) {
        const int c = tid + 256 * j;
        const uint16_t *src;
        if (r_contiguous) {
          const int row = min(kt * BK + c / (R / 8), K - 1);
          src = P + (int64_t)row * ld + (row == K - 1 ? min(at[j], rows - 8) : at[j] < rows ? at[j] : 0);
        } else {
          src = P + (at[j] >= 0 ? at[j] : other) + min(kt * BK + (c % (BK / 8)) * 8, K - 8);
        }
        __builtin_memcpy(&reg[j], src, 16);
      }
    };
    auto settle_tail = [&](auto of, auto &reg, bool r_contiguous, const auto &at, int64_t rows, int kt) {
      constexpr int R = decltype(of)::R, N = decltype(of)::N;
#pragma unroll
      for (int j = 0; j < N; j++) {
        const int c = tid + 256 * j;
        const int gk = kt * BK + (r_contiguous ? c / (R / 8) : (c % (BK / 8)) * 8);
        const int cut = !r_contiguous ? max(0, gk + 8 - K) : gk == K - 1 ? (int)max((int64_t)0, at[j] + 8 - rows) : 0;
        if (gk >= K) reg[j] = make_uint4(0, 0, 0, 0);
        else if (cut > 0 && cut < 8) reg[j] = without_first(reg[j], cut);
      }
    };
    auto load_any = [&](Tiles &t, int kt) {
      kt = min(kt, nk - 1);
      load_tail(of_a, t.a, A, a_r, a_at, a_first, p.lda, p.M, kt);
      load_tail(of_b, t.b, B, b_r, b_at, b_first, p.ldb, p.N, kt);
    };
    auto store_tiles = [&](Tiles &t, int buf, bool last) {
      if (last) {
        settle_tail(of_a, t.a, a_r, a_at, p.M, nk_all - 1);
        settle_tail(of_b, t.b, b_r, b_at, p.N, nk_all - 1);
      }
      uint16_t *As = smem + buf * Lds::BUFFER_ELEMS, *Bs = As + Lds::A_ELEMS;
      uint4 a[CA];
#pragma unroll
      for (int j = 0; j < CA; j++) a[j] = a_r || a_at[j] >= 0 ? t.a[j] : make_uint4(0, 0, 0, 0);
      store_operand(of_a, a, As, a_r);
      store_operand(of_b, t.b, Bs, b_r);
    };
    auto multiply = [&](int buf) {
      const uint16_t *As = smem + buf * Lds::BUFFER_ELEMS, *Bs = As + Lds::A_ELEMS;
#pragma unroll
      for (int ks = 0; ks < BK / 16; ks++) {
        uint4 af[TM], bf[TN];
#pragma unroll
        for (int i = 0; i < TM; i++) af[i] = fragment(of_a, As, a_r, wm * TM * 32 + i * 32, ks);
#pragma unroll
        for (int j = 0; j < TN; j++) bf[j] = fragment(of_b, Bs, b_r, wn * TN * 32 + j * 32, ks);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++) acc[i][j] = mfma32<BF16>(af[i], bf[j], acc[i][j]);
      }
    };
    Tiles even, odd;
    // Products of fewer than eight rows, columns or k have no eight elements to read: a tile at a time, chunks element by element.
    if (K < 8 || (a_r && (p.M < 8 || p.lda < 8)) || (b_r && (p.N < 8 || p.ldb < 8))) {
      for (int kt = k_begin; kt < nk; kt++) {
        load_operand(of_a, even.a, A, a_r, a_at, p.lda, p.M, a_vec, kt * BK);
        load_operand(of_b, even.b, B, b_r, b_at, p.ldb, p.N, b_vec, kt * BK);
        store_tiles(even, 0, false);
        __syncthreads();
        multiply(0);
        __syncthreads();
      }
      return;
    }
    if (nk <= k_begin) return;
    // Two K tiles are in flight in registers beside the two in LDS: a tile's loads are issued two products before they are stored.
    load_any(even, k_begin);
    load_any(odd, k_begin + 1);
    store_tiles(even, 0, k_begin == nk_all - 1);
    load_any(even, k_begin + 2);
    __syncthreads();
    int kt = k_begin;
    for (; kt + 4 < nwide; kt += 2) {  // loads tiles kt + 3 and kt + 4
      multiply(0);
      store_tiles(odd, 1, false);
      load_wide(odd, kt + 3);
      __syncthreads();
      multiply(1);
      store_tiles(even, 0, false);
      load_wide(even, kt + 4);
      __syncthreads();
    }
    for (; kt < nk; kt += 2) {
      multiply(0);
      if (kt + 1 >= nk) break;
      store_tiles(odd, 1, kt + 1 == nk_all - 1);
      load_any(odd, kt + 3);
      __syncthreads();
      multiply(1);
      if (kt + 2 >= nk) break;
      store_tiles(even, 0, kt + 2 == nk_all - 1);
      load_any(even, kt + 4);
      __syncthreads();
    }
  };
  if (p.a_trans) {
    if (p.b_trans) sweep_k(BoolConstant<true>(), BoolConstant<false>());
    else sweep_k(BoolConstant<true>(), BoolConstant<true>());
  } else {
    if (p.b_trans) sweep_k(BoolConstant<false>(), BoolConstant<false>());
    else sweep_k(BoolConstant<false>(), BoolConstant<true>());
  }

  if constexpr (SK) {  // (a lane's place in each 32 x 32 tile: see below)
    float *__restrict__ part = p.partial + (int64_t)slice * p.M * p.N;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int64_t col = n0 + wn * TN * 32 + j * 32 + (lane & 31);
#pragma unroll
        for (int v = 0; v < 16; v++) {
          const int64_t row = m0 + wm * TM * 32 + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
          if (row < p.M && col < p.N) part[row * p.N + col] = acc[i][j][v];
        }
      }
    return;
  }
  // epilogue: lane holds column (lane % 32), rows 8*(v/4) + 4*(lane/32) + v%4 of each 32x32 tile
  uint16_t *__restrict__ C = (uint16_t *)p.c;
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) {
      int64_t col = n0 + wn * TN * 32 + j * 32 + (lane & 31);
#pragma unroll
      for (int v = 0; v < 16; v++) {
        int64_t row = m0 + wm * TM * 32 + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (row < p.M && col < p.N) C[row * p.ldc + col] = BF16 ? f32_to_bf16(ep(acc[i][j][v], row, col)) : f32_to_f16(ep(acc[i][j][v], row, col));
      }
    }
}

// Adds the K slices' partial sums in slice order, applies the functor and narrows: one element per thread, for any N.  A
// workgroup's 256 threads are `across` columns (a power of two) of 256 / across rows; the grid is blocks of columns, fastest,
// by groups of rows.
template <bool BF16, class Ep>
__device__ __forceinline__ void gemm_splitk_reduce_body(const GemmParams &p, int across, int col_blocks, const Ep &ep) {
  const int64_t row = (int64_t)(blockIdx.x / col_blocks) * (256 / across) + threadIdx.x / across;
  const int64_t col = (int64_t)(blockIdx.x % col_blocks) * across + threadIdx.x % across;
  if (row >= p.M || col >= p.N) return;
  const float *__restrict__ src = p.partial + row * p.N + col;
  float t = src[0];
#pragma unroll 4
  for (int sl = 1; sl < p.split; sl++) t += src[(int64_t)sl * p.M * p.N];
  const float v = ep(t, row, col);
  ((uint16_t *)p.c)[row * p.ldc + col] = BF16 ? f32_to_bf16(v) : f32_to_f16(v);
}

// ------------------------------------------- 16-bit GEMM, full-tile fast path
// For problems made of whole 256 x 256 x 32 tiles with 16-byte aligned rows.
//
// Workgroup: 256 threads = 4 wavefronts (one per SIMD), wave grid 2 x 2, each wavefront
// 128 x 128 of C = 4 x 4 MFMA tiles of 32 x 32 (256 accumulator registers).
//
// Global -> LDS without passing through registers: `global_load_lds_dwordx4` writes the 64
// lanes' 16-byte chunks to 1 KB of consecutive LDS, so the LDS layout is fixed by which global
// chunk each lane fetches.
//   A stage [256 rows][64 bytes]: position q of row r holds chunk q ^ ((r / 4) & 3) of the row's
//     four; 16-byte fragment reads of 16 consecutive rows then fall into 16 distinct slots.
//   B stage [32 k rows][512 bytes], as in memory (N contiguous): position q of row k holds chunk
//     q ^ ((k & 3) << 2).  The MFMA operand wants K contiguous per lane; `ds_read_b64_tr_b16` does
//     that transposition on the way out: within 16 lanes, lane i receives element i % 4 of the
//     8-byte rows addressed by lanes i / 4, i / 4 + 4, i / 4 + 8, i / 4 + 12.  Lane r of a group
//     therefore addresses k row r / 4, columns 4 (r % 4) .. +3 of the group's 16 columns, and
//     two reads (k 0-3, k 4-7) make one 8-element operand.
// Both layouts were checked on the device: no LDS bank conflicts (SQ_LDS_BANK_CONFLICT = 0).
//
// Pipeline: STAGES LDS stages of one K tile each.  An iteration has two phases of 16 MFMAs (the
// tile's two K halves).  Every MFMA is followed by one LDS read or one direct-to-LDS load, which
// the matrix pipe hides: phase A reads the operands of phase B, phase B those of the next
// tile's phase A; a quarter of the way through each phase one load of tile t+STAGES-1 goes out,
// into the stage of tile t-1, which every wavefront finished reading before the previous barrier.
// One barrier per tile, between the phases: it follows the wait that tells this wavefront its
// own loads of tile t+1 have landed.  Loads past the last tile fetch the last tile again, so the
// wait count is the same in every iteration.
//
// The direct-to-LDS load is issued from inline assembly: the compiler orders every later LDS
// read behind such a load with a full vmcnt wait (it cannot tell the stages apart), which
// would serialise the pipeline.  Its own counting of ordinary loads stays conservative.
constexpr int F_BK = 32;
// Tile geometry of the direct-to-LDS kernel: 2 x 2 wavefronts of TM x TN MFMA tiles each.
template <int TM, int TN>
struct DmaTile {
  static constexpr int BM = 2 * TM * 32, BN = 2 * TN * 32;
  static constexpr int A_BYTES = BM * F_BK * 2, B_ROW_BYTES = BN * 2, STAGE_BYTES = A_BYTES + F_BK * B_ROW_BYTES;
  static constexpr int A_DMA = BM / 64, B_DMA = BN / 64;  // direct-to-LDS instructions per wavefront and K tile
  static constexpr int DMA = A_DMA + B_DMA;
  // Four stages everywhere: 128 KB (256 x 256), 96 KB (128 x 256, 256 x 128: one workgroup per CU, which is what a
  // problem that gives fewer than one 256 x 256 tile per CU gets anyway), 64 KB (128 x 128: two per CU).  With three
  // stages the 128 x 256 tile measured 46.3 us on 4096 x 2048 x 2048 against 40.4 with four (five and six: no better).
  static constexpr int STAGES = 4;
  static constexpr int LDS_BYTES = STAGES * STAGE_BYTES;
};
constexpr int F_BM = DmaTile<4, 4>::BM, F_BN = DmaTile<4, 4>::BN, F_STAGES = DmaTile<4, 4>::STAGES;
constexpr int F_A_BYTES = DmaTile<4, 4>::A_BYTES, F_STAGE_BYTES = DmaTile<4, 4>::STAGE_BYTES;
typedef short s16x4 __attribute__((ext_vector_type(4)));
#define TTS_LDS(p) ((__attribute__((address_space(3))) void *)(p))

// 64 lanes' 16-byte chunks, each `voff` bytes behind a base address that all lanes share, to 1 KB of LDS at `lds`.  The load
// has to stand one instruction behind the write of m0, and five behind a vector instruction that wrote the base address (a
// v_readfirstlane); the compiler does not look inside and counts neither.  Copying the base with a scalar instruction, which
// itself waits for the vector one, is both.
__device__ __forceinline__ void load_to_lds(const char *sbase, uint32_t voff, uint32_t lds) {
  uint64_t base;
  asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0" : "=&s"(base) : "s"(lds), "v"(voff), "s"(sbase) : "memory", "m0");
}

// s_waitcnt immediate: vmcnt in bits 3:0 and 15:14, expcnt (not waited for) in 6:4, lgkmcnt in 11:8
constexpr int waitcnt_imm(int vm, int lgkm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8); }

// The K slices of a tile become one without a second kernel: every workgroup leaves its sums in p.partial as its lanes hold them
// (written through: sc1), and the one that arrives last adds all of them in slice order into `acc` -- as the kernel that adds
// slices does, bit for bit -- and stores the tile.  false: this workgroup is done.  Nobody waits for anybody.  Bound by what one
// CU reads of others' sums, about 2.4 us per slice of 64 KiB with the trip through memory, where the second kernel has a launch
// and the whole chip: 1024 x 1024 x 1792 17.6 -> 14.7 us, 256 x 512 x 1600 14.6 -> 12.0.
template <int TM, int TN>
__device__ __forceinline__ bool slices_meet(const GemmParams &p, f32x16 (&acc)[TM][TN], int slice, int tile, int tiles, int wave, int lane) {
  typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
  constexpr int Q = TM * TN * 4;  // 16-byte pieces of a lane
  __shared__ int arrived;
  float *const slot = p.partial + ((int64_t)tile * 4 + wave) * (Q * 256);
  auto place = [&](int s) { return __builtin_amdgcn_make_buffer_rsrc(slot + (int64_t)s * tiles * (4 * Q * 256), 0, 0x7fffffff, 0x00027000); };
  {
    const auto own = place(slice);
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const f32x16 &a = acc[q / 4 / TN][q / 4 % TN];
      const f32x4 v = {a[4 * (q % 4)], a[4 * (q % 4) + 1], a[4 * (q % 4) + 2], a[4 * (q % 4) + 3]};
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), own, q * 1024 + lane * 16, 0, 16);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // in memory, and behind the barrier everybody's
  __syncthreads();
  if (threadIdx.x == 0) {
    arrived = __hip_atomic_fetch_add(p.counters + 32 * tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (arrived == p.split - 1) __hip_atomic_store(p.counters + 32 * tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
  }
  __syncthreads();
  if (arrived != p.split - 1) return false;
  f32x4 got[Q], next[Q];
  auto take = [&](f32x4 (&to)[Q], int s) {
    const auto from = place(s);
#pragma unroll
    for (int q = 0; q < Q; q++) to[q] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, q * 1024 + lane * 16, 0, 16));
  };
  take(got, 0);
  for (int s = 0; s < p.split; s++) {  // (the next slice's while one is added)
    take(next, s + 1 < p.split ? s + 1 : s);
#pragma unroll
    for (int q = 0; q < Q; q++) {
      f32x16 &a = acc[q / 4 / TN][q / 4 % TN];
#pragma unroll
      for (int e = 0; e < 4; e++) a[4 * (q % 4) + e] = s ? a[4 * (q % 4) + e] + got[q][e] : got[q][e];
      got[q] = next[q];
    }
  }
  return true;
}

// TM x TN = 4 x 4: the 256 x 256 tile described above.  Smaller tiles (2 x 2: 128 x 128, 2 x 4: 128 x 256, 4 x 2:
// 256 x 128) use the same stages, swizzles and phases with fewer rows and columns: an A instruction still covers 16
// rows of 64 bytes, a B instruction 1024 / (2 BN) k rows of 2 BN bytes (position q of k row k holds chunk
// q ^ ((k & 3) << 2) of the row's BN / 8).  They take A rows through an index vector and a matrix id per block of rows
// (p.a_rows, p.b_block): the A addresses are then 64-bit per lane.
// BT: B is column-major (p.b_trans: element (k, n) at b[k + n * ldb], the tutorial's `b.T` and the weight layout of a
// linear layer).  Its stage is then laid out like A's, [BN columns][64 bytes] with the same swizzle, and an operand is
// one 16-byte read; nothing needs transposing.
template <bool E> struct EdgeTile { static constexpr bool value = E; };
// AT: A is column-major (p.a_trans: element (m, k) at a[m + k * lda]).  Its stage is laid out like a row-major B's,
// [32 k rows][2 BM bytes], and read through the same transposing LDS read.
// PF: the workgroup has a fifth wavefront that fetches nothing into the stages; it touches lines of B some K tiles ahead
// of the four that work (below).
constexpr int F_PF_AHEAD = 8;
// SK: the grid holds p.split workgroups per tile; workgroup (tile, s) walks the s-th share of the K tiles and leaves its sums
// in p.partial.
template <bool BF16, int TM, int TN, class Ep, bool BT = false, bool AT = false, bool PF = false, bool SK = false, bool MEET = false>
__device__ __forceinline__ void gemm_dma_body(const GemmParams &p, int tiles_m, int tiles_n, const Ep &ep) {
  using T = DmaTile<TM, TN>;
  constexpr int BM = T::BM, BN = T::BN, STAGES = T::STAGES, A_BYTES = T::A_BYTES, STAGE_BYTES = T::STAGE_BYTES, ROWB = T::B_ROW_BYTES;
  constexpr int A_DMA = T::A_DMA, B_DMA = T::B_DMA, DMA = T::DMA;
  constexpr int B_KROWS = 1024 / ROWB;       // k rows one B instruction covers
  constexpr int B_CHUNKS = ROWB / 16;        // 16-byte chunks per k row
  constexpr bool GATHER = !(TM == 4 && TN == 4) && !AT;
  constexpr int A_ROWB = BM * 2, A_KROWS = 1024 / A_ROWB, A_CHUNKS = A_ROWB / 16;  // AT: bytes per k row, k rows per instruction, chunks per k row
  static_assert(DMA % 2 == 0, "half of a tile's loads go out in each phase");
#ifdef TTS_GEMM_RTC
  __shared__ __align__(16) char dma_smem[T::LDS_BYTES];
#else
  extern __shared__ __align__(16) char dma_smem[];
#endif
  char *smem = dma_smem;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  int bid = blockIdx.x;
  const int nwg = tiles_m * tiles_n;
  const int slice = SK ? bid / nwg : 0;
  if (SK) bid -= slice * nwg;
  if (nwg % 8 == 0) bid = (bid % 8) * (nwg / 8) + bid / 8;  // consecutive ids on one XCD
  const int group = 4 * tiles_n;                             // 4-tile-tall column groups
  const int g0 = (bid / group) * 4;
  const int gh = min(tiles_m - g0, 4);
  int tile_m = g0 + (bid % group) % gh;
  const int tile_n = (bid % group) / gh;
  int pf_share = tile_m - g0, pf_shares = gh;  // PF: this workgroup's part of the B lines its column group reads
  if (GATHER && p.b_block && tiles_m <= 256) {
    // Row tiles that multiply the same matrix should sit behind one L2: the workgroup takes the row tile whose place in
    // the order by matrix id (ties by position) is the one the tile order above gave it.  With ids 0..7 dealt round-robin
    // to 32 blocks of 128 rows, every XCD otherwise streams four of the eight matrices (measured past L2: 319 MB per
    // launch for 100 MB of operands).
    __shared__ int block_key[256], place_key[256], sorted_tile;
    if (tid < tiles_m) block_key[tid] = p.b_block[((int64_t)tid * BM) / p.b_block_rows];
    __syncthreads();
    if (tid < tiles_m) {
      const int mine = block_key[tid];
      int place = 0;
      for (int o = 0; o < tiles_m; o++) place += (block_key[o] < mine || (block_key[o] == mine && o < tid)) ? 1 : 0;
      if (place == tile_m) sorted_tile = tid;
      place_key[place] = mine;
    }
    __syncthreads();
    if (PF) {  // the row tiles of this column group that multiply the same matrix split its lines between them
      const int mine = place_key[tile_m];
      pf_share = 0, pf_shares = 0;
      for (int q = g0; q < g0 + gh; q++)
        if (place_key[q] == mine) {
          if (q < tile_m) pf_share++;
          pf_shares++;
        }
    }
    tile_m = sorted_tile;
  }
  const int64_t m0 = (int64_t)tile_m * BM, n0 = (int64_t)tile_n * BN;

  const char *b_base = (const char *)((const uint16_t *)p.b + (BT ? n0 * p.ldb : n0));
  int which = 0;
  if (GATHER && p.b_block) {  // the rows of this tile multiply a matrix of their own; a negative id: nothing to do for them
    which = p.b_block[m0 / p.b_block_rows];
    if (which < 0) return;
    b_base += 2 * ((p.gather_mul32 & 2) ? (int64_t)(int)((uint32_t)which * (uint32_t)p.b_block_stride) : (int64_t)which * p.b_block_stride);
  }

  const int nk_all = (int)(p.K / F_BK);
  const int k_begin = SK ? (int)((int64_t)slice * nk_all / p.split) : 0;
  const int nk = SK ? (int)((int64_t)(slice + 1) * nk_all / p.split) - k_begin : nk_all;
  // Row tiles with matrices of their own walk K from different starting tiles (matrix id tiles in, wrapping round): the
  // workgroups of a launch start together, and matrices that lie a power of two apart in memory would otherwise be read
  // at the same offsets at the same time.  (The sum over K is taken in that order; 1.5 us of 45 on the measured case.)
  const int k_first = (GATHER && p.b_block) ? (int)((uint32_t)which % (uint32_t)nk) : 0;
  if (PF && wave == 4) {
    // The working wavefronts' loads wait in the memory pipeline for as long as their lines take to arrive, and lines that
    // come from HBM (several weight matrices: nothing of B is read twice out of the Infinity Cache) take long enough that
    // more LDS stages do not help (five and six measured like four).  This wavefront asks for the lines first: a
    // 4-byte load per 128-byte line of its share of the B tile F_PF_AHEAD tiles ahead, into a patch of LDS nobody reads (a
    // load into a register would come back long after the compiler has given the register to something else).  It keeps
    // step with the others through the same barriers.  Measured on 4096 gathered rows x [8, 2048, 2048]: 50.0 -> 43.8 us
    // with operands from HBM; touching A's lines as well cost 1 us, touching every other line gained nothing.
    static_assert(!PF || (!BT && !AT), "the prefetching wavefront walks a row-major B");
    __shared__ int touched[64];
    const uint32_t sink = (uint32_t)(uintptr_t)TTS_LDS(touched);
    constexpr int LPR = ROWB / 128, LINES = F_BK * LPR;  // 128-byte lines per k row and per tile
    const int per = (LINES + pf_shares - 1) / pf_shares;
    const char *line_at[2];
    bool on[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {  // at most 128 lines per tile
      const int l = lane + 64 * h, line = pf_share * per + l;
      on[h] = l < per && line < LINES && n0 + (line % LPR) * 64 < p.N;
      line_at[h] = b_base + ((int64_t)(line / LPR) * p.ldb + (line % LPR) * 64) * 2;
    }
    auto touch = [&](int t) {
      if (t >= nk) return;
      t += k_first;
      if (t >= nk) t -= nk;
#pragma unroll
      for (int h = 0; h < 2; h++)
        if (on[h])
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(sink), "v"(line_at[h] + (int64_t)t * F_BK * p.ldb * 2) : "memory", "m0");
    };
    for (int t = STAGES - 1; t < F_PF_AHEAD; t++) touch(t);
    __syncthreads();  // the others' barrier after the prologue ...
    for (int t = 0; t < nk; t++) {
      touch(t + F_PF_AHEAD);
      __syncthreads();  // ... and the one of every K tile
    }
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));  // the patch of LDS goes away with the workgroup
    return;
  }

  // Wavefront w issues A instructions A_DMA w .. (rows 16 ia + lane / 4) and B instructions B_DMA w .. (k rows
  // B_KROWS ib + lane / B_CHUNKS) of a tile.  Per-lane byte offsets are constant; the tile's base address moves in
  // scalar registers (with gathered rows: per-lane 64-bit addresses that move by one K tile).
  uint32_t a_voff[A_DMA], b_voff[B_DMA];
  const char *a_lane[A_DMA];
#pragma unroll
  for (int i = 0; i < A_DMA; i++) {
    if (AT) {  // as a row-major B: k rows A_KROWS (A_DMA w + i) + lane / A_CHUNKS, chunks of rows past M fetch the last whole chunk (M % 8 == 0)
      const int krow = A_KROWS * (A_DMA * wave + i) + lane / A_CHUNKS;
      const int chunk = min((lane & (A_CHUNKS - 1)) ^ ((krow & 3) << 2), (int)((p.M - m0) / 8 - 1));
      a_voff[i] = (uint32_t)((krow * p.lda + 8 * chunk) * 2);
      continue;
    }
    // rows past M (the last row tile of a ragged problem) fetch row M - 1 again: they only reach outputs nobody stores
    const int row = min(16 * (A_DMA * wave + i) + lane / 4, (int)(p.M - 1 - m0));
    const int chunk = (lane & 3) ^ ((lane >> 4) & 3);
    a_voff[i] = (uint32_t)((row * p.lda + 8 * chunk) * 2);
    if (GATHER) {
      int64_t r = m0 + row;
      if (p.a_rows) r = (p.gather_mul32 & 1) ? (int64_t)(int)((uint32_t)p.a_rows[r] * (uint32_t)p.lda) : (int64_t)p.a_rows[r] * p.lda;
      else r *= p.lda;
      a_lane[i] = (const char *)((const uint16_t *)p.a + r + 8 * chunk);
    }
  }
#pragma unroll
  for (int i = 0; i < B_DMA; i++) {
    if (BT) {  // as A: columns 16 (B_DMA w + i) + lane / 4 of the tile, those past N fetch column N - 1
      const int col = min(16 * (B_DMA * wave + i) + lane / 4, (int)(p.N - 1 - n0));
      b_voff[i] = (uint32_t)((col * p.ldb + 8 * ((lane & 3) ^ ((lane >> 4) & 3))) * 2);
      continue;
    }
    const int krow = B_KROWS * (B_DMA * wave + i) + lane / B_CHUNKS;
    // likewise, chunks of columns past N fetch the last whole chunk of the row (N is a multiple of 8)
    const int chunk = min((lane & (B_CHUNKS - 1)) ^ ((krow & 3) << 2), (int)((p.N - n0) / 8 - 1));
    b_voff[i] = (uint32_t)((krow * p.ldb + 8 * chunk) * 2);
  }
  const char *a_base = (const char *)((const uint16_t *)p.a + (AT ? m0 : m0 * p.lda));
  const uint32_t lds0 = (uint32_t)(uintptr_t)TTS_LDS(smem);
  const uint32_t wave_u = __builtin_amdgcn_readfirstlane(wave);
  auto dma = [&](const char *sbase, uint32_t voff, uint32_t lds) {
#ifdef TTS_GEMM_RTC
    // the run-time compiler may be an older one than the library's (a process that loaded PyTorch first gets PyTorch's
    // hipRTC), and that one does not see that the tile's base address is the same in every lane: say so
    const uint64_t b = (uint64_t)(uintptr_t)sbase;
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));  // the builtin returns a signed int
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    sbase = (const char *)(uintptr_t)(((uint64_t)hi << 32) | (uint64_t)lo);
#endif
    load_to_lds(sbase, voff, lds);
  };
  auto dma_lane = [&](const char *addr, uint32_t lds) {  // every lane its own 64-bit address
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds), "v"(addr) : "memory", "m0");
  };
  auto dma_one = [&](int t, int n) {  // n < A_DMA: A part, else B part of tile t, into stage t % STAGES
    int tc = min(t, nk - 1) + k_first;
    if (tc >= nk) tc -= nk;
    tc += k_begin;
    const uint32_t st = lds0 + (t % STAGES) * STAGE_BYTES;
    if (n < A_DMA) {
      const uint32_t at = st + (A_DMA * wave_u + n) * 1024;
      if (GATHER) dma_lane(a_lane[n] + (int64_t)tc * F_BK * 2, at);
      else dma(a_base + (AT ? (int64_t)tc * F_BK * p.lda * 2 : (int64_t)tc * F_BK * 2), a_voff[n], at);
    } else {
      dma(b_base + (BT ? (int64_t)tc * F_BK * 2 : (int64_t)tc * F_BK * p.ldb * 2), b_voff[n - A_DMA], st + A_BYTES + (B_DMA * wave_u + n - A_DMA) * 1024);
    }
  };

  // fragment read offsets (bytes, within a stage)
  // A: row r = wm * TM * 32 + i * 32 + lane % 32, chunk c = 2 ks + lane / 32 at position c ^ ((r / 4) & 3)
  const int ar = wm * TM * 32 + (lane & 31);
  const int a_off = ar * 64, a_sw = (ar >> 2) & 3;
  // B: 16-lane group q = lane / 16, r16 = lane % 16: k row ks * 16 + 8 (q / 2) + 4 h + r16 / 4,
  // chunk wn * TN * 4 + 4 j + 2 (q & 1) + (r16 % 4) / 2, byte 8 (r16 & 1) within the chunk
  const int q = lane >> 4, r16 = lane & 15;
  const int b_chunk = wn * TN * 4 + 2 * (q & 1) + ((r16 & 3) >> 1), b_sw = (r16 >> 2) << 2;
  const int b_off = A_BYTES + (8 * (q >> 1) + (r16 >> 2)) * ROWB + 8 * (r16 & 1);

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

  // BT: column c = wn * TN * 32 + j * 32 + lane % 32 of the tile, chunk 2 ks + lane / 32 at position chunk ^ ((c / 4) & 3)
  const int bc = wn * TN * 32 + (lane & 31);
  const int bt_off = A_BYTES + bc * 64, bt_sw = (bc >> 2) & 3;
  // AT: as the row-major B below, with the wavefront's rows in place of its columns
  const int at_chunk = wm * TM * 4 + 2 * (q & 1) + ((r16 & 3) >> 1);
  const int at_off = (8 * (q >> 1) + (r16 >> 2)) * A_ROWB + 8 * (r16 & 1);
  constexpr int A_READS = AT ? 2 * TM : TM, READS = A_READS + (BT ? TN : 2 * TN), MFMAS = TM * TN;
  uint4 af[2][TM], bf[2][TN];
  // one fragment read (n < TM: A row block n; else B column block (n - TM) / 2, k half (n - TM) % 2)
  auto read_one = [&](int t, int ks, int n, uint4 (&a)[TM], uint4 (&b)[TN]) {
    const char *st = smem + (t % STAGES) * STAGE_BYTES;
    if (n < A_READS && AT) {
      const int i = n >> 1, h = n & 1;
      const char *ap = st + at_off + ks * 16 * A_ROWB + (((at_chunk + 4 * i) ^ b_sw) << 4) + h * 4 * A_ROWB;
      s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)TTS_LDS(ap));
      uint2 v2 = __builtin_bit_cast(uint2, v);
      if (h == 0) { a[i].x = v2.x; a[i].y = v2.y; } else { a[i].z = v2.x; a[i].w = v2.y; }
    } else if (n < A_READS) {
      a[n] = *reinterpret_cast<const uint4 *>(st + a_off + n * 2048 + (((2 * ks + (lane >> 5)) ^ a_sw) << 4));
    } else if (BT) {
      b[n - A_READS] = *reinterpret_cast<const uint4 *>(st + bt_off + (n - A_READS) * 2048 + (((2 * ks + (lane >> 5)) ^ bt_sw) << 4));
    } else {
      const int j = (n - A_READS) >> 1, h = (n - A_READS) & 1;
      const char *bp = st + b_off + ks * 16 * ROWB + (((b_chunk + 4 * j) ^ b_sw) << 4) + h * 4 * ROWB;
      s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)TTS_LDS(bp));
      uint2 v2 = __builtin_bit_cast(uint2, v);
      if (h == 0) { b[j].x = v2.x; b[j].y = v2.y; } else { b[j].z = v2.x; b[j].w = v2.y; }
    }
  };
  auto mfma_one = [&](int n, uint4 (&a)[TM], uint4 (&b)[TN]) {
    acc[n / TN][n % TN] = mfma32<BF16>(a[n / TN], b[n % TN], acc[n / TN][n % TN]);
  };
  // A phase: MFMAS matrix instructions, READS fragment reads for the next phase, DMA / 2 loads; they are dealt out
  // behind the matrix instructions as evenly as their numbers allow.
  constexpr int SLOTS = MFMAS > READS ? MFMAS : READS;
  auto phase = [&](uint4 (&a_use)[TM], uint4 (&b_use)[TN], uint4 (&a_next)[TM], uint4 (&b_next)[TN], int t_read, int ks_read, int t_load, int first_load) {
#pragma unroll
    for (int n = 0; n < SLOTS; n++) {
      __builtin_amdgcn_sched_barrier(0);
      if (n < MFMAS) mfma_one(n, a_use, b_use);
      if (n < READS) read_one(t_read, ks_read, n, a_next, b_next);
      constexpr int every = SLOTS / (DMA / 2);
      if (n % every == every - 1 && n / every < DMA / 2) dma_one(t_load, first_load + n / every);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // prologue: STAGES - 1 tiles in flight; tile 0 landed; its first operands read
  for (int t = 0; t < STAGES - 1; t++)
#pragma unroll
    for (int n = 0; n < DMA; n++) dma_one(t, n);
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(DMA * (STAGES - 2), 15));
  __syncthreads();
#pragma unroll
  for (int n = 0; n < READS; n++) read_one(0, 0, n, af[0], bf[0]);
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
  for (int t = 0; t < nk; t++) {
    // phase A: MFMAs of (tile t, first half); read (tile t, second half); first half of the loads of tile t + STAGES - 1
    phase(af[0], bf[0], af[1], bf[1], t, 1, t + STAGES - 1, 0);
    // own loads of tile t+1 have landed (later ones may be in flight); own reads of tile t are complete
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(DMA * (STAGES - 3) + DMA / 2, 0));
    __syncthreads();
    // phase B: MFMAs of (tile t, second half); read (tile t+1, first half); the rest of the loads
    phase(af[1], bf[1], af[0], bf[0], t + 1, 0, t + STAGES - 1, DMA / 2);
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));  // the surplus loads land before the LDS goes away

  // Epilogue.  A lane holds one column of each 32x32 block (rows 8 (v/4) + 4 (lane/32) + v%4 in element v).  Two rows
  // are narrowed at once (v_cvt_pk_bf16_f32 for bf16: round to nearest even, NaNs quieted), the pair is exchanged with
  // the neighbouring lane, and the even lane stores row r at columns (n, n+1), the odd lane row r+1 at (n-1, n):
  // half as many store instructions as one 2-byte store per element, and a handful of VALU ops per pair.
  if constexpr (MEET) {
    if (!slices_meet<TM, TN>(p, acc, slice, tile_m * tiles_n + tile_n, nwg, wave, lane)) return;
  }
  if constexpr (SK && !MEET) {
    // the slice's sums as they are: a lane's 32 x 32 block column by column, two rows of 32 consecutive floats per store
    float *__restrict__ part = p.partial + (int64_t)slice * p.M * p.N;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int64_t col = n0 + wn * TN * 32 + j * 32 + (lane & 31);
#pragma unroll
        for (int v = 0; v < 16; v++) {
          const int64_t row = m0 + wm * TM * 32 + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
          if (row < p.M && col < p.N) part[row * p.N + col] = acc[i][j][v];
        }
      }
    return;
  }
  uint16_t *__restrict__ C = (uint16_t *)p.c;
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  const bool odd = lane & 1;
  const uint32_t sel = odd ? 0x03020706u : 0x05040100u;  // odd: high halves of (neighbour, mine); even: low halves of (mine, neighbour)
  // EDGE: the tile sticks out of C (ragged M, or N that is not a multiple of the tile): elements outside are neither
  // evaluated (the functor may read a bias or a residual at the element's position) nor stored.
  auto store_tile = [&](auto edge) {
    constexpr bool EDGE = decltype(edge)::value;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int64_t col = n0 + wn * TN * 32 + j * 32 + (lane & 31) - (odd ? 1 : 0);
#pragma unroll
        for (int v = 0; v < 16; v += 2) {
          const int64_t er = m0 + wm * TM * 32 + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3), ec = n0 + wn * TN * 32 + j * 32 + (lane & 31);
          const bool in0 = !EDGE || (er < p.M && ec < p.N), in1 = !EDGE || (er + 1 < p.M && ec < p.N);
          const f32x2_t pr = {in0 ? ep(acc[i][j][v], er, ec) : 0.f, in1 ? ep(acc[i][j][v + 1], er + 1, ec) : 0.f};
          const uint32_t pk = BF16 ? __builtin_bit_cast(uint32_t, __builtin_convertvector(pr, bf16x2_t))
                                   : __builtin_bit_cast(uint32_t, __builtin_convertvector(pr, f16x2_t));
          const uint32_t nb = __builtin_amdgcn_mov_dpp(pk, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]: the neighbour's pair
          const uint32_t w = __builtin_amdgcn_perm(nb, pk, sel);
          const int64_t row = m0 + wm * TM * 32 + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3) + (odd ? 1 : 0);
          if (!EDGE || (row < p.M && col < p.N)) __builtin_nontemporal_store(w, reinterpret_cast<uint32_t *>(&C[row * p.ldc + col]));
        }
      }
  };
  if (m0 + BM > p.M || n0 + BN > p.N) store_tile(EdgeTile<true>());
  else store_tile(EdgeTile<false>());
}


// ------------------------- the 256 x 256 tile on v_mfma_f32_16x16x32 (row-major operands, whole K tiles)
// The same tile, the same ring of four direct-to-LDS stages and the same A swizzle as gemm_dma_body<4, 4>, with the matrix
// instruction of shape 16 x 16 x 32 instead of 32 x 32 x 16.  Under the board's power limit the time of a large product is the
// energy it dissipates, and on operands of the prescribed distribution the 16 x 16 x 32 instruction sustains 0.79 of the
// peak rate from registers where 32 x 32 x 16 sustains 0.70 to 0.73 (measured with no data movement at all; on all-zero
// operands both reach 0.90); LDS and global traffic per flop are the same for both.  4096^3: 101-104 us against 104-110 for
// the 32 x 32 x 16 body in the same runs, bit for bit the same result.
//
// A wavefront's 128 x 128 part of C is 8 x 8 blocks of 16 x 16, four accumulator registers each, held transposed (the B
// operand goes in as the instruction's first source): a lane holds four consecutive columns of one row, which the epilogue
// can narrow and pack without cross-lane moves.  One K tile of 32 is one instruction's depth.
//   A operand of row block i: row 16 i + lane % 16, k 8 (lane / 16) .. +7: one 16-byte LDS read (A's swizzle is chosen
//     for the order in which such a read serves its lanes: see a_swizzle).
//   B operand of column block j: `ds_read_b64_tr_b16` twice (k 0-3 and 4-7 of the lane's octet), lane r of a 16-lane group
//     addressing k row 8 (lane / 16) + r / 4, columns 4 (r % 4) .. +3 of the block.  Two k octets share a half wavefront, so
//     the stage's swizzle also flips chunk bit 1 with k bit 3: position q of k row k holds chunk q ^ ((k & 3) << 2) ^ (((k >> 3) & 1) << 1).
// Phases of a tile t: (0) the 32 products of column blocks 0-3, with the eight reads of B blocks 4-7 of tile t and half of
// the loads of tile t + 3 behind them; wait for the own loads of tile t + 1, barrier; (1) the 32 products of column blocks
// 4-7, with the reads of all of A (8) and of B blocks 0-3 (8) of tile t + 1 and the other half of the loads.  A's operands
// alternate between two register sets (the K loop is unrolled by two), B's blocks 0-3 and 4-7 each have one.
// The matrix instruction is issued from inline assembly, in place on the accumulation registers: left to the register
// allocator (the instruction's result may overlap its addend arbitrarily, so nothing ties them) the 64 accumulators rotate
// through both register files and are copied back at the loop's end, 520 moves per two tiles.
// Epilogue: every wavefront narrows 16 rows at a time into a patch of LDS of its own (the stages are free by then) and
// stores whole 256-byte row segments with 16-byte nontemporal stores: 33.5 MB written for 33.5 MB of C where 4-byte
// stores of 64-byte segments wrote 51 MB.
// Loops over compile-time indices, and every lambda of the body below is marked always_inline: the accumulators and
// operand registers must become registers whatever the size of the epilogue functor.  (With a functor of a few hundred
// operations the inliner left the epilogue's lambda out of line, the accumulators, passed to it by reference, lived in
// scratch memory, and the compiler read them right behind matrix instructions it had not seen being issued.)
template <int V>
struct IntConstant {
  static constexpr int value = V;
};
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (I < N) {
    f(IntConstant<I>());
    static_for<I + 1, N>(f);
  }
}

// SK: the grid holds p.split workgroups per tile; workgroup (tile, s) walks the s-th share of the K tiles and leaves its fp32
// sums in p.partial (a lane's four consecutive columns of a row are one 16-byte store, straight from the registers).
template <bool BF16, class Ep, bool SK = false>
__device__ __forceinline__ void gemm_dma16_body(const GemmParams &p, int tiles_m, int tiles_n, const Ep &ep) {
  using T = DmaTile<4, 4>;
  constexpr int BM = T::BM, BN = T::BN, STAGES = T::STAGES, A_BYTES = T::A_BYTES, STAGE_BYTES = T::STAGE_BYTES, ROWB = T::B_ROW_BYTES;
  constexpr int A_DMA = T::A_DMA, B_DMA = T::B_DMA, DMA = T::DMA;
  static_assert(A_DMA == 4 && B_DMA == 4 && ROWB == 512, "256 x 256 x 32 stages");
#ifdef TTS_GEMM_RTC
  __shared__ __align__(16) char dma_smem[T::LDS_BYTES];
#else
  extern __shared__ __align__(16) char dma_smem[];
#endif
  char *smem = dma_smem;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  int bid = blockIdx.x;
  const int nwg = tiles_m * tiles_n;
  const int slice = SK ? bid / nwg : 0;
  if (SK) bid -= slice * nwg;
  if (nwg % 8 == 0) bid = (bid % 8) * (nwg / 8) + bid / 8;  // consecutive ids on one XCD
  const int group = 4 * tiles_n;                             // 4-tile-tall column groups
  const int g0 = (bid / group) * 4;
  const int gh = min(tiles_m - g0, 4);
  const int tile_m = g0 + (bid % group) % gh, tile_n = (bid % group) / gh;
  const int64_t m0 = (int64_t)tile_m * BM, n0 = (int64_t)tile_n * BN;
  const char *a_base = (const char *)((const uint16_t *)p.a + m0 * p.lda);
  const char *b_base = (const char *)((const uint16_t *)p.b + n0);
  const int nk_all = (int)(p.K / F_BK);
  const int k_begin = SK ? (int)((int64_t)slice * nk_all / p.split) : 0;
  const int nk = SK ? (int)((int64_t)(slice + 1) * nk_all / p.split) - k_begin : nk_all;

  // A's swizzle: position q of row r holds chunk q ^ a_swizzle((r / 4) & 3).  A 16-byte LDS read serves sixteen lanes per
  // cycle, and not sixteen neighbours: lanes 0-3 go with 12-15, 20-23 and 24-27 (of the eight quads of a half wavefront,
  // those whose number has an even count of set bits, then the others; found by letting two lanes alone read one bank).
  // With this instruction's operand layout (lane l: row l % 16, chunk l / 16) such a cycle holds row quads 0 and 3 of one
  // chunk and 1 and 2 of the next, and the swizzle (0, 2, 3, 1) puts the four into different banks; the plain
  // (r / 4) & 3 of the 32 x 32 x 16 body, conflict-free for that body's layout, made every A read here take twice its cycles.
  auto a_swizzle = [](int row_quad) __attribute__((always_inline)) { return ((row_quad >> 1) & 1) | (((row_quad & 1) ^ ((row_quad >> 1) & 1)) << 1); };
  uint32_t a_voff[A_DMA], b_voff[B_DMA];
#pragma unroll
  for (int i = 0; i < A_DMA; i++) {
    // rows past M (the last row tile of a ragged problem) fetch row M - 1 again: they only reach outputs nobody stores
    const int row = min(16 * (A_DMA * wave + i) + lane / 4, (int)(p.M - 1 - m0));
    const int chunk = (lane & 3) ^ a_swizzle((lane >> 4) & 3);
    a_voff[i] = (uint32_t)((row * p.lda + 8 * chunk) * 2);
  }
#pragma unroll
  for (int i = 0; i < B_DMA; i++) {
    const int krow = 2 * (B_DMA * wave + i) + lane / 32;
    // likewise, chunks of columns past N fetch the last whole chunk of the row (N is a multiple of 8)
    const int chunk = min((lane & 31) ^ ((krow & 3) << 2) ^ (((krow >> 3) & 1) << 1), (int)((p.N - n0) / 8 - 1));
    b_voff[i] = (uint32_t)((krow * p.ldb + 8 * chunk) * 2);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)TTS_LDS(smem);
  const uint32_t wave_u = __builtin_amdgcn_readfirstlane(wave);
  // n < A_DMA: A part, else B part of tile t, into stage t % STAGES.  Loads past the last tile fetch the last tile again, so
  // that the wait count is the same in every iteration (a scalar branch around every load and between two waits instead
  // cost 5 us of 110: sixteen branches per tile in between the matrix instructions).
  auto base_of = [&](int t, bool of_b) __attribute__((always_inline)) {
    const int tc = min(t, nk - 1) + k_begin;
    const char *base = of_b ? b_base + (int64_t)tc * F_BK * p.ldb * 2 : a_base + (int64_t)tc * F_BK * 2;
#ifdef TTS_GEMM_RTC
    // (an older run-time compiler does not see that the tile's base address is the same in every lane: say so, here)
    const uint64_t b = (uint64_t)(uintptr_t)base;
    uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)), lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    asm volatile("" : "+s"(hi), "+s"(lo));
    base = (const char *)(uintptr_t)(((uint64_t)hi << 32) | (uint64_t)lo);
#endif
    return base;
  };
  auto lds_of = [&](int t, int n) __attribute__((always_inline)) {
    return lds0 + (t % STAGES) * STAGE_BYTES + (n < A_DMA ? (A_DMA * wave_u + n) * 1024 : A_BYTES + (B_DMA * wave_u + n - A_DMA) * 1024);
  };
  auto dma_one = [&](int t, int n) __attribute__((always_inline)) { load_to_lds(base_of(t, n >= A_DMA), n < A_DMA ? a_voff[n] : b_voff[n - A_DMA], lds_of(t, n)); };

  const int l16 = lane & 15, q = lane >> 4;
  const int a_off = (wm * 128 + l16) * 64 + ((q ^ a_swizzle((l16 >> 2) & 3)) << 4);
  const int b_sw = ((l16 >> 2) << 2) ^ ((q & 1) << 1);
  const int b_chunk = wn * 16 + ((l16 & 3) >> 1);
  const int b_off = A_BYTES + (8 * q + (l16 >> 2)) * ROWB + 8 * (l16 & 1);

  f32x4 acc[8][8];
  static_for<0, 64>([&](auto n) __attribute__((always_inline)) { acc[n.value / 8][n.value % 8] = (f32x4){0.f, 0.f, 0.f, 0.f}; });
  uint4 A[2][8], B0[4], B1[4];
  auto read_a = [&](int t, int i, uint4 (&a)[8]) {
    a[i] = *reinterpret_cast<const uint4 *>(smem + (t % STAGES) * STAGE_BYTES + a_off + i * 1024);
  };
  auto read_b = [&](int t, int j, int h, uint4 &b) __attribute__((always_inline)) {  // column block j of the wavefront's eight, k half h of the lane's octet
    const char *bp = smem + (t % STAGES) * STAGE_BYTES + b_off + h * 4 * ROWB + (((b_chunk + 2 * j) ^ b_sw) << 4);
    s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)TTS_LDS(bp));
    uint2 v2 = __builtin_bit_cast(uint2, v);
    if (h == 0) { b.x = v2.x; b.y = v2.y; } else { b.z = v2.x; b.w = v2.y; }
  };
  typedef uint32_t u32x4_r __attribute__((ext_vector_type(4)));
  auto mfma16 = [&](int i, int j, const uint4 &a, const uint4 &b) __attribute__((always_inline)) {
    if constexpr (BF16)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(__builtin_bit_cast(u32x4_r, b)), "v"(__builtin_bit_cast(u32x4_r, a)));
    else
      asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(__builtin_bit_cast(u32x4_r, b)), "v"(__builtin_bit_cast(u32x4_r, a)));
  };
  // A product and a load behind it.  The matrix instruction is what stands between the write of m0 and the load; a base address that
  // had to be read from a vector register is further behind, at the start of the phase.  (4096^3 bf16 against loads without either
  // wait: 95.3 / 96.4 us, with a compiled epilogue 96.4 / 99.3; through load_to_lds 100.1 / 98.6, 114.7 / 113.6.)
  auto mfma16_and_load = [&](int i, int j, const uint4 &a, const uint4 &b, const char *base, uint32_t voff, uint32_t lds) __attribute__((always_inline)) {
    if constexpr (BF16)
      asm volatile("s_mov_b32 m0, %3\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %4, %5"
                   : "+a"(acc[i][j]) : "v"(__builtin_bit_cast(u32x4_r, b)), "v"(__builtin_bit_cast(u32x4_r, a)), "s"(lds), "v"(voff), "s"(base) : "memory", "m0");
    else
      asm volatile("s_mov_b32 m0, %3\n\tv_mfma_f32_16x16x32_f16 %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %4, %5"
                   : "+a"(acc[i][j]) : "v"(__builtin_bit_cast(u32x4_r, b)), "v"(__builtin_bit_cast(u32x4_r, a)), "s"(lds), "v"(voff), "s"(base) : "memory", "m0");
  };
  auto tile = [&](int t, uint4 (&Ac)[8], uint4 (&An)[8]) __attribute__((always_inline)) {
    const char *base = base_of(t + STAGES - 1, false);
    static_for<0, 32>([&](auto slot) __attribute__((always_inline)) {
      constexpr int n = decltype(slot)::value;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (n % 8 == 7) mfma16_and_load(n >> 2, n & 3, Ac[n >> 2], B0[n & 3], base, a_voff[n / 8], lds_of(t + STAGES - 1, n / 8));
      else mfma16(n >> 2, n & 3, Ac[n >> 2], B0[n & 3]);
      if constexpr (n < 8) read_b(t, 4 + (n >> 1), n & 1, B1[n >> 1]);
    });
    __builtin_amdgcn_sched_barrier(0);
    // own loads of tile t + 1 have landed (later ones may be in flight); own reads of tile t are complete
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(DMA * (STAGES - 3) + DMA / 2, 0));
    __syncthreads();
    base = base_of(t + STAGES - 1, true);
    static_for<0, 32>([&](auto slot) __attribute__((always_inline)) {
      constexpr int n = decltype(slot)::value;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (n % 8 == 7) mfma16_and_load(n >> 2, 4 + (n & 3), Ac[n >> 2], B1[n & 3], base, b_voff[n / 8], lds_of(t + STAGES - 1, A_DMA + n / 8));
      else mfma16(n >> 2, 4 + (n & 3), Ac[n >> 2], B1[n & 3]);
      if constexpr (n < 8) read_a(t + 1, n, An);
      else if constexpr (n < 16) read_b(t + 1, (n - 8) >> 1, n & 1, B0[(n - 8) >> 1]);
    });
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
  };

  // prologue: STAGES - 1 tiles in flight; tile 0 landed; its first operands read
  for (int t = 0; t < STAGES - 1; t++) static_for<0, DMA>([&](auto n) __attribute__((always_inline)) { dma_one(t, n.value); });
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(DMA * (STAGES - 2), 15));
  __syncthreads();
  static_for<0, 8>([&](auto i) __attribute__((always_inline)) { read_a(0, i.value, A[0]); });
  static_for<0, 4>([&](auto j) __attribute__((always_inline)) {
    read_b(0, j.value, 0, B0[j.value]);
    read_b(0, j.value, 1, B0[j.value]);
  });
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
  int t = 0;
  for (; t + 1 < nk; t += 2) {  // two tiles per turn: A's register sets take turns
    tile(t, A[0], A[1]);
    tile(t + 1, A[1], A[0]);
  }
  if (t < nk) tile(t, A[0], A[1]);
  // The compiler does not know that the assembly above issued matrix instructions, so it leaves no wait states between
  // one of them and a read of its result (the epilogue's, or a spill the register allocator places right behind the
  // loop).  The sixteen accumulators the last tile wrote last pass through this statement, so whatever reads them comes
  // after its wait states; the others were written at least sixteen instructions (256 cycles) earlier.
  asm volatile("s_nop 15\n\ts_nop 15"
               : "+a"(acc[4][4]), "+a"(acc[4][5]), "+a"(acc[4][6]), "+a"(acc[4][7]), "+a"(acc[5][4]), "+a"(acc[5][5]), "+a"(acc[5][6]), "+a"(acc[5][7]),
                 "+a"(acc[6][4]), "+a"(acc[6][5]), "+a"(acc[6][6]), "+a"(acc[6][7]), "+a"(acc[7][4]), "+a"(acc[7][5]), "+a"(acc[7][6]), "+a"(acc[7][7])
               :
               : "memory");
  // Every wavefront has read its last operands: the last tile's stage is free.  The other three still receive the surplus
  // loads of the last iterations, which nobody waits for before the kernel's end.
  __syncthreads();

  // acc[i][j][v] is C(row 16 i + lane % 16, column 16 j + 4 (lane / 16) + v) of the wavefront's part
  if constexpr (SK) {
    float *__restrict__ part = p.partial + (int64_t)slice * p.M * p.N;
    static_for<0, 64>([&](auto bc) __attribute__((always_inline)) {
      constexpr int i = decltype(bc)::value / 8, j = decltype(bc)::value % 8;
      const int64_t row = m0 + wm * 128 + i * 16 + l16, col = n0 + wn * 128 + j * 16 + 4 * q;
      if (row < p.M && col < p.N) *reinterpret_cast<f32x4 *>(part + row * p.N + col) = acc[i][j];  // (N is a multiple of 8)
    });
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));  // the surplus loads land before the LDS goes away
    return;
  }
  uint16_t *__restrict__ C = (uint16_t *)p.c;
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  constexpr int PITCH = 272;  // bytes per staged row of 128 columns
  // (one patch of 16 rows per wavefront, in the last tile's stage; a wavefront's LDS accesses complete in order, so the
  // next 16 rows' writes come after this 16 rows' reads)
  static_assert(4 * 16 * PITCH <= STAGE_BYTES, "the four wavefronts' patches fit one stage");
  char *mine = smem + ((nk + STAGES - 1) % STAGES) * STAGE_BYTES + wave * (16 * PITCH);
  // A fused epilogue evaluates the stored value with the ids of the Triton program that owns the element (Ep::BM x Ep::BN
  // blocks; 0: no functor).  Blocks of 16 x 16 never straddle two owners, and a wavefront's 128 x 128 part has GI x GJ of
  // them: they are looked up once each, and what the functor computes from the program's ids alone is then the same
  // expression on the same values for every element of an owner, which the compiler evaluates once.  (Looked up per
  // element, every one of the 256 evaluations per lane is separate code: a functor with the tutorial's grouped tile
  // order and a bias per row and column took eight minutes to compile.)
  constexpr int EBM = Ep::BM, EBN = Ep::BN;
  constexpr bool OWNED = EBM >= 16 && EBN >= 16 && (128 % EBM == 0 || EBM % 128 == 0) && (128 % EBN == 0 || EBN % 128 == 0);
  constexpr int GI = OWNED && EBM < 128 ? 128 / EBM : 1, GJ = OWNED && EBN < 128 ? 128 / EBN : 1;
  int owner[GI][GJ];
  if constexpr (OWNED)
    static_for<0, GI * GJ>([&](auto gc) __attribute__((always_inline)) {
      constexpr int gi = decltype(gc)::value / GJ, gj = decltype(gc)::value % GJ;
      const int64_t r0 = m0 + wm * 128 + gi * (128 / GI), c0 = n0 + wn * 128 + gj * (128 / GJ);
      owner[gi][gj] = (r0 < p.M && c0 < p.N) ? ep.tile_pid[(r0 / EBM) * ep.tiles_n + c0 / EBN] : 0;  // (outside C: nobody's)
    });
  auto value = [&](auto ic, auto jc, float a, int64_t row, int64_t col) __attribute__((always_inline)) -> float {
    if constexpr (OWNED) return ep.at(owner[decltype(ic)::value * 16 / (128 / GI)][decltype(jc)::value * 16 / (128 / GJ)], a, (int)(row % EBM), (int)(col % EBN));
    else return ep(a, row, col);
  };
  // this lane's chunk of row lane / 16 of the wavefront's part
  uint16_t *c_lane = C + (m0 + wm * 128 + (lane >> 4)) * p.ldc + n0 + wn * 128 + (lane & 15) * 8;
  auto store_tile = [&](auto edge) __attribute__((always_inline)) {
    // EDGE: the tile sticks out of C (ragged M, or N that is not a multiple of the tile): elements outside are neither
    // evaluated (the functor may read a bias or a residual at the element's position) nor stored.
    constexpr bool EDGE = decltype(edge)::value;
    // rows and columns of the wavefront's part that lie inside C (N is a multiple of 8: a lane's four columns, and a
    // stored chunk's eight, are inside or outside together)
    const int rows_left = (int)min((int64_t)128, p.M - (m0 + wm * 128)), cols_left = (int)min((int64_t)128, p.N - (n0 + wn * 128));
    static_for<0, 8>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      char *reg = mine;
      const int64_t er = m0 + wm * 128 + i * 16 + l16;
      const bool row_in = !EDGE || i * 16 + l16 < rows_left;
      static_for<0, 8>([&](auto jc) __attribute__((always_inline)) {
        constexpr int j = decltype(jc)::value;
        const int64_t ec = n0 + wn * 128 + j * 16 + 4 * q;
        const bool in = !EDGE || (row_in && j * 16 + 4 * q < cols_left);
        float o[4];
        static_for<0, 4>([&](auto vc) __attribute__((always_inline)) {
          constexpr int v = decltype(vc)::value;
          o[v] = in ? value(ic, jc, acc[i][j][v], er, ec + v) : 0.f;
        });
        const f32x2_t p01 = {o[0], o[1]}, p23 = {o[2], o[3]};
        uint2 w;
        if (BF16) {
          w.x = __builtin_bit_cast(uint32_t, __builtin_convertvector(p01, bf16x2_t));
          w.y = __builtin_bit_cast(uint32_t, __builtin_convertvector(p23, bf16x2_t));
        } else {
          w.x = __builtin_bit_cast(uint32_t, __builtin_convertvector(p01, f16x2_t));
          w.y = __builtin_bit_cast(uint32_t, __builtin_convertvector(p23, f16x2_t));
        }
        *reinterpret_cast<uint2 *>(reg + l16 * PITCH + (j * 16 + 4 * q) * 2) = w;
      });
      // (a wavefront's LDS accesses complete in order: its reads below see its writes above)
      uint4 chunk[4];
      static_for<0, 4>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        chunk[k] = *reinterpret_cast<const uint4 *>(reg + (4 * k + (lane >> 4)) * PITCH + (lane & 15) * 16);
      });
      static_for<0, 4>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        const int row = 4 * k + (lane >> 4), ch = lane & 15;  // row of the sixteen, 16-byte chunk of the row
        // (rows of C need only be 4-byte aligned: a store of four dwords wants dword alignment, no more)
        typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
        const u32x4_a4 w = {chunk[k].x, chunk[k].y, chunk[k].z, chunk[k].w};
        if (!EDGE || (i * 16 + row < rows_left && ch * 8 < cols_left))
          __builtin_nontemporal_store(w, reinterpret_cast<u32x4_a4 *>(c_lane + (int64_t)(i * 16 + 4 * k) * p.ldc));
      });
    });
  };
  if (m0 + BM > p.M || n0 + BN > p.N) store_tile(EdgeTile<true>());
  else store_tile(EdgeTile<false>());
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));  // the surplus loads land before the LDS goes away
}

// ------------------------------------------------------------- fp32 GEMM
// tl.dot on fp32 blocks: the reference multiplies in fp32 (linalg.matmul on f32, ConversionPatterns.hpp:1128-1201; it
// ignores the dot's inputPrecision), so this kernel uses the fp32 matrix instruction (v_mfma_f32_32x32x2_f32), not a
// reduced-precision one.  Any shape and alignment, A and B row- or column-major.
// Largest workgroup: 128 x 128 of C, 2 x 2 wavefronts of 64 x 64 (2 x 2 MFMA tiles of 32 x 32, 64 accumulator registers), K in
// steps of 16.  Both operand tiles sit in LDS as [k][r] (r = row of A / column of B, pitch = tile + 4 floats): a lane's MFMA
// operand is element (k0 + lane / 32, r0 + lane % 32), so a wavefront reads two runs of 32 consecutive floats.
// Tiles go global -> registers -> LDS with the next tile's loads in flight during the current tile's arithmetic (two
// LDS buffers, one barrier per tile); 16-byte global loads along whichever dimension is contiguous in memory.
// T: MFMA tiles per wavefront and dimension, W: wavefronts per dimension: 2, 2 = 128 x 128 per workgroup; 1, 2 = 64 x 64 (for
// problems that give fewer than two of the large tiles per CU); 1, 1 = 32 x 32 (for those that do not fill the chip with 64 x 64:
// a tile's matrix instructions all run on one CU, 13 us of them for a 64 x 64 tile at K = 1000).
// G: groups of W x W wavefronts that split the K tiles among them and add their sums through LDS at the end, in group order:
// the chain of loads, LDS stores and matrix instructions of a group is 1 / G as long, and the SIMDs have several to run.
// All K tiles but the last load 16 bytes a chunk, at any alignment and without a test, two tiles ahead; the last goes element by
// element where a chunk sticks out (gemm_mfma_body reads that one in 16 bytes, too).
// 768^3: 39.3 -> 17.6 us; 16 x 1000 x 1000: 11.7 (27 with 64 x 64 tiles).  (Eight groups at 768^3: 25.3.)
constexpr int F32_BK = 16;

template <int T, int W, int G, class Ep>
__device__ __forceinline__ void gemm_f32_body(const GemmParams &p, int tiles_m, int tiles_n, const Ep &ep) {
  constexpr int BT = 32 * T * W;      // rows of A / columns of B per workgroup
  constexpr int PITCH = BT + 4;       // floats between k rows in LDS
  constexpr int NT = 64 * W * W;      // threads per group
  constexpr int CH = 4 * BT / NT;     // chunks of 4 floats per thread and operand tile (BT x 16 floats = 4 BT chunks)
  __shared__ __align__(16) float stage[G][2][2][F32_BK * PITCH];  // [group][buffer][A, B][k][r]
  static_assert(sizeof(stage) >= (size_t)(G - 1) * BT * BT * sizeof(float), "the groups' sums fit where the tiles were");
  const int tid = threadIdx.x % NT, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = G > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0;
  float(&smem)[2][2][F32_BK * PITCH] = stage[group];
  const int wm = wave / W, wn = wave % W;
  int bid = blockIdx.x;
  const int nwg = tiles_m * tiles_n;
  if (nwg % 8 == 0) bid = (bid % 8) * (nwg / 8) + bid / 8;  // consecutive ids on one XCD
  const int tall = 8 * tiles_n;
  const int g0 = (bid / tall) * 8;
  const int gh = min(tiles_m - g0, 8);
  const int tile_m = g0 + (bid % tall) % gh, tile_n = (bid % tall) / gh;
  const int64_t m0 = (int64_t)tile_m * BT, n0 = (int64_t)tile_n * BT;
  const float *__restrict__ A = (const float *)p.a;
  const float *__restrict__ B = (const float *)p.b;
  const int64_t K = p.K;
  const bool a_r = p.a_trans != 0, b_r = p.b_trans == 0;  // r contiguous in memory

  const int64_t nk_all = (K + F32_BK - 1) / F32_BK;
  const int64_t k_begin = nk_all * group / G, nk = nk_all * (group + 1) / G;  // this group's K tiles
  const int64_t steps = W > 1 ? (nk_all + G - 1) / G : nk - k_begin;          // the most any group has, where they meet at barriers
  // K tiles below nwide load whole chunks: rows (columns) beyond the problem are replaced by others whose results nobody
  // stores, and a chunk that ends behind its row reads into the next, which the last k row does not have
  int64_t nwide = K / F32_BK;
  if ((a_r && p.lda < 4) || (b_r && p.ldb < 4)) nwide = 0;
  else if (K % F32_BK == 0 && ((a_r && m0 + BT > p.M) || (b_r && n0 + BT > p.N))) nwide = nk_all - 1;
  nwide = min(nwide, nk);

  // An operand tile is BT r x 16 k = 4 BT chunks of 4 floats, CH per thread.  k contiguous in memory (A row-major, B
  // column-major): chunk c = (r = c / 4, k = 4 (c % 4)); r contiguous (A column-major, B row-major): (k = c / (BT / 4), r = 4 (c % (BT / 4))).
  struct Tiles { float4 a[CH], b[CH]; };
  const float *a_ptr[CH], *b_ptr[CH];
  auto chunk_ptr = [&](const float *P, bool r_contig, int64_t ld, int64_t r_base, int64_t rows, int c) {
    if (r_contig) {
      const int64_t r = r_base + 4 * (c % (BT / 4));
      return P + (int64_t)(c / (BT / 4)) * ld + (r < rows ? r : 0);
    }
    return P + min(r_base + c / 4, rows - 1) * ld + 4 * (c % 4);
  };
#pragma unroll
  for (int j = 0; j < CH; j++) {
    a_ptr[j] = chunk_ptr(A, a_r, p.lda, m0, p.M, tid + NT * j);
    b_ptr[j] = chunk_ptr(B, b_r, p.ldb, n0, p.N, tid + NT * j);
  }
  const int64_t a_step = F32_BK * (a_r ? p.lda : 1), b_step = F32_BK * (b_r ? p.ldb : 1);
  auto load_wide = [&](Tiles &t, int64_t kt) {
#pragma unroll
    for (int j = 0; j < CH; j++) __builtin_memcpy(&t.a[j], a_ptr[j] + kt * a_step, 16);
#pragma unroll
    for (int j = 0; j < CH; j++) __builtin_memcpy(&t.b[j], b_ptr[j] + kt * b_step, 16);
  };
  auto load_edge = [&](float4 (&reg)[CH], const float *P, bool r_contig, int64_t ld, int64_t r_base, int64_t rows, int64_t k0) {
#pragma unroll
    for (int j = 0; j < CH; j++) {
      const int c = tid + NT * j;
      float v[4] = {0.f, 0.f, 0.f, 0.f};
      if (r_contig) {
        const int64_t k = k0 + c / (BT / 4), r = r_base + 4 * (c % (BT / 4));
        if (k < K)
          for (int i = 0; i < 4; i++) if (r + i < rows) v[i] = P[k * ld + r + i];
      } else {
        const int64_t r = r_base + c / 4, k = k0 + 4 * (c % 4);
        if (r < rows)
          for (int i = 0; i < 4; i++) if (k + i < K) v[i] = P[r * ld + k + i];
      }
      reg[j] = make_float4(v[0], v[1], v[2], v[3]);
    }
  };
  auto load_any = [&](Tiles &t, int64_t kt) {
    if (kt < nwide) load_wide(t, kt);
    else if (kt < nk) {
      load_edge(t.a, A, a_r, p.lda, m0, p.M, kt * F32_BK);
      load_edge(t.b, B, b_r, p.ldb, n0, p.N, kt * F32_BK);
    }
  };
  auto store_tile = [&](const float4 (&reg)[CH], float *S, bool r_contig) {
#pragma unroll
    for (int j = 0; j < CH; j++) {
      const int c = tid + NT * j;
      if (r_contig) {
        *reinterpret_cast<float4 *>(S + (c / (BT / 4)) * PITCH + 4 * (c % (BT / 4))) = reg[j];
      } else {  // four k of one r: one float into each of four k rows
        float *dst = S + (4 * (c % 4)) * PITCH + c / 4;
        dst[0] = reg[j].x; dst[PITCH] = reg[j].y; dst[2 * PITCH] = reg[j].z; dst[3 * PITCH] = reg[j].w;
      }
    }
  };
  auto store_tiles = [&](const Tiles &t, int buf) {
    store_tile(t.a, smem[buf][0], a_r);
    store_tile(t.b, smem[buf][1], b_r);
  };
  f32x16 acc[T][T];
#pragma unroll
  for (int i = 0; i < T; i++)
#pragma unroll
    for (int j = 0; j < T; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
  auto multiply = [&](int buf) {
    const float *As = smem[buf][0] + (lane >> 5) * PITCH + wm * (32 * T) + (lane & 31);
    const float *Bs = smem[buf][1] + (lane >> 5) * PITCH + wn * (32 * T) + (lane & 31);
#pragma unroll
    for (int ks = 0; ks < F32_BK; ks += 2) {
      float af[T], bf[T];
#pragma unroll
      for (int i = 0; i < T; i++) af[i] = As[ks * PITCH + 32 * i];
#pragma unroll
      for (int j = 0; j < T; j++) bf[j] = Bs[ks * PITCH + 32 * j];
#pragma unroll
      for (int i = 0; i < T; i++)
#pragma unroll
        for (int j = 0; j < T; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i], bf[j], acc[i][j], 0, 0, 0);
    }
  };
  // Groups of one wavefront share nothing until the end: a wavefront's LDS accesses complete in order.  Others meet at
  // barriers (a turn of either loop has two: every group meets the same number, also when it has a tile fewer).
  auto sync = [&]() {
    if constexpr (W > 1) __syncthreads();
    else {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  };
  Tiles even, odd;
  load_any(even, k_begin);
  load_any(odd, k_begin + 1);
  if (k_begin < nk) store_tiles(even, 0);
  load_any(even, k_begin + 2);
  sync();
  int64_t kt = k_begin, step = 0;
  for (; kt + 4 < nwide; step += 2, kt += 2) {  // loads tiles kt + 3 and kt + 4
    multiply(0);
    store_tiles(odd, 1);
    load_wide(odd, kt + 3);
    sync();
    multiply(1);
    store_tiles(even, 0);
    load_wide(even, kt + 4);
    sync();
  }
  for (; step < steps; step += 2, kt += 2) {
    if (kt < nk) multiply(0);
    if (kt + 1 < nk) store_tiles(odd, 1);
    load_any(odd, kt + 3);
    sync();
    if (kt + 1 < nk) multiply(1);
    if (kt + 2 < nk) store_tiles(even, 0);
    load_any(even, kt + 4);
    sync();
  }
  if constexpr (G > 1) {
    if (W == 1) __syncthreads();  // (the last barrier of the loop otherwise) the tiles are free
    float *sums = reinterpret_cast<float *>(stage);
    auto place = [&](int g, int i, int j, int v) { return (((g * W * W + wave) * T + i) * T + j) * 1024 + v * 64 + lane; };
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
      for (int j = 0; j < T; j++)
#pragma unroll
        for (int v = 0; v < 16; v++)
          if (group > 0) sums[place(group - 1, i, j, v)] = acc[i][j][v];
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 0; g < G - 1; g++)
#pragma unroll
      for (int i = 0; i < T; i++)
#pragma unroll
        for (int j = 0; j < T; j++)
#pragma unroll
          for (int v = 0; v < 16; v++) acc[i][j][v] += sums[place(g, i, j, v)];
  }
  // lane holds column (lane % 32), rows 8 (v / 4) + 4 (lane / 32) + v % 4 of each 32 x 32 tile
  float *__restrict__ C = (float *)p.c;
#pragma unroll
  for (int i = 0; i < T; i++)
#pragma unroll
    for (int j = 0; j < T; j++) {
      const int64_t col = n0 + wn * (32 * T) + j * 32 + (lane & 31);
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int64_t row = m0 + wm * (32 * T) + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (row < p.M && col < p.N) C[row * p.ldc + col] = ep(acc[i][j][v], row, col);
      }
    }
}

}  // namespace tts_gemm_device

#ifdef TTS_GEMM_RTC
extern "C" __global__ __launch_bounds__(TTS_GEMM_RTC == 9 ? 512 : 256) void gemm_rtc(TtsGemmParams p, int tiles_m, int tiles_n, TtsEp ep) {
#if TTS_GEMM_RTC == 0
  tts_gemm_device::gemm_dma16_body<TTS_GEMM_BF16 != 0>(p, tiles_m, tiles_n, ep);
#elif TTS_GEMM_RTC == 2
  tts_gemm_device::gemm_splitk_reduce_body<TTS_GEMM_BF16 != 0>(p, tiles_m, tiles_n, ep);  // (across, col_blocks)
#elif TTS_GEMM_RTC >= 7
  constexpr int T = TTS_GEMM_RTC == 7 ? 2 : 1, W = TTS_GEMM_RTC == 8 ? 1 : 2, G = TTS_GEMM_RTC == 8 ? 4 : TTS_GEMM_RTC == 9 ? 2 : 1;
  tts_gemm_device::gemm_f32_body<T, W, G>(p, tiles_m, tiles_n, ep);
#elif TTS_GEMM_RTC >= 4
  constexpr int TM = TTS_GEMM_RTC == 5 ? 4 : 2, TN = TTS_GEMM_RTC == 4 ? 4 : 2;  // 128 x 256, 256 x 128, 128 x 128
  tts_gemm_device::gemm_dma_body<TTS_GEMM_BF16 != 0, TM, TN>(p, tiles_m, tiles_n, ep);
#else
  tts_gemm_device::gemm_mfma_body<TTS_GEMM_BF16 != 0, TTS_GEMM_RTC == 3 ? 1 : 2, 2, 64>(p, tiles_m, tiles_n, ep);
#endif
}
#endif
