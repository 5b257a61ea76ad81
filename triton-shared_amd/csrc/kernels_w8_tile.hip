// C[M,N] = A[M,K] x (f16(W[K,N]) * scale[N]) for more rows of A than the decode kernels are for: a tiled matrix product that
// widens the int8 weights on their way from LDS to the matrix instruction.
//
// What it replaces: a decode launch per 32 rows (every one reads all of W), and, from 193 rows, a pass that wrote the weights
// to memory as fp16 (twice their bytes) before an ordinary product.  Here W crosses the memory once per launch.  At
// [8192, 28672], before -> now, in one run: 32 rows 51.1 -> 43.8 us, 48 rows 92 -> 47, 100 rows 192 -> 68, 300 rows 371 -> 126 (1.12
// PFLOP/s; 136 on another device), 512 rows 451 -> 209, 1024 rows 523 -> 414; 64 x 4096 x 4096 63 -> 20.
//
// Workgroup: 4 wavefronts side by side, each 16 TM rows x 64 columns of C; all four share the A tile.  K advances by 64, two
// steps of one v_mfma_f32_16x16x32_f16 each.  Both operands go to LDS by `global_load_lds_dwordx4` into a ring of K tiles:
//   A stage [16 TM rows][128 bytes]: position q of row r holds chunk q ^ ((r >> 1) & 7), which puts the sixteen rows and two
//     chunks that a 16-byte LDS read serves in one cycle into different banks (see a_swizzle in gemm_dma16_body for which
//     those are).  Whole 128-byte lines: with K tiles of 32 a load fetched half of every line of A, and the loads alone
//     took 119 us of the 300-row product where they now take 91.
//   W stage [64 k rows][256 bytes] of int8; position q of row k holds chunk q ^ (((k >> 3) & 3) << 2), so that the four
//     k octets of a wavefront's dword reads fall into different banks.
// A lane reads the dword of its four columns in each of its eight k rows (one octet of k per 16 lanes).  Column c of the four
// gives one operand of the instruction: byte c of the eight dwords.  The source multiplies the widened weight b by its
// column's scale s in fp16, one rounding.  Here that is v_perm and one v_pk_fma_f16 per two weights: the byte with its sign
// flipped, b + 128, is the fp16 subnormal (b + 128) 2^-24; with s = m 2^e, 1 <= |m| < 2, that times m 2^14 minus m / 8 is b m
// 2^-10 rounded once, and b s has the same rounding at every scale up to 511.75 (its smallest value other than zero is normal
// where s is; where s is subnormal, products below 2^-13 are exact).  The fp32 sums are multiplied by 2^(e + 10), exactly.  40
// vector instructions per step where the byte widened first and multiplied after takes 72.  A workgroup that has a larger
// scale (whose products may overflow), an infinite one or a NaN among its columns takes those four: widen, times 512, times s.
// The weights go in as the first source, so a lane's results are sixteen neighbouring columns of one row (columns 16 q + 4 v +
// c for result v of instruction c, q = lane / 16): two 16-byte stores per row and lane.
// What bounds it at 300 rows: the matrix instructions alone take 101 us, widening and LDS reads add 12, the loads 23 (136 in all on that
// device; with weights of few significant bits instead of the rounded products 4 us less, which is the power the multipliers draw).  Eight
// wavefronts that share the rows two ways (the widening done twice) were slower at every size: 177 us.
#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "kernels.h"

namespace tts {

namespace {
using namespace tts_gemm_device;

constexpr int W8T_COLS = 256;  // columns of C per workgroup
constexpr int W8T_MAX_TM = 10;

template <int TM>
struct W8Tile {
  static constexpr int A_BYTES = TM * 2048, W_BYTES = 64 * W8T_COLS, STAGE = A_BYTES + W_BYTES;
  static constexpr int A_DMA = (2 * TM + 3) / 4, DMA = A_DMA + 4;  // direct-to-LDS instructions per wavefront and K tile
  static constexpr int STAGES = 160 * 1024 / STAGE < 6 ? 160 * 1024 / STAGE : 6;
  static constexpr int LDS = STAGES * STAGE;
};

// SK: the grid holds `split` workgroups per tile, each walks its share of the K tiles and leaves fp32 sums in `partial`
template <int TM, bool SK>
__global__ __launch_bounds__(256, 1) void gemm_w8a16_tile_kernel(GemmW8A16Params p, int tiles_m, int tiles_n, int split, float *partial) {
  using T = W8Tile<TM>;
  constexpr int STAGES = T::STAGES;
  extern __shared__ __align__(16) char w8_smem[];
  char *smem = w8_smem;
  const int tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  // the row tiles of one column of tiles (and its slices) are neighbours on one XCD: they read the same weights
  int bid = blockIdx.x;
  const int nwg = gridDim.x;
  if (nwg % 8 == 0) bid = (bid % 8) * (nwg / 8) + bid / 8;
  const int tile_m = bid % tiles_m, rest = bid / tiles_m;
  const int slice = SK ? rest % split : 0, tile_n = SK ? rest / split : rest;
  const int64_t m0 = (int64_t)tile_m * (16 * TM), n0 = (int64_t)tile_n * W8T_COLS;
  const int nk_all = (int)(p.K / 64);
  const int k_begin = SK ? (int)((int64_t)slice * nk_all / split) : 0;
  const int nk = SK ? (int)((int64_t)(slice + 1) * nk_all / split) - k_begin : nk_all;

  uint32_t a_voff[T::A_DMA], w_voff[4];
  static_for<0, T::A_DMA>([&](auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;
    // (a wavefront beyond the last eight rows fetches those again, so that all wait for equal numbers of loads; rows past M
    // fetch row M - 1: they only reach results nobody stores)
    const int in_tile = 8 * min((int)(T::A_DMA * wave) + i, 2 * TM - 1) + lane / 8;
    const int row = min(in_tile, (int)(p.M - 1 - m0));
    a_voff[i] = (uint32_t)((row * p.lda + 8 * ((lane & 7) ^ ((in_tile >> 1) & 7))) * 2);
  });
  static_for<0, 4>([&](auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;
    const int krow = 4 * (4 * (int)wave + i) + lane / 16;
    // columns past N (a multiple of 16) fetch the last whole chunk of the row
    const int chunk = min((lane & 15) ^ (((krow >> 3) & 3) << 2), (int)((p.N - n0) / 16 - 1));
    w_voff[i] = (uint32_t)(krow * p.ldw + 16 * chunk);
  });
  // the scales of the columns a lane widens and of those it holds results of, and whether any of the workgroup's columns has
  // one that needs the source's two steps (columns past N: some other column's)
  uint16_t s_in[4], s_out[16], s_any[4];
  const uint16_t *scales = (const uint16_t *)p.scale;
  __builtin_memcpy(s_in, scales + min(n0 + 64 * (int)wave + 4 * l16, p.N - 4), 8);
  __builtin_memcpy(s_any, scales + min(n0 + 4 * lane, p.N - 4), 8);
  __builtin_memcpy(s_out, scales + min(n0 + 64 * (int)wave + 16 * q, p.N - 16), 32);
  const bool literal = __builtin_amdgcn_ballot_w64(max(max(s_any[0] & 0x7fff, s_any[1] & 0x7fff), max(s_any[2] & 0x7fff, s_any[3] & 0x7fff)) > 0x5fff) != 0;
  // s = m 2^e, 1 <= |m| < 2 (m = s, e = 0 for zeros; of no use for the scales above 0x5fff)
  auto mantissa = [](uint16_t h) __attribute__((always_inline)) { return 2.f * __builtin_amdgcn_frexp_mantf((float)__builtin_bit_cast(_Float16, h)); };
  auto power = [](uint16_t h) __attribute__((always_inline)) {  // 2^(e + 10)
    return __builtin_amdgcn_ldexpf(1.f, __builtin_amdgcn_frexp_expf((float)__builtin_bit_cast(_Float16, h)) + 9);
  };
  uint32_t times[4], minus[4];  // per column, in both halves: what the subnormal is multiplied by and what is added; literal: the scale
  static_for<0, 4>([&](auto cc) __attribute__((always_inline)) {
    constexpr int c = decltype(cc)::value;
    const float m = mantissa(s_in[c]);
    const _Float16 t = literal ? __builtin_bit_cast(_Float16, s_in[c]) : (_Float16)(m * 16384.f), o = (_Float16)(m * -0.125f);
    times[c] = (uint32_t)__builtin_bit_cast(uint16_t, t) * 0x10001u;
    minus[c] = (uint32_t)__builtin_bit_cast(uint16_t, o) * 0x10001u;
  });
  const char *a_base = (const char *)((const uint16_t *)p.a + m0 * p.lda);
  const char *w_base = (const char *)p.w + n0;
  const uint32_t lds0 = (uint32_t)(uintptr_t)TTS_LDS(smem);
  // loads past the last tile fetch the last tile again: the wait count is the same in every iteration
  auto fetch = [&](int t, int stage, auto nc) __attribute__((always_inline)) {
    constexpr int n = decltype(nc)::value;
    const int tc = min(t, nk - 1) + k_begin;
    const uint32_t st = lds0 + stage * T::STAGE;
    if constexpr (n < T::A_DMA) load_to_lds(a_base + (int64_t)tc * 128, a_voff[n], st + min(T::A_DMA * wave + n, (uint32_t)(2 * TM - 1)) * 1024);
    else load_to_lds(w_base + (int64_t)tc * 64 * p.ldw, w_voff[n - T::A_DMA], st + T::A_BYTES + (4 * wave + n - T::A_DMA) * 1024);
  };

  // step s of a tile: k 32 s + 8 q .. +7
  const int a_off = l16 * 128, a_sw = (l16 >> 1) & 7;
  const int w_off = T::A_BYTES + 8 * q * W8T_COLS + (((4 * (int)wave + (l16 >> 2)) ^ (q << 2)) << 4) + 4 * (l16 & 3);
  f32x4 acc[TM][4];
  static_for<0, 4 * TM>([&](auto n) __attribute__((always_inline)) { acc[n.value / 4][n.value % 4] = (f32x4){0.f, 0.f, 0.f, 0.f}; });
  typedef uint32_t u32x4_r __attribute__((ext_vector_type(4)));
  uint4 A[2][TM];
  uint32_t raw[8], B[2][4][4];
  auto read_a = [&](int stage, int s, int i, uint4 (&a)[TM]) __attribute__((always_inline)) {
    a[i] = *reinterpret_cast<const uint4 *>(smem + stage * T::STAGE + a_off + i * 2048 + (((4 * s + q) ^ a_sw) << 4));
  };
  auto read_w = [&](int stage, int s, int j) __attribute__((always_inline)) {
    raw[j] = *reinterpret_cast<const uint32_t *>(smem + stage * T::STAGE + w_off + (32 * s + j) * W8T_COLS);
  };
  auto bias_w = [&](int j) __attribute__((always_inline)) { raw[j] ^= 0x80808080u; };  // bytes b + 128
  auto widen = [&](auto lit, int c, int tp, uint32_t (&b)[4][4]) __attribute__((always_inline)) {  // k 2 tp and 2 tp + 1 of column c
    const uint32_t sel = 0x0c000c00u | (uint32_t)c | ((uint32_t)(4 + c) << 16);
    const f16x2 v = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(raw[2 * tp + 1], raw[2 * tp], sel));
    const f16x2 t = __builtin_bit_cast(f16x2, times[c]), o = __builtin_bit_cast(f16x2, minus[c]);
    f16x2 w;
    if constexpr (decltype(lit)::value) {
      const f16x2 up = {(_Float16)32768.0f, (_Float16)32768.0f}, off = {(_Float16)-0.25f, (_Float16)-0.25f}, whole = {(_Float16)512.0f, (_Float16)512.0f};
      w = __builtin_elementwise_fma(v, up, off) * whole;  // b, exactly
      w = w * t;
    } else {
      w = __builtin_elementwise_fma(v, t, o);
    }
    b[c][tp] = __builtin_bit_cast(uint32_t, w);
  };
  // The matrix instruction from inline assembly, in place on the accumulation registers (see gemm_dma16_body).  The
  // compiler inserts no wait states in front of it: its operands are read from LDS or widened a phase earlier.
  auto mfma = [&](int i, int c, const uint4 &a, const uint32_t (&b)[4]) __attribute__((always_inline)) {
    const u32x4_r bv = {b[0], b[1], b[2], b[3]};
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[i][c]) : "v"(bv), "v"(__builtin_bit_cast(u32x4_r, a)));
  };
  // One step: its 4 TM products, with the reads and the widening of the next step (step ns of the tile at stage `next`)
  // dealt out behind them; LOAD: and the loads of tile t into `free`.
  auto step = [&](auto lit, auto load, int next, auto nsc, int t, int free, uint4 (&Ac)[TM], uint4 (&An)[TM], uint32_t (&Bc)[4][4], uint32_t (&Bn)[4][4]) __attribute__((always_inline)) {
    constexpr int ns = decltype(nsc)::value;
    static_for<0, 4 * TM>([&](auto slot) __attribute__((always_inline)) {
      constexpr int n = decltype(slot)::value;
      __builtin_amdgcn_sched_barrier(0);
      mfma(n / 4, n % 4, Ac[n / 4], Bc[n % 4]);
      if constexpr (n == 0) static_for<0, 8>([&](auto j) __attribute__((always_inline)) { read_w(next, ns, j.value); });
      else if constexpr (n <= TM) read_a(next, ns, n - 1, An);
      if constexpr (decltype(load)::value) {
        constexpr int d0 = n * T::DMA / (4 * TM), d1 = (n + 1) * T::DMA / (4 * TM);
        static_for<d0, d1>([&](auto d) __attribute__((always_inline)) { fetch(t, free, d); });
      }
      // sixteen pairs of weights over the slots behind the reads (the last slot is left free)
      constexpr int W0 = TM + 1, WN = 3 * TM - 2;
      if constexpr (n >= W0 && n < W0 + WN)
        static_for<(n - W0) * 24 / WN, (n - W0 + 1) * 24 / WN>([&](auto g) __attribute__((always_inline)) {
          if constexpr (g.value < 8) bias_w(g.value);
          else widen(lit, (g.value - 8) / 4, g.value % 4, Bn);
        });
    });
    __builtin_amdgcn_sched_barrier(0);
  };

  // prologue: STAGES tiles in flight; tile 0 landed, its first step read and widened
  for (int t = 0; t < STAGES; t++) static_for<0, T::DMA>([&](auto n) __attribute__((always_inline)) { fetch(t, t, n); });
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(T::DMA * (STAGES - 1), 15));
  __syncthreads();
  static_for<0, 8>([&](auto j) __attribute__((always_inline)) { read_w(0, 0, j.value); });
  static_for<0, TM>([&](auto i) __attribute__((always_inline)) { read_a(0, 0, i.value, A[0]); });
  static_for<0, 8>([&](auto j) __attribute__((always_inline)) { bias_w(j.value); });
  auto sweep_k = [&](auto lit) __attribute__((always_inline)) {
    static_for<0, 16>([&](auto g) __attribute__((always_inline)) { widen(lit, g.value / 4, g.value % 4, B[0]); });
    __builtin_amdgcn_sched_barrier(0);
    int stage = 0;
    for (int t = 0; t < nk; t++) {
      const int next = stage + 1 == STAGES ? 0 : stage + 1;
      step(lit, BoolConstant<false>(), stage, IntConstant<1>(), 0, 0, A[0], A[1], B[0], B[1]);
      // own loads of tile t + 1 have landed, own reads of tile t are complete: behind the barrier its stage is free
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(T::DMA * (STAGES - 2), 0));
      __syncthreads();
      step(lit, BoolConstant<true>(), next, IntConstant<0>(), t + STAGES, stage, A[1], A[0], B[1], B[0]);
      stage = next;
    }
  };
  if (literal) sweep_k(BoolConstant<true>());
  else sweep_k(BoolConstant<false>());
  // wait states between the last matrix instructions and the first read of their results (see gemm_dma16_body)
  asm volatile("s_nop 15\n\ts_nop 15" : : : "memory");
  auto settle = [](f32x4 &x) __attribute__((always_inline)) { asm volatile("" : "+a"(x) : : "memory"); };
  static_for<0, 4 * TM>([&](auto n) __attribute__((always_inline)) { settle(acc[n.value / 4][n.value % 4]); });

  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
  typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
  const int64_t col = n0 + 64 * (int)wave + 16 * q;
  const bool col_in = col < p.N;  // (N is a multiple of 16)
  static_for<0, 4>([&](auto vc) __attribute__((always_inline)) {
    static_for<0, 4>([&](auto cc) __attribute__((always_inline)) {
      constexpr int v = decltype(vc)::value, c = decltype(cc)::value;
      const float scale = literal ? 1.f : power(s_out[4 * v + c]);
      static_for<0, TM>([&](auto i) __attribute__((always_inline)) { acc[i.value][c][v] *= scale; });
    });
  });
  static_for<0, TM>([&](auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;
    const int64_t row = m0 + 16 * i + l16;
    if (row >= p.M || !col_in) return;
    if constexpr (SK) {
      float *at = partial + ((int64_t)slice * p.M + row) * p.N + col;
      static_for<0, 4>([&](auto vc) __attribute__((always_inline)) {
        constexpr int v = decltype(vc)::value;
        const f32x4 w = {acc[i][0][v], acc[i][1][v], acc[i][2][v], acc[i][3][v]};
        *reinterpret_cast<f32x4 *>(at + 4 * v) = w;
      });
    } else {
      uint16_t *at = (uint16_t *)p.c + row * p.ldc + col;
      static_for<0, 2>([&](auto hc) __attribute__((always_inline)) {
        u32x4_a4 w;
        static_for<0, 4>([&](auto dc) __attribute__((always_inline)) {
          constexpr int d = decltype(dc)::value, v = 2 * decltype(hc)::value + d / 2, c = 2 * (d % 2);
          const f32x2_t pr = {acc[i][c][v], acc[i][c + 1][v]};
          w[d] = __builtin_bit_cast(uint32_t, __builtin_convertvector(pr, f16x2_t));
        });
        __builtin_nontemporal_store(w, reinterpret_cast<u32x4_a4 *>(at + 8 * hc.value));
      });
    }
  });
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));  // the surplus loads land before the LDS goes away
}

struct W8TileChoice { int tm, tiles_m, tiles_n, split; };
// Row blocks per tile and K slices: the least modelled time.  A K tile of 64 takes a workgroup 0.2 us and 0.077 us per row
// block (the matrix pipe), 0.5 us at least (its loads); the weights cross the memory at 5.5 TB/s whatever the tiles; slices
// cost a second launch and their sums' way through memory.  (Measured at [8192, 28672], model in brackets: 48 rows 47 to 49 us (58),
// 300 rows 126 to 136 (131), 400 rows 191 to 204 (197), 512 rows 209 to 224 (216), 1024 rows 414 to 446 (425).)
W8TileChoice w8_tile_choice(const GemmW8A16Params &p) {
  W8TileChoice best{};
  double best_t = 0;
  const int64_t nk = p.K / 64;
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    return n;
  }();
  for (int tm = 1; tm <= W8T_MAX_TM; tm++) {
    W8TileChoice c;
    c.tm = tm;
    c.tiles_m = (int)((p.M + 16 * tm - 1) / (16 * tm));
    c.tiles_n = (int)((p.N + W8T_COLS - 1) / W8T_COLS);
    for (c.split = 1; c.split <= 16 && (c.split == 1 || nk / c.split >= 4); c.split++) {
      const int64_t wgs = (int64_t)c.tiles_m * c.tiles_n * c.split, rounds = (wgs + cus - 1) / cus;
      double t = std::max((double)(rounds * ((nk + c.split - 1) / c.split)) * std::max(0.5e-6, 0.2e-6 + 0.077e-6 * tm), (double)p.K * (double)p.N / 5.5e12) + 7e-6;
      if (c.split > 1) t += 3e-6 + 8.0 * c.split * (double)p.M * (double)p.N / 4.5e12;
      if (best.tm == 0 || t < best_t) { best = c; best_t = t; }
    }
  }
  return best;
}

template <int TM>
hipError_t w8_tile_launch(const GemmW8A16Params &p, const W8TileChoice &c, hipStream_t s) {
  using T = W8Tile<TM>;
  auto kern = c.split > 1 ? gemm_w8a16_tile_kernel<TM, true> : gemm_w8a16_tile_kernel<TM, false>;
  static const hipError_t attr = [] {
    hipError_t e = hipFuncSetAttribute((const void *)gemm_w8a16_tile_kernel<TM, false>, hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
    return e != hipSuccess ? e : hipFuncSetAttribute((const void *)gemm_w8a16_tile_kernel<TM, true>, hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
  }();
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(kern, dim3(c.tiles_m * c.tiles_n * c.split), dim3(256), T::LDS, s, p, c.tiles_m, c.tiles_n, c.split, p.partial);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || c.split == 1) return e;
  GemmParams g{};
  g.c = p.c; g.ldc = p.ldc; g.M = p.M; g.N = p.N; g.split = c.split; g.partial = p.partial; g.batches = 1;
  return launch_splitk_reduce(g, s);
}
}  // namespace

// Whole K tiles, 16-byte aligned rows of A and W, whole 16-column groups of C in 4-byte aligned rows, per-lane offsets of 32 bits.
bool w8_tile_ok(const GemmW8A16Params &p) {
  return p.M >= 1 && p.K % 64 == 0 && p.K >= 64 && p.N % 16 == 0 && p.N >= 16 && p.lda % 8 == 0 && p.ldw % 16 == 0 && p.ldc % 2 == 0 && ((uintptr_t)p.a & 15) == 0 &&
         ((uintptr_t)p.w & 15) == 0 && ((uintptr_t)p.c & 3) == 0 && p.lda < (1 << 22) && p.ldw < (1 << 25);
}

size_t w8_tile_partial_bytes(const GemmW8A16Params &p) {
  const W8TileChoice c = w8_tile_choice(p);
  return c.split > 1 ? (size_t)c.split * p.M * p.N * sizeof(float) : 0;
}

hipError_t launch_w8_tile(const GemmW8A16Params &p, hipStream_t s) {
  W8TileChoice c = w8_tile_choice(p);
  if (!p.partial) c.split = 1;
  switch (c.tm) {
    case 1: return w8_tile_launch<1>(p, c, s);
    case 2: return w8_tile_launch<2>(p, c, s);
    case 3: return w8_tile_launch<3>(p, c, s);
    case 4: return w8_tile_launch<4>(p, c, s);
    case 5: return w8_tile_launch<5>(p, c, s);
    case 6: return w8_tile_launch<6>(p, c, s);
    case 7: return w8_tile_launch<7>(p, c, s);
    case 8: return w8_tile_launch<8>(p, c, s);
    case 9: return w8_tile_launch<9>(p, c, s);
    default: return w8_tile_launch<10>(p, c, s);
  }
}

}  // namespace tts
