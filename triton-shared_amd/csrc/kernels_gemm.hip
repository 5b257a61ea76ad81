// MFMA kernel families for gfx950: 16-bit GEMM with fp32 accumulate, and the
// weight-only int8 GEMM at decode shapes (M <= 16).
//
// What they replace in the reference CPU path: per program and per K step, two
// malloc'd operand tiles filled with 0 and partially copied
// (StructuredToMemref.cpp:794-853), linalg.matmul on operands widened to f32 into
// a zero tile, an elementwise add into the loop-carried accumulator
// (ConversionPatterns.hpp:1171-1196), a truncf tile (RTNE) and a partial copy out
// (StructuredToMemref.cpp:1163-1196); the int8 variant adds a sitofp tile and a
// mulf tile per K step.  The launcher has proved that the grid of programs is a
// dense C = A*B, so these kernels choose their own tiling.
#include "kernels.h"

#include <cmath>
#include <cstring>

namespace tts {

namespace {

using namespace tts_gemm_device;

struct IdentityEp {
  static constexpr int BM = 0, BN = 0;  // (no owner to look up: see the generated functor, tile_codegen.cpp)
  __device__ __forceinline__ float operator()(float x, int64_t, int64_t) const { return x; }
};

// the kernels' device code is in gemm_device.h (it is also compiled at run time, with a fused epilogue)
template <bool BF16, int TM, int TN, int BK, bool SK>
__global__ __launch_bounds__(256) void gemm_mfma_kernel(GemmParams p, int tiles_m, int tiles_n) {
  gemm_mfma_body<BF16, TM, TN, BK, IdentityEp, SK>(of_batch(p, 2), tiles_m, tiles_n, IdentityEp());
}

template <bool BF16>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_any_kernel(GemmParams p, int across, int col_blocks) {
  gemm_splitk_reduce_body<BF16>(of_batch(p, 2), across, col_blocks, IdentityEp());
}

// the grid of gemm_splitk_reduce_body
struct ReduceGrid {
  int across, col_blocks, workgroups;
  explicit ReduceGrid(const GemmParams &p) {
    for (across = 16; across < 256 && across < p.N; across *= 2) {}
    col_blocks = (int)((p.N + across - 1) / across);
    workgroups = (int)((p.M + 256 / across - 1) / (256 / across)) * col_blocks;
  }
};

int device_cus() {  // of the current device (256 when the query fails)
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    return n;
  }();
  return cus;
}
// The height of the any-shape kernel's tiles, 64 or 128 rows (their width is 128).  What bounds the kernel on a full chip is the
// rate at which a CU takes 16-byte loads off the 16-byte grid, and the larger tile loads a third less for the same product
// (4001 x 4003 x 4005 bf16: 208 us against 298; 3001 x 3003 x 1001 52.8 / 56.4).  Up to one and a half of the larger tiles per CU
// the smaller ones spread better, or pad fewer rows (us with 128 / 64 rows: 33 x 4001 x 4001 21.2 / 13.5, 3001 x 401 x 2003 29.9 /
// 23.5, 64 x 1003 x 517 17.6 / 11.8, 2000 x 1000 x 520 16.8 / 11.9, 1000 x 3001 x 1003 26.4 / 25.2, 2001 x 2003 x 2005 43.3 / 44.2).
int any_rows(const GemmParams &p, int split) {
  static const char *env = getenv("TTS_GEMM_ROWS");  // tuning aid: "64" or "128"
  if (env) return atoi(env) == 64 ? 64 : 128;
  const int64_t tiles = ((p.M + 127) / 128) * ((p.N + 127) / 128) * std::max(1, p.batches) * split;
  return p.M <= 64 || 2 * tiles <= 3 * device_cus() ? 64 : 128;
}

// p.split > 1: the slices alone; whoever launches it adds them
template <bool BF16, bool SK, int TM>
hipError_t launch_gemm_any_t(const GemmParams &p, hipStream_t s) {
  constexpr size_t lds = GemmStageLds<64 * TM, 128, 64>::BYTES;
  auto kern = gemm_mfma_kernel<BF16, TM, 2, 64, SK>;
  static const hipError_t attr = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return attr;
  const int tiles_m = (int)((p.M + 64 * TM - 1) / (64 * TM)), tiles_n = (int)((p.N + 127) / 128);
  hipLaunchKernelGGL(kern, dim3(tiles_m * tiles_n * (SK ? p.split : 1), std::max(1, p.batches)), dim3(256), lds, s, p, tiles_m, tiles_n);
  return hipGetLastError();
}
template <bool BF16, bool SK>
hipError_t launch_gemm_any(const GemmParams &p, hipStream_t s) {
  return any_rows(p, SK ? p.split : 1) == 64 ? launch_gemm_any_t<BF16, SK, 1>(p, s) : launch_gemm_any_t<BF16, SK, 2>(p, s);
}
const char *any_name(int64_t rows, bool functor, bool sliced) {  // of the any-shape kernel in tiles of that height
  static const char *names[2][2][2] = {{{"gemm_mfma_kernel<128x128x64>", "gemm_mfma_kernel<128x128x64>, K slices"},
                                        {"gemm_mfma_kernel<128x128x64> + epilogue (hipRTC)", "gemm_mfma_kernel<128x128x64> + epilogue (hipRTC), K slices"}},
                                       {{"gemm_mfma_kernel<64x128x64>", "gemm_mfma_kernel<64x128x64>, K slices"},
                                        {"gemm_mfma_kernel<64x128x64> + epilogue (hipRTC)", "gemm_mfma_kernel<64x128x64> + epilogue (hipRTC), K slices"}}};
  return names[rows == 64][functor][sliced];
}
hipError_t launch_gemm_any_slices(const GemmParams &p, hipStream_t s) { return p.is_bf16 ? launch_gemm_any<true, true>(p, s) : launch_gemm_any<false, true>(p, s); }

// PF: a fifth wavefront that touches B's lines ahead of the four that work (gemm_device.h); the accumulators then sit in
// the 256 registers two wavefronts of a SIMD can have each, which the 128 x 256 tile fits without spilling.
template <bool BF16, int TM, int TN, bool BT, bool AT, bool PF, bool SK>
__global__ __launch_bounds__(PF ? 320 : 256) void gemm_dma_kernel(GemmParams p, int tiles_m, int tiles_n) {
  // whole 256 x 256 tiles of row-major operands: the body on the 16 x 16 x 32 matrix instruction (gemm_device.h)
  if constexpr (TM == 4 && TN == 4 && !BT && !AT && !PF) gemm_dma16_body<BF16, IdentityEp, SK>(of_batch(p, 2), tiles_m, tiles_n, IdentityEp());
  else gemm_dma_body<BF16, TM, TN, IdentityEp, BT, AT, PF, SK>(of_batch(p, 2), tiles_m, tiles_n, IdentityEp());
}

// Adds the K slices' partial sums in slice order and narrows: four columns per thread (N is a multiple of 8).
template <bool BF16>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(GemmParams batch) {
  const GemmParams p = of_batch(batch, 2);
  const int64_t quads = p.N / 4, idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= p.M * quads) return;
  const int64_t m = idx / quads, n = (idx % quads) * 4;
  const float4 *src = reinterpret_cast<const float4 *>(p.partial + m * p.N + n);
  float4 t = src[0];
  for (int sl = 1; sl < p.split; sl++) {
    const float4 u = src[(int64_t)sl * p.M * quads];
    t.x += u.x; t.y += u.y; t.z += u.z; t.w += u.w;
  }
  typedef float f32x4_t __attribute__((ext_vector_type(4)));
  typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
  typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
  const f32x4_t v = {t.x, t.y, t.z, t.w};
  uint16_t *dst = (uint16_t *)p.c + m * p.ldc + n;
  const uint2 w = BF16 ? __builtin_bit_cast(uint2, __builtin_convertvector(v, bf16x4_t)) : __builtin_bit_cast(uint2, __builtin_convertvector(v, f16x4_t));
  reinterpret_cast<uint32_t *>(dst)[0] = w.x;  // (rows of C are 4-byte aligned: gemm_dma_ok)
  reinterpret_cast<uint32_t *>(dst)[1] = w.y;
}

// p.split K slices of a product; whoever launches them adds them
template <bool BF16, int TM, int TN, bool BT, bool AT>
hipError_t launch_gemm_dma_slices(const GemmParams &p, hipStream_t s) {
  using T = DmaTile<TM, TN>;
  constexpr size_t lds = T::LDS_BYTES;
  auto kern = gemm_dma_kernel<BF16, TM, TN, BT, AT, false, true>;
  static const hipError_t attr = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return attr;
  int tiles_m = (int)((p.M + T::BM - 1) / T::BM), tiles_n = (int)((p.N + T::BN - 1) / T::BN);
  hipLaunchKernelGGL(kern, dim3(tiles_m * tiles_n * p.split, std::max(1, p.batches)), dim3(256), lds, s, p, tiles_m, tiles_n);
  return hipGetLastError();
}

// 128 x 128 tiles in K slices that meet in the kernel (slices_meet; chosen by choose_dma)
template <bool BF16, bool BT, bool AT>
__global__ __launch_bounds__(256) void gemm_dma_meeting_kernel(GemmParams p, int tiles_m, int tiles_n) {
  gemm_dma_body<BF16, 2, 2, IdentityEp, BT, AT, false, true, true>(p, tiles_m, tiles_n, IdentityEp());
}

template <bool BF16, int TM, int TN, bool BT, bool AT, bool PF = false>
hipError_t launch_gemm_dma_t(const GemmParams &p, hipStream_t s) {
  using T = DmaTile<TM, TN>;
  constexpr size_t lds = T::LDS_BYTES;
  if constexpr (!PF && TM == 2 && TN == 2) {
    if (p.split > 1 && p.counters) {
      auto kern = gemm_dma_meeting_kernel<BF16, BT, AT>;
      static const hipError_t attr = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (attr != hipSuccess) return attr;
      const int tiles_m = (int)((p.M + 127) / 128), tiles_n = (int)((p.N + 127) / 128);
      hipLaunchKernelGGL(kern, dim3(tiles_m * tiles_n * p.split), dim3(256), lds, s, p, tiles_m, tiles_n);
      return hipGetLastError();
    }
  }
  if constexpr (!PF) {
    if (p.split > 1) {
      hipError_t e = launch_gemm_dma_slices<BF16, TM, TN, BT, AT>(p, s);
      if (e != hipSuccess) return e;
      hipLaunchKernelGGL(gemm_splitk_reduce_kernel<BF16>, dim3((unsigned)((p.M * (p.N / 4) + 255) / 256), std::max(1, p.batches)), dim3(256), 0, s, p);
      return hipGetLastError();
    }
  }
  // Row tiles with weight matrices of their own (p.b_block) stream B from HBM: they get the prefetching wavefront.
  if constexpr (!PF && TM == 2 && TN == 4 && !BT && !AT) {
    static const char *pf = getenv("TTS_GEMM_PREFETCH");  // tuning aid: "0" = never, "2" = for every launch of this tile
    if (pf ? pf[0] == '2' || (pf[0] != '0' && p.b_block) : p.b_block != nullptr) return launch_gemm_dma_t<BF16, TM, TN, BT, AT, true>(p, s);
  }
  auto kern = gemm_dma_kernel<BF16, TM, TN, BT, AT, PF, false>;
  static const hipError_t attr = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return attr;
  int tiles_m = (int)((p.M + T::BM - 1) / T::BM), tiles_n = (int)((p.N + T::BN - 1) / T::BN);
  hipLaunchKernelGGL(kern, dim3(tiles_m * tiles_n, std::max(1, p.batches)), dim3(PF ? 320 : 256), lds, s, p, tiles_m, tiles_n);
  return hipGetLastError();
}

// one instantiation per layout of the operands in memory
template <bool BF16, int TM, int TN>
hipError_t launch_gemm_dma(const GemmParams &p, hipStream_t s) {
  if (p.a_trans) return p.b_trans ? launch_gemm_dma_t<BF16, TM, TN, true, true>(p, s) : launch_gemm_dma_t<BF16, TM, TN, false, true>(p, s);
  return p.b_trans ? launch_gemm_dma_t<BF16, TM, TN, true, false>(p, s) : launch_gemm_dma_t<BF16, TM, TN, false, false>(p, s);
}

// Whole K tiles of 32, N a multiple of 8 (whole 16-byte chunks of B rows), any M (a multiple of 8 when A is column-major);
// 16-byte aligned rows, and per-lane byte offsets that fit 32 bits.  Either operand may be column-major.  Tiles that
// stick out of C clamp their addresses and mask their stores.
bool gemm_dma_ok(const GemmParams &p, int64_t bm, int64_t bn) {
  if (p.a_trans && (p.M % 8 != 0 || p.a_rows || p.b_block)) return false;
  if ((p.a_rows || p.b_block) && bm != 128) return false;  // gathered rows: 128-row tiles (64-bit A addresses per lane)
  if (p.b_block && p.b_block_rows % bm != 0) return false;
  if (p.batches > 1 && (p.batch_a % 8 != 0 || p.batch_b % 8 != 0 || p.batch_c % 2 != 0)) return false;  // every product aligned like the first
  return p.M >= 1 && p.N >= 8 && p.N % 8 == 0 && p.K % F_BK == 0 && p.K >= F_BK && p.lda % 8 == 0 && p.ldb % 8 == 0 &&
         ((uintptr_t)p.a & 15) == 0 && ((uintptr_t)p.b & 15) == 0 && p.lda < (p.a_trans ? (1 << 25) : (1 << 22)) && p.ldb < (p.b_trans ? (1 << 22) : (1 << 25)) &&
         (!p.b_block || p.b_block_stride % 8 == 0) && p.ldc % 2 == 0 && ((uintptr_t)p.c & 3) == 0;  // C is written in 4-byte pairs
}
bool gemm_fast_path_ok(const GemmParams &p) { return !p.a_trans && !p.b_trans && gemm_dma_ok(p, F_BM, F_BN); }  // (the kernel compiled with an epilogue)

// ------------------------------------------------------------- fp32 GEMM (gemm_device.h: gemm_f32_body)
template <int T, int W, int G>
__global__ __launch_bounds__(64 * W * W * G) void gemm_f32_kernel(GemmParams batch, int tiles_m, int tiles_n) {
  gemm_f32_body<T, W, G>(of_batch(batch, 4), tiles_m, tiles_n, IdentityEp());
}

// The tilings gemm_f32_body is built for: edge of a workgroup's tile, threads.
struct F32Tiling { int edge, threads; };
constexpr F32Tiling F32_TILINGS[4] = {{128, 256}, {32, 256}, {64, 512}, {64, 256}};
int f32_tiling(const GemmParams &p) {
  const int cus = device_cus();
  auto tiles = [&](int64_t t) { return ((p.M + t - 1) / t) * ((p.N + t - 1) / t) * std::max(1, p.batches); };
  // Where the lines lie, us with 64 x 64 tiles / those in two groups / 32 x 32 tiles in four: 400 x 600 x 800 23.1 / 21.7 / 11.9;
  // 768^3 (576 small tiles) 22.3 / 20.7 / 17.6; 1000^3 (1024) 30.1 / 27.3 / 36.8; 1024 x 2048 x 1024 (512 tiles of 64) 49.0 /
  // 48.6 / 62.9; 1500 x 1500 x 1000 (576) 65.5 / 67.1 / 75.0.
  if (tiles(128) >= 2 * cus) return 0;
  if (2 * tiles(32) <= 5 * cus) return 1;
  return tiles(64) <= 2 * cus ? 2 : 3;
}
hipError_t launch_gemm_f32(const GemmParams &p, hipStream_t s) {
  const int which = f32_tiling(p), t = F32_TILINGS[which].edge;
  const int tiles_m = (int)((p.M + t - 1) / t), tiles_n = (int)((p.N + t - 1) / t);
  const auto kern = which == 0 ? gemm_f32_kernel<2, 2, 1> : which == 1 ? gemm_f32_kernel<1, 1, 4> : which == 2 ? gemm_f32_kernel<1, 2, 2> : gemm_f32_kernel<1, 2, 1>;
  hipLaunchKernelGGL(kern, dim3(tiles_m * tiles_n, std::max(1, p.batches)), dim3(F32_TILINGS[which].threads), 0, s, p, tiles_m, tiles_n);
  return hipGetLastError();
}

// ------------------------------------------------------ int8-weight GEMM
// Workgroup: NW wavefronts share one 128-column slab of W and split its K range
// in interleaved steps of 32 rows.  In a step, lane (j = lane % 16, g = lane / 16)
// streams rows 8g..8g+7 of the step, 8 columns (8 bytes) each, so that a
// 16-lane group reads 128 contiguous bytes of a row.  Bytes are widened to fp16
// exactly (bit pattern 0x6400 | (b ^ 0x80) is 1152 + b), multiplied by the
// column's fp16 scale in fp16 as the Triton source does, and fed to eight
// 16x16x32 MFMAs, one per column of the lane's eight.
constexpr int W8_COLS = 128;       // slab width of the 8-byte-load kernel
constexpr int W8_COLS_WIDE = 256;  // and of the 16-byte-load kernel

__device__ __forceinline__ uint32_t pk_sub_1152_mul(uint32_t biased, uint32_t scale2) {
  f16x2 v = __builtin_bit_cast(f16x2, biased);
  f16x2 s = __builtin_bit_cast(f16x2, scale2);
  const f16x2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
  v = v - off;  // exact: integers in [-128, 127]
  v = v * s;    // one fp16 rounding, as arith.mulf on f16
  return __builtin_bit_cast(uint32_t, v);
}

// FAST: K is a multiple of 32, N of 128, rows are 8/16-byte aligned: every load is unconditional,
// so that the compiler keeps all loads of a step (and of DEPTH steps) in flight.  Rows of A beyond
// M are read from row M-1: they only reach rows of the MFMA result that are never stored.
// CW: columns per lane (8: 8-byte weight loads, 128-column slabs; 16: 16-byte loads, 256-column
// slabs, FAST only).
template <int NW, int DEPTH, bool FAST, int CW>
__global__ __launch_bounds__(NW * 64) void gemm_w8a16_kernel(GemmW8A16Params p, int steps_per_slice) {
  static_assert(CW == 8 || (CW == 16 && FAST), "wide slabs exist on the unconditional path only");
  constexpr int W8_COLS = 16 * CW;
  constexpr int RW = NW > (CW == 8 ? 4 : 2) ? (CW == 8 ? 4 : 2) : NW;  // wavefronts combined per round
  using wvec = typename std::conditional<CW == 8, uint2, uint4>::type;
  __shared__ float red[RW][16][W8_COLS + 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int j = lane & 15, g = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * W8_COLS;
  const int slice = blockIdx.y;
  const uint16_t *__restrict__ A = (const uint16_t *)p.a;
  const int8_t *__restrict__ W = p.w;
  const uint16_t *__restrict__ S = (const uint16_t *)p.scale;
  const int K = (int)p.K;
  const bool a_vec = (p.lda % 8 == 0) && (((uintptr_t)A & 15) == 0);
  const bool w_vec = (p.ldw % 8 == 0) && (((uintptr_t)W & 7) == 0);
  const int64_t ncol = n0 + CW * j;                      // first of this lane's CW columns
  const int ncols = (int)max((int64_t)0, min((int64_t)CW, p.N - ncol));

  uint32_t scale2[CW];
#pragma unroll
  for (int c = 0; c < CW; c++) {
    uint32_t s = c < ncols ? S[ncol + c] : 0;
    scale2[c] = s | (s << 16);
  }
  f32x4 acc[CW];
#pragma unroll
  for (int c = 0; c < CW; c++) acc[c] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int step_begin = slice * steps_per_slice;
  const int step_end = min(step_begin + steps_per_slice, (K + 31) / 32);

  const int8_t *w_lane = W + (int64_t)(8 * g) * p.ldw + ncol;
  const uint16_t *a_lane = A + (int64_t)min(j, (int)p.M - 1) * p.lda + 8 * g;
  auto load_w = [&](int step, wvec (&q)[8]) {
    if constexpr (FAST) {
      const int8_t *src = w_lane + (int64_t)step * 32 * p.ldw;
#pragma unroll
      for (int t = 0; t < 8; t++) q[t] = *reinterpret_cast<const wvec *>(src + (int64_t)t * p.ldw);
      return;
    } else {
#pragma unroll
    for (int t = 0; t < 8; t++) {
      int k = step * 32 + 8 * g + t;
      if (k < K && ncols == 8 && w_vec) {
        q[t] = *reinterpret_cast<const uint2 *>(W + (int64_t)k * p.ldw + ncol);
      } else {
        uint32_t lo = 0, hi = 0;
        if (k < K)
          for (int c = 0; c < ncols; c++) {
            uint32_t b = (uint8_t)W[(int64_t)k * p.ldw + ncol + c];
            if (c < 4) lo |= b << (8 * c);
            else hi |= b << (8 * (c - 4));
          }
        q[t] = make_uint2(lo, hi);
      }
    }
    }
  };
  auto load_a = [&](int step) {
    if (FAST) return *reinterpret_cast<const uint4 *>(a_lane + step * 32);
    int k = step * 32 + 8 * g;
    return j < p.M ? load8(A + (int64_t)j * p.lda + k, K - k, a_vec) : make_uint4(0, 0, 0, 0);
  };

  auto word = [](const wvec &v, int i) -> uint32_t {
    if constexpr (CW == 8) return i == 0 ? v.x : v.y;
    else return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
  };
  auto consume = [&](const wvec (&q)[8], const uint4 &af) {
#pragma unroll
    for (int c = 0; c < CW; c++) {
      uint32_t frag[4];
#pragma unroll
      for (int tp = 0; tp < 4; tp++) {
        uint32_t w0 = word(q[2 * tp], c / 4);
        uint32_t w1 = word(q[2 * tp + 1], c / 4);
        // bytes [w0.b, 0, w1.b, 0], then flip the sign bit and set the exponent: 0x6400 | (b ^ 0x80)
        uint32_t sel = 0x0c000c00u | (uint32_t)(c & 3) | ((uint32_t)(4 + (c & 3)) << 16);
        uint32_t pair = __builtin_amdgcn_perm(w1, w0, sel) ^ 0x64806480u;
        frag[tp] = pk_sub_1152_mul(pair, scale2[c]);
      }
      uint4 bfrag = make_uint4(frag[0], frag[1], frag[2], frag[3]);
      acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, af), __builtin_bit_cast(f16x8, bfrag), acc[c], 0, 0, 0);
    }
  };
  // DEPTH steps are in flight in DEPTH register sets (the loop is unrolled over them, so no
  // copies), giving a step's loads the time of DEPTH steps' arithmetic to arrive
  wvec q[DEPTH][8];
  uint4 a[DEPTH];
  int step = step_begin + wave;
#pragma unroll
  for (int d = 0; d < DEPTH; d++)
    if (step + d * NW < step_end) { load_w(step + d * NW, q[d]); a[d] = load_a(step + d * NW); }
  for (; step < step_end; step += DEPTH * NW) {
#pragma unroll
    for (int d = 0; d < DEPTH; d++) {
      if (step + d * NW < step_end) {
        consume(q[d], a[d]);
        if (step + (d + DEPTH) * NW < step_end) { load_w(step + (d + DEPTH) * NW, q[d]); a[d] = load_a(step + (d + DEPTH) * NW); }
      }
    }
  }

  // combine the wavefronts' partial tiles through LDS, RW wavefronts at a time;
  // lane holds rows 4g+v (v = 0..3) of column n0 + CW*j + c
  constexpr int ROUNDS = (NW + RW - 1) / RW;
  constexpr int PER_THREAD = (16 * W8_COLS + NW * 64 - 1) / (NW * 64);
  float total[PER_THREAD];
#pragma unroll
  for (int e = 0; e < PER_THREAD; e++) total[e] = 0.f;
  for (int r = 0; r < ROUNDS; r++) {
    if (r) __syncthreads();
    if (wave / RW == r) {
#pragma unroll
      for (int c = 0; c < CW; c++)
#pragma unroll
        for (int v = 0; v < 4; v++) red[wave % RW][4 * g + v][CW * j + c] = acc[c][v];
    }
    __syncthreads();
    const int live = min(RW, NW - RW * r);
#pragma unroll
    for (int e = 0; e < PER_THREAD; e++) {
      int idx = tid + e * NW * 64;
      if (idx < 16 * W8_COLS) {
        int m = idx / W8_COLS, n = idx % W8_COLS;
        for (int w = 0; w < live; w++) total[e] += red[w][m][n];
      }
    }
  }
  uint16_t *__restrict__ C = (uint16_t *)p.c;
#pragma unroll
  for (int e = 0; e < PER_THREAD; e++) {
    int idx = tid + e * NW * 64;
    if (idx >= 16 * W8_COLS) continue;
    int m = idx / W8_COLS;
    int64_t n = n0 + idx % W8_COLS;
    if (m >= p.M || n >= p.N) continue;
    if (p.split > 1) p.workspace[((int64_t)slice * 16 + m) * p.N + n] = total[e];
    else C[(int64_t)m * p.ldc + n] = f32_to_f16(total[e]);
  }
}

// Ints from one slab's arrival counter to the next: the arrivals of many slices in one line would wait for each other.
__host__ __device__ constexpr int w8_counter_pitch(int split) { return split > 4 ? 32 : 1; }

// Partial tiles cross between workgroups (and so between the XCDs' L2 caches) through agent-scope
// relaxed atomic accesses: the stores are written through to memory and the loads bypass stale
// lines, without the whole-cache write-back and invalidate that a release/acquire pair costs
// (measured: 8 us per launch at the decode shape against 3 us this way).
__device__ __forceinline__ void store_through(float4 *dst, float4 v) {
  unsigned long long *d = reinterpret_cast<unsigned long long *>(dst);
  ulonglong2 u = __builtin_bit_cast(ulonglong2, v);
  __hip_atomic_store(d, u.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(d + 1, u.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float4 load_through(float4 *src) {
  unsigned long long *d = reinterpret_cast<unsigned long long *>(src);
  ulonglong2 u;
  u.x = __hip_atomic_load(d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  u.y = __hip_atomic_load(d + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return __builtin_bit_cast(float4, u);
}

// The decode shape's kernel: 256-column slabs, 16-byte weight loads (a lane holds 16 columns of
// 8 rows per step), one workgroup per (slab, K slice).  Requires K % 32 == 0, N % 16 == 0 (the last slab may have fewer columns),
// 16-byte-aligned rows of W and A.
//
// Tail: the NW wavefronts' partial tiles are summed through LDS in one round (float4 per lane,
// conflict-free).  With split > 1 every workgroup writes its slice's tile through to its workspace
// slot, waits for the stores' acknowledgement, and bumps the slab's arrival counter; the workgroup
// that arrives last adds the slices in slice order (so the sum does not depend on the order of
// arrival), writes C, and resets the counter for the next launch.  No workgroup waits for another.
// The counters are zero between launches (whoever allocates them clears them once).  Launches
// that share a workspace must not overlap.
// MT: groups of 16 rows of A a launch takes (1 or 2).  The weights are widened once per step and multiplied with every
// group's rows; the tails below (the sum over the wavefronts, the hand-over between K slices, the stores) run once per group.
// ANY: more than four slices, or a last slab of fewer columns (in a kernel of its own: whole slabs in few slices run 0.4 us of 42.4
// longer on it at the decode shape).
template <int NW, int MT, bool ANY>
__global__ __launch_bounds__(NW * 64) void gemm_w8a16_wide_kernel(GemmW8A16Params p, int first_steps, int other_steps) {
  extern __shared__ float4 w8_lds[];  // [NW][16][64]
  __shared__ int is_last;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int j = lane & 15, g = lane >> 4;
  const int slab = blockIdx.x, slice = blockIdx.y;
  const int64_t n0 = (int64_t)slab * W8_COLS_WIDE;
  const int col = ANY ? min(16 * j, (int)min(p.N - 16 - n0, (int64_t)W8_COLS_WIDE)) : 16 * j;  // this lane's sixteen of the slab (behind the last: others, which are not stored)
  const uint16_t *__restrict__ S = (const uint16_t *)p.scale;

  uint32_t scale2[16];
  {
    const uint4 *sp = reinterpret_cast<const uint4 *>(S + n0 + col);
    const bool s_vec = (((uintptr_t)S) & 15) == 0;
    uint16_t sv[16];
    if (s_vec) {
      uint4 lo = sp[0], hi = sp[1];
      uint32_t wds[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
      for (int c = 0; c < 16; c++) sv[c] = (uint16_t)(wds[c / 2] >> (16 * (c & 1)));
    } else {
#pragma unroll
      for (int c = 0; c < 16; c++) sv[c] = S[n0 + col + c];
    }
#pragma unroll
    for (int c = 0; c < 16; c++) scale2[c] = (uint32_t)sv[c] | ((uint32_t)sv[c] << 16);
  }
  f32x4 acc[MT][16];
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int c = 0; c < 16; c++) acc[m][c] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // slice 0 takes first_steps steps of 32 rows, every other slice other_steps
  const int step_begin = slice == 0 ? 0 : first_steps + (slice - 1) * other_steps;
  const int step_end = min(step_begin + (slice == 0 ? first_steps : other_steps), (int)(p.K / 32));
  const int8_t *w_lane = p.w + (int64_t)(8 * g) * p.ldw + n0 + col;
  const uint16_t *a_lane[MT];
#pragma unroll
  for (int m = 0; m < MT; m++) a_lane[m] = (const uint16_t *)p.a + (int64_t)min(16 * m + j, (int)p.M - 1) * p.lda + 8 * g;

  auto load_w = [&](int step, uint4 (&q)[8]) {
    const int8_t *src = w_lane + (int64_t)step * 32 * p.ldw;
#pragma unroll
    for (int t = 0; t < 8; t++) {
      // the weights are read once per launch: nontemporal, so that they do not displace A, the scales and the partial
      // tiles from the caches (46.2 -> 43.1 us at the decode shape with the weights coming from HBM)
      typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
      const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src + (int64_t)t * p.ldw));
      q[t] = make_uint4(v[0], v[1], v[2], v[3]);
    }
  };
  auto load_a = [&](int step, uint4 (&af)[MT]) {
#pragma unroll
    for (int m = 0; m < MT; m++) af[m] = *reinterpret_cast<const uint4 *>(a_lane[m] + step * 32);
  };
  auto word = [](const uint4 &v, int i) -> uint32_t { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; };
  auto consume = [&](const uint4 (&q)[8], const uint4 (&af)[MT]) {
#pragma unroll
    for (int c = 0; c < 16; c++) {
      uint32_t frag[4];
#pragma unroll
      for (int tp = 0; tp < 4; tp++) {
        // bytes [w0.b, 0, w1.b, 0], then flip the sign bit and set the exponent: 0x6400 | (b ^ 0x80)
        uint32_t sel = 0x0c000c00u | (uint32_t)(c & 3) | ((uint32_t)(4 + (c & 3)) << 16);
        uint32_t pair = __builtin_amdgcn_perm(word(q[2 * tp + 1], c / 4), word(q[2 * tp], c / 4), sel) ^ 0x64806480u;
        frag[tp] = pk_sub_1152_mul(pair, scale2[c]);
      }
      uint4 bfrag = make_uint4(frag[0], frag[1], frag[2], frag[3]);
#pragma unroll
      for (int m = 0; m < MT; m++)
        acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, af[m]), __builtin_bit_cast(f16x8, bfrag), acc[m][c], 0, 0, 0);
    }
  };
  // one step in flight per wavefront; two measured 1.2 us slower at the decode shape
  uint4 q[8];
  uint4 a[MT];
  int step = step_begin + wave;
  if (step < step_end) { load_w(step, q); load_a(step, a); }
  for (; step < step_end; step += NW) {
    consume(q, a);
    if (step + NW < step_end) { load_w(step + NW, q); load_a(step + NW, a); }
  }

  // sum the wavefronts' tiles: entry (c, lane) is rows 4g..4g+3 (of the group) of column n0 + 16j + c
  constexpr int PER = 1024 / (NW * 64);
  float4 tot[MT][PER];
#pragma unroll
  for (int m = 0; m < MT; m++) {
    if (m) __syncthreads();  // the previous group's tiles have been read
#pragma unroll
    for (int c = 0; c < 16; c++) w8_lds[(wave * 16 + c) * 64 + lane] = __builtin_bit_cast(float4, acc[m][c]);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < PER; e++) {
      const int idx = tid + e * NW * 64;
      float4 t = w8_lds[idx];
#pragma unroll
      for (int w = 1; w < NW; w++) {
        float4 u = w8_lds[w * 1024 + idx];
        t.x += u.x; t.y += u.y; t.z += u.z; t.w += u.w;
      }
      tot[m][e] = t;
    }
  }
  if (p.split > 1) {
    // a slab's slots: [slice][group][1024 float4]
    float4 *slots = reinterpret_cast<float4 *>(p.workspace) + (int64_t)slab * p.split * MT * 1024;
    int *counter = p.counters + w8_counter_pitch(p.split) * slab;
    // tot = the slices' tiles added in slice order, whoever adds them (so the sum does not depend on who arrived when);
    // `self` is this workgroup's slice, whose tile is tot.  Four or eight slices at a time, every load is issued before the first add: one round trip to memory instead of one per slice, of which 25 slices (15 x 2048 x 6400) made
    // most of 22.7 us (now 13.7).
    auto add_slices = [&](int self) {
      constexpr int EAGER = ANY && MT == 1 ? 8 : 4;
      float4 sum[MT][PER] = {};
      for (int s0 = 0; s0 < (ANY ? p.split : 1); s0 += EAGER) {
        float4 u[EAGER][MT][PER];
#pragma unroll
        for (int d = 0; d < EAGER; d++)
          if (s0 + d < p.split && s0 + d != self) {
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
              for (int e = 0; e < PER; e++) u[d][m][e] = load_through(slots + ((s0 + d) * MT + m) * 1024 + tid + e * NW * 64);
          }
#pragma unroll
        for (int d = 0; d < EAGER; d++)
          if (s0 + d < p.split) {
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
              for (int e = 0; e < PER; e++) {
                const float4 v = s0 + d == self ? tot[m][e] : u[d][m][e];
                float4 &t = sum[m][e];
                if (s0 + d == 0) t = v;
                else { t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w; }
              }
          }
      }
#pragma unroll
      for (int m = 0; m < MT; m++)
#pragma unroll
        for (int e = 0; e < PER; e++) tot[m][e] = sum[m][e];
    };
    bool others_done = false;
    if (slice == 0) {
      // Slice 0 is given slightly more of K than the others, so it usually ends last: if every other slice has arrived
      // already, nobody needs this slice's tile in memory, and the write, its acknowledgement and the counter update
      // drop out of the kernel's tail.  (If not, slice 0 goes the way of the others below.)
      if (tid == 0) is_last = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.split - 1;
      __syncthreads();
      others_done = is_last;
      __syncthreads();  // is_last is written again below
    }
    if (others_done) {
      if (tid == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      add_slices(0);
    } else {
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int e = 0; e < PER; e++) store_through(slots + (slice * MT + m) * 1024 + tid + e * NW * 64, tot[m][e]);
    __builtin_amdgcn_s_waitcnt(0);  // the stores have been acknowledged: the tile is in memory
    __syncthreads();                // ... every wavefront's part of it
    if (tid == 0) {
      int before = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      is_last = before == p.split - 1;
      if (before == p.split - 1) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!is_last) return;
    add_slices(slice);
    }
  }
  // to row-major through LDS, then 16-byte stores of eight fp16 values
  constexpr int PITCH = W8_COLS_WIDE + 4;
  float *tile = reinterpret_cast<float *>(w8_lds);
  uint16_t *__restrict__ C = (uint16_t *)p.c;
  const bool c_vec = (p.ldc % 8 == 0) && (((uintptr_t)C & 15) == 0);
#pragma unroll
  for (int grp = 0; grp < MT; grp++) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < PER; e++) {
      const int idx = tid + e * NW * 64;
      const int c = idx >> 6, jj = idx & 15, gg = (idx >> 4) & 3;
      float *dst = tile + (4 * gg) * PITCH + 16 * jj + c;
      dst[0] = tot[grp][e].x; dst[PITCH] = tot[grp][e].y; dst[2 * PITCH] = tot[grp][e].z; dst[3 * PITCH] = tot[grp][e].w;
    }
    __syncthreads();
    for (int item = tid; item < 16 * (W8_COLS_WIDE / 8); item += NW * 64) {
      const int m = item / (W8_COLS_WIDE / 8), n8 = (item % (W8_COLS_WIDE / 8)) * 8;
      if (16 * grp + m >= p.M || (ANY && n0 + n8 >= p.N)) continue;
      const float *src = tile + m * PITCH + n8;
      uint16_t h[8];
#pragma unroll
      for (int i = 0; i < 8; i++) h[i] = f32_to_f16(src[i]);
      uint16_t *dst = C + (int64_t)(16 * grp + m) * p.ldc + n0 + n8;
      if (c_vec) {
        *reinterpret_cast<uint4 *>(dst) = make_uint4(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16,
                                                     h[4] | (uint32_t)h[5] << 16, h[6] | (uint32_t)h[7] << 16);
      } else {
#pragma unroll
        for (int i = 0; i < 8; i++) dst[i] = h[i];
      }
    }
  }
}

__global__ __launch_bounds__(256) void gemm_w8a16_reduce_kernel(GemmW8A16Params p) {
  int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= p.M * p.N) return;
  int64_t m = idx / p.N, n = idx % p.N;
  float s = 0.f;
  for (int k = 0; k < p.split; k++) s += p.workspace[((int64_t)k * 16 + m) * p.N + n];
  ((uint16_t *)p.c)[m * p.ldc + n] = f32_to_f16(s);
}

constexpr int W8_WAVES = 16;

}  // namespace

namespace {
// Which direct-to-LDS tile a product runs on (null: none applies), and in how many K slices.
// round, turned, fill, fixed: us per K tile and round of workgroups, what a column-major B adds to it, us per K tile and workgroup
// per CU, and per launch; fitted at `time` below.
struct DmaCand { const char *tag; int64_t bm, bn; double eff, round, turned, fill, fixed; };
const DmaCand DMA_CANDS[4] = {{"256x256", 256, 256, 1.0, 0.59, 0.07, 0.04, 9}, {"128x256", 128, 256, 0.77, 0.48, 0.07, 0.05, 6},
                              {"256x128", 256, 128, 0.73, 0.51, 0.03, 0.04, 6.3}, {"128x128", 128, 128, 0.59, 0.34, 0, 0.03, 3.8}};
struct DmaChoice { const DmaCand *tile = nullptr; int split = 1; bool meet = false; };  // meet: the slices meet in the kernel

// us that K slices take to become one through a second kernel that the whole chip runs.
double added_us(const GemmParams &p, int split) { return 5.5 + 0.28e-6 * split * 4 * (double)p.M * (double)p.N * std::max(1, p.batches); }
// On 128 x 128 tiles the workgroup of a tile that arrives last can add the slices instead (slices_meet), reading 64 KiB of each alone.
// Two or three slices gain by it; more lose, every slice costing that workgroup a trip to memory, and so do tiles that stick out of C,
// which are handed over and stored as a whole where the second kernel reads only what belongs to C.  us of a product whose operands
// are in cache, by its second kernel in the slices that `time` says and by their meeting in two or three, both fitted (5 % rms) to 207
// sizes of 6 ... 140 tiles, K 1056 ... 8192; the host takes some 13 us for two launches from Python and 10.5 for one, whatever the GPU does.
// us, apart / together: 768 x 768 x 1536 16.4 / 14.1, 1024 x 1024 x 1792 17.7 / 14.6, 941 x 768 x 1376 15.9 / 13.1, 512 x 512 x 1536 13.8 / 12.1,
// 1024 x 2048 x 3072 24.7 / 23.3; where the rule keeps the second kernel 200 x 1600 x 1600 13.5 / 14.5, 808 x 1144 x 2816 19.2 / 21.3, 1024 x 1024
// x 4096 19.7 / 20.6, 183 x 3384 x 3968 21.6 / 23.0, 245 x 568 x 1664 13.0 / 13.8, 256 x 256 x 4096 in eight slices 12.8 / 17.4.
constexpr double APART_HOST_US = 13.0, TOGETHER_HOST_US = 10.5;
double apart_us(const GemmParams &p, int64_t tiles, int64_t nk, int split, int cus) {
  const double mb = 4e-6 * (double)p.M * (double)p.N, f = std::min(1.0, (double)tiles * split / cus);
  return std::max(APART_HOST_US, 5.6 + 0.38 * split + (0.4 + 0.33 * split) * mb + (0.237 - 0.026 * f) * (double)((nk + split - 1) / split) + (p.M % 128 ? 0.8 : 0) - (p.N % 128 ? 0.2 : 0));
}
double together_us(const GemmParams &p, int64_t tiles, int64_t nk, int split, int cus) {
  const double t = (double)tiles / 64, f = (double)tiles * split / cus;
  return std::max(TOGETHER_HOST_US, 4.8 + 1.03 * split + (0.81 * split - 0.09) * t + (0.2355 + 0.016 * f) * (double)((nk + split - 1) / split) + (p.M % 128 ? 0.5 : 0) + (p.N % 128 ? 0.9 : 0));
}

DmaChoice choose_dma(const GemmParams &p, int max_split) {
  static const char *dma_env = getenv("TTS_GEMM_DMA");      // tuning aid: "256x256", "128x256", "256x128", "128x128" or unset
  static const char *split_env = getenv("TTS_GEMM_SPLIT");  // tuning aid: the number of K slices (1 = never split)
  const int cus = device_cus();
  // (tiles of all the batch's products: they share the launch)
  auto tiles = [&](const DmaCand &c) { return ((p.M + c.bm - 1) / c.bm) * ((p.N + c.bn - 1) / c.bn) * std::max(1, p.batches); };
  // Rows with a weight matrix per block stream their weights from HBM, and the 128 x 256 tile's prefetching wavefront is ahead
  // from half a workgroup per CU on (us with 128 x 128 / 128 x 256 tiles: 144 of the latter 65 / 58, 160 42.4 / 40.1, 192 57.8 /
  // 50.8; below, 72 29.0 / 43.9, 28 16.4 / 19.6), but not where they make a second round that is mostly empty (288 73.3 / 79.1, 320
  // 77.4 / 80.3, 336 74.0 / 78.2, 396 87.4 / 92.0; 504 31.5 / 30.4, 510 47.8 / 45.1; beyond two rounds they are even: 576 110 / 110,
  // 800 210 / 210).  A few tiles over one round count as one: blocks of rows that pad the last matrix have nothing to do.
  const bool grouped = p.b_block != nullptr && !p.b_trans;
  auto grouped_wide = [&](int64_t t) { return 2 * t >= cus && !(10 * t > 11 * cus && 10 * t < 16 * cus); };
  // The other products: the least modelled time.  What decides is the number of rounds of workgroups over the chip, begun ones
  // included: a K tile of a round takes about the same however many of the CUs work (128 x 128 tiles, two of which share a CU,
  // up to 1 / 2 / 3 / 4 per CU: 0.38 / 0.69 / 1.0 / 1.4 us).  Few tiles (a skinny product, M = 16 ... 1024 against N, K in the thousands)
  // leave CUs idle while every workgroup walks all of K alone: K is then cut into slices, whose fp32 sums a second kernel adds, and
  // whose workgroups count in rounds like any others.
  // Fitted to 1820 products from HBM (M 16 ... 4200, N to 14336, K 512 ... 14336, powers of two and their like, model widths and sizes
  // nothing divides, either operand column-major) on every tile in 1 to 16 slices, for the choice rather than the times: it is
  // 1.9 % behind the best of each; the tile by the rule below and slices as if they filled the chip evenly are 9 % behind.
  // us: 3000 x 4096 x 2048 on 256 x 256 / 128 x 256 / 128 x 128 tiles 50.5 / 67.6 / 65.9; 3000 x 2048 x 4096 80.8 / 61.1 / 68.2; 2048 x 1536 x
  // 5120 on 128 x 128 tiles 64, in five slices of 256 x 256 50; 512 x 14336 x 4096 on 128 x 256 81, in two slices of 256 x 256 71; in 1 / 2 /
  // 3 / 4 slices 1504 x 3072 x 4096 on 256 x 256 84 / 64 / 56 / 79 (the fourth begins a second round).
  // Below K = 512 the fixed costs decide and the tiles measure alike: among the tiles that give every CU a workgroup (128 x 128:
  // always) the one with the least padded work per unit of the tile's measured efficiency at 4096^3 (105 / 136 / 144 / 179 us).
  const bool by_rounds = !grouped && p.K >= 512;
  const int64_t nk = p.K / F_BK;
  const double sums = (double)p.M * (double)p.N * std::max(1, p.batches) * 4;  // bytes of one slice's
  auto time = [&](const DmaCand &c, int split) {
    const double f = (double)tiles(c) * split / cus;
    return (double)((nk + split - 1) / split) * (std::ceil(f) * (c.round + (p.b_trans ? c.turned : 0)) + f * c.fill) + c.fixed +
           (split == 1 ? 0 : added_us(p, split));
  };
  DmaChoice best;
  double best_cost = 0;
  for (const DmaCand &c : DMA_CANDS) {
    if (!gemm_dma_ok(p, c.bm, c.bn)) continue;
    if (dma_env ? std::string(dma_env) != c.tag : !by_rounds && c.bm + c.bn != 256 && (grouped ? !grouped_wide(tiles(c)) : tiles(c) < cus)) continue;
    const double cost = by_rounds ? time(c, 1) : (double)(tiles(c) * c.bm * c.bn) / c.eff;
    if (!best.tile || cost < best_cost) { best.tile = &c; best_cost = cost; }
  }
  if (!best.tile || max_split < 2 || !by_rounds || p.a_rows || p.b_block) return best;
  // (the model's times of short walks are too long: in 128 x 128 tiles K to 1024 is ahead whole, us whole / in slices that a second
  // kernel adds / that meet: 256 x 1024 x 1024 11.0 / 13.6 / 11.9, 64 x 4096 x 1024 11.4 / 13.5 / 11.8; 512 x 1024 x 1216 11.9 / 14.3 / 11.8)
  if (best.tile == &DMA_CANDS[3] && p.K <= 1024 && !split_env && p.batches <= 1) return best;
  DmaChoice pick = best;
  double pick_t = best_cost;
  if (!(split_env && atoi(split_env) == 1))
    for (const DmaCand &c : DMA_CANDS) {
      if (!gemm_dma_ok(p, c.bm, c.bn) || (dma_env && std::string(dma_env) != c.tag)) continue;
      const int64_t most = std::min<int64_t>(std::min<int64_t>(std::min<int64_t>(16, max_split), nk / 8), (2 * cus + tiles(c) - 1) / tiles(c));
      for (int64_t sp = split_env ? atoi(split_env) : 2; sp <= most; sp++) {
        if (sp * sums > (double)((size_t)256 << 20)) break;
        const double t = time(c, (int)sp);
        if (t < pick_t || (split_env && pick.split == 1)) { pick.tile = &c; pick.split = (int)sp; pick_t = t; }
        if (split_env) break;
      }
    }
  // Slices that would meet in the kernel instead.  (What is ahead whole of slices that a second kernel adds stays whole: 1152 x 1536 x
  // 1024 11.5 us against 14.9 in two slices.)  From larger tiles, for which `time` knows what 128 x 128 in few slices would take with
  // their meeting in place of the second kernel: 1024 x 1536 x 4096 24.1 us against five slices of 128 x 256 at 26.9; only where the tiles are
  // filled (1715 x 408 x 7008 28.0 / 26.1).
  if (p.meet && pick.split > 1 && p.batches <= 1 && !split_env) {
    const DmaCand &c = DMA_CANDS[3];
    const int64_t t = tiles(c);
    const bool same = pick.tile == &c, filled = (double)p.M * (double)p.N >= 0.85 * 128 * 128 * (double)t;
    const double apart = same ? apart_us(p, t, nk, pick.split, cus) : 0;
    // us to be gained at least: of 207 sizes 66 gain 1.085 in the geometric mean, three lose 1.8 % at most (at 1.0 five, 3.6 %)
    double most = !same ? 0 : apart > APART_HOST_US ? 1.2 : 0.6;
    for (int sp = 2; sp <= 3; sp++) {
      if (!gemm_dma_ok(p, c.bm, c.bn) || (dma_env && std::string(dma_env) != c.tag) || sp > max_split || nk / 8 < sp || t * sp > cus || !(same || filled)) continue;
      const double gain = same ? apart - together_us(p, t, nk, sp, cus)
                               : pick_t - (time(c, sp) - added_us(p, sp) + 2.4 * sp - 4);
      if (gain > most) { pick = {&c, sp, true}; most = gain; }
    }
  }
  return pick;
}
}  // namespace

namespace {
// K slices of the any-shape kernel (1: none), at most max_split: where its tiles leave CUs without work, every workgroup
// would walk all of K alone.  Modelled like choose_dma's: the K tiles of 64 a workgroup walks -- 0.58 us each on 64 x 128 tiles
// with a CU to itself, 1.4 of that per workgroup beyond one, 1.19 us and 1.1 on 128 x 128 -- the slices' sums through memory and
// the second launch.  Measured in us per call with 1 / 2 / 4 / 8 / 16 slices: 33 x 4001 x 4001 40 / 25 / 17.7 / 15.0 / 17.3;
// 600 x 601 x 3001 33.8 / 24.3 / 18.9 / 20.8 / 30.8; 504 x 2000 x 3000 28.9 / 24.8 / 27 / 35 / 50; 100 x 700 x 2000 20.3 / 15.1 / 13.6 /
// 14.3 / 13.7; 1501^3 27 / 36; 500 x 600 x 700 11.9 / 14.4; 64 x 1003 x 517 11.9 / 14.0: the model takes 1 where two lose.
int any_split(const GemmParams &p, int max_split) {
  if (p.a_rows || p.b_block) return 1;
  const int64_t nk = (p.K + 63) / 64;
  const double sums = (double)p.M * (double)p.N * std::max(1, p.batches) * 4;
  auto model = [&](int split) {
    const int64_t rows = any_rows(p, split);
    const double w = (double)(((p.M + rows - 1) / rows) * ((p.N + 127) / 128) * std::max(1, p.batches) * split) / device_cus();
    double t = (w <= 1 ? 1.0 : (rows == 64 ? 1.4 : 1.1) * w) * (double)((nk + split - 1) / split) * (rows == 64 ? 0.58e-6 : 1.19e-6) + 5e-6;
    if (split > 1) t += 2 * split * sums / 6e12 + 4.5e-6;
    return t;
  };
  static const char *split_env = getenv("TTS_GEMM_SPLIT");  // tuning aid (see choose_dma)
  if (split_env) return std::max(1, std::min(atoi(split_env), std::min(16, max_split)));
  int pick = 1;
  double pick_t = 0.9 * model(1);
  for (int sp = 2; sp <= std::min<int64_t>(std::min(16, max_split), nk / 3); sp++) {
    if ((double)sp * sums > (double)((size_t)256 << 20)) break;
    const double t = model(sp);
    if (t < pick_t) { pick = sp; pick_t = t; }
  }
  return pick;
}
}  // namespace

GemmChoice gemm_choose(const GemmParams &p) {
  static const char *tile_env = getenv("TTS_GEMM_TILE");  // tuning aid: set = the any-shape kernel even for whole tiles
  GemmChoice c;
  if (p.is_f32 || tile_env) return c;
  const DmaChoice dma = choose_dma(p, 16);
  if (dma.tile) c.tile = (int)(dma.tile - DMA_CANDS);
  GemmParams q = p;
  q.split = c.split = dma.tile ? dma.split : any_split(p, 16);
  c.bytes = gemm_workspace_bytes(q);
  if (dma.meet) {
    c.meeting = (size_t)(((p.M + 127) / 128) * ((p.N + 127) / 128));
    c.bytes = (size_t)c.split * c.meeting * (128 * 128 * sizeof(float));
  }
  return c;
}
size_t gemm_workspace_bytes(const GemmParams &p) { return p.split > 1 ? (size_t)p.split * p.M * p.N * std::max(1, p.batches) * sizeof(float) : 0; }

// p.split: the most K slices p.partial has room for (what gemm_choose(p) said, or fewer; 1: none).
hipError_t launch_gemm(const GemmParams &p, hipStream_t s, const char **name, const GemmChoice *chosen) {
  if (p.is_f32) {
    if (p.a_rows || p.b_block) return hipErrorInvalidValue;  // (the matcher takes gathered rows on 16-bit operands only)
    *name = "gemm_f32_kernel";
    return launch_gemm_f32(p, s);
  }
  static const char *tile_env = getenv("TTS_GEMM_TILE");  // (as in gemm_choose)
  const bool kept = chosen && chosen->split == std::max(1, p.split);
  if (!tile_env) {
    // Whole K tiles go to the direct-to-LDS kernels.
    // at most p.split slices: what was chosen, or fewer when the caller's workspace holds no more (1: none)
    const DmaChoice choice = !kept ? choose_dma(p, std::max(1, p.split)) : chosen->tile < 0 ? DmaChoice{} : DmaChoice{&DMA_CANDS[chosen->tile], chosen->split};
    GemmParams q = p;
    q.split = choice.split;
    const DmaCand *best = choice.tile;
#define TTS_DMA(TM, TN, TAG)                                                                                  \
  do {                                                                                                        \
    *name = TAG;                                                                                              \
    return q.is_bf16 ? launch_gemm_dma<true, TM, TN>(q, s) : launch_gemm_dma<false, TM, TN>(q, s);            \
  } while (0)
    if (best && best->bm == 256 && best->bn == 256) TTS_DMA(4, 4, q.split > 1 ? "gemm_dma_kernel, K slices" : "gemm_dma_kernel");
    if (best && best->bm == 128 && best->bn == 256) TTS_DMA(2, 4, q.split > 1 ? "gemm_dma_kernel<128x256>, K slices" : "gemm_dma_kernel<128x256>");
    if (best && best->bm == 256 && best->bn == 128) TTS_DMA(4, 2, q.split > 1 ? "gemm_dma_kernel<256x128>, K slices" : "gemm_dma_kernel<256x128>");
    if (best) TTS_DMA(2, 2, q.split > 1 ? "gemm_dma_kernel<128x128>, K slices" : "gemm_dma_kernel<128x128>");
#undef TTS_DMA
  }
  // anything else: 128 x 128 x 64 tiles, two workgroups per CU, or half as high (a 256 x 256 x 32 form of the same kernel measured behind it
  // at every size tried: 4096^3: 202 against 197 us; 4096 x 2048 x 2048: 112 against 56 us)
  GemmParams q = p;
  q.split = tile_env || !p.partial ? 1 : kept ? chosen->split : any_split(p, std::max(1, p.split));
  *name = any_name(any_rows(q, q.split), false, q.split > 1);
  if (q.split == 1) return p.is_bf16 ? launch_gemm_any<true, false>(q, s) : launch_gemm_any<false, false>(q, s);
  hipError_t e = launch_gemm_any_slices(q, s);
  if (e != hipSuccess) return e;
  const ReduceGrid g(q);
  if (q.is_bf16) hipLaunchKernelGGL(gemm_splitk_reduce_any_kernel<true>, dim3(g.workgroups, std::max(1, q.batches)), dim3(256), 0, s, q, g.across, g.col_blocks);
  else hipLaunchKernelGGL(gemm_splitk_reduce_any_kernel<false>, dim3(g.workgroups, std::max(1, q.batches)), dim3(256), 0, s, q, g.across, g.col_blocks);
  return hipGetLastError();
}

namespace {
// The kernels compiled with a functor: 0 whole 256 x 256 x 32 tiles on the 16 x 16 x 32 instruction; 1 any shape in 128 x 128 x 64
// tiles; 2 the sum of K slices; 3 any shape in 64 x 128 x 64 tiles; 4 ... the other direct-to-LDS tiles, in the order of DMA_CANDS;
// 7 ... fp32 operands, in the order of F32_TILINGS (16 x 352 x 136, leaky_relu: 16.9 us on the generic kernel, 9.5 here).
int epilogue_dma_index(const DmaCand *tile) { return tile == &DMA_CANDS[0] ? 0 : 3 + (int)(tile - DMA_CANDS); }

template <int TM, int TN>
hipError_t launch_dma_slices(const GemmParams &p, hipStream_t s) {
  return p.is_bf16 ? launch_gemm_dma_slices<true, TM, TN, false, false>(p, s) : launch_gemm_dma_slices<false, TM, TN, false, false>(p, s);
}

// What a product with a functor runs on, in at most max_split K slices.  Row-major operands of whole K tiles take the
// direct-to-LDS tile and the slices that the plain product takes (choose_dma).  With leaky_relu in bf16, us, against 256 x 256
// tiles at every size: 128 x 4096 x 4096 22.5 / 80.6; 16 x 4096 x 4096 19 / 79; 512^3 12 / 17; 1024^3 13 / 25.5; 2048^3 24 / 44;
// 1000 x 4096 x 4096 53 / 88; 4096 x 2048 x 2048 40 / 48.6.  (A column-major operand goes to the any-shape kernel.)
struct EpilogueChoice { int whole, split; const DmaCand *tile; };  // the kernel without slices; the tile the slices run on (null: any shape)
EpilogueChoice choose_epilogue(const GemmParams &p, int max_split) {
  if (p.is_f32) return {7 + f32_tiling(p), 1, nullptr};
  if (!gemm_fast_path_ok(p)) return {any_rows(p, 1) == 64 ? 3 : 1, any_split(p, max_split), nullptr};
  const DmaChoice choice = choose_dma(p, max_split);
  if (!choice.tile) return {0, 1, &DMA_CANDS[0]};  // (only where a tuning variable names a tile that does not apply)
  return {epilogue_dma_index(choice.split > 1 ? choose_dma(p, 1).tile : choice.tile), choice.split, choice.tile};
}
// A kernel that is compiled already and computes what `whole` does: any direct-to-LDS tile for another of them, the any-shape
// kernel's 128 rows for its 64, any fp32 tiling (-1: none).
int compiled_epilogue(int whole, RtcModule *const *modules) {
  if (modules[whole]) return whole;
  if (whole >= 7) {
    for (int m = 7; m < GEMM_EPILOGUE_KERNELS; m++)
      if (modules[m]) return m;
    return -1;
  }
  if (whole == 1 || whole == 3) return modules[4 - whole] ? 4 - whole : -1;
  for (int m : {0, 4, 5, 6})
    if (modules[m]) return m;
  return -1;
}
}  // namespace

bool gemm_epilogue_compiled(const GemmParams &p, RtcModule *const *modules) { return compiled_epilogue(choose_epilogue(p, 1).whole, modules) >= 0; }
int gemm_epilogue_split(const GemmParams &p) { return choose_epilogue(p, 16).split; }

// Kernels are compiled from gemm_device.h plus the epilogue functor at the first launch that needs them.  A launch in slices
// (p.split > 1) also compiles the kernel it would be without, so that a later one of the same plan that may not use a workspace
// finds it; one that may not compile takes the kernel that is there.
hipError_t launch_gemm_epilogue(const GemmParams &p, const std::string &epilogue, RtcModule **modules, bool may_compile, const GemmEpilogueArgs &ep,
                                hipStream_t s, const char **name, std::string *err) {
  const EpilogueChoice choice = choose_epilogue(p, std::max(1, p.split));
  const bool sliced = choice.split > 1;
  const int whole = may_compile ? choice.whole : compiled_epilogue(choice.whole, modules), which = sliced ? 2 : whole;
  if (which < 0) return hipErrorInvalidValue;  // (gemm_epilogue_compiled said so)
  const bool any_shape = sliced ? !choice.tile : which == 1 || which == 3;
  *name = p.is_f32 ? "gemm_f32_kernel + epilogue (hipRTC)" : any_shape ? any_name(sliced ? any_rows(p, choice.split) : which == 3 ? 64 : 128, true, sliced)
                    : (sliced ? "gemm_dma_kernel + epilogue (hipRTC), K slices" : "gemm_dma_kernel + epilogue (hipRTC)");
  for (int m : {whole, which}) {
    if (modules[m]) continue;
    const std::string source = epilogue + "#define TTS_GEMM_RTC " + std::to_string(m) + "\n#define TTS_GEMM_BF16 " + std::to_string(p.is_bf16 ? 1 : 0) +
                               "\n" + gemm_device_source();
    hipError_t e = rtc_compile(source, "gemm_rtc", &modules[m], err);
    if (e != hipSuccess) {
      if (getenv("TTS_DUMP_RTC_SOURCE")) *err += "\n--- source ---\n" + source;
      return e;
    }
  }
  struct {
    GemmParams p;
    int tiles_m, tiles_n;  // (kernel 2: columns a workgroup spans, blocks of them)
    GemmEpilogueArgs ep;   // the functor: same layout as the generated struct TtsEp
  } a;
  a.p = p;
  a.p.split = choice.split;
  a.ep = ep;
  if (sliced) {
    const int t = choice.tile ? epilogue_dma_index(choice.tile) : 1;
    hipError_t e = t == 0 ? launch_dma_slices<4, 4>(a.p, s) : t == 4 ? launch_dma_slices<2, 4>(a.p, s) : t == 5 ? launch_dma_slices<4, 2>(a.p, s)
                 : t == 6 ? launch_dma_slices<2, 2>(a.p, s) : launch_gemm_any_slices(a.p, s);
    if (e != hipSuccess) return e;
    const ReduceGrid g(p);
    a.tiles_m = g.across;
    a.tiles_n = g.col_blocks;
    return rtc_launch(modules[2], g.workgroups, 1, 1, 256, &a, sizeof a, s);
  }
  if (p.is_f32) {
    const F32Tiling &t = F32_TILINGS[which - 7];
    a.tiles_m = (int)((p.M + t.edge - 1) / t.edge);
    a.tiles_n = (int)((p.N + t.edge - 1) / t.edge);
    return rtc_launch(modules[which], a.tiles_m * a.tiles_n, 1, 1, t.threads, &a, sizeof a, s);
  }
  const int64_t rows = which == 3 ? 64 : which == 0 || which == 5 ? 256 : 128, cols = which == 0 || which == 4 ? 256 : 128;
  a.tiles_m = (int)((p.M + rows - 1) / rows);
  a.tiles_n = (int)((p.N + cols - 1) / cols);
  return rtc_launch(modules[which], a.tiles_m * a.tiles_n, 1, 1, 256, &a, sizeof a, s);
}

namespace {
struct W8Config { int cw, nw, split; };

// Whether the 16-byte-load kernel takes a shape: N in whole slabs of 256, and from 1024 columns on in groups of 16 (below, a last slab that
// is half empty is a good part of all).  Whole slabs of 128 stay on the 8-byte kernel in two ranges where it is ahead, in 1 and in 16 rows, us 8-byte /
// 16-byte loads with the weights from memory (from cache as far apart), of 378 and 126 sizes measured:
//   * the 128-column slabs are a workgroup per CU at most and need no slices, K from 768 to below 3072: 28800 columns, K 512 10.3 / 10.2,
//     768 10.3 / 11.4, 1024 10.6 / 12.9, 2048 15.0 / 16.7, 2560 17.1 / 18.6, 3072 19.8 / 20.5 (16 rows 20.9 / 20.5), 4096 24.4 / 23.8.  In more
//     slabs than CUs it is behind: 32896 x 2048 25.1 / 17.7;
//   * K beyond 4096 where a step of 32 rows for each wavefront that the chip's CUs hold, 16, is all there is: 1152 columns x 12288
//     14.7 / 16.8, 2432 x 5888 12.4 / 14.0, 1920 x 8192 13.2 / 14.7, but two steps for some 1408 x 12288 20.9 / 17.2, 3200 x 5888 18.3 / 14.2, 2432 x 8192
//     18.6 / 14.9; K = 4096 behind by 2 to 6 % throughout.
// Other widths would take its form for any shape: 40016 x 2048 46.6 / 22.6, 2544 x 8192 25.8 / 16.2, 1040 x 8192 16.0 / 15.3.
bool w8_wide_shape(const GemmW8A16Params &p) {
  if (p.K % 32 != 0 || p.lda % 8 != 0 || p.ldw % 16 != 0) return false;
  if (p.N % W8_COLS_WIDE == 0) return true;
  if (p.N % 16 != 0 || p.N < 1024) return false;
  if (p.N % W8_COLS != 0) return true;
  const int64_t slabs = p.N / W8_COLS, steps = p.K / 32;
  if (slabs >= 192) return slabs > 256 || p.K < 768 || p.K >= 3072;  // (from 192 slabs on it takes no slices: w8_config)
  return p.K <= 4096 || slabs * steps > 16 * 256;
}

// The shape decides the kernel: 256-column slabs with 16-byte weight loads when N and the
// weight pitch allow, split over K so that about one workgroup lands on each CU.
// TTS_W8=cw,nw,split overrides the choice (tuning aid).
W8Config w8_config(const GemmW8A16Params &p) {
  const int64_t steps = (p.K + 31) / 32;
  W8Config c{8, 16, 1};
  if (w8_wide_shape(p)) c = W8Config{16, 8, 1};
  static const char *env = getenv("TTS_W8");
  int want_split = 0;
  if (env) {
    int cw = 0, nw = 0;
    if (sscanf(env, "%d,%d,%d", &cw, &nw, &want_split) >= 2 && (cw == 8 || (cw == 16 && c.cw == 16))) {
      c.cw = cw; c.nw = nw;
    }
  }
  const int64_t slabs = (p.N + 16 * c.cw - 1) / (16 * c.cw);
  if (want_split > 0) c.split = want_split;
  else if (c.cw == 16) {
    // At most one workgroup per CU (its LDS tile admits no more), and the least modelled time: a workgroup's round of eight steps takes
    // 1.35 us where the chip is idle and 12 ns per workgroup where memory is the limit, a meeting 0.35 us per slice beyond five.
    // Measured, us in 2 / 4 / 8 / 12 / 24 slices: 15 x 2048 x 6400 25.0 / 16.8 / 13.7 / 13.4 / 16.4; 9 x 6272 x 5376 22.3 / 16.1 / 14.5 / 19.9 / 26.9;
    // 3 x 9856 x 2432 13.9 / 12.1 / 16.5 / 18.5 / 27.9; 8 x 20096 x 7296 in 2 / 3 / 4 30.4 / 27.6 / 36.9.  (As many as fill the chip, as before: 16.8, 15.7, 12.3.)
    double best = 0;
    for (int64_t n = 1; n <= std::min<int64_t>(64, std::max<int64_t>(1, steps / c.nw)) && (n == 1 || slabs * n <= 256); n++) {
      const double rounds = std::max(1.0, (double)steps / (double)(c.nw * n)), memory = 0.0117 * (double)(slabs * n);
      const double t = rounds * std::sqrt(1.35 * 1.35 + memory * memory) + 0.35 * (double)std::max<int64_t>(0, n - 5);
      if (n == 1 || t < best) { c.split = (int)n; best = t; }
    }
  } else if (slabs < 192) {  // about one workgroup per CU, every wavefront busy
    const int64_t most = std::max<int64_t>(1, steps / c.nw);
    c.split = (int)std::max<int64_t>(1, std::min<int64_t>(std::min((256 + slabs - 1) / slabs, most), 64));
  }
  return c;
}

template <int NW, int DEPTH, bool FAST>
void w8_launch(const GemmW8A16Params &p, int steps_per_slice, hipStream_t s) {
  dim3 grid((unsigned)((p.N + W8_COLS - 1) / W8_COLS), p.split);
  hipLaunchKernelGGL((gemm_w8a16_kernel<NW, DEPTH, FAST, 8>), grid, dim3(NW * 64), 0, s, p, steps_per_slice);
}

template <int NW, int MT, bool ANY>
hipError_t w8_launch_wide(const GemmW8A16Params &p, int first_steps, int other_steps, hipStream_t s) {
  constexpr size_t lds = (size_t)NW * 16 * 64 * sizeof(float4);
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_w8a16_wide_kernel<NW, MT, ANY>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return attr;
  dim3 grid((unsigned)((p.N + W8_COLS_WIDE - 1) / W8_COLS_WIDE), p.split);
  hipLaunchKernelGGL((gemm_w8a16_wide_kernel<NW, MT, ANY>), grid, dim3(NW * 64), lds, s, p, first_steps, other_steps);
  return hipGetLastError();
}
}  // namespace

int gemm_w8a16_split(const GemmW8A16Params &p) { return w8_config(p).split; }

size_t gemm_w8a16_workspace_bytes(const GemmW8A16Params &p) {
  if (p.split <= 1) return 0;
  // per-slice partial tiles: 16 rows of fp32, 32 when a launch takes two groups of rows
  return (size_t)p.split * (p.M > 16 ? 32 : 16) * (size_t)((p.N + 255) / 256 * 256) * sizeof(float);
}

size_t gemm_w8a16_counters(const GemmW8A16Params &p) { return p.split <= 1 ? 0 : w8_counter_pitch(p.split) * (size_t)((p.N + 255) / 256); }

static hipError_t launch_gemm_w8a16_rows(const GemmW8A16Params &p, hipStream_t s, const char **name);

static bool w8_wide(const GemmW8A16Params &p);

// Many rows of A (a prefill-sized M): the decode kernels would read W once per 32 rows.  The weights are widened once,
// as the source does it -- w.to(f16) * scale[None, :], one fp16 rounding -- into a [K, N] fp16 matrix, and the tiled
// matmul kernels multiply (fp16 operands, fp32 accumulation: the same arithmetic as the decode kernels').  From 193
// rows up, where the passes of the decode kernel cost what widening (W read, twice its bytes written) and one tiled
// product do.  Eight columns per thread: 8-byte weight loads, 16-byte scale loads and stores.
// For shapes the tiled kernel of kernels_w8_tile.hip does not take.  Measured at [8192, 28672]: 304 us at M = 129, 351 at
// 256, 452 at 512, 952 at 2048, against 50 us per 32 rows on the decode kernels: from seven launches of those on, the widened
// product is ahead.
constexpr int64_t W8_WIDEN_FROM_ROWS = 193;
__global__ __launch_bounds__(256) void gemm_w8a16_widen_kernel(GemmW8A16Params p) {
  const int64_t octs = p.N / 8, idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= p.K * octs) return;
  const int64_t k = idx / octs, n = (idx % octs) * 8;
  const uint2 q = *reinterpret_cast<const uint2 *>(p.w + k * p.ldw + n);
  const uint4 sv = *reinterpret_cast<const uint4 *>((const uint16_t *)p.scale + n);
  const uint32_t qs[2] = {q.x, q.y}, ss[4] = {sv.x, sv.y, sv.z, sv.w};
  uint32_t out[4];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    // bytes 2c and 2c + 1 of the eight: [b0, 0, b1, 0], then 0x6400 | (b ^ 0x80) = 1152 + b as fp16 (exact), as in the decode kernels
    const uint32_t word = qs[c / 2] >> (16 * (c & 1));
    const uint32_t pair = ((word & 0xffu) | ((word & 0xff00u) << 8)) ^ 0x64806480u;
    out[c] = pk_sub_1152_mul(pair, ss[c]);
  }
  *reinterpret_cast<uint4 *>((uint16_t *)p.widened + k * p.N + n) = make_uint4(out[0], out[1], out[2], out[3]);
}
static bool w8_widens(const GemmW8A16Params &p) {
  return p.M >= W8_WIDEN_FROM_ROWS && p.N % 8 == 0 && p.ldw % 8 == 0 && ((uintptr_t)p.w & 7) == 0 && ((uintptr_t)p.scale & 15) == 0;
}

// More rows of A than a launch takes (32 on the 16-byte-load kernel, 16 on the other): the decode kernels once per
// group of rows, one launch after the other on the stream (they share the split-K workspace, which every launch leaves
// ready for the next).  W is read once per launch.
// The tiled kernel (kernels_w8_tile.hip) from 33 rows up, where the decode kernels read W once per 32 rows; from 17 rows when
// W holds 8 MB or more (32 x 4096 x 4096: 20 us against 33; 20 x 2048 x 2048, which the launches bound: 20 against 19).  Products
// of fewer than eight of its column tiles stay on the kernels below: the choice of kernel for them is part of what the
// tests hold fixed (the tiled kernel is faster there too: 100 x 1024 x 2048 in 20 us against 64).
static bool w8_tiles(const GemmW8A16Params &p) {
  return (p.M >= 33 || (p.M >= 17 && p.K * p.N >= (int64_t)8 << 20)) && p.N >= 2048 && w8_tile_ok(p);
}
bool gemm_w8a16_is_tiled(const GemmW8A16Params &p) { return w8_tiles(p); }
size_t gemm_w8a16_tile_bytes(const GemmW8A16Params &p) { return w8_tiles(p) ? w8_tile_partial_bytes(p) : 0; }
hipError_t launch_splitk_reduce(const GemmParams &p, hipStream_t s) {
  hipLaunchKernelGGL(gemm_splitk_reduce_kernel<false>, dim3((unsigned)((p.M * (p.N / 4) + 255) / 256), std::max(1, p.batches)), dim3(256), 0, s, p);
  return hipGetLastError();
}
size_t gemm_w8a16_widened_bytes(const GemmW8A16Params &p) { return w8_widens(p) && !w8_tiles(p) ? (size_t)p.K * p.N * 2 : 0; }

hipError_t launch_gemm_w8a16(const GemmW8A16Params &p, hipStream_t s, const char **name) {
  if (w8_tiles(p)) {
    *name = "gemm_w8a16_tile_kernel";
    return launch_w8_tile(p, s);
  }
  if (p.widened && w8_widens(p)) {
    hipLaunchKernelGGL(gemm_w8a16_widen_kernel, dim3((unsigned)((p.K * (p.N / 8) + 255) / 256)), dim3(256), 0, s, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    GemmParams g{};
    g.a = p.a; g.b = p.widened; g.c = p.c;
    g.M = p.M; g.N = p.N; g.K = p.K;
    g.lda = p.lda; g.ldb = p.N; g.ldc = p.ldc;
    g.split = 1;
    const char *inner = nullptr;
    e = launch_gemm(g, s, &inner);
    *name = "gemm_w8a16_widen_kernel + matmul";
    return e;
  }
  const int64_t rows = w8_wide(p) ? 32 : 16;
  if (p.M <= rows) return launch_gemm_w8a16_rows(p, s, name);
  for (int64_t m0 = 0; m0 < p.M; m0 += rows) {
    GemmW8A16Params q = p;
    q.M = std::min<int64_t>(rows, p.M - m0);
    q.a = (const uint16_t *)p.a + m0 * p.lda;
    q.c = (uint16_t *)p.c + m0 * p.ldc;
    hipError_t e = launch_gemm_w8a16_rows(q, s, name);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

static bool w8_fast(const GemmW8A16Params &p) {
  return p.K % 32 == 0 && p.N % W8_COLS == 0 && p.lda % 8 == 0 && p.ldw % 8 == 0 && ((uintptr_t)p.a & 15) == 0 && ((uintptr_t)p.w & 7) == 0;
}
static bool w8_wide(const GemmW8A16Params &p) {
  return w8_wide_shape(p) && w8_config(p).cw == 16 && ((uintptr_t)p.a & 15) == 0 && ((uintptr_t)p.w & 15) == 0;
}

static hipError_t launch_gemm_w8a16_rows(const GemmW8A16Params &p, hipStream_t s, const char **name) {
  const int steps = (int)((p.K + 31) / 32);
  const int sps = (steps + p.split - 1) / p.split;
  const bool fast = w8_fast(p);
  const bool wide = w8_wide(p);
  if (wide) {
    *name = "gemm_w8a16_wide_kernel";
    // slice 0 gets `bias` steps more than an even share (see the kernel's tail), taken evenly from the others
    int first = sps, other = sps;
    if (p.split > 1) {
      static const char *bias_env = getenv("TTS_W8_BIAS");  // tuning aid
      const int bias = bias_env ? atoi(bias_env) : 4;
      const int take = (bias + p.split - 2) / (p.split - 1);  // per other slice
      if (sps - take >= 8 && sps * p.split == steps) { first = sps + take * (p.split - 1); other = sps - take; }
    }
    const bool any = p.split > 4 || p.N % W8_COLS_WIDE != 0;
    if (p.M > 16) return any ? w8_launch_wide<8, 2, true>(p, first, other, s) : w8_launch_wide<8, 2, false>(p, first, other, s);
    return any ? w8_launch_wide<8, 1, true>(p, first, other, s) : w8_launch_wide<8, 1, false>(p, first, other, s);
  }
  *name = "gemm_w8a16_kernel";
  if (!fast) w8_launch<W8_WAVES, 2, false>(p, sps, s);
  else w8_launch<W8_WAVES, 2, true>(p, sps, s);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.split == 1) return e;
  int64_t outs = p.M * p.N;
  hipLaunchKernelGGL(gemm_w8a16_reduce_kernel, dim3((unsigned)((outs + 255) / 256)), dim3(256), 0, s, p);
  return hipGetLastError();
}

}  // namespace tts
