// C ABI (include/tts_hip.h) and the launcher: resolves a plan's symbolic
// bindings for the scalar arguments and grid of one launch, checks what the
// whole-grid kernels assume, and enqueues one kernel for the whole grid.
//
// The reference runs `for x, for y, for z: kernel(args, grid, x, y, z)` on the
// calling thread (backend/driver.py:116-133).  Here the per-program index
// arithmetic the reference executes inside each program (offsets, valid
// extents) is evaluated on the host once per distinct (scalars, grid) and
// cached; the device kernels receive closed forms of it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <list>
#include <map>
#include <memory>
#include <mutex>
#include <set>
#include <sstream>
#include <unordered_map>

#include "../../include/tts_hip.h"
#include "kernels.h"
#include "match.h"

using namespace tts;

namespace {

thread_local std::string g_error;

tts_status fail(tts_status st, const std::string &msg) {
  g_error = msg;
  return st;
}

char *dup_string(const std::string &s) {
  char *p = (char *)malloc(s.size() + 1);
  memcpy(p, s.c_str(), s.size() + 1);
  return p;
}

struct Invalid : std::runtime_error {
  using std::runtime_error::runtime_error;
};

// What tts_launch_noalloc refuses.  Not an Unsupported: a launch that the matrix-product families decline for a reason of
// their own goes on to the generic family's kernel and its binding is cached as such, whereas this refusal says nothing
// about the launch -- the same launch through tts_launch must still find the family's kernel, so nothing is cached.
struct WouldAllocate : std::runtime_error {
  using std::runtime_error::runtime_error;
};

thread_local bool g_no_alloc = false;  // set while tts_launch_noalloc runs on this thread
void may_allocate(const char *what) {
  if (g_no_alloc)
    throw WouldAllocate(std::string("tts_launch_noalloc: this launch needs ") + what + ", which allocates; run it once through tts_launch first");
}

// Whether the stream records a graph: nothing may be allocated then, and a workspace of the stream's would be shared by
// every replay.
bool is_capturing(hipStream_t s) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return false;
}

__global__ void clear_ints_kernel(int *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Everything a launch needs besides the pointers, resolved for one (scalars, grid).
struct Bound {
  Family family;
  Map1DParams map1d{};
  SoftmaxParams softmax{};
  LayerNormParams layernorm{};
  GemmParams gemm{};
  // What the product runs on (gemm_choose) with its operands as aligned as in some launch before, and its slices meeting in the
  // kernel or not: at the index the launcher makes of these; under the plan's mutex.
  GemmChoice gemm_choice[16];
  bool gemm_chosen[16] = {};
  GemmW8A16Params w8{};
  MapNParams mapn{};
  bool empty = false;  // nothing to do (e.g. zero trip count with nothing stored)
  bool fallback = false;  // the family's kernels do not take this launch; the generic family's kernel for the same program runs it
  int64_t slice_trips = 0;  // a generic program whose loop may run in slices: iterations of it (at most, over the grid's corners)
  double mean_trips = 0;    // and the mean of the corners'
  std::string describe;
  // matrix products with a fused epilogue: which program owns which BM x BN tile (device memory, owned by the binding)
  int *tile_pid = nullptr;
  int tiles_n = 0;
  Bound() = default;
  Bound(const Bound &) = delete;
  Bound &operator=(const Bound &) = delete;
  ~Bound() {
    if (tile_pid) (void)hipFree(tile_pid);
  }
};

}  // namespace

struct tts_plan {
  Plan plan;
  std::string family;
  TileTraits traits, fallback_traits;  // of plan.source and plan.fallback_source
  std::vector<int> arg_kinds;
  // bindings per (grid, scalar arguments), least recently used last; the oldest goes when there are more than 256
  struct CacheEntry {
    std::shared_ptr<Bound> bound;
    std::list<std::string>::iterator pos;
  };
  std::unordered_map<std::string, CacheEntry> cache;
  std::list<std::string> lru;
  std::mutex mu;
  const char *last_kernel = "";
  int last_slices = 1, last_meet = 0;
  // Split-K partial sums and arrival counters (device memory, owned by the plan), one set per stream the plan has been
  // launched on: launches on one stream run one after the other, launches on different streams may overlap and must
  // not share them.  Counters are zero between launches.
  struct SplitK {
    void *widened = nullptr;  // the int8-weight product's weights as fp16, for launches with many rows
    size_t widened_bytes = 0;
    float *workspace = nullptr;
    size_t workspace_bytes = 0;
    int *counters = nullptr;
    size_t counters_count = 0;
  };
  std::unordered_map<void *, SplitK> split_k;
  // Buffers a stream has outgrown.  Launches already enqueued (by this or another thread) may still use them, so they are
  // neither freed nor reused before the plan goes: growing never waits for the device.  A buffer grows to at least twice
  // its size, so the retired ones of a stream together are smaller than the one in use.
  std::vector<void *> retired;
  // A buffer of at least `need` bytes in *buf (of *have bytes); called with `mu` held.
  hipError_t grow(void **buf, size_t *have, size_t need) {
    if (*have >= need) return hipSuccess;
    size_t got = std::max(need, 2 * *have);
    void *fresh = nullptr;
    hipError_t e = hipMalloc(&fresh, got);
    if (e != hipSuccess && got > need) {
      (void)hipGetLastError();
      got = need;
      e = hipMalloc(&fresh, got);
    }
    if (e != hipSuccess) return e;
    if (*buf) retired.push_back(*buf);
    *buf = fresh;
    *have = got;
    return hipSuccess;
  }
  // At least `need` arrival counters for a stream; called with `mu` held.  New counters are cleared on the stream, in front of the
  // launches on it that use them, so that nothing waits for the device; the old ones, which launches in flight may still be
  // bumping, are retired.
  hipError_t grow_counters(SplitK &sk, size_t need, hipStream_t s) {
    if (sk.counters_count >= need) return hipSuccess;
    int *fresh = nullptr;
    const size_t count = std::max(need, 2 * sk.counters_count);
    hipError_t e = hipMalloc((void **)&fresh, count * sizeof(int));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(clear_ints_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, fresh, (int)count);
    e = hipGetLastError();
    retired.push_back(e == hipSuccess ? sk.counters : fresh);  // (freeing null is nothing)
    if (e != hipSuccess) return e;
    sk.counters = fresh;
    sk.counters_count = count;
    return hipSuccess;
  }
  // The stream's scratch memory, with at least so many bytes of workspace, counters and widened weights: null where that cannot be had,
  // because the stream records a graph and does not have it yet, or because there is no memory.  Called with `mu` held; every
  // caller has a way to launch without.  (Another stream may be recording: allocating is allowed beside that in the relaxed mode alone.)
  SplitK *room(hipStream_t s, size_t bytes, size_t counters, size_t widened = 0) {
    SplitK &sk = split_k[s];
    if (sk.workspace_bytes >= bytes && sk.counters_count >= counters && sk.widened_bytes >= widened) return &sk;
    if (is_capturing(s)) return nullptr;
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool changed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    hipError_t e = grow((void **)&sk.workspace, &sk.workspace_bytes, bytes);
    if (e == hipSuccess) e = grow(&sk.widened, &sk.widened_bytes, widened);
    if (e == hipSuccess) e = grow_counters(sk, counters, s);
    if (changed) (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e == hipSuccess) return &sk;
    (void)hipGetLastError();
    return nullptr;
  }
  RtcModule *fused = nullptr;  // the kernel compiled for this plan at its first launch (fused maps, tile programs)
  RtcModule *gemm_rtc[GEMM_EPILOGUE_KERNELS] = {};  // matrix products with a fused epilogue: launch_gemm_epilogue's kernels
  RtcModule *fallback = nullptr;  // the generic family's kernel for a matrix-product plan (launches the product kernels decline)
  ~tts_plan() {
    for (auto &kv : split_k) {
      if (kv.second.workspace) (void)hipFree(kv.second.workspace);
      if (kv.second.widened) (void)hipFree(kv.second.widened);
      if (kv.second.counters) (void)hipFree(kv.second.counters);
    }
    for (void *p : retired) (void)hipFree(p);
    rtc_release(fused);
    rtc_release(fallback);
    for (RtcModule *m : gemm_rtc) rtc_release(m);
  }
};

namespace {

struct Resolver {
  const Plan &pl;
  const ExprPool &X;
  std::vector<int64_t> ints;
  std::vector<double> floats;
  int g[3];
  Resolver(const Plan &p, const tts_arg *args, int n, int gx, int gy, int gz) : pl(p), X(p.prog.pool), g{gx, gy, gz} {
    ints.assign(n, 0);
    floats.assign(n, 0.0);
    for (int i = 0; i < n; i++) {
      if (args[i].kind == TTS_ARG_INT) ints[i] = args[i].v.i;
      if (args[i].kind == TTS_ARG_FLOAT) floats[i] = args[i].v.f;
    }
  }
  EvalEnv env(int px = 0, int py = 0, int pz = 0) const {
    EvalEnv e;
    e.args = ints.data();
    e.pid[0] = px; e.pid[1] = py; e.pid[2] = pz;
    e.nprog[0] = g[0]; e.nprog[1] = g[1]; e.nprog[2] = g[2];
    e.iv.assign(pl.prog.num_loops, 0);
    e.iter.assign(pl.prog.num_loops, {});
    e.result.assign(pl.prog.num_loops, {});
    return e;
  }
  int64_t ev(const std::string &name, const EvalEnv &e) const { return X.eval(pl.e.at(name), e); }
  int64_t ev0(const std::string &name) const { return ev(name, env()); }
  Affine affine(const std::string &name) const {
    const Lin &l = pl.lin.at(name);
    EvalEnv e = env();
    Affine a;
    a.c0 = X.eval(l.c0, e);
    for (int k = 0; k < 3; k++) a.c[k] = X.eval(l.coef[k], e);
    if (l.orig >= 0) {
      // the linear form was derived looking through i32 -> index extensions; confirm at every corner of the grid
      // (a coefficient may be negative, so the extreme offset can sit at any of them) that no 32-bit product wrapped
      for (int corner = 0; corner < 8; corner++) {
        const int px = (corner & 1) ? g[0] - 1 : 0, py = (corner & 2) ? g[1] - 1 : 0, pz = (corner & 4) ? g[2] - 1 : 0;
        if (((corner & 1) && g[0] == 1) || ((corner & 2) && g[1] == 1) || ((corner & 4) && g[2] == 1)) continue;  // same program as another corner
        EvalEnv at = env(px, py, pz);
        int64_t want = X.eval(l.orig, at);
        int64_t got = a.c0 + a.c[0] * px + a.c[1] * py + a.c[2] * pz;
        if (want != got)
          throw Invalid("32-bit overflow in the kernel's index arithmetic for '" + name + "' at program (" + std::to_string(px) + ", " +
                        std::to_string(py) + ", " + std::to_string(pz) + ") of the grid");
      }
    }
    return a;
  }
};

std::string show(const Affine &a) {
  std::ostringstream os;
  os << a.c0 << "+" << a.c[0] << "*x+" << a.c[1] << "*y+" << a.c[2] << "*z";
  return os.str();
}

void bind_map1d(const Resolver &r, Bound &b) {
  Map1DParams &p = b.map1d;
  p.xo = r.affine("x_off");
  p.yo = r.affine("y_off");
  p.zo = r.affine("z_off");
  p.block = (int)r.pl.k.at("block");
  p.masked = (int)r.pl.k.at("masked");
  p.op = (int)r.pl.k.at("op");
  p.swap = (int)r.pl.k.at("swap");
  if (p.masked) {
    p.m_start = r.affine("m_start");
    p.bound = r.ev0("bound");
  }
  std::ostringstream os;
  os << "kernel=map1d_f32\nop=" << p.op << "\nswap=" << p.swap << "\nblock=" << p.block << "\nmasked=" << p.masked
     << "\nx_off=" << show(p.xo) << "\ny_off=" << show(p.yo) << "\nz_off=" << show(p.zo) << "\nm_start=" << show(p.m_start)
     << "\nbound=" << p.bound << "\n";
  b.describe = os.str();
}

void bind_fused_map(const Resolver &r, Bound &b) {
  MapNParams &p = b.mapn;
  const auto &k = r.pl.k;
  p.block = (int)k.at("block");
  p.masked = (int)k.at("masked");
  p.n_in = (int)k.at("n_in");
  p.n_out = (int)k.at("n_out");
  p.n_ins = (int)k.at("n_ins");
  p.n_regs = (int)k.at("n_regs");
  if (p.masked) {
    p.m_start = r.affine("m_start");
    p.bound = r.ev0("bound");
  }
  std::ostringstream os;
  os << "kernel=mapn\nblock=" << p.block << "\nmasked=" << p.masked << "\nbound=" << p.bound << "\nm_start=" << show(p.m_start)
     << "\nregs=" << p.n_regs << "\n";
  for (int i = 0; i < p.n_in; i++) {
    std::string n = "in" + std::to_string(i);
    p.in_off[i] = r.affine(n + "_off");
    p.in_type[i] = (uint8_t)k.at(n + "_type");
    p.in_reg[i] = (uint8_t)k.at(n + "_reg");
    p.in_other[i] = (float)r.pl.f.at(n + "_other");
    os << n << "_off=" << show(p.in_off[i]) << "\n";
  }
  for (int j = 0; j < p.n_out; j++) {
    std::string n = "out" + std::to_string(j);
    p.out_off[j] = r.affine(n + "_off");
    p.out_type[j] = (uint8_t)k.at(n + "_type");
    p.out_reg[j] = (uint8_t)k.at(n + "_reg");
    os << n << "_off=" << show(p.out_off[j]) << "\n";
  }
  for (int q = 0; q < (int)k.at("n_imm"); q++) {
    int64_t arg = k.at("imm" + std::to_string(q) + "_arg");
    p.imm[q] = arg >= 0 ? (float)r.floats.at(arg) : (float)r.pl.f.at("imm" + std::to_string(q));
  }
  for (int t = 0; t < p.n_ins; t++) {
    uint64_t w = (uint64_t)k.at("ins" + std::to_string(t));
    MapIns &ins = p.ins[t];
    ins.op = w & 255; ins.dst = (w >> 8) & 255; ins.a = (w >> 16) & 255; ins.b = (w >> 24) & 255;
    ins.c = (w >> 32) & 255; ins.kinds = (w >> 40) & 255; ins.round = (w >> 48) & 255; ins.pad = 0;
    auto src = [&](int kind, int idx) {
      return kind == MS_PREV ? std::string("prev") : kind == MS_IMM ? "#" + std::to_string(p.imm[idx]) : "r" + std::to_string(idx);
    };
    os << "ins" << t << "=op" << (int)ins.op << " " << ((ins.kinds & 64) ? std::string("prev") : "r" + std::to_string(ins.dst)) << " <- "
       << src(ins.kinds & 3, ins.a) << ", " << src((ins.kinds >> 2) & 3, ins.b) << ", " << src((ins.kinds >> 4) & 3, ins.c)
       << (ins.round ? (ins.round == 1 ? " ->f16" : " ->bf16") : "") << "\n";
  }
  b.describe = os.str();
}

void bind_softmax(const Resolver &r, Bound &b) {
  SoftmaxParams &p = b.softmax;
  p.in_off = r.affine("in_off");
  p.out_off = r.affine("out_off");
  p.d_in = r.ev0("in_dims");
  p.d_out = r.ev0("out_dims");
  p.block = (int)r.pl.k.at("block");
  p.other = (float)r.pl.f.at("other");
  p.propagate_nan = r.pl.signature.find("maximumf") != std::string::npos;
  p.elem_kind = (int)r.pl.k.at("elem_kind");
  if (p.block > 65536) throw Unsupported("row_softmax: block sizes above 65536 are not implemented");
  std::ostringstream os;
  os << "kernel=softmax_f32\nelem=" << (p.elem_kind == 2 ? "f32" : p.elem_kind == 1 ? "bf16" : "f16") << "\nblock=" << p.block << "\nd_in=" << p.d_in << "\nd_out=" << p.d_out << "\nother=" << p.other
     << "\nin_off=" << show(p.in_off) << "\nout_off=" << show(p.out_off) << "\n";
  b.describe = os.str();
}

void bind_layernorm(const Resolver &r, Bound &b) {
  LayerNormParams &p = b.layernorm;
  p.x_off = r.affine("x_off");
  p.y_off = r.affine("y_off");
  p.w_off = r.affine("w_off");
  p.b_off = r.affine("b_off");
  p.mean_off = r.affine("mean_off");
  p.rstd_off = r.affine("rstd_off");
  p.N = r.ev0("N");
  p.eps = (float)r.floats.at(r.pl.k.at("eps_arg"));
  p.elem_kind = (int)r.pl.k.at("elem_kind");
  if (p.N > INT32_MAX) throw Invalid("layernorm_fwd: N does not fit 32 bits");
  std::ostringstream os;
  os << "kernel=layernorm_fwd\nN=" << p.N << "\neps=" << p.eps << "\nelem=" << (p.elem_kind == 2 ? "f32" : p.elem_kind == 1 ? "bf16" : "f16") << "\nx_off=" << show(p.x_off)
     << "\ny_off=" << show(p.y_off) << "\nw_off=" << show(p.w_off) << "\nb_off=" << show(p.b_off)
     << "\nmean_off=" << show(p.mean_off) << "\nrstd_off=" << show(p.rstd_off) << "\n";
  b.describe = os.str();
}

// Shared by both GEMM families: evaluates every program's tile origin and
// operand offsets, and proves that the grid of programs is exactly a dense
// C[M,N] = A[M,K] * B[K,N] tiled BM x BN, so that one kernel with its own
// tiling may compute it.
struct DenseGemm {
  int64_t M, N, K, lda, ldb, ldc;
  bool a_trans = false, b_trans = false;  // column-major operands (the tutorial's `b.T`): the pitch is the other stride
  std::vector<int> tile_pid;  // per BM x BN tile (row-major over the tile grid): linear id of the program that computes it
  int tiles_n = 0;
  // a batch of products of this shape: product b reads A and B and writes C batch_a * b, batch_b * b, batch_c * b elements further on
  int64_t batches = 1, batch_a = 0, batch_b = 0, batch_c = 0;
};

DenseGemm prove_dense_gemm(const Resolver &r, const char *F) {
  const Plan &pl = r.pl;
  const ExprPool &X = r.X;
  const int64_t BM = pl.k.at("BM"), BN = pl.k.at("BN"), BK = pl.k.at("BK");
  const int loop = (int)pl.k.at("loop");
  DenseGemm d;
  d.M = r.ev0("M");
  d.N = r.ev0("N");
  const int64_t sam = r.ev0("sam"), sak = r.ev0("sak"), sbk = r.ev0("sbk"), sbn = r.ev0("sbn"), scn = r.ev0("scn");
  d.ldc = r.ev0("scm");
  auto need = [&](bool ok, const std::string &why) {
    if (!ok) throw Unsupported(std::string(F) + ": " + why);
  };
  // the reference's lowering takes any strides (StructuredToMemref.cpp:105-138); these kernels want one stride of each
  // operand to be 1 and C row-major
  need(sak == 1 || sam == 1, "neither stride of A is 1");
  need(sbn == 1 || sbk == 1, "neither stride of B is 1");
  need(scn == 1, "the inner stride of C is not 1");
  d.a_trans = sak != 1;
  d.b_trans = sbn != 1;
  d.lda = d.a_trans ? sak : sam;
  d.ldb = d.b_trans ? sbn : sbk;
  need(d.M > 0 && d.N > 0, "empty problem");
  // a pitch of 0 is a broadcast operand, which the kernels read correctly; a negative one would become an unsigned byte
  // offset in the kernels, and rows of C that overlap or run backwards are not a dense product
  need(d.lda >= 0 && d.ldb >= 0, "a negative pitch of A or B");
  need(d.ldc > 0, "a pitch of C that is not positive");
  // K: the loop must sweep K in full blocks followed by at most one partial block
  int64_t trip = r.ev0("trip");
  need(trip >= 0 && trip < (1 << 24), "unreasonable K trip count");
  d.K = 0;
  {
    EvalEnv e = r.env();
    for (int64_t k = 0; k < trip; k++) {
      e.iv[loop] = k;
      int64_t kd = X.eval(pl.e.at("kdim"), e);
      need(kd == BK || (k == trip - 1 && kd >= 0), "the K mask does not describe a contiguous sweep of K");
      d.K += kd;
    }
  }
  need(r.ev0("a_kstep") == BK * sak && r.ev0("b_kstep") == BK * sbk, "operand pointers do not advance by one K block per iteration");
  // wraparound operands: the period is the whole matrix, so rows (columns) inside the problem are not affected
  const bool a_wraps = pl.e.count("a_mod"), b_wraps = pl.e.count("b_mod");
  if (a_wraps) need(r.ev0("a_mod") == d.M * sam, "A rows wrap around with a period other than M");
  if (b_wraps) need(r.ev0("b_mod") == d.N * sbn, "B columns wrap around with a period other than N");
  // tiles: every program's origin, offsets consistent with a dense layout, exact cover
  // A grid with a whole multiple of that many programs may be a batch of products (a batch index on another grid axis,
  // tutorial-style bmm): the programs then fall into groups that differ by constant offsets into A, B and C, each group
  // an exact cover of its own C, the offsets in arithmetic progression, the C's apart.
  const int64_t tm = (d.M + BM - 1) / BM, tn = (d.N + BN - 1) / BN;
  const int64_t programs = (int64_t)r.g[0] * r.g[1] * r.g[2];
  need(programs % (tm * tn) == 0 && programs >= tm * tn, "the grid does not have one program per output tile");
  d.batches = programs / (tm * tn);
  need(d.batches == 1 || (!a_wraps && !b_wraps), "a batch of products with wrapped operands");
  need(d.batches <= 65535, "more than 65535 products in a batch");
  std::map<std::array<int64_t, 3>, int> batch_of;  // offsets (A, B, C) of a product beyond those of a single one -> its place in `seen`
  std::vector<std::vector<char>> seen;
  d.tile_pid.assign(tm * tn, 0);
  d.tiles_n = (int)tn;
  for (int z = 0; z < r.g[2]; z++)
    for (int y = 0; y < r.g[1]; y++)
      for (int x = 0; x < r.g[0]; x++) {
        EvalEnv e = r.env(x, y, z);
        int64_t r0 = r.ev("r0", e), c0 = r.ev("c0", e);
        need(r0 >= 0 && c0 >= 0 && r0 % BM == 0 && c0 % BN == 0 && r0 / BM < tm && c0 / BN < tn, "a program's tile origin is off the tile grid");
        const std::array<int64_t, 3> off = {r.ev("a_base", e) - r0 * sam, r.ev("b_base", e) - c0 * sbn, r.ev("c_base", e) - (r0 * d.ldc + c0)};
        if (d.batches == 1) {
          need(off[0] == 0, "A tile offset is not row0 * its row stride");
          need(off[1] == 0, "B tile offset is not col0 * its column stride");
          need(off[2] == 0, "C tile offset is not row0 * ldc + col0");
        }
        auto at = batch_of.find(off);
        if (at == batch_of.end()) {
          need((int64_t)batch_of.size() < d.batches, "the programs do not fall into products of one shape");
          at = batch_of.emplace(off, (int)seen.size()).first;
          seen.emplace_back(tm * tn, 0);
        }
        char &s = seen[at->second][(r0 / BM) * tn + c0 / BN];
        need(!s, "two programs compute the same output tile");
        s = 1;
        if (d.batches == 1) d.tile_pid[(r0 / BM) * tn + c0 / BN] = x + r.g[0] * (y + r.g[1] * z);
        if (a_wraps) need(r.ev("a_wrapped", e) == r0 * sam, "the wrapped part of A's offset is not row0 * its row stride");
        if (b_wraps) need(r.ev("b_wrapped", e) == c0 * sbn, "the wrapped part of B's offset is not col0 * its column stride");
      }
  if (d.batches > 1) {
    // (every product has tm * tn distinct tiles, and there are batches * tm * tn programs: all covers are exact)
    need((int64_t)batch_of.size() == d.batches, "the programs do not fall into products of one shape");
    std::vector<std::array<int64_t, 3>> offs;
    for (auto &kv : batch_of) offs.push_back(kv.first);
    std::sort(offs.begin(), offs.end(), [](const std::array<int64_t, 3> &a, const std::array<int64_t, 3> &b) { return a[2] < b[2]; });
    need(offs[0][0] == 0 && offs[0][1] == 0 && offs[0][2] == 0, "the first product of a batch does not start at the arguments' addresses");
    d.batch_a = offs[1][0];
    d.batch_b = offs[1][1];
    d.batch_c = offs[1][2];
    for (int64_t b = 0; b < d.batches; b++)
      need(offs[b][0] == b * d.batch_a && offs[b][1] == b * d.batch_b && offs[b][2] == b * d.batch_c, "the products of a batch are not evenly spaced");
    need(d.batch_c >= (d.M - 1) * d.ldc + d.N, "the results of a batch's products overlap");
  }
  return d;
}

// The product with gathered rows (match.cpp: try_gemm_gathered): one program per BM x BN tile of C, rows of A through an
// index vector at rows_ptr + row0, the matrix of a block of BM rows picked by the id at block_ptr + row0 / BM.
void bind_gemm_gathered(const Resolver &r, Bound &b) {
  const Plan &pl = r.pl;
  const char *F = "gemm (gathered rows)";
  auto need = [&](bool ok, const std::string &why) {
    if (!ok) throw Unsupported(std::string(F) + ": " + why);
  };
  const int64_t BM = pl.k.at("BM"), BN = pl.k.at("BN"), BK = pl.k.at("BK");
  GemmParams &p = b.gemm;
  p.M = r.ev0("M"); p.N = r.ev0("N"); p.K = r.ev0("K");
  p.lda = r.ev0("sam"); p.ldb = r.ev0("sbk"); p.ldc = r.ev0("scm");
  p.is_bf16 = (int)pl.k.at("is_bf16");
  need(p.M > 0 && p.N > 0 && p.K >= 0, "empty problem");
  need(BM % 128 == 0, "blocks of rows that are not whole 128-row kernel tiles");
  need(r.ev0("b_kstep") == BK * p.ldb, "the B pointer does not advance by one K block per iteration");
  need(p.lda >= 0 && p.lda <= INT32_MAX && p.ldb >= 0, "negative or oversized pitches");
  const int64_t tm = (p.M + BM - 1) / BM, tn = (p.N + BN - 1) / BN;
  need((int64_t)r.g[0] * r.g[1] * r.g[2] == tm * tn, "the grid does not have one program per output tile");
  std::vector<char> seen(tm * tn, 0);
  for (int z = 0; z < r.g[2]; z++)
    for (int y = 0; y < r.g[1]; y++)
      for (int x = 0; x < r.g[0]; x++) {
        EvalEnv e = r.env(x, y, z);
        const int64_t r0 = r.ev("r0", e), c0 = r.ev("c0", e);
        need(r0 >= 0 && c0 >= 0 && r0 % BM == 0 && c0 % BN == 0 && r0 / BM < tm && c0 / BN < tn, "a program's tile origin is off the tile grid");
        char &s = seen[(r0 / BM) * tn + c0 / BN];
        need(!s, "two programs compute the same output tile");
        s = 1;
        need(r.ev("block_off", e) == r0 / BM, "the matrix id of a block of rows is not read from ids[row0 / BM]");
        need(r.ev("c_base", e) == r0 * p.ldc + c0, "C tile offset is not row0 * ldc + col0");
      }
  p.b_block_rows = (int)BM;
  p.b_block_stride = r.ev0("block_stride");
  p.gather_mul32 = 1 | (pl.k.at("mul32") ? 2 : 0);
  std::ostringstream os;
  os << "kernel=gemm_mfma\ngathered=1\nM=" << p.M << "\nN=" << p.N << "\nK=" << p.K << "\nlda=" << p.lda << "\nldb=" << p.ldb << "\nldc=" << p.ldc
     << "\nbf16=" << p.is_bf16 << "\nblock_rows=" << p.b_block_rows << "\nblock_stride=" << p.b_block_stride << "\n";
  b.describe = os.str();
}

void bind_gemm(const Resolver &r, Bound &b) {
  if (r.pl.k.count("gathered")) return bind_gemm_gathered(r, b);
  DenseGemm d = prove_dense_gemm(r, "gemm");
  GemmParams &p = b.gemm;
  p.M = d.M; p.N = d.N; p.K = d.K; p.lda = d.lda; p.ldb = d.ldb; p.ldc = d.ldc;
  p.a_trans = d.a_trans; p.b_trans = d.b_trans;
  p.is_bf16 = (int)r.pl.k.at("is_bf16");
  p.is_f32 = r.pl.k.count("is_f32") ? (int)r.pl.k.at("is_f32") : 0;
  p.batches = (int)d.batches; p.batch_a = d.batch_a; p.batch_b = d.batch_b; p.batch_c = d.batch_c;
  if (p.batches > 1 && !r.pl.source.empty()) throw Unsupported("gemm: a fused epilogue on a batch of products");
  if (!r.pl.source.empty() && !p.is_f32) {  // a fused epilogue on 16-bit results looks up the program that owns an element
    may_allocate("a table of tile owners on the device");
    hipError_t e = hipMalloc((void **)&b.tile_pid, d.tile_pid.size() * sizeof(int));
    if (e == hipSuccess) e = hipMemcpy(b.tile_pid, d.tile_pid.data(), d.tile_pid.size() * sizeof(int), hipMemcpyHostToDevice);
    if (e != hipSuccess) throw std::runtime_error(std::string("gemm: tile table: ") + hipGetErrorString(e));
    b.tiles_n = d.tiles_n;
  }
  std::ostringstream os;
  os << "kernel=gemm_mfma\nM=" << p.M << "\nN=" << p.N << "\nK=" << p.K << "\nlda=" << p.lda << "\nldb=" << p.ldb
     << "\nldc=" << p.ldc << "\nbf16=" << p.is_bf16 << "\nf32=" << p.is_f32 << "\na_trans=" << p.a_trans << "\nb_trans=" << p.b_trans << "\n";
  if (p.batches > 1) os << "batches=" << p.batches << "\nbatch_a=" << p.batch_a << "\nbatch_b=" << p.batch_b << "\nbatch_c=" << p.batch_c << "\n";
  if (r.pl.source.empty()) {  // what it runs on with operands that are aligned (as these null ones are) and memory to be had
    p.meet = 1;
    const GemmChoice &choice = b.gemm_choice[15] = gemm_choose(p);
    b.gemm_chosen[15] = true;
    os << "slices=" << choice.split << "\nmeet=" << (choice.meeting > 0) << "\n";
  }
  b.describe = os.str();
}

void bind_w8a16(const Resolver &r, Bound &b) {
  DenseGemm d = prove_dense_gemm(r, "gemm_w8a16");
  if (d.a_trans || d.b_trans) throw Unsupported("gemm_w8a16: only row-major operands are implemented");
  if (d.batches > 1) throw Unsupported("gemm_w8a16: a batch of products");
  GemmW8A16Params &p = b.w8;
  p.M = d.M; p.N = d.N; p.K = d.K; p.lda = d.lda; p.ldw = d.ldb; p.ldc = d.ldc;
  p.split = gemm_w8a16_split(p);
  std::ostringstream os;
  os << "kernel=gemm_w8a16\nM=" << p.M << "\nN=" << p.N << "\nK=" << p.K << "\nlda=" << p.lda << "\nldw=" << p.ldw
     << "\nldc=" << p.ldc << "\nsplit=" << p.split << "\n";
  b.describe = os.str();
}

std::shared_ptr<Bound> resolve(tts_plan *h, int gx, int gy, int gz, const tts_arg *args, int n) {
  if (n != (int)h->arg_kinds.size())
    throw Invalid("expected " + std::to_string(h->arg_kinds.size()) + " kernel arguments, got " + std::to_string(n));
  std::string key;
  key.reserve(16 + 8 * n);
  int g[3] = {gx, gy, gz};
  key.append((const char *)g, sizeof g);
  for (int i = 0; i < n; i++) {
    if (args[i].kind != h->arg_kinds[i])
      throw Invalid("kernel argument " + std::to_string(i) + " has the wrong kind (pointer/integer/float)");
    if (args[i].kind != TTS_ARG_PTR) key.append((const char *)&args[i].v, 8);
  }
  std::lock_guard<std::mutex> lock(h->mu);
  auto it = h->cache.find(key);
  if (it != h->cache.end()) {
    h->lru.splice(h->lru.begin(), h->lru, it->second.pos);
    return it->second.bound;
  }
  auto b = std::make_shared<Bound>();
  b->family = h->plan.family;
  Resolver r(h->plan, args, n, gx, gy, gz);
  switch (b->family) {
    case Family::Map1D: bind_map1d(r, *b); break;
    case Family::RowSoftmax: bind_softmax(r, *b); break;
    case Family::LayerNormFwd: bind_layernorm(r, *b); break;
    case Family::Gemm:
    case Family::GemmW8A16:
      // what these families can only check now (strides, M, the grid's shape) may fail for a launch that is a valid
      // Triton program all the same: the generic family's kernel for the same program runs it
      try {
        if (b->family == Family::Gemm) bind_gemm(r, *b);
        else bind_w8a16(r, *b);
      } catch (const Unsupported &e) {
        if (h->plan.fallback_source.empty()) throw;
        b->fallback = true;
        b->describe = std::string("kernel=tile_program\nfallback_reason=") + e.what() + "\n";
      }
      break;
    case Family::FusedMap: bind_fused_map(r, *b); break;
    case Family::TileProgram: {
      b->describe = "kernel=tile_program\n";
      if (h->traits.sliced)
        for (const SOp &s : h->plan.prog.body)
          if (s.kind == SK::For && s.loop == h->traits.loop)
            for (int corner = 0; corner < 2; corner++) {
              const EvalEnv e = corner ? r.env(gx - 1, gy - 1, gz - 1) : r.env();
              const int64_t lb = r.X.eval(s.lb, e), ub = r.X.eval(s.ub, e), step = r.X.eval(s.step, e);
              const int64_t trips = ub > lb && step > 0 ? (ub - lb + step - 1) / step : 0;
              b->slice_trips = std::max(b->slice_trips, trips);
              b->mean_trips += 0.5 * (double)trips;
            }
      break;
    }
  }
  h->lru.push_front(key);
  h->cache[key] = {b, h->lru.begin()};
  if (h->cache.size() > 256) {  // launches in flight hold their own reference to the binding they use
    h->cache.erase(h->lru.back());
    h->lru.pop_back();
  }
  return b;
}

template <class T>
T *ptr_arg(const tts_arg *args, const Plan &pl, const char *name) {
  return (T *)args[pl.k.at(name)].v.ptr;
}

template <class F>
tts_status guarded(F &&f) {
  try {
    return f();
  } catch (const Unsupported &e) {
    return fail(TTS_UNSUPPORTED, e.what());
  } catch (const WouldAllocate &e) {
    return fail(TTS_UNSUPPORTED, e.what());
  } catch (const Invalid &e) {
    return fail(TTS_INVALID, e.what());
  } catch (const std::exception &e) {
    return fail(TTS_INVALID, e.what());
  }
}

const char *PLAN_MAGIC = "tts.plan 1";

// ---- tts_launch_noalloc: the split-K scratch memory of callers that cannot allocate
// Partial tiles first, arrival counters behind them.  One copy of the array per GPU, held until the process ends.
constexpr size_t NOALLOC_WORKSPACE_BYTES = (size_t)8 << 20;
constexpr size_t NOALLOC_COUNTERS = 4096;
constexpr int NOALLOC_MAX_DEVICES = 64;

}  // namespace

// In host code this name is only a handle for hipGetSymbolAddress: the device address is looked up once per device
// (noalloc_scratch) and that pointer is what kernels and copies receive.
static __device__ __align__(256) unsigned char scratch[NOALLOC_WORKSPACE_BYTES + NOALLOC_COUNTERS * sizeof(int)];

namespace {

// the current device's copy of `scratch`
unsigned char *noalloc_scratch() {
  static std::mutex mu;
  static unsigned char *ptrs[NOALLOC_MAX_DEVICES] = {};
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) throw std::runtime_error(std::string("hipGetDevice: ") + hipGetErrorString(e));
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) throw Invalid("tts_launch_noalloc: device ordinal out of range");
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) throw std::runtime_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    ptrs[dev] = (unsigned char *)p;
  }
  return ptrs[dev];
}

}  // namespace

extern "C" {

const char *tts_last_error(void) { return g_error.c_str(); }
void tts_free(void *p) { free(p); }

tts_status tts_ttir_to_structured(const char *ttir_text, char **out) {
  if (!ttir_text || !out) return fail(TTS_INVALID, "null argument");
  return guarded([&]() {
    Func f = parse_ttir(ttir_text);
    Program p = lower_ttir(f);
    *out = dup_string(print_program(p));
    return TTS_OK;
  });
}

tts_status tts_structured_to_plan(const char *structured_text, char **out_plan, size_t *out_len, char **out_name) {
  if (!structured_text || !out_plan || !out_len) return fail(TTS_INVALID, "null argument");
  return guarded([&]() {
    Program p = read_program(structured_text);
    std::string name = p.name;
    Plan pl = make_plan(std::move(p));  // refuses here, at compile time, if no family matches
    std::string bytes = std::string(PLAN_MAGIC) + " family=" + family_name(pl.family) + "\n" + structured_text;
    *out_plan = dup_string(bytes);
    *out_len = bytes.size();
    if (out_name) *out_name = dup_string(name);
    return TTS_OK;
  });
}

tts_status tts_plan_load(const char *plan_bytes, size_t len, tts_plan **out) {
  if (!plan_bytes || !out) return fail(TTS_INVALID, "null argument");
  return guarded([&]() {
    std::string text(plan_bytes, len);
    if (text.rfind(PLAN_MAGIC, 0) != 0) throw Invalid("not a tts launch plan");
    size_t nl = text.find('\n');
    std::string header = text.substr(0, nl);
    auto h = std::make_unique<tts_plan>();
    h->plan = make_plan(read_program(text.substr(nl + 1)));
    h->family = family_name(h->plan.family);
    if (h->plan.family == Family::TileProgram) h->traits = tile_traits(h->plan.source);
    h->fallback_traits = tile_traits(h->plan.fallback_source);
    // (a plan written before its program had a family of its own says tile_program, which runs any)
    if (header.find("family=" + h->family) == std::string::npos && header.find("family=tile_program") == std::string::npos)
      throw Invalid("plan header and plan body disagree on the kernel family");
    for (auto &t : h->plan.prog.arg_types)
      h->arg_kinds.push_back(t.ptr ? TTS_ARG_PTR : t.is_float() ? TTS_ARG_FLOAT : TTS_ARG_INT);
    *out = h.release();
    return TTS_OK;
  });
}

void tts_plan_destroy(tts_plan *plan) { delete plan; }
const char *tts_plan_kernel_name(const tts_plan *plan) { return plan->plan.prog.name.c_str(); }
const char *tts_plan_family(const tts_plan *plan) { return plan->family.c_str(); }
const char *tts_plan_signature(const tts_plan *plan) { return plan->plan.signature.c_str(); }
int tts_plan_num_args(const tts_plan *plan) { return (int)plan->arg_kinds.size(); }
int tts_plan_arg_kind(const tts_plan *plan, int i) {
  return i >= 0 && i < (int)plan->arg_kinds.size() ? plan->arg_kinds[i] : -1;
}
const char *tts_plan_last_kernel(const tts_plan *plan) { return plan->last_kernel; }
int tts_plan_last_slices(const tts_plan *plan, int *meet) {
  if (meet) *meet = plan->last_meet;
  return plan->last_slices;
}

tts_status tts_plan_describe_launch(tts_plan *plan, int gx, int gy, int gz, const tts_arg *args, int n, char **out) {
  if (!plan || !out || (n > 0 && !args)) return fail(TTS_INVALID, "null argument");
  return guarded([&]() {
    if ((int64_t)gx * gy * gz <= 0) {
      *out = dup_string("kernel=none\n");
      return TTS_OK;
    }
    auto b = resolve(plan, gx, gy, gz, args, n);
    *out = dup_string("family=" + plan->family + "\n" + b->describe);
    return TTS_OK;
  });
}

}  // extern "C"

namespace {

int compute_units() {  // of the current device (256 when the query fails)
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    return n;
  }();
  return cus;
}

// Slices of an online softmax's loop (tile_mma.h): where its workgroups leave CUs idle each walks all of its blocks alone, and where
// they fill them about once the longest loops are what the launch waits for.  The least modelled time, in iterations of a
// workgroup alone on its CU (half as long again beside another): the longest slice, or the work of the chip and half of that
// where workgroups wait for a place; a meeting of n slices takes 1.5 + 0.8 n.  Measured, us in 1 / 2 / 3 / 4 / 8 slices: 2 heads x 4096 x 128 causal (64
// workgroups) 90 / 51 / 39 / 32 / 30.5; 8 x 1405 x 64 (88) 26.9 / 19.4 / 19.7 / 18.1 / 18.5; 15 x 638 x 128 causal (75 of at most ten iterations)
// 23.4 / 20.8 / 20.3 / 21.8 / 26.2; 8 x 4096 x 128 causal (256) 91 / 72 / 60 / 61 / 77; 23 x 225 x 128 (46 of at most four) 14.3 / 16.0 / 16.8.
int softmax_slices(int64_t workgroups, int64_t turns, double mean, int resident) {
  const double cus = compute_units();
  int pick = 1;
  double pick_t = 0;
  for (int64_t n = 1; n <= std::min<int64_t>(16, std::max<int64_t>(turns, 1)); n++) {
    const double per_cu = (double)(workgroups * n) / cus;
    if (n > 1 && per_cu > 3) break;
    double t = (double)((turns + n - 1) / n) * (1 + 0.5 * std::max(0.0, std::min(1.0, per_cu - 1)));
    if (per_cu > resident) t = std::max(t, (double)workgroups * mean / cus * 0.75 + 0.5 * t);
    if (n > 1) t += 1.5 + 0.8 * (double)n;
    if (n == 1 || t < pick_t) { pick = (int)n; pick_t = t; }
  }
  return pick;
}

// tts_launch and tts_launch_noalloc (no_alloc: nothing below may allocate device memory or compile)
tts_status launch_impl(tts_plan *plan, int gx, int gy, int gz, void *stream, const tts_arg *args, int n, bool no_alloc) {
  if (!plan || (n > 0 && !args)) return fail(TTS_INVALID, "null argument");
  struct Flag {
    bool saved;
    explicit Flag(bool v) : saved(g_no_alloc) { g_no_alloc = v; }
    ~Flag() { g_no_alloc = saved; }
  } flag(no_alloc);
  return guarded([&]() {
    if (gx < 0 || gy < 0 || gz < 0) throw Invalid("negative grid");
    if ((int64_t)gx * gy * gz == 0) return TTS_OK;  // backend/driver.py:117
    auto b = resolve(plan, gx, gy, gz, args, n);
    const Plan &pl = plan->plan;
    {
      // The device's grid holds 65535 along y and z; the reference's launcher loops over any extents
      // (backend/driver.py:116-133).  For larger ones every family launches one-dimensionally and numbers its programs
      // itself, as the compiled fused map and the row softmax always do (the matrix products use tilings of their own);
      // only the fused map's interpreter (a tuning aid) is left out.
      const char *mode = getenv("TTS_FUSED_MAP");
      const bool interpreter = pl.family == Family::FusedMap && !b->fallback && mode && std::string(mode) == "interpreter";
      if ((gy > 65535 || gz > 65535) && interpreter) throw Unsupported("grid y/z extents above 65535 on the fused map's interpreter");
      if ((int64_t)gx * gy * gz > INT32_MAX) throw Unsupported("more than 2^31 - 1 programs in a launch");
    }
    hipStream_t s = (hipStream_t)stream;
    hipError_t err = hipSuccess;
    const char *kname = "";
    int slices = 1, meet = 0;
    // one workgroup of 256 threads per Triton program, on the kernel generated for the program (compiled at its first use)
    auto run_tile_program = [&](RtcModule **slot, const std::string &source, const TileTraits &traits) -> tts_status {
      struct TileArgs { void *ptr[TILE_MAX_ARGS]; long long ival[TILE_MAX_ARGS]; double fval[TILE_MAX_ARGS]; int swap_xy, lgx, lgy, lgz; } a{};
      for (int i = 0; i < n; i++) {
        if (args[i].kind == TTS_ARG_PTR) a.ptr[i] = args[i].v.ptr;
        else if (args[i].kind == TTS_ARG_INT) a.ival[i] = args[i].v.i;
        else a.fval[i] = args[i].v.f;
      }
      {
        std::lock_guard<std::mutex> lock(plan->mu);
        if (!*slot) {
          may_allocate("to compile the program's kernel");
          std::string why;
          hipError_t ce = rtc_compile(source, "tile_program", slot, &why);
          if (ce != hipSuccess) return fail(TTS_HIP_ERROR, "tile_program: " + why + "\n--- source ---\n" + source);
        }
      }
      kname = "tile_program (hipRTC)";
      // A grid holds 2^32 - 1 threads along x and 65535 workgroups along y and z.  Launches beyond that are one-dimensional and the
      // kernel numbers the programs itself (x fastest), along y from 2^23 workgroups on, where surplus ones find no program.
      constexpr int64_t MOST_ALONG_X = 1 << 23;
      auto grid_fits = [&](bool swapped) { return (swapped ? gy : gx) <= MOST_ALONG_X && (swapped ? gx : gy) <= 65535 && gz <= 65535; };
      auto launch_numbered = [&](int64_t workgroups, void *arguments, size_t size) {
        const int64_t along_x = std::min(workgroups, MOST_ALONG_X);
        return rtc_launch(*slot, (int)along_x, (int)((workgroups + along_x - 1) / along_x), 1, 256, arguments, size, s);
      };
      if (traits.matrix) {  // a one-dimensional launch that numbers the programs itself
        kname = "tile_program (hipRTC, matrix layout)";
        int64_t e[3] = {gx, gy, gz};
        int64_t &shared = e[traits.axis < 0 ? 0 : traits.axis];
        shared = (shared + traits.programs - 1) / traits.programs;
        a.lgx = gx; a.lgy = gy; a.lgz = gz;
        // (a grid holds 2^32 - 1 threads along x: larger launches continue along y, where surplus workgroups find no program)
        const int64_t workgroups = e[0] * e[1] * e[2], along_x = std::min<int64_t>(workgroups, 1 << 23);
        if (traits.sliced) {
          struct { TileArgs t; int slices; float *partial; int *counters; } sa{};
          sa.t = a;
          sa.slices = softmax_slices(workgroups, b->slice_trips, b->mean_trips, rtc_resident_workgroups(*slot));
          if (sa.slices > 1 && (no_alloc || is_capturing(s))) sa.slices = 1;  // (as for the sums below)
          if (sa.slices > 1) {
            std::lock_guard<std::mutex> lock(plan->mu);
            if (const tts_plan::SplitK *sk = plan->room(s, (size_t)workgroups * sa.slices * traits.floats * sizeof(float), (size_t)workgroups * 32)) {  // (128 bytes apart)
              sa.partial = sk->workspace;
              sa.counters = sk->counters;
            } else {
              sa.slices = 1;
            }
          }
          slices = sa.slices;
          meet = slices > 1;
          const int64_t all = workgroups * sa.slices, x = std::min<int64_t>(all, 1 << 23);
          err = rtc_launch(*slot, (int)x, (int)((all + x - 1) / x), 1, traits.threads, &sa, sizeof sa, s);
          return TTS_OK;
        }
        err = rtc_launch(*slot, (int)along_x, (int)((workgroups + along_x - 1) / along_x), 1, traits.threads, &a, sizeof a, s);
        return TTS_OK;
      }
      if (traits.sliced) {
        // As many workgroups as the device holds at once, each program's loop dealt to an equal number of them, two
        // iterations each at least (dw and db of LayerNorm on fp16 [4096, 8192], 64 programs of 128 iterations: 341 us with
        // one workgroup per program, 27 us in 12 slices), and no more than 3 sqrt(iterations): an iteration takes some 0.75 us
        // of a slice and a slice some 0.08 us of the workgroup that adds them all (16 programs of 94 iterations: 47 / 23 / 11
        // slices 15.0 / 13.3 / 16.8 us; of 32 iterations: 16 / 8 / 4 slices 8.2 / 11.4 / 14.7 us).  A launch that may not
        // allocate keeps to one slice, and so does one that is recorded into a graph: the graph may be replayed beside
        // launches that use the same stream's workspace.
        const int64_t programs = (int64_t)gx * gy * gz;
        struct { TileArgs t; int slices; float *partial; int *counters; } sa{};
        sa.slices = (int)std::max<int64_t>(1, std::min({(int64_t)rtc_resident_workgroups(*slot) * compute_units() / programs, b->slice_trips / 2, 3 * (int64_t)std::sqrt((double)b->slice_trips), (int64_t)1024}));
        if (sa.slices > 1 && (no_alloc || is_capturing(s))) sa.slices = 1;
        if (sa.slices > 1) {
          std::lock_guard<std::mutex> lock(plan->mu);
          if (const tts_plan::SplitK *sk = plan->room(s, (size_t)programs * sa.slices * traits.floats * sizeof(float), (size_t)programs * 32)) {  // (128 bytes apart)
            sa.partial = sk->workspace;
            sa.counters = sk->counters;
          } else {
            sa.slices = 1;
          }
        }
        slices = sa.slices;
        meet = slices > 1;
        // one slice: the grid as it is, a workgroup per program, its x and y exchanged where the program asks for that (see below)
        const bool whole = sa.slices == 1, swap = whole && traits.swaps_grid && gy > 1 && gx <= 65535;
        if (whole && grid_fits(swap)) {
          a.swap_xy = swap ? 1 : 0;
          sa.t = a;
          err = swap ? rtc_launch(*slot, gy, gx, gz, 256, &sa, sizeof sa, s) : rtc_launch(*slot, gx, gy, gz, 256, &sa, sizeof sa, s);
          return TTS_OK;
        }
        a.lgx = gx; a.lgy = gy; a.lgz = gz;
        sa.t = a;
        err = launch_numbered(programs * sa.slices, &sa, sizeof sa);
        return TTS_OK;
      }
      // the program asks for neighbouring workgroups along program_id(1) (tile_codegen.cpp); grid.y holds 65535 at most
      a.swap_xy = traits.swaps_grid && gy > 1 && gx <= 65535 ? 1 : 0;
      // A workgroup per program.  (A few workgroups per CU that walk the programs with the weights they share held in
      // registers lose since every row moves in 16-byte accesses, us walking / a workgroup each: LayerNorm's dx bf16 [8192, 4096]
      // 54.3 / 42.8, [8192, 2048] 32.4 / 24.4, [8192, 3001] 57.8 / 45.3; RMSNorm fp16 [8000, 5120] 38.1 / 33.1, [8000, 4096]
      // 28.7 / 25.3; ahead only on some numbers of whole rows of 8192, [2000, 8192] 14.7 / 16.2, [2760, 8192] 18.6 / 20.0.)
      if (!grid_fits(a.swap_xy)) {
        a.swap_xy = 0;
        a.lgx = gx; a.lgy = gy; a.lgz = gz;
        err = launch_numbered((int64_t)gx * gy * gz, &a, sizeof a);
      } else {
        err = a.swap_xy ? rtc_launch(*slot, gy, gx, gz, 256, &a, sizeof a, s) : rtc_launch(*slot, gx, gy, gz, 256, &a, sizeof a, s);
      }
      return TTS_OK;
    };
    if (b->fallback) {
      tts_status st = run_tile_program(&plan->fallback, pl.fallback_source, plan->fallback_traits);
      if (st != TTS_OK) return st;
      plan->last_kernel = kname;
      plan->last_slices = slices;
      plan->last_meet = meet;
      if (err != hipSuccess) return fail(TTS_HIP_ERROR, std::string("kernel launch failed: ") + hipGetErrorString(err));
      return TTS_OK;
    }
    switch (b->family) {
      case Family::Map1D: {
        Map1DParams p = b->map1d;
        p.x = ptr_arg<const float>(args, pl, "x_arg");
        p.y = ptr_arg<const float>(args, pl, "y_arg");
        p.z = ptr_arg<float>(args, pl, "z_arg");
        err = launch_map1d(p, gx, gy, gz, s, &kname);
        break;
      }
      case Family::FusedMap: {
        MapNParams p = b->mapn;
        for (int i = 0; i < p.n_in; i++) p.in[i] = ptr_arg<const void>(args, pl, ("in" + std::to_string(i) + "_arg").c_str());
        for (int j = 0; j < p.n_out; j++) p.out[j] = ptr_arg<void>(args, pl, ("out" + std::to_string(j) + "_arg").c_str());
        // TTS_FUSED_MAP=interpreter keeps the program on the interpreter kernel; otherwise it is compiled
        // into a kernel of its own at the plan's first launch (scalar arguments stay arguments: one compile per plan)
        const char *mode = getenv("TTS_FUSED_MAP");
        if (mode && std::string(mode) == "interpreter") {
          err = launch_mapn(p, gx, gy, gz, s, &kname);
          break;
        }
        {
          std::lock_guard<std::mutex> lock(plan->mu);
          if (!plan->fused) {
            may_allocate("to compile the fused map's kernel");
            std::string why;
            hipError_t ce = fused_map_compile(p, &plan->fused, &why);
            if (ce != hipSuccess) return fail(TTS_HIP_ERROR, "fused_map: " + why);
          }
        }
        kname = "fused_map (hipRTC)";
        err = fused_map_launch(plan->fused, p, gx, gy, gz, s);
        break;
      }
      case Family::TileProgram: {
        tts_status st = run_tile_program(&plan->fused, pl.source, plan->traits);
        if (st != TTS_OK) return st;
        break;
      }
      case Family::RowSoftmax: {
        SoftmaxParams p = b->softmax;
        p.in = ptr_arg<const void>(args, pl, "in_arg");
        p.out = ptr_arg<void>(args, pl, "out_arg");
        err = launch_softmax(p, gx, gy, gz, s, &kname);
        break;
      }
      case Family::LayerNormFwd: {
        LayerNormParams p = b->layernorm;
        p.x = ptr_arg<const void>(args, pl, "x_arg");
        p.y = ptr_arg<void>(args, pl, "y_arg");
        p.w = ptr_arg<const void>(args, pl, "w_arg");
        p.b = ptr_arg<const void>(args, pl, "b_arg");
        p.mean = ptr_arg<float>(args, pl, "mean_arg");
        p.rstd = ptr_arg<float>(args, pl, "rstd_arg");
        err = launch_layernorm(p, gx, gy, gz, s, &kname);
        break;
      }
      case Family::Gemm: {
        GemmParams p = b->gemm;
        p.a = ptr_arg<const void>(args, pl, "a_arg");
        p.b = ptr_arg<const void>(args, pl, "b_arg");
        p.c = ptr_arg<void>(args, pl, "c_arg");
        if (pl.k.count("gathered")) {
          p.a_rows = ptr_arg<const int>(args, pl, "rows_arg");
          p.b_block = ptr_arg<const int>(args, pl, "block_arg");
        }
        p.split = 1;
        p.partial = nullptr;
        p.meet = 0;
        p.counters = nullptr;
        if (pl.source.empty()) {
          // a product with too few tiles for the chip runs in K slices, whose partial sums need memory: the stream's
          // workspace (as for the int8-weight product), or the static array of the call that may not allocate, when
          // they fit there (else that call runs the product without slices)
          // (the any-shape kernel keeps to whole products where the launch may not allocate or is recorded into a graph)
          // slices that meet in the kernel count their arrivals: not where a graph could be replayed beside other launches
          const bool recorded = is_capturing(s);
          auto choose = [&](bool meet) {
            p.meet = meet;
            const int at = (((uintptr_t)p.a & 15) == 0) | (((uintptr_t)p.b & 15) == 0) << 1 | (((uintptr_t)p.c & 3) == 0) << 2 | meet << 3;
            std::lock_guard<std::mutex> lock(plan->mu);
            if (!b->gemm_chosen[at]) {
              b->gemm_choice[at] = gemm_choose(p);
              b->gemm_chosen[at] = true;
            }
            return b->gemm_choice[at];
          };
          GemmChoice choice = choose(!no_alloc && !recorded);
          if (choice.split > 1 && !(choice.tile < 0 && (no_alloc || recorded))) {
            p.split = choice.split;
            if (no_alloc) {  // as many slices as the static array holds
              const size_t one = (size_t)p.M * p.N * std::max(1, p.batches) * sizeof(float);
              p.split = (int)std::min<size_t>((size_t)choice.split, NOALLOC_WORKSPACE_BYTES / one);
              if (p.split > 1) p.partial = reinterpret_cast<float *>(noalloc_scratch());
              else p.split = 1;
            } else {
              auto room = [&](size_t bytes, size_t counters) {
                std::lock_guard<std::mutex> lock(plan->mu);
                const tts_plan::SplitK *sk = plan->room(s, bytes, counters);
                if (!sk) return false;
                p.partial = sk->workspace;
                if (counters) p.counters = sk->counters;
                return true;
              };
              // without memory the second kernel's sums may still fit what the stream has, and the whole product needs none
              // (a later recording finds room for the sums that a second kernel adds)
              if (!room(choice.meeting ? std::max(choice.bytes, choose(false).bytes) : choice.bytes, 32 * choice.meeting)) {
                if (choice.meeting) choice = choose(false);
                else choice.split = 1;
                p.split = choice.split > 1 && room(choice.bytes, 0) ? choice.split : 1;
              }
            }
          }
          slices = p.split;
          meet = p.counters != nullptr;
          err = launch_gemm(p, s, &kname, &choice);
          break;
        }
        static_assert(TILE_MAX_ARGS == 32, "GemmEpilogueArgs holds 32 arguments");
        GemmEpilogueArgs a{};
        for (int i = 0; i < n; i++) {
          if (args[i].kind == TTS_ARG_PTR) a.ptr[i] = args[i].v.ptr;
          else if (args[i].kind == TTS_ARG_INT) a.ival[i] = args[i].v.i;
          else a.fval[i] = args[i].v.f;
        }
        a.tile_pid = b->tile_pid;
        a.tiles_n = b->tiles_n;
        a.gx = gx;
        a.gy = gy;
        a.gz = gz;
        std::string why;
        if (p.is_f32 && !pl.fallback_source.empty()) {
          // The generic kernel takes every launch of a product on fp32 operands, the matrix kernel most: the first launch compiles both, so
          // that later ones that may not compile find a kernel whichever they need.
          bool generic = false;
          {
            std::lock_guard<std::mutex> lock(plan->mu);
            const bool compiled = gemm_epilogue_compiled(p, plan->gemm_rtc);
            generic = plan->fallback && !compiled && (no_alloc || is_capturing(s));
            if (!plan->fallback && !no_alloc && !compiled) {
              const hipError_t ce = rtc_compile(pl.fallback_source, "tile_program", &plan->fallback, &why);
              if (ce != hipSuccess) return fail(TTS_HIP_ERROR, "tile_program: " + why);
            }
          }
          if (generic) {
            tts_status st = run_tile_program(&plan->fallback, pl.fallback_source, plan->fallback_traits);
            if (st != TTS_OK) return st;
            break;
          }
        }
        if (no_alloc) {
          std::lock_guard<std::mutex> lock(plan->mu);
          if (!gemm_epilogue_compiled(p, plan->gemm_rtc)) may_allocate("to compile the matrix product with its fused epilogue");
        }
        {
          std::lock_guard<std::mutex> lock(plan->mu);
          const int want = gemm_epilogue_split(p);
          const bool recorded = is_capturing(s);
          // (a launch that a graph records takes an equivalent kernel that is there, as one that may not allocate does: compiling
          // would load a module in the middle of the recording)
          const bool may_compile = !no_alloc && !(recorded && gemm_epilogue_compiled(p, plan->gemm_rtc));
          if (want > 1 && !no_alloc && !recorded) {
            p.split = want;
            if (const tts_plan::SplitK *sk = plan->room(s, gemm_workspace_bytes(p), 0)) p.partial = sk->workspace;
            else p.split = 1;
          }
          slices = p.split;
          err = launch_gemm_epilogue(p, pl.source, plan->gemm_rtc, may_compile, a, s, &kname, &why);
        }
        if (err != hipSuccess && !why.empty()) return fail(TTS_HIP_ERROR, "gemm epilogue: " + why);
        break;
      }
      case Family::GemmW8A16: {
        GemmW8A16Params p = b->w8;
        p.a = ptr_arg<const void>(args, pl, "a_arg");
        p.w = ptr_arg<const int8_t>(args, pl, "b_arg");
        p.scale = ptr_arg<const void>(args, pl, "s_arg");
        p.c = ptr_arg<void>(args, pl, "c_arg");
        const bool tiled = gemm_w8a16_is_tiled(p);  // (p.split is the decode kernels')
        if (p.split > 1 && no_alloc && !tiled) {
          const size_t need = gemm_w8a16_workspace_bytes(p), ncount = gemm_w8a16_counters(p);
          if (need > NOALLOC_WORKSPACE_BYTES || ncount > NOALLOC_COUNTERS)
            throw Unsupported("tts_launch_noalloc: the split-K partial tiles of this shape need " + std::to_string(need) + " bytes and " +
                              std::to_string(ncount) + " counters; the static scratch array holds " +
                              std::to_string(NOALLOC_WORKSPACE_BYTES) + " bytes and " + std::to_string(NOALLOC_COUNTERS) + " counters");
          unsigned char *base = noalloc_scratch();
          p.workspace = reinterpret_cast<float *>(base);
          p.counters = reinterpret_cast<int *>(base + NOALLOC_WORKSPACE_BYTES);
          // every call on this GPU shares the array: the counters start at zero whatever the last call left there
          // (a fill kernel rather than hipMemsetAsync, so that the call may be captured into a graph)
          if (ncount) {
            hipLaunchKernelGGL(clear_ints_kernel, dim3((unsigned)((ncount + 255) / 256)), dim3(256), 0, s, p.counters, (int)ncount);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return fail(TTS_HIP_ERROR, std::string("clearing the split-K counters: ") + hipGetErrorString(e));
          }
        } else if (p.split > 1 && !tiled) {
          std::lock_guard<std::mutex> lock(plan->mu);
          if (const tts_plan::SplitK *sk = plan->room(s, gemm_w8a16_workspace_bytes(p), gemm_w8a16_counters(p))) {
            p.workspace = sk->workspace;
            p.counters = sk->counters;
          } else {
            p.split = 1;
          }
        }
        p.widened = nullptr;
        if (!no_alloc) {  // (the call that may not allocate stays on the decode kernels, a launch per 32 rows)
          const size_t need = gemm_w8a16_widened_bytes(p);
          if (need) {
            std::lock_guard<std::mutex> lock(plan->mu);
            if (const tts_plan::SplitK *sk = plan->room(s, 0, 0, need)) p.widened = sk->widened;
          }
        }
        p.partial = nullptr;
        if (const size_t need = gemm_w8a16_tile_bytes(p)) {
          if (!no_alloc && !is_capturing(s)) {
            std::lock_guard<std::mutex> lock(plan->mu);
            if (const tts_plan::SplitK *sk = plan->room(s, need, 0)) p.partial = sk->workspace;
          } else if (no_alloc && need <= NOALLOC_WORKSPACE_BYTES) {
            p.partial = reinterpret_cast<float *>(noalloc_scratch());
          }
        }
        err = launch_gemm_w8a16(p, s, &kname);
        break;
      }
    }
    plan->last_kernel = kname;
    plan->last_slices = slices;
    plan->last_meet = meet;
    if (err != hipSuccess) return fail(TTS_HIP_ERROR, std::string("kernel launch failed: ") + hipGetErrorString(err));
    return TTS_OK;
  });
}

}  // namespace

extern "C" {

tts_status tts_launch(tts_plan *plan, int gx, int gy, int gz, void *stream, const tts_arg *args, int n) {
  return launch_impl(plan, gx, gy, gz, stream, args, n, false);
}

tts_status tts_launch_noalloc(tts_plan *plan, int gx, int gy, int gz, void *stream, const tts_arg *args, int n) {
  return launch_impl(plan, gx, gy, gz, stream, args, n, true);
}

}  // extern "C"
