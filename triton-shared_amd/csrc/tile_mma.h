// Matrix programs: the generic family's form for programs built around 16-bit matrix products (a flash-attention
// forward, its backward passes, a product with a chain of products behind it).  Included by tile_codegen.cpp, whose Gen
// prints index expressions, scalars and elementwise ops.
//
// Layout.  Every block of the program has BM rows, and a wavefront owns whole rows: 32 R of them (R = 1 throughout), row 32 rb + lane % 32
// in row block rb, both half wavefronts holding half of the row's columns each.  Products are computed transposed --
// result^T = b^T a^T on v_mfma_f32_32x32x16, so that the instruction's columns (lane % 32) are the block's rows -- and a
// lane then holds, of every 32 columns, columns 8 g + 4 (lane / 32) + {0..3}, g = 0..3.
//   * Reductions along the columns are folds of a lane's own registers and one exchange between the half wavefronts;
//     their results (and the carried vectors of an online softmax) are one register per row, in the lane that needs it.
//   * A block computed from one product and multiplied in the next needs no move at all: the registers 8 s .. 8 s + 7 of a
//     lane are, narrowed to 16 bits, its operand of the instruction for the 16 values of k that those registers hold.  The
//     order of k inside an instruction is free as long as both operands agree, so the other operand is read in that order.
//   * Only the right operands (a loaded block or its transpose) go through LDS: `global_load_lds_dwordx4`, two buffers
//     per load inside a loop, the next iteration's blocks in flight while the current one's are multiplied, one barrier
//     per iteration.  An operand whose k is contiguous in memory is read with 16-byte (or two 8-byte) LDS reads, any other
//     through `ds_read_b64_tr_b16`; the 16-byte chunks of a row are permuted so that neither form meets a bank conflict.
//     Blocks that stick out of their tensor or are not 16-byte aligned are staged through registers instead.
// What the ordinary form of the family spends its time on -- operands, products and every reduced row going through LDS
// element by element between some twenty barriers per iteration -- does not exist here: causal attention of 32 heads x
// 4096 x 128 in bf16 (64 x 64 blocks) 12.4 ms -> 170 us, 810 TFLOP/s; 32 x 4096 x 64 in fp16, no mask, 2.7 ms -> 205 us.
// What bounds it is the chain of an iteration, of which a SIMD holds two at most: the copies' way to LDS (a quarter of it while every
// wavefront sent its copies at once: with the next blocks' copies among the first product's instructions, fragments read four
// instructions ahead, the loop's tests in 32 bits and the row sums among the second product's instructions, 8 heads x 4096 x 128
// causal, a workgroup per CU, 120.7 -> 88.9 us, 3763 -> 3100 cycles an iteration), then the softmax between the two products.
//
// Programs of a grid axis on which no staged block depends (the query blocks of one head) share a workgroup, and with it
// the staged blocks: four wavefronts, each program taking BM / (32 R) of them.
struct MmaGen : Gen {
  enum Role { TILE = 1, ROW = 2, COL = 4, FRAG = 8, LDS = 16 };
  static constexpr int WAVES = 4;
  int64_t BM = 0;
  int R = 1, wpp = 1, G = 1, axis = -1;
  bool fast_exp = false;
  std::map<int, int> roles;             // value id -> roles it is needed in
  std::map<int, std::string> tile_of, row_of, col_of;  // materialised values
  std::map<int, std::string> factor_of;  // tiles held without a factor (a positive scalar) that their value has: see emit_scaled
  struct Image {
    int load = -1;
    int outer = 0, inner = 0;           // dimensions of the load: rows of the LDS image, and the dimension contiguous in memory
    int64_t rows = 0, cols = 0;
    int row_bytes = 0, chunks = 0;
    bool transposing = false;           // read through ds_read_b64_tr_b16 (the image's rows are k)
    int loop = -1;                      // staged per iteration of this loop (two buffers), or once (-1)
    int64_t offset = 0;                 // in the LDS array
    int64_t bytes() const { return rows * row_bytes; }
  };
  std::map<int, Image> images;          // load value id -> its image
  const SOp *meeting = nullptr;         // the loop that may run in slices: see softmax_loop
  size_t maximum_slot = 0;              // its carried row maximum
  std::string meeting_exp;              // and the exponential that rescales what it carries: math.exp or math.exp2
  int64_t lds_bytes = 0;
  int cur_loop = -1;

  explicit MmaGen(const Program &p) : Gen(p) {}
  [[noreturn]] static void decline(const std::string &why) { throw Unsupported("matrix program: " + why); }

  // ---- analysis -------------------------------------------------------------
  bool is_tile(const Value &v) const { return v.shape.size() == 2 && v.shape[0] == BM && v.shape[1] > 1; }
  const SOp *def_of(int v) const {
    auto d = def.find(v);
    return d == def.end() ? nullptr : d->second;
  }
  std::map<int, std::pair<const SOp *, size_t>> carried;  // a loop's region value or result -> (loop, slot)
  void collect(const std::vector<SOp> &ops, int loop) {
    for (const SOp &s : ops) {
      if (s.result >= 0) def[s.result] = &s;
      switch (s.kind) {
        case SK::Load: case SK::Store: case SK::Map: case SK::Splat: case SK::Const: case SK::Iota: case SK::FromIndex: case SK::ScalarArg:
        case SK::ExpandDims: case SK::Broadcast: break;
        case SK::Reduce:
          if (s.name == "region" || s.operands.size() != 1 || s.axis != 1) decline("a reduction other than one op along the columns");
          break;
        case SK::Dot:
          if (BM == 0) BM = val(s.result).shape.at(0);
          if (val(s.result).shape.at(0) != BM) decline("products with different numbers of rows");
          dots.push_back({&s, loop});
          break;
        case SK::For:
          if (loop >= 0) decline("nested loops");
          for (size_t q = 0; q < s.tile_args.size(); q++) {
            carried[s.tile_args[q]] = {&s, q};
            if (s.results[q] >= 0) carried[s.results[q]] = {&s, q};
          }
          collect(s.body, s.loop);
          break;
        default: decline("an op this form does not take");
      }
      if ((s.kind == SK::Load || s.kind == SK::Store) && (s.acc.gather >= 0 || s.acc.mask_value >= 0 || s.acc.other_value >= 0)) decline("an unstructured access");
    }
  }
  std::vector<std::pair<const SOp *, int>> dots;

  void need(int v, int role) {
    if (val(v).shape.empty()) return;  // scalars are written out where they are used
    int &r = roles[v];
    if (r & role) return;
    r |= role;
    auto c = carried.find(v);
    if (c != carried.end()) {
      const SOp &L = *c->second.first;
      const size_t q = c->second.second;
      if (role == COL) decline("a carried vector along the columns");
      need(L.tile_args[q], role);
      if (L.results[q] >= 0) need(L.results[q], role);
      need(L.tile_inits[q], role);
      need(L.tile_yields[q], role);
      return;
    }
    const SOp *d = def_of(v);
    if (!d) decline("a value without a definition");
    const Value &V = val(v);
    if (role == TILE && !is_tile(V)) decline("a block of another number of rows");
    if (role == TILE && V.shape[1] % 32) decline("a block of " + std::to_string(V.shape[1]) + " columns");  // (lanes hold columns in groups of 32)
    if (V.dtype == "f64" || (role == TILE && !scalar_ok(V.dtype))) decline("blocks of " + V.dtype);  // (rows are held in fp32 registers too)
    auto role_of = [&](int o) -> int {  // of an operand with its own shape, inside a rank-2 result
      const Value &O = val(o);
      if (O.shape.size() != 2) decline("an operand of rank " + std::to_string(O.shape.size()));
      if (is_tile(O)) return TILE;
      if (O.shape[0] == BM && O.shape[1] == 1) return ROW;
      if (O.shape[0] == 1 && O.shape[1] > 1) return COL;
      if (O.shape[0] == 1 && O.shape[1] == 1) return ROW;
      decline("a block of another number of rows");
    };
    if (V.shape.size() > 2) decline("blocks of rank above 2");
    if (role == ROW && V.shape[0] != BM && !(V.shape[0] == 1)) decline("a vector of another number of rows");
    switch (d->kind) {
      case SK::Const: case SK::Iota: break;
      case SK::Splat: break;
      case SK::Map: {
        static const char *shuffles[] = {"tt.trans", "tt.cat", "tt.join", "tt.split", "tt.reshape", "tt.unsplat"};
        for (const char *n : shuffles)
          if (d->name.rfind(n, 0) == 0) decline("an index shuffle");
        for (int o : d->operands) need(o, role);
        break;
      }
      case SK::ExpandDims: need(d->operands.at(0), d->axis == 1 ? ROW : COL); break;
      case SK::Broadcast: need(d->operands.at(0), val(d->operands[0]).shape.size() == 2 ? role_of(d->operands[0]) : role); break;
      case SK::Reduce:
        if (role != ROW) decline("a reduction's result along the columns");
        if (V.dtype != "f32") decline("a reduction of " + V.dtype + " values");
        need(d->operands[0], TILE);
        break;
      case SK::Load:
        for (int m : d->acc.mods)
          if (m >= 0) decline("a wrapped load read element by element");
        break;
      case SK::Dot: break;  // (its operands are looked at once, in analyse())
      default: decline("a value this form does not take");
    }
  }

  bool expr_uses_pid(int e, int ax, int depth = 0) const {
    if (e < 0) return false;
    if (depth > 64) return true;
    const Expr &x = P.pool.at(e);
    switch (x.k) {
      case EK::Const: case EK::Arg: case EK::NProg: return false;
      case EK::Pid: return x.a == ax;
      case EK::IV: {
        const SOp *L = loop_by_id(x.a);
        return !L || expr_uses_pid(L->lb, ax, depth + 1) || expr_uses_pid(L->step, ax, depth + 1);
      }
      case EK::Iter: {
        const SOp *L = loop_by_id(x.a);
        if (!L || x.b >= (int)L->int_iters.size()) return true;
        const IntIter &it = L->int_iters[x.b];
        if (expr_uses_pid(it.init, ax, depth + 1)) return true;
        // (the step's own mention of this iterator adds nothing new; any other leaf of it counts)
        return next_uses_pid(it.next, ax, x.a, depth + 1);
      }
      case EK::Result: case EK::Data: return true;
      case EK::Sext: case EK::Trunc: return expr_uses_pid(x.a, ax, depth + 1);
      default:
        for (int o : {x.a, x.b, x.c, x.d})
          if (expr_uses_pid(o, ax, depth + 1)) return true;
        return false;
    }
  }
  bool next_uses_pid(int e, int ax, int loop, int depth) const {
    if (e < 0) return false;
    if (depth > 64) return true;
    const Expr &x = P.pool.at(e);
    if (x.k == EK::Iter && x.a == loop) return false;
    if (x.k == EK::Const || x.k == EK::Arg || x.k == EK::NProg || x.k == EK::Pid || x.k == EK::IV || x.k == EK::Iter || x.k == EK::Result || x.k == EK::Data)
      return expr_uses_pid(e, ax, depth);
    for (int o : {x.a, x.b, x.c, x.d})
      if (next_uses_pid(o, ax, loop, depth + 1)) return true;
    return false;
  }
  const SOp *loop_by_id(int id) const {
    for (const SOp &s : P.body)
      if (s.kind == SK::For && s.loop == id) return &s;
    return nullptr;
  }
  static bool mentions(const ExprPool &X, int e, EK k) { return e >= 0 && X.depends_on(e, k); }

  const SOp *right_load(int b) const {  // the load behind a product's right operand (directly, or its transpose)
    const SOp *d = def_of(b);
    if (d && d->kind == SK::Map && d->name == "tt.trans") d = def_of(d->operands[0]);
    return d && d->kind == SK::Load ? d : nullptr;
  }

  void analyse() {
    collect(P.body, -1);
    if (dots.empty()) decline("no matrix product");
    if (BM % 32 || BM > 128) decline("blocks of " + std::to_string(BM) + " rows");
    if (128 % BM) decline("blocks of " + std::to_string(BM) + " rows");
    std::set<int> read, written;
    std::function<void(const std::vector<SOp> &)> bases = [&](const std::vector<SOp> &ops) {
      for (const SOp &s : ops) {
        if (s.kind == SK::Load) read.insert(s.acc.base_arg);
        if (s.kind == SK::Store) written.insert(s.acc.base_arg);
        bases(s.body);
      }
    };
    bases(P.body);
    for (int b : written)
      if (read.count(b)) decline("an argument that is both read and stored to");
    std::map<int, int> where;  // load -> the loop it stands in
    std::function<void(const std::vector<SOp> &, int)> places = [&](const std::vector<SOp> &ops, int loop) {
      for (const SOp &s : ops) {
        if (s.kind == SK::Load) where[s.result] = loop;
        if (s.kind == SK::For) places(s.body, s.loop);
      }
    };
    places(P.body, -1);
    for (auto &dl : dots) {
      const SOp &s = *dl.first;
      const Value &A = val(s.operands.at(0)), &B = val(s.operands.at(1)), &C = val(s.result);
      if (!is16(A.dtype) || A.dtype != B.dtype || C.dtype != "f32") decline("a product of other types than 16-bit floats into fp32");
      const int64_t K = A.shape[1], N = C.shape[1];
      if (N % 32 || N > 256 || K % 32 || K > 256) decline("a product of this shape");
      if (!is_tile(C)) decline("a product of this shape");
      need(s.result, TILE);
      need(s.operands.at(2), TILE);
      // left: a load in operand layout, or a block of 16-bit values computed from an fp32 one
      const SOp *a = def_of(s.operands[0]);
      if (a && a->kind == SK::Load) {
        int64_t st = 0;
        if (a->acc.sizes.size() != 2 || !P.pool.is_const(a->acc.strides[1], &st) || st != 1) decline("a left operand whose rows are not contiguous");
        if (a->acc.has_other && (a->acc.other_f != 0 || a->acc.other_i != 0)) decline("padding other than zero");
        for (int m : a->acc.mods)
          if (m >= 0) decline("a wrapped left operand");
        roles[s.operands[0]] |= FRAG;
      } else {
        if (!a || a->kind != SK::Map || a->name != "arith.truncf" || val(a->operands[0]).dtype != "f32") decline("a left operand that is not a narrowed block");
        need(s.operands[0], TILE);
      }
      const SOp *l = right_load(s.operands[1]);
      if (!l) decline("a right operand that is not loaded");
      if (images.count(l->result)) decline("a block used as the right operand of two products");
      const bool turned = def_of(s.operands[1])->kind == SK::Map;
      Image im;
      im.load = l->result;
      const Access &acc = l->acc;
      if (acc.sizes.size() != 2) decline("a right operand of this rank");
      if (acc.has_other && (acc.other_f != 0 || acc.other_i != 0)) decline("padding other than zero");
      for (int m : acc.mods)
        if (m >= 0) decline("a wrapped right operand");
      int64_t st = 0;
      if (P.pool.is_const(acc.strides[1], &st) && st == 1) im.inner = 1;
      else if (P.pool.is_const(acc.strides[0], &st) && st == 1) im.inner = 0;
      else decline("a right operand that is contiguous along neither dimension");
      im.outer = 1 - im.inner;
      im.rows = acc.sizes[im.outer];
      im.cols = acc.sizes[im.inner];
      const int k_dim = turned ? 1 : 0;  // the load's dimension that the product contracts
      im.transposing = im.inner != k_dim;
      im.row_bytes = (int)im.cols * 2;
      im.chunks = im.row_bytes / 16;
      if (im.cols < 32 || im.cols > 256 || (im.cols & (im.cols - 1)) || im.rows < 32 || im.rows > 256) decline("a right operand of this shape");
      im.loop = where.at(l->result);
      if (im.loop != dl.second) decline("a right operand loaded outside the loop that multiplies it");
      im.offset = lds_bytes;
      lds_bytes += im.bytes() * (im.loop >= 0 ? 2 : 1);
      images[im.load] = im;
    }
    if (lds_bytes > 128 * 1024) decline("right operands of " + std::to_string(lds_bytes) + " bytes in LDS");
    for (const SOp &s : P.body)
      if (s.kind == SK::Store) store_roles(s);
      else if (s.kind == SK::For)
        for (const SOp &t : s.body)
          if (t.kind == SK::Store) store_roles(t);
    // loads whose values are needed both as an operand and element by element would need both layouts
    for (auto &im : images)
      if (roles.count(im.first) && roles[im.first]) decline("a right operand that is also read element by element");
    for (auto &rv : roles)
      if ((rv.second & FRAG) && (rv.second & ~FRAG)) decline("a left operand that is also read element by element");
    wpp = (int)(BM / (32 * R));
    G = 1;
    axis = -1;
    // (a loop whose bounds another loop leaves behind: one program's value says nothing about another's, so none is shared)
    bool known = true;
    for (const SOp &s : P.body)
      if (s.kind == SK::For)
        for (int e : {s.lb, s.ub, s.step}) {
          if (mentions(P.pool, e, EK::Data)) decline("a loop bound that is data");
          known = known && !mentions(P.pool, e, EK::Result);
        }
    for (int ax = 0; ax < 3 && wpp < WAVES && axis < 0 && known; ax++) {
      bool free = true;
      for (auto &im : images) {
        const Access &a = def_of(im.first)->acc;
        for (const auto *v : {&a.offsets, &a.strides, &a.dims})
          for (int e : *v) free = free && !expr_uses_pid(e, ax);
        const SOp *L = im.second.loop >= 0 ? loop_by_id(im.second.loop) : nullptr;
        if (im.second.loop >= 0) free = free && L && !expr_uses_pid(L->lb, ax) && !expr_uses_pid(L->step, ax);
      }
      if (free) axis = ax;
    }
    if (axis >= 0) G = WAVES / wpp;
    // (the only loop, with nothing stored before it: workgroups whose slice is empty leave)
    size_t loops = 0;
    bool stored = false;
    for (const SOp &s : P.body) {
      if (s.kind == SK::For && ++loops == 1 && !stored && softmax_loop(s)) meeting = &s;
      stored = stored || s.kind == SK::Store;
    }
    if (loops > 1) meeting = nullptr;
    fast_exp = true;
    std::function<void(const std::vector<SOp> &)> outs = [&](const std::vector<SOp> &ops) {
      for (const SOp &s : ops) {
        if (s.kind == SK::Store && !is16(s.acc.elem)) fast_exp = false;
        outs(s.body);
      }
    };
    outs(P.body);
    for (const SOp &s : P.body)
      if (s.kind == SK::For)
        for (const IntIter &it : s.int_iters)
          if (mentions(P.pool, it.init, EK::Data) || mentions(P.pool, it.next, EK::Data)) decline("index state that is data");
  }
  static bool scalar_ok(const std::string &t) { return t == "f32" || t == "f16" || t == "bf16" || t == "i1" || t == "i32" || t == "i64"; }
  void store_roles(const SOp &s) {
    const Value &V = val(s.operands.at(0));
    for (int m : s.acc.mods)
      if (m >= 0) decline("a wrapped store");
    if (s.acc.sizes.size() == 2 && is_tile(V)) need(s.operands[0], TILE);
    else if (s.acc.sizes.size() == 1 && V.shape.size() == 1 && V.shape[0] == BM) need(s.operands[0], ROW);
    else decline("a store of this shape");
  }

  // ---- slices -------------------------------------------------------------------
  // An online softmax: a loop that carries a row maximum m' = max(m, max over x) and rows and blocks v' = v * exp(m - m') + s
  // where s is a row sum of, or a product with, p = exp(x - m') (narrowed or not) and x knows nothing of what is carried.
  // What such a loop has over some of its iterations is a state (m, v ...) like that of the others, and two states are one after
  // scaling both to the larger maximum: a program's iterations may be dealt to several workgroups (slices_meet).
  const SOp *seen_through(int v) const {  // the op behind broadcasts and added dimensions
    const SOp *d = def_of(v);
    while (d && (d->kind == SK::Broadcast || d->kind == SK::ExpandDims)) d = def_of(d->operands.at(0));
    return d;
  }
  int behind(int v) const {
    const SOp *d = def_of(v);
    while (d && (d->kind == SK::Broadcast || d->kind == SK::ExpandDims)) {
      v = d->operands.at(0);
      d = def_of(v);
    }
    return v;
  }
  bool reaches_carried(int v, const SOp &L, int depth = 0) const {
    if (depth > 64) return true;
    for (int a : L.tile_args)
      if (a == v) return true;
    const SOp *d = def_of(v);
    if (!d) return true;
    for (int o : d->operands)
      if (reaches_carried(o, L, depth + 1)) return true;
    return false;
  }
  bool softmax_loop(const SOp &L) {
    int64_t step = 0;
    if (!L.int_iters.empty() || !P.pool.is_const(L.step, &step) || step <= 0 || mentions(P.pool, L.lb, EK::Result) || mentions(P.pool, L.ub, EK::Result)) return false;
    for (const SOp &o : L.body)
      if (o.kind == SK::Store || o.kind == SK::For) return false;
    auto is_max = [](const std::string &n) { return n == "arith.maxnumf" || n == "arith.maximumf"; };
    for (size_t q = 0; q < L.tile_args.size(); q++) {
      const int m = L.tile_args[q], next = L.tile_yields[q];
      const SOp *y = def_of(next);
      if (val(m).shape.size() != 1 || val(m).dtype != "f32" || !y || y->kind != SK::Map || !is_max(y->name)) continue;
      const int other = y->operands.at(0) == m ? y->operands.at(1) : y->operands.at(1) == m ? y->operands.at(0) : -1;
      const SOp *r = other >= 0 ? def_of(other) : nullptr;
      if (!r || r->kind != SK::Reduce || r->name != y->name || reaches_carried(r->operands.at(0), L)) return false;
      std::string fn;
      auto exponential = [&](int v) -> const SOp * {  // exp(a - m'): the subtraction
        const SOp *e = seen_through(v);
        if (!e || e->kind != SK::Map || (e->name != "math.exp" && e->name != "math.exp2") || (!fn.empty() && e->name != fn)) return nullptr;
        const SOp *d = def_of(e->operands.at(0));
        if (!d || d->kind != SK::Map || d->name != "arith.subf" || behind(d->operands.at(1)) != next) return nullptr;
        fn = e->name;
        return d;
      };
      auto rescaled = [&](int v, int arg) {  // arg * exp(m - m')
        const SOp *d = def_of(v);
        if (!d || d->kind != SK::Map || d->name != "arith.mulf") return false;
        const int by = d->operands.at(0) == arg ? d->operands.at(1) : d->operands.at(1) == arg ? d->operands.at(0) : -1;
        const SOp *sub = by >= 0 ? exponential(by) : nullptr;
        return sub && behind(sub->operands.at(0)) == m;
      };
      auto probabilities = [&](int v) {  // exp(x - m'), narrowed or not
        const SOp *d = def_of(v);
        while (d && d->kind == SK::Map && (d->name == "arith.truncf" || d->name == "arith.extf")) d = def_of(v = d->operands.at(0));
        const SOp *sub = d && d->kind == SK::Map ? exponential(v) : nullptr;
        return sub && !reaches_carried(sub->operands.at(0), L);
      };
      auto product = [&](int v, int *into) {  // p . b + into
        const SOp *d = def_of(v);
        if (!d || d->kind != SK::Dot || !probabilities(d->operands.at(0)) || reaches_carried(d->operands.at(1), L)) return false;
        *into = d->operands.at(2);
        return true;
      };
      auto summand = [&](int v) {
        const SOp *d = def_of(v);
        int into = -1;
        if (d && d->kind == SK::Reduce) return d->name == "arith.addf" && probabilities(d->operands.at(0));
        const SOp *c = product(v, &into) ? def_of(into) : nullptr;
        return c && c->kind == SK::Const && c->fval == 0;
      };
      auto only_read_by = [&](int v, const std::set<const SOp *> &ops) {
        auto u = users.find(v);
        for (const SOp *o : u == users.end() ? std::vector<const SOp *>() : u->second)
          if (!ops.count(o)) return false;
        return true;
      };
      std::set<const SOp *> of_m = {y};
      for (size_t k = 0; k < L.tile_args.size(); k++) {
        if (k == q) continue;
        const int v = L.tile_args[k], w = L.tile_yields[k];
        const SOp *d = def_of(w);
        if (val(v).dtype != "f32" || !d) return false;
        int into = -1, kept = -1;
        if (d->kind == SK::Map && d->name == "arith.addf") {
          for (int t = 0; t < 2; t++)
            if (rescaled(d->operands.at(t), v) && summand(d->operands.at(1 - t))) kept = d->operands.at(t);
        } else if (product(w, &into) && rescaled(into, v)) {
          kept = into;
        }
        if (kept < 0 || !only_read_by(v, {def_of(kept)})) return false;
        const SOp *mul = def_of(kept);
        of_m.insert(def_of(seen_through(mul->operands.at(0) == v ? mul->operands.at(1) : mul->operands.at(0))->operands.at(0)));
      }
      // the maximum is read by itself and by its factors alone, the new one by exponentials alone
      if (of_m.size() < 2 || !only_read_by(m, of_m)) return false;
      std::function<bool(int)> fine = [&](int v) {
        auto u = users.find(v);
        for (const SOp *o : u == users.end() ? std::vector<const SOp *>() : u->second) {
          if (o == &L) continue;  // (the yield)
          if ((o->kind == SK::Broadcast || o->kind == SK::ExpandDims) && fine(o->result)) continue;
          if (o->kind != SK::Map || o->name != "arith.subf" || o->operands.at(1) != v) return false;
          for (const SOp *e : users.count(o->result) ? users.at(o->result) : std::vector<const SOp *>())
            if (e->kind != SK::Map || e->name != fn) return false;
        }
        return true;
      };
      if (!fine(next)) return false;
      maximum_slot = q;
      meeting_exp = fn;
      return true;
    }
    return false;
  }
  // floats of a lane's state: the carried rows, then the carried blocks
  int state_floats() const {
    int n = 0;
    for (int a : meeting->tile_args) n += R * (val(a).shape.size() == 1 ? 1 : NB(a) * 16);
    return (n + 3) / 4 * 4;
  }
  // The slices' states become one: every workgroup leaves its own in `partial` as its lanes hold it (written through, complete
  // before its arrival is counted), and the one that arrives last scales all of them to the largest maximum, adds them up in slice
  // order -- the result does not depend on who that is -- and goes on with the program.  Nobody waits for anybody.
  void slices_meet() {
    std::vector<std::string> regs;  // the maximum first
    auto add = [&](size_t q) {
      const int a = meeting->tile_args[q];
      for (int rb = 0; rb < R; rb++) {
        if (val(a).shape.size() == 1) regs.push_back(row_of.at(a) + "[" + std::to_string(rb) + "]");
        else
          for (int nb = 0; nb < NB(a); nb++)
            for (int i = 0; i < 16; i++) regs.push_back(tile_of.at(a) + "[" + std::to_string(rb) + "][" + std::to_string(nb) + "][" + std::to_string(i) + "]");
      }
    };
    add(maximum_slot);
    for (size_t q = 0; q < meeting->tile_args.size(); q++)
      if (q != maximum_slot) add(q);
    const int n = state_floats();
    const std::string N = std::to_string(n), Q = std::to_string(n / 4);
    line("if (parts > 1) {");
    indent++;
    line("__shared__ int arrived;");
    // this wavefront's place in slice h: 16 bytes of every lane, Q times
    line("const long long stride = (long long)(others * groups) * " + std::to_string(WAVES * 64 * n) + ";");
    line("float *const slot = partial + ((long long)wg * " + std::to_string(WAVES) + " + wave) * " + std::to_string(64 * n) + ";");
    line("{");
    indent++;
    line("const float st[" + N + "] = {");
    indent++;
    for (size_t r = 0; r < regs.size(); r += 8) {
      std::string t;
      for (size_t k = r; k < std::min(r + 8, regs.size()); k++) t += regs[k] + ", ";
      line(t);
    }
    indent--;
    line("};");
    line("const shared_memory_t at = shared_memory(slot + slice * stride);");
    line("#pragma unroll");
    line("for (int r = 0; r < " + Q + "; r++) put_through(at, r * 1024 + lane * 16, (f32x4_t){st[4 * r], st[4 * r + 1], st[4 * r + 2], st[4 * r + 3]});");
    indent--;
    line("}");
    line("asm volatile(\"s_waitcnt vmcnt(0)\" ::: \"memory\");");
    line("__syncthreads();");
    line("if (threadIdx.x == 0) {");
    line("  arrived = __hip_atomic_fetch_add(&counters[32 * wg], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);");
    line("  if (arrived == parts - 1) __hip_atomic_store(&counters[32 * wg], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch");
    line("}");
    line("__syncthreads();");
    line("if (arrived != parts - 1) return;");
    const std::string mx = row_of.at(meeting->tile_args[maximum_slot]) + "[0]";  // (R = 1)
    SOp op = *def_of(meeting->tile_yields[maximum_slot]);
    // (a load takes one or two microseconds, what the slices wrote sits behind other XCDs: all the maxima are loaded together, and
    // each slice's state while the one before it is added)
    line("float top = 0.f;");
    line("{");
    line("  float tops[16];");
    line("  #pragma unroll");
    line("  for (int h = 0; h < 16; h++) tops[h] = take_through(shared_memory(slot + (h < parts ? h : 0) * stride), lane * 16)[0];");
    line("  top = tops[0];");
    line("  #pragma unroll");
    line("  for (int h = 1; h < 16; h++) top = " + map_text_f32(op, "top", "tops[h]") + ";");
    line("}");
    line("float sum[" + N + "];");
    line("#pragma unroll");
    line("for (int r = 0; r < " + N + "; r++) sum[r] = 0.f;");
    line("f32x4_t got[" + Q + "], next[" + Q + "];");
    line("#pragma unroll");
    line("for (int r = 0; r < " + Q + "; r++) got[r] = take_through(shared_memory(slot), r * 1024 + lane * 16);");
    line("for (int h = 0; h < parts; h++) {");
    indent++;
    line("const shared_memory_t at = shared_memory(slot + (h + 1 < parts ? h + 1 : h) * stride);");
    line("#pragma unroll");
    line("for (int r = 0; r < " + Q + "; r++) next[r] = take_through(at, r * 1024 + lane * 16);");
    const std::string d = "(got[0][0] - top)";
    // (equal maxima are scaled by one, also where both are infinite)
    line("const float by = got[0][0] == top ? 1.0f : " + (fast_exp ? "hardware_exp2(" + d + (meeting_exp == "math.exp" ? " * TTS_LOG2E)" : ")") : (meeting_exp == "math.exp" ? "expf(" : "exp2f(") + d + ")") + ";");
    line("#pragma unroll");
    line("for (int r = 0; r < " + N + "; r++) sum[r] += got[r >> 2][r & 3] * by;");
    line("#pragma unroll");
    line("for (int r = 0; r < " + Q + "; r++) got[r] = next[r];");
    indent--;
    line("}");
    line(mx + " = top;");
    for (size_t r = 1; r < regs.size(); r++) line(regs[r] + " = sum[" + std::to_string(r) + "];");
    indent--;
    line("}");
  }

  // ---- elements ---------------------------------------------------------------
  // The element a lane holds is named by rb (row block), nb (block of 32 columns) and i (0..15) in the code around it.
  const char *ROWX = "(wrow + 32 * rb + l32)";
  const char *COLX = "(32 * nb + 8 * (i >> 2) + h4 + (i & 3))";
  std::string el(int v, int role) {
    const Value &V = val(v);
    if (V.shape.empty()) return at(v, "0", "0");
    if (role == TILE && tile_of.count(v)) {
      if (is16(V.dtype)) return std::string(V.dtype == "f16" ? "up_f16" : "up_bf16") + "((unsigned short)(" + tile_of[v] + "[rb][nb][i >> 1] >> (16 * (i & 1))))";
      const std::string x = tile_of[v] + "[rb][nb][i]";
      return factor_of.count(v) ? "(" + x + " * " + factor_of[v] + ")" : x;
    }
    if (role == ROW && row_of.count(v)) return row_of[v] + "[rb]";
    if (role == COL && col_of.count(v)) return col_of[v] + "[nb][i]";
    const SOp *d = def_of(v);
    if (!d) decline("a value without an element form");
    switch (d->kind) {
      case SK::Const: case SK::FromIndex: case SK::ScalarArg: return at(v, "0", "0");
      case SK::Splat: return at(d->operands[0], "0", "0");
      case SK::Iota: return "(int)(" + std::to_string(d->ival) + " + " + (V.shape[0] == 1 ? "0" : role == ROW ? ROWX : COLX) + ")";  // (one element: the same for every row)
      case SK::ExpandDims: return el(d->operands[0], d->axis == 1 ? ROW : COL);
      case SK::Broadcast: {
        const Value &O = val(d->operands[0]);
        if (O.shape.size() != 2) return el(d->operands[0], role);
        return el(d->operands[0], is_tile(O) ? TILE : O.shape[1] == 1 ? ROW : COL);
      }
      case SK::Map: {
        std::vector<std::string> a;
        for (int o : d->operands) a.push_back(el(o, role));
        return "(" + map_text(*d, a) + ")";
      }
      default: decline("a value without an element form");
    }
  }
  // The exponential of a difference against a maximum that its own minuend is one of (a softmax's scores against their row's
  // maximum, the old maximum against the new one) is at most 1, and what counts is its error next to the largest of the row,
  // which is 1: v_exp_f32 of the difference times log2 e is off by |d| 2^-24 of e^d at most, 0.4 2^-24 where that is largest, and
  // flushes what is below 2^-126.  That is how programs that only store 16-bit values compute those; every other exponential is
  // the library's, to an ulp over the whole range.
  bool is_maximum_over(int m, int x, int depth = 0) const {
    const SOp *d = def_of(m);
    if (!d || depth > 16) return m == x;
    if (m == x) return true;
    const bool max = d->name == "arith.maxnumf" || d->name == "arith.maximumf";
    if (d->kind == SK::Reduce) return max && d->operands.at(0) == x;
    if (d->kind == SK::Broadcast || d->kind == SK::ExpandDims) return is_maximum_over(d->operands.at(0), x, depth + 1);
    return d->kind == SK::Map && max && (is_maximum_over(d->operands.at(0), x, depth + 1) || is_maximum_over(d->operands.at(1), x, depth + 1));
  }
  // a product of a block (or row) with a scalar that is the same everywhere: the other factor and the scalar's value id
  bool scaled(int v, int *factor, int *scalar) const {
    const SOp *d = def_of(v);
    if (!d || d->kind != SK::Map || d->name != "arith.mulf" || val(v).dtype != "f32") return false;
    for (int q = 0; q < 2; q++) {
      const SOp *o = def_of(d->operands[q]);
      if (!o || o->kind != SK::Splat) continue;
      *scalar = o->operands.at(0);
      *factor = d->operands[1 - q];
      return true;
    }
    return false;
  }
  // is m a maximum of values one of which is `scalar` times a maximum over x?  (With scalar >= 0 that is one over scalar * x.)
  bool is_scaled_maximum_over(int m, int x, int scalar, int depth = 0) const {
    const SOp *d = def_of(m);
    if (!d || depth > 16) return false;
    int f = -1, s = -1;
    if (scaled(m, &f, &s) && s == scalar) return is_maximum_over(f, x);
    if (d->kind == SK::Broadcast || d->kind == SK::ExpandDims) return is_scaled_maximum_over(d->operands.at(0), x, scalar, depth + 1);
    const bool max = d->kind == SK::Map && (d->name == "arith.maxnumf" || d->name == "arith.maximumf");
    return max && (is_scaled_maximum_over(d->operands.at(0), x, scalar, depth + 1) || is_scaled_maximum_over(d->operands.at(1), x, scalar, depth + 1));
  }
  // The subtraction behind such an exponential; `*scalar`: it is one if this scalar is not negative (scores scaled after their
  // maximum was taken), which the kernel asks -- or -1.
  const SOp *difference_against_maximum(const SOp &s, int *scalar) const {
    *scalar = -1;
    if (!fast_exp || s.kind != SK::Map || (s.name != "math.exp" && s.name != "math.exp2") || val(s.result).dtype != "f32") return nullptr;
    const SOp *d = def_of(s.operands[0]);
    if (!d || d->kind != SK::Map || d->name != "arith.subf") return nullptr;
    if (is_maximum_over(d->operands[1], d->operands[0])) return d;
    int f = -1, by = -1;
    if (!scaled(d->operands[0], &f, &by) || !is_scaled_maximum_over(d->operands[1], f, by)) return nullptr;
    *scalar = by;
    return d;
  }
  std::string hardware_exp(const SOp &s, const std::string &x) const { return "__builtin_amdgcn_exp2f(" + x + (s.name == "math.exp" ? " * TTS_LOG2E)" : ")"); }
  std::string map_text(const SOp &s, const std::vector<std::string> &a) {
    int scalar = -1;
    return difference_against_maximum(s, &scalar) && scalar < 0 ? hardware_exp(s, a.at(0)) : map_expr(s, a);
  }
  // Scores that a positive scalar scales before such an exponential are held as the product left them (factor_of), and so are
  // they behind a select that puts -infinity in the place of some: the factor is in the exponential's fma, and a maximum
  // over them is scaled once it is taken (rounding keeps the order, so it is the same maximum).  A scalar outside of [2^-60,
  // 1] is multiplied in at once, and the factor is one: one above could take finite scores to infinity, whose difference is not a number, but
  // not in the fma.
  bool minus_infinity(int v) const {
    const SOp *d = def_of(v);
    while (d && (d->kind == SK::Splat || d->kind == SK::Broadcast)) d = def_of(d->operands.at(0));
    return d && d->kind == SK::Const && val(d->result).dtype == "f32" && d->fval == -__builtin_inf();
  }
  bool read_by_such_an_exponential(int v) const {
    auto u = users.find(v);
    if (u == users.end()) return false;
    int scalar = -1;
    for (const SOp *o : u->second) {
      if (o->name == "arith.subf" && o->operands.at(0) == v && folded_into_exp(*o)) {
        bool all = true;
        for (const SOp *e : users.at(o->result)) all = all && difference_against_maximum(*e, &scalar) && scalar < 0;
        if (all) return true;
      }
      if (o->name == "arith.select" && o->operands.at(1) == v && minus_infinity(o->operands.at(2)) && read_by_such_an_exponential(o->result)) return true;
    }
    return false;
  }
  bool emit_scaled(const SOp &s) {
    int x = -1, by = -1;
    if (!scaled(s.result, &x, &by) || !tile_of.count(x) || factor_of.count(x) || !read_by_such_an_exponential(s.result)) return false;
    const std::string n = declare_tile(s.result), f = "f" + std::to_string(s.result);
    line("const float s" + f + " = " + at(by, "0", "0") + ";");
    line("const bool fits_" + f + " = s" + f + " >= 0x1p-60f && s" + f + " <= 1.0f;");
    line("const float " + f + " = fits_" + f + " ? s" + f + " : 1.0f;");
    tile_loop(s.result, n + "[rb][nb][i] = " + el(x, TILE) + ";");
    line("if (!fits_" + f + ") {");
    indent++;
    tile_loop(s.result, n + "[rb][nb][i] *= s" + f + ";");
    indent--;
    line("}");
    tile_of[s.result] = n;
    factor_of[s.result] = f;
    return true;
  }
  // The same with the difference written where it is read.  It is taken before the factor log2 e, from scores that are held without
  // their factor as one fma, fma(x, factor, -m).  With both factors in the fma, exp2(fma(x, factor log2 e, -(m log2 e))), an instruction
  // less a score, m log2 e rounds by up to 2^-19 of a row's probabilities, by another amount in every block that raises the maximum: rms
  // error of the row sums against 64 bits, largest scores of 26, 6.7e-7 against 9.7e-8 here and with the scaled score rounded
  // first, of the results 2.2e-7 against 1.3e-7.
  bool emit_exp_of_difference(const SOp &s) {
    int scalar = -1;
    const SOp *d = difference_against_maximum(s, &scalar);
    if (!d) return false;
    const std::string n = declare_tile(s.result), m = el(d->operands[1], TILE);
    const std::string x = factor_of.count(d->operands[0]) ? "__builtin_fmaf(" + tile_of[d->operands[0]] + "[rb][nb][i], " + factor_of[d->operands[0]] + ", -(" + m + "))"
                                                          : "(" + el(d->operands[0], TILE) + " - " + m + ")";
    if (scalar >= 0) {
      line("if (" + at(scalar, "0", "0") + " >= 0.f) {");
      indent++;
    }
    tile_loop(s.result, n + "[rb][nb][i] = " + hardware_exp(s, x) + ";");
    if (scalar >= 0) {
      indent--;
      line("} else {");
      indent++;
      tile_loop(s.result, n + "[rb][nb][i] = " + map_expr(s, {x}) + ";");
      indent--;
      line("}");
    }
    tile_of[s.result] = n;
    return true;
  }
  bool folded_into_exp(const SOp &s) const {  // a difference that only such exponentials read is written there
    if (s.name != "arith.subf") return false;
    auto u = users.find(s.result);
    if (u == users.end()) return false;
    int scalar = -1;
    for (const SOp *o : u->second)
      if (!difference_against_maximum(*o, &scalar)) return false;
    return true;
  }

  // Lower and upper bound of an integer value over the rows of this wavefront and the columns of the block, as a scalar
  // expression and a constant beside it; conditions under which they hold (no 32-bit wrap) are added to `given`.
  struct Bound {
    std::string v;      // "": nothing but the constant
    int64_t c = 0;
    bool turns = false;  // v is one 32-bit value that changes from iteration to iteration
    bool mixed = false;  // v is a sum that holds such a value
    std::string text() const { return v.empty() ? std::to_string(c) + "LL" : "(" + v + " + " + std::to_string(c) + "LL)"; }
  };
  // a < b + slack, or something narrower.  A value that changes in the loop is compared in 32 bits with a bound that does not: one
  // scalar instruction and nothing else inside the loop.
  static std::string below(const Bound &a, const Bound &b, int64_t slack) {
    if (a.turns && !b.turns && !b.mixed) return "(int)" + a.v + " < sat32(" + (b.v.empty() ? "0LL" : b.v) + " + " + std::to_string(b.c + slack - a.c) + "LL)";
    if (b.turns && !a.turns && !a.mixed) return "(int)" + b.v + " > sat32(" + (a.v.empty() ? "0LL" : a.v) + " + " + std::to_string(a.c - slack - b.c) + "LL)";
    return a.text() + " < " + b.text() + " + " + std::to_string(slack) + "LL";
  }
  bool changes_in_a_loop(int v) const {  // may a scalar's value be another in the next iteration?
    const SOp *d = def_of(v);
    if (!d) return true;
    switch (d->kind) {
      case SK::Const: case SK::ScalarArg: return false;
      case SK::FromIndex: return mentions(P.pool, d->expr, EK::IV) || mentions(P.pool, d->expr, EK::Iter) || mentions(P.pool, d->expr, EK::Data);
      case SK::Map:
        for (int o : d->operands)
          if (changes_in_a_loop(o)) return true;
        return false;
      default: return true;
    }
  }
  bool bounds(int v, int role, Bound *lo, Bound *hi, std::string *given) {
    const Value &V = val(v);
    if (V.dtype != "i32" && V.dtype != "i64") return false;
    auto scalar = [&](int x) {
      *lo = Bound();
      lo->v = "(long long)" + at(x, "0", "0");
      const bool varies = changes_in_a_loop(x);
      lo->turns = varies && V.dtype == "i32";
      lo->mixed = varies && !lo->turns;
      *hi = *lo;
      return true;
    };
    if (V.shape.empty()) return scalar(v);
    const SOp *d = def_of(v);
    if (!d) return false;
    switch (d->kind) {
      case SK::Const: case SK::FromIndex: return scalar(v);
      case SK::Splat: return bounds(d->operands[0], role, lo, hi, given);
      case SK::Iota:
        *lo = *hi = Bound();
        lo->c = hi->c = d->ival;
        if (role == ROW && V.shape[0] > 1) {
          lo->v = hi->v = "wrow";
          hi->c += 32 * R - 1;
        } else {
          hi->c += V.shape[0] - 1;
        }
        return true;
      case SK::ExpandDims: return bounds(d->operands[0], d->axis == 1 ? ROW : COL, lo, hi, given);
      case SK::Broadcast: {
        const Value &O = val(d->operands[0]);
        if (O.shape.size() != 2) return bounds(d->operands[0], role, lo, hi, given);
        return bounds(d->operands[0], is_tile(O) ? TILE : O.shape[1] == 1 ? ROW : COL, lo, hi, given);
      }
      case SK::Map: {
        if (d->name != "arith.addi" && d->name != "arith.subi") return false;
        Bound a0, a1, b0, b1;
        if (!bounds(d->operands[0], role, &a0, &a1, given) || !bounds(d->operands[1], role, &b0, &b1, given)) return false;
        const bool minus = d->name == "arith.subi";
        auto sum = [&](const Bound &a, const Bound &b) {
          Bound r;
          r.c = minus ? a.c - b.c : a.c + b.c;
          r.v = b.v.empty() ? a.v : a.v.empty() ? (minus ? "-" + b.v : b.v) : "(" + a.v + (minus ? " - " : " + ") + b.v + ")";
          r.turns = (a.turns && b.v.empty()) || (b.turns && a.v.empty() && !minus);
          r.mixed = !r.turns && (a.turns || a.mixed || b.turns || b.mixed);
          return r;
        };
        *lo = sum(a0, minus ? b1 : b0);
        *hi = sum(a1, minus ? b0 : b1);
        if (V.dtype == "i32") {
          Bound least, most;
          least.c = INT32_MIN;
          most.c = INT32_MAX;
          *given += " && " + below(least, *lo, 1) + " && " + below(*hi, most, 1);
        }
        return true;
      }
      default: return false;
    }
  }
  // a scalar expression that is true only if the i1 block v is true for every element this wavefront holds
  bool all_true(int v, int role, std::string *text) {
    const Value &V = val(v);
    if (V.dtype != "i1") return false;
    if (V.shape.empty()) {
      *text = "(" + at(v, "0", "0") + ")";
      return true;
    }
    const SOp *d = def_of(v);
    if (!d) return false;
    switch (d->kind) {
      case SK::Splat: return all_true(d->operands[0], role, text);
      case SK::ExpandDims: return all_true(d->operands[0], d->axis == 1 ? ROW : COL, text);
      case SK::Broadcast: {
        const Value &O = val(d->operands[0]);
        if (O.shape.size() != 2) return all_true(d->operands[0], role, text);
        return all_true(d->operands[0], is_tile(O) ? TILE : O.shape[1] == 1 ? ROW : COL, text);
      }
      case SK::Map: {
        if (d->name == "arith.andi") {
          std::string a, b;
          if (!all_true(d->operands[0], role, &a) || !all_true(d->operands[1], role, &b)) return false;
          *text = "(" + a + " && " + b + ")";
          return true;
        }
        if (d->name.rfind("arith.cmpi.", 0) != 0) return false;
        const std::string p = d->name.substr(11);
        Bound a0, a1, b0, b1;
        std::string given;
        if (!bounds(d->operands[0], role, &a0, &a1, &given) || !bounds(d->operands[1], role, &b0, &b1, &given)) return false;
        if (p == "slt") *text = below(a1, b0, 0);
        else if (p == "sle") *text = below(a1, b0, 1);
        else if (p == "sgt") *text = below(b1, a0, 0);
        else if (p == "sge") *text = below(b1, a0, 1);
        else return false;
        *text = "(" + *text + given + ")";
        return true;
      }
      default: return false;
    }
  }

  // ---- code -------------------------------------------------------------------
  void line(const std::string &s) { os << pad() << s << "\n"; }
  int NB(int v) const { return (int)(val(v).shape[1] / 32); }
  std::string id(const char *p, int v) const { return p + std::to_string(v); }
  void open_tile(int v) {
    line("#pragma unroll");
    line("for (int rb = 0; rb < " + std::to_string(R) + "; rb++)");
    line("#pragma unroll");
    line("for (int nb = 0; nb < " + std::to_string(NB(v)) + "; nb++)");
    line("#pragma unroll");
  }
  void tile_loop(int v, const std::string &stmt) {
    open_tile(v);
    line("for (int i = 0; i < 16; i++) " + stmt);
  }
  void row_loop(const std::string &stmt) {
    line("#pragma unroll");
    line("for (int rb = 0; rb < " + std::to_string(R) + "; rb++) " + stmt);
  }
  std::string declare_tile(int v, const char *p = "v") {
    const std::string n = id(p, v);
    line(std::string(is16(val(v).dtype) ? "u32x8_t " : val(v).dtype == "f32" ? "f32x16_t " : "i32x16_t ") + n + "[" + std::to_string(R) + "][" + std::to_string(NB(v)) + "];");
    return n;
  }

  // the value of a 16-bit tile, two elements per dword
  void narrow_tile(const SOp &s) {
    const std::string n = declare_tile(s.result);
    const std::string x = el(s.operands[0], TILE);
    auto with_i = [&](const std::string &e, const std::string &to) {
      std::string out;
      for (size_t q = 0; q < e.size(); q++) {
        const bool word = e[q] == 'i' && (q == 0 || !(isalnum((unsigned char)e[q - 1]) || e[q - 1] == '_')) && (q + 1 == e.size() || !(isalnum((unsigned char)e[q + 1]) || e[q + 1] == '_'));
        out += word ? to : std::string(1, e[q]);
      }
      return out;
    };
    open_tile(s.result);
    line("for (int j = 0; j < 8; j++) " + n + "[rb][nb][j] = " + (val(s.result).dtype == "f16" ? "pack_f16(" : "pack_bf16(") + with_i(x, "(2 * j)") + ", " + with_i(x, "(2 * j + 1)") + ");");
    tile_of[s.result] = n;
  }

  void emit_map(const SOp &s) {
    const int v = s.result, r = roles.count(v) ? roles[v] : 0;
    const std::string &T = val(v).dtype;
    if ((r & TILE) && is_float(T)) {
      if (folded_into_exp(s)) return;
      if (is16(T)) {
        if (s.name != "arith.truncf" || val(s.operands[0]).dtype != "f32") decline("16-bit arithmetic on blocks");
        return narrow_tile(s);
      }
      std::string text;
      // a select that keeps the computed value wherever a mask holds: most blocks lie inside the mask as a whole
      if (s.name == "arith.select" && tile_of.count(s.operands[1]) && all_true(s.operands[0], TILE, &text)) {
        const std::string n = declare_tile(v);
        const bool held = factor_of.count(s.operands[1]) && minus_infinity(s.operands[2]);
        tile_loop(v, n + "[rb][nb][i] = " + (held ? tile_of[s.operands[1]] + "[rb][nb][i]" : el(s.operands[1], TILE)) + ";");
        if (held) factor_of[v] = factor_of[s.operands[1]];
        line("if (!" + text + ") {");
        indent++;
        tile_loop(v, "if (!" + el(s.operands[0], TILE) + ") " + n + "[rb][nb][i] = " + el(s.operands[2], TILE) + ";");
        indent--;
        line("}");
        tile_of[v] = n;
        return;
      }
      // a carried block times a row factor (the rescaling of an online softmax): multiplying by one changes nothing, so a
      // wavefront whose factors are all one skips it
      if (s.name == "arith.mulf" && cur_loop >= 0)
        for (int q = 0; q < 2; q++) {
          const int t = s.operands[q], f = s.operands[1 - q];
          const SOp *b = def_of(f);
          if (!carried.count(t) || !b || b->kind != SK::Broadcast || val(b->operands[0]).shape.size() != 2 || val(b->operands[0]).shape[1] != 1) continue;
          const std::string n = declare_tile(v), factor = el(f, TILE);
          tile_loop(v, n + "[rb][nb][i] = " + el(t, TILE) + ";");
          row_loop("if (__builtin_amdgcn_ballot_w64(" + factor + " != 1.0f)) {");
          indent++;
          line("#pragma unroll");
          line("for (int nb = 0; nb < " + std::to_string(NB(v)) + "; nb++)");
          line("#pragma unroll");
          line("for (int i = 0; i < 16; i++) " + n + "[rb][nb][i] = " + n + "[rb][nb][i] * " + factor + ";");
          indent--;
          line("}");
          tile_of[v] = n;
          return;
        }
      if (emit_exp_of_difference(s) || emit_scaled(s)) return;
      std::vector<std::string> a;
      for (int o : s.operands) a.push_back(el(o, TILE));
      text = map_text(s, a);
      const std::string n = declare_tile(v);
      tile_loop(v, n + "[rb][nb][i] = " + text + ";");
      tile_of[v] = n;
    }
    if ((r & ROW) && is_float(T)) {
      std::vector<std::string> a;
      for (int o : s.operands) a.push_back(el(o, ROW));
      const std::string text = map_text(s, a);
      const std::string n = id("r", v);
      line("float " + n + "[" + std::to_string(R) + "];");
      row_loop(n + "[rb] = " + text + ";");
      row_of[v] = n;
      if (meeting && v == meeting->tile_yields[maximum_slot]) {
        // A slice other than the first may begin with blocks in which a row is masked as a whole: its maximum is -infinity until then,
        // and what it adds to its sums is nothing.  (In the first slice that is as it is in the program: not a number.)
        next_maximum = n;
        line("float from" + n + "[" + std::to_string(R) + "];");
        row_loop("from" + n + "[rb] = " + n + "[rb] == nothing ? 0.f : " + n + "[rb];");
        row_of[v] = "from" + n;
      }
    }
  }
  std::string next_maximum;

  void emit_reduce(const SOp &s) {
    const int x = s.operands[0];
    const std::string n = id("r", s.result), T = "f32";
    SOp op = s;  // the combiner as an elementwise op on two values
    op.kind = SK::Map;
    auto combine = [&](const std::string &a, const std::string &b) { return map_text_f32(op, a, b); };
    line("float " + n + "[" + std::to_string(R) + "];");
    row_loop("{");
    indent++;
    const int nb = (int)(val(x).shape[1] / 32);
    // four chains, folded together at the end
    line("float f[4];");
    const bool held = factor_of.count(x) && (s.name == "arith.maxnumf" || s.name == "arith.maximumf");
    auto elem = [&](int b, int i) {
      std::string e = held ? tile_of[x] + "[rb][nb][i]" : el(x, TILE), out;
      for (size_t q = 0; q < e.size(); q++) {
        auto word = [&](const char *w) {
          const size_t l = strlen(w);
          return e.compare(q, l, w) == 0 && (q == 0 || !(isalnum((unsigned char)e[q - 1]) || e[q - 1] == '_')) && (q + l == e.size() || !(isalnum((unsigned char)e[q + l]) || e[q + l] == '_'));
        };
        if (word("nb")) { out += std::to_string(b); q++; }
        else if (word("i")) out += std::to_string(i);
        else out += e[q];
      }
      return out;
    };
    for (int c = 0; c < 4; c++) line("f[" + std::to_string(c) + "] = " + elem(0, c) + ";");
    for (int e = 4; e < 16 * nb; e++) {
      const std::string f = "f[" + std::to_string(e & 3) + "]";
      line(f + " = " + combine(f, elem(e / 16, e % 16)) + ";");
    }
    line("const float g0 = " + combine("f[0]", "f[1]") + ", g1 = " + combine("f[2]", "f[3]") + ", g = " + combine("g0", "g1") + ";");
    line("unsigned lo = __float_as_uint(g), hi = lo;");
    line("swap_halves(lo, hi);");
    line(n + "[rb] = " + combine("__uint_as_float(lo)", "__uint_as_float(hi)") + (held ? " * " + factor_of[x] : "") + ";");
    indent--;
    line("}");
    row_of[s.result] = n;
  }
  std::string map_text_f32(const SOp &op, const std::string &a, const std::string &b) {
    static const std::map<std::string, const char *> infix = {{"arith.addf", "+"}, {"arith.mulf", "*"}};
    static const std::map<std::string, const char *> call = {{"arith.maxnumf", "fmaxf"}, {"arith.minnumf", "fminf"}, {"arith.maximumf", "maximum_f"}, {"arith.minimumf", "minimum_f"}};
    if (infix.count(op.name)) return "(" + a + " " + infix.at(op.name) + " " + b + ")";
    if (call.count(op.name)) return std::string(call.at(op.name)) + "(" + a + ", " + b + ")";
    decline("a reduction with " + op.name);
  }

  // extent of an access along dimension d as a 32-bit scalar in [0, size] (the size itself when it is not masked)
  std::string extent(const Access &a, size_t d) {
    const std::string size = std::to_string(a.sizes[d]);
    if (a.dims.empty()) return size;
    int64_t c = 0;
    if (P.pool.is_const(a.dims[d], &c) && c >= a.sizes[d]) return size;
    return "(int)smin(smax(" + ex(a.dims[d]) + ", 0LL), " + size + "LL)";
  }
  bool full(const Access &a, size_t d) {
    int64_t c = 0;
    return a.dims.empty() || (P.pool.is_const(a.dims[d], &c) && c >= a.sizes[d]);
  }

  void emit_load(const SOp &s) {
    const int v = s.result, r = roles.count(v) ? roles[v] : 0;
    const Access &a = s.acc;
    if (r & FRAG) {
      const std::string n = id("a", v), ks = std::to_string(a.sizes[1] / 16);
      line("u32x4_t " + n + "[" + std::to_string(R) + "][" + ks + "];");
      line("{");
      indent++;
      line("const unsigned short *base = (const unsigned short *)p.ptr[" + std::to_string(a.base_arg) + "] + (" + ex(a.offsets[0]) + " + " + ex(a.offsets[1]) + ");");
      line("const long long pitch = " + ex(a.strides[0]) + ";");
      line("const int rows = mine ? " + extent(a, 0) + " : 0, cols = " + extent(a, 1) + ";");
      line("const bool vec = (((unsigned long long)base) & 15) == 0 && (pitch & 7) == 0;");
      line("#pragma unroll");
      line("for (int rb = 0; rb < " + std::to_string(R) + "; rb++)");
      line("#pragma unroll");
      line("for (int ks = 0; ks < " + ks + "; ks++) {");
      line("  const int row = " + std::string(ROWX) + ", col = 16 * ks + 2 * h4;");
      line("  " + n + "[rb][ks] = frag8(base + row * pitch + col, row < rows ? cols - col : 0, vec);");
      line("}");
      indent--;
      line("}");
      frag_of[v] = n;
    }
    auto elementwise = [&](const std::string &i0, const std::string &i1) {
      std::string pred, addr = address(a, i0, i1, pred);
      const std::string rd = mem_read(a, addr);
      pred = pred.empty() ? "mine" : "mine && " + pred;
      return "(" + pred + ") ? " + rd + " : " + other_of(a);
    };
    if (r & TILE) {
      if (!is_float(a.elem) || a.elem == "f64") decline("an elementwise load of " + a.elem);
      if (is16(a.elem)) {
        const std::string n = declare_tile(v);
        const std::string up = a.elem == "f16" ? "down_f16_exact(" : "down_bf16(";
        auto at_i = [&](const std::string &i) { return up + "(" + elementwise(ROWX, "(32 * nb + 8 * (" + i + " >> 2) + h4 + (" + i + " & 3))") + "))"; };
        open_tile(v);
        line("for (int j = 0; j < 8; j++) " + n + "[rb][nb][j] = (unsigned)" + at_i("(2 * j)") + " | ((unsigned)" + at_i("(2 * j + 1)") + " << 16);");
        tile_of[v] = n;
      } else {
        const std::string n = declare_tile(v);
        tile_loop(v, n + "[rb][nb][i] = " + elementwise(ROWX, COLX) + ";");
        tile_of[v] = n;
      }
    }
    if (r & ROW) {
      const std::string n = id("r", v), T = ctype(val(v).dtype);
      line(T + " " + n + "[" + std::to_string(R) + "];");
      row_loop(n + "[rb] = " + elementwise(a.sizes[0] == 1 ? "0" : ROWX, "0") + ";");
      row_of[v] = n;
    }
    if (r & COL) {
      const std::string n = id("c", v), T = ctype(val(v).dtype);
      const int64_t N = a.sizes.back();
      if (N % 32 || N > 256) decline("a vector of this length along the columns");
      line(T + " " + n + "[" + std::to_string(N / 32) + "][16];");
      line("#pragma unroll");
      line("for (int nb = 0; nb < " + std::to_string(N / 32) + "; nb++)");
      line("#pragma unroll");
      line("for (int i = 0; i < 16; i++) " + n + "[nb][i] = " + (a.sizes.size() == 2 ? elementwise("0", COLX) : elementwise(COLX, "0")) + ";");
      col_of[v] = n;
    }
  }
  std::map<int, std::string> frag_of;
  bool copies_due = false;  // the next product of the loop takes the copies of the next iteration's blocks

  // a scalar condition that is true only if every row (column) of dimension d is inside the access: for the usual extent
  // max(start, min(start + size, n)) - start with start the loop's own variable, start < n - size + 1 in 32 bits
  std::string whole(const Access &a, size_t d) {
    if (full(a, d)) return "true";
    const std::string size = std::to_string(a.sizes[d]);
    const Expr &e = P.pool.at(a.dims[d]);
    if (e.k == EK::Sub && P.pool.at(e.a).k == EK::MaxS) {
      const int start = e.b;
      const Expr &mx = P.pool.at(e.a);
      const int inner = mx.a == start ? mx.b : mx.b == start ? mx.a : -1;
      const Expr &st = P.pool.at(P.pool.at(start).k == EK::Sext ? P.pool.at(start).a : start);
      if (inner >= 0 && P.pool.at(inner).k == EK::MinS && st.k == EK::IV && P.pool.at(loop_by_id(st.a)->lb).bits == 32)
        for (int q = 0; q < 2; q++) {
          const Expr &mn = P.pool.at(inner);
          const int end = q ? mn.b : mn.a, n = q ? mn.a : mn.b;
          const Expr &en = P.pool.at(end);
          int64_t c = 0;
          if (en.k != EK::Add || !((en.a == start && P.pool.is_const(en.b, &c)) || (en.b == start && P.pool.is_const(en.a, &c))) || c < a.sizes[d]) continue;
          if (mentions(P.pool, n, EK::IV) || mentions(P.pool, n, EK::Iter)) continue;
          return "((int)" + ex(start) + " < sat32(" + ex(n) + " - " + std::to_string(a.sizes[d] - 1) + "LL))";
        }
    }
    return "(" + extent(a, d) + " >= " + size + ")";
  }
  // A copy of a right operand's block into its LDS image, as locals: the block's address, its pitch, and whether all of it can go by
  // direct-to-LDS loads (the same answer in every wavefront of the workgroup).
  void declare_stage(const Image &im) { line("const unsigned short *" + id("sb", im.load) + " = nullptr; long long " + id("sp", im.load) + " = 0; bool " + id("st", im.load) + " = false, " + id("sd", im.load) + " = false;"); }
  void locate_stage(const Image &im) {
    const Access &a = def_of(im.load)->acc;
    const std::string sb = id("sb", im.load), sp = id("sp", im.load), st = id("st", im.load);
    line(sb + " = (const unsigned short *)p.ptr[" + std::to_string(a.base_arg) + "] + (" + ex(a.offsets[0]) + " + " + ex(a.offsets[1]) + ");");
    line(sp + " = " + ex(a.strides[im.outer]) + ";");
    line(st + " = " + whole(a, im.inner) + " && (((unsigned long long)" + sb + ") & 15) == 0 && (" + sp + " & 7) == 0 && " + sp + " >= 0 && " + sp + " < " + std::to_string((int64_t)(1u << 30) / im.rows) + ";  // straight");
    line(id("sd", im.load) + " = " + st + " && " + whole(a, im.outer) + ";");
  }
  int stage_turns(const Image &im) const { return (int)((im.bytes() / 1024 + WAVES - 1) / WAVES); }  // direct-to-LDS loads per wavefront (1 KB each)
  std::string stage_copy(const Image &im, int turn, const std::string &from, const std::string &at_bytes) {
    const int NI = (int)(im.bytes() / 1024), RPI = 1024 / im.row_bytes;  // instructions of 1 KB, image rows per instruction
    const std::string ins = "(wave + " + std::to_string(WAVES * turn) + ")", row = "(" + ins + " * " + std::to_string(RPI) + " + lane / " + std::to_string(im.chunks) + ")";
    const std::string guard = WAVES * turn + WAVES > NI ? "if (wave < " + std::to_string(NI - WAVES * turn) + ") " : "";
    return guard + "copy_to_lds(" + from + ", (unsigned)(" + row + " * (int)" + id("sp", im.load) + " + 8 * ((lane & " + std::to_string(im.chunks - 1) + ") ^ (" + swizzle(im, row) + "))) * 2u, lds0 + " +
           at_bytes + " + " + ins + " * 1024);";
  }
  // Copies the block to byte offset `at` of the LDS array.  Whole blocks and last blocks of fewer rows go by direct-to-LDS loads, the
  // latter through a buffer resource that ends with the last row (what lies behind it is zero in LDS; rows must not overlap for
  // that); others through registers, which cost a loop 3 us where its last block is such a one (6 heads x 401 x 128: 16.8 -> 13.9 us).
  void emit_stage(const Image &im, const std::string &at_bytes) {
    const Access &a = def_of(im.load)->acc;
    const std::string sb = id("sb", im.load), sp = id("sp", im.load);
    line("if (" + id("sd", im.load) + ") {");
    indent++;
    for (int j = 0; j < stage_turns(im); j++) line(stage_copy(im, j, sb, at_bytes));
    indent--;
    line("} else {");
    indent++;
    line("const int rows = " + extent(a, im.outer) + ", cols = " + extent(a, im.inner) + ";");
    line("if (" + id("st", im.load) + " && " + sp + " >= " + std::to_string(im.cols) + " && " + sp + " < " + std::to_string((int64_t)(1u << 29) / im.rows) + ") {");
    indent++;
    line("const u32x4_t block = block_of(" + sb + ", rows > 0 ? (unsigned)((rows - 1) * (int)" + sp + " + " + std::to_string(im.cols) + ") * 2u : 0u);");
    for (int j = 0; j < stage_turns(im); j++) line(stage_copy(im, j, "block", at_bytes));
    indent--;
    line("} else {");
    indent++;
    line("const bool vec = (((unsigned long long)" + sb + ") & 15) == 0 && (" + sp + " & 7) == 0;");
    line("for (int c = threadIdx.x; c < " + std::to_string(im.rows * im.chunks) + "; c += " + std::to_string(64 * WAVES) + ") {");
    line("  const int row = c / " + std::to_string(im.chunks) + ", chunk = c & " + std::to_string(im.chunks - 1) + ";");
    line("  const u32x4_t w = frag8(" + sb + " + row * " + sp + " + 8 * chunk, row < rows ? cols - 8 * chunk : 0, vec);");
    line("  *(u32x4_t *)(lds + " + at_bytes + " + row * " + std::to_string(im.row_bytes) + " + ((chunk ^ (" + swizzle(im, "row") + ")) << 4)) = w;");
    line("}");
    indent--;
    line("}");
    indent--;
    line("}");
  }
  static std::string swizzle(const Image &im, const std::string &row) {
    if (!im.transposing) {
      if (im.chunks >= 16) return "(" + row + ") & 15";
      return "((" + row + ") / " + std::to_string(16 / im.chunks) + ") & " + std::to_string(im.chunks - 1);
    }
    if (im.chunks >= 16) return "((" + row + ") & 3) << 2";
    return "(((" + row + ") / " + std::to_string(16 / im.chunks) + ") & " + std::to_string(im.chunks / 4 - 1) + ") << 2";
  }

  void emit_dot(const SOp &s) {
    const int v = s.result;
    const SOp *l = right_load(s.operands[1]);
    const Image &im = images.at(l->result);
    const bool bf = val(s.operands[0]).dtype == "bf16";
    const bool natural = frag_of.count(s.operands[0]) != 0;  // the left operand's order of k inside an instruction
    const std::string n = declare_tile(v);
    const int nbs = NB(v), kss = (int)(val(s.operands[0]).shape[1] / 16);
    const SOp *c = def_of(s.operands[2]);
    if (c && c->kind == SK::Const && c->fval == 0) tile_loop(v, n + "[rb][nb][i] = 0.f;");
    else tile_loop(v, n + "[rb][nb][i] = " + el(s.operands[2], TILE) + ";");
    const std::string at_bytes = std::to_string(im.offset) + (im.loop >= 0 ? " + buf * " + std::to_string(im.bytes()) : "");
    line("{");
    indent++;
    line("const char *im = lds + " + at_bytes + ";");
    // The right operand's fragments are read DEPTH instructions ahead of the one that multiplies them (a read takes as long as
    // four), and the copies of the next iteration's blocks are spread among the instructions of the iteration's first product:
    // sent together, four wavefronts' copies of 32 KB hold the CU's memory pipe, and their senders, for some 640 cycles.
    const int frags = kss * nbs, depth = std::min(4, frags);
    std::vector<std::string> copies;
    if (copies_due) {
      for (auto &q : images)
        if (q.second.loop == cur_loop)
          for (int j = 0; j < stage_turns(q.second); j++)
            copies.push_back(stage_copy(q.second, j, id("sb", q.first), std::to_string(q.second.offset) + " + (buf ^ 1) * " + std::to_string(q.second.bytes())));
      copies_due = false;
    }
    const std::string RB = std::to_string(im.row_bytes), F = std::to_string(frags), D = std::to_string(depth), NBS = std::to_string(nbs);
    auto steps = [&](const std::vector<std::string> &between) {
      line("u32x4_t q[" + F + "];");
      line("#pragma unroll");
      line("for (int t = 0; t < " + F + " + " + D + "; t++) {");
      indent++;
      line("if (t < " + F + ") {");
      indent++;
      line("const int ks = t / " + NBS + ", nb = t % " + NBS + ";");
      if (!im.transposing) {
        line("const char *row = im + (32 * nb + l32) * " + RB + ";");
        line("const int sw = " + swizzle(im, "l32") + ";");  // (32 nb does not reach the swizzle: 32 / (16 / chunks) is a multiple of chunks)
        if (natural) {
          line("q[t] = *(const u32x4_t *)(row + (((2 * ks + (h4 >> 2)) ^ sw) << 4));");
        } else {
          line("const u32x2_t b0 = *(const u32x2_t *)(row + (((2 * ks) ^ sw) << 4) + 2 * h4), b1 = *(const u32x2_t *)(row + (((2 * ks + 1) ^ sw) << 4) + 2 * h4);");
          line("q[t] = (u32x4_t){b0.x, b0.y, b1.x, b1.y};");
        }
      } else {
        const std::string r0 = natural ? "16 * ks + 2 * h4 + (r16 >> 2)" : "16 * ks + h4 + (r16 >> 2)";
        const int second = natural ? 4 : 8;
        line("const int sw = " + swizzle(im, "r16 >> 2") + ";");
        line("const char *row = im + (" + r0 + ") * " + RB + " + 8 * (r16 & 1) + (((4 * nb + 2 * ((lane >> 4) & 1) + ((r16 & 3) >> 1)) ^ sw) << 4);");
        line("const u32x2_t b0 = read_tr(row), b1 = read_tr(row + " + std::to_string(second * im.row_bytes) + ");");
        line("q[t] = (u32x4_t){b0.x, b0.y, b1.x, b1.y};");
      }
      indent--;
      line("}");
      line("if (t >= " + D + ") {");
      indent++;
      line("const int ks = (t - " + D + ") / " + NBS + ", nb = (t - " + D + ") % " + NBS + ";");
      line("#pragma unroll");
      line("for (int rb = 0; rb < " + std::to_string(R) + "; rb++) {");
      if (natural) line("  const u32x4_t a = " + frag_of[s.operands[0]] + "[rb][ks];");
      else {
        const std::string t = tile_of.at(s.operands[0]);
        line("  const u32x4_t a = {" + t + "[rb][ks >> 1][4 * (ks & 1)], " + t + "[rb][ks >> 1][4 * (ks & 1) + 1], " + t + "[rb][ks >> 1][4 * (ks & 1) + 2], " + t +
             "[rb][ks >> 1][4 * (ks & 1) + 3]};");
      }
      line("  " + n + "[rb][nb] = mfma<" + (bf ? "true" : "false") + ">(q[t - " + D + "], a, " + n + "[rb][nb]);");
      line("}");
      indent--;
      line("}");
      for (size_t c = 0; c < between.size(); c++) line("if (t == " + std::to_string(depth + (int)(c * frags / between.size())) + ") " + (between[c].rfind("if", 0) == 0 ? "{ " + between[c] + " }" : between[c]));
      indent--;
      line("}");
      if (between.empty()) {  // (the compiler would read each fragment where it is used)
        const int reads = !im.transposing && natural ? 1 : 2;
        line("__builtin_amdgcn_sched_group_barrier(0x100, " + std::to_string(depth * reads) + ", 0);");
        for (int t = depth; t < frags; t++) line("__builtin_amdgcn_sched_group_barrier(0x008, " + std::to_string(R) + ", 0); __builtin_amdgcn_sched_group_barrier(0x100, " + std::to_string(reads) + ", 0);");
      }
    };
    if (!copies.empty()) {
      line("if (ahead) {");
      indent++;
      steps(copies);
      indent--;
      line("} else {");
      indent++;
    }
    steps({});
    if (!copies.empty()) {
      indent--;
      line("}");
    }
    indent--;
    line("}");
    tile_of[v] = n;
  }

  void emit_store(const SOp &s) {
    const Access &a = s.acc;
    const int v = s.operands[0];
    if (a.sizes.size() == 1) {
      std::string pred, addr = address(a, ROWX, "0", pred);
      line("if (mine && h4 == 0) {");
      indent++;
      line("#pragma unroll");
      line("for (int rb = 0; rb < " + std::to_string(R) + "; rb++) {");
      indent++;
      mem_write(a, addr, pred, el(v, ROW));
      indent--;
      line("}");
      indent--;
      line("}");
      return;
    }
    int64_t st = 0;
    const bool unit = P.pool.is_const(a.strides[1], &st) && st == 1;
    if (is16(a.elem) && unit && tile_of.count(v) && is16(val(v).dtype)) {
      const std::string t = tile_of.at(v);
      line("{");
      indent++;
      line("unsigned short *base = (unsigned short *)p.ptr[" + std::to_string(a.base_arg) + "] + (" + ex(a.offsets[0]) + " + " + ex(a.offsets[1]) + ");");
      line("const long long pitch = " + ex(a.strides[0]) + ";");
      line("const int rows = mine ? " + extent(a, 0) + " : 0, cols = " + extent(a, 1) + ";");
      line("const bool vec = (((unsigned long long)base) & 15) == 0 && (pitch & 7) == 0;");
      line("#pragma unroll");
      line("for (int rb = 0; rb < " + std::to_string(R) + "; rb++)");
      line("#pragma unroll");
      line("for (int nb = 0; nb < " + std::to_string(NB(v)) + "; nb++)");
      line("#pragma unroll");
      line("for (int g = 0; g < 2; g++) {  // the half wavefronts exchange four columns each: sixteen bytes of a row per lane");
      line("  unsigned x0 = " + t + "[rb][nb][4 * g], x1 = " + t + "[rb][nb][4 * g + 1], y0 = " + t + "[rb][nb][4 * g + 2], y1 = " + t + "[rb][nb][4 * g + 3];");
      line("  swap_halves(x0, y0);");
      line("  swap_halves(x1, y1);");
      line("  const int row = " + std::string(ROWX) + ", col = 32 * nb + 16 * g + 2 * h4;");
      line("  store8(base + row * pitch + col, row < rows ? cols - col : 0, vec, (u32x4_t){x0, x1, y0, y1});");
      line("}");
      indent--;
      line("}");
      return;
    }
    std::string pred, addr = address(a, ROWX, COLX, pred);
    line("if (mine) {");
    indent++;
    open_tile(v);
    line("for (int i = 0; i < 16; i++) {");
    indent++;
    mem_write(a, addr, pred, el(v, TILE));
    indent--;
    line("}");
    indent--;
    line("}");
  }

  void emit_ops(const std::vector<SOp> &ops) {
    for (const SOp &s : ops) {
      switch (s.kind) {
        case SK::Load:
          if (images.count(s.result)) {
            if (images.at(s.result).loop < 0) {
              line("{");
              indent++;
              declare_stage(images.at(s.result));
              locate_stage(images.at(s.result));
              emit_stage(images.at(s.result), std::to_string(images.at(s.result).offset));
              indent--;
              line("}");
              line("landed();");
            }
          } else emit_load(s);
          break;
        case SK::Map:
          if (roles.count(s.result)) emit_map(s);
          break;
        case SK::Reduce: if (roles.count(s.result)) emit_reduce(s); break;
        case SK::Dot: emit_dot(s); break;
        case SK::Store: emit_store(s); break;
        case SK::For: emit_for(s); break;
        default: break;
      }
    }
  }

  // The ops of a loop body with those that no product needs behind the last product: a softmax's row sums are then added up
  // between the second product's matrix instructions.  (Stores read nothing that is stored to: analyse().)
  std::vector<SOp> products_first(const std::vector<SOp> &ops) const {
    std::set<int> wanted;
    for (const SOp &o : ops)
      if (o.kind == SK::Dot) wanted.insert(o.result);
    for (size_t i = ops.size(); i-- > 0;)
      if (ops[i].result >= 0 && wanted.count(ops[i].result)) wanted.insert(ops[i].operands.begin(), ops[i].operands.end());
    std::vector<SOp> order;
    for (bool w : {true, false})
      for (const SOp &o : ops)
        if ((o.result >= 0 && wanted.count(o.result)) == w) order.push_back(o);
    return order;
  }

  void emit_for(const SOp &s) {
    const std::string L = std::to_string(s.loop);
    const bool i32 = P.pool.at(s.lb).bits == 32;
    for (size_t q = 0; q < s.tile_args.size(); q++) {
      const int a = s.tile_args[q];
      const Value &V = val(a);
      if (V.shape.empty()) decline("a carried scalar");
      const int r = roles.count(a) ? roles[a] : 0;
      const std::string n = "car" + L + "_" + std::to_string(q);
      const std::string later = meeting == &s && q != maximum_slot ? "slice ? 0.f : " : "";  // (what the sums start from counts once)
      if (r & TILE) {
        if (V.dtype != "f32") decline("a carried block of " + V.dtype);
        line("f32x16_t " + n + "[" + std::to_string(R) + "][" + std::to_string(NB(a)) + "];");
        tile_loop(a, n + "[rb][nb][i] = " + later + el(s.tile_inits[q], TILE) + ";");
        tile_of[a] = n;
      }
      if (r & ROW) {
        if (V.dtype != "f32") decline("a carried vector of " + V.dtype);
        line("float " + n + "r[" + std::to_string(R) + "];");
        row_loop(n + "r[rb] = " + later + el(s.tile_inits[q], ROW) + ";");
        row_of[a] = n + "r";
      }
    }
    for (size_t q = 0; q < s.int_iters.size(); q++) line("long long it" + L + "_" + std::to_string(q) + " = " + ex(s.int_iters[q].init) + ";");
    // Programs that share a workgroup turn together as often as the furthest of them: what one whose loop ends earlier carries
    // out of it is what it had there.
    const bool shared = G > 1;
    if (shared) for (size_t q = 0; q < s.int_iters.size(); q++) line("long long own" + L + "_" + std::to_string(q) + " = it" + L + "_" + std::to_string(q) + ";");
    bool staged = false;
    for (auto &im : images) staged = staged || im.second.loop == s.loop;
    const std::string iv = "iv" + L;
    // (32-bit loops count in 32 bits: a compare is one scalar instruction then, where a 64-bit one goes through the vector unit)
    const std::string T = i32 ? "int " : "long long ", cast = i32 ? "(int)" : "";
    line(T + iv + " = " + cast + ex(s.lb) + ";");
    line("const " + T + "ub" + L + " = mine ? " + cast + ex(s.ub) + " : " + iv + ";");
    if (G > 1) {
      const std::string px = std::string("pid") + "xyz"[axis], np = std::string("np") + "xyz"[axis];
      line("long long last" + L + " = " + iv + ";  // the furthest of this workgroup's programs");
      line("for (int g = 0; g < " + std::to_string(G) + "; g++) {");
      line("  const long long own = " + px + ", " + px + "_g = group0 + g;");
      line("  if (" + px + "_g < " + np + ") { const long long " + px + " = " + px + "_g; last" + L + " = smax(last" + L + ", " + ex(s.ub) + "); (void)" + px + "; }");
      line("  (void)own;");
      line("}");
    } else {
      // (every wavefront stages this program's blocks and meets its barriers, also one that has no rows of it)
      line("const long long last" + L + " = " + ex(s.ub) + ";");
    }
    if (meeting == &s) {
      int64_t step = 0;
      P.pool.is_const(s.step, &step);
      const std::string S = std::to_string(step) + "LL", whole = "whole" + L;
      // this workgroup's share of the iterations; more slices than iterations leave some workgroups without any
      line("const long long turns = last" + L + " > " + iv + " ? (last" + L + " - " + iv + " + " + std::to_string(step - 1) + "LL) / " + S + " : 0;");
      line("const int parts = (int)smax(1, smin(slices, turns));");
      line("if (slice >= parts) return;");
      line("const float nothing = slice > 0 ? -__builtin_inff() : __builtin_nanf(\"\");  // (equal to no maximum in the first slice)");
      line("const " + T + whole + " = " + cast + "last" + L + ";");
      line("const " + T + "end" + L + " = slice + 1 < parts ? " + cast + "(" + iv + " + turns * (slice + 1) / parts * " + S + ") : " + whole + ";");
      line(iv + " = " + cast + "(" + iv + " + turns * slice / parts * " + S + ");");
      line("const " + T + "own_ub" + L + " = ub" + L + " < end" + L + " ? ub" + L + " : end" + L + ";");
    } else {
      line("const " + T + "end" + L + " = " + cast + "last" + L + ";");
    }
    const std::string ub = (meeting == &s ? "own_ub" : "ub") + L;
    auto of_loop = [&](auto &&f) {
      for (auto &im : images)
        if (im.second.loop == s.loop) f(im.second);
    };
    auto stage_all = [&](const std::string &buf) {
      of_loop([&](const Image &im) { emit_stage(im, std::to_string(im.offset) + " + (" + buf + ") * " + std::to_string(im.bytes())); });
    };
    if (staged) {
      line("__syncthreads();");
      line("if (" + iv + " < end" + L + ") {");
      indent++;
      of_loop([&](const Image &im) { declare_stage(im); });
      of_loop([&](const Image &im) { locate_stage(im); });
      stage_all("0");
      indent--;
      line("}");
    }
    line("for (int buf = 0; " + iv + " < end" + L + "; buf ^= 1) {");
    indent++;
    line("const " + T + "next_iv" + L + " = " + cast + "(" + iv + " + " + ex(s.step) + ");");
    for (size_t q = 0; q < s.int_iters.size(); q++)
      line("const long long next" + L + "_" + std::to_string(q) + " = " + ex(s.int_iters[q].next) + ";");
    if (staged) {
      line("landed();");
      // The next iteration's blocks: a wavefront that has a product to do in this one sends their copies between its instructions
      // (emit_dot), any other, and every one whose blocks do not go by direct-to-LDS loads as a whole, sends them here.
      line("bool ahead = false;");
      of_loop([&](const Image &im) { declare_stage(im); });
      line("if (next_iv" + L + " < end" + L + ") {");
      indent++;
      // the names the index expressions use, at the next iteration's values
      line("const bool turn = " + iv + " < " + ub + ";");
      line("const " + T + "at_iv = next_iv" + L + ";");
      for (size_t q = 0; q < s.int_iters.size(); q++) line("const long long at_it" + std::to_string(q) + " = next" + L + "_" + std::to_string(q) + ";");
      line("{");
      indent++;
      line("const " + T + iv + " = at_iv; (void)" + iv + ";");
      for (size_t q = 0; q < s.int_iters.size(); q++) line("const long long it" + L + "_" + std::to_string(q) + " = at_it" + std::to_string(q) + "; (void)it" + L + "_" + std::to_string(q) + ";");
      std::string all = "turn";
      of_loop([&](const Image &im) {
        locate_stage(im);
        all += " && " + id("sd", im.load);
      });
      line("ahead = " + all + ";");
      line("if (!ahead) {");
      indent++;
      stage_all("buf ^ 1");
      indent--;
      line("}");
      indent--;
      line("}");
      indent--;
      line("}");
      copies_due = true;
    }
    line("if (" + iv + " < " + ub + ") {");
    indent++;
    auto saved_t = tile_of;
    auto saved_r = row_of;
    auto saved_c = col_of;
    cur_loop = s.loop;
    emit_ops(products_first(s.body));
    cur_loop = -1;
    copies_due = false;
    // every new value before the first assignment (a yield may name another carried value)
    for (size_t q = 0; q < s.tile_args.size(); q++) {
      const int a = s.tile_args[q], y = s.tile_yields[q];
      const int r = roles.count(a) ? roles[a] : 0;
      const std::string n = "new" + L + "_" + std::to_string(q);
      if (r & TILE) {
        line("f32x16_t " + n + "[" + std::to_string(R) + "][" + std::to_string(NB(a)) + "];");
        tile_loop(a, n + "[rb][nb][i] = " + el(y, TILE) + ";");
      }
      if (r & ROW) {
        line("float " + n + "r[" + std::to_string(R) + "];");
        row_loop(n + "r[rb] = " + (meeting == &s && q == maximum_slot ? next_maximum + "[rb]" : el(y, ROW)) + ";");
      }
    }
    for (size_t q = 0; q < s.tile_args.size(); q++) {
      const int a = s.tile_args[q];
      const int r = roles.count(a) ? roles[a] : 0;
      const std::string n = "new" + L + "_" + std::to_string(q);
      if (r & TILE) tile_loop(a, tile_of[a] + "[rb][nb][i] = " + n + "[rb][nb][i];");
      if (r & ROW) row_loop(row_of[a] + "[rb] = " + n + "r[rb];");
    }
    if (shared) for (size_t q = 0; q < s.int_iters.size(); q++) line("own" + L + "_" + std::to_string(q) + " = next" + L + "_" + std::to_string(q) + ";");
    tile_of = saved_t;
    row_of = saved_r;
    col_of = saved_c;
    indent--;
    line("}");
    line(iv + " = next_iv" + L + ";");
    for (size_t q = 0; q < s.int_iters.size(); q++) line("it" + L + "_" + std::to_string(q) + " = next" + L + "_" + std::to_string(q) + ";");
    indent--;
    line("}");
    for (size_t q = 0; q < s.int_iters.size(); q++) line("const long long res" + L + "_" + std::to_string(q) + " = " + (shared ? "own" : "it") + L + "_" + std::to_string(q) + "; (void)res" + L + "_" + std::to_string(q) + ";");
    for (size_t q = 0; q < s.tile_args.size(); q++) {
      const int a = s.tile_args[q], res = s.results[q];
      if (res < 0) continue;
      if (tile_of.count(a)) tile_of[res] = tile_of[a];
      if (row_of.count(a)) row_of[res] = row_of[a];
    }
    if (meeting == &s) slices_meet();
  }
};

// Registers a lane needs for the blocks that live through an iteration (a rough count, for the launch bounds): carried
// blocks and operand fragments, and two blocks of the widest kind being worked on.
inline int mma_registers(const MmaGen &g) {
  int64_t fixed = 0, widest = 0;
  std::set<int> steps;  // the new values of carried blocks take the old ones' registers
  for (const SOp &s : g.P.body) steps.insert(s.tile_yields.begin(), s.tile_yields.end());
  for (auto &r : g.roles) {
    const auto &V = g.val(r.first);
    if (r.second & MmaGen::FRAG) fixed += V.shape[1] / 4 * g.R;
    if (!(r.second & MmaGen::TILE) || V.dtype != "f32") continue;
    auto c = g.carried.find(r.first);
    if (c != g.carried.end() && c->second.first->tile_args[c->second.second] == r.first) fixed += V.shape[1] / 2 * g.R;
    else if (g.def.count(r.first) && g.def.at(r.first)->kind == SK::Dot && !steps.count(r.first) && V.shape[1] / 2 * g.R > widest) widest = V.shape[1] / 2 * g.R;
  }
  return (int)(fixed + 2 * widest);
}

const char *MMA_PRELUDE = R"SRC(
#define TTS_LOG2E 1.44269504088896340736f
typedef unsigned u32x8_t __attribute__((ext_vector_type(8)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
#define TTS_LDS(q) ((__attribute__((address_space(3))) void *)(q))
__device__ __forceinline__ float hardware_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ int sat32(long long x) { return (int)smin(smax(x, -2147483648LL), 2147483647LL); }
template <bool BF16>
__device__ __forceinline__ f32x16_t mfma(u32x4_t a, u32x4_t b, f32x16_t c) {
  if (BF16) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ unsigned pack_bf16(float a, float b) { const f32x2_t v = {a, b}; return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2_t)); }
// (the empty asm keeps a multiplication before it from being folded into the narrowing, as in down_f16)
__device__ __forceinline__ unsigned pack_f16(float a, float b) { asm("" : "+v"(a), "+v"(b)); const f32x2_t v = {a, b}; return __builtin_bit_cast(unsigned, __builtin_convertvector(v, f16x2_t)); }
// lanes 32-63 of x and lanes 0-31 of y change places
__device__ __forceinline__ void swap_halves(unsigned &x, unsigned &y) { asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y)); }
__device__ __forceinline__ u32x2_t read_tr(const char *q) {
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3))) *)TTS_LDS(q)));
}
// eight neighbouring 16-bit elements, zero beyond `valid`
__device__ __forceinline__ u32x4_t frag8(const unsigned short *q, int valid, bool vec) {
  if (valid >= 8 && vec) return *(const u32x4_t *)q;
  u32x4_t w = {0, 0, 0, 0};
  for (int e = 0; e < 8; e++)
    if (e < valid) w[e >> 1] |= (unsigned)q[e] << (16 * (e & 1));
  return w;
}
__device__ __forceinline__ void store8(unsigned short *q, int valid, bool vec, u32x4_t w) {
  if (valid >= 8 && vec) { *(u32x4_t *)q = w; return; }
  for (int e = 0; e < 8; e++)
    if (e < valid) q[e] = (unsigned short)(w[e >> 1] >> (16 * (e & 1)));
}
// 64 lanes' 16-byte chunks (each `off` bytes behind the wavefront's base address) to 1 KB of LDS
__device__ __forceinline__ void copy_to_lds(const void *base, unsigned off, unsigned to) {
  const unsigned long long b = (unsigned long long)base;
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32)), lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b);
  const void *s = (const void *)(((unsigned long long)hi << 32) | (unsigned long long)lo);
  // (the copy of the base keeps the load one instruction behind the write of m0, and off registers that v_readfirstlane has
  // just written, for which it would need five: the compiler counts neither)
  unsigned long long own;
  asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0" : "=&s"(own) : "s"(__builtin_amdgcn_readfirstlane((int)to)), "v"(off), "s"(s) : "memory", "m0");
}
// a block of `bytes` bytes as a buffer resource: loads behind its end give zeros.  (The s_nop is the distance described above.)
__device__ __forceinline__ u32x4_t block_of(const void *base, unsigned bytes) {
  const unsigned long long b = (unsigned long long)base;
  return (u32x4_t){(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b), (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32)), (unsigned)__builtin_amdgcn_readfirstlane((int)bytes), 0x00027000u};
}
__device__ __forceinline__ void copy_to_lds(u32x4_t block, unsigned off, unsigned to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" :: "s"(__builtin_amdgcn_readfirstlane((int)to)), "v"(off), "s"(block) : "memory", "m0");
}
// 16 bytes per lane behind a base address that a wavefront shares, written through to and read past the caches of an XCD (sc1): what
// workgroups on different XCDs hand over
typedef __amdgpu_buffer_rsrc_t shared_memory_t;
__device__ __forceinline__ shared_memory_t shared_memory(float *base) { return __builtin_amdgcn_make_buffer_rsrc(base, 0, 0x7fffffff, 0x00027000); }
__device__ __forceinline__ void put_through(shared_memory_t at, int offset, f32x4_t v) { __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), at, offset, 0, 16); }
__device__ __forceinline__ f32x4_t take_through(shared_memory_t at, int offset) { return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(at, offset, 0, 16)); }
// this wavefront's copies have arrived, and after the barrier everybody's
__device__ __forceinline__ void landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); __syncthreads(); }
)SRC";
