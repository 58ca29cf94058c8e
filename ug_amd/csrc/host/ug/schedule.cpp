// Scheduler: LazyBuffer DAG -> ordered kernels / matmuls / custom calls.  Mirrors
// ug-core/src/schedule.rs (fusion boundaries, argument order) and cache.rs.
#include <algorithm>
#include <set>
#include <unordered_map>
#include <unordered_set>

#include "lazy_buffer.h"

namespace ug {

// schedule.rs:23-39
op::Kernel KernelItem::kernel() const {
  op::Kernel k;
  k.name = "realize_" + std::to_string(dst.second.id());
  for (const auto& a : args) k.args.push_back(Arg{a.first, a.second.dtype(), true});
  op::Store st;
  st.dst = dst.first;
  st.layout = has_dst_layout ? dst_layout : Layout::from_shape(dst.second.shape());
  st.value = ast;
  k.ops.push_back(st);
  return k;
}

std::string normalized_kernel_key(const op::Kernel& k) {
  std::vector<std::pair<ArgId, size_t>> rename;
  std::string s;
  for (size_t i = 0; i < k.args.size(); ++i) {
    rename.push_back({k.args[i].id, i});
    s += "A" + std::to_string((int)k.args[i].dtype);
  }
  for (const op::Store& st : k.ops) {
    size_t idx = (size_t)-1;
    for (auto& p : rename)
      if (p.first == st.dst) idx = p.second;
    if (idx == (size_t)-1) bail("BUG: missing arg id");
    s += "|S" + std::to_string(idx) + st.layout.key() + op::ast_key(st.value, rename);
  }
  return s;
}

namespace {

// schedule.rs:480-520: use counts (1, or 2 for "twice or more"); realized nodes stop the walk.
void id_cnts(const LazyBuffer& b, std::unordered_map<size_t, size_t>& cnts) {
  if (b.realized()) return;
  size_t& cnt = cnts[b.id()];
  cnt += 1;
  if (cnt > 1) return;
  const Op& op = b.inner().op;
  switch (op.kind) {
    case Op::Value:
    case Op::Const: break;
    case Op::Reshape:
    case Op::Layout:
    case Op::Reduce:
    case Op::Unary: id_cnts(op.arg, cnts); break;
    case Op::Set:
      id_cnts(op.arg2, cnts);  // src
      id_cnts(op.arg, cnts);   // values
      break;
    case Op::MatMul:
    case Op::Binary:
      id_cnts(op.arg, cnts);
      id_cnts(op.arg2, cnts);
      break;
    case Op::CustomIp:
      for (const LazyBuffer& a : op.args) id_cnts(a, cnts);
      id_cnts(op.arg2, cnts);
      break;
    case Op::Ssa:
    case Op::Custom:
      for (const LazyBuffer& a : op.args) id_cnts(a, cnts);
      break;
  }
}

const LazyBuffer& buffer_of(const ArgBuffers& buffers, ArgId id) {
  auto it = std::lower_bound(buffers.begin(), buffers.end(), id.v, [](const auto& entry, size_t v) { return entry.first < v; });
  if (it == buffers.end() || it->first != id.v) bail("no arg for id " + std::to_string(id.v));
  return it->second;
}

// schedule.rs:308-475
struct Context {
  std::vector<ScheduleItem> items;
  ArgBuffers per_arg_id;
  std::unordered_map<size_t, op::Ast> ast_cache;
  std::unordered_map<size_t, ArgId> places;
  std::unordered_map<size_t, size_t> cnts;

  const LazyBuffer& get_arg_id(ArgId id) const { return buffer_of(per_arg_id, id); }

  ArgId new_arg(const LazyBuffer& b) {
    ArgId id = ArgId::fresh();
    per_arg_id.push_back({id.v, b});
    return id;
  }

  // Buffers that are an argument as they are, whoever asks: what exists, and what a custom call leaves.  A decode step is such calls on such buffers
  // alone, and without an expression (a load of the whole buffer) for each of them its schedule takes 78 -> 11 to 22 us for 33 calls on some 150 buffers,
  // and its thread, which had been the slower one of a reply of width 1024, no longer decides how long that takes: 198 -> 182 us a position (Tanolorn 290 -> 274).
  static bool is_place(const LazyBuffer& b) { return b.realized() || b.inner().op.kind == Op::Custom; }
  ArgId place(const LazyBuffer& b) {
    auto at = places.find(b.id());
    if (at != places.end()) return at->second;
    ArgId id;
    if (b.realized()) {
      id = new_arg(b);
    } else {
      const Op& op = b.inner().op;
      ScheduleItem it;
      it.kind = ScheduleItem::Custom;
      it.f = op.f;
      it.args.reserve(op.args.size() + 1);
      for (const LazyBuffer& a : op.args) it.args.push_back({push_schedule_item(a), a});
      id = new_arg(b);
      it.args.push_back({id, b});
      items.push_back(std::move(it));
    }
    places.emplace(b.id(), id);
    return id;
  }

  op::Ast walk(const LazyBuffer& b) {
    size_t id = b.id();
    auto cached = ast_cache.find(id);
    if (cached != ast_cache.end()) return cached->second;
    DType dtype = b.dtype();
    const Shape& shape = b.shape();
    op::Ast ast;
    if (is_place(b)) {
      ast = op::load(place(b), Layout::from_shape(shape), dtype);
      return ast_cache[id] = ast;
    } else {
      const Op& op = b.inner().op;
      switch (op.kind) {
        case Op::Unary: ast = op::unary(op.unary_op, walk(op.arg), op.cast_to); break;
        case Op::Binary: {
          op::Ast l = walk(op.arg);
          op::Ast r = walk(op.arg2);
          ast = op::binary(op.binary_op, l, r);
          break;
        }
        case Op::MatMul: {
          // Matmuls are not fused: both operands are materialised by their own kernels.
          push_schedule_item(op.arg);
          push_schedule_item(op.arg2);
          ArgId dst_id = new_arg(b);
          ScheduleItem it;
          it.kind = ScheduleItem::MatMul;
          it.dst = b;
          it.lhs = op.arg;
          it.rhs = op.arg2;
          it.b = op.b;
          it.m = op.m;
          it.n = op.n;
          it.k = op.k;
          it.transpose = op.transpose;
          items.push_back(std::move(it));
          ast = op::load(dst_id, Layout::from_shape(shape), dtype);
          break;
        }
        case Op::Reduce: ast = op::reduce(op.reduce_op, walk(op.arg), op.reduce_dim); break;
        case Op::Const: ast = op::cst(op.cst); break;
        case Op::Value: ast = op::load(new_arg(b), Layout::from_shape(shape), dtype); break;
        case Op::Reshape: {
          ArgId dst_id = push_schedule_item(op.arg);
          ast = op::load(dst_id, Layout::from_shape(shape), dtype);
          break;
        }
        case Op::Layout: ast = op::layout(op.layout_op, walk(op.arg), shape); break;
        case Op::Ssa: {
          Args args;
          for (const LazyBuffer& a : op.args) args.push_back({push_schedule_item(a), a});
          ArgId dst_id = new_arg(b);
          args.push_back({dst_id, b});
          ScheduleItem it;
          it.kind = ScheduleItem::Ssa;
          it.ssa = op.ssa;
          it.args = std::move(args);
          items.push_back(std::move(it));
          ast = op::load(dst_id, Layout::from_shape(shape), dtype);
          break;
        }
        case Op::Set: {
          ArgId arg_id = push_schedule_item(op.arg2);
          op::Ast values = walk(op.arg);
          push_kernel(op.arg2, values, &op.dst_layout);
          ast = op::load(arg_id, Layout::from_shape(shape), dtype);
          break;
        }
        case Op::CustomIp: {
          Args args;
          for (const LazyBuffer& a : op.args) args.push_back({push_schedule_item(a), a});
          ArgId arg_id = push_schedule_item(op.arg2);
          args.push_back({arg_id, op.arg2});
          ScheduleItem it;
          it.kind = ScheduleItem::Custom;
          it.f = op.f;
          it.args = std::move(args);
          items.push_back(std::move(it));
          ast = op::load(arg_id, Layout::from_shape(shape), dtype);
          break;
        }
        case Op::Custom: break;  // (a place)
      }
    }
    // A subtree used more than once gets a kernel of its own (schedule.rs:429-435).
    auto c = cnts.find(id);
    if (c != cnts.end() && c->second > 1) {
      ArgId dst_id = push_kernel(b, ast, nullptr);
      ast = op::load(dst_id, Layout::from_shape(shape), dtype);
    }
    ast_cache[id] = ast;
    return ast;
  }

  ArgId push_kernel(const LazyBuffer& buffer, const op::Ast& ast, const Layout* dst_layout) {
    if (ast.inner->kind == op::AstInner::Load) {
      const LazyBuffer& src = get_arg_id(ast.inner->load_src);
      // Loading and immediately storing the same buffer is a no-op (schedule.rs:446-453).
      if (src.data().get() == buffer.data().get()) return ast.inner->load_src;
    }
    ArgId dst_id = new_arg(buffer);
    std::set<ArgId> ids;
    op::arg_ids(ast, ids);
    ids.insert(dst_id);
    ScheduleItem it;
    it.kind = ScheduleItem::Kernel;
    for (const ArgId& a : ids) it.kernel.args.push_back({a, get_arg_id(a)});
    it.kernel.ast = ast;
    it.kernel.dst = {dst_id, buffer};
    if (dst_layout) {
      it.kernel.has_dst_layout = true;
      it.kernel.dst_layout = *dst_layout;
    }
    items.push_back(std::move(it));
    return dst_id;
  }

  ArgId push_schedule_item(const LazyBuffer& buffer) {
    if (is_place(buffer)) return place(buffer);
    op::Ast ast = walk(buffer);
    return push_kernel(buffer, ast, nullptr);
  }
};

}  // namespace

Schedule Schedule::create(const std::vector<LazyBuffer>& buffers) {
  if (buffers.empty()) bail("no buffers provided");
  Context ctx;
  for (const LazyBuffer& b : buffers) id_cnts(b, ctx.cnts);
  ctx.items.reserve(ctx.cnts.size());
  for (const LazyBuffer& b : buffers) ctx.push_schedule_item(b);
  Schedule s;
  s.device_ = buffers[0].device();
  s.items_ = std::move(ctx.items);
  s.per_arg_id_ = std::move(ctx.per_arg_id);
  return s;
}

const LazyBuffer& Schedule::get_arg_id(ArgId id) const {
  return buffer_of(per_arg_id_, id);
}

// A kernel item's place in the cache and its serial form, each made when it is first asked for.
struct Schedule::Prepared {
  std::optional<op::Kernel> kernel;
  CompilationCache::Entry* entry = nullptr;
  std::optional<ssa::Kernel> ssa;
  void of(const ScheduleItem& item, CompilationCache& cache) {
    if (kernel) return;
    kernel = item.kernel.kernel();
    entry = &cache.op_cache[normalized_kernel_key(*kernel)];
  }
  const ssa::Kernel& serial() {
    if (!ssa) ssa = kernel->optimize().lower(op::Opts());
    return *ssa;
  }
};

// schedule.rs:115-207
CompiledSchedule Schedule::compile_with_cache(CompilationCache& cache, bool pairs) const {
  CompiledSchedule out;
  out.device = device_;
  std::vector<Prepared> prepared(items_.size());
  std::optional<Holders> holders;
  out.funcs.reserve(items_.size());
  for (size_t i = 0; i < items_.size(); ++i) {
    CompiledFunc pair;
    if (!pairs || !device_->joins_rows() || !compile_pair(i, cache, prepared, holders, &pair)) {
      out.funcs.push_back(compile_item(items_[i], cache, &prepared[i]));
      continue;
    }
    // Neither kernel by itself is compiled or goes into the cache: a later schedule that has one alone compiles it then, and run() never does.
    out.funcs.push_back(pair);
    pair.in_pair = true;
    out.funcs.push_back(std::move(pair));
    ++i;
  }
  return out;
}

// Every handle that this schedule and the graph it was made from hold, counted in one walk.  (Behind buffers that were there already nothing is
// counted: a buffer that one of those holds is taken for somebody else's too, and written.)
Schedule::Holders Schedule::holders() const {
  Holders h;
  std::vector<const LazyBuffer*> todo;
  std::unordered_set<const LazyBufferInner*> results;
  auto note = [&](const LazyBuffer& x) {
    if (x.valid() && ++h.handles[&x.inner()] == 1) todo.push_back(&x);
  };
  for (size_t i = 0; i < items_.size(); ++i) {
    const ScheduleItem& it = items_[i];
    auto named = [&](const LazyBuffer& x) {
      if (!x.valid()) return;
      note(x);
      h.items.emplace(&x.inner(), std::make_pair(i, i)).first->second.second = i;
    };
    for (const auto& a : it.kernel.args) named(a.second);
    for (const auto& a : it.args) named(a.second);
    for (const LazyBuffer* x : {&it.kernel.dst.second, &it.dst, &it.lhs, &it.rhs}) named(*x);
    for (const LazyBuffer* x : {&it.kernel.dst.second, &it.dst})
      if (x->valid()) results.insert(&x->inner());
  }
  for (const auto& a : per_arg_id_) note(a.second);
  while (!todo.empty()) {
    const LazyBuffer& x = *todo.back();
    todo.pop_back();
    if (x.realized() && !results.count(&x.inner())) continue;
    const Op& op = x.inner().op;
    note(op.arg);
    note(op.arg2);
    for (const LazyBuffer& a : op.args) note(a);
  }
  return h;
}

// Whether nothing but items `first` and `first + 1` can ever ask for what the first one stores: no other item, no other buffer on the same storage,
// and every holder of the handle is this schedule or the graph it was made from.  (Handles are only ever copied from handles, so nobody can come
// by one later.)
bool Schedule::only_between(size_t first, const Holders& h) const {
  const LazyBuffer& b = items_[first].kernel.dst.second;
  if (b.data().use_count() != 1) return false;
  const auto at = h.items.find(&b.inner());
  return at != h.items.end() && at->second.first >= first && at->second.second <= first + 1 && b.use_count() == h.handles.at(&b.inner());
}

static bool reduces(const op::Ast& a) {
  switch (a.inner->kind) {
    case op::AstInner::Reduce: return true;
    case op::AstInner::Layout:
    case op::AstInner::Unary: return reduces(a.inner->arg);
    case op::AstInner::Binary: return reduces(a.inner->arg) || reduces(a.inner->rhs);
    default: return false;
  }
}

std::optional<Schedule::RowsPair> Schedule::pair_at(size_t first) const {
  if (first + 1 >= items_.size()) return {};
  const ScheduleItem &x = items_[first], &y = items_[first + 1];
  if (x.kind != ScheduleItem::Kernel || y.kind != ScheduleItem::Kernel || x.kernel.has_dst_layout || y.kernel.has_dst_layout) return {};
  const LazyBuffer& between = x.kernel.dst.second;
  if (between.elem_count() != y.kernel.dst.second.elem_count() || between.in_place_op() || y.kernel.dst.second.in_place_op()) return {};
  RowsPair p;
  // arguments by storage; a kernel that names one storage twice is refused when it runs, as ever
  const Args &xs = x.kernel.args, &ys = y.kernel.args;
  const auto at = [](const Args& args, size_t end, const LazyBuffer& b) {
    size_t i = 0;
    while (i < end && args[i].second.data() != b.data()) ++i;
    return i;
  };
  if (at(ys, ys.size(), between) == ys.size()) return {};
  for (size_t i = 0; i < xs.size(); ++i)
    if (at(xs, i, xs[i].second) < i) return {};
  const size_t link = at(xs, xs.size(), between);
  p.link = link < xs.size() ? (int)link : -1;
  p.shared.reserve(ys.size());
  for (size_t i = 0; i < ys.size(); ++i) {
    if (at(ys, i, ys[i].second) < i) return {};
    const size_t k = at(xs, xs.size(), ys[i].second);
    p.shared.push_back(k < xs.size() ? (int)k : -1);
  }
  // (row kernels reduce; asked last: it walks the expressions)
  if (p.link < 0 || !reduces(x.kernel.ast) || !reduces(y.kernel.ast)) return {};
  return p;
}

bool Schedule::compile_pair(size_t first, CompilationCache& cache, std::vector<Prepared>& prepared, std::optional<Holders>& held, CompiledFunc* out) const {
  const std::optional<RowsPair> p = pair_at(first);
  if (!p) return false;
  Prepared &x = prepared[first], &y = prepared[first + 1];
  x.of(items_[first], cache), y.of(items_[first + 1], cache);
  CompilationCache::Pair& known = cache.pair_cache[{x.entry, y.entry, p->link, p->shared}];
  if (known.stays_two) return false;
  if (!held) held = holders();
  const bool keep = !only_between(first, *held);
  std::shared_ptr<Func>& func = known.func[keep];
  if (!func) func = device_->compile_rows_pair(x.serial(), y.serial(), {x.kernel->ops[0].name(), y.kernel->ops[0].name()}, p->shared, p->link, keep);
  if (!func) {
    known.stays_two = true;
    return false;
  }
  out->kind = CompiledFunc::Kernel;
  out->func = func;
  const Args &xs = items_[first].kernel.args, &ys = items_[first + 1].kernel.args;
  for (size_t k = 0; k < xs.size(); ++k)
    if (keep || (int)k != p->link) out->args.push_back({xs[k].first, get_arg_id(xs[k].first)});
  for (size_t k = 0; k < ys.size(); ++k)
    if (p->shared[k] < 0) out->args.push_back({ys[k].first, get_arg_id(ys[k].first)});
  return true;
}

CompiledSchedule Schedule::compile_and_run(CompilationCache& cache) const {
  CompiledSchedule out;
  out.device = device_;
  out.funcs.reserve(items_.size());
  for (const ScheduleItem& item : items_) {
    Prepared prepared;
    out.funcs.push_back(compile_item(item, cache, &prepared));
    out.run_one(out.funcs.back());
  }
  return out;
}

// schedule.rs:162-188: grid heuristics, only for devices that ask for them.
static ssa::Kernel on_a_grid(const op::Kernel& kernel) {
  op::Opts opts;
  if (kernel.ops.size() == 1 && kernel.ops[0].layout.rank() >= 1 && kernel.ops[0].layout.num_elements() >= 1) {
    std::vector<std::pair<size_t, size_t>> dims;
    for (size_t i = 0; i < kernel.ops[0].layout.rank(); ++i) dims.push_back({i, kernel.ops[0].layout.dims()[i]});
    std::stable_sort(dims.begin(), dims.end(), [](const auto& a, const auto& b) { return a.second > b.second; });
    if (dims.size() >= 2 && dims[1].second > 1) opts = op::Opts().with_block_axis(dims[0].first).with_thread_block(dims[1].first, 32);
    else if (dims.size() > 1 && dims[0].second > 1) opts = op::Opts().with_global_axis(dims[0].first, 32);
  }
  return kernel.lower(opts);
}

CompiledFunc Schedule::compile_item(const ScheduleItem& item, CompilationCache& cache, Prepared* prepared) const {
  {
    CompiledFunc call;
    switch (item.kind) {
      case ScheduleItem::MatMul:
        call.kind = CompiledFunc::MatMul;
        call.dst = item.dst;
        call.lhs = item.lhs;
        call.rhs = item.rhs;
        call.b = item.b;
        call.m = item.m;
        call.n = item.n;
        call.k = item.k;
        call.transpose = item.transpose;
        break;
      case ScheduleItem::Custom:
        call.kind = CompiledFunc::Custom;
        call.f = item.f;
        call.args = item.args;
        break;
      case ScheduleItem::Ssa: {
        call.kind = CompiledFunc::Kernel;
        call.args = item.args;
        std::string key = item.ssa.instrs_key();
        auto it = cache.ssa_cache.find(key);
        if (it != cache.ssa_cache.end()) {
          call.func = it->second;
        } else {
          call.func = device_->compile(item.ssa, nullptr);
          cache.ssa_cache[key] = call.func;
        }
        break;
      }
      case ScheduleItem::Kernel: {
        call.kind = CompiledFunc::Kernel;
        prepared->of(item, cache);
        const op::Kernel& kernel = *prepared->kernel;
        for (const Arg& a : kernel.args) call.args.push_back({a.id, get_arg_id(a.id)});
        if (prepared->entry->func) {
          call.func = prepared->entry->func;
          break;
        }
        std::string kernel_name = kernel.ops.empty() ? "" : kernel.ops[0].name();
        const std::string* name = kernel.ops.empty() ? nullptr : &kernel_name;
        if (device_->use_grid()) call.func = device_->compile(on_a_grid(kernel.optimize()), name);
        else call.func = device_->compile(prepared->serial(), name);
        prepared->entry->func = call.func;
        break;
      }
    }
    return call;
  }
}

void CompiledSchedule::allocate_all() const {
  for (const CompiledFunc& f : funcs) {
    if (f.kind == CompiledFunc::MatMul) {
      f.dst.maybe_allocate_uninit();
      f.lhs.maybe_allocate_uninit();
      f.rhs.maybe_allocate_uninit();
    } else {
      for (const auto& a : f.args) a.second.maybe_allocate_uninit();
    }
  }
}

// schedule.rs:234-305
void CompiledSchedule::run() const {
  for (const CompiledFunc& f : funcs)
    if (!f.in_pair) run_one(f);
}

void CompiledSchedule::run_one(const CompiledFunc& f) const {
  thread_local std::vector<Slice*> bs;
  {
    switch (f.kind) {
      case CompiledFunc::Kernel:
      case CompiledFunc::Custom: {
        bs.clear();
        for (const auto& a : f.args) {
          a.second.maybe_allocate_uninit();
          // RefCell::try_borrow_mut: a cell may appear once.
          Slice* s = a.second.data()->slice.get();
          for (Slice* seen : bs)
            if (seen == s) bail("already borrowed: BorrowMutError");
          bs.push_back(s);
        }
        if (f.kind == CompiledFunc::Kernel) device->run(*f.func, bs);
        else (*f.f)(bs);
        break;
      }
      case CompiledFunc::MatMul: {
        const auto& ld = f.lhs.dims();
        const auto& rd = f.rhs.dims();
        size_t lr = ld.size(), rr = rd.size();
        std::vector<size_t> lp(ld), rp(rd);
        if (lr < rr) lp.insert(lp.begin(), rr - lr, 1);
        if (rr < lr) rp.insert(rp.begin(), lr - rr, 1);
        Layout lhs_l = Layout::from_shape(Shape(lp));
        Layout rhs_l = Layout::from_shape(Shape(rp));
        if (f.transpose) rhs_l = rhs_l.transpose();
        f.dst.maybe_allocate_uninit();
        f.lhs.maybe_allocate_uninit();
        f.rhs.maybe_allocate_uninit();
        if (f.dst.data().get() == f.lhs.data().get() || f.dst.data().get() == f.rhs.data().get()) bail("already borrowed: BorrowMutError");
        device->matmul(*f.dst.data()->slice, *f.lhs.data()->slice, *f.rhs.data()->slice, f.b, f.m, f.n, f.k, lhs_l, rhs_l);
        break;
      }
    }
  }
}

}  // namespace ug
