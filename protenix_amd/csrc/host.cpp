// The native host path: what protenix_amd/*.py does between a module call and the C ABI of
// libprotenix_amd.so (allocation, argument lists, streams, autograd bookkeeping), in C++.  One call
// per stack, update or operator instead of some twenty Python-level calls per block: below a few
// hundred tokens the GPU finishes a block's kernels faster than Python can enqueue them (93 tokens:
// 390 us of Python per block against 130 us of kernels).
//
// Weights are laid out here, from the modules' parameters, once per weight set (a plan), with a record of the
// parameters, sub-modules and hooks they came from: valid() compares identities and version
// counters, so that a parameter that was replaced or changed in place is noticed on the next call.
// The kernels and their arguments are those of ops.py; in a stack the single track's stages ride on the next block's
// pair kernels (Stages), where the Python path launches them on a second stream.
#include <torch/extension.h>

#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <cstring>
#include <mutex>
#include <set>

#include "../../include/protenix_amd.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using c10::optional;

void check(int rc, const char* what) {
  if (rc == PTX_OK) return;
  const char* kind = rc == 1 ? "bad argument" : rc == 2 ? "unsupported shape" : rc == 3 ? "launch failure" : "error";
  throw std::runtime_error(std::string(what) + ": " + kind + " (" + std::to_string(rc) + "): " + ptx_last_error_string());
}

int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return PTX_F32;
    case at::kBFloat16: return PTX_BF16;
    case at::kHalf: return PTX_F16;
    default: throw std::runtime_error(std::string("protenix_amd kernels take float32 or bfloat16 tensors, got ") + toString(t));
  }
}
// rows `z` with weights and workspaces in `compute`
int code_of_rows(at::ScalarType z, at::ScalarType compute) {
  return z == compute ? code_of(z) : PTX_MIXED;
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
hipStream_t current_stream(const Tensor& t) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

// ---- what a plan's weights were made from ---------------------------------------------------
// A plan stands in for a tree of modules only while every one of them is of a class it knows and runs that class's
// own forward; a sub-module of another type, a class changed under way or a `forward` set on an instance makes
// it stale.
struct Guard {
  struct Module {
    py::object dict;            // m.__dict__
    PyObject* m;                // (held by its parent's entry, or by the caller)
    py::object type;
  };
  std::vector<Module> modules;
  bool foreign = false;            // a module of a class that is not among `classes`
  struct Entry {
    py::object dict, key, value;   // dict[key] is value
    int64_t version = -1;          // of a parameter
    const void* data = nullptr;
  };
  std::vector<Entry> entries;
  std::vector<py::object> empty;   // dicts that must have no entries (hooks)

  void add(const py::dict& d, const py::handle& key) {
    Entry e;
    e.dict = d;
    e.key = py::reinterpret_borrow<py::object>(key);
    e.value = d[key];
    if (THPVariable_Check(e.value.ptr())) {
      const Tensor& t = THPVariable_Unpack(e.value.ptr());
      e.version = t.is_inference() ? -2 : (int64_t)t._version();
      e.data = t.data_ptr();
    }
    entries.push_back(std::move(e));
  }
  // `m` and everything below it; the plain attributes named in `attrs` where they exist
  Guard(const py::object& m, const py::list& attrs, const py::set& classes) { walk(m, attrs, classes); }
  void walk(const py::object& m, const py::list& attrs, const py::set& classes) {
    py::dict d = m.attr("__dict__");
    py::object type = py::reinterpret_borrow<py::object>((PyObject*)Py_TYPE(m.ptr()));
    if (!classes.contains(type)) {
      foreign = true;
      return;
    }
    modules.push_back(Module{d, m.ptr(), std::move(type)});
    py::dict params = d["_parameters"], mods = d["_modules"];
    for (auto item : params) add(params, item.first);
    empty.push_back(d["_forward_hooks"]);
    empty.push_back(d["_forward_pre_hooks"]);
    for (auto a : attrs)
      if (d.contains(a)) add(d, a);
    for (auto item : mods) {
      add(mods, item.first);
      if (!item.second.is_none()) walk(py::reinterpret_borrow<py::object>(item.second), attrs, classes);
    }
  }
  bool valid() const {
    static PyObject* const forward = PyUnicode_InternFromString("forward");
    if (foreign) return false;
    for (const Entry& e : entries) {
      PyObject* now = PyDict_GetItem(e.dict.ptr(), e.key.ptr());   // borrowed
      if (now != e.value.ptr()) return false;
      if (e.version != -1) {
        const Tensor& t = THPVariable_Unpack(now);
        if (e.version == -2 || t.is_inference() || (int64_t)t._version() != e.version || t.data_ptr() != e.data) return false;
      }
    }
    for (const py::object& d : empty)
      if (PyDict_Size(d.ptr()) != 0) return false;
    for (const Module& m : modules)   // (the entries hold: every module is still where it was)
      if ((PyObject*)Py_TYPE(m.m) != m.type.ptr() || PyDict_GetItem(m.dict.ptr(), forward)) return false;
    return true;
  }
};

// A point on a stream, to be waited for or timed.
struct Mark {
  hipEvent_t e = nullptr;
  explicit Mark(hipStream_t st, unsigned flags = hipEventDefault) {
    if (hipEventCreateWithFlags(&e, flags) != hipSuccess || hipEventRecord(e, st) != hipSuccess) throw std::runtime_error("cannot record an event");
  }
  Mark(const Mark&) = delete;
  ~Mark() { (void)hipEventDestroy(e); }
  float elapsed_time(const Mark& end) const {
    float ms = 0;
    if (hipEventElapsedTime(&ms, e, end.e) != hipSuccess) throw std::runtime_error("hipEventElapsedTime failed (synchronize first)");
    return ms;
  }
};

bool capturing(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone;
}

// What all plans are.  Weights are laid out on the stream of the call that made the plan; a call on another stream waits for
// them once, and they are not handed out again while that stream may still read them.
struct Plan {
  std::shared_ptr<const Guard> guard;
  explicit Plan(std::shared_ptr<const Guard> g) : guard(std::move(g)) {}
  Plan(const Plan&) = delete;
  virtual ~Plan() = default;
  bool valid() const { return guard->valid(); }
  // before this plan's launches on `st` (not while a graph is recorded, which takes no waits from outside: the recording's
  // owner has synchronised)
  void used_on(const c10::Stream& st, hipStream_t stream) const {
    if (!ready_ || stream == made_on_) return;
    const std::lock_guard<std::mutex> lock(mutex_);
    if (others_.count(stream) || capturing(stream)) return;
    others_.insert(stream);
    if (hipStreamWaitEvent(stream, ready_->e, 0) != hipSuccess) throw std::runtime_error("hipStreamWaitEvent failed");
    for (const Tensor& t : *weights_) t.record_stream(st);
  }

 protected:
  // all weights have been laid out, on `stream`
  void made(hipStream_t stream, const std::vector<Tensor>& weights) {
    if (capturing(stream)) return;   // (part of the recording)
    made_on_ = stream;
    weights_ = &weights;
    ready_ = std::make_unique<Mark>(stream, hipEventDisableTiming);
  }

 private:
  std::unique_ptr<Mark> ready_;
  hipStream_t made_on_ = nullptr;
  const std::vector<Tensor>* weights_ = nullptr;
  mutable std::mutex mutex_;
  mutable std::set<hipStream_t> others_;
};

// ---- a plan's weights ----------------------------------------------------------------------
// A configuration without a native path: the call goes to Python, which has it or the error message.
struct NotCovered {};
void require(bool ok) {
  if (!ok) throw NotCovered{};
}

// A module as Python holds it: plain attributes, sub-modules and parameters out of its dicts.  (Every class in the tree is
// one of this package's, see Guard.)
struct Module {
  py::dict d;
  explicit Module(const py::handle& m) : d(m.attr("__dict__")) {}
  py::object item(const char* name) const {
    require(d.contains(name));
    return d[name];
  }
  int number(const char* name) const { return item(name).cast<int>(); }
  double real(const char* name) const { return item(name).cast<double>(); }
  Module operator[](const char* name) const {
    const py::dict mods = d["_modules"];
    require(mods.contains(name) && !mods[name].is_none());
    return Module(mods[name]);
  }
  Tensor parameter(const char* name) const {   // undefined for None
    const py::dict params = d["_parameters"];
    require(params.contains(name));
    const py::object p = params[name];
    return p.is_none() ? Tensor() : p.cast<Tensor>();
  }
  // a linear layer's weight, of the size the kernels will take it for
  Tensor matrix(int64_t n_out, int64_t n_in) const {
    const Tensor w = parameter("weight");
    require(w.defined() && w.dim() == 2 && w.size(0) == n_out && w.size(1) == n_in);
    return w;
  }
  Tensor vector(const char* name, int64_t n) const {
    const Tensor v = parameter(name);
    require(!v.defined() || (v.dim() == 1 && v.size(0) == n));
    return v;
  }
};

// Parameters in the type and place the kernels want them: as they are where they qualify (dense, at a multiple of 16 bytes),
// otherwise converted, all of a plan's in one launch.
struct Weights {
  std::vector<Tensor> kept;        // what the pointers handed out point into
  Weights(at::Device device, hipStream_t stream) : device_(device), st_(stream) {}

  // *out: the parameter in `type` (null for none); valid after settle().  temporary: until done().
  void want(const void** out, const Tensor& t, at::ScalarType type, bool temporary = false) { add(out, t, type, temporary, false); }
  // *out: the matrices one below the other, packed for ptx_single_linear_stage
  void want_fragments(const void** out, std::initializer_list<Tensor> matrices, at::ScalarType type) {
    for (const Tensor& t : matrices) {
      add(out, t, type, false, true);
      out = nullptr;    // (it follows the one before)
    }
  }
  void settle() {
    int64_t bytes[2] = {0, 0};
    for (Wanted& w : wanted_) {
      int64_t& used = bytes[w.temporary];
      if (w.out) used = (used + 255) / 256 * 256;   // (whole cache lines; a matrix below another follows it)
      w.at = used;
      used += w.t.numel() * (int64_t)at::elementSize(w.type);
    }
    const auto options = at::TensorOptions().dtype(at::kByte).device(device_);
    char* base[2];
    for (int k = 0; k < 2; ++k) {
      Tensor buffer = at::empty({bytes[k]}, options);
      base[k] = (char*)buffer.data_ptr();
      (k ? temporaries_ : kept).push_back(std::move(buffer));
    }
    std::vector<ptx_param> list;
    for (const Wanted& w : wanted_) {
      char* dst = base[w.temporary] + w.at;
      if (w.out) *w.out = dst;
      const int64_t cols = w.t.dim() == 2 ? w.t.size(1) : w.t.numel();
      list.push_back(ptx_param{w.t.data_ptr(), dst, cols ? w.t.numel() / cols : 0, (int)cols, code_of(w.t.scalar_type()), code_of(w.type),
                               w.fragments});
    }
    check(ptx_param_pack(list.data(), (int)list.size(), st_), "param_pack");
    wanted_.clear();
  }
  // room for `elems` elements, kept
  void* room(int64_t elems, at::ScalarType type) {
    kept.push_back(at::empty({elems}, at::TensorOptions().dtype(type).device(device_)));
    return kept.back().data_ptr();
  }
  hipStream_t stream() const { return st_; }
  void done() { temporaries_.clear(); }   // (their memory is used again behind the launches on this stream)

 private:
  struct Wanted {
    Tensor t;
    const void** out;
    at::ScalarType type;
    bool temporary, fragments;
    int64_t at = 0;
  };
  void add(const void** out, const Tensor& p, at::ScalarType type, bool temporary, bool fragments) {
    if (!p.defined()) {
      *out = nullptr;
      return;
    }
    Tensor t = p.detach();
    if (t.device() != device_ || (t.scalar_type() != at::kFloat && t.scalar_type() != at::kBFloat16)) t = t.to(device_, type);
    t = t.contiguous();
    if (!fragments && t.scalar_type() == type && ((uintptr_t)t.data_ptr() & 15) == 0) {
      *out = t.data_ptr();
      (temporary ? temporaries_ : kept).push_back(std::move(t));
      return;
    }
    wanted_.push_back(Wanted{std::move(t), out, type, temporary, fragments});
  }
  at::Device device_;
  hipStream_t st_;
  std::vector<Wanted> wanted_;
  std::vector<Tensor> temporaries_;
};

// rows of c channels with this hidden width and arithmetic on the packed kernels
void require_width(int c, int hidden, at::ScalarType compute) {
  require((compute == at::kFloat || compute == at::kBFloat16) &&
          (((c == 64 || c == 128) && hidden == 128) || (c == 256 && hidden == 256 && compute == at::kBFloat16)));
}

struct TriMul {
  const void *ln_in_w, *ln_in_b, *ln_out_w, *ln_out_b, *packed = nullptr;
  int c_z, c_h;
  bool incoming;
  const void* w[6];     // while the plan is made
  TriMul(const Module& m, Weights& ws, at::ScalarType type) : c_z(m.number("c_z")), c_h(m.number("c_hidden")) {
    require_width(c_z, c_h, type);
    incoming = !m.item("_outgoing").cast<bool>();
    const Module in = m["layer_norm_in"], out = m["layer_norm_out"];
    ws.want(&ln_in_w, in.vector("weight", c_z), type);
    ws.want(&ln_in_b, in.vector("bias", c_z), type);
    ws.want(&ln_out_w, out.vector("weight", c_h), type);
    ws.want(&ln_out_b, out.vector("bias", c_h), type);
    const char* const names[4] = {"linear_a_p", "linear_a_g", "linear_b_p", "linear_b_g"};
    for (int i = 0; i < 4; ++i) ws.want(&w[i], m[names[i]].matrix(c_h, c_z), type, true);
    ws.want(&w[4], m["linear_z"].matrix(c_z, c_h), type, true);
    ws.want(&w[5], m["linear_g"].matrix(c_z, c_z), type, true);
  }
  void pack(Weights& ws, at::ScalarType type) {
    const int dt = code_of(type);
    void* p = ws.room(ptx_trimul_packed_elems(c_z, c_h, dt), type);
    check(ptx_trimul_pack(w[0], w[1], w[2], w[3], w[4], w[5], p, c_z, c_h, dt, ws.stream()), "trimul_pack");
    packed = p;
  }
};
struct TriAtt {
  const void *ln_w, *ln_b, *packed = nullptr;
  int c, heads;
  float inf;
  bool transposed;
  const void* w[6];     // while the plan is made: q, k, v, gate, bias, output
  TriAtt(const Module& m, Weights& ws, at::ScalarType type, bool transposed_)
      : c(m.number("c_in")), heads(m.number("no_heads")), inf((float)m.real("inf")), transposed(transposed_) {
    require(m.number("c_hidden") == 32);
    require_width(c, heads * 32, type);
    const Module ln = m["layer_norm"], mha = m["mha"];
    ws.want(&ln_w, ln.vector("weight", c), type);
    ws.want(&ln_b, ln.vector("bias", c), type);
    const char* const names[4] = {"linear_q", "linear_k", "linear_v", "linear_g"};
    for (int i = 0; i < 4; ++i) ws.want(&w[i], mha[names[i]].matrix(heads * 32, c), type, true);
    ws.want(&w[4], m["linear"].matrix(heads, c), type, true);
    ws.want(&w[5], mha["linear_o"].matrix(c, heads * 32), type, true);
  }
  void pack(Weights& ws, at::ScalarType type) {
    const int dt = code_of(type);
    void* p = ws.room(ptx_triattn_packed_elems(c, heads, dt), type);
    check(ptx_triattn_pack(w[0], w[1], w[2], w[3], w[4], w[5], p, c, heads, dt, ws.stream()), "triattn_pack");
    packed = p;
  }
};
struct Mask {   // of one pair tensor: as the triangle multiplications / the starting node read it, transposed, valid tokens
  Tensor m, mt;
  int n_valid = -1;
};
std::vector<Mask> masks_of(const py::list& l) {
  std::vector<Mask> v;
  for (auto h : l) {
    py::tuple t = py::reinterpret_borrow<py::tuple>(h);
    Mask m;
    if (!t[0].is_none()) m.m = t[0].cast<Tensor>();
    if (!t[1].is_none()) m.mt = t[1].cast<Tensor>();
    if (!t[2].is_none()) m.n_valid = t[2].cast<int>();
    v.push_back(std::move(m));
  }
  return v;
}

// One workspace, cut into 256-byte aligned parts; a triangle update's intermediates of one pair tensor.
struct Cut {
  char* base;
  int64_t used = 0;
  void* part(int64_t bytes) {
    void* p = base ? base + used : nullptr;
    used += (bytes + 255) / 256 * 256;
    return p;
  }
};
struct TriMulWs {
  void *a, *b, *x;
  TriMulWs(Cut& c, int n, int c_h, int64_t es) {
    a = c.part(ptx_trimul_operand_elems(n, c_h) * es);
    b = c.part(ptx_trimul_operand_elems(n, c_h) * es);
    x = c.part((int64_t)c_h * n * ((n + 7) / 8 * 8) * es);
  }
};
struct TriAttWs {
  void *q, *g, *k, *vt, *tb;
  TriAttWs(Cut& c, int n, int heads, int64_t es) {
    q = c.part((int64_t)heads * n * n * 32 * es);
    g = c.part((int64_t)heads * n * n * 32 * es);
    k = c.part(ptx_triattn_kv_elems(n, heads) * es);
    vt = c.part(ptx_triattn_kv_elems(n, heads) * es);
    tb = c.part(ptx_triattn_bias_elems(n, heads) * es);
  }
};
int64_t workspace_bytes(int n, int c_h, int heads, int64_t es) {
  Cut m{nullptr}, a{nullptr};
  if (c_h) TriMulWs(m, n, c_h, es);
  if (heads) TriAttWs(a, n, heads, es);
  return std::max(m.used, a.used);
}
// The same for updates whose output stage also projects for the next one (no gate tensors): what such a launch reads,
// x or o, lies apart from what it writes.
struct ChainWs {
  void *a, *b, *x, *q, *k, *vt, *tb, *o;
  ChainWs(Cut& c, int n, int c_h, int heads, int64_t es) {
    const int64_t ab = ptx_trimul_operand_elems(n, c_h) * es, row = (int64_t)heads * n * n * 32 * es;
    const int64_t kv = ptx_triattn_kv_elems(n, heads) * es;
    a = q = c.part(std::max(ab, row));
    b = k = c.part(std::max(ab, kv));
    vt = c.part(kv);
    tb = c.part(ptx_triattn_bias_elems(n, heads) * es);
    x = o = c.part(std::max((int64_t)c_h * n * ((n + 7) / 8 * 8) * es, row));
  }
};
int64_t chain_bytes(int n, int c_h, int heads, int64_t es) {
  Cut c{nullptr};
  ChainWs(c, n, c_h, heads, es);
  return c.used;
}

constexpr float kEps = 1e-5f;

// The stages of the single tracks of earlier blocks, in order: every pair launch that can carry one takes the
// first, so that a block's single track runs underneath the next block's pair kernels without launches,
// streams or waits of its own.  A block has seven stages and, its updates apart, seven such launches; where one of its projections is
// faster without (see Run::carry), the two LayerNorms, 5 us each, are launched by themselves; chained updates (Block::chain) have fewer
// launches, and their contractions, cores and transition take stages too.
struct Stages {
  struct Named {
    ptx_single_stage stage;
    const char* name;
    bool layernorm;
  };
  std::vector<Named> list;
  size_t next = 0;
  const ptx_single_stage* take() { return next < list.size() ? &list[next++].stage : nullptr; }
  ptx_single_stage* add(const char* name) {
    list.push_back(Named{{}, name, std::strcmp(name, "layernorm") == 0});
    return &list.back().stage;
  }
  void clear() {
    list.clear();
    next = 0;
  }
};

// One call: its stream, the single-track stages that wait for a launch to ride on, and what the caller
// wants to look at (ops.py): every launch bracketed by events, and workspaces filled with NaN first.
struct Run {
  c10::Stream stream;
  hipStream_t st;
  Stages singles;
  bool poison = false, timing = false;
  struct Span {
    const char* name;
    std::shared_ptr<Mark> begin, end;
  };
  std::vector<Span> spans;

  explicit Run(const Tensor& z)
      : stream(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(z.device().index()).unwrap()), st(current_stream(z)) {}

  template <typename F> void launch(const char* name, F&& f) {
    if (!timing) return check(f(), name);
    Span s{name, std::make_shared<Mark>(st), nullptr};
    check(f(), name);
    s.end = std::make_shared<Mark>(st);
    spans.push_back(std::move(s));
  }
  // What a pair launch carries: the next stage, or none for a projection (stage 0: of the triangle multiplications, 2: of the
  // attentions) that has a faster kernel for it - from 480 tokens on, below that the LayerNorms' launches cost what it saves
  // (16-bit rows, 384 tokens 528 us carrying / 533, 448 711 / 716, 480 881 / 872). On fp32 rows that is one of the two kinds at most, which leaves
  // five launches for the five other stages, on 16-bit rows it may be both, and stages left over are
  // launched.  us per block with a single track, always carrying / so: fp32 rows, 512 tokens 1107 / 1092, 640 1814 / 1785, 768
  // 2615 / 2595, 1024 5090 / 5047, 2048 28073 / 27832; 16-bit rows, 768 2403 / 2339, 1024 4656 / 4517, 1536 12661 / 12403.
  // Chained updates (Block::chain) have two launches fewer to carry: small products carry then, elsewhere the LayerNorms
  // are launched by themselves too.
  bool mul_alone = false, att_alone = false, contract_carries = false, chained = false, core_carries = false;
  void row_stages(int n, int c_z, int hidden, int dt) {
    mul_alone = ptx_row_stage_resident(0, n, c_z, hidden, dt);
    att_alone = n >= 480 && ptx_row_stage_resident(2, n, c_z, hidden, dt);
    contract_carries = ptx_trimul_contract_carries(n, dt);
  }
  // stage 4: of the contractions, which take part where the updates are chained (two launches fewer to carry), 5: of the
  // attention cores, see Block::joins_products
  const ptx_single_stage* carry(int stage) {
    if ((stage == 0 && mul_alone) || (stage == 2 && att_alone) || (stage == 4 && !(chained && contract_carries)) ||
        (stage == 5 && !core_carries))
      return nullptr;
    if ((mul_alone || att_alone || (chained && !contract_carries)) && singles.next < singles.list.size() && singles.list[singles.next].layernorm) run_next();
    return singles.take();
  }
  void run_next() {
    const char* name = singles.list[singles.next].name;
    const ptx_single_stage* s = singles.take();
    launch(name, [&] { return ptx_single_stage_run(s, st); });
  }
  void run_rest() {
    while (singles.next < singles.list.size()) run_next();
    singles.clear();
  }
  // The same in front of a launch that rewrites the pair bias but can carry a stage: the last one, which does not read it, is
  // left to it.
  optional<ptx_single_stage> run_rest_but_last() {
    optional<ptx_single_stage> last;
    while (singles.next + 1 < singles.list.size()) run_next();
    if (singles.next < singles.list.size()) last = *singles.take();
    singles.clear();
    return last;
  }
  // (0xff bytes are NaNs in every type)
  Tensor workspace(int64_t bytes, const at::TensorOptions& like) const {
    Tensor t = at::empty({bytes}, like.dtype(at::kByte));
    return poison ? t.fill_(255) : t;
  }
  // name -> [(begin, end)], appended to the caller's dict; with the interpreter's lock
  void hand_over(const py::object& timer) const {
    for (const Span& s : spans)
      py::reinterpret_borrow<py::dict>(timer).attr("setdefault")(s.name, py::list()).attr("append")(py::make_tuple(s.begin, s.end));
  }
};

void run_contraction(const TriMul& w, const void* a, const void* b, void* x, int n, int dt, Run& run) {
  const ptx_single_stage* carry4 = run.carry(4);
  run.launch("trimul_contract", [&] {
    return ptx_trimul_contract_carry(a, b, x, n, (n + 7) / 8 * 8, w.c_h, ptx_key_pitch(n), dt, carry4, run.st);
  });
}

// projection and product; the product is left in x
void run_trimul_product(const TriMul& w, const void* z, const Tensor& mask, int n, int dt, void* a, void* b, void* x, Run& run) {
  const ptx_single_stage* carry0 = run.carry(0);
  run.launch("trimul_project", [&] {
    return ptx_trimul_project_packed(z, ptr(mask), w.ln_in_w, w.ln_in_b, w.packed, a, b, n, w.c_z, w.c_h, ptx_key_pitch(n),
                                     w.incoming, kEps, dt, carry0, run.st);
  });
  run_contraction(w, a, b, x, n, dt, run);
}

void run_trimul_output(const TriMul& w, const void* x, const void* z, void* out, int n, bool add, int dt, Run& run) {
  const ptx_single_stage* carry1 = run.carry(1);
  run.launch("trimul_output", [&] {
    return ptx_trimul_output_packed(x, (n + 7) / 8 * 8, z, w.ln_in_w, w.ln_in_b, w.ln_out_w, w.ln_out_b, w.packed, out,
                                    n, w.c_z, w.c_h, add, kEps, dt, carry1, run.st);
  });
}

void run_trimul(const TriMul& w, const void* z, const Tensor& mask, void* out, int n, bool add, int dt, int64_t es, void* ws,
                Run& run) {
  Cut c{(char*)ws};
  TriMulWs s(c, n, w.c_h, es);
  run_trimul_product(w, z, mask, n, dt, s.a, s.b, s.x, run);
  run_trimul_output(w, s.x, z, out, n, add, dt, run);
}

// the attention of projected operands, gated unless the gate is null, into o
void run_attention(const TriAtt& w, const void* q, const void* k, const void* vt, const void* gate, const void* tb, void* o, const Mask& mask,
                   int n, int dt, Run& run) {
  const int pitch = ptx_key_pitch(n);
  const void* m = ptr(w.transposed ? mask.mt : mask.m);
  if (m && mask.n_valid >= 0) {
    // padding at the end: valid rows over valid keys without a mask, padded rows with it (ops.py)
    run.launch("triattn_fwd", [&] {
      return ptx_triattn_fwd_rows(q, k, vt, gate, tb, nullptr, o, n, w.heads, 32, pitch, 0, w.inf, 0, mask.n_valid,
                                  mask.n_valid, dt, run.st);
    });
    run.launch("triattn_fwd_padded_rows", [&] {
      return ptx_triattn_fwd_rows(q, k, vt, gate, tb, m, o, n, w.heads, 32, pitch, 0, w.inf, mask.n_valid, n - mask.n_valid, n,
                                  dt, run.st);
    });
  } else {
    const ptx_single_stage* carry5 = run.carry(5);
    run.launch("triattn_fwd", [&] {
      return ptx_triattn_fwd_carry(q, k, vt, gate, tb, m, o, n, w.heads, 32, pitch, 0, w.inf, dt, carry5, run.st);
    });
  }
}

// projection and core; the attention output is left in ws.g
TriAttWs run_triatt_core(const TriAtt& w, const void* z, const Mask& mask, int n, int dt, int64_t es, void* ws, Run& run) {
  Cut c{(char*)ws};
  TriAttWs s(c, n, w.heads, es);
  void* gate = ptx_triattn_late_gate(w.c, w.heads, dt) ? nullptr : s.g;
  const ptx_single_stage* carry2 = run.carry(2);
  run.launch("triattn_project", [&] {
    return ptx_triattn_project_packed(z, w.ln_w, w.ln_b, w.packed, s.q, s.k, s.vt, gate, s.tb, n, w.c, w.heads, ptx_key_pitch(n),
                                      w.transposed, kEps, dt, carry2, run.st);
  });
  run_attention(w, s.q, s.k, s.vt, gate, s.tb, s.g, mask, n, dt, run);
  return s;
}

void run_triatt(const TriAtt& w, const void* z, const Mask& mask, void* out, int n, bool add, int dt, int64_t es, void* ws,
                Run& run) {
  const TriAttWs s = run_triatt_core(w, z, mask, n, dt, es, ws, run);
  const ptx_single_stage* carry3 = run.carry(3);
  run.launch("triattn_output", [&] {
    return ptx_triattn_output_packed(s.g, z, w.ln_w, w.ln_b, w.packed, out, n, w.c, w.heads, w.transposed, add, kEps, dt,
                                     carry3, run.st);
  });
}

// ---- one Pairformer block ----------------------------------------------------------------------
struct Block : Plan {
  struct SingleWs;
  Weights weights;
  at::ScalarType compute;
  int c_z, c_s;
  TriMul out, in;
  TriAtt start, end;
  // pair transition (fused: with the ending node's output stage in front, one launch)
  int n_factor;
  bool fused;
  const void *tr_ln_w, *tr_ln_b, *tr_packed;
  // single track (matrices packed for ptx_single_linear_stage)
  int heads = 0, d = 0, hidden = 0;
  double a_eps = kEps, s_eps = kEps;
  const void *pb_ln_w = nullptr, *pb_ln_b = nullptr, *pb_w = nullptr, *a_ln_w, *a_ln_b, *w_in, *b_q, *w_o, *s_ln_w, *s_ln_b, *s_wa, *s_wb,
      *s_wo;

  // `module` on pair tensors like z (compute: their kernels' arithmetic) and single representations of type s_type; throws
  // NotCovered
  Block(std::shared_ptr<const Guard> guard_, const Module& m, const Tensor& z, at::ScalarType compute_, optional<at::ScalarType> s_type)
      : Plan(std::move(guard_)), weights(z.device(), current_stream(z)), compute(compute_), c_z((int)z.size(-1)), c_s(m.number("c_s")),
        out(m["tri_mul_out"], weights, compute), in(m["tri_mul_in"], weights, compute), start(m["tri_att_start"], weights, compute, false),
        end(m["tri_att_end"], weights, compute, true) {
    require(out.c_z == c_z && in.c_z == c_z && start.c == c_z && end.c == c_z);
    const Module tr = m["pair_transition"], tr_ln = tr["layernorm1"];
    n_factor = tr.number("n");
    require(tr.number("c_in") == c_z && n_factor > 0 && n_factor <= 64 && (n_factor * c_z) % 64 == 0);
    fused = c_z == 128 && end.heads == 4 && compute == at::kBFloat16;
    weights.want(&tr_ln_w, tr_ln.vector("weight", c_z), compute);
    weights.want(&tr_ln_b, tr_ln.vector("bias", c_z), compute);
    const void* w_tr[3];
    const int n_hidden = n_factor * c_z;
    weights.want(&w_tr[0], tr["linear_no_bias_a"].matrix(n_hidden, c_z), compute, true);
    weights.want(&w_tr[1], tr["linear_no_bias_b"].matrix(n_hidden, c_z), compute, true);
    weights.want(&w_tr[2], tr["linear_no_bias"].matrix(c_z, n_hidden), compute, true);
    if (c_s > 0) take_single(m, z, s_type);
    weights.settle();
    out.pack(weights, compute);
    in.pack(weights, compute);
    start.pack(weights, compute);
    end.pack(weights, compute);
    const int dt = code_of(compute);
    void* p = weights.room(fused ? ptx_triattn_output_transition_packed_elems(n_factor) : ptx_transition_packed_elems(c_z, n_factor), compute);
    if (fused)
      check(ptx_triattn_output_transition_pack(end.w[3], end.w[5], w_tr[0], w_tr[1], w_tr[2], p, n_factor, dt, weights.stream()), "transition_pack");
    else
      check(ptx_transition_pack(w_tr[0], w_tr[1], w_tr[2], p, c_z, n_factor, dt, weights.stream()), "transition_pack");
    tr_packed = p;
    weights.done();
    made(weights.stream(), weights.kept);
  }
  // The single track's stages ride on the pair kernels: same storage type, LayerNorm rows of whole vectors, on rows
  // of 128 or 256 channels; and not on widths that have a fused pair transition (64, 128, 256).
  void take_single(const Module& m, const Tensor& z, optional<at::ScalarType> s_type) {
    require(s_type && *s_type == z.scalar_type());
    const at::ScalarType type = *s_type;
    const Module apb = m["attention_pair_bias"], att = apb["attention"], st = m["single_transition"], ln_a = apb["layernorm_a"],
                 ln_z = apb["layernorm_z"], ln_s = st["layernorm1"];
    heads = att.number("num_heads");
    d = att.number("c_hidden");
    hidden = st.number("n") * c_s;
    const int hd = heads * d;
    require(c_s % 32 == 0 && c_s * (int64_t)at::elementSize(type) <= 2048 && c_s != 64 && c_s != 128 && c_s != 256 &&
            (c_z == 128 || c_z == 256) && heads >= 1 && heads <= 32 && apb.number("n_heads") == heads && att.number("c_q") == c_s &&
            att.number("c_k") == c_s && att.number("c_v") == c_s && st.number("c_in") == c_s && d > 0 && d % 8 == 0 && d <= 32 && hd % 32 == 0 &&
            hidden > 0);
    auto matrix = [&](const Module& parent, const char* name, int64_t n_out, int64_t n_in) {
      const Module l = parent[name];
      require(l.item("precision").is_none());
      return l.matrix(n_out, n_in);
    };
    weights.want(&pb_ln_w, ln_z.vector("weight", c_z), compute);
    weights.want(&pb_ln_b, ln_z.vector("bias", c_z), compute);
    weights.want(&pb_w, apb["linear_nobias_z"].matrix(heads, c_z), compute);
    weights.want(&a_ln_w, ln_a.vector("weight", c_s), type);
    weights.want(&a_ln_b, ln_a.vector("bias", c_s), type);
    weights.want(&s_ln_w, ln_s.vector("weight", c_s), type);
    weights.want(&s_ln_b, ln_s.vector("bias", c_s), type);
    weights.want(&b_q, att["linear_q"].vector("bias", hd), type);
    a_eps = ln_a.real("eps");
    s_eps = ln_s.real("eps");
    weights.want_fragments(&w_in, {matrix(att, "linear_q", hd, c_s), matrix(att, "linear_k", hd, c_s), matrix(att, "linear_g", hd, c_s),
                                   matrix(att, "linear_v", hd, c_s)}, type);
    weights.want_fragments(&w_o, {matrix(att, "linear_o", c_s, hd)}, type);
    weights.want_fragments(&s_wa, {matrix(st, "linear_no_bias_a", hidden, c_s)}, type);
    weights.want_fragments(&s_wb, {matrix(st, "linear_no_bias_b", hidden, c_s)}, type);
    weights.want_fragments(&s_wo, {matrix(st, "linear_no_bias", c_s, hidden)}, type);
  }

  // The five pair updates of the pair tensors `from` (like z; may be z) into z [batch][n][n][c_z]; the single attention's pair
  // bias (fp32 [batch][heads][n][n]) of the finished z into `bias` (null: none wanted).
  void pair_track(const void* from, const Tensor& z, const std::vector<Mask>& masks, int64_t batch, int n, void* ws, float* bias, Run& run) const {
    const int dt = code_of_rows(z.scalar_type(), compute);
    const int64_t es = at::elementSize(compute), plane = (int64_t)n * n * c_z * z.element_size();
    char* zp = (char*)z.data_ptr();
    const char* fp = (const char*)from;
    static const Mask none;
    auto mask = [&](int64_t b) -> const Mask& { return masks.empty() ? none : masks[b]; };
    const int64_t bias_plane = (int64_t)heads * n * n;
    if (run.chained) {
      for (int64_t b = 0; b < batch; ++b) {
        void* zb = zp + b * plane;
        chain(fp + b * plane, zb, mask(b), n, dt, es, ws, run);
        if (fused) {
          optional<ptx_single_stage> last;
          if (b == 0 && bias && ptx_triattn_output_transition_carries(n)) last = run.run_rest_but_last();
          else if (b == 0) run.run_rest();   // (the bias is about to be rewritten)
          output_transition(zb, attention_output(n, es, ws), n, dt, bias ? bias + b * bias_plane : nullptr, last ? &*last : nullptr, run);
        } else {
          output(end, zb, attention_output(n, es, ws), n, dt, run);
        }
      }
      if (fused) return;
    } else {
      for (int64_t b = 0; b < batch; ++b) run_trimul(out, fp + b * plane, mask(b).m, zp + b * plane, n, true, dt, es, ws, run);
      for (int64_t b = 0; b < batch; ++b) run_trimul(in, zp + b * plane, mask(b).m, zp + b * plane, n, true, dt, es, ws, run);
      for (int64_t b = 0; b < batch; ++b) run_triatt(start, zp + b * plane, mask(b), zp + b * plane, n, true, dt, es, ws, run);
      if (fused) {
        for (int64_t b = 0; b < batch; ++b) {
          void* zb = zp + b * plane;
          const TriAttWs s = run_triatt_core(end, zb, mask(b), n, dt, es, ws, run);
          if (b == 0) run.run_rest();   // (the bias is about to be rewritten)
          output_transition(zb, s.g, n, dt, bias ? bias + b * bias_plane : nullptr, nullptr, run);
        }
        return;
      }
      for (int64_t b = 0; b < batch; ++b) run_triatt(end, zp + b * plane, mask(b), zp + b * plane, n, true, dt, es, ws, run);
    }
    run.run_rest();   // (the bias is about to be rewritten)
    run.launch("transition", [&] {
      return ptx_transition_fwd(zp, tr_ln_w, tr_ln_b, tr_packed, zp, batch * n * n, c_z, n_factor, 1, kEps, dt, run.st);
    });
    if (bias)
      for (int64_t b = 0; b < batch; ++b)
        run.launch("pair_bias", [&] {
          return ptx_pair_bias_fwd(zp + b * plane, pb_ln_w, pb_ln_b, pb_w, bias + b * bias_plane, n, c_z, heads, 1, kEps, dt,
                                   run.st);
        });
  }

  // Whether an output stage projects for the update behind it (16-bit arithmetic; not where launches are timed one by one).
  bool chains(const Run& run, int n, int dt) const {
    return !run.timing && out.c_h == in.c_h && start.heads == end.heads && ptx_triattn_late_gate(c_z, start.heads, dt) &&
           ptx_row_stages_joined(1, n, c_z, out.c_h, dt);
  }
  // With a single track only where the block's other launches can carry its seven stages: two projections and output stages
  // and the two products carry six, the transition the last one or else an attention core one more.
  bool joins_products(int n, int dt) const {
    return ptx_row_stages_joined(0, n, c_z, out.c_h, dt) &&
           (c_s == 0 || (fused && ptx_trimul_contract_carries(n, dt) && (ptx_triattn_output_transition_carries(n) || ptx_triattn_fwd_carries(n, dt))));
  }
  bool core_carries(int n, int dt) const {
    return c_s > 0 && joins_products(n, dt) && !ptx_triattn_output_transition_carries(n);
  }
  // The block up to the ending node's attention output: pair tensor `from` (may be z) into z.
  void chain(const void* from, void* z, const Mask& mask, int n, int dt, int64_t es, void* ws, Run& run) const {
    Cut c{(char*)ws};
    const ChainWs s(c, n, out.c_h, start.heads, es);
    const int ldx = (n + 7) / 8 * 8, pitch = ptx_key_pitch(n);
    run_trimul_product(out, from, mask.m, n, dt, s.a, s.b, s.x, run);
    if (joins_products(n, dt)) {
      const ptx_single_stage* carry0 = run.carry(1);
      run.launch("trimul_output_trimul_project", [&] {
        return ptx_trimul_output_trimul_project(s.x, ldx, from, ptr(mask.m), out.ln_in_w, out.ln_in_b, out.ln_out_w, out.ln_out_b, out.packed, z,
                                                in.ln_in_w, in.ln_in_b, in.packed, s.a, s.b, n, c_z, out.c_h, pitch, kEps, dt, carry0, run.st);
      });
      run_contraction(in, s.a, s.b, s.x, n, dt, run);
    } else {
      run_trimul_output(out, s.x, from, z, n, true, dt, run);
      run_trimul_product(in, z, mask.m, n, dt, s.a, s.b, s.x, run);
    }
    const ptx_single_stage* carry1 = run.carry(1);
    run.launch("trimul_output_triattn_project", [&] {
      return ptx_trimul_output_triattn_project(s.x, ldx, z, in.ln_in_w, in.ln_in_b, in.ln_out_w, in.ln_out_b, in.packed, z, start.ln_w,
                                               start.ln_b, start.packed, s.q, s.k, s.vt, s.tb, n, c_z, in.c_h, start.heads, pitch, kEps, dt,
                                               carry1, run.st);
    });
    run_attention(start, s.q, s.k, s.vt, nullptr, s.tb, s.o, mask, n, dt, run);
    if (ptx_row_stages_joined(2, n, c_z, out.c_h, dt)) {
      const ptx_single_stage* carry3 = run.carry(3);
      run.launch("triattn_output_triattn_project", [&] {
        return ptx_triattn_output_triattn_project(s.o, z, start.ln_w, start.ln_b, start.packed, z, end.ln_w, end.ln_b, end.packed, s.q, s.k,
                                                  s.vt, s.tb, n, c_z, start.heads, pitch, kEps, dt, carry3, run.st);
      });
    } else {
      output(start, z, s.o, n, dt, run);
      project(end, z, s, n, dt, run);
    }
    run_attention(end, s.q, s.k, s.vt, nullptr, s.tb, s.o, mask, n, dt, run);
  }
  void project(const TriAtt& w, const void* z, const ChainWs& s, int n, int dt, Run& run) const {
    const ptx_single_stage* carry2 = run.carry(2);
    run.launch("triattn_project", [&] {
      return ptx_triattn_project_packed(z, w.ln_w, w.ln_b, w.packed, s.q, s.k, s.vt, nullptr, s.tb, n, w.c, w.heads, ptx_key_pitch(n),
                                        w.transposed, kEps, dt, carry2, run.st);
    });
  }
  const void* attention_output(int n, int64_t es, void* ws) const {
    Cut c{(char*)ws};
    return ChainWs(c, n, out.c_h, start.heads, es).o;
  }
  void output(const TriAtt& w, void* z, const void* o, int n, int dt, Run& run) const {
    const ptx_single_stage* carry3 = run.carry(3);
    run.launch("triattn_output", [&] {
      return ptx_triattn_output_packed(o, z, w.ln_w, w.ln_b, w.packed, z, n, w.c, w.heads, w.transposed, true, kEps, dt,
                                       carry3, run.st);
    });
  }
  // the ending node's output stage and the transition, with the pair bias where one is wanted
  void output_transition(void* z, const void* o, int n, int dt, float* bias, const ptx_single_stage* carry, Run& run) const {
    run.launch("triattn_output_transition", [&] {
      return ptx_triattn_output_transition_carry(o, z, end.ln_w, end.ln_b, tr_packed, tr_ln_w, tr_ln_b, z, n,
                                                 c_z, end.heads, end.transposed, n_factor, kEps, kEps, bias ? pb_ln_w : nullptr,
                                                 bias ? pb_ln_b : nullptr, bias ? pb_w : nullptr, bias,
                                                 bias ? heads : 0, 1, kEps, dt, carry, run.st);
    });
  }

  // bytes single_track() wants as scratch
  int64_t single_bytes(int64_t batch, int n, int64_t es) const {
    Cut c{nullptr};
    SingleWs(c, *this, batch, n, es);
    return c.used;
  }
  struct SingleWs {
    char *y, *qkg, *vt, *o, *h;
    int64_t qkg_plane, vt_plane, o_plane;   // bytes per batch element
    SingleWs(Cut& c, const Block& b, int64_t batch, int n, int64_t es) {
      const int64_t hd = (int64_t)b.heads * b.d, ldt = (n + 31) / 32 * 32;
      qkg_plane = (int64_t)n * 3 * hd * es;
      vt_plane = hd * ldt * es;
      o_plane = (int64_t)n * hd * es;
      y = (char*)c.part(batch * n * b.c_s * es);
      qkg = (char*)c.part(batch * qkg_plane);
      vt = (char*)c.part(batch * vt_plane);
      o = (char*)c.part(batch * o_plane);
      h = (char*)c.part(batch * n * b.hidden * es);
    }
  };
  // The stages of: mid = s + attention(LN(s); bias); s_out = mid + transition(LN(mid)).  The first two, which do not need the
  // pair bias:
  void single_projection(Stages& st, const void* s, at::ScalarType type, int64_t batch, int n, void* ws) const {
    const int dt = code_of(type), hd = heads * d, ldt = (n + 31) / 32 * 32;
    const int64_t es = at::elementSize(type), rows = batch * n;
    Cut c{(char*)ws};
    const SingleWs w(c, *this, batch, n, es);
    check(ptx_single_layernorm_stage(st.add("layernorm"), s, a_ln_w, a_ln_b, w.y, (int)rows, c_s, (float)a_eps, dt), "layernorm");
    for (int64_t b = 0; b < batch; ++b) {
      char* qkg = w.qkg + b * w.qkg_plane;
      check(ptx_single_linear_stage(st.add("linear"), w.y + b * n * c_s * es, w_in, nullptr, b_q, hd, nullptr, qkg, w.vt + b * w.vt_plane, 3 * hd, ldt, n, c_s, 4 * hd, dt, 1), "linear");
    }
  }
  // the others
  void single_track(Stages& st, const void* s, void* mid, void* s_out, const float* bias, at::ScalarType type, int64_t batch, int n,
                    void* ws) const {
    const int dt = code_of(type), hd = heads * d, ldt = (n + 31) / 32 * 32;
    const int64_t es = at::elementSize(type), rows = batch * n;
    Cut c{(char*)ws};
    const SingleWs w(c, *this, batch, n, es);
    for (int64_t b = 0; b < batch; ++b) {
      char* qkg = w.qkg + b * w.qkg_plane;
      check(ptx_single_attention_stage(st.add("single_attention"), qkg, qkg + hd * es, w.vt + b * w.vt_plane, qkg + 2 * hd * es,
                                       bias + b * heads * (int64_t)n * n, 1, w.o + b * w.o_plane, n, heads, d, 3 * hd, ldt, hd,
                                       (float)(1.0 / std::sqrt((double)d)), dt), "single_attention");
    }
    check(ptx_single_linear_stage(st.add("linear"), w.o, w_o, nullptr, nullptr, 0, s, mid, nullptr, c_s, 0,
                                  (int)rows, hd, c_s, dt, 1), "linear");
    check(ptx_single_layernorm_stage(st.add("layernorm"), mid, s_ln_w, s_ln_b, w.y, (int)rows, c_s, (float)s_eps, dt), "layernorm");
    check(ptx_single_linear_stage(st.add("swiglu"), w.y, s_wa, s_wb, nullptr, 0, nullptr,
                                  w.h, nullptr, hidden, 0, (int)rows, c_s, hidden, dt, 1), "swiglu");
    check(ptx_single_linear_stage(st.add("linear"), w.h, s_wo, nullptr, nullptr, 0, mid, s_out, nullptr, c_s, 0,
                                  (int)rows, hidden, c_s, dt, 1), "linear");
  }
};

// Owns the blocks it is given until the call ends: the caller's list is shared, and another thread may
// put a new plan into it while this one runs without the interpreter's lock.
using Blocks = std::vector<std::shared_ptr<Block>>;

// Blocks in sequence on the pair tensors `from` into z (contiguous; the same tensor: in place).  The single track of a block runs underneath the next
// block's pair kernels (see Stages), the last one's in finish().  The blocks may come in several lots: on new weights
// a plan is made while the kernels of the blocks before it run.
struct Call {
  // timer: None, or the dict that gets the launches' times; poison: see Run.
  Call(const optional<Tensor>& s, const Tensor& z, const Tensor& from, const py::list& masks, const py::object& timer, bool poison)
      : z_(z), from_(from), s_(s), masks_(masks_of(masks)), timer_(timer), run_(z) {
    run_.poison = poison;
    run_.timing = !timer.is_none();
    n_ = (int)z.size(-2);
    batch_ = z.numel() / ((int64_t)n_ * n_ * z.size(-1));
  }
  void blocks(const Blocks& list) {
    held_.insert(held_.end(), list.begin(), list.end());
    py::gil_scoped_release nogil;
    at::DeviceGuard dev(z_.device());
    for (const auto& b : list) {
      make_room(*b);   // (one allocation for all of a stack's)
      b->used_on(run_.stream, run_.st);
    }
    for (const auto& b : list) {
      make_room(*b);
      const bool single = b->c_s > 0;
      float* bias = single ? (float*)bias_.data_ptr() : nullptr;
      const int dt = code_of_rows(z_.scalar_type(), b->compute);
      run_.row_stages(n_, b->c_z, b->out.c_h, dt);
      run_.chained = b->chains(run_, n_, dt);
      run_.core_carries = run_.chained && b->core_carries(n_, dt);
      // (a first block's projection rides on its own pair kernels, where nothing waits from a block before)
      const bool early = single && run_.singles.list.empty();
      if (early) b->single_projection(run_.singles, s_now_, s_->scalar_type(), batch_, n_, sws_.data_ptr());
      b->pair_track(from_.data_ptr(), z_, masks_, batch_, n_, ws_.data_ptr(), bias, run_);
      from_ = z_;
      if (single) {
        if (!early) b->single_projection(run_.singles, s_now_, s_->scalar_type(), batch_, n_, sws_.data_ptr());
        b->single_track(run_.singles, s_now_, mid_.data_ptr(), s_out_.data_ptr(), bias, s_->scalar_type(), batch_, n_, sws_.data_ptr());
        s_now_ = s_out_.data_ptr();
      }
    }
  }
  // the new s (what was given, for blocks without a single track)
  optional<Tensor> finish() {
    {
      py::gil_scoped_release nogil;
      at::DeviceGuard dev(z_.device());
      run_.run_rest();
    }
    run_.hand_over(timer_);
    return s_out_.defined() ? optional<Tensor>(s_out_) : s_;
  }

 private:
  void make_room(const Block& b) {
    const int c_h = std::max(b.out.c_h, b.in.c_h), pair_heads = std::max(b.start.heads, b.end.heads);
    const int64_t es = at::elementSize(b.compute);
    enlarge(ws_, std::max(workspace_bytes(n_, c_h, pair_heads, es), chain_bytes(n_, c_h, pair_heads, es)));
    if (b.c_s == 0) return;
    enlarge(bias_, batch_ * b.heads * (int64_t)n_ * n_ * 4);
    enlarge(sws_, b.single_bytes(batch_, n_, (int64_t)s_->element_size()));
    if (s_out_.defined()) return;
    mid_ = at::empty_like(*s_);
    s_out_ = at::empty_like(*s_);
    s_now_ = s_->data_ptr();
  }
  void enlarge(Tensor& t, int64_t bytes) {
    if (t.defined() && t.numel() >= bytes) return;
    if (t.defined()) outgrown_.push_back(t);   // (stages that wait for a launch point into it)
    t = run_.workspace(bytes, z_.options());
  }
  Tensor z_, from_;   // (from_: until the first block has read it)
  optional<Tensor> s_;
  std::vector<Mask> masks_;
  py::object timer_;
  Run run_;
  int n_ = 0;
  int64_t batch_ = 0;
  Blocks held_;
  Tensor ws_, bias_, sws_, mid_, s_out_;
  std::vector<Tensor> outgrown_;
  const void* s_now_ = nullptr;
};

// ---- single updates ----------------------------------------------------------------------------
struct Update : Plan {
  Weights weights;
  at::ScalarType compute;
  optional<TriMul> mul;
  optional<TriAtt> att;
  // transposed: None for a triangle multiplication
  Update(std::shared_ptr<const Guard> guard_, const Module& m, const Tensor& z, at::ScalarType compute_, optional<bool> transposed)
      : Plan(std::move(guard_)), weights(z.device(), current_stream(z)), compute(compute_) {
    if (transposed) att.emplace(m, weights, compute, *transposed);
    else mul.emplace(m, weights, compute);
    require((att ? att->c : mul->c_z) == z.size(-1));
    weights.settle();
    if (att) att->pack(weights, compute);
    else mul->pack(weights, compute);
    weights.done();
    made(weights.stream(), weights.kept);
  }
  // out = [z +] update for every pair tensor of z (contiguous); out may be z
  void run(const Tensor& z, const Tensor& out, const py::list& mask_list, bool add, const py::object& timer, bool poison) const {
    const std::vector<Mask> masks = masks_of(mask_list);
    at::DeviceGuard dev(z.device());
    Run run(z);
    run.poison = poison;
    run.timing = !timer.is_none();
    {
      py::gil_scoped_release nogil;
      used_on(run.stream, run.st);
      run_on(run, z, out, masks, add);
    }
    run.hand_over(timer);
  }

 private:
  void run_on(Run& run, const Tensor& z, const Tensor& out, const std::vector<Mask>& masks, bool add) const {
    const int n = (int)z.size(-2), c = (int)z.size(-1);
    const int64_t batch = n ? z.numel() / ((int64_t)n * n * c) : 0, plane = (int64_t)n * n * c * z.element_size();
    const int dt = code_of_rows(z.scalar_type(), compute);
    const int64_t es = at::elementSize(compute);
    Tensor ws = run.workspace(workspace_bytes(n, mul ? mul->c_h : 0, att ? att->heads : 0, es), z.options());
    static const Mask none;
    for (int64_t b = 0; b < batch; ++b) {
      const Mask& m = masks.empty() ? none : masks[b];
      const char* zb = (const char*)z.data_ptr() + b * plane;
      char* ob = (char*)out.data_ptr() + b * plane;
      if (mul) run_trimul(*mul, zb, m.m, ob, n, add, dt, es, ws.data_ptr(), run);
      else run_triatt(*att, zb, m, ob, n, add, dt, es, ws.data_ptr(), run);
    }
  }
};

template <typename Plan, typename Kind>
std::shared_ptr<Plan> make_plan(std::shared_ptr<Guard> guard, const py::object& module, const Tensor& z, at::ScalarType compute, Kind kind) {
  at::DeviceGuard dev(z.device());
  try {
    return std::make_shared<Plan>(std::move(guard), Module(module), z, compute, kind);
  } catch (const NotCovered&) {
    return nullptr;
  }
}

// ---- LayerNorm ---------------------------------------------------------------------------------
Tensor same_as(const optional<Tensor>& t, const Tensor& x) {
  return t && t->defined() ? t->to(x.options()).contiguous() : Tensor();
}

struct LayerNormFn : torch::autograd::Function<LayerNormFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& input, const optional<Tensor>& weight,
                        const optional<Tensor>& bias, double eps) {
    at::DeviceGuard dev(input.device());
    const Tensor x = input.contiguous(), w = same_as(weight, x), b = same_as(bias, x);
    const int64_t cols = x.size(-1), rows = cols ? x.numel() / cols : 0;
    Tensor y = at::empty_like(x), stats = at::empty({2, rows}, x.options().dtype(at::kFloat));
    float* st = stats.data_ptr<float>();
    check(ptx_layernorm_fwd(ptr(x), ptr(w), ptr(b), ptr(y), st, st + rows, rows, (int)cols, (float)eps, code_of(x.scalar_type()),
                            current_stream(x)), "layernorm");
    ctx->save_for_backward({x, weight ? *weight : Tensor(), stats});
    // (needs_input_grad counts the tensors that were given)
    ctx->saved_data["w"] = weight ? (int64_t)1 : (int64_t)-1;
    ctx->saved_data["b"] = bias ? (int64_t)(weight ? 2 : 1) : (int64_t)-1;
    return y;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &weight = saved[1], &stats = saved[2];
    at::DeviceGuard dev(x.device());
    const Tensor dout = grads[0].to(x.scalar_type()).contiguous();
    const Tensor w = weight.defined() ? same_as(weight, x) : Tensor();
    const int64_t cols = x.size(-1), rows = cols ? x.numel() / cols : 0;
    auto needs = [&](const char* key) {
      const int64_t i = ctx->saved_data[key].toInt();
      return i >= 0 && ctx->needs_input_grad(i);
    };
    const bool need_w = needs("w"), need_b = needs("b");
    Tensor dx = at::empty_like(x), dw, db, ws;
    if (need_w) dw = at::empty({cols}, x.options());
    if (need_b) db = at::empty({cols}, x.options());
    if (need_w || need_b)
      ws = at::empty({ptx_layernorm_bwd_workspace_elems(std::max<int64_t>(rows, 1), (int)cols)}, x.options().dtype(at::kFloat));
    const float* st = stats.data_ptr<float>();
    check(ptx_layernorm_bwd(ptr(dout), ptr(x), st, st + rows, ptr(w), ptr(dx), ptr(dw), ptr(db), (float*)ptr(ws), rows, (int)cols,
                            code_of(x.scalar_type()), current_stream(x)), "layernorm_bwd");
    return {ctx->needs_input_grad(0) ? dx : Tensor(), dw, db, Tensor()};
  }
};

// LayerNorm over the last dimension of a GPU tensor, differentiable.
Tensor layer_norm(const Tensor& x, const optional<Tensor>& weight, const optional<Tensor>& bias, double eps, bool grad) {
  py::gil_scoped_release nogil;
  if (grad) return LayerNormFn::apply(x, weight, bias, eps);
  at::DeviceGuard dev(x.device());
  const Tensor xc = x.contiguous(), w = same_as(weight, xc), b = same_as(bias, xc);
  const int64_t cols = xc.size(-1), rows = cols ? xc.numel() / cols : 0;
  Tensor y = at::empty_like(xc);
  check(ptx_layernorm_fwd(ptr(xc), ptr(w), ptr(b), ptr(y), nullptr, nullptr, rows, (int)cols, (float)eps, code_of(xc.scalar_type()),
                          current_stream(xc)), "layernorm");
  return y;
}

// ---- the attention operator on standard-layout tensors ---------------------------------------------
struct TriAttentionFn : torch::autograd::Function<TriAttentionFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& Q, const Tensor& K, const Tensor& V,
                        const optional<Tensor>& bias1, const Tensor& bias2) {
    at::DeviceGuard dev(Q.device());
    const int64_t B = Q.size(0), N = Q.size(1), S = Q.size(2), H = Q.size(3), D = Q.size(4);
    const auto type = Q.scalar_type();
    const Tensor q = Q.contiguous(), k = K.to(type).contiguous(), v = V.to(type).contiguous();
    const Tensor b2 = bias2.to(type).expand({B, 1, H, S, S}).contiguous();
    const Tensor b1 = bias1 && bias1->defined() ? bias1->to(type).expand({B, N, 1, 1, S}).contiguous() : Tensor();
    Tensor o = at::empty_like(q), m = at::empty({B, N, S, H}, q.options().dtype(at::kFloat));
    Tensor ws = at::empty({ptx_triattn_core_workspace_elems((int)N, (int)S, (int)H)}, q.options());
    check(ptx_triattn_core_fwd(ptr(q), ptr(k), ptr(v), ptr(b1), ptr(b2), ptr(o), (float*)ptr(m), ptr(ws), (int)B, (int)N, (int)S, (int)H,
                               (int)D, code_of(type), current_stream(q)), "triattn_core_fwd");
    ctx->save_for_backward({q, k, v, b1, b2, o, m});
    ctx->saved_data["k"] = K.scalar_type();
    ctx->saved_data["v"] = V.scalar_type();
    ctx->saved_data["b2"] = bias2.scalar_type();
    ctx->saved_data["b2s"] = bias2.sizes().vec();
    ctx->saved_data["b2i"] = (int64_t)(bias1 ? 4 : 3);   // (needs_input_grad counts the tensors that were given)
    return o;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto t = ctx->get_saved_variables();
    const Tensor &q = t[0], &k = t[1], &v = t[2], &b1 = t[3], &b2 = t[4], &o = t[5], &m = t[6];
    at::DeviceGuard dev(q.device());
    const int64_t B = q.size(0), N = q.size(1), S = q.size(2), H = q.size(3), D = q.size(4);
    const Tensor dout = grads[0].to(q.scalar_type()).contiguous();
    const bool want_b2 = ctx->needs_input_grad(ctx->saved_data["b2i"].toInt());
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), db2 = want_b2 ? at::empty_like(b2) : Tensor();
    Tensor delta = at::empty({N * S * H}, q.options().dtype(at::kFloat));
    const int64_t n_parts = want_b2 ? ptx_triattn_core_bwd_partial_elems((int)N, (int)S, (int)H) : 0;
    Tensor parts = n_parts ? at::empty({n_parts}, q.options().dtype(at::kFloat)) : Tensor();
    check(ptx_triattn_core_bwd_sliced(ptr(q), ptr(k), ptr(v), ptr(b1), ptr(b2), ptr(o), (const float*)ptr(m), ptr(dout), ptr(dq), ptr(dk), ptr(dv),
                                      ptr(db2), (float*)ptr(delta), (float*)ptr(parts), (int)B, (int)N, (int)S, (int)H, (int)D,
                                      code_of(q.scalar_type()), current_stream(q)), "triattn_core_bwd");
    if (want_b2) {
      const auto shape = ctx->saved_data["b2s"].toIntVector();
      if (db2.sizes() != c10::IntArrayRef(shape)) db2 = at::sum_to(db2, shape);
      db2 = db2.to(ctx->saved_data["b2"].toScalarType());
    }
    return {dq, dk.to(ctx->saved_data["k"].toScalarType()), dv.to(ctx->saved_data["v"].toScalarType()), Tensor(), db2};
  }
};

Tensor tri_attention(const Tensor& q, const Tensor& k, const Tensor& v, const optional<Tensor>& b1, const Tensor& b2) {
  py::gil_scoped_release nogil;
  return TriAttentionFn::apply(q, k, v, b1, b2);
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.doc() = "native host path of protenix_amd (see csrc/host.cpp)";
  m.def("abi_version", []() { return ptx_version(); });
  py::class_<Guard, std::shared_ptr<Guard>>(m, "Guard")
      .def(py::init<const py::object&, const py::list&, const py::set&>(), py::arg("module"), py::arg("attrs"), py::arg("classes"))
      .def("valid", &Guard::valid);
  py::class_<Plan, std::shared_ptr<Plan>>(m, "Plan").def(py::init<std::shared_ptr<Guard>>()).def("valid", &Plan::valid);
  py::class_<Block, Plan, std::shared_ptr<Block>>(m, "Block");
  m.def("make_block", &make_plan<Block, optional<at::ScalarType>>, py::arg("guard"), py::arg("module"), py::arg("z"), py::arg("compute"),
        py::arg("s_type"), "a plan of the block `module` for pair tensors like z, or None where the Python path is to be taken");
  m.def("make_update", &make_plan<Update, optional<bool>>, py::arg("guard"), py::arg("module"), py::arg("z"), py::arg("compute"),
        py::arg("transposed"), "a plan of one triangle update; transposed: None for a multiplication");
  py::class_<Update, Plan, std::shared_ptr<Update>>(m, "Update")
      .def("run", &Update::run, py::arg("z"), py::arg("out"), py::arg("masks"), py::arg("add"), py::arg("timer") = py::none(),
           py::arg("poison") = false);
  m.def("first_stale", [](const std::vector<std::shared_ptr<Plan>>& blocks) {
    for (size_t i = 0; i < blocks.size(); ++i)
      if (!blocks[i]->valid()) return (int64_t)i;
    return (int64_t)-1;
  }, "index of the first block whose weights are no longer the module's, or -1");
  py::class_<Call>(m, "Call")
      .def(py::init<const optional<Tensor>&, const Tensor&, const Tensor&, const py::list&, const py::object&, bool>(), py::arg("s"),
           py::arg("z"), py::arg("from_"), py::arg("masks"), py::arg("timer") = py::none(), py::arg("poison") = false)
      .def("blocks", &Call::blocks)
      .def("finish", &Call::finish);
  py::class_<Mark, std::shared_ptr<Mark>>(m, "Mark").def("elapsed_time", &Mark::elapsed_time);
  m.def("layer_norm", &layer_norm);
  m.def("tri_attention", &tri_attention);
}
