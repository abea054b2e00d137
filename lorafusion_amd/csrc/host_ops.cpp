// Host side of the fused linears, the norm and the activation: allocation, launch through the C ABI, and the autograd nodes.
//
// A LoRA linear of a few hundred tokens runs on the GPU in well under 100 us, and Python took longer than that to get it
// there: its forward and backward are seven launches and nine allocations behind an autograd.Function whose backward runs
// on the engine's own thread, where every bytecode is cold and the interpreter lock changes hands (backward body 65 us
// there, 31 us when called from a warm loop).  Here one call validates, allocates and launches a forward, and the
// backward is a node of the engine that needs no interpreter at all: forward + backward of 100 x 1024 x 1024 went from 184 to
// 82 us of host time (torch.nn.functional.linear: 107), of four packed adapters from 259 to 130.  Argument rules, errors, saved tensors and results are
// those of the Python layer (lorafusion/ops/lora_v1.py:173-297, multi_lora.py:602-830); kernels are reached through
// lorafusion_hip.h only.
#include <ATen/ATen.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <cstring>
#include <optional>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/lorafusion_hip.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

namespace {

template <typename... A>
[[noreturn]] void bad_value(const A&... a) {
  std::ostringstream s;
  (s << ... << a);
  throw py::value_error(s.str());
}

class NotImplemented : public py::builtin_exception {
 public:
  using builtin_exception::builtin_exception;
  void set_error() const override { PyErr_SetString(PyExc_NotImplementedError, what()); }
};
// The kernels read the values alone: a forward-mode tangent of an operand would be lost without a word.
template <typename... L>
void refuse_tangents(const L&... operands) {
  if ((torch::autograd::isFwGradDefined(operands) || ...))
    throw NotImplemented("the fused LoRA, norm and activation functions have no forward-mode derivative.");
}
void refuse_tangents_of(const std::vector<Tensor>& t) {
  for (const Tensor& v : t) refuse_tangents(v);
}

void check(int rc, const char* what) {
  if (rc != LF_OK) throw std::runtime_error(std::string(what) + " failed: " + lf_strerror(rc) + " (code " + std::to_string(rc) + ")");
}

const char* dtype_name(at::ScalarType t) {   // torch's own spelling, for messages
  switch (t) {
    case at::kBFloat16: return "torch.bfloat16";
    case at::kHalf: return "torch.float16";
    case at::kFloat: return "torch.float32";
    case at::kDouble: return "torch.float64";
    case at::kByte: return "torch.uint8";
    case at::kChar: return "torch.int8";
    case at::kShort: return "torch.int16";
    case at::kInt: return "torch.int32";
    case at::kLong: return "torch.int64";
    case at::kBool: return "torch.bool";
    default: return c10::toString(t);
  }
}
std::string shape_name(at::IntArrayRef s) {   // a Python tuple
  std::ostringstream o;
  o << '(';
  for (size_t i = 0; i < s.size(); i++) o << (i ? ", " : "") << s[i];
  o << (s.size() == 1 ? ",)" : ")");
  return o.str();
}

int dtype_id(at::ScalarType t) {
  if (t == at::kBFloat16) return LF_BF16;
  if (t == at::kHalf) return LF_F16;
  bad_value("Unsupported dtype: ", dtype_name(t), "; expected torch.bfloat16 or torch.float16.");
}
void require_gpu(const Tensor& t, const char* name) {
  if (!t.is_cuda()) bad_value(name, " must live on the GPU (got device ", t.device().str(), "); the HIP kernels have no CPU path.");
}

const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void* mptr(const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }

struct Ptrs {
  const void* v[LF_MAX_SEG];
  explicit Ptrs(const std::vector<Tensor>& t) {
    for (size_t i = 0; i < t.size() && i < LF_MAX_SEG; i++) v[i] = t[i].const_data_ptr();
  }
};

// (a host tensor has no stream: the nodes run on host tensors where the kernels are stood in for)
void* stream_of(const Tensor& t) { return t.is_cuda() ? (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream() : nullptr; }

bool is_bits(const Tensor& mask, int64_t K) { return mask.defined() && mask.scalar_type() == at::kByte && mask.size(-1) * 8 == K; }
int64_t rows_of(const Tensor& t) {
  if (t.size(-1) == 0) throw std::runtime_error("the number of rows of a tensor of shape " + shape_name(t.sizes()) + " is not defined.");
  return t.numel() / t.size(-1);
}

Tensor scratch(size_t bytes, const Tensor& like) {
  return bytes ? at::empty({(int64_t)bytes}, like.options().dtype(at::kByte)) : Tensor();
}

lf_routing single_routing(int rank, float scale, float p) {
  lf_routing r;
  std::memset(&r, 0, sizeof r);
  r.n_seg = 1;
  r.block_size_m = 128;
  r.scale = scale;
  r.p = p;
  r.seg_rank[0] = rank;
  return r;
}
int round_rank(int r) { return (r + 15) / 16 * 16; }

// The base weight of a call: a 16-bit tensor [N, K], or NF4 codes with the tensors of their quant state (whose owner the caller holds).
struct Weight {
  Tensor w;
  bool nf4 = false;
  lf_nf4_weight c{};
};

// NF4, for a backward: a Python callable, codes -> (address of their lf_nf4_weight, its owner).  The struct holds addresses, and a
// weight may move between forward and backward (`p.data = ...` of an offloaded or gathered parameter, a hook that unpacks a
// copy, a quant state moved along with it): it is made from what codes and state are when the backward runs.
using PyRef = std::shared_ptr<py::object>;   // (let go of under the interpreter's lock, by whichever thread)
PyRef py_ref(py::handle h) {
  if (h.is_none()) return nullptr;
  return PyRef(new py::object(py::reinterpret_borrow<py::object>(h)), [](py::object* o) {
    py::gil_scoped_acquire gil;
    delete o;
  });
}
PyRef resolve_nf4(const py::object& of, const Tensor& codes, lf_nf4_weight& c) {
  py::gil_scoped_acquire gil;
  const py::tuple t = of(codes);
  c = *(const lf_nf4_weight*)t[0].cast<uintptr_t>();
  return py_ref(t[1]);
}

struct Forward { Tensor y, s, mask, dense; };

// Y (of shape y_sizes) and S for x [.., K] contiguous; the mask is drawn when a seed is given.
Forward run_forward(const Tensor& x, Weight& w, const std::vector<Tensor>& a, const std::vector<Tensor>& b, const lf_routing& r, int R, int N,
                    const Tensor& mask, std::optional<uint64_t> seed, bool packed, const Tensor& bias, bool keep_dense, at::IntArrayRef y_sizes) {
  const int M = (int)rows_of(x), K = (int)x.size(-1), dt = dtype_id(x.scalar_type());
  Forward f;
  f.y = at::empty(y_sizes, x.options());
  f.s = at::empty({M, R}, x.options());
  f.mask = mask;
  if (seed) f.mask = packed ? at::empty({M, K / 8}, x.options().dtype(at::kByte)) : at::empty({M, K}, x.options().dtype(at::kBool));
  if (keep_dense) f.dense = at::empty({N, K}, x.options());
  const size_t n = lf_workspace_bytes(w.nf4 && !keep_dense && !seed ? LF_OP_NF4_FWD : LF_OP_FWD, M, N, K, R, &r);
  // (a mask drawn over NF4 codes: the weight is dequantised here, in front of the forward's own workspace, and the 16-bit forward draws)
  const size_t head = w.nf4 && seed && !keep_dense ? ((size_t)N * K * 2 + 255) & ~(size_t)255 : 0;
  const Tensor ws = scratch(head + n, x);
  const Ptrs pa(a), pb(b);
  const int d = dt | (is_bits(f.mask, K) ? LF_MASK_BITS : 0);
  void* st = stream_of(x);
  if (seed) {
    const void* dense = ptr(w.w);
    if (w.nf4) {
      void* to = keep_dense ? mptr(f.dense) : mptr(ws);
      check(lf_nf4_dequant(w.c.packed, w.c.absmax, w.c.code2, w.c.absmax2, w.c.offset, to, (int64_t)N * K, w.c.blocksize, w.c.blocksize2, dt, st), "lf_nf4_dequant");
      dense = to;
    }
    check(lf_lora_fwd_seeded(ptr(x), dense, ptr(bias), (uint8_t*)mptr(f.mask), pa.v, pb.v, mptr(f.y), mptr(f.s), n ? (char*)mptr(ws) + head : nullptr, n, M, N, K, R,
                             &r, *seed, d, st), "lf_lora_fwd_seeded");
  } else if (w.nf4) {
    lf_nf4_weight c = w.c;
    c.dense = mptr(f.dense);
    c.dense_valid = 0;
    check(lf_nf4_lora_fwd(ptr(x), &c, ptr(bias), (const uint8_t*)ptr(f.mask), pa.v, pb.v, mptr(f.y), mptr(f.s), mptr(ws), n, M, N, K, R, &r, d, st),
          "lf_nf4_lora_fwd");
  } else {
    check(lf_lora_fwd(ptr(x), ptr(w.w), ptr(bias), (const uint8_t*)ptr(f.mask), pa.v, pb.v, mptr(f.y), mptr(f.s), mptr(ws), n, M, N, K, R, &r, d, st),
          "lf_lora_fwd");
  }
  return f;
}

struct Backward { Tensor dx; std::vector<Tensor> da, db; };

Backward run_backward(const Tensor& dy, const Tensor& x, const Weight& w, const std::vector<Tensor>& a, const std::vector<Tensor>& b, const Tensor& s,
                      const lf_routing& r, int R, const Tensor& mask, const Tensor& dense, bool need_dx, at::IntArrayRef dx_sizes) {
  const int M = (int)rows_of(dy), N = (int)dy.size(-1), K = (int)x.size(-1);
  Backward g;
  if (need_dx) g.dx = at::empty(dx_sizes, dy.options());
  for (const Tensor& t : a) g.da.push_back(at::empty({t.size(0), K}, dy.options()));
  for (const Tensor& t : b) g.db.push_back(at::empty({N, t.size(1)}, dy.options()));
  // no weight-sized head in the workspace when the dequantised weight is handed over, or not needed at all (no dX)
  const bool lean = !w.nf4 || dense.defined() || !need_dx;
  const size_t n = lf_workspace_bytes(lean ? LF_OP_BWD : LF_OP_NF4_BWD, M, N, K, R, &r);
  const size_t ds = ((size_t)M * R * 2 + 255) & ~(size_t)255;   // dS in front of the workspace
  const Tensor ws = scratch(ds + n, dy);
  const Ptrs pa(a), pb(b), oa(g.da), ob(g.db);
  const int d = dtype_id(dy.scalar_type()) | (is_bits(mask, K) ? LF_MASK_BITS : 0);
  char* wp = (char*)mptr(ws);
  void* st = stream_of(dy);
  void* const* da = const_cast<void* const*>(oa.v);
  void* const* db = const_cast<void* const*>(ob.v);
  if (w.nf4) {
    lf_nf4_weight c = w.c;
    c.dense = const_cast<void*>(ptr(dense));
    c.dense_valid = dense.defined();
    check(lf_nf4_lora_bwd(ptr(dy), ptr(x), &c, (const uint8_t*)ptr(mask), ptr(s), pa.v, pb.v, mptr(g.dx), da, db, wp, wp + ds, n, M, N, K, R, &r, d, st),
          "lf_nf4_lora_bwd");
  } else {
    check(lf_lora_bwd(ptr(dy), ptr(x), ptr(w.w), (const uint8_t*)ptr(mask), ptr(s), pa.v, pb.v, mptr(g.dx), da, db, wp, wp + ds, n, M, N, K, R, &r, d, st),
          "lf_lora_bwd");
  }
  return g;
}

// ------------------------------------------------------------------------------------------- autograd

bool wants_grad(std::initializer_list<Tensor> t, const std::vector<Tensor>& a = {}, const std::vector<Tensor>& b = {}) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor& v : t) if (v.defined() && v.requires_grad()) return true;
  return torch::autograd::any_variable_requires_grad(a) || torch::autograd::any_variable_requires_grad(b);
}

std::vector<SavedVariable> save_all(const std::vector<Tensor>& t) {
  std::vector<SavedVariable> s;
  s.reserve(t.size());
  for (const Tensor& v : t) s.emplace_back(v, false);
  return s;
}
std::vector<Tensor> unpack_all(std::vector<SavedVariable>& s) {
  std::vector<Tensor> t;
  t.reserve(s.size());
  for (SavedVariable& v : s) t.push_back(v.unpack());
  return t;
}

// the incoming gradient as a contiguous tensor (zeros where none came)
Tensor incoming(const variable_list& g, size_t i, at::IntArrayRef sizes, const at::TensorOptions& o) {
  return i < g.size() && g[i].defined() ? g[i].contiguous() : at::zeros(sizes, o);
}

// y = x W^T + scale_i (drop(x) A_i^T) B_i^T + bias; with `act` the input is silu(gate) * up and its gradient goes on to them.
struct LoraBackward : Node {
  SavedVariable x, w, mask, s, dense;
  std::vector<SavedVariable> a, b, act;   // act: the merged gate/up tensor, or gate and up
  PyRef nf4;                              // `w` holds NF4 codes: what makes their struct
  lf_routing r{};
  std::vector<Tensor> tables;
  int R = 0;
  std::vector<int64_t> in_sizes, y_sizes;  // of the differentiable input(s) and of y
  at::TensorOptions options;
  bool has_act = false;
  std::string label;

  std::string name() const override { return label; }
  void release_variables() override {
    PyRef state;   // (let go of behind the lock: that takes the interpreter's)
    std::lock_guard<std::mutex> lock(mutex_);
    for (SavedVariable* v : {&x, &w, &mask, &s, &dense}) v->reset_data();
    for (auto* l : {&a, &b, &act}) for (SavedVariable& v : *l) v.reset_data();
    tables.clear();
    state.swap(nf4);
  }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    const Tensor xs = x.unpack(), ms = mask.unpack(), ss = s.unpack(), dn = dense.unpack();
    const std::vector<Tensor> as = unpack_all(a), bs = unpack_all(b), in = unpack_all(act);
    Weight weight;
    weight.w = w.unpack();
    weight.nf4 = nf4 != nullptr;
    const size_t n_in = has_act ? in.size() : 1;
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard device(xs.device());
    const Tensor dy = incoming(grads, 0, y_sizes, options);
    bool need = task_should_compute_output(0) || (n_in > 1 && task_should_compute_output(1));
    // (no struct where nothing will be dequantised: the weight is at hand, or not needed)
    const PyRef owner = weight.nf4 && need && !dn.defined() ? resolve_nf4(*nf4, weight.w, weight.c) : nullptr;
    const int64_t K = xs.size(-1), M = rows_of(xs);
    const std::vector<int64_t> flat = {M, K};
    Backward g = run_backward(dy, xs.contiguous(), weight, as, bs, ss, r, R, ms, dn, need, has_act ? at::IntArrayRef(flat) : at::IntArrayRef(in_sizes));
    variable_list out;
    out.reserve(n_in + as.size() + bs.size());
    if (!has_act) {
      out.push_back(g.dx);
    } else if (!need) {
      out.resize(n_in);
    } else {
      const int dt = dtype_id(xs.scalar_type());
      void* st = stream_of(xs);
      if (n_in == 1) {
        // gate and up are the halves of one tensor, and so are their gradients
        const Tensor dg = at::empty(in_sizes, options);
        const char* gp = (const char*)in[0].const_data_ptr();
        char* dp = (char*)dg.mutable_data_ptr();
        check(lf_silu_mul_bwd(ptr(g.dx), gp, gp + K * 2, dp, dp + K * 2, (int)M, (int)K, K, 2 * K, 2 * K, 2 * K, 2 * K, dt, st), "lf_silu_mul_bwd");
        out.push_back(dg);
      } else {
        const Tensor dg = at::empty(in_sizes, options), du = at::empty(in_sizes, options);
        auto ld = [&](const Tensor& t) { return M > 1 ? t.stride(0) : K; };
        check(lf_silu_mul_bwd(ptr(g.dx), ptr(in[0]), ptr(in[1]), mptr(dg), mptr(du), (int)M, (int)K, K, ld(in[0]), ld(in[1]), K, K, dt, st),
              "lf_silu_mul_bwd");
        out.push_back(dg);
        out.push_back(du);
      }
    }
    for (Tensor& t : g.da) out.push_back(std::move(t));
    for (Tensor& t : g.db) out.push_back(std::move(t));
    out.resize(num_outputs());   // (none for the base weight and the bias)
    return out;
  }
};

// Make `y` the output of a LoraBackward whose inputs are `edges` (the differentiable input(s), then A_i, then B_i, then base weight
// and bias, as the caller holds them).  x, w, a, b: what the kernels read -- the same tensors where those are contiguous.
void attach(const Tensor& y, const variable_list& edges, const Tensor& x, const Tensor& w, const PyRef& nf4, const std::vector<Tensor>& a,
            const std::vector<Tensor>& b, const Tensor& mask, const Tensor& s, const Tensor& dense, const std::vector<Tensor>& act,
            const lf_routing& r, const std::vector<Tensor>& tables, int R, const char* label) {
  std::shared_ptr<LoraBackward> n(new LoraBackward(), torch::autograd::deleteNode);
  n->set_next_edges(torch::autograd::collect_next_edges(edges));
  n->x = SavedVariable(x, false);
  n->w = SavedVariable(w, false);
  n->mask = SavedVariable(mask, false);
  n->s = SavedVariable(s, false);
  n->dense = SavedVariable(dense, false);
  n->a = save_all(a);
  n->b = save_all(b);
  n->act = save_all(act);
  n->has_act = !act.empty();
  n->nf4 = nf4;
  n->r = r;
  n->tables = tables;
  n->R = R;
  n->in_sizes = edges[0].sizes().vec();
  n->y_sizes = y.sizes().vec();
  n->options = y.options();
  n->label = label;
  torch::autograd::set_history(y, n);
}

// ------------------------------------------------------------------------------------------- one adapter

void check_dims(int64_t M, int64_t N, int64_t K) {
  if (M <= 0) bad_value("M must be positive, got ", M, ".");
  if (K % 128 != 0) bad_value("K must be a multiple of 128, got ", K, ".");
  if (N % 128 != 0) bad_value("N must be a multiple of 128, got ", N, ".");
}
void check_rank(int64_t r) {
  if (r < 8 || r % 8 != 0 || r > 128) bad_value("LoRA rank must be a multiple of 8 in [8, 128], got ", r, ".");
}
// the caller's keep-mask as [M, K] bytes or [M, K / 8] bits
Tensor checked_mask(const Tensor& mask, int64_t M, int64_t K) {
  if (mask.scalar_type() != at::kBool && mask.scalar_type() != at::kByte)
    bad_value("dropout_mask must be a bool (or uint8) tensor, but got ", dtype_name(mask.scalar_type()), ".");
  const Tensor m = mask.reshape({M, -1});
  if (m.size(1) != K && !(m.scalar_type() == at::kByte && m.size(1) * 8 == K))
    bad_value("dropout_mask must have shape ", shape_name({M, K}), ", but got ", shape_name(m.sizes()), ".");
  if (!m.is_contiguous()) bad_value("dropout_mask must be contiguous.");
  require_gpu(m, "dropout_mask");
  return m;
}
// (read three times -- rank-r forward, dA, dX: an eighth of the bytes each)
Tensor packed_mask(const Tensor& m, int64_t K) {
  if (is_bits(m, K)) return m;
  const int64_t M = m.size(0);
  Tensor bits = at::empty({M, K / 8}, m.options().dtype(at::kByte));
  check(lf_mask_pack((const uint8_t*)ptr(m), (uint8_t*)mptr(bits), (int)M, (int)K, stream_of(m)), "lf_mask_pack");
  return bits;
}

// fused_linear_lora (lorafusion/ops/lora_v1.py:284-297).  seed: set when a mask is to be drawn.
Tensor linear_lora(const Tensor& x, const Tensor& w, const Tensor& a, const Tensor& b, double alpha, double p, std::optional<uint64_t> seed,
                   const OptTensor& bias_, const OptTensor& mask_) {
  if (x.dim() != 3 && x.dim() != 2) bad_value("Expected x to have 2 or 3 dimensions, got ", x.dim(), ".");
  require_gpu(w, "linear_w");
  const Tensor* named[] = {&x, &a, &b};
  const char* names[] = {"x", "lora_a", "lora_b"};
  for (int i = 0; i < 3; i++) {
    require_gpu(*named[i], names[i]);
    if (named[i]->scalar_type() != x.scalar_type())
      bad_value(names[i], " must have dtype ", dtype_name(x.scalar_type()), ", but got ", dtype_name(named[i]->scalar_type()), ".");
  }
  if (w.scalar_type() != x.scalar_type()) bad_value("linear_w must have dtype ", dtype_name(x.scalar_type()), ", but got ", dtype_name(w.scalar_type()), ".");
  dtype_id(x.scalar_type());
  const int64_t K = x.size(-1), M = K > 0 ? rows_of(x) : 0;
  if (w.dim() != 2 || w.size(1) != K) bad_value("linear_w must have shape [N, ", K, "], but got ", shape_name(w.sizes()), ".");
  const int64_t N = w.size(0);
  if (a.dim() != 2 || a.size(1) != K) bad_value("lora_a must have shape [r, ", K, "], but got ", shape_name(a.sizes()), ".");
  const int64_t rank = a.size(0);
  if (b.dim() != 2 || b.size(0) != N || b.size(1) != rank) bad_value("lora_b must have shape [", N, ", ", rank, "], but got ", shape_name(b.sizes()), ".");
  const Tensor bias = bias_.value_or(Tensor());
  if (bias.defined() && (bias.dim() != 1 || bias.size(0) != N || bias.scalar_type() != x.scalar_type()))
    bad_value("linear_bias must have shape [", N, "] and dtype ", dtype_name(x.scalar_type()), ".");
  check_dims(M, N, K);
  check_rank(rank);
  if (!(p >= 0.0 && p < 1.0)) bad_value("dropout_p must be in [0, 1), got ", p, ".");
  refuse_tangents(x, w, a, b, bias);

  Tensor mask;   // (as autograd sees it: an alias made below would not share its version counter)
  if (p > 0 && !seed) mask = checked_mask(*mask_, M, K);
  Weight wt;
  const int R = round_rank((int)rank);
  const lf_routing r = single_routing((int)rank, (float)alpha, (float)p);
  Tensor xs;
  std::vector<Tensor> as, bs;
  Forward f;
  {
    const at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard device(x.device());
    xs = x.contiguous(), wt.w = w.contiguous(), as = {a.contiguous()}, bs = {b.contiguous()};
    if (mask.defined()) mask = packed_mask(mask, K);
    std::vector<int64_t> ys = x.sizes().vec();
    ys.back() = N;
    f = run_forward(xs, wt, as, bs, r, R, (int)N, mask, p > 0 ? seed : std::nullopt, true, bias.defined() ? bias.contiguous() : bias, false, ys);
  }
  // (a base weight or bias that requires a gradient makes y differentiable; it receives none)
  if (wants_grad({x, a, b, w, bias})) attach(f.y, {x, a, b, w, bias}, xs, wt.w, nullptr, as, bs, f.mask, f.s, Tensor(), {}, r, {}, R, "FusedLinearLoRABackward");
  return f.y;
}

// ------------------------------------------------------------------------------------------- calls of the Python layer

lf_routing routing_at(uintptr_t addr) { return *(const lf_routing*)addr; }
Weight weight_at(const OptTensor& w, uintptr_t nf4) {
  Weight t;
  t.w = w.value_or(Tensor());
  t.nf4 = nf4 != 0;
  if (t.nf4) t.c = *(const lf_nf4_weight*)nf4;
  return t;
}

std::tuple<Tensor, Tensor, OptTensor, OptTensor> py_forward(const Tensor& x, const OptTensor& w, uintptr_t nf4, int N, const std::vector<Tensor>& a,
                                                           const std::vector<Tensor>& b, uintptr_t routing, int R, const OptTensor& mask,
                                                           std::optional<uint64_t> seed, bool packed, const OptTensor& bias, bool keep_dense) {
  refuse_tangents(x, w, bias);
  refuse_tangents_of(a);
  refuse_tangents_of(b);
  const at::AutoDispatchBelowADInplaceOrView below;
  const c10::DeviceGuard device(x.device());
  Weight wt = weight_at(w, nf4);
  Forward f = run_forward(x, wt, a, b, routing_at(routing), R, N, mask.value_or(Tensor()), seed, packed, bias.value_or(Tensor()), keep_dense, {rows_of(x), N});
  return {f.y, f.s, f.mask.defined() ? OptTensor(f.mask) : std::nullopt, f.dense.defined() ? OptTensor(f.dense) : std::nullopt};
}

std::tuple<OptTensor, std::vector<Tensor>, std::vector<Tensor>> py_backward(const Tensor& dy, const Tensor& x, const OptTensor& w, uintptr_t nf4,
                                                                           const std::vector<Tensor>& a, const std::vector<Tensor>& b, const Tensor& s,
                                                                           uintptr_t routing, int R, const OptTensor& mask, const OptTensor& dense,
                                                                           bool need_dx) {
  const at::AutoDispatchBelowADInplaceOrView below;
  const c10::DeviceGuard device(dy.device());
  const Weight wt = weight_at(w, nf4);
  Backward g = run_backward(dy, x, wt, a, b, s, routing_at(routing), R, mask.value_or(Tensor()), dense.value_or(Tensor()), need_dx, x.sizes());
  return {g.dx.defined() ? OptTensor(g.dx) : std::nullopt, g.da, g.db};
}

// `y` [M, N] as the differentiable result of a linear over `inputs` (x; or the merged gate/up tensor; or gate and up), of shape
// inputs[0].shape[:-1] + [N].  x: the contiguous [.., K] input of the kernels; a, b: as the caller holds them.
// others: operands that make y differentiable where they require a gradient, and receive none (base weight, bias).
// nf4: None (or 0), or what makes the struct of the codes `w`.
Tensor py_attach(const Tensor& y, const std::vector<Tensor>& inputs, const Tensor& x, const OptTensor& w, const py::object& nf4_of,
                 const std::vector<OptTensor>& others, const std::vector<Tensor>& a, const std::vector<Tensor>& b, const OptTensor& mask, const Tensor& s, const OptTensor& dense,
                 const std::vector<Tensor>& act, uintptr_t routing, const std::vector<Tensor>& tables, int R, const char* label) {
  const PyRef nf4 = PyCallable_Check(nf4_of.ptr()) ? py_ref(nf4_of) : nullptr;
  const py::gil_scoped_release nogil;
  Tensor out;
  std::vector<Tensor> as, bs;
  std::vector<int64_t> ys = inputs[0].sizes().vec();
  ys.back() = y.size(-1);
  {
    const at::AutoDispatchBelowADInplaceOrView below;   // (a plain alias: not a view that autograd would track)
    out = ys.size() == 2 ? y : y.view(ys);
    for (const Tensor& t : a) as.push_back(t.contiguous());
    for (const Tensor& t : b) bs.push_back(t.contiguous());
  }
  variable_list edges = inputs;
  edges.insert(edges.end(), a.begin(), a.end());
  edges.insert(edges.end(), b.begin(), b.end());
  refuse_tangents_of(edges);
  for (const OptTensor& t : others) edges.push_back(t.value_or(Tensor()));
  if (at::GradMode::is_enabled() && torch::autograd::any_variable_requires_grad(edges))
    attach(out, edges, x, w.value_or(Tensor()), nf4, as, bs, mask.value_or(Tensor()), s, dense.value_or(Tensor()), act, routing_at(routing), tables, R, label);
  return out;
}

// the adapters of a packed batch against its routing (messages of the Python layer)
void check_adapters(const std::vector<Tensor>& a, const std::vector<Tensor>& b, const std::vector<int64_t>& ranks, int64_t K, int64_t N, const Tensor& x) {
  auto one = [&](const Tensor& t, const char* name, int64_t rows, int64_t cols) {
    if (t.dim() != 2) bad_value(name, " must be a 2D tensor, but got ", t.dim(), "D.");
    if (t.scalar_type() != x.scalar_type()) bad_value(name, " must have dtype ", dtype_name(x.scalar_type()), ", but got ", dtype_name(t.scalar_type()), ".");
    require_gpu(t, name);
    if (t.size(0) != rows || t.size(1) != cols)
      bad_value(name, " must have shape [", rows, ", ", cols, "], but got ", shape_name(t.sizes()), ".");
  };
  if (a.size() != ranks.size() || b.size() != ranks.size()) bad_value("the batch info has ", ranks.size(), " adapter segments, got ", a.size(), " lora_a and ", b.size(), " lora_b.");
  for (size_t i = 0; i < a.size(); i++) one(a[i], "lora_a", ranks[i], K);
  for (size_t i = 0; i < b.size(); i++) one(b[i], "lora_b", N, ranks[i]);
}

// The operands of a packed batch over a 16-bit base weight against each other and the batch's routing (`rows` of it), in one call.  True:
// the kernels can read all of them as they lie.
bool check_multi(const Tensor& px, const Tensor& w, const std::vector<Tensor>& a, const std::vector<Tensor>& b, const std::vector<int64_t>& ranks, int64_t rows,
                 const OptTensor& bias) {
  if (px.dim() == 3) {
    if (px.size(0) != 1) bad_value("currently, we only support batch size 1 for multi-linear LoRA");
  } else if (px.dim() != 2) {
    bad_value("padded_x must be a 3D tensor, but got ", px.dim());
  }
  const int64_t M = px.size(-2), K = px.size(-1);
  if (M != rows) bad_value("padded_x has ", M, " rows but the batch info covers ", rows, ".");
  if (w.dim() != 2 || w.size(1) != K || w.scalar_type() != px.scalar_type())
    bad_value("linear_w must have shape [N, ", K, "] and dtype ", dtype_name(px.scalar_type()), ".");
  const int64_t N = w.size(0);
  require_gpu(px, "padded_x");
  dtype_id(px.scalar_type());
  check_dims(M, N, K);
  check_adapters(a, b, ranks, K, N, px);
  if (bias && (bias->dim() != 1 || bias->size(0) != N || bias->scalar_type() != px.scalar_type()))
    bad_value("linear_bias must have shape [", N, "] and dtype ", dtype_name(px.scalar_type()), ".");
  bool plain = px.is_contiguous() && w.is_contiguous() && (!bias || bias->is_contiguous());
  for (const Tensor& t : a) plain = plain && t.is_contiguous();
  for (const Tensor& t : b) plain = plain && t.is_contiguous();
  return plain;
}

// ------------------------------------------------------------------------------------------- RMSNorm, SiLU-multiply

struct RMSNormBackward : Node {
  SavedVariable x, w, rstd;
  std::vector<int64_t> sizes;
  std::string name() const override { return "RMSNormFunctionBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    x.reset_data(), w.reset_data(), rstd.reset_data();
  }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    const Tensor xv = x.unpack(), wv = w.unpack(), rs = rstd.unpack();
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard device(xv.device());
    const int M = (int)rows_of(xv), H = (int)xv.size(-1);
    const Tensor dy = incoming(grads, 0, sizes, xv.options());
    const Tensor dx = at::empty(sizes, xv.options());
    const bool need_dw = task_should_compute_output(1);
    const Tensor dw = need_dw ? (M > 0 ? at::empty({H}, xv.options()) : at::zeros({H}, xv.options())) : Tensor();
    if (M > 0) {
      const size_t n = need_dw ? lf_rmsnorm_bwd_workspace(M, H) : 0;
      const Tensor ws = scratch(n, xv);
      check(lf_rmsnorm_bwd(ptr(dy), ptr(xv), ptr(wv), (const float*)ptr(rs), mptr(dx), mptr(dw), M, H, dtype_id(xv.scalar_type()), mptr(ws), n, stream_of(xv)),
            "lf_rmsnorm_bwd");
    }
    return {dx, dw};
  }
};

Tensor rms_norm(const Tensor& x, const Tensor& w, double eps) {
  require_gpu(x, "x");
  require_gpu(w, "weight");
  if (w.scalar_type() != x.scalar_type()) bad_value("RMSNorm weight dtype ", dtype_name(w.scalar_type()), " differs from the input's ", dtype_name(x.scalar_type()), ".");
  const int64_t H = x.size(-1);
  if (w.dim() != 1 || w.size(0) != H) bad_value("RMSNorm weight shape ", shape_name(w.sizes()), " does not match the hidden size ", H, ".");
  refuse_tangents(x, w);
  Tensor xs, ws, y, rstd;
  {
    const at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard device(x.device());
    xs = x.contiguous(), ws = w.contiguous();
    const int64_t M = rows_of(xs);
    y = at::empty(x.sizes(), x.options());
    rstd = at::empty({M}, x.options().dtype(at::kFloat));
    if (M > 0)
      check(lf_rmsnorm_fwd(ptr(xs), ptr(ws), mptr(y), (float*)mptr(rstd), (int)M, (int)H, (float)eps, dtype_id(x.scalar_type()), stream_of(x)), "lf_rmsnorm_fwd");
  }
  if (wants_grad({x, w})) {
    std::shared_ptr<RMSNormBackward> n(new RMSNormBackward(), torch::autograd::deleteNode);
    n->set_next_edges(torch::autograd::collect_next_edges(x, w));
    n->x = SavedVariable(xs, false);
    n->w = SavedVariable(ws, false);
    n->rstd = SavedVariable(rstd, false);
    n->sizes = x.sizes().vec();
    torch::autograd::set_history(y, n);
  }
  return y;
}

// [M, I] rows with unit column stride (a copy only where the kernels could not read the tensor as it lies), and their stride
std::pair<Tensor, int64_t> rows_view(const Tensor& t) {
  Tensor t2 = t.dim() == 2 ? t : t.reshape({-1, t.size(-1)});
  if (t2.stride(1) != 1 || t2.stride(0) % 8 != 0 || (uintptr_t)t2.const_data_ptr() % 16 != 0 || (t2.size(0) > 1 && t2.stride(0) < t2.size(1))) t2 = t2.contiguous();
  return {t2, t2.size(0) > 1 ? t2.stride(0) : std::max(t2.stride(0), t2.size(1))};
}

// c = silu(a) * b; merged: a and b are the halves of one tensor
struct SiLUMulBackward : Node {
  SavedVariable a, b;
  std::vector<int64_t> sizes, c_sizes;   // of the input(s) and of c
  bool merged = false;
  std::string name() const override { return merged ? "SiLUMulMergedFunctionBackward" : "SiLUMulFunctionBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    a.reset_data(), b.reset_data();
  }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    const Tensor av = a.unpack(), bv = b.unpack();
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard device(av.device());
    const Tensor dc0 = grads[0].defined() ? grads[0] : at::zeros(c_sizes, av.options());
    const auto [dc, lddc] = rows_view(dc0);
    const int M = (int)dc.size(0), I = (int)dc.size(1), dt = dtype_id(av.scalar_type());
    void* st = stream_of(av);
    if (merged) {
      const Tensor dg = at::empty(sizes, av.options());
      const char* gp = (const char*)av.const_data_ptr();
      char* dp = (char*)dg.mutable_data_ptr();
      if (M > 0) check(lf_silu_mul_bwd(ptr(dc), gp, gp + 2 * (int64_t)I, dp, dp + 2 * (int64_t)I, M, I, lddc, 2 * I, 2 * I, 2 * I, 2 * I, dt, st), "lf_silu_mul_bwd");
      return {dg};
    }
    const auto [a2, lda] = rows_view(av);
    const auto [b2, ldb] = rows_view(bv);
    const Tensor da = at::empty(sizes, av.options()), db = at::empty(sizes, av.options());
    if (M > 0) check(lf_silu_mul_bwd(ptr(dc), ptr(a2), ptr(b2), mptr(da), mptr(db), M, I, lddc, lda, ldb, I, I, dt, st), "lf_silu_mul_bwd");
    return {da, db};
  }
};

Tensor silu_mul(const Tensor& a, const Tensor& b) {
  require_gpu(a, "a");
  if (a.sizes() != b.sizes() || a.scalar_type() != b.scalar_type())
    bad_value("silu_mul operands differ: ", shape_name(a.sizes()), " ", dtype_name(a.scalar_type()), " vs ", shape_name(b.sizes()), " ", dtype_name(b.scalar_type()), ".");
  if (a.size(-1) % 8 != 0) bad_value("the last dimension must be a multiple of 8, got ", a.size(-1), ".");
  refuse_tangents(a, b);
  Tensor c, as = a, bs = b;   // what the backward keeps: the caller's tensor where the kernel reads it as it lies, else the copy
  {
    const at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard device(a.device());
    const auto [a2, lda] = rows_view(a);
    const auto [b2, ldb] = rows_view(b);
    if (!a2.is_alias_of(a)) as = a2;
    if (!b2.is_alias_of(b)) bs = b2;
    c = at::empty(a.sizes(), a.options());
    if (a2.size(0) > 0)
      check(lf_silu_mul_fwd(ptr(a2), ptr(b2), mptr(c), (int)a2.size(0), (int)a2.size(1), lda, ldb, a2.size(1), dtype_id(a.scalar_type()), stream_of(a)), "lf_silu_mul_fwd");
  }
  if (wants_grad({a, b})) {
    std::shared_ptr<SiLUMulBackward> n(new SiLUMulBackward(), torch::autograd::deleteNode);
    n->set_next_edges(torch::autograd::collect_next_edges(a, b));
    n->a = SavedVariable(as, false);
    n->b = SavedVariable(bs, false);
    n->sizes = a.sizes().vec();
    n->c_sizes = n->sizes;
    torch::autograd::set_history(c, n);
  }
  return c;
}

Tensor silu_mul_merged(const Tensor& gu) {
  require_gpu(gu, "gate_up");
  const int64_t I2 = gu.size(-1), I = I2 / 2;
  if (I2 % 16 != 0) bad_value("the merged width must be a multiple of 16, got ", I2, ".");
  refuse_tangents(gu);
  Tensor g, c;
  std::vector<int64_t> cs = gu.sizes().vec();
  cs.back() = I;
  {
    const at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard device(gu.device());
    g = gu.contiguous();
    c = at::empty(cs, gu.options());
    const int64_t M = rows_of(g);
    const char* gp = (const char*)g.const_data_ptr();
    if (M > 0) check(lf_silu_mul_fwd(gp, gp + 2 * I, mptr(c), (int)M, (int)I, I2, I2, I, dtype_id(gu.scalar_type()), stream_of(gu)), "lf_silu_mul_fwd");
  }
  if (wants_grad({gu})) {
    std::shared_ptr<SiLUMulBackward> n(new SiLUMulBackward(), torch::autograd::deleteNode);
    n->set_next_edges(torch::autograd::collect_next_edges(gu));
    n->a = SavedVariable(g, false);
    n->merged = true;
    n->sizes = gu.sizes().vec();
    n->c_sizes = cs;
    torch::autograd::set_history(c, n);
  }
  return c;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  // (no Python object is touched inside; an exception is translated after the lock is back)
  using nogil = py::call_guard<py::gil_scoped_release>;
  m.def("linear_lora", &linear_lora, nogil());
  m.def("check_multi", &check_multi, nogil());
  m.def("forward", &py_forward, nogil());
  m.def("backward", &py_backward, nogil());
  m.def("attach", &py_attach);   // (takes a Python object: lets go of the lock itself)
  m.def("check_adapters", &check_adapters, nogil());
  m.def("rms_norm", &rms_norm, nogil());
  m.def("silu_mul", &silu_mul, nogil());
  m.def("silu_mul_merged", &silu_mul_merged, nogil());
}
