// One message-passing layer (GCLLayerFn of layer_fn.py) as a native autograd node.
//
// The kernels of a layer over a few graphs take less time than the Python around them (molecule-sized calls:
// 45 us of kernels behind 75 us of host work forward, 300 us behind 450 us forward and backward), most of it tensor
// allocations, argument conversion and the autograd engine's calls back into Python.  This is the same sequence of
// C-ABI calls with the allocations and the backward in C++.  It takes only calls whose tensors need no conversion
// (gcl_layer returns None for any other, and the Python node, which converts and reports errors, runs instead):
// plain device tensors of one dtype and device, contiguous, shapes that fit together.
#include <torch/extension.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <c10/hip/HIPStream.h>
#include "../../include/egnn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
typedef std::optional<Tensor> Opt;

// the status as the Python bindings report it (EgnnError); any thread
void check(const char* fn, int32_t status) {
  if (status == EGNN_OK) return;
  pybind11::gil_scoped_acquire gil;
  pybind11::module_::import("pymolecular_amd._capi").attr("check")(fn, status);
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
template <typename T = void> T* ptr(const Tensor& t) { return t.defined() ? (T*)t.data_ptr() : nullptr; }
Tensor get(const Opt& t) { return t.has_value() ? *t : Tensor(); }
bool aligned16(const Tensor& t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }
// unit-stride rows that start 16-byte aligned and do not overlap (an expanded gradient's have stride 0), else a copy
Tensor rowmajor(const Tensor& t) {
  return t.stride(1) == 1 && t.stride(0) >= t.size(1) && (t.stride(0) * t.element_size()) % 16 == 0 && aligned16(t)
             ? t : t.clone(at::MemoryFormat::Contiguous);
}

// no tensor subclass, functorch wrapper or functionalised tensor, on h's device
bool plain(const Tensor& t, const Tensor& h) {
  const auto ks = t.key_set();
  return t.is_cuda() && t.device() == h.device() && t.layout() == c10::kStrided && !t.is_conj() && !t.is_neg() &&
         !ks.has(c10::DispatchKey::Python) && !ks.has(c10::DispatchKey::FuncTorchBatched) &&
         !ks.has(c10::DispatchKey::FuncTorchGradWrapper) && !ks.has(c10::DispatchKey::Functionalize) &&
         !t._fw_grad(0).defined();
}
bool fits(const Tensor& t, const Tensor& h, at::ScalarType dt, std::initializer_list<int64_t> shape) {
  return plain(t, h) && t.scalar_type() == dt && t.sizes() == c10::IntArrayRef(shape) && t.is_contiguous();
}
bool fits_opt(const Opt& t, const Tensor& h, at::ScalarType dt, int64_t n) { return !t || fits(*t, h, dt, {n}); }

// the layer's tensors in the order they are saved
enum { kH, kX, kE, kRow, kCol, kPerm, kW1, kW2, kM1, kM2, kB1, kB2, kBx, kN0, kN2, kSched, kPQ, kAgg, kPre, kAct, kCount };

struct Layer {
  variable_list t;
  bool mean, residual, eq, nb0, nb2;
  EgnnDims dims() const {
    EgnnDims d{};
    const Tensor &h = t[kH], &w1 = t[kW1];
    d.N = h.size(0); d.E = t[kCol].numel(); d.F = (int32_t)h.size(1);
    d.FE = t[kE].defined() ? (int32_t)t[kE].size(1) : 0;
    d.H = (int32_t)w1.size(0); d.O = (int32_t)t[kW2].size(0); d.M = eq ? (int32_t)t[kM1].size(0) : d.O;
    d.equivariant = eq; d.mean_agg = mean;
    d.dtype = h.scalar_type() == at::kFloat ? EGNN_F32 : EGNN_BF16;
    d.weight_layout = EGNN_WEIGHTS_LINEAR;
    d.flags = eq ? EGNN_FLAG_COORD_RESIDUAL : 0;
    return d;
  }
  EgnnNodeDims node_dims() const {
    EgnnNodeDims d{};
    d.N = t[kH].size(0); d.K1 = (int32_t)t[kH].size(1); d.K2 = (int32_t)t[kW2].size(0);
    d.Hn = (int32_t)t[kN0].size(0); d.Fo = (int32_t)t[kN2].size(0);
    d.residual = residual; d.dtype = t[kH].scalar_type() == at::kFloat ? EGNN_F32 : EGNN_BF16;
    return d;
  }
};

class GclLayer : public torch::autograd::Function<GclLayer> {
 public:
  static variable_list forward(AutogradContext* ctx, const Tensor& h, const Opt& x, const Opt& ef, const Tensor& row,
                               const Tensor& col, const Opt& perm, const Tensor& e0w, const Opt& e0b, const Tensor& e2w,
                               const Opt& e2b, const Opt& c0w, const Opt& c0b, const Opt& c2w, const Tensor& n0w,
                               const Opt& n0b, const Tensor& n2w, const Opt& n2b, const Tensor& sched, bool mean,
                               bool residual, bool eq) {
    Layer a{{h, get(x), get(ef), row, col, get(perm), e0w, e2w, get(c0w), get(c2w), get(e0b), get(e2b), get(c0b), n0w,
             n2w, sched, {}, {}, {}, {}}, mean, residual, eq, n0b.has_value(), n2b.has_value()};
    const EgnnDims d = a.dims();
    const EgnnNodeDims nd = a.node_dims();
    const auto act = h.options(), bytes = act.dtype(at::kByte), f32 = act.dtype(at::kFloat);
    void* st = stream_of(h);
    a.t[kPQ] = at::empty({(int64_t)std::max<size_t>(egnn_node_proj_bytes(&d), 16)}, bytes);
    a.t[kAgg] = at::empty({d.N, d.O}, act);
    Tensor x_new = eq ? at::empty({d.N, 3}, f32) : Tensor();
    {
      const size_t nb = egnn_fwd_workspace_bytes(&d);
      const Tensor ws = at::empty({(int64_t)nb}, bytes);
      EgnnStrides s{};
      s.h = h.stride(0); s.coord = eq ? 3 : 4; s.edge = ef ? ef->stride(0) : 0; s.msg = d.O; s.mov = 3;
      check("egnn_fwd", egnn_fwd(&d, &s, ptr(h), ptr<float>(a.t[kX]), ptr(a.t[kE]), ptr<int32_t>(row), ptr<int32_t>(col),
                                 ptr<int32_t>(a.t[kPerm]), ptr(e0w), ptr(e2w), ptr(a.t[kM1]), ptr(a.t[kM2]), ptr(a.t[kB1]),
                                 ptr(a.t[kB2]), ptr(a.t[kBx]), ptr(a.t[kAgg]), ptr<float>(x_new), ptr(a.t[kPQ]), ptr(sched),
                                 ptr(ws), nb, st));
    }
    a.t[kPre] = at::empty({d.N, nd.Hn}, act);
    if (egnn_node_act_required(&nd)) a.t[kAct] = at::empty({d.N, nd.Hn}, act);
    Tensor out = at::empty({d.N, nd.Fo}, act);
    check("egnn_node_fwd", egnn_node_fwd(&nd, ptr(h), h.stride(0), ptr(a.t[kAgg]), d.O, ptr(n0w), ptr(get(n0b)), ptr(n2w),
                                         ptr(get(n2b)), ptr(a.t[kPre]), ptr(a.t[kAct]), ptr(out), nd.Fo, st));
    ctx->save_for_backward(a.t);
    ctx->saved_data["flags"] = (int64_t)(mean | residual << 1 | eq << 2 | a.nb0 << 3 | a.nb2 << 4);
    return eq ? variable_list{out, x_new} : variable_list{out};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const int64_t f = ctx->saved_data["flags"].toInt();
    Layer a{ctx->get_saved_variables(), bool(f & 1), bool(f & 2), bool(f & 4), bool(f & 8), bool(f & 16)};
    const Tensor &h = a.t[kH], &x = a.t[kX], &ef = a.t[kE], &w1 = a.t[kW1], &w2 = a.t[kW2];
    EgnnDims d = a.dims();
    const EgnnNodeDims nd = a.node_dims();
    const auto act = h.options(), bytes = act.dtype(at::kByte), f32 = act.dtype(at::kFloat);
    void* st = stream_of(h);
    // the node update's backward: grad_x = [dL/dh | dL/dagg]
    const Tensor gout = grads[0].defined() ? rowmajor(grads[0].to(h.scalar_type())) : at::zeros({d.N, nd.Fo}, act);
    const int64_t K = nd.K1 + nd.K2;
    const Tensor grad_x = at::empty({d.N, K}, act);
    const Tensor gn0 = at::empty_like(a.t[kN0]), gn2 = at::empty_like(a.t[kN2]);
    const Tensor gnb0 = a.nb0 ? at::empty({nd.Hn}, act) : Tensor(), gnb2 = a.nb2 ? at::empty({nd.Fo}, act) : Tensor();
    {
      const size_t nb = egnn_node_bwd_workspace_bytes(&nd);
      const Tensor ws = at::empty({(int64_t)std::max<size_t>(nb, 16)}, bytes);
      check("egnn_node_bwd", egnn_node_bwd(&nd, ptr(h), h.stride(0), ptr(a.t[kAgg]), d.O, ptr(a.t[kN0]), ptr(a.t[kN2]),
                                           ptr(a.t[kPre]), ptr(a.t[kAct]), ptr(gout), gout.stride(0), ptr(grad_x), ptr(gn0),
                                           ptr(gnb0), ptr(gn2), ptr(gnb2), ptr(ws), nb, st));
    }
    // the messages' backward, its gradient of h added to the node update's
    const Tensor grad_h = grad_x.narrow(1, 0, nd.K1);
    const Tensor gm = rowmajor(grad_x.narrow(1, nd.K1, nd.K2));
    Tensor gx, grad_c;
    if (a.eq) {
      gx = grads.size() > 1 && grads[1].defined() ? grads[1].to(at::kFloat).contiguous() : at::zeros({d.N, 3}, f32);
      grad_c = at::empty({d.N, 3}, f32);
    }
    auto like = [](const Tensor& t) { return t.defined() ? at::empty_like(t) : Tensor(); };
    const Tensor g1 = like(w1), g2 = like(w2), gm1 = like(a.t[kM1]), gm2 = like(a.t[kM2]);
    const Tensor gb1 = like(a.t[kB1]), gb2 = like(a.t[kB2]), gbx = like(a.t[kBx]);
    {
      d.flags |= EGNN_FLAG_ACCUMULATE_GRAD_H;
      const size_t nb = egnn_bwd_workspace_bytes(&d);
      const Tensor ws = at::empty({(int64_t)nb}, bytes);
      EgnnStrides s{};
      s.h = h.stride(0); s.coord = 3; s.edge = ef.defined() ? ef.stride(0) : 0; s.msg = gm.stride(0);
      s.mov = 3; s.grad_h = grad_h.stride(0);
      check("egnn_bwd", egnn_bwd(&d, &s, ptr(h), ptr<float>(x), ptr(ef), ptr<int32_t>(a.t[kRow]), ptr<int32_t>(a.t[kCol]),
                                 ptr<int32_t>(a.t[kPerm]), ptr(w1), ptr(w2), ptr(a.t[kM1]), ptr(a.t[kM2]), ptr(a.t[kB1]),
                                 ptr(a.t[kB2]), ptr(a.t[kBx]), ptr(gm), ptr<float>(gx), ptr(grad_h), ptr<float>(grad_c),
                                 ptr(g1), ptr(g2), ptr(gm1), ptr(gm2), ptr(gb1), ptr(gb2), ptr(gbx), ptr(a.t[kPQ]),
                                 ptr(a.t[kSched]), ptr(ws), nb, st));
    }
    return {grad_h, grad_c, {}, {}, {}, {}, g1, gb1, g2, gb2, gm1, gbx, gm2, gn0, gnb0, gn2, gnb2, {}, {}, {}, {}};
  }
};

// The layer, or None when a tensor would need a conversion or the dimensions are not supported
pybind11::object gcl_layer(const Tensor& h, const Opt& x, const Opt& ef, const Tensor& row, const Tensor& col,
                           const Opt& perm, const Tensor& e0w, const Opt& e0b, const Tensor& e2w, const Opt& e2b,
                           const Opt& c0w, const Opt& c0b, const Opt& c2w, const Tensor& n0w, const Opt& n0b,
                           const Tensor& n2w, const Opt& n2b, const Tensor& sched, bool mean, bool residual, bool eq) {
  const pybind11::object none = pybind11::none();
  if (torch::jit::tracer::isTracing() || h.dim() != 2 || h.size(0) < 1 || e0w.dim() != 2 || e2w.dim() != 2 ||
      n0w.dim() != 2 || n2w.dim() != 2 || col.dim() != 1)
    return none;
  const auto dt = h.scalar_type();
  if (dt != at::kFloat && dt != at::kBFloat16) return none;
  const int64_t N = h.size(0), F = h.size(1), H = e0w.size(0), O = e2w.size(0), Hn = n0w.size(0), Fo = n2w.size(0);
  const int64_t g = eq ? 1 : 0, FE = ef ? (ef->dim() == 2 ? ef->size(1) : -1) : 0;
  if (FE < 0 || (ef && (ef->size(0) < 1 || FE < 1)) || F % 16 || Hn % 8 || Fo % 8 || O % 8 || (residual && Fo != F)) return none;
  if (!fits(h, h, dt, {N, F}) || !aligned16(h) || !fits(e0w, h, dt, {H, 2 * F + g + FE}) || !fits(e2w, h, dt, {O, H}) ||
      !fits(n0w, h, dt, {Hn, F + O}) || !fits(n2w, h, dt, {Fo, Hn}) || !fits_opt(e0b, h, dt, H) ||
      !fits_opt(e2b, h, dt, O) || !fits_opt(n0b, h, dt, Hn) || !fits_opt(n2b, h, dt, Fo))
    return none;
  if (ef && !fits(*ef, h, dt, {ef->size(0), FE})) return none;
  if (!fits(row, h, at::kInt, {N + 1}) || !fits(col, h, at::kInt, {col.numel()}) ||
      (perm && !fits(*perm, h, at::kInt, {col.numel()})) || !plain(sched, h))
    return none;
  if (eq) {
    if (!x || !c0w || !c2w || c0w->dim() != 2 || !fits(*x, h, at::kFloat, {N, 3})) return none;
    const int64_t M = c0w->size(0);
    if (!fits(*c0w, h, dt, {M, O}) || !fits_opt(c0b, h, dt, M) || !plain(*c2w, h) || c2w->scalar_type() != dt ||
        c2w->numel() != M || !c2w->is_contiguous())
      return none;
  } else if (x || c0w || c0b || c2w) {
    return none;
  }
  {   // dimensions the library refuses are reported by the Python path
    Layer a{{h, get(x), get(ef), row, col, get(perm), e0w, e2w, get(c0w), get(c2w), {}, {}, {}, n0w, n2w, sched, {}, {}, {}, {}},
            mean, residual, eq, false, false};
    const EgnnDims d = a.dims();
    if (egnn_fwd_workspace_bytes(&d) == 0) return none;
  }
  variable_list r;
  {
    pybind11::gil_scoped_release nogil;
    r = GclLayer::apply(h, x, ef, row, col, perm, e0w, e0b, e2w, e2b, c0w, c0b, c2w, n0w, n0b, n2w, n2b, sched, mean,
                        residual, eq);
  }
  if (eq) return pybind11::make_tuple(r[0], r[1]);
  return pybind11::cast(r[0]);
}

}  // namespace

PYBIND11_MODULE(_egnn_torch, m) { m.def("gcl_layer", &gcl_layer); }
