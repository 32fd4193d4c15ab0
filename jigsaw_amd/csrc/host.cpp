// Host side of the small steps in native code: the distributed convolution (Step), ring attention over resident chunks, the
// sharded LayerNorm's pieces between its collectives, GroupNorm of a whole tensor, the projections around attention and the
// Swin block (SwinPass), and the backward of the functions that autograd calls here (_autograd.NativeFunction).
//
// The convolution: allocations, strips, pointer tables and the calls into
// libjigsaw_hip.so, in native code. A step of one layer is 10 launches of 3 to 60 us; worked through Python
// functions (checks, tuples of shapes, 14 allocations, up to 26 strips cut and looked up, ctypes calls) the host
// took about 165 us for it beside autograd's own 60, which is what small and ordinary layers then ran at
// (40 -> 72 channels of 2 x 217 x 301 bf16: 200 us of host time a step in one thread, 75 here).
// Everything that depends on shapes only is laid out once per layer and tile in a Step; a call allocates,
// fills the pointer tables and launches. A Step holds no tensors and is not changed after it is built (but for the
// note that the fused fold does not cover the layer), so that threads may share it.
//
// What a Step does not take (a strip of another shape or layout, tensors of mixed types) it declines by returning
// None before anything is launched; the callers' Python route then names the error or handles the case.
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <memory>
#include <tuple>
#include <utility>
#include <vector>

#include "../../include/jigsaw_hip.h"

namespace {

namespace py = pybind11;
using Shape = c10::SmallVector<int64_t, 5>;

struct Strip {
  py::object key;  // offset of the neighbour
  int slot;
  Shape shape;
  int64_t start, numel;  // in elements of the flat buffer (strips that are sent)
};

void check(int rc, const char* what) {
  if (rc != JG_OK) py::module_::import("jigsaw_amd._lib").attr("check")(rc, what);
}

Shape to_shape(const py::handle& seq) {
  Shape s;
  for (const auto& v : seq) s.push_back(v.cast<int64_t>());
  return s;
}

int64_t count(const Shape& s) {
  int64_t n = 1;
  for (int64_t v : s) n *= v;
  return n;
}

// What `Step.backward` leaves of the weight and bias gradient for `finish`, and the memory it is in.
struct SumsLeft {
  jg_conv_reduction sums = {};
  std::vector<at::Tensor> held;
};
// The most scratch that is held for it through the input gradient and the exchange. A launch of 4 to 10 us less is worth the workgroups'
// partials (up to 38 MB below 1000 channels), but not the copies of both tensors that fp32 layers on sums of bf16 parts have beside
// them: 3.1 GB for 1 x 64 -> 64 of 2048^2, which the input gradient (1.1 GB) and its own copies (1.6) have else the place of.
constexpr size_t kMostHeld = size_t(64) << 20;

class Step {
 public:
  // Strips: [(offset, slot, shape), ...] with the leading (batch, channel) entries in the shape.
  Step(const py::tuple& x_shape, const py::tuple& padded, const py::tuple& y_shape, const py::tuple& w_shape, int elem_size, int code,
       uintptr_t own, uintptr_t theirs, bool same, uintptr_t desc, const std::vector<size_t>& nbytes, const py::list& recv_fwd,
       const py::list& recv_bwd, const py::list& send_fwd, const py::list& send_bwd, bool try_fold)
      : x_shape_(to_shape(x_shape)), padded_(to_shape(padded)), y_shape_(to_shape(y_shape)), w_shape_(to_shape(w_shape)),
        elem_(elem_size), code_(code), own_(*reinterpret_cast<const jg_halo_geom*>(own)),
        theirs_(*reinterpret_cast<const jg_halo_geom*>(theirs)), same_(same), desc_(*reinterpret_cast<const jg_conv_desc*>(desc)),
        nbytes_(nbytes), recv_fwd_(strips(recv_fwd)), recv_bwd_(strips(recv_bwd)), send_fwd_(strips(send_fwd)),
        send_bwd_(strips(send_bwd)), beside_(nbytes_[JG_CONV_WGRAD] <= kMostHeld && jg_halo_fold_border_takes_sums(&theirs_, code) == 1),
        fold_(try_fold) {}

  bool sends() const { return !send_fwd_.empty(); }

  // Strips of the own tile for the neighbours, {offset: strip}.
  py::object pack(const at::Tensor& x, uintptr_t stream) const {
    if (x.sizes() != at::IntArrayRef(x_shape_) || !x.is_contiguous()) return py::none();
    return cut(x, send_fwd_, theirs_, 0, stream);
  }

  // (y, x_aug) from the own tile and the received strips, or None.
  py::object forward(const at::Tensor& x, const py::object& recv, const at::Tensor& w_any, const c10::optional<at::Tensor>& b_any,
                     uintptr_t stream) const {
    const void* src[27] = {};
    if (!takes(x, w_any, b_any) || !table(recv, recv_fwd_, x, src)) return py::none();
    at::AutoDispatchBelowADInplaceOrView below;
    const at::Tensor w = w_any.contiguous(), b = b_any ? b_any->contiguous() : at::Tensor();
    src[13] = x.data_ptr();
    at::Tensor x_aug = at::empty(padded_, x.options()), y = at::empty(y_shape_, x.options());
    check(jg_halo_assemble_3d(x_aug.data_ptr(), src, &own_, elem_, reinterpret_cast<void*>(stream)), "jg_halo_assemble_3d");
    const at::Tensor ws = scratch(nbytes_[JG_CONV_FWD], x);
    check(jg_conv_fwd(y.data_ptr(), x_aug.data_ptr(), w.data_ptr(), b.defined() ? b.data_ptr() : nullptr, &desc_, code_,
                      address(ws), nbytes_[JG_CONV_FWD], reinterpret_cast<void*>(stream)),
          "jg_conv_fwd");
    return py::make_tuple(y, x_aug);
  }

  // (input gradient, weight gradient, bias gradient, strips to send, folded, sums left) or None. The input gradient is the
  // padded one, or with `folded` the own tile's, to which only the neighbours' blocks are still missing. The
  // bias gradient is None where only the separate kernels cover the layer. Sums left (None, or for `finish`): what the weight
  // and bias gradient still miss.
  py::object backward(const at::Tensor& g_any, const at::Tensor& x_aug, const at::Tensor& w_any, bool need_x, bool need_w, bool need_b,
                      uintptr_t stream) {
    if (g_any.sizes() != at::IntArrayRef(y_shape_) || x_aug.sizes() != at::IntArrayRef(padded_) || !x_aug.is_contiguous() ||
        w_any.sizes() != at::IntArrayRef(w_shape_) || !same_kind(g_any, x_aug) || !same_kind(w_any, x_aug))
      return py::none();
    at::AutoDispatchBelowADInplaceOrView below;
    void* const s = reinterpret_cast<void*>(stream);
    const at::Tensor g = g_any.contiguous(), w = w_any.contiguous();
    py::object gw = py::none(), gb = py::none(), gx = py::none(), send = py::dict(), left = py::none();
    bool folded = false;
    SumsLeft later;
    if (need_w) {
      const at::Tensor gw_t = at::empty(w_shape_, g.options());
      const at::Tensor ws = scratch(nbytes_[JG_CONV_WGRAD], g);
      int rc = JG_ERR_UNSUPPORTED;
      if (need_b) {
        const at::Tensor gb_t = at::empty({w_shape_[0]}, g.options());
        if (need_x && beside_ && fold_.load(std::memory_order_relaxed)) {  // the last of the sums beside the border cells, in `finish`
          rc = jg_conv_wgrad_bias_later(&later.sums, gw_t.data_ptr(), gb_t.data_ptr(), x_aug.data_ptr(), g.data_ptr(), &desc_, code_,
                                        address(ws), nbytes_[JG_CONV_WGRAD], s);
          if (later.sums.kind != 0) later.held = {ws, gw_t, gb_t};
        } else {
          rc = jg_conv_wgrad_bias(gw_t.data_ptr(), gb_t.data_ptr(), x_aug.data_ptr(), g.data_ptr(), &desc_, code_, address(ws),
                                  nbytes_[JG_CONV_WGRAD], s);
        }
        if (rc != JG_ERR_UNSUPPORTED) {
          check(rc, "jg_conv_wgrad_bias");
          gb = py::cast(gb_t);
        }
      }
      if (rc == JG_ERR_UNSUPPORTED)
        check(jg_conv_wgrad(gw_t.data_ptr(), x_aug.data_ptr(), g.data_ptr(), &desc_, code_, address(ws), nbytes_[JG_CONV_WGRAD], s),
              "jg_conv_wgrad");
      gw = py::cast(gw_t);
    }
    if (need_x) {
      const at::Tensor ws = scratch(nbytes_[JG_CONV_DGRAD], g);
      if (fold_.load(std::memory_order_relaxed)) {
        // dgrad writes the owned cells and the strips itself
        const at::Tensor own = at::empty(x_shape_, g.options());
        void* tab[27] = {};
        py::dict out = new_strips(g, send_bwd_, tab);
        const int rc = jg_conv_dgrad_fold(own.data_ptr(), tab, w.data_ptr(), g.data_ptr(), &desc_, &own_, code_, address(ws),
                                          nbytes_[JG_CONV_DGRAD], s);
        if (rc != JG_ERR_UNSUPPORTED) {
          check(rc, "jg_conv_dgrad_fold");
          gx = py::cast(own);
          send = out;
          folded = true;
        } else {
          fold_.store(false, std::memory_order_relaxed);
        }
      }
      if (later.sums.kind != 0) {
        if (folded) {
          left = py::cast(std::move(later));
        } else {
          check(jg_conv_reduce(&later.sums, s), "jg_conv_reduce");
          later.held.clear();
        }
      }
      if (!folded) {
        const at::Tensor need = at::empty(padded_, g.options());
        check(jg_conv_dgrad(need.data_ptr(), w.data_ptr(), g.data_ptr(), &desc_, code_, address(ws), nbytes_[JG_CONV_DGRAD], s),
              "jg_conv_dgrad");
        gx = py::cast(need);
        if (!send_bwd_.empty()) send = cut(need, send_bwd_, own_, 1, stream);
      }
    }
    return py::make_tuple(gx, gw, gb, send, folded, left);
  }

  // The own tile's gradient from what `backward` returned and the neighbours' blocks, or None. The sums left are done in any case.
  py::object finish(const at::Tensor& part, bool folded, const py::object& recv, uintptr_t stream, const py::object& left) const {
    const void* tab[27] = {};
    void* const s = reinterpret_cast<void*>(stream);
    const jg_conv_reduction* const sums = left.is_none() ? nullptr : &left.cast<const SumsLeft&>().sums;
    if (!table(recv, recv_bwd_, part, tab)) {
      if (sums != nullptr) check(jg_conv_reduce(sums, s), "jg_conv_reduce");
      return py::none();
    }
    at::AutoDispatchBelowADInplaceOrView below;
    at::Tensor gx = part;
    const void* none[27] = {};
    if (!folded) {
      gx = at::empty(x_shape_, part.options());
      // where the neighbours' blocks are not as wide as the own halos, the own part first and the blocks by their widths
      check(jg_halo_fold_3d(gx.data_ptr(), part.data_ptr(), same_ ? tab : none, &own_, code_, s), "jg_halo_fold_3d");
    }
    if (sums != nullptr)
      check(jg_halo_fold_border_reduce_3d(gx.data_ptr(), tab, &theirs_, code_, sums, s), "jg_halo_fold_border_reduce_3d");
    else if (folded || !same_)
      check(jg_halo_fold_border_3d(gx.data_ptr(), tab, &theirs_, code_, s), "jg_halo_fold_border_3d");
    return py::cast(gx);
  }

  // Whether `forward` takes these, whatever strips arrive
  bool takes(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& b) const {
    return x.has_storage() && x.sizes() == at::IntArrayRef(x_shape_) && x.is_contiguous() && w.sizes() == at::IntArrayRef(w_shape_) && same_kind(w, x) &&
           (!b || (same_kind(*b, x) && b->dim() == 1 && b->size(0) == w_shape_[0]));
  }

 private:
  std::vector<Strip> strips(const py::list& rows) const {
    std::vector<Strip> out;
    int64_t at = 0;
    const int64_t per = 256 / elem_;  // every strip from a 256-byte boundary on
    for (const auto& row : rows) {
      const py::tuple t = row.cast<py::tuple>();
      Strip s{t[0], t[1].cast<int>(), to_shape(t[2]), at, 0};
      s.numel = count(s.shape);
      at += (s.numel + per - 1) / per * per;
      out.push_back(std::move(s));
    }
    return out;
  }
  static bool same_kind(const at::Tensor& t, const at::Tensor& like) {
    return t.scalar_type() == like.scalar_type() && t.device() == like.device();
  }
  static at::Tensor scratch(size_t n, const at::Tensor& like) {
    return n ? at::empty({(int64_t)n}, like.options().dtype(at::kByte)) : at::Tensor();
  }
  static void* address(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

  // Pointers of the strips in `recv` by slot; false where one is not what the geometry asks for.
  static bool table(const py::object& recv, const std::vector<Strip>& want, const at::Tensor& like, const void* out[27]) {
    if (!PyDict_Check(recv.ptr())) return false;
    if (PyDict_Size(recv.ptr()) == 0) return true;
    for (const Strip& s : want) {
      PyObject* o = PyDict_GetItemWithError(recv.ptr(), s.key.ptr());
      if (o == nullptr && PyErr_Occurred()) throw py::error_already_set();
      if (o == nullptr || o == Py_None) continue;
      if (!THPVariable_Check(o)) return false;
      const at::Tensor& t = THPVariable_Unpack(o);
      if (t.sizes() != at::IntArrayRef(s.shape) || !same_kind(t, like) || !t.is_contiguous()) return false;
      if (s.numel) out[s.slot] = t.data_ptr();
    }
    return true;
  }

  // Uninitialised strips in one allocation, {offset: strip}, and their addresses by slot.
  static py::dict new_strips(const at::Tensor& like, const std::vector<Strip>& want, void* tab[27]) {
    py::dict out;
    if (want.empty()) return out;
    const int64_t per = 256 / like.element_size();
    const Strip& last = want.back();
    const at::Tensor flat = at::empty({last.start + (last.numel + per - 1) / per * per}, like.options());
    char* const base = static_cast<char*>(flat.data_ptr());
    for (const Strip& s : want) {
      Shape strides(s.shape.size());
      int64_t step = 1;
      for (size_t a = s.shape.size(); a-- > 0;) {
        strides[a] = step;
        step *= s.shape[a] > 1 ? s.shape[a] : 1;
      }
      out[s.key] = at::as_strided(flat, s.shape, strides, s.start);
      if (s.numel) tab[s.slot] = base + s.start * like.element_size();
    }
    return out;
  }

  py::object cut(const at::Tensor& src, const std::vector<Strip>& want, const jg_halo_geom& geom, int from_padded, uintptr_t stream) const {
    at::AutoDispatchBelowADInplaceOrView below;
    void* tab[27] = {};
    py::dict out = new_strips(src, want, tab);
    check(jg_halo_pack_3d(tab, src.data_ptr(), &geom, from_padded, elem_, reinterpret_cast<void*>(stream)), "jg_halo_pack_3d");
    return std::move(out);
  }

  Shape x_shape_, padded_, y_shape_, w_shape_;
  int elem_, code_;
  jg_halo_geom own_, theirs_;
  bool same_;
  jg_conv_desc desc_;
  std::vector<size_t> nbytes_;
  std::vector<Strip> recv_fwd_, recv_bwd_, send_fwd_, send_bwd_;
  bool beside_;  // the border's launch takes the sums that the weight gradient leaves
  std::atomic<bool> fold_;
};

// ---- attention and norms: checks, allocations and calls of the Python routes in attention.py, layernorm.py, groupnorm.py,
// for tensors that need no conversion or copy; None for all others, before anything is allocated. Host time of a step, with
// autograd's own: ring of 4 heads x 128 x 2 chunks 49 us through Python, 20 here;
// LayerNorm of 4096 x 256 of 512 173 and 136 (its four collectives included); GroupNorm of 2 x 32 x 60 x 70 142 and 111.

int code_of(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return JG_F32;
    case at::kBFloat16: return JG_BF16;
    case at::kHalf: return JG_F16;
    default: return -1;
  }
}
bool on_gpu(const at::Tensor& t) { return t.is_cuda() && t.is_contiguous() && t.has_storage(); }
bool aligned(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }
void* pointer(uintptr_t p) { return reinterpret_cast<void*>(p); }

using List = std::vector<at::Tensor>;
constexpr size_t kMostChunks = 16;       // attention._MAX_CHUNKS_PER_CALL
constexpr int64_t kMostBatch = 65535;    // attention._MOST_BATCH
constexpr int64_t kMostRows = 1 << 23;   // attention._MOST_ROWS

// bf16 heads that may be better off with zero columns up to 64: attention._as_64_columns, which has the rule and the figures,
// decides, and whoever asked it calls the functions `_at_own_width`. Everything for which it can say yes has to be here.
bool may_want_64_columns(int64_t head_size, int64_t q_rows, int64_t keys) { return head_size < 64 && q_rows >= 2048 && keys >= 4096; }

// What the one-pass kernels take without copies, conversions or zero columns (attention._resident)
bool ring_ok(const at::Tensor& q, const List& k, const List& v, bool own_width, int64_t* batch) {
  const int64_t n = q.dim();
  if (n < 3 || k.empty() || k.size() > kMostChunks || v.size() != k.size() || q.numel() == 0 || k[0].numel() == 0) return false;
  const int64_t d = q.size(-1), sq = q.size(-2), sk = k[0].dim() == n ? k[0].size(-2) : 0;
  if ((q.scalar_type() != at::kBFloat16 && q.scalar_type() != at::kHalf) || d % 8 != 0 || d > 128 || sq > kMostRows || sk > kMostRows) return false;
  if (!own_width && q.scalar_type() == at::kBFloat16 && may_want_64_columns(d, sq, sk * (int64_t)k.size())) return false;
  *batch = q.numel() / (sq * d);
  if (*batch > kMostBatch || !on_gpu(q) || !aligned(q)) return false;
  for (int64_t a = 0; a < n; ++a)
    if (a != n - 2 && (k[0].dim() != n || k[0].size(a) != q.size(a))) return false;
  for (size_t j = 0; j < k.size(); ++j)
    for (const at::Tensor* t : {&k[j], &v[j]})
      if (t->sizes() != k[0].sizes() || t->scalar_type() != q.scalar_type() || t->device() != q.device() || !t->is_contiguous() || !aligned(*t))
        return false;
  return true;
}

template <typename P>
void addresses(const List& from, P* to) {
  for (size_t j = 0; j < from.size(); ++j) to[j] = from[j].data_ptr();
}

template <bool OWN_WIDTH>
py::object ring_forward(const at::Tensor& q, const List& k, const List& v, double scale, uintptr_t stream) {
  int64_t batch;
  if (!ring_ok(q, k, v, OWN_WIDTH, &batch)) return py::none();
  at::AutoDispatchBelowADInplaceOrView below;
  const at::Tensor out = at::empty_like(q), lse = at::empty(q.sizes().slice(0, q.dim() - 1), q.options().dtype(at::kFloat));
  const void *kp[kMostChunks], *vp[kMostChunks];
  addresses(k, kp);
  addresses(v, vp);
  check(jg_attn_fwd_chunks(out.data_ptr(), lse.data_ptr<float>(), q.data_ptr(), kp, vp, k.size(), batch, q.size(-2), k[0].size(-2),
                           q.size(-1), (float)scale, code_of(q), pointer(stream)),
        "jg_attn_fwd_chunks");
  return py::make_tuple(out, lse);
}

template <bool OWN_WIDTH>
py::object ring_backward(const at::Tensor& dout, const at::Tensor& q, const at::Tensor& out, const at::Tensor& lse, const List& k,
                         const List& v, double scale, uintptr_t stream) {
  int64_t batch;
  if (!ring_ok(q, k, v, OWN_WIDTH, &batch)) return py::none();
  for (const at::Tensor* t : {&dout, &out})
    if (t->sizes() != q.sizes() || t->scalar_type() != q.scalar_type() || t->device() != q.device() || !t->is_contiguous() || !aligned(*t)) return py::none();
  if (lse.scalar_type() != at::kFloat || lse.device() != q.device() || !lse.is_contiguous() || lse.sizes() != q.sizes().slice(0, q.dim() - 1))
    return py::none();
  at::AutoDispatchBelowADInplaceOrView below;
  const int64_t sq = q.size(-2), sk = k[0].size(-2), d = q.size(-1), P = (int64_t)k.size();
  Shape both{2 * P};
  both.append(k[0].sizes().begin(), k[0].sizes().end());
  const at::Tensor dq = at::empty_like(q), dkv = at::empty(both, q.options());
  const List views = dkv.unbind(0);
  const List dk(views.begin(), views.begin() + P), dv(views.begin() + P, views.end());
  const size_t nbytes = jg_attn_bwd_workspace_bytes(batch, sq, sk, d);
  const at::Tensor ws = at::empty({(int64_t)(nbytes > 4 ? nbytes : 4)}, q.options().dtype(at::kByte));
  const void *kp[kMostChunks], *vp[kMostChunks];
  void *dkp[kMostChunks], *dvp[kMostChunks];
  addresses(k, kp);
  addresses(v, vp);
  addresses(dk, dkp);
  addresses(dv, dvp);
  check(jg_attn_bwd_chunks(dq.data_ptr(), dkp, dvp, dout.data_ptr(), q.data_ptr(), kp, vp, P, out.data_ptr(), lse.data_ptr<float>(),
                           batch, sq, sk, d, (float)scale, code_of(q), ws.data_ptr(), nbytes, pointer(stream)),
        "jg_attn_bwd_chunks");
  return py::make_tuple(dq, dk, dv);
}

// (mean, var, the rank's own mean, room for the root): the row statistics before the collectives
py::object ln_partial(const at::Tensor& x, bool sharded, uintptr_t stream) {
  if (x.dim() < 1 || x.numel() == 0 || !on_gpu(x) || code_of(x) < 0) return py::none();
  at::AutoDispatchBelowADInplaceOrView below;
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  Shape shape{4};
  shape.append(x.sizes().begin(), x.sizes().end() - 1);
  shape.push_back(1);
  const List t = at::empty(shape, x.options().dtype(at::kFloat)).unbind(0);
  check(jg_ln_partial_fwd2(t[0].data_ptr<float>(), sharded ? t[2].data_ptr<float>() : nullptr, t[1].data_ptr<float>(), x.data_ptr(), rows, cols,
                           code_of(x), pointer(stream)),
        "jg_ln_partial_fwd2");
  return py::make_tuple(t[0], t[1], t[2], t[3]);
}

void ln_recentre(const at::Tensor& var, const at::Tensor& own, const at::Tensor& mean, uintptr_t stream) {
  check(jg_ln_recentre(var.data_ptr<float>(), own.data_ptr<float>(), mean.data_ptr<float>(), var.numel(), pointer(stream)), "jg_ln_recentre");
}

// (y, x_norm, var + eps) in w's type; `std` gets the root. x, w and b as the Python route has them at this point.
py::tuple ln_apply(const at::Tensor& x, const at::Tensor& mean, const at::Tensor& var, const at::Tensor& std, const at::Tensor& w,
                   const c10::optional<at::Tensor>& b, double eps, uintptr_t stream) {
  at::AutoDispatchBelowADInplaceOrView below;
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  const at::Tensor y = at::empty(x.sizes(), w.options()), x_norm = at::empty(x.sizes(), w.options()), var_eps = at::empty(mean.sizes(), w.options());
  check(jg_ln_apply2(y.data_ptr(), x_norm.data_ptr(), std.data_ptr<float>(), var_eps.data_ptr(), x.data_ptr(), mean.data_ptr<float>(),
                     var.data_ptr<float>(), w.data_ptr(), b ? b->data_ptr() : nullptr, rows, cols, (float)eps, code_of(x), code_of(w), pointer(stream)),
        "jg_ln_apply2");
  return py::make_tuple(y, x_norm, var_eps);
}

// Whether ln_apply takes these as they are: parameters in the type that y gets, nothing to be copied
bool ln_takes(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& b, const at::ScalarType type) {
  auto parameter = [&](const at::Tensor& t) {
    return on_gpu(t) && t.scalar_type() == type && t.device() == x.device() && t.dim() == 1 && t.size(0) == x.size(-1);
  };
  return x.dim() >= 1 && x.numel() > 0 && on_gpu(x) && code_of(x) >= 0 && parameter(w) && code_of(w) >= 0 && (!b || parameter(*b));
}

// (mean of g w, sum of g w x_norm, gw, gb): the backward before the collectives; parameter gradients in `like`'s type
py::object ln_partial_bwd(const at::Tensor& g, const at::Tensor& x_norm, const at::Tensor& w, const at::Tensor& std, bool need_w, bool need_b,
                          const at::ScalarType grad_type, uintptr_t stream) {
  if (g.numel() == 0 || !on_gpu(g) || !on_gpu(x_norm) || !on_gpu(w) || g.scalar_type() != x_norm.scalar_type() || g.sizes() != x_norm.sizes() ||
      w.scalar_type() != g.scalar_type() || code_of(g) < 0)
    return py::none();
  at::AutoDispatchBelowADInplaceOrView below;
  const int64_t cols = g.size(-1), rows = g.numel() / cols;
  Shape shape{2};
  shape.append(std.sizes().begin(), std.sizes().end());
  const List t = at::empty(shape, std.options()).unbind(0);
  const auto options = g.options().dtype(grad_type);
  const at::Tensor gw = need_w ? at::empty({cols}, options) : at::Tensor(), gb = need_b ? at::empty({cols}, options) : at::Tensor();
  const size_t nbytes = need_w || need_b ? jg_ln_bwd_workspace_bytes(rows, cols) : 0;
  const at::Tensor ws = at::empty({(int64_t)(nbytes > 4 ? nbytes : 4)}, g.options().dtype(at::kByte));
  const int code = grad_type == at::kFloat ? JG_F32 : grad_type == at::kBFloat16 ? JG_BF16 : JG_F16;
  check(jg_ln_partial_bwd2(t[0].data_ptr<float>(), t[1].data_ptr<float>(), need_w ? gw.data_ptr() : nullptr, need_b ? gb.data_ptr() : nullptr, code,
                           g.data_ptr(), x_norm.data_ptr(), w.data_ptr(), rows, cols, code_of(g), ws.data_ptr(), nbytes, pointer(stream)),
        "jg_ln_partial_bwd2");
  return py::make_tuple(t[0], t[1], need_w ? py::cast(gw) : py::none(), need_b ? py::cast(gb) : py::none());
}

at::Tensor ln_bwd_apply(const at::Tensor& g, const at::Tensor& x_norm, const at::Tensor& w, const at::Tensor& mean, const at::Tensor& dot,
                        const at::Tensor& std, int64_t n_global, uintptr_t stream) {
  at::AutoDispatchBelowADInplaceOrView below;
  const int64_t cols = g.size(-1), rows = g.numel() / cols;
  const at::Tensor gx = at::empty_like(g);
  check(jg_ln_bwd_apply(gx.data_ptr(), g.data_ptr(), x_norm.data_ptr(), w.data_ptr(), mean.data_ptr<float>(), dot.data_ptr<float>(),
                        std.data_ptr<float>(), rows, cols, n_global, code_of(g), pointer(stream)),
        "jg_ln_bwd_apply");
  return gx;
}

bool like_channels(const c10::optional<at::Tensor>& t, const at::Tensor& x) {
  return !t || (on_gpu(*t) && t->scalar_type() == x.scalar_type() && t->device() == x.device() && t->dim() == 1 && t->size(0) == x.size(1));
}

// (y, the copy of x or None, mean, rstd)
py::object gn_forward(const at::Tensor& x, int64_t groups, const c10::optional<at::Tensor>& w, const c10::optional<at::Tensor>& b, double eps,
                      bool keep, uintptr_t stream) {
  if (x.dim() < 2 || x.numel() == 0 || !on_gpu(x) || code_of(x) < 0 || !like_channels(w, x) || !like_channels(b, x)) return py::none();
  at::AutoDispatchBelowADInplaceOrView below;
  const int64_t n = x.size(0), c = x.size(1), s = x.numel() / (n * c);
  const at::Tensor y = at::empty_like(x), kept = keep ? at::empty_like(x) : at::Tensor();
  const List t = at::empty({2, n, groups}, x.options().dtype(at::kFloat)).unbind(0);
  const size_t nbytes = jg_gn_workspace_bytes(n, c, s);
  const at::Tensor ws = at::empty({(int64_t)nbytes}, x.options().dtype(at::kByte));
  check(jg_gn_forward_keep(y.data_ptr(), keep ? kept.data_ptr() : nullptr, t[0].data_ptr<float>(), t[1].data_ptr<float>(), x.data_ptr(),
                           w ? w->data_ptr() : nullptr, b ? b->data_ptr() : nullptr, n, c, s, groups, (float)eps, code_of(x), ws.data_ptr(), nbytes,
                           pointer(stream)),
        "jg_gn_forward_keep");
  return py::make_tuple(y, keep ? py::cast(kept) : py::none(), t[0], t[1]);
}

// (gx, gw, gb); the parameter gradients in `grad_type`
py::object gn_backward(const at::Tensor& g, const at::Tensor& x, const at::Tensor& mean, const at::Tensor& rstd, const c10::optional<at::Tensor>& w,
                       int64_t groups, bool need_x, bool need_w, bool need_b, const at::ScalarType grad_type, uintptr_t stream) {
  if (g.numel() == 0 || !on_gpu(g) || !on_gpu(x) || g.scalar_type() != x.scalar_type() || g.sizes() != x.sizes() || code_of(g) < 0 ||
      !like_channels(w, x))
    return py::none();
  at::AutoDispatchBelowADInplaceOrView below;
  const int64_t n = x.size(0), c = x.size(1), s = x.numel() / (n * c);
  const auto options = g.options().dtype(grad_type);
  const at::Tensor gx = need_x ? at::empty_like(g) : at::Tensor(), gw = need_w ? at::empty({c}, options) : at::Tensor(),
                   gb = need_b ? at::empty({c}, options) : at::Tensor();
  const size_t nbytes = jg_gn_workspace_bytes(n, c, s);
  const at::Tensor ws = at::empty({(int64_t)nbytes}, x.options().dtype(at::kByte));
  const int code = grad_type == at::kFloat ? JG_F32 : grad_type == at::kBFloat16 ? JG_BF16 : JG_F16;
  check(jg_gn_backward(need_x ? gx.data_ptr() : nullptr, need_w ? gw.data_ptr() : nullptr, need_b ? gb.data_ptr() : nullptr, g.data_ptr(), x.data_ptr(),
                       mean.data_ptr<float>(), rstd.data_ptr<float>(), w ? w->data_ptr() : nullptr, n, c, s, groups, code_of(x), code,
                       ws.data_ptr(), nbytes, pointer(stream)),
        "jg_gn_backward");
  auto given = [](const at::Tensor& t) -> py::object { return t.defined() ? py::cast(t) : py::none(); };
  return py::make_tuple(given(gx), given(gw), given(gb));
}

// ---- projections around attention and the Swin block: the launches of projection.py and swin._WholeBlock in their order, for
// tensors that need neither a cast nor a copy; None for all others, before anything is launched. Host time of a step, with
// autograd's own: Swin block 573 us through Python, 334 here (its kernels take about 450 of 65536 tokens of 128 channels, less of
// fewer); the two projections 213 and 164.
struct Heads {  // (B, H, S, D) of the head layout
  int64_t b = 1, h = 1, s = 1, d = 1;
};

at::Tensor f32(const at::Tensor& like, at::IntArrayRef shape) { return at::empty(shape, like.options().dtype(at::kFloat)); }
at::Tensor bytes(const at::Tensor& like, size_t n) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }

// out(r, n) = sum_k a(r, k) w[n][k] (+ b[n])
void nt(const at::Tensor& out, const at::Tensor& a, const at::Tensor& w, const at::Tensor* b, int64_t rows, bool a_heads, bool out_heads,
        const Heads& l, void* s) {
  check(jg_proj_nt(out.data_ptr(), a.data_ptr(), w.data_ptr(), b ? b->data_ptr() : nullptr, code_of(a), rows, w.size(0), w.size(1), a_heads, out_heads,
                   l.b, l.h, l.s, l.d, s),
        "jg_proj_nt");
}
void nt_fused(const at::Tensor& out, const at::Tensor& aux, int epilogue, const at::Tensor& a, const at::Tensor& w, const at::Tensor* b, int64_t rows, void* s) {
  check(jg_proj_nt_fused(out.data_ptr(), aux.data_ptr(), epilogue, a.data_ptr(), w.data_ptr(), b ? b->data_ptr() : nullptr, code_of(a), rows, w.size(0),
                         w.size(1), s),
        "jg_proj_nt_fused");
}
// (gw, gb): gradients of a weight (n, c) and its bias from the gradient and the input of its layer
// With `later` the sums of the partials are left to it, and the partials to `held`.
struct Later {
  jg_reductions sums = {};
  List held;
};
std::pair<at::Tensor, at::Tensor> tn(const at::Tensor& g, const at::Tensor& x, int64_t rows, int64_t n, int64_t c, bool g_heads, bool x_heads, const Heads& l,
                                     bool need_b, at::ScalarType grad_type, void* s, Later* later = nullptr) {
  const auto options = g.options().dtype(grad_type);
  const at::Tensor gw = at::empty({n, c}, options), gb = need_b ? at::empty({n}, options) : at::Tensor();
  const size_t nbytes = jg_proj_tn_workspace(rows, n, c);
  const at::Tensor ws = bytes(g, std::max<size_t>(nbytes, 16));
  if (later != nullptr) {
    later->held.push_back(ws);
    check(jg_proj_tn_later(&later->sums, gw.data_ptr(), need_b ? gb.data_ptr() : nullptr, g.data_ptr(), x.data_ptr(), code_of(g),
                           grad_type == at::kFloat ? JG_F32 : code_of(g), rows, n, c, g_heads, x_heads, l.b, l.h, l.s, l.d, ws.data_ptr(), nbytes, s),
          "jg_proj_tn_later");
    return {gw, gb};
  }
  check(jg_proj_tn(gw.data_ptr(), need_b ? gb.data_ptr() : nullptr, g.data_ptr(), x.data_ptr(), code_of(g), grad_type == at::kFloat ? JG_F32 : code_of(g),
                   rows, n, c, g_heads, x_heads, l.b, l.h, l.s, l.d, ws.data_ptr(), nbytes, s),
        "jg_proj_tn");
  return {gw, gb};
}
at::Tensor turned(const at::Tensor& w, void* s) {  // projection._transpose
  const int64_t n = w.size(0), k = w.size(1);
  if (w.element_size() != 2 || n % 8 != 0 || k % 8 != 0 || !aligned(w)) return w.t().contiguous();
  const at::Tensor out = at::empty({k, n}, w.options());
  check(jg_transpose16(out.data_ptr(), w.data_ptr(), n, k, s), "jg_transpose16");
  return out;
}

bool projection_ok(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& b) {
  return on_gpu(x) && on_gpu(w) && x.numel() > 0 && w.numel() > 0 && w.dim() == 2 && code_of(x) >= 0 && w.scalar_type() == x.scalar_type() &&
         w.device() == x.device() &&
         (!b || (on_gpu(*b) && b->dim() == 1 && b->size(0) == w.size(0) && b->scalar_type() == x.scalar_type() && b->device() == x.device()));
}

// (*lead, s, C) -> (3, *lead, heads, s, d)
py::object qkv_forward(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& b, int64_t heads, uintptr_t stream) {
  if (x.dim() < 2 || !projection_ok(x, w, b) || x.size(-1) != w.size(1) || heads < 1 || w.size(0) % (3 * heads) != 0) return py::none();
  at::AutoDispatchBelowADInplaceOrView below;
  const int64_t s = x.size(-2), rows = x.numel() / x.size(-1), d = w.size(0) / (3 * heads);
  Shape shape{3};
  shape.append(x.sizes().begin(), x.sizes().end() - 2);
  for (int64_t v : {heads, s, d}) shape.push_back(v);
  const at::Tensor out = at::empty(shape, x.options());
  nt(out, x, w, b ? &*b : nullptr, rows, false, true, {rows / s, heads, s, d}, pointer(stream));
  return py::cast(out);
}

// (*lead, heads, s, d) -> (*lead, s, n)
py::object heads_forward(const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& b, uintptr_t stream) {
  if (x.dim() < 3 || !projection_ok(x, w, b) || x.size(-3) * x.size(-1) != w.size(1)) return py::none();
  at::AutoDispatchBelowADInplaceOrView below;
  const int64_t h = x.size(-3), s = x.size(-2), d = x.size(-1), rows = x.numel() / (h * d);
  Shape shape(x.sizes().begin(), x.sizes().end() - 3);
  for (int64_t v : {s, w.size(0)}) shape.push_back(v);
  const at::Tensor out = at::empty(shape, x.options());
  nt(out, x, w, b ? &*b : nullptr, rows, true, false, {rows / s, h, s, d}, pointer(stream));
  return py::cast(out);
}

// (gx, gw, gb) of either; `qkv`: the gradient is in the head layout and x is not, else the other way round
py::object projection_backward(const at::Tensor& g, const at::Tensor& x, const at::Tensor& w, bool qkv, int64_t b, int64_t h, int64_t sq, int64_t d,
                               bool need_x, bool need_w, bool need_b, uintptr_t stream) {
  const int64_t n = w.size(0), c = w.size(1), rows = b * sq;
  if (!on_gpu(g) || !projection_ok(x, w, c10::nullopt) || g.scalar_type() != x.scalar_type() || g.device() != x.device() || g.numel() != rows * n ||
      x.numel() != rows * c)
    return py::none();
  at::AutoDispatchBelowADInplaceOrView below;
  void* const s = pointer(stream);
  const Heads l{b, h, sq, d};
  at::Tensor gx, gw, gb;
  if (need_x) {
    gx = at::empty_like(x);
    nt(gx, g, turned(w, s), nullptr, rows, qkv, !qkv, l, s);
  }
  if (need_w || need_b) std::tie(gw, gb) = tn(g, x, rows, n, c, qkv, !qkv, l, need_b, g.scalar_type(), s);
  auto given = [](const at::Tensor& t, bool wanted) -> py::object { return wanted ? py::cast(t) : py::none(); };
  return py::make_tuple(given(gx, need_x), given(gw, need_w), given(gb, need_b));
}

// One pass of swin._WholeBlock with bf16 tokens and fp32 parameters on a grid that wraps inside the rank: what its backward reads.
// The block's parameters in the order of swin._WholeBlock.forward.
enum Param { N1W, N1B, QKV_W, QKV_B, TABLE, PROJ_W, PROJ_B, N2W, N2B, FC1_W, FC1_B, FC2_W, FC2_B, PARAMS };

class SwinPass {
 public:
  // (result, pass) or None
  static py::object forward(const at::Tensor& x, const List& p, const c10::optional<at::Tensor>& side, int64_t heads, int64_t shift, double eps,
                            uintptr_t stream) {
    if (x.dim() != 4 || x.numel() == 0 || !on_gpu(x) || !aligned(x) || x.scalar_type() != at::kBFloat16 || p.size() != PARAMS) return py::none();
    const int64_t b = x.size(0), h = x.size(1), w = x.size(2), c = x.size(3), tokens = h * w, hidden = p[FC1_W].dim() == 2 ? p[FC1_W].size(0) : 0;
    if (c != 32 * heads || h % 8 != 0 || w % 8 != 0 || hidden == 0 || hidden % 8 != 0 || !jg_ln_plain_supported(c)) return py::none();
    const Shape want[PARAMS] = {{c}, {c}, {3 * c, c}, {3 * c}, {225, heads}, {c, c}, {c}, {c}, {c}, {hidden, c}, {hidden}, {c, hidden}, {c}};
    for (int i = 0; i < PARAMS; ++i)
      if (!on_gpu(p[i]) || p[i].scalar_type() != at::kFloat || p[i].device() != x.device() || p[i].sizes() != at::IntArrayRef(want[i])) return py::none();
    if (side && (!on_gpu(*side) || side->scalar_type() != at::kByte || side->numel() != tokens || side->device() != x.device())) return py::none();
    at::AutoDispatchBelowADInplaceOrView below;
    auto pass = std::make_unique<SwinPass>();
    SwinPass& t = *pass;
    void* const s = pointer(stream);
    const int64_t rows = b * tokens;
    t.x = x, t.n1w = p[N1W], t.n2w = p[N2W], t.table = p[TABLE], t.l = {b, heads, tokens, 32}, t.h = h, t.w = w, t.shift = shift;
    if (side) t.side = *side;
    t.cast(p, s);
    t.y1 = t.norm(x, p[N1W], p[N1B], t.mean1, t.rstd1, eps, s);
    t.qkv = at::empty({3, b, heads, tokens, 32}, x.options());
    nt(t.qkv, t.y1, t.wc[0], &t.bc[0], rows, false, true, t.l, s);
    t.out = at::empty({b, heads, tokens, 32}, x.options());
    t.lse = f32(x, {rows * heads});
    const char* const q = static_cast<const char*>(t.qkv.data_ptr());
    const int64_t part = 2 * rows * c;
    check(jg_attn_swin_shifted_fwd(t.out.data_ptr(), t.lse.data_ptr<float>(), q, q + part, q + 2 * part, t.table.data_ptr<float>(), t.codes(), b, heads, h,
                                   w, t.shift_y(), t.shift_x(), 32, (float)t.scale(), JG_BF16, s),
          "jg_attn_swin_shifted_fwd");
    t.x1 = at::empty_like(x);
    check(jg_proj_nt_fused_heads(t.x1.data_ptr(), x.data_ptr(), JG_EPI_ADD, t.out.data_ptr(), t.wc[1].data_ptr(), t.bc[1].data_ptr(), JG_BF16, rows, c, c, 1, b,
                                 heads, tokens, 32, s),
          "jg_proj_nt_fused_heads");
    t.y2 = t.norm(t.x1, p[N2W], p[N2B], t.mean2, t.rstd2, eps, s);
    t.pre = at::empty({b, h, w, hidden}, x.options());
    t.act = at::empty_like(t.pre);
    nt_fused(t.pre, t.act, JG_EPI_GELU, t.y2, t.wc[2], &t.bc[2], rows, s);
    const at::Tensor y = at::empty_like(x);
    nt_fused(y, t.x1, JG_EPI_ADD, t.act, t.wc[3], &t.bc[3], rows, s);
    return py::make_tuple(y, std::move(pass));
  }

  // Gradients of x (None unless wanted) and of the parameters, or None. A tensor goes with its last launch, what the forward kept
  // among them, so that there is room for the partials, which wait for the sums at the end: the peak over what the forward holds is 17 MB at
  // 65536 tokens of 128 channels and 68 at 262144 of 256, 279 and 1879 with all of it kept until the end (136 and 1080 through
  // Python), and the memory that comes back at once is still in the caches (the first step 441 -> 427 us). The pass keeps nothing afterwards.
  py::object backward(const at::Tensor& grad, bool need_x, uintptr_t stream) {
    if (!x.defined() || grad.sizes() != x.sizes() || !on_gpu(grad) || !aligned(grad) || grad.scalar_type() != at::kBFloat16 || grad.device() != x.device())
      return py::none();
    at::AutoDispatchBelowADInplaceOrView below;
    void* const s = pointer(stream);
    const int64_t c = x.size(3), rows = l.b * l.s, hidden = pre.size(3);
    const Heads flat;
    at::Tensor g[PARAMS];
    Later later;  // every parameter's sums of partials in one launch at the end
    auto drop = [](auto&... done) { (done.reset(), ...); };
    std::tie(g[FC2_W], g[FC2_B]) = tn(grad, act, rows, c, hidden, false, false, flat, true, at::kFloat, s, &later);
    drop(act);
    at::Tensor dpre = at::empty_like(pre);
    nt_fused(dpre, pre, JG_EPI_DGELU, grad, wt[3], nullptr, rows, s);
    drop(pre);
    std::tie(g[FC1_W], g[FC1_B]) = tn(dpre, y2, rows, hidden, c, false, false, flat, true, at::kFloat, s, &later);
    drop(y2);
    at::Tensor gy2 = at::empty_like(x);
    nt(gy2, dpre, wt[2], nullptr, rows, false, false, flat, s);
    drop(dpre);
    const at::Tensor gx1 = norm_backward(gy2, grad, x1, mean2, rstd2, n2w, true, &g[N2W], &g[N2B], later, s);
    drop(gy2, x1);
    at::Tensor gout = at::empty_like(out);
    nt(gout, gx1, wt[1], nullptr, rows, false, true, l, s);
    std::tie(g[PROJ_W], g[PROJ_B]) = tn(gx1, out, rows, c, c, false, true, l, true, at::kFloat, s, &later);
    at::Tensor dqkv = at::empty_like(qkv);
    g[TABLE] = at::empty_like(table);
    const size_t nbytes = jg_attn_swin_bwd_workspace_bytes(l.b, l.h, h, w);
    const at::Tensor ws = bytes(x, nbytes);
    const char* const q = static_cast<const char*>(qkv.data_ptr());
    char* const dq = static_cast<char*>(dqkv.data_ptr());
    const int64_t part = 2 * rows * c;
    check(jg_attn_swin_shifted_bwd_later(&later.sums, dq, dq + part, dq + 2 * part, g[TABLE].data_ptr<float>(), gout.data_ptr(), q, q + part, q + 2 * part,
                                         out.data_ptr(), lse.data_ptr<float>(), table.data_ptr<float>(), codes(), l.b, l.h, h, w, shift_y(), shift_x(), 32,
                                         (float)scale(), JG_BF16, ws.data_ptr(), nbytes, s),
          "jg_attn_swin_shifted_bwd_later");
    drop(gout, out, qkv);
    const at::Tensor gy = at::empty_like(x);
    nt(gy, dqkv, wt[0], nullptr, rows, true, false, l, s);
    std::tie(g[QKV_W], g[QKV_B]) = tn(dqkv, y1, rows, 3 * c, c, true, false, l, true, at::kFloat, s, &later);
    drop(dqkv, y1);
    const at::Tensor gx = norm_backward(gy, gx1, x, mean1, rstd1, n1w, need_x, &g[N1W], &g[N1B], later, s);
    check(jg_reduce_many(&later.sums, s), "jg_reduce_many");
    py::tuple all(1 + PARAMS);
    all[0] = need_x ? py::cast(gx) : py::none();
    for (int i = 0; i < PARAMS; ++i) all[1 + i] = py::cast(g[i]);
    *this = SwinPass();
    return std::move(all);
  }

 private:
  // bf16 copies of the four weights, their transposes and the biases in one launch (projection.cast_parameters)
  void cast(const List& p, void* s) {
    const int weight[4] = {QKV_W, PROJ_W, FC1_W, FC2_W}, bias[4] = {QKV_B, PROJ_B, FC1_B, FC2_B};
    int64_t total = 0;
    auto room = [&](const at::Tensor& t) { const int64_t at = total; total += (t.numel() + 7) / 8 * 8; return at; };
    int64_t at_w[4], at_wt[4], at_b[4];
    for (int i = 0; i < 4; ++i) at_w[i] = room(p[weight[i]]), at_wt[i] = room(p[weight[i]]), at_b[i] = room(p[bias[i]]);
    const at::Tensor flat_ = at::empty({total}, x.options());
    void *dst[8], *dst_t[8] = {};
    const void* src[8];
    int32_t rows[8], cols[8];
    for (int i = 0; i < 4; ++i) {
      const int64_t n = p[weight[i]].size(0), k = p[weight[i]].size(1);
      wc[i] = at::as_strided(flat_, {n, k}, {k, 1}, at_w[i]);
      wt[i] = at::as_strided(flat_, {k, n}, {n, 1}, at_wt[i]);
      bc[i] = at::as_strided(flat_, {n}, {1}, at_b[i]);
      dst[i] = wc[i].data_ptr(), dst_t[i] = wt[i].data_ptr(), src[i] = p[weight[i]].data_ptr(), rows[i] = n, cols[i] = k;
      dst[4 + i] = bc[i].data_ptr(), src[4 + i] = p[bias[i]].data_ptr(), rows[4 + i] = 1, cols[4 + i] = n;
    }
    check(jg_cast_params(dst, dst_t, src, rows, cols, 8, s), "jg_cast_params");
  }
  static at::Tensor norm(const at::Tensor& x, const at::Tensor& w, const at::Tensor& b, at::Tensor& mean, at::Tensor& rstd, double eps, void* s) {
    const int64_t cols = x.size(-1), rows = x.numel() / cols;
    const at::Tensor y = at::empty_like(x);
    mean = f32(x, {rows});
    rstd = f32(x, {rows});
    check(jg_ln_plain_fwd(y.data_ptr(), mean.data_ptr<float>(), rstd.data_ptr<float>(), x.data_ptr(), w.data_ptr<float>(), b.data_ptr<float>(), rows, cols,
                          (float)eps, JG_BF16, JG_BF16, s),
          "jg_ln_plain_fwd");
    return y;
  }
  // the gradient of the norm's input with what reaches it past the norm (`over`) added, if wanted; gw, gb
  static at::Tensor norm_backward(const at::Tensor& g, const at::Tensor& over, const at::Tensor& x, const at::Tensor& mean, const at::Tensor& rstd,
                                  const at::Tensor& w, bool need_x, at::Tensor* gw, at::Tensor* gb, Later& later, void* s) {
    const int64_t cols = x.size(-1), rows = x.numel() / cols;
    const at::Tensor gx = need_x ? at::empty_like(x) : at::Tensor();
    *gw = f32(x, {cols});
    *gb = f32(x, {cols});
    const size_t nbytes = jg_ln_plain_bwd_workspace_bytes(rows, cols);
    const at::Tensor ws = bytes(x, std::max<size_t>(nbytes, 4));
    later.held.push_back(ws);
    check(jg_ln_plain_bwd_later(&later.sums, need_x ? gx.data_ptr() : nullptr, gw->data_ptr<float>(), gb->data_ptr<float>(), g.data_ptr(), x.data_ptr(),
                                mean.data_ptr<float>(), rstd.data_ptr<float>(), w.data_ptr<float>(), rows, cols, JG_BF16, JG_BF16, ws.data_ptr(), nbytes,
                                need_x ? over.data_ptr() : nullptr, s),
          "jg_ln_plain_bwd_later");
    return gx;
  }
  const uint8_t* codes() const { return side.defined() ? side.data_ptr<uint8_t>() : nullptr; }
  int64_t shift_y() const { return (shift % h + h) % h; }
  int64_t shift_x() const { return (shift % w + w) % w; }
  static double scale() { return std::pow(32.0, -0.5); }

  at::Tensor x, n1w, n2w, table, side, y1, mean1, rstd1, qkv, out, lse, x1, y2, mean2, rstd2, pre, act;
  at::Tensor wc[4], wt[4], bc[4];  // qkv, output projection, the MLP's two layers
  Heads l;
  int64_t h = 0, w = 0, shift = 0;
};

// ---- backward(ctx, grad) of the functions of _autograd.NativeFunction. The engine calls them on a thread of its own with no Python function in
// between: there Python's objects come from the other thread's core one cache line at a time, and a function of 20 lines took 10 us and more.
uintptr_t current_stream(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(c10::hip::getCurrentHIPStream(t.device().index()).stream()); }

// What a function's ctx holds
struct Context {
  explicit Context(const py::object& ctx) : saved(ctx.attr("saved_tensors")), needs(ctx.attr("needs_input_grad")), rest(ctx.attr("rest")) {}
  // Saved tensor i row-major, as the kernels' pointers take it: hooks may have given it another layout
  at::Tensor rows(size_t i) const { return saved[i].cast<at::Tensor>().contiguous(); }
  bool need(size_t i) const { return needs[4 + i].cast<bool>(); }
  py::tuple saved, needs, rest;
};
// The gradients of (result, saved, rest, zeros, x, weight, bias)
py::tuple gradients(const py::object& x, const py::object& w, const py::object& b) {
  const py::object none = py::none();
  return py::make_tuple(none, none, none, none, x, w, b);
}

// rest: the plan, _ConvNd's arguments from the stride on, the tile's extents
py::object conv_backward(const py::object& ctx, const py::object& grad) {
  const py::object none = py::none();
  if (grad.is_none()) return gradients(none, none, none);
  const Context c(ctx);
  const at::Tensor g = grad.cast<at::Tensor>();
  const py::tuple args = c.rest[1];
  const py::handle config = args[5];
  Step& step = c.rest[0].cast<Step&>();
  const uintptr_t stream = current_stream(g);
  const bool need_x = c.need(0), need_w = c.need(1), need_b = c.need(2);
  const py::object got = step.backward(g, c.saved[0].cast<at::Tensor>(), c.saved[1].cast<at::Tensor>(), need_x, need_w, need_w && need_b, stream);
  if (got.is_none()) return py::module_::import("jigsaw_amd.conv").attr("_backward_without_plan")(ctx, grad);
  const py::tuple parts = got;
  const py::object gb = need_b && parts[2].is_none() ? py::object(config.attr("grad_bias")(g.contiguous())) : py::object(parts[2]);
  if (!need_x) return gradients(none, parts[1], gb);
  const py::object recv = step.sends() ? py::object(config.attr("halo_exchange").attr("backward")(parts[3])) : py::dict();
  py::object gx = step.finish(parts[0].cast<at::Tensor>(), parts[4].cast<bool>(), recv, stream, parts[5]);
  if (gx.is_none()) gx = py::module_::import("jigsaw_amd.conv").attr("_fold_without_plan")(parts[0], parts[4], recv, c.saved[1], c.rest[2], *args);
  return gradients(gx, parts[1], gb);
}

// rest: all_reduce(tensor, "avg" | "sum", group), the group, its size, the type of x and of the parameters
py::object ln_backward(const py::object& ctx, const py::object& grad) {
  const py::object none = py::none();
  if (grad.is_none()) return gradients(none, none, none);
  const Context c(ctx);
  const at::Tensor x_norm = c.rows(0), w = c.rows(1), std = c.rows(2), g = grad.cast<at::Tensor>().to(x_norm.scalar_type()).contiguous();
  const py::object& reduce = c.rest[0];
  const int64_t ranks = c.rest[2].cast<int64_t>();
  const uintptr_t stream = current_stream(g);
  const py::object got = ln_partial_bwd(g, x_norm, w, std, c.need(1), c.need(2), c.rest[4].cast<at::ScalarType>(), stream);
  TORCH_CHECK(!got.is_none(), "layer_norm: what the backward got is not what the forward saved");
  const py::tuple parts = got;
  if (!c.need(0)) return gradients(none, parts[2], parts[3]);
  if (ranks > 1) {
    reduce(parts[0], "avg", c.rest[1]);
    reduce(parts[1], "sum", c.rest[1]);
  }
  const at::Tensor gx = ln_bwd_apply(g, x_norm, w, parts[0].cast<at::Tensor>(), parts[1].cast<at::Tensor>(), std, x_norm.size(-1) * ranks, stream);
  return gradients(py::cast(gx.to(c.rest[3].cast<at::ScalarType>())), parts[2], parts[3]);
}

// rest: the number of groups, the type of the parameters
py::object gn_output_backward(const py::object& ctx, const at::Tensor& grad) {
  const Context c(ctx);
  const at::Tensor x = c.rows(0);
  const at::Tensor g = grad.to(x.scalar_type()).contiguous();
  const c10::optional<at::Tensor> w = c.saved[3].is_none() ? c10::nullopt : c10::optional<at::Tensor>(c.rows(3));
  const py::object got = gn_backward(g, x, c.rows(1), c.rows(2), w, c.rest[0].cast<int64_t>(), c.need(0), c.need(1), c.need(2),
                                     c.rest[1].cast<at::ScalarType>(), current_stream(g));
  TORCH_CHECK(!got.is_none(), "group_norm: what the backward got is not what the forward saved");
  const py::tuple all = got;
  return gradients(all[0], all[1], all[2]);
}

// rest: projection_backward, whether it is the qkv projection's, batch, heads, tokens and columns of a head
py::object projection_node_backward(const py::object& ctx, const at::Tensor& grad) {
  const Context c(ctx);
  const at::Tensor g = grad.contiguous();
  const py::object got = c.rest[0](g, c.rows(0), c.rows(1), c.rest[1], c.rest[2], c.rest[3], c.rest[4], c.rest[5], c.need(0), c.need(1), c.need(2), current_stream(g));
  TORCH_CHECK(!got.is_none(), "projection: what the backward got is not what the forward saved");
  const py::tuple all = got;
  return gradients(all[0], all[1], all[2]);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  // functions that a class may hold as methods
  auto method = [&](const char* name, auto f) { m.attr(name) = py::cpp_function(f, py::name(name), py::is_method(py::none())); };
  method("conv_backward", &conv_backward);
  method("ln_backward", &ln_backward);
  method("gn_output_backward", &gn_output_backward);
  method("projection_node_backward", &projection_node_backward);
  py::class_<SumsLeft>(m, "SumsLeft");
  py::class_<Step>(m, "Step")
      .def(py::init<const py::tuple&, const py::tuple&, const py::tuple&, const py::tuple&, int, int, uintptr_t, uintptr_t, bool,
                    uintptr_t, const std::vector<size_t>&, const py::list&, const py::list&, const py::list&, const py::list&, bool>())
      .def_property_readonly("sends", &Step::sends)
      .def("takes", &Step::takes)
      .def("pack", &Step::pack)
      .def("forward", &Step::forward)
      .def("backward", &Step::backward)
      .def("finish", &Step::finish);
  m.def("may_want_64_columns", &may_want_64_columns);
  m.def("ring_forward", &ring_forward<false>);
  m.def("ring_forward_at_own_width", &ring_forward<true>);
  m.def("ring_backward", &ring_backward<false>);
  m.def("ring_backward_at_own_width", &ring_backward<true>);
  m.def("ln_takes", &ln_takes);
  m.def("ln_partial", &ln_partial);
  m.def("ln_recentre", &ln_recentre);
  m.def("ln_apply", &ln_apply);
  m.def("ln_partial_bwd", &ln_partial_bwd);
  m.def("ln_bwd_apply", &ln_bwd_apply);
  m.def("gn_forward", &gn_forward);
  m.def("gn_backward", &gn_backward);
  m.def("qkv_forward", &qkv_forward);
  m.def("heads_forward", &heads_forward);
  m.def("projection_backward", &projection_backward);
  py::class_<SwinPass>(m, "SwinPass").def("backward", &SwinPass::backward);
  m.def("swin_forward", &SwinPass::forward);
}
