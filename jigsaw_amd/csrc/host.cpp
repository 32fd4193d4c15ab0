// Host side of the distributed convolution's step: allocations, strips, pointer tables and the calls into
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
#include <torch/extension.h>

#include <atomic>
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
        send_bwd_(strips(send_bwd)), fold_(try_fold) {}

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
    if (x.sizes() != at::IntArrayRef(x_shape_) || !x.is_contiguous() || w_any.sizes() != at::IntArrayRef(w_shape_) ||
        !same_kind(w_any, x) || (b_any && (!same_kind(*b_any, x) || b_any->dim() != 1 || b_any->size(0) != w_shape_[0])) ||
        !table(recv, recv_fwd_, x, src))
      return py::none();
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

  // (input gradient, weight gradient, bias gradient, strips to send, folded) or None. The input gradient is the
  // padded one, or with `folded` the own tile's, to which only the neighbours' blocks are still missing. The
  // bias gradient is None where only the separate kernels cover the layer.
  py::object backward(const at::Tensor& g_any, const at::Tensor& x_aug, const at::Tensor& w_any, bool need_x, bool need_w, bool need_b,
                      uintptr_t stream) {
    if (g_any.sizes() != at::IntArrayRef(y_shape_) || x_aug.sizes() != at::IntArrayRef(padded_) || !x_aug.is_contiguous() ||
        w_any.sizes() != at::IntArrayRef(w_shape_) || !same_kind(g_any, x_aug) || !same_kind(w_any, x_aug))
      return py::none();
    at::AutoDispatchBelowADInplaceOrView below;
    void* const s = reinterpret_cast<void*>(stream);
    const at::Tensor g = g_any.contiguous(), w = w_any.contiguous();
    py::object gw = py::none(), gb = py::none(), gx = py::none(), send = py::dict();
    bool folded = false;
    if (need_w) {
      const at::Tensor gw_t = at::empty(w_shape_, g.options());
      const at::Tensor ws = scratch(nbytes_[JG_CONV_WGRAD], g);
      int rc = JG_ERR_UNSUPPORTED;
      if (need_b) {
        const at::Tensor gb_t = at::empty({w_shape_[0]}, g.options());
        rc = jg_conv_wgrad_bias(gw_t.data_ptr(), gb_t.data_ptr(), x_aug.data_ptr(), g.data_ptr(), &desc_, code_, address(ws),
                                nbytes_[JG_CONV_WGRAD], s);
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
      if (!folded) {
        const at::Tensor need = at::empty(padded_, g.options());
        check(jg_conv_dgrad(need.data_ptr(), w.data_ptr(), g.data_ptr(), &desc_, code_, address(ws), nbytes_[JG_CONV_DGRAD], s),
              "jg_conv_dgrad");
        gx = py::cast(need);
        if (!send_bwd_.empty()) send = cut(need, send_bwd_, own_, 1, stream);
      }
    }
    return py::make_tuple(gx, gw, gb, send, folded);
  }

  // The own tile's gradient from what `backward` returned and the neighbours' blocks, or None.
  py::object finish(const at::Tensor& part, bool folded, const py::object& recv, uintptr_t stream) const {
    const void* tab[27] = {};
    if (!table(recv, recv_bwd_, part, tab)) return py::none();
    at::AutoDispatchBelowADInplaceOrView below;
    void* const s = reinterpret_cast<void*>(stream);
    at::Tensor gx = part;
    const void* none[27] = {};
    if (!folded) {
      gx = at::empty(x_shape_, part.options());
      // where the neighbours' blocks are not as wide as the own halos, the own part first and the blocks by their widths
      check(jg_halo_fold_3d(gx.data_ptr(), part.data_ptr(), same_ ? tab : none, &own_, code_, s), "jg_halo_fold_3d");
    }
    if (folded || !same_) check(jg_halo_fold_border_3d(gx.data_ptr(), tab, &theirs_, code_, s), "jg_halo_fold_border_3d");
    return py::cast(gx);
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
  std::atomic<bool> fold_;
};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  py::class_<Step>(m, "Step")
      .def(py::init<const py::tuple&, const py::tuple&, const py::tuple&, const py::tuple&, int, int, uintptr_t, uintptr_t, bool,
                    uintptr_t, const std::vector<size_t>&, const py::list&, const py::list&, const py::list&, const py::list&, bool>())
      .def_property_readonly("sends", &Step::sends)
      .def("pack", &Step::pack)
      .def("forward", &Step::forward)
      .def("backward", &Step::backward)
      .def("finish", &Step::finish);
}
