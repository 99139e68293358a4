// The eager front-end of the scans: what armhackathon_amd/op.py, mamba3.py,
// mamba3_noncausal.py, mamba3_block.py and ss2d.py do around the C ABI (the checks, the
// contiguous copies, the outputs, the stream), natively, for plain eager calls.
//
// Why: at the small end the kernels take 5 to 20 us and the host decides the time of a
// call. A custom op written in Python took 27 us before its kernel's launch (its
// dispatcher layers 10 to 15, the rest the wrapper and ctypes), and the stream-ordered
// allocation of the scratch of a scan 9 to 14 us more (hipMallocFromPoolAsync and
// hipFreeAsync, where torch's caching allocator takes 1). Host time of a call, before and
// with this: the two steps of a decode token 60 -> 16.5 us, a scan of L 64 31 -> 9, a
// Mamba-3 scan of L 64 66 -> 13.
//
// Every function returns None when the call is not the plain one it serves, and the
// Python caller then goes through the custom op, which checks, raises and dispatches as
// it always did. Plain means: CUDA float32 strided tensors of torch's own classes on one
// device, no gradient to record, no forward-mode tangent, and nothing between the caller
// and the kernels (no dispatch or function mode, functorch transform, tracer). Autocast is not
// looked at: the ops have no autocast rule, and float32 arguments stay float32 under it on
// either route.
// A shape or argument that a check would refuse is not plain either, nor is an error from
// the C ABI: the custom op's own path reports both.
//
// The C ABI's functions are given by address (bind()), so that they are those of the
// library that _ffi.py loaded.

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/version.h>

#include <array>
#include <initializer_list>
#include <vector>

#include "../../include/arm_scan_hip.h"

namespace py = pybind11;

namespace {

struct Abi {
  decltype(&arm_scan_selective_scan_f32) scan;
  decltype(&arm_scan_selective_scan_views_f32) scan_views;
  decltype(&arm_scan_selective_state_update_f32) step;
  decltype(&arm_scan_selective_scan_bidirectional_f32) bidir;
  decltype(&arm_scan_mamba3_scan_time_major_f32) m3;
  decltype(&arm_scan_mamba3_scan_angles_f32) m3_angles;
  decltype(&arm_scan_mamba3_scan_strided_f32) m3_strided;
  decltype(&arm_scan_mamba3_noncausal_f32) noncausal;
  decltype(&arm_scan_mamba3_angles_f32) angles;
  decltype(&arm_scan_mamba3_block_frontend_f32) frontend;
  decltype(&arm_scan_causal_conv1d_f32) conv;
  decltype(&arm_scan_causal_conv1d_update_f32) conv_step;
  decltype(&arm_scan_ss2d_f32) ss2d;
  decltype(&arm_scan_mamba3_grid_f32) grid;
  decltype(&arm_scan_thread_scratch) thread_scratch;
} abi{};

template <class F>
void bind_one(const py::dict& d, const char* name, F& f) {
  f = reinterpret_cast<F>(d[name].cast<uintptr_t>());
}

void bind(const py::dict& d) {
  bind_one(d, "arm_scan_selective_scan_f32", abi.scan);
  bind_one(d, "arm_scan_selective_scan_views_f32", abi.scan_views);
  bind_one(d, "arm_scan_selective_state_update_f32", abi.step);
  bind_one(d, "arm_scan_selective_scan_bidirectional_f32", abi.bidir);
  bind_one(d, "arm_scan_mamba3_scan_time_major_f32", abi.m3);
  bind_one(d, "arm_scan_mamba3_scan_angles_f32", abi.m3_angles);
  bind_one(d, "arm_scan_mamba3_scan_strided_f32", abi.m3_strided);
  bind_one(d, "arm_scan_mamba3_noncausal_f32", abi.noncausal);
  bind_one(d, "arm_scan_mamba3_angles_f32", abi.angles);
  bind_one(d, "arm_scan_mamba3_block_frontend_f32", abi.frontend);
  bind_one(d, "arm_scan_causal_conv1d_f32", abi.conv);
  bind_one(d, "arm_scan_causal_conv1d_update_f32", abi.conv_step);
  bind_one(d, "arm_scan_ss2d_f32", abi.ss2d);
  bind_one(d, "arm_scan_mamba3_grid_f32", abi.grid);
  bind_one(d, "arm_scan_thread_scratch", abi.thread_scratch);
}

using at::Tensor;
using Shape = std::initializer_list<int64_t>;

// Whether `ks` holds no functionality but those of `ok` (backend bits aside, which
// DispatchKeySet's subtraction leaves in).
bool within(c10::DispatchKeySet ks, c10::DispatchKeySet ok) {
  return ((ks - ok).raw_repr() & ~c10::full_backend_mask) == 0;
}

// Nothing of torch's sits between an eager call and the kernels on this thread.
bool plain_thread() {
  using c10::DispatchKey;
  const c10::DispatchKeySet ok({DispatchKey::BackendSelect, DispatchKey::ADInplaceOrView});
  return within(c10::impl::tls_local_dispatch_key_set().included_, ok) &&
         !at::impl::torch_function_mode_enabled();
}

// The tensors of one call: each is fetched with its shape, and `ok` goes false at the
// first that is not plain.
struct Call {
  bool ok;
  c10::Device device{c10::kCPU};
  bool have_device = false;

  Call() : ok(plain_thread()) {}

  // a tensor argument (None: undefined, where allowed)
  Tensor get(const py::handle& h, bool optional = false) {
    if (!ok) return {};
    if (h.is_none()) {
      ok = optional;
      return {};
    }
    PyObject* o = h.ptr();
    const PyTypeObject* type = Py_TYPE(o);
    if (type != reinterpret_cast<PyTypeObject*>(THPVariableClass) &&
        type != reinterpret_cast<PyTypeObject*>(ParameterClass)) {
      ok = false;
      return {};
    }
    Tensor t = THPVariable_Unpack(o);
    using c10::DispatchKey;
    using c10::DispatchKeySet;
    const DispatchKeySet keys_ok =
        DispatchKeySet({DispatchKey::CUDA, DispatchKey::AutogradCUDA,
                        DispatchKey::ADInplaceOrView, DispatchKey::AutocastCUDA});
    ok = t.defined() && t.is_cuda() && t.layout() == at::kStrided &&
         t.scalar_type() == at::kFloat && within(t.key_set(), keys_ok) && t.numel() > 0 &&
         !(at::GradMode::is_enabled() && t.requires_grad()) && !t._fw_grad(0).defined();
    if (!ok) return {};
    if (!have_device) {
      device = t.device();
      have_device = true;
    }
    ok = t.device() == device;
    return t;
  }
  // with a shape to match
  Tensor get(const py::handle& h, Shape shape, bool optional = false) {
    Tensor t = get(h, optional);
    if (ok && t.defined()) ok = t.sizes().equals(at::IntArrayRef(shape));
    return t;
  }
};

// The wrappers' own contiguous copies, made once nothing about the call is left to refuse: a
// call that goes on to the custom op, which makes them too, has paid for none here.
void lay(std::initializer_list<Tensor*> ts) {
  for (Tensor* t : ts)
    if (t->defined() && !t->is_contiguous()) *t = t->contiguous();
}

const float* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr<float>() : nullptr; }
float* out_ptr(Tensor& t) { return t.defined() ? t.mutable_data_ptr<float>() : nullptr; }
bool aligned(const Tensor& t) {
  return !t.defined() || reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
}

// Runs a call of the C ABI on the device's current stream, its scratch from torch's
// caching allocator (blocks that return to it when the call has been enqueued: what reuses
// them on this stream runs after it). False on any error.
struct Scratch {
  c10::Device device;
  std::vector<Tensor> held;
};
void* scratch_alloc(void* ctx, size_t bytes) {
  auto* s = static_cast<Scratch*>(ctx);
  try {
    s->held.push_back(at::empty({static_cast<int64_t>(bytes)},
                                at::TensorOptions().dtype(at::kByte).device(s->device)));
    return s->held.back().mutable_data_ptr();
  } catch (...) {  // out of memory: the library's error, reported by the custom op's path
    return nullptr;
  }
}
template <class F>
bool launch(c10::Device device, F&& f) {
  void* stream = c10::hip::getCurrentHIPStream(device.index()).stream();
  Scratch s{device, {}};
  py::gil_scoped_release nogil;
  abi.thread_scratch(scratch_alloc, &s);
  struct Unset {
    ~Unset() { abi.thread_scratch(nullptr, nullptr); }
  } unset;
  return f(stream) == 0;
}

Tensor empty(const Call& c, Shape shape) {
  return at::empty(at::IntArrayRef(shape),
                   at::TensorOptions().dtype(at::kFloat).device(c.device));
}
py::object wrap(const Tensor& t) {
  return t.defined() ? py::reinterpret_steal<py::object>(THPVariable_Wrap(t)) : py::none();
}

// ------------------------------------------------------------------ Mamba-1
// B, C (batch, state, len) or (batch, groups, state, len)
Tensor bc4(Call& c, const py::handle& h, int64_t batch, int64_t state, int64_t length,
           int64_t& groups) {
  Tensor t = c.get(h);
  if (!c.ok) return {};
  if (t.dim() == 3) t = t.unsqueeze(1);
  if (t.dim() != 4 || (groups && t.size(1) != groups)) {
    c.ok = false;
    return {};
  }
  groups = t.size(1);
  c.ok = t.size(0) == batch && t.size(2) == state && t.size(3) == length;
  return t;
}

struct M1 {
  Tensor u, delta, a, b, c, d, z, bias, h0;
  int64_t batch = 0, dim = 0, length = 0, state = 0, groups = 0;
  ArmScanDims dims() const {
    return {(size_t)batch, (size_t)dim, (size_t)length, (size_t)state, (size_t)groups};
  }
};

// Checked, as they lie: m1_lay makes the rows contiguous.
bool m1_args(Call& c, M1& m, const py::handle& u, const py::handle& delta,
             const py::handle& a, const py::handle& b, const py::handle& cc,
             const py::handle& d, const py::handle& z, const py::handle& bias,
             const py::handle& h0) {
  m.u = c.get(u);
  m.a = c.get(a);
  if (!c.ok || m.u.dim() != 3 || m.a.dim() != 2) return false;
  m.batch = m.u.size(0);
  m.dim = m.u.size(1);
  m.length = m.u.size(2);
  m.state = m.a.size(1);
  if (m.a.size(0) != m.dim) return false;
  m.delta = c.get(delta, {m.batch, m.dim, m.length});
  m.b = bc4(c, b, m.batch, m.state, m.length, m.groups);
  m.c = bc4(c, cc, m.batch, m.state, m.length, m.groups);
  m.d = c.get(d, {m.dim}, true);
  m.z = c.get(z, {m.batch, m.dim, m.length}, true);
  m.bias = c.get(bias, {m.dim}, true);
  m.h0 = c.get(h0, {m.batch, m.dim, m.state}, true);
  return c.ok && m.dim % m.groups == 0;
}
// views: u, z, B and C keep their strides
void m1_lay(M1& m, bool views) {
  lay({&m.delta, &m.a, &m.d, &m.bias, &m.h0});
  if (!views) lay({&m.u, &m.z, &m.b, &m.c});
}

py::object selective_scan(py::handle u, py::handle delta, py::handle a, py::handle b,
                          py::handle cc, py::handle d, py::handle z, py::handle bias,
                          py::handle h0, bool softplus, bool reverse) {
  Call c;
  M1 m;
  if (!m1_args(c, m, u, delta, a, b, cc, d, z, bias, h0)) return py::none();
  RECORD_FUNCTION("arm_scan::selective_scan", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  m1_lay(m, false);
  Tensor out = empty(c, {m.batch, m.dim, m.length}), last = empty(c, {m.batch, m.dim, m.state});
  const ArmScanDims dims = m.dims();
  if (!launch(c.device, [&](void* st) {
        return abi.scan(&dims, ptr(m.u), ptr(m.delta), ptr(m.a), ptr(m.b), ptr(m.c), ptr(m.d),
                        ptr(m.z), ptr(m.bias), softplus, reverse, 0, 0, out_ptr(out),
                        out_ptr(last), ptr(m.h0), st);
      }))
    return py::none();
  return py::make_tuple(wrap(out), wrap(last));
}

// Views that arm_scan_selective_scan_views_f32 reads in place, by the rule it states (the
// library refuses the rest with code 2, after the outputs are allocated), without broadcasts
// (the custom op materialises those).
bool views_ok(const M1& m) {
  auto fits = [&](at::IntArrayRef s) {
    return 4 * ((m.dim - 1) * s[1] + (m.length - 1) * s[2] + 1) < (int64_t(1) << 32) &&
           60 * s[2] < (int64_t(1) << 31);
  };
  auto view_ok = [&](const Tensor& t) {
    for (int i = 0; i < 3; ++i)
      if (t.stride(i) == 0 && t.size(i) > 1) return false;
    return fits(t.strides());
  };
  // 16-byte rows; what is not contiguous is delta's copy, or u by its strides
  auto lies16 = [](const Tensor& t) { return !t.is_contiguous() || aligned(t); };
  const bool whole = m.length % 4 == 0 && lies16(m.delta) && lies16(m.u);
  // other rows: z in 16-byte runs of channels (as out is), and more than 8 states
  const bool staged = !m.z.defined() ||
                      (m.z.stride(1) == 1 && m.z.stride(2) % 4 == 0 && m.z.stride(0) % 4 == 0 &&
                       aligned(m.z) && m.state > 8);
  const std::array<int64_t, 3> out{m.length * m.dim, 1, m.dim};
  return m.dim % 16 == 0 && (m.dim / m.groups) % 16 == 0 && (whole || staged) &&
         m.batch * m.groups <= 65535 && fits(out) && view_ok(m.u) &&
         (!m.z.defined() || view_ok(m.z));
}

template <int N>
std::array<long long, N> strides_of(const Tensor& t) {
  std::array<long long, N> s;
  for (int i = 0; i < N; ++i) s[i] = t.stride(i);
  return s;
}

py::object selective_scan_time_major(py::handle u, py::handle delta, py::handle a,
                                     py::handle b, py::handle cc, py::handle d, py::handle z,
                                     py::handle bias, py::handle h0, bool softplus,
                                     bool reverse) {
  Call c;
  M1 m;
  if (!m1_args(c, m, u, delta, a, b, cc, d, z, bias, h0) || !views_ok(m))
    return py::none();
  RECORD_FUNCTION("arm_scan::selective_scan_time_major", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  m1_lay(m, true);
  Tensor out = empty(c, {m.batch, m.length, m.dim}).transpose(1, 2);
  Tensor last = empty(c, {m.batch, m.dim, m.state});
  const ArmScanDims dims = m.dims();
  const auto us = strides_of<3>(m.u), os = strides_of<3>(out);
  const auto zs = m.z.defined() ? strides_of<3>(m.z) : us;
  const auto bs = strides_of<4>(m.b), cs = strides_of<4>(m.c);
  if (!launch(c.device, [&](void* st) {
        return abi.scan_views(&dims, ptr(m.u), m.u.is_contiguous() ? nullptr : us.data(),
                              ptr(m.delta), ptr(m.a), ptr(m.b), bs.data(), ptr(m.c), cs.data(),
                              ptr(m.d), ptr(m.z), m.z.defined() ? zs.data() : nullptr,
                              ptr(m.bias), softplus, reverse, out_ptr(out), os.data(),
                              out_ptr(last), ptr(m.h0), st);
      }))
    return py::none();
  return py::make_tuple(wrap(out), wrap(last));
}

py::object bidirectional(py::handle u, py::handle delta, py::handle a, py::handle b,
                         py::handle cc, py::handle d, py::handle z, py::handle bias,
                         bool softplus) {
  Call c;
  M1 m;
  if (!m1_args(c, m, u, delta, a, b, cc, d, z, bias, py::none())) return py::none();
  RECORD_FUNCTION("arm_scan::selective_scan_bidirectional", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  m1_lay(m, false);
  Tensor fwd = empty(c, {m.batch, m.dim, m.length}), bwd = empty(c, {m.batch, m.dim, m.length});
  const ArmScanDims dims = m.dims();
  if (!launch(c.device, [&](void* st) {
        return abi.bidir(&dims, ptr(m.u), ptr(m.delta), ptr(m.a), ptr(m.b), ptr(m.c), ptr(m.d),
                         ptr(m.z), ptr(m.bias), softplus, 0, 0, out_ptr(fwd), out_ptr(bwd),
                         nullptr, nullptr, st);
      }))
    return py::none();
  return py::make_tuple(wrap(fwd), wrap(bwd));
}

std::array<long long, 2> strides2(const Tensor& t) { return {t.stride(0), t.stride(1)}; }

// A tensor the call writes in place: as the dispatcher does for an op that mutates it.
void mutated(const Tensor& t) {
  if (!t.is_inference()) t.unsafeGetTensorImpl()->bump_version();
}

py::object state_update(py::handle state, py::handle x, py::handle dt, py::handle a,
                        py::handle b, py::handle cc, py::handle d, py::handle z,
                        py::handle bias, bool softplus) {
  Call c;
  Tensor s = c.get(state);
  if (!c.ok || s.dim() != 3 || !s.is_contiguous()) return py::none();
  const int64_t batch = s.size(0), dim = s.size(1), n = s.size(2);
  const Tensor tx = c.get(x, {batch, dim}), tdt = c.get(dt, {batch, dim}),
               tb = c.get(b, {batch, n}), tc = c.get(cc, {batch, n}),
               tz = c.get(z, {batch, dim}, true);
  Tensor ta = c.get(a, {dim, n}), td = c.get(d, {dim}, true), tbias = c.get(bias, {dim}, true);
  if (!c.ok) return py::none();
  RECORD_FUNCTION("arm_scan::selective_state_update", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  lay({&ta, &td, &tbias});
  Tensor out = empty(c, {batch, dim});
  const auto xs = strides2(tx), dts = strides2(tdt), bs = strides2(tb), cs = strides2(tc);
  const auto zs = tz.defined() ? strides2(tz) : xs;
  if (!launch(c.device, [&](void* st) {
        return abi.step(batch, dim, n, out_ptr(s), ptr(tx), xs.data(), ptr(tdt), dts.data(),
                        ptr(ta), ptr(tb), bs.data(), ptr(tc), cs.data(), ptr(td), ptr(tz),
                        tz.defined() ? zs.data() : nullptr, ptr(tbias), softplus, out_ptr(out),
                        st);
      }))
    return py::none();
  mutated(s);
  return wrap(out);
}

py::object causal_conv1d(py::handle x, py::handle weight, py::handle bias, bool silu,
                         bool time_major) {
  Call c;
  const Tensor tx = c.get(x);
  Tensor tw = c.get(weight);
  if (!c.ok || tx.dim() != 3 || tw.dim() != 2 || tw.size(0) != tx.size(1)) return py::none();
  const int64_t batch = tx.size(0), dim = tx.size(1), length = tx.size(2);
  Tensor tb = c.get(bias, {dim}, true);
  if (!c.ok) return py::none();
  RECORD_FUNCTION("arm_scan::causal_conv1d", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  lay({&tw, &tb});
  Tensor out = time_major ? empty(c, {batch, length, dim}).transpose(1, 2)
                          : empty(c, {batch, dim, length});
  const int64_t xs[3] = {tx.stride(0), tx.stride(1), tx.stride(2)};
  if (!launch(c.device, [&](void* st) {
        return abi.conv(batch, dim, length, tw.size(1), ptr(tx), xs, ptr(tw), ptr(tb), silu,
                        time_major, out_ptr(out), st);
      }))
    return py::none();
  return wrap(out);
}

py::object causal_conv1d_update(py::handle x, py::handle state, py::handle weight,
                                py::handle bias, bool silu) {
  Call c;
  const Tensor tx = c.get(x);
  Tensor tw = c.get(weight);
  if (!c.ok || tx.dim() != 2 || tw.dim() != 2 || tw.size(0) != tx.size(1)) return py::none();
  const int64_t batch = tx.size(0), dim = tx.size(1), width = tw.size(1);
  Tensor s = c.get(state, {batch, dim, width}), tb = c.get(bias, {dim}, true);
  if (!c.ok || !s.is_contiguous()) return py::none();
  RECORD_FUNCTION("arm_scan::causal_conv1d_update", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  lay({&tw, &tb});
  Tensor out = empty(c, {batch, dim});
  const int64_t xs[2] = {tx.stride(0), tx.stride(1)};
  if (!launch(c.device, [&](void* st) {
        return abi.conv_step(batch, dim, width, ptr(tx), xs, out_ptr(s), ptr(tw), ptr(tb), silu,
                             out_ptr(out), st);
      }))
    return py::none();
  mutated(s);
  return wrap(out);
}

// u, delta, z (b, d, h, w); b4, c4 (4, b, n, h, w); merge 0 none, 1 sum, 2 mean
py::object ss2d(py::handle u, py::handle delta, py::handle a, py::handle b4, py::handle c4,
                py::handle d, py::handle z, py::handle bias, bool softplus, int merge,
                bool want_last) {
  Call c;
  Tensor tu = c.get(u), ta = c.get(a);
  if (!c.ok || tu.dim() != 4 || ta.dim() != 2 || ta.size(0) != tu.size(1)) return py::none();
  const int64_t b = tu.size(0), dim = tu.size(1), h = tu.size(2), w = tu.size(3),
                n = ta.size(1);
  Tensor tdt = c.get(delta, {b, dim, h, w}), tb = c.get(b4, {4, b, n, h, w}),
         tc = c.get(c4, {4, b, n, h, w}), td = c.get(d, {dim}, true),
         tz = c.get(z, {b, dim, h, w}, true), tbias = c.get(bias, {dim}, true);
  if (!c.ok) return py::none();
  RECORD_FUNCTION("arm_scan::ss2d_scan", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  lay({&tu, &ta, &tdt, &tb, &tc, &td, &tz, &tbias});
  Tensor out = merge == 0 ? empty(c, {4, b, dim, h, w}) : empty(c, {b, dim, h, w}), last;
  if (want_last) last = empty(c, {4, b, dim, n});
  const ArmSS2DDims dims{(size_t)b, (size_t)dim, (size_t)h, (size_t)w, (size_t)n};
  if (!launch(c.device, [&](void* st) {
        return abi.ss2d(&dims, ptr(tu), ptr(tdt), ptr(ta), ptr(tb), ptr(tc), ptr(td), ptr(tz),
                        ptr(tbias), softplus, merge, out_ptr(out), out_ptr(last), st);
      }))
    return py::none();
  return py::make_tuple(wrap(out), wrap(last));
}

// ------------------------------------------------------------------ Mamba-3
struct M3 {
  Tensor q, k, v, adt, dt, trap, qb, kb, cos, sin, ang, d, z, psi, zeta, phi;
  int64_t b = 0, length = 0, h = 0, dv = 0, dqk = 0, rank = 1, groups = 0;
  bool mimo = false;
  ArmMamba3Dims dims() const {
    return {(size_t)b, (size_t)h, (size_t)dv, (size_t)dqk, (size_t)length, (size_t)rank,
            (size_t)groups};
  }
};

// Shapes as mamba3.py's _check_shapes; m3_lay makes all but v, z and the angles contiguous.
bool m3_args(Call& c, M3& m, const py::handle& q, const py::handle& k, const py::handle& v,
             const py::handle& adt, const py::handle& dt, const py::handle& trap,
             const py::handle& qb, const py::handle& kb, const py::handle& cos,
             const py::handle& sin, const py::handle& ang, const py::handle& d,
             const py::handle& z, const py::handle& psi, const py::handle& zeta,
             const py::handle& phi, bool mimo) {
  m.mimo = mimo;
  m.q = c.get(q);
  m.k = c.get(k);
  m.v = c.get(v);
  if (!c.ok || m.v.dim() != 4) return false;
  const int64_t full = mimo ? 5 : 4;
  if (m.q.dim() == full - 1) m.q = m.q.unsqueeze(full - 2);
  if (m.k.dim() == full - 1) m.k = m.k.unsqueeze(full - 2);
  if (m.q.dim() != full || !m.k.sizes().equals(m.q.sizes())) return false;
  m.b = m.v.size(0);
  m.length = m.v.size(1);
  m.h = m.v.size(2);
  m.dv = m.v.size(3);
  m.rank = mimo ? m.q.size(2) : 1;
  m.groups = m.q.size(full - 2);
  m.dqk = m.q.size(full - 1);
  if (m.q.size(0) != m.b || m.q.size(1) != m.length || m.dqk % 2 || m.h % m.groups) return false;
  m.adt = c.get(adt, {m.b, m.h, m.length});
  m.dt = c.get(dt, {m.b, m.h, m.length});
  m.trap = c.get(trap, {m.b, m.h, m.length});
  if (mimo) {
    m.qb = c.get(qb, {m.h, m.rank, m.dqk});
    m.kb = c.get(kb, {m.h, m.rank, m.dqk});
    m.psi = c.get(psi, {m.h, m.rank, m.dv});
    m.zeta = c.get(zeta, {m.h, m.rank, m.dv});
    m.phi = c.get(phi, {m.h, m.rank, m.dv});
  } else {
    m.qb = c.get(qb, {m.h, m.dqk});
    m.kb = c.get(kb, {m.h, m.dqk});
  }
  m.d = c.get(d, {m.h}, true);
  m.z = c.get(z, {m.b, m.length, m.h, m.dv}, true);
  if (!c.ok) return false;
  if (!cos.is_none() || !sin.is_none()) {  // then the angles are not read
    m.cos = c.get(cos, {m.b, m.length, m.h, m.dqk / 2});
    m.sin = c.get(sin, {m.b, m.length, m.h, m.dqk / 2});
    return c.ok && ang.is_none();
  }
  m.ang = c.get(ang);
  return c.ok && m.ang.dim() == 4 && m.ang.size(0) == m.b && m.ang.size(1) == m.length &&
         m.ang.size(2) == m.h && m.ang.size(3) >= 1 && m.ang.size(3) <= m.dqk / 2;
}
void m3_lay(M3& m) {
  lay({&m.q, &m.k, &m.adt, &m.dt, &m.trap, &m.qb, &m.kb, &m.psi, &m.zeta, &m.phi, &m.d, &m.cos,
       &m.sin});
}

// cos and sin from the raw angles (arm_scan_mamba3_angles_f32)
bool m3_rotations(const Call& c, M3& m) {
  if (m.cos.defined()) return true;
  const Tensor a = m.ang.contiguous();
  m.cos = empty(c, {m.b, m.length, m.h, m.dqk / 2});
  m.sin = empty(c, {m.b, m.length, m.h, m.dqk / 2});
  return launch(c.device, [&](void* st) {
    return abi.angles(ptr(a), ptr(m.dt), m.b, m.length, m.h, a.size(3), m.dqk / 2,
                      out_ptr(m.cos), out_ptr(m.sin), st);
  });
}

// Whether v and z ((batch, step) strides, heads dv apart, unit channel stride) or the
// angles can be read where they lie: mamba3.py's _inplace_strides.
bool in_place(const M3& m) {
  auto broadcast = [](const Tensor& t, int axis) {
    return t.stride(axis) == 0 && t.size(axis) > 1;
  };
  auto rows = [&](const Tensor& t) {
    return !(m.dv > 1 && t.stride(3) != 1) && !(m.h > 1 && t.stride(2) != m.dv) &&
           !broadcast(t, 0) && !broadcast(t, 1);
  };
  return rows(m.v) && (!m.z.defined() || rows(m.z)) &&
         !(m.ang.size(3) > 1 && m.ang.stride(3) != 1) && !broadcast(m.ang, 0) &&
         !broadcast(m.ang, 1);
}

py::object mamba3(py::handle q, py::handle k, py::handle v, py::handle adt, py::handle dt,
                  py::handle trap, py::handle qb, py::handle kb, py::handle cos, py::handle sin,
                  py::handle ang, py::handle d, py::handle z, py::handle psi, py::handle zeta,
                  py::handle phi, bool reverse, bool carry, bool mimo) {
  Call c;
  M3 m;
  if (!m3_args(c, m, q, k, v, adt, dt, trap, qb, kb, cos, sin, ang, d, z, psi, zeta, phi, mimo))
    return py::none();
  RECORD_FUNCTION("arm_scan::mamba3_scan", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  m3_lay(m);
  Tensor out = empty(c, {m.b, m.length, m.h, m.dv}), state, bx;
  const ArmMamba3Dims dims = m.dims();
  auto result = [&] {
    if (!carry) return py::object(wrap(out));
    return py::object(mimo ? py::make_tuple(wrap(out), wrap(state))
                           : py::make_tuple(wrap(out), wrap(state), wrap(bx)));
  };
  if (m.ang.defined() && !reverse && !carry &&
      !(m.v.is_contiguous() && m.ang.is_contiguous() &&
        (!m.z.defined() || m.z.is_contiguous())) &&
      in_place(m)) {
    const int64_t vs[2] = {m.v.stride(0), m.v.stride(1)};
    const int64_t zs[2] = {m.z.defined() ? m.z.stride(0) : 0, m.z.defined() ? m.z.stride(1) : 0};
    const int64_t as[3] = {m.ang.stride(0), m.ang.stride(1), m.ang.stride(2)};
    if (!launch(c.device, [&](void* st) {
          return abi.m3_strided(&dims, ptr(m.q), ptr(m.k), ptr(m.v), vs, ptr(m.adt), ptr(m.dt),
                                ptr(m.trap), ptr(m.qb), ptr(m.kb), ptr(m.ang), m.ang.size(3), as,
                                ptr(m.d), ptr(m.z), m.z.defined() ? zs : nullptr, ptr(m.psi),
                                ptr(m.zeta), ptr(m.phi), 0, 0, out_ptr(out), st);
        }))
      return py::none();
    return result();
  }
  lay({&m.v, &m.z});
  if (carry) {
    state = empty(c, {m.b, m.h, m.dv, m.dqk});
    if (!mimo) bx = empty(c, {m.b, m.h, m.dqk});
  }
  // the angle pre-pass fused into the scan: mamba3.py's _angles_fusable (SISO)
  if (m.ang.defined() && !mimo && !reverse && m.ang.size(3) % 4 == 0 && m.dv % 16 == 0 &&
      m.dqk % 16 == 0 && m.dqk <= 128) {
    m.ang = m.ang.contiguous();
    if (aligned(m.q) && aligned(m.k) && aligned(m.v) && aligned(m.qb) && aligned(m.kb) &&
        aligned(m.ang) && aligned(m.z)) {
      if (!launch(c.device, [&](void* st) {
            return abi.m3_angles(&dims, ptr(m.q), ptr(m.k), ptr(m.v), ptr(m.adt), ptr(m.dt),
                                 ptr(m.trap), ptr(m.qb), ptr(m.kb), ptr(m.ang), m.ang.size(3),
                                 ptr(m.d), ptr(m.z), nullptr, nullptr, nullptr, 0, 0,
                                 out_ptr(out), out_ptr(state), out_ptr(bx), st);
          }))
        return py::none();
      return result();
    }
  }
  if (!m3_rotations(c, m) || !launch(c.device, [&](void* st) {
        return abi.m3(&dims, ptr(m.q), ptr(m.k), ptr(m.v), ptr(m.adt), ptr(m.dt), ptr(m.trap),
                      ptr(m.qb), ptr(m.kb), ptr(m.cos), ptr(m.sin), ptr(m.d), ptr(m.z),
                      ptr(m.psi), ptr(m.zeta), ptr(m.phi), reverse, 0, 0, out_ptr(out),
                      out_ptr(state), out_ptr(bx), st);
      }))
    return py::none();
  return result();
}

py::object noncausal(py::handle q, py::handle k, py::handle v, py::handle adt, py::handle dt,
                     py::handle trap, py::handle qb, py::handle kb, py::handle cos,
                     py::handle sin, py::handle ang, py::handle d, py::handle z) {
  Call c;
  M3 m;
  const py::none none;
  if (!m3_args(c, m, q, k, v, adt, dt, trap, qb, kb, cos, sin, ang, d, z, none, none, none,
               false))
    return py::none();
  RECORD_FUNCTION("arm_scan::mamba3_noncausal", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  m3_lay(m);
  lay({&m.v, &m.z});
  Tensor out = empty(c, {m.b, m.length, m.h, m.dv});
  const ArmMamba3Dims dims = m.dims();
  if (!m3_rotations(c, m) || !launch(c.device, [&](void* st) {
        return abi.noncausal(&dims, ptr(m.q), ptr(m.k), ptr(m.v), ptr(m.adt), ptr(m.dt),
                             ptr(m.trap), ptr(m.qb), ptr(m.kb), ptr(m.cos), ptr(m.sin),
                             ptr(m.d), ptr(m.z), 0, 0, out_ptr(out), st);
      }))
    return py::none();
  return wrap(out);
}

// Both orderings of a token grid, scanned and merged: q, k (b, H, W, g, dqk); v, z (b, H, W,
// h, dv); adt, dt, trap (b, h, H, W); angles (b, H, W, h, r); merge 1 sum, 2 mean.
py::object grid_mamba3(py::handle q, py::handle k, py::handle v, py::handle adt, py::handle dt,
                       py::handle trap, py::handle qb, py::handle kb, py::handle ang,
                       py::handle d, py::handle z, bool noncausal, int merge) {
  Call c;
  const Tensor q0 = c.get(q), v0 = c.get(v), a0 = c.get(ang);
  if (!c.ok || q0.dim() != 5 || v0.dim() != 5 || a0.dim() != 5 || (merge != 1 && merge != 2))
    return py::none();
  const int64_t b = q0.size(0), H = q0.size(1), W = q0.size(2), g = q0.size(3),
                dqk = q0.size(4), h = v0.size(3), dv = v0.size(4), r = a0.size(4);
  if (dqk % 2 || h % g || r > dqk / 2 || H > 32768 || W > 32768) return py::none();
  Tensor tq = c.get(q, {b, H, W, g, dqk}), tk = c.get(k, {b, H, W, g, dqk}),
         tv = c.get(v, {b, H, W, h, dv}), tadt = c.get(adt, {b, h, H, W}),
         tdt = c.get(dt, {b, h, H, W}), ttrap = c.get(trap, {b, h, H, W}),
         tqb = c.get(qb, {h, dqk}), tkb = c.get(kb, {h, dqk}),
         ta = c.get(ang, {b, H, W, h, r}), td = c.get(d, {h}, true),
         tz = c.get(z, {b, H, W, h, dv}, true);
  if (!c.ok) return py::none();
  RECORD_FUNCTION("arm_scan::mamba3_grid", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  lay({&tq, &tk, &tv, &tadt, &tdt, &ttrap, &tqb, &tkb, &ta, &td, &tz});
  Tensor out = empty(c, {b, H, W, h, dv});
  const ArmMamba3Dims dims{(size_t)b, (size_t)h,       (size_t)dv, (size_t)dqk,
                           (size_t)(H * W), (size_t)1, (size_t)g};
  if (!launch(c.device, [&](void* st) {
        return abi.grid(&dims, H, W, ptr(tq), ptr(tk), ptr(tv), ptr(tadt), ptr(tdt), ptr(ttrap),
                        ptr(tqb), ptr(tkb), ptr(ta), r, ptr(td), ptr(tz), noncausal, merge,
                        out_ptr(out), st);
      }))
    return py::none();
  return wrap(out);
}

// The mixer between its projections: the front-end kernel, then the scan reading z, x and
// the angles where they lie in proj [z | x | B | C | dd_dt | dd_A | trap | angles].
py::object mixer_scan(py::handle proj, py::handle dt_bias, py::handle b_norm,
                      py::handle c_norm, py::handle b_bias, py::handle c_bias, py::handle d,
                      py::handle psi, py::handle zeta, py::handle phi, int64_t heads,
                      int64_t headdim, int64_t d_state, int64_t rank, int64_t groups,
                      int64_t n_angles, double a_floor, double eps) {
  Call c;
  const Tensor p = c.get(proj);
  if (!c.ok || p.dim() != 3 || !p.is_contiguous()) return py::none();
  const int64_t b = p.size(0), length = p.size(1), row = p.size(2);
  const int64_t inner = heads * headdim;
  const int64_t col_ang = 2 * inner + 2 * rank * groups * d_state + 3 * heads;
  const bool mimo = !psi.is_none();
  Tensor tdt = c.get(dt_bias, {heads}), tbn = c.get(b_norm, {d_state}),
         tcn = c.get(c_norm, {d_state}), tbb = c.get(b_bias, {heads, rank, d_state}),
         tcb = c.get(c_bias, {heads, rank, d_state}), td = c.get(d, {heads});
  Tensor tpsi, tzeta, tphi;
  if (mimo) {
    tpsi = c.get(psi, {heads, rank, headdim});
    tzeta = c.get(zeta, {heads, rank, headdim});
    tphi = c.get(phi, {heads, rank, headdim});
  }
  if (!c.ok || row != col_ang + n_angles) return py::none();
  RECORD_FUNCTION("arm_scan::mamba3_mixer_scan", std::vector<c10::IValue>());
  c10::DeviceGuard on_device(c.device);
  lay({&tdt, &tbn, &tcn, &tbb, &tcb, &td, &tpsi, &tzeta, &tphi});
  Tensor q = empty(c, {b, length, rank, groups, d_state}),
         k = empty(c, {b, length, rank, groups, d_state}), adt = empty(c, {b, heads, length}),
         dt = empty(c, {b, heads, length}), trap = empty(c, {b, heads, length}),
         out = empty(c, {b, length, heads, headdim});
  const float* base = ptr(p);
  const int64_t vs[2] = {length * row, row}, as[3] = {length * row, row, 0};
  const ArmMamba3Dims dims{(size_t)b, (size_t)heads, (size_t)headdim, (size_t)d_state,
                           (size_t)length, (size_t)rank, (size_t)groups};
  if (!launch(c.device, [&](void* st) {
        const int rc = abi.frontend(base, b, length, row, heads, headdim, d_state, rank, groups,
                                    n_angles, ptr(tdt), (float)a_floor, ptr(tbn), ptr(tcn),
                                    (float)eps, out_ptr(q), out_ptr(k), out_ptr(adt),
                                    out_ptr(dt), out_ptr(trap), st);
        if (rc) return rc;
        return abi.m3_strided(&dims, ptr(q), ptr(k), base + inner, vs, ptr(adt), ptr(dt),
                              ptr(trap), ptr(tcb), ptr(tbb), base + col_ang, n_angles, as,
                              ptr(td), base, vs, ptr(tpsi), ptr(tzeta), ptr(tphi), 0, 0,
                              out_ptr(out), st);
      }))
    return py::none();
  return wrap(out);
}

}  // namespace

PYBIND11_MODULE(_torch_front, m) {
  m.attr("torch_version") = TORCH_VERSION;
  m.def("bind", &bind);
  m.def("selective_scan", &selective_scan);
  m.def("selective_scan_time_major", &selective_scan_time_major);
  m.def("bidirectional", &bidirectional);
  m.def("state_update", &state_update);
  m.def("causal_conv1d", &causal_conv1d);
  m.def("causal_conv1d_update", &causal_conv1d_update);
  m.def("ss2d", &ss2d);
  m.def("mamba3", &mamba3);
  m.def("noncausal", &noncausal);
  m.def("grid_mamba3", &grid_mamba3);
  m.def("mixer_scan", &mixer_scan);
}
