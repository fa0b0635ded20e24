// native.cpp — the host path of kilat_amd's calls in C++: argument checks, output
// allocation, the launch through libkdecay.so's C ABI, and the autograd node of
// the training scan.
//
// scan() and decay_step() take the calls whose arguments the kernels read as
// they are, and return None for any other: the caller (triton_ops.py) then
// converts, copies, pads or raises.  What a call costs is host time: through
// Python and ctypes a forward took 10.5 us on the host, a decode step 12.4, and a
// training pass 145, of which autograd itself takes about 50 (the hand-over to
// the engine's thread).
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/torch.h>

#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include "kdecay.h"

namespace py = pybind11;
using at::Tensor;

namespace {

// -1: a type no kernel takes.
int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return KDECAY_F32;
    case at::kBFloat16: return KDECAY_BF16;
    case at::kHalf: return KDECAY_F16;
    case at::kDouble: return KDECAY_F64;
    default: return -1;
  }
}

bool chunked_head_dim(int64_t D, int64_t es) { return D == 16 || D == 32 || (D > 0 && D % (128 / es) == 0); }

// row_split of kdecay_rows.hip: whole rows of up to 16 vectors of 16 bytes,
// wider ones in the fewest equal streams; not less than one vector, and not a
// last stream of one vector that overlaps the stream before it.
bool row_vectors_ok(int64_t D, int64_t es) {
  const int64_t vw = 16 / es;
  if (D < vw) return false;
  const int64_t nv = (D + vw - 1) / vw, ng = (nv + 15) / 16;
  const int64_t left = nv - (ng - 1) * ((nv + ng - 1) / ng);
  return left >= 1 && (ng == 1 || left >= 2 || D % vw == 0);
}

// The chunked kernels' layout rule: d-stride 1, 16-byte base, and every other
// stride a multiple of 16 bytes (size-1 dims excepted).  For head dims they take,
// whose rows are whole 16-byte vectors.
bool vector_layout_ok(const Tensor& t) {
  if (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) return false;
  const int64_t vw = 16 / t.element_size();
  if (t.stride(3) != 1 && t.size(3) != 1) return false;
  for (int k = 0; k < 3; ++k)
    if (t.stride(k) % vw != 0 && t.size(k) != 1) return false;
  return true;
}

// The chunked backward's addressing rule: it reads one chunk of rows of V and of
// the upstream gradient through 32-bit byte offsets, so a chunk's rows must span
// less than 2^31 bytes (the library rejects other row strides).  A chunk holds at
// most 4 wavefronts x (64 lanes / lanes per row) x 16 rows per lane; the bound
// uses that largest chunk, so a tensor that passes is accepted whatever chunk
// size the library picks (whole 256-byte rows, 16 lanes each, make 256-row
// chunks: fewer rows).
bool bwd_rows_fit(int64_t N, int64_t D, int64_t es, int64_t row_stride) {
  const int64_t lanes_per_row = std::min(D, 128 / es) * es / 16;
  if (N <= 1 || lanes_per_row < 1) return true;
  return 4 * (64 / lanes_per_row) * 16 * row_stride * es <= 0x7FFFFFFF;
}

// Whether a head of 16 or 32 channels, less than a 128-byte line, runs on the
// row kernels although the chunked kernels take it: V of at least 4 MiB, where a
// row's line holds other heads' rows too (a projection's view) or the row is 32
// bytes.  The row kernels number adjacent heads onto one XCD and store pieces of
// lines through its cache.  Measured (us, chunked / row kernels, forward;
// backward): bf16 D=16 B=8 H=12 N=4096 projection view 20.1 / 13.6; 28.1 / 21.1,
// contiguous 14.9 / 13.0; 20.0 / 19.9; B=32 H=16 N=1000 view 24.3 / 13.7; 39.5 /
// 41.5, contiguous 20.1 / 12.8; 27.1 / 25.0; bf16 D=32 B=8 H=12 N=4096 view 16.6 /
// 13.1; 32.9 / 24.5, contiguous 13.2 / 13.6 and B=32 H=16 N=1000 contiguous 17.5 /
// 18.9; 26.2 / 29.4; fp32 D=16 B=8 H=12 N=4096 view 16.9 / 14.0; 32.2 / 26.0; but
// B=2 H=6 N=1024 bf16 D=32 view 7.9 / 7.8; 10.3 / 11.6.
//
// Where they lose among those (7483 forwards and training passes; time as a share
// of the chunked kernels', geometric mean, worst), for few (b,h) streams, whose
// chains are long and whose grids leave CUs idle, mostly:
//   - 64-byte rows, forward, fewer than 40 streams: to 8192 rows 1.01, 1.15; past
//     32256 rows where the grid is small (chunks of 8 wavefronts, rows_shape) 0.97, 1.13;
//   - 64-byte rows, training: fewer than 40 streams past 16384 rows, in fp32 up to
//     2^20 rows in all 0.96, 1.11, in 16 bits past 32768 rows with fewer than 24
//     streams 0.98, 1.07; 513 to 640 rows (a second backward chunk of 512, nearly
//     empty) 0.99, 1.10;
//   - 32-byte rows: fewer than 24 streams in less than 8 MiB 0.99, 1.13; fp32
//     outputs of a contiguous 2-byte V past 1024 rows, forward 1.00, 1.11.
// Without those 6729 are left: 0.72, 1.13, half a percent of them above 1.03.
//
// train: a pass with a backward (whose forward goes with it).  wide: fp32 outputs of a
// 2-byte V.
bool narrow_rows(const Tensor& V, bool train, bool wide) {
  const int64_t N = V.size(2), D = V.size(3), es = V.element_size(), streams = V.size(0) * V.size(1);
  const int64_t bytes = V.numel() * es;
  if (D > 32 || D * es >= 128 || bytes < (4 << 20)) return false;
  const bool view = V.stride(2) != D;
  if (D * es == 32) return (streams >= 24 || bytes >= (8 << 20)) && (view || train || !wide || N <= 1024);
  if (!view) return false;
  if (!train) return streams >= 40 || (N > 8192 && (N <= 32256 || streams * N > 416 * 1024));
  if (N > 512 && N <= 640) return false;
  if (streams >= 40 || N <= 16384) return true;
  return es == 2 ? streams >= 24 || N <= 32768 : streams * N > (1 << 20);
}

bool train_layout_ok(const Tensor& t, bool rows) {
  return rows ? t.stride(3) == 1 : vector_layout_ok(t) && bwd_rows_fit(t.size(2), t.size(3), t.element_size(), t.stride(2));
}

bool out_layout_ok(const Tensor& t, bool rows) { return rows ? t.stride(3) == 1 : vector_layout_ok(t); }

// Whether a scan from V into out goes to the channel-group kernels as they are.
bool chunked_route(const Tensor& V, const Tensor& out) {
  return chunked_head_dim(V.size(3), V.element_size()) && vector_layout_ok(V) && vector_layout_ok(out) &&
         !narrow_rows(V, false, out.scalar_type() != V.scalar_type());
}

// Whether the row kernels write `out` directly: adjacent channels, and no two
// elements in the same memory (Tensor::copy_ refuses those).
bool rows_out_ok(const Tensor& out) {
  for (int64_t k = 0; k < 3; ++k)
    if (out.stride(k) == 0 && out.size(k) > 1) return false;
  return out.stride(3) == 1;
}

void check(int rc, const char* what) {
  TORCH_CHECK(rc == 0, "kilat_amd: ", what, " failed (code ", rc, "): ", kdecay_last_error_string());
}

hipStream_t stream_of(const at::Device& d) { return c10::hip::getCurrentHIPStream(d.index()).stream(); }

// triton_ops._workspaces[(device index, stream)], or an undefined tensor.  That
// dictionary is the one place that holds workspaces; nothing here keeps one from
// call to call.  Called with the GIL held.
Tensor find_workspace(const at::Device& d, hipStream_t stream) {
  // Set under the GIL without a static's guard: the import may give the GIL up,
  // and a thread waiting for the guard would keep it from coming back.
  static PyObject* all = nullptr;
  if (!all) all = py::module_::import("kilat_amd.triton_ops").attr("_workspaces").cast<py::dict>().release().ptr();
  const py::tuple key = py::make_tuple(static_cast<int>(d.index()), reinterpret_cast<uintptr_t>(stream));
  PyObject* const t = PyDict_GetItemWithError(all, key.ptr());
  if (!t) {
    if (PyErr_Occurred()) throw py::error_already_set();
    return Tensor();
  }
  return THPVariable_Unpack(t);
}

// The workspace of at least nbytes, grown by triton_ops._workspace if need be
// (which raises under capture).
Tensor need_workspace(const at::Device& d, hipStream_t stream, size_t nbytes) {
  if (nbytes == 0) return Tensor();
  py::gil_scoped_acquire gil;
  Tensor ws = find_workspace(d, stream);
  if (ws.defined() && static_cast<size_t>(ws.numel()) >= nbytes) return ws;
  return py::module_::import("kilat_amd.triton_ops")
      .attr("_workspace")(py::cast(d), reinterpret_cast<uintptr_t>(stream), nbytes)
      .cast<Tensor>();
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
size_t bytes(const Tensor& ws) { return ws.defined() ? static_cast<size_t>(ws.numel()) : 0; }

// Floats of the saved states, and bytes of workspace that the training forward
// and its backward need.
std::pair<size_t, size_t> train_sizes(int64_t B, int64_t H, int64_t N, int64_t D, int code, bool rows) {
  if (rows)
    return {kdecay_scan_rows_saved_states_floats(B, H, N, D, code),
            std::max(kdecay_scan_rows_workspace_bytes(B, H, N, D, code),
                     kdecay_scan_rows_bwd_workspace_bytes(B, H, N, D, code))};
  return {kdecay_scan_saved_states_floats(B, H, N, D, code),
          std::max(kdecay_scan_workspace_bytes(B, H, N, D, code), kdecay_scan_bwd_workspace_bytes(B, H, N, D, code))};
}

// The scan with a backward: kdecay_scan_fwd_train / kdecay_scan_bwd, or their
// row-kernel forms.  Inputs: lam (fp32 [H]), V, init (fp32 [B,H,D] or undefined);
// outputs: y and the final state.  The reference's GPU path has no backward; its
// CPU path is differentiated by torch autograd through triton_ops.py:240-246,
// which this replaces on HIP tensors.  With `sequential`, y and the final state
// are then rewritten by the sequential kernel (its bits), while the backward uses
// the states the chunked training forward saved (equal to tolerance).
struct ScanNode : torch::autograd::Function<ScanNode> {
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& lam,
                                                const Tensor& V, const std::optional<Tensor>& init, int64_t t_offset,
                                                at::ScalarType out_dtype, bool rows, bool sequential) {
    const int64_t B = V.size(0), H = V.size(1), N = V.size(2), D = V.size(3);
    const int v_code = dtype_code(V.scalar_type()), o_code = dtype_code(out_dtype);
    // The saved V also feeds the backward kernel, whose addressing takes a
    // narrower range of row strides than the forward's.
    const Tensor Vk = train_layout_ok(V, rows) ? V : V.contiguous();
    // y is laid out like V; for head dims of the channel groups contiguous where
    // its type is another one or the chunked kernels would not take V as it is.
    const bool group = chunked_head_dim(D, V.element_size());
    const auto yopt = V.options().dtype(out_dtype);
    const bool like = !group || (out_dtype == V.scalar_type() && train_layout_ok(V, false));
    Tensor y = like ? at::empty_like(V, yopt) : at::empty(V.sizes(), yopt);
    if (group && !out_layout_ok(y, rows)) y = at::empty(V.sizes(), yopt);
    const Tensor out = out_layout_ok(y, rows) ? y : at::empty(V.sizes(), yopt);  // what the kernel writes
    const Tensor final = at::empty({B, H, D}, Vk.options().dtype(at::kFloat));
    const auto [nstates, nbytes] = train_sizes(B, H, N, D, v_code, rows);
    const Tensor states = at::empty({static_cast<int64_t>(std::max<size_t>(nstates, 1))}, final.options());
    const Tensor init32 = init.has_value() ? *init : Tensor();
    {
      const c10::DeviceGuard guard(V.device());
      const hipStream_t s = stream_of(V.device());
      const Tensor ws = need_workspace(V.device(), s, nbytes);
      check((rows ? kdecay_scan_fwd_rows_train : kdecay_scan_fwd_train)(
                Vk.data_ptr(), v_code, Vk.strides().data(), out.data_ptr(), o_code, out.strides().data(),
                lam.data_ptr<float>(), static_cast<float*>(ptr(init32)), final.data_ptr<float>(),
                states.data_ptr<float>(), states.numel(), B, H, N, D, t_offset, ptr(ws), bytes(ws), s),
            rows ? "kdecay_scan_fwd_rows_train" : "kdecay_scan_fwd_train");
      if (sequential)
        check(kdecay_scan_fwd_sequential(Vk.data_ptr(), v_code, Vk.strides().data(), out.data_ptr(), o_code,
                                         out.strides().data(), lam.data_ptr<float>(),
                                         static_cast<float*>(ptr(init32)), final.data_ptr<float>(), B, H, N, D,
                                         t_offset, s),
              "kdecay_scan_fwd_sequential");
    }
    if (!out.is_same(y)) y.copy_(out);
    ctx->set_materialize_grads(false);
    ctx->saved_data["t_offset"] = t_offset;
    ctx->saved_data["rows"] = rows;
    ctx->save_for_backward({lam, Vk, init32, states});
    return {y, final};
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &lam = saved[0], &V = saved[1], &init = saved[2], &states = saved[3];
    const bool rows = ctx->saved_data["rows"].toBool();
    const int64_t t_offset = ctx->saved_data["t_offset"].toInt();
    const int64_t B = V.size(0), H = V.size(1), N = V.size(2), D = V.size(3);
    const int code = dtype_code(V.scalar_type());
    Tensor gy = grads[0].defined() ? grads[0].to(V.scalar_type()).resolve_neg() : at::zeros_like(V);
    if (!train_layout_ok(gy, rows)) gy = gy.contiguous();
    const Tensor gfin = grads[1].defined() ? grads[1].to(at::kFloat).resolve_neg().contiguous() : Tensor();
    Tensor dV = at::empty_like(V);
    if (!out_layout_ok(dV, rows)) dV = at::empty(V.sizes(), V.options());
    const auto fopt = V.options().dtype(at::kFloat);
    const Tensor dlam = V.numel() ? at::empty({H}, fopt) : at::zeros({H}, fopt);  // nothing to sum: no launch writes it
    const Tensor dinit = init.defined() ? at::empty({B, H, D}, fopt) : Tensor();
    {
      const c10::DeviceGuard guard(V.device());
      const hipStream_t s = stream_of(V.device());
      const Tensor ws = need_workspace(
          V.device(), s,
          (rows ? kdecay_scan_rows_bwd_workspace_bytes : kdecay_scan_bwd_workspace_bytes)(B, H, N, D, code));
      check((rows ? kdecay_scan_rows_bwd : kdecay_scan_bwd)(
                V.data_ptr(), code, V.strides().data(), gy.data_ptr(), gy.strides().data(), dV.data_ptr(),
                dV.strides().data(), lam.data_ptr<float>(), static_cast<float*>(ptr(init)), states.data_ptr<float>(),
                static_cast<float*>(ptr(gfin)), dlam.data_ptr<float>(), static_cast<float*>(ptr(dinit)), B, H, N, D,
                t_offset, ptr(ws), bytes(ws), s),
            rows ? "kdecay_scan_rows_bwd" : "kdecay_scan_bwd");
    }
    return {dlam, dV, dinit, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

std::pair<Tensor, Tensor> scan_train(const Tensor& lam, const Tensor& V, const std::optional<Tensor>& init,
                                     int64_t t_offset, at::ScalarType out_dtype, bool rows, bool sequential) {
  const auto r = ScanNode::apply(lam, V, init, t_offset, out_dtype, rows, sequential);
  return {r[0], r[1]};
}

// Whether the kernels read `lam` as it is.
bool plain_lam(const Tensor& lam, int64_t H, const at::Device& d) {
  return lam.dim() == 1 && lam.size(0) == H && lam.scalar_type() == at::kFloat && lam.is_contiguous() &&
         lam.device() == d;
}

// Whether `s` is fp32 [B,H,D], contiguous, on device d.
bool plain_state(const Tensor& s, int64_t B, int64_t H, int64_t D, const at::Device& d) {
  return s.dim() == 3 && s.size(0) == B && s.size(1) == H && s.size(2) == D && s.scalar_type() == at::kFloat &&
         s.is_contiguous() && s.device() == d;
}

// A torch.Tensor or Parameter itself, whose memory holds its values: subclasses go
// through Python, where their __torch_function__ applies, and so do views that are
// negated when read (the imaginary part of a conjugate).
bool plain_tensor(PyObject* o) { return THPVariable_CheckExact(o) && !THPVariable_Unpack(o).is_neg(); }

// First byte and one past the last of a tensor's elements.
std::pair<uintptr_t, uintptr_t> extent(const Tensor& t) {
  const uintptr_t p = reinterpret_cast<uintptr_t>(t.const_data_ptr());
  if (t.numel() == 0) return {p, p};
  int64_t last = 0;
  for (int64_t k = 0; k < t.dim(); ++k) last += (t.size(k) - 1) * t.stride(k);
  return {p, p + (last + 1) * t.element_size()};
}

// Whether memory of `out` may be read by other workgroups after one has written
// it: `out` shares a byte range with V, other than being the very same view (each
// workgroup reads its rows before it writes them), or with another input.
bool meets(const Tensor& out, const Tensor& V, const Tensor& lam, const std::optional<Tensor>& init) {
  const auto [lo, hi] = extent(out);
  const auto shares = [lo = lo, hi = hi](const Tensor& t) {
    const auto [a, b] = extent(t);
    return a < hi && lo < b;
  };
  const bool same = out.const_data_ptr() == V.const_data_ptr() && out.strides() == V.strides() &&
                    out.scalar_type() == V.scalar_type();
  return (!same && shares(V)) || shares(lam) || (init.has_value() && shares(*init));
}

// Whether the kernels can read these tensors and write `out` as they lie: none
// lazily negated, and out apart from the inputs.  Anything but a tensor is left to
// the checks that follow.
bool as_they_lie(const py::object& lam_o, const py::object& V_o, const py::object& init_o, const py::object& out_o) {
  for (PyObject* o : {lam_o.ptr(), V_o.ptr(), init_o.ptr(), out_o.ptr()})
    if (THPVariable_Check(o) && THPVariable_Unpack(o).is_neg()) return false;
  if (!THPVariable_Check(out_o.ptr()) || !THPVariable_Check(V_o.ptr()) || !THPVariable_Check(lam_o.ptr())) return true;
  const bool has_init = THPVariable_Check(init_o.ptr());
  return !meets(THPVariable_Unpack(out_o.ptr()), THPVariable_Unpack(V_o.ptr()), THPVariable_Unpack(lam_o.ptr()),
                has_init ? std::optional<Tensor>(THPVariable_Unpack(init_o.ptr())) : std::nullopt);
}

// global_decay_scan(lam, V, ...) into a new y, for arguments the kernels read as
// they are; None (nothing launched) otherwise.
py::object scan(const py::object& lam_o, const py::object& V_o, const py::object& init_o, bool want_final,
                const py::object& t_offset_o, const py::object& out_dtype_o) {
  if (!plain_tensor(lam_o.ptr()) || !plain_tensor(V_o.ptr()) || !PyLong_CheckExact(t_offset_o.ptr())) return py::none();
  const Tensor &lam = THPVariable_Unpack(lam_o.ptr()), &V = THPVariable_Unpack(V_o.ptr());
  Tensor init;
  if (!init_o.is_none()) {
    if (!plain_tensor(init_o.ptr())) return py::none();
    init = THPVariable_Unpack(init_o.ptr());
  }
  if (!V.is_cuda() || V.dim() != 4 || V.numel() == 0) return py::none();
  const at::Device d = V.device();
  if (d.index() != c10::hip::current_device()) return py::none();
  const int64_t B = V.size(0), H = V.size(1), N = V.size(2), D = V.size(3);
  const at::ScalarType vt = V.scalar_type();
  // Not a torch.dtype: the general path, which takes what torch.empty_like does.
  if (!out_dtype_o.is_none() && !THPDtype_Check(out_dtype_o.ptr())) return py::none();
  const at::ScalarType ot = out_dtype_o.is_none() ? vt : out_dtype_o.cast<at::ScalarType>();
  const int v_code = dtype_code(vt), o_code = dtype_code(ot);
  if (v_code < 0 || (ot != vt && (ot != at::kFloat || vt == at::kDouble))) return py::none();
  if (!plain_lam(lam, H, d) || (init.defined() && !plain_state(init, B, H, D, d))) return py::none();
  int overflow = 0;  // the general path takes integers beyond 64 bits as ctypes does
  const int64_t t_offset = PyLong_AsLongLongAndOverflow(t_offset_o.ptr(), &overflow);
  if (overflow) return py::none();

  const bool train = at::GradMode::is_enabled() &&
                     (V.requires_grad() || lam.requires_grad() || (init.defined() && init.requires_grad()));
  const bool chunked = chunked_head_dim(D, V.element_size()) && !narrow_rows(V, train, ot != vt);
  if (!chunked && !row_vectors_ok(D, V.element_size())) return py::none();
  const hipStream_t s = stream_of(d);
  if (train) {
    if (vt == at::kDouble || V.is_inference()) return py::none();
    // The workspace is checked before the node is made: where it has to grow,
    // the caller decides what a stream capture does.
    const size_t nbytes = train_sizes(B, H, N, D, v_code, !chunked).second;
    if (nbytes && bytes(find_workspace(d, s)) < nbytes) return py::none();
    std::pair<Tensor, Tensor> r;
    {
      py::gil_scoped_release nogil;
      r = scan_train(lam, V, init.defined() ? std::optional<Tensor>(init) : std::nullopt, t_offset, ot, !chunked,
                     false);
    }
    const auto& [y, fin] = r;
    return want_final ? py::object(py::make_tuple(y, fin)) : py::cast(y);
  }

  if (chunked ? !vector_layout_ok(V) : V.stride(3) != 1) return py::none();
  const size_t nbytes =
      (chunked ? kdecay_scan_workspace_bytes : kdecay_scan_rows_workspace_bytes)(B, H, N, D, v_code);
  const Tensor ws = nbytes ? find_workspace(d, s) : Tensor();
  if (bytes(ws) < nbytes) return py::none();
  Tensor out, fin;
  int rc = 0;
  {
    py::gil_scoped_release nogil;
    at::AutoDispatchBelowADInplaceOrView below;  // new buffers only: nothing to record
    out = at::empty_like(V, V.options().dtype(ot));
    if (want_final) fin = at::empty({B, H, D}, V.options().dtype(at::kFloat));
    if (out_layout_ok(out, !chunked))
      rc = (chunked ? kdecay_scan_fwd : kdecay_scan_fwd_rows)(
          V.data_ptr(), v_code, V.strides().data(), out.data_ptr(), o_code, out.strides().data(),
          lam.data_ptr<float>(), static_cast<float*>(ptr(init)), static_cast<float*>(ptr(fin)), B, H, N, D, t_offset,
          ptr(ws), bytes(ws), s);
    else
      out = Tensor();
  }
  if (!out.defined()) return py::none();
  check(rc, chunked ? "kdecay_scan_fwd" : "kdecay_scan_fwd_rows");
  return want_final ? py::object(py::make_tuple(out, fin)) : py::cast(out);
}

// decay_step for arguments the kernel reads as they are; None (nothing launched)
// otherwise.
py::object decay_step(const py::object& lam_o, const py::object& state_o, const py::object& v_o,
                      const py::object& pos_o, const py::object& out_o, const py::object& new_o,
                      const py::object& out_dtype_o) {
  if (!plain_tensor(lam_o.ptr()) || !plain_tensor(state_o.ptr()) || !plain_tensor(v_o.ptr())) return py::none();
  const Tensor &lam = THPVariable_Unpack(lam_o.ptr()), &state = THPVariable_Unpack(state_o.ptr()),
               &v = THPVariable_Unpack(v_o.ptr());
  if (!state.is_cuda() || state.dim() != 3 || state.numel() == 0) return py::none();
  const at::Device d = state.device();
  if (d.index() != c10::hip::current_device()) return py::none();
  const int64_t B = state.size(0), H = state.size(1), D = state.size(2);
  const int v_code = dtype_code(v.scalar_type());
  if (!plain_state(state, B, H, D, d) || !plain_lam(lam, H, d)) return py::none();
  if (v_code < 0 || v_code == KDECAY_F64 || v.device() != d || v.numel() != B * H * D || !v.is_contiguous())
    return py::none();
  const int32_t* pos = nullptr;
  int64_t pos_all = 0;
  if (PyLong_CheckExact(pos_o.ptr())) {
    int overflow = 0;
    pos_all = PyLong_AsLongLongAndOverflow(pos_o.ptr(), &overflow);
    if (overflow) return py::none();
  } else {
    if (!plain_tensor(pos_o.ptr())) return py::none();
    const Tensor& p = THPVariable_Unpack(pos_o.ptr());
    if (p.scalar_type() != at::kInt || p.device() != d || p.numel() != B || !p.is_contiguous()) return py::none();
    pos = p.data_ptr<int32_t>();
  }
  Tensor out, next;
  if (!new_o.is_none()) {
    if (!plain_tensor(new_o.ptr())) return py::none();
    next = THPVariable_Unpack(new_o.ptr());
    if (!plain_state(next, B, H, D, d)) return py::none();
  }
  at::ScalarType ot = at::kFloat;
  if (!out_o.is_none()) {
    if (!plain_tensor(out_o.ptr())) return py::none();
    out = THPVariable_Unpack(out_o.ptr());
    if (!out.is_contiguous() || out.numel() != B * H * D || out.device() != d) return py::none();
    ot = out.scalar_type();
  } else {
    if (!THPDtype_Check(out_dtype_o.ptr())) return py::none();
    ot = out_dtype_o.cast<at::ScalarType>();
  }
  const int o_code = dtype_code(ot);
  if (o_code < 0 || o_code == KDECAY_F64) return py::none();
  const bool given_out = out.defined(), given_next = next.defined();
  int rc;
  {
    py::gil_scoped_release nogil;
    at::AutoDispatchBelowADInplaceOrView below;  // new buffers only: nothing to record
    if (!given_next) next = at::empty({B, H, D}, state.options());
    if (!given_out) out = at::empty({B, H, D}, state.options().dtype(ot));
    rc = kdecay_step(lam.data_ptr<float>(), state.data_ptr<float>(), v.data_ptr(), v_code, next.data_ptr<float>(),
                     out.data_ptr(), o_code, pos, pos_all, B, H, D, stream_of(d));
  }
  check(rc, "kdecay_step");
  return py::make_tuple(given_out ? out_o : py::cast(out), given_next ? new_o : py::cast(next));
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  m.doc() = "Host path of kilat_amd (see native.cpp).";
  m.def("scan", &scan);
  m.def("decay_step", &decay_step);
  m.def("scan_train", &scan_train, py::call_guard<py::gil_scoped_release>());
  m.def("chunked_route", &chunked_route);
  m.def("rows_out_ok", &rows_out_ok);
  m.def("as_they_lie", &as_they_lie);
  m.def("meets", &meets);
  m.def("chunked_head_dim", &chunked_head_dim);
  m.def("row_vectors_ok", &row_vectors_ok);
  m.def("vector_layout_ok", &vector_layout_ok);
  m.def("bwd_rows_fit", &bwd_rows_fit);
  m.def("narrow_rows", &narrow_rows, py::arg("V"), py::arg("train") = false, py::arg("wide") = false);
}
