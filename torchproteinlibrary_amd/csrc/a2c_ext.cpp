// a2c_ext.cpp -- the Angles2Coords part of the pybind11 module
// `_FullAtomModel`: tensor glue over the C ABI in include/tpl_a2c.h, with the
// reference's entry-point names and argument orders
// (Layers/FullAtomModel/main.cpp:10-14,
// Layers/FullAtomModel/Angles2Coords/angles2coords_interface.cpp:8-144).
// The reference takes CPU tensors; these take GPU tensors (the sequences as a
// uint8 [batch, length] tensor on the same device).  Work goes to torch's
// current HIP stream of the angles' device.
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <string>
#include <tuple>
#include <vector>

#include "a2c_flagged.h"
#include "host_flags.h"
#include "native_fn.h"
#include "tpl_a2c.h"

namespace {

#define A2C_CHECK_GPU(x)                                                      \
    TORCH_CHECK((x).is_cuda(), #x " must be a GPU tensor");                   \
    TORCH_CHECK((x).is_contiguous(), #x " must be contiguous")

void check_rc(int rc, const char* what) {
    TORCH_CHECK(rc == TPL_A2C_OK, what, " failed: ", tpl_a2c_strerror(rc));
}

int dtype_code(const torch::Tensor& t) {
    if (t.scalar_type() == torch::kFloat) return TPL_A2C_F32;
    if (t.scalar_type() == torch::kDouble) return TPL_A2C_F64;
    TORCH_CHECK(false, "angles must be float32 or float64, got ", t.scalar_type());
    return -1;
}

void check_common(const torch::Tensor& seqs, const torch::Tensor& angles) {
    A2C_CHECK_GPU(seqs);
    A2C_CHECK_GPU(angles);
    TORCH_CHECK(seqs.scalar_type() == torch::kByte && seqs.dim() == 2, "sequences must be uint8 [batch, length]");
    TORCH_CHECK(angles.dim() == 3 && angles.size(1) == 8, "angles must be [batch, 8, length], got ", angles.sizes());
    TORCH_CHECK(seqs.size(0) == angles.size(0), "sequences and angles differ in batch");
    TORCH_CHECK(seqs.device() == angles.device(), "sequences must be on the device of the angles");
    TORCH_CHECK(angles.size(0) <= INT32_MAX && angles.size(2) <= INT32_MAX / 8 && seqs.size(1) <= INT32_MAX,
                "inputs too large");
}

uint32_t* status_ptr(const c10::optional<torch::Tensor>& status, const torch::Tensor& like) {
    if (!status.has_value() || !status->defined()) return nullptr;
    A2C_CHECK_GPU(*status);
    TORCH_CHECK(status->scalar_type() == torch::kInt && status->numel() >= 1, "status must be an int32 tensor");
    TORCH_CHECK(status->device() == like.device(), "status must be on the device of the angles");
    return reinterpret_cast<uint32_t*>(status->data_ptr());
}

// The optional scheduling order (tpl_a2c_forward_ordered): int32 [batch] on
// the angles' device.
const int32_t* order_ptr(const c10::optional<torch::Tensor>& order, const torch::Tensor& like) {
    if (!order.has_value() || !order->defined()) return nullptr;
    A2C_CHECK_GPU(*order);
    TORCH_CHECK(order->scalar_type() == torch::kInt && order->dim() == 1 && order->size(0) == like.size(0),
                "order must be int32 [batch]");
    TORCH_CHECK(order->device() == like.device(), "order must be on the device of the angles");
    return order->data_ptr<int32_t>();
}

hipStream_t stream_of(const torch::Tensor& t) {
    return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// `need` bytes of workspace from torch's allocator, or none if there is no
// memory for them: the kernels without a workspace do the same.
torch::Tensor workspace(size_t need, const torch::Tensor& like) {
    if (need == 0) return torch::Tensor();
    try {
        return torch::empty({(int64_t)need}, like.options().dtype(torch::kByte));
    } catch (const c10::OutOfMemoryError&) {
        return torch::Tensor();
    }
}
void* ptr(const torch::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// The workspaces of the two directions, where the form that they take reads one.
torch::Tensor forward_workspace(const torch::Tensor& angles, int64_t atoms_stride, bool names) {
    const int B = (int)angles.size(0), L = (int)angles.size(2);
    const bool groups =
        tplx_a2c_forward_form(dtype_code(angles), B, L, (int)atoms_stride, names, 1) == TPLX_A2C_FWD_GROUPS;
    return workspace(groups ? tplx_a2c_workspace_bytes(B, L) : 0, angles);
}
torch::Tensor backward_workspace(const torch::Tensor& grad_angles, int64_t atoms_stride) {
    const int B = (int)grad_angles.size(0), L = (int)grad_angles.size(2);
    const bool groups =
        tplx_a2c_backward_form(dtype_code(grad_angles), B, L, (int)atoms_stride, 1) == TPLX_A2C_BWD_GROUPS;
    return workspace(groups ? tplx_a2c_backward_workspace_bytes(B, L) : 0, grad_angles);
}

void forward_on(const torch::Tensor& sequences, const torch::Tensor& input_angles,
                const torch::Tensor& output_coords, const torch::Tensor& res_names, const torch::Tensor& atom_names,
                uint32_t* status, uint32_t* flags, const c10::optional<torch::Tensor>& order, hipStream_t stream) {
    check_common(sequences, input_angles);
    A2C_CHECK_GPU(output_coords);
    A2C_CHECK_GPU(res_names);
    A2C_CHECK_GPU(atom_names);
    const int64_t B = input_angles.size(0);
    TORCH_CHECK(output_coords.scalar_type() == input_angles.scalar_type(), "coordinates must have the dtype of the angles");
    TORCH_CHECK(output_coords.dim() == 2 && output_coords.size(0) == B && output_coords.size(1) % 3 == 0,
                "output_coords must be [batch, 3*atoms]");
    const int64_t A = output_coords.size(1) / 3;
    TORCH_CHECK(A <= INT32_MAX / 3, "output_coords too large");
    for (const auto* n : {&res_names, &atom_names}) {
        TORCH_CHECK(n->scalar_type() == torch::kByte && n->dim() == 3 && n->size(0) == B && n->size(1) == A &&
                        n->size(2) == 4,
                    "names must be uint8 [batch, atoms, 4]");
        TORCH_CHECK(n->device() == input_angles.device(), "names must be on the device of the angles");
    }
    TORCH_CHECK(output_coords.device() == input_angles.device(), "coordinates must be on the device of the angles");
    const torch::Tensor ws = forward_workspace(input_angles, A, true);
    check_rc(tplx_a2c_forward(TPLX_A2C_FWD_AUTO, order_ptr(order, input_angles), dtype_code(input_angles),
                              sequences.data_ptr<uint8_t>(), (int)sequences.size(1), input_angles.data_ptr(),
                              (int)input_angles.size(2), output_coords.data_ptr(), res_names.data_ptr<uint8_t>(),
                              atom_names.data_ptr<uint8_t>(), (int)A, ptr(ws), status, flags, (int)B, stream),
             "Angles2Coords_forward");
}

void forward(torch::Tensor sequences, torch::Tensor input_angles, torch::Tensor output_coords,
             torch::Tensor res_names, torch::Tensor atom_names, c10::optional<torch::Tensor> status,
             c10::optional<torch::Tensor> order) {
    check_common(sequences, input_angles);
    c10::DeviceGuard guard(input_angles.device());
    forward_on(sequences, input_angles, output_coords, res_names, atom_names, status_ptr(status, input_angles),
               nullptr, order, stream_of(input_angles));
}

// As forward without a status; waits for the work and returns its status bits
// (a2c_flagged.h).
int64_t forward_checked(torch::Tensor sequences, torch::Tensor input_angles, torch::Tensor output_coords,
                        torch::Tensor res_names, torch::Tensor atom_names, c10::optional<torch::Tensor> order) {
    check_common(sequences, input_angles);
    c10::DeviceGuard guard(input_angles.device());
    hipStream_t stream = stream_of(input_angles);
    return host_flags::run(stream, [&](uint32_t* flags) {
        forward_on(sequences, input_angles, output_coords, res_names, atom_names, nullptr, flags, order, stream);
    });
}

void backward_on(const torch::Tensor& grad_atoms, const torch::Tensor& grad_angles, const torch::Tensor& sequences,
                 const torch::Tensor& coords, uint32_t* status, uint32_t* flags,
                 const c10::optional<torch::Tensor>& order, hipStream_t stream) {
    A2C_CHECK_GPU(grad_atoms);
    A2C_CHECK_GPU(coords);
    const int64_t B = grad_angles.size(0);
    TORCH_CHECK(grad_atoms.scalar_type() == grad_angles.scalar_type() &&
                    coords.scalar_type() == grad_angles.scalar_type(),
                "gradients and coordinates must have one dtype");
    TORCH_CHECK(grad_atoms.dim() == 2 && grad_atoms.size(0) == B && grad_atoms.size(1) % 3 == 0,
                "grad_atoms must be [batch, 3*atoms]");
    TORCH_CHECK(coords.sizes() == grad_atoms.sizes(), "coords must have the shape of grad_atoms");
    TORCH_CHECK(grad_atoms.device() == grad_angles.device() && coords.device() == grad_angles.device(),
                "gradients and coordinates must be on one device");
    const int64_t A = grad_atoms.size(1) / 3;
    TORCH_CHECK(A <= INT32_MAX / 3, "grad_atoms too large");
    const torch::Tensor ws = backward_workspace(grad_angles, A);
    check_rc(tplx_a2c_backward(TPLX_A2C_BWD_AUTO, order_ptr(order, grad_angles), dtype_code(grad_angles),
                               sequences.data_ptr<uint8_t>(), (int)sequences.size(1), coords.data_ptr(),
                               grad_atoms.data_ptr(), (int)A, grad_angles.data_ptr(), (int)grad_angles.size(2),
                               ptr(ws), status, flags, (int)B, stream),
             "Angles2Coords_backward");
}

// From the forward's coordinates (what the Python layer saves).
void backward_coords(torch::Tensor grad_atoms, torch::Tensor grad_angles, torch::Tensor sequences,
                     torch::Tensor coords, c10::optional<torch::Tensor> status,
                     c10::optional<torch::Tensor> order) {
    check_common(sequences, grad_angles);
    c10::DeviceGuard guard(grad_angles.device());
    backward_on(grad_atoms, grad_angles, sequences, coords, status_ptr(status, grad_angles), nullptr, order,
                stream_of(grad_angles));
}

// As backward_coords without a status; waits for the work and returns its
// status bits (a2c_flagged.h).
int64_t backward_checked(torch::Tensor grad_atoms, torch::Tensor grad_angles, torch::Tensor sequences,
                         torch::Tensor coords, c10::optional<torch::Tensor> order) {
    check_common(sequences, grad_angles);
    c10::DeviceGuard guard(grad_angles.device());
    hipStream_t stream = stream_of(grad_angles);
    return host_flags::run(stream, [&](uint32_t* flags) {
        backward_on(grad_atoms, grad_angles, sequences, coords, nullptr, flags, order, stream);
    });
}

// The reference's signature (angles, not coordinates): the coordinates are
// computed again first, as the reference rebuilds its conformation.
void backward(torch::Tensor grad_atoms, torch::Tensor grad_angles, torch::Tensor sequences,
              torch::Tensor input_angles, c10::optional<torch::Tensor> status) {
    check_common(sequences, input_angles);
    A2C_CHECK_GPU(grad_atoms);
    TORCH_CHECK(grad_angles.sizes() == input_angles.sizes(), "grad_angles must have the shape of the angles");
    TORCH_CHECK(grad_atoms.dim() == 2 && grad_atoms.size(0) == input_angles.size(0) && grad_atoms.size(1) % 3 == 0,
                "grad_atoms must be [batch, 3*atoms]");
    const int64_t A = grad_atoms.size(1) / 3;
    TORCH_CHECK(A <= INT32_MAX / 3, "grad_atoms too large");
    c10::DeviceGuard guard(input_angles.device());
    auto coords = torch::empty_like(grad_atoms);
    check_rc(tpl_a2c_forward(dtype_code(input_angles), sequences.data_ptr<uint8_t>(), (int)sequences.size(1),
                             input_angles.data_ptr(), (int)input_angles.size(2), coords.data_ptr(), nullptr,
                             nullptr, (int)A, status_ptr(status, input_angles), (int)input_angles.size(0),
                             stream_of(input_angles)),
             "Angles2Coords_backward");
    backward_coords(grad_atoms, grad_angles, sequences, coords, status, c10::nullopt);
}

// The autograd function of a plain call (native_fn.h); what it does is written
// at Angles2CoordsFunction.
constexpr const char* kLayer = "torchproteinlibrary_amd.FullAtomModel.Angles2Coords.Angles2Coords";
using native_fn::variable_list;
using torch::Tensor;
using torch::autograd::AutogradContext;

struct Angles2Coords : torch::autograd::Function<Angles2Coords> {
    static variable_list forward(AutogradContext* ctx, Tensor angles, Tensor sequences, int64_t max_atoms,
                                 c10::optional<Tensor> order) {
        angles = angles.contiguous();
        const torch::Device dev = angles.device();
        c10::DeviceGuard guard(dev);
        const Tensor seqs = sequences.to(dev).contiguous();
        check_common(seqs, angles);
        if (order.has_value()) order = order->to(dev).contiguous();
        const int64_t B = angles.size(0);
        const auto bytes = angles.options().dtype(torch::kByte);
        Tensor coords = torch::empty({B, 3 * max_atoms}, angles.options());
        Tensor res_names = torch::empty({B, max_atoms, 4}, bytes), atom_names = torch::empty({B, max_atoms, 4}, bytes);
        const hipStream_t s = stream_of(angles);
        const uint32_t bits = native_fn::run(s, [&](uint32_t* flags) {
            forward_on(seqs, angles, coords, res_names, atom_names, nullptr, flags, order, s);
        });
        if (bits) native_fn::python(kLayer, "_check", bits, coords, "forward");
        ctx->save_for_backward({seqs, coords});
        ctx->saved_data["length"] = angles.size(2);
        ctx->saved_data["order"] = order;
        ctx->mark_non_differentiable({res_names, atom_names});
        ctx->set_materialize_grads(false);  // the names' would be filled with zeros for nothing
        return {coords, res_names, atom_names};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        return native_fn::backward(grads, [&]() -> variable_list {
            const Tensor &seqs = saved[0], &coords = saved[1];
            const Tensor g = grads[0].defined() ? grads[0].contiguous() : torch::zeros_like(coords);
            c10::DeviceGuard guard(coords.device());
            const hipStream_t s = stream_of(coords);
            Tensor out = torch::empty({coords.size(0), 8, ctx->saved_data["length"].toInt()}, coords.options());
            check_common(seqs, out);
            const auto order = ctx->saved_data["order"].toOptional<Tensor>();
            const uint32_t bits = native_fn::run(s, [&](uint32_t* flags) {
                backward_on(g, out, seqs, coords, nullptr, flags, order, s);
            });
            if (bits) native_fn::python(kLayer, "_check", bits, out, "backward");
            return {out, Tensor(), Tensor(), Tensor()};
        });
    }
};

// (coords, res_names, atom_names), or nothing if the call is not a plain one.
// max_atoms < 0: the largest of num_atoms, read from wherever it is (B integers
// straight to the host; the largest found by a kernel first takes longer).
c10::optional<std::tuple<Tensor, Tensor, Tensor>> apply(Tensor angles, Tensor sequences, Tensor num_atoms,
                                                        c10::optional<Tensor> order, int64_t max_atoms) {
    if (!native_fn::plain({&angles}) || sequences.requires_grad() || num_atoms.requires_grad() ||
        !torch::isIntegralType(num_atoms.scalar_type(), false) || angles.dim() != 3 || angles.size(1) != 8)
        return c10::nullopt;
    if (max_atoms < 0) {
        const Tensor n = num_atoms.to(torch::kCPU).to(torch::kLong).contiguous();
        const int64_t* p = n.data_ptr<int64_t>();
        max_atoms = n.numel() ? *std::max_element(p, p + n.numel()) : 0;
    }
    auto out = Angles2Coords::apply(angles, sequences, max_atoms, order);
    return std::make_tuple(out[0], out[1], out[2]);
}

// The sequences of a call as the device wants them: (atom counts, the uint8
// [batch, longest + 1] tensor of convertStringList on the device, the counts as
// int32 on the device), copied from pinned memory without a wait; None if
// a sequence is not a string of the 20 letters, the call is not a plain one (a
// mode may hand out tensors without memory), or a capture is open (the copies
// would read their staging memory again on each replay).
pybind11::object prepare(pybind11::list sequences, torch::Tensor angles) {
    namespace py = pybind11;
    const size_t B = sequences.size();
    if (B == 0 || !native_fn::plain({&angles})) return py::none();
    c10::DeviceGuard guard(angles.device());
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream_of(angles), &capture) != hipSuccess || capture != hipStreamCaptureStatusNone)
        return py::none();
    std::vector<std::pair<const char*, size_t>> s(B);
    size_t longest = 0;
    std::vector<int32_t> counts(B);
    for (size_t i = 0; i < B; ++i) {
        PyObject* o = PyList_GET_ITEM(sequences.ptr(), (Py_ssize_t)i);
        if (!PyUnicode_CheckExact(o) || !PyUnicode_IS_COMPACT_ASCII(o)) return py::none();
        s[i] = {reinterpret_cast<const char*>(PyUnicode_1BYTE_DATA(o)), (size_t)PyUnicode_GET_LENGTH(o)};
        counts[i] = tpl_a2c_num_atoms(s[i].first);
        if (counts[i] < 0 || std::strlen(s[i].first) != s[i].second) return py::none();
        longest = std::max(longest, s[i].second);
    }
    const auto pinned = torch::TensorOptions().pinned_memory(true);
    const Tensor seqs = torch::empty({(int64_t)B, (int64_t)longest + 1}, pinned.dtype(torch::kByte));
    const Tensor n = torch::empty({(int64_t)B}, pinned.dtype(torch::kInt));
    std::memset(seqs.data_ptr(), 0, seqs.nbytes());
    for (size_t i = 0; i < B; ++i)
        std::memcpy(seqs.data_ptr<uint8_t>() + i * (longest + 1), s[i].first, s[i].second);
    std::memcpy(n.data_ptr(), counts.data(), B * sizeof(int32_t));
    const Tensor dseqs = seqs.to(angles.device(), /*non_blocking=*/true);
    const Tensor dn = n.to(angles.device(), /*non_blocking=*/true);
    return py::make_tuple(counts, dseqs, dn);
}

int num_atoms(const std::string& sequence) {
    const int n = tpl_a2c_num_atoms(sequence.c_str());
    TORCH_CHECK(n >= 0, "getSeqNumAtoms: sequence holds a letter outside the 20 amino acids: ", sequence);
    return n;
}

// Timing loop for bench.py: sets of [sequences, angles, coords, grad_coords,
// grad_angles] (and optionally the scheduling order, int32 [batch]) rotated
// per launch (no names, no status).  Returns the average
// HIP-event ms of (fwd+bwd step, fwd alone, bwd alone) over `steps` launches
// each, after `warmup`.
std::tuple<double, double, double> bench(std::vector<std::vector<torch::Tensor>> sets, int64_t steps,
                                         int64_t warmup) {
    TORCH_CHECK(!sets.empty() && steps > 0 && warmup >= 0, "bench: bad arguments");
    for (auto& t : sets) {
        TORCH_CHECK(t.size() == 5 || t.size() == 6, "bench: a set has 5 tensors (6 with an order)");
        if (t.size() == 6) (void)order_ptr(t[5], t[1]);
        check_common(t[0], t[1]);
        for (int k = 2; k < 5; ++k) {
            A2C_CHECK_GPU(t[k]);
            TORCH_CHECK(t[k].scalar_type() == t[1].scalar_type(), "bench: dtype mismatch");
        }
        TORCH_CHECK(t[2].sizes() == t[3].sizes() && t[4].sizes() == t[1].sizes(), "bench: shape mismatch");
    }
    c10::DeviceGuard guard(sets[0][1].device());
    hipStream_t stream = stream_of(sets[0][1]);
    const int dt = dtype_code(sets[0][1]);
    const torch::Tensor ws = forward_workspace(sets[0][1], sets[0][2].size(1) / 3, false),
                        bws = backward_workspace(sets[0][1], sets[0][2].size(1) / 3);
    for (auto& t : sets) TORCH_CHECK(t[1].sizes() == sets[0][1].sizes(), "bench: sets differ in shape");
    auto fwd = [&](std::vector<torch::Tensor>& t) {
        const int32_t* order = t.size() == 6 ? t[5].data_ptr<int32_t>() : nullptr;
        check_rc(tplx_a2c_forward(TPLX_A2C_FWD_AUTO, order, dt, t[0].data_ptr<uint8_t>(), (int)t[0].size(1),
                                  t[1].data_ptr(), (int)t[1].size(2), t[2].data_ptr(), nullptr, nullptr,
                                  (int)(t[2].size(1) / 3), ptr(ws), nullptr, nullptr, (int)t[1].size(0), stream),
                 "forward");
    };
    auto bwd = [&](std::vector<torch::Tensor>& t) {
        const int32_t* order = t.size() == 6 ? t[5].data_ptr<int32_t>() : nullptr;
        check_rc(tplx_a2c_backward(TPLX_A2C_BWD_AUTO, order, dt, t[0].data_ptr<uint8_t>(), (int)t[0].size(1),
                                   t[2].data_ptr(), t[3].data_ptr(), (int)(t[3].size(1) / 3), t[4].data_ptr(),
                                   (int)t[4].size(2), ptr(bws), nullptr, nullptr, (int)t[1].size(0), stream),
                 "backward");
    };
    hipEvent_t e0, e1;
    TORCH_CHECK(hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess, "hipEventCreate failed");
    auto timed = [&](int which) {
        auto body = [&](std::vector<torch::Tensor>& t) {
            if (which != 2) fwd(t);
            if (which != 1) bwd(t);
        };
        for (int64_t i = 0; i < warmup; ++i) body(sets[i % sets.size()]);
        TORCH_CHECK(hipEventRecord(e0, stream) == hipSuccess, "hipEventRecord failed");
        for (int64_t i = 0; i < steps; ++i) body(sets[i % sets.size()]);
        TORCH_CHECK(hipEventRecord(e1, stream) == hipSuccess, "hipEventRecord failed");
        TORCH_CHECK(hipEventSynchronize(e1) == hipSuccess, "hipEventSynchronize failed");
        float ms = 0.f;
        TORCH_CHECK(hipEventElapsedTime(&ms, e0, e1) == hipSuccess, "hipEventElapsedTime failed");
        return (double)ms / steps;
    };
    const double step = timed(0), f = timed(1), b = timed(2);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return {step, f, b};
}

}  // namespace

void register_a2c(pybind11::module& m) {
    namespace py = pybind11;
    auto st = py::arg("status") = py::none();
    auto od = py::arg("order") = py::none();
    m.def("Angles2Coords_forward", &forward, "full-atom coordinates and names from angles (GPU)",
          py::arg("sequences"), py::arg("input_angles"), py::arg("output_coords"), py::arg("res_names"),
          py::arg("atom_names"), st, od);
    m.def("Angles2Coords_forward_checked", &forward_checked, "status bits of the forward, once it has run",
          py::arg("sequences"), py::arg("input_angles"), py::arg("output_coords"), py::arg("res_names"),
          py::arg("atom_names"), od, py::call_guard<py::gil_scoped_release>());
    m.def("Angles2Coords_backward", &backward, "gradient of the coordinates with respect to the angles (GPU)",
          py::arg("grad_atoms"), py::arg("grad_angles"), py::arg("sequences"), py::arg("input_angles"), st);
    m.def("Angles2Coords_backward_coords", &backward_coords,
          "the same from the forward's coordinates (GPU)", py::arg("grad_atoms"), py::arg("grad_angles"),
          py::arg("sequences"), py::arg("coords"), st, od);
    m.def("Angles2Coords_backward_checked", &backward_checked, "status bits of the backward, once it has run",
          py::arg("grad_atoms"), py::arg("grad_angles"), py::arg("sequences"), py::arg("coords"), od,
          py::call_guard<py::gil_scoped_release>());
    m.def("Angles2Coords_apply", &apply, "a plain differentiable call: (coords, names, names), or None",
          py::call_guard<py::gil_scoped_release>());
    m.def("Angles2Coords_prepare", &prepare, "atom counts and device tensors of sequences, or None");
    m.def("getSeqNumAtoms", &num_atoms, "atoms of a sequence", py::arg("sequence"));
    m.def("a2c_bench", &bench, "average event ms of Angles2Coords (step, fwd, bwd)");
}
