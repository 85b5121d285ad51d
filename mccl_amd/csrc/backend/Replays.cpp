// Replays.cpp -- allreduce replays over Python lists of tensors, without a Python statement
// per tensor: addresses, sizes and types are read here, the workspace comes from torch's
// allocator, and the calls into libmcclx run with the interpreter lock released.
//
// What is not a plain list of contiguous ROCm tensors, of one type and size within a group, is
// left to the Python form (the functions return None and have done nothing), which words the error.
#include "backend/Replays.hpp"

#include <torch/extension.h>

#include <torch/csrc/autograd/python_variable.h>

#include <cctype>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "backend/Device.hpp"
#include "mcclx.h"

namespace py = pybind11;

namespace mccl {
namespace {

int dtype_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return MCCLX_F32;
        case at::kHalf: return MCCLX_F16;
        case at::kBFloat16: return MCCLX_BF16;
        default: return -1;
    }
}

struct How {
    int op, algo, wire, mode, acc;
};

// One group: `tensors` is a list or tuple of the virtual ranks' tensors; their addresses go to
// `ptrs` (r->tensors is set by the caller, once `ptrs` has stopped growing).
bool read_group(PyObject* tensors, const How& how, mcclx_replay* r, std::vector<void*>& ptrs) {
    if (!PyList_Check(tensors) && !PyTuple_Check(tensors)) return false;
    const Py_ssize_t world = PySequence_Fast_GET_SIZE(tensors);
    if (world < 1) return false;
    PyObject** items = PySequence_Fast_ITEMS(tensors);
    std::memset(r, 0, sizeof *r);
    for (Py_ssize_t i = 0; i < world; ++i) {
        if (!THPVariable_Check(items[i])) return false;
        const at::Tensor& t = THPVariable_Unpack(items[i]);
        if (!dev::on_device(t) || !t.is_contiguous()) return false;
        if (i == 0) {
            r->dtype = dtype_code(t);
            r->numel = static_cast<uint64_t>(t.numel());
            if (r->dtype < 0) return false;
        } else if (dtype_code(t) != r->dtype || static_cast<uint64_t>(t.numel()) != r->numel) {
            return false;
        }
        ptrs.push_back(t.data_ptr());
    }
    r->world = static_cast<int32_t>(world);
    r->op = how.op;
    r->algo = how.algo;
    r->wire_bf16 = how.wire;
    r->mode = how.mode;
    r->acc = how.acc;
    return true;
}

constexpr uint32_t kWaitSpinUs = 1000;

uint64_t aligned(uint64_t n) { return (n + 255) / 256 * 256; }

// Orders the queue behind torch's current stream, issues the replays in a workspace of
// their own and waits for them.
int run(mcclx_ctx* ctx, int device, std::vector<mcclx_replay>& reps) {
    uint64_t total = 0;
    const mcclx_replay* before = nullptr;
    for (mcclx_replay& r : reps) {  // (operation, algorithm, mode and wire form are the call's)
        const bool alike = before && r.world == before->world && r.dtype == before->dtype && r.numel == before->numel;
        r.workspace_bytes = alike ? before->workspace_bytes : aligned(mcclx_replay_workspace_bytes(&r));
        total += r.workspace_bytes;
        before = &r;
    }
    at::Tensor ws;
    if (total) {
        ws = dev::empty_bytes(static_cast<int64_t>(total + 256), device);
        char* at = reinterpret_cast<char*>(aligned(reinterpret_cast<uintptr_t>(ws.data_ptr())));
        for (mcclx_replay& r : reps) {
            if (r.workspace_bytes) r.workspace = at;
            at += r.workspace_bytes;
        }
    }
    void* stream = dev::current_stream(device);
    py::gil_scoped_release unlocked;
    // The call waits in any case: the workspace goes back to the allocator.  Tensors and workspace are device
    // memory, so the end of the queue may be seen early (mcclx_queue_wait); not for a list, where that gains nothing.
    const bool early = reps.size() == 1;
    const int rc = mcclx_queue_wait_stream(ctx, stream);
    if (rc != MCCLX_OK) return rc;  // nothing has been issued
    return mcclx_allreduce_replay_wait(ctx, reps.data(), static_cast<uint32_t>(reps.size()), early ? kWaitSpinUs : 0);
}

py::object replay_many(uintptr_t ctx, int device, py::handle groups, int op, int algo, bool wire, int mode, int acc) {
    if (!PyList_Check(groups.ptr()) && !PyTuple_Check(groups.ptr())) return py::none();
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(groups.ptr());
    PyObject** items = PySequence_Fast_ITEMS(groups.ptr());
    const How how{op, algo, wire ? 1 : 0, mode, acc};
    std::vector<mcclx_replay> reps(static_cast<size_t>(n));
    std::vector<void*> ptrs;
    for (Py_ssize_t i = 0; i < n; ++i) {
        if (!read_group(items[i], how, &reps[static_cast<size_t>(i)], ptrs)) return py::none();
        if (i == 0) ptrs.reserve(static_cast<size_t>(n) * static_cast<size_t>(reps[0].world));
    }
    size_t at = 0;
    for (mcclx_replay& r : reps) {
        r.tensors = ptrs.data() + at;
        at += static_cast<size_t>(r.world);
    }
    return py::int_(run(reinterpret_cast<mcclx_ctx*>(ctx), device, reps));
}

// The workspace is taken from torch's allocator, so the call waits for the queue.
py::object replay_one(uintptr_t ctx, int device, py::handle tensors, int op, int algo, bool wire, int mode, int acc) {
    std::vector<mcclx_replay> reps(1);
    std::vector<void*> ptrs;
    if (!read_group(tensors.ptr(), How{op, algo, wire ? 1 : 0, mode, acc}, &reps[0], ptrs)) return py::none();
    reps[0].tensors = ptrs.data();
    return py::int_(run(reinterpret_cast<mcclx_ctx*>(ctx), device, reps));
}

// ProcessGroupMCCL::allreduce for the virtual ranks (ProcessGroupMCCL.cpp:105-186): the wire form and
// the algorithm from the environment, read on every call.  Returns (code, algorithm), or None.
py::object allreduce(uintptr_t ctx, int device, py::handle tensors, int op, int mode) {
    const char* wire_env = std::getenv("MCCL_WIRE_DTYPE");                // :117-120
    const char* below_env = std::getenv("MCCL_TREE_BELOW");               // :138-139
    const int wire = wire_env && std::strcmp(wire_env, "bf16") == 0;
    int64_t below = -1;
    if (below_env) {
        while (*below_env && std::isspace(static_cast<unsigned char>(*below_env))) ++below_env;
        below = std::isdigit(static_cast<unsigned char>(*below_env)) ? static_cast<int64_t>(std::strtoull(below_env, nullptr, 10)) : 0;
    }
    std::vector<mcclx_replay> reps(1);
    std::vector<void*> ptrs;
    mcclx_replay& r = reps[0];
    if (!read_group(tensors.ptr(), How{op, 0, wire, mode, MCCLX_ACC_STEP}, &r, ptrs)) return py::none();
    r.tensors = ptrs.data();
    const bool use_wire = wire && r.dtype == MCCLX_F32;
    r.algo = mcclx_select_algo(std::getenv("MCCL_ALLREDUCE_ALGO"), below, r.numel * (use_wire || r.dtype != MCCLX_F32 ? 2u : 4u),
                               static_cast<int64_t>(r.numel), r.world);   // :134-145
    const int algo = r.algo;
    return py::make_tuple(run(reinterpret_cast<mcclx_ctx*>(ctx), device, reps), algo);
}

}  // namespace

void bind_replays(py::module_& m) {
    m.def("_allreduce", &allreduce);
    m.def("_allreduce_replay", &replay_one);
    m.def("_allreduce_replay_many", &replay_many);
}

}  // namespace mccl
