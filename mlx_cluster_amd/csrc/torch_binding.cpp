// Compiled fast path of the Python surface for the common call: every array a
// torch tensor of the right dtype, contiguous, on the current device, the
// call on torch's current stream.  It does what walks.py does for such calls
// (check the arguments, allocate the outputs and workspace from torch's
// caching allocator, launch through the C ABI, read the status word) without
// the Python layer's per-call cost, which bounds the reference tests' own
// calls (2,000 walks of 5 steps on a Cora-sized graph).  Any other call
// returns None and walks.py takes it.  Errors raise as in walks.py.
//
// Mirrors: random_walk / rejection_sampling of /root/reference/bindings.cpp:12-63.
#include <ATen/hip/HIPContext.h>
#include <hip/hip_runtime.h>
#include <pybind11/pybind11.h>
#include <torch/extension.h>

#include <chrono>
#include <optional>
#include <string>

#include "mlxc.h"

namespace py = pybind11;

namespace {

// Whether t can be passed as is: a contiguous tensor of dtype on device.
bool usable(const at::Tensor& t, at::ScalarType dtype, const at::Device& device) {
    return t.scalar_type() == dtype && t.device() == device && t.is_contiguous();
}

const void* data_or_null(const at::Tensor& t) { return t.numel() ? t.data_ptr() : nullptr; }

void raise_code(int rc, const char* what) {
    const std::string msg = std::string(what) + ": " + mlxc_last_error();
    if (rc == MLXC_ERR_INVALID_ARGUMENT) throw py::value_error(msg);
    throw std::runtime_error(msg);
}

// The calling thread's host words for mlxc_set_status_target: allocated at
// the thread's first validated call (one pinned page) and kept for the rest
// of the process, since freeing them at thread exit could run after the HIP
// runtime has shut down; null if the allocation failed.
int64_t* status_words() {
    thread_local int64_t* words = [] {
        void* p = nullptr;
        if (hipHostMalloc(&p, 3 * sizeof(int64_t),
                          hipHostMallocCoherent | hipHostMallocMapped | hipHostMallocPortable) !=
            hipSuccess) {
            (void)hipGetLastError();
            return static_cast<int64_t*>(nullptr);
        }
        return static_cast<int64_t*>(p);
    }();
    return words;
}

// For a validated call: makes the library publish the call's status word into
// the calling thread's host words (mlxc_set_status_target), and puts the
// target that the thread had before back afterwards.
class StatusTarget {
public:
    explicit StatusTarget(bool check) : before(mlxc_status_target()) {
        int64_t* h = check ? status_words() : nullptr;
        if (!h) return;
        __atomic_store_n(&h[0], int64_t{0}, __ATOMIC_RELAXED);
        if (mlxc_set_status_target(h) == MLXC_OK) words = h;
    }
    ~StatusTarget() {
        if (words || before) mlxc_set_status_target(before);
    }
    int64_t* words = nullptr;

private:
    int64_t* const before;
};

// The status word of the call just enqueued on `stream`.  Its last launch
// stores it into `h` and the host waits for the flag: spinning for up to about
// 200 us (the reference tests' calls take tens), then in hipStreamSynchronize.
// Without the host words, torch's scalar read (a copy ordered on the stream,
// about 13 us more per call).
bool wait_published(hipStream_t stream, const int64_t* h) {
    if (!h) return false;
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
    for (unsigned i = 1;; ++i) {
        if (__atomic_load_n(&h[0], __ATOMIC_ACQUIRE)) return true;
        __builtin_ia32_pause();
        if (i % 64 == 0 && std::chrono::steady_clock::now() > until) break;
    }
    if (hipStreamSynchronize(stream) != hipSuccess)
        throw std::runtime_error(std::string("hipStreamSynchronize: ") +
                                 hipGetErrorString(hipGetLastError()));
    return __atomic_load_n(&h[0], __ATOMIC_ACQUIRE) != 0;
}
// Word k of the call's workspace (0, or 1 after a CSR build).
int64_t read_word(const at::Tensor& work, hipStream_t stream, const int64_t* h, int k) {
    if (wait_published(stream, h)) return __atomic_load_n(&h[1 + k], __ATOMIC_RELAXED);
    return work.select(0, k).item<int64_t>();
}

// Waits for the call and raises ValueError for status bits, as walks.py's
// check=True does.
void check_status(const at::Tensor& work, hipStream_t stream, const int64_t* words,
                  const char* what) {
    const int64_t bits = read_word(work, stream, words, 0);
    if (bits == 0) return;
    std::string msg = std::string(what) + ": ";
    if (bits & MLXC_STATUS_BAD_NODE) msg += "a start or col entry is outside [0, num_nodes)";
    if (bits & MLXC_STATUS_BAD_ROW) {
        if (bits & MLXC_STATUS_BAD_NODE) msg += "; ";
        msg += "rowptr is malformed (an entry outside [0, num_edges] or decreasing)";
    }
    throw py::value_error(msg);
}

py::object outputs(const at::Tensor& n_out, const at::Tensor& e_out, bool return_edges) {
    if (return_edges) return py::make_tuple(n_out, e_out);
    return py::cast(n_out);
}

// random_walk(rowptr, col, start, rand or None, walk_length, seed or None,
// check, return_edges, int32_out) -> walks, (walks, edges) or None.
py::object random_walk(const at::Tensor& rowptr, const at::Tensor& col, const at::Tensor& start,
                       std::optional<at::Tensor> rand, int64_t walk_length,
                       std::optional<uint64_t> seed, bool check, bool return_edges,
                       bool int32_out) {
    if (!rowptr.is_cuda() || rowptr.dim() != 1 || rowptr.numel() < 1 || col.dim() != 1 ||
        start.dim() != 1 || walk_length < 0 || walk_length > INT32_MAX - 1 ||
        rand.has_value() == seed.has_value())
        return py::none();
    const at::Device device = rowptr.device();
    if (device.index() != c10::hip::current_device()) return py::none();
    if (!usable(rowptr, at::kLong, device) || !usable(col, at::kLong, device) ||
        !usable(start, at::kLong, device))
        return py::none();
    const int64_t N = start.numel(), L = walk_length;
    if (rand && (!usable(*rand, at::kFloat, device) || rand->numel() != N * L)) return py::none();
    const int64_t V = rowptr.numel() - 1, E = col.numel();
    const auto dtype = int32_out ? at::kInt : at::kLong;
    const auto opts = at::TensorOptions().dtype(dtype).device(device);
    at::Tensor n_out = at::empty({N, L + 1}, opts);
    at::Tensor e_out = return_edges ? at::empty({N, L}, opts) : at::Tensor();
    const size_t ws = mlxc_random_walk_preferred_bytes(V, E, N, static_cast<int32_t>(L));
    at::Tensor work = at::empty({static_cast<int64_t>((ws + 7) / 8)},
                                at::TensorOptions().dtype(at::kLong).device(device));
    hipStream_t stream = at::hip::getCurrentHIPStream().stream();
    const int out_type = int32_out ? MLXC_OUT_INT32 : MLXC_OUT_INT64;
    const StatusTarget target(check);
    int rc;
    if (rand)
        rc = mlxc_random_walk(
            static_cast<const int64_t*>(data_or_null(rowptr)), V,
            static_cast<const int64_t*>(data_or_null(col)), E,
            static_cast<const int64_t*>(data_or_null(start)), N,
            static_cast<const float*>(data_or_null(*rand)), static_cast<int32_t>(L),
            n_out.numel() ? n_out.data_ptr() : nullptr,
            return_edges && e_out.numel() ? e_out.data_ptr() : nullptr, out_type,
            work.data_ptr(), static_cast<size_t>(work.numel()) * 8, stream);
    else
        rc = mlxc_random_walk_seeded(
            static_cast<const int64_t*>(data_or_null(rowptr)), V,
            static_cast<const int64_t*>(data_or_null(col)), E,
            static_cast<const int64_t*>(data_or_null(start)), N, static_cast<int32_t>(L), *seed,
            0, n_out.numel() ? n_out.data_ptr() : nullptr,
            return_edges && e_out.numel() ? e_out.data_ptr() : nullptr, out_type,
            work.data_ptr(), static_cast<size_t>(work.numel()) * 8, stream);
    if (rc != MLXC_OK) raise_code(rc, "random_walk");
    if (check) check_status(work, stream, target.words, "random_walk");
    return outputs(n_out, e_out, return_edges);
}

// rejection_sampling(rowptr, col, start, walk_length, p, q, seed, rule, rows,
// check, return_edges, int32_out) -> walks, (walks, edges) or None.
py::object rejection_sampling(const at::Tensor& rowptr, const at::Tensor& col,
                              const at::Tensor& start, int64_t walk_length, double p, double q,
                              uint64_t seed, int32_t rule, int32_t rows, bool check,
                              bool return_edges, bool int32_out) {
    if (!rowptr.is_cuda() || rowptr.dim() != 1 || rowptr.numel() < 1 || col.dim() != 1 ||
        start.dim() != 1 || walk_length < 0 || walk_length > INT32_MAX - 1)
        return py::none();
    const at::Device device = rowptr.device();
    if (device.index() != c10::hip::current_device()) return py::none();
    if (!usable(rowptr, at::kLong, device) || !usable(col, at::kLong, device) ||
        !usable(start, at::kLong, device))
        return py::none();
    const int64_t N = start.numel(), L = walk_length;
    const int64_t V = rowptr.numel() - 1, E = col.numel();
    const auto dtype = int32_out ? at::kInt : at::kLong;
    const auto opts = at::TensorOptions().dtype(dtype).device(device);
    at::Tensor n_out = at::empty({N, L + 1}, opts);
    at::Tensor e_out = return_edges ? at::empty({N, L}, opts) : at::Tensor();
    const size_t ws = mlxc_rejection_sampling_preferred_bytes(V, E, N, static_cast<int32_t>(L), p,
                                                              q, rule);
    at::Tensor work = at::empty({static_cast<int64_t>((ws + 7) / 8)},
                                at::TensorOptions().dtype(at::kLong).device(device));
    hipStream_t stream = at::hip::getCurrentHIPStream().stream();
    const StatusTarget target(check);
    const int rc = mlxc_rejection_sampling(
        static_cast<const int64_t*>(data_or_null(rowptr)), V,
        static_cast<const int64_t*>(data_or_null(col)), E,
        static_cast<const int64_t*>(data_or_null(start)), N, static_cast<int32_t>(L), p, q, seed,
        0, rule, rows, n_out.numel() ? n_out.data_ptr() : nullptr,
        return_edges && e_out.numel() ? e_out.data_ptr() : nullptr,
        int32_out ? MLXC_OUT_INT32 : MLXC_OUT_INT64, work.data_ptr(),
        static_cast<size_t>(work.numel()) * 8, stream);
    if (rc != MLXC_OK) raise_code(rc, "rejection_sampling");
    if (check) check_status(work, stream, target.words, "rejection_sampling");
    return outputs(n_out, e_out, return_edges);
}

// to_csr(edge_index, num_nodes, flags) -> (rowptr, col) or None.
py::object to_csr(const at::Tensor& edge_index, int64_t num_nodes, int32_t flags) {
    if (!edge_index.is_cuda() || edge_index.dim() != 2 || edge_index.size(0) != 2 || num_nodes < 0)
        return py::none();
    const at::Device device = edge_index.device();
    if (device.index() != c10::hip::current_device() || !usable(edge_index, at::kLong, device))
        return py::none();
    const int64_t E = edge_index.size(1);
    const size_t ws = mlxc_csr_build_workspace_bytes(num_nodes, E, flags);
    if (ws == 0) return py::none();
    const int64_t* row = E ? edge_index.data_ptr<int64_t>() : nullptr;
    const int64_t* col = E ? row + E : nullptr;
    const auto opts = at::TensorOptions().dtype(at::kLong).device(device);
    at::Tensor rowptr = at::empty({num_nodes + 1}, opts);
    at::Tensor col_out = at::empty({flags & MLXC_CSR_SYMMETRIZE ? 2 * E : E}, opts);
    at::Tensor work = at::empty({static_cast<int64_t>((ws + 7) / 8)}, opts);
    hipStream_t stream = at::hip::getCurrentHIPStream().stream();
    int rc;
    int64_t bits = 0, count = 0;
    {
        // A build takes up to milliseconds: other Python threads (a data
        // loader's) run while this one launches it and waits.
        const py::gil_scoped_release other_threads_run;
        const StatusTarget target(true);
        rc = mlxc_csr_build(row, col, E, num_nodes, flags, rowptr.data_ptr<int64_t>(),
                            col_out.numel() ? col_out.data_ptr<int64_t>() : nullptr,
                            work.data_ptr(), static_cast<size_t>(work.numel()) * 8, stream);
        if (rc == MLXC_OK) {
            bits = read_word(work, stream, target.words, 0);
            count = read_word(work, stream, target.words, 1);
        }
    }
    if (rc != MLXC_OK) raise_code(rc, "to_csr");
    if (bits & MLXC_STATUS_BAD_NODE)
        throw py::value_error("edge_index holds ids outside [0, num_nodes)");
    return py::make_tuple(rowptr, col_out.narrow(0, 0, count));
}

}  // namespace

PYBIND11_MODULE(_mlxc_torch, m) {
    m.doc() = "Compiled fast path of mlx_cluster_amd.random_walk / rejection_sampling / to_csr";
    m.def("random_walk", &random_walk);
    m.def("rejection_sampling", &rejection_sampling);
    m.def("to_csr", &to_csr);
}
