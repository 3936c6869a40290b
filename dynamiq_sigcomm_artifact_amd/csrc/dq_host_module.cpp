// Python module `_host`: the package's own host path in native code.
//
// A codec launch on a small bucket takes 3 us on the GPU, and a call that goes through ctypes -- an argument conversion
// per parameter, a Python function per tensor check -- takes 8 us of host time in front of it.  The functions and objects
// here take the tensors as they are, check them, find torch's current stream and call the C ABI, in well under a
// microsecond besides the launch itself.  What they compute, accept and refuse is what the Python wrappers they stand
// behind document (capi.py, dynamiq_pipeline.py).
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/autograd/python_variable.h>

#include <stdexcept>
#include <string>
#include <vector>

#include "dynamiq_eden.h"

namespace py = pybind11;

namespace {

[[noreturn]] void refuse(const std::string &text) { throw std::runtime_error(text); }

void check(int status)
{
    if (status != DQ_OK) refuse(dq_last_error());
}

// The kernels dereference whatever address they are given: a host pointer, a strided view or a buffer of another GPU is a
// memory fault on the device, not an error code.  Every tensor whose address goes into the library passes through ptr().
struct Args {
    int device = -1;

    const at::Tensor &tensor(PyObject *o)
    {
        if (!THPVariable_Check(o)) refuse(std::string("a tensor argument is required, got ") + Py_TYPE(o)->tp_name);
        const at::Tensor &t = THPVariable_Unpack(o);
        if (!t.is_cuda()) refuse("tensor arguments must live on the GPU (got a " + std::string(c10::DeviceTypeName(t.device().type(), true)) + " tensor)");
        if (!t.is_contiguous()) refuse("tensor arguments must be contiguous");
        const int d = t.device().index();
        if (device < 0)
            device = d;
        else if (device != d)
            refuse("tensor arguments live on different devices");
        return t;
    }
    const at::Tensor &tensor(py::handle h) { return tensor(h.ptr()); }
    void *ptr(py::handle h) { return tensor(h.ptr()).data_ptr(); }
    void *ptr_or_null(py::handle h) { return h.is_none() ? nullptr : ptr(h); }
    const at::Tensor &typed(py::handle h, at::ScalarType dtype, int64_t count, const char *what)
    {
        const at::Tensor &t = tensor(h);
        if (t.scalar_type() != dtype || t.numel() < count) refuse(std::string(what) + ": wrong dtype or too few entries");
        return t;
    }
};

int dtype_code(const at::Tensor &t)
{
    switch (t.scalar_type()) {
    case at::kHalf: return DQ_F16;
    case at::kBFloat16: return DQ_BF16;
    case at::kFloat: return DQ_F32;
    default: refuse(std::string("unsupported element dtype ") + c10::toString(t.scalar_type()));
    }
}

// None: torch's current stream; a raw handle; a torch stream
dq_stream_t stream_of(py::handle s)
{
    if (s.is_none()) return c10::hip::getCurrentHIPStream().stream();
    if (PyLong_Check(s.ptr())) return reinterpret_cast<dq_stream_t>(PyLong_AsUnsignedLongLong(s.ptr()));
    return reinterpret_cast<dq_stream_t>(static_cast<uintptr_t>(py::cast<uint64_t>(s.attr("cuda_stream"))));
}

// u of the width rule: a number, or a float64 device tensor
struct Offset {
    double value = 0.0;
    const double *dev = nullptr;
    Offset(Args &a, py::handle u)
    {
        if (THPVariable_Check(u.ptr())) {
            const at::Tensor &t = a.tensor(u);
            if (t.scalar_type() != at::kDouble || t.numel() < 1) refuse("a tensor u must be float64 on the device of the vectors");
            dev = t.data_ptr<double>();
        } else {
            value = py::cast<double>(u);
        }
    }
};

uint32_t *hist_of(Args &a, py::handle h, int64_t *entries)
{
    *entries = 0;
    if (h.is_none()) return nullptr;
    const at::Tensor &t = a.tensor(h);
    if (t.scalar_type() != at::kInt) refuse("hist must be int32");
    *entries = t.numel();
    return reinterpret_cast<uint32_t *>(t.data_ptr<int32_t>());
}

// ---- buckets of one rank ----------------------------------------------------------------------------------

// The state of a SinglePassBuckets object.  Its buckets share scratch and run on the caller's stream; a caller that comes
// back on another stream is ordered behind the one before.
struct Buckets {
    int strategy, device;
    uint64_t seed, pending = 0; // training steps begun since the last launch
    py::object step_dev, u_dev, hist, stats, counts;
    uint64_t *step_ptr = nullptr;
    const double *u_ptr = nullptr;
    uint32_t *hist_ptr = nullptr;
    int64_t hist_ints = 0;
    char *stats_ptr = nullptr;
    int64_t stats_room = 0, counts_room = 0;
    int32_t *counts_ptr = nullptr;
    hipStream_t last = nullptr;
    bool used = false;

    Buckets(int strategy_, uint64_t seed_, py::object step, py::object u, py::object h) : strategy(strategy_), seed(seed_)
    {
        Args a;
        step_ptr = reinterpret_cast<uint64_t *>(a.typed(step, at::kLong, 1, "step counter").data_ptr());
        u_ptr = a.typed(u, at::kDouble, 1, "u").data_ptr<double>();
        hist_ptr = hist_of(a, h, &hist_ints);
        device = a.device;
        step_dev = step;
        u_dev = u;
        hist = h;
    }
    void scratch(py::object stats_, py::object counts_)
    {
        Args a;
        const at::Tensor &s = a.typed(stats_, at::kBFloat16, 0, "stats"), &c = a.typed(counts_, at::kInt, 0, "counts");
        stats_ptr = static_cast<char *>(s.data_ptr());
        counts_ptr = c.data_ptr<int32_t>();
        stats_room = s.numel() / 2;
        counts_room = c.numel() / 4;
        stats = stats_;
        counts = counts_;
    }
    void follow(hipStream_t s)
    {
        if (used && s != last) check(dq_stream_order_after(s, last, device));
        last = s;
        used = true;
    }
    void join()
    {
        const hipStream_t s = c10::hip::getCurrentHIPStream(device).stream();
        if (used && s != last) follow(s);
    }
};

// buckets that are enqueued together: addresses, not tensors (whoever calls launch() keeps those alive)
struct Batch {
    std::vector<dq_roundtrip_t> desc;
    int dtype = DQ_BF16;

    // rows: where each bucket's counts go
    Batch(Buckets &b, py::sequence pairs, const std::vector<uint64_t> &steps, const std::vector<int64_t> &rows)
    {
        const size_t count = py::len(pairs);
        if (count == 0 || steps.size() != count || rows.size() != count) refuse("buckets and scratch do not match");
        int64_t at = 0;
        for (size_t k = 0; k < count; k++) {
            const py::tuple p = py::cast<py::tuple>(pairs[k]);
            if (p.size() != 2) refuse("a bucket is a pair (x, out)");
            Args a;
            a.device = b.device;
            const at::Tensor &x = a.tensor(p[0]), &out = a.tensor(p[1]);
            const int code = dtype_code(x);
            if (k == 0) dtype = code;
            if (code != dtype || out.scalar_type() != x.scalar_type() || out.numel() < x.numel())
                refuse("the buckets of a list and their outputs must have one dtype, and every output its bucket's size");
            dq_roundtrip_t d;
            d.src = x.data_ptr();
            d.out = out.data_ptr();
            d.n = x.numel();
            d.stats = b.stats_ptr + 4 * at;
            if (rows[k] < 0 || rows[k] >= b.counts_room) refuse("buckets and scratch do not match");
            d.counts = b.counts_ptr + 4 * rows[k];
            d.step = steps[k];
            at += (d.n + 255) / 256;
            desc.push_back(d);
        }
        if (at > b.stats_room) refuse("buckets and scratch do not match");
    }
    // the same buffers in the same order?
    bool matches(py::handle pairs) const
    {
        PyObject *list = pairs.ptr();
        if (!PyList_CheckExact(list) || PyList_GET_SIZE(list) != (Py_ssize_t)desc.size()) return false;
        for (size_t k = 0; k < desc.size(); k++) {
            PyObject *p = PyList_GET_ITEM(list, k);
            if (!PyTuple_CheckExact(p) || PyTuple_GET_SIZE(p) != 2) return false;
            PyObject *xo = PyTuple_GET_ITEM(p, 0), *oo = PyTuple_GET_ITEM(p, 1);
            if (!THPVariable_Check(xo) || !THPVariable_Check(oo)) return false;
            const at::Tensor &x = THPVariable_Unpack(xo), &out = THPVariable_Unpack(oo);
            if (x.data_ptr() != desc[k].src || out.data_ptr() != desc[k].out || x.numel() != desc[k].n || out.numel() < x.numel() ||
                !x.is_contiguous() || !out.is_contiguous() || out.scalar_type() != x.scalar_type() || dtype_code(x) != dtype)
                return false;
        }
        return true;
    }
    void launch(Buckets &b)
    {
        const hipStream_t s = c10::hip::getCurrentHIPStream(b.device).stream();
        b.follow(s);
        const uint64_t more = b.pending;
        int rc;
        {
            py::gil_scoped_release nogil;
            rc = dq_bucket_roundtrip(desc.data(), (int)desc.size(), dtype, b.strategy, 1, 0.0, b.u_ptr, b.seed, b.step_ptr, more, b.hist_ptr,
                                     b.hist_ints, b.device, s);
        }
        check(rc);
        b.pending = 0;
    }
};

// one bucket of one rank outside a SinglePassBuckets object
void roundtrip(py::handle x, py::handle out, int64_t n, py::handle stats, py::handle counts, py::handle u, py::handle hist,
               uint64_t seed, int strategy, py::handle stream)
{
    Args a;
    const at::Tensor &src = a.tensor(x);
    const at::Tensor &dst = a.tensor(out);
    if (src.numel() < n || dst.numel() < n || dst.scalar_type() != src.scalar_type()) refuse("the output must have the vector's dtype and size");
    dq_roundtrip_t d;
    d.src = src.data_ptr();
    d.out = dst.data_ptr();
    d.n = n;
    d.stats = a.typed(stats, at::kBFloat16, 2 * ((n + 255) / 256), "stats").data_ptr();
    d.counts = a.typed(counts, at::kInt, 4, "counts").data_ptr<int32_t>();
    d.step = 0;
    const Offset o(a, u);
    int64_t hist_ints;
    uint32_t *h = hist_of(a, hist, &hist_ints);
    const dq_stream_t s = stream_of(stream);
    const int code = dtype_code(src);
    int rc;
    {
        py::gil_scoped_release nogil;
        rc = dq_bucket_roundtrip(&d, 1, code, strategy, 1, o.value, o.dev, seed, nullptr, 0, h, hist_ints, a.device, s);
    }
    check(rc);
}

// ---- ranks that share the GPU's memory ---------------------------------------------------------------------

struct Ranks {
    std::vector<const void *> src;
    std::vector<void *> out;
    dq_ranks_t r;

    Ranks(Args &a, py::sequence vecs, py::sequence outs, int64_t n, py::handle total, py::handle mean, py::handle order,
          py::handle work, int strategy)
    {
        memset(&r, 0, sizeof(r));
        const size_t world = py::len(vecs);
        if (world == 0 || py::len(outs) != world) refuse("one vector and one output per rank");
        at::ScalarType dtype = at::kBFloat16;
        for (size_t k = 0; k < world; k++) {
            const py::object x = vecs[k], o = outs[k];
            const at::Tensor &s = a.tensor(x), &d = a.tensor(o);
            if (k == 0) {
                dtype = s.scalar_type();
                r.dtype = dtype_code(s);
            }
            if (s.scalar_type() != dtype || d.scalar_type() != dtype || s.numel() < n || d.numel() < n)
                refuse("the ranks' vectors and outputs must have one dtype and size");
            src.push_back(s.data_ptr());
            out.push_back(d.data_ptr());
        }
        const int64_t nsc = (n + 255) / 256;
        r.src = src.data();
        r.out = out.data();
        r.n = n;
        r.world = (int)world;
        r.strategy = strategy;
        r.total = a.typed(total, at::kBFloat16, 2 * nsc, "total").data_ptr();
        r.mean = a.typed(mean, at::kFloat, (int64_t)world * nsc, "mean").data_ptr<float>();
        r.order = a.typed(order, at::kInt, 3 * nsc, "order").data_ptr<int32_t>();
        const at::Tensor &w = a.typed(work, at::kInt, 4, "work");
        r.work = w.data_ptr<int32_t>();
        r.work_ints = w.numel();
    }
    void enqueue(int stages, int device, dq_stream_t s)
    {
        int rc;
        {
            py::gil_scoped_release nogil;
            rc = dq_ranks_allreduce(&r, stages, device, s);
        }
        check(rc);
    }
};

void ranks_dynamic(py::sequence vecs, py::sequence outs, int64_t n, py::handle total, py::handle mean, py::handle order,
                   py::handle work, py::handle u, py::handle hist, uint64_t seed, int strategy, py::handle stream)
{
    Args a;
    Ranks k(a, vecs, outs, n, total, mean, order, work, strategy);
    const Offset o(a, u);
    k.r.u = o.value;
    k.r.u_dev = o.dev;
    k.r.hist = hist_of(a, hist, &k.r.hist_ints);
    k.r.seed = seed;
    k.enqueue(DQ_RANKS_STATS | DQ_RANKS_PLAN | DQ_RANKS_RING, a.device, stream_of(stream));
}

} // namespace

PYBIND11_MODULE(_host, m)
{
    m.doc() = "native host path of dynamiq_sigcomm_artifact_amd";
    py::class_<Buckets>(m, "Buckets")
        .def(py::init<int, uint64_t, py::object, py::object, py::object>())
        .def("scratch", &Buckets::scratch)
        .def("join", &Buckets::join)
        .def("begin_step", [](Buckets &b) { b.pending++; });
    py::class_<Batch>(m, "Batch")
        .def(py::init([](Buckets &b, py::sequence pairs, py::sequence steps, py::sequence rows) {
            std::vector<uint64_t> s;
            std::vector<int64_t> at;
            for (size_t k = 0; k < py::len(steps); k++) s.push_back(py::cast<uint64_t>(steps[k]));
            for (size_t k = 0; k < py::len(rows); k++) at.push_back(py::cast<int64_t>(rows[k]));
            return new Batch(b, pairs, s, at);
        }))
        .def("matches", &Batch::matches)
        .def("launch", &Batch::launch);
    m.def("roundtrip", &roundtrip);
    m.def("ranks_dynamic", &ranks_dynamic);
}
