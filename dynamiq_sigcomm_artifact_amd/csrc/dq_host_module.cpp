// Python module `_host`: the package's own host path in native code.
//
// A codec launch on a small bucket takes 3 us on the GPU, and a call that goes through ctypes -- an argument conversion
// per parameter, a Python function per tensor check -- takes 8 us of host time in front of it.  The functions and objects
// here take the tensors as they are, check them, find torch's current stream and call the C ABI, in well under a
// microsecond besides the launch itself.  What they compute, accept and refuse is what the Python wrappers they stand
// behind document (capi.py, dynamiq_pipeline.py).
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Generator.h>
#include <torch/csrc/autograd/python_variable.h>

#include <string.h>

#include <algorithm>
#include <mutex>
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

// modulo 2^64: seeds, steps and handles, whatever int() takes; `whole`: whole numbers only
uint64_t word(PyObject *o, bool whole = false)
{
    const py::object made = py::reinterpret_steal<py::object>(whole ? PyNumber_Index(o) : PyNumber_Long(o));
    if (!made) throw py::error_already_set();
    return PyLong_AsUnsignedLongLongMask(made.ptr());
}

// None: torch's current stream, of that device if one is named; a raw handle; a torch stream
dq_stream_t stream_of(py::handle s, int device = -1)
{
    if (s.is_none()) return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    const py::object raw = PyLong_Check(s.ptr()) || !py::hasattr(s, "cuda_stream") ? py::reinterpret_borrow<py::object>(s) : s.attr("cuda_stream");
    return reinterpret_cast<dq_stream_t>(static_cast<uintptr_t>(word(raw.ptr())));
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

// memory that a tensor's first n elements take
struct Span {
    uintptr_t begin, end;
    Span(const at::Tensor &t, int64_t n) : begin(reinterpret_cast<uintptr_t>(t.data_ptr())), end(begin + (uintptr_t)(n * t.element_size())) {}
    bool meets(const Span &o) const { return begin < o.end && o.begin < end; }
    // The kernels of one pass read a superchunk and write it where it was, or elsewhere: an output that lies across a source at
    // another address would be written while other waves still read there.
    bool across(const Span &o) const { return begin != o.begin && meets(o); }
};

// ---- buckets of one rank ----------------------------------------------------------------------------------

// The state of a SinglePassBuckets object.  Its buckets share scratch and run on the caller's stream; a caller that comes
// back on another stream is ordered behind the one before.  The object lets one thread in at a time: launch() gives up the
// interpreter's lock between choosing the order and the steps and the launches that these belong to.
//
// A launch takes the steps begun since the last one along and advances the counter in device memory itself.  That holds for
// eager launches only: a recorded launch is replayed without this object taking part.  So a step begun while recording is a
// node of the graph, steps begun before the recording that no launch has taken along yet go into `base`, a constant of every
// later launch, and once a graph exists a step is begun on the device at once, where the next replay finds it.
struct Buckets {
    int strategy, device;
    uint64_t seed, pending = 0; // training steps begun since the last launch
    uint64_t base = 0;          // steps that the counter in device memory never gets
    bool recorded = false;      // a graph with launches of this object may exist
    py::object step_dev, u_dev, hist, counts, stats, spare;
    uint64_t *step_ptr = nullptr;
    const double *u_ptr = nullptr;
    uint32_t *hist_ptr = nullptr;
    int64_t hist_ints = 0;
    int32_t *counts_ptr = nullptr, *spare_ptr = nullptr; // rows of four: of the slots, and of buckets beside them
    char *stats_ptr = nullptr;
    int64_t counts_rows = 0, stats_room = 0, spare_rows = 0;
    hipStream_t last = nullptr; // of the last eager launch, at first of the tensors' making
    bool used = false;
    std::vector<hipStream_t> kept_for; // streams beside the one that the tensors were made on
    hipStream_t last_recorded = nullptr; // of the last launch of the recording with this id
    unsigned long long recording = 0;

    Buckets(int strategy_, uint64_t seed_, py::object step, py::object u, py::object h, py::object counts_)
        : strategy(strategy_), seed(seed_)
    {
        Args a;
        step_ptr = reinterpret_cast<uint64_t *>(a.typed(step, at::kLong, 1, "step counter").data_ptr());
        u_ptr = a.typed(u, at::kDouble, 1, "u").data_ptr<double>();
        hist_ptr = hist_of(a, h, &hist_ints);
        const at::Tensor &c = a.typed(counts_, at::kInt, 4, "counts");
        counts_ptr = c.data_ptr<int32_t>();
        counts_rows = c.numel() / 4;
        device = a.device;
        step_dev = step;
        u_dev = u;
        hist = h;
        counts = counts_;
        follow(c10::hip::getCurrentHIPStream(device).stream()); // on which the caller has filled them
    }
    // scratch that grows.  A recorded launch has the addresses of its day: whoever replaces the tensors keeps the old ones.
    void scratch(py::object stats_, py::object spare_)
    {
        Args a;
        const at::Tensor &s = a.typed(stats_, at::kBFloat16, 0, "stats"), &c = a.typed(spare_, at::kInt, 0, "spare counts");
        stats_ptr = static_cast<char *>(s.data_ptr());
        spare_ptr = c.data_ptr<int32_t>();
        stats_room = s.numel() / 2;
        spare_rows = c.numel() / 4;
        stats = stats_;
        spare = spare_;
        kept_for.clear();
    }
    // is s recording a graph, and which?
    static bool capturing(hipStream_t s, unsigned long long *id)
    {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (hipStreamGetCaptureInfo(s, &status, id) != hipSuccess) {
            (void)hipGetLastError(); // (of the null stream while another one records)
            return false;
        }
        return status == hipStreamCaptureStatusActive;
    }
    // the memory may not go to another tensor before s, torch's current stream, is done with it
    void keep_for(hipStream_t s)
    {
        if (std::find(kept_for.begin(), kept_for.end(), s) != kept_for.end()) return;
        const py::object stream = py::module_::import("torch.cuda").attr("current_stream")(device);
        for (const py::object *o : {&step_dev, &u_dev, &hist, &counts, &stats, &spare})
            if (*o && !o->is_none()) o->attr("record_stream")(stream);
        kept_for.push_back(s);
    }
    // orders s behind what was enqueued so far; true while s is recording.  (A recording cannot wait for eager work: whoever
    // records has waited for it, as torch.cuda.graph does.)
    bool follow(hipStream_t s)
    {
        unsigned long long id = 0;
        if (capturing(s, &id)) {
            if (recording == id && s != last_recorded) check(dq_stream_order_after(s, last_recorded, device));
            recording = id;
            last_recorded = s;
            recorded = true;
            base += pending;
            pending = 0;
            return true;
        }
        if (used && s != last) {
            check(dq_stream_order_after(s, last, device));
            keep_for(s);
        }
        last = s;
        used = true;
        return false;
    }
    // the next launch is ordered behind s too: a replay on s right after this call is in order with the launches around it
    void join()
    {
        const hipStream_t s = c10::hip::getCurrentHIPStream(device).stream();
        unsigned long long id = 0;
        const bool now = capturing(s, &id);
        if (now ? recording == id && s != last_recorded : used && s != last) follow(s);
    }
    // would join() have to wait?
    bool behind() const { return used && c10::hip::getCurrentHIPStream(device).stream() != last; }
    // the counter in device memory takes the steps that wait for a launch
    void settle()
    {
        if (pending == 0) return;
        if (!follow(c10::hip::getCurrentHIPStream(device).stream())) { // (a recording has put them into `base`)
            at::Tensor counter = THPVariable_Unpack(step_dev.ptr());
            counter.add_((int64_t)pending);
            pending = 0;
        }
    }
    void begin_step()
    {
        const hipStream_t s = c10::hip::getCurrentHIPStream(device).stream();
        unsigned long long id = 0;
        if (!recorded && !capturing(s, &id)) {
            pending++;
            return;
        }
        follow(s);
        at::Tensor counter = THPVariable_Unpack(step_dev.ptr());
        counter.add_(1);
    }
};

// buckets that are enqueued with one call: addresses, not tensors (whoever calls launch() keeps those alive).  A run of
// buckets of one element type that leave one another's memory alone shares launches; the runs follow one another in the
// list's order, so a bucket may read what an earlier one of the list has written.
struct Batch {
    struct Run {
        int dtype, count;
    };
    // does bucket b write what a reads or writes, or read what a writes?
    static bool clash(const Span &a_src, const Span &a_out, const Span &b_src, const Span &b_out)
    {
        return b_out.meets(a_src) || b_out.meets(a_out) || b_src.meets(a_out);
    }
    // do any two of the spans meet, those of one bucket aside?  (Sorted: each against the one that reaches furthest so far.)
    static bool any_meet(std::vector<std::pair<Span, size_t>> spans)
    {
        std::sort(spans.begin(), spans.end(), [](const auto &a, const auto &b) { return a.first.begin < b.first.begin; });
        for (size_t k = 1, far = 0; k < spans.size(); k++) {
            if (spans[k].first.meets(spans[far].first) && spans[k].second != spans[far].second) return true;
            if (spans[k].first.end > spans[far].first.end) far = k;
        }
        return false;
    }
    std::vector<dq_roundtrip_t> desc;
    std::vector<Run> runs;

    // rows: where each bucket's counts go, those of the slots first, then the spare ones
    Batch(Buckets &b, py::sequence pairs, const std::vector<uint64_t> &steps, const std::vector<int64_t> &rows)
    {
        const size_t count = py::len(pairs);
        if (count == 0 || steps.size() != count || rows.size() != count) refuse("buckets and scratch do not match");
        int64_t at = 0;
        std::vector<int> codes;
        std::vector<std::pair<Span, size_t>> spans; // of source and output, one after the other
        for (size_t k = 0; k < count; k++) {
            const py::tuple p = py::cast<py::tuple>(pairs[k]);
            if (p.size() != 2) refuse("a bucket is a pair (x, out)");
            Args a;
            a.device = b.device;
            const at::Tensor &x = a.tensor(p[0]), &out = a.tensor(p[1]);
            const int code = dtype_code(x);
            if (out.scalar_type() != x.scalar_type() || out.numel() < x.numel())
                refuse("an output must have its bucket's dtype and size");
            dq_roundtrip_t d;
            d.src = x.data_ptr();
            d.out = out.data_ptr();
            d.n = x.numel();
            d.stats = b.stats_ptr + 4 * at;
            const int64_t spare = rows[k] - b.counts_rows;
            if (rows[k] < 0 || spare >= b.spare_rows) refuse("buckets and scratch do not match");
            d.counts = spare < 0 ? b.counts_ptr + 4 * rows[k] : b.spare_ptr + 4 * spare;
            d.step = steps[k];
            at += (d.n + 255) / 256;
            desc.push_back(d);
            codes.push_back(code);
            spans.emplace_back(Span(x, d.n), k);
            spans.emplace_back(Span(out, d.n), k);
            if (spans[2 * k + 1].first.across(spans[2 * k].first)) refuse("an output lies across its bucket at another address");
        }
        const bool meet = any_meet(spans);
        for (size_t k = 0; k < count; k++) {
            bool joins = !runs.empty() && runs.back().dtype == codes[k];
            for (size_t i = joins && meet ? k - runs.back().count : k; joins && i < k; i++)
                joins = !clash(spans[2 * i].first, spans[2 * i + 1].first, spans[2 * k].first, spans[2 * k + 1].first);
            if (joins)
                runs.back().count++;
            else
                runs.push_back(Run{codes[k], 1});
        }
        if (at > b.stats_room) refuse("buckets and scratch do not match");
    }
    // the same buffers in the same order?
    bool matches(py::handle pairs) const
    {
        PyObject *list = pairs.ptr();
        if (!PyList_CheckExact(list) || PyList_GET_SIZE(list) != (Py_ssize_t)desc.size()) return false;
        size_t run = 0;
        int left = runs[0].count;
        for (size_t k = 0; k < desc.size(); k++, left--) {
            if (left == 0) left = runs[++run].count;
            PyObject *p = PyList_GET_ITEM(list, k);
            if (!PyTuple_CheckExact(p) || PyTuple_GET_SIZE(p) != 2) return false;
            PyObject *xo = PyTuple_GET_ITEM(p, 0), *oo = PyTuple_GET_ITEM(p, 1);
            if (!THPVariable_Check(xo) || !THPVariable_Check(oo)) return false;
            const at::Tensor &x = THPVariable_Unpack(xo), &out = THPVariable_Unpack(oo);
            if (x.data_ptr() != desc[k].src || out.data_ptr() != desc[k].out || x.numel() != desc[k].n || out.numel() < x.numel() ||
                !x.is_contiguous() || !out.is_contiguous() || out.scalar_type() != x.scalar_type() || dtype_code(x) != runs[run].dtype)
                return false;
        }
        return true;
    }
    void launch(Buckets &b)
    {
        const hipStream_t s = c10::hip::getCurrentHIPStream(b.device).stream();
        b.follow(s);
        const dq_roundtrip_t *buckets = desc.data();
        std::vector<dq_roundtrip_t> moved;
        if (b.base) {
            moved = desc;
            for (dq_roundtrip_t &d : moved) d.step += b.base;
            buckets = moved.data();
        }
        for (const Run &r : runs) {
            const uint64_t more = b.pending; // (of the first run: it advances the counter)
            int rc;
            {
                py::gil_scoped_release nogil;
                rc = dq_bucket_roundtrip(buckets, r.count, r.dtype, b.strategy, 1, 0.0, b.u_ptr, b.seed, b.step_ptr, more, b.hist_ptr,
                                         b.hist_ints, b.device, s);
            }
            check(rc);
            b.pending -= more;
            buckets += r.count;
        }
    }
};

// one bucket of one rank outside a SinglePassBuckets object; false: the output lies across the vector, nothing done
bool roundtrip(py::handle x, py::handle out, int64_t n, py::handle stats, py::handle counts, py::handle u, py::handle hist,
               uint64_t seed, int strategy, py::handle stream)
{
    Args a;
    const at::Tensor &src = a.tensor(x);
    const at::Tensor &dst = a.tensor(out);
    if (src.numel() < n || dst.numel() < n || dst.scalar_type() != src.scalar_type()) refuse("the output must have the vector's dtype and size");
    if (Span(dst, n).across(Span(src, n))) return false;
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
    const dq_stream_t s = stream_of(stream, a.device);
    const int code = dtype_code(src);
    int rc;
    {
        py::gil_scoped_release nogil;
        rc = dq_bucket_roundtrip(&d, 1, code, strategy, 1, o.value, o.dev, seed, nullptr, 0, h, hist_ints, a.device, s);
    }
    check(rc);
    return true;
}

// ---- ranks that share the GPU's memory ---------------------------------------------------------------------

struct Ranks {
    std::vector<const void *> src;
    std::vector<void *> out;
    bool across = false; // an output lies across a vector at another address
    dq_ranks_t r;

    Ranks(Args &a, py::sequence vecs, py::sequence outs, int64_t n, int strategy)
    {
        memset(&r, 0, sizeof(r));
        const size_t world = py::len(vecs);
        if (world == 0 || py::len(outs) != world) refuse("one vector and one output per rank");
        at::ScalarType dtype = at::kBFloat16;
        std::vector<Span> reads, writes;
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
            reads.emplace_back(s, n);
            writes.emplace_back(d, n);
        }
        for (const Span &w : writes)
            for (const Span &x : reads) across = across || w.across(x);
        r.src = src.data();
        r.out = out.data();
        r.n = n;
        r.world = (int)world;
        r.strategy = strategy;
    }
    Ranks(Args &a, py::sequence vecs, py::sequence outs, int64_t n, py::handle total, py::handle mean, py::handle order,
          py::handle work, int strategy)
        : Ranks(a, vecs, outs, n, strategy)
    {
        const int64_t nsc = (n + 255) / 256;
        r.total = a.typed(total, at::kBFloat16, 2 * nsc, "total").data_ptr();
        r.mean = a.typed(mean, at::kFloat, (int64_t)r.world * nsc, "mean").data_ptr<float>();
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

// false: an output lies across a vector, nothing done
bool ranks_dynamic(py::sequence vecs, py::sequence outs, int64_t n, py::handle total, py::handle mean, py::handle order,
                   py::handle work, py::handle u, py::handle hist, uint64_t seed, int strategy, py::handle stream)
{
    Args a;
    Ranks k(a, vecs, outs, n, total, mean, order, work, strategy);
    if (k.across) return false;
    const Offset o(a, u);
    k.r.u = o.value;
    k.r.u_dev = o.dev;
    k.r.hist = hist_of(a, hist, &k.r.hist_ints);
    k.r.seed = seed;
    k.enqueue(DQ_RANKS_STATS | DQ_RANKS_PLAN | DQ_RANKS_RING | DQ_RANKS_NO_LISTS, a.device, stream_of(stream, a.device));
    return true;
}

// ---- compressor objects ------------------------------------------------------------------------------------

void need(bool ok, const char *text)
{
    if (!ok) refuse(text);
}

// The calls of a compressor object (compressors.py): element counts, the rows of the random pool and their LCG, the
// checks and texts of the module's scaling_* functions, torch's current stream, the launch.
struct Codec {
    int nbits, chunk, strategy;
    bool extended; // float32 buffers and 3/5/6/7-bit codes
    uint32_t rand_seed;
    bool philox = false;
    uint64_t philox_seed = 0, philox_step = 0;
    py::object base;  // the pool as drawn or loaded, [rows, chunk]
    py::dict pools;   // dtype -> the pool in that dtype

    Codec(int nbits_, int chunk_, int strategy_, bool extended_, uint32_t seed, py::object base_, py::dict pools_)
        : nbits(nbits_), chunk(chunk_), strategy(strategy_), extended(extended_), rand_seed(seed), base(base_), pools(pools_)
    {
    }
    uint32_t next_rand()
    {
        rand_seed = rand_seed * 671431u + 1000000007u; // utils_aggregation.py:391-393
        return rand_seed;
    }
    const at::Tensor &pool(at::ScalarType dtype)
    {
        PyObject *key = reinterpret_cast<PyObject *>(torch::getTHPDtype(dtype));
        PyObject *have = PyDict_GetItem(pools.ptr(), key);
        if (!have) {
            if (!THPVariable_Check(base.ptr())) refuse("this compressor has no random pool");
            const py::object made = base.attr("to")(py::reinterpret_borrow<py::object>(key));
            PyDict_SetItem(pools.ptr(), key, made.ptr());
            have = made.ptr(); // the dictionary holds it
        }
        return THPVariable_Unpack(have);
    }
    // first of n / chunk consecutive rows, where the LCG points (utils_aggregation.py:409-420).  The pool is an attribute that
    // a caller may replace: what the kernels read is checked on every call.
    int64_t first_row(const at::Tensor &p, int64_t n, at::ScalarType dtype)
    {
        need(chunk > 0, "chunk_size must be positive");
        need(p.scalar_type() == dtype, "rand_pool dtype must match input dtype");
        need(p.dim() >= 2, "rand_pool must have rows");
        need(n % chunk || n / chunk * row_width(p) >= n, "rand_pool is too small"); // (a ragged n is refused further on)
        const int64_t choices = p.size(0) - n / chunk - 1;
        need(choices > 0, "randomized_vec_pool is too small for scaling quantization");
        return (int64_t)next_rand() % choices;
    }
    static int64_t row_width(const at::Tensor &p) { return p.size(0) ? p.numel() / p.size(0) : 0; }
    const void *random_rows(const at::Tensor &like, int64_t n)
    {
        const at::Tensor &p = pool(like.scalar_type());
        need(p.is_cuda(), "rand_pool must be a CUDA tensor");
        need(p.is_contiguous(), "rand_pool must be contiguous");
        need(p.device() == like.device(), "tensor arguments live on different devices");
        const int64_t first = first_row(p, n, like.scalar_type());
        return static_cast<const char *>(p.data_ptr()) + first * row_width(p) * (int64_t)p.element_size();
    }
    void check_common(int64_t n) const
    {
        need(n > 0, "n must be positive");
        if (!extended) need(nbits == 2 || nbits == 4 || nbits == 8, "nbits must be one of {2, 4, 8}");
        const int rc = dq_scaling_check_common(n, nbits, chunk, strategy, 0);
        if (rc) refuse(dq_last_error());
    }
    bool data_dtype(const at::Tensor &t) const
    {
        const at::ScalarType d = t.scalar_type();
        return d == at::kBFloat16 || d == at::kHalf || (d == at::kFloat && (extended || philox));
    }
    static bool empty(py::handle h) { return THPVariable_Check(h.ptr()) && THPVariable_Unpack(h.ptr()).numel() == 0; }
    static const at::Tensor &cuda(py::handle h, const char *text)
    {
        if (!THPVariable_Check(h.ptr())) refuse(std::string("a tensor argument is required, got ") + Py_TYPE(h.ptr())->tp_name);
        const at::Tensor &t = THPVariable_Unpack(h.ptr());
        need(t.is_cuda(), text);
        return t;
    }
    int64_t bytes(int64_t n) const { return dq_scaling_required_bytes(n, nbits, chunk, strategy); }

    void compress(py::handle input, py::handle send)
    {
        if (empty(input)) return; // nothing to do, wherever it lives
        const at::Tensor &src = cuda(input, "input must be a CUDA tensor");
        const int64_t n = src.numel();
        const at::Tensor &dst = cuda(send, "output must be a CUDA tensor");
        need(data_dtype(src), "input must be torch.float16 or torch.bfloat16");
        const void *rnd = philox ? nullptr : random_rows(src, n);
        need(dst.scalar_type() == at::kByte, "output must be torch.uint8");
        need(src.is_contiguous(), "input must be contiguous");
        need(dst.is_contiguous(), "output must be contiguous");
        need(dst.device() == src.device(), "tensor arguments live on different devices");
        check_common(n);
        need(dst.numel() >= bytes(n), "output buffer is too small");
        const void *x = src.data_ptr();
        uint8_t *y = dst.data_ptr<uint8_t>();
        const int code = dtype_code(src), device = src.device().index();
        const dq_stream_t s = c10::hip::getCurrentHIPStream().stream();
        const uint64_t step = philox ? ++philox_step : 0;
        int rc;
        {
            py::gil_scoped_release nogil;
            rc = philox ? dq_scaling_compress_philox(x, y, n, nbits, chunk, code, device, strategy, philox_seed, step, s)
                        : dq_scaling_compress(x, y, rnd, n, nbits, chunk, code, device, strategy, s);
        }
        check(rc);
    }
    void decompress(py::handle recv, py::handle output, bool add)
    {
        if (empty(output)) return;
        const at::Tensor &dst = cuda(output, "output must be a CUDA tensor");
        const int64_t n = dst.numel();
        const at::Tensor &src = cuda(recv, "input must be a CUDA tensor");
        need(src.scalar_type() == at::kByte, "input must be torch.uint8");
        need(data_dtype(dst), "output must be torch.float16 or torch.bfloat16");
        need(src.is_contiguous(), "input must be contiguous");
        need(dst.is_contiguous(), "output must be contiguous");
        need(dst.device() == src.device(), "tensor arguments live on different devices");
        check_common(n);
        need(src.numel() >= bytes(n), "input buffer is too small");
        const uint8_t *x = src.data_ptr<uint8_t>();
        void *y = dst.data_ptr();
        const int code = dtype_code(dst), device = dst.device().index();
        const dq_stream_t s = c10::hip::getCurrentHIPStream().stream();
        int rc;
        {
            py::gil_scoped_release nogil;
            rc = dq_scaling_decompress(x, y, n, nbits, chunk, code, device, strategy, s, add ? 1 : 0);
        }
        check(rc);
    }
    void dec_comp(py::handle recv_, py::handle input, py::handle send_)
    {
        if (empty(input)) return;
        const at::Tensor &inp = cuda(input, "inp must be a CUDA tensor");
        const int64_t n = inp.numel();
        const at::Tensor &recv = cuda(recv_, "recv must be a CUDA tensor"), &send = cuda(send_, "send must be a CUDA tensor");
        need(recv.scalar_type() == at::kByte, "recv must be torch.uint8");
        need(data_dtype(inp), "inp must be torch.float16 or torch.bfloat16");
        const void *rnd = philox ? nullptr : random_rows(inp, n);
        need(send.scalar_type() == at::kByte, "send must be torch.uint8");
        need(recv.is_contiguous(), "recv must be contiguous");
        need(inp.is_contiguous(), "inp must be contiguous");
        need(send.is_contiguous(), "send must be contiguous");
        need(recv.device() == inp.device() && send.device() == inp.device(), "tensor arguments live on different devices");
        check_common(n);
        need(recv.numel() >= bytes(n), "recv buffer is too small");
        need(send.numel() >= bytes(n), "send buffer is too small");
        const uint8_t *r = recv.data_ptr<uint8_t>();
        void *x = inp.data_ptr();
        uint8_t *y = send.data_ptr<uint8_t>();
        const int code = dtype_code(inp), device = inp.device().index();
        const dq_stream_t s = c10::hip::getCurrentHIPStream().stream();
        const uint64_t step = philox ? ++philox_step : 0;
        int rc;
        {
            py::gil_scoped_release nogil;
            rc = philox ? dq_scaling_dec_comp_philox(r, x, y, n, nbits, chunk, code, device, strategy, philox_seed, step, s)
                        : dq_scaling_dec_comp(r, x, y, rnd, n, nbits, chunk, code, device, strategy, s);
        }
        check(rc);
    }
};

// ---- ranks with random pools --------------------------------------------------------------------------------

void enqueue_pooled(Args &a, Ranks &k, at::ScalarType dtype, const py::sequence &codecs, const int64_t (&size)[3], int stages)
{
    const int world = k.r.world;
    std::vector<const void *> pool(3 * world, nullptr);
    std::vector<int32_t> first(3 * world * world, 0);
    for (int g = 0; g < 3; g++) {
        if (size[g] == 0) continue;
        const py::sequence of_width = codecs[g];
        std::vector<Codec *> codec;
        for (int r = 0; r < world; r++) codec.push_back(&py::cast<Codec &>(of_width[r]));
        const int64_t per = (size[g] + world - 1) / world;
        // step by step, as the ring's calls go: ranks may share a compressor
        for (int step = 0; step < world; step++) {
            for (int r = 0; r < world; r++) {
                Codec &c = *codec[r];
                const at::Tensor &p = c.pool(dtype);
                need(p.is_cuda() && p.is_contiguous() && p.device().index() == a.device, "rand_pool must be a contiguous tensor on the vectors' device");
                pool[g * world + r] = p.data_ptr();
                const int chunk = (r - step + world) % world;
                const int64_t rows = std::max<int64_t>(0, std::min(per, size[g] - per * chunk));
                if (rows == 0) continue;
                need(p.dim() == 2 && p.size(1) == 16, "rand_pool must have rows of 16 values");
                const int64_t at = c.first_row(p, rows * 256, dtype);
                need(at <= 0x7fffffff, "randomized_vec_pool has too many rows");
                first[(g * world + r) * world + step] = (int32_t)at;
            }
        }
    }
    k.r.pool = pool.data();
    k.r.first = first.data();
    k.r.sorted_plan = 1;
    k.r.top_count = size[0];
    k.r.bottom_count = size[2];
    k.enqueue(stages, a.device, c10::hip::getCurrentHIPStream().stream());
}

// One bucket of the fixed-proportion (sorted_plan) or dynamic all-reduce with compressor objects: codecs holds one list per
// width (8, 4, 2 bits), group sizes counts.  Walks every codec's LCG as the ring's calls on its non-empty chunks would, in
// the order of the widths, the steps and the ranks: rank r works on chunk (r - step) mod world in that step.  False: an output
// lies across a vector, nothing done.
bool ranks_pooled(py::sequence vecs, py::sequence outs, int64_t n, py::handle total, py::handle mean, py::handle order,
                  py::handle work, py::sequence codecs, py::sequence counts, int stages, int strategy)
{
    Args a;
    Ranks k(a, vecs, outs, n, total, mean, order, work, strategy);
    if (k.across) return false;
    const int64_t size[3] = {py::cast<int64_t>(counts[0]), py::cast<int64_t>(counts[1]), py::cast<int64_t>(counts[2])};
    enqueue_pooled(a, k, THPVariable_Unpack(py::object(vecs[0]).ptr()).scalar_type(), codecs, size, stages);
    return true;
}

// fixed_proportion_allreduce_grouped with compressors of the package: (reduced statistics, row lists), or None where an output lies across
// a vector and nothing was done.  One block of scratch: row lists, means, plan.
py::object ranks_fixed(py::sequence vecs, py::sequence outs, int64_t n, py::sequence codecs, int64_t top, int64_t middle, int64_t bottom,
                       int strategy)
{
    Args a;
    Ranks k(a, vecs, outs, n, strategy);
    if (k.across) return py::none();
    const int64_t nsc = (n + 255) / 256, world = k.r.world, plan = dq_group_plan_sorted_work_ints(nsc);
    const at::Tensor total = at::empty({nsc, 2}, at::TensorOptions().dtype(at::kBFloat16).device(at::kCUDA, (c10::DeviceIndex)a.device));
    const at::Tensor ints = at::empty({3 * nsc + world * nsc + plan}, at::TensorOptions().dtype(at::kInt).device(at::kCUDA, (c10::DeviceIndex)a.device));
    k.r.total = total.data_ptr();
    k.r.order = ints.data_ptr<int32_t>();
    k.r.mean = reinterpret_cast<float *>(k.r.order + 3 * nsc);
    k.r.work = k.r.order + 3 * nsc + world * nsc;
    k.r.work_ints = plan;
    const int64_t size[3] = {top, middle, bottom};
    enqueue_pooled(a, k, THPVariable_Unpack(py::object(vecs[0]).ptr()).scalar_type(), codecs, size, DQ_RANKS_STATS | DQ_RANKS_PLAN | DQ_RANKS_RING);
    return py::make_tuple(py::reinterpret_steal<py::object>(THPVariable_Wrap(total)),
                          py::reinterpret_steal<py::object>(THPVariable_Wrap(ints.narrow(0, 0, 3 * nsc))));
}

// ---- EDEN and THC (eden.py, thc.py) --------------------------------------------------------------------------

at::Tensor empty_on(int device, int64_t n, at::ScalarType dtype)
{
    return at::empty({n}, at::TensorOptions().dtype(dtype).device(at::kCUDA, (c10::DeviceIndex)device));
}

// Eden.compress: slices as (start, elements, padded size, rotations); returns one (packed, scale) per slice
py::list eden_compress(py::handle vec, py::handle boundaries, py::handle centroids, int nbits, py::handle seed, py::sequence slices)
{
    Args a;
    const at::Tensor &v = a.tensor(vec);
    const int64_t levels = (int64_t)1 << nbits;
    const float *b = a.typed(boundaries, at::kFloat, levels - 1, "boundaries").data_ptr<float>();
    const float *c = a.typed(centroids, at::kFloat, levels, "centroids").data_ptr<float>();
    const int elem = (int)v.element_size();
    std::vector<dq_eden_slice_t> all;
    std::vector<at::Tensor> planes;
    const int64_t many = (int64_t)py::len(slices);
    const at::Tensor results = empty_on(a.device, 4 * many, at::kFloat);
    int64_t room = 0;
    for (int64_t k = 0; k < many; k++) {
        const py::sequence s = slices[k];
        const int64_t start = py::cast<int64_t>(s[0]);
        dq_eden_slice_t x;
        x.count = py::cast<int64_t>(s[1]);
        x.n = py::cast<int64_t>(s[2]);
        x.rotations = py::cast<int>(s[3]);
        if (start < 0 || x.count <= 0 || start + x.count > v.numel()) refuse("a slice lies outside the vector");
        x.vec = static_cast<char *>(v.data_ptr()) + start * elem;
        x.seed = (int64_t)word(seed.ptr(), true);
        x.nbits = nbits;
        x.boundaries = b;
        x.centroids = c;
        planes.push_back(empty_on(a.device, x.n / 32 * nbits, at::kInt));
        x.packed = reinterpret_cast<uint32_t *>(planes.back().data_ptr<int32_t>());
        x.result = results.data_ptr<float>() + 4 * k;
        room += dq_eden_slice_bytes(x.n);
        all.push_back(x);
    }
    at::Tensor scratch = empty_on(a.device, room, at::kByte);
    check(dq_eden_compress(all.data(), (int)all.size(), dtype_code(v), scratch.data_ptr(), room, a.device, c10::hip::getCurrentHIPStream().stream()));
    py::list out;
    for (size_t k = 0; k < all.size(); k++)
        out.append(py::make_tuple(py::reinterpret_steal<py::object>(THPVariable_Wrap(planes[k])),
                                  py::reinterpret_steal<py::object>(THPVariable_Wrap(results.select(0, 4 * (int64_t)k + 2)))));
    return out;
}

// Eden.decompress: slices as (packed, nbits, centroids, scale, elements, rotations, seed), stored one after the other to out
void eden_decompress(py::handle out, py::sequence slices)
{
    Args a;
    const at::Tensor &y = a.tensor(out);
    const int64_t elem = y.element_size();
    std::vector<dq_eden_slice_t> all;
    int64_t room = 0, total = 0;
    for (size_t k = 0; k < py::len(slices); k++) {
        const py::sequence s = slices[k];
        dq_eden_slice_t x;
        const at::Tensor &p = a.typed(py::object(s[0]), at::kInt, 1, "packed_bins");
        x.nbits = py::cast<int>(s[1]);
        if (x.nbits < 1 || x.nbits > 8) refuse("nbits must be in [1, 8]");
        x.packed = reinterpret_cast<uint32_t *>(p.data_ptr<int32_t>());
        x.n = p.numel() / x.nbits * 32;
        x.centroids = a.typed(py::object(s[2]), at::kFloat, (int64_t)1 << x.nbits, "centroids").data_ptr<float>();
        x.boundaries = nullptr;
        x.result = a.typed(py::object(s[3]), at::kFloat, 1, "scale").data_ptr<float>();
        x.count = py::cast<int64_t>(s[4]);
        x.rotations = py::cast<int>(s[5]);
        x.seed = (int64_t)word(py::object(s[6]).ptr(), true);
        x.vec = static_cast<char *>(y.data_ptr()) + total * elem;
        total += x.count;
        room += dq_eden_slice_bytes(x.n);
        all.push_back(x);
    }
    if (total > y.numel()) refuse("out is too small");
    at::Tensor scratch = empty_on(a.device, room, at::kByte);
    check(dq_eden_decompress(all.data(), (int)all.size(), dtype_code(y), scratch.data_ptr(), room, a.device, c10::hip::getCurrentHIPStream().stream()));
}

// norm: a float32 device scalar, with (t, inv_sqrt, inv_levels, inv_clients); or None, with (lo, spacing, step) numbers
dq_thc_grid_t thc_grid(Args &a, py::handle norm, const py::tuple &numbers)
{
    dq_thc_grid_t g;
    memset(&g, 0, sizeof(g));
    if (norm.is_none()) {
        g.lo = py::cast<float>(numbers[0]);
        g.spacing = py::cast<float>(numbers[1]);
        g.step = py::cast<float>(numbers[2]);
    } else {
        g.norm = a.typed(norm, at::kFloat, 1, "max_norm").data_ptr<float>();
        g.t = py::cast<float>(numbers[0]);
        g.inv_sqrt = py::cast<float>(numbers[1]);
        g.inv_levels = py::cast<float>(numbers[2]);
        g.inv_clients = py::cast<float>(numbers[3]);
    }
    return g;
}

py::object thc_compress(py::handle src, int64_t count, py::handle work, py::handle bits, py::handle uniform, double scale,
                        py::handle norm, py::tuple numbers, int levels)
{
    Args a;
    const at::Tensor &x = a.tensor(src), &w = a.tensor(work);
    const int64_t n = w.numel();
    if (x.numel() < count || w.scalar_type() != at::kFloat) refuse("thc_compress: a buffer is too small or of the wrong dtype");
    const uint32_t *sign = reinterpret_cast<const uint32_t *>(a.typed(bits, at::kInt, n / 32, "sign").data_ptr<int32_t>());
    const float *u = a.typed(uniform, at::kFloat, n, "uniform").data_ptr<float>();
    const dq_thc_grid_t g = thc_grid(a, norm, numbers);
    at::Tensor out = empty_on(a.device, n, at::kBFloat16);
    check(dq_thc_compress(x.data_ptr(), dtype_code(x), count, w.data_ptr<float>(), sign, u, out.data_ptr(), n, (float)scale, &g, levels,
                          a.device, c10::hip::getCurrentHIPStream().stream()));
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(out));
}

// thc_compress with the uniform values that generator.uniform_() would fill a vector with, drawn in the kernel: the generator is
// moved on as that call moves it.  None where it cannot be: a generator of another device, a stream that records (torch
// keeps the generator's state on the device then), a GPU whose resident threads are no power of two, a length that the kernel does
// not draw for.  (thc.py asks only beside the torch releases whose launch of uniform_ this restates.)
py::object thc_compress_drawn(py::handle src, int64_t count, py::handle work, py::handle bits, py::handle generator, double scale,
                              py::handle norm, py::tuple numbers, int levels)
{
    Args a;
    const at::Tensor &x = a.tensor(src), &w = a.tensor(work);
    const int64_t n = w.numel();
    if (x.numel() < count || w.scalar_type() != at::kFloat) refuse("thc_compress: a buffer is too small or of the wrong dtype");
    const uint32_t *sign = reinterpret_cast<const uint32_t *>(a.typed(bits, at::kInt, n / 32, "sign").data_ptr<int32_t>());
    const dq_thc_grid_t g = thc_grid(a, norm, numbers);
    if (!THPGenerator_Check(generator.ptr())) return py::none();
    at::Generator gen = reinterpret_cast<THPGenerator *>(generator.ptr())->cdata;
    if (!gen.device().is_cuda() || gen.device().index() != a.device || n < (1 << 19) || n > (1 << 25)) return py::none();
    const hipStream_t stream = c10::hip::getCurrentHIPStream().stream();
    unsigned long long id = 0;
    if (Buckets::capturing(stream, &id)) return py::none();
    int cus = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, a.device) != hipSuccess ||
        hipDeviceGetAttribute(&per_cu, hipDeviceAttributeMaxThreadsPerMultiProcessor, a.device) != hipSuccess)
        return py::none();
    dq_uniform_stream_t drawn;
    drawn.threads = std::min((int64_t)cus * (per_cu / 256), (n + 255) / 256) * 256;
    if (drawn.threads <= 0 || (drawn.threads & (drawn.threads - 1)) != 0) return py::none();
    at::Tensor out = empty_on(a.device, n, at::kBFloat16);
    {
        const std::lock_guard<std::mutex> lock(gen.mutex());
        drawn.seed = gen.current_seed();
        drawn.offset = gen.get_offset();
        gen.set_offset(drawn.offset + 4 * ((uint64_t)((n - 1) / (4 * drawn.threads)) + 1));
    }
    check(dq_thc_compress_drawn(x.data_ptr(), dtype_code(x), count, w.data_ptr<float>(), sign, &drawn, out.data_ptr(), n, (float)scale, &g, levels,
                                a.device, stream));
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(out));
}

void thc_decompress(py::handle levels, py::handle bits, py::handle out, int64_t count, double scale, py::handle norm, py::tuple numbers)
{
    Args a;
    const at::Tensor &y = a.tensor(out);
    const int64_t n = y.numel();
    if (y.scalar_type() != at::kFloat) refuse("thc_decompress: out must be float32");
    const void *l = a.typed(levels, at::kBFloat16, n, "levels").data_ptr();
    const uint32_t *sign = reinterpret_cast<const uint32_t *>(a.typed(bits, at::kInt, n / 32, "sign").data_ptr<int32_t>());
    const dq_thc_grid_t g = thc_grid(a, norm, numbers);
    check(dq_thc_decompress(l, sign, y.data_ptr<float>(), count, n, (float)scale, &g, a.device, c10::hip::getCurrentHIPStream().stream()));
}

// ---- codec calls on tensors (capi.py) ------------------------------------------------------------------------
// positional arguments only, no argument-conversion layer: capi.py's functions give them in order

template <class F> PyObject *guarded(Py_ssize_t have, Py_ssize_t want, F body)
{
    try {
        if (have != want) refuse("wrong number of arguments");
        body();
    } catch (py::error_already_set &e) {
        e.restore();
        return nullptr;
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
    Py_RETURN_NONE;
}

int64_t integer(PyObject *o)
{
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw py::error_already_set();
    return v;
}

int small_integer(PyObject *o) { return (int)integer(o); }

float real(PyObject *o)
{
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw py::error_already_set();
    return (float)v;
}

// fp32 elements may come with a bf16 pool
int pair_code(const at::Tensor &elem, const at::Tensor &pool)
{
    const int code = dtype_code(elem);
    if (pool.scalar_type() == elem.scalar_type()) return code;
    if (code == DQ_F32 && pool.scalar_type() == at::kBFloat16) return code | DQ_RAND_BF16;
    refuse("rand_pool dtype must match input dtype");
}

// src, dst, rand_pool, n, nbits, chunk_size, strategy, stream
PyObject *scaling_compress(PyObject *, PyObject *const *v, Py_ssize_t have)
{
    return guarded(have, 8, [&] {
        Args a;
        const at::Tensor &src = a.tensor(v[0]), &dst = a.tensor(v[1]), &pool = a.tensor(v[2]);
        const int code = pair_code(src, pool), nbits = small_integer(v[4]), chunk = small_integer(v[5]), strategy = small_integer(v[6]);
        const int64_t n = integer(v[3]);
        const dq_stream_t s = stream_of(v[7]);
        const void *x = src.data_ptr(), *r = pool.data_ptr();
        uint8_t *y = static_cast<uint8_t *>(dst.data_ptr());
        int rc;
        {
            py::gil_scoped_release nogil;
            rc = dq_scaling_compress(x, y, r, n, nbits, chunk, code, a.device, strategy, s);
        }
        check(rc);
    });
}

// src, dst, n, nbits, chunk_size, strategy, add, stream
PyObject *scaling_decompress(PyObject *, PyObject *const *v, Py_ssize_t have)
{
    return guarded(have, 8, [&] {
        Args a;
        const at::Tensor &src = a.tensor(v[0]), &dst = a.tensor(v[1]);
        const int code = dtype_code(dst), nbits = small_integer(v[3]), chunk = small_integer(v[4]), strategy = small_integer(v[5]);
        const int64_t n = integer(v[2]);
        const int add = PyObject_IsTrue(v[6]);
        const dq_stream_t s = stream_of(v[7]);
        const uint8_t *x = static_cast<const uint8_t *>(src.data_ptr());
        void *y = dst.data_ptr();
        int rc;
        {
            py::gil_scoped_release nogil;
            rc = dq_scaling_decompress(x, y, n, nbits, chunk, code, a.device, strategy, s, add);
        }
        check(rc);
    });
}

// recv, inp, send, rand_pool, n, nbits, chunk_size, strategy, stream
PyObject *scaling_dec_comp(PyObject *, PyObject *const *v, Py_ssize_t have)
{
    return guarded(have, 9, [&] {
        Args a;
        const at::Tensor &recv = a.tensor(v[0]), &inp = a.tensor(v[1]), &send = a.tensor(v[2]), &pool = a.tensor(v[3]);
        const int code = pair_code(inp, pool), nbits = small_integer(v[5]), chunk = small_integer(v[6]), strategy = small_integer(v[7]);
        const int64_t n = integer(v[4]);
        const dq_stream_t s = stream_of(v[8]);
        const uint8_t *x = static_cast<const uint8_t *>(recv.data_ptr());
        uint8_t *y = static_cast<uint8_t *>(send.data_ptr());
        void *i = inp.data_ptr();
        const void *r = pool.data_ptr();
        int rc;
        {
            py::gil_scoped_release nogil;
            rc = dq_scaling_dec_comp(x, i, y, r, n, nbits, chunk, code, a.device, strategy, s);
        }
        check(rc);
    });
}

const void *sign_of(Args &a, PyObject *sign, int *packed)
{
    *packed = 0;
    if (sign == Py_None) return nullptr;
    const at::Tensor &t = a.tensor(sign);
    *packed = t.scalar_type() == at::kInt ? 1 : 0;
    return t.data_ptr();
}

// src, sign, dst, block, scale, nbits, strategy, rand_pool, seed, step, stream
PyObject *rht_scaling_compress(PyObject *, PyObject *const *v, Py_ssize_t have)
{
    return guarded(have, 11, [&] {
        Args a;
        const at::Tensor &src = a.tensor(v[0]);
        need(src.scalar_type() == at::kFloat, "rht_scaling_compress: src must be float32");
        int packed, rcode = 0;
        const void *sign = sign_of(a, v[1], &packed);
        uint8_t *y = static_cast<uint8_t *>(a.tensor(v[2]).data_ptr());
        const void *pool = nullptr;
        if (v[7] != Py_None) {
            const at::Tensor &p = a.tensor(v[7]);
            rcode = dtype_code(p);
            pool = p.data_ptr();
        }
        const int64_t block = integer(v[3]), n = src.numel();
        const float scale = real(v[4]), *x = static_cast<const float *>(src.data_ptr());
        const int nbits = small_integer(v[5]), strategy = small_integer(v[6]);
        const uint64_t seed = word(v[8]), step = word(v[9]);
        const dq_stream_t s = stream_of(v[10]);
        int rc;
        {
            py::gil_scoped_release nogil;
            rc = dq_rht_scaling_compress(x, sign, packed, y, pool, rcode, n, block, scale, nbits, a.device, strategy, seed, step, s);
        }
        check(rc);
    });
}

// src, sign, dst, block, scale, nbits, strategy, stream
PyObject *scaling_decompress_irht(PyObject *, PyObject *const *v, Py_ssize_t have)
{
    return guarded(have, 8, [&] {
        Args a;
        const uint8_t *x = static_cast<const uint8_t *>(a.tensor(v[0]).data_ptr());
        int packed;
        const void *sign = sign_of(a, v[1], &packed);
        const at::Tensor &dst = a.tensor(v[2]);
        need(dst.scalar_type() == at::kFloat, "scaling_decompress_irht: dst must be float32");
        const int64_t block = integer(v[3]), n = dst.numel();
        float *y = static_cast<float *>(dst.data_ptr());
        const float scale = real(v[4]);
        const int nbits = small_integer(v[5]), strategy = small_integer(v[6]);
        const dq_stream_t s = stream_of(v[7]);
        int rc;
        {
            py::gil_scoped_release nogil;
            rc = dq_scaling_decompress_irht(x, sign, packed, y, n, block, scale, nbits, a.device, strategy, s);
        }
        check(rc);
    });
}

PyMethodDef kFunctions[] = {
    {"scaling_compress", reinterpret_cast<PyCFunction>(scaling_compress), METH_FASTCALL, nullptr},
    {"scaling_decompress", reinterpret_cast<PyCFunction>(scaling_decompress), METH_FASTCALL, nullptr},
    {"scaling_dec_comp", reinterpret_cast<PyCFunction>(scaling_dec_comp), METH_FASTCALL, nullptr},
    {"rht_scaling_compress", reinterpret_cast<PyCFunction>(rht_scaling_compress), METH_FASTCALL, nullptr},
    {"scaling_decompress_irht", reinterpret_cast<PyCFunction>(scaling_decompress_irht), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

} // namespace

PYBIND11_MODULE(_host, m)
{
    PyModule_AddFunctions(m.ptr(), kFunctions);
    py::class_<Codec>(m, "Codec")
        .def(py::init<int, int, int, bool, uint32_t, py::object, py::dict>())
        .def_readwrite("nbits", &Codec::nbits)
        .def_readwrite("chunk", &Codec::chunk)
        .def_readwrite("strategy", &Codec::strategy)
        .def_readwrite("rand_seed", &Codec::rand_seed)
        .def_readwrite("philox", &Codec::philox)
        .def_readwrite("philox_seed", &Codec::philox_seed)
        .def_readwrite("philox_step", &Codec::philox_step)
        .def_readwrite("base", &Codec::base)
        .def_readwrite("pools", &Codec::pools)
        .def("compress", &Codec::compress)
        .def("decompress", &Codec::decompress)
        .def("dec_comp", &Codec::dec_comp);
    m.def("ranks_pooled", &ranks_pooled);
    m.def("ranks_fixed", &ranks_fixed);
    m.def("eden_compress", &eden_compress);
    m.def("eden_decompress", &eden_decompress);
    m.def("thc_compress", &thc_compress);
    m.def("thc_compress_drawn", &thc_compress_drawn);
    m.def("thc_decompress", &thc_decompress);
    m.doc() = "native host path of dynamiq_sigcomm_artifact_amd";
    py::class_<Buckets>(m, "Buckets")
        .def(py::init<int, uint64_t, py::object, py::object, py::object, py::object>())
        .def_readonly("recorded", &Buckets::recorded)
        .def("scratch", &Buckets::scratch)
        .def("join", &Buckets::join)
        .def("behind", &Buckets::behind)
        .def("settle", &Buckets::settle)
        .def("begin_step", &Buckets::begin_step);
    py::class_<Batch>(m, "Batch")
        .def(py::init([](Buckets &b, py::sequence pairs, py::sequence steps, py::sequence rows) {
            std::vector<uint64_t> s;
            std::vector<int64_t> at;
            for (size_t k = 0; k < py::len(steps); k++) s.push_back(py::cast<uint64_t>(steps[k]));
            for (size_t k = 0; k < py::len(rows); k++) at.push_back(py::cast<int64_t>(rows[k]));
            return new Batch(b, pairs, s, at);
        }))
        .def("matches", &Batch::matches)
        .def("launch", &Batch::launch)
        .def_property_readonly("runs", [](const Batch &b) {
            py::list counts;
            for (const Batch::Run &r : b.runs) counts.append(r.count);
            return counts;
        });
    m.def("roundtrip", &roundtrip);
    m.def("ranks_dynamic", &ranks_dynamic);
}
