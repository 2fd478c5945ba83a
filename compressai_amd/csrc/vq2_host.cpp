// vq2_host.cpp -- the argument checks and launches of the entries that small
// calls spend their time in, in native code (module compressai_amd._vq2_host).
//
// A batch-1 projection takes ~7 us on the GPU and its Python entry (checks,
// ctypes structures, allocation, launch) took ~18 us of host time.  Each
// function here takes the arguments of the kernels.py entry of its name and
// makes the same checks; a call that passes them is launched and its results
// returned, any other returns None before anything happened, and the Python
// entry goes on to refuse it or to handle it.  Nothing is kept between calls:
// every pointer, shape and type is read from the arguments of the call.
#include <torch/extension.h>

#include <algorithm>

#include "vq2_amd.h"

namespace py = pybind11;
using OptTensor = std::optional<at::Tensor>;

namespace {

constexpr int64_t CB_ROWS = 65536;

int dt_code(at::ScalarType t)
{
    switch (t) {
    case at::kFloat: return VQ2_DT_F32;
    case at::kHalf: return VQ2_DT_F16;
    case at::kBFloat16: return VQ2_DT_BF16;
    default: return -1;
    }
}

const void* ptr(const at::Tensor& t) { return t.const_data_ptr(); }
const void* ptr(const OptTensor& t) { return t ? t->const_data_ptr() : nullptr; }

// Collects what a call needs of its tensors; ok turns false at the first that
// the Python entry has to look at.
struct Check {
    bool ok = true;
    std::optional<at::Device> dev;
    void need(bool c) { ok = ok && c; }
    void on_gpu(const at::Tensor& t)
    {
        if (!dev) dev = t.device();
        need(t.is_cuda() && t.device() == *dev);
    }
    void dense(const at::Tensor& t)
    {
        on_gpu(t);
        need(t.is_contiguous());
    }
    void table(const OptTensor& t, at::ScalarType dt, int64_t n)
    {
        if (!t) return;
        dense(*t);
        need(t->scalar_type() == dt && t->numel() == n);
    }
    // a codebook of at least `rows` rows
    void book(const at::Tensor& t, int64_t rows)
    {
        dense(t);
        need(t.dim() == 2 && t.size(0) >= rows && t.size(1) == 8);
    }
    void scales(const at::Tensor& t, int64_t n)
    {
        dense(t);
        need(t.numel() == n && dt_code(t.scalar_type()) >= 0);
    }
};

int64_t attr_int(py::handle o, const char* name) { return py::cast<int64_t>(o.attr(name)); }

void* stream_of(const at::Device& dev)
{
    // a handle that is never given back: an object would be released after the
    // interpreter has ended
    static const py::handle get = py::object(py::module_::import("torch._C").attr("_cuda_getCurrentRawStream")).release();
    return (void*)py::cast<uintptr_t>(get((int)dev.index()));
}

// Runs a library call without the interpreter lock, as ctypes does: a launch
// waits while the GPU's queue is full, and the other Python threads stood
// still with it (600 ms behind 0.6 s of queued work).  The call may touch no
// Python object and throws nothing.
template <class F>
int unlocked(F call)
{
    PyThreadState* const state = PyEval_SaveThread();
    const int status = call();
    PyEval_RestoreThread(state);
    return status;
}

void check_status(int status, const char* name)
{
    if (status == VQ2_OK) return;
    py::module_::import("compressai_amd._lib").attr("check")(status, name);
}

// (workspace pointer, bytes) from kernels._workspace for the sorted launches
std::pair<void*, size_t> sorted_workspace(py::handle get, const at::Device& dev, size_t bytes)
{
    if (bytes == 0) return {nullptr, 0};
    py::object buf = get(py::cast(dev), bytes, py::arg("sorted_kind") = true);
    const at::Tensor t = py::cast<at::Tensor>(buf);
    return {t.data_ptr(), (size_t)t.numel()};
}

// The rule of kernels.sorted_slices (tests/test_launch_chunks.py compares the
// two); chunks >= 1.
int64_t sorted_slices(int64_t chunks, int64_t min_ipc, int64_t cu)
{
    const int64_t fit = cu / chunks;
    return fit >= 3 ? std::max<int64_t>(1, std::min<int64_t>({32, fit, min_ipc / 20})) : 1;
}

// vq_sorted_gemv(x, mats, cb0, cb1, n, perm, sign, hb, rht_scale, rs, out_dtype=...)
py::object sorted_gemv(const at::Tensor& x, const py::sequence& mats, const at::Tensor& cb0, const OptTensor& cb1, int64_t n,
                       const OptTensor& perm, const OptTensor& sign, int64_t hb, std::optional<double> rht_scale, double rs,
                       at::ScalarType out_dtype, int64_t cu, py::handle workspace)
{
    const size_t k = mats.size();
    Check c;
    c.dense(x);
    c.need(k >= 1 && k <= 4 && x.numel() == n && dt_code(x.scalar_type()) >= 0 && dt_code(out_dtype) >= 0);
    c.table(perm, at::kInt, n);
    c.table(sign, at::kChar, n);
    c.book(cb0, CB_ROWS);
    c.need(cb0.scalar_type() == at::kHalf || cb0.scalar_type() == at::kBFloat16);
    if (!c.ok) return py::none();
    vq2_sorted_mat m[4] = {};
    int64_t chunks = 0, min_ipc = INT64_MAX, s2 = -1;
    at::ScalarType s_dt = at::kFloat;
    py::list ys;
    for (size_t i = 0; i < k; i++) {
        py::tuple pair = mats[i];
        if (pair.size() != 2) return py::none();
        py::handle p = pair[0];
        const at::Tensor scale = py::cast<at::Tensor>(pair[1]), ent = py::cast<at::Tensor>(p.attr("entries"));
        const int64_t rows = attr_int(p, "out_rows"), kind = attr_int(p, "s2_kind");
        c.scales(scale, rows);
        c.on_gpu(ent);
        c.need(attr_int(p, "n") == n && (i == 0 || (kind == s2 && scale.scalar_type() == s_dt)));
        s2 = kind;
        s_dt = scale.scalar_type();
        m[i] = vq2_sorted_mat{(const uint32_t*)ptr(ent), attr_int(p, "iters_per_chunk"), attr_int(p, "stage1_iters"),
                              attr_int(p, "n_iters"), attr_int(p, "rows_per_chunk"), (int)kind, ptr(scale), nullptr, rows};
        chunks += attr_int(p, "n_chunks");
        min_ipc = std::min(min_ipc, m[i].iters_per_chunk);
    }
    if (s2 != 0) {
        if (!cb1) return py::none();
        c.book(*cb1, s2 == 2 ? 256 : CB_ROWS);
        c.need(cb1->scalar_type() == cb0.scalar_type());
    } else if (cb1) {
        c.on_gpu(*cb1);
    }
    if (!c.ok || chunks < 1) return py::none();
    for (size_t i = 0; i < k; i++) {
        at::Tensor y = at::empty({m[i].out_rows}, x.options().dtype(out_dtype));
        m[i].y = y.data_ptr();
        ys.append(y);
    }
    const int slices = (int)sorted_slices(chunks, min_ipc, cu);
    const auto ws = sorted_workspace(workspace, *c.dev, vq2_sorted_gemv_workspace(m, (int)k, slices));
    const float sc = rht_scale ? (float)*rht_scale : (hb ? (float)(1.0 / std::sqrt((double)hb)) : 1.0f);
    void* const st = stream_of(*c.dev);
    check_status(unlocked([&] {
                     return vq2_sorted_gemv(ptr(x), dt_code(x.scalar_type()), (const int32_t*)ptr(perm), (const int8_t*)ptr(sign),
                                            hb, sc, (int)k, m, ptr(cb0), s2 ? ptr(cb1) : nullptr, dt_code(cb0.scalar_type()),
                                            dt_code(s_dt), dt_code(out_dtype), n, (float)rs, slices, ws.first, ws.second, st);
                 }),
                 "vq2_sorted_gemv");
    return ys;
}

// The matrices of vq_gemv_rht / vq_rows_gemm: (i0, i1 or None, scale, rows)
// each, as kernels.check_gemv_rht_mats takes them.
struct Mats {
    size_t k = 0;
    vq2_seg seg[4] = {};
    int s2 = VQ2_S2_NONE;
    at::ScalarType s_dt = at::kFloat;
};

void read_mats(Check& c, Mats& r, const py::sequence& mats, const at::Tensor& cb0, const OptTensor& cb1, int64_t n)
{
    r.k = mats.size();
    c.need(r.k >= 1 && r.k <= 4 && n % 8 == 0);
    c.book(cb0, CB_ROWS);
    c.need(dt_code(cb0.scalar_type()) >= 0);
    if (!c.ok) return;
    for (size_t i = 0; i < r.k; i++) {
        py::tuple t = mats[i];
        if (t.size() != 4) return c.need(false);
        const at::Tensor i0 = py::cast<at::Tensor>(t[0]), scale = py::cast<at::Tensor>(t[2]);
        const OptTensor i1 = py::cast<OptTensor>(t[1]);
        const int64_t rows = py::cast<int64_t>(t[3]);
        c.dense(i0);
        c.need(i0.scalar_type() == at::kShort && i0.numel() == rows * (n / 8));
        c.scales(scale, rows);
        int s2 = VQ2_S2_NONE;
        if (i1) {
            c.dense(*i1);
            s2 = i1->scalar_type() == at::kByte ? VQ2_S2_U8 : VQ2_S2_U16;
            c.need((s2 == VQ2_S2_U8 || i1->scalar_type() == at::kShort) && i1->numel() == i0.numel() && cb1.has_value());
            if (!c.ok) return;
            c.book(*cb1, s2 == VQ2_S2_U8 ? 256 : CB_ROWS);
            c.need(cb1->scalar_type() == cb0.scalar_type());
        }
        c.need(i == 0 || (s2 == r.s2 && scale.scalar_type() == r.s_dt));
        if (!c.ok) return;
        r.s2 = s2;
        r.s_dt = scale.scalar_type();
        r.seg[i] = vq2_seg{(const int16_t*)ptr(i0), ptr(i1), ptr(scale), nullptr, rows, rows};
    }
    if (cb1) c.on_gpu(*cb1);
}

py::list make_outputs(Mats& r, const at::Tensor& x, std::optional<int64_t> batch, at::ScalarType out_dtype)
{
    py::list ys;
    for (size_t i = 0; i < r.k; i++) {
        const int64_t rows = r.seg[i].out_rows;
        at::Tensor y = batch ? at::empty({*batch, rows}, x.options().dtype(out_dtype))
                             : at::empty({rows}, x.options().dtype(out_dtype));
        r.seg[i].y = y.data_ptr();
        ys.append(y);
    }
    return ys;
}

// vq_gemv_rht within the fused width
py::object gemv_rht(const at::Tensor& x, const py::sequence& mats, const at::Tensor& cb0, const OptTensor& cb1, int64_t n,
                    const OptTensor& perm, const OptTensor& sign, int64_t hb, std::optional<double> rht_scale, double rs,
                    at::ScalarType out_dtype)
{
    Check c;
    c.dense(x);
    c.need(n > 0 && x.numel() % std::max<int64_t>(n, 1) == 0 && dt_code(x.scalar_type()) >= 0 && dt_code(out_dtype) >= 0);
    c.table(perm, at::kInt, n);
    c.table(sign, at::kChar, n);
    if (!c.ok) return py::none();
    Mats r;
    read_mats(c, r, mats, cb0, cb1, n);
    if (!c.ok) return py::none();
    const int64_t batch = x.numel() / n;
    py::list ys = make_outputs(r, x, x.dim() == 2 ? std::optional<int64_t>(batch) : std::nullopt, out_dtype);
    if (x.dim() != 2 && batch != 1) return py::none();
    const float sc = rht_scale ? (float)*rht_scale : (float)(1.0 / std::sqrt((double)hb));
    void* const st = stream_of(*c.dev);
    check_status(unlocked([&] {
                     return vq2_gemv_rht(ptr(x), dt_code(x.scalar_type()), batch, n, (const int32_t*)ptr(perm),
                                         (const int8_t*)ptr(sign), hb, sc, (int)r.k, r.seg, r.s2, ptr(cb0), ptr(cb1),
                                         dt_code(cb0.scalar_type()), dt_code(r.s_dt), dt_code(out_dtype), n, (float)rs, st);
                 }),
                 "vq2_gemv_rht");
    return ys;
}

// vq_rows_gemm
py::object rows_gemm(const at::Tensor& x, const py::sequence& mats, const at::Tensor& cb0, const OptTensor& cb1, int64_t n,
                     const OptTensor& perm, const OptTensor& sign, int64_t hb, std::optional<double> rht_scale, double rs,
                     at::ScalarType act_dtype, at::ScalarType out_dtype)
{
    Check c;
    c.dense(x);
    c.need(n >= 64 && n % 64 == 0 && n <= 8192 && x.numel() > 0 && x.numel() % n == 0 && dt_code(x.scalar_type()) >= 0 &&
           dt_code(out_dtype) >= 0 && dt_code(act_dtype) >= 0);
    c.table(perm, at::kInt, n);
    c.table(sign, at::kChar, n);
    if (!c.ok) return py::none();
    Mats r;
    read_mats(c, r, mats, cb0, cb1, n);
    if (!c.ok) return py::none();
    const int64_t batch = x.numel() / n;
    const int cdt = dt_code(cb0.scalar_type());
    const size_t bytes = vq2_rows_gemm_workspace(batch, n, (int)r.k, r.seg, r.s2, cdt);
    if (bytes == 0) return py::none();
    py::list ys = make_outputs(r, x, batch, out_dtype);
    const at::Tensor ws = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte));
    const float sc = rht_scale ? (float)*rht_scale : (hb ? (float)(1.0 / std::sqrt((double)hb)) : 1.0f);
    void* const st = stream_of(*c.dev);
    check_status(unlocked([&] {
                     return vq2_rows_gemm(ptr(x), dt_code(x.scalar_type()), batch, n, (const int32_t*)ptr(perm),
                                          (const int8_t*)ptr(sign), hb, sc, dt_code(act_dtype), (int)r.k, r.seg, r.s2,
                                          ptr(cb0), ptr(cb1), cdt, dt_code(r.s_dt), dt_code(out_dtype), n, (float)rs,
                                          ws.data_ptr(), bytes, st);
                 }),
                 "vq2_rows_gemm");
    return ys;
}

bool read_rot(Check& c, vq2_rot_tables& r, const py::tuple& t, int64_t n, OptTensor& perm, OptTensor& sign)
{
    if (t.size() != 4) return false;
    perm = py::cast<OptTensor>(t[0]);
    sign = py::cast<OptTensor>(t[1]);
    c.table(perm, at::kInt, n);
    c.table(sign, at::kChar, n);
    r = vq2_rot_tables{(const int32_t*)ptr(perm), (const int8_t*)ptr(sign), py::cast<int64_t>(t[2]),
                       (float)py::cast<double>(t[3])};
    return c.ok;
}

struct Pool {
    int64_t experts, rows, ng, chunks;
    vq2_sorted_pool p;
};

Pool read_pool(Check& c, py::handle o, const at::Tensor& scale)
{
    const at::Tensor ent = py::cast<at::Tensor>(o.attr("entries"));
    Pool r;
    r.experts = attr_int(o, "n_experts");
    r.rows = attr_int(o, "rows");
    r.ng = attr_int(o, "ng");
    r.chunks = attr_int(o, "chunks");
    c.on_gpu(ent);
    c.scales(scale, r.experts * r.rows);
    c.need(attr_int(o, "s2_kind") == 0);  // two-stage pools: the Python entry
    const int64_t ipc = attr_int(o, "iters_per_chunk");
    r.p = vq2_sorted_pool{(const uint32_t*)ptr(ent), ipc, attr_int(o, "n_iters"), attr_int(o, "rows_per_chunk"), r.rows, r.ng,
                          ptr(scale), std::max(dt_code(scale.scalar_type()), 0), attr_int(o, "stage1_iters"), 0, nullptr};
    return r;
}

// vq_sorted_moe of one-stage pools, with ids and w or with the router built
// in; slices as kernels.moe_slices chooses them (asked through `slices`)
py::object sorted_moe(const at::Tensor& h, py::handle gate_up, const at::Tensor& gu_scale, py::handle down,
                      const at::Tensor& dn_scale, const at::Tensor& cb, const py::tuple& rot_h, const py::tuple& rot_i,
                      const OptTensor& ids, const OptTensor& w, const OptTensor& logits, std::optional<int64_t> top_k,
                      std::optional<int64_t> shared_id, const OptTensor& gate, at::ScalarType out_dtype,
                      py::handle slices, py::handle workspace)
{
    Check c;
    c.dense(h);
    const Pool gp = read_pool(c, gate_up, gu_scale), dp = read_pool(c, down, dn_scale);
    const int64_t H = gp.ng * 8, I = dp.ng * 8;
    c.need(gp.rows == 2 * I && dp.rows == H && gp.experts == dp.experts && h.numel() > 0 && h.numel() % H == 0 &&
           dt_code(h.scalar_type()) >= 0 && dt_code(out_dtype) >= 0);
    c.book(cb, CB_ROWS);
    c.need(cb.scalar_type() == at::kHalf || cb.scalar_type() == at::kBFloat16);
    vq2_rot_tables rh, ri;
    OptTensor keep[4];
    if (!c.ok || !read_rot(c, rh, rot_h, H, keep[0], keep[1]) || !read_rot(c, ri, rot_i, I, keep[2], keep[3]))
        return py::none();
    const int64_t T = h.numel() / H;
    const bool router = logits.has_value();
    int64_t P, n_routed = 0;
    at::Tensor ids_out, w_out;
    if (router) {
        if (!gate || !top_k || !shared_id || ids || w) return py::none();
        c.dense(*logits);
        c.dense(*gate);
        c.need(gate->numel() == H && dt_code(gate->scalar_type()) >= 0 && dt_code(logits->scalar_type()) >= 0 &&
               *top_k >= 1 && logits->numel() % T == 0);
        if (!c.ok) return py::none();
        P = *top_k + 1;
        n_routed = logits->numel() / T;
        ids_out = at::empty({T, P}, h.options().dtype(at::kInt));
        w_out = at::empty({T, P}, h.options().dtype(at::kFloat));
    } else {
        if (!ids || !w) return py::none();
        c.dense(*ids);
        c.dense(*w);
        c.need(ids->numel() % T == 0 && w->numel() == ids->numel() && w->scalar_type() == at::kFloat &&
               (ids->scalar_type() == at::kInt || ids->scalar_type() == at::kLong));
        if (!c.ok) return py::none();
        P = ids->numel() / T;
    }
    const py::tuple sl = slices(T, P, gate_up, down, py::cast(*c.dev), H, I, rh.hb, ri.hb);
    const int sg = py::cast<int>(sl[0]), sd = py::cast<int>(sl[1]);
    const auto ws = sorted_workspace(workspace, *c.dev, vq2_sorted_moe_workspace(T, (int)P, H, I, sg, sd));
    at::Tensor out = at::empty({T, H}, h.options().dtype(out_dtype));
    int32_t* const io = router ? ids_out.data_ptr<int32_t>() : nullptr;
    float* const wo = router ? w_out.data_ptr<float>() : nullptr;
    void* const st = stream_of(*c.dev);
    check_status(unlocked([&] {
                     return vq2_sorted_moe(
                         ptr(h), dt_code(h.scalar_type()), T, (int)P, router ? nullptr : ptr(ids),
                         !router && ids->scalar_type() == at::kLong, router ? nullptr : (const float*)ptr(w),
                         router ? ptr(logits) : nullptr, router ? dt_code(logits->scalar_type()) : 0, n_routed,
                         router ? (int)*top_k : 0, router ? *shared_id : 0, router ? ptr(gate) : nullptr,
                         router ? dt_code(gate->scalar_type()) : 0, io, wo, gp.experts, H, I, &gp.p, &dp.p, ptr(cb),
                         dt_code(cb.scalar_type()), &rh, &ri, out.data_ptr(), dt_code(out_dtype), sg, sd, ws.first, ws.second,
                         st);
                 }),
                 "vq2_sorted_moe");
    if (router) return py::make_tuple(out, ids_out, w_out);
    return py::cast(out);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.def("sorted_gemv", &sorted_gemv);
    m.def("gemv_rht", &gemv_rht);
    m.def("rows_gemm", &rows_gemm);
    m.def("sorted_moe", &sorted_moe);
    m.def("sorted_slices", [](int64_t chunks, int64_t min_ipc, int64_t cu) {
        return sorted_slices(std::max<int64_t>(1, chunks), min_ipc, cu);
    });
}
