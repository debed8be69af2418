// Tensor front end of the entry points that a training or inference step calls,
// as a Python extension (distdl_amd._front).  A call through ctypes costs the host
// 15 to 20 us beside the launch's four: attribute reads of every tensor, output and
// workspace allocations, marshalling; the same here costs two to four.
//
// Every function takes the forms that layers hand over step by step (device tensors
// of one type, contiguous but for the weight's pitch) and returns None for any other:
// the callers in hip_ops.py then go their general way, which converts, copies or
// raises.  A failing entry point raises RuntimeError as _lib.check does.  The
// interpreter lock is released while a function runs.
#include "front.h"

namespace ddl_front {

int float_code(const Tensor& t) {   // 0: none of the three
    switch (t.scalar_type()) {
        case at::kFloat: return DDL_DT_F32;
        case at::kBFloat16: return DDL_DT_BF16;
        case at::kHalf: return DDL_DT_F16;
        default: return 0;
    }
}

namespace {

int sum_code(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kDouble: return DDL_DT_F64;
        case at::kInt: return DDL_DT_I32;
        case at::kLong: return DDL_DT_I64;
        default: return float_code(t);
    }
}

Tensor floats(const Tensor& like, at::IntArrayRef shape) { return at::empty(shape, like.options().dtype(at::kFloat)); }
Tensor shaped(const Tensor& like, const std::optional<std::vector<int64_t>>& shape) { return shape ? at::empty(*shape, like.options()) : Tensor(); }
int64_t clamped(int64_t n, int64_t most) { return n < 1 ? 1 : n > most ? most : n; }

}  // namespace

// ---------------------------------------------------------------- linear --

// Is `w` the [n, k] matrix of a product with `x`, in any number of dimensions of which the leading ones have one element?
static bool weight_matrix(const Tensor& w, const Tensor& x) {
    if (!w.is_cuda() || w.scalar_type() != x.scalar_type() || w.dim() < 2) return false;
    for (int64_t d = 0; d < w.dim() - 2; ++d)
        if (w.size(d) != 1) return false;
    return w.size(-2) > 0 && w.size(-1) > 0 && (w.size(-1) == 1 || w.stride(-1) == 1);
}

MaybeTensor product(const Tensor& x, const Tensor& w, const MaybeTensor& bias) {
    const int dt = float_code(x);
    if (!dt || !plain(x) || !weight_matrix(w, x) || x.dim() < 1 || x.numel() == 0) return std::nullopt;
    const int64_t n = w.size(-2), k = w.size(-1);
    if (x.size(-1) != k) return std::nullopt;
    if (bias && (!plain(*bias) || bias->scalar_type() != x.scalar_type() || bias->numel() != n)) return std::nullopt;
    const int64_t m = x.numel() / k, ldw = n > 1 ? w.stride(-2) : k;
    const void *px = x.data_ptr(), *pw = w.data_ptr();
    const bool aligned = multiple(px, 16) && multiple(pw, 16);
    if (dt != DDL_DT_F32 && !(k % 8 == 0 && aligned && (n <= 1 || ldw % 8 == 0)) && !ddl_gemm_in_place(dt, aligned, k, 1, ldw, 1, m, n, k))
        return std::nullopt;
    auto shape = x.sizes().vec();
    shape.back() = n;
    Tensor y = at::empty(shape, x.options()), work;
    const int64_t elems = ddl_gemm_workspace_at(dt, aligned, k, 1, ldw, 1, m, n, k);
    if (elems) work = floats(x, {elems});
    check(ddl_gemm_ws(px, k, 1, pw, ldw, 1, pointer(bias), y.data_ptr(), dt, n, m, n, k, static_cast<float*>(pointer(work)), elems, current_stream()),
          "ddl_gemm");
    return y;
}

std::optional<std::tuple<Tensor, Tensor, Tensor>> product_backward(const Tensor& x, const Tensor& w, const Tensor& dy, bool need_x, bool need_w,
                                                                  const MaybeShape& bias_shape) {
    const int dt = float_code(x);
    if (!dt || !plain(x) || !plain(dy) || !weight_matrix(w, x) || dy.scalar_type() != x.scalar_type()) return std::nullopt;
    const int64_t n = w.size(-2), k = w.size(-1);
    const bool need_b = bias_shape.has_value();
    if (x.numel() == 0 || x.numel() % k != 0) return std::nullopt;
    const int64_t m = x.numel() / k, ldw = n > 1 ? w.stride(-2) : k;
    if (dy.numel() != m * n) return std::nullopt;
    const void *px = x.data_ptr(), *pw = w.data_ptr(), *pdy = dy.data_ptr();
    if (dt != DDL_DT_F32) {   // the conditions of hip_ops.linear_backward for reading every operand where it lies
        auto along_k = [](const void* p, int64_t pitch, int64_t depth) { return depth % 8 == 0 && pitch % 8 == 0 && pitch <= 0x3FFFFF && multiple(p, 16); };
        auto along_rows = [](const void* p, int64_t pitch, int64_t rows, int64_t depth) {
            return rows % 8 == 0 && pitch % 8 == 0 && pitch <= 0x3FFFFF && multiple(p, 16) && (depth + 64) * pitch <= 0x3FFFFFFF;
        };
        if (need_x && !(along_k(pdy, n, n) && along_rows(pw, ldw, k, n)) && !ddl_gemm_in_place(dt, multiple(pdy, 16) && multiple(pw, 16), n, 1, 1, ldw, m, k, n))
            return std::nullopt;
        if (need_w && !(along_rows(pdy, n, n, m) && along_rows(px, k, k, m)) && !ddl_gemm_in_place(dt, multiple(pdy, 16) && multiple(px, 16), 1, n, 1, k, n, k, m))
            return std::nullopt;
    }
    Tensor dx, dw, db, work;
    if (need_x) dx = at::empty(x.sizes(), x.options());
    if (need_w) dw = at::empty(w.sizes(), x.options());
    if (need_b) db = at::empty(*bias_shape, x.options());
    const bool aligned = multiple(px, 16) && multiple(pw, 16) && multiple(pdy, 16);
    const int64_t elems = ddl_linear_backward_workspace_at(dt, aligned, m, n, k, k, ldw, n, need_x, need_w, need_b);
    if (elems) work = floats(x, {elems});
    check(ddl_linear_backward(px, pw, pdy, pointer(dx), pointer(dw), pointer(db), dt, m, n, k, k, ldw, n, static_cast<float*>(pointer(work)), elems,
                              current_stream()),
          "ddl_linear_backward");
    return std::make_tuple(dx, dw, db);
}

// ------------------------------------------------------------ layer norm --

namespace {

bool ln_operands(const Tensor& x, const MaybeTensor& gamma, const MaybeTensor& beta, int64_t cols) {
    if (!float_code(x) || !plain(x) || cols < 1 || x.numel() == 0 || x.numel() % cols != 0 || gamma.has_value() != beta.has_value()) return false;
    if (!gamma) return true;
    return plain(*gamma) && plain(*beta) && gamma->scalar_type() == x.scalar_type() && beta->scalar_type() == x.scalar_type() &&
           gamma->numel() == cols && beta->numel() == cols;
}

}  // namespace

std::optional<Normalized> layer_norm(const Tensor& x, const MaybeTensor& gamma, const MaybeTensor& beta, int64_t cols, double eps) {
    if (!ln_operands(x, gamma, beta, cols)) return std::nullopt;
    const int64_t rows = x.numel() / cols;
    Tensor y = at::empty(x.sizes(), x.options()), mean = floats(x, {rows}), rstd = floats(x, {rows});
    check(ddl_layer_norm(x.data_ptr(), float_code(x), rows, cols, cols, pointer(gamma), pointer(beta), static_cast<float>(eps), y.data_ptr(), cols,
                         mean.data_ptr<float>(), rstd.data_ptr<float>(), current_stream()),
          "ddl_layer_norm");
    return Normalized(y, x.detach().view({rows, cols}), mean, rstd, gamma ? gamma->detach().view({cols}) : Tensor());
}

namespace {

bool ln_backward_operands(const Tensor& dy, const Tensor& x2d, const Tensor& mean, const Tensor& rstd, const MaybeTensor& gamma) {
    return float_code(x2d) && plain(dy) && plain(x2d) && plain(mean) && plain(rstd) && x2d.dim() == 2 && x2d.numel() > 0 &&
           dy.scalar_type() == x2d.scalar_type() && dy.numel() == x2d.numel() &&
           (!gamma || (plain(*gamma) && gamma->scalar_type() == x2d.scalar_type() && gamma->numel() == x2d.size(1)));
}

}  // namespace

// Rows this worker holds whole: dx and the parameters' gradients in one pass.  dy may have any shape of as many elements.
std::optional<std::tuple<Tensor, Tensor, Tensor>> ln_backward_whole(const Tensor& dy, const Tensor& x2d, const Tensor& mean, const Tensor& rstd,
                                                                    const MaybeTensor& gamma, const MaybeShape& gamma_shape, const MaybeShape& beta_shape) {
    if (!ln_backward_operands(dy, x2d, mean, rstd, gamma)) return std::nullopt;
    const int64_t rows = x2d.size(0), cols = x2d.size(1), quad = 4 * x2d.element_size();
    const bool vec = cols % 4 == 0 && multiple(x2d.data_ptr(), quad) && multiple(dy.data_ptr(), quad) && (!gamma || multiple(gamma->data_ptr(), quad));
    const bool one_pass = vec && cols <= 1024;
    if (!one_pass && (!(gamma_shape || beta_shape) || cols <= 512 || (cols > 8192 && !(vec && cols <= 16384)))) return std::nullopt;
    const int64_t splits = one_pass ? clamped((rows + 31) / 32, 256) : clamped((rows + 3) / 4, 256);
    Tensor dx = at::empty(dy.sizes(), dy.options()), dg = shaped(dy, gamma_shape), db = shaped(dy, beta_shape), work = floats(dy, {2 * splits * cols});
    const float weight = static_cast<float>(1.0 / static_cast<double>(cols));
    const int dt = float_code(x2d);
    if (one_pass)
        check(ddl_ln_bwd_one_pass(dy.data_ptr(), x2d.data_ptr(), dt, rows, cols, cols, cols, mean.data_ptr<float>(), rstd.data_ptr<float>(), pointer(gamma),
                                  nullptr, 1, 0, weight, dx.data_ptr(), cols, work.data_ptr<float>(), work.numel(), pointer(dg), pointer(db),
                                  current_stream()),
              "ddl_ln_bwd_one_pass");
    else
        check(ddl_ln_bwd_whole_rows(dy.data_ptr(), x2d.data_ptr(), dt, rows, cols, cols, cols, mean.data_ptr<float>(), rstd.data_ptr<float>(),
                                    pointer(gamma), weight, dx.data_ptr(), cols, work.data_ptr<float>(), work.numel(), pointer(dg), pointer(db),
                                    current_stream()),
              "ddl_ln_bwd_whole_rows");
    return std::make_tuple(dx, dg, db);
}

// Rows shared with other workers: this worker's row sums and partial column sums ...
std::optional<std::tuple<Tensor, Tensor>> ln_backward_partial_params(const Tensor& dy, const Tensor& x2d, const Tensor& mean, const Tensor& rstd,
                                                                     const MaybeTensor& gamma) {
    if (!ln_backward_operands(dy, x2d, mean, rstd, gamma) || dy.sizes() != x2d.sizes()) return std::nullopt;
    const int64_t rows = x2d.size(0), cols = x2d.size(1);
    Tensor sums = floats(dy, {rows, 2}), work = floats(dy, {ddl_ln_bwd_partial_params_workspace(rows, cols)});
    check(ddl_ln_bwd_partial_params(dy.data_ptr(), x2d.data_ptr(), float_code(x2d), rows, cols, cols, cols, mean.data_ptr<float>(), rstd.data_ptr<float>(),
                                    pointer(gamma), sums.data_ptr<float>(), work.data_ptr<float>(), work.numel(), current_stream()),
          "ddl_ln_bwd_partial_params");
    return std::make_tuple(sums, work);
}

// ... and dx and the parameters' gradients from all workers' row sums.
std::optional<std::tuple<Tensor, Tensor, Tensor>> ln_backward_input_params(const Tensor& dy, const Tensor& x2d, const Tensor& mean, const Tensor& rstd,
                                                                           const MaybeTensor& gamma, const Tensor& part_sums, double weight,
                                                                           const Tensor& work, const MaybeShape& gamma_shape, const MaybeShape& beta_shape) {
    if (!ln_backward_operands(dy, x2d, mean, rstd, gamma) || dy.sizes() != x2d.sizes() || !plain(part_sums) || !plain(work) || part_sums.scalar_type() != at::kFloat ||
        work.scalar_type() != at::kFloat || part_sums.dim() != 3 || part_sums.size(1) != x2d.size(0) || part_sums.size(2) != 2)
        return std::nullopt;
    const int64_t rows = x2d.size(0), cols = x2d.size(1);
    Tensor dx = at::empty(dy.sizes(), dy.options()), dg = shaped(dy, gamma_shape), db = shaped(dy, beta_shape);
    check(ddl_ln_bwd_input_params(dy.data_ptr(), x2d.data_ptr(), float_code(x2d), rows, cols, cols, cols, mean.data_ptr<float>(), rstd.data_ptr<float>(),
                                  pointer(gamma), part_sums.data_ptr<float>(), static_cast<int>(part_sums.size(0)), static_cast<float>(weight),
                                  dx.data_ptr(), cols, work.data_ptr<float>(), work.numel(), pointer(dg), pointer(db), current_stream()),
          "ddl_ln_bwd_input_params");
    return std::make_tuple(dx, dg, db);
}

// ------------------------------------------------------------- embedding --

static bool id_tensor(const Tensor& ids) { return plain(ids) && (ids.scalar_type() == at::kLong || ids.scalar_type() == at::kInt); }

MaybeTensor embedding_gather(const Tensor& weight, const Tensor& ids, int64_t lo, int64_t hi) {
    if (!plain(weight) || weight.dim() != 2 || weight.size(0) != hi - lo || !id_tensor(ids)) return std::nullopt;
    auto shape = ids.sizes().vec();
    const int64_t dim = weight.size(1);
    shape.push_back(dim);
    Tensor out = at::empty(shape, weight.options());
    check(ddl_embedding_gather(weight.data_ptr(), dim, dim, static_cast<int>(weight.element_size()), ids.data_ptr(), ids.scalar_type() == at::kLong,
                               ids.numel(), lo, hi, out.data_ptr(), current_stream()),
          "ddl_embedding_gather");
    return out;
}

MaybeTensor embedding_backward(const Tensor& dy, const Tensor& ids, int64_t lo, int64_t hi, int64_t padding_idx, bool by_freq) {
    const int dt = float_code(dy);
    if (!dt || !plain(dy) || !id_tensor(ids) || dy.dim() != ids.dim() + 1 || dy.sizes().slice(0, ids.dim()) != ids.sizes() || dy.size(-1) == 0 || hi < lo)
        return std::nullopt;
    const int64_t dim = dy.size(-1), rows = hi - lo, n = ids.numel();
    const int64_t few = 3 * rows + 1 + n, all = ddl_embedding_backward_workspace(n, rows), elems = few > all ? few : all;
    Tensor dw = at::empty({rows, dim}, dy.options()), work = at::empty({elems}, dy.options().dtype(at::kInt));
    check(ddl_embedding_backward(dy.data_ptr(), dt, dim, dim, ids.data_ptr(), ids.scalar_type() == at::kLong, n, lo, hi, padding_idx, by_freq, dw.data_ptr(),
                                 dim, work.data_ptr<int32_t>(), elems, current_stream()),
          "ddl_embedding_backward");
    return dw;
}

// ----------------------------------------------------------------- boxes --

Boxes::Boxes(const std::string& descriptors, const std::vector<Place>& places, int elem_size) : places_(places), elem_size_(elem_size) {
    if (descriptors.size() != places.size() * sizeof(ddl_box_t)) throw std::invalid_argument("Boxes: descriptors and places disagree");
    boxes_.resize(places.size());
    if (!places.empty()) memcpy(boxes_.data(), descriptors.data(), descriptors.size());
    for (const Place& p : places) {
        if (std::get<0>(p) >= bases_) bases_ = std::get<0>(p) + 1;
        if (std::get<2>(p) >= bases_) bases_ = std::get<2>(p) + 1;
    }
}

void Boxes::run(const std::vector<int64_t>& bases, int op, int dtype) const {
    if (boxes_.empty()) return;
    if (bases.size() < bases_) throw std::invalid_argument("Boxes: too few base addresses");
    std::vector<ddl_box_t> boxes(boxes_);
    for (size_t i = 0; i < boxes.size(); ++i) {
        boxes[i].src = reinterpret_cast<const void*>(bases[std::get<0>(places_[i])] + std::get<1>(places_[i]));
        boxes[i].dst = reinterpret_cast<void*>(bases[std::get<2>(places_[i])] + std::get<3>(places_[i]));
    }
    check(ddl_copy_boxes(boxes.data(), static_cast<int>(boxes.size()), elem_size_, op, dtype, current_stream()), "ddl_copy_boxes");
}

// The sum over the sources, in order, of elements [start, start + extent) along `axis`, each divided first.
static MaybeTensor sum_slab(const std::vector<Tensor>& srcs, int64_t axis, int64_t start, int64_t extent, double divisor) {
    if (srcs.empty() || srcs.size() > 64) return std::nullopt;
    const Tensor& first = srcs[0];
    const int dt = sum_code(first), nd = static_cast<int>(first.dim());
    if (!dt || nd < 1 || nd > DDL_MAX_DIMS || axis < 0 || axis >= nd || start < 0 || extent < 1 || start + extent > first.size(axis) || first.numel() == 0)
        return std::nullopt;
    ddl_box_t box{};
    box.ndim = nd;
    auto shape = first.sizes().vec();
    shape[axis] = extent;
    int64_t run = 1;
    for (int d = nd - 1; d >= 0; --d) {
        box.shape[d] = shape[d], box.src_stride[d] = first.stride(d), box.dst_stride[d] = run;
        run *= shape[d];
    }
    std::vector<const void*> ptrs;
    for (const Tensor& t : srcs) {
        if (!plain(t) || t.scalar_type() != first.scalar_type() || t.sizes() != first.sizes() || t.strides() != first.strides()) return std::nullopt;
        ptrs.push_back(static_cast<const char*>(t.data_ptr()) + start * first.stride(axis) * first.element_size());
        if ((reinterpret_cast<intptr_t>(ptrs.back()) - reinterpret_cast<intptr_t>(ptrs[0])) % 16 != 0) return std::nullopt;
    }
    Tensor out = at::empty(shape, first.options());
    box.dst = out.data_ptr();
    check(ddl_sum_boxes(&box, ptrs.data(), static_cast<int>(ptrs.size()), static_cast<int>(first.element_size()), dt, divisor, current_stream()),
          "ddl_sum_boxes");
    return out;
}

// The pieces joined along `axis`.
static MaybeTensor join(const Tensor& local, const std::vector<Tensor>& parts, int64_t axis) {
    const int nd = static_cast<int>(local.dim());
    if (parts.empty() || nd < 1 || nd > DDL_MAX_DIMS || axis < 0 || axis >= nd || !local.is_cuda()) return std::nullopt;
    auto shape = local.sizes().vec();
    shape[axis] = 0;
    for (const Tensor& t : parts) {
        if (!plain(t) || t.scalar_type() != local.scalar_type() || t.dim() != nd || t.numel() == 0) return std::nullopt;
        for (int d = 0; d < nd; ++d)
            if (d != axis && t.size(d) != local.size(d)) return std::nullopt;
        shape[axis] += t.size(axis);
    }
    Tensor out = at::empty(shape, local.options());
    std::vector<ddl_box_t> boxes(parts.size());
    int64_t start = 0;
    for (size_t q = 0; q < parts.size(); ++q) {
        ddl_box_t& box = boxes[q];
        box = ddl_box_t{};
        box.ndim = nd;
        for (int d = 0; d < nd; ++d) box.shape[d] = parts[q].size(d), box.dst_stride[d] = out.stride(d);
        int64_t run = 1;
        for (int d = nd - 1; d >= 0; --d) {
            box.src_stride[d] = run;
            run *= box.shape[d];
        }
        box.src = parts[q].data_ptr();
        box.dst = static_cast<char*>(out.data_ptr()) + start * out.stride(axis) * out.element_size();
        start += parts[q].size(axis);
    }
    check(ddl_copy_boxes(boxes.data(), static_cast<int>(boxes.size()), static_cast<int>(out.element_size()), DDL_OP_COPY, DDL_DT_BITS, current_stream()),
          "ddl_copy_boxes");
    return out;
}

}  // namespace ddl_front

PYBIND11_MODULE(_front, m) {
    namespace py = pybind11;
    using namespace ddl_front;
    typedef py::call_guard<py::gil_scoped_release> unlocked;
    // as hip_ops has them: the weight as a matrix, its bias as a vector
    m.def("linear", [](const Tensor& x, const Tensor& w, const MaybeTensor& bias) { return w.dim() == 2 ? product(x, w, bias) : std::nullopt; }, unlocked());
    m.def("linear_backward",
          [](const Tensor& x, const Tensor& w, const Tensor& dy, bool need_x, bool need_w, bool need_b) -> std::optional<std::tuple<Tensor, Tensor, Tensor>> {
              if (w.dim() != 2) return std::nullopt;
              return product_backward(x, w, dy, need_x, need_w, need_b ? MaybeShape(std::vector<int64_t>{w.size(0)}) : std::nullopt);
          },
          unlocked());
    m.def("layer_norm", &layer_norm, unlocked());
    m.def("ln_backward_whole", &ln_backward_whole, unlocked());
    m.def("ln_backward_partial_params", &ln_backward_partial_params, unlocked());
    m.def("ln_backward_input_params", &ln_backward_input_params, unlocked());
    m.def("embedding_gather", &embedding_gather, unlocked());
    m.def("embedding_backward", &embedding_backward, unlocked());
    m.def("sum_slab", &sum_slab, unlocked());
    m.def("join", &join, unlocked());
    py::class_<Boxes, std::shared_ptr<Boxes>>(m, "Boxes")
        .def(py::init([](const py::bytes& descriptors, const std::vector<Boxes::Place>& places, int elem_size) {
            return new Boxes(static_cast<std::string>(descriptors), places, elem_size);
        }))
        .def("run", &Boxes::run, unlocked());
    define_nodes(m);
}
