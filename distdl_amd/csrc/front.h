// Tensor front ends of the entry points (front.cpp) and what the autograd nodes
// (front_nodes.cpp) use of them.
#ifndef DDL_FRONT_H
#define DDL_FRONT_H
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <memory>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/distdl_hip.h"

namespace ddl_front {

using at::Tensor;
typedef std::optional<Tensor> MaybeTensor;
typedef std::optional<std::vector<int64_t>> MaybeShape;   // of a parameter's gradient, if that is wanted

inline void check(int rc, const char* what) {
    if (rc != 0) throw std::runtime_error(std::string(what) + " failed with code " + std::to_string(rc) + ": " + ddl_last_error());
}
inline void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }
inline bool plain(const Tensor& t) { return t.is_cuda() && t.is_contiguous(); }
inline bool multiple(const void* p, int64_t bytes) { return reinterpret_cast<uintptr_t>(p) % bytes == 0; }
inline const void* pointer(const MaybeTensor& t) { return t ? t->data_ptr() : nullptr; }
inline void* pointer(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
int float_code(const Tensor& t);   // 0: none of the three

// Every one of these answers nothing to forms that it does not take, see front.cpp.
MaybeTensor product(const Tensor& x, const Tensor& w, const MaybeTensor& bias);
std::optional<std::tuple<Tensor, Tensor, Tensor>> product_backward(const Tensor& x, const Tensor& w, const Tensor& dy, bool need_x, bool need_w,
                                                                  const MaybeShape& bias_shape);
typedef std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> Normalized;   // y, the rows as [rows, cols], mean, rstd, gamma as [cols]
std::optional<Normalized> layer_norm(const Tensor& x, const MaybeTensor& gamma, const MaybeTensor& beta, int64_t cols, double eps);
std::optional<std::tuple<Tensor, Tensor, Tensor>> ln_backward_whole(const Tensor& dy, const Tensor& x2d, const Tensor& mean, const Tensor& rstd,
                                                                    const MaybeTensor& gamma, const MaybeShape& gamma_shape, const MaybeShape& beta_shape);
std::optional<std::tuple<Tensor, Tensor>> ln_backward_partial_params(const Tensor& dy, const Tensor& x2d, const Tensor& mean, const Tensor& rstd,
                                                                     const MaybeTensor& gamma);
std::optional<std::tuple<Tensor, Tensor, Tensor>> ln_backward_input_params(const Tensor& dy, const Tensor& x2d, const Tensor& mean, const Tensor& rstd,
                                                                           const MaybeTensor& gamma, const Tensor& part_sums, double weight,
                                                                           const Tensor& work, const MaybeShape& gamma_shape, const MaybeShape& beta_shape);
MaybeTensor embedding_gather(const Tensor& weight, const Tensor& ids, int64_t lo, int64_t hi);
MaybeTensor embedding_backward(const Tensor& dy, const Tensor& ids, int64_t lo, int64_t hi, int64_t padding_idx, bool by_freq);

// The boxes of one launch with everything but the base addresses: a call adds those
// of the slots.  Calls only read the object.
class Boxes {
public:
    typedef std::tuple<size_t, int64_t, size_t, int64_t> Place;   // source slot and byte offset, destination slot and byte offset
    // descriptors: ddl_box_t after ddl_box_t, without the pointers.
    Boxes(const std::string& descriptors, const std::vector<Place>& places, int elem_size);
    void run(const std::vector<int64_t>& bases, int op, int dtype) const;

private:
    std::vector<ddl_box_t> boxes_;
    std::vector<Place> places_;
    size_t bases_ = 0;
    int elem_size_;
};

void define_nodes(pybind11::module_& m);   // front_nodes.cpp

}  // namespace ddl_front
#endif  // DDL_FRONT_H
