// torch.ops.llmopt.w4a16_linear's kernel for ROCm tensors: the calls that every step of a program makes (contiguous half
// tensors of matching shapes on one device) go from torch's dispatcher to llmopt_hip_launch here.  Everything else - arguments to
// refuse, tensors to lay out anew, empty results, a device's first call, a launch that fails - is the business of
// llmopt::w4a16_linear_general, the same operator in Python, which also says what is wrong.
//
// One token of a small model, 1 x 576 x 1536, is a kernel of 4.7 us, and the checks, the output and the launch took 12.1 us a
// call in Python.
#include <ATen/Functions.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <array>
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <limits>
#include <mutex>
#include <optional>
#include <shared_mutex>

namespace {

using Launch = int (*)(void *library, const char *name, void *const *pointers, const size_t *lengths, uint32_t count,
                       const void *parameters, uint32_t parameter_bytes, void *hip_stream);

constexpr int64_t kGroup = 64;
std::atomic<Launch> launch{nullptr};
std::array<std::atomic<void *>, 64> libraries{};  // by device: a context's library, while there is one
std::shared_mutex in_use;                         // shared: a library is being launched from; alone: one comes or goes

bool plain(const at::Tensor &t, at::ScalarType type, c10::Device device) {
  return t.scalar_type() == type && t.device() == device && t.is_contiguous();
}

at::Tensor general(const at::Tensor &input, const at::Tensor &packed, const at::Tensor &scale, const std::optional<at::Tensor> &bias) {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("llmopt::w4a16_linear_general", "")
                             .typed<at::Tensor(const at::Tensor &, const at::Tensor &, const at::Tensor &,
                                               const std::optional<at::Tensor> &)>();
  return op.call(input, packed, scale, bias);
}

at::Tensor w4a16_linear(const at::Tensor &input, const at::Tensor &packed, const at::Tensor &scale,
                        const std::optional<at::Tensor> &bias) {
  const c10::Device device = input.device();
  const int index = device.index();
  if (index < 0 || index >= (int)libraries.size() || libraries[index].load(std::memory_order_relaxed) == nullptr)
    return general(input, packed, scale, bias);
  if (input.dim() == 0 || packed.dim() != 2 || scale.dim() != 2 || !plain(input, at::kHalf, device) ||
      !plain(packed, at::kByte, device) || !plain(scale, at::kHalf, device) || (bias && !plain(*bias, at::kHalf, device)))
    return general(input, packed, scale, bias);
  const int64_t n = packed.size(0), k = packed.size(1) * 2, limit = std::numeric_limits<uint32_t>::max();
  if (n == 0 || k == 0 || k % kGroup != 0 || input.size(-1) != k || scale.size(0) != n || scale.size(1) != k / kGroup ||
      (bias && bias->numel() != n) || n > limit || k > limit || input.numel() == 0 || input.numel() / k > limit)
    return general(input, packed, scale, bias);
  const int64_t m = input.numel() / k;
  c10::SmallVector<int64_t, 5> shape(input.sizes().begin(), input.sizes().end());
  shape.back() = n;
  const at::Tensor output = at::empty(shape, input.options());
  const at::Tensor &addend = bias ? *bias : scale;
  void *const pointers[] = {const_cast<void *>(input.const_data_ptr()), const_cast<void *>(packed.const_data_ptr()),
                            const_cast<void *>(scale.const_data_ptr()), const_cast<void *>(addend.const_data_ptr()),
                            output.mutable_data_ptr()};
  const size_t lengths[] = {input.nbytes(), packed.nbytes(), scale.nbytes(), addend.nbytes(), output.nbytes()};
  const uint32_t parameters[] = {(uint32_t)m, (uint32_t)n, (uint32_t)k, bias ? 1u : 0u, 0u};  // rows, columns, k, bias, its stride
  // queued on torch's stream; the tensors outlive the launch call
  int status = -1;
  {
    std::shared_lock<std::shared_mutex> held(in_use);
    if (void *library = libraries[index].load(std::memory_order_relaxed))  // (another thread may have closed it meanwhile)
      status = launch.load(std::memory_order_relaxed)(
          library, m == 1 ? "llmopt_w4a16_linear_f16_g64" : "llmopt_w4a16_linear_f16_g64_m4", pointers, lengths, 5, parameters,
          sizeof(parameters), c10::hip::getCurrentHIPStream(index).stream());
  }
  return status < 0 ? general(input, packed, scale, bias) : output;
}

TORCH_LIBRARY_IMPL(llmopt, CUDA, m) { m.impl("w4a16_linear", w4a16_linear); }  // (ROCm tensors carry the CUDA dispatch key)

}  // namespace

// From here on calls on `device` go to `library` through `function` (llmopt_hip_launch); without a library they go to Python, and
// no launch from the former one is under way any more.
extern "C" __attribute__((visibility("default"))) void llmopt_torch_bind(int device, void *library, void *function) {
  if (device < 0 || device >= (int)libraries.size()) return;
  std::unique_lock<std::shared_mutex> alone(in_use);
  if (library != nullptr) launch.store(reinterpret_cast<Launch>(function), std::memory_order_relaxed);
  libraries[device].store(library, std::memory_order_relaxed);
}
