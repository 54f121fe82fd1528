// Router top-k (+ routing mask and merge probs), one wavefront per row; the
// per-row routine and its math citation are in topk_device.h.
#include <type_traits>

#include "topk_device.h"

namespace moe {
namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / kWave;

template <int kEPL, bool kSorted>
__global__ __launch_bounds__(kThreads) void topk_kernel(const float *logits, int64_t T, int E, int k,
                                                        float *values, int64_t *indices,
                                                        uint8_t *routing_map, float *probs) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + threadIdx.x / kWave;
  if (t >= T) return;
  const float *row = logits + t * E;
  topk_row<kEPL, kSorted>([&](int e) { return row[e]; }, t, E, k, values, indices, routing_map, probs);
}

// go(n, sorted) with the slots per lane that E experts need (n = 64-element pieces, 16 above 512 experts).
template <typename Go>
void by_slots(int E, bool searched, Go go) {
  const std::true_type sorted{};
  const std::false_type unsorted{};
  switch ((E + kWave - 1) / kWave) {
    case 1: go(std::integral_constant<int, 1>{}, sorted); break;
    case 2: go(std::integral_constant<int, 2>{}, sorted); break;
    case 3: go(std::integral_constant<int, 3>{}, sorted); break;
    case 4: go(std::integral_constant<int, 4>{}, sorted); break;
    case 5: go(std::integral_constant<int, 5>{}, sorted); break;
    case 6: searched ? go(std::integral_constant<int, 6>{}, unsorted) : go(std::integral_constant<int, 6>{}, sorted); break;
    case 7: searched ? go(std::integral_constant<int, 7>{}, unsorted) : go(std::integral_constant<int, 7>{}, sorted); break;
    case 8: searched ? go(std::integral_constant<int, 8>{}, unsorted) : go(std::integral_constant<int, 8>{}, sorted); break;
    default: go(std::integral_constant<int, 16>{}, unsorted); break;
  }
}

}  // namespace
}  // namespace moe

extern "C" {

int moe_topk(const float *logits, int64_t T, int64_t E, int64_t k, float *values, int64_t *indices,
             uint8_t *routing_map, float *probs, void *stream) {
  using namespace moe;
  if (T < 0 || E < 0) return fail(MOE_ERR_SHAPE, "moe_topk: negative size (T=%lld E=%lld)", (long long)T, (long long)E);
  if (k < 1 || k > E) return fail(MOE_ERR_SHAPE, "moe_topk: k=%lld out of range for E=%lld", (long long)k, (long long)E);
  if (k > 64) return fail(MOE_ERR_CAPACITY, "moe_topk: k=%lld exceeds the 64 supported", (long long)k);
  if (E > 1024) return fail(MOE_ERR_CAPACITY, "moe_topk: E=%lld exceeds the 1024 supported", (long long)E);
  if (T == 0) return MOE_OK;
  if (logits == nullptr || values == nullptr || indices == nullptr) {
    return fail(MOE_ERR_INVALID_ARG, "moe_topk: null logits, values or indices");
  }
  const int64_t grid = ceil_div(T, kWavesPerBlock);
  if (grid > 0x7fffffff) return fail(MOE_ERR_CAPACITY, "moe_topk: T=%lld too large", (long long)T);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int e = static_cast<int>(E), kk = static_cast<int>(k);
  auto go = [&](auto epl, auto sorted) {
    topk_kernel<decltype(epl)::value, decltype(sorted)::value><<<dim3(grid), dim3(kThreads), 0, s>>>(logits, T, e, kk, values, indices, routing_map, probs);
  };
  by_slots(e, topk_searches(T, k), go);
  return check_launch("moe_topk");
}

}  // extern "C"
