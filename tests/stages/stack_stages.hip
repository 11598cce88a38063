// stack_stages.hip -- the traversal's per-lane stack (LaneStack) step by step,
// for tests: a wave of lanes with the same entries takes one inner step.
#include "../../rendiation_amd/csrc/trace_device.h"

namespace {

using namespace rdrt;

// Lane l starts with sp[l] entries, entry i being 100 + i, takes a step whose
// node has kids[l] hit children 1, 2, 3, 4 (farthest first) and writes sp, the
// step's result, then its entries.
template <int K, int S, int LAYOUT>
__global__ __launch_bounds__(64) void k_stack(const uint32_t *sp, const uint32_t *kids, uint32_t *status,
                                              uint32_t *out, uint32_t words) {
  using Stack = LaneStack<K, S, 64>;
  __shared__ uint32_t lds[Stack::kRows * 64];
  volatile uint32_t spill[Stack::kSpill];
  const uint32_t lane = threadIdx.x, n = kids[lane];
  Stack stk{lds + lane, spill, status + lane, 0u};
  for (uint32_t i = 0; i < sp[lane]; i++) stk.push(100u + i);
  const uint32_t ref = stk.template step<LAYOUT>([&]() { return Kids{n, {1u, 2u, 3u, 4u}}; });
  uint32_t *o = out + (size_t)lane * words;
  o[0] = stk.sp;
  o[1] = ref;
  for (uint32_t i = 0; i < stk.sp && i + 2u < words; i++) o[2 + i] = stk.get(i);
}

template <int K, int S>
hipError_t launch(uint32_t layout, const uint32_t *sp, const uint32_t *kids, uint32_t *status, uint32_t *out,
                  uint32_t words) {
  if (layout == 0) hipLaunchKernelGGL((k_stack<K, S, 0>), dim3(1), dim3(64), 0, 0, sp, kids, status, out, words);
  else hipLaunchKernelGGL((k_stack<K, S, 1>), dim3(1), dim3(64), 0, 0, sp, kids, status, out, words);
  return hipGetLastError();
}

}  // namespace

// The arrays hold 64 values each, `out` 64 * words.
extern "C" int stack_step(uint32_t lds, uint32_t entries, uint32_t layout, const uint32_t *sp, const uint32_t *kids,
                          uint32_t *status, uint32_t *out, uint32_t words) {
  if (lds == 8 && entries == 8) return (int)launch<8, 8>(layout, sp, kids, status, out, words);
  if (lds == 16 && entries == 16) return (int)launch<16, 16>(layout, sp, kids, status, out, words);
  if (lds == 8 && entries == 24) return (int)launch<8, 24>(layout, sp, kids, status, out, words);
  if (lds == 16 && entries == 48) return (int)launch<16, 48>(layout, sp, kids, status, out, words);
  return (int)hipErrorInvalidValue;
}
