// Tail splitting: which items of a launch are cut into parts (see SplitPlan in fba_kernels.h).
#include <cstdlib>
#include <mutex>

#include "fba_kernels.h"

namespace fba {

namespace {

// Compute units of the current device (looked up once per device).
int compute_units() {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static int cache[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  std::lock_guard<std::mutex> lock(mu);
  if (cache[dev] == 0) {
    int n = 0;
    cache[dev] = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
  }
  return cache[dev];
}

}  // namespace

int device_compute_units() { return compute_units(); }

namespace {
constexpr int kQueueBytes = 256;
__global__ void queue_reset_kernel(int* queue) { queue[threadIdx.x] = 0; }
}  // namespace

bool claims_wanted(int items_per_xcd, int total_work, int wgs_per_cu) {
  const char* e = getenv("FBA_CLAIM_WORK");
  const bool off = e != nullptr && e[0] == '0';
  (void)items_per_xcd;  // either mapping deals grid index i to XCD i % 8, which is all a claim relies on
  return !off && total_work >= 4 * compute_units() * wgs_per_cu;
}

int* work_queue_in(void* ws, int64_t ws_bytes, int64_t partial_bytes) {
  if (ws == nullptr) return nullptr;
  const int64_t off = (ws_bytes - kQueueBytes) & ~(int64_t)15;
  if (off < partial_bytes) return nullptr;
  return reinterpret_cast<int*>(static_cast<char*>(ws) + off);
}

hipError_t launch_queue_reset(int* queue, hipStream_t stream) {
  hipLaunchKernelGGL(queue_reset_kernel, dim3(1), dim3(kQueueBytes / 4), 0, stream, queue);
  return hipGetLastError();
}

// The hardware hands work-groups to free slots in index order.  With n items on s slots the last n % s items form a
// partial round; when that round would fill at most half of the slots, each of its items is cut into up to floor(s / (n % s))
// parts (at most 8), so that the parts fill the slots once and take 1 / parts of a round.  Launches smaller than the
// machine (n < s) are split the same way.
//
// How many parts pay: every part writes its partial results, and the merge reads them back, so with m items of at most
// max_steps steps each the round takes about  max_steps step_cost / parts + m parts  in units of what one part's results
// cost, least at parts = sqrt(max_steps step_cost / m).  The lists are on the device: step_cost assumes that 40 % of the
// longest possible list is there.  One part's 64 KiB cost 27 ns at what the stores and the merge sustain (2.4 TB/s) and a
// forward step of such a round 0.65 us, so forward has step_cost 9.  Measured, forward / backward in us (always as many
// parts as slots allow, against this rule): B1 H8 S768, 128-token blocks, half kept 22.0 / 54.9 -> 15.8 / 43.0; H4 S1536
// 23.9 / 58.5 -> 19.8 / 54.7; H8 S4096, a quarter kept 43.2 / 104.8 -> 37.0 / 92.9.
SplitPlan plan_split(int num_items, int wgs_per_cu, int max_steps, double step_cost, int64_t slot_bytes, void* ws, int64_t ws_bytes) {
  SplitPlan plan{nullptr, num_items, 1, 0};
  if (ws == nullptr || num_items <= 0) return plan;
  int slots = compute_units() * wgs_per_cu;
  if (slots > kSplitMaxSlots) slots = kSplitMaxSlots;
  const int rest = num_items % slots;
  if (rest == 0 || 2 * rest > slots) return plan;
  int parts = slots / rest;
  if (parts > 8) parts = 8;
  const double whole = max_steps * step_cost;
  while (parts >= 2 && (double)parts * parts * rest > whole) --parts;
  while (parts >= 2 && (int64_t)rest * parts * slot_bytes > ws_bytes) --parts;
  if (parts < 2 || whole / parts + (double)rest * parts > 0.9 * whole) return plan;
  plan.ws = static_cast<float*>(ws);
  plan.first = num_items - rest;
  plan.parts = parts;
  return plan;
}

}  // namespace fba
