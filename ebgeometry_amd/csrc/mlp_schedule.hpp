// The steps that train the bound network and the rows and partial gradients each of them touches, for the
// trainer and for the host check of its launches.
#pragma once

#include <algorithm>
#include <cstdint>
#include <string>

namespace ebgpu {

constexpr int kTrainRows = 64;  // rows per tile
constexpr int kTrainBlk  = 128; // most workgroups of a step (each strides over tiles)

// Workgroups, hence partial gradients, of a step of `rows` rows.
inline int mlp_train_blocks(int rows) { return std::min((rows + kTrainRows - 1) / kTrainRows, kTrainBlk); }

// An epoch over n samples: step k takes `rows` samples from `first` on.
struct TrainStep
{
  uint64_t first;
  int      rows;
};
inline uint64_t  train_steps(uint64_t n, int batch) { return (n + uint64_t(batch) - 1) / uint64_t(batch); }
inline TrainStep train_step(uint64_t n, int batch, uint64_t k)
{
  const uint64_t first = k * uint64_t(batch);
  return {first, int(std::min<uint64_t>(uint64_t(batch), n - first))};
}

// Whether a step of `rows` rows keeps within its arrays: `samples` points and targets from the step's
// first on, `partials` partial gradients. The kernel reads every row below `rows` and no other; each of
// its workgroups writes one partial gradient, and the update sums them. On failure *why (nullable) says
// what does not fit.
inline bool check_train_step(int rows, uint64_t samples, uint64_t partials, std::string* why)
{
  const char* w = nullptr;
  if (rows < 1) w = "empty training batch";
  else if (uint64_t(rows) > samples) w = "training batch reaches past the samples";
  else if (uint64_t(mlp_train_blocks(rows)) > partials) w = "training batch larger than its buffers";
  if (w && why) *why = w;
  return !w;
}

// The same for the epochs over n samples in batches of `batch`, for arrays of `samples` rows and
// `partials` partial gradients: the steps (all but the last are alike) follow each other, end at n, and
// keep within the arrays.
inline bool check_train_schedule(uint64_t n, int batch, uint64_t samples, uint64_t partials, std::string* why)
{
  const uint64_t steps = batch < 1 ? 0 : train_steps(n, batch);
  if (steps < 1) {
    if (why) *why = "no training steps";
    return false;
  }
  for (const uint64_t k : {uint64_t(0), steps - 1}) {
    const TrainStep t = train_step(n, batch, k);
    if (t.rows > batch || t.first + uint64_t(t.rows) != std::min(n, (k + 1) * uint64_t(batch)) || t.first > samples) {
      if (why) *why = "training steps do not cover the samples";
      return false;
    }
    if (!check_train_step(t.rows, samples - t.first, partials, why)) return false;
  }
  return true;
}

} // namespace ebgpu
