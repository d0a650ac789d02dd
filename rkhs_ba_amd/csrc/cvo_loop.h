// The resident iteration loop's launch interface (cvo_loop.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "cvo_internal.h"

namespace cvo {

constexpr int kMaxLoopDevices = 64;
constexpr size_t kLoopMaxLds = 128 * 1024;  // dynamic LDS of a block, beside up to 8 KB of static LDS

// Arguments of a launch, in device memory.
struct LoopArgs {
  KConsts kc;
  AssocProblem prob[3];  // the registration; adaptive lengthscale: and its two self problems
  int32_t rows;          // LDS rows of a block
  int32_t max_iters;     // iterations of this launch
  uint32_t tag0;         // tag of its first iteration (never 0, never used before on these words)
  uint32_t* fail;        // set when a wait ran out
  uint64_t* xa;          // words of the two exchanges
  uint64_t* xb;
  uint64_t wait_ticks;   // longest wait of an exchange, in ticks of the 100 MHz clock
};

struct LoopShape {
  int blocks = 0, rows = 0;
  size_t lds = 0;
};

// The compute units a resident launch holds until the object goes.
struct LoopUnits {
  int device = 0, n = 0;
  ~LoopUnits();
  bool claim(int dev, int blocks, int units);
};

size_t loop_words_bytes();
uint64_t* loop_step_words(uint64_t* words);  // the step exchange's part of them
// Shape of a launch over problems of rows[q] source rows; false where the loop
// does not take them.
bool loop_shape(const KConsts& kc, const int* rows, int n_probs, int units, LoopShape* out);
hipError_t launch_loop(const LoopArgs* a, const KConsts& kc, const LoopShape& s, hipStream_t st);

}  // namespace cvo
