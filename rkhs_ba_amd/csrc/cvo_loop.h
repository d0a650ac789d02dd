// The resident iteration loop's launch interface (cvo_loop.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "cvo_internal.h"

namespace cvo {

constexpr int kMaxLoopDevices = 64;
constexpr size_t kLoopMaxLds = 128 * 1024;  // dynamic LDS of a block, beside up to 8 KB of static LDS

// Arguments of the launches of one shape, in device memory.
struct LoopArgs {
  KConsts kc;
  AssocProblem prob[3];  // the registration; adaptive lengthscale: and its two self problems
  int32_t rows;          // LDS rows of a block
  int32_t max_iters;     // iterations of a launch
  uint32_t* flags;       // [0] set when a wait ran out, [1] the registration is done
  uint64_t* xa;          // words of the two exchanges
  uint64_t* xb;
  uint64_t wait_ticks;   // longest wait of an exchange, in ticks of the 100 MHz clock
};

struct LoopShape {
  int blocks = 0, rows = 0;
  size_t lds = 0;
};

// A call that uses the device, counted while the object lives (once a context).
class ActiveCall {
 public:
  explicit ActiveCall(cvo_ctx* ctx);
  ~ActiveCall();

 private:
  cvo_ctx* ctx_;
};

// Blocks that a resident launch may have of a device's units: all of them for the
// process's only call, an equal part beside others; 0 where that is too small.
int loop_share(int dev, int units);

// The compute units a resident launch holds until the object goes.
class LoopUnits {
 public:
  ~LoopUnits();
  // Waits up to wait_ms for other launches to give units back.
  bool claim(int dev, int blocks, int units, int wait_ms);

 private:
  int device_ = 0, n_ = 0;
};

size_t loop_words_bytes();
uint64_t* loop_step_words(uint64_t* words);  // the step exchange's part of them
// Shape of a launch over problems of rows[q] source rows; false where the loop
// does not take them.
bool loop_shape(const KConsts& kc, const int* rows, int n_probs, int units, LoopShape* out);
hipError_t launch_loop(const LoopArgs* a, const KConsts& kc, const LoopShape& s, hipStream_t st);

}  // namespace cvo
