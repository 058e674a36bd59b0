// FP32 convolutions on the padded-NHWC kernels (conv_nhwc.hip), for the FP32 family to run in place of its own where they
// are expected to be faster.
#pragma once

#include "gpu_inference/kernel_registry.h"

namespace gie {

struct NhwcF32 {
  int config = -1;  // -1: no configuration takes the problem in `room` bytes of workspace
  int split = 1;
  double us = 0.0;  // expected time beyond two dispatches
};

// The fastest configuration and split for prob on `cus` CUs whose padded copies and partials fit `room` bytes.
NhwcF32 nhwc_f32_best(const ConvProblem& prob, int cus, size_t room);

// Runs it (stages 0: repack, 1: convolution, 2: reduce).
void nhwc_f32_launch(const NhwcF32& how, const LaunchArgs& la);

}  // namespace gie
