// The small-convolution kernel (conv_mini.hip) as the other families see it: which configurations run a problem and
// what each is expected to take. The FP32 family sends its small problems there (f32_family.cpp).
#pragma once

#include "gpu_inference/conv2d.h"

namespace gie {

// Modeled time (us, without dispatch) of configuration `config` on `cus` CUs.
double mini_busy_us(int config, const ConvProblem& prob, int cus);
// The configuration expected to be fastest for the problem, or -1 when none runs it; *us (optional): its time.
int mini_best_config(const ConvProblem& prob, int cus, double* us);
// Enqueues configuration `config` (mini_best_config has accepted the problem).
void mini_launch(int config, const ConvProblem& prob, const void* x, const void* w, const void* bias, void* y,
                 void* stream);

}  // namespace gie
