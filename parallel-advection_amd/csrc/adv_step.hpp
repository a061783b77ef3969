// One advection step of a whole array outside the executors' own kernels
// (adv_step.hip).
#pragma once

#include "common.hpp"

namespace bkma {

// Takes the step if a faster kernel covers the shape and the parameters
// (*done = true), with the executors' values.
bkma_status adv_step_whole(const AdvDev &p, bkma_dtype dt, void *data, hipStream_t s, bool *done);

}  // namespace bkma
