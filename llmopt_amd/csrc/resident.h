// The layers of a retained decode step as one resident launch (kernels/decode_resident.hip).
#pragma once

#include "kernels/kernels.h"
#include "runtime.h"

namespace llmopt {

// Records [first, first + count) of a plan are whole layers that one resident launch stands for.
struct ResidentRun {
  size_t first = 0, count = 0;
  ResidentArgs args = {};  // layers, hand, tag and failed unset
  std::vector<ResidentLayer> layers;
};

// The run of a list of records, if it has one: layers in the forms that a decode step is made of (the three launches of
// small batches, the five of larger ones), one behind the other on one stream of rows, of sizes that the kernel takes, whose
// buffers between the records are scratch (llmopt_hip_buffer_set_scratch) and not read outside the run, in a step that may run
// again from its first record after the resident launch gave up: no record writes what the step finds there and reads.
bool find_resident_run(const std::vector<DispatchRecord> &records, ResidentRun *out);

}  // namespace llmopt
