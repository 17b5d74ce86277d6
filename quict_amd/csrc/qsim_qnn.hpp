// What a context keeps for its batches of variational circuits (qs_qnn_batch): a
// stream (inputs and outputs are in host memory, so nothing orders it with the
// caller's), buffers that grow on demand and are given back with the context, and the
// planned programs.  One batch at a time.
#pragma once
#include "qsim_sweep.hpp"

#include <map>
#include <mutex>

namespace qs {

constexpr int QNN_MAX_W = 20;

struct QnnState {
  std::mutex mu;
  hipStream_t stream = nullptr;
  char* dev = nullptr;
  char* host = nullptr;  // pinned
  uint64_t dev_bytes = 0, host_bytes = 0;
  std::map<std::pair<int, int>, VarImage> images;  // (width, layers)

  int open(int device);
  // At least these bytes; QS_ERR_UNSUPPORTED if the device has not so much to give.
  int room(uint64_t dev_need, uint64_t host_need);
};

}  // namespace qs
