// Work on a second stream beside the first.
#pragma once

#include <hip/hip_runtime_api.h>

#include "pool.hpp"

namespace mxg {

// The second stream's work starts after what the first holds now; done() ends it
// and wait() makes the first stream wait for it. If an error unwinds in between,
// the first stream waits all the same: buffers that the caller then gives back are
// handed out again in the order of the first stream alone, while kernels on the
// second may still use them.
class Fork {
 public:
  Fork(hipStream_t first, hipStream_t second, hipEvent_t fork, hipEvent_t join) : first_(first), second_(second), join_(join) {
    check(hipEventRecord(fork, first_));
    check(hipStreamWaitEvent(second_, fork, 0));
  }
  ~Fork() {
    if (waited_) return;
    if (!done_) (void)hipEventRecord(join_, second_);
    (void)hipStreamWaitEvent(first_, join_, 0);
  }
  Fork(const Fork&) = delete;
  Fork& operator=(const Fork&) = delete;
  void done() {
    check(hipEventRecord(join_, second_));
    done_ = true;
  }
  void wait() {
    check(hipStreamWaitEvent(first_, join_, 0));
    waited_ = true;
  }

 private:
  static void check(hipError_t e) {
    if (e != hipSuccess) throw Error(MXG_ERR_HIP, std::string("stream fork failed: ") + hipGetErrorString(e));
  }
  hipStream_t first_, second_;
  hipEvent_t join_;
  bool done_ = false, waited_ = false;
};

}  // namespace mxg
