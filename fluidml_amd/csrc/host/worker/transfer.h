// Arguments of a run between the caller's arrays and HBM, through pinned host memory that stays with the plan.
#ifndef FLUIDML_AMD_HOST_WORKER_TRANSFER_H_
#define FLUIDML_AMD_HOST_WORKER_TRANSFER_H_

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace fluidml {
namespace worker {

class Transfer {
 public:
  // One argument: its device buffer and its size.  The device buffer is readable and writable up to the next multiple
  // of 256 bytes (fluidml_hip_arena_create pads that far).
  struct Slot {
    void *device = nullptr;
    size_t bytes = 0;
    size_t offset = 0;  // in the pinned memory of its direction
  };

  // Allocates the pinned memory; throws std::runtime_error on HIP errors.
  Transfer(std::vector<Slot> &&inputs, std::vector<Slot> &&outputs);
  ~Transfer();
  Transfer(const Transfer &) = delete;

  // Copies host[i] into the device buffer of input i on `stream`.  The host arrays may be changed as soon as it returns.
  void In(const std::vector<const void *> &host, void *stream);
  // Copies the device buffer of output i into host[i] once everything issued on `stream` before is done, and returns
  // when all of it is there: the nanoseconds from the end of the last In on that stream to the start of this copy.
  double Out(const std::vector<void *> &host, void *stream);

 private:
  void Release();

  class InJob;
  class OutJob;

  std::vector<Slot> inputs_, outputs_;
  size_t in_bytes_ = 0, out_bytes_ = 0, out_slice_ = 0;
  char *in_ = nullptr, *out_ = nullptr;
  // host: kFlagBase bytes with the elapsed ticks, then one flag per outbound slice
  char *mailbox_ = nullptr;
  uint64_t *clock_ = nullptr;     // device
  uint32_t *counters_ = nullptr;  // device: one per outbound slice and one per outbound launch
  uint32_t value_ = 0;
  double wait_ns_ = 0;  // from queueing the last outbound copy to its first flag
  double ns_per_tick_ = 10.0;
};

}  // namespace worker
}  // namespace fluidml

#endif
