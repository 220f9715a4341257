// Device state to host arrays: one packing kernel, staged copies, and for large
// states several host threads, each filling its part of the caller's arrays
// while the next parts are on their way.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <vector>

#include "beads_amd.h"
#include "common.hpp"
#include "real.hpp"

namespace beads_amd {

// The per-atom device arrays of one system (null tag / molid: not available).
struct StateSource {
  uint32_t n = 0;
  const real4* pos = nullptr;
  const real4* vel = nullptr;
  const real4* force = nullptr;
  const int4* image = nullptr;
  const uint32_t* tag = nullptr;
  const uint32_t* molid = nullptr;
};

class StateReader {
 public:
  StateReader() = default;
  ~StateReader();
  StateReader(const StateReader&) = delete;
  StateReader& operator=(const StateReader&) = delete;

  // Fills the non-null arrays of out in the stream's order; they are complete
  // on return.
  void read(const StateSource& src, const beads_state_out_t& out, hipStream_t stream);

 private:
  struct Field {  // bytes [offset, offset + size) of the staged state go to dst
    size_t offset, size;
    unsigned char* dst;
  };
  static void deliver(const std::vector<Field>& fields, const unsigned char* bytes, size_t offset,
                      size_t size);
  void deliver_in_chunks(const std::vector<Field>& fields, size_t total, hipStream_t stream);

  DeviceBuffer<unsigned char> stage_;
  PinnedBuffer<unsigned char> host_;
  std::vector<hipEvent_t> events_;
};

}  // namespace beads_amd
