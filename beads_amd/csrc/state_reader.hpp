// Device state to host arrays: a packing kernel, staged copies, and for large
// states several host threads, each filling its part of the caller's arrays
// while the next parts are on their way.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>
#include <vector>

#include "beads_amd.h"
#include "common.hpp"
#include "real.hpp"

namespace beads_amd {

struct PackStateParams;

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
  StateReader();
  ~StateReader();
  StateReader(const StateReader&) = delete;
  StateReader& operator=(const StateReader&) = delete;

  // Fills the non-null arrays of out in the stream's order; they are complete
  // on return. Callable from several threads, one read at a time.
  void read(const StateSource& src, const beads_state_out_t& out, hipStream_t stream);

  // The most a read copies at once, the most it stages on the device, and the
  // size of a copy above the first.
  void set_sizes(size_t whole, size_t window, size_t piece);

 private:
  // A wanted field: its bytes per atom, the caller's array, and where the
  // packing kernel is told the field's place in a window.
  struct Field {
    size_t bytes;
    unsigned char* dst;
    uint64_t PackStateParams::* place;
  };
  // The atoms staged on the device together (the last window may hold fewer).
  struct Window {
    size_t first, count;
  };
  size_t reserve(size_t n, size_t per_atom);
  void pack(const std::vector<Field>& fields, PackStateParams p, Window w, hipStream_t stream);
  static void deliver(const std::vector<Field>& fields, Window w, const unsigned char* bytes,
                      size_t offset, size_t size);
  void read_windows(const std::vector<Field>& fields, const PackStateParams& p, size_t per_atom,
                    size_t window_atoms, hipStream_t stream);

  std::mutex mutex_;
  size_t whole_bytes_, window_bytes_, piece_bytes_;
  DeviceBuffer<unsigned char> stage_;
  PinnedBuffer<unsigned char> host_;
  std::vector<hipEvent_t> events_;
};

}  // namespace beads_amd
