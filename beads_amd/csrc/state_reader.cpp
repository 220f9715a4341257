#include "state_reader.hpp"

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <exception>
#include <system_error>
#include <thread>

#include "kernels.hpp"

namespace beads_amd {

namespace {

// States up to kWhole bytes come over in one copy; larger ones in kPiece pieces
// by up to kThreads threads with kSlots pieces in flight each, because what
// bounds them is not the link but the first touch of the caller's pages and the
// copy out of the staging memory, about 4 GB/s in one thread.
// The device stages a window of kWindow bytes at a time, so that a system that
// fills the card can still be read; where even that is not free, windows shrink
// down to kSmallest. One packing kernel a window: with one for each piece the
// stream goes back and forth between kernels and copies (1,000,000 atoms 3.1 ms
// against 2.7, 2,000,000 8.1 against 6.4).
constexpr size_t kPiece = size_t{1} << 20;
constexpr size_t kWhole = size_t{4} << 20;
constexpr size_t kWindow = size_t{16} << 20;
constexpr size_t kSmallest = size_t{1} << 14;
constexpr unsigned kThreads = 8;
constexpr unsigned kSlots = 2;

}  // namespace

StateReader::StateReader() : whole_bytes_(kWhole), window_bytes_(kWindow), piece_bytes_(kPiece) {}

StateReader::~StateReader() {
  for (auto& e : events_) (void)hipEventDestroy(e);
}

void StateReader::set_sizes(size_t whole, size_t window, size_t piece) {
  require(window >= kSmallest && piece > 0, "state windows hold at least " +
                                                std::to_string(kSmallest) + " bytes.");
  const std::lock_guard<std::mutex> lock(mutex_);
  whole_bytes_ = whole;
  window_bytes_ = window;
  piece_bytes_ = piece;
}

// Device memory for the windows of a state; the atoms that a window holds.
size_t StateReader::reserve(size_t n, size_t per_atom) {
  size_t bytes = std::min(n * per_atom, std::max(whole_bytes_, window_bytes_));
  for (;;) {
    try {
      stage_.resize(bytes);
      return bytes / per_atom;
    } catch (const Error&) {
      if (bytes / 2 < kSmallest) throw;
      (void)hipGetLastError();  // the exception has reported it
      bytes /= 2;
    }
  }
}

void StateReader::pack(const std::vector<Field>& fields, PackStateParams p, Window w,
                       hipStream_t stream) {
  p.first = static_cast<uint32_t>(w.first);
  p.n = static_cast<uint32_t>(w.count);
  p.out = stage_.data();
  size_t at = 0;
  for (const Field& f : fields) {
    p.*f.place = at;
    at += f.bytes * w.count;
  }
  launch_pack_state(p, stream);
  BEADS_HIP(hipGetLastError());
}

// Bytes [offset, offset + size) of a window to the caller's arrays.
void StateReader::deliver(const std::vector<Field>& fields, Window w, const unsigned char* bytes,
                          size_t offset, size_t size) {
  size_t at = 0;
  for (const Field& f : fields) {
    const size_t end = at + f.bytes * w.count;
    const size_t b = std::max(offset, at), e = std::min(offset + size, end);
    if (b < e) {
      std::memcpy(f.dst + f.bytes * w.first + (b - at), bytes + (b - offset), e - b);
    }
    at = end;
  }
}

void StateReader::read_windows(const std::vector<Field>& fields, const PackStateParams& p,
                               size_t per_atom, size_t window_atoms, hipStream_t stream) {
  const size_t n = p.n, piece = piece_bytes_;
  const size_t per_window = (window_atoms * per_atom + piece - 1) / piece;
  const size_t windows = (n + window_atoms - 1) / window_atoms;
  const size_t last = ((n - (windows - 1) * window_atoms) * per_atom + piece - 1) / piece;
  const size_t pieces = (windows - 1) * per_window + last;
  const unsigned cores = std::max(1u, std::thread::hardware_concurrency());
  const unsigned threads =
      static_cast<unsigned>(std::min<size_t>(std::min(kThreads, cores), (pieces + 1) / 2));
  host_.resize(static_cast<size_t>(threads) * kSlots * piece);
  while (events_.size() < static_cast<size_t>(threads) * kSlots) {
    hipEvent_t e;
    BEADS_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    events_.push_back(e);
  }
  int device = 0;
  BEADS_HIP(hipGetDevice(&device));
  size_t next = 0;
  bool failed = false;
  std::mutex next_mutex;
  std::exception_ptr error;
  auto window_of = [&](size_t k) {
    const size_t first = k / per_window * window_atoms;
    return Window{first, std::min(window_atoms, n - first)};
  };
  auto work = [&](unsigned t) {
    try {
      BEADS_HIP(hipSetDevice(device));
      struct {
        size_t k, offset, size;
      } in_slot[kSlots];
      // Takes the next piece and enqueues its copy, with the packing of its
      // window before the window's first: the pieces are enqueued in order, so
      // in the stream a window is packed after the one before has been copied.
      auto take = [&](unsigned s) {
        const std::lock_guard<std::mutex> lock(next_mutex);
        const size_t k = failed ? pieces : next++;
        in_slot[s].k = k;
        if (k >= pieces) return;
        const Window w = window_of(k);
        const size_t offset = k % per_window * piece;
        const size_t size = std::min(piece, w.count * per_atom - offset);
        in_slot[s].offset = offset;
        in_slot[s].size = size;
        failed = true;  // unless all of it succeeds
        if (offset == 0) pack(fields, p, w, stream);
        BEADS_HIP(hipMemcpyAsync(host_.data() + (t * kSlots + s) * piece, stage_.data() + offset,
                                 size, hipMemcpyDeviceToHost, stream));
        BEADS_HIP(hipEventRecord(events_[t * kSlots + s], stream));
        failed = false;
      };
      for (unsigned s = 0; s < kSlots; ++s) take(s);
      for (unsigned s = 0; in_slot[s].k < pieces; s = (s + 1) % kSlots) {
        BEADS_HIP(hipEventSynchronize(events_[t * kSlots + s]));
        deliver(fields, window_of(in_slot[s].k), host_.data() + (t * kSlots + s) * piece,
                in_slot[s].offset, in_slot[s].size);
        take(s);
      }
    } catch (...) {
      const std::lock_guard<std::mutex> lock(next_mutex);
      if (!error) error = std::current_exception();
    }
  };
  std::vector<std::thread> helpers;
  helpers.reserve(threads);
  try {
    for (unsigned t = 1; t < threads; ++t) helpers.emplace_back(work, t);
  } catch (const std::system_error&) {
    // fewer threads: the ones there are share the pieces
  }
  work(0);
  for (auto& h : helpers) h.join();
  if (error) {
    (void)hipStreamSynchronize(stream);  // no copy into the staging memory outlives the call
    std::rethrow_exception(error);
  }
}

void StateReader::read(const StateSource& src, const beads_state_out_t& o, hipStream_t stream) {
  const std::lock_guard<std::mutex> lock(mutex_);
  std::vector<Field> fields;
  size_t per_atom = 0;
  PackStateParams p{};
  p.n = src.n;
  p.pos = src.pos;
  p.vel = src.vel;
  p.force = src.force;
  p.image = src.image;
  p.tag = src.tag;
  p.molid = src.molid;
  // Reals first, so that every field keeps its alignment.
  auto add = [&](void* dst, size_t bytes, bool available, uint64_t PackStateParams::* place) {
    p.*place = kNoField;
    if (dst == nullptr || !available) return;
    fields.push_back({bytes, static_cast<unsigned char*>(dst), place});
    per_atom += bytes;
  };
  add(o.positions, 3 * sizeof(real_t), true, &PackStateParams::positions);
  add(o.velocities, 3 * sizeof(real_t), true, &PackStateParams::velocities);
  add(o.forces, 3 * sizeof(real_t), true, &PackStateParams::forces);
  add(o.masses, sizeof(real_t), true, &PackStateParams::masses);
  add(o.images, 3 * sizeof(int32_t), true, &PackStateParams::images);
  add(o.types, sizeof(int32_t), true, &PackStateParams::types);
  add(o.tags, sizeof(uint32_t), src.tag != nullptr, &PackStateParams::tags);
  add(o.molecule_ids, sizeof(uint32_t), src.molid != nullptr, &PackStateParams::molecule_ids);
  if (per_atom == 0 || p.n == 0) {
    BEADS_HIP(hipStreamSynchronize(stream));
    return;
  }
  const size_t n = p.n, total = n * per_atom;
  const size_t window_atoms = reserve(n, per_atom);
  if (total > whole_bytes_ || window_atoms < n) {
    read_windows(fields, p, per_atom, window_atoms, stream);
    return;
  }
  const Window all{0, n};
  host_.resize(total);
  pack(fields, p, all, stream);
  BEADS_HIP(hipMemcpyAsync(host_.data(), stage_.data(), total, hipMemcpyDeviceToHost, stream));
  BEADS_HIP(hipStreamSynchronize(stream));
  deliver(fields, all, host_.data(), 0, total);
}

}  // namespace beads_amd
