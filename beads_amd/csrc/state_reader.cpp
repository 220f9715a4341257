#include "state_reader.hpp"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <system_error>
#include <thread>

#include "kernels.hpp"

namespace beads_amd {

namespace {

// States up to kWhole bytes come over in one copy; larger ones in kChunk
// pieces by up to kThreads threads with two pieces in flight each, because what
// bounds them is not the link but the first touch of the caller's pages and
// the copy out of the staging memory, about 4 GB/s in one thread.
constexpr size_t kChunk = size_t{1} << 20;
constexpr size_t kWhole = size_t{4} << 20;
constexpr unsigned kThreads = 8;
constexpr unsigned kSlots = 2;

}  // namespace

StateReader::~StateReader() {
  for (auto& e : events_) (void)hipEventDestroy(e);
}

void StateReader::deliver(const std::vector<Field>& fields, const unsigned char* bytes,
                          size_t offset, size_t size) {
  for (const Field& f : fields) {
    const size_t b = std::max(offset, f.offset), e = std::min(offset + size, f.offset + f.size);
    if (b < e) std::memcpy(f.dst + (b - f.offset), bytes + (b - offset), e - b);
  }
}

void StateReader::deliver_in_chunks(const std::vector<Field>& fields, size_t total,
                                    hipStream_t stream) {
  const size_t chunks = (total + kChunk - 1) / kChunk;
  const unsigned cores = std::max(1u, std::thread::hardware_concurrency());
  const unsigned threads =
      static_cast<unsigned>(std::min<size_t>(std::min(kThreads, cores), (chunks + 1) / 2));
  host_.resize(static_cast<size_t>(threads) * kSlots * kChunk);
  while (events_.size() < static_cast<size_t>(threads) * kSlots) {
    hipEvent_t e;
    BEADS_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    events_.push_back(e);
  }
  int device = 0;
  BEADS_HIP(hipGetDevice(&device));
  std::atomic<size_t> next{0};
  std::mutex error_mutex;
  std::exception_ptr error;
  auto work = [&](unsigned t) {
    try {
      BEADS_HIP(hipSetDevice(device));
      size_t in_slot[kSlots];
      auto request = [&](unsigned s) {
        in_slot[s] = next.fetch_add(1);
        if (in_slot[s] >= chunks) return;
        const size_t at = in_slot[s] * kChunk;
        BEADS_HIP(hipMemcpyAsync(host_.data() + (t * kSlots + s) * kChunk, stage_.data() + at,
                                 std::min(kChunk, total - at), hipMemcpyDeviceToHost, stream));
        BEADS_HIP(hipEventRecord(events_[t * kSlots + s], stream));
      };
      for (unsigned s = 0; s < kSlots; ++s) request(s);
      for (unsigned s = 0; in_slot[s] < chunks; s = (s + 1) % kSlots) {
        BEADS_HIP(hipEventSynchronize(events_[t * kSlots + s]));
        const size_t at = in_slot[s] * kChunk;
        deliver(fields, host_.data() + (t * kSlots + s) * kChunk, at, std::min(kChunk, total - at));
        request(s);
      }
    } catch (...) {
      const std::lock_guard<std::mutex> lock(error_mutex);
      if (!error) error = std::current_exception();
    }
  };
  std::vector<std::thread> helpers;
  helpers.reserve(threads);
  try {
    for (unsigned t = 1; t < threads; ++t) helpers.emplace_back(work, t);
  } catch (const std::system_error&) {
    // fewer threads: the ones there are share the chunks
  }
  work(0);
  for (auto& h : helpers) h.join();
  if (error) {
    (void)hipStreamSynchronize(stream);  // no copy into the staging memory outlives the call
    std::rethrow_exception(error);
  }
}

void StateReader::read(const StateSource& src, const beads_state_out_t& o, hipStream_t stream) {
  const size_t n = src.n;
  std::vector<Field> fields;
  size_t total = 0;
  PackStateParams p{};
  p.n = src.n;
  p.pos = src.pos;
  p.vel = src.vel;
  p.force = src.force;
  p.image = src.image;
  p.tag = src.tag;
  p.molid = src.molid;
  // Reals first, so that every field keeps its alignment.
  auto add = [&](void* dst, size_t bytes, bool available, uint64_t& offset) {
    offset = kNoField;
    if (dst == nullptr || !available) return;
    offset = total;
    fields.push_back({total, bytes, static_cast<unsigned char*>(dst)});
    total += bytes;
  };
  add(o.positions, 3 * n * sizeof(real_t), true, p.positions);
  add(o.velocities, 3 * n * sizeof(real_t), true, p.velocities);
  add(o.forces, 3 * n * sizeof(real_t), true, p.forces);
  add(o.masses, n * sizeof(real_t), true, p.masses);
  add(o.images, 3 * n * sizeof(int32_t), true, p.images);
  add(o.types, n * sizeof(int32_t), true, p.types);
  add(o.tags, n * sizeof(uint32_t), src.tag != nullptr, p.tags);
  add(o.molecule_ids, n * sizeof(uint32_t), src.molid != nullptr, p.molecule_ids);
  if (total == 0) {
    BEADS_HIP(hipStreamSynchronize(stream));
    return;
  }
  stage_.resize(total);
  p.out = stage_.data();
  launch_pack_state(p, stream);
  BEADS_HIP(hipGetLastError());
  if (total > kWhole) {
    deliver_in_chunks(fields, total, stream);
    return;
  }
  host_.resize(total);
  BEADS_HIP(hipMemcpyAsync(host_.data(), stage_.data(), total, hipMemcpyDeviceToHost, stream));
  BEADS_HIP(hipStreamSynchronize(stream));
  deliver(fields, host_.data(), 0, total);
}

}  // namespace beads_amd
