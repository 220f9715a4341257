// gfx950 kernels of the per-step MD path.
//
// Design (CDNA4): 256-wide workgroups (4 wave64s), one work-item per atom
// except in the force pass and the build (a team of lanes per atom), real4 SoA
// streams (float4, or double4 in the BEADS_REAL64 build), FP64 for LJ pair
// values and global reductions. Kernels that gather
// neighbour positions map workgroups onto atoms XCD by XCD so each XCD's L2
// holds one contiguous (spatially sorted) slab of positions. The two kernels of
// the neighbour-rebuild sequence read the device control block first and exit
// when no rebuild is due, so a step never waits on the host. No kernel that runs
// every step fences at device scope (on gfx950 that is an L2 write-back and
// invalidate of the XCD): cross-workgroup totals are formed by a one-workgroup
// kernel launched after the workgroups that wrote the partials. Only a reorder,
// inside the rebuild kernel, hands bulk data between workgroups with one.
//
// Reference counterparts (paths under native/src):
//   control/bin/scan/scatter/sort  simulation/neighbor/cell_list_build.cu:110-219,347-414,
//                                  neighbor_system.cpp:79-146,198-216
//   build                          simulation/neighbor/full/*.cu,
//                                  full_neighbor_path_common.cuh:49-94,
//                                  rebuild_tracker.cu:26-53 (reference capture)
//   force                          forcefield/pair/pair_lj.cu:21-167,
//                                  bond/bond_harmonic.cu:24-99, angle/angle_harmonic.cu:47-178,
//                                  dihedral/dihedral_harmonic.cu:65-227,
//                                  dynamics/integrator/velocity_verlet.cu:97-111,
//                                  dynamics/thermostat/berendsen_thermostat.cu:104-163
//   integrate                      velocity_verlet.cu:59-95, rebuild_tracker.cu:55-94
#include "kernels.hpp"

#include <hip/hip_runtime.h>

#include <type_traits>

#include "beads_amd.h"
#include "device_common.hpp"

namespace beads_amd {
namespace {

using namespace dev;

// ---------------------------------------------------------------- rebuild --

// Rebuild bookkeeping of NeighborSystem::update_after_position_change /
// rebuild_now (neighbor_system.cpp:79-146, 198-207), on the device. The sort
// cadence counts builds (neighbor_system.cpp:198-202) or, with
// sort_every_steps, steps: a build sorts when at least that many steps have
// passed since the last sort (the sort needs the rebuild that follows it).
__device__ __forceinline__ bool reorder_due(const Ctrl* ctrl, const NeighborControl& nc,
                                            uint64_t steps) {
  const bool due = nc.sort_every_steps != 0
                       ? ctrl->clock + steps - ctrl->last_sort >= nc.sort_every_steps
                       : ((ctrl->build_count + 1) % nc.sort_every) == 0;
  return nc.path != 0 && due;
}

// One thread: the counters of a step, with the decisions taken from them.
__device__ __forceinline__ void update_control(Ctrl* ctrl, const NeighborControl& nc, bool forced,
                                               bool rebuild, bool reorder, uint64_t steps) {
  ctrl->clock += steps;
  if (!forced) {
    const bool first = ctrl->checked == 0;
    ctrl->checked = 1;
    if (rebuild && nc.check_every > 1 && first) {
      ctrl->dangerous += 1;
    }
  }
  if (rebuild) {
    ctrl->rebuild = 1;
    ctrl->build_count += 1;
    ctrl->reorder = reorder ? 1u : 0u;
    ctrl->reorder_count += reorder ? 1u : 0u;
    if (reorder) ctrl->last_sort = ctrl->clock;
    ctrl->checked = 0;
  }
}

// Direct path: the bookkeeping alone, no cells to bin.
__global__ __launch_bounds__(kNeighborParts) void control_kernel(
    Ctrl* ctrl, NeighborControl nc, int forced, uint64_t steps, unsigned long long* neighbor_parts) {
  const bool rebuild = forced || ctrl->rebuild;
  if (rebuild) neighbor_parts[threadIdx.x * kNeighborPartStride] = 0;
  __syncthreads();
  if (threadIdx.x == 0) {
    update_control(ctrl, nc, forced != 0, rebuild, rebuild && reorder_due(ctrl, nc, steps), steps);
  }
}

// ----------------------------------------------------- one-launch rebuild --
//
// Binning, scan, scatter, in-cell sort and reorder are phases of one kernel:
// as kernels of their own, with the bookkeeping, they were seven launches a
// step, most of which find no rebuild due (about 2 us each inside a step
// graph). The phases are separated by barriers over the grid's workgroups.
// 100 steps of a 48,000-bead melt 4.98 -> 4.06 ms. A rebuild itself takes
// 26 us there, 85 us for the 1,000,000-bead melt (95 us as separate kernels)
// and 305 us with a reorder, most of it memory; of a small one (25 us at 4,000
// beads) most is the barriers, 4 us each.
//
// Which workgroups take part is settled at run time, so that no wait depends
// on how many of them the GPU holds at once: a workgroup that starts joins by
// taking a rank; rank 0 closes the list when all have joined, or join_ticks
// after its own start, and a workgroup that starts later leaves at once. The
// members are all running when the list closes and wait only for each other,
// so every wait ends. Work is divided by rank over the members there are.
//
// Every wait is bounded all the same (wait_polls). Past the bound a member
// stores Ctrl::stalled and leaves, which fails the others' next barrier; up to
// it each phase has read only what the barriers before it completed. From then
// on the cells, and a reorder's arrays, may be half done, so the state is
// final: no later launch bins, sorts or builds (counts that were not cleared
// would run the scatter past its array), the force pass keeps the last whole
// list, whose slots stay inside every array, and every host call that
// waits for the engine reports the stall.
//
// Each member has a cache line of its own to arrive on and one to be released
// on: polls and stores of 256 workgroups on one word would serialise (33 ns
// each past the L2).
constexpr int kRebuildBlock = 1024;
constexpr uint32_t kRebuildWaves = kRebuildBlock / 64;
constexpr uint32_t kJoinClosed = 0x80000000u;
constexpr uint32_t kRankBits = 9;  // ranks and counts up to kRebuildMaxBlocks
static_assert(kRebuildMaxBlocks < (1u << kRankBits) && kRebuildMaxBlocks <= kRebuildBlock,
              "rank 0 polls one member per thread");
struct Members {
  uint64_t* lines;  // [member][2 * kSyncLine]: arrival word, release word a line later
  uint32_t* stalled_host;
  uint32_t wait_polls;
  uint32_t rank, count;
  uint64_t epoch;   // unique to this rebuild and barrier, advanced by each barrier
};

template <typename T>
__device__ __forceinline__ T agent_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void agent_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until *word holds the epoch above its kRankBits; false past the bound.
__device__ __forceinline__ bool await_epoch(const uint64_t* word, const Members& m) {
  for (uint32_t polls = 0; (agent_load(word) >> kRankBits) != m.epoch; ++polls) {
    if (polls >= m.wait_polls) return false;
    __builtin_amdgcn_s_sleep(1);
  }
  return true;
}

__device__ __forceinline__ void report_stall(Ctrl* ctrl, const Members& m) {
  agent_store(&ctrl->stalled, 1u);
  __hip_atomic_store(m.stalled_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Joins the rebuild's members. Returns false (in every thread) where the
// workgroup has nothing to do. epoch0 is above 0, which the lines start with.
__device__ __forceinline__ bool join_members(Ctrl* ctrl, const RebuildParams& p, uint64_t epoch0,
                                             Members& m) {
  __shared__ uint32_t rank_lds, count_lds;
  const RebuildLimits& limits = p.limits;
  uint64_t* const lines = p.sync_lines;
  if (threadIdx.x == 0) {
    // Nobody joins after a stall (looked at by one thread: a stall in this very
    // launch may come between the looks of two).
    const uint32_t v = agent_load(&ctrl->stalled) != 0
                           ? kJoinClosed
                           : __hip_atomic_fetch_add(&ctrl->joined, 1u, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
    rank_lds = v;
    count_lds = 0;
    if (v == 0) {
      const uint32_t all = min(static_cast<uint32_t>(gridDim.x), limits.members);
      const long long start = wall_clock64();
      while (agent_load(&ctrl->joined) < all && wall_clock64() - start < limits.join_ticks) {
        __builtin_amdgcn_s_sleep(1);
      }
      count_lds = min(__hip_atomic_fetch_or(&ctrl->joined, kJoinClosed, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT),
                      limits.members);
      agent_store(&ctrl->members, count_lds);
    }
  }
  __syncthreads();
  const uint32_t rank = rank_lds;
  if (rank >= limits.members) return false;  // closed (kJoinClosed) or full
  m.lines = lines;
  m.stalled_host = p.stalled_host;
  m.wait_polls = limits.wait_polls;
  m.rank = rank;
  m.epoch = epoch0;
  if (rank == 0) {
    const uint32_t count = count_lds;
    if (threadIdx.x > 0 && threadIdx.x < count) {
      agent_store(lines + (2 * threadIdx.x + 1) * kSyncLine, (epoch0 << kRankBits) | count);
    }
  } else if (threadIdx.x == 0) {
    const uint64_t* const release = lines + (2 * rank + 1) * kSyncLine;
    if (await_epoch(release, m)) {
      count_lds = static_cast<uint32_t>(agent_load(release)) & ((1u << kRankBits) - 1u);
    } else {
      report_stall(ctrl, m);
    }
  }
  __syncthreads();
  m.count = count_lds;
  return m.count != 0;
}

// Barrier over the members. What they stored at agent scope (agent_store,
// atomics) before it is seen by agent_load and atomics after it: such accesses
// go past the L2, which another XCD does not see, so all the barrier has to do
// is wait for them. FULL also hands over ordinary stores, by writing back and
// emptying the L2, 2 us a barrier and more where it holds much: only the
// reorder moves enough data to want it. Returns false (in every thread) past
// the bound on a wait.
template <bool FULL>
__device__ __forceinline__ bool member_barrier(Ctrl* ctrl, Members& m) {
  __shared__ int ok_lds;
  m.epoch += 1;
  if (threadIdx.x == 0) ok_lds = 1;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores are acknowledged
  __syncthreads();
  if (threadIdx.x == 0) {
    if (FULL) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    if (m.rank != 0) agent_store(m.lines + 2 * m.rank * kSyncLine, m.epoch << kRankBits);
  }
  if (m.rank == 0) {
    if (threadIdx.x > 0 && threadIdx.x < m.count &&
        !await_epoch(m.lines + 2 * threadIdx.x * kSyncLine, m)) {
      ok_lds = 0;
    }
    __syncthreads();
    if (threadIdx.x > 0 && threadIdx.x < m.count && ok_lds) {
      agent_store(m.lines + (2 * threadIdx.x + 1) * kSyncLine, m.epoch << kRankBits);
    }
  } else if (threadIdx.x == 0 &&
             !await_epoch(m.lines + (2 * m.rank + 1) * kSyncLine, m)) {
    ok_lds = 0;
  }
  __syncthreads();
  const bool ok = ok_lds != 0;
  if (!ok && threadIdx.x == 0) report_stall(ctrl, m);
  // One wave's acquire empties the caches the workgroup reads through.
  if (FULL && threadIdx.x < 64) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  __syncthreads();
  return ok;
}

// Exclusive scan of a value over the workgroup's threads; total gets the sum.
__device__ __forceinline__ uint32_t block_exclusive(uint32_t v, uint32_t* lds, uint32_t& total) {
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t incl = v;
#pragma unroll
  for (uint32_t off = 1; off < 64; off <<= 1) {
    const uint32_t u = __shfl_up(incl, off, 64);
    incl += lane >= off ? u : 0u;
  }
  __syncthreads();
  if (lane == 63) lds[wave] = incl;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
#pragma unroll
  for (uint32_t w = 0; w < kRebuildWaves; ++w) {
    const uint32_t x = lds[w];
    before += w < wave ? x : 0u;
    total += x;
  }
  return before + incl - v;
}

// cell_list_build.cu:135-166: cell index in the storage precision and atomic
// counts, one atomic per distinct cell of the wave.
__device__ __forceinline__ void bin_atom(const CellScanParams& p, Ctrl* ctrl, uint32_t i) {
  const real4 x = p.pos[i];
  const uint32_t c = cell_of_position(x, p.box, p.grid);
  p.cell_of[i] = c;
  wave_increment(p.cell_count, c);
  raise_flag(outside_cells(x, p.box, p.grid), &ctrl->outside);
}

// Cells up to which a member sums the counts before its own tile by itself
// (at most 64 KB from the L2) instead of a further barrier.
constexpr uint32_t kOwnPrefixCells = 16384;

// Exclusive scan of the cell counts into cell_start[0..n_cells], copied to the
// scatter cursor; clears the counts for the next rebuild. Each member scans
// its own tile of consecutive cells.
__device__ __forceinline__ bool scan_cells(const CellScanParams& p, Ctrl* ctrl, Members& m,
                                           uint32_t* tile_sums) {
  __shared__ uint32_t lds[kRebuildWaves];
  const uint32_t t = threadIdx.x;
  const uint32_t per = (p.n_cells + m.count - 1) / m.count;
  const uint32_t begin = min(p.n_cells, m.rank * per), end = min(p.n_cells, begin + per);
  uint32_t mine = 0, carry = 0;
  if (p.n_cells <= kOwnPrefixCells) {
    for (uint32_t c = t; c < begin; c += kRebuildBlock) mine += agent_load(p.cell_count + c);
    block_exclusive(mine, lds, carry);
  } else {
    uint32_t total;
    for (uint32_t c = begin + t; c < end; c += kRebuildBlock) mine += agent_load(p.cell_count + c);
    block_exclusive(mine, lds, total);
    if (t == 0) agent_store(tile_sums + m.rank, total);
    if (!member_barrier<false>(ctrl, m)) return false;
    block_exclusive(t < m.rank ? agent_load(tile_sums + t) : 0u, lds, carry);
  }
  // Other members may still sum this tile's counts: they are cleared past the
  // next barrier.
  for (uint32_t base = begin; base < end; base += kRebuildBlock) {
    const uint32_t c = base + t;
    const uint32_t cnt = c < end ? agent_load(p.cell_count + c) : 0u;
    uint32_t total;
    const uint32_t start = carry + block_exclusive(cnt, lds, total);
    if (c < end) {
      agent_store(p.cell_start + c, start);
      agent_store(p.cell_cursor + c, start);
    }
    carry += total;
  }
  if (end == p.n_cells && t == 0) agent_store(p.cell_start + p.n_cells, carry);
  if (!member_barrier<false>(ctrl, m)) return false;
  for (uint32_t c = begin + t; c < end; c += kRebuildBlock) p.cell_count[c] = 0;
  return true;
}

// Counting-sort scatter of an atom into its cell; sort_cell orders the members.
__device__ __forceinline__ void scatter_atom(const CellScanParams& p, uint32_t i) {
  const uint32_t slot = wave_increment(p.cell_cursor, p.cell_of[i]);
  agent_store(p.cell_atoms + slot, i);
}

// Order each cell's members by (x, slot): with the counting sort this is a
// deterministic order, where the reference's atomic scatter
// (cell_list_build.cu:168-181) leaves each cell's members in arbitrary order;
// the sets a build finds are the same for any order inside a cell. Ordering
// by x makes the members of an x-row of cells ascending in x, so a build can
// scan a row as one run and skip its ends beyond r_s (cell_xbins). One wave
// per cell: for up to 64 members lane l holds member l, whose rank is the
// number of members before it in (x, slot) order, and stores it at start +
// rank; the x-bin prefix counts come from one ballot per bin. Larger cells:
// sort_large_cell. When no reorder follows, the kernel also
// writes the members' positions in cell order with the slot in .w (the
// build's candidate stream); after a reorder, commit_atom writes them.
__device__ __forceinline__ real4 cell_entry(real4 x, uint32_t slot) {
  return make_real4(x.x, x.y, x.z, real_of_id(slot));
}

// v of lane `lane` (uniform over the wave).
__device__ __forceinline__ real_t read_lane(real_t v, int lane) {
#ifdef BEADS_REAL64
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = static_cast<uint32_t>(
      __builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(b)), lane));
  const uint32_t hi = static_cast<uint32_t>(
      __builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(b >> 32)), lane));
  return __builtin_bit_cast(real_t, (static_cast<uint64_t>(hi) << 32) | lo);
#else
  return __builtin_bit_cast(real_t, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
#endif
}

// Bin of coordinate x inside x-cell cx (0 .. kXBins - 1), monotone in x: the
// cell coordinate of axis_cell, offset by the cell and scaled by the bin count
// (a power of two).
__device__ __forceinline__ int x_bin(real_t x, real_t lo, real_t inv, uint32_t cx) {
#pragma clang fp contract(off)
  const real_t f = ((x - lo) * inv - static_cast<real_t>(cx)) * static_cast<real_t>(kXBins);
  return f <= real_t(0) ? 0
                        : (f >= static_cast<real_t>(kXBins - 1) ? kXBins - 1 : static_cast<int>(f));
}

// The order's key: NaN, which no comparison would place (two members would take
// one entry and another keep what was there before), comes last.
__device__ __forceinline__ real_t order_key(real_t x) {
  return x == x ? x : static_cast<real_t>(__builtin_huge_val());
}

__device__ __forceinline__ bool before_in_cell(real_t xa, uint32_t sa, real_t xb, uint32_t sb) {
  return xa < xb || (xa == xb && sa < sb);
}

// Position of member v (x = its key) of a wave's chunk of cnt members, one a lane.
__device__ __forceinline__ uint32_t rank_in_chunk(uint32_t v, real_t x, uint32_t cnt) {
  uint32_t rank = 0;
  for (uint32_t m = 0; m < cnt; ++m) {
    const uint32_t w = static_cast<uint32_t>(
        __builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(m)));
    const real_t xw = read_lane(x, static_cast<int>(m));
    rank += before_in_cell(xw, w, x, v) ? 1u : 0u;
  }
  return rank;
}

// The members [b, b + cnt) of a cell of more than 64, ordered by one wave:
// chunks of 64 by rank, then runs of twice the length until one is left, each
// member's place in the other run found by bisection. The passes go back and
// forth between cell_atoms and scratch; returns the array with the last one's
// result. Such cells are rare, but have to end: a system that has flown apart
// has all its atoms in the corner cells, and one lane inserting one member after
// another took m^2 / 4 moves of 0.4 us (80 ms at 937 members, 1.5 hours at
// 242,771, which take 155 ms now: a chain of dependent loads per bisection).
__device__ __forceinline__ const uint32_t* sort_large_cell(const CellScanParams& p, uint32_t b,
                                                        uint32_t cnt, uint32_t* scratch) {
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t *src = p.cell_atoms + b, *dst = scratch + b;
  auto key = [&p](uint32_t v) { return order_key(p.pos[v].x); };
  for (uint32_t base = 0; base < cnt; base += 64) {
    const uint32_t here = min(64u, cnt - base);
    const uint32_t v = lane < here ? agent_load(src + base + lane) : 0xffffffffu;
    const real_t x = lane < here ? key(v) : real_t(0);
    const uint32_t rank = rank_in_chunk(v, x, here);
    if (lane < here) dst[base + rank] = v;
  }
  for (uint32_t w = 64; w < cnt; w *= 2) {  // cnt < 2^28
    uint32_t* const done = dst;
    dst = src;
    src = done;
    // The wave's stores are in the caches it reads through.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    for (uint32_t k = lane; k < cnt; k += 64) {
      const uint32_t first = k & ~(w - 1);  // of the member's run
      const uint32_t pair = k & ~(2 * w - 1);
      const uint32_t other = first == pair ? first + w : pair;
      uint32_t lo = other, hi = other < cnt ? min(cnt, other + w) : other;
      const uint32_t v = src[k];
      const real_t x = key(v);
      while (lo < hi) {
        const uint32_t mid = (lo + hi) / 2;
        const uint32_t u = src[mid];
        if (before_in_cell(key(u), u, x, v)) {
          lo = mid + 1;
        } else {
          hi = mid;
        }
      }
      dst[pair + (k - first) + (lo - other)] = v;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  return dst - b;
}

// One wave orders cell c; stream: also write the candidate stream. scratch: an
// entry per atom, used for large cells.
__device__ __forceinline__ void sort_cell(const CellScanParams& p, uint32_t c, bool stream,
                                          uint32_t* scratch) {
  const uint32_t lane = threadIdx.x & 63u;
  const real_t lo = p.box.lo[0], inv = p.grid.inv_cell[0];
  const uint32_t b = agent_load(p.cell_start + c), e = agent_load(p.cell_start + c + 1);
  const uint32_t cnt = e - b;
  const uint32_t cx = c % p.grid.nx;
  uint32_t* a = p.cell_atoms;
  if (cnt <= 64) {
    const uint32_t v = lane < cnt ? agent_load(a + b + lane) : 0xffffffffu;
    const real4 xv4 = lane < cnt ? p.pos[v] : make_real4(0, 0, 0, 0);
    const real_t xv = order_key(xv4.x);
    const uint32_t rank = rank_in_chunk(v, xv, cnt);
    if (lane < cnt) {
      a[b + rank] = v;
      if (stream) p.cell_pos[b + rank] = cell_entry(xv4, v);
    }
    const int bin = lane < cnt ? x_bin(xv, lo, inv, cx) : kXBins;
    uint32_t pre[kXBins];
#pragma unroll
    for (int m = 1; m <= kXBins; ++m) {
      pre[m - 1] = static_cast<uint32_t>(__builtin_popcountll(__ballot(bin < m)));
    }
    if (lane == 0) {
      p.cell_xbins[c] = make_uint4(pre[0] | (pre[1] << 16), pre[2] | (pre[3] << 16),
                                   pre[4] | (pre[5] << 16), pre[6] | (pre[7] << 16));
    }
    return;
  }
  const uint32_t* const sorted = sort_large_cell(p, b, cnt, scratch);
  uint32_t pre[kXBins] = {};
  for (uint32_t k = lane; k - lane < cnt; k += 64) {
    int bin = kXBins;
    if (k < cnt) {
      const uint32_t v = sorted[b + k];
      const real4 xv4 = p.pos[v];
      a[b + k] = v;
      if (stream) p.cell_pos[b + k] = cell_entry(xv4, v);
      bin = x_bin(order_key(xv4.x), lo, inv, cx);
    }
#pragma unroll
    for (int m = 1; m <= kXBins; ++m) {
      pre[m - 1] += static_cast<uint32_t>(__builtin_popcountll(__ballot(bin < m)));
    }
  }
  if (lane == 0 && cnt <= kXBinsMaxCount) {
    p.cell_xbins[c] = make_uint4(pre[0] | (pre[1] << 16), pre[2] | (pre[3] << 16),
                                 pre[4] | (pre[5] << 16), pre[6] | (pre[7] << 16));
  }
}

// trajectory_output.cu:183-250: one record per atom in slot order, fields in
// the file's order (tag, type, position, image, velocity, force); the type is
// stored 1-based as in the spec.
__global__ __launch_bounds__(kBlock) void pack_records_kernel(PackParams p) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= p.n) {
    return;
  }
  uint32_t* r = p.out + static_cast<size_t>(i) * p.words;
  const real4 x = p.pos[i];
  uint32_t k = 0;
  // A real as one word (binary32) or two, low word first (binary64).
  auto put = [&](real_t v) {
#ifdef BEADS_REAL64
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    r[k++] = static_cast<uint32_t>(b);
    r[k++] = static_cast<uint32_t>(b >> 32);
#else
    r[k++] = __builtin_bit_cast(uint32_t, v);
#endif
  };
  r[k++] = p.tag[i];
  if (p.mask & BEADS_TRAJ_TYPE) r[k++] = id_of(x.w) + 1u;
  if (p.mask & BEADS_TRAJ_POSITION) {
    put(x.x);
    put(x.y);
    put(x.z);
  }
  if (p.mask & BEADS_TRAJ_IMAGE) {
    const int4 m = p.image[i];
    r[k++] = static_cast<uint32_t>(m.x);
    r[k++] = static_cast<uint32_t>(m.y);
    r[k++] = static_cast<uint32_t>(m.z);
  }
  if (p.mask & BEADS_TRAJ_VELOCITY) {
    const real4 v = p.vel[i];
    put(v.x);
    put(v.y);
    put(v.z);
  }
  if (p.mask & BEADS_TRAJ_FORCE) {
    const real4 f = p.force[i];
    put(f.x);
    put(f.y);
    put(f.z);
  }
}

// The wanted fields of every atom, each an array of its own (a host copy of
// whole records would leave the taking apart, and a quarter more bytes, to one
// host thread).
__global__ __launch_bounds__(kBlock) void pack_state_kernel(PackStateParams p) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= p.n) {
    return;
  }
  const uint32_t a = p.first + i;
  auto put3 = [&](uint64_t field, auto x, auto y, auto z) {
    auto* o = reinterpret_cast<decltype(x)*>(p.out + field) + 3 * static_cast<size_t>(i);
    o[0] = x;
    o[1] = y;
    o[2] = z;
  };
  if (p.positions != kNoField || p.types != kNoField) {
    const real4 x = p.pos[a];
    if (p.positions != kNoField) put3(p.positions, x.x, x.y, x.z);
    if (p.types != kNoField) {
      reinterpret_cast<int32_t*>(p.out + p.types)[i] = static_cast<int32_t>(id_of(x.w)) + 1;
    }
  }
  if (p.velocities != kNoField || p.masses != kNoField) {
    const real4 v = p.vel[a];
    if (p.velocities != kNoField) put3(p.velocities, v.x, v.y, v.z);
    if (p.masses != kNoField) reinterpret_cast<real_t*>(p.out + p.masses)[i] = v.w;
  }
  if (p.forces != kNoField) {
    const real4 f = p.force[a];
    put3(p.forces, f.x, f.y, f.z);
  }
  if (p.images != kNoField) {
    const int4 m = p.image[a];
    put3(p.images, m.x, m.y, m.z);
  }
  if (p.tags != kNoField) reinterpret_cast<uint32_t*>(p.out + p.tags)[i] = p.tag[a];
  if (p.molecule_ids != kNoField) {
    reinterpret_cast<uint32_t*>(p.out + p.molecule_ids)[i] = p.molid[a];
  }
}

// cell_list_build.cu:183-219: gather every per-atom array into cell order
// (new slot s takes old slot cell_atoms[s]) and record the inverse map.
__device__ __forceinline__ void gather_atom(const ReorderParams& p, uint32_t s) {
  const uint32_t o = p.cell_atoms[s];
  p.new_of_old[o] = s;
  p.s_pos[s] = p.pos[o];
  p.s_vel[s] = p.vel[o];
  p.s_image[s] = p.image[o];
  p.s_tag[s] = p.tag[o];
  p.s_molid[s] = p.molid[o];
  p.s_cell_of[s] = p.cell_of[o];
  p.s_topo_count[s] = p.topo_count[o];
  const size_t n = p.n;
  for (uint32_t k = 0; k < p.bcap; ++k) p.s_bond[k * n + s] = p.bond[k * n + o];
  for (uint32_t k = 0; k < p.acap; ++k) p.s_angle[k * n + s] = p.angle[k * n + o];
  for (uint32_t k = 0; k < p.dcap; ++k) p.s_dih[k * n + s] = p.dih[k * n + o];
  for (uint32_t k = 0; k < p.ecap; ++k) p.s_excl[k * n + s] = p.excl[k * n + o];
  if (p.spill_index != nullptr) p.s_spill_index[s] = p.spill_index[o];
}

// Copy back and translate partner slots through the inverse permutation.
__device__ __forceinline__ void commit_atom(const ReorderParams& p, uint32_t s) {
  p.pos[s] = p.s_pos[s];
  p.vel[s] = p.s_vel[s];
  p.image[s] = p.s_image[s];
  p.tag[s] = p.s_tag[s];
  p.molid[s] = p.s_molid[s];
  p.cell_of[s] = p.s_cell_of[s];
  p.cell_atoms[s] = s;
  p.cell_pos[s] = cell_entry(p.s_pos[s], s);
  const uint32_t cw = p.s_topo_count[s];
  p.topo_count[s] = cw;
  const size_t n = p.n;
  const uint32_t* m = p.new_of_old;
  const uint32_t nb = cw & 255u, na = (cw >> 8) & 255u, nd = (cw >> 16) & 255u, ne = cw >> 24;
  for (uint32_t k = 0; k < nb; ++k) {
    uint2 r = p.s_bond[k * n + s];
    r.x = m[r.x];
    p.bond[k * n + s] = r;
  }
  for (uint32_t k = 0; k < na; ++k) {
    uint4 r = p.s_angle[k * n + s];
    r.x = m[r.x];
    r.y = m[r.y];
    p.angle[k * n + s] = r;
  }
  for (uint32_t k = 0; k < nd; ++k) {
    uint4 r = p.s_dih[k * n + s];
    r.x = m[r.x];
    r.y = m[r.y];
    r.z = m[r.z];
    p.dih[k * n + s] = r;
  }
  for (uint32_t k = 0; k < ne; ++k) {
    p.excl[k * n + s] = m[p.s_excl[k * n + s]];
  }
  if (p.spill_index != nullptr) {
    // The particle's spill segments stay where they are; their partner slots
    // are remapped here by their one owner.
    const uint32_t si = p.s_spill_index[s];
    p.spill_index[s] = si;
    if (si != kNoSpill) {
      const SpillEntry e = p.spill[si];
      for (uint32_t k = 0; k < e.cnt[0]; ++k) {
        uint2& r = p.spill_bond[e.off[0] + k];
        r.x = m[r.x];
      }
      for (uint32_t k = 0; k < e.cnt[1]; ++k) {
        uint4& r = p.spill_angle[e.off[1] + k];
        r.x = m[r.x];
        r.y = m[r.y];
      }
      for (uint32_t k = 0; k < e.cnt[2]; ++k) {
        uint4& r = p.spill_dih[e.off[2] + k];
        r.x = m[r.x];
        r.y = m[r.y];
        r.z = m[r.z];
      }
      for (uint32_t k = 0; k < e.cnt[3]; ++k) {
        uint32_t& r = p.spill_excl[e.off[3] + k];
        r = m[r];
      }
    }
  }
}

// Phases 1 to 6 of a rebuild for the atoms and cells of this member; see the
// section's head. The build that follows is a launch of its own: it wants far
// more workgroups than wait at a barrier.
__global__ __launch_bounds__(kRebuildBlock) void rebuild_kernel(CellScanParams cp, ReorderParams rp,
                                                                RebuildParams p) {
  Ctrl* const ctrl = p.ctrl;
  const bool forced = p.forced != 0;
  const bool rebuild = forced || ctrl->rebuild != 0;
  if (!rebuild) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      update_control(ctrl, p.control, false, false, false, p.steps);
    }
    return;
  }
  const bool reorder = reorder_due(ctrl, p.control, p.steps);
  Members m;
  // The epochs of a rebuild differ from those of every other one: each whole
  // one counts a build, and none follows one that stalled.
  if (!join_members(ctrl, p, (ctrl->build_count + 1) * 8u, m)) return;
  const uint32_t n = cp.n;
  const uint32_t first = m.rank * kRebuildBlock + threadIdx.x;
  const uint32_t stride = m.count * kRebuildBlock;
  for (uint64_t i = first; i < n; i += stride) bin_atom(cp, ctrl, static_cast<uint32_t>(i));
  if (!member_barrier<false>(ctrl, m)) return;
  // Every member has read the counters that its decisions come from.
  if (m.rank == 0) {
    if (threadIdx.x < kNeighborParts) p.neighbor_parts[threadIdx.x * kNeighborPartStride] = 0;
    if (threadIdx.x == 0) update_control(ctrl, p.control, forced, true, reorder, p.steps);
  }
  if (!scan_cells(cp, ctrl, m, p.tile_sums)) return;
  for (uint64_t i = first; i < n; i += stride) scatter_atom(cp, static_cast<uint32_t>(i));
  if (!member_barrier<false>(ctrl, m)) return;
  for (uint32_t c = m.rank * kRebuildWaves + threadIdx.x / 64; c < cp.n_cells;
       c += m.count * kRebuildWaves) {  // uniform over the wave
    sort_cell(cp, c, !reorder, rp.new_of_old);
  }
  if (!reorder) return;
  if (!member_barrier<true>(ctrl, m)) return;
  for (uint64_t s = first; s < n; s += stride) gather_atom(rp, static_cast<uint32_t>(s));
  if (!member_barrier<true>(ctrl, m)) return;
  for (uint64_t s = first; s < n; s += stride) commit_atom(rp, static_cast<uint32_t>(s));
}

constexpr int kBuildTeam = 4;
constexpr int kBuildSlots = 4;
constexpr uint32_t kBuildAtoms = kBlock / kBuildTeam;

// LDS bytes a build workgroup may use to stage the union of its atoms' row
// runs (more LDS per workgroup costs occupancy).
constexpr uint32_t kStageBytesMax = 24576;

// Rows path: regular grid, at least 5 cells per axis, no atom outside the
// cells, atom i not in an x-boundary cell, so that each row is one run. Writes row r's run for r = t,
// t + kBuildTeam, ... (the team's lanes share the rows), widens the block's
// span of row r, [lo[r], hi[r]), to cover a nonempty run, and returns false
// off the rows path.
__device__ inline bool row_runs(const BuildParams& p, uint32_t i, uint32_t t, uint2* rows,
                                uint32_t* lo_r, uint32_t* hi_r) {
  const CellGridView& g = p.grid;
  if (g.path != 1 || g.nx < 5 || g.ny < 5 || g.nz < 5 || p.ctrl->outside != 0) return false;
  const uint32_t c = p.cell_of[i];
  const uint32_t cx = c % g.nx, cyz = c / g.nx, cy = cyz % g.ny, cz = cyz / g.ny;
  if (cx < 1 || cx + 1 >= g.nx) return false;
  const real4 xi = p.pos[i];
#pragma unroll 1
  for (uint32_t r = t; r < static_cast<uint32_t>(kRows); r += kBuildTeam) {
    const uint2 d =
        row_run_pair(g, p.box, p.rs2, p.cell_start, p.cell_xbins, true, xi, cx, cy, cz, r).a;
    rows[r] = d;
    const uint32_t b = d.x, e = d.y & kRunIndexMask;
    if (b < e) {
      atomicMin(lo_r + r, b);
      atomicMax(hi_r + r, e);
    }
  }
  return true;
}

// The append rule's test of one atom's candidates: self, distance, exclusions.
// EXCL: 0 = no exclusions, 4 or 8 = up to that many partners held in
// registers, -1 = any count read from memory (the spilled ones too).
template <int EXCL, bool HALF>
struct BuildAccept {
  const BuildParams& p;
  const uint32_t i;
  const real4 xi;
  uint32_t ex[EXCL > 0 ? EXCL : 1];
  uint32_t ne = 0;
  uint32_t spill_ne = 0, spill_off = 0;  // exclusions past the inline capacity

  __device__ __forceinline__ BuildAccept(const BuildParams& params, uint32_t slot, real4 x)
      : p(params), i(slot), xi(x) {
    if (EXCL < 0 && p.spill_index != nullptr) {
      const uint32_t si = p.spill_index[i];
      if (si != kNoSpill) {
        spill_off = p.spill[si].off[3];
        spill_ne = p.spill[si].cnt[3];
      }
    }
    if (EXCL != 0) {
      ne = p.topo_count[i] >> 24;
      if (EXCL > 0) {
#pragma unroll
        for (int k = 0; k < EXCL; ++k) {
          ex[k] = k < static_cast<int>(ne) ? p.excl[static_cast<size_t>(k) * p.n + i] : 0xffffffffu;
        }
      }
    }
  }

  // sh: the image shift of the candidate's cell, with mic(xi - xj) equal to
  // (xi - xj) + sh on every axis (cells of a grid with at least 5 cells per
  // axis). mode: kShift adds sh on every axis, kShiftYZ only on y and z (a run
  // that does not wrap has no x shift; adding a zero would change nothing but
  // the sign of a zero difference, which r^2 squares away), kGeneric takes
  // mic() per candidate.
  // Returns the wave's lanes that accept their candidate, as a lane mask:
  // every test is a compare whose ballot is its lane mask, so the tests
  // combine as scalar ANDs without branches.
  template <typename Mode>
  __device__ __forceinline__ uint64_t operator()(uint32_t j, real4 xj, Mode, real3 sh) const {
    real_t dx, dy, dz;
    if (Mode::value == kGeneric) {
      dx = mic(xi.x - xj.x, p.box.L[0], p.box.hL[0]);
      dy = mic(xi.y - xj.y, p.box.L[1], p.box.hL[1]);
      dz = mic(xi.z - xj.z, p.box.L[2], p.box.hL[2]);
    } else {
      dx = Mode::value == kShift ? (xi.x - xj.x) + sh.x : xi.x - xj.x;
      dy = (xi.y - xj.y) + sh.y;
      dz = (xi.z - xj.z) + sh.z;
    }
    const real_t r2 = r2_strict(dx, dy, dz);
    uint64_t m = __builtin_amdgcn_ballot_w64(!(r2 > p.rs2)) &
                 __builtin_amdgcn_ballot_w64(HALF ? j > i : j != i);
    if (EXCL > 0) {
#pragma unroll
      for (int k = 0; k < EXCL; ++k) {
        m &= __builtin_amdgcn_ballot_w64(ex[k] != j);
      }
    } else if (EXCL < 0) {
      bool ok = __builtin_amdgcn_inverse_ballot_w64(m);
      if (ok) {
        for (uint32_t k = 0; k < ne; ++k) {
          if (p.excl[static_cast<size_t>(k) * p.n + i] == j) ok = false;
        }
        for (uint32_t k = 0; k < spill_ne; ++k) {
          if (p.spill_excl[spill_off + k] == j) ok = false;
        }
      }
      m = __builtin_amdgcn_ballot_w64(ok);
    }
    return m;
  }
};

// Stored neighbours and overflow of a workgroup's atoms (stored: this lane's
// share of the total; over: some atom of this lane found more than fit).
__device__ __forceinline__ void publish_build(const BuildParams& p, uint32_t stored, bool over,
                                              double* red_lds) {
  const double total = block_sum<kBlock>(static_cast<double>(stored), red_lds);
  if (threadIdx.x == 0) {
    atomicAdd(&p.neighbor_parts[(blockIdx.x % kNeighborParts) * kNeighborPartStride],
              static_cast<unsigned long long>(total));
  }
  raise_flag(over, &p.ctrl->overflow);
}

// Full-list build with the append rule of full_neighbor_path_common.cuh:49-94:
// skip self, skip excluded, keep r2 <= r_s^2 (reference minimum image and
// operation order), overflow past max_neighbors. Each atom has a team of
// kBuildTeam adjacent lanes; lane t takes candidates k + u*kBuildTeam + t
// (u < kBuildSlots) of every candidate run, so the team's loads are
// consecutive 16-byte entries of the cell-ordered position stream (slot in
// .w), one load per candidate with no index gather; slots past a run's end
// load whatever follows it (the streams are padded past the last atom) and
// test nothing. Accepted candidates are appended in
// candidate order (the order of a one-lane scan) through a ballot of the
// team's lanes and written straight into the atom's chunks. EXCL: 0 = no
// exclusions, 4 or 8 = up to that many partners held in registers (every
// candidate within r_s is compared with all of them), -1 = any count read
// from memory. Also captures the positions the displacement check compares
// against. HALF keeps only partners with a higher slot, so every pair is
// stored once.
template <int EXCL, bool HALF>
__global__ __launch_bounds__(kBlock) void build_kernel(BuildParams p) {
  if (p.ctrl->rebuild == 0 || p.ctrl->stalled != 0) {
    return;
  }
  __shared__ double red_lds[4];
  const uint32_t t = threadIdx.x & (kBuildTeam - 1);
  const uint32_t team_lane0 = (threadIdx.x & 63u) & ~static_cast<uint32_t>(kBuildTeam - 1);
  const uint32_t below = (1u << t) - 1u;
  // The workgroup's atoms: kBuildAtoms consecutive entries of the candidate
  // stream (cell order) on the cell paths, consecutive slots on the direct
  // path.
  const uint32_t q = xcd_block(blockIdx.x, gridDim.x) * kBuildAtoms + threadIdx.x / kBuildTeam;
  const uint32_t i = q < p.n && p.grid.path != 0 ? id_of(p.cell_pos[q].w) : q;
  uint32_t count = 0;  // the same in every lane of a team
  // Rows path: each team's row runs, and the workgroup's span of each row,
  // staged in LDS (stage_off[r] - lo[r] is row r's stream-to-LDS offset)
  // when the spans fit; the teams then read their candidates from LDS.
  __shared__ uint2 row_lds[kBuildAtoms * kRows];
  extern __shared__ real4 stage[];  // p.stage_cap + kCandidatePad entries
  __shared__ uint32_t row_lo[kRows], row_hi[kRows], stage_off[kRows + 1];
  if (threadIdx.x < kRows) {
    row_lo[threadIdx.x] = 0xffffffffu;
    row_hi[threadIdx.x] = 0u;
  }
  __syncthreads();
  uint2* const team_rows = row_lds + (threadIdx.x / kBuildTeam) * kRows;
  const bool rows_path = i < p.n && row_runs(p, i, t, team_rows, row_lo, row_hi);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t off = 0;
    for (int r = 0; r < kRows; ++r) {
      stage_off[r] = off;
      off += row_hi[r] > row_lo[r] ? row_hi[r] - row_lo[r] : 0u;
    }
    stage_off[kRows] = off;
  }
  __syncthreads();
  const bool staged = stage_off[kRows] <= p.stage_cap;  // uniform over the workgroup
  if (staged) {
    for (int r = 0; r < kRows; ++r) {
      const uint32_t len = stage_off[r + 1] - stage_off[r];
      for (uint32_t k = threadIdx.x; k < len; k += kBlock) {
        stage[stage_off[r] + k] = p.cell_pos[row_lo[r] + k];
      }
    }
    if (rows_path) {
      // Re-base this lane's rows onto the stage (nonempty runs lie inside
      // their row's span).
      for (uint32_t r = t; r < static_cast<uint32_t>(kRows); r += kBuildTeam) {
        const uint2 d = team_rows[r];
        const uint32_t b_run = d.x, e_run = d.y & kRunIndexMask;
        if (b_run < e_run) {
          const uint32_t shift = stage_off[r] - row_lo[r];
          team_rows[r] = make_uint2(b_run + shift, ((e_run + shift) & kRunIndexMask) | (d.y & ~kRunIndexMask));
        }
      }
    }
  }
  __syncthreads();
  if (i < p.n) {  // uniform over a team
    const real4 xi = p.pos[i];
    const uint32_t n = p.n;
    const BuildAccept<EXCL, HALF> accept(p, i, xi);
    const real_t L0 = p.box.L[0], L1 = p.box.L[1], L2 = p.box.L[2];
    const uint32_t maxn = p.max_neighbors;
    // Candidates [b, e) of a run (b < e) whose entry s is entry(s) = {x, y,
    // z, slot bits}, kBuildTeam * kBuildSlots per round.
    // Atom i's entries of chunk c start at c * chunk_words + row_word.
    const uint32_t row_word = i * kNbrChunk;
    const uint32_t chunk_words = n * kNbrChunk;
    // One round: candidates k + u * kBuildTeam + t (u < kBuildSlots) of the
    // run ending at e (k < e).
    auto round = [&](uint32_t k, uint32_t e, auto entry, auto mode, real3 sh) {
      // Entries past the run (at most kCandidatePad - 1 past the stream's
      // last atom) are loaded and then ignored.
      static_assert(kBuildTeam * kBuildSlots <= kCandidatePad, "candidate padding");
      real4 x[kBuildSlots];
#pragma unroll
      for (int u = 0; u < kBuildSlots; ++u) {
        x[u] = entry(k + t, u);
      }
      // Slot u of this lane is in the run while u * kBuildTeam < left.
      const int left = static_cast<int>(e - k) - static_cast<int>(t);
#pragma unroll
      for (int u = 0; u < kBuildSlots; ++u) {
        const uint32_t j = id_of(x[u].w);
        const uint64_t m =
            __builtin_amdgcn_ballot_w64(u * kBuildTeam < left) & accept(j, x[u], mode, sh);
        const uint32_t bits = static_cast<uint32_t>(m >> team_lane0) & ((1u << kBuildTeam) - 1u);
        if (__builtin_amdgcn_inverse_ballot_w64(m)) {
          const uint32_t slot = count + __builtin_popcount(bits & below);
          if (slot < maxn) {
            // Entry (chunk slot / kNbrChunk, atom i, slot % kNbrChunk);
            // a chunk holds n * kNbrChunk < 2^32 entries.
            const uint64_t w = static_cast<uint64_t>(slot / kNbrChunk) * chunk_words +
                               (row_word | (slot & (kNbrChunk - 1)));
            p.nbr[w] = j;
          }
        }
        count += __builtin_popcount(bits);
      }
    };
    auto scan_range = [&](uint32_t b, uint32_t e, auto entry, auto mode, real3 sh) {
      for (uint32_t k = b; k < e; k += kBuildTeam * kBuildSlots) {
        round(k, e, entry, mode, sh);
      }
    };
    const real3 no_shift = make_real3(0, 0, 0);
    // entry(k0, u): the stream's entry k0 + u * kBuildTeam, addressed by a
    // 32-bit byte offset from the stream's base ((n + kCandidatePad) *
    // sizeof(real4) < 2^32) plus u's constant, so that the slots of a round
    // are immediate offsets of one address.
    constexpr uint32_t kEntryBytes = sizeof(real4);
    constexpr size_t kSlotBytes = kBuildTeam * sizeof(real4);
    if (p.grid.path == 0) {
      const char* pos_bytes = reinterpret_cast<const char*>(p.pos);
      const auto entry = [pos_bytes](uint32_t k0, int u) {
        const real4 q = *reinterpret_cast<const real4*>(
            pos_bytes + static_cast<size_t>(k0 * kEntryBytes) + u * kSlotBytes);
        return make_real4(q.x, q.y, q.z, real_of_id(k0 + u * kBuildTeam));
      };
      scan_range(0, n, entry, kGenericMode{}, no_shift);
    } else {
      const uint32_t c = p.cell_of[i];
      const CellGridView& g = p.grid;
      const uint32_t cx = c % g.nx, cyz = c / g.nx, cy = cyz % g.ny, cz = cyz / g.ny;
      const char* cp_bytes = reinterpret_cast<const char*>(p.cell_pos);
      const auto entry = [cp_bytes](uint32_t k0, int u) {
        return *reinterpret_cast<const real4*>(
            cp_bytes + static_cast<size_t>(k0 * kEntryBytes) + u * kSlotBytes);
      };
      // The team's rows in order, one run after another: a team moves to its
      // next row as soon as its run ends, so that the wave's lanes wait only
      // for the team with the most rounds in all, not in each row.
      auto scan_rows = [&](auto row_entry) {
        uint32_t r = 0, k = 0, e = 0;
        real3 sh = make_real3(0, 0, 0);
        for (;;) {
          if (k >= e) {
            bool more = true;
            do {
              if (r == static_cast<uint32_t>(kRows)) {
                more = false;
                break;
              }
              const uint2 d = team_rows[r++];
              k = d.x;
              e = d.y & kRunIndexMask;
              const uint32_t code = d.y >> kRunCodeShift;
              sh = make_real3(0, shift_of(code & 3u, L1), shift_of(code >> 2, L2));
            } while (k >= e);
            if (!more) break;
          }
          round(k, e, row_entry, kShiftYZMode{}, sh);
          k += kBuildTeam * kBuildSlots;
        }
      };
      // Boundary cells, grids of fewer than 5 cells per axis, and any grid while
      // some atom is outside the cells (then nothing is pruned, and a wrapped
      // cell says nothing about the image): the rows one after another, each
      // one run or two.
      const bool pruned = p.ctrl->outside == 0;
      auto rows_in_turn = [&](auto mode) {
#pragma unroll 1
        for (uint32_t r = 0; r < static_cast<uint32_t>(kRows); ++r) {
          const RunPair q = row_run_pair(g, p.box, p.rs2, p.cell_start, p.cell_xbins, pruned, xi,
                                         cx, cy, cz, r);
#pragma unroll 1
          for (int part = 0; part < 2; ++part) {
            const uint2 d = part == 0 ? q.a : q.b;
            const uint32_t yz = d.y >> kRunCodeShift;
            scan_range(d.x & kRunIndexMask, d.y & kRunIndexMask, entry, mode,
                       make_real3(shift_of(d.x >> kRunCodeShift, L0), shift_of(yz & 3u, L1),
                                  shift_of(yz >> 2, L2)));
          }
        }
      };
      if (rows_path && staged) {
        scan_rows([](uint32_t k0, int u) { return stage[k0 + u * kBuildTeam]; });
      } else if (rows_path) {
        scan_rows(entry);
      } else if (pruned && g.path == 1 && g.nx >= 5 && g.ny >= 5 && g.nz >= 5) {
        rows_in_turn(kShiftMode{});
      } else {
        rows_in_turn(kGenericMode{});
      }
    }
    if (t == 0) {
      p.nbr_count[i] = min(count, maxn);
      p.ref_pos[i] = xi;
      p.ref_image[i] = p.image[i];
    }
  }
  const bool counted = t == 0 && i < p.n;
  publish_build(p, counted ? min(count, p.max_neighbors) : 0u, counted && count > p.max_neighbors,
                red_lds);
}

// The build for systems whose atoms make too few waves at kBuildTeam lanes
// each: TEAM lanes per atom, no LDS stage and no workgroup-wide phase. What
// bounds the smallest is one atom's serial chain (its runs' bounds, then a load
// per round), so the next round's candidates are in flight while this one's are
// tested; larger ones are bound by the candidates tested, so a round is two
// slots a lane: with four, half of a short row's round is idle (100,000-bead
// mixture 78 us against 65, 48,000-bead melt 66 against 58).
constexpr int kWideSlots = 2;

template <int EXCL, bool HALF, int TEAM>
__global__ __launch_bounds__(kBlock) void build_wide_kernel(BuildParams p) {
  if (p.ctrl->rebuild == 0 || p.ctrl->stalled != 0) {
    return;
  }
  constexpr uint32_t kWideAtoms = kBlock / TEAM;
  __shared__ double red_lds[4];
  __shared__ uint2 run_lds[kWideAtoms * kMaxRuns];
  const uint32_t t = threadIdx.x & (TEAM - 1);
  const uint32_t team_lane0 = (threadIdx.x & 63u) & ~static_cast<uint32_t>(TEAM - 1);
  const uint32_t q = xcd_block(blockIdx.x, gridDim.x) * kWideAtoms + threadIdx.x / TEAM;
  uint2* const runs = run_lds + (threadIdx.x / TEAM) * kMaxRuns;
  const bool direct = p.grid.path == 0;
  const bool pruned = p.ctrl->outside == 0;  // as in build_kernel
  const CellGridView& g = p.grid;
  real4 xi = make_real4(0, 0, 0, 0);
  uint32_t i = q, n_runs = 0, count = 0;
  if (q < p.n) {  // uniform over a team
    if (direct) {
      xi = p.pos[q];
      if (t == 0) runs[0] = make_uint2(0u, p.n);
      n_runs = 1;
    } else {
      xi = p.cell_pos[q];  // the atom's position, .w its slot
      i = id_of(xi.w);
      n_runs = team_runs<TEAM>(g, p.box, p.rs2, p.cell_start, p.cell_xbins, pruned, xi,
                               cell_of_position(xi, p.box, g), t, team_lane0, runs);
    }
  }
  __syncthreads();
  if (q < p.n) {
    const BuildAccept<EXCL, HALF> accept(p, i, xi);
    const uint32_t maxn = p.max_neighbors;
    const uint32_t row_word = i * kNbrChunk;
    const uint32_t chunk_words = p.n * kNbrChunk;
    const auto put = [&](uint32_t slot, uint32_t j) {
      if (slot < maxn) {
        p.nbr[static_cast<uint64_t>(slot / kNbrChunk) * chunk_words +
              (row_word | (slot & (kNbrChunk - 1)))] = j;
      }
    };
    if (direct) {
      const auto entry = [&](uint32_t k) {
        const real4 x = p.pos[k];
        return make_real4(x.x, x.y, x.z, real_of_id(k));
      };
      count = scan_runs<TEAM, kWideSlots>(runs, n_runs, t, team_lane0, p.box, entry, accept,
                                               put, kGenericMode{});
    } else {
      const char* cp_bytes = reinterpret_cast<const char*>(p.cell_pos);
      const auto entry = [cp_bytes](uint32_t k) {
        return *reinterpret_cast<const real4*>(cp_bytes +
                                               k * static_cast<uint32_t>(sizeof(real4)));
      };
      if (pruned && g.nx >= 5 && g.ny >= 5 && g.nz >= 5) {
        count = scan_runs<TEAM, kWideSlots>(runs, n_runs, t, team_lane0, p.box, entry, accept,
                                                 put, kShiftMode{});
      } else {
        count = scan_runs<TEAM, kWideSlots>(runs, n_runs, t, team_lane0, p.box, entry, accept,
                                                 put, kGenericMode{});
      }
    }
    if (t == 0) {
      p.nbr_count[i] = min(count, maxn);
      p.ref_pos[i] = xi;
      p.ref_image[i] = p.image[i];
    }
  }
  const bool counted = t == 0 && q < p.n;
  publish_build(p, counted ? min(count, p.max_neighbors) : 0u, counted && count > p.max_neighbors,
                red_lds);
}

// ------------------------------------------------------------------ force --

// LJ over one atom's stored list by one lane (pair_lj.cu:21-167), used by the
// half-list pair pass. The loop reads two 16-byte quads of indices and issues
// the eight position gathers together before any arithmetic. The decision
// r^2 < r_c^2 is binary32 on the exact-intermediate minimum image; the pair
// value is FP64. REACT adds the reaction -s d of every pair to pair_acc[j].
// TYPES: 0 = single type (coefficients in registers), 1 = table in LDS,
// 2 = table in global memory.
template <bool OBS, int TYPES, bool REACT>
__device__ __forceinline__ void lj_list(const ForceParams& p, uint32_t i, real4 xi4,
                                        const LjCoeff* lj_lds, const LjCoeff& c0, double& fxd,
                                        double& fyd, double& fzd, double& e_pair,
                                        double& w_pair) {
  const int T = p.n_types;
  const int ti = static_cast<int>(id_of(xi4.w));
  const uint32_t n = p.n;
  const real_t L0 = p.box.L[0], L1 = p.box.L[1], L2 = p.box.L[2];
  const real_t h0 = p.box.hL[0], h1 = p.box.hL[1], h2 = p.box.hL[2];
  const uint32_t cnt = p.nbr_count[i];
  // Eight slots per iteration: both index quads of a half chunk, then eight
  // gathers in flight before any arithmetic. Slots at or past cnt gather
  // atom i itself (never used), so every load stays inside pos and inside the
  // atom's allocated chunks (kNbrChunk is a multiple of 8).
  static_assert(kNbrChunk % 8 == 0, "neighbour chunks hold whole 8-slot groups");
  for (uint32_t base = 0; base < cnt; base += 8) {
    const uint32_t* cp = p.nbr + nbr_chunk_base(base / kNbrChunk, i, n) + (base & (kNbrChunk - 1));
    const uint4 qa = *reinterpret_cast<const uint4*>(cp);
    const uint4 qb = *reinterpret_cast<const uint4*>(cp + 4);
    const uint32_t jj[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
    real4 xj[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      xj[u] = p.pos[base + u < cnt ? jj[u] : i];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const real_t dx = mic_diff(xi4.x, xj[u].x, L0, h0);
      const real_t dy = mic_diff(xi4.y, xj[u].y, L1, h1);
      const real_t dz = mic_diff(xi4.z, xj[u].z, L2, h2);
      const real_t r2 = r2_strict(dx, dy, dz);
      if (base + u < cnt && r2 < p.rc2) {
        LjCoeff c;
        if (TYPES == 0) {
          c = c0;
        } else if (TYPES == 1) {
          c = lj_lds[ti * T + static_cast<int>(id_of(xj[u].w))];
        } else {
          c = p.lj[ti * T + static_cast<int>(id_of(xj[u].w))];
        }
        double rr, u_pair;
        const double s = lj_pair(dx, dy, dz, c, rr, u_pair);
        fxd += s * dx;
        fyd += s * dy;
        fzd += s * dz;
        if (REACT) {
          double* acc = p.pair_acc + 3 * static_cast<size_t>(jj[u]);
          unsafeAtomicAdd(acc, -s * dx);
          unsafeAtomicAdd(acc + 1, -s * dy);
          unsafeAtomicAdd(acc + 2, -s * dz);
        }
        if (OBS) {
          e_pair += u_pair;
          w_pair += s * rr;
        }
      }
    }
  }
}

// LJ over atom i's stored list, shared by the TEAM lanes of its team: lane t
// takes slots base + u*TEAM + t, u < SLOTS, and keeps FP64 partial sums
// (pair_lj.cu:21-167; same decision and pair value as lj_list). Slots at or
// past cnt neither load an index nor count; they gather atom i itself.
template <bool OBS, int TYPES, int TEAM, int SLOTS>
__device__ __forceinline__ void lj_team(const ForceParams& p, uint32_t i, uint32_t t, real4 xi4,
                                        const LjCoeff* lj_lds, const LjCoeff& c0, double& fxd,
                                        double& fyd, double& fzd, double& e_pair,
                                        double& w_pair) {
  static_assert(kNbrChunk % TEAM == 0, "a team's slots of one load share a chunk");
  static_assert(kNbrRound % (TEAM * SLOTS) == 0, "a round stays inside the padded capacity");
  const int T = p.n_types;
  const int ti = static_cast<int>(id_of(xi4.w));
  const uint32_t n = p.n;
  const real_t L0 = p.box.L[0], L1 = p.box.L[1], L2 = p.box.L[2];
  const real_t h0 = p.box.hL[0], h1 = p.box.hL[1], h2 = p.box.hL[2];
  const real_t xm0 = xi4.x - L0, xm1 = xi4.y - L1, xm2 = xi4.z - L2;
  const real_t hmin = shortest_half(p.box);
  const uint32_t cnt = p.nbr_count[i];
  for (uint32_t base = 0; base < cnt; base += TEAM * SLOTS) {
    // Every slot of the round lies inside the atom's padded capacity; slots
    // at or past the count read whatever the chunk holds and become i.
    uint32_t jj[SLOTS];
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      const uint32_t s = base + u * TEAM + t;
      jj[u] = p.nbr[nbr_chunk_base(s / kNbrChunk, i, n) + (s & (kNbrChunk - 1))];
    }
    // slot base + u * TEAM + t holds a neighbour iff u * TEAM < rem
    const int rem = static_cast<int>(cnt) - static_cast<int>(base + t);
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      jj[u] = u * TEAM < rem ? jj[u] : i;
    }
    // Gathers as a 32-bit byte offset from the array base (n * sizeof(real4)
    // < 2^32, checked at set-up).
    const char* pos_bytes = reinterpret_cast<const char*>(p.pos);
    real4 xj[SLOTS];
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      xj[u] = *reinterpret_cast<const real4*>(
          pos_bytes + jj[u] * static_cast<uint32_t>(sizeof(real4)));
    }
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      // mic_diff_sel returns the raw difference unless it exceeds half the
      // box; the folded forms are formed only when some lane of the wave
      // may need them (pairs across a periodic boundary), the same values.
      real_t dx = xi4.x - xj[u].x;
      real_t dy = xi4.y - xj[u].y;
      real_t dz = xi4.z - xj[u].z;
      if (past_half(dx, dy, dz, hmin)) {
        dx = mic_diff_sel(xi4.x, xm0, xj[u].x, L0, h0);
        dy = mic_diff_sel(xi4.y, xm1, xj[u].y, L1, h1);
        dz = mic_diff_sel(xi4.z, xm2, xj[u].z, L2, h2);
      }
      const real_t r2 = r2_strict(dx, dy, dz);
      if (u * TEAM < rem && r2 < p.rc2) {
        LjCoeff c;
        if (TYPES == 0) {
          c = c0;
        } else if (TYPES == 1) {
          c = lj_lds[ti * T + static_cast<int>(id_of(xj[u].w))];
        } else {
          c = p.lj[ti * T + static_cast<int>(id_of(xj[u].w))];
        }
        double rr, u_pair;
        const double s = lj_pair(dx, dy, dz, c, rr, u_pair);
        fxd += s * dx;
        fyd += s * dy;
        fzd += s * dz;
        if (OBS) {
          e_pair += u_pair;
          w_pair += s * rr;
        }
      }
    }
  }
}

template <int TYPES>
__device__ __forceinline__ void load_lj_table(const ForceParams& p, LjCoeff* lj_lds) {
  if (TYPES == 1) {
    for (int k = threadIdx.x; k < p.n_types * p.n_types; k += kBlock) {
      lj_lds[k] = p.lj[k];
    }
    __syncthreads();
  }
}

// Half-list pair pass (no reference counterpart; the reference keeps a full
// list): every stored pair (i, j > i) is evaluated once, the force on i is
// summed in registers and the reaction on j added to pair_acc with FP64
// atomics; i's own sum is added last. Pair energy and virial are summed per
// workgroup and added to ctrl->half_pair. The force pass that follows adds the
// listed terms, kicks, reduces and clears pair_acc.
template <bool OBS, int TYPES>
__global__ __launch_bounds__(kBlock) void half_pair_kernel(ForceParams p) {
  __shared__ LjCoeff lj_lds[TYPES == 1 ? kMaxLdsTypes * kMaxLdsTypes : 1];
  __shared__ double red_lds[4];
  load_lj_table<TYPES>(p, lj_lds);
  const LjCoeff c0 = TYPES == 0 ? p.lj[0] : LjCoeff{0.0, 0.0, 0.0, 0.0};
  const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  double e_pair = 0.0, w_pair = 0.0;
  if (i < p.n) {
    double fxd = 0.0, fyd = 0.0, fzd = 0.0;
    lj_list<OBS, TYPES, true>(p, i, p.pos[i], lj_lds, c0, fxd, fyd, fzd, e_pair, w_pair);
    double* acc = p.pair_acc + 3 * static_cast<size_t>(i);
    unsafeAtomicAdd(acc, fxd);
    unsafeAtomicAdd(acc + 1, fyd);
    unsafeAtomicAdd(acc + 2, fzd);
  }
  if (OBS) {
    const double e = block_sum<kBlock>(e_pair, red_lds);
    const double w = block_sum<kBlock>(w_pair, red_lds);
    if (threadIdx.x == 0) {
      unsafeAtomicAdd(&p.ctrl->half_pair[0], e);
      unsafeAtomicAdd(&p.ctrl->half_pair[1], w);
    }
  }
}

// Atom i's total force (rounded once from FP64), the force store, optionally
// the post-force half-kick (velocity_verlet.cu:97-111), and the atom's
// kinetic energy. Run by one lane of the team.
template <bool KICK>
__device__ __forceinline__ void finish_atom(const ForceParams& p, uint32_t i, double fxd,
                                            double fyd, double fzd, StepSums& sums) {
  const real_t fx = static_cast<real_t>(fxd);
  const real_t fy = static_cast<real_t>(fyd);
  const real_t fz = static_cast<real_t>(fzd);
  p.force[i] = make_real4(fx, fy, fz, 0);
  real4 v = p.vel[i];
  if (KICK) {
    const real_t h = real_t(0.5) * p.dt / v.w;
    v.x += h * fx;
    v.y += h * fy;
    v.z += h * fz;
    p.vel[i] = v;
  }
  const double vx = v.x, vy = v.y, vz = v.z;
  sums.ke += 0.5 * static_cast<double>(v.w) * (vx * vx + vy * vy + vz * vz);
}

// Workgroup sums of one force pass: thread 0 writes partials[q * nbk + block]
// (q = 0 kinetic energy; with OBS 1..4 energies, 5..8 virials).
template <bool OBS>
__device__ __forceinline__ void store_step_partials(const ForceParams& p, const StepSums& sums,
                                                    double* red_lds) {
  const uint32_t nbk = gridDim.x;
  double* part = p.partials;
  double s = block_sum<kBlock>(sums.ke, red_lds);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
  if (OBS) {
    const double vals[8] = {0.5 * sums.e_pair, sums.e_bond, sums.e_angle, sums.e_dih,
                            0.5 * sums.w_pair, sums.w_bond, sums.w_angle, sums.w_dih};
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      s = block_sum<kBlock>(vals[q], red_lds);
      if (threadIdx.x == 0) part[(q + 1) * static_cast<size_t>(nbk) + blockIdx.x] = s;
    }
  }
}

// One workgroup after the force pass: FP64 totals of the nbk workgroups'
// partials and the Berendsen factor (berendsen_thermostat.cu:109-163). Steps
// whose sums nobody reads (ForceParams::sums) do without it. A kernel of its own, so the force pass publishes
// its partials at the kernel boundary instead of with a device-scope fence
// (an L2 write-back and invalidate on gfx950) in every workgroup.
constexpr int kReduceBlock = 1024;

// This thread's shares of NQ arrays v[q * n ..][0..n) for kReduceBlock-wide
// sums: elements threadIdx.x + m*kReduceBlock, four loads of each array in
// flight.
template <int NQ>
__device__ __forceinline__ void strided_sums(const double* v, uint32_t n, double* out) {
  double a[NQ][4] = {};
  uint32_t b = threadIdx.x;
  for (; b + 3 * kReduceBlock < n; b += 4 * kReduceBlock) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
#pragma unroll
      for (int m = 0; m < 4; ++m) a[q][m] += v[q * static_cast<size_t>(n) + b + m * kReduceBlock];
    }
  }
  for (; b < n; b += kReduceBlock) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) a[q][0] += v[q * static_cast<size_t>(n) + b];
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) out[q] = (a[q][0] + a[q][1]) + (a[q][2] + a[q][3]);
}

// All sums at once: with observables a chain of nine sums one after another,
// each a pass of loads and two barriers, took 13 us at 100,000 atoms and 35 us
// at 1,000,000; together they take 8.4 and 26.
template <bool KICK, bool OBS, bool HALF>
__global__ __launch_bounds__(kReduceBlock) void step_reduce_kernel(ForceParams p, uint32_t nbk) {
  constexpr int kSums = OBS ? 9 : 1;
  constexpr int kWaves = kReduceBlock / 64;
  __shared__ double lds[kSums][kWaves];
  double part[kSums];
  strided_sums<kSums>(p.partials, nbk, part);
#pragma unroll
  for (int q = 0; q < kSums; ++q) {
    part[q] = wave_sum(part[q]);
    if ((threadIdx.x & 63u) == 0) lds[q][threadIdx.x >> 6] = part[q];
  }
  __syncthreads();
  const int q = static_cast<int>(threadIdx.x);
  if (q < kSums) {
    double acc = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) acc += lds[q][w];
    Ctrl* ctrl = p.ctrl;
    if (q == 0) {
      ctrl->ke_pre = acc;
      double lambda = 1.0;
      if (KICK && p.berendsen && acc > 0.0 && p.dof > 0.0) {
        const double current = 2.0 * acc / p.dof;
        const double arg = 1.0 + p.dt_over_tau * (p.target_thermal / current - 1.0);
        lambda = sqrt(arg > 0.0 ? arg : 0.0);
      }
      ctrl->lambda = lambda;
      if (!KICK) ctrl->ke = acc;
    } else if (q <= 4) {
      ctrl->pe[q - 1] = (HALF && q == 1) ? ctrl->half_pair[0] : acc;
    } else {
      ctrl->virial[q - 5] = (HALF && q == 5) ? ctrl->half_pair[1] : acc;
    }
  }
  if (HALF) {
    __syncthreads();  // half_pair is read before it is cleared
    if (threadIdx.x == 0) {
      p.ctrl->half_pair[0] = 0.0;
      p.ctrl->half_pair[1] = 0.0;
    }
  }
}

// Fused force pass: LJ over the stored full list (pair_lj.cu:21-167), or the
// half-list pair pass's sums (HALF), plus the listed terms, then optionally
// the post-force half-kick (velocity_verlet.cu:97-111) and the kinetic-energy
// reduction for the Berendsen factor (berendsen_thermostat.cu:109-163) as
// per-workgroup partials, which step_reduce_kernel totals in FP64.
//
// Each atom has a team of TEAM adjacent lanes. Lane t reads list slots
// base + u*TEAM + t (u < SLOTS), so one gather instruction fetches
// TEAM consecutive entries of each of the wave's 64/TEAM lists: mostly
// consecutive slots of one cell, a few cache lines per atom instead of one
// line per lane. The team's FP64 partial sums meet in a shuffle butterfly and
// the atom's total is rounded to binary32 once.
template <bool KICK, bool OBS, int TYPES, bool HALF, bool SPILL, bool LISTED, int TEAM, int SLOTS>
__global__ __launch_bounds__(kBlock) void force_kernel(ForceParams p) {
  __shared__ LjCoeff lj_lds[TYPES == 1 && !HALF ? kMaxLdsTypes * kMaxLdsTypes : 1];
  __shared__ double red_lds[4];
  if (!HALF) load_lj_table<TYPES>(p, lj_lds);
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // the step's rebuild is done
    p.ctrl->rebuild = 0;
    p.ctrl->reorder = 0;
    p.ctrl->joined = 0;
    p.ctrl->outside = 0;
  }
  const LjCoeff c0 = TYPES == 0 && !HALF ? p.lj[0] : LjCoeff{0.0, 0.0, 0.0, 0.0};
  const uint32_t t = threadIdx.x & (TEAM - 1);
  const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * (kBlock / TEAM) + threadIdx.x / TEAM;
  StepSums sums;
  if (i < p.n) {  // uniform over a team
    const real4 xi4 = p.pos[i];
    double fxd = 0.0, fyd = 0.0, fzd = 0.0;
    if (HALF) {
      if (t == 0) {
        double* acc = p.pair_acc + 3 * static_cast<size_t>(i);
        fxd = acc[0];
        fyd = acc[1];
        fzd = acc[2];
        acc[0] = 0.0;
        acc[1] = 0.0;
        acc[2] = 0.0;
      }
    } else {
      lj_team<OBS, TYPES, TEAM, SLOTS>(p, i, t, xi4, lj_lds, c0, fxd, fyd, fzd, sums.e_pair, sums.w_pair);
    }
    if (LISTED && p.topo.has_listed) {
      listed_team<OBS, SPILL, TEAM>(p.pos, p.topo, p.box, p.n, i, t, xi4, fxd, fyd, fzd, sums);
    }
    fxd = team_sum<TEAM>(fxd);
    fyd = team_sum<TEAM>(fyd);
    fzd = team_sum<TEAM>(fzd);
    if (t == 0) {
      finish_atom<KICK>(p, i, fxd, fyd, fzd, sums);
    }
  }
  if (p.sums) store_step_partials<OBS>(p, sums, red_lds);
}

// Apply the pending Berendsen factor and reduce the kinetic energy of the
// stored velocities (output steps; berendsen_thermostat.cu:135-163 and
// thermo_output.cu:60-85).
template <bool THERMO>
__global__ __launch_bounds__(kBlock) void scale_kernel(ScaleParams p) {
  __shared__ double red_lds[4];
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  double ke = 0.0;
  if (i < p.n) {
    real4 v = p.vel[i];
    if (THERMO) {
      const real_t lam = static_cast<real_t>(p.ctrl->lambda);
      v.x *= lam;
      v.y *= lam;
      v.z *= lam;
      p.vel[i] = v;
    }
    const double vx = v.x, vy = v.y, vz = v.z;
    ke = 0.5 * static_cast<double>(v.w) * (vx * vx + vy * vy + vz * vz);
  }
  const double s = block_sum<kBlock>(ke, red_lds);
  if (threadIdx.x == 0) p.partials[blockIdx.x] = s;
}

// One workgroup after scale_kernel: FP64 total of its nbk partials.
__global__ __launch_bounds__(kReduceBlock) void scale_reduce_kernel(ScaleParams p, uint32_t nbk) {
  __shared__ double red_lds[kReduceBlock / 64];
  double part[1];
  strided_sums<1>(p.partials, nbk, part);
  const double acc = block_sum<kReduceBlock>(part[0], red_lds);
  if (threadIdx.x == 0) {
    p.ctrl->ke = acc;
    p.ctrl->lambda = 1.0;
  }
}

// Pending Berendsen factor, first half-kick, drift and wrap
// (velocity_verlet.cu:59-95; box_geometry_view.cuh:92-102), then the
// displacement test against the last build (rebuild_tracker.cu:55-94).
template <bool THERMO, bool CHECK>
__global__ __launch_bounds__(kBlock) void integrate_kernel(IntegrateParams p) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= p.n) {
    return;
  }
  real4 v = p.vel[i];
  const real4 f = p.force[i];
  real4 x = p.pos[i];
  if (THERMO) {
    // Rounded on its own, as the reference's separate rescale kernel and
    // scale_kernel (output steps) round it: never fused into the kick.
#pragma clang fp contract(off)
    const real_t lam = static_cast<real_t>(p.ctrl->lambda);
    v.x *= lam;
    v.y *= lam;
    v.z *= lam;
  }
  const real_t h = real_t(0.5) * p.dt / v.w;
  v.x += h * f.x;
  v.y += h * f.y;
  v.z += h * f.z;
  x.x += p.dt * v.x;
  x.y += p.dt * v.y;
  x.z += p.dt * v.z;
  real_t c[3];
  {
#pragma clang fp contract(off)
    c[0] = floor((x.x - p.box.lo[0]) * p.box.invL[0]);
    c[1] = floor((x.y - p.box.lo[1]) * p.box.invL[1]);
    c[2] = floor((x.z - p.box.lo[2]) * p.box.invL[2]);
    x.x -= c[0] * p.box.L[0];
    x.y -= c[1] * p.box.L[1];
    x.z -= c[2] * p.box.L[2];
  }
  p.pos[i] = x;
  p.vel[i] = v;
  const bool wrapped = c[0] != real_t(0) || c[1] != real_t(0) || c[2] != real_t(0);
  int4 im = make_int4(0, 0, 0, 0);
  if (wrapped || CHECK) {
    im = p.image[i];
  }
  if (wrapped) {
    im.x += static_cast<int>(c[0]);
    im.y += static_cast<int>(c[1]);
    im.z += static_cast<int>(c[2]);
    p.image[i] = im;
  }
  if (CHECK) {
#pragma clang fp contract(off)
    const real4 r = p.ref_pos[i];
    const int4 ri = p.ref_image[i];
    const real_t dx = (x.x - r.x) + static_cast<real_t>(im.x - ri.x) * p.box.L[0];
    const real_t dy = (x.y - r.y) + static_cast<real_t>(im.y - ri.y) * p.box.L[1];
    const real_t dz = (x.z - r.z) + static_cast<real_t>(im.z - ri.z) * p.box.L[2];
    raise_flag(dx * dx + dy * dy + dz * dz > p.threshold_sq, &p.ctrl->rebuild);
  }
}


}  // namespace

void launch_control(Ctrl* ctrl, NeighborControl control, bool forced, uint64_t steps,
                    unsigned long long* neighbor_parts, hipStream_t stream) {
  control_kernel<<<1, kNeighborParts, 0, stream>>>(ctrl, control, forced ? 1 : 0, steps,
                                                   neighbor_parts);
}

void launch_rebuild(const CellScanParams& cells, const ReorderParams& reorder,
                    const RebuildParams& p, hipStream_t stream) {
  // More workgroups than the atoms fill shorten the per-cell phase; four times
  // as many as kRebuildBlock asks for took 39 instead of 43 us per rebuild at
  // 100,000 atoms, 26 instead of 30 at 48,000 and 25 instead of 27 at 4,000.
  // Half the cap costs 134 instead of 85 us at 1,000,000.
  const unsigned g = grid_for(cells.n, kRebuildBlock / 4);
  rebuild_kernel<<<g < kRebuildMaxBlocks ? g : kRebuildMaxBlocks, kRebuildBlock, 0, stream>>>(
      cells, reorder, p);
}

void launch_pack_records(const PackParams& p, hipStream_t stream) {
  pack_records_kernel<<<grid_for(p.n), kBlock, 0, stream>>>(p);
}

// Atoms up to which the wide build is used, and its 32-lane shape. Measured,
// 4 lanes / 16 / 32, us per build (equilibrated systems): LJ fluid of 4,000
// beads 65 / 18 / 14, of 32,000 65 / 32 / 39; bead-spring melt of 8,000
// 96 / 24 / 21, of 48,000 103 / 58 / 67. 4 / 16 around the upper line: melt of
// 100,000 144 / 100, of 150,000 166 / 140, of 216,000 210 / 196, of 288,000
// 247 / 255; fluid of 108,000 99 / 82, of 144,000 112 / 106, of 256,000
// 162 / 175; mixture of 100,000 77 / 66, of 150,000 96 / 91, of 216,000
// 124 / 125, of 288,000 150 / 162; solvent in a caller's order of 100,000
// 138 / 101, of 150,000 168 / 143, of 216,000 214 / 206, of 288,000 257 / 264.
// The upper line was set when nothing larger than 100,000 had been timed with
// two slots a round; by these figures it belongs at about 200,000.
constexpr uint32_t kWideBuild32Max = 12000;
constexpr uint32_t kWideBuildMax = 100000;

void launch_pack_state(const PackStateParams& p, hipStream_t stream) {
  pack_state_kernel<<<grid_for(p.n), kBlock, 0, stream>>>(p);
}

void launch_build(const BuildParams& params, hipStream_t stream) {
  const unsigned g = grid_for(params.n, kBuildAtoms);
  // Stage capacity from the mean cell occupancy m: a workgroup's kBuildAtoms
  // atoms span about kBuildAtoms / m cells of one row of cells, so each of the
  // kRows rows of the stencil holds about kBuildAtoms + 2m members; 15 %
  // margin, whole multiples of 64 entries, at most kStageBytesMax.
  BuildParams p = params;
  const double m = p.grid.n_cells > 0 ? static_cast<double>(p.n) / p.grid.n_cells : 0.0;
  const uint32_t want = static_cast<uint32_t>(1.15 * kRows * (kBuildAtoms + 2.0 * m) + 63.0) & ~63u;
  const uint32_t most = kStageBytesMax / sizeof(real4) - kCandidatePad;
  p.stage_cap = p.grid.path == 1 ? (want < most ? want : most) : 0u;
  const size_t lds = p.grid.path == 1 ? (p.stage_cap + kCandidatePad) * sizeof(real4) : 0;
  // Exclusion registers: the fewest of 4 / 8 that hold every slot's
  // exclusions (ecap is the largest count), else read from memory.
  const int ex = p.spill_index != nullptr
                     ? -1
                     : (p.ecap == 0 ? 0 : (p.ecap <= 4 ? 4 : (p.ecap <= 8 ? 8 : -1)));
  const int team = p.n <= kWideBuild32Max ? 32 : (p.n <= kWideBuildMax ? 16 : kBuildTeam);
  const unsigned gw = grid_for(params.n, kBlock / team);
#define BEADS_BUILD_CASE(E, H)                                          \
  if (ex == E && (p.half != 0) == H) {                                  \
    if (team == 32) {                                                   \
      build_wide_kernel<E, H, 32><<<gw, kBlock, 0, stream>>>(p);        \
    } else if (team == 16) {                                            \
      build_wide_kernel<E, H, 16><<<gw, kBlock, 0, stream>>>(p);        \
    } else {                                                            \
      build_kernel<E, H><<<g, kBlock, lds, stream>>>(p);                \
    }                                                                   \
  }
  BEADS_BUILD_CASE(0, false)
  BEADS_BUILD_CASE(4, false)
  BEADS_BUILD_CASE(8, false)
  BEADS_BUILD_CASE(-1, false)
  BEADS_BUILD_CASE(0, true)
  BEADS_BUILD_CASE(4, true)
  BEADS_BUILD_CASE(8, true)
  BEADS_BUILD_CASE(-1, true)
#undef BEADS_BUILD_CASE
}

// Lanes per atom and slots per lane of the force pass. Four lanes an atom cost
// least per slot and per listed term; below some tens of thousands of atoms
// they leave the GPU too few waves, and the pass lasts as long as one atom's
// chain of rounds and terms, which more lanes shorten. Measured 4x8 / 8x4 /
// 16x2, us per pass: LJ fluid of 500 beads 8.7 / 6.7 / 5.4, of 4,000
// 8.6 / 6.3 / 5.4, of 32,000 10.1 / 9.0 / 10.2; bead-spring melt of 8,000
// 14.2 / 10.7 / 10.7, of 18,000 16.8 / 14.6 / 14.8, of 48,000
// 22.5 / 23.1 / 29.1; mixture of 8,000 8.9 / 7.7 / 5.9, of 64,000
// 13.9 / 14.3 / 16.7. More slots in flight (8x8, 16x4, 16x8) gain at most 0.5
// us and would widen the lists' padding.
constexpr uint32_t kForceTeam16Max = 12000;
constexpr uint32_t kForceTeam8Max = 40000;

static ForceShape force_shape(uint32_t n) {
  if (n <= kForceTeam16Max) return {16, 2};
  if (n <= kForceTeam8Max) return {8, 4};
  return {4, 8};
}

void launch_force(const ForceParams& params, bool kick, bool obs, bool sums, hipStream_t stream) {
  ForceParams p = params;
  p.sums = sums ? 1 : 0;
  const unsigned g = grid_for(p.n);
  const int types = p.n_types == 1 ? 0 : (p.n_types <= kMaxLdsTypes ? 1 : 2);
  const bool half = p.half != 0;
  if (half) {
#define BEADS_HALF_CASE(O, T)                                           \
    if (obs == O && types == T) half_pair_kernel<O, T><<<g, kBlock, 0, stream>>>(p);
    BEADS_HALF_CASE(false, 0)
    BEADS_HALF_CASE(false, 1)
    BEADS_HALF_CASE(false, 2)
    BEADS_HALF_CASE(true, 0)
    BEADS_HALF_CASE(true, 1)
    BEADS_HALF_CASE(true, 2)
#undef BEADS_HALF_CASE
  }
  const bool spill = p.topo.spill_index != nullptr;
  // The half list's and the spill's variants exist in the widest-work shape only.
  const ForceShape shape = half || spill ? ForceShape{4, 8} : force_shape(p.n);
  const unsigned gf = grid_for(p.n, kBlock / shape.team);
#define BEADS_FORCE_SHAPE(K, O, T, N, S)                                               \
  if (shape.team == N && shape.slots == S) {                                           \
    if (p.topo.has_listed) {                                                           \
      force_kernel<K, O, T, false, false, true, N, S><<<gf, kBlock, 0, stream>>>(p);   \
    } else {                                                                           \
      force_kernel<K, O, T, false, false, false, N, S><<<gf, kBlock, 0, stream>>>(p);  \
    }                                                                                  \
  }
#define BEADS_FORCE_CASE(K, O, T)                                                      \
  if (kick == K && obs == O && (half || types == T)) {                                 \
    if (half) {                                                                        \
      if (spill) {                                                                     \
        force_kernel<K, O, 0, true, true, true, 4, 8><<<gf, kBlock, 0, stream>>>(p);         \
      } else {                                                                         \
        force_kernel<K, O, 0, true, false, true, 4, 8><<<gf, kBlock, 0, stream>>>(p);        \
      }                                                                                \
      if (sums) step_reduce_kernel<K, O, true><<<1, kReduceBlock, 0, stream>>>(p, gf); \
    } else {                                                                           \
      if (spill) {                                                                     \
        force_kernel<K, O, T, false, true, true, 4, 8><<<gf, kBlock, 0, stream>>>(p);        \
      } else {                                                                         \
        BEADS_FORCE_SHAPE(K, O, T, 4, 8)                                               \
        BEADS_FORCE_SHAPE(K, O, T, 8, 4)                                               \
        BEADS_FORCE_SHAPE(K, O, T, 16, 2)                                              \
      }                                                                                \
      if (sums) step_reduce_kernel<K, O, false><<<1, kReduceBlock, 0, stream>>>(p, gf); \
    }                                                                                  \
    return;                                                                            \
  }
  BEADS_FORCE_CASE(true, false, 0)
  BEADS_FORCE_CASE(true, false, 1)
  BEADS_FORCE_CASE(true, false, 2)
  BEADS_FORCE_CASE(true, true, 0)
  BEADS_FORCE_CASE(true, true, 1)
  BEADS_FORCE_CASE(true, true, 2)
  BEADS_FORCE_CASE(false, false, 0)
  BEADS_FORCE_CASE(false, false, 1)
  BEADS_FORCE_CASE(false, false, 2)
  BEADS_FORCE_CASE(false, true, 0)
  BEADS_FORCE_CASE(false, true, 1)
  BEADS_FORCE_CASE(false, true, 2)
#undef BEADS_FORCE_CASE
#undef BEADS_FORCE_SHAPE
}

void launch_integrate(const IntegrateParams& p, bool thermostat, bool check,
                      bool /*force_rebuild*/, hipStream_t stream) {
  const unsigned g = grid_for(p.n);
  if (thermostat) {
    if (check) integrate_kernel<true, true><<<g, kBlock, 0, stream>>>(p);
    else integrate_kernel<true, false><<<g, kBlock, 0, stream>>>(p);
  } else {
    if (check) integrate_kernel<false, true><<<g, kBlock, 0, stream>>>(p);
    else integrate_kernel<false, false><<<g, kBlock, 0, stream>>>(p);
  }
}

void launch_scale(const ScaleParams& p, bool thermostat, hipStream_t stream) {
  const unsigned g = grid_for(p.n);
  if (thermostat) scale_kernel<true><<<g, kBlock, 0, stream>>>(p);
  else scale_kernel<false><<<g, kBlock, 0, stream>>>(p);
  scale_reduce_kernel<<<1, kReduceBlock, 0, stream>>>(p, g);
}

}  // namespace beads_amd
