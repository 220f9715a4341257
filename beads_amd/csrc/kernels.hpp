// Host-side launchers for the gfx950 kernels in kernels.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "device.hpp"

namespace beads_amd {

constexpr int kBlock = 256;

struct CellScanParams {
  uint32_t n;
  uint32_t n_cells;
  uint32_t* cell_of;
  uint32_t* cell_count;
  uint32_t* cell_start;
  uint32_t* cell_cursor;
  uint32_t* cell_atoms;
  const real4* pos;
  real4* cell_pos;  // written in cell order when no reorder follows
  uint4* cell_xbins; // per cell: x-bin prefix counts of its x-sorted members
  BoxView box;
  CellGridView grid;
};

// The rebuild kernel's bookkeeping and the memory its workgroups meet in.
constexpr uint32_t kRebuildMaxBlocks = 256;
constexpr uint32_t kSyncLine = 16;  // 8-byte words of a member's arrival or release line

// How a rebuild's workgroups meet (rebuild_kernel).
struct RebuildLimits {
  uint32_t members = kRebuildMaxBlocks;  // most that take part
  int64_t join_ticks = 3000;             // how long the first waits for the grid to start,
                                         // in wall_clock64 ticks (rebuild_join_ticks)
  // Polls before any other wait is given up: at about a microsecond each some
  // two minutes of running, far above the longest phase (one wave orders a large
  // cell: 155 ms at 242,771 members). Polls and not time, which passes for a
  // workgroup whose queue is off the GPU too.
  uint32_t wait_polls = 1u << 27;
};

// Ticks of 10 ns. An idle GPU starts the grid in a few microseconds; beside
// another stream's kernels a rebuild of a large system by half the grid costs
// more than the wait. Next to copies that fill the GPU (x *= 1 over 1 GiB), 96
// steps of an LJ fluid with 17 rebuilds and 2 reorders, ms by window of 0 / 10 /
// 30 / 100 / 200 us: 4,000,000 beads 234 / 190 / 170 / 163.6 / 162.9 (half the
// grid joins in 30 us, all of it in 200), 1,000,000 beads 59.7 / 57.4 / 54.2 /
// 52.8 to 54.1 / 55.1. As seven launches, which start as the GPU comes free,
// these were 162.0 and 49.5 (engine and copies together 225 and 57.6 against
// 222 and 56.7). At 48,000 beads 30 us is as long as a rebuild takes (12.1 ms,
// 14.6 as seven launches).
constexpr int64_t rebuild_join_ticks(uint32_t n) {
  return n < 300000 ? 3000 : (n < 2000000 ? n / 100 : 20000);
}

struct RebuildParams {
  Ctrl* ctrl;
  NeighborControl control;
  int32_t forced;
  uint64_t steps;                      // steps advanced since the previous launch
  unsigned long long* neighbor_parts;  // cleared for the build
  uint64_t* sync_lines;                // [kRebuildMaxBlocks][2 * kSyncLine], zero at set-up
  uint32_t* tile_sums;                 // [kRebuildMaxBlocks]
  RebuildLimits limits;
  uint32_t* stalled_host;              // host memory: Ctrl::stalled for the host to look at
};

struct ScaleParams {
  uint32_t n;
  real4* vel;
  double* partials;
  Ctrl* ctrl;
};

inline unsigned grid_for(uint32_t n, int block = kBlock) {
  return static_cast<unsigned>((static_cast<uint64_t>(n) + block - 1) / block);
}

// The force pass gives every atom a team of adjacent lanes; each lane takes
// `slots` neighbour slots per round.
struct ForceShape {
  int team, slots;
};
constexpr int kForceTeamMax = 16;

// Entries allocated past the last atom in the build's candidate streams (the
// position array and its cell-ordered copy): a build round loads 16
// consecutive candidates without a bounds test and ignores those past the run.
constexpr uint32_t kCandidatePad = 16;

// Neighbour-rebuild sequence; every kernel is predicated on ctrl->rebuild so
// the host never waits for the displacement check.
// The bookkeeping alone (direct path). steps: steps advanced since the
// previous launch (0 at set-up).
void launch_control(Ctrl* ctrl, NeighborControl control, bool forced, uint64_t steps,
                    unsigned long long* neighbor_parts, hipStream_t stream);
// Binning, scan, scatter, sort and (when due) reorder: one launch.
void launch_rebuild(const CellScanParams& cells, const ReorderParams& reorder,
                    const RebuildParams& p, hipStream_t stream);
void launch_build(const BuildParams& p, hipStream_t stream);

// Trajectory records in file order (slot order), one `words`-word record per
// atom: tag, then type, position, image, velocity, force as `mask` selects.
struct PackParams {
  uint32_t n;
  uint32_t mask;   // BEADS_TRAJ_* bits
  uint32_t words;  // record size in 32-bit words
  const real4* pos;
  const real4* vel;
  const real4* force;
  const int4* image;
  const uint32_t* tag;
  uint32_t* out;
};
void launch_pack_records(const PackParams& p, hipStream_t stream);

// The state of n atoms from `first` on as arrays of one field each: byte
// offsets into out (kNoField: not wanted).
constexpr uint64_t kNoField = ~uint64_t{0};
struct PackStateParams {
  uint32_t first, n;
  const real4* pos;
  const real4* vel;
  const real4* force;
  const int4* image;
  const uint32_t* tag;
  const uint32_t* molid;
  unsigned char* out;
  uint64_t positions, velocities, forces, masses, images, types, tags, molecule_ids;
};
void launch_pack_state(const PackStateParams& p, hipStream_t stream);

// One step's work.
// sums: total the kinetic energy (with observables also energies and virials)
// and form the Berendsen factor.
void launch_force(const ForceParams& p, bool kick, bool observables, bool sums,
                  hipStream_t stream);
void launch_integrate(const IntegrateParams& p, bool thermostat, bool check,
                      bool force_rebuild, hipStream_t stream);
void launch_scale(const ScaleParams& p, bool thermostat, hipStream_t stream);

}  // namespace beads_amd
