// Device helpers shared by the per-step kernels (kernels.hip) and the batched
// replica kernel (replicas.hip): minimum image, decision arithmetic in the
// storage precision real_t, cell indexing, wavefront/workgroup reductions,
// listed-term algebra.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "device.hpp"

namespace beads_amd {
namespace dev {

// Workgroups are dispatched round-robin over the 8 XCDs; give XCD x the
// contiguous logical range [x * nb / 8, (x + 1) * nb / 8).
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb) {
  const uint32_t q = nb >> 3, r = nb & 7u;
  const uint32_t xcd = b & 7u, idx = b >> 3;
  return xcd < r ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
}

// box_geometry_view.cuh:50-62 (minimum image of an already-formed difference).
__device__ __forceinline__ real_t mic(real_t d, real_t L, real_t hL) {
  return d > hL ? d - L : (d < -hL ? d + L : d);
}

// Minimum-image displacement xi - xj with exact intermediates: when the raw
// difference crosses half the box, xi - L (xi > L/2) or xj - L (xj > L/2) is
// exact by Sterbenz, so only the final small difference rounds. mic(xi - xj)
// instead rounds at the scale of L before folding back (about 1e-6 nm at
// L ~ 50 nm), which the r^-13 force amplifies past 1e-5.
__device__ __forceinline__ real_t mic_diff(real_t xi, real_t xj, real_t L, real_t hL) {
  const real_t d = xi - xj;
  return d > hL ? (xi - L) - xj : (d < -hL ? xi - (xj - L) : d);
}

// mic_diff with both folded forms evaluated and one selected (no branches):
// xi_m = xi - L is the caller's, hoisted out of a loop over partners.
__device__ __forceinline__ real_t mic_diff_sel(real_t xi, real_t xi_m, real_t xj, real_t L,
                                              real_t hL) {
  const real_t d = xi - xj;
  const real_t up = xi_m - xj;
  const real_t dn = xi - (xj - L);
  real_t r = __builtin_unpredictable(d > hL) ? up : d;
  r = __builtin_unpredictable(d < -hL) ? dn : r;
  return r;
}

// Whether some lane's raw difference may lie past half the box on some axis:
// one compare of the largest component with the shortest half length, where a
// compare per axis costs three (1M-bead melt force pass 262 -> 255 us at the
// median, 2M mixture 230 -> 228). A wave that only may need the folded forms
// takes them and gets the same values.
__device__ __forceinline__ real_t shortest_half(const BoxView& b) {
  return fmin(b.hL[0], fmin(b.hL[1], b.hL[2]));
}
__device__ __forceinline__ bool past_half(real_t dx, real_t dy, real_t dz, real_t shortest) {
  return __builtin_amdgcn_ballot_w64(fmax(fmax(fabs(dx), fabs(dy)), fabs(dz)) > shortest) != 0;
}

// Squared distance exactly as written in the reference source (no FMA), so the
// r^2 <= r_s^2 and r^2 < r_c^2 decisions match a host evaluation in real_t.
__device__ __forceinline__ real_t r2_strict(real_t dx, real_t dy, real_t dz) {
#pragma clang fp contract(off)
  return dx * dx + dy * dy + dz * dz;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    v += __shfl_xor(v, o, 64);
  }
  return v;
}

// Sum of a value over an aligned team of TEAM adjacent lanes (xor butterfly:
// every lane ends with the same bits, since a + b == b + a exactly).
template <int TEAM>
__device__ __forceinline__ double team_sum(double v) {
#pragma unroll
  for (int m = TEAM / 2; m > 0; m >>= 1) {
    v += __shfl_xor(v, m, TEAM);
  }
  return v;
}

// counter[key] += 1 for every active lane of the wave. Up to kSharedKeys
// distinct keys are served with one atomic each: the lanes sharing a key add
// their count through the first of them and take consecutive values in lane
// order. Lanes whose key has not come up by then add for themselves: spatially
// sorted atoms of a wave lie in a handful of cells, but atoms in a caller's
// order have a cell each, and one returning atomic after another is a chain of
// up to 64 memory latencies (the scatter of 100,000 shuffled beads). Returns
// the counter's value before this lane's increment.
constexpr int kSharedKeys = 6;

__device__ __forceinline__ uint32_t wave_increment(uint32_t* counter, uint32_t key) {
  const uint32_t lane = threadIdx.x & 63u;
  uint64_t pending = __ballot(1);
  uint32_t result = 0;
  for (int shared = 0; pending != 0 && shared < kSharedKeys; ++shared) {
    const int first = __builtin_ctzll(pending);
    const uint32_t lead = static_cast<uint32_t>(__shfl(static_cast<int>(key), first));
    const uint64_t group = __ballot(key == lead) & pending;
    if ((group >> lane) & 1ull) {
      const uint32_t rank = static_cast<uint32_t>(__builtin_popcountll(group & ((1ull << lane) - 1ull)));
      uint32_t base = 0;
      if (rank == 0) {
        base = atomicAdd(&counter[lead], static_cast<uint32_t>(__builtin_popcountll(group)));
      }
      result = static_cast<uint32_t>(__shfl(static_cast<int>(base), first)) + rank;
    }
    pending &= ~group;
  }
  if ((pending >> lane) & 1ull) result = atomicAdd(&counter[key], 1u);
  return result;
}

// Sets *flag, read by later kernels only, when hit holds in some active lane:
// one store per wave, into this XCD's L2 (the kernel's end writes it back; all
// writers store the same word). Stores at agent scope go past the L2 one after
// another, 37 ns each on one address, which is what a frame_load whose every
// atom has moved spent its time on (57 of 61 us at 100,000 beads).
__device__ __forceinline__ void raise_flag(bool hit, uint32_t* flag) {
  const uint64_t m = __builtin_amdgcn_ballot_w64(hit);
  if (m != 0 && (threadIdx.x & 63u) == static_cast<uint32_t>(__builtin_ctzll(m))) {
    __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
}

// 1/x in FP64: the hardware reciprocal (relative error <= 4.6e-8 measured on
// gfx950) refined by one Newton step (<= 2.3e-15).
__device__ __forceinline__ double rcp_f64(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  return r * (2.0 - x * r);
}

// 1/sqrt(x) in FP64 for x > 0: the hardware reciprocal square root refined by
// one Newton step (the hardware value's relative error squared, about 1e-15).
__device__ __forceinline__ double rsq_f64(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  return r * (1.5 - 0.5 * x * r * r);
}

// Sum over a BLOCK-wide workgroup (BLOCK a multiple of 64, at most 1024);
// result valid in thread 0. lds needs BLOCK / 64 doubles.
template <int BLOCK>
__device__ __forceinline__ double block_sum(double v, double* lds) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) {
    lds[wave] = v;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    v = 0.0;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; ++w) v += lds[w];
  }
  return v;
}

// cell_list_build.cu:110-123: cell index in real_t, clamped.
__device__ __forceinline__ uint32_t axis_cell(real_t x, real_t lo, real_t inv, uint32_t count) {
  const real_t s = (x - lo) * inv;
  uint32_t i = s <= real_t(0) ? 0u : static_cast<uint32_t>(s);
  return i >= count ? count - 1 : i;
}

__device__ __forceinline__ uint32_t cell_of_position(real4 x, const BoxView& box,
                                                     const CellGridView& g) {
  const uint32_t ix = axis_cell(x.x, box.lo[0], g.inv_cell[0], g.nx);
  const uint32_t iy = axis_cell(x.y, box.lo[1], g.inv_cell[1], g.ny);
  const uint32_t iz = axis_cell(x.z, box.lo[2], g.inv_cell[2], g.nz);
  return ix + g.nx * (iy + g.ny * iz);
}

// Whether the clamp puts x into a cell that does not hold it, on some axis: the
// wrap leaves a coordinate outside the box by its rounding, which after a
// displacement of millions of box lengths is a good part of a cell. Up to
// kOutsideSlack of a cell counts as inside (a build's pruning allows for twice
// that, kGapSlack); NaN is outside.
constexpr real_t kOutsideSlack = static_cast<real_t>(1.0 / 128.0);
__device__ __forceinline__ bool outside_cells(real4 x, const BoxView& box, const CellGridView& g) {
  auto inside = [](real_t v, real_t lo, real_t inv, uint32_t count) {
    const real_t s = (v - lo) * inv;
    return s >= -kOutsideSlack && s <= static_cast<real_t>(count) + kOutsideSlack;
  };
  return !(inside(x.x, box.lo[0], g.inv_cell[0], g.nx) &&
           inside(x.y, box.lo[1], g.inv_cell[1], g.ny) &&
           inside(x.z, box.lo[2], g.inv_cell[2], g.nz));
}

// regular_cell_neighbor_builder.cu:40-53.
__device__ __forceinline__ uint32_t wrapped_axis(uint32_t c, int d, uint32_t count) {
  if (d < 0) return c == 0 ? count - 1 : c - 1;
  if (d > 0) return c + 1 == count ? 0 : c + 1;
  return c;
}

// small_dimension_neighbor_builder.cu:56-76.
__device__ __forceinline__ int unique_axis(uint32_t c, uint32_t count, uint32_t out[3]) {
  if (count <= 1) {
    out[0] = 0;
    return 1;
  }
  if (count == 2) {
    out[0] = c == 0 ? 1u : 0u;
    out[1] = c;
    return 2;
  }
  out[0] = wrapped_axis(c, -1, count);
  out[1] = c;
  out[2] = wrapped_axis(c, 1, count);
  return 3;
}

// Candidate cells of the regular and small-dimension builders, z outermost.
struct CellNeighborhood {
  uint32_t xs[3], ys[3], zs[3];
  int nx, ny, nz;
};

__device__ __forceinline__ CellNeighborhood neighborhood(uint32_t c, const CellGridView& g) {
  CellNeighborhood h;
  const uint32_t cx = c % g.nx;
  const uint32_t cyz = c / g.nx;
  const uint32_t cy = cyz % g.ny;
  const uint32_t cz = cyz / g.ny;
  if (g.path == 1) {
    for (int d = -1; d <= 1; ++d) {
      h.xs[d + 1] = wrapped_axis(cx, d, g.nx);
      h.ys[d + 1] = wrapped_axis(cy, d, g.ny);
      h.zs[d + 1] = wrapped_axis(cz, d, g.nz);
    }
    h.nx = h.ny = h.nz = 3;
  } else {
    h.nx = unique_axis(cx, g.nx, h.xs);
    h.ny = unique_axis(cy, g.ny, h.ys);
    h.nz = unique_axis(cz, g.nz, h.zs);
  }
  return h;
}

// ------------------------------------------------- candidate runs of a build ---
//
// A build visits the 27 cells around an atom's cell (fewer on short axes), z
// outermost, x innermost. Cells adjacent in x are adjacent in the cell-ordered
// stream, so the three x-cells of a row are one run of the stream, or two where
// the row wraps around the box (or, with two cells, starts at the upper one).

// Neighbour k (0, 1, 2) along an axis of count cells, in the order of
// unique_axis, and its image shift code (0: none, 1: +L, 2: -L): with at
// least 5 cells per axis a candidate in a wrapped neighbour cell lies more
// than L/2 away (mic adds +L or -L), and in any other neighbour cell less
// than L/2 away (mic adds 0).
__device__ inline uint32_t neighbour_cell(uint32_t cc, uint32_t count, int k, uint32_t& code) {
  code = 0;
  if (count <= 1) return 0u;
  if (count == 2) return k == 0 ? (cc == 0 ? 1u : 0u) : cc;
  if (k == 0) {
    if (cc == 0) {
      code = 1;
      return count - 1;
    }
    return cc - 1;
  }
  if (k == 2) {
    if (cc + 1 == count) {
      code = 2;
      return 0u;
    }
    return cc + 1;
  }
  return cc;
}

__device__ inline real_t shift_of(uint32_t code, real_t L) {
  return code == 0 ? static_cast<real_t>(0) : (code == 1 ? L : -L);
}

// Members of cell cc with x-bin below m (cell_xbins; m in 0..kXBins).
__device__ inline uint32_t members_below(const uint4* xbins, uint32_t cc, int m) {
  if (m <= 0) return 0u;
  const uint4 q = xbins[cc];
  const int f = m - 1;
  const uint32_t word = (f >> 1) == 0 ? q.x : ((f >> 1) == 1 ? q.y : ((f >> 1) == 2 ? q.z : q.w));
  return (word >> (16 * (f & 1))) & 0xffffu;
}

// Rows of x-adjacent cells around an atom (3 along z times 3 along y), and the
// most runs they make.
constexpr int kRows = 9;
constexpr int kMaxRuns = 2 * kRows;

// A run of the stream, [x, y) below 2^28, with the image shift codes of its
// cells in the top bits: x's in .x, y's and z's in .y.
constexpr int kRunCodeShift = 28;
constexpr uint32_t kRunIndexMask = (1u << kRunCodeShift) - 1u;

// The runs of row r (z neighbour r / 3, y neighbour r % 3) of an atom at xi in
// cell (cx, cy, cz); empty runs are {0, 0}. prune, with 5 or more cells per
// axis: a row whose cells lie at least gy along y and gz along z from the atom holds
// neighbours only within ext = sqrt(r_s^2 - gy^2 - gz^2) along x, and none when
// gy^2 + gz^2 > r_s^2: such rows are dropped, and with x-bin tables (xbins,
// members of a cell ascending in x) the row starts and ends at the bins within
// ext of the atom, one bin of margin on each side (a bin is an eighth of a
// cell). The gaps are taken kGapSlack of a cell short, far above the rounding
// of the cell coordinates, so a skipped member is farther than ext along x, or
// than the gaps along y and z, by a margin that no rounding of r^2 closes: the
// accepted candidates and their order are those of the full scan, provided that
// the cells hold their members. A member clamped into a face's cell from beyond
// the face is closer to the cells across it than its bin says, so a caller
// prunes only where no atom is outside (outside_cells).
struct RunPair {
  uint2 a, b;
};
__device__ inline RunPair row_run_pair(const CellGridView& g, const BoxView& box, real_t rs2,
                                       const uint32_t* cell_start, const uint4* xbins, bool prune,
                                       real4 xi, uint32_t cx, uint32_t cy, uint32_t cz,
                                       uint32_t r) {
  RunPair out;
  out.a = out.b = make_uint2(0u, 0u);
  const int iz = static_cast<int>(r / 3), iy = static_cast<int>(r % 3);
  if ((iz > 0 && static_cast<uint32_t>(iz) >= g.nz) || (iy > 0 && static_cast<uint32_t>(iy) >= g.ny))
    return out;
  uint32_t code_y, code_z;
  const uint32_t zc = neighbour_cell(cz, g.nz, iz, code_z);
  const uint32_t rowc = g.nx * (neighbour_cell(cy, g.ny, iy, code_y) + g.ny * zc);
  // The row's cells [l0, l1] then, where it wraps, [m0, m1]; x shift codes.
  uint32_t l0, l1, m0 = 1, m1 = 0, code_l = 0, code_m = 0;
  if (g.nx <= 2) {
    l0 = 0;
    l1 = g.nx - 1;
    if (g.nx == 2 && cx == 0) {
      l0 = l1 = 1;
      m0 = m1 = 0;
    }
  } else if (cx == 0) {
    l0 = l1 = g.nx - 1;
    code_l = 1;
    m0 = 0;
    m1 = 1;
  } else if (cx + 1 == g.nx) {
    l0 = cx - 1;
    l1 = cx;
    m0 = m1 = 0;
    code_m = 2;
  } else {
    l0 = cx - 1;
    l1 = cx + 1;
  }
  uint32_t skip = 0, keep = 0xffffffffu;  // members dropped at the row's start, kept of its last cell
  uint32_t n_last = 0;
  const uint32_t last = rowc + (m1 >= m0 ? m1 : l1);
  if (prune && g.nx >= 5 && g.ny >= 5 && g.nz >= 5) {
    constexpr real_t kGapSlack = static_cast<real_t>(1.0 / 64.0);
    static_assert(kGapSlack >= 2 * kOutsideSlack, "a member counted inside stays within the slack");
    const real_t fy = (xi.y - box.lo[1]) * g.inv_cell[1] - static_cast<real_t>(cy);
    const real_t fz = (xi.z - box.lo[2]) * g.inv_cell[2] - static_cast<real_t>(cz);
    // Gap to the row below (k = 0) and above (k = 2) along one axis.
    auto gap = [](real_t f, int k, real_t inv_cell) -> real_t {
      const real_t d = k == 0 ? f - kGapSlack : (static_cast<real_t>(1) - f) - kGapSlack;
      return k == 1 || d < 0 ? static_cast<real_t>(0) : d / inv_cell;
    };
    const real_t gz = gap(fz, iz, g.inv_cell[2]);
    const real_t gy = gap(fy, iy, g.inv_cell[1]);
    const real_t ext2 = rs2 - (gy * gy + gz * gz);
    if (ext2 < 0) return out;
    if (xbins != nullptr) {
      const real_t ext = sqrt(ext2);
      const real_t at = (xi.x - box.lo[0]) * g.inv_cell[0] - static_cast<real_t>(cx);
      const real_t reach = ext * g.inv_cell[0];
      // In bins from the start of the left and of the right neighbour cell.
      const int m_left =
          static_cast<int>(floor((at - reach + real_t(1)) * static_cast<real_t>(kXBins))) - 1;
      const int m_right =
          static_cast<int>(floor((at + reach - real_t(1)) * static_cast<real_t>(kXBins))) + 2;
      const int ml = m_left < 0 ? 0 : (m_left > kXBins ? kXBins : m_left);
      const int mr = m_right < 0 ? 0 : (m_right > kXBins ? kXBins : m_right);
      const uint32_t cl = rowc + l0;
      const uint32_t n_left = cell_start[cl + 1] - cell_start[cl];
      n_last = cell_start[last + 1] - cell_start[last];
      skip = n_left <= kXBinsMaxCount ? members_below(xbins, cl, ml) : 0u;
      keep = n_last <= kXBinsMaxCount ? members_below(xbins, last, mr) : n_last;
    }
  }
  const uint32_t yz = (code_y | (code_z << 2)) << kRunCodeShift;
  uint32_t b = cell_start[rowc + l0] + skip, e = cell_start[rowc + l1 + 1];
  if (m1 < m0 && keep != 0xffffffffu) e -= n_last - keep;
  if (b < e) out.a = make_uint2(b | (code_l << kRunCodeShift), e | yz);
  if (m1 >= m0) {
    b = cell_start[rowc + m0];
    e = cell_start[rowc + m1 + 1];
    if (keep != 0xffffffffu) e -= n_last - keep;
    if (b < e) out.b = make_uint2(b | (code_m << kRunCodeShift), e | yz);
  }
  return out;
}

// A team's runs in visiting order, empty ones left out, into its LDS entry
// list (kMaxRuns entries); returns how many, the same in every lane. Lane t of
// TEAM evaluates rows t, t + TEAM, ... Every lane of the team calls it.
template <int TEAM>
__device__ inline uint32_t team_runs(const CellGridView& g, const BoxView& box, real_t rs2,
                                     const uint32_t* cell_start, const uint4* xbins, bool prune,
                                     real4 xi, uint32_t c, uint32_t t, uint32_t team_lane0,
                                     uint2* runs) {
  const uint32_t cx = c % g.nx, cyz = c / g.nx, cy = cyz % g.ny, cz = cyz / g.ny;
  constexpr uint64_t kTeamMask = TEAM >= 64 ? ~0ull : (1ull << TEAM) - 1ull;
  uint32_t n = 0;
#pragma unroll 1
  for (uint32_t r0 = 0; r0 < static_cast<uint32_t>(kRows); r0 += TEAM) {
    RunPair p;
    p.a = p.b = make_uint2(0u, 0u);
    if (r0 + t < static_cast<uint32_t>(kRows)) {
      p = row_run_pair(g, box, rs2, cell_start, xbins, prune, xi, cx, cy, cz, r0 + t);
    }
    const bool has_a = p.a.y != 0, has_b = p.b.y != 0;  // a nonempty run ends past 0
    const uint64_t ma = (__ballot(has_a) >> team_lane0) & kTeamMask;
    const uint64_t mb = (__ballot(has_b) >> team_lane0) & kTeamMask;
    const uint64_t below = (1ull << t) - 1ull;
    uint32_t at = n + __builtin_popcountll(ma & below) + __builtin_popcountll(mb & below);
    if (has_a) runs[at++] = p.a;
    if (has_b) runs[at] = p.b;
    n += __builtin_popcountll(ma) + __builtin_popcountll(mb);
  }
  return n;
}

// How a build forms a candidate's minimum image.
constexpr int kShift = 0, kShiftYZ = 1, kGeneric = 2;
using kShiftMode = std::integral_constant<int, kShift>;
using kShiftYZMode = std::integral_constant<int, kShiftYZ>;
using kGenericMode = std::integral_constant<int, kGeneric>;

// One atom's runs scanned by its team of TEAM lanes, TEAM * SLOTS candidates
// per round, the next round's candidates loaded before this round's are
// tested (a small system has too few waves to hide a load otherwise). entry(q)
// is stream entry q = {x, y, z, slot bits}; accept(j, x, mode, shift) the
// wave's lanes whose candidate is a neighbour; put(slot, j) stores one.
// Candidates are taken in run order, so neighbours are appended in the order
// of a one-lane scan. Returns the atom's count, the same in every lane.
template <int TEAM, int SLOTS, typename Entry, typename Accept, typename Put, typename Mode>
__device__ __forceinline__ uint32_t scan_runs(const uint2* runs, uint32_t n_runs, uint32_t t,
                                              uint32_t team_lane0, const BoxView& box, Entry entry,
                                              Accept accept, Put put, Mode mode) {
  static_assert(TEAM <= 32, "a team's lane mask is one word");
  constexpr uint32_t kRound = TEAM * SLOTS;
  constexpr uint32_t kTeamMask = static_cast<uint32_t>((1ull << TEAM) - 1ull);
  const uint32_t below = (1u << t) - 1u;
  uint32_t count = 0;
  if (n_runs == 0) return count;
  uint32_t r = 0, k, e;
  real3 sh;
  auto open = [&]() {  // run r becomes the current one
    const uint2 d = runs[r++];
    k = d.x & kRunIndexMask;
    e = d.y & kRunIndexMask;
    const uint32_t yz = d.y >> kRunCodeShift;
    sh = make_real3(shift_of(d.x >> kRunCodeShift, box.L[0]), shift_of(yz & 3u, box.L[1]),
                    shift_of(yz >> 2, box.L[2]));
  };
  real4 next[SLOTS];
  auto load = [&]() {  // entries past the run's end repeat its last one
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      const uint32_t q = k + u * TEAM + t;
      next[u] = entry(q < e ? q : e - 1);
    }
  };
  open();
  load();
  for (;;) {
    real4 x[SLOTS];
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) x[u] = next[u];
    // Slot u of this lane is in the run while u * TEAM < left.
    const int left = static_cast<int>(e - k) - static_cast<int>(t);
    const real3 shift = sh;
    bool more = true;
    k += kRound;
    if (k >= e) {
      more = r < n_runs;
      if (more) open();
    }
    if (more) load();
#pragma unroll
    for (int u = 0; u < SLOTS; ++u) {
      const uint32_t j = id_of(x[u].w);
      const uint64_t m = __builtin_amdgcn_ballot_w64(u * TEAM < left) & accept(j, x[u], mode, shift);
      const uint32_t bits = static_cast<uint32_t>(m >> team_lane0) & kTeamMask;
      if (__builtin_amdgcn_inverse_ballot_w64(m)) {
        put(count + static_cast<uint32_t>(__builtin_popcount(bits & below)), j);
      }
      count += static_cast<uint32_t>(__builtin_popcount(bits));
    }
    if (!more) break;
  }
  return count;
}

// LJ pair value in FP64 from the displacement in real_t (exact in binary32
// too: FP64 VALU runs at the non-packed FP32 rate on CDNA4, and binary32 would
// amplify the rounding of r^2 six-fold through (sigma^2/r^2)^6). Returns the
// force scale s with f_i = s * d; energy gets 4 eps (sr12 - sr6) - shift.
__device__ __forceinline__ double lj_pair(real_t dx, real_t dy, real_t dz, const LjCoeff& c,
                                          double& rr, double& energy) {
  const double ddx = dx, ddy = dy, ddz = dz;
  rr = ddx * ddx + ddy * ddy + ddz * ddz;
  const double inv = rcp_f64(rr);
  const double sr2 = c.sigma2 * inv;
  const double sr6 = sr2 * sr2 * sr2;
  const double sr12 = sr6 * sr6;
  energy = c.eps4 * (sr12 - sr6) - c.shift;
  return c.eps24 * inv * (2.0 * sr12 - sr6);
}

// ------------------------------------------------------- listed terms ------

__device__ __forceinline__ real3 f3(real4 v) { return make_real3(v.x, v.y, v.z); }

// Minimum-image displacement p - q (wrapped coordinates), see mic_diff.
__device__ __forceinline__ real3 mic3(real3 p, real3 q, const BoxView& b) {
  return make_real3(mic_diff(p.x, q.x, b.L[0], b.hL[0]), mic_diff(p.y, q.y, b.L[1], b.hL[1]),
                    mic_diff(p.z, q.z, b.L[2], b.hL[2]));
}

// FP64 vectors for the listed terms. Their displacements come exact (or
// rounded once) from the positions through mic3; everything after that is
// FP64, because near-collinear triples make the angle and dihedral
// algebra ill-conditioned in binary32 (|v0 x v1| ~ 1e-5 |v0||v1| occurs in a
// million-bead melt and costs binary32 three significant digits there).
struct d3 {
  double x, y, z;
};
__device__ __forceinline__ d3 dbl(real3 v) { return {v.x, v.y, v.z}; }
__device__ __forceinline__ real3 flt(d3 v) {
  return make_real3(static_cast<real_t>(v.x), static_cast<real_t>(v.y), static_cast<real_t>(v.z));
}
__device__ __forceinline__ d3 dsub(d3 a, d3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ d3 dadd(d3 a, d3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ d3 dscale(d3 a, double s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ double ddot(d3 a, d3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ d3 dcross(d3 a, d3 b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// The listed terms take square roots and quotients as products with the
// FP64 reciprocal (square root) of rcp_f64 / rsq_f64 (one Newton step each,
// about 1e-15 relative) instead of IEEE division and square root, whose
// correctly rounded sequences cost several times the instructions.

// Harmonic bond U = k/2 (r - r0)^2 (bond_harmonic.cu:41-79) on the displacement
// d = x_self - x_partner; returns the force on self and the term's energy and
// virial d.f.
__device__ __forceinline__ real3 bond_force(real3 df, real2 kc, double& energy,
                                            double& virial) {
  const d3 d = dbl(df);
  const double k = kc.x, r0 = kc.y;
  const double r2 = ddot(d, d);
  if (r2 == 0.0) {
    energy = 0.5 * k * r0 * r0;
    virial = 0.0;
    return make_real3(0, 0, 0);
  }
  const double inv_r = rsq_f64(r2);
  const double stretch = r2 * inv_r - r0;
  energy = 0.5 * k * stretch * stretch;
  const double s = -k * stretch * inv_r;
  virial = s * r2;
  return flt(dscale(d, s));
}

// Harmonic angle U = k/2 (theta - theta0)^2 (angle_harmonic.cu:61-158) for one
// role. Same mathematics as the reference, in a stable form: theta =
// atan2(|a x b|, a.b) and sin(theta) = |a x b| / (|a||b|) instead of acos(c)
// and sqrt(1 - c^2), and the force directions as a x (a x b), b x (a x b)
// instead of differences of nearly parallel vectors. The reference's floor
// (sin theta replaced by kSinFloor at or below it, angle_harmonic.cu:25, 126;
// real_t{0.001}: the binary32 value in the binary32 build) is kept.
__device__ __forceinline__ real3 angle_role_force(real3 xi, real3 xj, real3 xk, real2 kc,
                                                  int role, const BoxView& box, double& energy,
                                                  double& virial) {
  const d3 a = dbl(mic3(xi, xj, box));
  const d3 b = dbl(mic3(xk, xj, box));
  const double k = kc.x, theta0 = kc.y;
  const double ra2 = ddot(a, a), rb2 = ddot(b, b);
  if (ra2 == 0.0 || rb2 == 0.0) {
    energy = 0.5 * k * theta0 * theta0;
    virial = 0.0;
    return make_real3(0, 0, 0);
  }
  const double ia = rsq_f64(ra2), ib = rsq_f64(rb2);
  const d3 nrm = dcross(a, b);
  const double nn2 = ddot(nrm, nrm);
  const double nn = nn2 > 0.0 ? nn2 * rsq_f64(nn2) : 0.0;
  // The FP64 arguments are well conditioned; in the binary32 build an atan2
  // of them in binary32 is accurate to a few 1e-8 relative (below the
  // force's own rounding) and keeps the pass's register budget.
  const double theta = kReal64 ? atan2(nn, ddot(a, b))
                               : atan2f(static_cast<float>(nn), static_cast<float>(ddot(a, b)));
  const double dth = theta - theta0;
  energy = 0.5 * k * dth * dth;
  const double sn_true = nn * ia * ib;
  constexpr double kSinFloor = static_cast<double>(static_cast<real_t>(0.001));
  const double sn = sn_true <= kSinFloor ? kSinFloor : sn_true;
  const double A = -k * dth * rcp_f64(sn);
  const double aib = A * ia * ib;
  const d3 fi = dscale(dcross(a, nrm), aib * ia * ia);
  const d3 fk = dscale(dcross(b, nrm), -aib * ib * ib);
  virial = ddot(a, fi) + ddot(b, fk);
  if (role == 0) return flt(fi);
  if (role == 2) return flt(fk);
  return flt(dscale(dadd(fi, fk), -1.0));
}

// Harmonic dihedral k[1 + d cos(n phi)] (dihedral_harmonic.cu:83-206), one role.
// phi = atan2(|v1| v0.c1, c0.c1) carries the reference's sign convention
// (negative when v0.c1 < 0) without the ill-conditioned acos near 0 and pi.
__device__ __forceinline__ real3 dihedral_role_force(real3 xi, real3 xj, real3 xk, real3 xl,
                                                     real4 kc, int role, const BoxView& box,
                                                     double& energy, double& virial) {
  const d3 v0 = dbl(mic3(xi, xj, box));
  const d3 v1 = dbl(mic3(xk, xj, box));
  const d3 v2 = dbl(mic3(xk, xl, box));
  const d3 c0 = dcross(v0, v1), c1 = dcross(v1, v2);
  const double n1 = ddot(v1, v1), nc0 = ddot(c0, c0), nc1 = ddot(c1, c1);
  const double k = kc.x, dsign = kc.y, nmul = kc.z;
  if (n1 == 0.0 || nc0 == 0.0 || nc1 == 0.0) {
    energy = nmul == 0.0 ? k * (1.0 + dsign) : k;
    virial = 0.0;
    return make_real3(0, 0, 0);
  }
  const double inb = rsq_f64(n1);
  const double nb = n1 * inb;
  // cos(phi) and sin(phi) from the cross products (sin carries the sign of
  // v0.c1), then cos(n phi), sin(n phi) by the angle-addition recurrence:
  // the reference's k[1 + d cos(n phi)] and its derivative without a
  // transcendental call.
  const double ic0 = rsq_f64(nc0), ic1 = rsq_f64(nc1);
  const double inv_c = ic0 * ic1;
  const double c1phi = ddot(c0, c1) * inv_c;
  const double s1phi = nb * ddot(v0, c1) * inv_c;
  double cs = 1.0, sn = 0.0;
  for (int m = 0; m < static_cast<int>(nmul); ++m) {
    const double c2 = cs * c1phi - sn * s1phi;
    sn = sn * c1phi + cs * s1phi;
    cs = c2;
  }
  energy = k * (1.0 + dsign * cs);
  const double dE = -k * dsign * nmul * sn;
  const d3 fi = dscale(c0, -dE * nb * ic0 * ic0);
  const d3 fl = dscale(c1, dE * nb * ic1 * ic1);
  const double inv_n1 = inb * inb;
  const d3 sv = dsub(dscale(fi, ddot(v0, v1) * inv_n1), dscale(fl, ddot(v2, v1) * inv_n1));
  const d3 fj = dsub(sv, fi);
  const d3 fk = dscale(dadd(sv, fl), -1.0);
  virial = ddot(v0, fi) + ddot(v1, fk) + ddot(dsub(v1, v2), fl);
  if (role == 0) return flt(fi);
  if (role == 1) return flt(fj);
  if (role == 2) return flt(fk);
  return flt(fl);
}

// Per-thread sums of one force pass.
struct StepSums {
  double ke = 0.0;
  double e_pair = 0.0, w_pair = 0.0;
  double e_bond = 0.0, w_bond = 0.0, e_angle = 0.0, w_angle = 0.0, e_dih = 0.0, w_dih = 0.0;
};

// Listed terms, atom-centric: atom i evaluates every term it belongs to and
// keeps its own role's force (no atomics, deterministic; the reference adds
// each term's forces with float atomics, bond_harmonic.cu, angle_harmonic.cu,
// dihedral_harmonic.cu). A term's energy and virial are counted once, by role
// 0 (bonds: the flag bit of the coefficient word). Records hold partner slots
// of the same position array; topo's per-slot arrays have stride n.
template <bool OBS>
__device__ __forceinline__ real3 bond_term(const real4* pos, const TopologyView& topo,
                                            const BoxView& box, real3 xi, uint2 r,
                                            StepSums& sums) {
  double e, w;
  const real3 f =
      bond_force(mic3(xi, f3(pos[r.x]), box), topo.bond_coeff[r.y & 0x7fffffffu], e, w);
  if (OBS && (r.y >> 31) != 0) {
    sums.e_bond += e;
    sums.w_bond += w;
  }
  return f;
}

template <bool OBS>
__device__ __forceinline__ real3 angle_term(const real4* pos, const TopologyView& topo,
                                             const BoxView& box, real3 xi, uint4 r,
                                             StepSums& sums) {
  const int role = static_cast<int>(r.w);
  const real3 a = f3(pos[r.x]);
  const real3 b = f3(pos[r.y]);
  const real3 pi = role == 0 ? xi : a;
  const real3 pj = role == 0 ? a : (role == 1 ? xi : b);
  const real3 pk = role == 2 ? xi : b;
  double e, w;
  const real3 f = angle_role_force(pi, pj, pk, topo.angle_coeff[r.z], role, box, e, w);
  if (OBS && role == 0) {
    sums.e_angle += e;
    sums.w_angle += w;
  }
  return f;
}

template <bool OBS>
__device__ __forceinline__ real3 dihedral_term(const real4* pos, const TopologyView& topo,
                                                const BoxView& box, real3 xi, uint4 r,
                                                StepSums& sums) {
  const int role = static_cast<int>(r.w >> 30);
  const real3 a = f3(pos[r.x]);
  const real3 b = f3(pos[r.y]);
  const real3 c = f3(pos[r.z]);
  real3 q0, q1, q2, q3;
  if (role == 0) { q0 = xi; q1 = a; q2 = b; q3 = c; }
  else if (role == 1) { q0 = a; q1 = xi; q2 = b; q3 = c; }
  else if (role == 2) { q0 = a; q1 = b; q2 = xi; q3 = c; }
  else { q0 = a; q1 = b; q2 = c; q3 = xi; }
  double e, w;
  const real3 f =
      dihedral_role_force(q0, q1, q2, q3, topo.dih_coeff[r.w & 0x3fffffffu], role, box, e, w);
  if (OBS && role == 0) {
    sums.e_dih += e;
    sums.w_dih += w;
  }
  return f;
}

// The listed terms of atom i shared over its team of TEAM lanes: lane t takes
// terms t, t + TEAM, ... of each kind and adds their forces to its FP64
// partial sums.
template <bool OBS, bool SPILL, int TEAM>
__device__ __forceinline__ void listed_team(const real4* pos, const TopologyView& topo,
                                            const BoxView& box, size_t n, uint32_t i, uint32_t t,
                                            real4 xi4, double& fxd, double& fyd, double& fzd,
                                            StepSums& sums) {
  const uint32_t cw = topo.count[i];
  const uint32_t nbond = cw & 255u, nang = (cw >> 8) & 255u, ndih = (cw >> 16) & 255u;
  const real3 xi = f3(xi4);
  auto add = [&](real3 f) {
    fxd += f.x;
    fyd += f.y;
    fzd += f.z;
  };
  for (uint32_t k = t; k < nbond; k += TEAM) {
    add(bond_term<OBS>(pos, topo, box, xi, topo.bond[k * n + i], sums));
  }
  for (uint32_t k = t; k < nang; k += TEAM) {
    add(angle_term<OBS>(pos, topo, box, xi, topo.angle[k * n + i], sums));
  }
  for (uint32_t k = t; k < ndih; k += TEAM) {
    add(dihedral_term<OBS>(pos, topo, box, xi, topo.dih[k * n + i], sums));
  }
  if (SPILL) {  // some particle spills: its records past the inline capacities
    const uint32_t si = topo.spill_index[i];
    if (si != kNoSpill) {  // uniform over the team
      const SpillEntry e = topo.spill[si];
      for (uint32_t k = t; k < e.cnt[0]; k += TEAM) {
        add(bond_term<OBS>(pos, topo, box, xi, topo.spill_bond[e.off[0] + k], sums));
      }
      for (uint32_t k = t; k < e.cnt[1]; k += TEAM) {
        add(angle_term<OBS>(pos, topo, box, xi, topo.spill_angle[e.off[1] + k], sums));
      }
      for (uint32_t k = t; k < e.cnt[2]; k += TEAM) {
        add(dihedral_term<OBS>(pos, topo, box, xi, topo.spill_dih[e.off[2] + k], sums));
      }
    }
  }
}

// Neighbour storage: each atom's list is cut into chunks of kNbrChunk entries;
// chunk c of atom i is kNbrChunk consecutive words at ((c * N) + i) * kNbrChunk.
// A build appends into an LDS staging row and writes whole 64-byte chunks; the
// force pass reads a chunk as four 16-byte loads.
__device__ __forceinline__ size_t nbr_chunk_base(uint32_t c, uint32_t i, uint32_t n) {
  return (static_cast<size_t>(c) * n + i) * kNbrChunk;
}

}  // namespace dev
}  // namespace beads_amd
