// mc_grid_limit.h - how much of a large lattice one launch takes.
#pragma once

namespace mcb {

// A launch has fewer than 2^32 threads.  The tiles of 64 lattice points (a
// multiple of 8, whole rounds over the XCDs) that a launch with `groups`
// wavefronts a tile takes: with 16 groups, 2.7e8 points.
inline unsigned tiles_per_launch(unsigned groups) { return ((1u << 26) - 1) / groups / 8 * 8; }

}  // namespace mcb
