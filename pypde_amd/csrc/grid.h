// Extents of a launch of many workgroups.
//
// gridDim.x * blockDim.x has to stay below 2^32 (hip_runtime_api.h).  A module
// launch past it returns success all the same and leaves work out: with 2^25 + 1
// face points of 128 threads (nine variables, one wavefront per matrix), every cell
// of the grid came out wrong.  Variants that give a point or a cell several
// threads come near it on grids that fit the GPU, so workgroups that do not fit in
// x continue in y; kernels number them x + y gridDim.x (blk_x) and those past the
// last one, fewer than the grid has rows, find no work.
#pragma once

namespace pypde {

constexpr unsigned long GRID_THREADS = (1ul << 32) - 1;

struct Grid {
  unsigned int x, y;
};

// The fewest rows of equal length that hold `blocks` workgroups of `threads`.
inline Grid grid_of(unsigned long blocks, unsigned int threads,
                    unsigned long limit = GRID_THREADS) {
  const unsigned long fit = limit / threads > 0 ? limit / threads : 1;
  const unsigned long rows = blocks > fit ? (blocks + fit - 1) / fit : 1;
  return {(unsigned int)((blocks + rows - 1) / rows), (unsigned int)rows};
}

}  // namespace pypde
