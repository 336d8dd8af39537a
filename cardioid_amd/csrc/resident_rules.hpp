// resident_rules.hpp -- the rules of the resident form that need no device:
// plain functions, the same on the host and in the kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace cdh {

// The tiles of a slab that can hold neighbours of one of its tiles' cells on
// one side: part 0 the planes one step back in x, 1 level, 2 one step on.
// first(t) is the box point of tile t's first cell; the tile's own cells lie
// in box points lo .. hi; plane and row are the box's steps in x and y.  A
// slab's cells are in box order, so the tiles with cells in a range of box
// points are a range too, found by the tiles' first box points; it may hold a
// tile too many at its start.  The range is {begin, end}.
struct TileRange {
   int begin, end;
};
template <class First>
__host__ __device__ inline TileRange tile_range(int part, int64_t lo, int64_t hi, int64_t plane,
                                                int64_t row, int ntile, First &&first)
{
   const int64_t reach = part == 1 ? row + 1 : row;
   // the number of tiles whose first box point is at most x
   auto upto = [&](int64_t x) {
      int n0 = 0, n1 = ntile;
      while (n0 < n1) {
         const int m = (n0 + n1) / 2;
         if (first(m) <= x) n0 = m + 1;
         else n1 = m;
      }
      return n0;
   };
   const int e = upto(hi + (part - 1) * plane + reach);
   const int f = upto(lo + (part - 1) * plane - reach);
   return e > 0 ? TileRange{f > 0 ? f - 1 : 0, e} : TileRange{0, 0};
}

// Whether a cooperative launch that ended with `e` was turned down for what it
// asks of the device, so that step kernels take the run; any other error is
// the caller's.
inline bool resident_refused(hipError_t e)
{
   return e == hipErrorCooperativeLaunchTooLarge || e == hipErrorNotSupported;
}

}  // namespace cdh
