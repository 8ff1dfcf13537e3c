// hr_slices.h -- how the grid builds split the cells of large triangles.
//
// A wave of the pair passes has 64 triangles, whose candidate cells (the cells
// of their boxes) form one list.  Host and device share the arithmetic.
#pragma once

#include <stdint.h>

namespace hr {

// Waves of 64 triangles with many candidates (large triangles: walls, a ground)
// are listed by the count pass and their candidates are spread over the launch
// in kPairSlices slices each, in place of one wave that the whole launch waits
// for.  A slice has at least kSliceMin candidates, so that reading the 64
// triangles again is a small part of its work.  Two ground triangles of a
// 74-cells-wide exact grid (82,000 triangles): 640 us a pass before, rebuild and
// frame 1718 -> 645 us; 768 wall triangles of a two-level grid of 20,480: write
// pass 12.6 -> 5.1 us.
constexpr uint32_t kPairsHeavy = 1024;     // candidates of a wave from which it is listed
constexpr uint32_t kPairSlices = 32;
constexpr uint32_t kSliceMin = 256;
constexpr uint32_t kSliceStep = 64;        // candidates of a wave's step

// The most candidates that one wave's list may have.  Past it the build reports
// 2^32 - 1 pairs, which no buffer holds: 64 walls across a grid of 1e8 cells
// have 6e9 candidates, and a sum that wraps would drop most of their
// references.  Below it no step of a list and no end of a slice passes 2^32.
constexpr uint32_t kPairsWaveMax = 0xFFFFFF00u;

constexpr uint32_t pairs_count_or_refuse(uint32_t candidates, uint32_t count)
{
    return candidates > kPairsWaveMax ? 0xFFFFFFFFu : count;
}

constexpr uint32_t slice_len(uint32_t total)
{
    const uint32_t n = ((total + kPairSlices - 1u) / kPairSlices + kSliceStep - 1u) / kSliceStep * kSliceStep;
    return n < kSliceMin ? kSliceMin : n;
}

// candidates [slice_begin, slice_end) of slice s; none where the begin is past the total
constexpr uint32_t slice_begin(uint32_t total, uint32_t s) { return s * slice_len(total); }
constexpr uint32_t slice_end(uint32_t total, uint32_t s)
{
    const uint32_t b = slice_begin(total, s), n = slice_len(total);
    return total - b < n ? total : b + n;
}

// whether a lane that owns the cnt candidates from ex on has one in the step from j0 on
constexpr bool owns_in_step(uint32_t ex, uint32_t cnt, uint32_t j0)
{
    return cnt != 0u && ex < j0 + kSliceStep && ex + cnt > j0;
}

}  // namespace hr
