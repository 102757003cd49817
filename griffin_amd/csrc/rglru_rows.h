// Where lanes read a row that may end inside a step of a contraction.  Plain C++, so that the host can check it for every lane.
#pragma once

namespace rglru {

// First element of the vector of `per_lane` elements that quarter `q` of a wave reads in the contraction step that starts at element
// `first` of a row of `width` elements (whole vectors): its own vector, or the row's first one where its own lies past the row.
// Offsets from the row's start: the caller adds nothing to them, and drops the products of a vector that is not its own.
constexpr int row_vector(int first, int q, int per_lane, int width) {
  return first + q * per_lane < width ? first + q * per_lane : 0;
}

}  // namespace rglru
