// Window of a record that an image tile reaches (integer arithmetic of
// k_kdm_forward_tile, in a header of its own so that it can be checked on the
// host).
#pragma once

namespace seisfat {

struct SampleWindow {
  int first, len;
};

// The samples [first, first + len) of a record of nt that the time indices from
// i_lo to i_hi (>= -1) reach; len <= 0 when none.  An index past the record may
// be any value up to INT_MAX (t_index), so it is bounded before one is added:
// 0 <= first and first + len <= nt whenever len > 0.
constexpr SampleWindow sample_window(int i_lo, int i_hi, int nt) {
  const int first = i_lo > 0 ? i_lo : 0;
  const int last = i_hi < nt - 1 ? i_hi : nt - 1;
  return {first, last - first + 1};
}

}  // namespace seisfat
