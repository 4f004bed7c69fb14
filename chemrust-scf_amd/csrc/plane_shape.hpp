// Row buffers of the plane kernels: how many lane groups of a workgroup
// transform rows. Host arithmetic only (no HIP), so that its bounds are checked
// without a device.
#pragma once
#include <algorithm>
#include <cstddef>

namespace chs {

// `groups` lane groups, of which 1 / div at most get a buffer; an n-point plane
// (cmp_bytes) of n_act active columns, row_bytes a buffer, tab_bytes of tables,
// lim bytes of LDS a workgroup. 0: the plane does not fit with one buffer.
// Group g < result starts on row g, whose V_eff the plane kernel loads ahead of
// its loop: the result is never above n (a 512-thread workgroup has more groups
// than a 32- or 36-point plane has rows).
inline int plane_row_buffers(size_t lim, size_t cmp_bytes, size_t row_bytes, size_t tab_bytes,
                             int n, int n_act, int groups, int div) {
  if (cmp_bytes + row_bytes + tab_bytes > lim) return 0;
  const size_t fit = (lim - cmp_bytes - tab_bytes) / row_bytes;
  int nrb = (int)std::min(fit, (size_t)groups);
  nrb = std::min(std::max(1, nrb / std::max(1, div)), n);
  // the fewest that keep the rounds over the rows and over the active columns,
  // where that lets another workgroup onto the CU (complex64 at 72 points, 512
  // threads: 36 of 56 groups, three workgroups in place of two, 0.191 -> 0.174
  // ms for 160 bands); otherwise whole wavefronts of groups are better
  // (complex128 at 72 points: 24 in place of 28 groups cost 4%)
  const int rr = (n + nrb - 1) / nrb, ry = (n_act + nrb - 1) / nrb;
  const int few = std::max((n + rr - 1) / rr, ry > 0 ? (n_act + ry - 1) / ry : 1);
  auto per_cu = [&](int g) { return lim / (cmp_bytes + (size_t)g * row_bytes + tab_bytes); };
  return per_cu(few) > per_cu(nrb) ? few : nrb;
}

}  // namespace chs
