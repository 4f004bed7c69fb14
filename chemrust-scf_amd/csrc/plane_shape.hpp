// Row buffers of the plane kernels: how many lane groups of a workgroup
// transform rows. Host arithmetic only (no HIP), so that its bounds are checked
// without a device.
#pragma once
#include <algorithm>
#include <cstddef>

namespace chs {

// `groups` lane groups, of which 1 / div at most get a buffer; an n-point plane
// (cmp_bytes) of n_act active columns, row_bytes a buffer, tab_bytes of tables,
// lim bytes of LDS a workgroup, csz a complex number's bytes. 0: the plane does
// not fit with one buffer. Group g < result starts on row g, whose V_eff the plane kernel loads ahead of
// its loop: the result is never above n (a 512-thread workgroup has more groups
// than a 32- or 36-point plane has rows).
inline int plane_row_buffers(size_t lim, size_t cmp_bytes, size_t row_bytes, size_t tab_bytes,
                             size_t csz, int n, int n_act, int groups, int div) {
  if (cmp_bytes + row_bytes + tab_bytes > lim) return 0;
  const size_t fit = (lim - cmp_bytes - tab_bytes) / row_bytes;
  int nrb = (int)std::min(fit, (size_t)groups);
  nrb = std::min(std::max(1, nrb / std::max(1, div)), n);
  // complex64: the fewest that keep the rounds over the rows and over the active
  // columns, where that lets another workgroup into the CU's LDS (160 bands, 512
  // threads: 72 points 0.189 -> 0.168 ms, 96 points 0.667 -> 0.423; grids of 48
  // points and fewer, which wavefronts and registers limit, the same either way).
  // complex128 keeps all its groups: registers limit its workgroups, and partly
  // filled wavefronts cost it time (256 threads, 48 points 0.172 ms against
  // 0.185, 512 threads, 72 points 0.412 against 0.454; density of 20 bands, 48
  // points 51 against 55 us)
  if (csz != 8) return nrb;
  const int rr = (n + nrb - 1) / nrb, ry = (n_act + nrb - 1) / nrb;
  const int few = std::max((n + rr - 1) / rr, ry > 0 ? (n_act + ry - 1) / ry : 1);
  auto per_cu = [&](int g) { return lim / (cmp_bytes + (size_t)g * row_bytes + tab_bytes); };
  return per_cu(few) > per_cu(nrb) ? few : nrb;
}

}  // namespace chs
