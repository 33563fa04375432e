// The box of cells that a launch's beams may reach, for
// tests/test_beam_reach.py.
#include "../../adamantine_amd/csrc/adm_device.hpp"

// The cells of a mesh that a beam may touch though they lie outside the box
// (there must be none); outside: the cells outside it.
extern "C" int64_t missed_cells(const adm_beam_state *beams, int n_beams,
                                const double *origin, const double *h,
                                const int32_t *nc, int64_t *outside) {
  const double o[3] = {origin[0], origin[1], origin[2]};
  const double inv_h[3] = {1.0 / h[0], 1.0 / h[1], 1.0 / h[2]};
  int32_t lo[3], hi[3];
  adm::beam_reach(beams, n_beams, o, inv_h, lo, hi);
  int64_t missed = 0;
  *outside = 0;
  for (int z = 0; z < nc[2]; ++z)
    for (int y = 0; y < nc[1]; ++y)
      for (int x = 0; x < nc[0]; ++x) {
        const int c[3] = {x, y, z};
        bool in = true;
        double a[3], b[3];
        for (int d = 0; d < 3; ++d) {
          in = in && c[d] >= lo[d] && c[d] <= hi[d];
          a[d] = o[d] + c[d] * h[d];
          b[d] = o[d] + (c[d] + 1) * h[d];
        }
        if (in) continue;
        ++*outside;
        for (int k = 0; k < n_beams; ++k)
          if (adm::beam_may_touch(beams[k], a, b)) {
            ++missed;
            break;
          }
      }
  return missed;
}
