// Device and host helpers of the library as plain C entry points, for their
// unit tests only (libpicopic_unit.so; the library itself does not contain
// this file).
#include <hip/hip_runtime.h>

#include "../pcp32.hpp"
#include "../pcp_pair_schedule.hpp"

using namespace pcp;

extern "C" {

// split_coordinate of n coordinates u of a grid of nc cells: inside[k], and
// where inside the cell and the offset
void unit_split(long n, const double *u, long nc, int *inside, long *cell, float *f) {
  for (long k = 0; k < n; ++k) inside[k] = split_coordinate(u[k], nc, cell[k], f[k]) ? 1 : 0;
}

// below_edge of the cells i[k]
void unit_below_edge(long n, const long *i, double dx, double *x) {
  for (long k = 0; k < n; ++k) x[k] = below_edge(i[k], dx);
}

// the unlike pairs of a cell of nel electrons and nion ions, chain after chain:
// particle of the less and of the more numerous species; returns their number,
// or -1 where a chain past long_chains holds more than one
long unit_unlike_pairs(int nel, int nion, int *near_, int *far_) {
  UnlikeChains U;
  U.set(nel, nion);
  long n = 0;
  for (int e = 0; e < U.n; ++e) {
    const int len = U.length(e);
    if (len > 1 && e >= U.long_chains() && U.big != U.n) return -1;
    for (int j = 0; j < len; ++j, ++n) {
      near_[n] = e;
      far_[n] = U.partner(e, j);
    }
  }
  return n;
}

// sort keys of the global cells (cr[k], cz[k]) of a grid of Dr x Dz domains of
// nr x nz cells in bins of bin_r x bin_z
void unit_sort_keys(long n, const long *cr, const long *cz, int Dr, int Dz, int nr, int nz, int bin_r, int bin_z,
                    uint32_t *key) {
  Geom g{};
  g.Dr = Dr; g.Dz = Dz; g.nr = nr; g.nz = nz;
  g.bin_r = bin_r; g.bin_z = bin_z; g.nbz = nz / bin_z;
  g.div_nr = make_fastdiv((uint32_t)nr); g.div_nz = make_fastdiv((uint32_t)nz);
  g.div_bin_r = make_fastdiv((uint32_t)bin_r); g.div_bin_z = make_fastdiv((uint32_t)bin_z);
  for (long k = 0; k < n; ++k) {
    const int I = (int)g.div_nr.div((uint32_t)cr[k]), J = (int)g.div_nz.div((uint32_t)cz[k]);
    key[k] = sort_cell_key(g, I * Dz + J, cr[k] - (long)I * nr, cz[k] - (long)J * nz);
  }
}

}  // extern "C"
