// Device and host helpers of the library as plain C entry points, for their
// unit tests only (libpicopic_unit.so; the library itself does not contain
// this file).
#include <hip/hip_runtime.h>

#include <initializer_list>
#include <utility>

#include "../pcp32.hpp"
#include "../pcp_pair_schedule.hpp"
#include "../pcp_physics.hpp"
#include "../pcp_wave.hpp"

using namespace pcp;

namespace {

// Run sums along the runs of equal keys of a wavefront of x and of masks of the
// runs themselves (0 or 1).  FORM 4 and 3: four and three values at once (the
// masks dead after it), 1: value by value.
template <int FORM>
__global__ void k_run_sums(const uint32_t *key, const float *x, float *out) {
  const Runs R = runs_of(key[threadIdx.x]);
  float a[4] = {run_mask_f(R, 5), run_mask_f(R, 1), run_mask_f(R, 4), x[threadIdx.x]};
  if (FORM == 4) run_sums_f(a[0], a[1], a[2], a[3], R);
  if (FORM == 3) run_sums_f(a[0], a[1], a[2], R);
  for (int k = 0; k < 4; ++k) out[k * 64 + threadIdx.x] = FORM == 1 ? run_sum_f(a[k], R) : a[k];
}

// reserve_groups of a wavefront: head, size and rank of every lane
__global__ void k_reserve_groups(const uint32_t *key, const int *active, int *out) {
  const ReserveGroup G = reserve_groups(key[threadIdx.x], active[threadIdx.x] != 0);
  out[threadIdx.x] = G.head;
  out[64 + threadIdx.x] = (int)G.size;
  out[128 + threadIdx.x] = (int)G.rank;
}

// out[0] a / b, out[1] a / b with b's reciprocal at hand, out[2] sqrt(b),
// out[3] a / c^2, out[4] the cell of a in cells of size b
__global__ void k_quotients(long n, const double *a, const double *b, double *out) {
  for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x) {
    out[k] = quot(a[k], b[k]);
    out[n + k] = quot(a[k], b[k], recip(b[k]));
    out[2 * n + k] = sqrt_normal(b[k]);
    out[3 * n + k] = over_c2(a[k]);
    out[4 * n + k] = (double)cell_number(a[k], b[k]);
  }
}

// a kernel's arrays on the device: inputs copied in, outputs copied back
template <class F>
int on_device(std::initializer_list<std::pair<const void *, size_t>> in, void *out, size_t out_bytes, F launch) {
  void *d[5] = {};
  int n = 0, rc = 0;
  for (const auto &a : in) {
    if (hipMalloc(&d[n], a.second) != hipSuccess ||
        hipMemcpy(d[n], a.first, a.second, hipMemcpyHostToDevice) != hipSuccess)
      rc = -1;
    ++n;
  }
  if (hipMalloc(&d[n], out_bytes) != hipSuccess) rc = -1;
  if (rc == 0) {
    launch(d, d[n]);
    if (hipGetLastError() != hipSuccess || hipMemcpy(out, d[n], out_bytes, hipMemcpyDeviceToHost) != hipSuccess) rc = -1;
  }
  for (void *p : d) (void)hipFree(p);
  return rc;
}

}  // namespace

extern "C" {

int unit_run_sums(int form, const uint32_t *key, const float *x, float *out) {
  return on_device({{key, 64 * sizeof(uint32_t)}, {x, 64 * sizeof(float)}}, out, 4 * 64 * sizeof(float),
                   [form](void **d, void *o) {
                     auto f = form == 4 ? k_run_sums<4> : form == 3 ? k_run_sums<3> : k_run_sums<1>;
                     hipLaunchKernelGGL(f, dim3(1), dim3(64), 0, 0, (const uint32_t *)d[0], (const float *)d[1],
                                        (float *)o);
                   });
}

int unit_reserve_groups(const uint32_t *key, const int *active, int *out) {
  return on_device({{key, 64 * sizeof(uint32_t)}, {active, 64 * sizeof(int)}}, out, 3 * 64 * sizeof(int),
                   [](void **d, void *o) {
                     hipLaunchKernelGGL(k_reserve_groups, dim3(1), dim3(64), 0, 0, (const uint32_t *)d[0],
                                        (const int *)d[1], (int *)o);
                   });
}

int unit_quotients(long n, const double *a, const double *b, double *out) {
  return on_device({{a, n * sizeof(double)}, {b, n * sizeof(double)}}, out, 5 * n * sizeof(double),
                   [n](void **d, void *o) {
                     hipLaunchKernelGGL(k_quotients, dim3(1024), dim3(256), 0, 0, n, (const double *)d[0],
                                        (const double *)d[1], (double *)o);
                   });
}

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
