// Binary Coulomb collisions on the device: the Collisions base pass
// (src/collisions.cpp:87-236: sort_to_cells, random_sort,
// collect_weighted_params_tot_grid) and the pairing loop shared by
// CollisionsP12 / TA77S / SK98 (collisionsP12.cpp:330-530), plus TA77S
// correct_velocities (collisionsTA77S.cpp:419-566).
//
// Pipeline per pass (two species: electrons `se`, ions `si`):
//   k_coll_count    particles per (domain, cell) bucket
//   scan            bucket offsets (hipCUB)
//   k_coll_fill     bucket lists of particle indices
//   k_coll_classify cells with both species into lists by size (at most 16,
//                   32, 64, 128, 256 or more particles of either species; a
//                   cell missing a species ends its r-row as the reference's
//                   `break` does)
//   k_coll_prep     per group of listed cells (512 particle slots of one size
//                   class, one workgroup): shuffle each bucket by ranking its
//                   particles on a Philox key of (particle id, pass), and the
//                   per-cell sums in the shuffled order
//   k_coll_stats    per listed cell, a lane each: density / temperature / Debye
//                   length, and the first cell of each r-row whose values are
//                   not normal (the reference's `break` ends the rest of that
//                   row)
//   k_coll_pairs    per group (1024 slots): the reference's pair schedule as
//                   dense lists of independent pairs over the group's cells,
//                   velocities staged in FP64; pair q of global cell c draws
//                   the uniforms Philox(seed; c << 24 | q, 2 pass + 1)
// A cell above 256 has a workgroup and a global stage of its own
// (k_coll_prep_crowd, with its statistics, and k_coll_pairs_crowd).
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <climits>

#include "pcp32.hpp"
#include "pcp_collide.hpp"
#include "pcp_collide_physics.hpp"
#include "pcp_mlp.hpp"
#include "pcp_pair_schedule.hpp"
#include "pcp_rng.hpp"
#include "pcp_wave.hpp"

namespace pcp {

namespace {

constexpr int COLL_BLOCK = 64;   // one wavefront per cell

// particle access for FP64 and FP32 split storage
struct View64 {
  SpeciesDev s;
  int cur;
  __device__ __forceinline__ bool cell_of(const Geom &g, long p, int &cr, int &cz) const {
    double r = s.r[cur][p];
    if (!(r >= 0)) return false;
    cr = cell_number(r, g.dr);
    cz = cell_number(s.z[cur][p], g.dz);
    return cr < g.Nr && cz >= 0 && cz < g.Nz;   // (the phase "move" may leave the grid)
  }
  __device__ __forceinline__ void load(long p, double v[3]) const {
    v[0] = s.vr[p]; v[1] = s.vphi[p]; v[2] = s.vz[p];
  }
  __device__ __forceinline__ void store(long p, const double v[3]) const {
    s.vr[p] = v[0]; s.vphi[p] = v[1]; s.vz[p] = v[2];
  }
  __device__ __forceinline__ double w(long p) const { return s.w[p]; }
  __device__ __forceinline__ uint64_t id(long p) const { return s.id[p]; }
  __device__ __forceinline__ long n() const { return s.n; }
};

struct View32 {
  Species32 s;
  int cur;    // position slot
  int vslot;  // velocity slot
  __device__ __forceinline__ bool cell_of(const Geom &g, long p, int &cr, int &cz) const {
    uint32_t c = s.cell[cur][p];
    if (c == DEAD_CELL) return false;
    cr = (int)g.div_Nz.div(c);
    cz = (int)(c - (uint32_t)cr * (uint32_t)g.Nz);
    return true;
  }
  __device__ __forceinline__ void load(long p, double v[3]) const {
    v[0] = s.vr[vslot][p]; v[1] = s.vphi[vslot][p]; v[2] = s.vz[vslot][p];
  }
  __device__ __forceinline__ void store(long p, const double v[3]) const {
    s.vr[vslot][p] = (float)v[0]; s.vphi[vslot][p] = (float)v[1]; s.vz[vslot][p] = (float)v[2];
  }
  __device__ __forceinline__ double w(long p) const { return (double)s.w[p]; }
  __device__ __forceinline__ uint64_t id(long p) const { return s.id[p]; }
  __device__ __forceinline__ long n() const { return s.n; }
};

// domain-major key of global cell (cr, cz): domain d = I Dz + J, then the
// cell's row-major index inside the domain (multiply-high divisions)
__device__ __forceinline__ uint32_t local_cell_key(const Geom &g, int cr, int cz) {
  const int I = (int)g.div_nr.div((uint32_t)cr), J = (int)g.div_nz.div((uint32_t)cz);
  const int lr = cr - I * g.nr, lz = cz - J * g.nz;
  return (uint32_t)(((long)(I * g.Dz + J) * g.nr + lr) * g.nz + lz);
}

// gate (optional): a device counter; the pass does nothing while it is 0.
// mask (optional): only particles of cells with mask[key] != 0 are bucketed.
__device__ __forceinline__ bool gate_closed(const unsigned long long *gate) { return gate && *gate == 0ull; }

// bucket of particle p (sentinel: removed, or its cell not in mask)
template <class V>
__device__ __forceinline__ uint32_t bucket_of(const Geom &g, const V &v, long p, long n, uint32_t sentinel,
                                              const int *mask) {
  uint32_t k = sentinel;
  int cr, cz;
  if (p < n && v.cell_of(g, p, cr, cz)) k = local_cell_key(g, cr, cz);
  if (mask && k != sentinel && !mask[k]) k = sentinel;
  return k;
}

// pass 1: particles per bucket (one atomic per run of a bucket's particles in a
// wavefront)
template <class V>
__global__ void __launch_bounds__(256) k_coll_count(Geom g, V v, uint32_t *cnt, uint32_t sentinel, const int *mask,
                                                    const unsigned long long *gate) {
  if (gate_closed(gate)) return;
  const long n = v.n();
  const long stride = (long)gridDim.x * blockDim.x;
  for (long b0 = (long)blockIdx.x * blockDim.x; b0 < n; b0 += stride) {
    const long p = b0 + threadIdx.x;
    const uint32_t k = bucket_of(g, v, p, n, sentinel, mask);
    const bool a = k != sentinel;
    (void)group_reserve(cnt, k, a);
  }
}

// pass 2: each particle's index at its bucket offset + a slot (fill counts
// from zero); the order inside a bucket is the atomics' -- the shuffle
// orders every bucket by its particles' keys
template <class V>
__global__ void __launch_bounds__(256) k_coll_fill(Geom g, V v, const uint32_t *off, uint32_t *fill, uint32_t *perm,
                                                   uint32_t sentinel, const int *mask,
                                                   const unsigned long long *gate) {
  if (gate_closed(gate)) return;
  const long n = v.n();
  const long stride = (long)gridDim.x * blockDim.x;
  for (long b0 = (long)blockIdx.x * blockDim.x; b0 < n; b0 += stride) {
    const long p = b0 + threadIdx.x;
    const uint32_t k = bucket_of(g, v, p, n, sentinel, mask);
    const bool a = k != sentinel;
    const uint32_t slot = group_reserve(fill, k, a);
    if (a) perm[off[k] + slot] = (uint32_t)p;
  }
}

__global__ void k_fill_i32(int *p, long n, int v) {
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) p[t] = v;
}

__global__ void k_fill_u32(uint32_t *p, long n) {
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) p[t] = 0;
}

// cell c (domain-major key) -> domain, local (i, j), global (cr, cz)
struct CellPos {
  int d, i, j;
  long cr, cz;
};
__device__ __forceinline__ CellPos cell_pos(const Geom &g, long c) {
  CellPos q;
  long per = (long)g.nr * g.nz;
  q.d = (int)(c / per);
  long lc = c - (long)q.d * per;
  q.i = (int)(lc / g.nz);
  q.j = (int)(lc - (long)q.i * g.nz);
  q.cr = (long)(q.d / g.Dz) * g.nr + q.i;
  q.cz = (long)(q.d % g.Dz) * g.nz + q.j;
  return q;
}

struct CellSums {
  double amount, energy, m[3];
};

// per-cell values kept between the two kernels
constexpr int TOT = 16;   // a_e E_e m_e[3] a_i E_i m_i[3] dens_e dens_i debye dens_e^(2/3) dens_i^(2/3)

// a cell's particles staged in LDS (FP64 velocities), up to MAXC per species
template <int MAXC>
struct CellStageT {
  double vx[2][MAXC], vy[2][MAXC], vz[2][MAXC], w[2][MAXC];
  uint32_t idx[2][MAXC];
};
using CellStage = CellStageT<COLL_MAXC>;

// cells are processed by size class: at most 16, 32, 64, 128 or COLL_MAXC
// particles of either species (a workgroup takes as many cells as fill its
// stage), the last class (crowded) a workgroup per cell, staged in global
// memory
constexpr int COLL_CLASSES = 6;
constexpr int COLL_GROUP_CLASSES = COLL_CLASSES - 1;
constexpr int COLL_CLASS0_SHIFT = 4;   // class k < 5 holds cells of at most 16 << k particles
static_assert((16 << (COLL_GROUP_CLASSES - 1)) == COLL_MAXC, "the last grouped class is COLL_MAXC");
// particles of all crowded cells of one pass that the global stage holds;
// beyond it a pass raises ERR_COLL_OVERFLOW
constexpr long COLL_CROWD_CAP = 1L << 22;
constexpr long COLL_CROWD_CELLS = COLL_CROWD_CAP / (COLL_MAXC + 1) + 1;
constexpr int COLL_CROWD_BLOCK = 256;

template <class V, int MAXC>
__device__ __forceinline__ void stage_species(const V &v, const uint32_t *perm, uint32_t o, int n, int s,
                                              CellStageT<MAXC> &S) {
  for (int k = threadIdx.x; k < n; k += COLL_BLOCK) {
    uint32_t p = perm[o + k];
    double vv[3];
    v.load(p, vv);
    S.idx[s][k] = p;
    S.vx[s][k] = vv[0]; S.vy[s][k] = vv[1]; S.vz[s][k] = vv[2];
    S.w[s][k] = v.w(p);
  }
}

// Cells with particles of both species go to the list of their size class;
// a cell missing a species has zero density and temperature, which ends
// the rest of its r-row (collisionsP12.cpp:351-354).
__global__ void k_coll_classify(Geom g, const uint32_t *off_e, const uint32_t *off_i, const int *mask,
                                uint32_t *lists, uint32_t *counts, uint32_t *crowd_off, int *row_bad, StepState *st,
                                const unsigned long long *gate) {
  if (gate_closed(gate)) return;
  const long ncells = (long)g.Dr * g.Dz * g.nr * g.nz;
  const long stride = (long)gridDim.x * blockDim.x;
  int err = 0;
  for (long c0 = (long)blockIdx.x * blockDim.x; c0 < ncells; c0 += stride) {
    const long c = c0 + threadIdx.x;
    int cls = -1;
    uint32_t crowd_at = 0;
    if (c < ncells && (!mask || mask[c])) {
      const int ne = (int)(off_e[c + 1] - off_e[c]), ni = (int)(off_i[c + 1] - off_i[c]);
      if (ne == 0 || ni == 0) {
        const CellPos q = cell_pos(g, c);
        atomicMin(&row_bad[(long)q.d * g.nr + q.i], q.j);
      } else {
        const int m = max(ne, ni);
        cls = 0;
        while (cls < COLL_GROUP_CLASSES && m > (16 << cls)) ++cls;
        if (cls == COLL_CLASSES - 1) {
          // a range of the crowded stage (counts[COLL_CLASSES] particles used)
          const uint32_t need = (uint32_t)(ne + ni);
          crowd_at = atomicAdd(&counts[COLL_CLASSES], need);
          if ((long)crowd_at + need > COLL_CROWD_CAP) {
            err |= ERR_COLL_OVERFLOW;
            cls = -1;
          }
        }
      }
    }
    // one counter atomic per class present in the wavefront
    const bool a = cls >= 0;
    const uint32_t at = wave_reserve(counts, a ? (uint32_t)cls : 0u, a);
    if (a) lists[(long)cls * ncells + at] = (uint32_t)c;
    if (cls == COLL_CLASSES - 1) crowd_off[at] = crowd_at;
  }
  if (err) atomicOr(&st->err, err);
}

// Collisions::collect_weighted_params_tot_grid's per-cell values from the
// cell's sums in shuffled order: density, temperature, Debye length, and
// the row break of a cell whose values are not normal
__device__ __forceinline__ void cell_stats(const Geom &g, long c, const CellSums &te, const CellSums &ti,
                                           double sum_el, double sum_ion, double *tot, int *row_bad) {
  const CellPos q = cell_pos(g, c);
  const double inv_e = 1. / EL_CHARGE;
  double temperature_el = te.energy / te.amount * inv_e;
  double temperature_ion = ti.energy / ti.amount * inv_e;
  // Collisions::geometry_cell_volume (collisions.cpp:162-170) passes
  // `i+shift` to CELL_VOLUME, which expands to 2.0 * i + shift + 1
  // (quirk kept: the macro argument is not parenthesised)
  const double shift = (double)((long)(q.d / g.Dz) * g.nr);
  const int i = q.i;
  double cell_volume = PCP_CELL_VOLUME(i+shift, g.dr, g.dz);
  double density_el = sum_el / cell_volume;
  double density_ion = sum_ion / cell_volume;
  double *t = tot + c * TOT;
  t[0] = te.amount; t[1] = te.energy; t[2] = te.m[0]; t[3] = te.m[1]; t[4] = te.m[2];
  t[5] = ti.amount; t[6] = ti.energy; t[7] = ti.m[0]; t[8] = ti.m[1]; t[9] = ti.m[2];
  t[10] = density_el; t[11] = density_ion;
  bool bad = !isnormal(temperature_ion) || !isnormal(temperature_el) || !isnormal(density_ion) ||
             !isnormal(density_el);
  t[12] = bad ? 0.0 : debye_length(density_el, density_ion, temperature_el, temperature_ion);
  // P12's s12 cap (collisionsP12.cpp) takes n^(2/3) of both species: once per cell here
  t[13] = pow(density_el, 2. / 3.);
  t[14] = pow(density_ion, 2. / 3.);
  if (bad) atomicMin(&row_bad[(long)q.d * g.nr + q.i], q.j);
}

// ---------------------------------------------------------------------------
// Grouped cells: a workgroup takes as many cells of one size class as fit its
// stage (512 or 1024 particle slots) at their class's size -- of 1024, 32 cells
// of at most 16 particles per species, ... 2 cells of at most 256.  Entry 2 g + s is species
// s of the group's cell g; its particles take the slots start[e] .. + n[e],
// one entry after another (starts at multiples of 4).
// ---------------------------------------------------------------------------
constexpr int COLL_GROUP_BLOCK = 256;
static_assert(COLL_GROUP_BLOCK == 4 * 64, "a wavefront per stage list");
constexpr int COLL_GROUP_SLOTS = 1024;   // k_coll_pairs
constexpr int COLL_PREP_SLOTS = 512;     // k_coll_prep
constexpr int COLL_GROUP_CELLS = COLL_GROUP_SLOTS >> (COLL_CLASS0_SHIFT + 1);   // the most cells of a group
static_assert(COLL_GROUP_CELLS * 2 <= 64, "a group's (cell, species) entries fit a wavefront");

// group number `it` over the class lists: its cells and their list entries
// (false: past the last group)
struct CellGroup {
  int cells;
  const uint32_t *list;
};
template <int SLOTS>
__device__ __forceinline__ bool cell_group(uint32_t it, const uint32_t *lists, const uint32_t *counts, long ncells,
                                           CellGroup &G) {
  // the largest cells first: their groups run longest
  for (int cls = COLL_GROUP_CLASSES - 1; cls >= 0; --cls) {
    const uint32_t n = counts[cls];
    const uint32_t per = SLOTS >> (COLL_CLASS0_SHIFT + cls + 1);
    const uint32_t ng = (n + per - 1) / per;
    if (it < ng) {
      G.cells = (int)min(per, n - it * per);
      G.list = lists + (long)cls * ncells + it * per;
      return true;
    }
    it -= ng;
  }
  return false;
}

// exclusive sum over a wavefront of one value per lane into out[0 .. 64]
__device__ __forceinline__ void wave_starts(int v, int lane, int out[65]) {
  int x = v;
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  out[lane + 1] = x;
  if (lane == 0) out[0] = 0;
}
// the e with start[e] <= t < start[e + 1]
__device__ __forceinline__ int entry_of(const int start[65], int t) {
  int e = 0, hi = 64;
  while (hi - e > 1) {
    const int mid = (e + hi) >> 1;
    if (start[mid] <= t) e = mid;
    else hi = mid;
  }
  return e;
}

// the buckets of a group: offset into perm, particles, first slot
struct GroupEntries {
  uint32_t off[64];
  int n[64];
  int start[65];
  // by the first wavefront; a barrier follows
  __device__ __forceinline__ void load(const CellGroup &G, const uint32_t *off_e, const uint32_t *off_i) {
    if (threadIdx.x >= 64) return;
    const int e = threadIdx.x;
    int cnt = 0;
    if (e < 2 * G.cells) {
      const long c = G.list[e >> 1];
      const uint32_t *o = (e & 1) ? off_i : off_e;
      off[e] = o[c];
      cnt = (int)(o[c + 1] - o[c]);
    }
    n[e] = cnt;
    wave_starts((cnt + 3) & ~3, e, start);
  }
};

// Shuffle and cell sums.  A particle's place is its rank among its bucket's
// 32-bit Philox keys (n comparisons against broadcast LDS reads of four keys,
// no barrier in the loop; equal keys, found by two particles claiming one
// place, are ranked again by (key, id, index)).  The sums run in the shuffled
// order, one thread per (quantity, species, cell).  Bound by latency: the
// bitonic sort and one-thread sums of a wavefront per cell took 6.2 ms per pass
// on a million cells of 32 + 32 FP64 particles on average (the ranks at a
// 1024-slot stage, 12 wavefronts per CU, still 2.7), this 2.1 with k_coll_stats.
template <class V>
__global__ void __launch_bounds__(COLL_GROUP_BLOCK) k_coll_prep(Geom g, V ve, V vi, const uint32_t *off_e,
                                                                const uint32_t *off_i, uint32_t *perm_e,
                                                                uint32_t *perm_i, double m_e, double m_i,
                                                                uint64_t seed, PassNo pass, double *tot,
                                                                const uint32_t *lists, const uint32_t *counts,
                                                                long ncells, const unsigned long long *gate) {
  __shared__ GroupEntries E;
  __shared__ __align__(16) uint32_t skey[COLL_PREP_SLOTS];
  __shared__ uint32_t sidx[COLL_PREP_SLOTS], claim[COLL_PREP_SLOTS];
  __shared__ double sx[COLL_PREP_SLOTS], sy[COLL_PREP_SLOTS], sz[COLL_PREP_SLOTS], sw[COLL_PREP_SLOTS];
  __shared__ int tie;
  if (gate_closed(gate)) return;
  const uint64_t step = pass.get();
  CellGroup G;
  for (uint32_t it = blockIdx.x; cell_group<COLL_PREP_SLOTS>(it, lists, counts, ncells, G); it += gridDim.x) {
    const int entries = 2 * G.cells;
    E.load(G, off_e, off_i);
    if (threadIdx.x == 0) tie = 0;
    __syncthreads();
    const int slots = E.start[64];
    for (int t = threadIdx.x; t < slots; t += COLL_GROUP_BLOCK) {
      const int e = entry_of(E.start, t), k = t - E.start[e];
      uint32_t key = 0xFFFFFFFFu;
      claim[t] = 0;
      if (k < E.n[e]) {
        const uint32_t p = ((e & 1) ? perm_i : perm_e)[E.off[e] + k];
        const uint64_t id = (e & 1) ? vi.id(p) : ve.id(p);
        uint32_t ph[4];
        philox4x32(id, (uint32_t)(2 * step), seed, ph);
        key = ph[0];
        sidx[t] = p;
      }
      skey[t] = key;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < slots; t += COLL_GROUP_BLOCK) {
      const int e = entry_of(E.start, t), base = E.start[e], n = E.n[e];
      if (t - base >= n) continue;
      const uint32_t key = skey[t], p = sidx[t];
      double v3[3], w;
      if (e & 1) { vi.load(p, v3); w = vi.w(p); }
      else { ve.load(p, v3); w = ve.w(p); }
      int r = 0;
#pragma unroll 4
      for (int j = 0; j < n; j += 4) {
        const uint4 q = *(const uint4 *)(skey + base + j);
        r += (int)(q.x < key) + (int)(q.y < key) + (int)(q.z < key) + (int)(q.w < key);
      }
      if (atomicExch(&claim[base + r], 1u)) tie = 1;
      ((e & 1) ? perm_i : perm_e)[E.off[e] + r] = p;
      sx[base + r] = v3[0]; sy[base + r] = v3[1]; sz[base + r] = v3[2];
      sw[base + r] = w;
    }
    __syncthreads();
    if (tie) {
      // two particles of a bucket drew the same key: rank by (key, low id bits, index)
      for (int t = threadIdx.x; t < slots; t += COLL_GROUP_BLOCK) {
        const int e = entry_of(E.start, t), base = E.start[e], n = E.n[e];
        if (t - base >= n) continue;
        const uint32_t key = skey[t], p = sidx[t];
        const uint32_t id = (uint32_t)((e & 1) ? vi.id(p) : ve.id(p));
        int r = 0;
        for (int j = 0; j < n; ++j) {
          bool less = skey[base + j] < key;
          if (skey[base + j] == key && base + j != t) {
            const uint32_t pj = sidx[base + j], idj = (uint32_t)((e & 1) ? vi.id(pj) : ve.id(pj));
            less = idj < id || (idj == id && pj < p);
          }
          r += less ? 1 : 0;
        }
        double v3[3], w;
        if (e & 1) { vi.load(p, v3); w = vi.w(p); }
        else { ve.load(p, v3); w = ve.w(p); }
        ((e & 1) ? perm_i : perm_e)[E.off[e] + r] = p;
        sx[base + r] = v3[0]; sy[base + r] = v3[1]; sz[base + r] = v3[2];
        sw[base + r] = w;
      }
      __syncthreads();
    }
    // collect_weighted_params_tot_grid: 0 weight, 1 energy, 2-4 momentum
    for (int t = threadIdx.x; t < 5 * 64; t += COLL_GROUP_BLOCK) {
      const int q = t >> 6, e = t & 63;
      if (e >= entries) continue;
      const int n = E.n[e], base = E.start[e];
      const double mass = (e & 1) ? m_i : m_e;
      const double *v = q == 2 ? sx : q == 3 ? sy : sz;
      double a = 0;
      if (q >= 2) {
#pragma unroll 4
        for (int k = 0; k < n; ++k) a += sw[base + k] * mass * v[base + k];
      } else if (q == 0) {
#pragma unroll 4
        for (int k = 0; k < n; ++k) a += sw[base + k];
      } else {
#pragma unroll 4
        for (int k = 0; k < n; ++k) {
          const double vr = sx[base + k], vphi = sy[base + k], vz = sz[base + k];
          const double v_sq = vr * vr + vphi * vphi + vz * vz;
          a += sw[base + k] * mass * v_sq / 2;
        }
      }
      tot[(long)G.list[e >> 1] * TOT + 5 * (e & 1) + q] = a;
    }
    __syncthreads();
  }
}

// density, temperature and Debye length of the grouped classes' cells from
// k_coll_prep's sums, a lane per cell (in k_coll_prep the few cells of a group
// kept 4 lanes of a wavefront busy for it)
__global__ void __launch_bounds__(256) k_coll_stats(Geom g, double *tot, int *row_bad, const uint32_t *lists,
                                                    const uint32_t *counts, long ncells,
                                                    const unsigned long long *gate) {
  if (gate_closed(gate)) return;
  for (int cls = 0; cls < COLL_GROUP_CLASSES; ++cls) {
    const uint32_t n = counts[cls];
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
      const long c = lists[(long)cls * ncells + t];
      const double *s = tot + c * TOT;
      const CellSums te{s[0], s[1], {s[2], s[3], s[4]}}, ti{s[5], s[6], {s[7], s[8], s[9]}};
      cell_stats(g, c, te, ti, te.amount, ti.amount, tot, row_bad);
    }
  }
}

struct CrowdStage {
  double *b;     // the cell's range of the crowded stage
  int n0;        // electrons first, then ions
  __device__ __forceinline__ double &at(int c, int s, int k) const { return b[c * COLL_CROWD_CAP + s * n0 + k]; }
  __device__ __forceinline__ double &vx(int s, int k) const { return at(0, s, k); }
  __device__ __forceinline__ double &vy(int s, int k) const { return at(1, s, k); }
  __device__ __forceinline__ double &vz(int s, int k) const { return at(2, s, k); }
  __device__ __forceinline__ double &w(int s, int k) const { return at(3, s, k); }
};

// One pair, out of line: the schedule below calls it from several places.  Only
// the arithmetic is: with the draws and the stage's loads inside the call the
// runner's state went through scratch (SK98 146 -> 244 registers).  The serial
// sums of a crowded cell (correct_params, k_coll_prep_crowd) are unrolled so
// that four particles' loads are under way at once, and the addresses that this
// file's build forms anew in each trip count less.  A pass over 7000 cells of
// 300 + 300 FP64 particles, P12 / TA77S / SK98: 4.02 / 5.24 / 4.04 ms, now
// 3.03 / 3.65 / 3.00.
template <int SCHEME>
__device__ __noinline__ void collide_pair_call(double m_a, double m_b, double q_a, double q_b, double *va, double wa,
                                               double *vb, double wb, double dens_a, double dens_b, const P12Cell &K,
                                               double debye, double dt, PairDraws &R, int *err) {
  collide_pair<SCHEME>(m_a, m_b, q_a, q_b, va, wa, vb, wb, dens_a, dens_b, K, debye, dt, R, err);
}

// The pairs of a crowded cell, its independent pairs and chains spread over the
// workgroup's threads
template <int SCHEME>
struct PairRunner {
  CrowdStage S;
  double m[2], q[2];   // electrons, ions
  double dens[2], debye, dt;
  uint64_t seed, step, gcell;
  int *err;
  P12Cell K[3];   // P12: electron, unlike, ion pairs
  __device__ __forceinline__ void pair(int sa, int ka, int sb, int kb, uint32_t ord) {
    PairDraws R;
    uint64_t ctr = (gcell << 24) | (uint64_t)(ord & 0xFFFFFFu);
    uint32_t draw = (uint32_t)(2 * step + 1);
    uniform2(ctr, draw, seed, R.u[0], R.u[1]);
    uniform2(ctr ^ (1ull << 63), draw, seed, R.u[2], R.u[3]);
    R.pos = 0;
    double va[3] = {S.vx(sa, ka), S.vy(sa, ka), S.vz(sa, ka)};
    double vb[3] = {S.vx(sb, kb), S.vy(sb, kb), S.vz(sb, kb)};
    collide_pair_call<SCHEME>(m[sa], m[sb], q[sa], q[sb], va, S.w(sa, ka), vb, S.w(sb, kb), dens[sa], dens[sb],
                              K[sa + sb], debye, dt, R, err);
    S.vx(sa, ka) = va[0]; S.vy(sa, ka) = va[1]; S.vz(sa, ka) = va[2];
    S.vx(sb, kb) = vb[0]; S.vy(sb, kb) = vb[1]; S.vz(sb, kb) = vb[2];
  }
  // like-particle pairs of species s (cases 1a / 1b), ordinals from qb
  __device__ void like(int s, int n, uint32_t qb) {
    if (n % 2 == 0) {
      for (int k = threadIdx.x; k < n / 2; k += COLL_CROWD_BLOCK) pair(s, 2 * k, s, 2 * k + 1, qb + (uint32_t)k);
    } else {
      if (n >= 3 && threadIdx.x == 0) {
        pair(s, 0, s, 1, qb);
        pair(s, 1, s, 2, qb + 1);
        pair(s, 2, s, 0, qb + 2);
      }
      if (n >= 5)
        for (int k = threadIdx.x; k < (n - 3) / 2; k += COLL_CROWD_BLOCK)
          pair(s, 3 + 2 * k, s, 4 + 2 * k, qb + 3 + (uint32_t)k);
    }
    __syncthreads();
  }
  __device__ void run(int nel, int nion) {
    // cases 1a/1b in reference order: ion pairs if nion is even, electron pairs
    // if nel is even, ion pairs if nion is odd, electron pairs if nel is odd
    const uint32_t n_ion = like_pairs(nion), n_el = like_pairs(nel);
    const bool el_first = nion % 2 != 0 && nel % 2 == 0;
    like(1, nion, el_first ? n_el : 0);
    like(0, nel, el_first ? 0 : n_ion);
    // case 2a / 2b
    UnlikeChains U;
    U.set(nel, nion);
    for (int e = threadIdx.x; e < U.n; e += COLL_CROWD_BLOCK) {
      const int len = U.length(e);
      for (int j = 0; j < len; ++j) {
        const int far = U.partner(e, j);
        pair(0, nel <= nion ? e : far, 1, nel <= nion ? far : e, n_ion + n_el + (uint32_t)far);
      }
    }
    __syncthreads();
  }
};

// TA77S correct_velocities for species s of the staged cell; t = the cell's
// {amount, energy, moment[3]} from before the collisions
struct CorrParams {
  double ok, alpha, V0[3], dV[3];
};
template <class Stage>
__device__ CorrParams correct_params(const Stage &S, int s, int n, double mass, const double *t) {
  CorrParams P;
  double m_new[3] = {0, 0, 0}, E_new = 0;
#pragma unroll 4
  for (int k = 0; k < n; ++k) {
    double vr = S.vx(s, k), vphi = S.vy(s, k), vz = S.vz(s, k);
    double v_sq = vr * vr + vphi * vphi + vz * vz;
    double mass_m = mass * S.w(s, k);
    m_new[0] += mass_m * vr;
    m_new[1] += mass_m * vphi;
    m_new[2] += mass_m * vz;
    E_new += mass_m * v_sq / 2;
  }
  const double amount = t[0], energy = t[1];
  double mass_tot = amount * mass;
  double dV[3], V0[3];
  for (int k = 0; k < 3; ++k) dV[k] = (m_new[k] - t[2 + k]) / mass_tot;
  for (int k = 0; k < 3; ++k) V0[k] = t[2 + k] / mass_tot;
  double delta_E = E_new - energy;
  double V0_sq = V0[0] * V0[0] + V0[1] * V0[1] + V0[2] * V0[2];
  double alpha = (energy - mass_tot * V0_sq / 2) /
                 (energy + delta_E -
                  mass_tot * (pow(V0[0] + dV[0], 2) + pow(V0[1] + dV[1], 2) + pow(V0[2] + dV[2], 2)) / 2);
  bool ok = isnormal(alpha);
  if (ok) {
    if (alpha < 0) alpha = -alpha;
    if (alpha == 0) alpha = 1;
    alpha = sqrt(alpha);
  }
  P.ok = ok ? 1.0 : 0.0;
  P.alpha = alpha;
  for (int k = 0; k < 3; ++k) { P.V0[k] = V0[k]; P.dV[k] = dV[k]; }
  return P;
}

__device__ void correct_species(const CrowdStage &S, int s, int n, double mass, const double *t) {
  __shared__ CorrParams shared_p;
  if (threadIdx.x == 0) shared_p = correct_params(S, s, n, mass, t);
  __syncthreads();
  const CorrParams P = shared_p;
  if (P.ok != 0.0) {
    const double alpha = P.alpha;
    for (int k = threadIdx.x; k < n; k += COLL_CROWD_BLOCK) {
      double vr = S.vx(s, k), vphi = S.vy(s, k), vz = S.vz(s, k);
      S.vx(s, k) = P.V0[0] + alpha * (vr - P.V0[0] - P.dV[0]);
      S.vy(s, k) = P.V0[1] + alpha * (vphi - P.V0[1] - P.dV[1]);
      S.vz(s, k) = P.V0[2] + alpha * (vz - P.V0[2] - P.dV[2]);
    }
  }
  __syncthreads();
}

// what a pair takes from its cell
struct CellStatsLds {
  double dens[2], debye;
  uint64_t gcell;
  UnlikeChains chains;
  int active;
};

// one bucket's slots, for correct_params
struct SlotStage {
  const double *x, *y, *z, *wt;
  __device__ __forceinline__ double vx(int, int k) const { return x[k]; }
  __device__ __forceinline__ double vy(int, int k) const { return y[k]; }
  __device__ __forceinline__ double vz(int, int k) const { return z[k]; }
  __device__ __forceinline__ double w(int, int k) const { return wt[k]; }
};

struct PairStage {
  double vx[COLL_GROUP_SLOTS], vy[COLL_GROUP_SLOTS], vz[COLL_GROUP_SLOTS], w[COLL_GROUP_SLOTS];
};

// The pairs of a group run as stages of independent pairs or chains, each a
// dense list over the group's cells that the workgroup's wavefronts take 64
// entries at a time: the like pairs with the first of an odd bucket's three
// chained ones, the rest of those chains, the first pair of every unlike
// chain, the rest of the unlike chains.  Bound by FP64 instruction issue, so
// what counts is how many of a wavefront's lanes hold a pair: a wavefront per
// cell ran 40 + 40 particles as passes of 20, 20 and 40 of 64 lanes, and a lane
// per cell the cells of up to 16.  One P12 pass over a million cells of 32 + 32
// FP64 particles on average: 21.5 ms that way, 10.6 with the dense lists (and
// the same pair arithmetic), 6.7 with p12_collide's shared reciprocals, 5.4 at
// three wavefronts per SIMD (two without the limit; with the machine LICM pass
// off, which kept the pair's FP64 constants in registers over the whole loop,
// the limit spills 10 registers instead of 92; four spill 51 and measure the
// same).
template <int SCHEME, class V>
__global__ void __launch_bounds__(COLL_GROUP_BLOCK) __attribute__((amdgpu_waves_per_eu(3))) k_coll_pairs(
    Geom g, V ve, V vi, const uint32_t *off_e, const uint32_t *off_i, const uint32_t *perm_e, const uint32_t *perm_i,
    double m_e, double m_i, double q_e, double q_i, uint64_t seed, PassNo pass, const double *tot, const int *row_bad,
    const uint32_t *lists, const uint32_t *counts, long ncells, StepState *st, const unsigned long long *gate) {
  constexpr int STAGES = 4;
  __shared__ PairStage S;
  __shared__ GroupEntries E;
  __shared__ CellStatsLds C[COLL_GROUP_CELLS];
  __shared__ P12Cell K[SCHEME == COLL_P12 ? COLL_GROUP_CELLS : 1][3];
  __shared__ int pre[STAGES][65];
  __shared__ uint32_t ticket[STAGES];
  if (gate_closed(gate)) return;
  const uint64_t step = pass.get();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int err = 0;
  CellGroup G;
  for (uint32_t it = blockIdx.x; cell_group<COLL_GROUP_SLOTS>(it, lists, counts, ncells, G); it += gridDim.x) {
    const int entries = 2 * G.cells;
    E.load(G, off_e, off_i);
    if (wave == 1 && lane < G.cells) {
      const long c = G.list[lane];
      const CellPos q = cell_pos(g, c);
      const double *t = tot + c * TOT;
      CellStatsLds &L = C[lane];
      L.dens[0] = t[10]; L.dens[1] = t[11]; L.debye = t[12];
      L.gcell = (uint64_t)q.cr * (uint64_t)g.Nz + (uint64_t)q.cz;
      L.active = q.j < row_bad[(long)q.d * g.nr + q.i];
      L.chains.set((int)(off_e[c + 1] - off_e[c]), (int)(off_i[c + 1] - off_i[c]));
    }
    if (SCHEME == COLL_P12 && wave >= 2) {
      const int t = (int)threadIdx.x - 128;
      if (t < 3 * G.cells) {
        const int i = t / 3, k = t - 3 * i;
        K[i][k].set_species(k, m_e, m_i, q_e, q_i, tot + (long)G.list[i] * TOT + 10, g.dt);
      }
    }
    if (threadIdx.x < STAGES) ticket[threadIdx.x] = 0;
    __syncthreads();
    const int slots = E.start[64];
    for (int t = threadIdx.x; t < slots; t += COLL_GROUP_BLOCK) {
      const int e = entry_of(E.start, t), k = t - E.start[e];
      if (k >= E.n[e]) continue;
      const uint32_t p = ((e & 1) ? perm_i : perm_e)[E.off[e] + k];
      double v3[3], w;
      if (e & 1) { vi.load(p, v3); w = vi.w(p); }
      else { ve.load(p, v3); w = ve.w(p); }
      S.vx[t] = v3[0]; S.vy[t] = v3[1]; S.vz[t] = v3[2];
      S.w[t] = w;
    }
    // list starts of the stages, a wavefront each: (cell, species) entries of
    // stages 0 and 1, cells of 2 and 3
    {
      int v = 0;
      if (wave < 2) {
        if (lane < entries && C[lane >> 1].active) {
          const int n = E.n[lane];
          v = wave == 0 ? n >> 1 : (n % 2 != 0 && n >= 3) ? 1 : 0;
        }
      } else if (lane < G.cells && C[lane].active) {
        const UnlikeChains &U = C[lane].chains;
        v = wave == 2 ? U.n : U.big == U.n ? 0 : U.long_chains();
      }
      wave_starts(v, lane, pre[wave]);
    }
    __syncthreads();
    for (int stage = 0; stage < STAGES; ++stage) {
      const int total = pre[stage][64];
      if (total == 0) continue;
      for (;;) {
        uint32_t b = 0;
        if (lane == 0) b = atomicAdd(&ticket[stage], 64u);
        const int p = __builtin_amdgcn_readfirstlane((int)b) + lane;
        if (p - lane >= total) break;
        // this lane's chain: pairs j0 .. j1 of number k of entry e
        int e = 0, k = 0, j0 = 0, j1 = 0;
        if (p < total) {
          e = entry_of(pre[stage], p);
          k = p - pre[stage][e];
          if (stage == 0) j1 = 1;
          else if (stage == 1) { j0 = 1; j1 = 3; }
          else {
            const int len = C[e].chains.length(k);
            j0 = stage - 2;
            j1 = stage == 2 ? min(len, 1) : len;
          }
        }
        for (int j = j0; j < j1; ++j) {
          int cell, sa, sb, ka, kb;
          uint32_t ord;
          if (stage < 2) {
            cell = e >> 1;
            sa = sb = e & 1;
            const int n = E.n[e], nel = E.n[2 * cell], nion = E.n[2 * cell + 1];
            // ordinals in reference order: ion pairs if nion is even, electron
            // pairs if nel is even, ion pairs if nion is odd, electron pairs if
            // nel is odd
            const bool el_first = nion % 2 != 0 && nel % 2 == 0;
            ord = sa == 0 ? (el_first ? 0 : like_pairs(nion)) : (el_first ? like_pairs(nel) : 0);
            if (n % 2 == 0) {
              ka = 2 * k;
              kb = ka + 1;
              ord += (uint32_t)k;
            } else if (k == 0) {
              // the chain (0, 1), (1, 2), (2, 0)
              ka = j;
              kb = j == 2 ? 0 : j + 1;
              ord += (uint32_t)j;
            } else {
              ka = 2 * k + 1;
              kb = ka + 1;
              ord += (uint32_t)(k + 2);
            }
          } else {
            cell = e;
            sa = 0;
            sb = 1;
            const int nel = E.n[2 * cell], nion = E.n[2 * cell + 1];
            const int far = C[cell].chains.partner(k, j);
            ka = nel <= nion ? k : far;
            kb = nel <= nion ? far : k;
            ord = like_pairs(nel) + like_pairs(nion) + (uint32_t)far;
          }
          const CellStatsLds &L = C[cell];
          const int ta = E.start[2 * cell + sa] + ka, tb = E.start[2 * cell + sb] + kb;
          PairDraws R;
          const uint64_t ctr = (L.gcell << 24) | (uint64_t)(ord & 0xFFFFFFu);
          const uint32_t draw = (uint32_t)(2 * step + 1);
          const double wa = S.w[ta], wb = S.w[tb];
          uniform2(ctr, draw, seed, R.u[0], R.u[1]);
          // P12 takes one more, compared with the weights: below them when both are 1 or more
          R.u[2] = 0;
          if (SCHEME != COLL_P12 || !(wa >= 1 && wb >= 1)) uniform2(ctr ^ (1ull << 63), draw, seed, R.u[2], R.u[3]);
          R.pos = 0;
          double va[3] = {S.vx[ta], S.vy[ta], S.vz[ta]};
          double vb[3] = {S.vx[tb], S.vy[tb], S.vz[tb]};
          collide_pair<SCHEME>(sa ? m_i : m_e, sb ? m_i : m_e, sa ? q_i : q_e, sb ? q_i : q_e, va, wa, vb, wb,
                               L.dens[sa], L.dens[sb], K[SCHEME == COLL_P12 ? cell : 0][sa + sb], L.debye, g.dt, R,
                               &err);
          S.vx[ta] = va[0]; S.vy[ta] = va[1]; S.vz[ta] = va[2];
          S.vx[tb] = vb[0]; S.vy[tb] = vb[1]; S.vz[tb] = vb[2];
        }
      }
      __syncthreads();
    }
    if (SCHEME == COLL_TA77S) {
      // correct_velocities runs over every cell
      __shared__ CorrParams corr[64];
      if ((int)threadIdx.x < entries) {
        const int e = threadIdx.x, o = E.start[e];
        const SlotStage T{S.vx + o, S.vy + o, S.vz + o, S.w + o};
        corr[e] = correct_params(T, 0, E.n[e], (e & 1) ? m_i : m_e, tot + (long)G.list[e >> 1] * TOT + 5 * (e & 1));
      }
      __syncthreads();
      for (int t = threadIdx.x; t < slots; t += COLL_GROUP_BLOCK) {
        const CorrParams &P = corr[entry_of(E.start, t)];
        if (P.ok == 0.0) continue;
        S.vx[t] = P.V0[0] + P.alpha * (S.vx[t] - P.V0[0] - P.dV[0]);
        S.vy[t] = P.V0[1] + P.alpha * (S.vy[t] - P.V0[1] - P.dV[1]);
        S.vz[t] = P.V0[2] + P.alpha * (S.vz[t] - P.V0[2] - P.dV[2]);
      }
    }
    // every thread stores the slots that it staged (and corrected)
    for (int t = threadIdx.x; t < slots; t += COLL_GROUP_BLOCK) {
      const int e = entry_of(E.start, t), k = t - E.start[e];
      if (k >= E.n[e]) continue;
      const uint32_t p = ((e & 1) ? perm_i : perm_e)[E.off[e] + k];
      const double v3[3] = {S.vx[t], S.vy[t], S.vz[t]};
      if (e & 1) vi.store(p, v3);
      else ve.store(p, v3);
    }
    __syncthreads();
  }
  if (err) atomicOr(&st->err, err);
}

// ---------------------------------------------------------------------------
// Crowded cells (more than COLL_MAXC particles of a species): a workgroup per
// cell.  The shuffle sorts the cell's keys in the global key array with a
// bitonic network whose comparators all run ascending (the first merge step
// of each stage mirrors), so entries past n act as +inf and are skipped; the
// pairs run the same schedule on an FP64 stage in global memory.
// ---------------------------------------------------------------------------
template <class V>
__device__ void crowd_shuffle(const V &v, uint32_t *perm, uint32_t o, int n, uint64_t seed, uint64_t step,
                              uint64_t *key, uint32_t *idx) {
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    const uint32_t p = perm[o + k];
    const uint64_t id = v.id(p);
    uint32_t ph[4];
    philox4x32(id, (uint32_t)(2 * step), seed, ph);
    key[k] = ((uint64_t)ph[0] << 32) | (id & 0xFFFFFFFFull);
    idx[k] = p;
  }
  __syncthreads();
  int P = 1;
  while (P < n) P <<= 1;
  for (int kk = 2; kk <= P; kk <<= 1)
    for (int j = kk >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < P; i += blockDim.x) {
        const int l = j == (kk >> 1) ? (i ^ (kk - 1)) : (i ^ j);
        if (l > i && l < n) {
          const uint64_t a = key[i], b = key[l];
          if (a > b || (a == b && idx[i] > idx[l])) {
            key[i] = b;
            key[l] = a;
            const uint32_t x = idx[i];
            idx[i] = idx[l];
            idx[l] = x;
          }
        }
      }
      __syncthreads();
    }
  for (int k = threadIdx.x; k < n; k += blockDim.x) perm[o + k] = idx[k];
  __syncthreads();
}

template <class V>
__device__ __forceinline__ void crowd_stage_species(const V &v, const uint32_t *perm, uint32_t o, int n, int s,
                                                    const CrowdStage &S) {
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    const uint32_t p = perm[o + k];
    double vv[3];
    v.load(p, vv);
    S.vx(s, k) = vv[0]; S.vy(s, k) = vv[1]; S.vz(s, k) = vv[2];
    S.w(s, k) = v.w(p);
  }
}

template <class V>
__global__ void __launch_bounds__(COLL_CROWD_BLOCK) k_coll_prep_crowd(
    Geom g, V ve, V vi, const uint32_t *off_e, const uint32_t *off_i, uint32_t *perm_e, uint32_t *perm_i, double m_e,
    double m_i, uint64_t seed, PassNo pass, double *tot, int *row_bad, const uint32_t *list, const uint32_t *count,
    const uint32_t *crowd_off, uint64_t *ckey, uint32_t *cidx, double *cstage, const unsigned long long *gate) {
  const uint64_t step = pass.get();
  if (gate_closed(gate)) return;
  const uint32_t nlist = *count;
  for (uint32_t li = blockIdx.x; li < nlist; li += gridDim.x) {
    const long c = list[li];
    const int nn[2] = {(int)(off_e[c + 1] - off_e[c]), (int)(off_i[c + 1] - off_i[c])};
    const uint32_t base = crowd_off[li];
    crowd_shuffle(ve, perm_e, off_e[c], nn[0], seed, step, ckey + base, cidx + base);
    crowd_shuffle(vi, perm_i, off_i[c], nn[1], seed, step, ckey + base + nn[0], cidx + base + nn[0]);
    const CrowdStage S{cstage + base, nn[0]};
    crowd_stage_species(ve, perm_e, off_e[c], nn[0], 0, S);
    crowd_stage_species(vi, perm_i, off_i[c], nn[1], 1, S);
    __syncthreads();
    if (threadIdx.x == 0) {
      // cell_sums in the shuffled order, from the stage
      CellSums t[2];
      double sum_w[2];
      const double mass[2] = {m_e, m_i};
      for (int sp = 0; sp < 2; ++sp) {
        t[sp] = CellSums{0, 0, {0, 0, 0}};
        sum_w[sp] = 0;
#pragma unroll 4
        for (int k = 0; k < nn[sp]; ++k) {
          double vr = S.vx(sp, k), vphi = S.vy(sp, k), vzz = S.vz(sp, k), w = S.w(sp, k);
          double v_sq = vr * vr + vphi * vphi + vzz * vzz;
          double weighted_m = w * mass[sp];
          t[sp].m[0] += weighted_m * vr;
          t[sp].m[1] += weighted_m * vphi;
          t[sp].m[2] += weighted_m * vzz;
          t[sp].amount += w;
          t[sp].energy += weighted_m * v_sq / 2;
        }
#pragma unroll 4
        for (int k = 0; k < nn[sp]; ++k) sum_w[sp] += S.w(sp, k);
      }
      cell_stats(g, c, t[0], t[1], sum_w[0], sum_w[1], tot, row_bad);
    }
    __syncthreads();
  }
}

template <int SCHEME, class V>
__global__ void __launch_bounds__(COLL_CROWD_BLOCK) k_coll_pairs_crowd(
    Geom g, V ve, V vi, const uint32_t *off_e, const uint32_t *off_i, const uint32_t *perm_e, const uint32_t *perm_i,
    double m_e, double m_i, double q_e, double q_i, uint64_t seed, PassNo pass, const double *tot,
    const int *row_bad, const uint32_t *list, const uint32_t *count, const uint32_t *crowd_off, double *cstage,
    StepState *st, const unsigned long long *gate) {
  const uint64_t step = pass.get();
  if (gate_closed(gate)) return;
  const uint32_t nlist = *count;
  int err = 0;
  for (uint32_t li = blockIdx.x; li < nlist; li += gridDim.x) {
    const long c = list[li];
    const int nn[2] = {(int)(off_e[c + 1] - off_e[c]), (int)(off_i[c + 1] - off_i[c])};
    const CrowdStage S{cstage + crowd_off[li], nn[0]};
    crowd_stage_species(ve, perm_e, off_e[c], nn[0], 0, S);
    crowd_stage_species(vi, perm_i, off_i[c], nn[1], 1, S);
    __syncthreads();
    const CellPos q = cell_pos(g, c);
    const double *t = tot + c * TOT;
    if (q.j < row_bad[(long)q.d * g.nr + q.i]) {
      PairRunner<SCHEME> P{S, {m_e, m_i}, {q_e, q_i}, {t[10], t[11]}, t[12], g.dt, seed, step,
                           (uint64_t)q.cr * (uint64_t)g.Nz + (uint64_t)q.cz, &err, {}};
      if (SCHEME == COLL_P12)
        for (int k = 0; k < 3; ++k) P.K[k].set_species(k, m_e, m_i, q_e, q_i, t + 10, g.dt);
      P.run(nn[0], nn[1]);
    }
    if (SCHEME == COLL_TA77S) {
      correct_species(S, 1, nn[1], m_i, t + 5);
      correct_species(S, 0, nn[0], m_e, t + 0);
    }
    for (int k = threadIdx.x; k < nn[0]; k += COLL_CROWD_BLOCK) {
      double v3[3] = {S.vx(0, k), S.vy(0, k), S.vz(0, k)};
      ve.store(perm_e[off_e[c] + k], v3);
    }
    for (int k = threadIdx.x; k < nn[1]; k += COLL_CROWD_BLOCK) {
      double v3[3] = {S.vx(1, k), S.vy(1, k), S.vz(1, k)};
      vi.store(perm_i[off_i[c] + k], v3);
    }
    __syncthreads();
  }
  if (err) atomicOr(&st->err, err);
}

// ---------------------------------------------------------------------------
// collision surrogate (no reference counterpart)
// ---------------------------------------------------------------------------
// per-cell moments, per species: count, sum w, sum w v (3), sum w v_z^2,
// sum w (v_r^2 + v_phi^2)
constexpr int SST = 16;

template <class V>
__device__ __forceinline__ void species_moments(const V &v, const uint32_t *perm, uint32_t o, int n, double *out) {
  double a[7] = {0, 0, 0, 0, 0, 0, 0};
  for (int k = threadIdx.x; k < n; k += COLL_BLOCK) {
    const uint32_t p = perm[o + k];
    double vv[3];
    v.load(p, vv);
    const double w = v.w(p);
    a[0] += 1.0;
    a[1] += w;
    a[2] += w * vv[0];
    a[3] += w * vv[1];
    a[4] += w * vv[2];
    a[5] += w * vv[2] * vv[2];
    a[6] += w * (vv[0] * vv[0] + vv[1] * vv[1]);
  }
#pragma unroll
  for (int q = 0; q < 7; ++q) a[q] = wave_sum(a[q]);
  if (threadIdx.x == 0)
    for (int q = 0; q < 7; ++q) out[q] = a[q];
}

template <class V>
__global__ void __launch_bounds__(COLL_BLOCK) k_surr_moments(Geom g, V ve, V vi, const uint32_t *off_e,
                                                             const uint32_t *off_i, const uint32_t *perm_e,
                                                             const uint32_t *perm_i, double *mom) {
  const long ncells = (long)g.Dr * g.Dz * g.nr * g.nz;
  for (long c = blockIdx.x; c < ncells; c += gridDim.x) {
    species_moments(ve, perm_e, off_e[c], (int)(off_e[c + 1] - off_e[c]), mom + c * SST);
    species_moments(vi, perm_i, off_i[c], (int)(off_i[c + 1] - off_i[c]), mom + c * SST + 8);
  }
}

// temperatures [eV] of one species from its moments: T_par (z), T_perp
// (per degree of freedom of r, phi), and the mean velocity
__device__ __forceinline__ bool species_temps(const double *m, double mass, double &tpar, double &tperp, double V[3]) {
  const double sw = m[1];
  if (!(m[0] >= SURR_MIN_PARTICLES) || !(sw > 0)) return false;
  V[0] = m[2] / sw; V[1] = m[3] / sw; V[2] = m[4] / sw;
  tpar = mass * (m[5] / sw - V[2] * V[2]) / EL_CHARGE;
  tperp = mass * (m[6] / sw - V[0] * V[0] - V[1] * V[1]) / (2.0 * EL_CHARGE);
  return isnormal(tpar) && tpar > 0 && isnormal(tperp) && tperp > 0;
}

// Collision-rate scale of each target (relative changes of Te_par,
// Te_perp, Ti_par, Ti_perp over one pass): the network learns the relative
// change divided by dt times the species' collision frequency up to a
// constant -- electrons n_e / (Te_perp sqrt(Te_par)) (the isotropisation
// rate of a bi-Maxwellian), ions n_i / Ti^1.5 -- so that its outputs stay
// of order one across the density and temperature range.
__device__ __forceinline__ bool surr_rate_scale(const double *me, const double *mi, double m_e, double m_i,
                                                double vol, double dt, double sc[MLP_OUT]) {
  double tep, tet, tip, tit, V[3];
  if (!species_temps(me, m_e, tep, tet, V) || !species_temps(mi, m_i, tip, tit, V)) return false;
  const double t = dt * 1e10;
  const double se = (me[1] / vol) * 1e-20 * t / (tet * sqrt(tep));
  const double ti = (tip + 2.0 * tit) / 3.0;
  const double si = (mi[1] / vol) * 1e-20 * t / (ti * sqrt(ti));
  sc[0] = sc[1] = se;
  sc[2] = sc[3] = si;
  return isnormal(se) && isnormal(si);
}

// features: log10 n_e, log10 n_i, log10 Te_par, log10 Te_perp, log10 Ti,
// log10 dt; normalised by the fitted mean / std when `norm` is given.
// ok[c] = 1 for a cell the network may handle.
__global__ void k_surr_features(Geom g, const double *mom, double m_e, double m_i, SurrNorm norm, int normalise,
                                float *X, int *ok) {
  const long ncells = (long)g.Dr * g.Dz * g.nr * g.nz;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncells; c += (long)gridDim.x * blockDim.x) {
    const double *me = mom + c * SST, *mi = me + 8;
    double tep, tet, tip, tit, Ve[3], Vi[3];
    bool good = species_temps(me, m_e, tep, tet, Ve) && species_temps(mi, m_i, tip, tit, Vi);
    const CellPos q = cell_pos(g, c);
    const double vol = PCP_CELL_VOLUME((double)q.cr, g.dr, g.dz);
    double f[MLP_IN] = {log10(me[1] / vol), log10(mi[1] / vol), log10(tep), log10(tet),
                        log10((tip + 2.0 * tit) / 3.0), log10(g.dt)};
    for (int k = 0; k < MLP_IN; ++k) {
      float x = (float)f[k];
      if (normalise) {
        x = (x - norm.mean[k]) / norm.std[k];
        if (!(fabsf(x) <= SURR_MAX_Z)) good = false;
      }
      X[c * MLP_XSTRIDE + k] = good ? x : 0.f;
    }
    X[c * MLP_XSTRIDE + 6] = 0.f;
    X[c * MLP_XSTRIDE + 7] = 0.f;
    ok[c] = good ? 1 : 0;
  }
}

// training rows of the cells that collided: relative changes of Te_par,
// Te_perp, Ti_par, Ti_perp over the pass, each over its rate scale
// a training row of cell c: valid when the cell collided (not after a row
// break) and its moments are normal before and after the pass
__device__ __forceinline__ bool surr_row(const Geom &g, long c, const double *before, const double *after, double m_e,
                                         double m_i, const int *ok, const int *row_bad, double rel[MLP_OUT]) {
  if (!ok[c]) return false;
  const CellPos q = cell_pos(g, c);
  if (q.j >= row_bad[(long)q.d * g.nr + q.i]) return false;
  double b[4], a[4], V[3], sc[MLP_OUT];
  if (!species_temps(before + c * SST, m_e, b[0], b[1], V) || !species_temps(before + c * SST + 8, m_i, b[2], b[3], V) ||
      !species_temps(after + c * SST, m_e, a[0], a[1], V) || !species_temps(after + c * SST + 8, m_i, a[2], a[3], V))
    return false;
  const double vol = PCP_CELL_VOLUME((double)q.cr, g.dr, g.dz);
  if (!surr_rate_scale(before + c * SST, before + c * SST + 8, m_e, m_i, vol, g.dt, sc)) return false;
  for (int k = 0; k < MLP_OUT; ++k) rel[k] = (a[k] - b[k]) / b[k] / sc[k];
  return true;
}

__global__ void k_surr_rowflag(Geom g, const double *before, const double *after, double m_e, double m_i,
                               const int *ok, const int *row_bad, uint32_t *flag) {
  const long ncells = (long)g.Dr * g.Dz * g.nr * g.nz;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c <= ncells; c += (long)gridDim.x * blockDim.x) {
    double rel[MLP_OUT];
    flag[c] = c < ncells && surr_row(g, c, before, after, m_e, m_i, ok, row_bad, rel) ? 1u : 0u;
  }
}

// training rows of the cells that collided, in cell order from row n0 on:
// relative changes of Te_par, Te_perp, Ti_par, Ti_perp over the pass, each
// over its rate scale
__global__ void k_surr_targets(Geom g, const double *before, const double *after, double m_e, double m_i,
                               const int *ok, const int *row_bad, const float *X, const uint32_t *offset, long n0,
                               float *DX, float *DT, long cap) {
  const long ncells = (long)g.Dr * g.Dz * g.nr * g.nz;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncells; c += (long)gridDim.x * blockDim.x) {
    double rel[MLP_OUT];
    if (!surr_row(g, c, before, after, m_e, m_i, ok, row_bad, rel)) continue;
    const long slot = n0 + (long)offset[c];
    if (slot >= cap) continue;
    for (int k = 0; k < MLP_XSTRIDE; ++k) DX[slot * MLP_XSTRIDE + k] = X[c * MLP_XSTRIDE + k];
    for (int k = 0; k < MLP_OUT; ++k) DT[slot * MLP_YSTRIDE + k] = (float)rel[k];
  }
}

// The network's relative temperature changes applied per species as
// rescalings of the thermal velocity about the species' mean velocity (z
// by alpha_par, r and phi by alpha_perp), then one common factor on both
// species' thermal velocities restores the cell's total kinetic energy:
// each species' momentum and the cell's energy are conserved exactly (up to
// rounding).  Cells the network may not handle are flagged for the binary
// collision fallback.
template <class V>
__global__ void __launch_bounds__(COLL_BLOCK) k_surr_apply(Geom g, V ve, V vi, const uint32_t *off_e,
                                                           const uint32_t *off_i, const uint32_t *perm_e,
                                                           const uint32_t *perm_i, const double *mom, double m_e,
                                                           double m_i, const float *Y, SurrNorm norm, const int *ok,
                                                           int *fallback, unsigned long long *n_fallback) {
  __shared__ CellStage S;
  __shared__ double red[4];
  const long ncells = (long)g.Dr * g.Dz * g.nr * g.nz;
  for (long c = blockIdx.x; c < ncells; c += gridDim.x) {
    const int nn[2] = {(int)(off_e[c + 1] - off_e[c]), (int)(off_i[c + 1] - off_i[c])};
    const bool use = ok[c] && nn[0] <= COLL_MAXC && nn[1] <= COLL_MAXC;
    if (threadIdx.x == 0) {
      fallback[c] = use ? 0 : 1;
      if (!use && (nn[0] > 0 || nn[1] > 0)) atomicAdd(n_fallback, 1ull);
    }
    if (!use) continue;
    stage_species(ve, perm_e, off_e[c], nn[0], 0, S);
    stage_species(vi, perm_i, off_i[c], nn[1], 1, S);
    __syncthreads();
    double Vs[2][3], apar[2], aperp[2], sc[MLP_OUT];
    const double mass[2] = {m_e, m_i};
    const CellPos q = cell_pos(g, c);
    // ok[c] guarantees normal moments, hence a normal rate scale
    (void)surr_rate_scale(mom + c * SST, mom + c * SST + 8, m_e, m_i, PCP_CELL_VOLUME((double)q.cr, g.dr, g.dz), g.dt,
                          sc);
    for (int s = 0; s < 2; ++s) {
      const double *m = mom + c * SST + 8 * s;
      for (int k = 0; k < 3; ++k) Vs[s][k] = m[2 + k] / m[1];
      const double ypar = (double)Y[c * MLP_YSTRIDE + 2 * s] * norm.tscale[2 * s] * sc[2 * s];
      const double yperp = (double)Y[c * MLP_YSTRIDE + 2 * s + 1] * norm.tscale[2 * s + 1] * sc[2 * s + 1];
      apar[s] = sqrt(fmax(1.0 + ypar, SURR_MIN_FACTOR));
      aperp[s] = sqrt(fmax(1.0 + yperp, SURR_MIN_FACTOR));
    }
    // thermal energy before and after the per-species rescaling
    double e0 = 0, e1 = 0;
    for (int s = 0; s < 2; ++s)
      for (int k = threadIdx.x; k < nn[s]; k += COLL_BLOCK) {
        const double dx = S.vx[s][k] - Vs[s][0], dy = S.vy[s][k] - Vs[s][1], dz = S.vz[s][k] - Vs[s][2];
        const double wm = S.w[s][k] * mass[s];
        e0 += wm * (dx * dx + dy * dy + dz * dz);
        const double nx = aperp[s] * dx, ny = aperp[s] * dy, nz = apar[s] * dz;
        e1 += wm * (nx * nx + ny * ny + nz * nz);
      }
    e0 = wave_sum(e0);
    e1 = wave_sum(e1);
    if (threadIdx.x == 0) red[0] = e1 > 0 ? sqrt(e0 / e1) : 1.0;
    __syncthreads();
    const double beta = red[0];
    for (int s = 0; s < 2; ++s)
      for (int k = threadIdx.x; k < nn[s]; k += COLL_BLOCK) {
        double v3[3];
        v3[0] = Vs[s][0] + beta * (aperp[s] * (S.vx[s][k] - Vs[s][0]));
        v3[1] = Vs[s][1] + beta * (aperp[s] * (S.vy[s][k] - Vs[s][1]));
        v3[2] = Vs[s][2] + beta * (apar[s] * (S.vz[s][k] - Vs[s][2]));
        if (s == 0) ve.store(S.idx[0][k], v3);
        else vi.store(S.idx[1][k], v3);
      }
    __syncthreads();
  }
}

__global__ void k_fill_zero_ull(unsigned long long *p) { *p = 0ull; }

// ---------------------------------------------------------------------------
// Fused surrogate phase of an FP32 step.  The push kernel (k32_push_mom)
// leaves each global cell's moments of the pushed velocities in mom; the
// network runs on the features of every cell; k_fsurr_params turns its
// outputs into per-cell rescalings that the move kernel applies to each
// particle on the fly (no buckets, no staging).  The rescaling is the one of
// k_surr_apply, with the energy-restoring factor beta computed from the
// moments: for species s with thermal sums P_perp = sum w (v_r^2 + v_phi^2)
// - |sum w v_perp|^2 / sum w and P_par likewise,
//   beta^2 = sum_s m_s (P_perp + P_par) / sum_s m_s (a_perp^2 P_perp + a_par^2 P_par).
// Cells the network does not cover keep their velocities here and are
// flagged (by local cell key) for the P12 fallback.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void global_cell(const Geom &g, long c, long &cr, long &cz) {
  cr = (long)g.div_Nz.div((uint32_t)c);
  cz = c - cr * g.Nz;
}

__global__ void k_fsurr_features(Geom g, const double *mom, double m_e, double m_i, SurrNorm norm, float *X,
                                 int *ok) {
  const long ncells = g.Nr * g.Nz;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncells; c += (long)gridDim.x * blockDim.x) {
    const double *me = mom + c * SURR_PAR_STRIDE, *mi = me + 8;
    double tep, tet, tip, tit, Ve[3], Vi[3];
    bool good = species_temps(me, m_e, tep, tet, Ve) && species_temps(mi, m_i, tip, tit, Vi);
    long cr, cz;
    global_cell(g, c, cr, cz);
    const double vol = PCP_CELL_VOLUME((double)cr, g.dr, g.dz);
    const double f[MLP_IN] = {log10(me[1] / vol), log10(mi[1] / vol), log10(tep), log10(tet),
                              log10((tip + 2.0 * tit) / 3.0), log10(g.dt)};
    for (int k = 0; k < MLP_IN; ++k) {
      float x = ((float)f[k] - norm.mean[k]) / norm.std[k];
      if (!(fabsf(x) <= SURR_MAX_Z)) good = false;
      X[c * MLP_XSTRIDE + k] = good ? x : 0.f;
    }
    X[c * MLP_XSTRIDE + 6] = 0.f;
    X[c * MLP_XSTRIDE + 7] = 0.f;
    ok[c] = good ? 1 : 0;
  }
}

// also writes the P12 fallback's bucket counts (local cell keys) from the
// moments' particle counts: the particles are still in the cells the push
// counted them in
__global__ void k_fsurr_params(Geom g, double *mom, double m_e, double m_i, const float *Y, SurrNorm norm,
                               const int *ok, float *par, int *fallback, unsigned long long *n_fallback,
                               uint32_t *cnt_e, uint32_t *cnt_i) {
  const long ncells = g.Nr * g.Nz;
  if (blockIdx.x == 0 && threadIdx.x == 0) cnt_e[ncells] = cnt_i[ncells] = 0;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncells; c += (long)gridDim.x * blockDim.x) {
    double *m = mom + c * SURR_PAR_STRIDE;
    float *P = par + c * SURR_PAR_STRIDE;
    long cr, cz;
    global_cell(g, c, cr, cz);
    const uint32_t lk = local_cell_key(g, (int)cr, (int)cz);
    if (ok[c]) {
      double sc[MLP_OUT];
      (void)surr_rate_scale(m, m + 8, m_e, m_i, PCP_CELL_VOLUME((double)cr, g.dr, g.dz), g.dt, sc);
      const double mass[2] = {m_e, m_i};
      double V[2][3], ap[2], az[2], pp[2], pz[2];
      double e0 = 0, e1 = 0;
      for (int s = 0; s < 2; ++s) {
        const double *q = m + 8 * s;
        for (int k = 0; k < 3; ++k) V[s][k] = q[2 + k] / q[1];
        const double ypar = (double)Y[c * MLP_YSTRIDE + 2 * s] * norm.tscale[2 * s] * sc[2 * s];
        const double yperp = (double)Y[c * MLP_YSTRIDE + 2 * s + 1] * norm.tscale[2 * s + 1] * sc[2 * s + 1];
        az[s] = sqrt(fmax(1.0 + ypar, SURR_MIN_FACTOR));
        ap[s] = sqrt(fmax(1.0 + yperp, SURR_MIN_FACTOR));
        pp[s] = fmax(q[6] - (q[2] * q[2] + q[3] * q[3]) / q[1], 0.0);
        pz[s] = fmax(q[5] - q[4] * q[4] / q[1], 0.0);
        e0 += mass[s] * (pp[s] + pz[s]);
        e1 += mass[s] * (ap[s] * ap[s] * pp[s] + az[s] * az[s] * pz[s]);
      }
      const double beta = e1 > 0 ? sqrt(e0 / e1) : 1.0;
      for (int s = 0; s < 2; ++s) {
        P[8 * s + 0] = (float)V[s][0];
        P[8 * s + 1] = (float)V[s][1];
        P[8 * s + 2] = (float)V[s][2];
        P[8 * s + 3] = (float)(beta * ap[s]);
        P[8 * s + 4] = (float)(beta * az[s]);
      }
      fallback[lk] = 0;
      cnt_e[lk] = cnt_i[lk] = 0;
    } else {
      for (int s = 0; s < 2; ++s) {
        P[8 * s + 0] = P[8 * s + 1] = P[8 * s + 2] = 0.f;
        P[8 * s + 3] = P[8 * s + 4] = 1.f;
      }
      const bool any = m[0] > 0 || m[8] > 0;
      fallback[lk] = any ? 1 : 0;
      cnt_e[lk] = any ? (uint32_t)m[0] : 0u;
      cnt_i[lk] = any ? (uint32_t)m[8] : 0u;
    }
    // fallback cells counted with one atomic per wavefront
    const bool fb = !ok[c] && (m[0] > 0 || m[8] > 0);
    const unsigned long long bal = __ballot(fb);
    if (bal && __lane_id() == __ffsll((long long)__ballot(1)) - 1) atomicAdd(n_fallback, (unsigned long long)__popcll(bal));
    // the next step's push accumulates into zeroed moments
    for (int k = 0; k < SURR_PAR_STRIDE; ++k) m[k] = 0.0;
  }
}

__global__ void k_fill_zero_f64(double *p, long n) {
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) p[t] = 0.0;
}

}  // namespace

struct CollBuffers {
  uint32_t *cnt[2] = {nullptr, nullptr}, *off[2] = {nullptr, nullptr};
  uint32_t *fill[2] = {nullptr, nullptr}, *perm[2] = {nullptr, nullptr};
  uint32_t *lists = nullptr, *lcount = nullptr;   // cells per size class
  uint32_t *crowd_off = nullptr;                  // crowded cells: range of each listed cell
  uint64_t *crowd_key = nullptr;                  // shuffle keys, indices and FP64 stage of
  uint32_t *crowd_idx = nullptr;                  // the crowded cells (COLL_CROWD_CAP particles)
  double *crowd_stage = nullptr;
  long cap[2] = {0, 0};
  double *tot = nullptr;
  int *row_bad = nullptr;
  void *scan_tmp = nullptr;
  size_t scan_bytes = 0;
  long ncells = 0;
  // surrogate
  double *mom = nullptr, *mom2 = nullptr;
  float *feat = nullptr, *pred = nullptr;
  int *ok = nullptr, *fallback = nullptr;
  unsigned long long *counter = nullptr;   // [0] fallback cells
  // fused surrogate phase (per global cell)
  double *fmom = nullptr;
  float *fX = nullptr, *fY = nullptr, *fpar = nullptr;
  int *fok = nullptr;
  long fcells = 0;
};

void coll_free(pcp_ctx *c) {
  CollBuffers *b = c->coll;
  if (!b) return;
  for (int s = 0; s < 2; ++s) {
    (void)hipFree(b->cnt[s]); (void)hipFree(b->off[s]); (void)hipFree(b->fill[s]);
    (void)hipFree(b->perm[s]);
  }
  (void)hipFree(b->lists); (void)hipFree(b->lcount);
  (void)hipFree(b->crowd_off); (void)hipFree(b->crowd_key); (void)hipFree(b->crowd_idx); (void)hipFree(b->crowd_stage);
  (void)hipFree(b->tot); (void)hipFree(b->row_bad); (void)hipFree(b->scan_tmp);
  (void)hipFree(b->mom); (void)hipFree(b->mom2); (void)hipFree(b->feat); (void)hipFree(b->pred);
  (void)hipFree(b->ok); (void)hipFree(b->fallback); (void)hipFree(b->counter);
  (void)hipFree(b->fmom); (void)hipFree(b->fX); (void)hipFree(b->fY); (void)hipFree(b->fpar); (void)hipFree(b->fok);
  delete b;
  c->coll = nullptr;
}

static int coll_alloc(pcp_ctx *c, long cap_e, long cap_i) {
  CollBuffers *b = c->coll;
  const long ncells = (long)c->D * c->g.nr * c->g.nz;
  if (b && b->cap[0] >= cap_e && b->cap[1] >= cap_i) return 0;
  coll_free(c);
  b = new CollBuffers();
  c->coll = b;
  b->ncells = ncells;
  const long caps[2] = {std::max(cap_e, 1L), std::max(cap_i, 1L)};
  for (int s = 0; s < 2; ++s) {
    b->cap[s] = caps[s];
    if (hipMalloc(&b->cnt[s], (ncells + 1) * sizeof(uint32_t)) != hipSuccess ||
        hipMalloc(&b->off[s], (ncells + 1) * sizeof(uint32_t)) != hipSuccess ||
        hipMalloc(&b->fill[s], (ncells + 1) * sizeof(uint32_t)) != hipSuccess ||
        hipMalloc(&b->perm[s], caps[s] * sizeof(uint32_t)) != hipSuccess)
      return -1;
  }
  if (hipMalloc(&b->lists, (size_t)COLL_CLASSES * ncells * sizeof(uint32_t)) != hipSuccess ||
      hipMalloc(&b->lcount, (COLL_CLASSES + 1) * sizeof(uint32_t)) != hipSuccess ||
      hipMalloc(&b->crowd_off, COLL_CROWD_CELLS * sizeof(uint32_t)) != hipSuccess ||
      hipMalloc(&b->crowd_key, COLL_CROWD_CAP * sizeof(uint64_t)) != hipSuccess ||
      hipMalloc(&b->crowd_idx, COLL_CROWD_CAP * sizeof(uint32_t)) != hipSuccess ||
      hipMalloc(&b->crowd_stage, 4 * COLL_CROWD_CAP * sizeof(double)) != hipSuccess)
    return -1;
  if (hipMalloc(&b->tot, ncells * TOT * sizeof(double)) != hipSuccess ||
      hipMalloc(&b->row_bad, (long)c->D * c->g.nr * sizeof(int)) != hipSuccess ||
      hipMalloc(&b->mom, ncells * SST * sizeof(double)) != hipSuccess ||
      hipMalloc(&b->mom2, ncells * SST * sizeof(double)) != hipSuccess ||
      hipMalloc(&b->feat, ncells * MLP_XSTRIDE * sizeof(float)) != hipSuccess ||
      hipMalloc(&b->pred, ncells * MLP_YSTRIDE * sizeof(float)) != hipSuccess ||
      hipMalloc(&b->ok, ncells * sizeof(int)) != hipSuccess ||
      hipMalloc(&b->fallback, ncells * sizeof(int)) != hipSuccess ||
      hipMalloc(&b->counter, 2 * sizeof(unsigned long long)) != hipSuccess)
    return -1;
  if (hipMemset(b->counter, 0, 2 * sizeof(unsigned long long)) != hipSuccess) return -1;
  if (hipcub::DeviceScan::ExclusiveSum(nullptr, b->scan_bytes, b->cnt[0], b->off[0], (int)(ncells + 1)) !=
      hipSuccess)
    return -1;
  if (hipMalloc(&b->scan_tmp, std::max<size_t>(b->scan_bytes, 16)) != hipSuccess) return -1;
  return 0;
}

// bucket lists of both species (sort_to_cells)
// `counted`: the bucket counts are already in cnt (the fused surrogate phase
// writes them from the push's per-cell particle counts)
template <class V>
static int coll_buckets(pcp_ctx *c, V ve, V vi, long n_e, long n_i, const int *mask = nullptr,
                        const unsigned long long *gate = nullptr, bool counted = false) {
  CollBuffers *b = c->coll;
  const Geom &g = c->g;
  const long ncells = b->ncells;
  const uint32_t sentinel = (uint32_t)ncells;
  const long nn[2] = {n_e, n_i};
  unsigned gz = (unsigned)std::min<long>((ncells + 256) / 256, (long)c->n_cu * 16);
  for (int s = 0; s < 2; ++s) {
    hipLaunchKernelGGL(k_fill_u32, dim3(gz), dim3(256), 0, c->stream, b->fill[s], ncells + 1);
    unsigned gp = (unsigned)std::max(1L, std::min<long>((nn[s] + 255) / 256, (long)c->n_cu * 16));
    if (!counted) {
      hipLaunchKernelGGL(k_fill_u32, dim3(gz), dim3(256), 0, c->stream, b->cnt[s], ncells + 1);
      if (nn[s] > 0)
        hipLaunchKernelGGL(k_coll_count<V>, dim3(gp), dim3(256), 0, c->stream, g, s == 0 ? ve : vi, b->cnt[s],
                           sentinel, mask, gate);
    }
    size_t bytes = b->scan_bytes;
    if (hipcub::DeviceScan::ExclusiveSum(b->scan_tmp, bytes, b->cnt[s], b->off[s], (int)(ncells + 1), c->stream) !=
        hipSuccess)
      return -1;
    if (nn[s] > 0)
      hipLaunchKernelGGL(k_coll_fill<V>, dim3(gp), dim3(256), 0, c->stream, g, s == 0 ? ve : vi, b->off[s],
                         b->fill[s], b->perm[s], sentinel, mask, gate);
  }
  return 0;
}

// shuffle and statistics of every listed cell: the grouped classes in one
// launch, the crowded cells in another
template <class V>
static void coll_prep(pcp_ctx *c, V ve, V vi, double m_e, double m_i, uint64_t seed, PassNo step,
                      const unsigned long long *gate) {
  CollBuffers *b = c->coll;
  const Geom &g = c->g;
  hipLaunchKernelGGL((k_coll_prep<V>), dim3((unsigned)c->n_cu * 12), dim3(COLL_GROUP_BLOCK), 0, c->stream, g, ve, vi,
                     b->off[0], b->off[1], b->perm[0], b->perm[1], m_e, m_i, seed, step, b->tot, b->lists,
                     b->lcount, b->ncells, gate);
  hipLaunchKernelGGL(k_coll_stats, dim3((unsigned)std::max(1L, std::min<long>((b->ncells + 255) / 256, (long)c->n_cu * 8))),
                     dim3(256), 0, c->stream, g, b->tot, b->row_bad, b->lists, b->lcount, b->ncells, gate);
  hipLaunchKernelGGL((k_coll_prep_crowd<V>), dim3((unsigned)c->n_cu * 2), dim3(COLL_CROWD_BLOCK), 0, c->stream, g, ve,
                     vi, b->off[0], b->off[1], b->perm[0], b->perm[1], m_e, m_i, seed, step, b->tot, b->row_bad,
                     b->lists + (size_t)COLL_GROUP_CLASSES * b->ncells, b->lcount + COLL_GROUP_CLASSES, b->crowd_off,
                     b->crowd_key, b->crowd_idx, b->crowd_stage, gate);
}

template <int SCHEME, class V>
static void coll_pairs(pcp_ctx *c, V ve, V vi, double m_e, double m_i, double q_e, double q_i, uint64_t seed,
                       PassNo step, const unsigned long long *gate) {
  CollBuffers *b = c->coll;
  const Geom &g = c->g;
  hipLaunchKernelGGL((k_coll_pairs<SCHEME, V>), dim3((unsigned)c->n_cu * 8), dim3(COLL_GROUP_BLOCK), 0, c->stream, g,
                     ve, vi, b->off[0], b->off[1], b->perm[0], b->perm[1], m_e, m_i, q_e, q_i, seed, step, b->tot,
                     b->row_bad, b->lists, b->lcount, b->ncells, c->st, gate);
  hipLaunchKernelGGL((k_coll_pairs_crowd<SCHEME, V>), dim3((unsigned)c->n_cu * 2), dim3(COLL_CROWD_BLOCK), 0,
                     c->stream, g, ve, vi, b->off[0], b->off[1], b->perm[0], b->perm[1], m_e, m_i, q_e, q_i, seed,
                     step, b->tot, b->row_bad, b->lists + (size_t)COLL_GROUP_CLASSES * b->ncells,
                     b->lcount + COLL_GROUP_CLASSES, b->crowd_off, b->crowd_stage, c->st, gate);
}

// the binary pass on the cells of `mask` (all cells when null): cells
// classified by size, then shuffle + statistics of every cell (the row
// breaks are final only after all of them), then the pairs
template <class V>
static void coll_binary(pcp_ctx *c, int scheme, V ve, V vi, double m_e, double m_i, double q_e, double q_i,
                        uint64_t seed, PassNo step, const int *mask, const unsigned long long *gate = nullptr) {
  CollBuffers *b = c->coll;
  const Geom &g = c->g;
  const long ncells = b->ncells;
  const long rows = (long)c->D * g.nr;
  hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)std::max<long>(1, std::min<long>((rows + 255) / 256, 1024))),
                     dim3(256), 0, c->stream, b->row_bad, rows, INT_MAX);
  hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, c->stream, b->lcount, (long)COLL_CLASSES + 1);
  const unsigned gz = (unsigned)std::max(1L, std::min<long>((ncells + 255) / 256, (long)c->n_cu * 16));
  hipLaunchKernelGGL(k_coll_classify, dim3(gz), dim3(256), 0, c->stream, g, b->off[0], b->off[1], mask, b->lists,
                     b->lcount, b->crowd_off, b->row_bad, c->st, gate);
  coll_prep(c, ve, vi, m_e, m_i, seed, step, gate);
  if (scheme == COLL_TA77S) coll_pairs<COLL_TA77S>(c, ve, vi, m_e, m_i, q_e, q_i, seed, step, gate);
  else if (scheme == COLL_SK98) coll_pairs<COLL_SK98>(c, ve, vi, m_e, m_i, q_e, q_i, seed, step, gate);
  else coll_pairs<COLL_P12>(c, ve, vi, m_e, m_i, q_e, q_i, seed, step, gate);
}

template <class V>
static void surr_moments(pcp_ctx *c, V ve, V vi, double *mom) {
  CollBuffers *b = c->coll;
  unsigned gc = (unsigned)std::min<long>(b->ncells, (long)c->n_cu * 32);
  hipLaunchKernelGGL(k_surr_moments<V>, dim3(gc), dim3(COLL_BLOCK), 0, c->stream, c->g, ve, vi, b->off[0], b->off[1],
                     b->perm[0], b->perm[1], mom);
}

static SurrNorm surr_norm(const pcp_ctx *c) {
  SurrNorm nm;
  const MlpState *m = c->mlp;
  for (int k = 0; k < MLP_IN; ++k) {
    nm.mean[k] = m ? m->feat_mean[k] : 0.f;
    nm.std[k] = m ? m->feat_std[k] : 1.f;
  }
  for (int k = 0; k < MLP_OUT; ++k) nm.tscale[k] = m ? m->targ_scale[k] : 1.f;
  return nm;
}

template <class V>
static int coll_run(pcp_ctx *c, int scheme, V ve, V vi, long n_e, long n_i, double m_e, double m_i, double q_e,
                    double q_i, uint64_t seed, PassNo step) {
  CollBuffers *b = c->coll;
  if (coll_buckets(c, ve, vi, n_e, n_i) < 0) return -1;
  if (scheme != COLL_SURROGATE) {
    coll_binary(c, scheme, ve, vi, m_e, m_i, q_e, q_i, seed, step, nullptr);
    return 0;
  }
  // network on the cells it covers, P12 on the others
  if (!c->mlp || !c->mlp->trained) return -2;
  const long ncells = b->ncells;
  unsigned gc = (unsigned)std::min<long>(ncells, (long)c->n_cu * 32);
  unsigned gt = (unsigned)std::min<long>((ncells + 255) / 256, (long)c->n_cu * 16);
  surr_moments(c, ve, vi, b->mom);
  hipLaunchKernelGGL(k_surr_features, dim3(gt), dim3(256), 0, c->stream, c->g, b->mom, m_e, m_i, surr_norm(c), 1,
                     b->feat, b->ok);
  mlp_forward(c, b->feat, ncells, b->pred);
  hipLaunchKernelGGL(k_fill_zero_ull, dim3(1), dim3(1), 0, c->stream, b->counter);
  hipLaunchKernelGGL(k_surr_apply<V>, dim3(gc), dim3(COLL_BLOCK), 0, c->stream, c->g, ve, vi, b->off[0], b->off[1],
                     b->perm[0], b->perm[1], b->mom, m_e, m_i, b->pred, surr_norm(c), b->ok, b->fallback,
                     b->counter);
  coll_binary(c, COLL_P12, ve, vi, m_e, m_i, q_e, q_i, seed, step, b->fallback);
  return 0;
}

// one P12 pass that also appends (features, relative temperature changes)
// rows of the cells it collided to the network's training set
template <class V>
static int coll_collect(pcp_ctx *c, V ve, V vi, long n_e, long n_i, double m_e, double m_i, double q_e, double q_i,
                        uint64_t seed, PassNo step) {
  CollBuffers *b = c->coll;
  MlpState *m = c->mlp;
  if (coll_buckets(c, ve, vi, n_e, n_i) < 0) return -1;
  const long ncells = b->ncells;
  unsigned gt = (unsigned)std::min<long>((ncells + 255) / 256, (long)c->n_cu * 16);
  surr_moments(c, ve, vi, b->mom);
  hipLaunchKernelGGL(k_surr_features, dim3(gt), dim3(256), 0, c->stream, c->g, b->mom, m_e, m_i, surr_norm(c), 0,
                     b->feat, b->ok);
  coll_binary(c, COLL_P12, ve, vi, m_e, m_i, q_e, q_i, seed, step, nullptr);
  surr_moments(c, ve, vi, b->mom2);
  // rows in cell order (the bucket arrays of species 0 are free again):
  // flags, their exclusive sum, then the rows at their offsets
  const long n0 = m->n;
  unsigned gf = (unsigned)std::min<long>((ncells + 256) / 256, (long)c->n_cu * 16);
  hipLaunchKernelGGL(k_surr_rowflag, dim3(gf), dim3(256), 0, c->stream, c->g, b->mom, b->mom2, m_e, m_i, b->ok,
                     b->row_bad, b->cnt[0]);
  size_t bytes = b->scan_bytes;
  if (hipcub::DeviceScan::ExclusiveSum(b->scan_tmp, bytes, b->cnt[0], b->off[0], (int)(ncells + 1), c->stream) !=
      hipSuccess)
    return -1;
  hipLaunchKernelGGL(k_surr_targets, dim3(gt), dim3(256), 0, c->stream, c->g, b->mom, b->mom2, m_e, m_i, b->ok,
                     b->row_bad, b->feat, b->off[0], n0, m->X, m->T, m->cap);
  uint32_t rows = 0;
  if (hipMemcpyAsync(&rows, b->off[0] + ncells, sizeof rows, hipMemcpyDeviceToHost, c->stream) != hipSuccess)
    return -1;
  if (hipStreamSynchronize(c->stream) != hipSuccess) return -1;
  m->n = std::min<long>(n0 + (long)rows, m->cap);
  return 0;
}

int coll_prepare(pcp_ctx *c, int se, int si) {
  if (c->s32) return coll_alloc(c, c->s32->sp[se].cap, c->s32->sp[si].cap);
  return coll_alloc(c, c->sp[se].cap, c->sp[si].cap);
}

int launch_collide(pcp_ctx *c, int scheme, int se, int si, uint64_t seed, PassNo step, int vslot) {
  if (c->s32) {
    Species32 &e = c->s32->sp[se], &i = c->s32->sp[si];
    if (coll_alloc(c, e.cap, i.cap) < 0) return -1;
    View32 ve{e, c->cur, vslot}, vi{i, c->cur, vslot};
    return coll_run(c, scheme, ve, vi, e.n, i.n, e.m, i.m, e.q, i.q, seed, step);
  }
  SpeciesDev &e = c->sp[se], &i = c->sp[si];
  if (coll_alloc(c, e.cap, i.cap) < 0) return -1;
  View64 ve{e, c->cur}, vi{i, c->cur};
  return coll_run(c, scheme, ve, vi, e.n, i.n, e.m, i.m, e.q, i.q, seed, step);
}

int fsurr_prepare(pcp_ctx *c, int se, int si) {
  if (!c->s32) return -1;
  if (coll_alloc(c, c->s32->sp[se].cap, c->s32->sp[si].cap) < 0) return -1;
  CollBuffers *b = c->coll;
  const long nc = c->g.Nr * c->g.Nz;
  if (b->fcells == nc) return 0;
  if (hipMalloc(&b->fmom, nc * SURR_PAR_STRIDE * sizeof(double)) != hipSuccess ||
      hipMalloc(&b->fX, nc * MLP_XSTRIDE * sizeof(float)) != hipSuccess ||
      hipMalloc(&b->fY, nc * MLP_YSTRIDE * sizeof(float)) != hipSuccess ||
      hipMalloc(&b->fpar, nc * SURR_PAR_STRIDE * sizeof(float)) != hipSuccess ||
      hipMalloc(&b->fok, nc * sizeof(int)) != hipSuccess)
    return -1;
  unsigned gz = (unsigned)std::min<long>((nc * SURR_PAR_STRIDE + 255) / 256, (long)c->n_cu * 16);
  hipLaunchKernelGGL(k_fill_zero_f64, dim3(gz), dim3(256), 0, c->stream, b->fmom, nc * SURR_PAR_STRIDE);
  b->fcells = nc;
  return 0;
}

double *fsurr_mom(pcp_ctx *c) { return c->coll ? c->coll->fmom : nullptr; }
const float *fsurr_par(pcp_ctx *c) { return c->coll ? c->coll->fpar : nullptr; }

int fsurr_cells(pcp_ctx *c, int se, int si, uint64_t seed, PassNo step) {
  CollBuffers *b = c->coll;
  if (!b || !b->fmom || !c->mlp || !c->mlp->trained) return -2;
  Species32 &e = c->s32->sp[se], &i = c->s32->sp[si];
  const long nc = b->fcells;
  const unsigned gt = (unsigned)std::min<long>((nc + 255) / 256, (long)c->n_cu * 16);
  hipLaunchKernelGGL(k_fsurr_features, dim3(gt), dim3(256), 0, c->stream, c->g, b->fmom, e.m, i.m, surr_norm(c),
                     b->fX, b->fok);
  mlp_forward(c, b->fX, nc, b->fY);
  hipLaunchKernelGGL(k_fill_zero_ull, dim3(1), dim3(1), 0, c->stream, b->counter);
  hipLaunchKernelGGL(k_fsurr_params, dim3(gt), dim3(256), 0, c->stream, c->g, b->fmom, e.m, i.m, b->fY,
                     surr_norm(c), b->fok, b->fpar, b->fallback, b->counter, b->cnt[0], b->cnt[1]);
  // P12 on the cells the network does not cover, on the pushed velocities
  // (every kernel returns at once while no cell is flagged)
  View32 ve{e, c->cur, c->cur ^ 1}, vi{i, c->cur, c->cur ^ 1};
  if (coll_buckets(c, ve, vi, e.n, i.n, b->fallback, b->counter, true) < 0) return -1;
  coll_binary(c, COLL_P12, ve, vi, e.m, i.m, e.q, i.q, seed, step, b->fallback, b->counter);
  return 0;
}

int surrogate_collect(pcp_ctx *c, int se, int si, uint64_t seed, uint64_t pass) {
  const PassNo step{nullptr, pass};
  if (c->s32) {
    Species32 &e = c->s32->sp[se], &i = c->s32->sp[si];
    if (coll_alloc(c, e.cap, i.cap) < 0) return -1;
    View32 ve{e, c->cur, c->cur}, vi{i, c->cur, c->cur};
    return coll_collect(c, ve, vi, e.n, i.n, e.m, i.m, e.q, i.q, seed, step);
  }
  SpeciesDev &e = c->sp[se], &i = c->sp[si];
  if (coll_alloc(c, e.cap, i.cap) < 0) return -1;
  View64 ve{e, c->cur}, vi{i, c->cur};
  return coll_collect(c, ve, vi, e.n, i.n, e.m, i.m, e.q, i.q, seed, step);
}

long surrogate_fallback_cells(pcp_ctx *c) {
  if (!c->coll) return 0;
  unsigned long long n = 0;
  if (hipMemcpy(&n, c->coll->counter, sizeof n, hipMemcpyDeviceToHost) != hipSuccess) return -1;
  return (long)n;
}

}  // namespace pcp
