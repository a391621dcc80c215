// gfx950 kernels of the GEMS force-evaluation hot path.
//
// Data layout (HBM, cell-sorted order after each rebuild):
//   pos    double4[ncap]   x, y, z, w unused             32 B/atom
//   vel, acc, frc          3 x double[ncap] (SoA)         24 B/atom each
//   epa, rho, eband        double[ncap]
//   eband32                float[ncap] (mixed precision: 1/sqrt(rho) - e0)
//   type, orig, cellof     int[ncap]
//   list   uint32[ncap][cap]: the row of an atom is contiguous (a wavefront
//          reads one row).  entry = j | (image code << 27); image code w = (wx+1)+3(wy+1)+9(wz+1)
//          with the neighbour's periodic image at x_j + wd*L_d.
// Wavefronts are 64 lanes; per-atom kernels use 256-thread workgroups.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "gh_device.h"


namespace {
using namespace ghd;


__global__ void k_fill_int(int *__restrict__ p, int v, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---------------------------------------------------------------------------
// Rebuild decision (test_update, Neighbour.F90:1305-1346).  The reference
// rebuilds when the two largest displacements since the last build sum past
// the skin.  Here the displacement is the true (minimum-image) one, and the
// test uses 2*max, which bounds d1+d2 from above.  Integrators fold each
// workgroup's max |x - x_old|^2 into GhStatus::maxdisp2 with at most one
// atomicMax (non-negative doubles order as their bit patterns); it runs over
// the steps since the last build and the first kernel of a rebuild sequence
// reads it (rebuild_due, rebuild_book).  State-changing kernels return at
// once while GhStatus::halt is set (raise_halt).
// ---------------------------------------------------------------------------
// The O(N^2) list mode tests the rule in its first kernel of a step (every
// workgroup the same words, which that kernel does not change except for the
// next step's displacement maximum) and books it in the second (n2_decide,
// n2_book); k_n2_book where no second kernel follows.
// One decision per workgroup (a stop raised meanwhile must not divide it); all
// threads call it, it ends with a barrier.
__device__ __forceinline__ bool n2_decide(GhStatus *st, double skin, long long step) {
  __shared__ int sdue;
  if (threadIdx.x == 0) {
    const bool due = !halted(st) && rebuild_due(st, skin, step);
    if (blockIdx.x == 0) {
      st->rebuild = due;
      if (due) disp2_clear(st, step + 1);
    }
    sdue = due;
  }
  __syncthreads();
  return sdue != 0;
}
__device__ __forceinline__ void n2_book(GhStatus *st, long long step) {  // one thread
  if (!st->rebuild) return;
  st->rebuild = 0;
  st->nupd += 1;
  st->force_rebuild = 0;
  // (a build whose rows are all empty has left the tag of an earlier one)
  st->maxnn = (st->maxnn_tag >> 32) == (unsigned long long)st->nupd ? (int)(unsigned)st->maxnn_tag : 0;
  disp2_clear(st, step);
}
__global__ void k_n2_book(GhStatus *st, long long step) { n2_book(st, step); }

struct GridArgs {
  int nc[3], gn[3], gofs[3], pbc[3];
  double L[3], one_cell[3];
  int ncell;
  int ghost;
};



// ---------------------------------------------------------------------------
// Rows of atom numbers: the O(N^2) list mode (free clusters, boxes of a few
// cells, masked pairs; FP64 and mixed) and smaller FP64 boxes in cell mode
// (gh_rows_path).  Row of atom i at i * cap, entry = j | image code << 27; the
// passes gather neighbours from global memory (such systems' positions sit in
// the caches) with G lanes per atom:
//  - 64 in the O(N^2) mode, whose systems hold tens to a few thousand atoms:
//    with one lane per atom a 201-atom cluster ran on four wavefronts whose
//    lanes walked ~200 candidates or ~50 neighbours one dependent load after
//    another; now a row is one load and one round of pair terms.  201 Ag-Cu
//    atoms, FP64: build 45 -> 5.1 us, density 32 -> 4.2, forces 41 -> 4.5.
//  - 16 in cell mode.  The tiled passes spend most of a small system's time on
//    each brick's halo (tables, barriers, three rounds of staging) and leave
//    compute units without a brick: Au 32,000 atoms density 14.3 -> 9.4 us,
//    fused forces 18.8 -> 13.0.  Rows are the tiled build's,
//    entry for entry, and lane l sums entries l, l + 16, ..., as lane l / 4 of
//    the tiled passes does in its accumulator l % 4, so both give the same
//    bits.
// ---------------------------------------------------------------------------
struct N2Build {
  const double4 *pos;
  int n, cap, ncap;
  GridArgs g;
  double rl2;
  int *nn;
  unsigned *list;
  double *xold;
  const int *orig, *mfeel, *mfelt;
};

// List build (verlet_self, Neighbour.F90:676-759): rd > rl^2 -> skip, so
// equality is kept.  Minimum image by rounding as vdistance does; or, with
// ghost images (box mic F), every first-shell image x_j + w L, w in {-1,0,1}
// on each periodic axis, of every atom j including i itself (not w = 0), as
// the reference's ghost atoms are (pbcghost / pbcfullghost,
// Neighbour.F90:1520-1794).  Positions are wrapped into [0, L) just before a
// ghost-image build, as do_pbc does before the reference creates its ghosts,
// so the window is the reference's: it holds every image within the cut when
// each periodic side is at least the cut plus skin.  With pair masks (a
// one-sided `feels` interaction: a cross group with half and newton off,
// Interaction.f90:69-77, 128-131) atom i lists j only when
// mfeel[i] & mfelt[j] is nonzero; i then takes the whole pair force and half
// the pair energy, j no reaction.
// A wavefront builds the rows of R consecutive atoms from s0 (uniform): its
// lanes take 64 consecutive candidates (of (j, image) pairs with ghost
// images), the ballot of the test gives each kept one its place, so a row is
// in candidate order.  Returns the longest row asked for (uniform).
template <int R>
__device__ __forceinline__ int n2_rows(const N2Build &B, int s0) {
  const GridArgs &g = B.g;
  const int lane = threadIdx.x & 63, n = B.n, cap = B.cap;
  if (s0 >= n) return 0;
  double4 pi[R];
  int m[R], fi[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int s = min(s0 + r, n - 1);
    pi[r] = B.pos[s];
    m[r] = 0;
    fi[r] = B.mfeel ? B.mfeel[B.orig[s]] : -1;
  }
  auto put = [&](int r, bool keep, unsigned e) {
    const unsigned long long k = __ballot(keep);
    const int d = m[r] + lane_rank(k);
    if (keep && d < cap) B.list[(size_t)(s0 + r) * cap + d] = e;
    m[r] += __popcll(k);
  };
  if (g.ghost) {
    const long long nw = 27ll * n;
    for (long long t0 = 0; t0 < nw; t0 += 64) {
      const long long t = min(t0 + lane, nw - 1);
      const int j = (int)(t / 27), w = (int)(t - 27ll * j);
      const int wx = w % 3 - 1, wy = (w / 3) % 3 - 1, wz = w / 9 - 1;
      const bool live = t0 + lane < nw && !((wx && !g.pbc[0]) || (wy && !g.pbc[1]) || (wz && !g.pbc[2]));
      const int fj = B.mfelt ? B.mfelt[B.orig[j]] : -1;
      const double4 pj = B.pos[j];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double ux = pj.x - pi[r].x, uy = pj.y - pi[r].y, uz = pj.z - pi[r].z;
        const double rd = dist2_rn(ux + wx * g.L[0], uy + wy * g.L[1], uz + wz * g.L[2]);
        put(r, live && s0 + r < n && (fi[r] & fj) && !(j == s0 + r && w == 13) && rd <= B.rl2,
            (unsigned)j | ((unsigned)w << 27));
      }
    }
  } else {
    const bool wrap = g.pbc[0] || g.pbc[1] || g.pbc[2];
    const double ob0 = 1.0 / g.L[0], ob1 = 1.0 / g.L[1], ob2 = 1.0 / g.L[2];
    for (int j0 = 0; j0 < n; j0 += 64) {
      const int j = min(j0 + lane, n - 1);
      const int fj = B.mfelt ? B.mfelt[B.orig[j]] : -1;
      const double4 pj = B.pos[j];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        double vx = pj.x - pi[r].x, vy = pj.y - pi[r].y, vz = pj.z - pi[r].z;
        int wx = 0, wy = 0, wz = 0;
        if (wrap) {
          if (g.pbc[0]) { wx = -(int)round(vx * ob0); vx = vx + wx * g.L[0]; }
          if (g.pbc[1]) { wy = -(int)round(vy * ob1); vy = vy + wy * g.L[1]; }
          if (g.pbc[2]) { wz = -(int)round(vz * ob2); vz = vz + wz * g.L[2]; }
        }
        const double rd = dist2_rn(vx, vy, vz);
        put(r, j0 + lane < n && j != s0 + r && s0 + r < n && (fi[r] & fj) && rd <= B.rl2,
            (unsigned)j | ((unsigned)((wx + 1) + 3 * (wy + 1) + 9 * (wz + 1)) << 27));
      }
    }
  }
  int most = 0;
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (s0 + r < n) {
      most = max(most, m[r]);
      if (lane == 0) B.nn[s0 + r] = min(m[r], cap);
      if (lane < 3)
        B.xold[lane * B.ncap + s0 + r] = lane == 0 ? pi[r].x : lane == 1 ? pi[r].y : pi[r].z;
    }
  return most;
}

// The wavefront's first atom: R per wavefront.
template <int R>
__device__ __forceinline__ int n2_first() {
  const int w = (int)(blockIdx.x * (GH_BLOCK / 64) + (threadIdx.x >> 6));
  return __builtin_amdgcn_readfirstlane(w) * R;
}

// The workgroup's longest row: the status word of the build, and an overflow.
__device__ __forceinline__ void n2_rows_max(int m, GhStatus *st, int cap, long long step) {
  __shared__ int part[GH_BLOCK / 64];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < GH_BLOCK / 64; ++w) m = max(m, part[w]);
    if (m > 0) atomicMax(&st->maxnn_tag, ((unsigned long long)(st->nupd + 1) << 32) | (unsigned)m);
    if (m > cap) {
      st->overflow = 1;
      if (cap > 0) raise_halt(st, GH_HALT_OVERFLOW, step);  // cap 0: the sizing count
    }
  }
}

template <int R>
__global__ __launch_bounds__(GH_BLOCK) void k_build_n2(GhStatus *st, N2Build B, double skin,
                                                       long long step) {
  if (!n2_decide(st, skin, step)) return;
  n2_rows_max(n2_rows<R>(B, n2_first<R>()), st, B.cap, step);
}

// Image shift table in LDS: shift[w] = (wx*L0, wy*L1, wz*L2).
struct ShiftLds {
  double x[27], y[27], z[27];
};
__device__ __forceinline__ void load_shift(ShiftLds &sh, double L0, double L1, double L2) {
  if (threadIdx.x < 27) {
    int w = threadIdx.x;
    sh.x[w] = (w % 3 - 1) * L0;
    sh.y[w] = ((w / 3) % 3 - 1) * L1;
    sh.z[w] = (w / 9 - 1) * L2;
  }
}

// A pair pass over one row, G lanes per atom: f(j, pj, vx, vy, vz) for every
// listed pair, 64 entries a round; the first round's entries are loaded
// before the row's length is known.
// (The passes skip pairs beyond the cut, so that a distance that is not a
// number reaches the sums.)
template <int G>
struct Row {
  static constexpr int U = 64 / G;  // entries of a lane in a round
  const unsigned *list;
  int m;
  unsigned e[U];
};
template <int G>
__device__ __forceinline__ Row<G> row_head(const unsigned *list, const int *nn, int cap, int i,
                                           bool on) {
  Row<G> r;
  r.list = list + (size_t)i * cap;
  r.m = on ? nn[i] : 0;
#pragma unroll
  for (int u = 0; u < r.U; ++u) r.e[u] = r.list[min((int)(threadIdx.x & (G - 1)) + u * G, cap - 1)];
  return r;
}
template <int G, class F>
__device__ __forceinline__ void row_each(Row<G> &r, const double4 *pos, const double4 &pi,
                                         const ShiftLds &sh, F &&f) {
  const int sub = threadIdx.x & (G - 1);
  for (int k0 = 0; k0 < r.m; k0 += 64) {
    double4 p[Row<G>::U];
#pragma unroll
    for (int u = 0; u < r.U; ++u) {
      const int k = k0 + sub + u * G;
      if (k0 > 0 && k < r.m) r.e[u] = r.list[k];
      if (k < r.m) p[u] = pos[r.e[u] & GH_JMASK];
    }
#pragma unroll
    for (int u = 0; u < r.U; ++u)
      if (k0 + sub + u * G < r.m) {
        const int w = (int)(r.e[u] >> 27);
        f((int)(r.e[u] & GH_JMASK), p[u], (p[u].x + sh.x[w]) - pi.x, (p[u].y + sh.y[w]) - pi.y,
          (p[u].z + sh.z[w]) - pi.z);
      }
  }
}
template <int G>
__device__ __forceinline__ double lanes_total(double v) {
  return G == 64 ? wave_total(v) : row_total(v);
}

// ---------------------------------------------------------------------------
// Integrators.  Per-type masses come in the kernel argument block.
// ---------------------------------------------------------------------------
struct MassArgs {
  double om[GH_MAXT];   // 1/m
  double osm[GH_MAXT];  // sqrt(1/m)
};

struct WrapArgs {
  int pbc[3];
  double L[3];
};

// Positions are not wrapped between neighbour rebuilds: the list stores each
// pair's periodic image, which stays valid while atoms move continuously.
// They are wrapped into the box at every rebuild (k_wrap_rebuild) and when
// copied out, which reproduces do_pbc_1 (Set_Properties.f90:444-470).
// Workgroup maximum of |x - x_old|^2 folded into the device-wide maximum (at
// most one atomicMax, no fence: the next kernel reads it).
template <bool STABLE = true>
__device__ __forceinline__ void disp_reduce(double d2, GhStatus *st, long long step) {
  __shared__ double part[GH_BLOCK / 64];
  d2 = wave_max(d2);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = d2;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < GH_BLOCK / 64; ++w) d2 = fmax(d2, part[w]);
    fold_disp2<STABLE>(st, d2, step);
  }
}

// velocity_verlet_a (Integration.F90:1150-1169) + do_pbc + displacement.
__global__ __launch_bounds__(GH_BLOCK) void k_vv_a(
    int n, int ncap, double dt, MassArgs ma,
    const int *__restrict__ type, double4 *__restrict__ pos, double *__restrict__ vel,
    double *__restrict__ acc, const double *__restrict__ frc, const double *__restrict__ xold,
    GhStatus *st, long long step) {
  if (halted(st)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double d2 = 0.0;
  if (i < n) {
    const double acel_dv = dt * 0.5, acel_dx = acel_dv * dt;
    const double om = ma.om[type[i]];
    double4 p = pos[i];
    double x[3] = {p.x, p.y, p.z};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double a = frc[d * ncap + i] * om;
      const double v = vel[d * ncap + i];
      x[d] = x[d] + dt * v + acel_dx * a;
      vel[d * ncap + i] = v + acel_dv * a;
      acc[d * ncap + i] = a;
      const double dd = x[d] - xold[d * ncap + i];
      d2 += dd * dd;
    }
    p.x = x[0];
    p.y = x[1];
    p.z = x[2];
    pos[i] = p;
  }
  disp_reduce(d2, st, step);
}

// velocity_verlet_b (Integration.F90:1171-1186).
__global__ __launch_bounds__(GH_BLOCK) void k_vv_b(int n, int ncap, double dt, MassArgs ma,
                                                   const int *__restrict__ type,
                                                   double *__restrict__ vel,
                                                   double *__restrict__ acc,
                                                   const double *__restrict__ frc,
                                                   const GhStatus *st) {
  if (halted(st)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double acel_dv = dt * 0.5;
  const double om = ma.om[type[i]];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double a = frc[d * ncap + i] * om;
    acc[d * ncap + i] = a;
    vel[d * ncap + i] = vel[d * ncap + i] + acel_dv * a;
  }
}

__device__ __forceinline__ void ermak_gauss(const ErmakArgs &k, int id,
                                            const double *__restrict__ gauss, int ncap,
                                            double g[6]) {
  if (k.philox) {
    philox_normals(k.seed, k.step, id, g);
  } else {
#pragma unroll
    for (int q = 0; q < 6; ++q) g[q] = gauss[(size_t)q * ncap + id];
  }
}

// ermak_a (Integration.F90:963-1011) + do_pbc + displacement.
__global__ __launch_bounds__(GH_BLOCK) void k_ermak_a(
    int n, int ncap, ErmakArgs k, MassArgs ma,
    const int *__restrict__ type,
    const int *__restrict__ orig, const double *__restrict__ gauss, double4 *__restrict__ pos,
    const double *__restrict__ vel, const double *__restrict__ acc,
    const double *__restrict__ xold, GhStatus *st) {
  if (halted(st)) return;
  const long long step = k.step;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double d2 = 0.0;
  if (i < n) {
    double g[6];
    ermak_gauss(k, orig[i], gauss, ncap, g);
    const double f_lan = k.skt * ma.osm[type[i]];
    double4 p = pos[i];
    double x[3] = {p.x, p.y, p.z};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double pos_v = f_lan * k.sdr * g[2 * d];
      x[d] = x[d] + k.c1 * vel[d * ncap + i] + k.c2 * k.dt * acc[d * ncap + i] + pos_v;
      const double dd = x[d] - xold[d * ncap + i];
      d2 += dd * dd;
    }
    p.x = x[0];
    p.y = x[1];
    p.z = x[2];
    pos[i] = p;
  }
  disp_reduce(d2, st, step);
}

// ermak_b (Integration.F90:1013-1031); vel_v is re-derived from the same
// normals that ermak_a used (same stream entry), not stored.
__global__ __launch_bounds__(GH_BLOCK) void k_ermak_b(
    int n, int ncap, ErmakArgs k, MassArgs ma, const int *__restrict__ type,
    const int *__restrict__ orig, const double *__restrict__ gauss, double *__restrict__ vel,
    double *__restrict__ acc, const double *__restrict__ frc, const GhStatus *st) {
  if (halted(st)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double g[6];
  ermak_gauss(k, orig[i], gauss, ncap, g);
  const int t = type[i];
  const double f_lan = k.skt * ma.osm[t];
  const double om = ma.om[t];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double vel_v = f_lan * k.sdv * (k.crv1 * g[2 * d] + k.crv2 * g[2 * d + 1]);
    const double f = frc[d * ncap + i];
    vel[d * ncap + i] = k.c0 * vel[d * ncap + i] + (k.c1 - k.c2) * acc[d * ncap + i] +
                        k.c2 * f * om + vel_v;
    acc[d * ncap + i] = f * om;
  }
}

// ermak_b of step k.step - 1 and ermak_a of k.step in one kernel (Philox
// stream), where the force pass does not apply them.
__global__ __launch_bounds__(GH_BLOCK) void k_ermak_ba(
    int n, int ncap, ErmakArgs k, MassArgs ma, const int *__restrict__ type,
    const int *__restrict__ orig, double4 *__restrict__ pos, double *__restrict__ vel,
    double *__restrict__ acc, const double *__restrict__ frc, const double *__restrict__ xold,
    GhStatus *st) {
  if (halted(st)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double d2 = 0.0;
  if (i < n) {
    double g[6], h[6];
    const int id = orig[i], t = type[i];
    philox_normals(k.seed, k.step - 1, id, g);
    philox_normals(k.seed, k.step, id, h);
    const double f_lan = k.skt * ma.osm[t], om = ma.om[t];
    double4 p = pos[i];
    double x[3] = {p.x, p.y, p.z};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double vel_v = f_lan * k.sdv * (k.crv1 * g[2 * d] + k.crv2 * g[2 * d + 1]);
      const double f = frc[d * ncap + i];
      const double v = k.c0 * vel[d * ncap + i] + (k.c1 - k.c2) * acc[d * ncap + i] +
                       k.c2 * f * om + vel_v;
      const double a = f * om;
      vel[d * ncap + i] = v;
      acc[d * ncap + i] = a;
      x[d] = x[d] + k.c1 * v + k.c2 * k.dt * a + f_lan * k.sdr * h[2 * d];
      const double dd = x[d] - xold[d * ncap + i];
      d2 += dd * dd;
    }
    p.x = x[0];
    p.y = x[1];
    p.z = x[2];
    pos[i] = p;
  }
  disp_reduce(d2, st, k.step);
}

// ---------------------------------------------------------------------------
// Energies (write_energy, Output.F90:824-831): deterministic two-stage sums,
// compensated: every running sum carries its rounding error beside it
// (TwoSum, Knuth), partial sums travel as (sum, error) pairs and the result
// is sum + error, so the total does not depend on the grid's order of
// accumulation beyond the last bit.  (The reference sums per atom with an
// OpenMP reduction, TB.F90:472-477.)
// stage A: [epot, M, Px, Py, Pz] partials; stage B: sum m |v - vcm|^2.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void dd_add(double &s, double &c, double x) {
  const double t = s + x;
  const double bp = t - s;
  c += (s - (t - bp)) + (x - bp);
  s = t;
}

// Block-wide compensated sums of NV values; deterministic order.  Result
// (sum, error) valid in thread 0.
template <int NV>
__device__ __forceinline__ void block_sum_dd(double (&s)[NV], double (&c)[NV]) {
  __shared__ double part[GH_BLOCK / 64][NV][2];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k)
    for (int o = 32; o > 0; o >>= 1) {
      const double s2 = __shfl_xor(s[k], o, 64), c2 = __shfl_xor(c[k], o, 64);
      dd_add(s[k], c[k], s2);
      c[k] += c2;
    }
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      part[wid][k][0] = s[k];
      part[wid][k][1] = c[k];
    }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double ss = 0.0, cc = 0.0;
      for (int w = 0; w < GH_BLOCK / 64; ++w) {
        dd_add(ss, cc, part[w][k][0]);
        cc += part[w][k][1];
      }
      s[k] = ss;
      c[k] = cc;
    }
  }
}

// True in every thread of the grid's last workgroup to arrive, whose reads then
// see the others' writes; the ticket is left at zero.  (256 workgroups at
// most in the reductions, 512 in k_row_force's sum of the calls without
// allocation: each arrival is a fence.)
__device__ __forceinline__ bool last_block(unsigned *ticket) {
  __shared__ bool last;
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    last = atomicAdd(ticket, 1u) == gridDim.x - 1;
  }
  __syncthreads();
  if (!last) return false;
  __threadfence();
  if (threadIdx.x == 0) *ticket = 0u;
  return true;
}

// The workgroups' compensated sums of NV values to their grid total, formed by
// the last workgroup; true there, the totals in v of thread 0.  (A launch of
// its own for the totals cost 4-6 us per energy row.)
template <int NV>
__device__ __forceinline__ bool grid_sum_dd(double (&v)[NV], double (&e)[NV], double *part,
                                            unsigned *ticket) {
  block_sum_dd<NV>(v, e);
  if (threadIdx.x == 0)
    for (int k = 0; k < NV; ++k) {
      part[(blockIdx.x * NV + k) * 2] = v[k];
      part[(blockIdx.x * NV + k) * 2 + 1] = e[k];
    }
  if (!last_block(ticket)) return false;
  for (int k = 0; k < NV; ++k) v[k] = e[k] = 0.0;
  for (int b = threadIdx.x; b < (int)gridDim.x; b += blockDim.x)
    for (int k = 0; k < NV; ++k) {
      dd_add(v[k], e[k], part[(b * NV + k) * 2]);
      e[k] += part[(b * NV + k) * 2 + 1];
    }
  block_sum_dd<NV>(v, e);
  for (int k = 0; k < NV; ++k) v[k] += e[k];
  return true;
}

// The status to pinned host memory, by a workgroup.
__device__ __forceinline__ void report_status(GhReport *rep, const GhStatus *st) {
  static_assert(sizeof(GhStatus) % 8 == 0, "copied by words");
  const unsigned long long *in = reinterpret_cast<const unsigned long long *>(st);
  unsigned long long *out = reinterpret_cast<unsigned long long *>(&rep->st);
  for (int k = threadIdx.x; k < (int)(sizeof(GhStatus) / 8); k += blockDim.x) out[k] = in[k];
}

// Potential energy alone (gh_compute).
__global__ __launch_bounds__(GH_BLOCK) void k_red_epot(int n, const double *__restrict__ epa,
                                                       double *part, unsigned *ticket,
                                                       GhReport *rep) {
  double v[1] = {0.0}, e[1] = {0.0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    dd_add(v[0], e[0], epa[i]);
  if (grid_sum_dd<1>(v, e, part, ticket) && threadIdx.x == 0) rep->epot = v[0];
}

__global__ __launch_bounds__(GH_BLOCK) void k_red_a(int n, int ncap, MassArgs ma,
                                                    const int *__restrict__ type,
                                                    const double *__restrict__ epa,
                                                    const double *__restrict__ vel, double *part,
                                                    unsigned *ticket, double *sums,
                                                    GhReport *rep) {
  double v[5] = {0, 0, 0, 0, 0}, e[5] = {0, 0, 0, 0, 0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const double m = 1.0 / ma.om[type[i]];
    dd_add(v[0], e[0], epa[i]);
    dd_add(v[1], e[1], m);
    dd_add(v[2], e[2], m * vel[i]);
    dd_add(v[3], e[3], m * vel[ncap + i]);
    dd_add(v[4], e[4], m * vel[2 * ncap + i]);
  }
  if (grid_sum_dd<5>(v, e, part, ticket) && threadIdx.x == 0) {
    rep->epot = v[0];
    for (int k = 0; k < 5; ++k) sums[k] = v[k];
  }
}

__global__ __launch_bounds__(GH_BLOCK) void k_red_b(int n, int ncap, MassArgs ma,
                                                    const int *__restrict__ type,
                                                    const double *__restrict__ vel,
                                                    const double *__restrict__ sums, double *part,
                                                    unsigned *ticket, const GhStatus *st,
                                                    GhReport *rep) {
  const double M = sums[1];
  const double cx = sums[2] / M, cy = sums[3] / M, cz = sums[4] / M;
  double v[1] = {0}, e[1] = {0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const double m = 1.0 / ma.om[type[i]];
    const double wx = vel[i] - cx, wy = vel[ncap + i] - cy, wz = vel[2 * ncap + i] - cz;
    dd_add(v[0], e[0], (wx * wx + wy * wy + wz * wz) * m);
  }
  if (grid_sum_dd<1>(v, e, part, ticket)) {
    if (threadIdx.x == 0) rep->ekin2 = v[0];
    report_status(rep, st);
  }
}

// ---------------------------------------------------------------------------
// Passes over rows of atom numbers.
// ---------------------------------------------------------------------------
// The parameter block of a pair: kernel argument (one type) or LDS table.
// FP64 (Tb64) and mixed precision (TbF in Angstrom; the pair vector stays
// FP64, the pair terms are FP32, sums FP64).
template <bool MIXED>
using TbForm = typename std::conditional<MIXED, TbF, Tb64>::type;
template <bool MIXED>
__device__ __forceinline__ const TbForm<MIXED> &tb_form(const TbDev &d) {
  if constexpr (MIXED) return d.f;
  else return d.d;
}

struct RowArgs {
  GhStatus *st;
  StepArgs sa;
  int cell;     // cell mode: the step's first pass tests the rebuild rule (step_gate)
  int inline_build;  // O(N^2) mode: SMA-TB's density pass builds the rows itself
  double4 *pos;
  const int *type, *nn;
  const unsigned *list;
  int n, cap, ncap, nt;
  double L[3];
  const TbDev *tbd;
  double *rho;
  double e0, ev_ui;
  double *frc, *epa;
  // FUSE 3 (forces without allocation): the caller's arrays
  double *F_out, *epot_out, *part;
  int *status_out;
  unsigned *ticket;
};

// First pass of a step in cell mode: gated and published as the tiled ones;
// in the O(N^2) mode published.  True: nothing to do.
__device__ __forceinline__ bool rows_gate(const RowArgs &A) {
  if (A.cell) return step_gate(A.st, A.sa);
  if (blockIdx.x == 0 && threadIdx.x == 0)
    step_publish(A.sa.prog, A.sa.step, halted(A.st), A.st->halt_step,
                 disp2_max(A.st, A.sa.step));
  return false;
}
// The atom of the thread's G lanes; workgroups in XCD order.
template <int G>
__device__ __forceinline__ int row_atom() {
  return (int)(xcd_block() * GH_BLOCK + threadIdx.x) / G;
}

// 1/sqrt(rho) (FP64) or its FP32 offset from e0 and the type (mixed), held in
// the fourth word of an atom's position from the density pass on.
template <bool MIXED>
__device__ __forceinline__ double eb_word(double eb, double e0, int t) {
  if (!MIXED) return eb;
  return __hiloint2double(t, __float_as_int((float)(eb - e0)));
}

// SMA-TB pass 1 (smatb_preinteraction, TB.F90:367-455):
//   rho_i = sum_j [ r < rci ? xi^2 exp(-2q(r/r0-1)) : (b1 x^5 + b2 x^4 + b3 x^3)^2 ]
//   with x = r - rce and r > rce skipped.
template <bool MIXED, bool SINGLE, int G>
__global__ __launch_bounds__(GH_BLOCK) void k_row_rho(RowArgs A, N2Build B, TbForm<MIXED> p1) {
  if (rows_gate(A)) return;
  __shared__ ShiftLds sh;
  __shared__ TbForm<MIXED> sp[SINGLE ? 1 : GH_MAXT * GH_MAXT];
  load_shift(sh, A.L[0], A.L[1], A.L[2]);
  if (!SINGLE) load_params(sp, A.tbd, A.nt);
  bool due = false;
  if (G == 64 && A.inline_build) due = n2_decide(A.st, A.sa.skin, A.sa.step);
  else __syncthreads();
  const int i0 = row_atom<G>(), sub = threadIdx.x & (G - 1);
  const bool live = i0 < A.n;
  const int i = min(i0, A.n - 1);
  if (due) {
    n2_rows_max(n2_rows<1>(B, __builtin_amdgcn_readfirstlane(i0)), A.st, B.cap, A.sa.step);
    __threadfence_block();  // the wavefront reads the row its own lanes wrote
  }
  Row<G> row = row_head<G>(A.list, A.nn, A.cap, i, live);
  const double4 pi = A.pos[i];
  const int ti = SINGLE ? 0 : A.type[i];
  double acc = 0.0;
  row_each<G>(row, A.pos, pi, sh, [&](int j, const double4 &, double vx, double vy, double vz) {
    const TbForm<MIXED> &P = SINGLE ? p1 : sp[ti * GH_MAXT + A.type[j]];
    const double rd = fma(vx, vx, fma(vy, vy, vz * vz));
    if constexpr (MIXED) {
      float band;
      if (tb_rho_fx(P, rd, band)) acc += (double)band;
    } else if (!(rd > P.rce2)) {
      double dr, ir;
      sqrt_rsq64(rd, dr, ir);
      acc = __dadd_rn(acc, tb_band64(P, dr));
    }
  });
  acc = lanes_total<G>(acc);
  if (live && sub == 0) {
    A.rho[i] = acc;
    // (other lanes read this position's first three words only)
    A.pos[i].w = eb_word<MIXED>(1.0 / sqrt(acc), A.e0, ti);
  }
}

// Velocity Verlet or Ermak update of an atom whose force its G lanes hold:
// lanes 0..2 an axis each, new positions to pos_next (other atoms' lanes still
// read pos); the Ermak update draws the next step's normals in lanes 4..6.
// Returns |x_new - x_old|^2 in lane 0 (FUSE 1: stepb and stepa as fused_vv; 2:
// ermak_b of this step and ermak_a of the next).
template <int FUSE>
using FuseT = typename std::conditional<FUSE == 2, FuseErmak, FuseVV>::type;
struct AxisLoad {
  double v, a, xo;
  int id;
};
template <int FUSE>
__device__ __forceinline__ AxisLoad axis_load(const FuseT<FUSE> &f, int i, int ax) {
  AxisLoad l{0.0, 0.0, 0.0, 0};
  if constexpr (FUSE == 1 || FUSE == 2) {
    l.v = f.vel[ax * f.ncap + i];
    l.xo = f.xold[ax * f.ncap + i];
    if constexpr (FUSE == 2) {
      l.a = f.acc[ax * f.ncap + i];
      l.id = f.orig[i];
    }
  }
  return l;
}
template <int FUSE>
__device__ __forceinline__ double axis_update(const FuseT<FUSE> &f, const AxisLoad &l, int i,
                                              int lane, int ax, const double4 &p, int t, double F,
                                              bool live) {
  double x = ax == 0 ? p.x : ax == 1 ? p.y : p.z, v;
  if constexpr (FUSE == 2) {
    const ErmakArgs &k = f.k;
    float ga, gb;
    axis_normals(k.seed, k.step + (lane >= 4 ? 1 : 0), l.id, ax, ga, gb);
    const float gn = __shfl_down(ga, 4, 64);
    const double f_lan = k.skt * f.osm[t];
    const double vel_v = f_lan * k.sdv * (k.crv1 * (double)ga + k.crv2 * (double)gb);
    const double a = F * f.om[t];
    v = k.c0 * l.v + (k.c1 - k.c2) * l.a + k.c2 * F * f.om[t] + vel_v;
    x = x + k.c1 * v + k.c2 * k.dt * a + f_lan * k.sdr * (double)gn;
    if (live && lane < 3) f.acc[ax * f.ncap + i] = a;
  } else {
    const double a = __dmul_rn(F, f.om[t]);  // rounded as in fused_vv
    v = fma(f.acel_dv, a, l.v);                      // stepb
    x = fma(f.acel_dx, a, fma(f.dt, v, x));          // stepa
    v = fma(f.acel_dv, a, v);
  }
  if (live && lane < 3) {
    f.vel[ax * f.ncap + i] = v;
    reinterpret_cast<double *>(f.pos_next + i)[ax] = x;
  }
  const double dd = x - l.xo;
  double d2 = live && lane < 3 ? dd * dd : 0.0;
  d2 += dpp64<0xB1>(d2);
  d2 += dpp64<0x4E>(d2);
  return d2;
}

// Forces f = {Fx, Fy, Fz, energy sum} (ui/A and eV) of an atom, the same in
// its G lanes, to where the launch wants them.  FUSE 0: stored with the
// per-atom energy e; 1, 2: the update; 3: stored in the caller's layout, the
// total energy by the last workgroup.  All threads call it.
template <int G, int FUSE>
__device__ __forceinline__ void row_result(const RowArgs &A, const FuseT<FUSE> &fv,
                                           const AxisLoad &ld, int i, bool live, const double4 &pi,
                                           int t, const double (&F)[3], double e) {
  const int lane = threadIdx.x & (G - 1), ax = min(lane & 3, 2);
  const double Fa = ax == 0 ? F[0] : ax == 1 ? F[1] : F[2];
  if constexpr (FUSE == 1 || FUSE == 2) {
    const double d2 = axis_update<FUSE>(fv, ld, i, lane, ax, pi, t, Fa, live);
    // (the O(N^2) mode's first workgroup books the rebuild in this kernel)
    if (A.cell) disp_reduce(d2, A.st, A.sa.step + 1);
    else disp_reduce<false>(d2, A.st, A.sa.step + 1);
  } else {
    if (live && lane < 3) {
      if (FUSE == 3) A.F_out[3 * i + lane] = Fa;
      else A.frc[lane * A.ncap + i] = Fa;
    } else if (live && lane == 3) {
      A.epa[i] = e;
    }
    if constexpr (FUSE == 3) {
      double v[1] = {live && lane == 3 ? e : 0.0}, c[1] = {0.0};
      if (grid_sum_dd<1>(v, c, A.part, A.ticket) && threadIdx.x == 0) {
        *A.epot_out = v[0];
        *A.status_out = A.st->overflow ? GH_EOVERFLOW : 0;
      }
    }
  }
}

// SMA-TB pass 2 (smatb_interact, TB.F90:457-586), full list, newton off:
//   r <= rci: repul = A e^{-p(r/r0-1)};
//             factor = 2 repul p/r0 - xi^2/2 e^{-2q(r/r0-1)} (2q/r0)(eb_i+eb_j)
//   rci < r <= rce: factor = P P' (eb_i+eb_j) - 2 R';  repul = R
//   F_i -= factor * vd / r  (vd = x_j - x_i), e_i = sum repul - sqrt(rho_i).
template <bool MIXED, bool SINGLE, int G, int FUSE>
__global__ __launch_bounds__(GH_BLOCK) void k_row_force(RowArgs A, TbForm<MIXED> p1,
                                                        FuseT<FUSE> fv) {
  if (!A.cell && blockIdx.x == 0 && threadIdx.x == 0) n2_book(A.st, A.sa.step);
  if ((FUSE == 1 || FUSE == 2 || A.cell) && halted(A.st)) return;
  __shared__ ShiftLds sh;
  __shared__ TbForm<MIXED> sp[SINGLE ? 1 : GH_MAXT * GH_MAXT];
  load_shift(sh, A.L[0], A.L[1], A.L[2]);
  if (!SINGLE) load_params(sp, A.tbd, A.nt);
  __syncthreads();
  const int i0 = row_atom<G>(), lane = threadIdx.x & (G - 1);
  const bool live = i0 < A.n;
  const int i = min(i0, A.n - 1);
  Row<G> row = row_head<G>(A.list, A.nn, A.cap, i, live);
  const double4 pi = A.pos[i];
  const int ti = SINGLE ? 0 : A.type[i];
  const AxisLoad ld = axis_load<FUSE>(fv, i, min(lane & 3, 2));
  double f[4] = {0.0, 0.0, 0.0, 0.0};
  row_each<G>(row, A.pos, pi, sh, [&](int j, const double4 &pj, double vx, double vy, double vz) {
    const double rd = fma(vx, vx, fma(vy, vy, vz * vz));
    double s, rep;
    if constexpr (MIXED) {
      const TbForm<MIXED> &P = SINGLE ? p1 : sp[ti * GH_MAXT + __double2hiint(pj.w)];
      float sf, repul;
      if (!tb_force_fx<true>(P, rd,
                             __int_as_float(__double2loint(pi.w)) +
                                 __int_as_float(__double2loint(pj.w)),
                             sf, repul))
        return;
      s = (double)sf;
      rep = (double)repul;
    } else {
      const TbForm<MIXED> &P = SINGLE ? p1 : sp[ti * GH_MAXT + A.type[j]];
      if (rd > P.rce2) return;
      double dr, ir, factor;
      sqrt_rsq64(rd, dr, ir);
      tb_pair64(P, dr, pi.w + pj.w, factor, rep);
      s = factor * ir;
    }
    f[0] = fma(-s, vx, f[0]);
    f[1] = fma(-s, vy, f[1]);
    f[2] = fma(-s, vz, f[2]);
    f[3] = __dadd_rn(f[3], rep);
  });
#pragma unroll
  for (int d = 0; d < (FUSE == 1 || FUSE == 2 ? 3 : 4); ++d) f[d] = lanes_total<G>(f[d]);
  const double F[3] = {f[0] * A.ev_ui, f[1] * A.ev_ui, f[2] * A.ev_ui};
  const double e = FUSE == 1 || FUSE == 2 ? 0.0 : (f[3] - sqrt(A.rho[i])) * A.ev_ui;
  row_result<G, FUSE>(A, fv, ld, i, live, pi, ti, F, e);
}

// Pair potentials, full list, newton off: e_i += p/2; F_i -= f vd / r.
// POT: GH_POT_LJ (lj_interact, Pairs.F90:207-279: r^2 > rc^2 skipped; p =
// 4e(s6^2 - s6); f = e(48 s6 - 24) s6 / r) or a tabulated form per type pair
// (plj_interact, Pairs.F90:293-370; slj_interact, :403-493; wca_interact,
// :508-560; sm1_interact, :916-990).
// The step's first pass in cell mode; the O(N^2) mode's is the list build.
template <bool MIXED, int POT, int FUSE>
__global__ __launch_bounds__(GH_BLOCK) void k_row_pair(RowArgs A, const PljDev *__restrict__ pljd,
                                                       double eps, double sig2, double rc2,
                                                       FuseT<FUSE> fv) {
  constexpr int G = 16;
  constexpr bool TAB = POT != GH_POT_LJ;
  if (rows_gate(A)) return;
  if (!A.cell && blockIdx.x == 0 && threadIdx.x == 0) n2_book(A.st, A.sa.step);
  if (FUSE && halted(A.st)) return;
  __shared__ ShiftLds sh;
  __shared__ PljDev pp[TAB ? GH_MAXT * GH_MAXT : 1];
  load_shift(sh, A.L[0], A.L[1], A.L[2]);
  if (TAB)
    for (int k = threadIdx.x; k < GH_MAXT * GH_MAXT; k += blockDim.x) pp[k] = pljd[k];
  __syncthreads();
  const int i0 = row_atom<G>(), lane = threadIdx.x & (G - 1);
  const bool live = i0 < A.n;
  const int i = min(i0, A.n - 1);
  Row<G> row = row_head<G>(A.list, A.nn, A.cap, i, live);
  const double4 pi = A.pos[i];
  const int ti = A.type[i];
  const AxisLoad ld = axis_load<FUSE>(fv, i, min(lane & 3, 2));
  const double e4 = 4.0 * eps, e24 = 24.0 * eps, e48 = 48.0 * eps;
  double f[4] = {0.0, 0.0, 0.0, 0.0};
  row_each<G>(row, A.pos, pi, sh, [&](int j, const double4 &, double vx, double vy, double vz) {
    const double r2 = MIXED ? fma(vx, vx, fma(vy, vy, vz * vz)) : dist2_rn(vx, vy, vz);
    if (r2 > rc2) return;
    double p, s;
    if constexpr (TAB) {
      const PljDev &P = pp[ti * GH_MAXT + A.type[j]];
      if (r2 > P.rc2) return;  // this pair's cut
      if constexpr (MIXED) {
        float pf, fr;
        table_pair32<POT>(P, (float)r2, pf, fr);
        p = (double)pf;
        s = (double)fr;
      } else {
        table_pair64<POT>(P, r2, p, s);
      }
    } else if constexpr (MIXED) {
      const float ef = (float)eps, ir2 = __builtin_amdgcn_rcpf((float)r2);
      const float s2 = (float)sig2 * ir2, s6 = s2 * s2 * s2;
      p = (double)(4.0f * ef * (s6 * s6 - s6));
      s = (double)(ef * fmaf(48.0f, s6, -24.0f) * s6 * ir2);  // f / r
    } else {
      const double ir2 = rcp64(r2);
      const double s2 = sig2 * ir2, s6 = s2 * s2 * s2;
      p = e4 * (s6 * s6 - s6);
      s = fma(e48, s6, -e24) * s6 * ir2;
    }
    f[0] = fma(-s, vx, f[0]);
    f[1] = fma(-s, vy, f[1]);
    f[2] = fma(-s, vz, f[2]);
    f[3] = __dadd_rn(f[3], p);
  });
#pragma unroll
  for (int d = 0; d < (FUSE ? 3 : 4); ++d) f[d] = lanes_total<G>(f[d]);
  const double F[3] = {f[0] * A.ev_ui, f[1] * A.ev_ui, f[2] * A.ev_ui};
  row_result<G, FUSE>(A, fv, ld, i, live, pi, ti, F, f[3] * 0.5 * A.ev_ui);
}

// Wraps positions into [0, L) on periodic axes (used when the box or the
// atoms change; the timestep kernels apply do_pbc_1's single shift).
__global__ void k_wrap(int n, WrapArgs wa, double4 *__restrict__ pos) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double4 p = pos[i];
  double x[3] = {p.x, p.y, p.z};
#pragma unroll
  for (int d = 0; d < 3; ++d)
    if (wa.pbc[d]) {
      x[d] = x[d] - wa.L[d] * floor(x[d] / wa.L[d]);
      if (x[d] >= wa.L[d]) x[d] -= wa.L[d];
    }
  p.x = x[0];
  p.y = x[1];
  p.z = x[2];
  pos[i] = p;
}

// State in the caller's order (AoS), one thread per value so that the writes
// are consecutive: they may go to pinned host memory directly.  Any output may
// be null.  Positions are reported wrapped as do_pbc_1 does (they run
// continuously between rebuilds, at most half a skin outside the box).
__global__ __launch_bounds__(GH_BLOCK) void k_get(int n, int ncap, WrapArgs wa,
                                                  const int *__restrict__ inv,
                                                  const double4 *__restrict__ pos,
                                                  const double *__restrict__ vel,
                                                  const double *__restrict__ frc,
                                                  const double *__restrict__ epa, double *x,
                                                  double *v, double *F, double *e,
                                                  const GhStatus *st, GhReport *rep) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == 0 && rep) report_status(rep, st);
  if (k >= 3 * n) return;
  const int i = k / 3, d = k - 3 * i, s = inv[i];
  if (x) {
    double p = reinterpret_cast<const double *>(pos + s)[d];
    if (wa.pbc[d]) {
      if (p >= wa.L[d]) p -= wa.L[d];
      else if (p < 0.0) p += wa.L[d];
    }
    x[k] = p;
  }
  if (v) v[k] = vel[d * ncap + s];
  if (F) F[k] = frc[d * ncap + s];
  if (e && k < n) e[k] = epa[inv[k]];
}
// Vectors of the caller's atoms (3n, AoS) into a sorted array [3][ncap].
__global__ __launch_bounds__(GH_BLOCK) void k_put3(int n, int ncap, const int *__restrict__ inv,
                                                   const double *__restrict__ in,
                                                   double *__restrict__ dst) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= 3 * n) return;
  const int i = k / 3, d = k - 3 * i;
  dst[d * ncap + inv[i]] = in[k];
}

// New positions from the host, in caller order (x: 3n, AoS): each atom's
// coordinate moves to the periodic image nearest its current one (a host-side
// wrap is no displacement), and its displacement since the last build joins
// the rebuild test.
__global__ __launch_bounds__(GH_BLOCK) void k_set_positions(
    int n, int ncap, WrapArgs wa, const int *__restrict__ inv, const double *__restrict__ x,
    double4 *__restrict__ pos, const double *__restrict__ xold, GhStatus *st, long long step) {
  const int o = blockIdx.x * blockDim.x + threadIdx.x;
  double d2 = 0.0;
  if (o < n) {  // in the caller's order: x may be in host memory
    double v[3] = {x[3 * (size_t)o], x[3 * (size_t)o + 1], x[3 * (size_t)o + 2]};
    const int s = inv[o];
    double4 p = pos[s];
    const double old[3] = {p.x, p.y, p.z};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (wa.pbc[d]) v[d] += wa.L[d] * rint((old[d] - v[d]) / wa.L[d]);
      const double dd = v[d] - xold[d * ncap + s];
      d2 += dd * dd;
    }
    p.x = v[0];
    p.y = v[1];
    p.z = v[2];
    pos[s] = p;
  }
  disp_reduce(d2, st, step);
}

// Before the kernel that decides (n2_decide): the same test.
__global__ void k_wrap_rebuild(const GhStatus *st, double skin, long long step, int n, WrapArgs wa,
                               double4 *__restrict__ pos) {
  if (halted(st) || !rebuild_due(st, skin, step)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double4 p = pos[i];
  double x[3] = {p.x, p.y, p.z};
#pragma unroll
  for (int d = 0; d < 3; ++d)
    if (wa.pbc[d]) {
      x[d] = x[d] - wa.L[d] * floor(x[d] / wa.L[d]);
      if (x[d] >= wa.L[d]) x[d] -= wa.L[d];
    }
  p.x = x[0];
  p.y = x[1];
  p.z = x[2];
  pos[i] = p;
}

inline int nblocks(int n) { return (n + GH_BLOCK - 1) / GH_BLOCK; }

GridArgs make_grid(const gh_ctx *c) {
  GridArgs g;
  for (int d = 0; d < 3; ++d) {
    g.nc[d] = c->nc[d];
    g.gn[d] = c->gn[d];
    g.gofs[d] = c->gofs[d];
    g.pbc[d] = c->pbc[d];
    g.L[d] = c->L[d];
    g.one_cell[d] = 1.0 / c->cell[d];
  }
  g.ncell = c->ncell;
  g.ghost = c->ghost;
  return g;
}

inline int n2_blocks(int n, int rows) {
  const int per = GH_BLOCK / 64 * rows;
  return (n + per - 1) / per;
}

N2Build make_n2_build(const gh_ctx *c) {
  const double rl = c->rcut + c->skin;
  return N2Build{c->pos, c->n, c->cap, c->ncap, make_grid(c), rl * rl, c->nn,
                 c->list, c->xold, c->orig,
                 c->masked ? c->mfeel : nullptr, c->masked ? c->mfelt : nullptr};
}

// Workgroups of a pass with G lanes per atom, in XCD order.
inline int row_blocks(int n, int lanes) {
  const int per = GH_BLOCK / lanes;
  return xgrid((n + per - 1) / per);
}

RowArgs make_row_args(const gh_ctx *c) {
  RowArgs A;
  memset(&A, 0, sizeof(A));
  A.st = c->status;
  A.sa = StepArgs{c->step, c->skin, c->prog_d};
  A.cell = c->list_mode == 1;
  A.inline_build = !A.cell && c->pot == GH_POT_SMATB && c->n <= 1024;
  A.pos = c->pos;
  A.type = c->type;
  A.nn = c->nn;
  A.list = c->list;
  A.n = c->n;
  A.cap = c->cap;
  A.ncap = c->ncap;
  A.nt = c->nt;
  for (int d = 0; d < 3; ++d) A.L[d] = c->L[d];
  A.tbd = c->tbd;
  A.rho = c->rho;
  A.e0 = c->tb_e0;
  A.ev_ui = ghc::ev_ui();
  A.frc = c->frc;
  A.epa = c->epa;
  return A;
}

MassArgs make_mass(const gh_ctx *c) {
  MassArgs m;
  for (int t = 0; t < GH_MAXT; ++t) {
    m.om[t] = 1.0 / c->mass_t[t];
    m.osm[t] = sqrt(m.om[t]);
  }
  return m;
}

WrapArgs make_wrap(const gh_ctx *c) {
  WrapArgs w;
  for (int d = 0; d < 3; ++d) {
    w.pbc[d] = c->boxed ? c->pbc[d] : 0;
    w.L[d] = c->L[d];
  }
  return w;
}

ErmakArgs make_ermak(const gh_ctx *c) {
  ErmakArgs k;
  const double dt = c->dt, gama = c->gamma;
  k.c0 = exp(-dt * gama);
  k.c1 = (1.0 - k.c0) / gama;
  k.c2 = (1.0 - k.c1 / dt) / gama;
  k.sdr = sqrt(dt / gama * (2.0 - (3.0 - 4.0 * k.c0 + k.c0 * k.c0) / (dt * gama)));
  k.sdv = sqrt(1.0 - k.c0 * k.c0);
  k.crv1 = (1.0 - k.c0) * (1.0 - k.c0) / (gama * k.sdr * k.sdv);
  k.crv2 = sqrt(1.0 - (k.crv1 * k.crv1));
  k.skt = sqrt(ghc::kB_ui() * c->T);
  k.dt = dt;
  k.philox = c->rng_mode == GH_RNG_PHILOX;
  k.seed = c->philox_seed;
  k.step = c->step;
  return k;
}

}  // namespace

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// Neighbour rebuild.  force: request a rebuild regardless of displacement.
// Every kernel of the rebuild tests the rule or reads the flag its first one set, so the
// sequence can be enqueued every step without a host round trip.
using namespace ghd;

int gh_request_rebuild(gh_ctx *c) {
  hipStream_t s = c->stream;
  GhStatus h;
  GH_HIP(c, hipMemcpyAsync(&h, c->status, sizeof(GhStatus), hipMemcpyDeviceToHost, s));
  GH_HIP(c, hipStreamSynchronize(s));
  h.force_rebuild = 1;
  GH_HIP(c, hipMemcpyAsync(c->status, &h, sizeof(GhStatus), hipMemcpyHostToDevice, s));
  GH_HIP(c, hipStreamSynchronize(s));
  return 0;
}

// forces_follow: a force evaluation is enqueued next.  The O(N^2) mode's
// SMA-TB density pass then builds the rows itself (one wavefront per atom has
// the row's atom at hand: one launch and its gap less per step); its
// second kernel of the step books the rebuild.
static bool n2_inline(const gh_ctx *c) { return c->pot == GH_POT_SMATB && c->n <= 1024; }

int gh_launch_rebuild(gh_ctx *c, bool force, bool forces_follow) {
  hipStream_t s = c->stream;
  if (force) GH_TRY(gh_request_rebuild(c));
  const int n = c->n, nb = nblocks(n);
  if (c->list_mode == 1) return gh_launch_rebuild_cells(c);  // decides in its first kernels
  if (c->boxed && (c->pbc[0] || c->pbc[1] || c->pbc[2]))
    { k_wrap_rebuild<<<nb, GH_BLOCK, 0, s>>>(c->status, c->skin, c->step, n, make_wrap(c), c->pos); ++c->launches; }
  if (!forces_follow || !n2_inline(c)) {
    const N2Build B = make_n2_build(c);
    // rows per wavefront: one where the atoms do not fill the chip's wavefront
    // slots anyway, several where every wavefront reads all positions (32 n^2
    // bytes through the caches: 130 MB at 2,048 atoms, 33 MB with four rows)
    if (n <= 1024) k_build_n2<1><<<n2_blocks(n, 1), GH_BLOCK, 0, s>>>(c->status, B, c->skin, c->step);
    else if (n <= 8192) k_build_n2<4><<<n2_blocks(n, 4), GH_BLOCK, 0, s>>>(c->status, B, c->skin, c->step);
    else k_build_n2<8><<<n2_blocks(n, 8), GH_BLOCK, 0, s>>>(c->status, B, c->skin, c->step);
    ++c->launches;
  }
  if (!forces_follow) { k_n2_book<<<1, 1, 0, s>>>(c->status, c->step); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

// Cell mode by rows of atom numbers instead of tiles: FP64, whatever the shape
// asked for.  200 velocity Verlet steps, tiled -> rows, ms: Au 2,048 atoms
// 6.7 -> 3.0, 32,000 7.7 -> 5.5, 119,164 17.8 -> 14.0 (the same bits either
// way, tiles taking four lanes per atom there); above, with one lane per atom,
// tiles win for one type (Au 256,000 21.3 against 28.2; a row entry is four
// bytes and its neighbour's 32 come from the L2).  With several types a pair's
// parameters come from LDS, which the tiles' positions and lists already load:
// 40 steps Ag-Cu 143,748 9.5 -> 7.4, 256,000 14.9 -> 11.4; 442,368 21.6 and, at
// the best shape, 18.6 against 18.7; 1M 39.3 against 42.7.  Pair potentials
// have one pass and less to save: LJ 2,048 4.6 -> 3.4, 32,000 7.2 -> 5.9, 55,296
// 8.3 -> 8.2, 119,164 12.6 against 14.2.  The environment's choice of a tiled
// list build or of workgroups per brick keeps the tiles.
bool gh_rows_path(const gh_ctx *c) {
  const int most = c->pot != GH_POT_SMATB ? 65536 : c->nt == 1 ? 131072 : 393216;
  return c->precision == GH_FP64 && c->n < most && c->list_rows == 0 && c->chunks_env == 0;
}

bool gh_can_fuse(const gh_ctx *c) {
  if (c->integ == GH_INT_VV) return true;
  return c->rng_mode == GH_RNG_PHILOX && (c->list_mode == 0 || c->rows);
}

FuseVV gh_fuse_vv(const gh_ctx *c) {
  FuseVV fv;
  fv.dt = c->dt;
  fv.acel_dv = c->dt * 0.5;
  fv.acel_dx = fv.acel_dv * c->dt;
  for (int t = 0; t < GH_MAXT; ++t) fv.om[t] = 1.0 / c->mass_t[t];
  fv.vel = c->vel;
  fv.xold = c->xold;
  fv.pos_next = c->pos_next;
  fv.ncap = c->ncap;
  return fv;
}

static FuseErmak make_fuse_ermak(const gh_ctx *c) {
  FuseErmak f;
  f.k = make_ermak(c);
  const MassArgs m = make_mass(c);
  for (int t = 0; t < GH_MAXT; ++t) {
    f.om[t] = m.om[t];
    f.osm[t] = m.osm[t];
  }
  f.vel = c->vel;
  f.acc = c->acc;
  f.xold = c->xold;
  f.orig = c->orig;
  f.pos_next = c->pos_next;
  f.ncap = c->ncap;
  return f;
}

int gh_launch_forces(gh_ctx *c, hipEvent_t mid, bool fuse) {
  if (c->list_mode == 1 && !c->rows) return gh_launch_forces_tiled(c, mid, fuse);
  hipStream_t s = c->stream;
  const bool single = c->nt == 1, mixed = c->precision == GH_MIXED, cell = c->list_mode == 1;
  const int fu = !fuse ? 0 : c->integ == GH_INT_VV ? 1 : 2;
  const FuseVV fv = gh_fuse_vv(c);
  FuseErmak fe{};
  if (fu == 2) fe = make_fuse_ermak(c);
  const RowArgs A = make_row_args(c);
  if (c->pot == GH_POT_SMATB) {
    const N2Build B = make_n2_build(c);
    const int nb = row_blocks(c->n, cell ? 16 : 64);
#define ROW_RHO(MX, SG, GG, P) k_row_rho<MX, SG, GG><<<nb, GH_BLOCK, 0, s>>>(A, B, P)
#define ROW_FORCE(MX, SG, GG, P)                                                            \
  do {                                                                                      \
    if (fu == 0) k_row_force<MX, SG, GG, 0><<<nb, GH_BLOCK, 0, s>>>(A, P, fv);               \
    else if (fu == 1) k_row_force<MX, SG, GG, 1><<<nb, GH_BLOCK, 0, s>>>(A, P, fv);          \
    else k_row_force<MX, SG, GG, 2><<<nb, GH_BLOCK, 0, s>>>(A, P, fe);                       \
  } while (0)
#define ROW_TB(KERNEL)                                                                      \
  do {                                                                                      \
    if (cell) {                                                                             \
      if (single) KERNEL(false, true, 16, c->tb64_0);                                       \
      else KERNEL(false, false, 16, c->tb64_0);                                             \
    } else if (mixed) {                                                                     \
      if (single) KERNEL(true, true, 64, c->tbf_a0);                                        \
      else KERNEL(true, false, 64, c->tbf_a0);                                              \
    } else {                                                                                \
      if (single) KERNEL(false, true, 64, c->tb64_0);                                       \
      else KERNEL(false, false, 64, c->tb64_0);                                             \
    }                                                                                       \
    ++c->launches;                                                                          \
  } while (0)
    ROW_TB(ROW_RHO);
    if (mid) GH_HIP(c, hipEventRecord(mid, s));
    ROW_TB(ROW_FORCE);
#undef ROW_TB
#undef ROW_FORCE
#undef ROW_RHO
  } else if (c->pot == GH_POT_LJ || gh_is_table_pot(c->pot)) {
    if (mid) GH_HIP(c, hipEventRecord(mid, s));
    const double rc2 = c->lj_rc * c->lj_rc, sig2 = c->lj_sigma * c->lj_sigma;
    const int nb = row_blocks(c->n, 16);
#define ROW_PAIR3(MX, PT, FU, F) \
  k_row_pair<MX, PT, FU><<<nb, GH_BLOCK, 0, s>>>(A, c->pljd, c->lj_eps, sig2, rc2, F)
#define ROW_PAIR2(MX, PT)                                                                   \
  do {                                                                                      \
    if (fu == 0) ROW_PAIR3(MX, PT, 0, fv);                                                  \
    else if (fu == 1) ROW_PAIR3(MX, PT, 1, fv);                                             \
    else ROW_PAIR3(MX, PT, 2, fe);                                                          \
  } while (0)
#define ROW_PAIR(PT)                                                                        \
  do {                                                                                      \
    if (mixed) ROW_PAIR2(true, PT);                                                         \
    else ROW_PAIR2(false, PT);                                                              \
    ++c->launches;                                                                          \
  } while (0)
    switch (c->pot) {
      case GH_POT_SLJ: ROW_PAIR(GH_POT_SLJ); break;
      case GH_POT_WCA: ROW_PAIR(GH_POT_WCA); break;
      case GH_POT_SM1: ROW_PAIR(GH_POT_SM1); break;
      case GH_POT_PLJ: ROW_PAIR(GH_POT_PLJ); break;
      default: ROW_PAIR(GH_POT_LJ);
    }
#undef ROW_PAIR
#undef ROW_PAIR2
#undef ROW_PAIR3
  } else {
    return gh_fail(c, GH_ESTATE, "no potential set");
  }
  GH_HIP(c, hipGetLastError());
  return 0;
}

int gh_launch_vv_a(gh_ctx *c) {
  { k_vv_a<<<nblocks(c->n), GH_BLOCK, 0, c->stream>>>(c->n, c->ncap, c->dt,
                                                    make_mass(c), c->type, c->pos, c->vel,
                                                    c->acc, c->frc, c->xold, c->status,
                                                    c->step); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

int gh_launch_ermak_ba(gh_ctx *c) {
  { k_ermak_ba<<<nblocks(c->n), GH_BLOCK, 0, c->stream>>>(
      c->n, c->ncap, make_ermak(c), make_mass(c), c->type, c->orig, c->pos, c->vel, c->acc, c->frc,
      c->xold, c->status); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

int gh_launch_vv_b(gh_ctx *c) {
  { k_vv_b<<<nblocks(c->n), GH_BLOCK, 0, c->stream>>>(c->n, c->ncap, c->dt, make_mass(c), c->type,
                                                    c->vel, c->acc, c->frc, c->status); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

int gh_launch_ermak_a(gh_ctx *c) {
  { k_ermak_a<<<nblocks(c->n), GH_BLOCK, 0, c->stream>>>(
      c->n, c->ncap, make_ermak(c), make_mass(c), c->type, c->orig,
      c->gauss, c->pos, c->vel, c->acc, c->xold, c->status); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

int gh_launch_ermak_b(gh_ctx *c) {
  { k_ermak_b<<<nblocks(c->n), GH_BLOCK, 0, c->stream>>>(c->n, c->ncap, make_ermak(c),
                                                       make_mass(c), c->type, c->orig,
                                                       c->gauss, c->vel, c->acc, c->frc,
                                                       c->status); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

// Reduction grids: 256 workgroups at most (last_block).
static int red_blocks(int n) { return std::min(256, std::max(1, nblocks(n))); }

// epot of the current forces into the report; asynchronous.
int gh_launch_epot(gh_ctx *c) {
  { k_red_epot<<<red_blocks(c->n), GH_BLOCK, 0, c->stream>>>(c->n, c->epa, c->red, c->red_tick,
                                                             c->rep_h); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

// epot and ekin (ui) of the current state, and the status; host-synchronous.
int gh_launch_energies(gh_ctx *c, double *epot_ui, double *ekin_ui, GhStatus *st) {
  hipStream_t s = c->stream;
  const int nblk = red_blocks(c->n);
  const MassArgs ma = make_mass(c);
  double *part = c->red, *sums = c->red + 2 * 5 * 256;
  { k_red_a<<<nblk, GH_BLOCK, 0, s>>>(c->n, c->ncap, ma, c->type, c->epa, c->vel, part, c->red_tick,
                                      sums, c->rep_h); ++c->launches; }
  { k_red_b<<<nblk, GH_BLOCK, 0, s>>>(c->n, c->ncap, ma, c->type, c->vel, sums, part, c->red_tick,
                                      c->status, c->rep_h); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  GH_HIP(c, hipStreamSynchronize(s));
  *epot_ui = c->rep_h->epot;
  *ekin_ui = c->rep_h->ekin2 * 0.5;
  if (st) *st = c->rep_h->st;
  return 0;
}

int gh_launch_get(gh_ctx *c, double *x, double *v, double *F, double *e, bool status) {
  { k_get<<<nblocks(3 * c->n), GH_BLOCK, 0, c->stream>>>(
      c->n, c->ncap, make_wrap(c), c->inv, c->pos, c->vel, c->frc, c->epa, x, v, F, e, c->status,
      status ? c->rep_h : nullptr); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

int gh_launch_put3(gh_ctx *c, double *dst, const double *in) {
  { k_put3<<<nblocks(3 * c->n), GH_BLOCK, 0, c->stream>>>(c->n, c->ncap, c->inv, in, dst); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

int gh_launch_set_positions(gh_ctx *c, const double *x_dev, long long step) {
  { k_set_positions<<<nblocks(c->n), GH_BLOCK, 0, c->stream>>>(
      c->n, c->ncap, make_wrap(c), c->inv, x_dev, c->pos, c->xold, c->status,
      step); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

int gh_launch_wrap(gh_ctx *c) {
  { k_wrap<<<nblocks(c->n), GH_BLOCK, 0, c->stream>>>(c->n, make_wrap(c), c->pos); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

// Fill helper for host code (no hipMemset in code that may be captured).
int gh_fill_int(gh_ctx *c, int *p, int v, int n) {
  if (n <= 0) return 0;
  { k_fill_int<<<nblocks(n), GH_BLOCK, 0, c->stream>>>(p, v, n); ++c->launches; }
  GH_HIP(c, hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// gh_cluster_forces_static: gh_compute of one free cluster (no box: the
// O(N^2) verlet_self list and the SMA-TB passes above) from the caller's
// device arrays, every intermediate in one file-scope device array.  No
// device memory is allocated; the array lives as long as the process, one
// copy per device.  Calls that overlap on one device share it and race.
// ---------------------------------------------------------------------------
#define GH_STATIC_MAXN 2048  // atoms per call
#define GH_STATIC_CAP 160    // list row capacity (a free cluster's rows hold < 90)
#define GH_STATIC_MAXT 2     // atom types per call
namespace {
constexpr size_t al256(size_t b) { return (b + 255) / 256 * 256; }
constexpr size_t kSOffPos = al256(sizeof(GhStatus));
constexpr size_t kSOffList = kSOffPos + al256(sizeof(double4) * GH_STATIC_MAXN);
constexpr size_t kSOffNn = kSOffList + al256(sizeof(unsigned) * GH_STATIC_CAP * GH_STATIC_MAXN);
constexpr size_t kSOffXold = kSOffNn + al256(sizeof(int) * GH_STATIC_MAXN);
constexpr size_t kSOffRho = kSOffXold + al256(sizeof(double) * 3 * GH_STATIC_MAXN);
constexpr size_t kSOffTick = kSOffRho + al256(sizeof(double) * GH_STATIC_MAXN);
constexpr size_t kSOffPart = kSOffTick + 256;
constexpr size_t kSOffTb = kSOffPart + al256(sizeof(double) * 2 * GH_STATIC_MAXN);
constexpr size_t kScratchBytes = kSOffTb + al256(sizeof(TbDev) * GH_MAXT * GH_MAXT);

// the parameter blocks of up to GH_STATIC_MAXT types, by value
struct StaticTb {
  TbDev t[GH_STATIC_MAXT * GH_STATIC_MAXT];
};

// Re-arms the status for one build, stages positions (3n AoS -> double4)
// and writes the parameter table.  Every field the later kernels read is
// written here: nothing depends on an earlier call's contents.
__global__ __launch_bounds__(GH_BLOCK) void k_static_init(unsigned char *scr, int n, int nt,
                                                          const double *__restrict__ x,
                                                          StaticTb tb) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  GhStatus *st = reinterpret_cast<GhStatus *>(scr);
  if (i == 0) {
    disp2_clear(st, 0);
    disp2_clear(st, 1);
    st->force_rebuild = 1;
    st->rebuild = 0;
    st->overflow = 0;
    st->maxnn = 0;
    st->maxnn_tag = 0ull;
    st->nupd = 0;
    st->outside = 0;
    st->halt = 0;
    st->halt_step = 0;
    *reinterpret_cast<unsigned *>(scr + kSOffTick) = 0u;
  }
  TbDev *tbd = reinterpret_cast<TbDev *>(scr + kSOffTb);
  if (i < nt * nt) tbd[(i / nt) * GH_MAXT + i % nt] = tb.t[i];
  if (i < n) {
    double4 *pos = reinterpret_cast<double4 *>(scr + kSOffPos);
    pos[i] = make_double4(x[3 * i], x[3 * i + 1], x[3 * i + 2], 0.0);
  }
}
}  // namespace

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Device address of `scratch` on each device, taken once per device with
// that device current (the host-side name is only a stand-in).
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[64];

extern "C" int gh_cluster_forces_static(int device, int precision, int n, int nt,
                                        const double *x, const int *type, const double *A,
                                        const double *xi, const double *p, const double *q,
                                        const double *r0, const double *rci, const double *rce,
                                        double skin, double *F, double *e_atom, double *epot,
                                        int *status, void *stream) {
  if (device < 0 || device >= 64 || (precision != GH_FP64 && precision != GH_MIXED))
    return GH_EINVAL;
  if (n < 1 || n > GH_STATIC_MAXN || nt < 1 || nt > GH_STATIC_MAXT || !(skin >= 0.0))
    return GH_EINVAL;  // n <= GH_STATIC_MAXN atoms, nt <= GH_STATIC_MAXT types
  if (!x || !type || !A || !xi || !p || !q || !r0 || !rci || !rce || !F || !e_atom || !epot ||
      !status)
    return GH_EINVAL;
  int prev = 0;
  if (hipGetDevice(&prev) != hipSuccess || hipSetDevice(device) != hipSuccess) return GH_EHIP;
  int rc = 0;
  unsigned char *scr = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
      void *ptr = nullptr;
      if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) rc = GH_EHIP;
      else g_scratch_ptr[device] = ptr;
    }
    scr = static_cast<unsigned char *>(g_scratch_ptr[device]);
  }
  // parameter blocks (TB.F90:106-170) as gh_set_smatb and gh_upload_tb build them
  StaticTb tb;
  memset(&tb, 0, sizeof(tb));
  double rcut = 0.0;
  const GhTbPair t00{A[0], xi[0], p[0], q[0], r0[0], rci[0], rce[0], 0, 0, 0, 0, 0, 0};
  const double e0 = gh_tb_e0(&t00);
  for (int a = 0; a < nt && rc == 0; ++a)
    for (int b = 0; b < nt; ++b) {
      const int k = a * nt + b;
      if (!(r0[k] > 0) || !(rci[k] > 0) || !(rce[k] > rci[k])) rc = GH_EINVAL;
      GhTbPair t{A[k], xi[k], p[k], q[k], r0[k], rci[k], rce[k], 0, 0, 0, 0, 0, 0};
      gh_tb_coeffs(t);
      gh_tbdev_fill(t, e0, tb.t[k]);
      rcut = std::max(rcut, t.rce);
    }
  if (rc == 0) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    GhStatus *st = reinterpret_cast<GhStatus *>(scr);
    double4 *pos = reinterpret_cast<double4 *>(scr + kSOffPos);
    unsigned *list = reinterpret_cast<unsigned *>(scr + kSOffList);
    int *nn = reinterpret_cast<int *>(scr + kSOffNn);
    double *xold = reinterpret_cast<double *>(scr + kSOffXold);
    double *rho = reinterpret_cast<double *>(scr + kSOffRho);
    const TbDev *tbd = reinterpret_cast<const TbDev *>(scr + kSOffTb);
    const int nb = nblocks(n), nw = row_blocks(n, 64);
    const double L = 1e6, rl = rcut + skin;
    N2Build B;
    memset(&B, 0, sizeof(B));
    for (int d = 0; d < 3; ++d) {
      B.g.nc[d] = B.g.gn[d] = 1;
      B.g.L[d] = L;
      B.g.one_cell[d] = 1.0 / L;
    }
    B.g.ncell = 1;
    B.pos = pos;
    B.n = n;
    B.cap = GH_STATIC_CAP;
    B.ncap = GH_STATIC_MAXN;
    B.rl2 = rl * rl;
    B.nn = nn;
    B.list = list;
    B.xold = xold;
    RowArgs P;
    memset(&P, 0, sizeof(P));
    P.st = st;
    P.sa = StepArgs{0, skin, nullptr};
    P.inline_build = n <= 1024;
    P.pos = pos;
    P.type = type;
    P.nn = nn;
    P.list = list;
    P.n = n;
    P.cap = GH_STATIC_CAP;
    P.ncap = GH_STATIC_MAXN;
    P.nt = nt;
    for (int d = 0; d < 3; ++d) P.L[d] = L;
    P.tbd = tbd;
    P.rho = rho;
    P.e0 = e0;
    P.ev_ui = ghc::ev_ui();
    P.epa = e_atom;
    P.F_out = F;
    P.epot_out = epot;
    P.status_out = status;
    P.part = reinterpret_cast<double *>(scr + kSOffPart);
    P.ticket = reinterpret_cast<unsigned *>(scr + kSOffTick);
    const bool single = nt == 1;
    const FuseVV none{};
    k_static_init<<<std::max(nb, 1), GH_BLOCK, 0, s>>>(scr, n, nt, x, tb);
    if (n > 1024) k_build_n2<4><<<n2_blocks(n, 4), GH_BLOCK, 0, s>>>(st, B, skin, 0);
    if (precision == GH_MIXED) {
      if (single) {
        k_row_rho<true, true, 64><<<nw, GH_BLOCK, 0, s>>>(P, B, tb.t[0].f);
        k_row_force<true, true, 64, 3><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].f, none);
      } else {
        k_row_rho<true, false, 64><<<nw, GH_BLOCK, 0, s>>>(P, B, tb.t[0].f);
        k_row_force<true, false, 64, 3><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].f, none);
      }
    } else {
      if (single) {
        k_row_rho<false, true, 64><<<nw, GH_BLOCK, 0, s>>>(P, B, tb.t[0].d);
        k_row_force<false, true, 64, 3><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].d, none);
      } else {
        k_row_rho<false, false, 64><<<nw, GH_BLOCK, 0, s>>>(P, B, tb.t[0].d);
        k_row_force<false, false, 64, 3><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].d, none);
      }
    }
    if (hipGetLastError() != hipSuccess) rc = GH_EHIP;
  }
  (void)hipSetDevice(prev);
  return rc;
}
