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
// workgroup's max |x - x_old|^2 into GhStatus::maxdisp2 with one
// atomicMax (non-negative doubles order as their bit patterns); it runs over
// the steps since the last build and the first kernel of a rebuild sequence
// reads it (rebuild_due, rebuild_book).  State-changing kernels return at
// once while GhStatus::halt is set (raise_halt).
// ---------------------------------------------------------------------------
// Decision of the O(N^2) list mode (one thread).
__global__ void k_decide(GhStatus *st, double skin, long long step) {
  st->rebuild = !st->halt && rebuild_due(st, skin, step);
  rebuild_book(st);
}

struct GridArgs {
  int nc[3], gn[3], gofs[3], pbc[3];
  double L[3], one_cell[3];
  int ncell;
  int ghost;
};



// ---------------------------------------------------------------------------
// The O(N^2) list mode (free clusters, boxes of a few cells, masked pairs):
// a wavefront per atom, in the list build and in every pair pass.  These
// systems hold tens to a few thousand atoms: with one lane per atom a 201-atom
// cluster runs on four wavefronts whose lanes walk ~200 candidates or ~50
// neighbours one dependent load after another; with a wavefront per atom its
// row (rows are contiguous: entry k of atom i at i * cap + k) is one load and
// one round of pair terms.  201 Ag-Cu atoms, FP64: build 45 -> 5.1 us, density
// 32 -> 4.2, forces 41 -> 4.5.
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

template <int R>
__global__ __launch_bounds__(GH_BLOCK) void k_build_n2(GhStatus *st, N2Build B, long long step) {
  if (!st->rebuild) return;
  __shared__ int part[GH_BLOCK / 64];
  const int m = n2_rows<R>(B, n2_first<R>());
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    int wm = m;
    for (int w = 1; w < GH_BLOCK / 64; ++w) wm = max(wm, part[w]);
    if (wm > 0) atomicMax(&st->maxnn, wm);
    if (wm > B.cap) {
      st->overflow = 1;
      if (B.cap > 0) raise_halt(st, GH_HALT_OVERFLOW, step);  // cap 0: the sizing count
    }
  }
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

// A pair pass over one row: f(j, vx, vy, vz) for every listed pair, the
// wavefront's lanes 64 entries at a time.
struct N2Row {
  const double4 *pos;
  const unsigned *list;  // the atom's row
  int m;
};
template <class F>
__device__ __forceinline__ void n2_each(const N2Row &row, const double4 &pi, const ShiftLds &sh,
                                        F &&f) {
  for (int k = threadIdx.x & 63; k < row.m; k += 64) {
    const unsigned e = row.list[k];
    const int j = (int)(e & GH_JMASK), w = (int)(e >> 27);
    const double4 pj = row.pos[j];
    f(j, (pj.x - pi.x) + sh.x[w], (pj.y - pi.y) + sh.y[w], (pj.z - pi.z) + sh.z[w]);
  }
}

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

// SMA-TB pass 1 of one atom (smatb_preinteraction, TB.F90:367-455):
//   rho_i = sum_j [ r < rci ? xi^2 exp(-2q(r/r0-1)) : (b1 x^5 + b2 x^4 + b3 x^3)^2 ]
//   with x = r - rce and r > rce skipped.  The same value in every lane.
template <bool MIXED, bool SINGLE>
__device__ __forceinline__ double n2_rho(const N2Row &row, const double4 &pi, const ShiftLds &sh,
                                         const int *__restrict__ type, int ti,
                                         const TbForm<MIXED> *sp, const TbForm<MIXED> &p1) {
  double acc = 0.0;
  n2_each(row, pi, sh, [&](int j, double vx, double vy, double vz) {
    const TbForm<MIXED> &P = SINGLE ? p1 : sp[ti * GH_MAXT + type[j]];
    const double rd = fma(vx, vx, fma(vy, vy, vz * vz));
    if constexpr (MIXED) {
      float band;
      if (tb_rho_fx(P, rd, band)) acc += (double)band;
    } else {
      if (rd > P.rce2) return;
      double dr, ir;
      sqrt_rsq64(rd, dr, ir);
      acc += tb_band64(P, dr);
    }
  });
  return wave_total(acc);
}

// SMA-TB pass 2 of one atom (smatb_interact, TB.F90:457-586), full list,
// newton off:
//   r <= rci: repul = A e^{-p(r/r0-1)};
//             factor = 2 repul p/r0 - xi^2/2 e^{-2q(r/r0-1)} (2q/r0)(eb_i+eb_j)
//   rci < r <= rce: factor = P P' (eb_i+eb_j) - 2 R';  repul = R
//   F_i -= factor * vd / r  (vd = x_j - x_i), e_i = sum repul - sqrt(rho_i).
// eb is 1/sqrt(rho) (FP64) or its FP32 offset from e0 (mixed); f = {Fx, Fy,
// Fz, sum repul} in every lane.
template <bool MIXED, bool SINGLE, class EB>
__device__ __forceinline__ void n2_force(const N2Row &row, const double4 &pi, const ShiftLds &sh,
                                         const int *__restrict__ type, int ti,
                                         const TbForm<MIXED> *sp, const TbForm<MIXED> &p1,
                                         const EB *eb, EB ebi, double (&f)[4]) {
  f[0] = f[1] = f[2] = f[3] = 0.0;
  n2_each(row, pi, sh, [&](int j, double vx, double vy, double vz) {
    const TbForm<MIXED> &P = SINGLE ? p1 : sp[ti * GH_MAXT + type[j]];
    const double rd = fma(vx, vx, fma(vy, vy, vz * vz));
    double s, rep;
    if constexpr (MIXED) {
      float sf, repul;
      if (!tb_force_fx<true>(P, rd, ebi + eb[j], sf, repul)) return;
      s = (double)sf;
      rep = (double)repul;
    } else {
      if (rd > P.rce2) return;
      double dr, ir, factor;
      sqrt_rsq64(rd, dr, ir);
      tb_pair64(P, dr, ebi + eb[j], factor, rep);
      s = factor * ir;
    }
    f[0] = fma(-s, vx, f[0]);
    f[1] = fma(-s, vy, f[1]);
    f[2] = fma(-s, vz, f[2]);
    f[3] += rep;
  });
#pragma unroll
  for (int d = 0; d < 4; ++d) f[d] = wave_total(f[d]);
}

struct N2Pass {
  const double4 *pos;
  const int *type, *nn;
  const unsigned *list;
  int n, cap, ncap, nt;
  double L[3];
  const TbDev *tbd;
  double *rho, *eband;
  float *eband32;
  double e0, ev_ui;
  double *frc, *epa;
};

template <bool MIXED, bool SINGLE>
__global__ __launch_bounds__(GH_BLOCK) void k_n2_rho(N2Pass A, TbForm<MIXED> p1) {
  __shared__ ShiftLds sh;
  __shared__ TbForm<MIXED> sp[SINGLE ? 1 : GH_MAXT * GH_MAXT];
  load_shift(sh, A.L[0], A.L[1], A.L[2]);
  if (!SINGLE) load_params(sp, A.tbd, A.nt);
  __syncthreads();
  const int i = n2_first<1>();
  if (i >= A.n) return;
  const N2Row row{A.pos, A.list + (size_t)i * A.cap, A.nn[i]};
  const double rho = n2_rho<MIXED, SINGLE>(row, A.pos[i], sh, A.type, SINGLE ? 0 : A.type[i], sp, p1);
  if ((threadIdx.x & 63) == 0) {
    A.rho[i] = rho;
    const double eb = 1.0 / sqrt(rho);
    A.eband[i] = eb;
    A.eband32[i] = (float)(eb - A.e0);
  }
}

template <bool MIXED, bool SINGLE>
__global__ __launch_bounds__(GH_BLOCK) void k_n2_force(N2Pass A, TbForm<MIXED> p1) {
  __shared__ ShiftLds sh;
  __shared__ TbForm<MIXED> sp[SINGLE ? 1 : GH_MAXT * GH_MAXT];
  load_shift(sh, A.L[0], A.L[1], A.L[2]);
  if (!SINGLE) load_params(sp, A.tbd, A.nt);
  __syncthreads();
  const int i = n2_first<1>();
  if (i >= A.n) return;
  const N2Row row{A.pos, A.list + (size_t)i * A.cap, A.nn[i]};
  const double4 pi = A.pos[i];
  const int ti = SINGLE ? 0 : A.type[i];
  double f[4];
  if constexpr (MIXED) n2_force<true, SINGLE>(row, pi, sh, A.type, ti, sp, p1, A.eband32, A.eband32[i], f);
  else n2_force<false, SINGLE>(row, pi, sh, A.type, ti, sp, p1, A.eband, A.eband[i], f);
  const int lane = threadIdx.x & 63;
  if (lane < 3) A.frc[lane * A.ncap + i] = (lane == 0 ? f[0] : lane == 1 ? f[1] : f[2]) * A.ev_ui;
  else if (lane == 3) A.epa[i] = (f[3] - sqrt(A.rho[i])) * A.ev_ui;
}

// Pair potentials, full list, newton off: e_i += p/2; F_i -= f vd / r.
// POT: GH_POT_LJ (lj_interact, Pairs.F90:207-279: r^2 > rc^2 skipped; p =
// 4e(s6^2 - s6); f = e(48 s6 - 24) s6 / r) or a tabulated form per type pair
// (plj_interact, Pairs.F90:293-370; slj_interact, :403-493; wca_interact,
// :508-560; sm1_interact, :916-990).
template <bool MIXED, int POT>
__global__ __launch_bounds__(GH_BLOCK) void k_n2_pair(N2Pass A, const PljDev *__restrict__ pljd,
                                                      double eps, double sig2, double rc2) {
  constexpr bool TAB = POT != GH_POT_LJ;
  __shared__ ShiftLds sh;
  __shared__ PljDev pp[TAB ? GH_MAXT * GH_MAXT : 1];
  load_shift(sh, A.L[0], A.L[1], A.L[2]);
  if (TAB)
    for (int k = threadIdx.x; k < GH_MAXT * GH_MAXT; k += blockDim.x) pp[k] = pljd[k];
  __syncthreads();
  const int i = n2_first<1>();
  if (i >= A.n) return;
  const N2Row row{A.pos, A.list + (size_t)i * A.cap, A.nn[i]};
  const int ti = TAB ? A.type[i] : 0;
  double f[4] = {0.0, 0.0, 0.0, 0.0};
  n2_each(row, A.pos[i], sh, [&](int j, double vx, double vy, double vz) {
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
      p = 4.0 * eps * (s6 * s6 - s6);
      s = eps * fma(48.0, s6, -24.0) * s6 * ir2;
    }
    f[0] = fma(-s, vx, f[0]);
    f[1] = fma(-s, vy, f[1]);
    f[2] = fma(-s, vz, f[2]);
    f[3] += p;
  });
#pragma unroll
  for (int d = 0; d < 4; ++d) f[d] = wave_total(f[d]);
  const int lane = threadIdx.x & 63;
  if (lane < 3) A.frc[lane * A.ncap + i] = (lane == 0 ? f[0] : lane == 1 ? f[1] : f[2]) * A.ev_ui;
  else if (lane == 3) A.epa[i] = f[3] * 0.5 * A.ev_ui;
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
// Workgroup maximum of |x - x_old|^2 folded into the device-wide maximum with
// one atomicMax (no fence: the next kernel reads it).
__device__ __forceinline__ void disp_reduce(double d2, GhStatus *st, long long step) {
  __shared__ double part[GH_BLOCK / 64];
  d2 = wave_max(d2);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = d2;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < GH_BLOCK / 64; ++w) d2 = fmax(d2, part[w]);
    fold_disp2(st, d2, step);
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

// velocity_verlet_b of one step fused with velocity_verlet_a of the next
// (Integration.F90:1171-1186 then 1150-1169): the same operations in the same
// order as the two kernels, with a = F/m formed once.  The acceleration is
// not stored (stepa recomputes it; the last stepb of a run stores it).
__global__ __launch_bounds__(GH_BLOCK) void k_vv_ba(
    int n, int ncap, double dt, MassArgs ma,
    const int *__restrict__ type, double4 *__restrict__ pos, double *__restrict__ vel,
    const double *__restrict__ frc, const double *__restrict__ xold, GhStatus *st,
    long long step) {
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
      const double v = vel[d * ncap + i] + acel_dv * a;  // stepb
      x[d] = x[d] + dt * v + acel_dx * a;                // stepa
      vel[d * ncap + i] = v + acel_dv * a;
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

struct ErmakArgs {
  double c0, c1, c2, sdr, sdv, crv1, crv2, skt, dt;
  int philox;
  unsigned long long seed;
  long long step;
};

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
// most: each arrival is a fence.)
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
  if (grid_sum_dd<1>(v, e, part, ticket) && threadIdx.x == 0) {
    rep->ekin2 = v[0];
    rep->st = *st;
  }
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
  if (k == 0 && rep) rep->st = *st;
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

__global__ void k_wrap_rebuild(const GhStatus *st, int n, WrapArgs wa,
                               double4 *__restrict__ pos) {
  if (!st->rebuild) return;
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
                 reinterpret_cast<unsigned *>(c->list), c->xold, c->orig,
                 c->masked ? c->mfeel : nullptr, c->masked ? c->mfelt : nullptr};
}

N2Pass make_n2_pass(const gh_ctx *c) {
  return N2Pass{c->pos, c->type, c->nn, reinterpret_cast<const unsigned *>(c->list),
                c->n, c->cap, c->ncap, c->nt, {c->L[0], c->L[1], c->L[2]}, c->tbd,
                c->rho, c->eband, c->eband32, c->tb_e0, ghc::ev_ui(), c->frc, c->epa};
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
// Every kernel of the rebuild reads the device flag set by k_decide, so the
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

int gh_launch_rebuild(gh_ctx *c, bool force) {
  hipStream_t s = c->stream;
  if (force) GH_TRY(gh_request_rebuild(c));
  const int n = c->n, nb = nblocks(n);
  if (c->list_mode == 1) return gh_launch_rebuild_cells(c);  // decides in its first kernels
  { k_decide<<<1, 1, 0, s>>>(c->status, c->skin, c->step); ++c->launches; }
  if (c->list_mode == 0 && c->boxed && (c->pbc[0] || c->pbc[1] || c->pbc[2]))
    { k_wrap_rebuild<<<nb, GH_BLOCK, 0, s>>>(c->status, n, make_wrap(c), c->pos); ++c->launches; }
  const N2Build B = make_n2_build(c);
  // rows per wavefront: one where the atoms do not fill the chip's wavefront
  // slots anyway, several where every wavefront reads all positions (32 n^2
  // bytes through the caches: 130 MB at 2,048 atoms, 33 MB with four rows)
  if (n <= 1024) k_build_n2<1><<<n2_blocks(n, 1), GH_BLOCK, 0, s>>>(c->status, B, c->step);
  else if (n <= 8192) k_build_n2<4><<<n2_blocks(n, 4), GH_BLOCK, 0, s>>>(c->status, B, c->step);
  else k_build_n2<8><<<n2_blocks(n, 8), GH_BLOCK, 0, s>>>(c->status, B, c->step);
  ++c->launches;
  GH_HIP(c, hipGetLastError());
  return 0;
}

bool gh_can_fuse_vv(const gh_ctx *c) {
  return c->list_mode == 1 && c->integ == GH_INT_VV &&
         (c->pot == GH_POT_SMATB || c->pot == GH_POT_LJ || gh_is_table_pot(c->pot));
}

int gh_launch_forces(gh_ctx *c, hipEvent_t mid, bool fuse_vv) {
  if (c->list_mode == 1) return gh_launch_forces_tiled(c, mid, fuse_vv);
  if (fuse_vv) return gh_fail(c, GH_ESTATE, "fused integration needs the tiled path");
  hipStream_t s = c->stream;
  const int nb = n2_blocks(c->n, 1);
  const bool single = c->nt == 1, mixed = c->precision == GH_MIXED;
  const N2Pass A = make_n2_pass(c);
  if (c->pot == GH_POT_SMATB) {
#define N2_TB(KERNEL)                                                                       \
  do {                                                                                      \
    if (mixed) {                                                                            \
      if (single) KERNEL<true, true><<<nb, GH_BLOCK, 0, s>>>(A, c->tbf_a0);                  \
      else KERNEL<true, false><<<nb, GH_BLOCK, 0, s>>>(A, c->tbf_a0);                        \
    } else {                                                                                \
      if (single) KERNEL<false, true><<<nb, GH_BLOCK, 0, s>>>(A, c->tb64_0);                 \
      else KERNEL<false, false><<<nb, GH_BLOCK, 0, s>>>(A, c->tb64_0);                       \
    }                                                                                       \
    ++c->launches;                                                                          \
  } while (0)
    N2_TB(k_n2_rho);
    if (mid) GH_HIP(c, hipEventRecord(mid, s));
    N2_TB(k_n2_force);
#undef N2_TB
  } else if (c->pot == GH_POT_LJ || gh_is_table_pot(c->pot)) {
    if (mid) GH_HIP(c, hipEventRecord(mid, s));
    const double rc2 = c->lj_rc * c->lj_rc, sig2 = c->lj_sigma * c->lj_sigma;
#define N2_PAIR(PT)                                                                         \
  do {                                                                                      \
    if (mixed) k_n2_pair<true, PT><<<nb, GH_BLOCK, 0, s>>>(A, c->pljd, c->lj_eps, sig2, rc2); \
    else k_n2_pair<false, PT><<<nb, GH_BLOCK, 0, s>>>(A, c->pljd, c->lj_eps, sig2, rc2);      \
    ++c->launches;                                                                          \
  } while (0)
    switch (c->pot) {
      case GH_POT_SLJ: N2_PAIR(GH_POT_SLJ); break;
      case GH_POT_WCA: N2_PAIR(GH_POT_WCA); break;
      case GH_POT_SM1: N2_PAIR(GH_POT_SM1); break;
      case GH_POT_PLJ: N2_PAIR(GH_POT_PLJ); break;
      default: N2_PAIR(GH_POT_LJ);
    }
#undef N2_PAIR
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

int gh_launch_vv_ba(gh_ctx *c) {
  { k_vv_ba<<<nblocks(c->n), GH_BLOCK, 0, c->stream>>>(c->n, c->ncap, c->dt,
                                                     make_mass(c), c->type, c->pos, c->vel,
                                                     c->frc, c->xold, c->status,
                                                     c->step); ++c->launches; }
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

int gh_launch_set_positions(gh_ctx *c, const double *x_dev) {
  { k_set_positions<<<nblocks(c->n), GH_BLOCK, 0, c->stream>>>(
      c->n, c->ncap, make_wrap(c), c->inv, x_dev, c->pos, c->xold, c->status,
      c->step); ++c->launches; }
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
constexpr size_t kSOffEband = kSOffRho + al256(sizeof(double) * GH_STATIC_MAXN);
constexpr size_t kSOffEb32 = kSOffEband + al256(sizeof(double) * GH_STATIC_MAXN);
constexpr size_t kSOffFrc = kSOffEb32 + al256(sizeof(float) * GH_STATIC_MAXN);
constexpr size_t kSOffTb = kSOffFrc + al256(sizeof(double) * 3 * GH_STATIC_MAXN);
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
    st->maxdisp2[0].bits = st->maxdisp2[1].bits = 0ull;
    st->rebuild = 1;
    st->overflow = 0;
    st->maxnn = 0;
    st->outside = 0;
    st->halt = 0;
    st->halt_step = 0;
  }
  TbDev *tbd = reinterpret_cast<TbDev *>(scr + kSOffTb);
  if (i < nt * nt) tbd[(i / nt) * GH_MAXT + i % nt] = tb.t[i];
  if (i < n) {
    double4 *pos = reinterpret_cast<double4 *>(scr + kSOffPos);
    pos[i] = make_double4(x[3 * i], x[3 * i + 1], x[3 * i + 2], 0.0);
  }
}

// Forces to the caller's AoS layout; one workgroup then sums the energies
// (compensated) and reports the build's row overflow.
__global__ __launch_bounds__(GH_BLOCK) void k_static_out(const unsigned char *scr, int n,
                                                         double *__restrict__ F) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double *frc = reinterpret_cast<const double *>(scr + kSOffFrc);
#pragma unroll
  for (int d = 0; d < 3; ++d) F[3 * i + d] = frc[d * GH_STATIC_MAXN + i];
}
__global__ __launch_bounds__(GH_BLOCK) void k_static_sum(const unsigned char *scr, int n,
                                                         const double *__restrict__ e,
                                                         double *__restrict__ epot,
                                                         int *__restrict__ status) {
  double v[1] = {0.0}, c[1] = {0.0};
  for (int i = threadIdx.x; i < n; i += blockDim.x) dd_add(v[0], c[0], e[i]);
  block_sum_dd<1>(v, c);
  if (threadIdx.x == 0) {
    *epot = v[0] + c[0];
    const GhStatus *st = reinterpret_cast<const GhStatus *>(scr);
    *status = st->overflow ? GH_EOVERFLOW : 0;
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
    double *eband = reinterpret_cast<double *>(scr + kSOffEband);
    float *eb32 = reinterpret_cast<float *>(scr + kSOffEb32);
    double *frc = reinterpret_cast<double *>(scr + kSOffFrc);
    const TbDev *tbd = reinterpret_cast<const TbDev *>(scr + kSOffTb);
    const int nb = nblocks(n), nw = n2_blocks(n, 1);
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
    const N2Pass P{pos, type, nn, list, n, GH_STATIC_CAP, GH_STATIC_MAXN, nt, {L, L, L}, tbd,
                   rho, eband, eb32, e0, ghc::ev_ui(), frc, e_atom};
    const bool single = nt == 1;
    k_static_init<<<std::max(nb, 1), GH_BLOCK, 0, s>>>(scr, n, nt, x, tb);
    if (n <= 1024) k_build_n2<1><<<nw, GH_BLOCK, 0, s>>>(st, B, 0);
    else k_build_n2<4><<<n2_blocks(n, 4), GH_BLOCK, 0, s>>>(st, B, 0);
    if (precision == GH_MIXED) {
      if (single) {
        k_n2_rho<true, true><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].f);
        k_n2_force<true, true><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].f);
      } else {
        k_n2_rho<true, false><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].f);
        k_n2_force<true, false><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].f);
      }
    } else {
      if (single) {
        k_n2_rho<false, true><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].d);
        k_n2_force<false, true><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].d);
      } else {
        k_n2_rho<false, false><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].d);
        k_n2_force<false, false><<<nw, GH_BLOCK, 0, s>>>(P, tb.t[0].d);
      }
    }
    k_static_out<<<nb, GH_BLOCK, 0, s>>>(scr, n, F);
    k_static_sum<<<1, GH_BLOCK, 0, s>>>(scr, n, e_atom, epot, status);
    if (hipGetLastError() != hipSuccess) rc = GH_EHIP;
  }
  (void)hipSetDevice(prev);
  return rc;
}
