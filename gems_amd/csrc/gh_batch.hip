// Batched free clusters: many independent unboxed systems on one device.
//
// GEMS has no batching (one system per process, replica exchange over MPI
// ranks, src/ReplicaExchange.f90:27-151); per system the work is the same hot
// path: the O(N^2) verlet_self list (Neighbour.F90:676-759, rd <= rl^2 kept),
// the two SMA-TB passes (TB.F90:367-586) and the Ermak update
// (Integration.F90:963-1031).  A system's atoms are contiguous; all state is
// FP64 in HBM (SoA with stride ld).
//
// Forces and most Langevin dynamics run over the atoms of all systems at once, 16
// or 8 lanes per atom, two launches per step (density; forces with the update to
// the next step): a step then costs the chip's throughput, not the time one
// compute unit needs for the largest cluster (a workgroup per system took 170
// us per step for 2,000 atoms while the compute units of the smaller systems
// idled; 128 Ag-Cu clusters of 38..2000 atoms, mixed: 206 -> 68 us per step;
// 16 clusters of 38..600 96 -> 18).  Mixed batches that fill the chip with a
// workgroup per system all the same, or whose systems are tiny, take all Langevin
// steps in one launch (k_batch_langevin, by batch_staged), and FIRE, whose every
// iteration needs sums over each system, all iterations (largest system first).
//
// Neighbour rows: cap 16-bit indices local to the system, contiguous per
// atom; the pairs inside the inner bound at build time fill a row from its
// front, the others from its back, so the 16 lanes of an atom take one branch
// of the pair function per round.
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <numeric>
#include <type_traits>
#include <vector>

#include "gh_device.h"

#define GH_FBS 256  // smallest workgroup of the FIRE kernel

namespace {
struct FireState;
}
struct gh_batch {
  int device = 0;
  hipStream_t stream = nullptr;
  int precision = GH_FP64;
  std::string err;
  int nsys = 0, ntot = 0, ld = 0;
  int nt = 1;
  int types = 1;  // one past the largest type of an atom
  double mass_t[GH_MAXT] = {1, 1, 1, 1, 1, 1, 1, 1};
  GhTbPair tb[GH_MAXT * GH_MAXT];
  bool have_pot = false;
  double rcut = 0.0, skin = 1.0;
  int cap = 0;
  int cap_req = 0;  // row capacity asked for by the last overflow
  long long step = 0;
  bool lists_valid = false;
  bool forces_valid = false;
  std::vector<int> off_h, order_h;
  std::vector<double> T_h, epot_h;
  // device
  int *off = nullptr, *order = nullptr, *type = nullptr, *flags = nullptr;
  unsigned *nn = nullptr;
  int *sysof = nullptr, *a0of = nullptr;   // each atom's system and that system's first atom
  GhLine *dmax = nullptr;                  // [2][nsys] largest |x - x_old|^2, by step parity
  double4 *pos = nullptr, *pos_next = nullptr;  // x, y, z, type
  double4 *pk = nullptr;  // what the force pass reads of a neighbour (density pass)
  double *vel = nullptr, *acc = nullptr, *frc = nullptr, *e = nullptr, *rho = nullptr,
         *xold = nullptr, *T = nullptr, *out = nullptr, *scale = nullptr;
  FireState *fst = nullptr;         // [nsys] between the FIRE launches
  unsigned short *list = nullptr;
  TbDev *tbd = nullptr;
  TbF *tbf = nullptr;
  TbDev tbd0;           // host copies of tbd[0] and tbf[0] (one-type kernel arguments)
  TbF tbf0;
  double tb_e0 = 0.0;
  int nst = 0;   // LDS staging slots per workgroup (largest system + sentinel)
  // systems of one lane per atom and of four run beside one another (launch_split)
  hipStream_t stream2 = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
};

namespace {
using namespace ghd;

struct BatchArgs {
  const int *off, *order, *type, *sysof, *a0of;
  int first;  // FIRE: this launch's workgroup b works on system order[first + b]
  int nsys, ntot;
  double4 *pos, *pos_next, *pk;
  double *vel, *acc, *frc, *e, *rho, *xold;
  unsigned *nn;  // row lengths: pairs at the front | pairs at the back << 16
  unsigned short *list;
  int cap, ld;
  const TbDev *tbd;
  const TbF *tbf;
  int nt;
  double om[GH_MAXT], osm[GH_MAXT];
  double rl2, near2;  // build: list cut, inner-branch bound
  // the same in steps of 2^-GH_BFXK A, squared: surely outside the cut above
  // hi2q, surely inside below lo2q; within band2q of near2q neither side is sure
  float hi2q, lo2q, near2q, band2q;
  int nst;            // LDS staging slots (largest system + sentinel); 0 = none
  double ev_ui;
  const double *T;
  GhLine *dmax;
  double *out;  // per system: [0] epot ui, [1] ekin ui, [2] rebuilds, [3] fmax eV/A,
                // [4] iterations, [5] converged
  int *flags;   // [0] list overflow, [1] longest row asked for past the capacity
  double e0;    // eband reference of the FP32 pair forms
};

#define OUTW 6

// BS threads; 0: as launched (256, 512 or 1024).
template <int BS>
struct BlockRed {
  double v[BS ? BS / 64 : 16][8];  // up to 8 values per reduction
};
// Runs f(w) for every wavefront of the workgroup, four at a time (fully
// unrolled, 16 wavefronts x 8 values would all sit in registers).
template <int BS, class F>
__device__ __forceinline__ void each_wave(F &&f) {
  if constexpr (BS > 0) {
#pragma unroll 4
    for (int w = 0; w < BS / 64; ++w) f(w);
  } else {
    for (int w0 = 0; w0 < (int)(blockDim.x >> 6); w0 += 4)
#pragma unroll
      for (int u = 0; u < 4; ++u) f(w0 + u);
  }
}

// Block-wide sums of NV values; the result is returned to every thread.
template <int BS, int NV>
__device__ __forceinline__ void bsum(BlockRed<BS> &R, double (&v)[NV]) {
  static_assert(NV <= 8, "BlockRed holds 8 values per wave");
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) R.v[threadIdx.x >> 6][k] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double s = 0.0;
    each_wave<BS>([&](int w) { s += R.v[w][k]; });
    v[k] = s;
  }
  __syncthreads();
}

// Block-wide sums of the first NV values of v and the maximum of m, returned
// to every thread; two barriers, the second before the next use of R.
template <int BS, int NV>
__device__ __forceinline__ void bred(BlockRed<BS> &R, double (&v)[3], double &m) {
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_total(v[k]);
  m = wave_top(m);
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) R.v[threadIdx.x >> 6][k] = v[k];
    R.v[threadIdx.x >> 6][3] = m;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = 0.0;
  each_wave<BS>([&](int w) {
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] += R.v[w][k];
    m = fmax(m, R.v[w][3]);
  });
  __syncthreads();
}

// Lane groups of G = 16, 8, 4 or 1: the group's bits of a wave mask, and sums
// over a group in every lane of it.
template <int G>
__device__ __forceinline__ unsigned group_bits(unsigned long long m) {
  return (unsigned)(m >> (threadIdx.x & 63 & ~(G - 1))) & ((1u << G) - 1);
}
template <int G>
__device__ __forceinline__ double group_total(double v) {
  if (G >= 4) v += dpp64<0xB1>(v);    // quad_perm [1,0,3,2]
  if (G >= 4) v += dpp64<0x4E>(v);    // quad_perm [2,3,0,1]
  if (G >= 8) v += dpp64<0x141>(v);   // row_half_mirror
  if (G == 16) v += dpp64<0x140>(v);  // row_mirror
  return v;
}

// A row's lengths and its atom's build position, by the row's 16 lanes.
__device__ __forceinline__ void row_end(const BatchArgs &B, bool on, int i, int m0, int m1,
                                        const double4 &pi) {
  const int sub = threadIdx.x & 15, cap = B.cap;
  if (!on) return;
  if (sub == 0) {
    if (m0 + m1 > cap) {
      B.flags[0] = 1;
      atomicMax(&B.flags[1], m0 + m1);
    }
    const int f = min(m0, cap);
    B.nn[i] = (unsigned)f | ((unsigned)min(m1, cap - f) << 16);
  }
  if (sub < 3) B.xold[sub * B.ld + i] = sub == 0 ? pi.x : sub == 1 ? pi.y : pi.z;
}

// The row of atom k of a system (verlet_self, Neighbour.F90:676-759: all
// pairs with rd <= rl^2, itself excluded; rd rounded as the reference's
// dot_product) by 16 lanes, 64 candidates per round; inner pairs fill it from
// the front, the others from the back.  `on` is the same in the 16 lanes;
// every lane of the wavefront calls it.
__device__ __forceinline__ void batch_row(const BatchArgs &B, bool on, int a0, int n, int k) {
  const int sub = threadIdx.x & 15, i = a0 + k, cap = B.cap;
  const unsigned below = (1u << sub) - 1;
  const double4 pi = B.pos[i];
  unsigned short *row = B.list + (size_t)i * cap;
  int m0 = 0, m1 = 0;
  for (int j0 = 0; __any(on && j0 < n); j0 += 64) {
    double4 p[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) p[u] = B.pos[a0 + min(j0 + 16 * u + sub, n - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + 16 * u + sub;
      const double rd = dist2_rn(p[u].x - pi.x, p[u].y - pi.y, p[u].z - pi.z);
      const bool keep = on && j < n && j != k && rd <= B.rl2, near = rd < B.near2;
      const unsigned b0 = group_bits<16>(__ballot(keep && near));
      const unsigned b1 = group_bits<16>(__ballot(keep && !near));
      const int d = near ? m0 + __popc(b0 & below) : cap - 1 - (m1 + __popc(b1 & below));
      if (keep && d >= 0 && d < cap) row[d] = (unsigned short)j;
      m0 += __popc(b0);
      m1 += __popc(b1);
    }
  }
  row_end(B, on, i, m0, m1, pi);
}

// The row of atom i: its ends and, for 16 and 8 lanes, the first 16 pairs of
// the front and the first 48 of the back, which are nearly always all of them.
// These loads need nothing but the atom's number, so they are in flight
// together with the atom's own data.
template <int G>
struct RowHead {
  static constexpr int NF = G >= 8 ? 16 / G : 0, NB = G >= 8 ? 48 / G : 0;  // entries of a lane
  const unsigned short *row;
  int m0, m1, s[G >= 8 ? NF + NB : 1];
};
template <int G>
__device__ __forceinline__ RowHead<G> row_head(const BatchArgs &B, int i, bool on) {
  RowHead<G> r;
  r.row = B.list + (size_t)i * B.cap;
  const unsigned w = on ? B.nn[i] : 0u;
  r.m0 = (int)(w & 0xFFFFu);
  r.m1 = (int)(w >> 16);
  if constexpr (G >= 8) {
    const int sub = threadIdx.x & (G - 1);
#pragma unroll
    for (int u = 0; u < r.NF; ++u) r.s[u] = r.row[min(sub + G * u, B.cap - 1)];
#pragma unroll
    for (int u = 0; u < r.NB; ++u) r.s[r.NF + u] = r.row[max(B.cap - 1 - (sub + G * u), 0)];
  }
  return r;
}
// Runs f(u) for every pair of a row after load(u, s), s the neighbour's index
// in the system, four payloads in flight.  16 and 8 lanes: lane sub takes
// entries sub, sub + G, ... of the front, then of the back.  4 lanes and one:
// lane sub takes the quads sub, sub + G, ... (one 8-byte load each, the next one
// in flight while one is used).
template <int G, class LOAD, class F>
__device__ __forceinline__ void batch_each(const BatchArgs &B, const RowHead<G> &r, LOAD &&load,
                                           F &&f) {
  const int sub = threadIdx.x & (G - 1);
  if constexpr (G >= 8) {
#pragma unroll
    for (int c = 0; c < r.NF + r.NB; c += 4) {
      bool on[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int e = c + u;
        on[u] = e < r.NF ? sub + G * e < r.m0 : sub + G * (e - r.NF) < r.m1;
        if (on[u]) load(u, r.s[e]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (on[u]) f(u);
    }
    auto run = [&](int k0, int m, const unsigned short *first, int dir) {
      for (; k0 < m; k0 += 4 * G) {
        int s[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) s[u] = first[dir * min(k0 + u * G, m - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u) load(u, s[u]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (k0 + u * G < m) f(u);
      }
    };
    run(sub + 16, r.m0, r.row, 1);
    run(sub + 48, r.m1, r.row + (B.cap - 1), -1);
  } else {
    static_assert(G == 4 || G == 1, "16, 8, 4 lanes per atom or one");
    // virtual quads: the front's, padded to whole rounds of the lanes, then the
    // back's
    const unsigned long long *qf = reinterpret_cast<const unsigned long long *>(r.row);
    const int nf = (r.m0 + 4 * G - 1) / (4 * G) * G, nq = nf + ((r.m1 + 3) >> 2),
              last = (B.cap >> 2) - 1;
    auto quad = [&](int v) { return v < nf ? qf[min(v, last)] : qf[max(last - (v - nf), 0)]; };
    unsigned long long w = nq > 0 ? quad(sub) : 0ull;
    for (int v = sub; v < nq; v += G) {
      const unsigned long long nw = quad(min(v + G, nq));
      const bool front = v < nf;
      const int k0 = 4 * (front ? v : v - nf), m = front ? r.m0 : r.m1;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        load(u, k0 + u < m ? GH_QSLOT(w, front ? u : 3 - u) : 0);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (k0 + u < m) f(u);
      w = nw;
    }
  }
}

// One SMA-TB form of the passes.  FP64: Tb64.  Mixed: the FP32 forms on
// positions quantised to 2^-GH_BFXK A about the system's first atom (QUANT:
// pair vectors are then exact differences of integers below 2^53, held in
// FP64) with TbF in that unit, or on FP64 positions with TbF in Angstrom
// (systems whose staging does not fit LDS in the FIRE kernel; one rule for
// all kernels, so a system's forces do not depend on the kernel).
template <bool MIXED>
using BForm = typename std::conditional<MIXED, TbF, Tb64>::type;

template <bool QUANT>
__device__ __forceinline__ double bq(double p, double o) {
  return QUANT ? rint((p - o) * GH_BFXS) : p;
}

template <bool MIXED, bool SINGLE>
struct BTable {
  BForm<MIXED> t[SINGLE ? 1 : GH_MAXT * GH_MAXT];
};
template <bool MIXED, bool QUANT, bool SINGLE>
__device__ __forceinline__ void load_table(BTable<MIXED, SINGLE> &T, const BatchArgs &B) {
  if (SINGLE) return;
  for (int k = threadIdx.x; k < GH_MAXT * GH_MAXT; k += blockDim.x)
    if (k / GH_MAXT < B.nt && k % GH_MAXT < B.nt) {
      if constexpr (!MIXED) T.t[k] = B.tbd[k].d;
      else if constexpr (QUANT) T.t[k] = B.tbf[k];
      else T.t[k] = B.tbd[k].f;
    }
  __syncthreads();
}

// What the force pass reads of an atom: its position (quantised, QUANT), and
// 1/sqrt(rho) (FP64) or its FP32 offset and the type (mixed) in w.
template <bool MIXED>
__device__ __forceinline__ double pk_w(double eb, double e0, int t) {
  if (!MIXED) return eb;
  return __hiloint2double(t, __float_as_int((float)(eb - e0)));
}

// Density of atom i (smatb_preinteraction, TB.F90:367-455) by G lanes, stored
// with its pack.  Positions from global memory (a system's are cached).
template <bool MIXED, bool QUANT, bool SINGLE, int G>
__device__ __forceinline__ void batch_rho(const BatchArgs &B, const BTable<MIXED, SINGLE> &T,
                                          const BForm<MIXED> &p1, int a0, int i, bool on,
                                          const RowHead<G> &row) {
  const double4 o = QUANT ? B.pos[a0] : make_double4(0, 0, 0, 0);
  const double4 pi = B.pos[i];
  const double xi = bq<QUANT>(pi.x, o.x), yi = bq<QUANT>(pi.y, o.y), zi = bq<QUANT>(pi.z, o.z);
  const int ti = SINGLE ? 0 : (int)pi.w;
  double acc = 0.0;
  double4 p[4];
  batch_each<G>(
      B, row, [&](int u, int s) { p[u] = B.pos[a0 + s]; },
      [&](int u) {
        const double vx = bq<QUANT>(p[u].x, o.x) - xi, vy = bq<QUANT>(p[u].y, o.y) - yi,
                     vz = bq<QUANT>(p[u].z, o.z) - zi;
        const double rd = fma(vx, vx, fma(vy, vy, vz * vz));
        const BForm<MIXED> &P = SINGLE ? p1 : T.t[ti * GH_MAXT + (int)p[u].w];
        if constexpr (MIXED) {
          float band;
          if (tb_rho_fx(P, rd, band)) acc += (double)band;
        } else if (rd <= P.rce2) {
          double dr, ir;
          sqrt_rsq64(rd, dr, ir);
          acc += tb_band64(P, dr);
        }
      });
  acc = group_total<G>(acc);
  if (on && (threadIdx.x & (G - 1)) == 0) {
    B.rho[i] = acc;
    B.pk[i] = make_double4(xi, yi, zi, pk_w<MIXED>(1.0 / sqrt(acc), B.e0, ti));
  }
}

// Forces and repulsion of atom i (smatb_interact, TB.F90:457-586) by G lanes:
// f = {Fx, Fy, Fz, sum of repulsions} (eV units) in each.
template <bool MIXED, bool SINGLE, int G, bool ENERGY = true>
__device__ __forceinline__ void batch_force(const BatchArgs &B, const BTable<MIXED, SINGLE> &T,
                                            const BForm<MIXED> &p1, int a0, int i,
                                            const RowHead<G> &row, double (&f)[4]) {
  const double4 pi = B.pk[i];
  const int ti = SINGLE ? 0 : MIXED ? __double2hiint(pi.w) : B.type[i];
  f[0] = f[1] = f[2] = f[3] = 0.0;
  double4 p[4];
  int t[4];
  batch_each<G>(
      B, row,
      [&](int u, int s) {
        p[u] = B.pk[a0 + s];
        if (!MIXED && !SINGLE) t[u] = B.type[a0 + s];
      },
      [&](int u) {
        const double vx = p[u].x - pi.x, vy = p[u].y - pi.y, vz = p[u].z - pi.z;
        const double rd = fma(vx, vx, fma(vy, vy, vz * vz));
        const int tj = SINGLE ? 0 : MIXED ? __double2hiint(p[u].w) : t[u];
        const BForm<MIXED> &P = SINGLE ? p1 : T.t[ti * GH_MAXT + tj];
        double s, rep;
        if constexpr (MIXED) {
          float sf, repul;
          if (!tb_force_fx<ENERGY>(P, rd,
                                   __int_as_float(__double2loint(pi.w)) +
                                       __int_as_float(__double2loint(p[u].w)),
                                   sf, repul))
            return;
          s = (double)sf;  // factor / r per unit of the pair vector
          if (ENERGY) rep = (double)repul;
        } else {
          if (!(rd <= P.rce2)) return;
          double dr, ir, factor;
          sqrt_rsq64(rd, dr, ir);
          tb_pair64(P, dr, pi.w + p[u].w, factor, rep);
          s = factor * ir;
        }
        f[0] = fma(-s, vx, f[0]);
        f[1] = fma(-s, vy, f[1]);
        f[2] = fma(-s, vz, f[2]);
        if (ENERGY) f[3] += rep;
      });
#pragma unroll
  for (int d = 0; d < (ENERGY ? 4 : 3); ++d) f[d] = group_total<G>(f[d]);
}

// ---------------------------------------------------------------------------
// Forces and Langevin steps over all systems: 16 lanes per atom.  What bounds
// a step is the vector issue of the pair terms and, for small batches, the
// two launches.
// ---------------------------------------------------------------------------
#define GH_BWG 256
// Step `par` (parity): builds the rows of the systems whose atoms have moved
// past the skin (`always`: of every system), then the densities.
template <bool MIXED, bool QUANT, bool SINGLE, int G>
__global__ __launch_bounds__(GH_BWG) void k_batch_rho(BatchArgs B, BForm<MIXED> p1, double skin,
                                                      int par, int always) {
  __shared__ BTable<MIXED, SINGLE> T;
  load_table<MIXED, QUANT, SINGLE>(T, B);
  const int i0 = (int)(blockIdx.x * GH_BWG + threadIdx.x) / G;
  const bool live = i0 < B.ntot;
  const int i = min(i0, B.ntot - 1), sub = threadIdx.x & (G - 1);
  const int s = B.sysof[i], a0 = B.a0of[i];
  RowHead<G> row = row_head<G>(B, i, live);
  const double d2 = __longlong_as_double((long long)B.dmax[par * B.nsys + s].bits);
  const bool due = live && (always || 2.0 * sqrt(d2) > skin);
  if (live && i == a0 && sub == 0) {
    // the next step's maximum starts from nothing (its writer is the force pass)
    B.dmax[(par ^ 1) * B.nsys + s].bits = 0ull;
    if (due && !always) B.out[s * OUTW + 2] += 1.0;
  }
  if (__any(due)) {
    // 16 lanes build the rows of their 16 / G atoms one after the other
#pragma unroll
    for (int h = 0; h < 16 / G; ++h) {
      const int src = (int)(threadIdx.x & 63 & ~15) + h * G;
      const int ih = __shfl(i, src, 64), sh = __shfl(s, src, 64);
      const bool on = __shfl((int)due, src, 64) != 0;
      const int b0 = B.off[sh];
      batch_row(B, on, b0, B.off[sh + 1] - b0, ih - b0);
    }
    __threadfence_block();  // the wavefront reads the rows its own lanes wrote
    row = row_head<G>(B, i, live);
  }
  batch_rho<MIXED, QUANT, SINGLE, G>(B, T, p1, a0, i, live, row);
}

struct ErmakC {
  double c0, c1, c2, sdr, sdv, crv1, crv2, dt, kB_ui;
};

// The workgroup's displacements folded into their systems' maxima: one atomic
// where its atoms share a system, one per atom otherwise.  Each maximum has a
// cache line of its own (128 of them on eight lines, one atomic per
// wavefront: 66 us per step more at 67,896 atoms).  d2: the same in a group's
// lanes; all threads call it.
template <int G>
__device__ __forceinline__ void fold_sys_disp2(const BatchArgs &B, double d2, int s, bool live,
                                               int par) {
  __shared__ double part[GH_BWG / 64];
  __shared__ int same[2];
  if (threadIdx.x == 0) same[0] = s;
  if (threadIdx.x == GH_BWG - 1) same[1] = s;
  d2 = live ? d2 : 0.0;
  const double w = wave_max(d2);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = w;
  __syncthreads();
  GhLine *dst = B.dmax + (size_t)par * B.nsys;
  if (same[0] == same[1]) {  // systems are contiguous
    if (threadIdx.x == 0) {
      double m = part[0];
      for (int k = 1; k < GH_BWG / 64; ++k) m = fmax(m, part[k]);
      atomicMax(&dst[s].bits, (unsigned long long)__double_as_longlong(m));
    }
  } else if (live && (threadIdx.x & (G - 1)) == 0) {
    atomicMax(&dst[s].bits, (unsigned long long)__double_as_longlong(d2));
  }
}

// ermak_a of the first step (Integration.F90:963-1011) for every atom, its
// 16 lanes as in k_batch_force; positions move in place.
__global__ __launch_bounds__(GH_BWG) void k_batch_ermak_a(BatchArgs B, ErmakC k,
                                                          unsigned long long seed, long long step) {
  const int i0 = (int)(blockIdx.x * GH_BWG + threadIdx.x) >> 4;
  const bool live = i0 < B.ntot;
  const int i = min(i0, B.ntot - 1), sub = threadIdx.x & 15, s = B.sysof[i];
  double d2 = 0.0;
  if (live && sub < 3) {
    float ga, gb;
    axis_normals(seed, step, i, sub, ga, gb);
    const double f_lan = sqrt(k.kB_ui * B.T[s]) * B.osm[B.type[i]];
    double *x = reinterpret_cast<double *>(B.pos + i) + sub;
    const double v = *x + k.c1 * B.vel[sub * B.ld + i] + k.c2 * k.dt * B.acc[sub * B.ld + i] +
                     f_lan * k.sdr * (double)ga;
    *x = v;
    const double dd = v - B.xold[sub * B.ld + i];
    d2 = dd * dd;
  }
  fold_sys_disp2<16>(B, group_total<16>(d2), s, live, (int)(step & 1));
}

// Forces; MODE 0: stored with the per-atom energies (batch_compute); 1: then
// ermak_b of `step` (Integration.F90:1013-1031) and ermak_a of the next, the
// new positions to pos_next; 2: the run's last step, ermak_b and energies.
// Lanes 0..2 of an atom's group hold its axes, lanes 4..6 draw the next
// step's normals beside them.
template <bool MIXED, bool QUANT, bool SINGLE, int G, int MODE>
__global__ __launch_bounds__(GH_BWG) void k_batch_force(BatchArgs B, BForm<MIXED> p1, ErmakC k,
                                                        unsigned long long seed, long long step) {
  __shared__ BTable<MIXED, SINGLE> T;
  load_table<MIXED, QUANT, SINGLE>(T, B);
  const int i0 = (int)(blockIdx.x * GH_BWG + threadIdx.x) / G;
  const bool live = i0 < B.ntot;
  const int i = min(i0, B.ntot - 1), sub = threadIdx.x & (G - 1);
  const int s = B.sysof[i], a0 = B.a0of[i];
  const RowHead<G> row = row_head<G>(B, i, live);
  const int ax = min(sub & 3, 2);
  double v = 0.0, a = 0.0, xo = 0.0, x = 0.0;
  if (MODE != 0) {  // issued before the pair loop
    v = B.vel[ax * B.ld + i];
    a = B.acc[ax * B.ld + i];
    if (MODE == 1) {
      xo = B.xold[ax * B.ld + i];
      x = reinterpret_cast<const double *>(B.pos + i)[ax];
    }
  }
  double f[4];
  batch_force<MIXED, SINGLE, G>(B, T, p1, a0, i, row, f);
  if (MODE != 1 && live && sub == 3) B.e[i] = (f[3] - sqrt(B.rho[i])) * B.ev_ui;
  const double F = (ax == 0 ? f[0] : ax == 1 ? f[1] : f[2]) * B.ev_ui;
  if (MODE == 0) {
    if (live && sub < 3) B.frc[sub * B.ld + i] = F;
    return;
  }
  float ga, gb;
  axis_normals(seed, step + (sub >= 4 ? 1 : 0), i, ax, ga, gb);
  const float ga_next = __shfl_down(ga, 4, 64);
  const int t = B.type[i];
  const double f_lan = sqrt(k.kB_ui * B.T[s]) * B.osm[t], om = B.om[t];
  const double vel_v = f_lan * k.sdv * (k.crv1 * (double)ga + k.crv2 * (double)gb);
  v = k.c0 * v + (k.c1 - k.c2) * a + k.c2 * F * om + vel_v;
  a = F * om;
  double d2 = 0.0;
  if (MODE == 1) {
    x = x + k.c1 * v + k.c2 * k.dt * a + f_lan * k.sdr * (double)ga_next;
    d2 = x - xo;
    d2 = live && sub < 3 ? d2 * d2 : 0.0;
  }
  if (live && sub < 3) {
    B.vel[sub * B.ld + i] = v;
    B.acc[sub * B.ld + i] = a;
    if (MODE == 1) reinterpret_cast<double *>(B.pos_next + i)[sub] = x;
  }
  if (MODE == 1) fold_sys_disp2<G>(B, group_total<G>(d2), s, live, (int)((step + 1) & 1));
}

// epot (ui) and ekin about the centre of mass (ui) of one system.
template <int BS>
__device__ void sys_energies(const BatchArgs &B, BlockRed<BS> &R, int a0, int a1, double &epot,
                             double &ekin) {
  double s[5] = {0, 0, 0, 0, 0};
  for (int i = a0 + threadIdx.x; i < a1; i += blockDim.x) {
    const double m = 1.0 / B.om[B.type[i]];
    s[0] += B.e[i];
    s[1] += m;
    s[2] += m * B.vel[i];
    s[3] += m * B.vel[B.ld + i];
    s[4] += m * B.vel[2 * B.ld + i];
  }
  bsum<BS, 5>(R, s);
  const double cx = s[2] / s[1], cy = s[3] / s[1], cz = s[4] / s[1];
  double k[1] = {0.0};
  for (int i = a0 + threadIdx.x; i < a1; i += blockDim.x) {
    const double m = 1.0 / B.om[B.type[i]];
    const double wx = B.vel[i] - cx, wy = B.vel[B.ld + i] - cy, wz = B.vel[2 * B.ld + i] - cz;
    k[0] += (wx * wx + wy * wy + wz * wz) * m;
  }
  bsum<BS, 1>(R, k);
  epot = s[0];
  ekin = 0.5 * k[0];
}
// The energies of every system, a workgroup each.
__global__ __launch_bounds__(GH_BWG) void k_batch_energies(BatchArgs B) {
  __shared__ BlockRed<GH_BWG> R;
  const int s = blockIdx.x;
  double ep, ek;
  sys_energies(B, R, B.off[s], B.off[s + 1], ep, ek);
  if (threadIdx.x == 0) {
    B.out[s * OUTW + 0] = ep;
    B.out[s * OUTW + 1] = ek;
  }
}

// ---------------------------------------------------------------------------
// FIRE (Bitzek et al. 2006), a workgroup per system and all its iterations in
// one launch: velocity-Verlet MD step, then P = F.v; v <- (1-a) v + a |v|
// F/|F|; P > 0 for more than N_min steps grows dt (x1.1, capped at dt_max) and
// shrinks a (x0.99); P <= 0 halves dt, zeroes v and resets a.  Mixed
// precision: a first launch runs every system with the FP32 pair terms until
// max|F| < fswitch, a second goes on in FP64; convergence is max|F| < ftol in
// FP64.  (Both in one kernel held 146 registers, three wavefronts per SIMD;
// the mixed one fits the 128 of four.)
//
// An iteration is a chain of passes over the system's atoms with barriers
// between them, so what counts is how few trips to memory it makes and how
// many systems a compute unit holds: four lanes per atom in the passes; one
// loop over the atoms does the mixing of the last iteration, the first half
// kick and the drift and stages the new positions (every thread forms the
// new position of the first atom, the staging's origin, itself); the force
// pass does the second half kick and the sums.  1024 Au clusters of 13..309
// atoms, mixed: 54 us per iteration with one lane per atom and a loop per
// operation, 44 now.
// ---------------------------------------------------------------------------
struct FireC {
  double dt_max, alpha0, fstop, ui_ev;  // fstop: fswitch (mixed) or ftol, eV/A
  int max_iter, resume;
};
struct FireState {  // between the launches, per system
  double dt, alpha, fmax;
  int npos, it, done, conv;
};

#define GH_FG 4  // lanes per atom
// LDS staging of a mixed system: positions in steps of 2^-GH_BFXK A about its
// first atom with eband32 as the fourth word, and types; `far`: an atom lies
// 64 A or more away, the passes then quantise positions from global memory.
struct Stage {
  int4 *q;
  unsigned char *ty;
  int *far;
};
__device__ __forceinline__ void stage_atom(const Stage &S, int k, const double (&x)[3],
                                           const double (&o)[3]) {
  const double dx = (x[0] - o[0]) * GH_BFXS, dy = (x[1] - o[1]) * GH_BFXS,
               dz = (x[2] - o[2]) * GH_BFXS;
  if (!(fabs(dx) < GH_FXLIM && fabs(dy) < GH_FXLIM && fabs(dz) < GH_FXLIM)) *S.far = 1;
  S.q[k] = make_int4(__double2int_rn(dx), __double2int_rn(dy), __double2int_rn(dz), 0);
}

// The row of atom k as batch_row builds it, entry for entry, from the staged
// positions: FP32 decides all pairs but those near a bound, which the FP64 rd
// decides (150 systems of 2,000 atoms, 50 Langevin steps: 8.6 -> 8.3 ms).
__device__ __forceinline__ void batch_row_staged(const BatchArgs &B, const Stage &S, bool on,
                                                 int a0, int n, int k) {
  const int sub = threadIdx.x & 15, i = a0 + k, cap = B.cap;
  const unsigned below = (1u << sub) - 1;
  const double4 pi = B.pos[i];
  const int4 qi = S.q[k];
  unsigned short *row = B.list + (size_t)i * cap;
  int m0 = 0, m1 = 0;
  for (int j0 = 0; __any(on && j0 < n); j0 += 64) {
    int4 q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) q[u] = S.q[min(j0 + 16 * u + sub, n - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + 16 * u + sub;
      const float ux = (float)(int)((unsigned)q[u].x - (unsigned)qi.x),
                  uy = (float)(int)((unsigned)q[u].y - (unsigned)qi.y),
                  uz = (float)(int)((unsigned)q[u].z - (unsigned)qi.z);
      const float r2 = fmaf(ux, ux, fmaf(uy, uy, uz * uz));
      bool keep = on && j < n && j != k && r2 <= B.hi2q, near = r2 < B.near2q;
      if (keep && (r2 >= B.lo2q || fabsf(r2 - B.near2q) <= B.band2q)) {
        const double4 p = B.pos[a0 + j];
        const double rd = dist2_rn(p.x - pi.x, p.y - pi.y, p.z - pi.z);
        keep = rd <= B.rl2;
        near = rd < B.near2;
      }
      const unsigned long long kept = __ballot(keep);
      if (kept == 0ull) continue;
      const unsigned b0 = group_bits<16>(kept & __ballot(near));
      const unsigned b1 = group_bits<16>(kept & ~__ballot(near));
      const int d = near ? m0 + __popc(b0 & below) : cap - 1 - (m1 + __popc(b1 & below));
      if (keep && d >= 0 && d < cap) row[d] = (unsigned short)j;
      m0 += __popc(b0);
      m1 += __popc(b1);
    }
  }
  row_end(B, on, i, m0, m1, pi);
}

// The rows of the system's atoms; ends with a barrier.
template <bool QUANT>
__device__ void sys_build(const BatchArgs &B, const Stage &S, int a0, int n) {
  const int per = (int)blockDim.x >> 4, g = (int)threadIdx.x >> 4;
  const bool lds = QUANT && !*S.far;
  for (int k0 = 0; k0 < n; k0 += per) {
    const bool on = k0 + g < n;
    const int k = min(k0 + g, n - 1);
    if (lds) batch_row_staged(B, S, on, a0, n, k);
    else batch_row(B, on, a0, n, k);
  }
  __syncthreads();
}

template <bool MIXED, bool QUANT, bool SINGLE, int G>
__device__ __forceinline__ void fire_rho(const BatchArgs &B, const Stage &S,
                                         const BTable<MIXED, SINGLE> &T, const BForm<MIXED> &p1,
                                         int a0, int n) {
  const int sub = threadIdx.x & (G - 1), g = (int)threadIdx.x / G;
  const int per = (int)blockDim.x / G;
  const bool lds = QUANT && !*S.far;
  for (int k0 = 0; k0 < n; k0 += per) {
    const bool on = k0 + g < n;
    const int k = min(k0 + g, n - 1), i = a0 + k;
    const RowHead<G> row = row_head<G>(B, i, on);
    if (!lds) {
      batch_rho<MIXED, QUANT, SINGLE, G>(B, T, p1, a0, i, on, row);
    } else if constexpr (QUANT) {
      const int4 qi = S.q[k];
      const int ti = SINGLE ? 0 : S.ty[k];
      double acc = 0.0;
      int4 q[4];
      int t[4];
      batch_each<G>(
          B, row,
          [&](int u, int s) {
            q[u] = S.q[s];
            t[u] = SINGLE ? 0 : S.ty[s];
          },
          [&](int u) {
            const double dx = fxd(q[u].x, qi.x), dy = fxd(q[u].y, qi.y), dz = fxd(q[u].z, qi.z);
            float band;
            if (tb_rho_fx(SINGLE ? p1 : T.t[ti * GH_MAXT + t[u]],
                          fma(dx, dx, fma(dy, dy, dz * dz)), band))
              acc += (double)band;
          });
      acc = group_total<G>(acc);
      if (on && sub == 0) {
        B.rho[i] = acc;
        S.q[k].w = __float_as_int((float)(1.0 / sqrt(acc) - B.e0));
      }
    }
  }
  __syncthreads();
}

// WHAT 0: forces; 1: the per-atom energies of the last ones; 2: both.  A
// quench reads energies at its end only, so the iterations of a mixed one don't
// sum them (6.9 -> 6.5 ms with the order above; in FP64, where the repulsion is
// part of the force anyway, a pass of its own for them costs registers: 12.1 ms
// against 13.9).  hdt > 0: then the second half kick (v += hdt F / m) and the sums pv = {F.v, |v|^2, |F|^2} of
// the thread's atoms.  fm2: the largest |F|^2 of its atoms.
template <bool MIXED, bool QUANT, bool SINGLE, int WHAT, int G>
__device__ __forceinline__ void fire_force(const BatchArgs &B, const Stage &S,
                                           const BTable<MIXED, SINGLE> &T, const BForm<MIXED> &p1,
                                           int a0, int n, double hdt, double (&pv)[3],
                                           double &fm2) {
  const int sub = threadIdx.x & (G - 1), g = (int)threadIdx.x / G;
  const int per = (int)blockDim.x / G;
  const bool lds = QUANT && !*S.far;
  for (int k0 = 0; k0 < n; k0 += per) {
    const bool on = k0 + g < n;
    const int k = min(k0 + g, n - 1), i = a0 + k;
    const RowHead<G> row = row_head<G>(B, i, on);
    const int ax = min(sub, 2);
    const double v0 = G == 4 && WHAT != 1 && hdt > 0.0 ? B.vel[ax * B.ld + i] : 0.0;
    double f[4] = {0.0, 0.0, 0.0, 0.0};
    if (!lds) {
      batch_force<MIXED, SINGLE, G, (WHAT > 0)>(B, T, p1, a0, i, row, f);
    } else if constexpr (QUANT) {
      const int4 qi = S.q[k];
      const int ti = SINGLE ? 0 : S.ty[k];
      const float di = __int_as_float(qi.w);
      int4 q[4];
      int t[4];
      batch_each<G>(
          B, row,
          [&](int u, int s) {
            q[u] = S.q[s];
            t[u] = SINGLE ? 0 : S.ty[s];
          },
          [&](int u) {
            const double dx = fxd(q[u].x, qi.x), dy = fxd(q[u].y, qi.y), dz = fxd(q[u].z, qi.z);
            float sf, repul;
            if (tb_force_fx<(WHAT > 0)>(SINGLE ? p1 : T.t[ti * GH_MAXT + t[u]],
                                        fma(dx, dx, fma(dy, dy, dz * dz)),
                                        di + __int_as_float(q[u].w), sf, repul)) {
              const double sfd = (double)sf;
              f[0] = fma(-sfd, dx, f[0]);
              f[1] = fma(-sfd, dy, f[1]);
              f[2] = fma(-sfd, dz, f[2]);
              if (WHAT > 0) f[3] += (double)repul;
            }
          });
#pragma unroll
      for (int d = WHAT == 1 ? 3 : 0; d < (WHAT > 0 ? 4 : 3); ++d) f[d] = group_total<G>(f[d]);
    }
    if (WHAT > 0 && on && sub == G - 1) B.e[i] = (f[3] - sqrt(B.rho[i])) * B.ev_ui;
    if (WHAT == 1) continue;
    if constexpr (G == 1) {
      if (!on) continue;
      double F2 = 0.0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double F = f[d] * B.ev_ui;
        B.frc[d * B.ld + i] = F;
        F2 += F * F;
        if (hdt > 0.0) {
          const double v = B.vel[d * B.ld + i] + hdt * F * B.om[SINGLE ? 0 : B.type[i]];
          B.vel[d * B.ld + i] = v;
          pv[0] += F * v;
          pv[1] += v * v;
        }
      }
      pv[2] += F2;
      fm2 = fmax(fm2, F2);
      continue;
    }
    const double F = (ax == 0 ? f[0] : ax == 1 ? f[1] : f[2]) * B.ev_ui;
    if (on && sub < 3) {
      B.frc[sub * B.ld + i] = F;
      if (hdt > 0.0) {
        const double v = v0 + hdt * F * B.om[SINGLE ? 0 : B.type[i]];
        B.vel[sub * B.ld + i] = v;
        pv[0] += F * v;
        pv[1] += v * v;
        pv[2] += F * F;
      }
    }
    if (on && sub == 0) {
      const double Fy = f[1] * B.ev_ui, Fz = f[2] * B.ev_ui;
      fm2 = fmax(fm2, F * F + Fy * Fy + Fz * Fz);
    }
  }
}

// (G lanes per atom; BS threads, 0: as launched)
template <bool MIXED, bool QUANT, bool SINGLE, int G, int BS>
__global__ __launch_bounds__(BS ? BS : 1024, 4) void k_batch_fire(BatchArgs B, FireC fc_arg, double skin_arg,
                                                       FireState *fst, BForm<MIXED> p_arg) {
  // The constants live in LDS and are read where they are used: held in
  // scalar registers for a whole kernel of this kind they were spilled, and
  // the ROCm 7.2 compiler has mis-allocated such spills (a later
  // kernel-argument load overwrote the registers before they were saved).
  __shared__ FireC fc;
  __shared__ double skin;
  __shared__ BForm<MIXED> p1;
  extern __shared__ int4 dyn_q[];
  __shared__ BTable<MIXED, SINGLE> T;
  __shared__ BlockRed<BS> R;
  __shared__ int sfar;
  // Systems come largest first and 256 workgroups fill one slot on each CU:
  // every other 256 run in reverse, so that a CU's systems add up alike (1024
  // Au clusters of 13 to 309 atoms, a quench of 100 iterations: 6.75 -> 6.58 ms).
  const int wr = (int)blockIdx.x & ~255, ww = min(256, (int)gridDim.x - wr);
  const int s = B.order[B.first + ((wr >> 8) & 1 ? 2 * wr + ww - 1 - (int)blockIdx.x : (int)blockIdx.x)];
  FireState st = fst[s];
  if (fc_arg.resume && st.done) return;
  if (threadIdx.x == 0) {
    fc = fc_arg;
    skin = skin_arg;
    p1 = p_arg;
    sfar = 0;
  }
  load_table<MIXED, QUANT, SINGLE>(T, B);
  const int a0 = B.off[s], a1 = B.off[s + 1], n = a1 - a0;
  Stage S{dyn_q, reinterpret_cast<unsigned char *>(dyn_q + B.nst), &sfar};
  __syncthreads();
  if (!fc.resume) {
    for (int i = a0 + threadIdx.x; i < a1; i += blockDim.x)
      for (int d = 0; d < 3; ++d) B.vel[d * B.ld + i] = 0.0;
    st.dt = fc.dt_max * 0.1;
    st.alpha = fc.alpha0;
    st.npos = st.it = st.done = st.conv = 0;
  }
  if (QUANT) {
    const double4 o4 = B.pos[a0];
    const double o[3] = {o4.x, o4.y, o4.z};
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
      const double4 p = B.pos[a0 + k];
      const double x[3] = {p.x, p.y, p.z};
      stage_atom(S, k, x, o);
      if (!SINGLE) S.ty[k] = (unsigned char)B.type[a0 + k];
    }
    __syncthreads();
  }
  if (!fc.resume) sys_build<QUANT>(B, S, a0, n);
  constexpr int kForce = MIXED ? 0 : 2;
  double pv[3] = {0.0, 0.0, 0.0}, fm2 = 0.0;
  fire_rho<MIXED, QUANT, SINGLE, G>(B, S, T, p1, a0, n);
  fire_force<MIXED, QUANT, SINGLE, kForce, G>(B, S, T, p1, a0, n, 0.0, pv, fm2);
  // the mixing of the last iteration, still to be applied to v: v <- cm v + mixv F
  double cm = 1.0, mixv = 0.0;
  bool pend = false;
  bred<BS, 0>(R, pv, fm2);
  double dt = st.dt, alpha = st.alpha, fnow = sqrt(fm2) * fc.ui_ev;  // eV/A
  int it = st.it, npos = st.npos;
  bool stop = false;
  st.fmax = fnow;  // (no iterations: of the starting positions)
  for (; it < fc.max_iter; ++it) {
    st.fmax = fnow;
    if (fnow < fc.fstop) {
      stop = true;
      break;
    }
    // mixing, first half kick, drift; the origin of the staging first
    double o[3] = {0.0, 0.0, 0.0}, d2 = 0.0;
    auto move = [&](int i, double (&x)[3], bool store) {
      const double4 p = B.pos[i];
      const double om = B.om[SINGLE ? 0 : (int)p.w];
      x[0] = p.x;
      x[1] = p.y;
      x[2] = p.z;
      double e2 = 0.0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double F = B.frc[d * B.ld + i];
        double v = B.vel[d * B.ld + i];
        if (pend) v = cm * v + mixv * F;
        v = v + 0.5 * dt * F * om;
        x[d] += dt * v;
        if (store) {
          B.vel[d * B.ld + i] = v;
          const double dd = x[d] - B.xold[d * B.ld + i];
          e2 += dd * dd;
        }
      }
      if (store) B.pos[i] = make_double4(x[0], x[1], x[2], p.w);
      return e2;
    };
    if (QUANT) {
      move(a0, o, false);
      if (threadIdx.x == 0) sfar = 0;
      __syncthreads();  // every thread has read atom a0 before it moves
    }
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
      double x[3];
      d2 = fmax(d2, move(a0 + k, x, true));
      if (QUANT) stage_atom(S, k, x, o);
    }
    double none[3] = {0.0, 0.0, 0.0};
    bred<BS, 0>(R, none, d2);
    if (2.0 * sqrt(d2) > skin) sys_build<QUANT>(B, S, a0, n);
    pv[0] = pv[1] = pv[2] = fm2 = 0.0;
    fire_rho<MIXED, QUANT, SINGLE, G>(B, S, T, p1, a0, n);
    fire_force<MIXED, QUANT, SINGLE, kForce, G>(B, S, T, p1, a0, n, 0.5 * dt, pv, fm2);
    bred<BS, 3>(R, pv, fm2);
    fnow = sqrt(fm2) * fc.ui_ev;
    pend = true;
    if (pv[0] > 0.0) {
      cm = 1.0 - alpha;
      mixv = pv[2] > 0.0 ? alpha * sqrt(pv[1]) / sqrt(pv[2]) : 0.0;
      ++npos;
      if (npos > 5) {
        dt = fmin(dt * 1.1, fc.dt_max);
        alpha *= 0.99;
      }
    } else {
      cm = mixv = 0.0;
      npos = 0;
      dt *= 0.5;
      alpha = fc.alpha0;
    }
  }
  if (pend)
    for (int i = a0 + threadIdx.x; i < a1; i += blockDim.x)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double v = B.vel[d * B.ld + i];
        B.vel[d * B.ld + i] = cm == 0.0 && mixv == 0.0 ? 0.0 : cm * v + mixv * B.frc[d * B.ld + i];
      }
  const bool done = !MIXED || !stop;  // a mixed system below fswitch goes on in FP64
  double ep = 0.0, ek = 0.0;
  if (done) {
    if (MIXED) {
      fire_force<MIXED, QUANT, SINGLE, 1, G>(B, S, T, p1, a0, n, 0.0, pv, fm2);
      __syncthreads();
    }
    sys_energies(B, R, a0, a1, ep, ek);
  }
  if (threadIdx.x == 0) {
    st.dt = dt;
    st.alpha = alpha;
    st.npos = npos;
    st.it = it;
    st.done = done;
    st.conv = !MIXED && stop;
    fst[s] = st;
    if (done) {
      B.out[s * OUTW + 0] = ep;
      B.out[s * OUTW + 3] = st.fmax;
      B.out[s * OUTW + 4] = it;
      B.out[s * OUTW + 5] = st.conv;
    }
  }
}

// Langevin steps of mixed systems staged in LDS, a workgroup per system (largest
// first) and all steps in one launch: no random gathers from the L2, which bound
// the passes over all atoms, and no launches per step.  Chosen by batch_staged,
// its threads by staged_threads; the first step's ermak_a has run.
//
// G lanes per atom: four, or one in large systems (launch_split).  The update
// takes a thread per atom and axis and draws each normal once: the next step's
// pair waits in pos_next, which the passes over all atoms rewrite (150 systems of
// 2,000 Ag-Cu atoms, 50 steps: 8.3 -> 7.9 ms).
template <bool SINGLE, int G>
__global__ __launch_bounds__(1024, 4) void k_batch_langevin(BatchArgs B, ErmakC k_arg, double skin,
                                                            TbF p_arg, unsigned long long seed,
                                                            long long step0, int nsteps) {
  __shared__ ErmakC k;
  __shared__ TbF p1;
  extern __shared__ int4 dyn_q[];
  __shared__ BTable<true, SINGLE> T;
  __shared__ double top[16];
  __shared__ int sfar;
  const int s = B.order[B.first + blockIdx.x], a0 = B.off[s], n = B.off[s + 1] - a0;
  if (threadIdx.x == 0) {
    k = k_arg;
    p1 = p_arg;
  }
  load_table<true, true, SINGLE>(T, B);
  Stage S{dyn_q, reinterpret_cast<unsigned char *>(dyn_q + B.nst), &sfar};
  const double skt = sqrt(k_arg.kB_ui * B.T[s]);
  auto normals = [&](int q) { return reinterpret_cast<float2 *>(B.pos_next + a0 + q / 3) + q % 3; };
  for (int q = threadIdx.x; q < 3 * n; q += blockDim.x) {
    float2 g;
    axis_normals(seed, step0, a0 + q / 3, q % 3, g.x, g.y);
    *normals(q) = g;
  }
  for (int st = 0; st < nsteps; ++st) {
    if (threadIdx.x == 0) sfar = 0;
    __syncthreads();
    const double4 o4 = B.pos[a0];
    const double o[3] = {o4.x, o4.y, o4.z};
    double d2 = 0.0, none[3] = {0.0, 0.0, 0.0}, fm2 = 0.0;
    for (int q = threadIdx.x; q < n; q += blockDim.x) {
      const double4 p = B.pos[a0 + q];
      const double x[3] = {p.x, p.y, p.z};
      double e2 = 0.0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double dd = x[d] - B.xold[d * B.ld + a0 + q];
        e2 += dd * dd;
      }
      d2 = fmax(d2, e2);
      stage_atom(S, q, x, o);
      if (!SINGLE) S.ty[q] = (unsigned char)(int)p.w;
    }
    d2 = wave_top(d2);
    if ((threadIdx.x & 63) == 0) top[threadIdx.x >> 6] = d2;
    __syncthreads();
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) d2 = fmax(d2, top[w]);
    if (2.0 * sqrt(d2) > skin) {
      sys_build<true>(B, S, a0, n);
      if (threadIdx.x == 0) B.out[s * OUTW + 2] += 1.0;
    }
    const bool last = st + 1 == nsteps;
    fire_rho<true, true, SINGLE, G>(B, S, T, p1, a0, n);
    if (last) fire_force<true, true, SINGLE, 2, G>(B, S, T, p1, a0, n, 0.0, none, fm2);
    else fire_force<true, true, SINGLE, 0, G>(B, S, T, p1, a0, n, 0.0, none, fm2);
    __syncthreads();
    // ermak_b, and ermak_a of the next step (the passes read positions from LDS)
    const long long step = step0 + st;
    for (int q = threadIdx.x; q < 3 * n; q += blockDim.x) {
      const int i = a0 + q / 3, ax = q % 3, t = SINGLE ? 0 : S.ty[q / 3];
      float2 g = *normals(q);
      const double F = B.frc[ax * B.ld + i], om = B.om[t], f_lan = skt * B.osm[t];
      const double vel_v = f_lan * k.sdv * (k.crv1 * (double)g.x + k.crv2 * (double)g.y);
      const double v = k.c0 * B.vel[ax * B.ld + i] + (k.c1 - k.c2) * B.acc[ax * B.ld + i] +
                       k.c2 * F * om + vel_v;
      const double a = F * om;
      B.vel[ax * B.ld + i] = v;
      B.acc[ax * B.ld + i] = a;
      if (!last) {
        axis_normals(seed, step + 1, i, ax, g.x, g.y);
        *normals(q) = g;
        double *x = reinterpret_cast<double *>(B.pos + i) + ax;
        *x = *x + k.c1 * v + k.c2 * k.dt * a + f_lan * k.sdr * (double)g.x;
      }
    }
    __syncthreads();
  }
}

__global__ void k_batch_zero(GhLine *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i].bits = 0ull;
}

__global__ void k_batch_scale(int nsys, const int *__restrict__ off,
                              const double *__restrict__ scale, double *__restrict__ vel,
                              int ld) {
  const int s = blockIdx.x;
  if (s >= nsys) return;
  const double f = scale[s];
  for (int i = off[s] + threadIdx.x; i < off[s + 1]; i += blockDim.x)
    for (int d = 0; d < 3; ++d) vel[d * ld + i] *= f;
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static int bfail(gh_batch *b, int code, const std::string &m) {
  if (b) b->err = m;
  return code;
}
#define BH(b, call)                                                                      \
  do {                                                                                   \
    hipError_t e_ = (call);                                                              \
    if (e_ != hipSuccess)                                                                \
      return bfail(b, GH_EHIP, std::string(#call) + ": " + hipGetErrorString(e_));        \
  } while (0)
#define BT(x)                 \
  do {                        \
    int rc_ = (x);            \
    if (rc_ != 0) return rc_; \
  } while (0)

template <typename T>
static int balloc(gh_batch *b, T **p, size_t n) {
  if (*p) {
    BH(b, hipFree(*p));
    *p = nullptr;
  }
  if (n) BH(b, hipMalloc((void **)p, sizeof(T) * n));
  return 0;
}

static BatchArgs bargs(const gh_batch *b) {
  BatchArgs A;
  A.off = b->off;
  A.order = b->order;
  A.first = 0;
  A.type = b->type;
  A.sysof = b->sysof;
  A.a0of = b->a0of;
  A.nsys = b->nsys;
  A.ntot = b->ntot;
  A.pos = b->pos;
  A.pos_next = b->pos_next;
  A.pk = b->pk;
  A.vel = b->vel;
  A.acc = b->acc;
  A.frc = b->frc;
  A.e = b->e;
  A.rho = b->rho;
  A.xold = b->xold;
  A.nn = b->nn;
  A.list = b->list;
  A.cap = b->cap;
  A.ld = b->ld;
  A.tbd = b->tbd;
  A.tbf = b->tbf;
  A.e0 = b->tb_e0;
  A.nt = std::max(b->nt, b->types);  // (entries past the potential's are zero: no interaction)
  A.nst = b->nst;
  A.dmax = b->dmax;
  for (int t = 0; t < GH_MAXT; ++t) {
    A.om[t] = 1.0 / b->mass_t[t];
    A.osm[t] = sqrt(A.om[t]);
  }
  const double rl = b->rcut + b->skin;
  A.rl2 = rl * rl;
  double rci = 1e300;
  for (int i = 0; i < b->nt; ++i)
    for (int j = 0; j < b->nt; ++j) rci = std::min(rci, b->tb[i * GH_MAXT + j].rci);
  A.near2 = rci * rci;
  // FP32 on the staged positions: its error on r^2 stays below 1e-4 A^2 for
  // pairs near the bounds; the margins are thirty times that
  const double q2 = GH_BFXS * GH_BFXS, margin = std::max(3e-3, 1e-4 * A.rl2);
  A.hi2q = (float)((A.rl2 + margin) * q2);
  A.lo2q = (float)((A.rl2 - margin) * q2);
  A.near2q = (float)(A.near2 * q2);
  A.band2q = (float)(std::max(3e-3, 1e-4 * A.near2) * q2);
  A.ev_ui = ghc::ev_ui();
  A.T = b->T;
  A.out = b->out;
  A.flags = b->flags;
  return A;
}

// Reports a row overflow of the last call and re-arms the flags; the next
// call re-sizes the rows to the longest one asked for (plus a quarter).
static int check_flags(gh_batch *b) {
  int f[2] = {0, 0};
  BH(b, hipMemcpyAsync(f, b->flags, sizeof(f), hipMemcpyDeviceToHost, b->stream));
  BH(b, hipStreamSynchronize(b->stream));
  if (f[0]) {
    const int zero[2] = {0, 0};
    BH(b, hipMemcpyAsync(b->flags, zero, sizeof(zero), hipMemcpyHostToDevice, b->stream));
    BH(b, hipStreamSynchronize(b->stream));
    b->lists_valid = false;
    b->forces_valid = false;
    b->cap_req = f[1] + std::max(16, f[1] / 4);
    const int cap = b->cap;
    b->cap = 0;
    return bfail(b, GH_EOVERFLOW,
                 "a cluster's neighbour row exceeded the capacity (" + std::to_string(f[1]) +
                     " > " + std::to_string(cap) + "); results of this call are invalid; "
                     "the next call re-sizes the rows");
  }
  return 0;
}

static int fetch_out(gh_batch *b, std::vector<double> &o) {
  o.resize((size_t)b->nsys * OUTW);
  BH(b, hipMemcpyAsync(o.data(), b->out, sizeof(double) * o.size(), hipMemcpyDeviceToHost,
                       b->stream));
  BH(b, hipStreamSynchronize(b->stream));
  return 0;
}

// capacity of a list row: every other atom of the largest system, capped by
// the densest packing within rcut+skin (fcc metals: < 90 neighbours)
static int batch_ready(gh_batch *b) {
  if (!b->nsys) return bfail(b, GH_ESTATE, "no systems");
  if (!b->have_pot) return bfail(b, GH_ESTATE, "no potential");
  if (b->cap == 0) {
    int nmax = 0;
    for (int s = 0; s < b->nsys; ++s) nmax = std::max(nmax, b->off_h[s + 1] - b->off_h[s]);
    const double rl = b->rcut + b->skin;
    // close packing density of the smallest pair distance (0.8 r0 at most)
    double rmin = 1e30;
    for (int i = 0; i < b->nt; ++i)
      for (int j = 0; j < b->nt; ++j) rmin = std::min(rmin, 0.8 * b->tb[i * GH_MAXT + j].r0);
    const double dens = 1.4142135623730951 / (rmin * rmin * rmin);
    int est = (int)(4.18879 * rl * rl * rl * dens) + 16;
    b->cap = std::max(8, std::min(nmax, std::max(est, b->cap_req)));
    b->cap = (b->cap + 7) / 8 * 8;
    BT(balloc(b, &b->list, (size_t)b->cap * b->ld));
    // LDS staging of the largest system (int4 + type byte per atom, and the
    // sentinel) beside tables of 344 B per type pair and the sums of eight
    // wavefronts, within 64 KB: 3,799 atoms of one type, 2,525 of several; larger
    // systems use global memory.  The rule also says which FP32 form a mixed
    // batch computes (quantised positions where it holds), so it follows neither
    // the size of the tables' structures nor the kernels' threads (with 1024 they
    // hold up to 65.8 KB in all, of the 160 KB of a compute unit).
    const size_t stat = (b->nt > 1 ? GH_MAXT * GH_MAXT : 1) * 344 +
                        sizeof(double) * 8 * 8 + 64;
    const size_t need = 17 * (size_t)(nmax + 1);
    b->nst = stat + need <= 65536 ? nmax + 1 : 0;
  }
  return 0;
}

static int largest_system(const gh_batch *b) {
  const int big = b->order_h[0];
  return b->off_h[big + 1] - b->off_h[big];
}

// Threads of the workgroups of k_batch_langevin.  A CU runs 16 of its wavefronts:
// as one workgroup while the atoms' sum is at most one system of the largest size
// per CU, as two, four, ... of half, a quarter, ... the wavefronts where it is
// two, four, ..., so that all systems are in flight; no fewer than the largest
// power of two in the largest system's atoms (more systems in flight then only
// outgrow the L2), and no more than four lanes for each of them.  50 steps of Ag-Cu
// systems, ms, 64 / 128 / 256 / 512 / 1024 threads, with the largest systems per CU:
// 10,000 of 13 atoms (40) 1.7 / 2.5 / 4.3 / 7.9 / 15; 6000 of 147 (23) 12.5 / 10.9 / 12.2 /
// 16 / 18; 2000 of 147 (7.8) 6.7 / 3.8 / 4.3 / 5.4 / 6.1; 4000 of 309 (16) 27 / 16.1 / 15.5 /
// 17.0 / 21; 1000 of 309 (3.9) 13 / 7.0 / 4.2 / 4.5 / 5.5; 600 of 147 (2.3) 5.8 / 3.4 / 2.0 /
// 2.4 / 2.3; 400 of 1000 (1.6) - / 20 / 10 / 6.5 / 6.7; 1024 of 13 to 309, log-uniform
// (1.2) 11 / 5.8 / 3.1 / 1.9 / 2.9; 512 of 38 to 1000, log-uniform (0.57) 38 / 20 / 10 /
// 5.7 / 3.8.
static int staged_threads(const gh_batch *b) {
  const int nmax = largest_system(b);
  const double r = b->ntot / (256.0 * nmax);
  int bs = 1024;
  while (bs > 64 && r > 1024.0 / bs && bs > nmax) bs /= 2;
  while (bs > 64 && bs / 2 >= GH_FG * nmax) bs /= 2;
  return bs;
}

// Runs launch(lanes, first, count, stream) for the systems of one lane per atom,
// those of `least` atoms and more (systems come largest first), and of four, on
// two streams where there are both.  One and a half times the workgroup's threads:
// its wavefronts are full either way, and four lanes pay a row's padding and the
// sums four times (50 Langevin steps, Ag-Cu, ms, four lanes and one: 150 systems of
// 2,000 atoms 9.2 and 7.9, 1000 of 400 5.6 and 5.1, 1000 of 309 4.2 and 4.3, 600 of 147
// 2.0 and 2.5).
template <class LAUNCH>
static int launch_split(gh_batch *b, int least, LAUNCH &&launch) {
  int one = 0;
  for (; one < b->nsys; ++one) {
    const int s = b->order_h[one];
    if (b->off_h[s + 1] - b->off_h[s] < least) break;
  }
  const bool both = one > 0 && one < b->nsys;
  if (both) {
    BH(b, hipEventRecord(b->ev_fork, b->stream));
    BH(b, hipStreamWaitEvent(b->stream2, b->ev_fork, 0));
  }
  // (the large ones first)
  if (one > 0) launch(1, 0, one, b->stream);
  BH(b, hipGetLastError());
  if (one < b->nsys) launch(GH_FG, one, b->nsys - one, both ? b->stream2 : b->stream);
  BH(b, hipGetLastError());
  if (both) {
    BH(b, hipEventRecord(b->ev_join, b->stream2));
    BH(b, hipStreamWaitEvent(b->stream, b->ev_join, 0));
  }
  return 0;
}

// Threads of the FIRE kernel's workgroups: 256 where four systems share a compute
// unit and hide each other's barriers (1024 Au clusters, mixed, a quench of 100
// iterations: 128 threads 9.9 ms, 256 6.7, 512 7.2; registers for five wavefronts
// per SIMD instead of four spill: 9.0); fewer systems leave units idle, and a
// system's rounds of atoms, one memory round trip after another, bound its
// iteration: 512 up to 768 systems, 1024 up to 256.  80 iterations, clusters to 309
// atoms, 256 / 512 / 1024 threads, ms, mixed (FP64): 200 systems 3.4 / 2.4 / 2.2
// (5.3 / 4.2 / 4.2), 500 4.4 / 3.2 / 4.0 (7.0 / 5.6 / 7.3), 700 5.0 / 4.2 / 5.4
// (8.2 / 7.4 / 9.4).  But by the atoms' sum per CU in systems of the largest size:
// where it is more than two, 256 instead of 512 (40 iterations, Ag-Cu, ms, mixed and
// FP64, 256 / 512: 600 systems of 147 atoms 1.65 / 2.08 and 2.87 / 3.47), and where it
// is below three quarters and the largest needs more than three rounds of 512
// threads, 1024 (512 of 38 to 1000, log-uniform, 512 / 1024: 4.5 / 3.2 and 7.5 / 5.6);
// 512 also for more systems where the largest needs that many (2000 of 13 to 2000,
// log-uniform, 256 / 512: 16 / 11 and 26 / 20).
// No more than the largest system has lanes for.
static int fire_threads(const gh_batch *b) {
  const int nmax = largest_system(b);
  const double r = b->ntot / (256.0 * nmax);
  int bs = GH_FBS;
  if (b->nsys <= 256 || (nmax > 384 && r <= 0.75)) bs = 1024;
  else if (r <= 2.1 && (b->nsys <= 768 || nmax > 384)) bs = 512;
  while (bs > GH_FBS && bs / 2 >= GH_FG * nmax) bs /= 2;
  return bs;
}

// The FIRE kernel over all systems, a workgroup each.
template <bool MIXED, bool QUANT>
static int launch_fire(gh_batch *b, const BatchArgs &A, const FireC &fc, const BForm<MIXED> &p) {
  const size_t lds = QUANT ? 17 * (size_t)b->nst : 0;
  const int bs = fire_threads(b);
  BatchArgs A1 = A;
  auto launch = [&](int lanes, int first, int count, hipStream_t stream) {
    A1.first = first;
#define LAUNCH_FIRE(SG, G, BS) \
  k_batch_fire<MIXED, QUANT, SG, G, BS><<<count, bs, lds, stream>>>(A1, fc, b->skin, b->fst, p)
    if (b->nt == 1) {
      if (lanes == 1) LAUNCH_FIRE(true, 1, 0);
      else if (bs == 1024) LAUNCH_FIRE(true, GH_FG, 1024);
      else if (bs == 512) LAUNCH_FIRE(true, GH_FG, 512);
      else LAUNCH_FIRE(true, GH_FG, GH_FBS);
    } else {
      if (lanes == 1) LAUNCH_FIRE(false, 1, 0);
      else if (bs == 1024) LAUNCH_FIRE(false, GH_FG, 1024);
      else if (bs == 512) LAUNCH_FIRE(false, GH_FG, 512);
      else LAUNCH_FIRE(false, GH_FG, GH_FBS);
    }
#undef LAUNCH_FIRE
  };
  // (FP64 of one type is short of registers either way: 40 iterations, four lanes and
  // one, 1000 systems of 400 atoms 8.3 and 8.9 ms, 300 of 2000 27.3 and 26.4)
  return launch_split(b, !MIXED && b->nt == 1 ? 3 * bs : bs + bs / 2, launch);
}

static int batch_blocks(const gh_batch *b, int lanes) {
  const int per = GH_BWG / lanes;
  return (b->ntot + per - 1) / per;
}
// Lanes per atom of the passes: 16, or 8 where 16 would fill the chip's
// wavefront slots many times over and the fixed work per wavefront (sums,
// random numbers, update) counts more than the wavefronts in flight.
// Langevin step, mixed, 16 against 8 lanes: 2,600 atoms 18 and 23 us, 80,000
// 72 and 81, 320,000 200 and 186 (FP64 230 and 206).
static bool batch_g8(const gh_batch *b) { return b->ntot >= 200000; }

// Launches kernel<MIXED, QUANT, SINGLE, lanes, ...> for the batch's form
// (mixed batches on quantised positions where their systems would fit the LDS
// staging).
#define BATCH_FORM(KERNEL, MX, QU, ARGS, ...)                                                \
  do {                                                                                       \
    const bool one = b->nt == 1;                                                             \
    if (batch_g8(b)) {                                                                       \
      const int gr = batch_blocks(b, 8);                                                     \
      if (one) KERNEL<MX, QU, true, 8 __VA_ARGS__><<<gr, GH_BWG, 0, b->stream>>> ARGS;        \
      else KERNEL<MX, QU, false, 8 __VA_ARGS__><<<gr, GH_BWG, 0, b->stream>>> ARGS;           \
    } else {                                                                                 \
      const int gr = batch_blocks(b, 16);                                                    \
      if (one) KERNEL<MX, QU, true, 16 __VA_ARGS__><<<gr, GH_BWG, 0, b->stream>>> ARGS;       \
      else KERNEL<MX, QU, false, 16 __VA_ARGS__><<<gr, GH_BWG, 0, b->stream>>> ARGS;          \
    }                                                                                        \
  } while (0)

static void launch_rho(gh_batch *b, const BatchArgs &A, int par, int always) {
  if (b->precision != GH_MIXED) BATCH_FORM(k_batch_rho, false, false, (A, b->tbd0.d, b->skin, par, always));
  else if (b->nst > 0) BATCH_FORM(k_batch_rho, true, true, (A, b->tbf0, b->skin, par, always));
  else BATCH_FORM(k_batch_rho, true, false, (A, b->tbd0.f, b->skin, par, always));
}
template <int MODE>
static void launch_force(gh_batch *b, const BatchArgs &A, const ErmakC &k, uint64_t seed,
                         long long step) {
  if (b->precision != GH_MIXED) BATCH_FORM(k_batch_force, false, false, (A, b->tbd0.d, k, seed, step), , MODE);
  else if (b->nst > 0) BATCH_FORM(k_batch_force, true, true, (A, b->tbf0, k, seed, step), , MODE);
  else BATCH_FORM(k_batch_force, true, false, (A, b->tbd0.f, k, seed, step), , MODE);
}
#undef BATCH_FORM

extern "C" {

int gh_batch_create(gh_batch **out, int device, int precision) {
  if (!out) return GH_EINVAL;
  *out = nullptr;
  if (precision != GH_FP64 && precision != GH_MIXED) return GH_EINVAL;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return GH_EHIP;
  gh_batch *b = new gh_batch();
  b->device = device;
  b->precision = precision;
  if (hipSetDevice(device) != hipSuccess ||
      hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess ||
      hipStreamCreateWithFlags(&b->stream2, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&b->ev_fork, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&b->ev_join, hipEventDisableTiming) != hipSuccess ||
      hipMalloc((void **)&b->flags, sizeof(int) * 4) != hipSuccess ||
      hipMemsetAsync(b->flags, 0, sizeof(int) * 4, b->stream) != hipSuccess ||
      hipStreamSynchronize(b->stream) != hipSuccess) {
    delete b;
    return GH_EHIP;
  }
  *out = b;
  return 0;
}

void gh_batch_destroy(gh_batch *b) {
  if (!b) return;
  (void)hipSetDevice(b->device);
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  if (b->stream2) (void)hipStreamSynchronize(b->stream2);
  void *p[] = {b->off, b->order, b->type, b->nn, b->flags, b->pos, b->vel, b->acc, b->frc,
               b->e, b->rho, b->xold, b->T, b->out, b->scale, b->list,
               b->tbd, b->tbf, b->sysof, b->a0of, b->dmax, b->pos_next, b->pk, b->fst};
  for (void *q : p)
    if (q) (void)hipFree(q);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  if (b->stream2) (void)hipStreamDestroy(b->stream2);
  if (b->ev_fork) (void)hipEventDestroy(b->ev_fork);
  if (b->ev_join) (void)hipEventDestroy(b->ev_join);
  delete b;
}

const char *gh_batch_last_error(const gh_batch *b) { return b ? b->err.c_str() : "null batch"; }

int gh_batch_set_precision(gh_batch *b, int precision) {
  if (!b) return GH_EINVAL;
  if (precision != GH_FP64 && precision != GH_MIXED) return bfail(b, GH_EINVAL, "precision");
  b->precision = precision;
  b->forces_valid = false;
  return 0;
}

int gh_batch_set_systems(gh_batch *b, int nsys, const int *off, const double *x,
                         const int *type) {
  if (!b || nsys <= 0 || !off || !x) return bfail(b, GH_EINVAL, "gh_batch_set_systems");
  if (off[0] != 0) return bfail(b, GH_EINVAL, "off[0] must be 0");
  for (int s = 0; s < nsys; ++s) {
    const int n = off[s + 1] - off[s];
    if (n < 1 || n > 65535) return bfail(b, GH_EINVAL, "systems need 1..65535 atoms");
  }
  // (a refused call leaves the batch's systems as they are)
  for (int i = 0; type && i < off[nsys]; ++i)
    if (type[i] < 0 || type[i] >= GH_MAXT) return bfail(b, GH_EINVAL, "type out of range");
  BH(b, hipSetDevice(b->device));
  b->nsys = nsys;
  b->ntot = off[nsys];
  b->ld = (b->ntot + 255) / 256 * 256;
  const int ld = b->ld;
  b->off_h.assign(off, off + nsys + 1);
  b->order_h.resize(nsys);
  std::iota(b->order_h.begin(), b->order_h.end(), 0);
  std::stable_sort(b->order_h.begin(), b->order_h.end(), [&](int a, int c) {
    return off[a + 1] - off[a] > off[c + 1] - off[c];
  });
  b->T_h.assign(nsys, 0.0);
  BT(balloc(b, &b->off, nsys + 1));
  BT(balloc(b, &b->order, nsys));
  BT(balloc(b, &b->type, ld));
  BT(balloc(b, &b->nn, ld));
  BT(balloc(b, &b->pos, ld));
  BT(balloc(b, &b->vel, 3 * (size_t)ld));
  BT(balloc(b, &b->acc, 3 * (size_t)ld));
  BT(balloc(b, &b->frc, 3 * (size_t)ld));
  BT(balloc(b, &b->e, ld));
  BT(balloc(b, &b->rho, ld));
  BT(balloc(b, &b->pos_next, ld));
  BT(balloc(b, &b->pk, ld));
  BT(balloc(b, &b->sysof, ld));
  BT(balloc(b, &b->a0of, ld));
  BT(balloc(b, &b->dmax, 2 * (size_t)nsys));
  BT(balloc(b, &b->xold, 3 * (size_t)ld));
  BT(balloc(b, &b->T, nsys));
  BT(balloc(b, &b->out, (size_t)nsys * OUTW));
  BT(balloc(b, &b->scale, nsys));
  BT(balloc(b, &b->fst, nsys));
  b->cap = 0;
  b->cap_req = 0;
  if (b->list) {
    BH(b, hipFree(b->list));
    b->list = nullptr;
  }
  std::vector<double4> hp(ld, make_double4(0, 0, 0, 0));
  std::vector<int> ht(ld, 0);
  for (int i = 0; i < b->ntot; ++i) {
    ht[i] = type ? type[i] : 0;
    hp[i] = make_double4(x[3 * i], x[3 * i + 1], x[3 * i + 2], (double)ht[i]);
  }
  b->types = 1 + *std::max_element(ht.begin(), ht.end());
  std::vector<int> hs(ld, nsys - 1), ha(ld, off[nsys - 1]);
  for (int k = 0; k < nsys; ++k) {
    std::fill(hs.begin() + off[k], hs.begin() + off[k + 1], k);
    std::fill(ha.begin() + off[k], ha.begin() + off[k + 1], off[k]);
  }
  // every upload and clear is ordered on the batch stream (a non-blocking
  // stream does not wait for work on the null stream)
  hipStream_t st = b->stream;
  BH(b, hipMemcpyAsync(b->pos, hp.data(), sizeof(double4) * ld, hipMemcpyHostToDevice, st));
  BH(b, hipMemcpyAsync(b->pos_next, hp.data(), sizeof(double4) * ld, hipMemcpyHostToDevice, st));
  BH(b, hipMemcpyAsync(b->type, ht.data(), sizeof(int) * ld, hipMemcpyHostToDevice, st));
  BH(b, hipMemcpyAsync(b->off, off, sizeof(int) * (nsys + 1), hipMemcpyHostToDevice, st));
  BH(b, hipMemcpyAsync(b->sysof, hs.data(), sizeof(int) * ld, hipMemcpyHostToDevice, st));
  BH(b, hipMemcpyAsync(b->a0of, ha.data(), sizeof(int) * ld, hipMemcpyHostToDevice, st));
  BH(b, hipMemcpyAsync(b->order, b->order_h.data(), sizeof(int) * nsys, hipMemcpyHostToDevice,
                       st));
  BH(b, hipMemsetAsync(b->vel, 0, sizeof(double) * 3 * ld, st));
  BH(b, hipMemsetAsync(b->acc, 0, sizeof(double) * 3 * ld, st));
  BH(b, hipMemsetAsync(b->frc, 0, sizeof(double) * 3 * ld, st));
  BH(b, hipMemsetAsync(b->out, 0, sizeof(double) * nsys * OUTW, st));
  BH(b, hipMemsetAsync(b->T, 0, sizeof(double) * nsys, st));
  BH(b, hipStreamSynchronize(st));
  b->lists_valid = false;
  b->forces_valid = false;
  return 0;
}

int gh_batch_set_smatb(gh_batch *b, int nt, const double *A, const double *xi, const double *p,
                       const double *q, const double *r0, const double *rci, const double *rce) {
  if (!b || nt <= 0 || nt > GH_MAXT) return bfail(b, GH_EINVAL, "gh_batch_set_smatb");
  // reuse the single-system parameter upload through a scratch context
  gh_ctx tmp;
  tmp.device = b->device;
  tmp.tbf_k = GH_BFXK;  // the FP32 forms in the unit of the staged positions
  int rc = gh_set_smatb(&tmp, nt, A, xi, p, q, r0, rci, rce);
  if (rc) return bfail(b, rc, tmp.err);
  for (int k = 0; k < GH_MAXT * GH_MAXT; ++k) b->tb[k] = tmp.tb[k];
  if (b->tbd) BH(b, hipFree(b->tbd));
  b->tbd = tmp.tbd;  // ownership moves to the batch
  tmp.tbd = nullptr;
  if (b->tbf) BH(b, hipFree(b->tbf));
  b->tbf = tmp.tbf;
  tmp.tbf = nullptr;
  b->tb_e0 = tmp.tb_e0;
  b->tbd0.d = tmp.tb64_0;
  b->tbd0.f = tmp.tbf_a0;
  b->tbf0 = tmp.tbf0;
  b->nt = nt;
  b->rcut = tmp.rcut;
  b->have_pot = true;
  b->cap = 0;
  b->lists_valid = false;
  b->forces_valid = false;
  return 0;
}

int gh_batch_set_masses(gh_batch *b, int nt, const double *mass) {
  if (!b || nt <= 0 || nt > GH_MAXT || !mass) return bfail(b, GH_EINVAL, "gh_batch_set_masses");
  for (int t = 0; t < nt; ++t) {
    if (!(mass[t] > 0)) return bfail(b, GH_EINVAL, "masses must be positive");
    b->mass_t[t] = mass[t];
  }
  return 0;
}

int gh_batch_set_skin(gh_batch *b, double skin) {
  if (!b || !(skin >= 0)) return bfail(b, GH_EINVAL, "skin must be >= 0");
  b->skin = skin;
  b->cap = 0;
  b->lists_valid = false;
  return 0;
}

int gh_batch_set_velocities(gh_batch *b, const double *v) {
  if (!b || !b->nsys) return bfail(b, GH_ESTATE, "no systems");
  std::vector<double> h(3 * (size_t)b->ld, 0.0);
  if (v)
    for (int i = 0; i < b->ntot; ++i)
      for (int d = 0; d < 3; ++d) h[(size_t)d * b->ld + i] = v[3 * (size_t)i + d];
  BH(b, hipMemcpyAsync(b->vel, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice,
                       b->stream));
  BH(b, hipStreamSynchronize(b->stream));
  return 0;
}

int gh_batch_set_temperatures(gh_batch *b, const double *T) {
  if (!b || !b->nsys || !T) return bfail(b, GH_ESTATE, "no systems");
  b->T_h.assign(T, T + b->nsys);
  BH(b, hipMemcpyAsync(b->T, T, sizeof(double) * b->nsys, hipMemcpyHostToDevice, b->stream));
  BH(b, hipStreamSynchronize(b->stream));
  return 0;
}

int gh_batch_compute(gh_batch *b, double *F, double *epot) {
  if (!b) return GH_EINVAL;
  BH(b, hipSetDevice(b->device));
  BT(batch_ready(b));
  const BatchArgs A = bargs(b);
  launch_rho(b, A, 0, 1);
  launch_force<0>(b, A, ErmakC{}, 0, 0);
  k_batch_energies<<<b->nsys, GH_BWG, 0, b->stream>>>(A);
  BH(b, hipGetLastError());
  BT(check_flags(b));
  b->lists_valid = true;
  b->forces_valid = true;
  std::vector<double> o;
  BT(fetch_out(b, o));
  const double ui_ev = ghc::ui_ev();
  b->epot_h.resize(b->nsys);
  for (int s = 0; s < b->nsys; ++s) b->epot_h[s] = o[s * OUTW] * ui_ev;
  if (epot)
    for (int s = 0; s < b->nsys; ++s) epot[s] = b->epot_h[s];
  if (F) {
    std::vector<double> h(3 * (size_t)b->ld);
    BH(b, hipMemcpyAsync(h.data(), b->frc, sizeof(double) * h.size(), hipMemcpyDeviceToHost,
                         b->stream));
    BH(b, hipStreamSynchronize(b->stream));
    for (int i = 0; i < b->ntot; ++i)
      for (int d = 0; d < 3; ++d) F[3 * (size_t)i + d] = h[(size_t)d * b->ld + i];
  }
  return 0;
}

// Mixed Langevin steps by a workgroup per system (k_batch_langevin) or over all
// atoms.  The former takes the largest system's time, the latter the sum's, so
// by their ratio: 50 steps, Ag-Cu, ms, over all atoms and per system: 512 systems of
// 38 to 2000 atoms, log-uniform, 6.8 and 7.8 (129 of the largest in all), 150 of 2000
// 9.5 and 8.0, 304 of 38 to 500 2.1 and 1.8 (124), 120 of 13 0.67 and 0.43; 64 of 309
// 1.2 and 1.4, 16 of 2000 1.9 and 7.6.  And where the largest system's step takes
// less than two launches, whatever their number: one of 13 0.61 and 0.41, ten of 38
// 0.68 and 0.68, ten of 55 0.67 and 0.71.
static bool batch_staged(const gh_batch *b) {
  const int nmax = largest_system(b);
  return b->precision == GH_MIXED && b->nst > 0 &&
         (nmax <= 32 || b->ntot >= (nmax <= 512 ? 115ll : 144ll) * nmax);
}
int gh_batch_langevin(gh_batch *b, int nsteps, double dt, double gamma, uint64_t seed,
                      double *epot, double *ekin) {
  if (!b || nsteps < 0 || !(dt > 0) || !(gamma > 0))
    return bfail(b, GH_EINVAL, "langevin needs nsteps >= 0, dt > 0, gamma > 0");
  BH(b, hipSetDevice(b->device));
  // (cap 0: the skin changed since the rows were sized)
  if (!b->forces_valid || b->cap == 0) BT(gh_batch_compute(b, nullptr, nullptr));
  ErmakC k;
  k.c0 = exp(-dt * gamma);
  k.c1 = (1.0 - k.c0) / gamma;
  k.c2 = (1.0 - k.c1 / dt) / gamma;
  k.sdr = sqrt(dt / gamma * (2.0 - (3.0 - 4.0 * k.c0 + k.c0 * k.c0) / (dt * gamma)));
  k.sdv = sqrt(1.0 - k.c0 * k.c0);
  k.crv1 = (1.0 - k.c0) * (1.0 - k.c0) / (gamma * k.sdr * k.sdv);
  k.crv2 = sqrt(1.0 - (k.crv1 * k.crv1));
  k.dt = dt;
  k.kB_ui = ghc::kB_ui();
  if (nsteps > 0) {
    const long long step0 = b->step + 1;
    BatchArgs A = bargs(b);
    k_batch_zero<<<(2 * b->nsys + GH_BWG - 1) / GH_BWG, GH_BWG, 0, b->stream>>>(b->dmax, 2 * b->nsys);
    k_batch_ermak_a<<<batch_blocks(b, 16), GH_BWG, 0, b->stream>>>(A, k, seed, step0);
    if (batch_staged(b)) {
      const size_t lds = 17 * (size_t)b->nst;
      const int bs = staged_threads(b);
      auto launch = [&](int lanes, int first, int count, hipStream_t stream) {
        A.first = first;
#define LAUNCH_LANGEVIN(SG, G) \
  k_batch_langevin<SG, G><<<count, bs, lds, stream>>>(A, k, b->skin, b->tbf0, seed, step0, nsteps)
        if (b->nt == 1 && lanes == 1) LAUNCH_LANGEVIN(true, 1);
        else if (b->nt == 1) LAUNCH_LANGEVIN(true, GH_FG);
        else if (lanes == 1) LAUNCH_LANGEVIN(false, 1);
        else LAUNCH_LANGEVIN(false, GH_FG);
#undef LAUNCH_LANGEVIN
      };
      BT(launch_split(b, bs + bs / 2, launch));
    }
    for (int st = 0; st < nsteps && !batch_staged(b); ++st) {
      const long long step = step0 + st;
      launch_rho(b, A, (int)(step & 1), 0);
      if (st + 1 < nsteps) {
        launch_force<1>(b, A, k, seed, step);
        std::swap(b->pos, b->pos_next);
        std::swap(A.pos, A.pos_next);
      } else {
        launch_force<2>(b, A, k, seed, step);
      }
    }
  }
  k_batch_energies<<<b->nsys, GH_BWG, 0, b->stream>>>(bargs(b));
  BH(b, hipGetLastError());
  b->step += nsteps;
  BT(check_flags(b));
  std::vector<double> o;
  BT(fetch_out(b, o));
  const double ui_ev = ghc::ui_ev();
  b->epot_h.resize(b->nsys);
  for (int s = 0; s < b->nsys; ++s) {
    b->epot_h[s] = o[s * OUTW] * ui_ev;
    if (epot) epot[s] = b->epot_h[s];
    if (ekin) ekin[s] = o[s * OUTW + 1] * ui_ev;
  }
  return 0;
}

// splitmix64: host stream for the Metropolis draws of the exchanges
static double smix_u01(uint64_t &st) {
  uint64_t z = (st += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return ((z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
}

int gh_batch_exchange(gh_batch *b, int nladder, int R, int *sys, int parity, uint64_t seed,
                      int *naccept) {
  if (!b || nladder <= 0 || R < 2 || !sys) return bfail(b, GH_EINVAL, "gh_batch_exchange");
  if ((int)b->epot_h.size() != b->nsys) return bfail(b, GH_ESTATE, "no energies yet");
  BH(b, hipSetDevice(b->device));
  const double kB = ghc::kB_ui(), ev_ui = ghc::ev_ui();
  std::vector<double> scale(b->nsys, 1.0);
  uint64_t st = seed;
  int acc = 0;
  for (int l = 0; l < nladder; ++l)
    for (int r = parity & 1; r + 1 < R; r += 2) {
      const int lo = sys[l * R + r], hi = sys[l * R + r + 1];
      // ReplicaExchange.f90:86-110: deltab = beta - beta_partner,
      // deltau = (E_partner - E) deltab; swap if deltau <= 0 or u < e^{-deltau}
      const double beta = 1.0 / (kB * b->T_h[lo]), betap = 1.0 / (kB * b->T_h[hi]);
      const double du = (b->epot_h[hi] - b->epot_h[lo]) * ev_ui * (beta - betap);
      bool swap = true;
      if (du > 0) swap = smix_u01(st) < exp(-du);
      if (!swap) continue;
      ++acc;
      // the configurations trade temperatures: velocities scale by sqrt(T_new/T_old)
      std::swap(b->T_h[lo], b->T_h[hi]);
      scale[lo] = sqrt(b->T_h[lo] / b->T_h[hi]);
      scale[hi] = sqrt(b->T_h[hi] / b->T_h[lo]);
      std::swap(sys[l * R + r], sys[l * R + r + 1]);
    }
  BH(b, hipMemcpyAsync(b->T, b->T_h.data(), sizeof(double) * b->nsys, hipMemcpyHostToDevice,
                       b->stream));
  BH(b, hipMemcpyAsync(b->scale, scale.data(), sizeof(double) * b->nsys, hipMemcpyHostToDevice,
                       b->stream));
  k_batch_scale<<<b->nsys, 256, 0, b->stream>>>(b->nsys, b->off, b->scale, b->vel, b->ld);
  BH(b, hipGetLastError());
  BH(b, hipStreamSynchronize(b->stream));
  if (naccept) *naccept = acc;
  return 0;
}

int gh_batch_fire(gh_batch *b, int max_iter, double dt_max, double alpha0, double fswitch,
                  double ftol, int *iters, int *converged, double *epot, double *fmax) {
  if (!b || max_iter < 0 || !(dt_max > 0)) return bfail(b, GH_EINVAL, "gh_batch_fire");
  BH(b, hipSetDevice(b->device));
  BT(batch_ready(b));
  const BatchArgs A = bargs(b);
  FireC fc;
  fc.dt_max = dt_max;
  fc.alpha0 = alpha0;
  fc.ui_ev = ghc::ui_ev();
  fc.max_iter = max_iter;
  fc.resume = 0;
  if (b->precision == GH_MIXED) {
    fc.fstop = fswitch;
    if (b->nst > 0) BT((launch_fire<true, true>(b, A, fc, b->tbf0)));
    else BT((launch_fire<true, false>(b, A, fc, b->tbd0.f)));
    fc.resume = 1;
  }
  fc.fstop = ftol;
  BT((launch_fire<false, false>(b, A, fc, b->tbd0.d)));
  BT(check_flags(b));
  b->lists_valid = true;
  b->forces_valid = false;  // the last forces may be FP64 while precision is mixed
  std::vector<double> o;
  BT(fetch_out(b, o));
  const double ui_ev = ghc::ui_ev();
  b->epot_h.resize(b->nsys);
  for (int s = 0; s < b->nsys; ++s) {
    b->epot_h[s] = o[s * OUTW] * ui_ev;
    if (epot) epot[s] = b->epot_h[s];
    if (fmax) fmax[s] = o[s * OUTW + 3];
    if (iters) iters[s] = (int)o[s * OUTW + 4];
    if (converged) converged[s] = (int)o[s * OUTW + 5];
  }
  return 0;
}

int gh_batch_get_state(gh_batch *b, double *x, double *v) {
  if (!b || !b->nsys) return bfail(b, GH_ESTATE, "no systems");
  if (x) {
    std::vector<double4> h(b->ld);
    BH(b, hipMemcpyAsync(h.data(), b->pos, sizeof(double4) * b->ld, hipMemcpyDeviceToHost,
                         b->stream));
    BH(b, hipStreamSynchronize(b->stream));
    for (int i = 0; i < b->ntot; ++i) {
      x[3 * (size_t)i] = h[i].x;
      x[3 * (size_t)i + 1] = h[i].y;
      x[3 * (size_t)i + 2] = h[i].z;
    }
  }
  if (v) {
    std::vector<double> h(3 * (size_t)b->ld);
    BH(b, hipMemcpyAsync(h.data(), b->vel, sizeof(double) * h.size(), hipMemcpyDeviceToHost,
                         b->stream));
    BH(b, hipStreamSynchronize(b->stream));
    for (int i = 0; i < b->ntot; ++i)
      for (int d = 0; d < 3; ++d) v[3 * (size_t)i + d] = h[(size_t)d * b->ld + i];
  }
  return 0;
}

}  // extern "C"
