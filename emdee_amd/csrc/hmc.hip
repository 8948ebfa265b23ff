// hmc.hip -- batched hybrid Monte Carlo of many independent Lennard-Jones
// replicas in one persistent launch.
//
// There is no counterpart in the reference: a reference user runs replicas
// one after another, each a tEmDee driven by EmDee_upload("momenta"),
// EmDee_boost / EmDee_displace / EmDee_boost (velocity Verlet, mass 1,
// pair_lj_cut) and a Metropolis test on the total energy.  Here one
// workgroup owns one replica for a whole HMC cycle (momentum refresh, an
// nsteps-long trajectory, accept/reject, restore on rejection), and one
// kernel launch runs several cycles for every replica; the launch is
// captured once in a HIP graph and replayed.
//
// Per replica (N <= 8192 atoms) the workgroup keeps, in LDS, the 32-bit
// fixed-point coordinates of the current step, so all pair gathers of the
// mixed form are LDS reads.  Pairs come from a Verlet list per replica in
// global memory (16-bit indices, column-major; kept between launches with
// its build coordinates): built from a cell list
// (counting sort into cells of side >= (rc + skin)/DIV, stencil of
// (2 DIV + 1)^3 cells) and rebuilt before a force evaluation whenever some
// atom has moved more than skin/2 since the last build -- the rule of
// neighbor_lists.f90:41-59 in its simplest sufficient form -- which also
// covers the coordinates restored after a rejected move.  A replica whose
// list would overflow its capacity (denser than LJ close packing) takes every
// atom as a candidate instead.  The pair set is the reference's: r^2 < rc^2 on the FP64
// scaled coordinates (neighbor_lists.f90:244), with FP32 candidates in the
// band around the cutoff re-tested in FP64.  Pair terms are FP32 (mixed form)
// or FP64 (plain form), accumulated per atom in FP64.
//
// Random numbers come from a counter-based generator (splitmix64 finaliser,
// Steele, Lea & Flood 2014) keyed by (seed, replica, cycle, atom, component),
// so the momenta and uniforms do not depend on the launch shape; Gaussian
// momenta use the Box-Muller transform.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <numeric>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/emdee_gpu.h"
#include "device_state.h"
#include "readback.h"

namespace emdee {

namespace {
constexpr int HMC_NMAX = 8192;   // atoms per replica
constexpr int HMC_CMAX = 6144;   // cells per replica
constexpr int HMC_HIST = 1024;   // cycles of potential-energy history
const double TWO_PI_D = 6.283185307179586;

// (padded to whole 16-byte groups, as it is loaded: without the pads the plain
// form's spills fall differently and 512 replicas take 9.4 ms a cycle for 8.8)
struct ReplicaDesc {
  int off, N, pad0, M;     // atom offset and count; cells per edge for the list build
  double L, kT;
  float K, lo, hi, pad1;   // fixed-point cutoff band (mixed form)
  double Rc2s, unit;       // FP64 scaled cutoff; L / 2^32
  double Rl2s, trig2s;     // list radius (rc + skin)^2 and (skin/2)^2, scaled units^2
};
// per-atom vectors of all replicas, component by component: x of atom i at
// [i], y at [total + i], z at [2 total + i]
struct HmcState {
  double *R, *P, *F, *Rsave, *Fsave;
  // plain form only: R / L atom by atom, so that a partner costs one 32-byte
  // gather and no division (291 replicas: 2.77 -> 2.17 ms a cycle; component
  // by component 2.50)
  double4 *S;
  size_t total;
};
constexpr double HMC_SKIN = 0.3;   // list skin (LJ units; 0.2 and 0.45 measured slower)

__host__ __device__ inline uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}
// uniform in (0, 1) for (seed, stream, counter)
__host__ __device__ inline double hmc_uniform(uint64_t seed, uint64_t stream, uint64_t counter) {
  uint64_t x = mix64(seed ^ mix64(stream * 0x9E3779B97F4A7C15ULL + counter));
  return ((double)(x >> 11) + 0.5) * (1.0 / 9007199254740992.0);
}
__host__ __device__ inline uint64_t hmc_stream(int replica, int cycle) {
  return ((uint64_t)(uint32_t)replica << 32) | (uint32_t)cycle;
}
constexpr uint64_t HMC_ACCEPT_COUNTER = 1ULL << 40;

__device__ __forceinline__ double wave_max(double v) {
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  return v;
}

template <int BS>
__device__ double block_total(double v, double* red) {
  v = wave_sum(v);
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  for (int k = 0; k < BS / 64; k++) s += red[k];
  return s;
}
}  // namespace

// LDS of a workgroup.  qz lies below qxy so that both are reached from a list
// entry (8 j, the byte offset of qxy[j]) with constant offsets.
struct HmcLds {
  unsigned int qz[HMC_NMAX];
  uint2 qxy[HMC_NMAX];
  unsigned short clist[HMC_NMAX];
  unsigned short cstart[HMC_CMAX + 2];
  unsigned int ccount2[HMC_CMAX / 2];   // 16-bit cell counts, two per word
};

// One HMC workgroup per replica.  mode 0: forces and potential energy of the
// current coordinates only; mode 1: ncycles full cycles.
//
// A step is two passes over the atoms with a barrier after each.  The force
// pass walks an atom's list and gives it both half kicks that its force takes
// part in (the end of this step and the start of the next), so forces stay in
// registers except at a trajectory's end; the drift pass moves the atom and
// renews its fixed-point coordinates.  Per step and atom that is 136 bytes of
// state instead of 370 (momenta 72, positions 48, build coordinates 16), and
// 64 more in the plain form for the scaled positions.  The list holds packets
// of eight 16-bit entries, one 16-byte load each (four, and the next in flight,
// instead of eight loads with an address and a bound test apiece), padded with
// the atom itself, which the pair terms mask.  Bound by instruction issue (54 %
// of the chip's, the tail of the launch included) and the latency of one
// replica's 16 wavefronts per CU: the mixed form spends 46 % of its time in the
// force passes and 44 % in the 1.7 list builds of a cycle, the plain form 76 and
// 19 %.  512 replicas of 256 to 8,192 atoms, ten steps: 4.41 -> 3.82 ms a cycle.
// Partners read two, four or eight at a time and
// masked instead of branched over: 3.93, 4.11 and 4.04 ms with 1,024 threads,
// 10 % less with 256, which no replica set of these sizes chooses.
template <int BS, int DIV, bool MIXED>
__global__ void __launch_bounds__(BS)
k_hmc(const ReplicaDesc* __restrict__ desc, const int* __restrict__ order, HmcState st, double* __restrict__ U,
      int* __restrict__ cycle, long long* __restrict__ accepted, double* __restrict__ lastDH, double dt, int nsteps,
      uint64_t seed, int ncycles, int mode, unsigned short* __restrict__ nlist, unsigned short* __restrict__ nnb,
      uint4* __restrict__ qbuild, int cap, int* __restrict__ lstate, double* __restrict__ Uhist, int histLen) {
  __shared__ HmcLds s;
  __shared__ double red[BS / 64];
  __shared__ int scanTmp[BS / 64];
  __shared__ int cycleNow;
  __shared__ double Unow;
  __shared__ int listState;   // 0: no valid list, 1: valid list, 2: overflow (every atom)

  const int r = order[blockIdx.x];
  const ReplicaDesc d = desc[r];
  const int N = d.N;
  const size_t T = st.total;   // stride between the components of a vector array
  double* __restrict__ Rr = st.R + d.off;
  double* __restrict__ Pr = st.P + d.off;
  double* __restrict__ Fr = st.F + d.off;
  double* __restrict__ Rs = st.Rsave + d.off;
  double* __restrict__ Fs = st.Fsave + d.off;
  double4* __restrict__ Sr = MIXED ? nullptr : st.S + d.off;
  uint4* __restrict__ qb = qbuild + d.off;
  unsigned short* __restrict__ list = nlist + (size_t)d.off * cap;
  const double L = d.L, hdt = 0.5 * dt;
  const float c0 = 4.0f, c1 = 24.0f, c2 = 1.0f;   // pair_lj_cut with epsilon = sigma = 1

  // cell list of the current coordinates (fixed point in LDS)
  auto count_of = [&](int c) { return (int)((s.ccount2[c >> 1] >> ((c & 1) * 16)) & 0xffffu); };
  auto bump = [&](int c) {   // returns the previous count of cell c
    unsigned int old = atomicAdd(&s.ccount2[c >> 1], 1u << ((c & 1) * 16));
    return (int)((old >> ((c & 1) * 16)) & 0xffffu);
  };
  // fixed-point coordinates of x (atom i) into LDS; returns the squared
  // displacement since the last list build (scaled units^2)
  auto place = [&](int i, const double (&x)[3]) __attribute__((always_inline)) {
    unsigned int u[3];
    if (!MIXED) Sr[i] = make_double4(x[0] / L, x[1] / L, x[2] / L, 0.0);
    for (int c = 0; c < 3; c++) {
      double v = x[c] / L, f = v - floor(v);
      u[c] = (unsigned int)(unsigned long long)llrint(f * 4294967296.0);
    }
    s.qxy[i] = make_uint2(u[0], u[1]);
    s.qz[i] = u[2];
    uint4 b = qb[i];
    double ex = (double)(int)(u[0] - b.x), ey = (double)(int)(u[1] - b.y), ez = (double)(int)(u[2] - b.z);
    return (ex * ex + ey * ey + ez * ez) * (1.0 / 18446744073709551616.0);
  };
  auto block_max = [&](double m) {
    m = wave_max(m);
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = m;
    __syncthreads();
    double t = 0.0;
    for (int k = 0; k < BS / 64; k++) t = fmax(t, red[k]);
    return t;
  };
  // cell list of the coordinates in LDS, cells of side L / Mc
  auto build_cells = [&](int Mc) {
    const int ncc = Mc * Mc * Mc;
    for (int c = threadIdx.x; c < (ncc + 1) / 2; c += BS) s.ccount2[c] = 0;
    __syncthreads();
    auto cell_of = [&](int i) {
      const uint2 xy = s.qxy[i];
      return (int)(((unsigned long long)xy.x * Mc) >> 32) +
             Mc * ((int)(((unsigned long long)xy.y * Mc) >> 32) + Mc * (int)(((unsigned long long)s.qz[i] * Mc) >> 32));
    };
    for (int i = threadIdx.x; i < N; i += BS) bump(cell_of(i));
    __syncthreads();
    // exclusive scan of the counts: per-thread chunk sums, a scan over the
    // wave and over the waves' totals, chunks
    int chunk = (ncc + BS - 1) / BS, c0i = min(ncc, (int)threadIdx.x * chunk), c1i = min(ncc, c0i + chunk);
    int local = 0;
    for (int c = c0i; c < c1i; c++) local += count_of(c);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int incl = local;
    for (int off = 1; off < 64; off <<= 1) {
      int v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    if (lane == 63) scanTmp[w] = incl;
    __syncthreads();
    int run = incl - local;
    for (int k = 0; k < w; k++) run += scanTmp[k];
    for (int c = c0i; c < c1i; c++) { s.cstart[c] = (unsigned short)run; run += count_of(c); }
    if (threadIdx.x == 0) s.cstart[ncc] = (unsigned short)N;
    __syncthreads();
    for (int c = threadIdx.x; c < (ncc + 1) / 2; c += BS) s.ccount2[c] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < N; i += BS) {
      int c = cell_of(i);
      s.clist[s.cstart[c] + bump(c)] = (unsigned short)i;
    }
    __syncthreads();
  };
  // gives visit, for atom i, the ranges of cell-sorted places (s.clist) of the
  // cells within Mc-cell reach that can lie within sqrt(R2s) (scaled units) of
  // it, culled row by row; the atom itself is among them.  Mc < 2 DIV + 1: one
  // cell holds every atom.
  auto walk = [&](int i, int Mc, double R2s, auto&& visit) __attribute__((always_inline)) {
    const int w = (Mc >= 2 * DIV + 1) ? DIV : 0;
    // cutoff^2 in cell units, with margins far above the FP32 rounding of the
    // culling (which can then only keep extra cells)
    const float rcell2 = (float)(R2s * (double)Mc * (double)Mc * (1.0 + 1e-5) + 1e-5);
    const uint2 xy = s.qxy[i];
    unsigned long long px = (unsigned long long)xy.x * Mc, py = (unsigned long long)xy.y * Mc,
                       pz = (unsigned long long)s.qz[i] * Mc;
    int cx = (int)(px >> 32), cy = (int)(py >> 32), cz = (int)(pz >> 32);
    // position of atom i inside its cell, in cell units
    const float ox = (float)(unsigned int)px * 2.3283064e-10f, oy = (float)(unsigned int)py * 2.3283064e-10f,
                oz = (float)(unsigned int)pz * 2.3283064e-10f;
    // cells are numbered x fastest, so the cells x-w..x+w of one (y, z) row
    // are one contiguous slot range (two where the row wraps, visited in
    // the order of increasing dx); w = 0 takes every atom at once
    for (int dz = -w; dz <= w; dz++) {
      int z = cz + dz; z = z < 0 ? z + Mc : (z >= Mc ? z - Mc : z);
      float gz = fmaxf(dz > 0 ? dz - oz : (dz < 0 ? oz - dz - 1 : 0.0f), 0.0f);
      for (int dy = -w; dy <= w; dy++) {
        int y = cy + dy; y = y < 0 ? y + Mc : (y >= Mc ? y - Mc : y);
        int base = Mc * (y + Mc * z), xa = cx - w, xb = cx + w;
        if (w > 0) {   // rows and cells beyond the cutoff sphere hold no partner
          float gy = fmaxf(dy > 0 ? dy - oy : (dy < 0 ? oy - dy - 1 : 0.0f), 0.0f);
          float rem = rcell2 - gy * gy - gz * gz;
          if (rem <= 0.0f) continue;
          float ex = sqrtf(rem) + 1e-4f;
          xa = cx + max((int)floorf(ox - ex), -w);
          xb = cx + min((int)floorf(ox + ex), w);
        }
        int r0a, r0b, r1a = 0, r1b = -1;   // cell ranges [r0a, r0b] then [r1a, r1b]
        if (xa < 0) { r0a = xa + Mc; r0b = Mc - 1; r1a = 0; r1b = xb; }
        else if (xb >= Mc) { r0a = xa; r0b = Mc - 1; r1a = 0; r1b = xb - Mc; }
        else { r0a = xa; r0b = xb; }
        for (int part = 0; part < 2; part++) {
          int ca = part == 0 ? r0a : r1a, cb = part == 0 ? r0b : r1b;
          if (cb < ca) continue;
          visit((w == 0) ? 0 : (int)s.cstart[base + ca], (w == 0) ? N : (int)s.cstart[base + cb + 1]);
        }
      }
    }
  };
  // Verlet list at radius sqrt(d.Rl2s) from the coordinates in LDS (every
  // atom within it, in walk order; the FP32 test keeps a margin, so the list
  // may hold a few more); the build coordinates are kept for the trigger.
  // Entry n of atom i is 8 j at list[8 ((n/8) N + i) + n%8]; four entries are
  // gathered in a register pair and stored together, and the last packet is
  // padded with the atom itself.
  // Measured (same replicas): one 16-bit store per entry 4.00 ms a cycle, this
  // 3.82; atoms taken in cell order, whose lanes read the same candidates but
  // store apart, 4.35; candidates read four at a time 4.48.
  auto build_list = [&]() {
    build_cells(d.M);
    const float rl2 = (float)(d.Rl2s * 18446744073709551616.0 * (1.0 + 1e-4));
    int over = 0;
    for (int i = threadIdx.x; i < N; i += BS) {
      const uint2 xy = s.qxy[i];
      const unsigned int wi = s.qz[i];
      int n = 0;
      unsigned int lo = 0, hi = 0;   // the last four entries, the oldest lowest
      unsigned short* __restrict__ li = list + 8 * (size_t)i;
      auto put = [&](int j) __attribute__((always_inline)) {
        lo = __builtin_amdgcn_alignbit(hi, lo, 16);
        hi = __builtin_amdgcn_alignbit((unsigned int)(8 * j), hi, 16);
        if ((n & 3) == 3 && n < cap)
          *reinterpret_cast<uint2*>(li + 8 * (size_t)(n >> 3) * N + (n & 4)) = make_uint2(lo, hi);
        n++;
      };
      walk(i, d.M, d.Rl2s, [&](int a, int b) __attribute__((always_inline)) {
        for (int q = a; q < b; q++) {
          const int j = s.clist[q];
          const uint2 v = s.qxy[j];
          float ddx = (float)(int)(xy.x - v.x), ddy = (float)(int)(xy.y - v.y), ddz = (float)(int)(wi - s.qz[j]);
          float r2 = ddx * ddx + ddy * ddy + ddz * ddz;
          if (r2 < rl2 && j != i) put(j);
        }
      });
      const int cnt = n;
      while (n & 7) put(i);
      nnb[d.off + i] = (unsigned short)min(cnt, cap);
      qb[i] = make_uint4(xy.x, xy.y, wi, 0u);
      over |= cnt > cap;
    }
    // any overflow: this replica takes every atom from now on
    over = __syncthreads_or(over);
    if (threadIdx.x == 0) listState = over ? 2 : 1;
    __syncthreads();
  };

  // force on atom i from its partners, and with E_ true its pair energies
  auto force_of = [&](int i, bool useList, auto E_, double (&f)[3], double& ei) __attribute__((always_inline)) {
    constexpr bool WANT_E = decltype(E_)::value;
    const uint2 xy = s.qxy[i];
    const unsigned int wi = s.qz[i], io = 8u * (unsigned int)i;
    double fx = 0, fy = 0, fz = 0, e = 0;
    double xi[3] = { 0, 0, 0 };
    if (!MIXED) { const double4 a = Sr[i]; xi[0] = a.x; xi[1] = a.y; xi[2] = a.z; }
    // o: 8 j
    auto pair = [&](unsigned int o) __attribute__((always_inline)) {
      // the pair's r^2 in scaled units and its separation, in FP64
      auto exact = [&](double (&q)[3]) {
        const size_t j = o >> 3;
        if (MIXED) {
          for (int c = 0; c < 3; c++) q[c] = Rr[c * T + i] / L - Rr[c * T + j] / L;
        } else {
          const double4 b = Sr[j];
          q[0] = xi[0] - b.x; q[1] = xi[1] - b.y; q[2] = xi[2] - b.z;
        }
        for (int c = 0; c < 3; c++) q[c] = q[c] - rint(q[c]);
        double q2;
        {
#pragma clang fp contract(off)
          q2 = q[0] * q[0] + q[1] * q[1] + q[2] * q[2];
        }
        return q2;
      };
      if (MIXED) {
        // the atom itself (zero separation) is masked, not branched over
        const uint2 v = *reinterpret_cast<const uint2*>(reinterpret_cast<const char*>(s.qxy) + o);
        const unsigned int vz = *reinterpret_cast<const unsigned int*>(reinterpret_cast<const char*>(s.qz) + (o >> 1));
        float ddx = (float)(int)(xy.x - v.x), ddy = (float)(int)(xy.y - v.y), ddz = (float)(int)(wi - vz);
        float r2 = ddx * ddx + ddy * ddy + ddz * ddz;
        bool in = r2 < d.lo && o != io;
        if (r2 >= d.lo && r2 < d.hi) {
          double q[3];
          in = exact(q) < d.Rc2s;
        }
        if (in) {
          float invR2 = d.K * __builtin_amdgcn_rcpf(r2);
          float sr2 = c2 * invR2, sr6 = sr2 * sr2 * sr2;
          float W = c1 * sr6 * (sr6 + sr6 - 1.0f);
          float g = W * invR2;
          fx += (double)(g * ddx);
          fy += (double)(g * ddy);
          fz += (double)(g * ddz);
          if (WANT_E) e += (double)(c0 * sr6 * (sr6 - 1.0f));
        }
      } else {
        if (o == io) return;
        double q[3];
        const double q2 = exact(q);
        if (q2 < d.Rc2s) {
          double invR2 = 1.0 / (L * L * q2);
          double sr2 = invR2, sr6 = sr2 * sr2 * sr2, sr12 = sr6 * sr6;
          double W = 24.0 * (sr12 + sr12 - sr6);
          double g = W * invR2;
          fx += g * q[0];
          fy += g * q[1];
          fz += g * q[2];
          if (WANT_E) e += 4.0 * (sr12 - sr6);
        }
      }
    };
    if (useList) {
      // packets of eight, the next one loaded before this one's pairs
      const int np = ((int)nnb[d.off + i] + 7) >> 3;
      const uint4* __restrict__ lp = reinterpret_cast<const uint4*>(list) + i;
      uint4 nx = np > 0 ? lp[0] : make_uint4(0, 0, 0, 0);
      for (int p = 0; p < np; p++) {
        const uint4 c = nx;
        if (p + 1 < np) nx = lp[(size_t)(p + 1) * N];
        const unsigned int w[4] = { c.x, c.y, c.z, c.w };
#pragma unroll
        for (int u = 0; u < 4; u++) {
          pair(w[u] & 0xffffu);
          pair(w[u] >> 16);
        }
      }
    } else {
      // a list that would overflow its capacity (more neighbours within
      // rc + skin than LJ atoms at close packing hold): every atom
      for (int j = 0; j < N; j++) pair(8u * (unsigned int)j);
    }
    const double sc = MIXED ? d.unit : L;
    f[0] = sc * fx; f[1] = sc * fy; f[2] = sc * fz;
    ei = e;
  };
  // the list for the coordinates in LDS: rebuilt when it is missing or an atom
  // moved more than skin/2
  auto check_list = [&](double moved) {
    if (listState != 2 && (listState == 0 || moved > d.trig2s)) build_list();
    return listState == 1;
  };

  // the list and its build coordinates persist between launches (written
  // together), so a list still valid for the current coordinates is kept
  if (threadIdx.x == 0) listState = lstate[r];
  __syncthreads();
  if (mode == 0) {
    double m = 0.0;
    for (int i = threadIdx.x; i < N; i += BS) {
      const double x[3] = { Rr[i], Rr[T + i], Rr[2 * T + i] };
      m = fmax(m, place(i, x));
    }
    const bool useList = check_list(block_max(m));
    double e = 0.0;
    for (int i = threadIdx.x; i < N; i += BS) {
      double f[3], ei;
      force_of(i, useList, std::true_type(), f, ei);
      for (int c = 0; c < 3; c++) Fr[c * T + i] = f[c];
      e += ei;
    }
    e = 0.5 * block_total<BS>(e, red);
    if (threadIdx.x == 0) { U[r] = e; lstate[r] = listState; }
    return;
  }
  const double sq = sqrt(d.kT);
  // per-replica scalars live in LDS for the whole launch
  if (threadIdx.x == 0) { cycleNow = cycle[r]; Unow = U[r]; }
  __syncthreads();
  for (int cyc = 0; cyc < ncycles; cyc++) {
    const int cnum = cycleNow;
    const uint64_t stream = hmc_stream(r, cnum);
    // momentum refresh (mass 1), saved state, and the first half kick and drift
    double k = 0.0, moved = 0.0;
    for (int i = threadIdx.x; i < N; i += BS) {
      double x[3];
      for (int c = 0; c < 3; c++) {
        double u1 = hmc_uniform(seed, stream, 6ULL * i + 2 * c), u2 = hmc_uniform(seed, stream, 6ULL * i + 2 * c + 1);
        double p = sq * (sqrt(-2.0 * log(u1)) * cos(TWO_PI_D * u2));
        x[c] = Rr[c * T + i];
        const double f = Fr[c * T + i];
        Rs[c * T + i] = x[c];
        Fs[c * T + i] = f;
        k += p * p;
        if (nsteps > 0) {
          p = p + hdt * f;
          x[c] = x[c] + dt * p;
          Pr[c * T + i] = p;
          Rr[c * T + i] = x[c];
        }
      }
      if (nsteps > 0) moved = fmax(moved, place(i, x));
    }
    const double U0 = Unow, H0 = U0 + 0.5 * block_total<BS>(k, red);
    double U1 = U0, K1 = k;
    for (int st = 0; st < nsteps; st++) {
      const bool useList = check_list(block_max(moved));
      if (st < nsteps - 1) {
        // force, the end of this step and the first half kick of the next
        for (int i = threadIdx.x; i < N; i += BS) {
          double f[3], ei;
          force_of(i, useList, std::false_type(), f, ei);
          for (int c = 0; c < 3; c++) {
            double p = Pr[c * T + i];
            p = p + hdt * f[c];
            p = p + hdt * f[c];
            Pr[c * T + i] = p;
          }
        }
        __syncthreads();   // every force of the old coordinates before any drift
        moved = 0.0;
        for (int i = threadIdx.x; i < N; i += BS) {
          double x[3];
          for (int c = 0; c < 3; c++) {
            x[c] = Rr[c * T + i] + dt * Pr[c * T + i];
            Rr[c * T + i] = x[c];
          }
          moved = fmax(moved, place(i, x));
        }
      } else {
        double e = 0.0;
        K1 = 0.0;
        for (int i = threadIdx.x; i < N; i += BS) {
          double f[3], ei, p[3];
          force_of(i, useList, std::true_type(), f, ei);
          for (int c = 0; c < 3; c++) {
            Fr[c * T + i] = f[c];
            p[c] = Pr[c * T + i] + hdt * f[c];
          }
          e += ei;
          K1 += p[0] * p[0] + p[1] * p[1] + p[2] * p[2];
        }
        U1 = 0.5 * block_total<BS>(e, red);
      }
    }
    const double H1 = U1 + 0.5 * block_total<BS>(K1, red);
    const double dH = H1 - H0;
    const bool accept = dH <= 0.0 || hmc_uniform(seed, stream, HMC_ACCEPT_COUNTER) < exp(-dH / d.kT);
    if (!accept)
      for (int i = threadIdx.x; i < N; i += BS)
        for (int c = 0; c < 3; c++) { Rr[c * T + i] = Rs[c * T + i]; Fr[c * T + i] = Fs[c * T + i]; }
    __syncthreads();
    if (threadIdx.x == 0) {
      Unow = accept ? U1 : U0;
      cycleNow = cnum + 1;
      U[r] = Unow;
      accepted[r] += accept ? 1 : 0;
      lastDH[r] = dH;
      cycle[r] = cycleNow;
      Uhist[(size_t)(cnum % histLen) * gridDim.x + r] = Unow;   // the grid holds one workgroup per replica
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) lstate[r] = listState;
}

// Elements first .. first + count of all replicas' coordinates, atom by atom,
// to pinned host memory
__global__ void __launch_bounds__(BLOCK)
k_hmc_coords(double* __restrict__ host, const double* __restrict__ R, size_t total, size_t first, size_t count) {
  const size_t x = (size_t)blockIdx.x * BLOCK + threadIdx.x, e = first + x, atom = e / 3;
  if (x < count) host[x] = R[(e - 3 * atom) * total + atom];
}
__global__ void k_hmc_post(unsigned long long* hostSeq, unsigned long long seq) {
  __threadfence_system();
  *(volatile unsigned long long*)hostSeq = seq;
}

}  // namespace emdee

// ------------------------------------------------------------ host side

using namespace emdee;

struct EmDeeHMC {
  int nrep = 0, total = 0, nsteps = 0, cyclesPerLaunch = 1, precision = 1;
  double rc = 2.5, dt = 0.005;
  uint64_t seed = 0;
  hipStream_t stream = nullptr;
  std::vector<ReplicaDesc> hdesc;
  std::vector<int> offsets, hN;
  DBuf<ReplicaDesc> desc;
  DBuf<int> order, cycle;
  DBuf<double> R, P, F, Rsave, Fsave;   // [3][total]
  DBuf<double4> S;
  // pinned coherent host memory that EmDeeHMC_get reads through: HMC_RING
  // doubles and the number of the last chunk posted
  double* ring = nullptr;
  double* ringDev = nullptr;
  unsigned long long posted = 0;
  DBuf<double> U, lastDH;
  DBuf<long long> accepted;
  int cap = 0;                   // Verlet-list entries per atom
  DBuf<unsigned short> nlist, nnb;
  DBuf<uint4> qbuild;
  DBuf<int> lstate;              // per replica: 0 no list, 1 valid list, 2 overflow
  DBuf<double> Uhist;            // potential energy after each of the last HMC_HIST cycles [cycle % HMC_HIST][replica]
  int variant = -1;            // index into the variant table
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  double tuneMs[6] = { 0, 0, 0, 0, 0, 0 };
};

namespace {
using HmcKernel = void (*)(const ReplicaDesc*, const int*, HmcState, double*, int*, long long*, double*, double, int,
                           uint64_t, int, int, unsigned short*, unsigned short*, uint4*, int, int*, double*, int);
struct Variant { int bs, div; HmcKernel mixed, plain; };
const Variant VARIANTS[] = {
  { 256, 1, k_hmc<256, 1, true>, k_hmc<256, 1, false> },
  { 512, 1, k_hmc<512, 1, true>, k_hmc<512, 1, false> },
  { 1024, 1, k_hmc<1024, 1, true>, k_hmc<1024, 1, false> },
  { 256, 2, k_hmc<256, 2, true>, k_hmc<256, 2, false> },
  { 512, 2, k_hmc<512, 2, true>, k_hmc<512, 2, false> },
  { 1024, 2, k_hmc<1024, 2, true>, k_hmc<1024, 2, false> },
};
constexpr int NVARIANTS = 6;
constexpr size_t HMC_RING = 4 * READ_CHUNK;   // 8 MB

// cells per edge: of side at least (rc + skin) / div, or one cell
double edge_cells(const EmDeeHMC* h, const ReplicaDesc& d, int div) {
  const double M = std::floor(div * d.L / (h->rc + HMC_SKIN));
  return M >= 2 * div + 1 ? M : 1.0;
}

bool variant_fits(const EmDeeHMC* h, int v) {
  for (const ReplicaDesc& d : h->hdesc) {
    const double M = edge_cells(h, d, VARIANTS[v].div);
    if (M * M * M > HMC_CMAX) return false;
  }
  return true;
}

void set_cells(EmDeeHMC* h, int div) {
  for (ReplicaDesc& d : h->hdesc) d.M = (int)edge_cells(h, d, div);
  HIP_CHECK(hipMemcpy(h->desc.p, h->hdesc.data(), sizeof(ReplicaDesc) * h->nrep, hipMemcpyHostToDevice));
}

void launch(EmDeeHMC* h, int v, int ncycles, int mode) {
  const Variant& var = VARIANTS[v];
  HmcKernel k = h->precision ? var.mixed : var.plain;
  const HmcState st{ h->R.p, h->P.p, h->F.p, h->Rsave.p, h->Fsave.p, h->S.p, (size_t)h->total };
  hipLaunchKernelGGL(k, dim3(h->nrep), dim3(var.bs), 0, h->stream, h->desc.p, h->order.p, st, h->U.p, h->cycle.p,
                     h->accepted.p, h->lastDH.p, h->dt, h->nsteps, h->seed, ncycles, mode, h->nlist.p, h->nnb.p,
                     h->qbuild.p, h->cap, h->lstate.p, h->Uhist.p, HMC_HIST);
  launch_check("hmc");
}
}  // namespace

extern "C" {

EmDeeHMC* EmDeeHMC_create(int nrep, const int* natoms, const double* box, const double* kT, const double* R,
                          double rc, double dt, int nsteps, unsigned long long seed, int precision) {
  const char* task = "batched HMC set-up";
  if (nrep < 1) fatal(task, "no replicas");
  EmDeeHMC* h = new EmDeeHMC();
  h->nrep = nrep; h->rc = rc; h->dt = dt; h->nsteps = nsteps; h->seed = seed; h->precision = precision ? 1 : 0;
  HIP_CHECK(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
  h->offsets.resize(nrep);
  h->hN.assign(natoms, natoms + nrep);
  h->hdesc.resize(nrep);
  int off = 0;
  for (int r = 0; r < nrep; r++) {
    if (natoms[r] < 2 || natoms[r] > HMC_NMAX) fatal(task, "replica sizes must be between 2 and 8192 atoms");
    if (box[r] < 2.0 * rc) fatal(task, "replica box shorter than twice the cutoff");
    ReplicaDesc& d = h->hdesc[r];
    d.off = off; d.N = natoms[r]; d.L = box[r]; d.kT = kT[r];
    double two32 = 4294967296.0, rc2s = (rc * rc) / (box[r] * box[r]), rc2u = rc2s * two32 * two32;
    d.K = (float)(two32 * two32 / (box[r] * box[r]));
    // FP32 rounding plus the quantisation of the fixed-point coordinates
    const double q = 1.0 / two32, band = 2e-6 + 4.0 * q / std::sqrt(rc2s) + 3.0 * q * q / rc2s;
    d.lo = (float)(rc2u * (1.0 - band));
    d.hi = (float)(rc2u * (1.0 + band));
    d.Rc2s = rc2s;
    d.unit = box[r] / two32;
    const double rl = rc + HMC_SKIN;
    d.Rl2s = (rl * rl) / (box[r] * box[r]);
    d.trig2s = (0.25 * HMC_SKIN * HMC_SKIN) / (box[r] * box[r]);
    h->offsets[r] = off;
    off += natoms[r];
  }
  h->total = off;
  // list capacity: 1.6 times the mean count at the densest replica's
  // density, plus room for fluctuations (a replica that overflows takes
  // every atom instead), in whole packets of eight
  {
    double rho = 0.0, rl = rc + HMC_SKIN;
    for (int r = 0; r < nrep; r++) rho = std::max(rho, natoms[r] / (box[r] * box[r] * box[r]));
    int cap = (int)(1.6 * 4.18879020478639 * rl * rl * rl * rho) + 24;
    h->cap = std::min(((cap + 7) / 8) * 8, HMC_NMAX);
  }
  // largest replicas first: the dispatcher hands out workgroups in order
  std::vector<int> ord(nrep);
  std::iota(ord.begin(), ord.end(), 0);
  std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return natoms[a] > natoms[b]; });
  h->desc.alloc(nrep); h->order.alloc(nrep); h->cycle.alloc(nrep); h->U.alloc(nrep); h->lastDH.alloc(nrep);
  h->accepted.alloc(nrep);
  for (DBuf<double>* b : { &h->R, &h->P, &h->F, &h->Rsave, &h->Fsave }) b->alloc(3 * (size_t)off);
  if (!h->precision) h->S.alloc(off);
  h->nlist.alloc((size_t)off * h->cap); h->nnb.alloc(off); h->qbuild.alloc(off); h->lstate.alloc(nrep);
  h->Uhist.alloc((size_t)HMC_HIST * nrep);
  HIP_CHECK(hipHostMalloc((void**)&h->ring, sizeof(double) * (HMC_RING + 8), hipHostMallocCoherent));
  HIP_CHECK(hipHostGetDevicePointer((void**)&h->ringDev, h->ring, 0));
  *reinterpret_cast<unsigned long long*>(h->ring + HMC_RING) = 0;
  std::vector<double> Rc(3 * (size_t)off);
  for (int i = 0; i < off; i++) for (int c = 0; c < 3; c++) Rc[(size_t)c * off + i] = R[3 * (size_t)i + c];
  HIP_CHECK(hipMemcpy(h->R.p, Rc.data(), sizeof(double) * Rc.size(), hipMemcpyHostToDevice));
  HIP_CHECK(hipMemcpy(h->order.p, ord.data(), sizeof(int) * nrep, hipMemcpyHostToDevice));
  std::vector<int> zeroI(nrep, 0);
  std::vector<long long> zeroL(nrep, 0);
  HIP_CHECK(hipMemcpy(h->cycle.p, zeroI.data(), sizeof(int) * nrep, hipMemcpyHostToDevice));
  HIP_CHECK(hipMemcpy(h->lstate.p, zeroI.data(), sizeof(int) * nrep, hipMemcpyHostToDevice));
  HIP_CHECK(hipMemcpy(h->accepted.p, zeroL.data(), sizeof(long long) * nrep, hipMemcpyHostToDevice));
  // default variant: the first that fits; forces of the initial coordinates
  for (int v = 0; v < NVARIANTS; v++)
    if (variant_fits(h, v)) { h->variant = v; break; }
  if (h->variant < 0) fatal(task, "replica boxes too large for the cell table");
  set_cells(h, VARIANTS[h->variant].div);
  launch(h, h->variant, 0, 0);
  HIP_CHECK(hipStreamSynchronize(h->stream));
  return h;
}

// Autotuner: times one cycle of every variant that fits (block size x cell
// division) from the same state, restores the state, and keeps the fastest.
int EmDeeHMC_tune(EmDeeHMC* h) {
  int n = h->total, nr = h->nrep;
  DBuf<double> R0, F0;
  DBuf<double> U0;
  DBuf<int> c0;
  DBuf<long long> a0;
  R0.alloc(3 * (size_t)n); F0.alloc(3 * (size_t)n); U0.alloc(nr); c0.alloc(nr); a0.alloc(nr);
  HIP_CHECK(hipMemcpyAsync(R0.p, h->R.p, 3 * sizeof(double) * n, hipMemcpyDeviceToDevice, h->stream));
  HIP_CHECK(hipMemcpyAsync(F0.p, h->F.p, 3 * sizeof(double) * n, hipMemcpyDeviceToDevice, h->stream));
  HIP_CHECK(hipMemcpyAsync(U0.p, h->U.p, sizeof(double) * nr, hipMemcpyDeviceToDevice, h->stream));
  HIP_CHECK(hipMemcpyAsync(c0.p, h->cycle.p, sizeof(int) * nr, hipMemcpyDeviceToDevice, h->stream));
  HIP_CHECK(hipMemcpyAsync(a0.p, h->accepted.p, sizeof(long long) * nr, hipMemcpyDeviceToDevice, h->stream));
  hipEvent_t e0, e1;
  HIP_CHECK(hipEventCreate(&e0));
  HIP_CHECK(hipEventCreate(&e1));
  int best = -1;
  double bestMs = 1e300;
  for (int v = 0; v < NVARIANTS; v++) {
    h->tuneMs[v] = -1.0;
    if (!variant_fits(h, v)) continue;
    set_cells(h, VARIANTS[v].div);
    HIP_CHECK(hipEventRecord(e0, h->stream));
    launch(h, v, 1, 1);
    HIP_CHECK(hipEventRecord(e1, h->stream));
    HIP_CHECK(hipEventSynchronize(e1));
    float ms = 0;
    HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
    h->tuneMs[v] = ms;
    if (ms < bestMs) { bestMs = ms; best = v; }
    HIP_CHECK(hipMemcpyAsync(h->R.p, R0.p, 3 * sizeof(double) * n, hipMemcpyDeviceToDevice, h->stream));
    HIP_CHECK(hipMemcpyAsync(h->F.p, F0.p, 3 * sizeof(double) * n, hipMemcpyDeviceToDevice, h->stream));
    HIP_CHECK(hipMemcpyAsync(h->U.p, U0.p, sizeof(double) * nr, hipMemcpyDeviceToDevice, h->stream));
    HIP_CHECK(hipMemcpyAsync(h->cycle.p, c0.p, sizeof(int) * nr, hipMemcpyDeviceToDevice, h->stream));
    HIP_CHECK(hipMemcpyAsync(h->accepted.p, a0.p, sizeof(long long) * nr, hipMemcpyDeviceToDevice, h->stream));
  }
  HIP_CHECK(hipStreamSynchronize(h->stream));
  HIP_CHECK(hipEventDestroy(e0));
  HIP_CHECK(hipEventDestroy(e1));
  R0.release(); F0.release(); U0.release(); c0.release(); a0.release();
  h->variant = best;
  set_cells(h, VARIANTS[best].div);
  if (h->exec) { (void)hipGraphExecDestroy(h->exec); h->exec = nullptr; }
  if (h->graph) { (void)hipGraphDestroy(h->graph); h->graph = nullptr; }
  return best;
}

// Runs `launches` graph launches of `cycles` HMC cycles each (the graph is
// captured on the first call and whenever the number of cycles changes).
void EmDeeHMC_run(EmDeeHMC* h, int launches, int cycles) {
  if (cycles < 1 || launches < 1) return;
  if (!h->exec || cycles != h->cyclesPerLaunch) {
    if (h->exec) { (void)hipGraphExecDestroy(h->exec); h->exec = nullptr; }
    if (h->graph) { (void)hipGraphDestroy(h->graph); h->graph = nullptr; }
    h->cyclesPerLaunch = cycles;
    HIP_CHECK(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
    launch(h, h->variant, cycles, 1);
    HIP_CHECK(hipStreamEndCapture(h->stream, &h->graph));
    HIP_CHECK(hipGraphInstantiate(&h->exec, h->graph, nullptr, nullptr, 0));
  }
  for (int k = 0; k < launches; k++) HIP_CHECK(hipGraphLaunch(h->exec, h->stream));
}

void EmDeeHMC_synchronize(EmDeeHMC* h) { HIP_CHECK(hipStreamSynchronize(h->stream)); }

// Coordinates (3 * total atoms, replica order), potential energies, accepted
// moves and the last energy change of every replica; any pointer may be null.
void EmDeeHMC_get(EmDeeHMC* h, double* R, double* U, long long* accepted, double* lastDH) {
  HIP_CHECK(hipStreamSynchronize(h->stream));
  if (R) {
    const volatile unsigned long long* seq = reinterpret_cast<unsigned long long*>(h->ring + HMC_RING);
    const ReadRing ring{ h->ring, h->ringDev, seq, HMC_RING };
    const size_t T = h->total;
    read_back(R, 3 * T, ring, h->posted + 1, [&](size_t first, size_t count, double* to, unsigned long long number) {
      hipLaunchKernelGGL(k_hmc_coords, dim3(div_up((long)count, BLOCK)), dim3(BLOCK), 0, h->stream, to, h->R.p, T, first,
                         count);
      hipLaunchKernelGGL(k_hmc_post, dim3(1), dim3(1), 0, h->stream,
                         reinterpret_cast<unsigned long long*>(h->ringDev + HMC_RING), number);
      launch_check("hmc coordinates");
      h->posted = number;
    }, [&](unsigned long long number) {
      for (int k = 0; k < (1 << 20) && *seq < number; k++) __builtin_ia32_pause();
      if (*seq < number) HIP_CHECK(hipStreamSynchronize(h->stream));
      if (*seq < number) fatal("batched HMC", "the coordinates did not arrive");
      std::atomic_thread_fence(std::memory_order_acquire);
    });
  }
  if (U) HIP_CHECK(hipMemcpy(U, h->U.p, sizeof(double) * h->nrep, hipMemcpyDeviceToHost));
  if (accepted) HIP_CHECK(hipMemcpy(accepted, h->accepted.p, sizeof(long long) * h->nrep, hipMemcpyDeviceToHost));
  if (lastDH) HIP_CHECK(hipMemcpy(lastDH, h->lastDH.p, sizeof(double) * h->nrep, hipMemcpyDeviceToHost));
}

// Potential energies after each of the last `cycles` cycles (at most 1024
// and at most the cycles run), oldest first: U[c * nrep + replica].  Returns
// the number of cycles copied.  Every replica runs the same cycles, so the
// first replica's cycle counter numbers them.
int EmDeeHMC_history(EmDeeHMC* h, int cycles, double* U) {
  HIP_CHECK(hipStreamSynchronize(h->stream));
  int done = 0;
  HIP_CHECK(hipMemcpy(&done, h->cycle.p, sizeof(int), hipMemcpyDeviceToHost));
  int n = std::max(0, std::min({ cycles, HMC_HIST, done }));
  if (n == 0 || !U) return n;
  std::vector<double> all((size_t)HMC_HIST * h->nrep);
  HIP_CHECK(hipMemcpy(all.data(), h->Uhist.p, sizeof(double) * all.size(), hipMemcpyDeviceToHost));
  for (int c = 0; c < n; c++) {
    int row = (done - n + c) % HMC_HIST;
    std::copy(all.begin() + (size_t)row * h->nrep, all.begin() + (size_t)(row + 1) * h->nrep, U + (size_t)c * h->nrep);
  }
  return n;
}

// Chosen variant {block size, cell division} and the autotuner's timings.
void EmDeeHMC_variant(EmDeeHMC* h, int* blockSize, int* cellDivision, double* tuneMs) {
  if (blockSize) *blockSize = VARIANTS[h->variant].bs;
  if (cellDivision) *cellDivision = VARIANTS[h->variant].div;
  if (tuneMs) for (int v = 0; v < NVARIANTS; v++) tuneMs[v] = h->tuneMs[v];
}

void EmDeeHMC_destroy(EmDeeHMC* h) {
  if (!h) return;
  (void)hipStreamSynchronize(h->stream);
  if (h->exec) (void)hipGraphExecDestroy(h->exec);
  if (h->graph) (void)hipGraphDestroy(h->graph);
  h->desc.release(); h->order.release(); h->cycle.release(); h->U.release(); h->lastDH.release(); h->accepted.release();
  for (DBuf<double>* b : { &h->R, &h->P, &h->F, &h->Rsave, &h->Fsave }) b->release();
  h->S.release();
  h->nlist.release(); h->nnb.release(); h->qbuild.release(); h->lstate.release(); h->Uhist.release();
  if (h->ring) (void)hipHostFree(h->ring);
  (void)hipStreamDestroy(h->stream);
  delete h;
}

// The generator of the momenta and acceptance uniforms, for hosts that
// replay a run (3 * n Gaussian momenta of unit mass at kT, then the uniform
// of the Metropolis test).
void EmDeeHMC_momenta(unsigned long long seed, int replica, int cycle, int n, double kT, double* P) {
  uint64_t stream = hmc_stream(replica, cycle);
  double sq = std::sqrt(kT);
  for (int i = 0; i < n; i++)
    for (int x = 0; x < 3; x++) {
      double u1 = hmc_uniform(seed, stream, 6ULL * i + 2 * x), u2 = hmc_uniform(seed, stream, 6ULL * i + 2 * x + 1);
      P[3 * i + x] = sq * (std::sqrt(-2.0 * std::log(u1)) * std::cos(TWO_PI_D * u2));
    }
}
double EmDeeHMC_uniform(unsigned long long seed, int replica, int cycle) {
  return hmc_uniform(seed, hmc_stream(replica, cycle), HMC_ACCEPT_COUNTER);
}

}  // extern "C"
