// ewald.hip -- reciprocal-space Ewald sum on the GPU (kspace_ewald.f90:188-314).
//
// The reference stores qeikr(k, j) = q_j e^{i k.r_j} for every k-vector and
// charge (nvecs x Ncharged complex FP64: 1.4 GB for 12,288 charges and 7,073
// vectors) and reads it twice.  Here both passes are contractions of small
// per-charge tables on the FP64 matrix cores, and nothing of that size exists.
//   * With c_x(p), s_x(p) = cos, sin of 2 pi p r_x / L, the vectors
//     (n1, +-n2, +-n3) share the eight real sums
//       M[e1 e2 e3] = sum_j q_j X1(n1, e1) X2(n2, e2) X3(n3, e3),  X = c or s,
//     of which S(k) of each sign combination is four terms.  A "quad" is one
//     (n1, n2 >= 0) with its four (e1, e2) rows; its columns are the (n3, e3)
//     with n3 <= m, the largest n3 of the quad in the sphere.  Four
//     multiply-adds per charge and vector are left of the complex recursion's
//     six to twelve, and no chain of products runs along a row.
//   * k_ew_tables: X1 (times q), X2, X3 for p = 0, 1, ... by the reference's
//     recursion (kspace_ewald.f90:232-246).
//   * k_ew_structure: M as a product (quad rows x charges) . (charges x
//     columns) per chunk of charges of one type; k_ew_sigma adds the chunks in
//     a fixed order (deterministic), forms S, sigma = S lambda, the energy and
//     the coefficients D of every charge's potential,
//       phi_j = sum D[e1 e2 e3] q_j X1 X2 X3 = sum_k 2 prefac Re(q_j e^{ik.r_j} conj(sigma)).
//   * k_ew_forces: D contracted with X3 and with its derivative on the matrix
//     cores, then with X1 and X2 and their derivatives per charge:
//     F_j = -grad phi_j (kspace_ewald.f90:297), the quads split over blocks for
//     occupancy; k_ew_force_add adds the partial forces in a fixed order into
//     F (cell-sorted slots).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "device_state.h"
#include "kspace.h"

namespace emdee {

namespace {
const double TWO_PI = 2.0 * 3.14159265358979324;   // 2 pi with global.f90:38
constexpr int EW_P = 16;                            // columns n3 per block of columns
constexpr int EW_CHUNKS = 128;                      // charge chunks of the structure factors (about)
constexpr int EW_TARGET_WAVES_F = 4096;             // quad split target of the forces: four waves per SIMD
constexpr int EW_FA = 2;                            // 16-charge tiles per wavefront of the forces
constexpr int EW_ADD_LANES = 16;                    // lanes per charge adding the partial forces
typedef double f64x4 __attribute__((ext_vector_type(4)));
}  // namespace

struct EwaldState {
  int nm = 0, nvecs = 0, nt = 0, nl = 0, nslots = 0, ngroups = 0;
  int nq = 0, npb = 1, nchunks = 0, ksF = 1;   // quads (multiple of 8), column blocks, charge chunks, quad splits
  double unit = 0;                             // 2 pi / L of the set-up
  DBuf<int4> quad;        // n1, n2, m (-1: padding), unused; m descending
  DBuf<double> wq, vq;    // [quad][npb * EW_P]: prefac (0 beyond m), 1 - k^2 / (2 alpha^2) when the virial is wanted
  DBuf<int> item, groupType, chunkStart, typeChunks;
  DBuf<double> q, lambda, selfc;
  // scratch of one evaluation, one allocation: tables, partial structure
  // factors, force coefficients, partial forces and energies
  DBuf<double2> work;
  double2* T = nullptr;
  double *Mpart = nullptr, *D = nullptr, *Fpart = nullptr, *part = nullptr;
  std::vector<int4> hostQuad;
};

static EwaldState* ewald_of(Device* d) {
  if (!d->ewald) d->ewald = new EwaldState();
  return d->ewald;
}

static void release_state(EwaldState* e) {
  e->quad.release(); e->wq.release(); e->vq.release(); e->item.release(); e->groupType.release();
  e->chunkStart.release(); e->typeChunks.release(); e->q.release(); e->lambda.release(); e->selfc.release();
  e->work.release();
  delete e;
}

void dev_ewald_release(Device* d) {
  if (!d->ewald) return;
  release_state(d->ewald);
  d->ewald = nullptr;
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// {cos, sin} of 2 pi p r_x / L, kspace_ewald.f90:209-246, axis blockIdx.y:
// axes 0 (times q) and 1 for p <= nm, axis 2 for every column p < np.
// Axis x, order p at T[(x*(nm+1) + p)*nslots + slot].
__global__ void k_ew_tables(double2* __restrict__ T, const int* __restrict__ item, const int* __restrict__ iperm,
                            const double* __restrict__ R, const double* __restrict__ q, double L, int nm, int np,
                            int nslots, int Npad) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, x = blockIdx.y;
  if (j >= nslots) return;
  const int i = item[j], s = i >= 0 ? iperm[i] : -1;
  double2 Z = make_double2(1.0, 0.0);
  if (s >= 0) {
    double th = TWO_PI * (R[(size_t)x * Npad + s] / L);
    double sn, cs;
    sincos(th, &sn, &cs);
    Z = make_double2(cs, sn);
  }
  const double f = x == 0 ? q[j] : 1.0;
  const int top = x == 2 ? np - 1 : nm;
  double2* Tx = T + (size_t)x * (nm + 1) * nslots + j;
  Tx[0] = make_double2(f, 0.0);
  double2 b = Z;
  for (int p = 1; p <= top; p++) {
    Tx[(size_t)p * nslots] = make_double2(f * b.x, f * b.y);
    b = cmul(b, Z);
  }
}

// M of eight quads x EW_P columns over one chunk of charges: block (chunk,
// eight quads, column block), four wavefronts, each with a quarter of every
// 256-slot group.  v_mfma_f64_16x16x4: rows i = (quad, e2) with e1 = c in one
// tile and e1 = s in the other, columns j = n3 with e3 = c and e3 = s in two
// tiles, four charges per step, so a step's three table loads (X1, X2, X3)
// feed four products.  12,288 charges, 7,073 vectors took 55 us by complex
// recursion on the vector units, and take 22 (28 TF/s, where a large FP64
// product reaches 72) here, with two or four wavefronts per block.  Bound by
// the latency of the table loads and the ends of a short kernel: the matrix
// cores are busy for 45 % of the time, the waves wait for 74 % of theirs.
// Mpart[((chunk * nq + quad) * npb + block) * 128 + 64 e1 + 32 e2 + 16 e3 + n3].
constexpr int EW_SW = 4;                             // wavefronts per block
__global__ void __launch_bounds__(64 * EW_SW) k_ew_structure(double* __restrict__ Mpart, const double2* __restrict__ T,
                                                      const int4* __restrict__ quad, const int* __restrict__ chunkStart,
                                                      int nm, int nslots, int nq, int npb) {
  __shared__ double red[EW_SW - 1][16][64];
  const int lane = threadIdx.x & 63, h = threadIdx.x >> 6, r = lane & 15, kk = lane >> 4;
  const int q0 = blockIdx.y * 8, pb = blockIdx.z;
  if (quad[q0].z < pb * EW_P) return;   // no quad of the eight reaches these columns (m descending)
  const int4 qd = quad[q0 + (r >> 1)];
  const int e2 = r & 1;
  const size_t plane = (size_t)(nm + 1) * nslots;
  const double2* __restrict__ t1 = T + (size_t)qd.x * nslots + kk;
  const double* __restrict__ t2 = reinterpret_cast<const double*>(T + plane + (size_t)qd.y * nslots + kk) + e2;
  const double2* __restrict__ t3 = T + 2 * plane + (size_t)(pb * EW_P + r) * nslots + kk;
  f64x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) acc[a][b] = (f64x4){ 0.0, 0.0, 0.0, 0.0 };
  const int g0 = chunkStart[blockIdx.x], g1 = chunkStart[blockIdx.x + 1];
  for (int g = g0; g < g1; g++) {
    const int base = g * EWALD_GROUP + h * (EWALD_GROUP / EW_SW);
#pragma unroll 8
    for (int k = 0; k < EWALD_GROUP / EW_SW; k += 4) {
      const double2 x1 = t1[base + k], x3 = t3[base + k];
      const double x2 = t2[2 * (base + k)];
      const double ac = x1.x * x2, as = x1.y * x2;
      acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ac, x3.x, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ac, x3.y, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(as, x3.x, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(as, x3.y, acc[1][1], 0, 0, 0);
    }
  }
  if (h > 0) {
#pragma unroll
    for (int u = 0; u < 16; u++) red[h - 1][u][lane] = acc[u >> 3][(u >> 2) & 1][u & 3];
  }
  __syncthreads();
  if (h == 0) {
    // lane holds rows i = lane/16 + 4u of column lane%16
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int e1 = u >> 3, e3 = (u >> 2) & 1, i = kk + 4 * (u & 3);
      double v = acc[e1][e3][u & 3];
#pragma unroll
      for (int w = 0; w < EW_SW - 1; w++) v += red[w][u][lane];
      Mpart[(((size_t)blockIdx.x * nq + q0 + (i >> 1)) * npb + pb) * 128 + 64 * e1 + 32 * (i & 1) + 16 * e3 + r] = v;
    }
  }
}

// One quad and column block per workgroup: M of every charged type (chunks
// added in a fixed order by four groups of 128 threads), then per vector
// (n3, signs of n2 and n3) S_I(k) (kspace_ewald.f90:226-228), sigma(k) =
// S(k) lambda (:284) and the energy prefac * sum_I S_I . sigma_I (:287), and
// the coefficients D of the forces in the lane order of k_ew_forces:
// D[((t * nq/4 + quad/4) * 8 npb + n3/2) * 64 + lane].  With vq (a partial k
// set standing in for part of the sum), the partials also carry the virial of
// the energy, sum_k E_k (1 - k^2/(2 alpha^2)) = -dE/dln(lambda) when positions
// and box scale by lambda: part[2 b + 1].
constexpr int EW_SIGMA_MAXT = 8;
__global__ void __launch_bounds__(512) k_ew_sigma(double* __restrict__ D, double* __restrict__ part,
                                                  const double* __restrict__ Mpart, const int4* __restrict__ quad,
                                                  const double* __restrict__ wq, const double* __restrict__ vq,
                                                  const int* __restrict__ typeChunks, const double* __restrict__ lam,
                                                  int nt, int nq, int npb) {
  __shared__ double red[4][EW_SIGMA_MAXT][128];
  __shared__ double sg[EW_SIGMA_MAXT][2][64];
  const int tid = threadIdx.x, c = tid & 127, sub = tid >> 7;
  const int qi = blockIdx.x, pb = blockIdx.y;
  const int4 qd = quad[qi];
  const bool any = qd.z >= pb * EW_P;   // uniform over the block
  if (any) {
    const size_t stride = (size_t)nq * npb * 128, o = ((size_t)qi * npb + pb) * 128 + c;
    for (int t = 0; t < nt; t++) {
      double s = 0.0;
#pragma unroll 4
      for (int g = typeChunks[t] + sub; g < typeChunks[t + 1]; g += 4) s += Mpart[g * stride + o];
      red[sub][t][c] = s;
    }
  }
  __syncthreads();
  double e = 0.0, v = 0.0;
  if (tid < 64) {
    const int p = tid & 15, col = pb * EW_P + p;
    const bool neg2 = (tid & 16) != 0, neg3 = (tid & 32) != 0;   // signs of n2 and n3
    // each vector of the half space once: n1 > 0 or n2 > 0 or n3 > 0, and no
    // second copy of a zero component
    const bool on = any && col <= qd.z && !(neg2 && qd.y == 0) && !(neg3 && col == 0) && !(qd.x == 0 && neg2) &&
                    !(qd.x == 0 && qd.y == 0 && (neg3 || col == 0));
    const double s2 = neg2 ? -1.0 : 1.0, s3 = neg3 ? -1.0 : 1.0;
    const double w = on ? wq[(size_t)qi * npb * EW_P + col] : 0.0;
    double sr[EW_SIGMA_MAXT], si[EW_SIGMA_MAXT];
#pragma unroll
    for (int t = 0; t < EW_SIGMA_MAXT; t++) {
      sr[t] = si[t] = 0.0;
      if (t < nt && on) {
        double m[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {   // u = 4 e1 + 2 e2 + e3
          const int k = 16 * u + p;
          m[u] = (red[0][t][k] + red[1][t][k]) + (red[2][t][k] + red[3][t][k]);
        }
        // (c1 + i s1)(c2 + i s2 sn2)(c3 + i s3 sn3)
        sr[t] = (m[0] - s2 * m[6]) - s3 * (m[5] + s2 * m[3]);
        si[t] = (m[4] + s2 * m[2]) + s3 * (m[1] - s2 * m[7]);
      }
    }
#pragma unroll
    for (int t2 = 0; t2 < EW_SIGMA_MAXT; t2++) {
      if (t2 < nt) {
        double gr = 0.0, gi = 0.0;
#pragma unroll
        for (int t1 = 0; t1 < EW_SIGMA_MAXT; t1++) {
          if (t1 < nt) {
            gr += sr[t1] * lam[t1 + nt * t2];
            gi += si[t1] * lam[t1 + nt * t2];
          }
        }
        e += sr[t2] * gr + si[t2] * gi;
        sg[t2][0][tid] = 2.0 * w * gr;
        sg[t2][1][tid] = 2.0 * w * gi;
      }
    }
    e *= w;
    if (vq) v = on ? e * vq[(size_t)qi * npb * EW_P + col] : 0.0;
    e = wave_sum(e);
    v = wave_sum(v);
    if (tid == 0) {
      const int b = qi * npb + pb;
      if (vq) { part[2 * b] = e; part[2 * b + 1] = v; } else part[b] = e;
    }
  }
  __syncthreads();
  // phi_j = sum over the vectors of gr Re(e) + gi Im(e), e = q (c1 + i s1)(c2 + i s2 sn2)(c3 + i s3 sn3)
  const int p = c & 15, e3 = (c >> 4) & 1, e2 = (c >> 5) & 1, e1 = c >> 6;
  const int par = e1 + e2 + e3;   // number of sines: the term is i^par
  for (int t = sub; t < nt; t += 4) {
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const double f = ((e2 && (u & 1)) ? -1.0 : 1.0) * ((e3 && (u & 2)) ? -1.0 : 1.0);
      const double g = sg[t][par & 1][16 * u + p];
      s += (par >= 2 ? -f : f) * g;
    }
    const int kk = 2 * (p & 1) + e3, lane = 16 * kk + (qi & 3) + 4 * (2 * e1 + e2);
    D[(((size_t)t * (nq >> 2) + (qi >> 2)) * (8 * npb) + 8 * pb + (p >> 1)) * 64 + lane] = s;
  }
}

// Partial k-space forces over the quads of blockIdx.y:
// Fpart[(y*4 + x)*nslots + j], x = 0..2; x = 3 holds the atom's share of the
// reciprocal energy, phi_j / 2, whose sum over atoms is kspace_ewald.f90:287.
// A block's four wavefronts take 32 slots each of one group (one charged
// type), so they read the same D.  Per tile of four quads, with rows
// i = quad + 4 (2 e1 + e2), D times X3 and D times -dX3/d(angle) over the
// columns give T and T' of 4 x 16 charges: the lane of quad lane/16 and charge
// lane%16 holds its four (e1, e2) values and finishes with X1 and X2.  12,288
// charges, 7,073 vectors: 73 us by recursion, 32 here (28 TF/s of products),
// with the matrix cores 41 % busy, VALU issue at 46 % and the waves waiting for
// 49 % of their cycles.  EW_FA = 2 tiles of 16 charges per wavefront
// share each load of D at four wavefronts per SIMD; one tile took 34-36 us,
// four (two wavefronts per SIMD for registers) 35-40.
__global__ void __launch_bounds__(256) k_ew_forces(double* __restrict__ Fpart, const double2* __restrict__ T,
                                                   const int4* __restrict__ quad, const double* __restrict__ D,
                                                   const int* __restrict__ groupType, double unit, int nm, int nslots,
                                                   int nq, int npb, int ks) {
  const int lane = threadIdx.x & 63, r = lane & 15, kk = lane >> 4;
  const int j0 = blockIdx.x * (64 * EW_FA) + (threadIdx.x >> 6) * (16 * EW_FA) + r;
  const int ntile = nq >> 2;
  const double* __restrict__ Dt = D + (size_t)groupType[blockIdx.x * (64 * EW_FA) / EWALD_GROUP] * ntile * (8 * npb) * 64 + lane;
  const size_t plane = (size_t)(nm + 1) * nslots;
  const double2* __restrict__ t1 = T + j0;
  const double2* __restrict__ t2 = T + plane + j0;
  const double2* __restrict__ t3 = T + 2 * plane + (size_t)(kk >> 1) * nslots + j0;
  const bool e3 = (kk & 1) != 0;
  double fx[EW_FA], fy[EW_FA], fz[EW_FA], er[EW_FA];
#pragma unroll
  for (int a = 0; a < EW_FA; a++) fx[a] = fy[a] = fz[a] = er[a] = 0.0;
  for (int tile = blockIdx.y; tile < ntile; tile += ks) {
    const int m = quad[4 * tile].z;   // the largest of the four
    if (m < 0) break;                 // padding only from here on
    f64x4 tv[EW_FA], td[EW_FA];
#pragma unroll
    for (int a = 0; a < EW_FA; a++) tv[a] = td[a] = (f64x4){ 0.0, 0.0, 0.0, 0.0 };
    const double* __restrict__ dm = Dt + (size_t)tile * (8 * npb) * 64;
#pragma unroll 2
    for (int s = 0; 2 * s <= m; s++) {
      const double d = dm[64 * s], n3 = 2 * s + (kk >> 1);
      double2 z[EW_FA];
#pragma unroll
      for (int a = 0; a < EW_FA; a++) z[a] = t3[(size_t)(2 * s) * nslots + 16 * a];
#pragma unroll
      for (int a = 0; a < EW_FA; a++) {
        tv[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(d, e3 ? z[a].y : z[a].x, tv[a], 0, 0, 0);
        td[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(d, n3 * (e3 ? -z[a].x : z[a].y), td[a], 0, 0, 0);
      }
    }
    const int4 qd = quad[4 * tile + kk];
    const double n1 = qd.x, n2 = qd.y;
#pragma unroll
    for (int a = 0; a < EW_FA; a++) {
      const double2 x1 = t1[(size_t)qd.x * nslots + 16 * a], x2 = t2[(size_t)qd.y * nslots + 16 * a];
      const double pc = x2.x * tv[a][0] + x2.y * tv[a][1], ps = x2.x * tv[a][2] + x2.y * tv[a][3];
      const double qc = x2.y * tv[a][0] - x2.x * tv[a][1], qs = x2.y * tv[a][2] - x2.x * tv[a][3];
      const double dc = x2.x * td[a][0] + x2.y * td[a][1], ds = x2.x * td[a][2] + x2.y * td[a][3];
      er[a] += x1.x * pc + x1.y * ps;
      fx[a] += n1 * (x1.y * pc - x1.x * ps);
      fy[a] += n2 * (x1.x * qc + x1.y * qs);
      fz[a] += x1.x * dc + x1.y * ds;
    }
  }
  // the four quads of a tile lie in lanes 16 apart; component kk leaves by lane group kk
  const size_t o = ((size_t)blockIdx.y * 4 + kk) * nslots + j0;
#pragma unroll
  for (int a = 0; a < EW_FA; a++) {
    double v[4] = { unit * fx[a], unit * fy[a], unit * fz[a], 0.5 * er[a] };
#pragma unroll
    for (int x = 0; x < 4; x++) {
      v[x] += __shfl_xor(v[x], 16, 64);
      v[x] += __shfl_xor(v[x], 32, 64);
    }
    Fpart[o + 16 * a] = kk == 0 ? v[0] : kk == 1 ? v[1] : kk == 2 ? v[2] : v[3];
  }
}

// F(slot of atom) += sum over k ranges (fixed order), kspace_ewald.f90:297;
// with eatom, also the atom's reciprocal and self energies
// (self: -lambda_II alpha q^2 / sqrt(pi), modelClass_kspace.f90:223-229).
// EW_ADD_LANES lanes per charge: lane u adds the ranges u, u + 16, ... in
// order, and a fixed butterfly adds the lanes' sums.  The last block adds k_ew_sigma's
// energy (and with virial its virial) partials instead and posts them, which
// as a launch of its own (k_reduce_post) held ten steps of 12,288 charges up (2.02 -> 1.99 ms).
__global__ void k_ew_force_add(double* __restrict__ F, double* __restrict__ eatom, const double* __restrict__ Fpart,
                               const int* __restrict__ item, const int* __restrict__ iperm,
                               const double* __restrict__ q, const int* __restrict__ groupType,
                               const double* __restrict__ selfc, int nslots, int ks, int Npad, Post post,
                               const double* __restrict__ part, int nparts, bool virial) {
  if (blockIdx.x == gridDim.x - 1) {
    double v[2] = { 0.0, 0.0 };
    if (virial) {
      sum_partials<2>(v, part, nparts);
    } else {
      double e[1];
      sum_partials<1>(e, part, nparts);
      v[0] = e[0];
    }
    if (threadIdx.x == 0) {
      post.host[0] = v[0];
      if (virial) post.host[1] = v[1];
      __threadfence_system();
      *(volatile unsigned long long*)post.hostSeq = post.seq;
    }
    return;
  }
  int gt = blockIdx.x * blockDim.x + threadIdx.x;
  int j = gt / EW_ADD_LANES, u = gt % EW_ADD_LANES;
  bool ok = j < nslots;
  double f[4] = { 0.0, 0.0, 0.0, 0.0 };
  if (ok) {
    for (int y = u; y < ks; y += EW_ADD_LANES)
#pragma unroll
      for (int x = 0; x < 4; x++) f[x] += Fpart[((size_t)y * 4 + x) * nslots + j];
  }
#pragma unroll
  for (int off = EW_ADD_LANES / 2; off > 0; off >>= 1)
#pragma unroll
    for (int x = 0; x < 4; x++) f[x] += __shfl_xor(f[x], off, EW_ADD_LANES);
  if (!ok || u != 0) return;
  int i = item[j];
  if (i < 0) return;
  int s = iperm[i];
  for (int x = 0; x < 3; x++) F[x * (size_t)Npad + s] += f[x];
  if (eatom) eatom[s] += f[3] + selfc[groupType[j / EWALD_GROUP]] * q[j] * q[j];
}

static void ewald_state_setup(EwaldState* e, const EwaldSetup& s) {
  e->nm = s.nm; e->nvecs = s.nvecs; e->nt = s.nt; e->nl = s.nl; e->nslots = s.nslots; e->unit = s.unit;
  e->ngroups = s.nslots / EWALD_GROUP;
  auto put = [&](auto& buf, const auto& host) {
    buf.alloc(host.size());
    HIP_CHECK(hipMemcpy(buf.p, host.data(), host.size() * sizeof(host[0]), hipMemcpyHostToDevice));
  };
  if (s.nslots % EWALD_GROUP || (int)s.groupType.size() != s.nslots / EWALD_GROUP)
    fatal("kspace set-up", "charge slots are not grouped");
  if (s.nt > EW_SIGMA_MAXT) fatal("kspace set-up", "more than 8 charged types");
  // quads (n1, n2 >= 0) with their largest n3, and prefac by n3; the half
  // space holds every sign combination of a quad's vectors
  std::vector<int4> quads;
  std::vector<int> at((size_t)(s.nm + 1) * (s.nm + 1), -1);
  for (int k = 0; k < s.nvecs; k++) {
    const int n1 = s.kn[3 * k], n2 = std::abs(s.kn[3 * k + 1]), n3 = std::abs(s.kn[3 * k + 2]);
    if (n1 < 0 || n1 > s.nm || n2 > s.nm || n3 > s.nm)
      fatal("kspace set-up", "k-vector outside the half space of the table");
    int& q = at[(size_t)n1 * (s.nm + 1) + n2];
    if (q < 0) { q = (int)quads.size(); quads.push_back(make_int4(n1, n2, n3, 0)); }
    quads[q].z = std::max(quads[q].z, n3);
  }
  std::stable_sort(quads.begin(), quads.end(), [](const int4& a, const int4& b) { return a.z > b.z; });
  while (quads.size() % 8) quads.push_back(make_int4(0, 0, -1, 0));
  for (size_t q = 0; q < quads.size(); q++) if (quads[q].z >= 0) at[(size_t)quads[q].x * (s.nm + 1) + quads[q].y] = (int)q;
  e->nq = (int)quads.size();
  e->npb = (s.nm + 1 + EW_P - 1) / EW_P;
  std::vector<double> wq((size_t)e->nq * e->npb * EW_P, 0.0);
  std::vector<int> seen(wq.size(), 0);
  for (int k = 0; k < s.nvecs; k++) {
    const int n2 = std::abs(s.kn[3 * k + 1]), n3 = std::abs(s.kn[3 * k + 2]);
    const size_t o = (size_t)at[(size_t)s.kn[3 * k] * (s.nm + 1) + n2] * e->npb * EW_P + n3;
    wq[o] = s.prefac[k];
    seen[o]++;
  }
  for (size_t q = 0; q < quads.size(); q++)
    for (int n3 = 0; n3 <= quads[q].z; n3++) {
      const bool z1 = quads[q].x == 0, z2 = quads[q].y == 0, z3 = n3 == 0;
      const int want = z1 && z2 && z3 ? 0 : (z1 ? (z2 ? 1 : (z3 ? 1 : 2)) : (z2 ? 1 : 2) * (z3 ? 1 : 2));
      if (seen[q * e->npb * EW_P + n3] != want) fatal("kspace set-up", "the k-vectors do not fill a sphere");
    }
  e->hostQuad = quads;
  put(e->quad, quads);
  put(e->wq, wq);
  put(e->item, s.slotItem);
  put(e->q, s.slotQ);
  put(e->groupType, s.groupType);
  put(e->lambda, s.lambda);
  // chunks of whole groups of one type, about EW_CHUNKS in all
  const int per = std::max(1, div_up(e->ngroups, EW_CHUNKS));
  std::vector<int> chunk, typeChunks(s.nt + 1, 0);
  for (int t = 0; t < s.nt; t++) {
    for (int g = s.typeGroups[t]; g < s.typeGroups[t + 1]; g += per) chunk.push_back(g);
    typeChunks[t + 1] = (int)chunk.size();
  }
  e->nchunks = (int)chunk.size();
  chunk.push_back(e->ngroups);
  put(e->chunkStart, chunk);
  put(e->typeChunks, typeChunks);
  e->ksF = std::max(1, std::min(e->nq / 4, EW_TARGET_WAVES_F / std::max(1, s.nslots / (16 * EW_FA))));
  // every part a multiple of 16 bytes (nslots, 128 and 64 are even)
  const size_t nT = (2 * (size_t)(s.nm + 1) + e->npb * EW_P) * s.nslots,
               nM = (size_t)e->nchunks * e->nq * e->npb * 64, nD = (size_t)s.nt * (e->nq / 4) * (8 * e->npb) * 32,
               nF = (size_t)e->ksF * 2 * s.nslots, nP = (size_t)e->nq * e->npb;
  e->work.alloc(nT + nM + nD + nF + nP);
  e->T = e->work.p;
  e->Mpart = reinterpret_cast<double*>(e->T + nT);
  e->D = e->Mpart + 2 * nM;
  e->Fpart = e->D + 2 * nD;
  e->part = e->Fpart + 2 * nF;
}

void dev_ewald_setup(Device* d, const EwaldSetup& s) {
  EwaldState* e = ewald_of(d);
  ewald_state_setup(e, s);
  std::vector<double> selfc((size_t)s.nl * s.nt);
  for (int l = 0; l < s.nl; l++)
    for (int t = 0; t < s.nt; t++)
      selfc[(size_t)l * s.nt + t] = -s.alpha * s.lambda[(size_t)l * s.nt * s.nt + t * s.nt + t] / std::sqrt(3.14159265358979324);
  e->selfc.alloc(selfc.size());
  HIP_CHECK(hipMemcpy(e->selfc.p, selfc.data(), selfc.size() * sizeof(double), hipMemcpyHostToDevice));
}

// One evaluation of the sum over the state's k-vectors with the type-pair
// weights lam and self-energy coefficients selfc (null: none): forces added
// to F (slot order), atom shares to eatom (may be null); returns the energy
// and, with the state's virial factors, its virial in *W.
static unsigned long long ewald_launch(Device* d, EwaldState* e, double* F, const double* lam, const double* selfc,
                                       double* eatom, double L, bool virial, int slot) {
  // shapes the kernels assume
  if (e->nslots % EWALD_GROUP || e->ngroups * EWALD_GROUP != e->nslots || e->nq % 8 || e->nm < 1 ||
      e->npb * EW_P <= e->nm || e->nchunks < 1)
    fatal("kspace computation", "inconsistent k-space set-up");
  if (eatom && !selfc) fatal("kspace computation", "atom energies need the self-energy coefficients");
  int Np = d->Npad;
  const double* vf = virial ? e->vq.p : nullptr;
  if (virial && !vf) fatal("kspace computation", "no virial factors for this k set");
  hipLaunchKernelGGL(k_ew_tables, dim3(div_up(e->nslots, BLOCK), 3), dim3(BLOCK), 0, d->stream, e->T, e->item.p,
                     d->iperm.p, d->R.p, e->q.p, L, e->nm, e->npb * EW_P, e->nslots, Np);
  launch_check("ewald tables");
  hipLaunchKernelGGL(k_ew_structure, dim3(e->nchunks, e->nq / 8, e->npb), dim3(64 * EW_SW), 0, d->stream, e->Mpart, e->T,
                     e->quad.p, e->chunkStart.p, e->nm, e->nslots, e->nq, e->npb);
  launch_check("ewald structure factors");
  hipLaunchKernelGGL(k_ew_sigma, dim3(e->nq, e->npb), dim3(512), 0, d->stream, e->D, e->part, e->Mpart, e->quad.p,
                     e->wq.p, vf, e->typeChunks.p, lam, e->nt, e->nq, e->npb);
  launch_check("ewald sigma");
  hipLaunchKernelGGL(k_ew_forces, dim3(e->nslots / (64 * EW_FA), e->ksF), dim3(256), 0, d->stream, e->Fpart, e->T, e->quad.p,
                     e->D, e->groupType.p, e->unit, e->nm, e->nslots, e->nq, e->npb, e->ksF);
  launch_check("ewald forces");
  // with the energy (and virial), straight into pinned host memory
  Post post{};
  post.host = d->hpostDev + slot;
  post.hostSeq = d->hseqDev;
  post.seq = ++d->seq;
  hipLaunchKernelGGL(k_ew_force_add, dim3(div_up((long)e->nslots * EW_ADD_LANES, BLOCK) + 1), dim3(BLOCK), 0, d->stream, F,
                     eatom, e->Fpart, e->item.p, d->iperm.p, e->q.p, e->groupType.p, selfc, e->nslots, e->ksF, Np, post,
                     e->part, e->nq * e->npb, vf != nullptr);
  launch_check("ewald force add");
  return post.seq;
}

// the same, read once its energy (and virial) have been posted
static double ewald_eval(Device* d, EwaldState* e, double* F, const double* lam, const double* selfc, double* eatom,
                         double L, double* W, int slot) {
  dev_post_wait(d, ewald_launch(d, e, F, lam, selfc, eatom, L, W != nullptr, slot));
  if (W) *W = d->hpost[slot + 1];
  return d->hpost[slot];
}

bool dev_ewald_launch(Device* d, int layer, double L) {
  EwaldState* e = d->ewald;
  if (!e || e->nvecs == 0 || e->nslots == 0) return false;
  double* F = d->F.p + 3 * (size_t)d->Npad * layer;
  ewald_launch(d, e, F, e->lambda.p + (size_t)layer * e->nt * e->nt, e->selfc.p + (size_t)layer * e->nt,
               d->wantAtomE ? d->eatom.p : nullptr, L, false, POST_EWALD);
  return true;
}

double dev_ewald_energy(const Device* d) { return d->hpost[POST_EWALD]; }

double dev_ewald_compute(Device* d, int layer, double L) {
  if (!dev_ewald_launch(d, layer, L)) return 0.0;
  dev_wait_posts(d);
  return dev_ewald_energy(d);
}

// A reciprocal-space sum over a partial k set (set-up by lowk_setup): one
// weight table (layer 0 of s.lambda), no self energy, with its virial.
EwaldState* dev_lowk_create(const EwaldSetup& s) {
  if (s.nl != 1) fatal("kspace set-up", "a partial k set has one weight table");
  EwaldState* e = new EwaldState();
  ewald_state_setup(e, s);
  std::vector<double> vq((size_t)e->nq * e->npb * EW_P, 0.0), zero(s.nt, 0.0);
  for (int q = 0; q < e->nq; q++)
    for (int n3 = 0; n3 <= e->hostQuad[q].z; n3++) {
      const int4 n = e->hostQuad[q];
      const double k2 = s.unit * s.unit * ((double)n.x * n.x + (double)n.y * n.y + (double)n3 * n3);
      vq[(size_t)q * e->npb * EW_P + n3] = 1.0 - k2 / (2.0 * s.alpha * s.alpha);
    }
  e->vq.alloc(vq.size());
  HIP_CHECK(hipMemcpy(e->vq.p, vq.data(), vq.size() * sizeof(double), hipMemcpyHostToDevice));
  e->selfc.alloc(s.nt);
  HIP_CHECK(hipMemcpy(e->selfc.p, zero.data(), zero.size() * sizeof(double), hipMemcpyHostToDevice));
  return e;
}

double dev_lowk_compute(Device* d, EwaldState* e, double* F, double* eatom, double L, double* W) {
  if (!e || e->nvecs == 0 || e->nslots == 0) { *W = 0.0; return 0.0; }
  return ewald_eval(d, e, F, e->lambda.p, e->selfc.p, eatom, L, W, POST_LOWK);
}

bool dev_lowk_launch(Device* d, EwaldState* e, double* F, double* eatom, double L) {
  if (!e || e->nvecs == 0 || e->nslots == 0) return false;
  ewald_launch(d, e, F, e->lambda.p, e->selfc.p, eatom, L, true, POST_LOWK);
  return true;
}

double dev_lowk_result(const Device* d, double* W) {
  *W = d->hpost[POST_LOWK + 1];
  return d->hpost[POST_LOWK];
}

int dev_lowk_vectors(const EwaldState* e) { return e ? e->nvecs : 0; }

void dev_lowk_release(EwaldState* e) {
  if (e) release_state(e);
}

}  // namespace emdee
