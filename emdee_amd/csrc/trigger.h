// What the kernels that move atoms share with the rebuild trigger: the scaled
// positions that the pair kernels read, and pass A's maximum.
#pragma once
#include "device_state.h"

namespace emdee {

// Scaled positions of a slot: Rs = R / L (EmDeeCode.f90:1228, IEEE division)
// packed with the type, so that a neighbour costs one 32-byte gather, and, when Q4 is given, the mixed form's fixed-point copy
// u = round(2^32 (s - floor s)) mod 2^32 and FP32 charge.
// Q4.w holds the type; a slot whose scaled position is not finite also
// carries Q4_NONFINITE, so that the fixed-point prefilter of the list build
// leaves its candidates to the FP64 test (which rejects them, as the
// reference's r^2 comparison does with NaN).
constexpr int Q4_NONFINITE = 1 << 30, Q4_TYPE = Q4_NONFINITE - 1;
struct Scaled {
  double4* Rs4;
  int4* Q4;
  float* qf;
  const int* type;
  const double* charge;
  const int* charged;
  double L;
};
__device__ __forceinline__ void scale_vals(const Scaled& sc, double x, double y, double z, int s, int t, bool charged,
                                           double charge, double (&v)[3], int4& q4) {
  v[0] = x / sc.L; v[1] = y / sc.L; v[2] = z / sc.L;
  if (sc.Rs4) sc.Rs4[s] = make_double4(v[0], v[1], v[2], (double)t);
  if (sc.Q4) {
    unsigned int u[3];
    for (int x = 0; x < 3; x++) {
      double f = v[x] - floor(v[x]);
      u[x] = (unsigned int)(unsigned long long)llrint(f * 4294967296.0);
    }
    bool fin = isfinite(v[0]) && isfinite(v[1]) && isfinite(v[2]);
    q4 = make_int4((int)u[0], (int)u[1], (int)u[2], fin ? t : (t | Q4_NONFINITE));
    sc.Q4[s] = q4;
    if (sc.qf) sc.qf[s] = charged ? (float)charge : 0.0f;
  }
}
__device__ __forceinline__ void scale_vals(const Scaled& sc, double x, double y, double z, int s) {
  double v[3];
  int4 q4;
  const bool q = sc.Q4 && sc.qf && sc.charged[s];
  scale_vals(sc, x, y, z, s, sc.type[s], q, q ? sc.charge[s] : 0.0, v, q4);
}

// (max, first index) of a set of pairs: the larger value wins, ties go to the
// smaller index, so any combination order gives the same pair.
__device__ __forceinline__ void max_first(double& v, double& idx, double ov, double oi) {
  if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
}
// Reduces nb blocks' {max, first index} into trig and posts them to the host
// (as k_reduce_post); one block.
__device__ __forceinline__ void trig_post(double* __restrict__ trig, const double* __restrict__ part, int nb,
                                          double* __restrict__ host, unsigned long long* __restrict__ hostSeq,
                                          unsigned long long seq) {
  __shared__ double smax[BLOCK / 64], sidx[BLOCK / 64];
  double v = -1.0, idx = 2147483647.0;
#pragma unroll 8
  for (int b = threadIdx.x; b < nb; b += BLOCK) max_first(v, idx, part[2 * b], part[2 * b + 1]);
  for (int off = 32; off > 0; off >>= 1) max_first(v, idx, __shfl_down(v, off, 64), __shfl_down(idx, off, 64));
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) { smax[w] = v; sidx[w] = idx; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < BLOCK / 64; k++) max_first(v, idx, smax[k], sidx[k]);
    trig[0] = v;
    trig[1] = idx;
    host[0] = v;
    host[1] = idx;
    __threadfence_system();
    *(volatile unsigned long long*)hostSeq = seq;
  }
}
// Thread 0's {max, first index} of a block of pass A: left in part, and posted
// by the last block when the grid finishes it (finish_sums)
__device__ __forceinline__ void finish_trig(const Post& post, double* __restrict__ trig, double* __restrict__ part,
                                            double v, int idx) {
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = v;
    part[2 * blockIdx.x + 1] = (double)idx;
  }
  if (post.ticket && last_block(post.ticket, gridDim.x))
    trig_post(trig, part, gridDim.x, post.host, post.hostSeq, post.seq);
}
// This block's {max, first index} from its threads' (all threads call it),
// then finish_trig.
__device__ __forceinline__ void trig_block(const Post& post, double* __restrict__ trig, double* __restrict__ part,
                                           double v, int idx) {
  __shared__ double smax[BLOCK / 64];
  __shared__ int sidx[BLOCK / 64];
  for (int off = 32; off > 0; off >>= 1) {
    double ov = __shfl_down(v, off, 64);
    int oi = __shfl_down(idx, off, 64);
    if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
  }
  int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) { smax[wid] = v; sidx[wid] = idx; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < BLOCK / 64; w++)
      if (smax[w] > v || (smax[w] == v && sidx[w] < idx)) { v = smax[w]; idx = sidx[w]; }
  }
  finish_trig(post, trig, part, v, idx);
}

// For a kernel that moves atoms and forms the next trigger's pass A, in the
// last trigger's set-up (d->trigKnown): the scaled positions to write, and the
// note that it did (g blocks, for the positions of d->posWrites).
inline Scaled dev_trig_scaled(const Device* d) {
  return Scaled{ d->trigRs4 ? d->Rs4.p : nullptr, d->trigMixed ? d->Q4.p : nullptr, nullptr, d->type.p, d->charge.p,
                 d->chargedFlag.p, d->trigL };
}
inline void dev_trig_formed(Device* d, const Post& post, int g) {
  d->trigPreSeq = post.ticket ? post.seq : 0;
  d->trigPreAt = d->posWrites;
  d->trigPreBlocks = g;
  d->trigPreMixed = d->trigMixed;
  d->trigPreRs4 = d->trigRs4;
  d->trigPreL = d->trigL;
}

}  // namespace emdee
