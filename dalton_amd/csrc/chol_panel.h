// The pivot search and column pass of the pivoted Cholesky (cholesky.hip), in a
// file of their own so that a host build can run a block's threads in a chosen
// order.  Includes nothing: the includer brings the device intrinsics in.
#pragma once

namespace ccgpu {

namespace {

// Largest remaining diagonal and its index (smallest index on ties), in two
// stages so that the search spreads over the whole chip: every block of a
// grid-stride pass writes the best (value, index) of its elements to
// part[2 b], part[2 b + 1], and one block reduces the nb partials in a fixed
// order (the pivot is the same as that of a sequential scan).
__device__ __forceinline__ void better(double& bv, long& bi, double ov, long oi) {
  if (ov > bv || (ov == bv && oi < bi)) {
    bv = ov;
    bi = oi;
  }
}

// Block reduction of (bv, bi) over 256 threads into part[2 blockIdx.x ...].
__device__ __forceinline__ void block_best(double bv, long bi, double* __restrict__ part) {
  __shared__ double sv[4];
  __shared__ long si[4];
  for (int off = 32; off > 0; off >>= 1) {
    const double ov = __shfl_down(bv, off, 64);
    const long oi = __shfl_down(bi, off, 64);
    better(bv, bi, ov, oi);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    sv[w] = bv;
    si[w] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < (int)(blockDim.x >> 6); ++q) better(bv, bi, sv[q], si[q]);
    part[2 * (long)blockIdx.x] = bv;
    part[2 * (long)blockIdx.x + 1] = (double)bi;
  }
}

// Step j of the panel that starts at vector K0: pivot p = argmax of the
// remaining diagonal, then
//   L[K0 + j][q] = (R[p][q] - sum_{i<j} L[K0+i][p] L[K0+i][q]) / sqrt(d_p),
//   d[q] -= L[K0 + j][q]^2, d[p] = 0,
// where R = V minus the vectors of earlier panels.  Stops (st[0] = 1,
// st[1] = vectors made) once the largest diagonal is below thr.
// Every block reduces the npart stage-1 partials of the last step (pin) to
// the pivot by itself and writes its own of the updated diagonal to pout, so
// a vector is one launch; a step after the stop leaves them as they are.  The
// block that finds the stop writes st[0] in the launch whose other blocks may
// still be starting: one thread reads it for its whole block, so that no wave
// leaves while others go on to sums it has not written to LDS.
// Bound by latency: the panel's elements of column p go through LDS and the
// sum over them reads eight rows at a time.  nbas = 90, 576 steps: 6.3 us each;
// 11.4 us and 4.1 us for the pivot before.
__global__ __launch_bounds__(256) void k_chol_panel_col(double* __restrict__ L, double* __restrict__ d,
                                                        const double* __restrict__ R, const double* __restrict__ pin,
                                                        int npart, long* __restrict__ st, long M, long K0, int j,
                                                        double thr, double* __restrict__ pout) {
  __shared__ double cp[64], bestv[4];
  __shared__ long besti[4], stop;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (t == 0) stop = st[0];
  double dp = -1.0;
  long p = M;
  for (int q = t; q < npart; q += 256) better(dp, p, pin[2 * q], (long)pin[2 * q + 1]);
  for (int off = 32; off > 0; off >>= 1) {
    const double ov = __shfl_xor(dp, off, 64);
    const long oi = __shfl_xor(p, off, 64);
    better(dp, p, ov, oi);
  }
  if (lane == 0) {
    bestv[wave] = dp;
    besti[wave] = p;
  }
  __syncthreads();
  if (stop != 0) return;
  dp = bestv[0];
  p = besti[0];
  for (int q = 1; q < 4; ++q) better(dp, p, bestv[q], besti[q]);
  if (dp < thr) {
    if (blockIdx.x == 0 && t == 0) {
      st[0] = 1;
      st[1] = K0 + j;
    }
    return;
  }
  const double* Lp = L + K0 * M;
  if (t < j) cp[t] = Lp[t * M + p];
  __syncthreads();
  const double rs = 1.0 / sqrt(dp);
  double bv = -1.0;
  long bi = M;
  for (long q = (long)blockIdx.x * 256 + t; q < M; q += (long)gridDim.x * 256) {
    double s = R[p * M + q];
    const double dq0 = d[q];
#pragma unroll 8
    for (int i = 0; i < j; ++i) s -= cp[i] * Lp[i * M + q];
    const double l = s * rs;
    L[(K0 + j) * M + q] = l;
    const double dq = (q == p) ? 0.0 : dq0 - l * l;
    d[q] = dq;
    better(bv, bi, dq, q);
  }
  block_best(bv, bi, pout);
  if (blockIdx.x == 0 && t == 0) st[1] = K0 + j + 1;
}

}  // namespace

}  // namespace ccgpu
