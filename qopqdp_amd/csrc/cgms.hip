// Device-side pieces of the multi-shift CG (lib/invert_cg_p.c:130-402):
// the per-iteration scalar recurrences (zeta, beta, alpha in FP64) run in a
// one-block kernel, and the vector updates of all shifts are fused into two
// passes.  The host only intervenes for the solution fold / true-residual
// check, which the reference does every 100 iterations or on convergence.
#include "solver.h"

namespace qop {

template <int P> struct QT;
template <> struct QT<P64> { using R = double; using S = double2; };
template <> struct QT<P32> { using R = float; using S = float2; };

__device__ __forceinline__ double wsum(double v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Fixed-order sums of m partials of one or two arrays by one 1024-thread
// block: four independent accumulators per thread and array keep the loads in
// flight (with 256 threads and one accumulator the sums of 2 x 5184 partials
// took 12.8 us, all of it load latency).
constexpr int SUM_THREADS = 1024;
template <int N>
__device__ __forceinline__ void block_sums(const double *const (&p)[N], int m, double *sh, double (&out)[N]) {
  double s[N][4];
#pragma unroll
  for (int k = 0; k < N; k++)
#pragma unroll
    for (int j = 0; j < 4; j++) s[k][j] = 0;
  int i = threadIdx.x;
  for (; i + 3 * SUM_THREADS < m; i += 4 * SUM_THREADS)
#pragma unroll
    for (int k = 0; k < N; k++)
#pragma unroll
      for (int j = 0; j < 4; j++) s[k][j] += p[k][i + j * SUM_THREADS];
  for (; i < m; i += SUM_THREADS)
#pragma unroll
    for (int k = 0; k < N; k++) s[k][0] += p[k][i];
#pragma unroll
  for (int k = 0; k < N; k++) {
    const double t = wsum((s[k][0] + s[k][1]) + (s[k][2] + s[k][3]));
    if ((threadIdx.x & 63) == 0) sh[k * (SUM_THREADS / 64) + (threadIdx.x >> 6)] = t;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; k++) {  // only the first wave's result is used
    const double t = threadIdx.x < SUM_THREADS / 64 ? sh[k * (SUM_THREADS / 64) + threadIdx.x] : 0.0;
    out[k] = wsum(t);
  }
}

// After linop: pkp, b[imin] and the zeta/beta recurrences (:203-238).
__global__ void __launch_bounds__(SUM_THREADS)
cgms_scalarA(CgmsDev d, int nch) {
  __shared__ double sh[2 * SUM_THREADS / 64];
  CgmsState *s = d.st;
  if (s->status != 0) {
    if (threadIdx.x == 0) s->xpend = 0;  // the x update of the stopping iteration is done
    return;
  }
  const double *const parts[2] = {d.partA, d.partB};
  double sums[2];
  block_sums<2>(parts, nch, sh, sums);
  if (threadIdx.x != 0) return;
  s->oldrsq = s->rsq;
  double pkp = sums[0] + s->m2 * sums[1];  // ddagd_norm2 return value
  s->pkp = pkp;
  s->iteration++;
  s->total++;
  s->xpend = 0;
  if (pkp <= 0) { s->status = 2; s->break_reason = 1; return; }
  const int imin = s->imin, ns = s->ns;
  s->b[imin] = s->rsq / pkp;
  s->zn[imin] = 1;
  for (int i = 0; i < ns; i++) {
    if (i == imin) continue;
    double zn = s->z[i] * s->zo[i] * s->bo[imin];
    double c1 = s->b[imin] * s->a[imin] * (s->zo[i] - s->z[i]);
    c1 += s->zo[i] * s->bo[imin] * (1 + s->shifts[i] * s->b[imin]);
    if (c1 != 0.0) zn /= c1; else zn = 0;
    if (s->z[i] != 0.0) s->b[i] = s->b[imin] * zn / s->z[i];
    else { zn = 0; s->b[i] = 0; }
    s->zn[i] = zn;
  }
}

// Relative-residual reduction (only when relmin > 0): r vs out[irel].
template <int P>
__global__ void __launch_bounds__(256)
cgms_relnorm(CgmsDev d, int Vh, VecView r, VecView x) {
  using S = typename QT<P>::S;
  const CgmsState *s = d.st;
  if (s->status != 0) return;
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  double acc = 0;
  if (h < Vh) {
    double r2 = 0, x2 = 0;
    for (int c = 0; c < 3; c++) {
      S a = ((const S *)r.data)[c * Vh + h], b = ((const S *)x.data)[c * Vh + h];
      r2 += (double)a.x * a.x + (double)a.y * a.y;
      x2 += (double)b.x * b.x + (double)b.y * b.y;
    }
    acc = x2 == 0.0 ? 1.0 : r2 / x2;
  }
  const int nch = (Vh + 63) / 64;
  acc = wsum(acc);
  if ((threadIdx.x & 63) == 0 && (h >> 6) < nch) d.partD[h >> 6] = acc;
}

// After the update: rsq, stopping tests, then alpha and the shift-over of
// zeta/beta (:254-275, 349-376).  Sets status 1 when the host must fold the
// solution and check the true residual.
__global__ void __launch_bounds__(SUM_THREADS)
cgms_scalarB(CgmsDev d, int nch, int with_rel, int Vh) {
  __shared__ double sh[2 * SUM_THREADS / 64];
  CgmsState *s = d.st;
  if (s->status != 0) return;
  double rsq, rel = 0;
  if (with_rel) {
    const double *const parts[2] = {d.partC, d.partD};
    double sums[2];
    block_sums<2>(parts, nch, sh, sums);
    rsq = sums[0];
    rel = sums[1];
  } else {
    const double *const parts[1] = {d.partC};
    double sums[1];
    block_sums<1>(parts, nch, sh, sums);
    rsq = sums[0];
  }
  if (threadIdx.x != 0) return;
  s->rsq = rsq;
  const int it = s->iteration;
  s->xpend = with_rel ? 0 : 1;  // read only once the status is raised
  if (s->cg) {  // the restart / stopping test at the top of lib/invert_cg_p.c's loop
    if (with_rel) s->relnorm2 = rel / (double)Vh;
    if (it >= s->restart || s->total >= s->max_iter || rsq < s->rsqstop ||
        (with_rel && s->relnorm2 < s->relstop)) {
      s->status = 1;
      return;
    }
    s->a[0] = rsq / s->oldrsq;
    return;
  }
  double rsqc = s->zn[s->irsq] * s->zn[s->irsq] * rsq;
  if (with_rel) s->relnorm2 = s->zn[s->irel] * s->zn[s->irel] * (rel / (double)Vh);
  if (it >= s->restart || it >= s->max_iter) { s->status = 2; s->break_reason = 2; return; }
  if (rsqc * s->trueRsqFac < s->rsqstop) s->nextRsqCheck = it;
  if (with_rel && s->relnorm2 * s->trueRelFac < s->relstop) s->nextRelCheck = it;
  if (s->nextRsqCheck <= it || (s->relstop > 0 && s->nextRelCheck <= it)) {
    s->status = 1;
    return;
  }
  // alpha and shift-over
  const int imin = s->imin, ns = s->ns;
  s->a[imin] = rsq / s->oldrsq;
  for (int i = 0; i < ns; i++) {
    if (i == imin) continue;
    double c2 = s->z[i] * s->b[imin];
    s->a[i] = c2 != 0.0 ? s->a[imin] * s->zn[i] * s->b[i] / c2 : 0;
  }
  for (int i = 0; i < ns; i++) { s->bo[i] = s->b[i]; s->zo[i] = s->z[i]; s->z[i] = s->zn[i]; }
}

// The solution and search directions of all shifts in one pass
// (:209-252, 349-376): x_i += b_i p_i with the directions of this iteration,
// then p_i = zn_i r + a_i p_i (the base: p = r + a p) and the partials of the
// base |p|^2 for the next iteration's <p, A p>.  pms[imin] is p.
// Streaming, 4 vectors per shift (x and p read and written) + r: with x and p
// updated in separate passes it was 5, and A p was stored and read back
// besides.  In the iteration that raises the status only x is updated; after a
// host check only p (what = CGMS_P).  FP32 vectors: sums formed in FP64 and
// rounded once.
template <int P>
__global__ void __launch_bounds__(256)
cgms_xp(CgmsDev d, int Vh, VecView r, int ns, int what) {
  using R = typename QT<P>::R;
  using S = typename QT<P>::S;
  const CgmsState *s = d.st;
  if (s->status != 0) {
    if (what != CGMS_XP || !s->xpend) return;
    what = CGMS_X;
  }
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  double acc = 0;
  if (h < Vh) {
    S rv[3];
    if (what & CGMS_P) {
      const S *rr = (const S *)r.data;
#pragma unroll
      for (int c = 0; c < 3; c++) rv[c] = rr[c * Vh + h];
    }
    for (int i = 0; i < ns; i++) {
      const bool base = i == s->imin;
      const double ai = s->a[i], zi = s->zn[i], bi = s->b[i];
      S *pm = (S *)d.pms[i].data;
      S *x = (S *)d.xs[i].data;
      S pv[3];
#pragma unroll
      for (int c = 0; c < 3; c++) pv[c] = pm[c * Vh + h];
      if (what & CGMS_X) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          S xv = x[c * Vh + h];
          xv.x = (R)fma(bi, (double)pv[c].x, (double)xv.x);
          xv.y = (R)fma(bi, (double)pv[c].y, (double)xv.y);
          x[c * Vh + h] = xv;
        }
      }
      if (what & CGMS_P) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const double tx = base ? (double)rv[c].x : zi * (double)rv[c].x;
          const double ty = base ? (double)rv[c].y : zi * (double)rv[c].y;
          pv[c].x = (R)fma(ai, (double)pv[c].x, tx);
          pv[c].y = (R)fma(ai, (double)pv[c].y, ty);
          pm[c * Vh + h] = pv[c];
          if (base) acc += (double)pv[c].x * pv[c].x + (double)pv[c].y * pv[c].y;
        }
      }
    }
  }
  if (what & CGMS_P) {
    const int nch = (Vh + 63) / 64;
    acc = wsum(acc);
    if ((threadIdx.x & 63) == 0 && (h >> 6) < nch) d.partB[h >> 6] = acc;
  }
}

void cgms_launch_scalarA(CgmsDev d, int nch, hipStream_t st) {
  launch_kernel(cgms_scalarA, dim3(1), dim3(SUM_THREADS), 0, st, d, nch);
  QOP_CHECK_HIP(hipGetLastError());
}
void cgms_launch_relnorm(CgmsDev d, int prec, int Vh, VecView r, VecView x,
                         hipStream_t st) {
  dim3 g((Vh + 255) / 256), b(256);
  if (prec == P64) launch_kernel(cgms_relnorm<P64>, g, b, 0, st, d, Vh, r, x);
  else launch_kernel(cgms_relnorm<P32>, g, b, 0, st, d, Vh, r, x);
  QOP_CHECK_HIP(hipGetLastError());
}
void cgms_launch_scalarB(CgmsDev d, int nch, int with_rel, int Vh, hipStream_t st) {
  launch_kernel(cgms_scalarB, dim3(1), dim3(SUM_THREADS), 0, st, d, nch, with_rel, Vh);
  QOP_CHECK_HIP(hipGetLastError());
}
void cgms_launch_xp(CgmsDev d, int prec, int Vh, VecView r, int ns, int what, hipStream_t st) {
  dim3 g((Vh + 255) / 256), b(256);
  if (prec == P64) launch_kernel(cgms_xp<P64>, g, b, 0, st, d, Vh, r, ns, what);
  else launch_kernel(cgms_xp<P32>, g, b, 0, st, d, Vh, r, ns, what);
  QOP_CHECK_HIP(hipGetLastError());
}

}  // namespace qop
