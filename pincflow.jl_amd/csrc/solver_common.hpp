// Deterministic reductions and the BiCGSTAB scalar updates shared by the
// FP64 solve (poisson.hip) and the mixed-precision solve (mixed.hip).
// Each translation unit gets its own copies (anonymous namespace).
#pragma once

#include "pcf_internal.hpp"

namespace pcf {
namespace {

// ---------------------------------------------------------------------------
// block reduction of up to 3 values (blockDim.x * blockDim.y == 256)
// ---------------------------------------------------------------------------
template <int ND>
__device__ __forceinline__ void block_partials(double (&val)[ND], double* partials, int block) {
  __shared__ double red[ND][kReduceBlock / 64];
  const int tid = threadIdx.x + blockDim.x * threadIdx.y;
  const int lane = tid & 63, wid = tid >> 6;
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    double x = val[d];
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
    if (lane == 0) red[d][wid] = x;
  }
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      double s = red[d][0];
      for (int q = 1; q < kReduceBlock / 64; ++q) s += red[d][q];
      partials[(size_t)d * kPartialStride + block] = s;
    }
  }
}

// Sum nparts partials of dot slot d with one block of 1024 threads, in a
// fixed order.
__device__ double finalize_sum(const double* partials, int d, int nparts) {
  __shared__ double red[16];
  const int tid = threadIdx.x;
  const int stride = blockDim.x;
  const double* pp = partials + (size_t)d * kPartialStride;
  double s = 0.0;
  // the same order as one partial at a time, with 8 loads in flight
  int q = tid;
  for (; q + 7 * stride < nparts; q += 8 * stride) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = pp[q + u * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; q < nparts; q += stride) s += pp[q];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((tid & 63) == 0) red[tid >> 6] = s;
  __syncthreads();
  double r = 0.0;
  if (tid == 0)
    for (int q = 0; q < (int)(blockDim.x / 64); ++q) r += red[q];
  __syncthreads();
  return r;  // valid in thread 0
}

// Initial residual and convergence test (apply_bicgstab!.jl:56-69).  Partial
// slot 0 holds <r0, r0>; with a nonzero initial guess (guessed = 1) slot 1
// holds <b, b> and the criterion stays |r| / |b|, as for x0 = 0.
__global__ void k_bicg_start(const double* partials, int nparts, SolverScalars* sc, double nxyz, double tol,
                             int guessed) {
  double rr = finalize_sum(partials, 0, nparts);
  double bb = guessed ? finalize_sum(partials, 1, nparts) : rr;
  if (threadIdx.x == 0) {
    double res = sqrt(rr / nxyz);
    double b_norm = guessed ? sqrt(bb / nxyz) : res;
    sc->b_norm = b_norm;
    sc->res = res;
    sc->tol = tol;
    sc->niter = 0;
    sc->rr0 = rr;  // <r0, r0> = <r, r0> for r = r0
    sc->done = (res == 0.0 || res / b_norm <= tol) ? 1 : 0;
    sc->fresh = 1;
    sc->next.done = sc->done;
  }
}

// The scalar steps below are one block of 1024 threads per solve: the
// single-solve kernels run them on their state's scalars, the ensemble
// kernels (poisson.hip) on each member's, one block per member.

// alpha = <r, r0> / <v, r0>, from the partials of the A p kernel
__device__ __forceinline__ void bicg_alpha(const double* partials, int nparts, SolverScalars* sc) {
  if (sc->done) return;
  double vr0 = finalize_sum(partials, 0, nparts);
  if (threadIdx.x == 0) {
    sc->vr0 = vr0;
    sc->alpha = sc->rr0 / vr0;
  }
}
__global__ void k_bicg_alpha(const double* partials, int nparts, SolverScalars* sc) {
  bicg_alpha(partials, nparts, sc);
}

// omega = <t, s> / <t, t>
__device__ __forceinline__ void bicg_omega(const double* partials, int nparts, SolverScalars* sc) {
  if (sc->done) return;
  double ts = finalize_sum(partials, 0, nparts);
  double tt = finalize_sum(partials, 1, nparts);
  if (threadIdx.x == 0) {
    sc->ts = ts;
    sc->tt = tt;
    sc->omega = ts / tt;
  }
}
__global__ void k_bicg_omega(const double* partials, int nparts, SolverScalars* sc) {
  bicg_omega(partials, nparts, sc);
}

// residual, convergence and beta (apply_bicgstab!.jl:116-142).  maxit > 0
// (the ensemble solve) stops a solve that reaches maxit iterations without
// converging with done = 2; the single solve stops by its host loop.
__device__ __forceinline__ void bicg_check(const double* partials, int nparts, SolverScalars* sc, double nxyz,
                                           int maxit) {
  if (sc->done) return;
  double rr = finalize_sum(partials, 0, nparts);
  double rr0n = finalize_sum(partials, 1, nparts);
  if (threadIdx.x == 0) {
    double res = sqrt(rr / nxyz);
    sc->rr = rr;
    sc->res = res;
    sc->niter = sc->niter + 1;
    if (res / sc->b_norm <= sc->tol) {
      sc->done = 1;
    } else {
      sc->beta = sc->alpha / sc->omega * rr0n / sc->rr0;
      sc->rr0 = rr0n;
      if (maxit > 0 && sc->niter >= maxit) sc->done = 2;
    }
    sc->rr0_new = rr0n;
  }
}
__global__ void k_bicg_check(const double* partials, int nparts, SolverScalars* sc, double nxyz) {
  bicg_check(partials, nparts, sc, nxyz, 0);
}

// ---------------------------------------------------------------------------
// Fused iterations: on grids where an iteration's time is that of its
// launches, the scalar steps run inside the kernels that use them.  Every
// block sums the partials itself (a few thousand values from L2), which costs
// about 1.5 us against 4.5 us for a kernel of one block between two others.
// ---------------------------------------------------------------------------

// finalize_sum's values of ND dots, in its order, in every thread of a block
// of any number of full wavefronts
template <int ND>
__device__ __forceinline__ void block_sums(const double* partials, int nparts, double (&sum)[ND]) {
  __shared__ double red[ND][16];
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  // the 16 wavefronts of finalize_sum's block, four at a time so that their
  // loads are in flight together
  constexpr int G = 4;
  for (int w0 = threadIdx.x >> 6; w0 < 16; w0 += G * nw) {
    double s[G][ND] = {};
    for (int q0 = lane; q0 < nparts; q0 += 2 * 1024) {
      double v[G][ND][2];
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int q = q0 + 64 * (w0 + g * nw) + u * 1024;
            v[g][d][u] = w0 + g * nw < 16 && q < nparts ? partials[(size_t)d * kPartialStride + q] : 0.0;
          }
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int u = 0; u < 2; ++u) s[g][d] += v[g][d][u];
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        double x = s[g][d];
        for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
        if (lane == 0 && w0 + g * nw < 16) red[d][w0 + g * nw] = x;
      }
  }
  __syncthreads();
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    sum[d] = 0.0;
#pragma unroll
    for (int w = 0; w < 16; ++w) sum[d] += red[d][w];
  }
}

// What the kernel of the preconditioner's first pseudo-time step does before
// it: nothing, the previous iteration's check and p = r + beta (p - omega v),
// or alpha and s = r - alpha v (apply_bicgstab!.jl:71-142).
enum { FUSE_NONE = 0, FUSE_P = 1, FUSE_S = 2 };
// The operands of a fused step at a thread's N cells.  They, the partials and
// the scalars are loaded together, before anything waits for one of them: a
// load that follows another costs a round trip of 1 us here.  own: cell o is
// the thread's own; threads beyond a column's top load another's, of vectors
// that the kernel does not write (dst is stored by the cell's own thread
// while others still load).
template <int FUSE, int N>
struct FuseOperands {
  double r[N], v[N], p[N];
  __device__ __forceinline__ void load(const BicgFuse& F, int u, size_t o, bool own) {
    const double* p_or_r = own ? F.dst : F.r;
    r[u] = F.r[o];
    v[u] = F.v[o];
    p[u] = FUSE == FUSE_P ? p_or_r[o] : 0.0;
  }
};
struct FuseScalars {
  double c0, c1;
  bool fresh;
};
// The scalars of a fused step in every thread; false if the solve has ended.
// Block 0 records them (in sc->next where other blocks still read sc).
template <int FUSE>
__device__ __forceinline__ bool fuse_scalars(const BicgFuse& F, FuseScalars& S) {
  SolverScalars* sc = F.sc;
  const int done = sc->done;
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  const double rr0 = sc->rr0;
  if constexpr (FUSE == FUSE_P) {
    const double alpha = sc->alpha, omega = sc->omega, b_norm = sc->b_norm, tol = sc->tol;
    const int niter = sc->niter;
    S.fresh = sc->fresh != 0;
    double sum[2];
    block_sums<2>(F.partials, F.nparts, sum);
    if (done) return false;
    S.c0 = alpha / omega * sum[1] / rr0;
    S.c1 = omega;
    if (S.fresh) return true;  // p = r already (k_bicg_init)
    const double res = sqrt(sum[0] / F.nxyz);
    const bool end = res / b_norm <= tol;
    if (first) {
      sc->next.rr = sum[0];
      sc->next.res = res;
      sc->next.beta = S.c0;
      sc->next.rr0 = sum[1];
      sc->next.niter = niter + 1;
      sc->next.done = end ? 1 : 0;
    }
    return !end;
  } else {
    double sum[1];
    block_sums<1>(F.partials, F.nparts, sum);
    if (done) return false;
    S.c0 = rr0 / sum[0];
    S.c1 = 0.0;
    S.fresh = false;
    if (first) {
      sc->vr0 = sum[0];
      sc->alpha = S.c0;
    }
    return true;
  }
}
// the vector's new value
template <int FUSE, int N>
__device__ __forceinline__ double fuse_value(const FuseOperands<FUSE, N>& X, const FuseScalars& S, int u) {
  if constexpr (FUSE == FUSE_P) return S.fresh ? X.p[u] : X.r[u] + S.c0 * (X.p[u] - S.c1 * X.v[u]);
  else return X.r[u] - S.c0 * X.v[u];
}
// The kernel after a FUSE_P one: moves the check over; false if it ended the
// solve.
__device__ __forceinline__ bool fuse_commit(SolverScalars* sc) {
  const bool done = sc->next.done != 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (sc->fresh) {
      sc->fresh = 0;
    } else if (!sc->done) {
      sc->rr = sc->next.rr;
      sc->res = sc->next.res;
      sc->niter = sc->next.niter;
      sc->rr0_new = sc->next.rr0;
      if (!done) {
        sc->beta = sc->next.beta;
        sc->rr0 = sc->next.rr0;
      }
      sc->done = sc->next.done;
    }
  }
  return !done;
}

}  // namespace
}  // namespace pcf
