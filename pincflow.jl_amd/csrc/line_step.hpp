// One pseudo-time step of the z-line preconditioner in one kernel: the
// right-hand side s + deta (H s - b) (H: the horizontal 22-point part of the
// operator; FIRST: deta (0 - b), from s = 0) and the line solve in z that
// follows it (apply_preconditioner!.jl:40-124), shared by the FP64
// preconditioner and the FP32 one.
#pragma once

#include <type_traits>

#include "pcf_internal.hpp"

namespace pcf {
namespace {

// The grid is cut into tiles of columns (FP32: 32 x 2, whose bf16 rows fill a
// 128-byte line; FP64: 16 x 1).  A tile's coefficients lie together in
// memory, [tile][k][coefficient][column], and so do its line-solve factors,
// [tile][k][P, E, Q][column] (k_line_pack): the levels of a block's columns
// are then one contiguous stream.  With x-fastest
// arrays every level and coefficient of a column lies on a page of its own,
// and the same kernel took 234 us instead of 120 at 256 x 256 x 128 (bf16).
//
// A block takes one tile; thread (x, seg) owns the NPL consecutive levels
// from seg NPL of W adjacent columns, so the block has CX ceil(nz / NPL)
// threads, CX = the tile's columns / W.  A thread evaluates the right-hand side of
// its levels in registers.  The two recurrences of the line solve,
// s_k = (r_k + e_k s_(k-1)) p_k upwards and y_k = s_k + q_k y_(k+1)
// downwards, are affine maps: a thread composes those of its levels, the
// segments' maps meet in LDS, and each thread composes the segments below
// (above) it and replays its own levels with the value that enters them.  So
// the right-hand side never goes to memory, all loads of a column are
// independent of each other, and a grid with few columns still fills the
// chip with nz / NPL threads per column.
//
// What bounds it: on a large grid memory traffic (72 B per cell with bf16
// coefficients and an FP64 right-hand side: 604 MB in 122 us, 5.0 TB/s, at
// 256 x 256 x 128; a horizontal kernel and a line solve apart took 128), on a
// small one the round trips of a thread's loads (48 x 40 x 64: 11 us against
// 23).  Before, a thread walked each column alone: 30 us for the first step
// at 128 x 128 x 128, 10.5 now.

// x-fastest coefficients and line-solve factors
template <typename T>
struct LineCoefs {
  const T* a[T_COUNT];
  const T *P, *E, *Q;
};

template <typename R>
struct LineTile {
  static constexpr int X = sizeof(R) == 8 ? 16 : 32, Y = sizeof(R) == 8 ? 1 : 2, cols = X * Y;
  static __host__ __device__ int count(int nx, int ny) { return ((nx + X - 1) / X) * ((ny + Y - 1) / Y); }
};

// The columns and levels of a thread of a tile; seg0: the block's first
// segment.
template <typename R, int W, int NPL>
struct LineThread {
  int tx, seg, i, j, k0;
  bool act;
  size_t o, c;  // the first cell in the x-fastest arrays; its level in the tile's arrays
  __device__ __forceinline__ LineThread(int tile, int nx, int ny, int nz, int seg0 = 0) {
    using T = LineTile<R>;
    constexpr int CX = T::cols / W;
    const int tiles_x = (nx + T::X - 1) / T::X;
    tx = threadIdx.x % CX;
    seg = seg0 + threadIdx.x / CX;
    i = (tile % tiles_x) * T::X + (tx * W) % T::X;
    j = (tile / tiles_x) * T::Y + (tx * W) / T::X;
    act = i < nx && j < ny;
    if (i >= nx) i = nx - W;  // idle threads read cells of the grid
    if (j >= ny) j = ny - 1;
    k0 = seg * NPL;
    o = (size_t)i + (size_t)nx * (j + (size_t)ny * k0);
    c = (size_t)tile * nz + k0;
  }
};

// bytes of dynamic LDS of a block of `threads` threads
template <typename R, int W>
constexpr unsigned line_lds(int threads) {
  return (unsigned)(4 * threads * W * sizeof(R));
}

// W consecutive values of a vector (W a power of two, the address aligned to
// them), cached or streamed past the caches
template <int W, typename T>
struct LineVec {
  typedef T type __attribute__((ext_vector_type(W)));
};
template <typename T>
struct LineVec<1, T> {
  typedef T type;
};
template <int W, bool STREAM, typename T>
__device__ __forceinline__ void line_load(const T* p, T (&o)[W]) {
  using V = typename LineVec<W, T>::type;
  V v;
  if constexpr (STREAM) v = __builtin_nontemporal_load((const V*)p);
  else v = *(const V*)p;
  if constexpr (W == 1) o[0] = v;
  else
#pragma unroll
    for (int c = 0; c < W; ++c) o[c] = v[c];
}
template <int W, typename T, typename R>
__device__ __forceinline__ void line_store(T* p, const R (&o)[W]) {
  typename LineVec<W, T>::type v;
  if constexpr (W == 1) v = (T)o[0];
  else
#pragma unroll
    for (int c = 0; c < W; ++c) v[c] = (T)o[c];
  *(typename LineVec<W, T>::type*)p = v;
}
// W coefficients as loaded (FP64, FP32, or bf16 bits, two to a word) and one
// of them in the arithmetic type
template <int W, typename CT>
struct LineCoef {
  static constexpr bool pairs = sizeof(CT) == 2 && W > 1;
  static constexpr int N = pairs ? W / 2 : W;
  using T = std::conditional_t<pairs, unsigned, CT>;
  T v[N];
  __device__ __forceinline__ void load(const CT* p) { line_load<N, true>((const T*)p, v); }
  template <typename R>
  __device__ __forceinline__ R get(int c) const {
    if constexpr (pairs) return __uint_as_float(c & 1 ? v[c / 2] & 0xffff0000u : v[c / 2] << 16);
    else if constexpr (sizeof(CT) == 2) return __uint_as_float((unsigned)v[c] << 16);
    else return v[c];
  }
};

// The line solve of the right-hand sides r of a thread's levels; y: the
// solution there, left in r.  f: the packed factors (of k_pc_factors) of the
// thread's first level and column; lds: line_lds bytes.
template <typename R, int W, int NPL>
__device__ __forceinline__ void line_solve_segments(const R* __restrict__ f, int k0, int nz, int tx, int seg, int nseg,
                                                    R (&r)[NPL][W], R* lds) {
  constexpr int cols = LineTile<R>::cols, CX = cols / W;
  R *la = lds, *lb = lds + CX * W * nseg, *lc = lb + CX * W * nseg, *ld = lc + CX * W * nseg;
  const int at = (seg * CX + tx) * W;
  R e[NPL][W], p[NPL][W], q[NPL][W];
  R A[W], B[W];
#pragma unroll
  for (int c = 0; c < W; ++c) {
    A[c] = 0;
    B[c] = 1;
  }
#pragma unroll
  for (int u = 0; u < NPL; ++u) {
    const R* fu = f + 3 * cols * (min(k0 + u, nz - 1) - k0);
    line_load<W, true>(fu, p[u]);
    line_load<W, true>(fu + cols, e[u]);
    line_load<W, true>(fu + 2 * cols, q[u]);
  }
#pragma unroll
  for (int u = 0; u < NPL; ++u) {
    const int k = k0 + u;
    const bool in = k < nz;  // else the identity map
#pragma unroll
    for (int c = 0; c < W; ++c) {
      const bool bottom = u == 0 && k == 0;  // the lowest level's P is the pivot itself
      const R rr = bottom ? r[u][c] / p[u][c] : r[u][c];
      r[u][c] = in ? rr : (R)0;
      p[u][c] = in && !bottom ? p[u][c] : (R)1;
      e[u][c] = bottom ? (R)0 : (in ? e[u][c] : (R)1);
      q[u][c] = k == nz - 1 ? (R)0 : (in ? q[u][c] : (R)1);
      A[c] = (r[u][c] + e[u][c] * A[c]) * p[u][c];
      B[c] = e[u][c] * B[c] * p[u][c];
    }
  }
#pragma unroll
  for (int c = 0; c < W; ++c) {
    la[at + c] = A[c];
    lb[at + c] = B[c];
  }
  __syncthreads();
  R sv[W];
#pragma unroll
  for (int c = 0; c < W; ++c) sv[c] = 0;
#pragma unroll 4
  for (int t = 0; t < seg; ++t)
#pragma unroll
    for (int c = 0; c < W; ++c) sv[c] = la[(t * CX + tx) * W + c] + lb[(t * CX + tx) * W + c] * sv[c];
#pragma unroll
  for (int u = 0; u < NPL; ++u)
#pragma unroll
    for (int c = 0; c < W; ++c) {
      sv[c] = (r[u][c] + e[u][c] * sv[c]) * p[u][c];
      r[u][c] = k0 + u < nz ? sv[c] : (R)0;
    }
#pragma unroll
  for (int c = 0; c < W; ++c) {
    A[c] = 0;
    B[c] = 1;
  }
#pragma unroll
  for (int u = NPL - 1; u >= 0; --u)
#pragma unroll
    for (int c = 0; c < W; ++c) {
      A[c] = r[u][c] + q[u][c] * A[c];
      B[c] = q[u][c] * B[c];
    }
#pragma unroll
  for (int c = 0; c < W; ++c) {
    lc[at + c] = A[c];
    ld[at + c] = B[c];
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < W; ++c) sv[c] = 0;
#pragma unroll 4
  for (int t = nseg - 1; t > seg; --t)
#pragma unroll
    for (int c = 0; c < W; ++c) sv[c] = lc[(t * CX + tx) * W + c] + ld[(t * CX + tx) * W + c] * sv[c];
#pragma unroll
  for (int u = NPL - 1; u >= 0; --u)
#pragma unroll
    for (int c = 0; c < W; ++c) {
      sv[c] = r[u][c] + q[u][c] * sv[c];
      r[u][c] = sv[c];
    }
}

// The same line solve for columns of any height, one column wide (W = 1), CB
// columns a block: its first `own` segments take the levels in chunks of own NPL, upwards
// and then downwards, the value at a chunk's edge going on to the next one in
// LDS; idle threads of a wider block run identity maps.  rhs(k0, r): the
// right-hand sides of the NPL levels from k0; f: the tile's packed factors at
// the thread's column; keep(k, s) and kept(k): a thread's own scratch for the
// upward sweep of all chunks but the last, inside the column; put(k, y): the
// solution at a level inside it.  lds: 2 blockDim.x + CB values.
template <typename R, int CB, int NPL, class Rhs, class Keep, class Kept, class Put>
__device__ __forceinline__ void line_solve_chunks(const R* __restrict__ f, int nz, int own, Rhs rhs,
                                                  Keep keep, Kept kept, Put put, R* lds) {
  constexpr int cols = LineTile<R>::cols;
  R *la = lds, *lb = la + blockDim.x, *edge = lb + blockDim.x;
  const int tx = threadIdx.x % CB, seg = threadIdx.x / CB;
  const int chunk = own * NPL, chunks = (nz + chunk - 1) / chunk;
  R r[NPL][1], in = 0;
  for (int ch = 0; ch < chunks; ++ch) {
    const int k0 = seg < own ? ch * chunk + seg * NPL : nz;
    rhs(k0, r);
    R p[NPL], e[NPL], A = 0, B = 1;
#pragma unroll
    for (int u = 0; u < NPL; ++u) {
      const R* fu = f + (size_t)3 * cols * min(k0 + u, nz - 1);
      p[u] = __builtin_nontemporal_load(fu);
      e[u] = __builtin_nontemporal_load(fu + cols);
    }
#pragma unroll
    for (int u = 0; u < NPL; ++u) {
      const bool lev = k0 + u < nz, bottom = u == 0 && k0 == 0;  // the lowest level's P is the pivot itself
      const R rr = bottom ? r[u][0] / p[u] : r[u][0];
      r[u][0] = lev ? rr : (R)0;
      p[u] = lev && !bottom ? p[u] : (R)1;
      e[u] = bottom ? (R)0 : (lev ? e[u] : (R)1);
      A = (r[u][0] + e[u] * A) * p[u];
      B = e[u] * B * p[u];
    }
    la[threadIdx.x] = A;
    lb[threadIdx.x] = B;
    __syncthreads();
    R s = in;
#pragma unroll 4
    for (int t = 0; t < seg; ++t) s = la[t * CB + tx] + lb[t * CB + tx] * s;
#pragma unroll
    for (int u = 0; u < NPL; ++u) {
      s = (r[u][0] + e[u] * s) * p[u];
      r[u][0] = k0 + u < nz ? s : (R)0;
    }
    if (seg == own - 1) edge[tx] = s;
    if (ch + 1 < chunks)
#pragma unroll
      for (int u = 0; u < NPL; ++u)
        if (k0 + u < nz) keep(k0 + u, r[u][0]);
    __syncthreads();  // the readers of la, lb; edge
    in = edge[tx];
  }
  in = 0;
  for (int ch = chunks - 1; ch >= 0; --ch) {
    const int k0 = seg < own ? ch * chunk + seg * NPL : nz;
    R q[NPL], A = 0, B = 1;
    if (ch + 1 < chunks)
#pragma unroll
      for (int u = 0; u < NPL; ++u) r[u][0] = k0 + u < nz ? kept(k0 + u) : (R)0;
#pragma unroll
    for (int u = 0; u < NPL; ++u)
      q[u] = __builtin_nontemporal_load(f + (size_t)3 * cols * min(k0 + u, nz - 1) + 2 * cols);
#pragma unroll
    for (int u = NPL - 1; u >= 0; --u) {
      const int k = k0 + u;
      q[u] = k == nz - 1 ? (R)0 : (k < nz ? q[u] : (R)1);
      A = r[u][0] + q[u] * A;
      B = q[u] * B;
    }
    la[threadIdx.x] = A;
    lb[threadIdx.x] = B;
    __syncthreads();
    R y = in;
#pragma unroll 4
    for (int t = own - 1; t > seg; --t) y = la[t * CB + tx] + lb[t * CB + tx] * y;
#pragma unroll
    for (int u = NPL - 1; u >= 0; --u) {
      y = r[u][0] + q[u] * y;
      if (k0 + u < nz) put(k0 + u, y);
    }
    if (seg == 0) edge[tx] = y;
    __syncthreads();
    in = edge[tx];
  }
}

// Pack a grid's x-fastest coefficients and factors (SrcT) into tiles: block
// (tile, group of levels) of cols x 256 / cols threads.  The columns beyond
// the grid of a partial tile get zero coefficients and the identity's factors.
template <typename SrcT, typename CT, typename R>
__global__ void __launch_bounds__(256) k_line_pack(LineCoefs<SrcT> A, CT* __restrict__ coefs, R* __restrict__ factors,
                                                   int nx, int ny, int nz) {
  using L = LineTile<R>;
  const int lane = threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y, tile = blockIdx.x;
  if (k >= nz) return;
  const int tx = (nx + L::X - 1) / L::X;
  const int i = (tile % tx) * L::X + lane % L::X, j = (tile / tx) * L::Y + lane / L::X;
  const bool in = i < nx && j < ny;
  const size_t o = in ? (size_t)i + (size_t)nx * (j + (size_t)ny * k) : 0;
  CT* c = coefs + ((size_t)tile * nz + k) * T_COUNT * L::cols + lane;
  R* f = factors + ((size_t)tile * nz + k) * 3 * L::cols + lane;
  for (int t = 0; t < T_COUNT; ++t) {
    if constexpr (sizeof(CT) == 2) {
      const unsigned u = in ? __float_as_uint((float)A.a[t][o]) : 0u;
      c[t * L::cols] = (CT)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);  // round to nearest even
    } else {
      c[t * L::cols] = in ? (CT)A.a[t][o] : (CT)0;
    }
  }
  f[0] = in ? (R)A.P[o] : (R)1;
  f[L::cols] = in ? (R)A.E[o] : (R)0;
  f[2 * L::cols] = in ? (R)A.Q[o] : (R)0;
}
template <typename SrcT, typename CT, typename R>
void launch_line_pack(hipStream_t s, const LineCoefs<SrcT>& A, CT* coefs, R* factors, int nx, int ny, int nz) {
  constexpr int cols = LineTile<R>::cols, rows = 256 / cols;
  hipLaunchKernelGGL((k_line_pack<SrcT, CT, R>), dim3(LineTile<R>::count(nx, ny), (nz + rows - 1) / rows),
                     dim3(cols, rows), 0, s, A, coefs, factors, nx, ny, nz);
}

// The block a launch's b-th workgroup takes: consecutive workgroups go to
// the 8 XCDs in turn, so each XCD gets a contiguous range of blocks (rows
// whose neighbours are then in its own L2).
__device__ __forceinline__ int xcd_block(int b, int nb) {
  const int per = nb / 8;
  return b < 8 * per ? (b % 8) * per + b / 8 : b;
}

// At a thread's levels k0 ... k0 + NPL - 1 of the columns (i ... i + W - 1, j)
// of an x-fastest grid: the right-hand side s + deta (H s - b), or with
// RESID the residual b - A s of all 25 points.  a: the packed coefficients of
// the thread's first level and column; rd(ii, jj, kk, v[W]) and
// rd(ii, jj, kk): the iterate at W cells and at one cell inside the grid.
// The walk up the levels keeps the five levels of s it needs in registers, so
// each is loaded once per thread.
template <typename R, int W, int NPL, int DEPTH, bool RESID, typename CT, typename BT, class Rd>
__device__ __forceinline__ void line_rhs(const CT* __restrict__ a, Rd rd, const BT* __restrict__ b, int nx, int ny,
                                         int nz, R deta, int i, int j, int k0, R (&r)[NPL][W]) {
  const size_t sxy = (size_t)nx * ny;
  const int im = i == 0 ? nx - 1 : i - 1, ip = i + W == nx ? 0 : i + W;
  const int jm = j == 0 ? ny - 1 : j - 1, jp = j + 1 == ny ? 0 : j + 1;
  // s on the levels k0 - 2 ... k0 + NPL + 1.  Every load is unconditional (at
  // a level inside the grid; those beyond the walls are zeroed where they are
  // used), so that no branch comes between the loads.  DEPTH >= 0: the
  // coefficients of the next DEPTH levels are loaded before a level is
  // evaluated and those beyond it after, which a compiler barrier at the
  // level's result keeps (without it the loads are hoisted until the registers
  // spill); DEPTH < 0 leaves the order to the compiler.
  constexpr int cols = LineTile<R>::cols;
  constexpr int LAG = DEPTH < 0 ? 0 : DEPTH, AHEAD = 4 + LAG;  // levels of s loaded before the first is evaluated
  R C[NPL + 4][W + 2], F[NPL + 4][W], B[NPL + 4][W];  // C with its x neighbours
  auto level = [&](int w) {
    const int kk = min(max(k0 - 2 + w, 0), nz - 1);
    R v[W];
    rd(i, j, kk, v);
#pragma unroll
    for (int c = 0; c < W; ++c) C[w][c + 1] = v[c];
    C[w][0] = rd(im, j, kk);
    C[w][W + 1] = rd(ip, j, kk);
    rd(i, jp, kk, F[w]);
    rd(i, jm, kk, B[w]);
  };
  LineCoef<W, CT> T[LAG + 1][T_COUNT];
  BT bv[LAG + 1][W];
  auto coefs = [&](int u) {
    const int d = u % (LAG + 1), v = min(k0 + u, nz - 1) - k0;  // v < 0 only for idle segments
    const CT* av = a + T_COUNT * cols * v;
#pragma unroll
    for (int t = 0; t < T_COUNT; ++t)
      if (RESID || (t != T_AC && t != T_AD && t != T_AU)) T[d][t].load(av + t * cols);
    line_load<W, true>(b + ((size_t)i + (size_t)nx * j + sxy * (size_t)(k0 + v)), bv[d]);
  };
#pragma unroll
  for (int w = 0; w < AHEAD && w < NPL + 4; ++w) level(w);
#pragma unroll
  for (int u = 0; u < LAG; ++u) coefs(u);
#pragma unroll
  for (int u = 0; u < NPL; ++u) {
    const int m = u + 2, d = u % (LAG + 1);
    if (AHEAD + u < NPL + 4) level(AHEAD + u);
    if (u + LAG < NPL) coefs(u + LAG);
    // (without it the 16-level kernel's bf16 loads sink to their uses, one
    // round trip each: 152 us against 42 at 64 x 64 x 160, 650 against 204 at
    // 256 x 256 x 160)
    if constexpr (DEPTH == 0 && sizeof(CT) == 2) asm volatile("" ::: "memory");
    const int k = k0 + u;
#pragma unroll
    for (int c = 0; c < W; ++c) {
      auto A = [&](int t) -> R { return T[d][t].template get<R>(c); };
      // the levels two below ... two above; zero beyond the walls
      auto Z = [&](R x, int w) -> R {
        const int kk = k0 + w - 2;
        return w == m ? x : ((unsigned)kk < (unsigned)nz ? x : (R)0);
      };
      auto XL = [&](int w) -> R { return Z(C[w][c], w); };
      auto XR = [&](int w) -> R { return Z(C[w][c + 2], w); };
      auto X0 = [&](int w) -> R { return Z(C[w][c + 1], w); };
      auto YF = [&](int w) -> R { return Z(F[w][c], w); };
      auto YB = [&](int w) -> R { return Z(B[w][c], w); };
      R v = A(T_AL) * XL(m) + A(T_AR) * XR(m) + A(T_AF) * YF(m) + A(T_AB) * YB(m);
      if constexpr (RESID) v += A(T_AU) * X0(m + 1) + A(T_AD) * X0(m - 1) + A(T_AC) * X0(m);
      v += A(T_ARU) * XR(m + 1) + A(T_ARD) * XR(m - 1) + A(T_ALU) * XL(m + 1) + A(T_ALD) * XL(m - 1) +
           A(T_AFU) * YF(m + 1) + A(T_AFD) * YF(m - 1) + A(T_ABU) * YB(m + 1) + A(T_ABD) * YB(m - 1) +
           A(T_AUU) * X0(m + 2) + A(T_ADD) * X0(m - 2) + A(T_ARUU) * XR(m + 2) + A(T_ARDD) * XR(m - 2) +
           A(T_ALUU) * XL(m + 2) + A(T_ALDD) * XL(m - 2) + A(T_AFUU) * YF(m + 2) + A(T_AFDD) * YF(m - 2) +
           A(T_ABUU) * YB(m + 2) + A(T_ABDD) * YB(m - 2);
      const R rr = RESID ? (R)bv[d][c] - v : X0(m) + deta * (v - (R)bv[d][c]);
      r[u][c] = k < nz ? rr : (R)0;
      if constexpr (DEPTH >= 0) asm volatile("" : "+v"(r[u][c])::"memory");
    }
  }
}

}  // namespace
}  // namespace pcf
