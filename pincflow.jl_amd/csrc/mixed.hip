// Mixed-precision pressure solve (precision = PCF_PRECISION_MIXED).
//
// BiCGSTAB keeps the reference's FP64 Krylov iteration (apply_bicgstab!.jl:
// 24-150): the operator applies, the residual recurrence, the dot products,
// norms and scalars and the solution update stay FP64.  The preconditioner
// (apply_preconditioner!.jl:40-124) runs in FP32 on FP32 copies of the 22
// horizontal operator coefficients and of the line-solve factors, which
// halves its traffic.  Because an FP32 M^-1 is not exactly linear, the
// solution is accumulated in the textbook form x += alpha M^-1 p + omega M^-1 s
// (bicgstab_core, k_bicg_xr_yz), which keeps x consistent with the FP64
// residual recurrence; the stopping test is the reference criterion.
//
// Optionally (initial_guess = PCF_GUESS_PREVIOUS) each implicit stage starts
// from the same stage's solution of the previous time step, rescaled by the
// ratio of the time steps (the solution is proportional to dt times the
// pressure correction), or (PCF_GUESS_EXTRAPOLATED) from the linear
// extrapolation in time of the last two; the criterion stays |r| / |b|.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "line_step.hpp"
#include "pcf_device.hpp"
#include "solver_common.hpp"

namespace pcf {

namespace {

// Memory layout of a level's arrays: x fastest (the finest level and the
// levels smoothed with row-parallel kernels) or z fastest (the coarse levels
// smoothed one column per wavefront, whose accesses are then contiguous
// across the lanes of a wavefront).
struct Lay {
  int nx, ny, nz;
  bool zf;
  __host__ __device__ size_t at(int i, int j, int k) const {
    return zf ? (size_t)k + (size_t)nz * ((size_t)i + (size_t)nx * j)
              : (size_t)i + (size_t)nx * ((size_t)j + (size_t)ny * k);
  }
  // 32-bit form for the levels smoothed column by column (at most
  // kCoarseColumnCols x kScanMaxNz cells)
  __device__ int at32(int i, int j, int k) const { return zf ? k + nz * (i + nx * j) : i + nx * (j + ny * k); }
  __host__ __device__ size_t count() const { return (size_t)nx * ny * nz; }
  // the cell of the t-th element in memory order
  __device__ void cell(size_t t, int& i, int& j, int& k) const {
    if (zf) {
      k = (int)(t % nz);
      const size_t c = t / nz;
      i = (int)(c % nx);
      j = (int)(c / nx);
    } else {
      i = (int)(t % nx);
      const size_t r = t / nx;
      j = (int)(r % ny);
      k = (int)(r / ny);
    }
  }
};

// A pseudo-time step's operands on an x-fastest grid: the packed coefficients
// (CT: float, or uint16_t holding bf16 bits, the upper half of an FP32) and
// factors, and the iterate.
template <typename CT>
struct LineArgs {
  const CT* coefs;
  const float* factors;
  const float* s;
  int nx, ny, nz;
  float deta;
  // coarse-level correction added to s first (PRO = true): s + omega e at
  // the coarse cell (i >> sx, j >> sy, k) in layout cl
  const float* e;
  float omega;
  int sx, sy;
  Lay cl;
};

// The iterate of a step: s, or with PRO s + omega P e, the multigrid
// prolongation of the coarse-level correction fused into the first
// post-smoothing step.
template <int W, bool PRO, typename CT>
struct LineRead {
  const LineArgs<CT>& A;
  __device__ __forceinline__ float operator()(int i, int j, int k) const {
    float v = A.s[(size_t)i + (size_t)A.nx * (j + (size_t)A.ny * k)];
    if constexpr (PRO) v += A.omega * A.e[A.cl.at(i >> A.sx, j >> A.sy, k)];
    return v;
  }
  __device__ __forceinline__ void operator()(int i, int j, int k, float (&v)[W]) const {
    line_load<W, false>(A.s + ((size_t)i + (size_t)A.nx * (j + (size_t)A.ny * k)), v);
    if constexpr (PRO) {
      if constexpr (W == 4) {
        if (A.sx == 1 && !A.cl.zf) {  // the two coarse cells of the four fine ones
          float e[2];
          line_load<2, false>(A.e + A.cl.at(i >> 1, j >> A.sy, k), e);
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] += A.omega * e[c / 2];
          return;
        }
      }
#pragma unroll
      for (int c = 0; c < W; ++c) v[c] += A.omega * A.e[A.cl.at((i + c) >> A.sx, j >> A.sy, k)];
    }
  }
};

constexpr int kTileCols = LineTile<float>::cols, kTileX = LineTile<float>::X;

// One pseudo-time step in FP32 of a tile (line_step.hpp); s and out must
// differ.
template <int W, int NPL, bool FIRST, bool PRO, typename CT, typename BT, typename OutT>
__device__ __forceinline__ void line_step32(const LineArgs<CT>& A, const BT* __restrict__ b, OutT* __restrict__ out,
                                            int tile) {
  extern __shared__ float line_shared[];
  const int nx = A.nx, ny = A.ny, nz = A.nz;
  const LineThread<float, W, NPL> t(tile, nx, ny, nz);
  const size_t sxy = (size_t)nx * ny;
  float r[NPL][W];
  if constexpr (FIRST) {
#pragma unroll
    for (int u = 0; u < NPL; ++u) {
      BT v[W];
      line_load<W, false>(b + (t.o + sxy * (ptrdiff_t)(min(t.k0 + u, nz - 1) - t.k0)), v);
#pragma unroll
      for (int c = 0; c < W; ++c) r[u][c] = t.k0 + u < nz ? A.deta * (0.0f - (float)v[c]) : 0.0f;
    }
  } else {
    // what the registers allow
    constexpr int DEPTH = W == 1 && NPL <= 8 && !PRO ? 1 : W == 4 && !PRO && sizeof(CT) == 2 ? -1 : 0;
    line_rhs<float, W, NPL, DEPTH, false, CT, BT>(A.coefs + t.c * T_COUNT * kTileCols + t.tx * W, LineRead<W, PRO, CT>{A}, b,
                                           nx, ny, nz, A.deta, t.i, t.j, t.k0, r);
  }
  line_solve_segments<float, W, NPL>(A.factors + t.c * 3 * kTileCols + t.tx * W, t.k0, nz, t.tx, t.seg,
                                     blockDim.x / (kTileCols / W), r, line_shared);
  if (t.act) {
#pragma unroll
    for (int u = 0; u < NPL; ++u)
      if (t.k0 + u < nz) line_store<W>(out + t.o + sxy * u, r[u]);
  }
}
// commit: the kernel before was a FUSE_P one
template <int W, int NPL, bool FIRST, bool PRO, typename CT, typename BT, typename OutT>
__global__ void __launch_bounds__(W == 4 ? 512 : 1024) __attribute__((amdgpu_waves_per_eu(W == 4 ? 2 : 4, W == 4 ? 2 : 4)))
    k_line_step32(LineArgs<CT> A, const BT* __restrict__ b, OutT* __restrict__ out, const SolverScalars* sc,
                  SolverScalars* commit) {
  if (!FIRST && commit) {
    if (!fuse_commit(commit)) return;
  } else if (sc && sc->done) {
    return;
  }
  line_step32<W, NPL, FIRST, PRO, CT, BT, OutT>(A, b, out, xcd_block(blockIdx.x, gridDim.x));
}

// The first pseudo-time step of the vector that a fused BiCGSTAB step updates
// first.
template <int NPL, int FUSE>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4, 4)))
    k_line_fuse32(LineArgs<float> A, BicgFuse F, float* __restrict__ out) {
  extern __shared__ float line_shared[];
  const LineThread<float, 1, NPL> t(xcd_block(blockIdx.x, gridDim.x), A.nx, A.ny, A.nz);
  const size_t sxy = (size_t)A.nx * A.ny;
  FuseOperands<FUSE, NPL> X;
  if (t.act) {
#pragma unroll
    for (int u = 0; u < NPL; ++u)
      X.load(F, u, t.o + sxy * (ptrdiff_t)(min(t.k0 + u, A.nz - 1) - t.k0), t.k0 + u < A.nz);
  }
  FuseScalars S;
  if (!fuse_scalars<FUSE>(F, S)) return;
  float r[NPL][1];
#pragma unroll
  for (int u = 0; u < NPL; ++u) {
    r[u][0] = 0.0f;
    if (t.act && t.k0 + u < A.nz) {
      const double x = fuse_value(X, S, u);
      F.dst[t.o + sxy * u] = x;
      r[u][0] = A.deta * (0.0f - (float)x);
    }
  }
  line_solve_segments<float, 1, NPL>(A.factors + t.c * 3 * kTileCols + t.tx, t.k0, A.nz, t.tx, t.seg,
                                     blockDim.x / kTileCols, r, line_shared);
  if (t.act) {
#pragma unroll
    for (int u = 0; u < NPL; ++u)
      if (t.k0 + u < A.nz) out[t.o + sxy * u] = r[u][0];
  }
}

constexpr int kLineMaxNz = 256;  // most levels of k_line_step32's columns (taller ones, and on few tiles those of
                                 // more than 128: k_line_tall32)

// A block of a tall column's step: CB columns of a tile, NPL levels per
// thread, and the segments of its chunks, the fewest chunks that 1024 threads
// allow with the levels spread over them.
template <int CB, int NPL>
struct TallBlock {
  static constexpr int columns = CB, npl = NPL, parts = kTileCols / CB;  // blocks per tile
  static __host__ __device__ int segments(int nz) {
    const int most = 1024 / CB * NPL, chunks = (nz + most - 1) / most, levels = (nz + chunks - 1) / chunks;
    return (levels + NPL - 1) / NPL;
  }
};
// Whole tiles, and half tiles on grids of few tiles, whose twice as many blocks
// do not yet outnumber the 256 CUs and take half the chunks.  Whole / half
// tiles, bf16, one application of two steps at 300 levels: 76 / 55 us on 64
// tiles (64 x 64), 88 / 76 on 128 (128 x 64), 92 / 108 on 144 (96 x 96).  The
// step that adds the coarse correction (PRO) spills with 16 levels per thread
// and takes smaller blocks of 8 on few tiles: V-cycles of 1105 / 1007 us at
// 64 x 64 x 600, 270 / 241 at 48 x 40 x 200.
constexpr int kTallFewTiles = 128;
template <bool PRO, class F>
__host__ __device__ inline void with_tall_block(int nx, int ny, int nz, F&& f) {
  const bool few = LineTile<float>::count(nx, ny) <= kTallFewTiles;
  if (PRO && few && nz <= 256) f(TallBlock<32, 8>{});
  else if (PRO && few) f(TallBlock<16, 8>{});
  else if (few) f(TallBlock<32, 16>{});
  else f(TallBlock<64, 16>{});
}

// The same step for tall columns, chunk by chunk;
// col: FP32 scratch of the grid's size, which keeps the upward sweep of all
// chunks but the last (null up to kLineMaxNz levels, one chunk).  Like
// the shorter columns it is bound by memory on a large grid and by the round
// trips of a chunk on a small one.  One application of two steps, FP32 / bf16
// storage, with a horizontal kernel and a line solve apart, with a thread per
// column for both, and chunk by chunk:
//   64 x 64 x 300    145 / 138   632 / 614    63 /  55 us
//   256 x 128 x 320  382 / 307   836 / 802   312 / 232 us
template <class TB, bool FIRST, bool PRO, typename CT, typename BT, typename OutT>
__device__ __forceinline__ void line_tall32(const LineArgs<CT>& A, const BT* __restrict__ b, OutT* __restrict__ out,
                                            float* col, int block) {
  extern __shared__ float line_shared[];
  constexpr int NPL = TB::npl;
  const int nx = A.nx, ny = A.ny, nz = A.nz, tile = block / TB::parts;
  const int tx = block % TB::parts * TB::columns + threadIdx.x % TB::columns, tiles_x = (nx + kTileX - 1) / kTileX;
  int i = tile % tiles_x * kTileX + tx % kTileX, j = tile / tiles_x * LineTile<float>::Y + tx / kTileX;
  const bool act = i < nx && j < ny;
  i = min(i, nx - 1);  // idle threads read cells of the grid
  j = min(j, ny - 1);
  const size_t sxy = (size_t)nx * ny, c = (size_t)i + (size_t)nx * j, tc = (size_t)tile * nz;
  auto rhs = [&](int k0, float (&r)[NPL][1]) {
    if constexpr (FIRST) {
#pragma unroll
      for (int u = 0; u < NPL; ++u)
        r[u][0] = A.deta * (0.0f - (float)__builtin_nontemporal_load(b + c + sxy * min(k0 + u, nz - 1)));
    } else {
      line_rhs<float, 1, NPL, 0, false, CT, BT>(
          A.coefs + (tc + k0) * T_COUNT * kTileCols + tx, LineRead<1, PRO, CT>{A}, b, nx, ny, nz, A.deta, i, j, k0, r);
    }
  };
  // (idle columns of a partial tile keep nothing: their cells are another's)
  line_solve_chunks<float, TB::columns, NPL>(
      A.factors + tc * 3 * kTileCols + tx, nz, TB::segments(nz), rhs,
      [&](int k, float s) { if (act) col[c + sxy * k] = s; },
      [&](int k) { return act ? col[c + sxy * k] : 0.0f; },
      [&](int k, float y) { if (act) out[c + sxy * k] = (OutT)y; }, line_shared);
}
template <class TB, bool FIRST, bool PRO, typename CT, typename BT, typename OutT>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4, 4)))
    k_line_tall32(LineArgs<CT> A, const BT* __restrict__ b, OutT* __restrict__ out, float* col,
                  const SolverScalars* sc, SolverScalars* commit) {
  if (!FIRST && commit) {
    if (!fuse_commit(commit)) return;
  } else if (sc && sc->done) {
    return;
  }
  line_tall32<TB, FIRST, PRO, CT, BT, OutT>(A, b, out, col, xcd_block(blockIdx.x, gridDim.x));
}

__global__ void k_to_f32(const double* a, float* b, size_t n) {
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    b[q] = (float)a[q];
}

// g = q1 + r (q1 - q2): the linear extrapolation in time of the last two
// solutions per unit time step (r: this step over the previous one)
__global__ void k_extrapolate(const double* q1, const double* q2, double* g, size_t n, double r) {
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    g[q] = q1[q] + r * (q1[q] - q2[q]);
}

// g = c x (the saved warm start, c = 1 / dt)
__global__ void k_scale_copy(const double* x, double* g, size_t n, double c) {
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    g[q] = c * x[q];
}

// ---------------------------------------------------------------------------
// Multigrid preconditioner (FP32).  The coarse operator of level l+1 is the
// Galerkin product R A P of level l with piecewise-constant aggregation of
// fx x fy columns (P: copy a coarse value to its fine cells, R = P^T: sum
// over them); z is never coarsened, so the z-line pseudo-time step of the
// reference preconditioner remains the smoother on every level.  Because
// the fine stencil couples a cell with x or y neighbours but never with
// diagonal ones, R A P has the same 25-point shape.
// ---------------------------------------------------------------------------
constexpr float kMgOmega = 1.5f;     // over-correction of the coarse-level correction
constexpr int kMgMinSize = 8;        // a dimension is coarsened while even and >= this

// (di, dj, dk) of the 25 coefficients in the order of T_AC ... T_AFUU
__device__ constexpr int kOffI[T_COUNT] = {0, -1, 1, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0};
__device__ constexpr int kOffJ[T_COUNT] = {0, 0, 0, -1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1};
__device__ constexpr int kOffK[T_COUNT] = {0, 0, 0, 0, 0, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1, -2, 2, -2, 2, -2, 2, -2, 2, -2, 2};

// coefficient index of the offset (di, dj, dk); -1 if none
__host__ __device__ constexpr int coef_of(int di, int dj, int dk) {
  for (int t = 0; t < T_COUNT; ++t) {
    const int oi[T_COUNT] = {0, -1, 1, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0};
    const int oj[T_COUNT] = {0, 0, 0, -1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1};
    const int ok[T_COUNT] = {0, 0, 0, 0, 0, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1, -2, 2, -2, 2, -2, 2, -2, 2, -2, 2};
    if (oi[t] == di && oj[t] == dj && ok[t] == dk) return t;
  }
  return -1;
}
__host__ __device__ constexpr int floor_div(int a, int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }

struct MgCoefs {
  float* a[T_COUNT];
};

// R A P: one thread per coarse cell, in the coarse level's memory order.
// FT: the fine coefficients, FP32, or the finest level's in FP64, each rounded
// to FP32 where it is added: the same sums as from FP32 copies, without the 28
// conversions a solve (23 us each at 256 x 256 x 128) and the arrays' memory.
template <int FX, int FY, typename FT>
__global__ void k_mg_coarsen(LineCoefs<FT> fine, MgCoefs coarse, Lay fl, Lay cl) {
  const size_t t0 = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (t0 >= cl.count()) return;
  int I, J, k;
  cl.cell(t0, I, J, k);
  constexpr int oi[T_COUNT] = {0, -1, 1, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0};
  constexpr int oj[T_COUNT] = {0, 0, 0, -1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1};
  constexpr int ok[T_COUNT] = {0, 0, 0, 0, 0, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1, -2, 2, -2, 2, -2, 2, -2, 2, -2, 2};
  float acc[T_COUNT];
#pragma unroll
  for (int t = 0; t < T_COUNT; ++t) acc[t] = 0.0f;
#pragma unroll
  for (int b = 0; b < FY; ++b)
#pragma unroll
    for (int a = 0; a < FX; ++a) {
      const size_t o = fl.at(FX * I + a, FY * J + b, k);
#pragma unroll
      for (int t = 0; t < T_COUNT; ++t) {
        const int target = coef_of(floor_div(a + oi[t], FX), floor_div(b + oj[t], FY), ok[t]);
        acc[target] += (float)fine.a[t][o];
      }
    }
#pragma unroll
  for (int t = 0; t < T_COUNT; ++t) coarse.a[t][t0] = acc[t];
}

// Line-solve factors (see k_pc_factors) of a coarse operator, in FP32: one
// thread per column.
__global__ void __launch_bounds__(64) k_mg_factors(const float* ac, const float* ad, const float* au, float* P, float* E,
                                                   float* Q, Lay l, float deta) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= l.nx * l.ny) return;
  const int i = c % l.nx, j = c / l.nx;
  size_t o = l.at(i, j, 0);
  const float denom = 1 - deta * ac[o];
  float qk = deta * au[o] / denom;
  P[o] = denom;
  E[o] = deta * ad[o];
  Q[o] = qk;
  for (int k = 1; k < l.nz; ++k) {
    o = l.at(i, j, k);
    const float e = deta * ad[o];
    const float p = 1 / (1 - deta * ac[o] - e * qk);
    qk = deta * au[o] * p;
    P[o] = p;
    E[o] = e;
    Q[o] = qk;
  }
}

// The operands of A s at cell (i, j, k) of a level: a and x, zero beyond the walls.
__device__ __forceinline__ void resid_operands(const MgCoefs& A, const float* __restrict__ s, const Lay& l, int i, int j,
                                               int k, float (&a)[T_COUNT], float (&x)[T_COUNT]) {
  constexpr int oi[T_COUNT] = {0, -1, 1, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0};
  constexpr int oj[T_COUNT] = {0, 0, 0, -1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0, 0, 0, -1, -1, 1, 1};
  constexpr int ok[T_COUNT] = {0, 0, 0, 0, 0, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1, -2, 2, -2, 2, -2, 2, -2, 2, -2, 2};
  const size_t o = l.at(i, j, k);
#pragma unroll
  for (int t = 0; t < T_COUNT; ++t) {
    int ii = i + oi[t], jj = j + oj[t];
    ii = ii < 0 ? ii + l.nx : (ii >= l.nx ? ii - l.nx : ii);
    jj = jj < 0 ? jj + l.ny : (jj >= l.ny ? jj - l.ny : jj);
    a[t] = A.a[t][o];
    x[t] = s[l.at(ii, jj, min(max(k + ok[t], 0), l.nz - 1))];
  }
#pragma unroll
  for (int t = 0; t < T_COUNT; ++t) x[t] = (unsigned)(k + ok[t]) < (unsigned)l.nz ? x[t] : 0.0f;
}

// b_coarse = R (b - A s) on a z-fastest level: block (64, FX FY) of 64
// levels of one coarse column, one thread per fine cell, whose residuals are
// summed in LDS in the order of the fine columns.
template <int FX, int FY, typename BT>
__global__ void __launch_bounds__(256) k_resid_restrict_columns(MgCoefs A, const BT* __restrict__ b,
                                                            const float* __restrict__ s, float* __restrict__ bc,
                                                            Lay l, Lay cl, const SolverScalars* sc) {
  if (sc && sc->done) return;
  __shared__ float part[FX * FY][64];
  const int nz = l.nz, nkb = (nz + 63) / 64;
  const int col = blockIdx.x / nkb, k = 64 * (blockIdx.x % nkb) + threadIdx.x;
  const int I = col % cl.nx, J = col / cl.nx, n = threadIdx.y;
  const int i = FX * I + n % FX, j = FY * J + n / FX;
  const int kc = min(k, nz - 1);
  float a[T_COUNT], x[T_COUNT], v = 0.0f;
  resid_operands(A, s, l, i, j, kc, a, x);
#pragma unroll
  for (int t = 0; t < T_COUNT; ++t) v += a[t] * x[t];
  part[n][threadIdx.x] = (float)b[l.at(i, j, kc)] - v;
  __syncthreads();
  if (n == 0 && k < nz) {
    float sum = 0.0f;
#pragma unroll
    for (int q = 0; q < FX * FY; ++q) sum += part[q][threadIdx.x];
    bc[cl.at(I, J, k)] = sum;
  }
}

// The same on an x-fastest level without packed 2 x 2 tiles: one thread per
// fine x position, level and coarse row, in memory order, so that a
// wavefront's accesses are contiguous (the kernel above, whose lanes run over
// z, took 2941 us against 1308 for a V-cycle at 255 x 256 x 64).  The x pairs
// are summed across lanes.
template <int FX, int FY, typename BT>
__global__ void __launch_bounds__(256) k_resid_restrict_rows(MgCoefs A, const BT* __restrict__ b,
                                                             const float* __restrict__ s, float* __restrict__ bc,
                                                             Lay l, Lay cl, const SolverScalars* sc) {
  if (sc && sc->done) return;
  const unsigned nx = l.nx, cy = cl.ny;
  const unsigned q = xcd_block(blockIdx.x, gridDim.x) * 256u + threadIdx.x;
  if (q >= nx * cy * l.nz) return;  // a pair's lanes stay or leave together
  const int i = q % nx, J = q / nx % cy, k = q / nx / cy;
  float sum = 0.0f;
#pragma unroll
  for (int n = 0; n < FY; ++n) {
    const int j = FY * J + n;
    float a[T_COUNT], x[T_COUNT], v = 0.0f;
    resid_operands(A, s, l, i, j, k, a, x);
#pragma unroll
    for (int t = 0; t < T_COUNT; ++t) v += a[t] * x[t];
    const float r = (float)b[l.at(i, j, k)] - v;
    sum += r;
    if constexpr (FX == 2) sum += __shfl_down(r, 1);
  }
  if (i % FX == 0) bc[cl.at(i / FX, J, k)] = sum;
}

// b_coarse = R (b - A s) for 2 x 2 aggregation of a level with packed tiles: a
// block per tile (blockIdx.y: its part of a column of more levels than a block
// has) as in the line steps; the x pairs are summed in the thread (W = 4) or
// across lanes, the rows j and j + 1 of a tile across lanes.
template <int W, int NPL, typename BT, typename CT>
__global__ void __launch_bounds__(W == 4 ? 512 : 1024)
    __attribute__((amdgpu_waves_per_eu(W == 4 ? 2 : 4, W == 4 ? 2 : 4))) k_resid_restrict(LineArgs<CT> A, const BT* __restrict__ b,
                                                         float* __restrict__ bc, const SolverScalars* sc) {
  if (sc && sc->done) return;
  const int nx = A.nx, ny = A.ny, nz = A.nz;
  const int tile = xcd_block(blockIdx.x, gridDim.x);
  const LineThread<float, W, NPL> t(tile, nx, ny, nz, blockIdx.y * (blockDim.x / (kTileCols / W)));
  float r[NPL][W];
  line_rhs<float, W, NPL, W == 1 && NPL == 8 ? 1 : 0, true, CT, BT>(A.coefs + t.c * T_COUNT * kTileCols + t.tx * W, LineRead<W, false, CT>{A}, b,
                                        nx, ny, nz, A.deta, t.i, t.j, t.k0, r);
  constexpr int row = kTileX / W;  // threads per row of the tile
#pragma unroll
  for (int u = 0; u < NPL; ++u) {
    const int k = t.k0 + u;
    if constexpr (W == 4) {
      const float c0 = r[u][0] + r[u][1], c1 = r[u][2] + r[u][3];
      // every lane takes part in the exchange
      const float u0 = __shfl_down(c0, row), u1 = __shfl_down(c1, row);
      if (t.act && k < nz && (t.tx & row) == 0) {
        bc[A.cl.at(t.i / 2, t.j / 2, k)] = c0 + u0;
        bc[A.cl.at(t.i / 2 + 1, t.j / 2, k)] = c1 + u1;
      }
    } else {
      const float c0 = r[u][0] + __shfl_down(r[u][0], 1);
      const float u0 = __shfl_down(c0, row);
      if (t.act && k < nz && (t.tx & row) == 0 && (t.i & 1) == 0) bc[A.cl.at(t.i / 2, t.j / 2, k)] = c0 + u0;
    }
  }
}

// ---------------------------------------------------------------------------
// Line solves with one wavefront per column.  The z recurrences of the line
// solve are affine maps, s_k = fa_k + fb_k s_(k-1) upwards and
// y_k = col_k + q_k y_(k+1) downwards; lane l holds NPL consecutive levels,
// composes its maps and an inclusive scan over the 64 lanes (shuffles)
// composes the rest, so a column costs one round trip to memory instead of
// nz dependent steps.  Used where there are too few columns to hide the
// latency of the thread-per-column sweep.
// ---------------------------------------------------------------------------
template <int NPL>
__device__ __forceinline__ void scan_line(const float (&fa)[NPL], const float (&fb)[NPL], const float (&q)[NPL],
                                          int nz, float (&y)[NPL]) {
  const int lane = threadIdx.x & 63;
  float A = 0.0f, B = 1.0f;
#pragma unroll
  for (int u = 0; u < NPL; ++u) {
    A = fa[u] + fb[u] * A;
    B = fb[u] * B;
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float Ap = __shfl_up(A, off), Bp = __shfl_up(B, off);
    if (lane >= off) {
      A = A + B * Ap;
      B = B * Bp;
    }
  }
  float sv = __shfl_up(A, 1);
  if (lane == 0) sv = 0.0f;  // the map of level 0 does not depend on it
  float col[NPL];
#pragma unroll
  for (int u = 0; u < NPL; ++u) {
    sv = fa[u] + fb[u] * sv;
    col[u] = NPL * lane + u < nz ? sv : 0.0f;
  }
  float Cc = 0.0f, D = 1.0f;
#pragma unroll
  for (int u = NPL - 1; u >= 0; --u) {
    Cc = col[u] + q[u] * Cc;
    D = q[u] * D;
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float Cn = __shfl_down(Cc, off), Dn = __shfl_down(D, off);
    if (lane + off < 64) {
      Cc = Cc + D * Cn;
      D = D * Dn;
    }
  }
  float t = __shfl_down(Cc, 1);
  if (lane == 63) t = 0.0f;  // above the top level: q = 0 there
#pragma unroll
  for (int u = NPL - 1; u >= 0; --u) {
    t = col[u] + q[u] * t;
    y[u] = t;
  }
}

// The forward map of level k of a column from its line-solve factors p, e, q
// (those of a level inside the column) and right-hand side r (k = 0: p holds
// the pivot itself); identity maps above nz.
__device__ __forceinline__ void line_maps(float p, float e, float qv, int k, int nz, float r, float& fa, float& fb,
                                          float& q) {
  const bool in = k < nz;
  const float a = k == 0 ? r / p : r * p, b = k == 0 ? 0.0f : e * p;
  fa = in ? a : 0.0f;
  fb = in ? b : 1.0f;
  q = in ? (k == nz - 1 ? 0.0f : qv) : 1.0f;
}

// One pseudo-time step of column (i, j): the right-hand side
// s + deta (H s - b) at the lane's levels (FIRST: deta (0 - b), from s = 0),
// then the line solve.  rd(i, j, k) reads the current iterate; the level's
// arrays are in layout l.
template <int NPL, bool FIRST, typename BT, class Rd>
__device__ __forceinline__ void column_step(const MgCoefs& A, const float* P, const float* E, const float* Q,
                                            const BT* b, Rd rd, const Lay& l, int i, int j, float deta,
                                            float (&y)[NPL]) {
  const int lane = threadIdx.x & 63;
  const int nx = l.nx, ny = l.ny, nz = l.nz;
  const int im = i == 0 ? nx - 1 : i - 1, ip = i + 1 == nx ? 0 : i + 1;
  const int jm = j == 0 ? ny - 1 : j - 1, jp = j + 1 == ny ? 0 : j + 1;
  float fa[NPL], fb[NPL], q[NPL];
  // every load is unconditional, at a level inside the column (zeroed beyond
  // the walls where it is used): a branch per neighbour made each load wait
  // for the one before (14 us against 7 for a first post-smoothing step at
  // 32 x 32 x 128).  With four levels per lane or more the barrier below keeps
  // one level's loads in flight: those of all spilt (k_coarse_solve at 10 x 1 x
  // 160: 15.4 us a step against 6.7; the 26 x 16 x 400 level's post-smoothing
  // 55 against 52).
#pragma unroll
  for (int u = 0; u < NPL; ++u) {
    const int k = NPL * lane + u;
    const int kc = k < nz ? k : nz - 1;
    const int o = l.at32(i, j, kc);
    const float p = P[o], e = E[o], qv = Q[o];
    float r;
    if constexpr (FIRST) {
      r = deta * (0.0f - (float)b[o]);
    } else {
      float a[T_COUNT], s[5][5];  // s: the column and its x and y neighbours on levels k - 2 ... k + 2
#pragma unroll
      for (int t = 0; t < T_COUNT; ++t)
        if (t != T_AC && t != T_AD && t != T_AU) a[t] = A.a[t][o];
#pragma unroll
      for (int w = 0; w < 5; ++w) {
        const int kk = min(max(kc - 2 + w, 0), nz - 1);
        s[0][w] = rd(i, j, kk);
        s[1][w] = rd(im, j, kk);
        s[2][w] = rd(ip, j, kk);
        s[3][w] = rd(i, jm, kk);
        s[4][w] = rd(i, jp, kk);
      }
      const float bv = (float)b[o];
#pragma unroll
      for (int w = 0; w < 5; ++w)
#pragma unroll
        for (int n = 0; n < 5; ++n) s[n][w] = (unsigned)(kc - 2 + w) < (unsigned)nz ? s[n][w] : 0.0f;
      float v = a[T_AL] * s[1][2] + a[T_AR] * s[2][2] + a[T_AF] * s[4][2] + a[T_AB] * s[3][2];
      v += a[T_ARU] * s[2][3] + a[T_ARD] * s[2][1] + a[T_ALU] * s[1][3] + a[T_ALD] * s[1][1] + a[T_AFU] * s[4][3] +
           a[T_AFD] * s[4][1] + a[T_ABU] * s[3][3] + a[T_ABD] * s[3][1] + a[T_AUU] * s[0][4] + a[T_ADD] * s[0][0] +
           a[T_ARUU] * s[2][4] + a[T_ARDD] * s[2][0] + a[T_ALUU] * s[1][4] + a[T_ALDD] * s[1][0] +
           a[T_AFUU] * s[4][4] + a[T_AFDD] * s[4][0] + a[T_ABUU] * s[3][4] + a[T_ABDD] * s[3][0];
      r = s[0][2] + deta * (v - bv);
    }
    line_maps(p, e, qv, k, nz, r, fa[u], fb[u], q[u]);
    if (!FIRST && NPL >= 4 && u + 1 < NPL) asm volatile("" : "+v"(fa[u])::"memory");
  }
  scan_line<NPL>(fa, fb, q, nz, y);
}

// One smoothing step of a level with few columns, one wavefront per column
// (block 256 = 4 columns); s_old and out must differ.  PRO: the iterate is
// s_old + omega P e (e: the coarse-level correction in layout cl,
// fx = 1 << sx, fy = 1 << sy).  ol: the layout of out.
template <int NPL, bool FIRST, bool PRO, typename BT, typename OutT>
__global__ void __launch_bounds__(256) k_col_smooth(MgCoefs A, const float* __restrict__ P,
                                                    const float* __restrict__ E, const float* __restrict__ Q,
                                                    const BT* __restrict__ b, const float* __restrict__ s_old,
                                                    const float* __restrict__ e, float omega, int sx, int sy, Lay l,
                                                    Lay cl, OutT* __restrict__ out, Lay ol, float deta,
                                                    const SolverScalars* sc) {
  if (sc && sc->done) return;
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= l.nx * l.ny) return;  // uniform over the wavefront
  const int i = c % l.nx, j = c / l.nx;
  auto rd = [&](int ii, int jj, int kk) -> float {
    float v = s_old[l.at32(ii, jj, kk)];
    if (PRO) v += omega * e[cl.at32(ii >> sx, jj >> sy, kk)];
    return v;
  };
  float y[NPL];
  column_step<NPL, FIRST, BT>(A, P, E, Q, b, rd, l, i, j, deta, y);
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int u = 0; u < NPL; ++u) {
    const int k = NPL * lane + u;
    if (k < l.nz) out[ol.at32(i, j, k)] = (OutT)y[u];
  }
}

// All smoothing steps of the coarsest level in one workgroup of up to 16
// wavefronts, wavefront w smoothing the columns w, w + 16, ... (nx ny <= 16),
// the iterate ping-ponging between two z-fastest LDS buffers (2 nx ny nz
// floats of dynamic shared memory), so a column's new values are stored as
// soon as they are computed.
template <int NPL, typename BT, typename OutT>
__global__ void __launch_bounds__(1024) k_coarse_solve(MgCoefs A, const float* __restrict__ P,
                                                       const float* __restrict__ E, const float* __restrict__ Q,
                                                       const BT* __restrict__ b, OutT* __restrict__ out, Lay l,
                                                       Lay ol, float deta, int steps, const SolverScalars* sc) {
  if (sc && sc->done) return;
  extern __shared__ float lds[];
  const int nx = l.nx, nz = l.nz;
  const int ncols = l.nx * l.ny, n = ncols * nz;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  for (int step = 0; step < steps; ++step) {
    const float* cur = lds + (step & 1) * n;
    float* nxt = lds + ((step + 1) & 1) * n;
    auto rd = [&](int ii, int jj, int kk) -> float { return cur[kk + nz * (ii + nx * jj)]; };
#pragma unroll 1
    for (int c = w; c < ncols; c += nw) {  // uniform over the wavefront
      float y[NPL];
      if (step == 0)
        column_step<NPL, true, BT>(A, P, E, Q, b, rd, l, c % nx, c / nx, deta, y);
      else
        column_step<NPL, false, BT>(A, P, E, Q, b, rd, l, c % nx, c / nx, deta, y);
#pragma unroll
      for (int u = 0; u < NPL; ++u) {
        const int k = NPL * lane + u;
        if (k < nz) {
          if (step + 1 < steps)
            nxt[k + nz * c] = y[u];
          else
            out[ol.at32(c % nx, c / nx, k)] = (OutT)y[u];
        }
      }
    }
    __syncthreads();  // the step's writes before the next step's reads
  }
}

Lay lay_of(const MgLevel& L) { return Lay{L.nx, L.ny, L.nz, L.zf}; }

// The layout in which level L reads the coarse correction of level C: its
// own.  (A z-fastest correction read by an x-fastest level's line step costs
// a cache line per lane: 42 us against 27 for the first post-smoothing step
// at 64 x 64 x 128; the coarse level's last smoothing step stores it across
// instead.)
Lay correction_layout(const MgLevel& L, const MgLevel& C) { return Lay{C.nx, C.ny, C.nz, L.zf}; }

bool bf16_storage(const pcf_state* st) { return st->cfg.preconditioner_storage == PCF_STORAGE_BF16; }

// f(W, NPL), the columns and levels per thread of a grid's line steps.  Eight
// levels per thread up to 128 levels, 16 above (a block has at most 1024
// threads).  Four columns per thread (16-byte loads, a quarter of the memory
// instructions) pay where the tiles alone fill the chip: with bf16
// coefficients 120 us against 125 at 256 x 256 x 128, but 30 against 28 at
// 128 x 128 x 128 and 18 against 14 at 48 x 40 x 64, where the threads do.
// The results do not depend on W.
constexpr long long kLineWideCells = 4 << 20;
__host__ __device__ inline bool line_wide(int nx, int ny, int nz) {
  return nx % 4 == 0 && (long long)nx * ny * nz >= kLineWideCells;
}
// STEP (a step that is not from zero, with coefficients CT): four levels per
// thread on a flat grid where eight would leave half a segment or more beyond
// the top, with bf16 coefficients on a wide grid only.  Eight / four levels:
// FP32 166 / 145 us at 512 x 512 x 17, 341 / 309 at 512 x 512 x 41, 64 / 54 at
// 300 x 200 x 25; bf16 202 / 189 at 512 x 512 x 33, but 44 / 46 at 300 x 200 x 25.
__host__ __device__ inline bool line_short(int nx, int ny, int nz, bool bf16) {
  return nz <= 64 && (nz - 1) % 8 < 4 && (!bf16 || line_wide(nx, ny, nz));
}
template <bool STEP, typename CT, class F>
void with_line_shape(int nx, int ny, int nz, F&& f) {
  using std::integral_constant;
  if constexpr (STEP)
    if (line_short(nx, ny, nz, sizeof(CT) == 2)) {
      if (line_wide(nx, ny, nz)) f(integral_constant<int, 4>{}, integral_constant<int, 4>{});
      else if constexpr (sizeof(CT) == 4) f(integral_constant<int, 1>{}, integral_constant<int, 4>{});
      return;
    }
  if (nz > 128)
    f(integral_constant<int, 1>{}, integral_constant<int, 16>{});
  else if (line_wide(nx, ny, nz))
    f(integral_constant<int, 4>{}, integral_constant<int, 8>{});
  else
    f(integral_constant<int, 1>{}, integral_constant<int, 8>{});
}

template <typename CT>
LineArgs<CT> line_args(const MgLevel& L, const float* s, const float* e = nullptr, const MgLevel* C = nullptr) {
  LineArgs<CT> A;
  A.coefs = (const CT*)L.coefs;
  A.factors = L.factors;
  A.s = s;
  A.nx = L.nx;
  A.ny = L.ny;
  A.nz = L.nz;
  A.deta = L.deta;
  A.e = e;
  A.omega = kMgOmega;
  A.sx = L.fx == 2;
  A.sy = L.fy == 2;
  A.cl = C ? (e ? correction_layout(L, *C) : lay_of(*C)) : Lay{1, 1, 1, false};
  return A;
}

// One pseudo-time step of an x-fastest level: out = the line solve of
// s + deta (H s - b), or of deta (0 - b) with FIRST; e (with the coarser
// level C): s is s + omega P e.  out must differ from s.
template <bool FIRST, typename BT, typename OutT>
void line_step(pcf_state* st, const MgLevel& L, const BT* b, const float* s, OutT* out, const SolverScalars* sc,
               const float* e = nullptr, const MgLevel* C = nullptr, SolverScalars* commit = nullptr) {
  ProfScope prof(st, FIRST ? PCF_K_PC_THOMAS : PCF_K_PC_RHS);
  auto go = [&](auto ct, auto pro) {
    constexpr bool PRO = decltype(pro)::value;
    using CT = decltype(ct);
    const LineArgs<CT> A = line_args<CT>(L, s, e, C);
    const dim3 grd(LineTile<float>::count(L.nx, L.ny));
    if (L.nz > kLineMaxNz || (L.nz > 128 && LineTile<float>::count(L.nx, L.ny) <= kTallFewTiles)) {
      with_tall_block<PRO>(L.nx, L.ny, L.nz, [&](auto tb) {
        using TB = decltype(tb);
        const int threads = TB::columns * TB::segments(L.nz);
        hipLaunchKernelGGL((k_line_tall32<TB, FIRST, PRO, CT, BT, OutT>), dim3(grd.x * TB::parts), dim3(threads),
                           (line_lds<float, 1>(threads)), st->stream, A, b, out, L.col, sc, commit);
      });
    } else {
      with_line_shape<!FIRST, CT>(L.nx, L.ny, L.nz, [&](auto w, auto npl) {
        constexpr int W = decltype(w)::value, NPL = decltype(npl)::value;
        const int threads = kTileCols / W * ((L.nz + NPL - 1) / NPL);
        hipLaunchKernelGGL((k_line_step32<W, NPL, FIRST, PRO, CT, BT, OutT>), grd, dim3(threads),
                           (line_lds<float, W>(threads)), st->stream, A, b, out, sc, commit);
      });
    }
  };
  if constexpr (FIRST) {
    go(float{}, std::false_type{});
  } else {
    auto pick = [&](auto ct) {
      if (e) go(ct, std::true_type{});
      else go(ct, std::false_type{});
    };
    if (L.bf16) pick(uint16_t{});
    else pick(float{});
  }
}

// The first pseudo-time step of the finest level with a fused BiCGSTAB step.
void line_fuse(pcf_state* st, const MgLevel& L, const BicgFuse& F, int fuse, float* out) {
  ProfScope prof(st, PCF_K_PC_THOMAS);
  const LineArgs<float> A = line_args<float>(L, nullptr);
  auto go = [&](auto npl) {
    constexpr int NPL = decltype(npl)::value;
    const dim3 grd(LineTile<float>::count(L.nx, L.ny)), blk(kTileCols * ((L.nz + NPL - 1) / NPL));
    const unsigned lds = line_lds<float, 1>((int)blk.x);
    if (fuse == FUSE_P) hipLaunchKernelGGL((k_line_fuse32<NPL, FUSE_P>), grd, blk, lds, st->stream, A, F, out);
    else hipLaunchKernelGGL((k_line_fuse32<NPL, FUSE_S>), grd, blk, lds, st->stream, A, F, out);
  };
  if (L.nz > 128) go(std::integral_constant<int, 16>{});
  else go(std::integral_constant<int, 8>{});
}

// Pack a level's coefficients and factors for the line steps.
template <typename SrcT>
void line_pack(pcf_state* st, const MgLevel& L, const LineCoefs<SrcT>& A) {
  if (L.bf16) launch_line_pack(st->stream, A, (uint16_t*)L.coefs, L.factors, L.nx, L.ny, L.nz);
  else launch_line_pack(st->stream, A, (float*)L.coefs, L.factors, L.nx, L.ny, L.nz);
}

// Level paths.  Coarse levels of at most kCoarseColumnCols columns are stored
// z fastest and smoothed one wavefront per column, larger ones x fastest by
// line steps (48 x 40 x 64: 5 us per step against 11, where a tile per
// workgroup leaves the chip empty; 64 x 64 x 128 keeps line steps).  A finest
// level, always x fastest, is smoothed column by column up to kColumnCols
// columns, 256 levels and kColumnCells cells: lanes along z of an x-fastest
// array touch a cache line each, which a small grid's caches hold (V-cycle by
// column / by line steps: 208 / 238 us at 16 x 16 x 200, 234 / 236 at
// 28 x 28 x 200, 373 / 302 at 32 x 32 x 200, 323 / 293 at 16 x 16 x 300).
// The coarsest level runs all its steps in one workgroup when it has at most
// 16 columns.
constexpr size_t kColumnCols = 1024, kCoarseColumnCols = 2048, kColumnCells = 160000;
constexpr int kScanMaxNz = 512;
constexpr size_t kCoarseLdsFloats = 16384;

size_t columns(const MgLevel& L) { return (size_t)L.nx * L.ny; }
bool column_path(const MgLevel& L) {
  if (L.zf) return L.nz <= kScanMaxNz;
  return columns(L) <= kColumnCols && L.nz <= 256 && columns(L) * L.nz <= kColumnCells;
}

MgCoefs coefs_of(const MgLevel& L) {
  MgCoefs A;
  for (int t = 0; t < T_COUNT; ++t) A.a[t] = L.a[t];
  return A;
}

__global__ void k_round_bf16(MgCoefs A, size_t n) {
  float* a = A.a[blockIdx.y];
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
    const unsigned u = __float_as_uint(a[q]);
    a[q] = __uint_as_float((u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u);  // round to nearest even
  }
}

// The preconditioner's copies of the current operator: the packed
// coefficients and line-solve factors of the levels smoothed by line steps,
// and FP32 arrays of the multigrid's levels.
int prepare_mixed(pcf_state* st) {
  if (st->t32_valid) return PCF_OK;
  int rc = pc_factors(st);
  if (rc) return rc;
  const size_t N = st->g.nv();
  const MgLevel& L0 = st->mg[0];
  if (L0.coefs) {
    LineCoefs<double> A;
    for (int t = 0; t < T_COUNT; ++t) A.a[t] = st->T.a[t];
    A.P = st->pc_P;
    A.E = st->pc_E;
    A.Q = st->pc_Q;
    line_pack(st, L0, A);
  }
  if (L0.a[0]) {
    for (int t = 0; t < T_COUNT; ++t)
      hipLaunchKernelGGL(k_to_f32, dim3(1024), dim3(256), 0, st->stream, st->T.a[t], L0.a[t], N);
    hipLaunchKernelGGL(k_to_f32, dim3(1024), dim3(256), 0, st->stream, st->pc_P, L0.P, N);
    hipLaunchKernelGGL(k_to_f32, dim3(1024), dim3(256), 0, st->stream, st->pc_E, L0.E, N);
    hipLaunchKernelGGL(k_to_f32, dim3(1024), dim3(256), 0, st->stream, st->pc_Q, L0.Q, N);
  }
  // coarse operators and their line-solve factors
  for (size_t l = 1; l < st->mg.size(); ++l) {
    const MgLevel& F = st->mg[l - 1];
    const MgLevel& C = st->mg[l];
    const MgCoefs ca = coefs_of(C);
    const Lay fl = lay_of(F), cl = lay_of(C);
    const dim3 grd(blocks_for(cl.count(), 256)), blk(256);
    auto coarsen = [&](auto ft, auto* const* src) {
      using FT = decltype(ft);
      LineCoefs<FT> fa{};
      for (int t = 0; t < T_COUNT; ++t) fa.a[t] = src[t];
      if (F.fx == 2 && F.fy == 2)
        hipLaunchKernelGGL((k_mg_coarsen<2, 2, FT>), grd, blk, 0, st->stream, fa, ca, fl, cl);
      else if (F.fx == 2)
        hipLaunchKernelGGL((k_mg_coarsen<2, 1, FT>), grd, blk, 0, st->stream, fa, ca, fl, cl);
      else
        hipLaunchKernelGGL((k_mg_coarsen<1, 2, FT>), grd, blk, 0, st->stream, fa, ca, fl, cl);
    };
    if (l == 1) coarsen(double{}, st->T.a);
    else coarsen(float{}, F.a);
    hipLaunchKernelGGL(k_mg_factors, dim3(blocks_for((long long)C.nx * C.ny, 64)), dim3(64), 0, st->stream,
                       C.a[T_AC], C.a[T_AD], C.a[T_AU], C.P, C.E, C.Q, cl, C.deta);
    if (C.coefs) {
      LineCoefs<float> A;
      for (int t = 0; t < T_COUNT; ++t) A.a[t] = C.a[t];
      A.P = C.P;
      A.E = C.E;
      A.Q = C.Q;
      line_pack(st, C, A);
    }
  }
  // bf16 storage covers the levels of more than kColumnCols columns; those
  // smoothed column by column keep the rounded values in FP32 arrays (after
  // the coarser levels have been formed from the unrounded ones)
  if (bf16_storage(st))
    for (size_t l = 1; l < st->mg.size(); ++l) {
      const MgLevel& C = st->mg[l];
      if (C.zf && columns(C) > kColumnCols)
        hipLaunchKernelGGL(k_round_bf16, dim3(64, T_COUNT), dim3(256), 0, st->stream, coefs_of(C), lay_of(C).count());
    }
  PCF_HIP(hipGetLastError());
  st->t32_valid = true;
  return PCF_OK;
}

template <class F>
void with_npl(int nz, F&& f) {
  if (nz <= 64)
    f(std::integral_constant<int, 1>{});
  else if (nz <= 128)
    f(std::integral_constant<int, 2>{});
  else if (nz <= 256)
    f(std::integral_constant<int, 4>{});
  else
    f(std::integral_constant<int, 8>{});
}

// steps smoothing steps on level L.  s: the buffer holding the current
// iterate, null to start from zero; e (with the coarser level C): the coarse
// correction, s += omega P e before the first step.  The last step writes to
// out64 when given (the FP64 result of the finest level); otherwise returns
// the buffer holding the result.
template <typename BT>
float* mg_smooth(pcf_state* st, const MgLevel& L, const BT* b, float* s, const float* e, const MgLevel* C, int steps,
                 double* out64, const Lay& ol, const SolverScalars* sc, const BicgFuse* F = nullptr,
                 int fuse = FUSE_NONE) {
  const bool col = column_path(L);
  const size_t nc = columns(L);
  int step = 0;
  if (!s) {  // first step from zero
    const bool last = steps == 1;
    if (col) {
      ProfScope prof(st, PCF_K_PC_THOMAS);
      with_npl(L.nz, [&](auto npl) {
        constexpr int NPL = decltype(npl)::value;
        const Lay l = lay_of(L);
        if (last && out64)
          hipLaunchKernelGGL((k_col_smooth<NPL, true, false, BT, double>), dim3(blocks_for(nc, 4)), dim3(256), 0,
                             st->stream, coefs_of(L), L.P, L.E, L.Q, b, nullptr, nullptr, 0.0f, 0, 0, l, l, out64, l,
                             L.deta, sc);
        else
          hipLaunchKernelGGL((k_col_smooth<NPL, true, false, BT, float>), dim3(blocks_for(nc, 4)), dim3(256), 0,
                             st->stream, coefs_of(L), L.P, L.E, L.Q, b, nullptr, nullptr, 0.0f, 0, 0, l, l, L.s,
                             last ? ol : l, L.deta, sc);
      });
    } else if (fuse != FUSE_NONE) {
      line_fuse(st, L, *F, fuse, L.s);
    } else {
      if (last && out64)
        line_step<true, BT, double>(st, L, b, nullptr, out64, sc);
      else
        line_step<true, BT, float>(st, L, b, nullptr, L.s, sc);
    }
    s = L.s;
    step = 1;
  }
  for (; step < steps; ++step) {
    const bool last = step == steps - 1;
    if (col) {
      const bool pro = e && step == 0;
      float* dst = s == L.s ? L.rhs : L.s;
      ProfScope prof(st, PCF_K_PC_THOMAS);
      with_npl(L.nz, [&](auto npl) {
        constexpr int NPL = decltype(npl)::value;
        const int sx = L.fx == 2, sy = L.fy == 2;
        const Lay l = lay_of(L), cl = C ? correction_layout(L, *C) : l;
        const dim3 g(blocks_for(nc, 4)), blk(256);
        if (last && out64) {
          if (pro)
            hipLaunchKernelGGL((k_col_smooth<NPL, false, true, BT, double>), g, blk, 0, st->stream, coefs_of(L), L.P,
                               L.E, L.Q, b, s, e, kMgOmega, sx, sy, l, cl, out64, l, L.deta, sc);
          else
            hipLaunchKernelGGL((k_col_smooth<NPL, false, false, BT, double>), g, blk, 0, st->stream, coefs_of(L), L.P,
                               L.E, L.Q, b, s, e, kMgOmega, sx, sy, l, cl, out64, l, L.deta, sc);
        } else {
          if (pro)
            hipLaunchKernelGGL((k_col_smooth<NPL, false, true, BT, float>), g, blk, 0, st->stream, coefs_of(L), L.P,
                               L.E, L.Q, b, s, e, kMgOmega, sx, sy, l, cl, dst, last ? ol : l, L.deta,
                               sc);
          else
            hipLaunchKernelGGL((k_col_smooth<NPL, false, false, BT, float>), g, blk, 0, st->stream, coefs_of(L), L.P,
                               L.E, L.Q, b, s, e, kMgOmega, sx, sy, l, cl, dst, last ? ol : l, L.deta,
                               sc);
        }
      });
      s = dst;
      continue;
    }
    const float* pro = step == 0 ? e : nullptr;
    float* dst = s == L.s ? L.rhs : L.s;
    SolverScalars* commit = fuse == FUSE_P && step == 1 ? F->sc : nullptr;
    if (last && out64)
      line_step<false, BT, double>(st, L, b, s, out64, sc, pro, C, commit);
    else
      line_step<false, BT, float>(st, L, b, s, dst, sc, pro, C, commit);
    s = dst;
  }
  return s;
}

// b_coarse = R (b - A s)
template <typename BT>
void mg_restrict(pcf_state* st, const MgLevel& L, const MgLevel& C, const BT* b, const float* s,
                 const SolverScalars* sc) {
  ProfScope prof(st, PCF_K_PC_RHS);
  if (L.coefs && L.fx == 2 && L.fy == 2) {
    auto go = [&](auto ct) {
      using CT = decltype(ct);
      // 8 levels per thread at any height, as no level waits for another (16:
      // 20 us against 13 at 44 x 44 x 130)
      auto launch = [&](auto w) {
        constexpr int W = decltype(w)::value, NPL = 8, most = (W == 4 ? 512 : 1024) / (kTileCols / W);
        const int segs = (L.nz + NPL - 1) / NPL, parts = (segs + most - 1) / most;
        hipLaunchKernelGGL((k_resid_restrict<W, NPL, BT, CT>), dim3(LineTile<float>::count(L.nx, L.ny), parts),
                           dim3(kTileCols / W * ((segs + parts - 1) / parts)), 0, st->stream,
                           line_args<CT>(L, s, nullptr, &C), b, C.b, sc);
      };
      if (line_wide(L.nx, L.ny, L.nz)) launch(std::integral_constant<int, 4>{});
      else launch(std::integral_constant<int, 1>{});
    };
    if (L.bf16) go(uint16_t{});
    else go(float{});
    return;
  }
  const MgCoefs A = coefs_of(L);
  const Lay fl = lay_of(L), cl = lay_of(C);
  auto go = [&](auto fx, auto fy) {
    constexpr int FX = decltype(fx)::value, FY = decltype(fy)::value;
    if (L.zf)
      hipLaunchKernelGGL((k_resid_restrict_columns<FX, FY, BT>), dim3((unsigned)columns(C) * blocks_for(L.nz, 64)),
                         dim3(64, FX * FY), 0, st->stream, A, b, s, C.b, fl, cl, sc);
    else
      hipLaunchKernelGGL((k_resid_restrict_rows<FX, FY, BT>), dim3(blocks_for((long long)L.nx * C.ny * L.nz, 256)),
                         dim3(256), 0, st->stream, A, b, s, C.b, fl, cl, sc);
  };
  using std::integral_constant;
  if (L.fx == 2 && L.fy == 2) go(integral_constant<int, 2>{}, integral_constant<int, 2>{});
  else if (L.fx == 2) go(integral_constant<int, 2>{}, integral_constant<int, 1>{});
  else go(integral_constant<int, 1>{}, integral_constant<int, 2>{});
}

// The coarsest level: mg_coarse_steps smoothing steps from zero.
template <typename BT>
float* mg_coarsest(pcf_state* st, const MgLevel& L, const BT* b, double* out64, const Lay& ol,
                   const SolverScalars* sc) {
  const size_t nc = columns(L);
  const size_t n = nc * (size_t)L.nz;
  if (nc <= 16 && L.nz <= 256 && 2 * n <= kCoarseLdsFloats) {
    ProfScope prof(st, PCF_K_PC_THOMAS);
    const unsigned lds = (unsigned)(2 * n * sizeof(float));
    const dim3 blk(64 * (unsigned)nc);
    with_npl(L.nz, [&](auto npl) {
      constexpr int NPL = decltype(npl)::value;
      if constexpr (NPL <= 4) {
        if (out64)
          hipLaunchKernelGGL((k_coarse_solve<NPL, BT, double>), dim3(1), blk, lds, st->stream, coefs_of(L), L.P, L.E,
                             L.Q, b, out64, lay_of(L), lay_of(L), L.deta, st->cfg.mg_coarse_steps, sc);
        else
          hipLaunchKernelGGL((k_coarse_solve<NPL, BT, float>), dim3(1), blk, lds, st->stream, coefs_of(L), L.P, L.E,
                             L.Q, b, L.s, lay_of(L), ol, L.deta, st->cfg.mg_coarse_steps, sc);
      }
    });
    return L.s;
  }
  return mg_smooth<BT>(st, L, b, nullptr, nullptr, nullptr, st->cfg.mg_coarse_steps, out64, ol, sc);
}

// One V-cycle on level l for the right-hand side b; the finest level writes
// its result to out64; returns the buffer holding the level's result, in
// layout ol.
template <typename BT>
float* mg_vcycle(pcf_state* st, size_t l, const BT* b, double* out64, const Lay& ol, const SolverScalars* sc,
                 const BicgFuse* F = nullptr, int fuse = FUSE_NONE) {
  const MgLevel& L = st->mg[l];
  if (l + 1 == st->mg.size()) return mg_coarsest<BT>(st, L, b, out64, ol, sc);
  const MgLevel& C = st->mg[l + 1];
  float* s =
      mg_smooth<BT>(st, L, b, nullptr, nullptr, nullptr, st->cfg.mg_smoothing_steps, nullptr, lay_of(L), sc, F, fuse);
  mg_restrict<BT>(st, L, C, b, s, sc);
  const Lay el = correction_layout(L, C);
  const float* e = mg_vcycle<float>(st, l + 1, C.b, nullptr, el, sc);
  return mg_smooth<BT>(st, L, b, s, e, &C, st->cfg.mg_smoothing_steps, out64, ol, sc);
}

}  // namespace

// Whether the solve's first two kernels are line steps of the finest level.
bool fusable_mixed(const pcf_state* st) {
  const MgLevel& L = st->mg[0];
  if (!L.coefs || L.nz > kLineMaxNz) return false;
  if (st->cfg.preconditioner_type == PCF_PC_MULTIGRID) return st->mg.size() > 1 && st->cfg.mg_smoothing_steps >= 2;
  return st->cfg.preconditioner_iterations >= 2;
}

// M^-1 sin -> sout (FP64 in and out, FP32 inside); sout must not alias sin.
int precondition_mixed(pcf_state* st, const double* sin, double* sout, const SolverScalars* sc, const BicgFuse* F,
                       int fuse) {
  int rc = prepare_mixed(st);
  if (rc) return rc;
  if (st->cfg.preconditioner_type == PCF_PC_MULTIGRID) {
    mg_vcycle<double>(st, 0, sin, sout, lay_of(st->mg[0]), sc, F, fuse);
    PCF_HIP(hipGetLastError());
    return PCF_OK;
  }
  const MgLevel& L = st->mg[0];
  const int iters = st->cfg.preconditioner_iterations;
  if (iters == 1) {
    line_step<true, double, double>(st, L, sin, nullptr, sout, sc);
  } else {
    float* cur = L.s;  // FP32 iterate between pseudo-time steps
    if (fuse != FUSE_NONE) line_fuse(st, L, *F, fuse, cur);
    else line_step<true, double, float>(st, L, sin, nullptr, cur, sc);
    for (int it = 2; it <= iters; ++it) {
      float* next = cur == L.s ? L.rhs : L.s;
      SolverScalars* commit = fuse == FUSE_P && it == 2 ? F->sc : nullptr;
      if (it == iters)
        line_step<false, double, double>(st, L, sin, cur, sout, sc, nullptr, nullptr, commit);
      else
        line_step<false, double, float>(st, L, sin, cur, next, sc, nullptr, nullptr, commit);
      cur = next;
    }
  }
  PCF_HIP(hipGetLastError());
  return PCF_OK;
}

int apply_bicgstab_mixed(pcf_state* st, double tolref, double dt, int* niter_out) {
  const pcf_config& n = st->cfg;
  int rc = prepare_mixed(st);
  if (rc) return rc;
  const int slot = st->solve_slot;
  const bool stage = slot >= 0 && slot < 2 && dt > 0.0;
  const bool extrap = n.initial_guess == PCF_GUESS_EXTRAPOLATED;
  const bool use_prev =
      (n.initial_guess == PCF_GUESS_PREVIOUS || n.initial_guess == PCF_GUESS_LEARNED || extrap) && stage;
  const double* prev = use_prev && st->m_prev_valid[slot] ? st->m_prev[slot] : nullptr;
  const double* guess = n.initial_guess == PCF_GUESS_PREVIOUS || extrap ? prev : nullptr;
  const size_t N = st->g.nv();
  if (extrap && prev && st->m_prev2_valid[slot] && st->m_prev_dt[slot] > 0.0) {
    hipLaunchKernelGGL(k_extrapolate, dim3(2048), dim3(256), 0, st->stream, prev, st->m_prev2[slot], st->m_guess, N,
                       dt / st->m_prev_dt[slot]);
    PCF_HIP(hipGetLastError());
    guess = st->m_guess;
  }
  double scale = dt;
  if (n.initial_guess == PCF_GUESS_LEARNED && stage) {
    if ((rc = learned_guess(st, dt, prev, &guess))) return rc;
    scale = 1.0;
  }
  rc = bicgstab_core(st, tolref, true, guess, scale, niter_out);
  if (rc == PCF_E_NOCONV && st->stage_net && st->stage_iterations > 0) {
    // the flexible solve with the learned stage failed: the plain
    // preconditioned BiCGSTAB from zero is the fallback
    const int failed = *niter_out;
    pcf_net* keep = st->stage_net;
    st->stage_net = nullptr;
    rc = bicgstab_core(st, tolref, true, nullptr, 0.0, niter_out);
    st->stage_net = keep;
    st->stage_fallbacks += 1;
    *niter_out += failed;
  }
  if (rc) return rc;
  if (use_prev) {  // keep solution / dt for the same stage of the next step
    if (extrap) {  // and the one before it
      std::swap(st->m_prev[slot], st->m_prev2[slot]);
      st->m_prev2_valid[slot] = st->m_prev_valid[slot];
    }
    hipLaunchKernelGGL(k_scale_copy, dim3(2048), dim3(256), 0, st->stream, st->solution, st->m_prev[slot], N,
                       1.0 / dt);
    PCF_HIP(hipGetLastError());
    st->m_prev_valid[slot] = true;
    st->m_prev_dt[slot] = dt;
  }
  return PCF_OK;
}

// ---------------------------------------------------------------------------
// Ensemble batch: the FP32 line preconditioner over the solves of a batched
// iteration (see the ensemble kernels of poisson.hip).  Each member runs the
// line steps of its single solve (precondition_mixed), with the same segments
// and so the same bits.
// ---------------------------------------------------------------------------
namespace {

__device__ __forceinline__ int ens_member32(const int* start, int count, int b) {
  int lo = 0, hi = count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (start[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// One pseudo-time step of every solve: from the FP64 vector v[in] (FIRST) or
// the member's FP32 iterate `from` (0: cur32, 1: rhs32), to v[out] (OutT
// double) or the other FP32 buffer.  The members' columns may have different
// heights: the segments beyond a column's top are identity maps.
// TALL: columns of more than kLineMaxNz levels, in the blocks of line_step.
template <bool TALL, bool FIRST, typename CT, typename OutT>
__global__ void __launch_bounds__(1024) kEm_line(const EnsTable* __restrict__ E, const EnsList* __restrict__ L, int in,
                                                 int from, int out) {
  const int a = ens_member32(L->line_start, L->count, blockIdx.x);
  const EnsMember& M = E->m[L->member[a]];
  if (M.sc->done) return;
  const int b = blockIdx.x - L->line_start[a];
  LineArgs<CT> A;
  A.coefs = (const CT*)M.coefs32;
  A.factors = M.factors32;
  A.s = from == 0 ? M.cur32 : M.rhs32;
  A.nx = M.nx;
  A.ny = M.ny;
  A.nz = M.nz;
  A.deta = (float)M.deta;
  A.e = nullptr;
  A.omega = 0.0f;
  A.sx = A.sy = 0;
  A.cl = Lay{1, 1, 1, false};
  OutT* dst;
  if constexpr (sizeof(OutT) == 8) dst = M.v[out];
  else dst = FIRST || from == 1 ? M.cur32 : M.rhs32;
  const double* v = M.v[in];
  if constexpr (TALL)
    with_tall_block<false>(M.nx, M.ny, M.nz, [&](auto tb) {
      line_tall32<decltype(tb), FIRST, false, CT, double, OutT>(A, v, dst, M.col32, b);
    });
  else if (!FIRST && line_short(M.nx, M.ny, M.nz, sizeof(CT) == 2))
    line_step32<1, 4, FIRST, false, CT, double, OutT>(A, v, dst, b);
  else if (M.nz > 128)
    line_step32<1, 16, FIRST, false, CT, double, OutT>(A, v, dst, b);
  else
    line_step32<1, 8, FIRST, false, CT, double, OutT>(A, v, dst, b);
}

}  // namespace

// blocks and threads per block of a member's line steps
bool ensemble_line_tall(const pcf_state* st) { return st->g.nz > kLineMaxNz; }
int ensemble_line_blocks(const pcf_state* st) {
  const Geo& g = st->g;
  int blocks = LineTile<float>::count(g.nx, g.ny);
  if (ensemble_line_tall(st))
    with_tall_block<false>(g.nx, g.ny, g.nz, [&](auto tb) { blocks *= decltype(tb)::parts; });
  return blocks;
}
int ensemble_line_threads(const pcf_state* st) {
  const Geo& g = st->g;
  int threads = 0;
  if (ensemble_line_tall(st)) {
    with_tall_block<false>(g.nx, g.ny, g.nz,
                           [&](auto tb) { threads = decltype(tb)::columns * decltype(tb)::segments(g.nz); });
  } else {
    const int npl = line_short(g.nx, g.ny, g.nz, st->mg[0].bf16) ? 4 : g.nz > 128 ? 16 : 8;
    threads = kTileCols * ((g.nz + npl - 1) / npl);
  }
  return threads;
}

// M^-1 v[in] -> v[out] for every solve of the list (precondition_mixed's
// line branch); threads: the largest of the members' blocks
template <bool TALL>
static void precondition_members(hipStream_t s, const EnsTable* dT, const EnsList* dL, const EnsList& L, int threads,
                                 int iters, bool bf16, int in, int out) {
  const dim3 grd(L.line_start[L.count]), blk(threads);
  const unsigned lds = 4 * threads * sizeof(float);
  if (iters == 1) {
    hipLaunchKernelGGL((kEm_line<TALL, true, float, double>), grd, blk, lds, s, dT, dL, in, 0, out);
    return;
  }
  hipLaunchKernelGGL((kEm_line<TALL, true, float, float>), grd, blk, lds, s, dT, dL, in, 0, out);
  int from = 0;
  for (int it = 2; it <= iters; ++it, from ^= 1) {
    if (it == iters && bf16)
      hipLaunchKernelGGL((kEm_line<TALL, false, uint16_t, double>), grd, blk, lds, s, dT, dL, in, from, out);
    else if (it == iters)
      hipLaunchKernelGGL((kEm_line<TALL, false, float, double>), grd, blk, lds, s, dT, dL, in, from, out);
    else if (bf16)
      hipLaunchKernelGGL((kEm_line<TALL, false, uint16_t, float>), grd, blk, lds, s, dT, dL, in, from, out);
    else
      hipLaunchKernelGGL((kEm_line<TALL, false, float, float>), grd, blk, lds, s, dT, dL, in, from, out);
  }
}
void ensemble_precondition_mixed(hipStream_t s, const EnsTable* dT, const EnsList* dL, const EnsList& L, int threads,
                                 bool tall, int iters, bool bf16, int in, int out) {
  if (tall) precondition_members<true>(s, dT, dL, L, threads, iters, bf16, in, out);
  else precondition_members<false>(s, dT, dL, L, threads, iters, bf16, in, out);
}

// Allocation of the mixed-precision buffers (pcf_create, precision MIXED).
int alloc_mixed(pcf_state* st) {
  const size_t N = st->g.nv();
  const bool multigrid = st->cfg.preconditioner_type == PCF_PC_MULTIGRID;
  auto af = [&](float** p) -> int { return device_alloc(st, p, N); };
  // the packed arrays of a level smoothed by line steps; in multigrid, bf16
  // storage covers the levels of more than kColumnCols columns and those too
  // tall to be smoothed column by column
  auto packed = [&](MgLevel& L) -> int {
    L.bf16 = bf16_storage(st) && (!multigrid || columns(L) > kColumnCols || L.nz > kScanMaxNz);
    const size_t n = (size_t)LineTile<float>::count(L.nx, L.ny) * kTileCols * L.nz;
    int rc1 = device_alloc(st, &L.coefs, n * T_COUNT * (L.bf16 ? 2 : 4));
    if (!rc1) rc1 = device_alloc(st, &L.factors, 3 * n);
    if (!rc1 && L.nz > kLineMaxNz) rc1 = device_alloc(st, &L.col, columns(L) * L.nz);
    return rc1;
  };
  int rc;
  double** dl[] = {&st->bzpc, &st->m_prev[0], &st->m_prev[1]};
  for (double** p : dl)
    if ((rc = device_alloc(st, p, N))) return rc;
  if (st->cfg.initial_guess == PCF_GUESS_EXTRAPOLATED) {
    double** el[] = {&st->m_prev2[0], &st->m_prev2[1], &st->m_guess};
    for (double** p : el)
      if ((rc = device_alloc(st, p, N))) return rc;
  }
  // level 0, the only one of the line relaxation
  const Geo& g = st->g;
  MgLevel L0;
  L0.nx = g.nx;
  L0.ny = g.ny;
  L0.nz = g.nz;
  L0.deta = (float)st->deta;
  for (float** p : {&L0.s, &L0.rhs})
    if ((rc = af(p))) return rc;
  if (!multigrid || !column_path(L0))
    if ((rc = packed(L0))) return rc;
  // FP32 arrays of the finest level where the column kernels or the general
  // residual read them; the line steps read the packed ones
  const bool pair = g.nx % 2 == 0 && g.nx >= kMgMinSize && g.ny % 2 == 0 && g.ny >= kMgMinSize;
  if (multigrid && (!L0.coefs || !pair)) {
    for (int t = 0; t < T_COUNT; ++t)
      if ((rc = af(&L0.a[t]))) return rc;
    for (float** p : {&L0.P, &L0.E, &L0.Q})
      if ((rc = af(p))) return rc;
  }
  st->mg.clear();
  st->mg.push_back(L0);
  if (!multigrid) return PCF_OK;
  // the coarse levels' "grid spacings": Galerkin aggregation of fx x fy
  // columns multiplies the x couplings by fy and the y couplings by fx, which
  // sets the pseudo-time step of each level's smoother like the reference's
  // deta = dtau / (2 (1/dx^2 + 1/dy^2)) (apply_preconditioner!.jl:58)
  double cx = 1.0 / (g.dx * g.dx), cy = 1.0 / (g.dy * g.dy);
  for (;;) {
    MgLevel& F = st->mg.back();
    const int fx = (F.nx % 2 == 0 && F.nx >= kMgMinSize) ? 2 : 1;
    const int fy = (F.ny % 2 == 0 && F.ny >= kMgMinSize) ? 2 : 1;
    if (fx == 1 && fy == 1) break;
    F.fx = fx;
    F.fy = fy;
    MgLevel C;
    C.nx = F.nx / fx;
    C.ny = F.ny / fy;
    C.nz = F.nz;
    cx *= fy;
    cy *= fx;
    C.deta = (float)(st->cfg.dtau / (2.0 * (cx + cy)));
    const size_t Nc = (size_t)C.nx * C.ny * C.nz;
    auto ac = [&](float** p) -> int { return device_alloc(st, p, Nc); };
    for (int t = 0; t < T_COUNT; ++t)
      if ((rc = ac(&C.a[t]))) return rc;
    float** v[] = {&C.P, &C.E, &C.Q, &C.b, &C.s, &C.rhs};
    for (float** p : v)
      if ((rc = ac(p))) return rc;
    C.zf = columns(C) <= kCoarseColumnCols && C.nz <= kScanMaxNz;  // smoothed column by column
    if (!C.zf && (rc = packed(C))) return rc;
    st->mg.push_back(C);
  }
  return PCF_OK;
}

}  // namespace pcf
