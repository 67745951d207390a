// Banded overlap of a B-spline rank: Cholesky factor S = U^H U (zpbtrf 'U') and the
// fibre-wise triangular multiplies / solves of core/representation/overlapmatrix.cpp:
//   multiply  x <- U^H (U x)        (ztbmv 'U','N' then 'C', :123-128)
//   solve     x <- U^-1 (U^-H x)    (ztbsv 'U','C' then 'N', :130-135)
//   sqrt      x <- U x | U^H x, x <- U^-1 x | U^-H x (:137-149)
// applied to every 1-D fibre of one rank of a C-ordered tensor (MapToRank3 loops,
// :155-229).
//
// Up to kTileRows rows and not too many fibres (in_tiles) a workgroup holds a tile of whole fibres in
// LDS: the multiplies are banded sums out of LDS and S^-1 x is a product with the dense inverse, which
// the host forms in extended precision (overlap_tile_kernel); U^-1 x and U^-H x are substitutions by
// one lane per fibre with the rows and coefficients staged (overlap_chain_kernel).  Beyond, one thread
// owns one fibre (substitution) or one element (multiply).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "pp_common.h"
#include "pp_internal.h"

namespace pp {

// U(i, j), j - sd <= i <= j, stored at u[j * (sd + 1) + sd + i - j]
__device__ inline double uel(const double* u, int sd, int i, int j) { return u[j * (sd + 1) + sd + i - j]; }

template <int OP, bool CONJ>
__global__ void overlap_fibre_kernel(const double* __restrict__ u, int n, int sd, long long pre, long long post,
                                     double2* __restrict__ data) {
  const long long fib = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (fib >= pre * post) return;
  const long long p = fib / post, q = fib % post;
  double2* x = data + p * n * post + q;
  const long long st = post;
  auto X = [&](int i) -> double2& { return x[i * st]; };
  // x <- U x (ascending, uses x_j for j >= i)
  auto mul_u = [&]() {
    for (int i = 0; i < n; ++i) {
      double2 acc = make_double2(0, 0);
      const int jmax = min(n - 1, i + sd);
      for (int j = i; j <= jmax; ++j) {
        const double a = uel(u, sd, i, j);
        const double2 v = X(j);
        acc.x = fma(a, v.x, acc.x);
        acc.y = fma(a, v.y, acc.y);
      }
      X(i) = acc;
    }
  };
  // x <- U^H x (descending, uses x_j for j <= i); U is real
  auto mul_uh = [&]() {
    for (int i = n - 1; i >= 0; --i) {
      double2 acc = make_double2(0, 0);
      const int jmin = max(0, i - sd);
      for (int j = jmin; j <= i; ++j) {
        const double a = uel(u, sd, j, i);
        const double2 v = X(j);
        acc.x = fma(a, v.x, acc.x);
        acc.y = fma(a, v.y, acc.y);
      }
      X(i) = acc;
    }
  };
  // x <- U^-1 x (back substitution)
  auto solve_u = [&]() {
    for (int i = n - 1; i >= 0; --i) {
      double2 acc = X(i);
      const int jmax = min(n - 1, i + sd);
      for (int j = i + 1; j <= jmax; ++j) {
        const double a = uel(u, sd, i, j);
        const double2 v = X(j);
        acc.x = fma(-a, v.x, acc.x);
        acc.y = fma(-a, v.y, acc.y);
      }
      const double d = uel(u, sd, i, i);
      X(i) = make_double2(acc.x / d, acc.y / d);
    }
  };
  // x <- U^-H x (forward substitution)
  auto solve_uh = [&]() {
    for (int i = 0; i < n; ++i) {
      double2 acc = X(i);
      const int jmin = max(0, i - sd);
      for (int j = jmin; j < i; ++j) {
        const double a = uel(u, sd, j, i);
        const double2 v = X(j);
        acc.x = fma(-a, v.x, acc.x);
        acc.y = fma(-a, v.y, acc.y);
      }
      const double d = uel(u, sd, i, i);
      X(i) = make_double2(acc.x / d, acc.y / d);
    }
  };
  if (OP == PP_OVERLAP_MULTIPLY) { mul_u(); mul_uh(); }
  else if (OP == PP_OVERLAP_SOLVE) { solve_uh(); solve_u(); }
  else if (OP == PP_OVERLAP_SQRT_MULTIPLY) { if (CONJ) mul_uh(); else mul_u(); }
  else { if (CONJ) solve_uh(); else solve_u(); }
}

// The solves with the band width fixed at compile time: each thread keeps a sliding
// window of the last SD unknowns in registers, so every element of the fibre is loaded and
// stored exactly once per pass and the recurrences run out of registers.  The band
// coefficients of row/column i are uniform across the wave (scalar loads).
template <int OP, bool CONJ, int SD>
__global__ __launch_bounds__(128) void overlap_window_kernel(const double* __restrict__ u, int n, long long pre,
                                                            long long post, double2* __restrict__ data) {
  const long long fib = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (fib >= pre * post) return;
  const long long p = fib / post, q = fib % post;
  double2* x = data + p * n * post + q;
  const long long st = post;
  auto U = [&](int i, int j) { return u[j * (SD + 1) + SD + i - j]; };
  // x <- U^-1 x, descending; window holds the SD most recently solved values x_{i+1..i+SD}
  auto solve_u = [&]() {
    double2 w[SD + 1];
#pragma unroll
    for (int d = 0; d <= SD; ++d) w[d] = make_double2(0, 0);
    for (int i = n - 1; i >= 0; --i) {
      double2 acc = x[i * st];
#pragma unroll
      for (int d = 1; d <= SD; ++d) {
        if (i + d < n) {
          const double a = U(i, i + d);
          acc.x = fma(-a, w[d - 1].x, acc.x);
          acc.y = fma(-a, w[d - 1].y, acc.y);
        }
      }
      const double dg = U(i, i);
      acc = make_double2(acc.x / dg, acc.y / dg);
      x[i * st] = acc;
#pragma unroll
      for (int d = SD; d > 0; --d) w[d] = w[d - 1];
      w[0] = acc;
    }
  };
  // x <- U^-H x, ascending; window holds x_{i-1..i-SD}
  auto solve_uh = [&]() {
    double2 w[SD + 1];
#pragma unroll
    for (int d = 0; d <= SD; ++d) w[d] = make_double2(0, 0);
    for (int i = 0; i < n; ++i) {
      double2 acc = x[i * st];
#pragma unroll
      for (int d = 1; d <= SD; ++d) {
        if (i - d >= 0) {
          const double a = U(i - d, i);
          acc.x = fma(-a, w[d - 1].x, acc.x);
          acc.y = fma(-a, w[d - 1].y, acc.y);
        }
      }
      const double dg = U(i, i);
      acc = make_double2(acc.x / dg, acc.y / dg);
      x[i * st] = acc;
#pragma unroll
      for (int d = SD; d > 0; --d) w[d] = w[d - 1];
      w[0] = acc;
    }
  };
  if (OP == PP_OVERLAP_SOLVE) { solve_uh(); solve_u(); }
  else { if (CONJ) solve_uh(); else solve_u(); }
}

// Element-parallel triangular multiplies (no recurrence): one thread per tensor element,
// out-of-place.  mode 0: y = U x, mode 1: y = U^H x along the rank of extent n with
// stride `post`.  Used for the multiply ops, which need no sequential sweep.
template <int SD, int MODE>
__global__ __launch_bounds__(256) void overlap_elem_kernel(const double* __restrict__ u, int n, long long post,
                                                           long long total, const double2* __restrict__ x,
                                                           double2* __restrict__ y) {
  const long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const long long q = idx % post;
  const int i = (int)((idx / post) % n);
  const long long base = idx - (long long)i * post;  // element 0 of this fibre
  double2 acc = make_double2(0, 0);
#pragma unroll
  for (int d = 0; d <= SD; ++d) {
    const int j = MODE == 0 ? i + d : i - d;
    if (j >= 0 && j < n) {
      const double a = MODE == 0 ? u[j * (SD + 1) + SD - d] : u[i * (SD + 1) + SD - d];
      const double2 v = x[base + (long long)j * post];
      acc.x = fma(a, v.x, acc.x);
      acc.y = fma(a, v.y, acc.y);
    }
  }
  (void)q;
  y[idx] = acc;
}

constexpr int kTileRows = 512;

// A tile of FT fibres: where it starts, how many fibres it has, and the strides of a row and of a
// fibre (consecutive fibres are neighbours in memory when the rank is not the last one).
struct FibreTile {
  long long base, row, fibre;
  int cnt;
};
// Workgroup b runs on XCD b % 8: each XCD takes a contiguous range of tiles, so that a cache line that
// two tiles share comes into one L2.
template <int FT>
__device__ inline FibreTile fibre_tile(int n, long long pre, long long post) {
  const unsigned id = blockIdx.x, per_xcd = gridDim.x >> 3;
  const long long tile = (id & 7) * per_xcd + min(id & 7, gridDim.x & 7) + (id >> 3);
  if (post > 1) {
    const long long tiles = (post + FT - 1) / FT, p = tile / tiles, q0 = (tile - p * tiles) * FT;
    return {p * n * post + q0, post, 1, (int)min((long long)FT, post - q0)};
  }
  const long long p0 = tile * FT;
  return {p0 * n, 1, n, (int)min((long long)FT, pre - p0)};
}
// element e of the tile in memory order: consecutive threads on consecutive addresses
template <int FT>
__device__ inline void tile_element(const FibreTile& t, int n, int e, int& i, int& f) {
  if (t.row > 1) {
    i = e / FT;
    f = e % FT;
  } else {
    f = e / n;
    i = e - f * n;
  }
}
template <int FT>
__device__ inline void load_tile(const FibreTile& t, int n, const double2* src, double2* X) {
  for (int e = threadIdx.x; e < n * FT; e += blockDim.x) {
    int i, f;
    tile_element<FT>(t, n, e, i, f);
    X[i * FT + f] = f < t.cnt ? src[t.base + i * t.row + f * t.fibre] : make_double2(0, 0);
  }
}
static long long tile_count(long long pre, long long post, int ft) {
  return post > 1 ? pre * ((post + ft - 1) / ft) : (pre + ft - 1) / ft;
}

// Without Sinv: x <- U x, U^H x or U^H (U x), in the order of the sums above.  With it: x <- S^-1 x,
// S^-1 as rows [j][i] of which lanes i read consecutive values: wave (g, k) sums rows
// 64 g .. 64 g + 63 over the k-th part of j for all FT fibres, and the parts are added in order.
// dst may be src: a workgroup has read its tile before it writes it.  Two substitutions are a chain
// of 2 n dependent rows with one lane per fibre, 50.5 us per rank at 42 x 60 x 60; the product has
// none, 10.9 us.  The two banded passes of U^H U in one launch: 2 x 5.0 us -> 5.6 (42 x 512 x 60: 31 us
// -> 25, 72 with one fibre per workgroup and consecutive tiles on different XCDs).
template <int FT>
__global__ __launch_bounds__(1024) void overlap_tile_kernel(const double* __restrict__ u,
                                                            const double* __restrict__ Sinv, int mul_first,
                                                            int mul_second, int n, int sd, int parts, long long pre,
                                                            long long post, const double2* src, double2* dst) {
  extern __shared__ double2 tile[];
  double2* X = tile;           // [n][FT]
  double2* Y = tile + n * FT;  // [parts][n][FT]
  const FibreTile t = fibre_tile<FT>(n, pre, post);
  load_tile<FT>(t, n, src, X);
  if (!Sinv) {
    double* C = reinterpret_cast<double*>(tile + (mul_second >= 0 ? 2 : 1) * n * FT);
    for (int e = threadIdx.x; e < n * (sd + 1); e += blockDim.x) C[e] = u[e];
    __syncthreads();
    auto band = [&](const double2* in, int mode, int i, int f) {
      double2 acc = make_double2(0, 0);
      const int step = mode == 0 ? 1 : -1;
#pragma unroll 4
      for (int d = 0; d <= sd; ++d) {
        const int j = i + step * d;
        const bool in_range = j >= 0 && j < n;
        const double c = C[(mode == 0 && in_range ? j : i) * (sd + 1) + sd - d];
        const double2 x = in[(in_range ? j : i) * FT + f];
        acc.x = in_range ? fma(c, x.x, acc.x) : acc.x;
        acc.y = in_range ? fma(c, x.y, acc.y) : acc.y;
      }
      return acc;
    };
    const double2* last = X;
    if (mul_second >= 0) {
      for (int e = threadIdx.x; e < n * FT; e += blockDim.x) Y[e] = band(X, mul_first, e / FT, e % FT);
      __syncthreads();
      last = Y;
    }
    const int mode = mul_second >= 0 ? mul_second : mul_first;
    for (int e = threadIdx.x; e < n * FT; e += blockDim.x) {
      int i, f;
      tile_element<FT>(t, n, e, i, f);
      if (f < t.cnt) dst[t.base + i * t.row + f * t.fibre] = band(last, mode, i, f);
    }
    return;
  }
  __syncthreads();
  const int groups = (n + 63) / 64, wave = threadIdx.x >> 6, g = wave % groups, k = wave / groups;
  const int i = 64 * g + (threadIdx.x & 63);
  const int j0 = n * k / parts, j1 = n * (k + 1) / parts;
  if (i < n) {
    double2 acc[FT];
#pragma unroll
    for (int f = 0; f < FT; ++f) acc[f] = make_double2(0, 0);
#pragma unroll 8
    for (int j = j0; j < j1; ++j) {
      const double m = Sinv[(long long)j * n + i];
#pragma unroll
      for (int f = 0; f < FT; ++f) {
        const double2 x = X[j * FT + f];
        acc[f].x = fma(m, x.x, acc[f].x);
        acc[f].y = fma(m, x.y, acc[f].y);
      }
    }
#pragma unroll
    for (int f = 0; f < FT; ++f) Y[(k * n + i) * FT + f] = acc[f];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n * FT; e += blockDim.x) {
    int r, f;
    tile_element<FT>(t, n, e, r, f);
    if (f >= t.cnt) continue;
    double2 s = Y[r * FT + f];
    for (int p = 1; p < parts; ++p) {
      s.x += Y[(p * n + r) * FT + f].x;
      s.y += Y[(p * n + r) * FT + f].y;
    }
    dst[t.base + r * t.row + f * t.fibre] = s;
  }
}

// coefficients of sd superdiagonals (-1: none)
static size_t tile_lds(int n, int ft, int parts, int sd) {
  return (size_t)n * ft * (1 + parts) * sizeof(double2) + (size_t)n * (sd + 1) * sizeof(double);
}

// A launch holds fewer than 2^32 threads.
static bool launchable(long long blocks, int threads) { return blocks * threads < (1LL << 32); }

// false: more tiles than a launch can hold, nothing was done
static bool overlap_tile(const OverlapFactor& ov, int op, bool conj, long long pre, long long post, const double2* src,
                         double2* dst, hipStream_t s) {
  const int n = ov.n, groups = (n + 63) / 64;
  const long long fibres = pre * post;
  const bool solve = op == PP_OVERLAP_SOLVE;
  const int first = op == PP_OVERLAP_MULTIPLY ? 0 : conj ? 1 : 0, second = op == PP_OVERLAP_MULTIPLY ? 1 : -1;
  // few fibres: one per workgroup, so that as many CUs as there are take part; many: tiles whose
  // coefficients are read once for FT fibres.  A solve's are as wide as leaves 64 KB of LDS for the
  // partial sums; a multiply's have four fibres, as narrower ones of a rank that is not the last take
  // less than 64 bytes of a row and a cache line then goes to several XCDs
  const bool few = fibres <= (solve || post == 1 || n <= 160 ? 512 : 128);
  const int ft = few ? 1 : post == 2 ? 2 : solve && n <= 64 ? 8 : n <= 160 || (!solve && post > 1) ? 4 : n <= 320 ? 2 : 1;
  const int parts = solve ? std::max(1, std::min(ft >= 4 ? 4 : 8, 16 / groups)) : second < 0 ? 0 : 1;
  const int threads = solve ? 64 * groups * parts : std::max(256, std::min(1024, (n * ft + 63) / 64 * 64));
  const size_t lds = tile_lds(n, ft, parts, solve ? -1 : ov.sd);
  const long long blocks = tile_count(pre, post, ft);
  if (!launchable(blocks, threads)) return false;
#define PP_TILE(F)                                                                                             \
  case F:                                                                                                      \
    hipLaunchKernelGGL(overlap_tile_kernel<F>, dim3((unsigned)blocks), dim3(threads), lds, s, ov.u.ptr,        \
                       solve ? ov.s_inv.ptr : nullptr, first, second, n, ov.sd, parts, pre, post, src, dst);   \
    break;
  switch (ft) {
    PP_TILE(1) PP_TILE(2) PP_TILE(4) PP_TILE(8)
  }
#undef PP_TILE
  PP_HIP(hipGetLastError());
  return true;
}

// x / c for r = 1 / c rounded: two residual corrections of x r give the rounded quotient (P. Markstein,
// IBM J. Res. Dev. 34 (1990) 111), the bits of the division (0 for x = -0), in five dependent
// operations instead of its ten.  Where a residual could underflow or a value is not finite, and for
// r = 0 (a divisor outside 2^+-100), the division itself, behind a branch of the whole wave: the
// compiler would otherwise compute both.
__device__ inline double divide_by(double x, double c, double r) {
  double q = x * r;
  const bool plain = (fabs(q) > 1e-250 && fabs(q) < 1e250) || x == 0.0;
  q = fma(fma(-q, c, x), r, q);
  q = fma(fma(-q, c, x), r, q);
  if (__ballot(!plain)) q = plain ? q : x / c;
  return q;
}

// x <- U^-1 x (LOWER false, descending rows) or U^-H x (ascending) with the arithmetic of
// overlap_window_kernel, term by term: a Krylov exponential amplifies the rounding of these solves
// from step to step, so another order of the same sums would move its results.  What is left is the
// chain itself, SD dependent FMAs and a division per row.  The tile and the coefficients (zeros
// outside the matrix, then the diagonal and its reciprocal) sit in LDS with the rows in the order
// they are solved, padded to a multiple of SD by rows that are never read back; U is real, so the
// real and imaginary parts are solved by lanes of their own in the first wave.  A lane reads two
// rows ahead and keeps the last SD unknowns in registers that rotate through an unrolled loop.
// 8 fibres of 120 rows: 58 (U^-1) and 31 us (U^-H) with every row loaded from memory in turn,
// 14.4 us here; with the compiler's division and a bounds test per row 26.
template <int SD, int FT, bool LOWER>
__global__ __launch_bounds__(256) void overlap_chain_kernel(const double* __restrict__ u, int n, int rows,
                                                            long long pre, long long post, const double2* src,
                                                            double2* dst) {
  constexpr int W = SD + 2, P = 2 * FT;
  extern __shared__ double2 tile[];
  double2* X = tile;                                              // [rows + 2][FT]
  double* C = reinterpret_cast<double*>(tile + (rows + 2) * FT);  // [rows + 2][W]
  const FibreTile t = fibre_tile<FT>(n, pre, post);
  for (int e = threadIdx.x; e < n * FT; e += blockDim.x) {
    int i, f;
    tile_element<FT>(t, n, e, i, f);
    X[(LOWER ? i : n - 1 - i) * FT + f] = f < t.cnt ? src[t.base + i * t.row + f * t.fibre] : make_double2(0, 0);
  }
  for (int e = n * FT + threadIdx.x; e < (rows + 2) * FT; e += blockDim.x) X[e] = make_double2(0, 0);
  for (int e = threadIdx.x; e < (rows + 2) * (SD + 1); e += blockDim.x) {
    const int r = e / (SD + 1), d = e % (SD + 1) + 1, i = LOWER ? r : n - 1 - r;
    if (d <= SD) {
      double c = 0.0;
      if (r < n && LOWER && i - d >= 0) c = u[i * (SD + 1) + SD - d];
      if (r < n && !LOWER && i + d < n) c = u[(i + d) * (SD + 1) + SD - d];
      C[r * W + d - 1] = c;
    } else {
      const double c = r < n ? u[i * (SD + 1) + SD] : 1.0;
      C[r * W + SD] = c;
      C[r * W + SD + 1] = c > 0x1p-100 && c < 0x1p100 ? 1.0 / c : 0.0;
    }
  }
  __syncthreads();
  if (threadIdx.x < P) {
    double* x = reinterpret_cast<double*>(X) + threadIdx.x;
    double w[SD];  // the unknown of row r sits in w[r % SD]
#pragma unroll
    for (int d = 0; d < SD; ++d) w[d] = 0.0;
    double xa = x[0], xb = x[P], ca[W], cb[W];
#pragma unroll
    for (int d = 0; d < W; ++d) {
      ca[d] = C[d];
      cb[d] = C[W + d];
    }
    for (int r0 = 0; r0 < rows; r0 += SD) {
#pragma unroll
      for (int q = 0; q < SD; ++q) {
        const int r = r0 + q;
        const double xc = x[(r + 2) * P];
        double cc[W];
#pragma unroll
        for (int d = 0; d < W; ++d) cc[d] = C[(r + 2) * W + d];
#pragma unroll
        for (int d = 1; d <= SD; ++d) xa = fma(-ca[d - 1], w[(q + SD - d) % SD], xa);
        w[q] = divide_by(xa, ca[SD], ca[SD + 1]);
        x[r * P] = w[q];
        xa = xb;
        xb = xc;
#pragma unroll
        for (int d = 0; d < W; ++d) {
          ca[d] = cb[d];
          cb[d] = cc[d];
        }
      }
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n * FT; e += blockDim.x) {
    int i, f;
    tile_element<FT>(t, n, e, i, f);
    if (f < t.cnt) dst[t.base + i * t.row + f * t.fibre] = X[(LOWER ? i : n - 1 - i) * FT + f];
  }
}

template <int SD>
static void overlap_chain(const OverlapFactor& ov, bool lower, long long pre, long long post, const double2* src,
                          double2* dst, hipStream_t s) {
  // few fibres: two per workgroup (the chain costs the same for any number; the copies shrink);
  // many: 16, as long as the tile leaves a CU several workgroups (or, if only two of them are filled, all)
  const int n = ov.n, ft = pre * post <= 512 || (post == 2 && n > 128) || n > 160 ? 2 : 16;
  const int rows = (n + SD - 1) / SD * SD;
  const size_t lds = (size_t)(rows + 2) * (ft * sizeof(double2) + (SD + 2) * sizeof(double));
  const long long blocks = tile_count(pre, post, ft);  // (of at most 32768 fibres: in_tiles)
#define PP_CHAIN(F, L)                                                                                             \
  hipLaunchKernelGGL((overlap_chain_kernel<SD, F, L>), dim3((unsigned)blocks), dim3(256), lds, s, ov.u.ptr, n, rows, \
                     pre, post, src, dst)
  if (ft == 2) {
    if (lower) PP_CHAIN(2, true);
    else PP_CHAIN(2, false);
  } else {
    if (lower) PP_CHAIN(16, true);
    else PP_CHAIN(16, false);
  }
#undef PP_CHAIN
  PP_HIP(hipGetLastError());
}

// S^-1 = U^-1 U^-H of the factor, rounded once from extended precision
static void invert_overlap(OverlapFactor& o) {
  const int n = o.n, sd = o.sd;
  auto U = [&](int i, int j) -> long double { return o.u_host[(size_t)j * (sd + 1) + sd + i - j]; };
  std::vector<double> si((size_t)n * n);
  std::vector<long double> x(n);
  for (int c = 0; c < n; ++c) {
    for (int i = 0; i < n; ++i) {  // U^-H e_c
      long double t = i == c ? 1.0L : 0.0L;
      for (int j = std::max(c, i - sd); j < i; ++j) t -= U(j, i) * x[j];
      x[i] = i < c ? 0.0L : t / U(i, i);
    }
    for (int i = n - 1; i >= 0; --i) {  // U^-1 of it
      long double t = x[i];
      for (int j = i + 1; j <= std::min(n - 1, i + sd); ++j) t -= U(i, j) * x[j];
      x[i] = t / U(i, i);
      si[(size_t)c * n + i] = (double)x[i];
    }
  }
  o.s_inv.upload(si.data(), si.size());
  PP_HIP(hipDeviceSynchronize());  // the upload reads a host vector that goes out of scope
}

template <int SD>
static void launch_window(int op, bool conj, const double* u, int n, long long pre, long long post, double2* data,
                          int blocks, int threads, hipStream_t s) {
#define PP_OW(OPC, CJ) \
  hipLaunchKernelGGL((overlap_window_kernel<OPC, CJ, SD>), dim3(blocks), dim3(threads), 0, s, u, n, pre, post, data)
  switch (op) {
    case PP_OVERLAP_SOLVE: PP_OW(PP_OVERLAP_SOLVE, false); break;
    default:
      if (conj) PP_OW(PP_OVERLAP_SQRT_SOLVE, true); else PP_OW(PP_OVERLAP_SQRT_SOLVE, false);
  }
#undef PP_OW
}

// Whether an operation runs on tiles of fibres in LDS; otherwise a thread takes a fibre or an element.
// A substitution by threads is a chain of n rows that takes the same time for any number of fibres
// until they fill the chip; on tiles it is several times shorter, but a workgroup has few chains (or
// multiplies by n^2 values), so its time grows with the fibres.  us by threads / on tiles, six
// superdiagonals:
//   fibres x rows   2520 x 60  20000 x 60  80000 x 60  20000 x 160  2520 x 200  20000 x 200  2520 x 512
//   S^-1              46 / 9     48 / 29     91 / 101    137 / 132    150 / 35    175 / 241    406 / 311
//     (two superdiagonals, 20000 x 160: 108 / 131; 10000 x 320: 272 / 241)
//   U^-1              35 / 11    36 / 15     51 / 45     110 / 57     114 / 45    139 / 181    287 / 134
//   U^-H              22 / 11    21 / 15     48 / 45      61 / 58      69 / 45     78 / 180    173 / 135
// and 20000 x 512 up to five times slower on tiles.
// The multiplies have no chain, and spare a pass over memory on tiles.
static bool in_tiles(const OverlapFactor& ov, int op, bool conj, long long fibres) {
  const int n = ov.n;
  if (n > kTileRows) return false;
  const long long values = fibres * n;
  if (op == PP_OVERLAP_SOLVE)
    return fibres <= 32768 && values <= (n > 320 ? 1300000 : n > 256 || (n <= 160 && ov.sd >= 6) ? 3200000 : 2500000);
  if (op == PP_OVERLAP_SQRT_SOLVE) {
    if (ov.sd < 1 || ov.sd > 8) return false;
    if (n <= 160) return fibres <= 32768 && (!conj || values <= 3200000);
    const long long work = values * (std::max(ov.sd, 6) + 2);
    return conj ? fibres <= 4000 && work <= 8 * 1300000 : work <= 8 * (n > 256 ? 3300000 : 2600000);
  }
  return ov.sd <= 8;
}

void overlap_apply(const OverlapFactor& ov, int op, bool conj, int ndim, const int* extents, int rank,
                   const double2* src, double2* data, hipStream_t s, double2* work) {
  PP_REQUIRE(rank >= 0 && rank < ndim, "rank out of range");
  PP_REQUIRE(extents[rank] == ov.n, "overlap size does not match the rank extent");
  long long pre = 1, post = 1;
  for (int r = 0; r < rank; ++r) pre *= extents[r];
  for (int r = rank + 1; r < ndim; ++r) post *= extents[r];
  const long long fibres = pre * post;
  const int threads = 128;
  const int blocks = ceil_div(fibres, threads);
  if (blocks == 0) return;
  PP_REQUIRE(op >= 0 && op <= 3, "unknown overlap op");
  if (in_tiles(ov, op, conj, fibres)) {
    switch (op == PP_OVERLAP_SQRT_SOLVE ? ov.sd : 0) {
#define PP_CH(K) case K: overlap_chain<K>(ov, conj, pre, post, src, data, s); return;
      PP_CH(1) PP_CH(2) PP_CH(3) PP_CH(4) PP_CH(5) PP_CH(6) PP_CH(7) PP_CH(8)
#undef PP_CH
      default:
        if (overlap_tile(ov, op, conj, pre, post, src, data, s)) return;
    }
  }
  if (ov.sd >= 1 && ov.sd <= 8 && (op == PP_OVERLAP_MULTIPLY || op == PP_OVERLAP_SQRT_MULTIPLY)) {
    const long long total = pre * ov.n * post;
    if (!work && ov.work.count < (size_t)total) ov.work.resize(total);
    const int eb = ceil_div(total, 256);
    double2* w = work ? work : ov.work.ptr;
    auto pass = [&](int mode, const double2* in, double2* out) {
      switch (ov.sd * 2 + mode) {
#define PP_EL(K) \
  case 2 * K: hipLaunchKernelGGL((overlap_elem_kernel<K, 0>), dim3(eb), dim3(256), 0, s, ov.u.ptr, ov.n, post, total, in, out); break; \
  case 2 * K + 1: hipLaunchKernelGGL((overlap_elem_kernel<K, 1>), dim3(eb), dim3(256), 0, s, ov.u.ptr, ov.n, post, total, in, out); break;
        PP_EL(1) PP_EL(2) PP_EL(3) PP_EL(4) PP_EL(5) PP_EL(6) PP_EL(7) PP_EL(8)
#undef PP_EL
      }
    };
    if (op == PP_OVERLAP_MULTIPLY) {
      pass(0, src, w);      // U x
      pass(1, w, data);     // U^H (U x)
    } else if (src != data) {
      pass(conj ? 1 : 0, src, data);
    } else {
      pass(conj ? 1 : 0, data, w);
      PP_HIP(hipMemcpyAsync(data, w, total * sizeof(double2), hipMemcpyDeviceToDevice, s));
    }
    PP_HIP(hipGetLastError());
    return;
  }
  if (src != data) vec_copy(fibres * ov.n, src, data, s);
  if (ov.sd >= 1 && ov.sd <= 8) {
    switch (ov.sd) {
#define PP_SD(K) case K: launch_window<K>(op, conj, ov.u.ptr, ov.n, pre, post, data, blocks, threads, s); break;
      PP_SD(1) PP_SD(2) PP_SD(3) PP_SD(4) PP_SD(5) PP_SD(6) PP_SD(7) PP_SD(8)
#undef PP_SD
    }
    PP_HIP(hipGetLastError());
    return;
  }
#define PP_OV_LAUNCH(OPC, CJ) \
  hipLaunchKernelGGL((overlap_fibre_kernel<OPC, CJ>), dim3(blocks), dim3(threads), 0, s, ov.u.ptr, ov.n, ov.sd, pre, post, data)
  switch (op) {
    case PP_OVERLAP_MULTIPLY: PP_OV_LAUNCH(PP_OVERLAP_MULTIPLY, false); break;
    case PP_OVERLAP_SOLVE: PP_OV_LAUNCH(PP_OVERLAP_SOLVE, false); break;
    case PP_OVERLAP_SQRT_MULTIPLY:
      if (conj) PP_OV_LAUNCH(PP_OVERLAP_SQRT_MULTIPLY, true); else PP_OV_LAUNCH(PP_OVERLAP_SQRT_MULTIPLY, false);
      break;
    case PP_OVERLAP_SQRT_SOLVE:
      if (conj) PP_OV_LAUNCH(PP_OVERLAP_SQRT_SOLVE, true); else PP_OV_LAUNCH(PP_OVERLAP_SQRT_SOLVE, false);
      break;
    default: throw Error(PP_ERR_INVALID, "unknown overlap op");
  }
#undef PP_OV_LAUNCH
  PP_HIP(hipGetLastError());
}

// Upper banded Cholesky S = U^T U of a real symmetric positive definite band matrix
// (the arithmetic of zpbtrf('U') for a real matrix).
void band_cholesky_upper_host(int n, int sd, const double* s, std::vector<double>& u) {
  const int ld = sd + 1;
  u.assign(s, s + (size_t)n * ld);
  auto U = [&](int i, int j) -> double& { return u[(size_t)j * ld + sd + i - j]; };
  for (int j = 0; j < n; ++j) {
    const int i0 = std::max(0, j - sd);
    for (int i = i0; i <= j; ++i) {
      double sum = U(i, j);
      const int k0 = std::max(i0, std::max(0, i - sd));
      for (int k = k0; k < i; ++k) sum -= U(k, i) * U(k, j);
      if (i < j) {
        U(i, j) = sum / U(i, i);
      } else {
        if (!(sum > 0.0)) throw Error(PP_ERR_INVALID, "overlap matrix is not positive definite");
        U(j, j) = std::sqrt(sum);
      }
    }
  }
}

}  // namespace pp

using namespace pp;

extern "C" int pp_overlap_create(int n, int superdiagonals, const double* s_upper, pp_overlap** out) {
  return guarded([&] {
    PP_REQUIRE(out && s_upper && n > 0 && superdiagonals >= 0 && superdiagonals < n, "invalid overlap arguments");
    auto* o = new pp_overlap();
    try {
      o->f.n = n;
      o->f.sd = superdiagonals;
      band_cholesky_upper_host(n, superdiagonals, s_upper, o->f.u_host);
      o->f.u.upload(o->f.u_host.data(), o->f.u_host.size());
      if (n <= kTileRows) {
        invert_overlap(o->f);
        // 102 KB at 512 rows of 8 superdiagonals
        PP_HIP(hipFuncSetAttribute((const void*)overlap_tile_kernel<4>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)tile_lds(kTileRows, 4, 1, 8)));
      }
      PP_HIP(hipDeviceSynchronize());
    } catch (...) {
      delete o;
      throw;
    }
    *out = o;
  });
}

extern "C" int pp_overlap_get_factor(const pp_overlap* ov, double* u_upper) {
  return guarded([&] {
    PP_REQUIRE(ov && u_upper, "NULL argument");
    std::copy(ov->f.u_host.begin(), ov->f.u_host.end(), u_upper);
  });
}

extern "C" int pp_overlap_destroy(pp_overlap* ov) {
  return guarded([&] { delete ov; });
}

extern "C" int pp_overlap_apply(const pp_overlap* ov, int op, int conj, int ndim, const int* extents, int rank,
                                pp_cplx* data, pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(ov && extents && data, "NULL argument");
    double2* d = reinterpret_cast<double2*>(data);
    overlap_apply(ov->f, op, conj != 0, ndim, extents, rank, d, d, (hipStream_t)stream);
  });
}
