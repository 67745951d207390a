// Block-diagonal ("radial") preconditioner of the Cayley step for rank-3 (two-electron)
// wavefunctions: for every angular channel c an exact solve of
//   M_c = scaling_s (S1 x S2) + scaling_h P_c        (n1*n2 x n1*n2)
// where P_c is the angular-diagonal part of H (RadialTwoElectronPreconditioner.Setup,
// examples/tensor/helium_stabilization/preconditioner.py:113-146; the SuperLU variant,
// :156-198, solves the same systems exactly).
//
// M_c is block banded: n2 x n2 blocks (I, J) with |I - J| <= b (b = B-spline order - 1).
//
// Symmetric M_c (real symmetric S and P: every Hamiltonian of this library) of which some multiple has a
// definite Hermitian part (S x S + i dt/2 P_c; H - sigma S for sigma below the spectrum), b n2 <= 512: b
// block rows together form a superblock s of m = b n2 unknowns, and M_c is block tridiagonal in them with
// the sparse couplings A_s,s+1 (S and P entries).  Superblocks are eliminated from both ends towards
// the middle one; with the pivot blocks D_s = A_ss - A_s,s-+1 D_s-+1^-1 A_s-+1,s inverted on the host
//   w_s = D_s^-1 (b_s - A_s,s-+1 w_s-+1)      from the ends inwards (two chains at once)
//   x_mid = D_mid^-1 (b_mid - A w of both neighbours)
//   x_s = w_s - D_s^-1 (A_s,s+-1 x_s+-1)      from the middle outwards
// D_s^-1 is symmetric, so only its upper triangle is read: 0.44 GB per sweep at helium's 42 channels
// (10 superblocks of 360), against 0.87 GB of L' or U' in the general form below, by two workgroups
// per channel instead of one, in 10 steps instead of 60.  See pc_sym_kernel for the figures.
//
// Otherwise the host factors it once per channel by a right-looking block LU without pivoting, and stores for each block row I
//   L_II^-1,  L'_IJ = L_II^-1 L_IJ (J = I-b..I-1),  U_II^-1,  U'_IJ = U_II^-1 U_IJ.
// The device solve is then
//   c_I = L_II^-1 b_I        (all I in parallel)
//   y_I = c_I - sum_J L'_IJ y_J   (sequential over I, one workgroup per channel, LDS resident)
//   d_I = U_II^-1 y_I        (all I in parallel)
//   x_I = d_I - sum_J U'_IJ x_J   (sequential, descending I)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <complex>
#include <limits>
#include <string>
#include <thread>
#include <utility>
#include <vector>

#include "pp_common.h"
#include "pp_internal.h"
#include "pp_krylov.h"

namespace pp {

using cd = std::complex<double>;

namespace {

// dense n x n row-major helpers
void lu_nopivot(int n, cd* a) {
  for (int k = 0; k < n; ++k) {
    const cd piv = a[k * n + k];
    if (piv == cd(0)) throw Error(PP_ERR_INVALID, "zero pivot in preconditioner block LU");
    for (int i = k + 1; i < n; ++i) {
      cd l = a[i * n + k] / piv;
      a[i * n + k] = l;
      for (int j = k + 1; j < n; ++j) a[i * n + j] -= l * a[k * n + j];
    }
  }
}

// X U = A, U upper (from a packed LU), in place on A
void right_upper_solve(int n, const cd* lu, cd* a) {
  for (int r = 0; r < n; ++r) {
    cd* row = a + (size_t)r * n;
    for (int j = 0; j < n; ++j) {
      cd s = row[j];
      for (int k = 0; k < j; ++k) s -= row[k] * lu[k * n + j];
      row[j] = s / lu[j * n + j];
    }
  }
}

// L X = A, L unit lower (from a packed LU), in place on A
void left_unit_lower_solve(int n, const cd* lu, cd* a) {
  for (int i = 0; i < n; ++i)
    for (int k = 0; k < i; ++k) {
      const cd l = lu[i * n + k];
      if (l == cd(0)) continue;
      for (int j = 0; j < n; ++j) a[i * n + j] -= l * a[k * n + j];
    }
}

// C -= A B
void gemm_sub(int n, const cd* A, const cd* B, cd* C) {
  for (int i = 0; i < n; ++i)
    for (int k = 0; k < n; ++k) {
      const cd a = A[i * n + k];
      if (a == cd(0)) continue;
      const cd* b = B + (size_t)k * n;
      cd* c = C + (size_t)i * n;
      for (int j = 0; j < n; ++j) c[j] -= a * b[j];
    }
}

// C = A B
void gemm(int n, const cd* A, const cd* B, cd* C) {
  std::fill(C, C + (size_t)n * n, cd(0));
  for (int i = 0; i < n; ++i)
    for (int k = 0; k < n; ++k) {
      const cd a = A[i * n + k];
      if (a == cd(0)) continue;
      const cd* b = B + (size_t)k * n;
      cd* c = C + (size_t)i * n;
      for (int j = 0; j < n; ++j) c[j] += a * b[j];
    }
}

void unit_lower_inverse(int n, const cd* lu, cd* out) {
  std::fill(out, out + (size_t)n * n, cd(0));
  for (int i = 0; i < n; ++i) out[i * n + i] = 1;
  left_unit_lower_solve(n, lu, out);
}

void upper_inverse(int n, const cd* lu, cd* out) {
  // solve U X = I by back substitution, column by column
  std::fill(out, out + (size_t)n * n, cd(0));
  for (int c = 0; c < n; ++c) {
    for (int i = n - 1; i >= 0; --i) {
      cd s = (i == c) ? cd(1) : cd(0);
      for (int k = i + 1; k < n; ++k) s -= lu[i * n + k] * out[k * n + c];
      out[i * n + c] = s / lu[i * n + i];
    }
  }
}

struct HostFactors {
  std::vector<cd> linv, lp, uinv, up;
};

}  // namespace

static void factor_channel(int c, int n1, int n2, int b, const double* s1, const double* s2, const cd* pdata,
                           int p1, const std::vector<int>& pos1, int p2, const std::vector<int>& pos2, cd sh,
                           cd ss, HostFactors& F) {
  const size_t bs = (size_t)n2 * n2;
  const int nb = 2 * b + 1;
  std::vector<cd> A((size_t)n1 * nb * bs, cd(0));
  auto blk = [&](int I, int J) -> cd* { return A.data() + ((size_t)I * nb + (J - I + b)) * bs; };
  const cd* pc = pdata + (size_t)c * p1 * p2;
  for (int I = 0; I < n1; ++I)
    for (int J = std::max(0, I - b); J <= std::min(n1 - 1, I + b); ++J) {
      cd* a = blk(I, J);
      const double sIJ = s1[(size_t)I * n1 + J];
      const int q1 = pos1[(size_t)I * n1 + J];
      for (int i = 0; i < n2; ++i)
        for (int j = std::max(0, i - b); j <= std::min(n2 - 1, i + b); ++j) {
          cd v = ss * (sIJ * s2[(size_t)i * n2 + j]);
          const int q2 = pos2[(size_t)i * n2 + j];
          if (q1 >= 0 && q2 >= 0) v += sh * pc[(size_t)q1 * p2 + q2];
          a[i * n2 + j] = v;
        }
    }
  // right-looking block LU
  for (int K = 0; K < n1; ++K) {
    cd* akk = blk(K, K);
    lu_nopivot(n2, akk);
    const int hi = std::min(n1 - 1, K + b);
    for (int I = K + 1; I <= hi; ++I) right_upper_solve(n2, akk, blk(I, K));
    for (int J = K + 1; J <= hi; ++J) left_unit_lower_solve(n2, akk, blk(K, J));
    for (int I = K + 1; I <= hi; ++I)
      for (int J = K + 1; J <= hi; ++J) gemm_sub(n2, blk(I, K), blk(K, J), blk(I, J));
  }
  // derived blocks
  std::vector<cd> tmp(bs);
  for (int I = 0; I < n1; ++I) {
    cd* li = F.linv.data() + ((size_t)c * n1 + I) * bs;
    cd* ui = F.uinv.data() + ((size_t)c * n1 + I) * bs;
    unit_lower_inverse(n2, blk(I, I), li);
    upper_inverse(n2, blk(I, I), ui);
    for (int q = 0; q < b; ++q) {
      const int J = I - b + q;
      cd* dst = F.lp.data() + ((size_t)c * n1 + I) * b * bs;  // [row][q*n2 + j]
      if (J >= 0) gemm(n2, li, blk(I, J), tmp.data());
      else std::fill(tmp.begin(), tmp.end(), cd(0));
      for (int i = 0; i < n2; ++i)
        for (int j = 0; j < n2; ++j) dst[(size_t)i * b * n2 + q * n2 + j] = tmp[i * n2 + j];
    }
    for (int q = 0; q < b; ++q) {
      const int J = I + 1 + q;
      cd* dst = F.up.data() + ((size_t)c * n1 + I) * b * bs;
      if (J < n1) gemm(n2, ui, blk(I, J), tmp.data());
      else std::fill(tmp.begin(), tmp.end(), cd(0));
      for (int i = 0; i < n2; ++i)
        for (int j = 0; j < n2; ++j) dst[(size_t)i * b * n2 + q * n2 + j] = tmp[i * n2 + j];
    }
  }
}

// ------------------------------------------------------------------------------------
// host factorisation of the symmetric form
// ------------------------------------------------------------------------------------
// An n x n complex block as separate real and imaginary arrays (the products vectorise).
struct SplitBlock {
  std::vector<double> re, im;
  explicit SplitBlock(size_t n = 0) : re(n, 0.0), im(n, 0.0) {}
};

// C -= A B (n x n, row-major); AT: A is used transposed, BT: B transposed first into scratch
static void split_gemm_sub(int n, const SplitBlock& A, bool at, const SplitBlock& B, bool bt, SplitBlock& C,
                           SplitBlock& scratch) {
  const SplitBlock* Bp = &B;
  if (bt) {
    for (int i = 0; i < n; ++i)
      for (int j = 0; j < n; ++j) {
        scratch.re[(size_t)i * n + j] = B.re[(size_t)j * n + i];
        scratch.im[(size_t)i * n + j] = B.im[(size_t)j * n + i];
      }
    Bp = &scratch;
  }
  for (int i = 0; i < n; ++i) {
    double* __restrict__ cr = C.re.data() + (size_t)i * n;
    double* __restrict__ ci = C.im.data() + (size_t)i * n;
    for (int k = 0; k < n; ++k) {
      const size_t e = at ? (size_t)k * n + i : (size_t)i * n + k;
      const double ar = A.re[e], ai = A.im[e];
      const double* __restrict__ br = Bp->re.data() + (size_t)k * n;
      const double* __restrict__ bi = Bp->im.data() + (size_t)k * n;
      for (int j = 0; j < n; ++j) {
        cr[j] -= ar * br[j] - ai * bi[j];
        ci[j] -= ar * bi[j] + ai * br[j];
      }
    }
  }
}

// The directions of an elimination's pivots in the complex plane, relative to the first diagonal entry.
// Without pivoting the elimination is stable where they stay well within a half plane: where some multiple of M
// has a definite Hermitian part, so has every Schur complement.  Otherwise (sigma inside the spectrum) the
// superblocks' explicit inverses lose more digits than the block LU: 20 x 20 with band 5, random symmetric
// P + 0.3 S: error 1.5e-8, with the block LU 4.9e-11 (S + 0.3i P: 6.0e-16 and 5.4e-16).
struct PivotFan {
  cd ref;
  double lo = 0.0, hi = 0.0;
  static constexpr double kWidest = 2.1;  // 120 degrees; a Crank-Nicolson step's span just over 90
  bool add(cd piv) {  // false: zero, not a number, or too far from the others
    const double a = std::arg(piv * std::conj(ref));
    lo = std::min(lo, a);
    hi = std::max(hi, a);
    return piv != cd(0) && std::isfinite(a) && hi - lo <= kWidest;
  }
};

// A <- A^-1 (n x n), Gauss-Jordan without pivoting; false as soon as a pivot does not fit the others
static bool split_invert(int n, SplitBlock& A, PivotFan& fan) {
  for (int k = 0; k < n; ++k) {
    double* kr = A.re.data() + (size_t)k * n;
    double* ki = A.im.data() + (size_t)k * n;
    const cd piv(kr[k], ki[k]);
    if (!fan.add(piv)) return false;
    const cd inv = 1.0 / piv;
    kr[k] = 1.0;
    ki[k] = 0.0;
    for (int j = 0; j < n; ++j) {
      const cd t = cd(kr[j], ki[j]) * inv;
      kr[j] = t.real();
      ki[j] = t.imag();
    }
    for (int i = 0; i < n; ++i) {
      if (i == k) continue;
      double* __restrict__ ir = A.re.data() + (size_t)i * n;
      double* __restrict__ ii = A.im.data() + (size_t)i * n;
      const double fr = ir[k], fi = ii[k];
      ir[k] = ii[k] = 0.0;
      for (int j = 0; j < n; ++j) {
        ir[j] -= fr * kr[j] - fi * ki[j];
        ii[j] -= fr * ki[j] + fi * kr[j];
      }
    }
  }
  return true;
}

// The entries of channel c's M_c, upper triangle in the radial indices.
struct SymMatrix {
  int n1, n2, b, p2;
  const double *s1, *s2;
  const cd* p;
  const int *pos1, *pos2;
  cd sh, ss;
  double pval(int I, int J, int i, int j) const {
    const int q1 = pos1[(size_t)I * n1 + J], q2 = pos2[(size_t)i * n2 + j];
    return q1 >= 0 && q2 >= 0 ? p[(size_t)q1 * p2 + q2].real() : 0.0;
  }
  cd operator()(int I, int J, int i, int j) const {
    return ss * (s1[(size_t)I * n1 + J] * s2[(size_t)i * n2 + j]) + sh * pval(I, J, i, j);
  }
};

// Whether P_c is real and M_c symmetric to rounding: the potentials are sums of products whose order
// differs between (I, J) and (J, I), so entries may differ in their last bits; measured against the
// geometric mean of the two diagonal entries, as a perturbation of a definite matrix is.
static bool is_symmetric(const SymMatrix& M, int p1) {
  for (size_t k = 0; k < (size_t)p1 * M.p2; ++k)
    if (M.p[k].imag() != 0.0) return false;
  const double tol = 256 * std::numeric_limits<double>::epsilon();
  for (int I = 0; I < M.n1; ++I)
    for (int J = I; J <= std::min(M.n1 - 1, I + M.b); ++J)
      for (int i = 0; i < M.n2; ++i)
        for (int j = std::max(0, i - M.b); j <= std::min(M.n2 - 1, i + M.b); ++j) {
          const cd u = M(I, J, i, j), l = M(J, I, j, i);
          if (u == l) continue;
          const double scale = std::sqrt(std::abs(M(I, I, i, i)) * std::abs(M(J, J, j, j)));
          if (!(std::abs(u - l) <= tol * scale)) return false;
        }
  return true;
}

// Inverse pivot blocks of one channel into dinv [ns][m][m] (upper triangle, halved diagonal); false, with
// dinv unfinished, where the pivots spread too far.
static bool factor_symmetric(const SymMatrix& M, int ns, int mid, cd* dinv) {
  const int n2 = M.n2, b = M.b, m = b * n2;
  const size_t bs = (size_t)n2 * n2;
  auto rows = [&](int s) { return std::min(b, M.n1 - s * b); };
  // M is given in both triangles to rounding; the upper one is used for both
  auto entry = [&](int I, int J, int i, int j) {
    return I < J || (I == J && i <= j) ? M(I, J, i, j) : M(J, I, j, i);
  };
  std::vector<SplitBlock> D, W, Dl, Dr;  // blocks (q, q') of a pivot block, its inverse, the chains' last inverses
  SplitBlock scratch(bs), pivot(bs);
  std::vector<SplitBlock> panel(b, SplitBlock(bs));
  PivotFan fan{M(0, 0, 0, 0)};
  // D -= A_s,f Dinv_f A_f,s with the sparse couplings A
  auto subtract = [&](int s, int f, const std::vector<SplitBlock>& inv) {
    const int rs = rows(s), rf = rows(f);
    const int lds = rf * n2, cols = rs * n2;
    std::vector<double> tr((size_t)lds * cols, 0.0), ti((size_t)lds * cols, 0.0);  // T = Dinv_f A_f,s
    for (int qs = 0; qs < rs; ++qs)
      for (int qf = 0; qf < rf; ++qf) {
        const int I = f * b + qf, J = s * b + qs;
        if (std::abs(I - J) > b) continue;
        for (int i = 0; i < n2; ++i)
          for (int j = std::max(0, i - b); j <= std::min(n2 - 1, i + b); ++j) {
            const cd a = entry(I, J, i, j);  // row (qf, i) of f, column (qs, j) of s
            for (int q = 0; q < rf; ++q) {
              const SplitBlock& B = inv[q * b + qf];
              for (int r = 0; r < n2; ++r) {
                const double xr = B.re[(size_t)r * n2 + i], xi = B.im[(size_t)r * n2 + i];
                const size_t e = (size_t)(qs * n2 + j) * lds + q * n2 + r;  // T stored by columns
                tr[e] += xr * a.real() - xi * a.imag();
                ti[e] += xr * a.imag() + xi * a.real();
              }
            }
          }
      }
    for (int qs = 0; qs < rs; ++qs)
      for (int qf = 0; qf < rf; ++qf) {
        const int I = s * b + qs, J = f * b + qf;
        if (std::abs(I - J) > b) continue;
        for (int i = 0; i < n2; ++i)
          for (int j = std::max(0, i - b); j <= std::min(n2 - 1, i + b); ++j) {
            const cd a = entry(I, J, i, j);  // row (qs, i) of s, column (qf, j) of f
            for (int q = qs; q < rs; ++q) {  // upper blocks only
              SplitBlock& B = D[qs * b + q];
              for (int r = 0; r < n2; ++r) {
                const size_t e = (size_t)(q * n2 + r) * lds + qf * n2 + j;
                B.re[(size_t)i * n2 + r] -= a.real() * tr[e] - a.imag() * ti[e];
                B.im[(size_t)i * n2 + r] -= a.real() * ti[e] + a.imag() * tr[e];
              }
            }
          }
      }
  };
  // D (upper blocks) <- D^-1 (all blocks), sweeping one block row after the other: D becomes -D^-1
  auto invert = [&](int rs) {  // false: see split_invert
    for (int k = 0; k < rs; ++k) {
      pivot = D[k * b + k];
      // the pivot block is symmetric to rounding: use its upper triangle
      for (int i = 0; i < n2; ++i)
        for (int j = 0; j < i; ++j) {
          pivot.re[(size_t)i * n2 + j] = pivot.re[(size_t)j * n2 + i];
          pivot.im[(size_t)i * n2 + j] = pivot.im[(size_t)j * n2 + i];
        }
      if (!split_invert(n2, pivot, fan)) return false;
      for (int i = 0; i < rs; ++i) {  // panel_i = -D_ik pivot^-1
        if (i == k) continue;
        std::fill(panel[i].re.begin(), panel[i].re.end(), 0.0);
        std::fill(panel[i].im.begin(), panel[i].im.end(), 0.0);
        const bool below = i > k;  // D_ik = D_ki^T
        split_gemm_sub(n2, below ? D[k * b + i] : D[i * b + k], below, pivot, false, panel[i], scratch);
      }
      for (int i = 0; i < rs; ++i)
        for (int j = i; j < rs; ++j) {
          if (i == k || j == k) continue;
          // D_ij -= D_ik pivot^-1 D_kj = -panel_i D_kj: the negated product through a negated panel
          SplitBlock& P = panel[i];
          for (auto& z : P.re) z = -z;
          for (auto& z : P.im) z = -z;
          if (j > k) split_gemm_sub(n2, P, false, D[k * b + j], false, D[i * b + j], scratch);
          else split_gemm_sub(n2, P, false, D[j * b + k], true, D[i * b + j], scratch);
          for (auto& z : P.re) z = -z;
          for (auto& z : P.im) z = -z;
        }
      for (int i = 0; i < rs; ++i) {
        if (i == k) continue;
        // swept: D_ik <- D_ik pivot^-1 = -panel_i (stored in the upper block, transposed below)
        SplitBlock& B = i < k ? D[i * b + k] : D[k * b + i];
        for (int r = 0; r < n2; ++r)
          for (int q = 0; q < n2; ++q) {
            const size_t e = i < k ? (size_t)r * n2 + q : (size_t)q * n2 + r;
            B.re[e] = -panel[i].re[(size_t)r * n2 + q];
            B.im[e] = -panel[i].im[(size_t)r * n2 + q];
          }
      }
      D[k * b + k] = pivot;
      for (auto& z : D[k * b + k].re) z = -z;
      for (auto& z : D[k * b + k].im) z = -z;
    }
    for (int i = 0; i < rs; ++i)
      for (int j = i; j < rs; ++j) {
        SplitBlock& B = D[i * b + j];
        for (auto& z : B.re) z = -z;
        for (auto& z : B.im) z = -z;
        if (j == i) continue;
        SplitBlock& T = D[j * b + i];
        for (int r = 0; r < n2; ++r)
          for (int q = 0; q < n2; ++q) {
            T.re[(size_t)q * n2 + r] = B.re[(size_t)r * n2 + q];
            T.im[(size_t)q * n2 + r] = B.im[(size_t)r * n2 + q];
          }
      }
    return true;
  };
  auto pivot_block = [&](int s) {
    const int rs = rows(s);
    D.assign((size_t)b * b, SplitBlock(bs));
    for (int q = 0; q < rs; ++q)
      for (int qq = q; qq < rs; ++qq) {
        SplitBlock& B = D[q * b + qq];
        for (int i = 0; i < n2; ++i)
          for (int j = std::max(0, i - b); j <= std::min(n2 - 1, i + b); ++j) {
            const cd a = entry(s * b + q, s * b + qq, i, j);
            B.re[(size_t)i * n2 + j] = a.real();
            B.im[(size_t)i * n2 + j] = a.imag();
          }
      }
  };
  auto store = [&](int s) {
    const int rs = rows(s);
    cd* out = dinv + (size_t)s * m * m;
    for (int q = 0; q < rs; ++q)
      for (int qq = q; qq < rs; ++qq) {
        const SplitBlock& B = D[q * b + qq];
        for (int i = 0; i < n2; ++i)
          for (int j = q == qq ? i : 0; j < n2; ++j) {
            const cd z(B.re[(size_t)i * n2 + j], B.im[(size_t)i * n2 + j]);
            out[(size_t)(q * n2 + i) * m + qq * n2 + j] = q == qq && i == j ? 0.5 * z : z;
          }
      }
  };
  for (int s = 0; s < mid; ++s) {
    pivot_block(s);
    if (s > 0) subtract(s, s - 1, Dl);
    if (!invert(rows(s))) return false;
    store(s);
    Dl = D;
  }
  for (int s = ns - 1; s > mid; --s) {
    pivot_block(s);
    if (s < ns - 1) subtract(s, s + 1, Dr);
    if (!invert(rows(s))) return false;
    store(s);
    Dr = D;
  }
  pivot_block(mid);
  if (mid > 0) subtract(mid, mid - 1, Dl);
  if (mid < ns - 1) subtract(mid, mid + 1, Dr);
  if (!invert(rows(mid))) return false;
  store(mid);
  return true;
}

// out_I = B_I x_I for all blocks I of all channels; 8 threads per row
__global__ __launch_bounds__(512) void pc_diag_kernel(const double2* __restrict__ B, double2* __restrict__ psi, int n2) {
  extern __shared__ double2 xs[];
  const long long blkid = blockIdx.x;  // c * n1 + I
  double2* x = psi + blkid * n2;
  for (int j = threadIdx.x; j < n2; j += blockDim.x) xs[j] = x[j];
  __syncthreads();
  const double2* M = B + blkid * (long long)n2 * n2;
  const int part = threadIdx.x & 7;
  for (int row = threadIdx.x >> 3; row < n2; row += blockDim.x >> 3) {
    double2 acc = make_double2(0, 0);
    for (int j = part; j < n2; j += 8) cfma(acc, M[(long long)row * n2 + j], xs[j]);
    for (int off = 4; off > 0; off >>= 1) {
      acc.x += __shfl_xor(acc.x, off, 8);
      acc.y += __shfl_xor(acc.y, off, 8);
    }
    if (part == 0) x[row] = acc;
  }
}

// Sequential block sweep over one channel held in LDS (generic fallback, any n2).
__global__ __launch_bounds__(512) void pc_sweep_kernel(const double2* __restrict__ Mp, double2* __restrict__ psi, int n1,
                                                       int n2, int b, int forward) {
  extern __shared__ double2 y[];
  const int c = blockIdx.x;
  double2* g = psi + (long long)c * n1 * n2;
  for (int i = threadIdx.x; i < n1 * n2; i += blockDim.x) y[i] = g[i];
  __syncthreads();
  const int part = threadIdx.x & 7;
  const int width = b * n2;
  for (int step = 0; step < n1; ++step) {
    const int I = forward ? step : n1 - 1 - step;
    const double2* M = Mp + ((long long)c * n1 + I) * (long long)b * n2 * n2;
    for (int row = threadIdx.x >> 3; row < n2; row += blockDim.x >> 3) {
      double2 acc = make_double2(0, 0);
      const double2* mrow = M + (long long)row * width;
      for (int q = 0; q < b; ++q) {
        const int J = forward ? I - b + q : I + 1 + q;
        if (J < 0 || J >= n1) continue;
        const double2* yj = y + J * n2;
        for (int j = part; j < n2; j += 8) cfma(acc, mrow[q * n2 + j], yj[j]);
      }
      for (int off = 4; off > 0; off >>= 1) {
        acc.x += __shfl_xor(acc.x, off, 8);
        acc.y += __shfl_xor(acc.y, off, 8);
      }
      if (part == 0) {
        double2 v = y[I * n2 + row];
        y[I * n2 + row] = make_double2(v.x - acc.x, v.y - acc.y);
      }
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < n1 * n2; i += blockDim.x) g[i] = y[i];
}

// Block sweep for n2 <= 64: 16 threads per row, 1024 threads; all B*4 matrix elements a
// thread needs for a block step are loaded before any is used, so the step costs one
// memory latency plus the transfer of the block row instead of a chain of dependent
// loads.  The matrix is streamed with non-temporal loads (read once per solve).
typedef double pc_d2v __attribute__((ext_vector_type(2)));
template <int B>
__global__ __launch_bounds__(1024) void pc_sweep16_kernel(const double2* __restrict__ Mp, double2* __restrict__ psi,
                                                          int n1, int n2, int forward) {
  constexpr int JPER = 4;  // ceil(64 / 16)
  extern __shared__ double2 y[];
  const int c = blockIdx.x;
  double2* g = psi + (long long)c * n1 * n2;
  for (int i = threadIdx.x; i < n1 * n2; i += blockDim.x) y[i] = g[i];
  __syncthreads();
  const int part = threadIdx.x & 15;
  const int row = threadIdx.x >> 4;
  const bool active = row < n2;
  const int width = B * n2;
  for (int step = 0; step < n1; ++step) {
    const int I = forward ? step : n1 - 1 - step;
    const double2* mrow = Mp + ((long long)c * n1 + I) * (long long)B * n2 * n2 + (long long)row * width;
    double2 m[B][JPER];
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int J = forward ? I - B + q : I + 1 + q;
#pragma unroll
      for (int u = 0; u < JPER; ++u) {
        const int j = part + 16 * u;
        if (active && J >= 0 && J < n1 && j < n2) {
          const pc_d2v v = __builtin_nontemporal_load(reinterpret_cast<const pc_d2v*>(mrow + q * n2 + j));
          m[q][u] = make_double2(v.x, v.y);
        } else {
          m[q][u] = make_double2(0, 0);
        }
      }
    }
    double2 acc = make_double2(0, 0);
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int J = forward ? I - B + q : I + 1 + q;
      if (J < 0 || J >= n1) continue;
      const double2* yj = y + J * n2;
#pragma unroll
      for (int u = 0; u < JPER; ++u) {
        const int j = part + 16 * u;
        if (j < n2) cfma(acc, m[q][u], yj[j]);
      }
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
      acc.x += __shfl_xor(acc.x, off, 16);
      acc.y += __shfl_xor(acc.y, off, 16);
    }
    if (active && part == 0) {
      const double2 v = y[I * n2 + row];
      y[I * n2 + row] = make_double2(v.x - acc.x, v.y - acc.y);
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < n1 * n2; i += blockDim.x) g[i] = y[i];
}

static void launch_sweep(const Precond& pc, const double2* M, double2* psi, int forward, hipStream_t s) {
  const size_t lds = (size_t)pc.n1 * pc.n2 * sizeof(double2);
  if (pc.n2 <= 64 && pc.b >= 1 && pc.b <= 8) {
    switch (pc.b) {
#define PP_SW(BB) case BB: hipLaunchKernelGGL(pc_sweep16_kernel<BB>, dim3(pc.nchan), dim3(1024), lds, s, M, psi, pc.n1, pc.n2, forward); break;
      PP_SW(1) PP_SW(2) PP_SW(3) PP_SW(4) PP_SW(5) PP_SW(6) PP_SW(7) PP_SW(8)
#undef PP_SW
    }
  } else {
    hipLaunchKernelGGL(pc_sweep_kernel, dim3(pc.nchan), dim3(512), lds, s, M, psi, pc.n1, pc.n2, pc.b, forward);
  }
}

// ------------------------------------------------------------------------------------
// symmetric superblock form
// ------------------------------------------------------------------------------------
struct SymArgs {
  const double2* dinv;
  const double* pc;
  const double* s1;
  const double* s2;
  double2 sh, ss;
  double2* psi;
  int n1, n2, b, ns, mid;
};

constexpr int kSymWaves = 8;
constexpr int kSymOff = 0x40000000;  // past every buffer read through a descriptor here (at most 4 MB), with any row added
typedef unsigned pc_u4 __attribute__((ext_vector_type(4)));
enum { kSymForward = 0, kSymMiddle = 1, kSymBackward = 2 };

// v + v of the lane that the DPP control names
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
  return v + __hiloint2double(hi, lo);
}
// Wave sums of a.x (in lanes 0-31) and a.y (in lanes 32-63): one exchange that halves the values a
// lane carries, one between rows of 16 lanes, then four steps within a row.
__device__ __forceinline__ double wave_sum2(double2 a) {
  const bool up = threadIdx.x & 32;
  double v = (up ? a.y : a.x) + __shfl_xor(up ? a.x : a.y, 32, 64);
  v += __shfl_xor(v, 16, 64);
  v = dpp_add<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v = dpp_add<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v = dpp_add<0x141>(v);  // row_half_mirror
  v = dpp_add<0x140>(v);  // row_mirror
  return v;
}

// Row r of an upper triangle whose diagonal lies in tile T0: lane j of tile t takes column 64 t + j,
// at byte lane_off[t] of a row (past the buffer for columns past the matrix).  Entries left of the
// diagonal are masked by such an offset too, and rows past the matrix end past the buffer, so that
// every load reads zeros there and none sits behind a branch.
template <int NT, int T0>
__device__ __forceinline__ void sym_load(__amdgpu_buffer_rsrc_t D, int r, int lane, int row_bytes,
                                         const int (&lane_off)[NT], double2 (&d)[NT]) {
#pragma unroll
  for (int t = T0; t < NT; ++t) {
    const int off = r * row_bytes + lane_off[t];
    d[t] = __builtin_bit_cast(double2,
                              __builtin_amdgcn_raw_buffer_load_b128(D, t == T0 && lane < r - 64 * T0 ? kSymOff : off, 0, 0));
  }
}

template <class F, int... T>
__device__ __forceinline__ void for_each_tile(F&& f, std::integer_sequence<int, T...>) {
  (f(std::integral_constant<int, T>{}), ...);
}

// One workgroup of 8 waves per (channel, chain).  Each superblock is a symmetric matrix-vector
// product: wave w takes rows w, w + 8, ..., keeps its columns' sums (y_j += d_rj v_r) in registers over
// all its rows, sums each row across the lanes (y_r += d_rj v_j; the stored diagonal is halved, so that
// both parts take it) and has two more rows' loads in flight meanwhile, as well as the next
// superblock's first rows during the coupling.  Bound by what one CU pulls from HBM:
// two rows ahead it is about 31 GB/s, 84 workgroups at once.  Helium, 42 x 60 x 60: 170 + 49 + 170 us
// (inwards, middle, outwards) per solve, against 2 x 549 + 2 x 30 us
// for the general form; 15 x 13 x 13: 16 + 12 + 16 us against 2 x 22.8 + 2 x 4.5 us.
template <int NT, int W>
__global__ __launch_bounds__(64 * kSymWaves) void pc_sym_kernel(SymArgs a, int mode) {
  extern __shared__ double2 lds[];
  constexpr int M = 64 * NT;
  const int n2 = a.n2, b = a.b, m = b * n2, w2 = 2 * b + 1;
  const int c = mode == kSymMiddle ? blockIdx.x : blockIdx.x >> 1, end = mode == kSymMiddle ? 0 : blockIdx.x & 1;
  double2* v = lds;                 // [M] operand of the product
  double2* x = v + M;               // [M] the last superblock's result
  double2* rowsum = x + M;          // [M]
  double2* red = rowsum + M;        // [8][M] column sums per wave, or the coupling's parts [b b][n2]
  double* s2 = reinterpret_cast<double*>(red + kSymWaves * M);  // [w2][n2]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double2* psi = a.psi + (long long)c * a.n1 * n2;
  for (int e = tid; e < w2 * n2; e += blockDim.x) s2[e] = a.s2[e];
  auto block_rows = [&](int s) { return min(b, a.n1 - s * b); };
  // part[q b + q'][i] = sum over block q' of superblock `from` of the coupling to block row q of `to`
  // (neighbours) times x.  Wave w takes the block pairs w, w + 8, ...; a pair's W diagonals are read
  // while the pair before is summed (masked as above past the band, the matrix and the last pair).
  auto couple = [&](int to, int from) {
    const int low = min(to, from), rt = block_rows(to), rf = block_rows(from);
    int i = min(lane, n2 - 1);
    asm volatile("" : "+v"(i));  // as in product(): the diagonals' offsets stay inside the loop
    const __amdgpu_buffer_rsrc_t P = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<double*>(a.pc + ((long long)c * a.n1 + low * b) * b * w2 * n2), (short)0,
        min(b, a.n1 - low * b) * b * w2 * n2 * (int)sizeof(double), 0x00020000);
    struct Job {
      int q, qf, delta;
    };
    Job at = {0, -1, 0};
    int skip = wave + 1;
    auto next = [&]() {  // the wave's next pair; q = rt when there is none
      while (skip > 0 && at.q < rt) {
        if (++at.qf >= rf) {
          at.qf = 0;
          ++at.q;
        }
        at.delta = to < from ? b + at.qf - at.q : b + at.q - at.qf;
        if (at.delta <= b && at.q < rt) --skip;
      }
      skip = kSymWaves;
      return at;
    };
    // row i couples to column i + d - b when `to` is the lower superblock, else it is the column of
    // the stored row i - d + b
    auto other = [&](int d) { return to < from ? i + d - b : i - d + b; };
    auto load = [&](const Job& k, double (&p)[W], double& s1) {
      s1 = a.s1[(low * b + min(to < from ? k.q : k.qf, b - 1)) * (b + 1) + min(max(k.delta, 0), b)];
#pragma unroll
      for (int d = 0; d < W; ++d) {
        const int j = other(d), row = ((to < from ? k.q : k.qf) * b + k.delta - 1) * w2 + d;
        const bool in = k.q < rt && d < w2 && j >= 0 && j < n2;
        const int off = in ? (row * n2 + (to < from ? i : j)) * (int)sizeof(double) : kSymOff;
        p[d] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(P, off, 0, 0));
      }
    };
    auto sum = [&](const Job& k, const double (&p)[W], double s1) {
      double2 acc = make_double2(0, 0);
#pragma unroll
      for (int d = 0; d < W; ++d) {
        const int j = other(d), jc = min(max(j, 0), n2 - 1);
        const bool in = d < w2 && j == jc;
        const double sv = s1 * s2[min(d, w2 - 1) * n2 + (to < from ? i : jc)];
        const double2 xv = x[k.qf * n2 + jc];
        const double2 av = make_double2(fma(a.sh.x, p[d], a.ss.x * sv), fma(a.sh.y, p[d], a.ss.y * sv));
        double2 t = acc;
        cfma(t, av, xv);
        acc.x = in ? t.x : acc.x;
        acc.y = in ? t.y : acc.y;
      }
      if (lane < n2) red[(k.q * b + k.qf) * n2 + lane] = acc;
    };
    double pa[W], pb[W], sa, sb;
    Job ja = next(), jb;
    load(ja, pa, sa);
    while (true) {
      jb = next();
      load(jb, pb, sb);
      if (ja.q >= rt) break;
      sum(ja, pa, sa);
      ja = next();
      load(ja, pa, sa);
      if (jb.q >= rt) break;
      sum(jb, pb, sb);
    }
    __syncthreads();
  };
  // sum of the parts of row e of superblock `to`
  auto coupled = [&](int to, int from, int e) {
    const int q = e / n2, i = e - q * n2;
    double2 s = make_double2(0, 0);
    for (int qf = 0; qf < block_rows(from); ++qf)
      if (to < from ? qf <= q : qf >= q) s = cadd(s, red[(q * b + qf) * n2 + i]);
    return s;
  };
  double2 d[3][NT];  // rows in flight
  int lane_off[NT];
  __amdgpu_buffer_rsrc_t D;
  const int row_bytes = m * (int)sizeof(double2);
  auto first_rows = [&](int s) {
    const int ms = block_rows(s) * n2;
    D = __builtin_amdgcn_make_buffer_rsrc(const_cast<double2*>(a.dinv + ((long long)c * a.ns + s) * m * m), (short)0,
                                          m * row_bytes, 0x00020000);
#pragma unroll
    for (int t = 0; t < NT; ++t) lane_off[t] = 64 * t + lane < ms ? (64 * t + lane) * (int)sizeof(double2) : kSymOff;
    sym_load<NT, 0>(D, wave, lane, row_bytes, lane_off, d[0]);
    sym_load<NT, 0>(D, wave + kSymWaves, lane, row_bytes, lane_off, d[1]);
  };
  // x (LDS) = D_s^-1 v
  auto product = [&](int s) {
    const int ms = block_rows(s) * n2;
    double2 vj[NT], col[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      vj[t] = v[64 * t + lane];
      col[t] = make_double2(0, 0);
    }
    // the rows whose diagonal lies in tile T0 (64 rows, 8 of them per wave): only tiles T0 .. NT - 1
    auto rows_of_tile = [&](auto tile) {
      constexpr int T0 = decltype(tile)::value;
      if (64 * T0 >= ms) return;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        // The row offsets are the same for every superblock: kept apart from the loop over them, or
        // hundreds of them are formed ahead of it and spilt; likewise the scheduler may not pull the
        // loads of later rows forward.
        int first = wave, l = lane;
        asm volatile("" : "+s"(first), "+v"(l));
        const int r = 64 * T0 + kSymWaves * k + first;
        constexpr int TN = T0 + 1 < NT ? T0 + 1 : T0;  // two rows on: the next tile's after the sixth
        double2(&ahead)[NT] = d[(8 * T0 + k + 2) % 3];
        if (k < 6 || TN == T0) sym_load<NT, T0>(D, r + 2 * kSymWaves, l, row_bytes, lane_off, ahead);
        else sym_load<NT, TN>(D, r + 2 * kSymWaves, l, row_bytes, lane_off, ahead);
        __builtin_amdgcn_sched_barrier(0);
        const double2(&row)[NT] = d[(8 * T0 + k) % 3];
        const double2 vr = v[r];
        double2 sum = make_double2(0, 0);
#pragma unroll
        for (int t = T0; t < NT; ++t) {
          cfma(sum, row[t], vj[t]);
          cfma(col[t], row[t], vr);
        }
        // formed here, not put off with the row kept: nothing reads them before the last row
#pragma unroll
        for (int t = T0; t < NT; ++t) asm volatile("" : "+v"(col[t].x), "+v"(col[t].y));
        // every lane of a half holds its total
        reinterpret_cast<double*>(rowsum + r)[lane >> 5] = wave_sum2(sum);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    for_each_tile(rows_of_tile, std::make_integer_sequence<int, NT>{});
#pragma unroll
    for (int t = 0; t < NT; ++t) red[wave * M + 64 * t + lane] = col[t];
    __syncthreads();
    if (tid < ms) {
      double2 y = rowsum[tid];
#pragma unroll
      for (int k = 0; k < kSymWaves; ++k) y = cadd(y, red[k * M + tid]);
      x[tid] = y;
    }
    __syncthreads();
  };
  // element tid of a superblock (M <= 512 threads)
  auto element = [&](int s) { return tid < block_rows(s) * n2 ? psi[(long long)s * m + tid] : make_double2(0, 0); };
  const int steps = mode == kSymMiddle ? 1 : end ? a.ns - 1 - a.mid : a.mid;
  if (steps == 0) return;
  if (mode == kSymBackward && tid < M) x[tid] = element(a.mid);
  __syncthreads();
  for (int k = 0; k < steps; ++k) {
    // the superblock, and the neighbours whose results are known: outside it on the way in, both for
    // the middle, inside it on the way out
    int s = a.mid, near[2] = {-1, -1};
    if (mode == kSymForward) {
      s = end ? a.ns - 1 - k : k;
      if (k > 0) near[0] = end ? s + 1 : s - 1;
    } else if (mode == kSymBackward) {
      s = end ? a.mid + 1 + k : a.mid - 1 - k;
      near[0] = end ? s - 1 : s + 1;
    } else {
      near[0] = s - 1;
      near[1] = s + 1 < a.ns ? s + 1 : -1;
    }
    const bool on = tid < block_rows(s) * n2;
    first_rows(s);
    const double2 own = element(s);
    double2 coupling = make_double2(0, 0);
    for (int side = 0; side < 2; ++side) {
      const int from = near[side];
      if (from < 0) continue;
      if (mode == kSymMiddle) {
        if (tid < M) x[tid] = element(from);
        __syncthreads();
      }
      couple(s, from);
      if (on) coupling = cadd(coupling, coupled(s, from, tid));
      __syncthreads();
    }
    if (tid < M) v[tid] = !on ? make_double2(0, 0) : mode == kSymBackward ? coupling : csub(own, coupling);
    __syncthreads();
    product(s);
    if (on) {
      const double2 xs = mode == kSymBackward ? csub(own, x[tid]) : x[tid];
      x[tid] = xs;
      psi[(long long)s * m + tid] = xs;
    }
    __syncthreads();
  }
}

static size_t sym_lds(int nt, int n2, int b) {
  return (size_t)(3 + kSymWaves) * 64 * nt * sizeof(double2) + (size_t)(2 * b + 1) * n2 * sizeof(double);
}

// (column tiles, widest band): b <= 4, 6 and 8 with n2 <= 64
#define PP_SYM_FORMS(X)                                                                                    \
  X(1, 9) X(2, 9) X(3, 9) X(4, 9) X(1, 13) X(2, 13) X(3, 13) X(4, 13) X(5, 13) X(6, 13) X(1, 17) X(2, 17) \
  X(3, 17) X(4, 17) X(5, 17) X(6, 17) X(7, 17) X(8, 17)
static int sym_form(const Precond& pc) {
  return (pc.b * pc.n2 + 63) / 64 * 32 + (pc.b <= 4 ? 9 : pc.b <= 6 ? 13 : 17);
}

// The LDS limit belongs to the kernel, not to a preconditioner: the most that any of this form needs.
static void sym_prepare(const Precond& pc) {
  switch (sym_form(pc)) {
#define PP_SYM(NT, W)                                                                                          \
  case NT * 32 + W:                                                                                            \
    PP_HIP(hipFuncSetAttribute((const void*)pc_sym_kernel<NT, W>, hipFuncAttributeMaxDynamicSharedMemorySize,  \
                               (int)sym_lds(NT, 64, W / 2)));                                                  \
    break;
    PP_SYM_FORMS(PP_SYM)
#undef PP_SYM
  }
}

static void sym_solve(const Precond& pc, double2* psi, hipStream_t s) {
  const int nt = (pc.b * pc.n2 + 63) / 64;
  const SymArgs a = {pc.dinv.ptr, pc.pc.ptr, pc.s1.ptr, pc.s2.ptr, pc.sh, pc.ss, psi, pc.n1, pc.n2, pc.b, pc.ns, pc.mid};
  auto launch = [&](int mode) {
    const dim3 grid(mode == kSymMiddle ? pc.nchan : 2 * pc.nchan);
    switch (sym_form(pc)) {
#define PP_SYM(NT, W)                                                                                              \
  case NT * 32 + W:                                                                                                \
    hipLaunchKernelGGL((pc_sym_kernel<NT, W>), grid, dim3(64 * kSymWaves), sym_lds(nt, pc.n2, pc.b), s, a, mode);  \
    break;
      PP_SYM_FORMS(PP_SYM)
#undef PP_SYM
    }
  };
  if (pc.ns > 1) launch(kSymForward);
  launch(kSymMiddle);
  if (pc.ns > 1) launch(kSymBackward);
  PP_HIP(hipGetLastError());
}

void precond_solve(const Precond& pc, double2* psi, hipStream_t s) {
  if (pc.sym) {
    sym_solve(pc, psi, s);
    return;
  }
  const int nblk = pc.nchan * pc.n1;
  const size_t lds_diag = pc.n2 * sizeof(double2);
  const size_t lds_sweep = (size_t)pc.n1 * pc.n2 * sizeof(double2);
  (void)lds_sweep;
  hipLaunchKernelGGL(pc_diag_kernel, dim3(nblk), dim3(512), lds_diag, s, pc.linv.ptr, psi, pc.n2);
  launch_sweep(pc, pc.lp.ptr, psi, 1, s);
  hipLaunchKernelGGL(pc_diag_kernel, dim3(nblk), dim3(512), lds_diag, s, pc.uinv.ptr, psi, pc.n2);
  launch_sweep(pc, pc.up.ptr, psi, 0, s);
  PP_HIP(hipGetLastError());
}

}  // namespace pp

using namespace pp;

extern "C" int pp_precond_create(int nchan, int n1, int n2, int band, const double* s1, const double* s2,
                                 const pp_cplx* p_data, int p1_count, const int32_t* pairs1, int p2_count,
                                 const int32_t* pairs2, pp_cplx scaling_h, pp_cplx scaling_s, pp_precond** out) {
  return guarded([&] {
    PP_REQUIRE(out && s1 && s2 && p_data && pairs1 && pairs2, "NULL argument");
    PP_REQUIRE(nchan > 0 && n1 > 0 && n2 > 0 && band >= 0 && band < n1, "invalid sizes");
    PP_REQUIRE((size_t)n1 * n2 * sizeof(double2) <= 64 * 1024, "channel block exceeds 64 KiB of LDS");
    std::vector<int> pos1((size_t)n1 * n1, -1), pos2((size_t)n2 * n2, -1);
    for (int p = 0; p < p1_count; ++p) {
      const int r = pairs1[2 * p], c = pairs1[2 * p + 1];
      PP_REQUIRE(r >= 0 && r < n1 && c >= 0 && c < n1, "pair out of range");
      pos1[(size_t)r * n1 + c] = p;
    }
    for (int p = 0; p < p2_count; ++p) {
      const int r = pairs2[2 * p], c = pairs2[2 * p + 1];
      PP_REQUIRE(r >= 0 && r < n2 && c >= 0 && c < n2, "pair out of range");
      pos2[(size_t)r * n2 + c] = p;
    }
    const cd sh(scaling_h.re, scaling_h.im), ss(scaling_s.re, scaling_s.im);
    const cd* pd = reinterpret_cast<const cd*>(p_data);
    const unsigned nthreads = std::max(1u, std::min({std::thread::hardware_concurrency(), 16u, (unsigned)nchan}));
    auto each_channel = [&](auto&& work) {
      std::vector<std::thread> pool;
      std::vector<std::string> errors(nthreads);
      for (unsigned t = 0; t < nthreads; ++t) {
        pool.emplace_back([&, t] {
          try {
            for (int c = (int)t; c < nchan; c += (int)nthreads) work(c);
          } catch (const std::exception& e) {
            errors[t] = e.what();
          }
        });
      }
      for (auto& th : pool) th.join();
      for (auto& e : errors)
        if (!e.empty()) throw Error(PP_ERR_INVALID, e);
    };
    auto matrix = [&](int c) {
      return SymMatrix{n1, n2, band, p2_count, s1, s2, pd + (size_t)c * p1_count * p2_count, pos1.data(), pos2.data(),
                       sh, ss};
    };
    // the superblock kernel's limits: lanes for a block row, 8 column tiles
    bool sym = band >= 1 && band <= 8 && n2 <= 64;
    if (sym) {
      std::vector<char> ok(nchan, 0);
      each_channel([&](int c) { ok[c] = is_symmetric(matrix(c), p1_count); });
      for (char o : ok) sym = sym && o;
    }
    if (sym) {
      const int ns = (n1 + band - 1) / band, mid = ns / 2, m = band * n2, w = 2 * band + 1;
      std::vector<cd> dinv((size_t)nchan * ns * m * m);
      std::vector<double> pc((size_t)nchan * n1 * band * w * n2, 0.0), s1b((size_t)n1 * (band + 1), 0.0),
          s2b((size_t)w * n2, 0.0);
      for (int I = 0; I < n1; ++I)
        for (int d = 0; d <= band && I + d < n1; ++d) s1b[(size_t)I * (band + 1) + d] = s1[(size_t)I * n1 + I + d];
      for (int d = 0; d < w; ++d)
        for (int i = 0; i < n2; ++i)
          if (i + d - band >= 0 && i + d - band < n2) s2b[(size_t)d * n2 + i] = s2[(size_t)i * n2 + i + d - band];
      std::atomic<bool> fits{true};
      each_channel([&](int c) {
        const SymMatrix M = matrix(c);
        if (!fits || !factor_symmetric(M, ns, mid, dinv.data() + (size_t)c * ns * m * m)) {
          fits = false;
          return;
        }
        for (int I = 0; I < n1; ++I)
          for (int delta = 1; delta <= band && I + delta < n1; ++delta)
            for (int d = 0; d < w; ++d)
              for (int i = 0; i < n2; ++i)
                if (i + d - band >= 0 && i + d - band < n2)
                  pc[((((size_t)c * n1 + I) * band + delta - 1) * w + d) * n2 + i] = M.pval(I, I + delta, i, i + d - band);
      });
      if (fits) {
        auto* p = new pp_precond();
        try {
          Precond& q = p->p;
          q.nchan = nchan;
          q.n1 = n1;
          q.n2 = n2;
          q.b = band;
          q.sym = true;
          q.ns = ns;
          q.mid = mid;
          q.sh = make_double2(sh.real(), sh.imag());
          q.ss = make_double2(ss.real(), ss.imag());
          q.dinv.upload(reinterpret_cast<const double2*>(dinv.data()), dinv.size());
          q.pc.upload(pc.data(), pc.size());
          q.s1.upload(s1b.data(), s1b.size());
          q.s2.upload(s2b.data(), s2b.size());
          sym_prepare(q);
          PP_HIP(hipDeviceSynchronize());
        } catch (...) {
          delete p;
          throw;
        }
        *out = p;
        return;
      }
    }
    const size_t bs = (size_t)n2 * n2;
    HostFactors F;
    F.linv.assign((size_t)nchan * n1 * bs, 0);
    F.uinv.assign((size_t)nchan * n1 * bs, 0);
    F.lp.assign((size_t)nchan * n1 * band * bs, 0);
    F.up.assign((size_t)nchan * n1 * band * bs, 0);
    each_channel([&](int c) {
      factor_channel(c, n1, n2, band, s1, s2, pd, p1_count, pos1, p2_count, pos2, sh, ss, F);
    });
    auto* p = new pp_precond();
    try {
      p->p.nchan = nchan;
      p->p.n1 = n1;
      p->p.n2 = n2;
      p->p.b = band;
      static_assert(sizeof(cd) == sizeof(double2), "complex layout");
      p->p.linv.upload(reinterpret_cast<const double2*>(F.linv.data()), F.linv.size());
      p->p.uinv.upload(reinterpret_cast<const double2*>(F.uinv.data()), F.uinv.size());
      p->p.lp.upload(reinterpret_cast<const double2*>(F.lp.data()), F.lp.size());
      p->p.up.upload(reinterpret_cast<const double2*>(F.up.data()), F.up.size());
      PP_HIP(hipDeviceSynchronize());
    } catch (...) {
      delete p;
      throw;
    }
    *out = p;
  });
}

extern "C" int pp_precond_destroy(pp_precond* pc) {
  return guarded([&] { delete pc; });
}

extern "C" int pp_precond_solve(const pp_precond* pc, pp_cplx* psi, pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(pc && psi, "NULL argument");
    precond_solve(pc->p, reinterpret_cast<double2*>(psi), (hipStream_t)stream);
  });
}
