// CTMRG renormalisation step, its reverse sweep, the top-k FP64 eigensolver
// and the energy chain, orchestrated on one HIP stream.
//
// Reference: src/ctmrg.jl:110-153 (ctmrg, ctmrgstep), src/fixedpoint.jl:11-41
// (fixedpoint, StopFunction), src/trg.jl:72-106 (svd_back), src/autodiff.jl:23-29
// (norm adjoint), src/variationalipeps.jl:28-56 (energy, expectationvalue).
//
// Notation: chi = environment bond, D = double-layer bond (Dd = d^2 in the
// reference), n = chi*D.  Every tensor is column-major with the reference's
// index order; contractions are issued as the reference's einsum strings
// through contract_desc (tc_build.cpp).
//
// The n x n "corner matrix" cpmat + cpmat^T is symmetric, so its SVD is
// obtained from an eigendecomposition: s = |lambda| sorted descending,
// U = eigenvectors, V = U sign(lambda).
#include "ctmrg.h"
#include "resolvent.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>

namespace tnad {

static inline size_t esize(Prec p) { return p == Prec::F64 ? 8 : 4; }

// --------------------------------------------------------------------------
// small kernels private to this file
// --------------------------------------------------------------------------
namespace {

constexpr int NT = 256;

// out[j] = |Y[:, j] - theta_j X[:, j]| for j < gridDim.x; block 0 also writes out[gridDim.x] = theta_0 and
// out[gridDim.x + 1] = the Rayleigh-Ritz flag (*gate, or 1 without one), so that the host reads the
// iteration's whole status with one transfer
__global__ void resid_norms_kernel(const double* __restrict__ X, const double* __restrict__ Y,
                                   const double* __restrict__ theta, int n, double* __restrict__ out,
                                   const int* __restrict__ gate) {
  __shared__ double red[4];
  const int j = blockIdx.x;
  if (j == 0 && threadIdx.x == 0) {
    out[gridDim.x] = theta[0];
    out[gridDim.x + 1] = gate ? (double)*gate : 1.0;
  }
  const double th = theta[j];
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    double r = Y[i + (long long)j * n] - th * X[i + (long long)j * n];
    acc += r * r;
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) out[j] = sqrt(red[0] + red[1] + red[2] + red[3]);
}

// Next subspace block from the Rayleigh-Ritz pairs:
// Z[:, j] = Yr[:, j] / theta_j = Xr[:, j] + R[:, j] / theta_j (R = Yr - Xr Theta is orthogonal to Xr, so
// Z^T Z = I + (R Theta^-1)^T (R Theta^-1) >= I stays well conditioned however collinear the residuals are);
// numerically null Ritz values keep Z[:, j] = Xr[:, j].  One block of 256 threads per column j.
__global__ __launch_bounds__(256) void ritz_scale_kernel(const double* __restrict__ Xr, const double* __restrict__ Yr,
                                                         const double* __restrict__ theta, int n,
                                                         double* __restrict__ Z) {
  const int j = blockIdx.x;
  const double t0 = fabs(theta[0]), th = theta[j];
  const bool use_y = fabs(th) > 1e-14 * t0;
  const size_t o = (size_t)n * j;
  for (int i = threadIdx.x; i < n; i += 256) Z[o + i] = use_y ? Yr[o + i] / th : Xr[o + i];
}

// *out = sum_ij (G_ij - delta_ij)^2 (one workgroup; G is k x k)
// |G - I|_F^2 of a k x k matrix (k <= 256): one workgroup of GD_NT threads, thread (row i, column
// phase jo) sums rows i over columns jo, jo + GD_NT / 256, ... (coalesced along rows)
constexpr int GD_NT = 1024;
// (next to the Cholesky kernel's smallest pivot and breakdown column, so the host reads the pass's status with
// one transfer)
__global__ __launch_bounds__(GD_NT) void gram_dev_kernel(const double* __restrict__ G, int k,
                                                         double* __restrict__ out) {
  __shared__ double red[GD_NT / 64];
  const int t = threadIdx.x, i = t & 255, jo = t >> 8;
  double acc = 0.0;
  if (i < k)
#pragma unroll 8
    for (int j = jo; j < k; j += GD_NT / 256) {   // (eight loads in flight; one at a time 14.6 us on average at k up to 192, now 6.4)
      const double v = G[i + (size_t)k * j] - (i == j ? 1.0 : 0.0);
      acc += v * v;
    }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o);
  if ((t & 63) == 0) red[t >> 6] = acc;
  __syncthreads();
  if (t == 0) {
    double s = 0.0;
    for (int w = 0; w < GD_NT / 64; ++w) s += red[w];
    out[0] = s;
  }
}

// F = (I + E)^{-1/2} to second order for G = I + E (binomial series: I - E/2 + 3/8 E^2), written from G and
// G2 = G G as 15/8 I - 5/4 G + 3/8 G2; F may overwrite G2 (each entry is read before it is written)
__global__ void inv_sqrt2_coef_kernel(const double* __restrict__ G, const double* G2, int k, double* F) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= k * k) return;
  const int i = q % k, j = q / k;
  F[q] = 0.375 * G2[q] - 1.25 * G[q] + (i == j ? 1.875 : 0.0);
}

// *out = max(*out, max |A_i|), as bits (the order of non-negative doubles is that of their bits; NaNs are passed over)
__global__ void max_bits_kernel(const double* __restrict__ A, size_t n, unsigned long long* __restrict__ out) {
  double m = 0.0;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    m = fmax(m, fabs(A[i]));
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_down(m, o));
  if ((threadIdx.x & 63) == 0) atomicMax(out, (unsigned long long)__double_as_longlong(m));
}

// make the largest-|.| entry of every column positive (first occurrence wins);
// the same sign is applied to the companion block Y (A*X) when given.
__global__ void canon_sign_kernel(double* __restrict__ X, double* __restrict__ Y, int n) {
  __shared__ double bv[4];
  __shared__ int bi[4];
  const int j = blockIdx.x;
  double best = -1.0;
  int idx = 0x7fffffff;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    double v = fabs(X[i + (long long)j * n]);
    if (v > best || (v == best && i < idx)) { best = v; idx = i; }
  }
  for (int o = 32; o > 0; o >>= 1) {
    double ob = __shfl_down(best, o);
    int oi = __shfl_down(idx, o);
    if (ob > best || (ob == best && oi < idx)) { best = ob; idx = oi; }
  }
  if ((threadIdx.x & 63) == 0) { bv[threadIdx.x >> 6] = best; bi[threadIdx.x >> 6] = idx; }
  __syncthreads();
  __shared__ double sgn;
  if (threadIdx.x == 0) {
    double b = bv[0];
    int ii = bi[0];
    for (int w = 1; w < 4; ++w)
      if (bv[w] > b || (bv[w] == b && bi[w] < ii)) { b = bv[w]; ii = bi[w]; }
    sgn = ii < n && X[ii + (long long)j * n] < 0 ? -1.0 : 1.0;   // (no such entry in a column of NaNs)
  }
  __syncthreads();
  if (sgn < 0) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      X[i + (long long)j * n] = -X[i + (long long)j * n];
      if (Y) Y[i + (long long)j * n] = -Y[i + (long long)j * n];
    }
  }
}

// coefficient block (rows x chi) of the eigen adjoint (see eig_adjoint below).  Rows i < chi, the kept pairs:
//   coef = Kt/2 with Kt = R11 Sigma + Sigma R11^T + C1bar,  R11_ij = (F_ij g_ij + F_ji g_ji) s_j,
// F_ij = (s_j^2 - s_i^2) / ((s_j^2 - s_i^2)^2 + eta),  s = |lambda|.
// Evaluated without FP contraction: the reference forms S2 = S.^2 first and then
// S2' .- S2 (src/trg.jl:76-78), so the diagonal difference is exactly zero and the
// Lorentzian F vanishes there; a fused multiply-add would leave the rounding residual of
// s^2 (~1e-17) in place of that zero and F would blow up to ~1e23.
// Rows i >= chi (only with the whole spectrum, rows = n): the pairs of a kept and a discarded vector,
//   (lambda_j + lambda_i) L(s_j^2 - s_i^2) g_ij,
// the difference of squares formed as (lambda_j - lambda_i)(lambda_j + lambda_i), so that the quotient stays
// accurate for a (+s, -s) pair; nothing for a kept value at the rounding level (s_j <= 1e-14 s_0, as in
// resolvent_pcg).
__global__ void eigback_coef_kernel(const double* __restrict__ g, const double* __restrict__ lam,
                                    const double* __restrict__ C1bar, int chi, int rows, double eta,
                                    double* __restrict__ coef) {
#pragma clang fp contract(off)
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= rows * chi) return;
  int i = e % rows, j = e / rows;
  double li = lam[i], lj = lam[j];
  if (i >= chi) {
    const double p = lj + li, d = (lj - li) * p;
    coef[e] = fabs(lj) > 1e-14 * fabs(lam[0]) ? p * (d / (d * d + eta)) * g[e] : 0.0;
    return;
  }
  double si2 = li * li, sj2 = lj * lj;
  double Fij = (sj2 - si2) / ((sj2 - si2) * (sj2 - si2) + eta);
  double Fji = -Fij;
  double gij = g[i + (long long)j * rows];
  double gji = g[j + (long long)i * rows];
  double sj = fabs(lj), si = fabs(li);
  double sigj = lj < 0 ? -1.0 : 1.0, sigi = li < 0 ? -1.0 : 1.0;
  double R_ij = (Fij * gij + Fji * gji) * sj;   // R11[i,j]
  double R_ji = (Fji * gji + Fij * gij) * si;   // R11[j,i]
  double Kt = R_ij * sigj + sigi * R_ji + C1bar[i + (long long)j * chi];
  coef[e] = 0.5 * Kt;
}

// W[:, j] += lambda_j * Xr[:, j] + AXr[:, j]
__global__ void add_lam_cols_kernel(double* __restrict__ W, const double* __restrict__ Xr,
                                    const double* __restrict__ AXr, const double* __restrict__ lam, int n,
                                    int chi) {
  size_t tot = (size_t)n * chi;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot; e += (size_t)gridDim.x * blockDim.x) {
    int j = e / n;
    W[e] += lam[j] * Xr[e] + AXr[e];
  }
}

// lbar[abc, x, y] += f * *coef * tr[abc] * delta_xy
__global__ void add_trace_diag_kernel(double* __restrict__ lbar, const double* __restrict__ tr,
                                      const double* __restrict__ coef, double f, int m, int s) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m * s) return;
  int abc = e % m, x = e / m;
  const double c = f * *coef;
  lbar[abc + (size_t)m * (x + s * x)] += c * tr[abc];
}

// tr[abc] = sum_x l[abc, x, x]
__global__ void trace_last2_kernel(const double* __restrict__ l, int m, int s, double* __restrict__ tr) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m) return;
  double acc = 0.0;
  for (int x = 0; x < s; ++x) acc += l[e + (size_t)m * (x + s * x)];
  tr[e] = acc;
}

// out = a / b  and the energy-adjoint scalars (ebar = 1/nn, nnbar = -e/nn^2), all on device
__global__ void energy_scalars_kernel(const double* e, const double* nn, double* out) {
  out[0] = e[0] / nn[0];
  out[1] = 1.0 / nn[0];
  out[2] = -e[0] / (nn[0] * nn[0]);
}

// norm adjoint: out = ybar/|x| + nbar * x / (|x| + eps(0f0)),  nbar = -<x,ybar>/|x|^2
__global__ void norm_back_kernel(const double* __restrict__ x, const double* __restrict__ ybar,
                                 const double* __restrict__ sumsq, const double* __restrict__ dot,
                                 double* __restrict__ out, size_t n) {
  const double nrm = sqrt(*sumsq);
  const double nbar = -(*dot) / (nrm * nrm);
  const double eps0 = 1.401298464324817e-45;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    out[i] = ybar[i] / nrm + nbar * x[i] / (nrm + eps0);
}

inline unsigned nb(size_t n) {
  size_t b = (n + NT - 1) / NT;
  if (b > 65535ull * 8) b = 65535ull * 8;
  return (unsigned)(b ? b : 1);
}

}  // namespace

// --------------------------------------------------------------------------
// typed buffer helpers
// --------------------------------------------------------------------------
PBuf::PBuf(Ctx* c, Prec p_, size_t n_) : p(p_), n(n_), b(c, n_ * esize(p_)) {}

void to_prec(Ctx* c, const double* src, PBuf& dst) {
  if (dst.p == Prec::F64) k_copy(src, dst.b.as<double>(), dst.n, c->stream);
  else k_cast_from<float>(src, dst.b.as<float>(), dst.n, c->stream);
}
void from_prec(Ctx* c, const PBuf& src, double* dst) {
  if (src.p == Prec::F64) k_copy(src.b.as<double>(), dst, src.n, c->stream);
  else k_cast<float>(src.b.as<float>(), dst, src.n, c->stream);
}

// src at precision p: the buffer itself when the storage type already matches,
// otherwise a converted copy held in tmp (FP64 <-> float storage)
const PBuf& at_prec(Ctx* c, const PBuf& src, Prec p, PBuf& tmp) {
  const bool src64 = src.p == Prec::F64, want64 = p == Prec::F64;
  if (src64 == want64) return src;
  tmp = PBuf(c, p, src.n);
  if (src64) {
    to_prec(c, src.b.as<double>(), tmp);
  } else {
    k_cast<float>(src.b.as<float>(), tmp.b.as<double>(), src.n, c->stream);
  }
  return tmp;
}

// src at precision p as a kernel operand: src itself for FP64, else a converted copy held in tmp
static const void* as_prec(Ctx* c, const double* src, size_t n, Prec p, PBuf& tmp) {
  if (p == Prec::F64) return src;
  tmp = PBuf(c, p, n);
  to_prec(c, src, tmp);
  return tmp.ptr();
}

void tc(Ctx* c, Prec p, const TView& A, const void* a, const TView& B, const void* b, const TView& C, void* o,
        double alpha, double beta) {
  tc_launch(c, p, contract_desc(A, B, C, alpha, beta), a, b, o, c->stream);
}

// Opt-in diagnostics (TNAD_DEBUG_EIG=1): report whether a device array holds a non-finite value.
static void dbg_finite(Ctx* c, const char* what, const double* dev, size_t n) {
  static const bool on = [] {
    const char* e = std::getenv("TNAD_DEBUG_FINITE");
    return e && *e && *e != '0';
  }();
  if (!on) return;
  std::vector<double> h(n);
  c->read_async(h.data(), dev, n * 8);
  c->sync();
  size_t bad = 0;
  double mx = 0.0;
  for (double v : h) {
    if (!std::isfinite(v)) ++bad;
    else mx = std::max(mx, std::fabs(v));
  }
  std::fprintf(stderr, "[tnad eig]   %s: %zu non-finite of %zu, max |finite| %.3e\n", what, bad, n, mx);
}

// ==========================================================================
// Eigensolver: top-k eigenpairs of a symmetric n x n FP64 matrix by |lambda|
// ==========================================================================
// light: one pass is enough (the block goes through another product and orthonormalisation before a
// Rayleigh-Ritz step looks at it, so only its span and a deviation well below 1 matter): X^T X is not formed
// range (nullable): set, and nothing done to Y, when the first pass finds a squared column norm outside 1e-200 .. 1e200
static void orthonormalize(Ctx* c, double* Y, int n, int k, double* X, EigWork& w, unsigned seed, bool light = false,
                           bool* range = nullptr) {
  hipStream_t s = c->stream;
  // (the columns' scale is taken out of the Gram matrix by the Cholesky kernel: Y itself is only normalised,
  // with a random refill of null columns, when a pass fails)
  // A well-conditioned block takes plain CholeskyQR passes: one when the result is orthonormal to
  // working precision (|X^T X - I|_F <= 1e-12, the usual case once the iteration converges), else a
  // second: X (X^T X)^{-1/2} to second order when |X^T X - I|_F <= 1e-5, CholeskyQR2 above.  A pass counts when the
  // Cholesky pivots of the Gram matrix (unit columns) stay above 1e-6, and, unless it is a light one, when it leaves a
  // deviation below 1e-2: pivots alone bound no condition number, but a light block meets another product and a
  // measured pass before anything is read off it.  The first pass and the test run before
  // the host looks at the pivots, so that one round trip serves both.  A block that fails (condition
  // number up to ~1e10: the first product with a random block) takes one shifted CholeskyQR pass, which
  // keeps its small directions (to an accuracy of u over their relative size, all that the iteration needs of
  // them), and the plain pass again.  If that fails too, the block has lower rank than k (a rank-deficient
  // corner matrix): columns that a shifted pass finds linearly dependent on earlier ones (pivot at the
  // shift's level) are replaced by random directions, so the block always spans k dimensions, and what
  // still fails takes shifted CholeskyQR followed by two plain passes (sCholQR3).
  std::vector<double> piv(k);
  std::vector<int> dead(k);
  const double u = 1.1102230246251565e-16;
  const double shift = 11.0 * ((double)n * k + (double)k * (k + 1)) * u * (double)k;
  // a column with less than 1% of its (unit) norm outside the span of the earlier ones is replaced:
  // it adds next to no new direction, and keeping it would leave the block so ill-conditioned that
  // plain passes could break down
  const double dead_thresh = std::max(2.0 * std::sqrt(shift), 1e-2);
  // shifted Cholesky of the Gram matrix of Y: its pivots flag the dependent columns (returns how many)
  auto find_dead = [&](unsigned fill_seed, bool refill) {
    tc_launch(c, Prec::F64, gemm_desc('T', 'N', k, k, n, n, n, k), Y, Y, w.G.as<double>(), s);
    chol_inv(w.G.as<double>(), k, shift, w.Rinv.as<double>(), w.info.as<int>(), w.res.as<double>(), s);
    c->read_async(piv.data(), w.res.ptr, (size_t)k * 8);
    c->sync();
    int ndead = 0;
    for (int j = 0; j < k; ++j) {
      dead[j] = !(piv[j] > dead_thresh);
      ndead += dead[j];
    }
    if (ndead > 0 && refill) {
      c->write_async(w.info.ptr, dead.data(), (size_t)k * sizeof(int));
      k_random_fill_flagged(Y, n, k, w.info.as<int>(), fill_seed, s);
      k_col_norms(Y, n, k, w.nrm.as<double>(), s);
      k_scale_cols(Y, n, k, w.nrm.as<double>(), 1, s);
    }
    return ndead;
  };
  // Plain CholeskyQR as described above, then the shifted pass (round 0) or the refill of dependent columns
  // (round 1), each followed by the plain pass again.  What still fails takes sCholQR3 below.
  for (int round = 0; round < 3; ++round) {
    double* scal = w.scal.as<double>();   // [0] smallest pivot, [1] breakdown column, [2] |X^T X - I|_F^2
    tc_launch(c, Prec::F64, gemm_desc('T', 'N', k, k, n, n, n, k), Y, Y, w.G.as<double>(), s);
    chol_inv(w.G.as<double>(), k, 0.0, w.Rinv.as<double>(), w.info.as<int>(), nullptr, s, scal, true);
    tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, k, k, n, k, n), Y, w.Rinv.as<double>(), X, s);
    if (!light) {
      tc_launch(c, Prec::F64, gemm_desc('T', 'N', k, k, n, n, n, k), X, X, w.H.as<double>(), s);
      hipLaunchKernelGGL(gram_dev_kernel, dim3(1), dim3(GD_NT), 0, s, w.H.as<double>(), k, scal + 2);
      TNAD_HIP_TRY(hipGetLastError());
    }
    double hs[3] = {0.0, 0.0, 0.0};   // smallest pivot, breakdown column, |X^T X - I|_F^2
    c->read_async(hs, scal, (light ? 2 : 3) * sizeof(double));
    c->sync();
    int info = (int)hs[1];
    const double dev = std::sqrt(hs[2]);
    if (round == 0 && info == -1 && range) {
      *range = true;
      return;
    }
    if (std::getenv("TNAD_DEBUG_EIG"))
      std::fprintf(stderr, "[tnad eig] plain Cholesky info=%d min pivot=%.3e |X^T X - I|_F=%.3e\n", info, hs[0], dev);
    if (info == 0 && hs[0] > 1e-6 && dev <= 1e-2) {
      if (light || dev <= 1e-12) return;
      if (dev <= 1e-5) {
        // X^T X = I + E with |E|_F <= 1e-5: X F with F = (I + E)^{-1/2} to second order is orthonormal to
        // O(|E|^3) (below 1e-15) and spans the same columns, which is all the iteration keeps; it takes
        // two small products instead of a second Cholesky and its host check
        tc_launch(c, Prec::F64, gemm_desc('N', 'N', k, k, k, k, k, k), w.H.as<double>(), w.H.as<double>(),
                  w.Rinv.as<double>(), s);
        hipLaunchKernelGGL(inv_sqrt2_coef_kernel, dim3((k * k + 255) / 256), dim3(256), 0, s, w.H.as<double>(),
                           w.Rinv.as<double>(), k, w.Rinv.as<double>());
        TNAD_HIP_TRY(hipGetLastError());
        tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, k, k, n, k, n), X, w.Rinv.as<double>(), Y, s);
        k_copy(Y, X, (size_t)n * k, s);
        return;
      }
      chol_inv(w.H.as<double>(), k, 0.0, w.Rinv.as<double>(), w.info.as<int>(), nullptr, s);
      c->read_async(&info, w.info.ptr, sizeof(int));
      c->sync();
      if (info != 0)   // breakdown (pivot <= 0): factor the shifted Gram instead
        chol_inv(w.H.as<double>(), k, shift, w.Rinv.as<double>(), w.info.as<int>(), nullptr, s);
      tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, k, k, n, k, n), X, w.Rinv.as<double>(), Y, s);
      k_copy(Y, X, (size_t)n * k, s);
      return;
    }
    if (round == 2) break;
    if (round == 0) {   // ill-conditioned: the shifted factor of the same Gram matrix, columns back to unit norm
      chol_inv(w.G.as<double>(), k, shift, w.Rinv.as<double>(), w.info.as<int>(), nullptr, s, nullptr, true);
      tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, k, k, n, k, n), Y, w.Rinv.as<double>(), X, s);
      k_copy(X, Y, (size_t)n * k, s);
      k_normalize_cols(Y, n, k, w.nrm.as<double>(), 1e-13, seed + 104729u, s);
      continue;
    }
    const int ndead = find_dead(seed + 7919u, true);
    if (std::getenv("TNAD_DEBUG_EIG"))
      std::fprintf(stderr, "[tnad eig] shifted CholeskyQR: %d dependent columns refilled\n", ndead);
    if (ndead == 0) break;   // ill-conditioned without dependent columns: sCholQR3
  }
  // the Cholesky factor used below must belong to the block as it finally is: the last attempt
  // factors without refilling afterwards
  for (int attempt = 0;; ++attempt) {
    const int ndead = find_dead(seed + 7919u * (attempt + 2), attempt < 3);
    if (std::getenv("TNAD_DEBUG_EIG"))
      std::fprintf(stderr, "[tnad eig] shifted CholeskyQR attempt %d: %d dependent columns\n", attempt, ndead);
    if (ndead == 0 || attempt == 3) break;
  }
  dbg_finite(c, "shifted Rinv", w.Rinv.as<double>(), (size_t)k * k);
  tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, k, k, n, k, n), Y, w.Rinv.as<double>(), X, s);
  double* src = X;
  double* dst = Y;
  for (int pass = 1; pass < 3; ++pass) {
    tc_launch(c, Prec::F64, gemm_desc('T', 'N', k, k, n, n, n, k), src, src, w.G.as<double>(), s);
    chol_inv(w.G.as<double>(), k, 0.0, w.Rinv.as<double>(), w.info.as<int>(), nullptr, s);
    int info = 0;
    c->read_async(&info, w.info.ptr, sizeof(int));
    c->sync();
    if (info != 0)   // breakdown (pivot <= 0): factor the shifted Gram instead
      chol_inv(w.G.as<double>(), k, shift, w.Rinv.as<double>(), w.info.as<int>(), nullptr, s);
    dbg_finite(c, "plain pass Rinv", w.Rinv.as<double>(), (size_t)k * k);
    tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, k, k, n, k, n), src, w.Rinv.as<double>(), dst, s);
    std::swap(src, dst);
  }
  // passes alternate X -> Y -> X: the orthonormal block ends in X (Y is scratch)
}

// the power of two that brings the largest entry of A into [1, 2) when that lies outside 2^-300 .. 2^300, else 1
static double unit_scale(Ctx* c, const double* A, size_t nn, EigWork& w) {
  double* top = w.scal.as<double>() + 8;
  k_fill(top, 1, 0.0, c->stream);
  hipLaunchKernelGGL(max_bits_kernel, dim3(256), dim3(NT), 0, c->stream, A, nn, reinterpret_cast<unsigned long long*>(top));
  TNAD_HIP_TRY(hipGetLastError());
  double mx = 0.0;
  c->read_async(&mx, top, sizeof(double));
  c->sync();
  if (!(mx > 0.0) || !std::isfinite(mx)) return 1.0;
  const int ex = std::ilogb(mx);
  return std::abs(ex) > 300 ? std::ldexp(1.0, -std::max(-1020, std::min(ex, 1020))) : 1.0;
}

EigWork::EigWork(Ctx* c, int n, int k)
    : Y(c, (size_t)n * k * 8), Xr(c, (size_t)n * k * 8), Yr(c, (size_t)n * k * 8), H(c, (size_t)k * k * 8),
      W(c, (size_t)k * k * 8), Vw(c, syev_dc_work_doubles(k) * 8), G(c, (size_t)k * k * 8), Rinv(c, (size_t)k * k * 8),
      nrm(c, (size_t)k * 8), res(c, (size_t)(k + 2) * 8), info(c, (size_t)k * sizeof(int) + 16), scal(c, 16 * 8) {}

int topk_eig(Ctx* c, const double* A, int n, int want, int k, const double* X0, int maxit, double tol,
             double* X, double* AX, double* theta, EigStats* st, EigPlan* plan) {
  hipStream_t s = c->stream;
  if (n <= JACOBI_MAX) {
    // full spectrum: exact reference semantics (all n singular values / vectors), by divide and conquer
    // (2-3.5x faster than Jacobi sweeps to convergence at n = 40..192)
    DevBuf Vw(c, syev_dc_work_doubles(n) * 8);
    syev_dc(A, n, n, theta, X, Vw.as<double>(), s);
    tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, n, n, n, n, n), A, X, AX, s);
    if (st) { st->iters = 1; st->k = n; st->resid = 0.0; }
    return n;
  }
  k = eig_block_width(n, want, k);
  // the entry points reject want > JACOBI_MAX for n > JACOBI_MAX (tnad_limits.h); the residual kernel and the
  // status transfer below are sized by want and need want <= k
  if (want < 1 || want > k) throw Error(TNAD_ERR_UNSUPPORTED, "eigensolver: kept block wider than 192");
  EigWork w(c, n, k);
  // starting block: the previous step's Ritz vectors, or a random one (its columns' norms lie within a few per
  // cent of each other, and only its span counts: it needs no orthonormalisation)
  auto start_block = [&] {
    if (X0) k_copy(X0, X, (size_t)n * k, s);
    else k_random_matrix(X, (size_t)n * k, 0x1234567u, s);
  };
  start_block();
  if (maxit < 2) {   // the Rayleigh-Ritz step comes at once: it needs an orthonormal block
    k_copy(X, w.Y.as<double>(), (size_t)n * k, s);
    orthonormalize(c, w.Y.as<double>(), n, k, X, w, 0x9e3779b9u);
  }
  std::vector<double> hres(k + 2), hth(k);
  // opt-in trace of the iteration (TNAD_DEBUG_EIG=1), to stderr
  static const bool dbg = [] {
    const char* e = std::getenv("TNAD_DEBUG_EIG");
    return e && *e && *e != '0';
  }();
  // Orthogonal iteration X <- orth(A X), with a Rayleigh-Ritz step only where the kept residual is expected to
  // have reached tol: the span after p products is the same whether or not Ritz vectors were formed on
  // the way, and a Rayleigh-Ritz step (0.65 ms of eigensolver at k = 192, two n x k x k products, a host round
  // trip) costs as much as three or four products with their CholeskyQR passes.  The first one comes after the
  // product count that the caller's previous, similar matrix needed (plan), else after the second
  // product; it measures the residual and the rate |theta_k / theta_want| per product, which place the next
  // one.  At chi = 128, D = 4: ~6 Rayleigh-Ritz steps per eigenproblem before, 1 to 2 now.
  int it = 0, n_exact = 0, last_rr = 0, best_it = 0;
  int next_rr = 2;
  if (plan && plan->products > 0 && plan->rate > 0.0) {
    int d;   // products to add (or leave out) for this tolerance at that matrix's rate
    if (plan->resid < 3e-15) d = -std::max(1, plan->products / 4);   // rounding level: reached some products earlier
    else d = (int)std::ceil(std::max(-16.0, std::min(16.0, std::log(tol / plan->resid) / std::log(plan->rate))));
    next_rr = std::max(2, plan->products + d);
  }
  next_rr = std::min(next_rr, std::max(maxit, 1));
  double rel = 0.0, best = HUGE_VAL, best_mark = HUGE_VAL, prev_rel = HUGE_VAL, rate = 0.0;
  bool force_exact = false;
  // The Gram matrices hold squares, so a matrix far from order one (below 1e-100, above 1e100: the first product's columns
  // tell) is taken times a power of two, exactly, from there on: Y = scale A X, and theta and A X divided by it at the end.
  double scale = 1.0;
  while (true) {
    tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, k, n, n, n, n, scale), A, X, w.Y.as<double>(), s);   // Y = A X
    ++it;
    if (it < next_rr) {
      bool range = false;
      const bool light = it + 1 < next_rr;
      orthonormalize(c, w.Y.as<double>(), n, k, X, w, 0x51ed2701u + it, light, it == 1 && scale == 1.0 ? &range : nullptr);
      if (range) {
        scale = unit_scale(c, A, (size_t)n * n, w);
        if (scale != 1.0) {
          start_block();
          it = 0;
        } else {   // only null columns
          orthonormalize(c, w.Y.as<double>(), n, k, X, w, 0x51ed2701u + it, light);
        }
      }
      continue;
    }
    // Rayleigh-Ritz: H = X^T Y ; H = W diag(theta) W^T ; Xr = X W ; Yr = Y W.  One product after the last
    // Ritz basis (H nearly diagonal) a few rotations of near-degenerate pairs plus second-order perturbation
    // theory (ritz_select) may stand in for the eigendecomposition of H; otherwise H is decomposed exactly,
    // by divide and conquer: after products without a Rayleigh-Ritz step between (there the columns mix,
    // and the perturbation theory's remainder, not the span, set the residual: up to 96 products instead of
    // 12 on the 800 x 800 splits of TRG at chi = 20), whenever H is not close enough to diagonal, and
    // whenever the residual stopped falling.  ritz_select's flag gates the exact solver's kernels on the
    // device: no host round trip.
    tc_launch(c, Prec::F64, gemm_desc('T', 'N', k, k, n, n, n, k), X, w.Y.as<double>(), w.H.as<double>(), s);
    dbg_finite(c, "X", X, (size_t)n * k);
    dbg_finite(c, "H", w.H.as<double>(), (size_t)k * k);
    const bool exact_forced = force_exact || last_rr == 0 || it - last_rr > 1;
    int* gate = w.info.as<int>();
    if (!exact_forced) ritz_select(w.H.as<double>(), k, k, want, 1e-2, theta, w.W.as<double>(), gate, s);
    syev_dc(w.H.as<double>(), k, k, theta, w.W.as<double>(), w.Vw.as<double>(), s, exact_forced ? nullptr : gate);
    dbg_finite(c, "W", w.W.as<double>(), (size_t)k * k);
    dbg_finite(c, "theta", theta, (size_t)k);
    tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, k, k, n, k, n), X, w.W.as<double>(), w.Xr.as<double>(), s);
    tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, k, k, n, k, n), w.Y.as<double>(), w.W.as<double>(),
              w.Yr.as<double>(), s);
    hipLaunchKernelGGL(resid_norms_kernel, dim3(want), dim3(NT), 0, s, w.Xr.as<double>(), w.Yr.as<double>(),
                       theta, n, w.res.as<double>(), exact_forced ? nullptr : gate);
    TNAD_HIP_TRY(hipGetLastError());
    c->read_async(hres.data(), w.res.ptr, (size_t)(want + 2) * 8);   // residuals, theta_0, flag
    c->read_async(hth.data(), theta, (size_t)k * 8);
    c->sync();
    const int flag = (int)hres[want + 1];
    const bool exact = flag != 0;   // the exact solver ran (forced, or the selective Rayleigh-Ritz declined)
    n_exact += exact;
    double mx = 0.0;
    bool nan = false;   // (the maximum passes over a NaN)
    for (int j = 0; j < want; ++j) {
      mx = std::max(mx, hres[j]);
      nan |= hres[j] != hres[j];
    }
    rel = mx / std::max(std::fabs(hth[0]), 1e-300);
    if (dbg)
      std::fprintf(stderr, "[tnad eig] n=%d k=%d want=%d it=%d rel_resid=%.3e theta0=%.6e rr=%s(%d)\n", n, k, want,
                   it, rel, hth[0], exact ? "exact" : "select", exact_forced ? -1 : flag);
    if (nan || !(rel == rel)) throw Error(TNAD_ERR_NAN, "eigensolver: NaN in Ritz residual");
    // residual ratio per product: observed between two Rayleigh-Ritz steps, else the guard's edge over the
    // last kept value
    rate = std::fabs(hth[k - 1]) / std::max(std::fabs(hth[want - 1]), 1e-300);
    if (last_rr > 0 && prev_rel > 0.0 && rel > 0.0) rate = std::pow(rel / prev_rel, 1.0 / (it - last_rr));
    rate = std::max(1e-3, std::min(0.9, rate));
    force_exact = last_rr > 0 && !(rel < 0.9 * prev_rel);
    prev_rel = rel;
    last_rr = it;
    if (rel <= tol || it >= maxit) break;
    // stagnation at the rounding level: no halving of the best residual in 8 iterations
    if (rel < best) { if (rel < 0.5 * best_mark) { best_mark = rel; best_it = it; } best = rel; }
    if (best < 1e3 * tol && it - best_it >= 8) break;
    // (bounded before the conversion: the quotient is infinite when tol / rel underflows)
    const int ahead = (int)std::ceil(std::max(1.0, std::min(std::log(tol / rel) / std::log(rate), 16.0)));
    next_rr = std::min(maxit, it + ahead);
    hipLaunchKernelGGL(ritz_scale_kernel, dim3(k), dim3(256), 0, s, w.Xr.as<double>(), w.Yr.as<double>(), theta, n,
                       w.Y.as<double>());
    TNAD_HIP_TRY(hipGetLastError());
    orthonormalize(c, w.Y.as<double>(), n, k, X, w, 0x51ed2701u + it, it + 1 < next_rr);
  }
  // A solve that ended above tol stopped falling (or hit maxit): the products past its best residual bought nothing, so
  // the next one looks where this one's residual last halved, and adds none for the tolerance it cannot reach.
  if (plan) {
    plan->products = rel <= tol ? it : best_it;
    plan->resid = rel <= tol ? rel : tol;
    plan->rate = rate;
  }
  k_copy(w.Xr.as<double>(), X, (size_t)n * k, s);
  if (scale == 1.0) {
    k_copy(w.Yr.as<double>(), AX, (size_t)n * k, s);
  } else {
    k_axpby(1.0 / scale, w.Yr.as<double>(), 0.0, AX, (size_t)n * k, s);
    k_axpby(1.0 / scale, theta, 0.0, theta, k, s);
  }
  hipLaunchKernelGGL(canon_sign_kernel, dim3(k), dim3(NT), 0, s, X, AX, n);
  TNAD_HIP_TRY(hipGetLastError());
  if (st) { st->iters = it; st->k = k; st->resid = rel; st->exact = n_exact; }
  return k;
}

// ==========================================================================
// CTMRG step (src/ctmrg.jl:126-153)
// ==========================================================================
StepTape::StepTape(Ctx* c, const StepDims& d, Prec p, int k)
    : prec(p), k(k), X(c, (size_t)d.n * k * 8), AX(c, (size_t)d.n * k * 8), theta(c, (size_t)k * 8),
      M(c, (size_t)d.n * d.n * 8), X2(c, p, (size_t)d.n * d.n), Y2(c, p, (size_t)d.n * d.n),
      C2(c, (size_t)d.chi * d.chi * 8), T2(c, (size_t)d.chi * d.D * d.chi * 8), nrm(c, 4 * 8) {}

void ctmrg_step(Ctx* c, const StepDims& d, const StepOpts& o, const double* a64, const PBuf& ap,
                const double* C, const double* T, const double* X0, double* X_keep, double* Cout, double* Tout,
                std::vector<double>& vals, StepTape* tape, StepState& state) {
  hipStream_t s = c->stream;
  const int chi = d.chi, D = d.D, n = d.n;
  const long long lc = chi, lD = D;
  const Prec p = o.prec;
  // operands at contraction precision
  PBuf Cq, Tq;
  const void* Cp = as_prec(c, C, (size_t)chi * chi, p, Cq);
  const void* Tp = as_prec(c, T, (size_t)chi * D * chi, p, Tq);
  PBuf X1(c, p, (size_t)n * chi);
  PBuf X2tmp;
  PBuf* X2 = tape ? &tape->X2 : nullptr;
  if (!X2) { X2tmp = PBuf(c, p, (size_t)n * n); X2 = &X2tmp; }
  PBuf cp(c, p, (size_t)n * n);
  // cp = ein"ad,iba,dcl,jkcb -> ijlk"(C, T, T, a)          (src/ctmrg.jl:130)
  tc(c, p, cm("iba", {lc, lD, lc}), Tp, cm("ad", {lc, lc}), Cp, cm("ibd", {lc, lD, lc}), X1.ptr());
  tc(c, p, cm("ibd", {lc, lD, lc}), X1.ptr(), cm("dcl", {lc, lD, lc}), Tp, cm("ibcl", {lc, lD, lD, lc}), X2->ptr());
  tc(c, p, cm("ibcl", {lc, lD, lD, lc}), X2->ptr(), cm("jkcb", {lD, lD, lD, lD}), ap.ptr(),
     cm("ijlk", {lc, lD, lc, lD}), cp.ptr());
  // cpmat = reshape(cp, n, n); cpmat += cpmat'                (src/ctmrg.jl:134-135)
  DevBuf Mtmp;
  double* M = tape ? tape->M.as<double>() : nullptr;
  if (!M) { Mtmp = DevBuf(c, (size_t)n * n * 8); M = Mtmp.as<double>(); }
  if (p == Prec::F64) k_sym_add(cp.b.as<double>(), n, M, s);
  else k_sym_add(cp.b.as<float>(), n, M, s);
  // u, s, v = svd(cpmat) -> top-k eigenpairs by |lambda|        (src/ctmrg.jl:136)
  // block size: n (full spectrum) or 2.25 chi guard-extended (eig_block if set), capped at 192
  const int kreq = step_k(d, o);
  DevBuf Xtmp, AXtmp, thtmp;
  double *X = nullptr, *AX = nullptr, *theta = nullptr;
  if (tape) { X = tape->X.as<double>(); AX = tape->AX.as<double>(); theta = tape->theta.as<double>(); }
  else {
    Xtmp = DevBuf(c, (size_t)n * kreq * 8); AXtmp = DevBuf(c, (size_t)n * kreq * 8); thtmp = DevBuf(c, kreq * 8);
    X = Xtmp.as<double>(); AX = AXtmp.as<double>(); theta = thtmp.as<double>();
  }
  EigStats est;
  const bool warm = X0 != nullptr && n > JACOBI_MAX;
  c->mark(4);
  int k = topk_eig(c, M, n, chi, kreq, warm ? X0 : nullptr, warm ? o.eig_warm_iters : o.eig_max_iters,
                   p == Prec::F64 ? o.eig_tol : o.eig_tol_low, X, AX, theta, &est, &state.plan);
  c->mark(5);
  state.k = k;
  if (X_keep) k_copy(X, X_keep, (size_t)n * k, s);
  state.eig_iters = est.iters;
  state.eig_resid = est.resid;
  // z = reshape(u[:, 1:chi], chi, D, chi)                        (src/ctmrg.jl:137)
  const double* z = X;   // first chi columns
  // C' + C'^T = z^T (cpmat + cpmat^T) z  (src/ctmrg.jl:139,145), FP64
  double* C2 = tape ? tape->C2.as<double>() : nullptr;
  DevBuf C2tmp;
  if (!C2) { C2tmp = DevBuf(c, (size_t)chi * chi * 8); C2 = C2tmp.as<double>(); }
  tc_launch(c, Prec::F64, gemm_desc('T', 'N', chi, chi, n, n, n, chi), z, AX, C2, s);
  // T' = ein"abjcd,abi,dck -> ijk"(tp, z, z), tp = ein"iam,jkla -> ijklm"(T, a)  (src/ctmrg.jl:131,140)
  // evaluated as ((T z) a) z without materialising tp.
  PBuf zq;
  const void* zp = as_prec(c, z, (size_t)n * chi, p, zq);
  PBuf Y1(c, p, (size_t)n * n);
  PBuf Y2tmp;
  PBuf* Y2 = tape ? &tape->Y2 : nullptr;
  if (!Y2) { Y2tmp = PBuf(c, p, (size_t)n * n); Y2 = &Y2tmp; }
  PBuf T1p(c, p, (size_t)chi * D * chi);
  tc(c, p, cm("aed", {lc, lD, lc}), Tp, cm("abx", {lc, lD, lc}), zp, cm("edbx", {lD, lc, lD, lc}), Y1.ptr());
  tc(c, p, cm("edbx", {lD, lc, lD, lc}), Y1.ptr(), cm("bjce", {lD, lD, lD, lD}), ap.ptr(),
     cm("dcxj", {lc, lD, lc, lD}), Y2->ptr());
  tc(c, p, cm("dcxj", {lc, lD, lc, lD}), Y2->ptr(), cm("dcy", {lc, lD, lc}), zp, cm("xjy", {lc, lD, lc}), T1p.ptr());
  double* T2 = tape ? tape->T2.as<double>() : nullptr;
  DevBuf T2tmp;
  if (!T2) { T2tmp = DevBuf(c, (size_t)chi * D * chi * 8); T2 = T2tmp.as<double>(); }
  // edge += ein"ijk -> kji"(conj(edge)); corner /= norm(corner); edge /= norm(edge)   (src/ctmrg.jl:146-150)
  DevBuf red(c, 512 * 8), nr(c, 4 * 8);
  double* nrm = tape ? tape->nrm.as<double>() : nr.as<double>();
  if (p == Prec::F64) k_step_end(T1p.b.as<double>(), chi, D, C2, T2, red.as<double>(), nrm, Cout, Tout, s);
  else k_step_end(T1p.b.as<float>(), chi, D, C2, T2, red.as<double>(), nrm, Cout, Tout, s);
  if (tape) tape->eig_tol = p == Prec::F64 ? o.eig_tol : o.eig_tol_low;
  // vals = s ./ s[1]   (src/ctmrg.jl:142).  With the whole spectrum computed (n <= 192) all n
  // values; otherwise the k largest (the chi kept values, resolved to the eigensolver tolerance, and the
  // guard block's Ritz values, which are not), with the rest 0.  For n > 192 the step also measures the
  // norm of the spectrum beyond the kept chi values, rest = |M - Z Theta Z^T|_F / s[1] (Z the kept
  // eigenvectors): formed elementwise, it is accurate to ~n eps |M|_F even where rest is far below
  // sqrt(eps) (|M|_F^2 - sum theta^2 would lose it to cancellation).  The stop test uses it as a lower
  // bound on the change of the discarded values (run_ctmrg).
  const int nv = k;
  std::vector<double> th(nv);
  double sq[2] = {0.0, 0.0};
  DevBuf E, XT, sqd;
  if (n > JACOBI_MAX) {
    XT = DevBuf(c, (size_t)n * chi * 8);
    E = DevBuf(c, (size_t)n * n * 8);
    sqd = DevBuf(c, 2 * 8);
    k_scale_cols_to(X, n, chi, theta, XT.as<double>(), s);
    tc_launch(c, Prec::F64, gemm_desc('N', 'T', n, n, chi, n, n, n), XT.as<double>(), X, E.as<double>(), s);
    k_diff_sumsq(M, E.as<double>(), (size_t)n * n, red.as<double>(), sqd.as<double>(), s);
    c->read_async(sq, sqd.ptr, 2 * 8);
  }
  c->read_async(th.data(), theta, (size_t)nv * 8);
  c->sync();
  state.eig_ms = c->elapsed(4, 5);
  vals.assign(n, 0.0);
  double s0 = std::fabs(th[0]);
  for (int i = 0; i < nv; ++i) vals[i] = std::fabs(th[i]) / s0;
  for (int i = 0; i < nv; ++i)
    if (!(vals[i] == vals[i])) throw Error(TNAD_ERR_NAN, "ctmrgstep: NaN in singular values");
  if (n > JACOBI_MAX) {
    state.rest = std::sqrt(sq[0]) / s0;
    // rounding of the n^2 entries of E and of its sum (~n eps |M|_F), plus the kept residuals R = M Z - Z Theta:
    // |E - E_exact|_F <= sqrt(2) |R|_F <= sqrt(2 chi) max_j |r_j| (Mirsky)
    state.rest_err = (double)n * 2.3e-16 * std::sqrt(sq[1]) / s0 + std::sqrt(2.0 * chi) * est.resid;
    if (!(state.rest == state.rest)) throw Error(TNAD_ERR_NAN, "ctmrgstep: NaN in the discarded spectrum");
  }
}

// ==========================================================================
// Eigen adjoint: cotangent of z = U[:, 1:chi] (plus the C' chain's C1bar)
// -> cotangent of cpmat, i.e. svd_back (src/trg.jl:72-106) with dU nonzero in
// the first chi columns, dS = dV = nothing, followed by cpmat += cpmat'.
//
//   cpbar = W U1^T + U1 W^T,  W = U1 Kt/2 + (X_c Lambda1 + A X_c)
//
// Kt/2 holds the pairs among the kept chi eigenvectors (reference formula
// verbatim).  Every other eigenpair i contributes g_ij / (lambda_j - lambda_i)
// along u_i, i.e. (lambda_j - A)^-1 = (lambda_j + A)(lambda_j^2 - A^2)^-1 on the
// complement of the kept vectors: X_c solves (lambda_j^2 - A^2) x_j = P G_j there
// (resolvent_pcg, preconditioned by the extra Ritz pairs the eigensolver carries).
// With the whole spectrum known (n <= 192) those contributions are a coefficient
// each, in rows chi..n-1 of the coefficient block: W = U Kf over all n vectors, no
// solve (28 launches and two host round trips fewer per step).
// ==========================================================================
void eig_adjoint(Ctx* c, const StepDims& d, const StepTape& tp, const double* G, const double* C1bar,
                 double* cpbar, EigBackStats* st, double* sweep_ref) {
  hipStream_t s = c->stream;
  const int chi = d.chi, n = d.n, k = tp.k;
  const double* X = tp.X.as<double>();
  const double* lam = tp.theta.as<double>();
  const int rows = k == n ? n : chi;   // the vectors that enter by coefficients: all of them when all are known
  DevBuf g(c, (size_t)rows * chi * 8), coef(c, (size_t)rows * chi * 8), W(c, (size_t)n * chi * 8);
  // g = U^T G  (rows x chi)
  tc_launch(c, Prec::F64, gemm_desc('T', 'N', rows, chi, n, n, n, rows), X, G, g.as<double>(), s);
  hipLaunchKernelGGL(eigback_coef_kernel, dim3((rows * chi + NT - 1) / NT), dim3(NT), 0, s, g.as<double>(), lam,
                     C1bar, chi, rows, 1e-40, coef.as<double>());
  TNAD_HIP_TRY(hipGetLastError());
  // W = U coef  (n x rows . rows x chi)
  tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, chi, rows, n, rows, n), X, coef.as<double>(), W.as<double>(), s);
  int iters = 0;
  if (n > rows) {
    DevBuf sq(c, (size_t)k * 8), Xc(c, (size_t)n * chi * 8), AXc(c, (size_t)n * chi * 8),
        tmp(c, (size_t)n * chi * 8);
    k_square(lam, sq.as<double>(), k, s);
    const double* M = tp.M.as<double>();
    auto applyA2 = [&](const double* V, double* out, int nc) {
      tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, nc, n, n, n, n), M, V, tmp.as<double>(), s);
      tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, nc, n, n, n, n), M, tmp.as<double>(), out, s);
    };
    // A step computed with low-precision contractions resolved its eigenpairs only to the relative
    // residual its contractions can support (1e-8 and above), so this adjoint is no more accurate
    // than that whatever the solve does: its complement part is solved to 1e-6 instead of 1e-13, and
    // no further than 1e-13 of the reverse sweep's largest right-hand side (the early steps of a
    // converging CTMRG receive cotangents many orders smaller than the last ones, so that bound is the
    // one that holds their error down).  The same holds for an FP64 step whose eigensolver ran to a
    // looser residual than 1e-13 (the mixed path ties it to the step-to-step change).  At chi = 128,
    // D = 4 the relative bar at 1e-6 instead of 1e-8 cut the reverse sweep from 11.2 to 10.2 ms with the
    // gradient unchanged (relative difference to the FP64 path 4.8e-9 either way).
    const bool low = tp.prec != Prec::F64;
    const bool loose = low || tp.eig_tol > 1e-13;
    const double pcg_tol = loose ? 1e-6 : 1e-13;
    iters = resolvent_pcg(c, n, chi, k, X, sq.as<double>(), sq.as<double>() + chi, applyA2, G, Xc.as<double>(),
                          pcg_tol, 200, 1e-40, sweep_ref, loose ? 1e-13 : 0.0);
    static const bool dbg = [] {
      const char* e = std::getenv("TNAD_DEBUG_EIG");
      return e && *e && *e != '0';
    }();
    if (dbg)
      std::fprintf(stderr, "[tnad eig] adjoint n=%d chi=%d prec=%s eig_tol=%.1e: %d resolvent CG iterations (tol %.1e)\n",
                   n, chi, low ? "low" : "fp64", tp.eig_tol, iters, pcg_tol);
    // W += X_c Lambda1 + A X_c
    tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, chi, n, n, n, n), M, Xc.as<double>(), AXc.as<double>(), s);
    hipLaunchKernelGGL(add_lam_cols_kernel, dim3(nb((size_t)n * chi)), dim3(NT), 0, s, W.as<double>(),
                       Xc.as<double>(), AXc.as<double>(), lam, n, chi);
    TNAD_HIP_TRY(hipGetLastError());
  }
  // cpbar = W U1^T + U1 W^T
  tc_launch(c, Prec::F64, gemm_desc('N', 'T', n, n, chi, n, n, n), W.as<double>(), X, cpbar, s);
  tc_launch(c, Prec::F64, gemm_desc('N', 'T', n, n, chi, n, n, n, 1.0, 1.0), X, W.as<double>(), cpbar, s);
  if (st) st->pcg_iters = iters;
}

// ==========================================================================
// Reverse sweep of one ctmrgstep.  In: cotangents of the step outputs
// (C3bar, T3bar).  Out: cotangents of the step inputs (Cbar, Tbar) and the
// bulk contribution added into abar.
// ==========================================================================
void ctmrg_step_back(Ctx* c, const StepDims& d, Prec p, const StepTape& tp, const double* a64, const PBuf& ap,
                     const double* C3bar, const double* T3bar, double* Cbar, double* Tbar, double* abar,
                     double* sweep_ref) {
  hipStream_t s = c->stream;
  const int chi = d.chi, D = d.D, n = d.n;
  const long long lc = chi, lD = D;
  const size_t nC = (size_t)chi * chi, nT = (size_t)chi * D * chi, nA = (size_t)D * D * D * D;
  // --- adjoints of the normalisation and the symmetrisation (src/autodiff.jl:23-29) ---------
  DevBuf red(c, 512 * 8), C1bar(c, nC * 8), T1bar(c, nT * 8);
  k_step_end_back(tp.C2.as<double>(), C3bar, tp.T2.as<double>(), T3bar, chi, D, tp.nrm.as<double>(), red.as<double>(),
                  C1bar.as<double>(), T1bar.as<double>(), s);

  // tape intermediates stored at the forward step's precision, converted to the sweep's
  PBuf Y2tmp, X2tmp;
  const PBuf& Y2 = at_prec(c, tp.Y2, p, Y2tmp);
  const PBuf& X2 = at_prec(c, tp.X2, p, X2tmp);
  // --- T' chain adjoint (tp never materialised) ----------------------------
  // (an FP64 sweep uses the tape's tensors and accumulates into the results in place)
  const bool f64 = p == Prec::F64;
  PBuf T1q, zq, Tq, Cq;
  const void* T1b = as_prec(c, T1bar.as<double>(), nT, p, T1q);
  const void* zp = as_prec(c, tp.X.as<double>(), (size_t)n * chi, p, zq);   // first n*chi entries = z
  const void* Tp = as_prec(c, tp.T.as<double>(), nT, p, Tq);
  const void* Cp = as_prec(c, tp.C.as<double>(), nC, p, Cq);
  PBuf P1(c, p, (size_t)n * n), Q1(c, p, (size_t)n * n), S1(c, p, (size_t)n * n);
  DevBuf zbar(c, (size_t)n * chi * 8), Tacc, a_acc;
  PBuf Tbq, abq, zbq;
  if (!f64) {
    Tbq = PBuf(c, p, nT);
    abq = PBuf(c, p, nA);
    zbq = PBuf(c, p, (size_t)n * chi);
    Tacc = DevBuf(c, nT * 8);
    a_acc = DevBuf(c, nA * 8);
  }
  void* Tbp = f64 ? (void*)Tbar : Tbq.ptr();
  void* abp = f64 ? (void*)abar : abq.ptr();
  void* zbp = f64 ? zbar.ptr : zbq.ptr();
  const double acc = f64 ? 1.0 : 0.0;   // abar: added by the contraction itself, or from its own buffer below
  // P1[a,b,j,y] = sum_x z[a,b,x] T1bar[x,j,y]
  tc(c, p, cm("abx", {lc, lD, lc}), zp, cm("xjy", {lc, lD, lc}), T1b, cm("abjy", {lc, lD, lD, lc}),
     P1.ptr());
  // Q1[a,e,c,y] = sum_{b,j} P1[a,b,j,y] a[b,j,c,e] ; Tbar[a,e,d] = sum_{c,y} Q1[a,e,c,y] z[d,c,y]
  tc(c, p, cm("abjy", {lc, lD, lD, lc}), P1.ptr(), cm("bjce", {lD, lD, lD, lD}), ap.ptr(),
     cm("aecy", {lc, lD, lD, lc}), Q1.ptr());
  tc(c, p, cm("aecy", {lc, lD, lD, lc}), Q1.ptr(), cm("dcy", {lc, lD, lc}), zp, cm("aed", {lc, lD, lc}),
     Tbp);
  // S1[a,e,c,y] = sum_d T[a,e,d] z[d,c,y] ; abar[b,j,c,e] = sum_{a,y} P1[a,b,j,y] S1[a,e,c,y]
  tc(c, p, cm("aed", {lc, lD, lc}), Tp, cm("dcy", {lc, lD, lc}), zp, cm("aecy", {lc, lD, lD, lc}),
     S1.ptr());
  tc(c, p, cm("abjy", {lc, lD, lD, lc}), P1.ptr(), cm("aecy", {lc, lD, lD, lc}), S1.ptr(),
     cm("bjce", {lD, lD, lD, lD}), abp, 1.0, acc);
  // U1[a,b,j,y] = sum_{e,c} S1[a,e,c,y] a[b,j,c,e] (reuses P1) ; zbar[a,b,x] = sum_{j,y} U1 T1bar[x,j,y]
  tc(c, p, cm("aecy", {lc, lD, lD, lc}), S1.ptr(), cm("bjce", {lD, lD, lD, lD}), ap.ptr(),
     cm("abjy", {lc, lD, lD, lc}), P1.ptr());
  tc(c, p, cm("abjy", {lc, lD, lD, lc}), P1.ptr(), cm("xjy", {lc, lD, lc}), T1b, cm("abx", {lc, lD, lc}),
     zbp);
  // zbar[d,c,y] += sum_{x,j} Y2[d,c,x,j] T1bar[x,j,y]
  tc(c, p, cm("dcxj", {lc, lD, lc, lD}), Y2.ptr(), cm("xjy", {lc, lD, lc}), T1b, cm("dcy", {lc, lD, lc}),
     zbp, 1.0, 1.0);
  if (!f64) {
    from_prec(c, zbq, zbar.as<double>());
    from_prec(c, abq, a_acc.as<double>());
    k_axpby(1.0, a_acc.as<double>(), 1.0, abar, nA, s);
    from_prec(c, Tbq, Tacc.as<double>());
  }

  // --- C' chain: zbar += (cpmat + cpmat') z C1bar  (FP64; A z kept from the forward)
  tc_launch(c, Prec::F64, gemm_desc('N', 'N', n, chi, chi, n, chi, n, 1.0, 1.0), tp.AX.as<double>(),
            C1bar.as<double>(), zbar.as<double>(), s);

  // --- eigen adjoint -> cpbar (n x n, FP64) ---------------------------------
  DevBuf cpbar(c, (size_t)n * n * 8);
  eig_adjoint(c, d, tp, zbar.as<double>(), C1bar.as<double>(), cpbar.as<double>(), nullptr, sweep_ref);

  // --- cp chain adjoint -----------------------------------------------------
  PBuf cpq, X2b(c, p, (size_t)n * n), X1(c, p, (size_t)n * chi), X1b(c, p, (size_t)n * chi);
  const void* cpb = as_prec(c, cpbar.as<double>(), (size_t)n * n, p, cpq);
  PBuf Cbq;
  if (!f64) Cbq = PBuf(c, p, nC);
  void* Cbp = f64 ? (void*)Cbar : Cbq.ptr();
  // X1 = T C (recomputed)
  tc(c, p, cm("iba", {lc, lD, lc}), Tp, cm("ad", {lc, lc}), Cp, cm("ibd", {lc, lD, lc}), X1.ptr());
  // X2bar[i,b,c,l] = sum_{j,k} cpbar[i,j,l,k] a[j,k,c,b]
  tc(c, p, cm("ijlk", {lc, lD, lc, lD}), cpb, cm("jkcb", {lD, lD, lD, lD}), ap.ptr(), cm("ibcl", {lc, lD, lD, lc}),
     X2b.ptr());
  // abar[j,k,c,b] += sum_{i,l} cpbar[i,j,l,k] X2[i,b,c,l]
  tc(c, p, cm("ijlk", {lc, lD, lc, lD}), cpb, cm("ibcl", {lc, lD, lD, lc}), X2.ptr(), cm("jkcb", {lD, lD, lD, lD}), abp,
     1.0, acc);
  if (!f64) {
    from_prec(c, abq, a_acc.as<double>());
    k_axpby(1.0, a_acc.as<double>(), 1.0, abar, nA, s);
  }
  // X1bar[i,b,d] = sum_{c,l} X2bar[i,b,c,l] T[d,c,l] ; Tbar[d,c,l] += sum_{i,b} X1[i,b,d] X2bar[i,b,c,l]
  tc(c, p, cm("ibcl", {lc, lD, lD, lc}), X2b.ptr(), cm("dcl", {lc, lD, lc}), Tp, cm("ibd", {lc, lD, lc}), X1b.ptr());
  tc(c, p, cm("ibd", {lc, lD, lc}), X1.ptr(), cm("ibcl", {lc, lD, lD, lc}), X2b.ptr(), cm("dcl", {lc, lD, lc}), Tbp, 1.0,
     acc);
  // Cbar[a,d] = sum_{i,b} T[i,b,a] X1bar[i,b,d] ; Tbar[i,b,a] += sum_d X1bar[i,b,d] C[a,d]
  tc(c, p, cm("iba", {lc, lD, lc}), Tp, cm("ibd", {lc, lD, lc}), X1b.ptr(), cm("ad", {lc, lc}), Cbp);
  tc(c, p, cm("ibd", {lc, lD, lc}), X1b.ptr(), cm("ad", {lc, lc}), Cp, cm("iba", {lc, lD, lc}), Tbp, 1.0, 1.0);
  if (!f64) {
    from_prec(c, Cbq, Cbar);
    from_prec(c, Tbq, Tbar);
    k_axpby(1.0, Tacc.as<double>(), 1.0, Tbar, nT, s);
  }
  (void)a64;
}

// ==========================================================================
// expectationvalue (src/variationalipeps.jl:49-56), FP64, with reverse sweep
// l = ein"ab,ica,bde,cjfdlm,eg,gfk -> ijklm"(C, T, T, ap, C, T)
// ==========================================================================
EvCache::EvCache(Ctx* c, int chi, int D, int ph)
    : apn(c, (size_t)D * D * D * D * ph * ph * 8), E1(c, (size_t)chi * D * chi * 8),
      E2(c, (size_t)chi * D * D * chi * 8), E3(c, (size_t)chi * D * chi * 8),
      E4(c, (size_t)chi * D * chi * D * ph * ph * 8), l(c, (size_t)chi * D * chi * ph * ph * 8),
      tr(c, (size_t)chi * D * chi * 8), scal(c, 8 * 8) {}

void expectation_fwd(Ctx* c, int chi, int D, int ph, const double* h, const double* ap, const double* C,
                     const double* T, EvCache& ev, double* e_host) {
  hipStream_t s = c->stream;
  const long long lc = chi, lD = D, ls = ph;
  const long long n = lc * lD;
  const size_t nap = (size_t)D * D * D * D * ph * ph;
  DevBuf red(c, 300 * 8);
  // ap /= norm(ap)
  k_dot_to(ap, nullptr, nap, red.as<double>(), ev.scal.as<double>() + 3, s);   // |ap|^2
  k_scale_rsqrt(ap, nap, ev.scal.as<double>() + 3, ev.apn.as<double>(), s);
  const Prec F = Prec::F64;
  double* E1 = ev.E1.as<double>();
  double* E2 = ev.E2.as<double>();
  double* E3 = ev.E3.as<double>();
  double* E4 = ev.E4.as<double>();
  double* l = ev.l.as<double>();
  tc(c, F, cm("ica", {lc, lD, lc}), T, cm("ab", {lc, lc}), C, cm("icb", {lc, lD, lc}), E1);
  tc(c, F, cm("icb", {lc, lD, lc}), E1, cm("bde", {lc, lD, lc}), T, cm("icde", {lc, lD, lD, lc}), E2);
  tc(c, F, cm("eg", {lc, lc}), C, cm("gfk", {lc, lD, lc}), T, cm("efk", {lc, lD, lc}), E3);
  // E4[i,j,e,f,l,m] = sum_{c,d} E2[i,c,d,e] ap[c,j,f,d,l,m]  (one launch per physical pair (l,m))
  const long long e4s[4] = {1, lc, n, n * lc};
  for (int lm = 0; lm < ph * ph; ++lm) {
    tc(c, F, cm("icde", {lc, lD, lD, lc}), E2, cm("cjfd", {lD, lD, lD, lD}), ev.apn.as<double>() + (size_t)lm * D * D * D * D,
       with_strides("ijef", {lc, lD, lc, lD}, {e4s[0], e4s[1], e4s[2], e4s[3]}), E4 + (size_t)lm * n * n);
  }
  // l[i,j,k,l,m] = sum_{e,f} E4[i,j,e,f,l,m] E3[e,f,k]
  tc(c, F, with_strides("ijeflm", {lc, lD, lc, lD, ls, ls}, {1, lc, n, n * lc, n * n, n * n * ls}), E4,
     cm("efk", {lc, lD, lc}), E3, cm("ijklm", {lc, lD, lc, ls, ls}), l);
  // e = ein"abcij,abckl,ijkl -> "(l, l, h) ; n = ein"ijkaa,ijkbb -> "(l, l)
  DevBuf Lh(c, (size_t)n * chi * ph * ph * 8);
  tc(c, F, cm("abcij", {lc, lD, lc, ls, ls}), l, cm("ijkl", {ls, ls, ls, ls}), h, cm("abckl", {lc, lD, lc, ls, ls}),
     Lh.as<double>());
  const size_t nl = (size_t)n * chi * ph * ph, m3 = (size_t)n * chi;
  k_dot_to(Lh.as<double>(), l, nl, red.as<double>(), ev.scal.as<double>() + 0, s);   // e
  hipLaunchKernelGGL(trace_last2_kernel, dim3((m3 + NT - 1) / NT), dim3(NT), 0, s, l, (int)m3, ph, ev.tr.as<double>());
  k_dot_to(ev.tr.as<double>(), nullptr, m3, red.as<double>(), ev.scal.as<double>() + 1, s);   // nn
  // scal[5] = e/nn, scal[6] = 1/nn, scal[7] = -e/nn^2
  hipLaunchKernelGGL(energy_scalars_kernel, dim3(1), dim3(1), 0, s, ev.scal.as<double>() + 0,
                     ev.scal.as<double>() + 1, ev.scal.as<double>() + 5);
  TNAD_HIP_TRY(hipGetLastError());
  if (e_host) {
    c->read_async(e_host, ev.scal.as<double>() + 5, 8);
    c->sync();
  }
}

void expectation_back(Ctx* c, int chi, int D, int ph, const double* h, const double* ap, const double* C,
                      const double* T, EvCache& ev, double* apbar, double* Cbar, double* Tbar) {
  hipStream_t s = c->stream;
  const long long lc = chi, lD = D, ls = ph;
  const long long n = lc * lD;
  const size_t nap = (size_t)D * D * D * D * ph * ph;
  const size_t nl = (size_t)n * chi * ph * ph, m3 = (size_t)n * chi;
  const Prec F = Prec::F64;
  double* l = ev.l.as<double>();
  // lbar = ebar (l h^T + l h) + 2 nnbar tr (x) delta
  DevBuf lbar(c, nl * 8), tmp(c, nl * 8), red(c, 300 * 8);
  tc(c, F, cm("abcij", {lc, lD, lc, ls, ls}), l, cm("ijkl", {ls, ls, ls, ls}), h, cm("abckl", {lc, lD, lc, ls, ls}),
     lbar.as<double>());
  tc(c, F, cm("abckl", {lc, lD, lc, ls, ls}), l, cm("ijkl", {ls, ls, ls, ls}), h, cm("abcij", {lc, lD, lc, ls, ls}),
     tmp.as<double>());
  k_axpby(1.0, tmp.as<double>(), 1.0, lbar.as<double>(), nl, s);
  // scale by ebar (device scalar): lbar *= 1/nn  -> use scale_by_dev with nn
  k_scale_by_dev(lbar.as<double>(), nl, ev.scal.as<double>() + 1, s);
  // 2 nnbar = -2 e / nn^2, read on the device
  hipLaunchKernelGGL(add_trace_diag_kernel, dim3((m3 * ph + NT - 1) / NT), dim3(NT), 0, s, lbar.as<double>(),
                     ev.tr.as<double>(), ev.scal.as<double>() + 7, 2.0, (int)m3, ph);
  TNAD_HIP_TRY(hipGetLastError());
  double* E1 = ev.E1.as<double>();
  double* E2 = ev.E2.as<double>();
  double* E3 = ev.E3.as<double>();
  double* E4 = ev.E4.as<double>();
  const TView vE4 = with_strides("ijeflm", {lc, lD, lc, lD, ls, ls}, {1, lc, n, n * lc, n * n, n * n * ls});
  DevBuf E4b(c, (size_t)n * n * ph * ph * 8), E3b(c, (size_t)n * chi * 8), E2b(c, (size_t)n * n * 8),
      E1b(c, (size_t)n * chi * 8), apnb(c, nap * 8);
  tc(c, F, cm("ijklm", {lc, lD, lc, ls, ls}), lbar.as<double>(), cm("efk", {lc, lD, lc}), E3, vE4, E4b.as<double>());
  tc(c, F, vE4, E4, cm("ijklm", {lc, lD, lc, ls, ls}), lbar.as<double>(), cm("efk", {lc, lD, lc}), E3b.as<double>());
  const TView vE4s = with_strides("ijef", {lc, lD, lc, lD}, {1, lc, n, n * lc});
  for (int lm = 0; lm < ph * ph; ++lm) {
    const size_t oa = (size_t)lm * D * D * D * D, oe = (size_t)lm * n * n;
    tc(c, F, vE4s, E4b.as<double>() + oe, cm("cjfd", {lD, lD, lD, lD}), ev.apn.as<double>() + oa,
       cm("icde", {lc, lD, lD, lc}), E2b.as<double>(), 1.0, lm == 0 ? 0.0 : 1.0);
    tc(c, F, cm("icde", {lc, lD, lD, lc}), E2, vE4s, E4b.as<double>() + oe, cm("cjfd", {lD, lD, lD, lD}),
       apnb.as<double>() + oa);
  }
  tc(c, F, cm("icde", {lc, lD, lD, lc}), E2b.as<double>(), cm("bde", {lc, lD, lc}), T, cm("icb", {lc, lD, lc}),
     E1b.as<double>());
  tc(c, F, cm("icb", {lc, lD, lc}), E1, cm("icde", {lc, lD, lD, lc}), E2b.as<double>(), cm("bde", {lc, lD, lc}),
     Tbar, 1.0, 1.0);
  tc(c, F, cm("icb", {lc, lD, lc}), E1b.as<double>(), cm("ab", {lc, lc}), C, cm("ica", {lc, lD, lc}), Tbar, 1.0, 1.0);
  tc(c, F, cm("ica", {lc, lD, lc}), T, cm("icb", {lc, lD, lc}), E1b.as<double>(), cm("ab", {lc, lc}), Cbar, 1.0, 1.0);
  tc(c, F, cm("efk", {lc, lD, lc}), E3b.as<double>(), cm("gfk", {lc, lD, lc}), T, cm("eg", {lc, lc}), Cbar, 1.0, 1.0);
  tc(c, F, cm("eg", {lc, lc}), C, cm("efk", {lc, lD, lc}), E3b.as<double>(), cm("gfk", {lc, lD, lc}), Tbar, 1.0, 1.0);
  // ap /= norm(ap) adjoint
  DevBuf dd(c, 8);
  k_dot_to(ap, apnb.as<double>(), nap, red.as<double>(), dd.as<double>(), s);
  hipLaunchKernelGGL(norm_back_kernel, dim3(nb(nap)), dim3(NT), 0, s, ap, apnb.as<double>(),
                     ev.scal.as<double>() + 3, dd.as<double>(), apbar, nap);
  TNAD_HIP_TRY(hipGetLastError());
}

}  // namespace tnad
