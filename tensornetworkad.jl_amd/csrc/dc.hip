// Dense symmetric eigensolver for m <= 192 (FP64) in four stages, each a HIP kernel:
//
//  * trd_kernel : Householder reduction to tridiagonal form in one workgroup of 32 x 16 threads.  The
//    matrix stays in registers in a cyclic distribution (thread (ty, tx) holds the 6 x 12 elements
//    (ty + 32 a, tx + 16 b)), both triangles, so the product A v of each step is a per-thread partial
//    sum over its twelve columns finished by DPP butterflies across the 16 lanes of the same ty (one
//    row of a wavefront), and the symmetric rank-two update is local.  Per step: p = tau A v through
//    LDS, while the owner lanes of column j + 1 publish it as it stands; after the second barrier every
//    thread updates its elements, and wavefront 0 forms column j + 1 after the update from the published
//    column, v, p and p . v alone, then the next reflector from it, and publishes v and tau (the other
//    wavefronts never repeat its reductions, square root and division); two barriers per step; column
//    blocks that a step cannot touch are not emitted (template block index), finished row blocks are
//    skipped.
//    The reflectors (v with v[j+1] = 1, zeros above) and their tau are written for the back
//    transformation.
//  * dc_kernel : divide and conquer on the tridiagonal matrix T (Cuppen's method), a workgroup for each half of T.  A
//    half is torn recursively down to leaves of one or two rows (solved directly), T = diag(T1, T2) + |b| u u^T with
//    u = e_last + sign(b) e_first, and the tree is merged bottom-up, all merges of a level at once:
//    the children's eigenpairs give D + rho z z^T, z = Q^T u / sqrt 2, rho = 2 |b|; entries with
//    rho |z_i| below 8 eps max(|D|, rho |z|) deflate, and so does one of two entries whose Givens
//    rotation (zeroing one z) perturbs the matrix by less than that (Dongarra-Sorensen deflation);
//    the remaining K roots of the secular equation 1 + rho sum z_i^2 / (d_i - lambda) = 0 are found
//    in parallel, each as an offset tau from its nearer pole (so lambda - d_i is formed without
//    cancellation) by the two-pole rational model of the secular function (Li's "middle way"),
//    safeguarded by bisection on a bracket; z is then recomputed from the roots (Gu-Eisenstat, Lowner's
//    formula), which makes the eigenvectors (zhat_i / (d_i - lambda_j))_i orthogonal to working
//    accuracy; the merged eigenvectors are the children's (block-diagonal) eigenvector matrix times
//    that K x K matrix (deflated columns are copied), on the matrix cores.
//    A level is a chain of latencies, not of work: at m = 96, in one workgroup from single rows up, 325 k cycles, 127 k of
//    them in the roots (four lanes per root, terms reread from LDS in every iteration) and 80 k in products of narrow
//    merges, one output per thread.  Eight lanes per root hold their terms in registers (as many slots as the level needs)
//    and add by DPP (four or sixteen lanes: the same to 3 us more); the vectors are formed where their norms are;
//    every product goes to the matrix cores, a wavefront per 16 x 16 tile; up to 72 rows per half the eigenvector matrices
//    stay in LDS.  Divide and conquer with its top merge's roots, us at m = 48 / 80 / 96 / 128 / 192:
//    105 / 141 / 162 / 185 / 310 before, 51 / 73 / 75 / 82 / 134 now.
//  * dc_top_kernel, dc_sec_kernel, dc_zh_kernel : the merge of the two halves as far as its roots; it stops short of its
//    product: it leaves the children's eigenvectors Z in Qb and its kept poles, roots and recomputed z, since
//    H (Z M) = (H Z) M lets the product with the merge matrix M run over the whole chip.
//  * trd_back_kernel : Z <- H_0 H_1 ... H_(m-3) Z, one wavefront per column of Z (no barriers), four
//    reflectors per wavefront reduction.
//  * dc_final_kernel : W = Z M, a 16 x 16 tile of W per workgroup on the FP64 matrix cores.
// The eigenpairs are then sorted by |lambda| descending with the sign convention of the Jacobi path.
#include "dpp.h"
#include "tnad_internal.h"

#include <cfloat>

namespace tnad {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int TD_GX = 16, TD_GY = 32;       // thread grid: 32 rows x 16 columns of threads (512)
constexpr int TD_NT = TD_GX * TD_GY;
static_assert(TD_GX == 8 || TD_GX == 16 || TD_GX == 32, "row sums span half, one or two DPP rows");
static_assert(JACOBI_MAX % TD_GX == 0 && JACOBI_MAX % TD_GY == 0, "tridiagonalisation tiling");

struct TrdShared {
  double col[2][JACOBI_MAX];   // column j + 1 as it stands before step j's update (double-buffered by parity)
  double v[2][JACOBI_MAX];     // the reflector v (v[j+1] = 1, zeros elsewhere outside j+1..m-1)
  double p[2][JACOBI_MAX];     // tau A v
  double colb[JACOBI_MAX];     // the same for the last step of a column block (column j + 1 in the next block)
  double tv[2];                // tau
  double pp[2][TD_NT / 64];    // per wavefront: its rows' share of p . v
};

// 1 / x from the hardware estimate and two Newton steps (x finite and nonzero)
__device__ __forceinline__ double rcp_nr(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  return fma(r, fma(-x, r, 1.0), r);
}

// sqrt(x) and 1 / sqrt(x) from the hardware estimate, refined to the accuracy of the square root (x normal and positive)
__device__ __forceinline__ double sqrt_nr(double x, double& rs) {
  double y = __builtin_amdgcn_rsq(x);
  y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
  y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
  rs = y;
  const double q = x * y;
  return fma(fma(-q, q, x), 0.5 * y, q);
}

// the value of x in lane k (k uniform)
__device__ __forceinline__ double lane_of(double x, int k) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)b, k), hi = __builtin_amdgcn_readlane((int)(b >> 32), k);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// wavefront 0: the reflector H = I - tau v v^T with v[j+1] = 1 that maps column j's rows j+1.. (c: rows lane,
// lane + 64, lane + 128 of the lane) to (beta, 0, ..., 0); publishes v and tau (buffer j & 1) and writes v to
// Vh, tau and beta to the outputs
__device__ __forceinline__ void trd_reflect(const double (&c)[3], int j, int m, int lane, TrdShared& sh,
                                            double* __restrict__ Vh, double* __restrict__ tauo,
                                            double* __restrict__ eo) {
  double sg = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int r = lane + 64 * k;
    sg += (r > j + 1 && r < m) ? c[k] * c[k] : 0.0;
  }
  sg = wave_sum(sg);
  // alpha = c at row j + 1: read from its lane in each of the three slots, then the slot chosen (a select of
  // values, not of an index into c, which would send c to scratch memory)
  const int jr = j + 1, sl = jr >> 6;
  const double a0 = lane_of(c[0], jr & 63), a1 = lane_of(c[1], jr & 63), a2 = lane_of(c[2], jr & 63);
  const double al = sl == 0 ? a0 : (sl == 1 ? a1 : a2);
  double be = al, tv = 0.0, sc = 0.0;
  // below, beta d leaves the range of a double (a rank-one matrix gets there by rounding noise of noise); the largest entry
  // of the matrix is at least 1 here (trd_kernel), so a column below 1e-150 is nothing beside it
  if (sg > 1e-300) {
    // refined estimates in place of the square root and the division: they are a chain that every wavefront waits for
    double rs;
    const double nr = sqrt_nr(al * al + sg, rs);
    be = al >= 0.0 ? -nr : nr;
    const double d = al - be;                // |d| >= |al|: no cancellation
    const double inv = rcp_nr(be * d);       // tau = (beta - alpha) / beta = -d^2 inv, 1 / d = beta inv
    tv = -d * d * inv;
    sc = be * inv;
  }
  double* vv = sh.v[j & 1];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int r = lane + 64 * k;
    const double v = r == j + 1 ? 1.0 : ((r > j + 1 && r < m) ? c[k] * sc : 0.0);
    vv[r] = v;
    if (r < m) Vh[r + (size_t)j * m] = v;
  }
  if (lane == 0) {
    sh.tv[j & 1] = tv;
    tauo[j] = tv;
    eo[j] = be;
  }
}

// Householder steps j = TD_GX BJ .. min(TD_GX (BJ + 1) - 1, m - 3).  Columns below TD_GX BJ are finished (they lie
// left of every remaining step's column), so only column blocks b >= BJ are touched; row blocks whose
// rows all lie at or above j are skipped: those finished before the block's first step statically (A0),
// the others by a uniform test.  Step j finds v_j and tau_j published (by wavefront 0, during step j - 1, or
// before the first step); every thread forms its share of p = tau A v, and the owners of column j + 1
// publish it as it stands; after the second barrier every thread updates its elements while wavefront 0
// forms column j + 1 after the update from the published column, v, p and (p . v) alone, then the next
// reflector from it, so two barriers per step.
template <int RA, int RB, int BJ>
__device__ __forceinline__ void trd_block(double (&A)[RA][RB], int m, TrdShared& sh, int tx, int ty,
                                          int lane, int tid, double* __restrict__ Vh, double* __restrict__ tauo,
                                          double* __restrict__ eo) {
  constexpr int A0 = (BJ * TD_GX + 1) / TD_GY;   // row blocks a < A0 end at or above row BJ TD_GX
  const int j0 = BJ * TD_GX, j1 = min(m - 2, j0 + TD_GX);
  for (int j = j0; j < j1; ++j) {
    const int buf = j & 1;
    const double* vv = sh.v[buf];
    double* pv = sh.p[buf];
    const bool next = j + 1 < m - 2;   // uniform: a step j + 1 follows
    __syncthreads();
    const double tv = sh.tv[buf];
    // p = tau A v on the rows below j (finished row blocks are skipped and never stored); column by column,
    // so only the matrix, the row sums and one v entry are live
    double ps[RA] = {};
#pragma unroll
    for (int b = BJ; b < RB; ++b) {
      const double vcb = vv[tx + TD_GX * b];
#pragma unroll
      for (int a = A0; a < RA; ++a) {
        if (TD_GY * a + TD_GY - 1 <= j) continue;   // uniform: every row of the block is finished
        ps[a] = fma(A[a][b], vcb, ps[a]);
      }
    }
    // row sums over the TD_GX lanes of each row: pairs, quads, half rows (8 lanes), rows (16), row pairs (32)
#pragma unroll
    for (int a = A0; a < RA; ++a) ps[a] += dpp_d<0xB1>(ps[a]);
#pragma unroll
    for (int a = A0; a < RA; ++a) ps[a] += dpp_d<0x4E>(ps[a]);
#pragma unroll
    for (int a = A0; a < RA; ++a) ps[a] += dpp_d<0x141>(ps[a]);
    if constexpr (TD_GX >= 16) {
#pragma unroll
      for (int a = A0; a < RA; ++a) ps[a] += dpp_d<0x140>(ps[a]);
    }
    if constexpr (TD_GX == 32) {   // row_bcast15 adds row 0 into row 1, row 2 into row 3
#pragma unroll
      for (int a = A0; a < RA; ++a) ps[a] += dpp_d<0x142, 0xA>(ps[a]);
    }
    // the rows' share of p . v (v is zero on finished rows), summed over the wavefront's four rows of lanes
    double vr[RA], pq = 0.0;
#pragma unroll
    for (int a = A0; a < RA; ++a) {
      vr[a] = vv[ty + TD_GY * a];
      pq = fma(ps[a], vr[a], pq);
    }
    pq += dpp_d<0x142, 0xA>(pq);
    pq += dpp_d<0x143, 0x8>(pq);
    if (lane == 63) sh.pp[buf][tid >> 6] = tv * pq;
#pragma unroll
    for (int a = A0; a < RA; ++a) {
      if (TD_GY * a + TD_GY - 1 <= j) continue;
      const int r = ty + TD_GY * a;
      if (tx == (TD_GX == 32 ? 16 : 0)) pv[r] = (r > j && r < m) ? tv * ps[a] : 0.0;   // a lane that holds the row total
    }
    // column j + 1 before this step's update (its rows in finished blocks are never read)
    if (next) {
      double* cn = sh.col[buf];
      if (j + 1 < j0 + TD_GX) {
        if (tx == j + 1 - j0) {
#pragma unroll
          for (int a = A0; a < RA; ++a) cn[ty + TD_GY * a] = A[a][BJ];
        }
      } else if constexpr (BJ + 1 < RB) {   // a buffer of its own: one store merged from the two
        if (tx == 0) {                          // branches would index A dynamically (A in scratch memory)
#pragma unroll
          for (int a = A0; a < RA; ++a) sh.colb[ty + TD_GY * a] = A[a][BJ + 1];
        }
      }
    }
    __syncthreads();
    // w = p - (tau / 2) (p . v) v ;  A -= v w^T + w v^T
    const double* pp = sh.pp[buf];
    static_assert(TD_NT / 64 == 8, "eight shares");
    const double pw = ((pp[0] + pp[1]) + (pp[2] + pp[3])) + ((pp[4] + pp[5]) + (pp[6] + pp[7]));
    const double kc = 0.5 * tv * pw;
    if (next && tid < 64) {   // column j + 1 after the update (v[j+1] = 1), then the next reflector
      const double* cn = j + 1 < j0 + TD_GX ? sh.col[buf] : sh.colb;
      const double wj1 = pv[j + 1] - kc;
      double c[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int r = lane + 64 * k;
        const double x = cn[r] - vv[r] * wj1 - (pv[r] - kc * vv[r]);
        c[k] = r >= j + 2 ? x : 0.0;   // rows above hold stale values
      }
      trd_reflect(c, j + 1, m, lane, sh, Vh, tauo, eo);
    }
    // the thread's rows of v and w, then the update column by column (p is written this step only for
    // rows in unskipped blocks: columns at or left of j take w = 0)
    double wr[RA];
#pragma unroll
    for (int a = A0; a < RA; ++a) {
      const int r = ty + TD_GY * a;
      wr[a] = TD_GY * a + TD_GY - 1 <= j ? 0.0 : pv[r] - kc * vr[a];
    }
#pragma unroll
    for (int b = BJ; b < RB; ++b) {
      const int c = tx + TD_GX * b;
      const double vcb = vv[c], x = pv[c] - kc * vcb, wcb = c > j ? x : 0.0;
#pragma unroll
      for (int a = A0; a < RA; ++a) {
        if (TD_GY * a + TD_GY - 1 <= j) continue;
        A[a][b] = fma(-wr[a], vcb, fma(-vr[a], wcb, A[a][b]));
      }
    }
  }
}

// the column blocks BJ, BJ + 1, ..., RB - 1 in turn
template <int RA, int RB, int BJ>
__device__ __forceinline__ void trd_blocks(double (&A)[RA][RB], int m, TrdShared& sh, int tx, int ty,
                                           int lane, int tid, double* __restrict__ Vh, double* __restrict__ tauo,
                                           double* __restrict__ eo) {
  trd_block<RA, RB, BJ>(A, m, sh, tx, ty, lane, tid, Vh, tauo, eo);
  if constexpr (BJ + 1 < RB) trd_blocks<RA, RB, BJ + 1>(A, m, sh, tx, ty, lane, tid, Vh, tauo, eo);
}

// H (m x m, ld ldh; the upper triangle is read) -> of H / scale the diagonal dout (m), off-diagonal eout (m - 1),
// reflectors Vh (m x m, column j = v_j) and tauo (m - 2).  scale: the power of two that brings the largest entry
// into [1, 2), exact to divide by.  Squares of entries and of gaps are formed here and in the divide and conquer, and
// without it a matrix of norm 1e-133 lost eigenvectors with values 1e-14 of the largest, one of 1e-150 all of them.  RA x RB: elements per thread, the smallest of the
// instances in trd_launch that covers m: the padding of a larger one is multiplied and updated like the rest (the
// values are the same for each).
template <int RA, int RB>
__global__ __launch_bounds__(TD_NT) void trd_kernel(const double* __restrict__ H, int ldh, int m,
                                                    double* __restrict__ dout, double* __restrict__ eout,
                                                    double* __restrict__ Vh, double* __restrict__ tauo,
                                                    double* __restrict__ scale, const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  __shared__ TrdShared sh;
  const int tid = threadIdx.x, ty = tid / TD_GX, tx = tid % TD_GX, lane = tid & 63;
  double A[RA][RB];
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int r = ty + TD_GY * a, c = tx + TD_GX * b;
      const bool in = r < m && c < m;
      const double x = H[in ? min(r, c) + (size_t)max(r, c) * ldh : 0];   // branch-free, clamped address
      A[a][b] = in ? x : 0.0;
    }
  double mx = 0.0;
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < RB; ++b) mx = fmax(mx, fabs(A[a][b]));
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
  if (lane == 0) sh.pp[0][tid >> 6] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < TD_NT / 64; ++w) mx = fmax(mx, sh.pp[0][w]);
  const int ex = mx > 0.0 && mx <= DBL_MAX ? ilogb(mx) : 0;   // (zero and non-finite matrices as they are)
  if (tid == 0) *scale = ldexp(1.0, ex);
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < RB; ++b) A[a][b] = ldexp(A[a][b], -ex);
  if (m > 2) {   // the first reflector, from column 0 (published, then formed by wavefront 0)
    if (tx == 0) {
#pragma unroll
      for (int a = 0; a < RA; ++a) sh.col[1][ty + TD_GY * a] = A[a][0];
    }
    __syncthreads();
    if (tid < 64) {
      double c[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) c[k] = sh.col[1][lane + 64 * k];
      trd_reflect(c, 0, m, lane, sh, Vh, tauo, eout);
    }
  }
  trd_blocks<RA, RB, 0>(A, m, sh, tx, ty, lane, tid, Vh, tauo, eout);
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int r = ty + TD_GY * a, c = tx + TD_GX * b;
      if (r == c && r < m) dout[r] = A[a][b];
      if (r == m - 1 && c == m - 2) eout[m - 2] = A[a][b];
    }
}

// ---------------------------------------------------------------------------------------------------
// divide and conquer
// ---------------------------------------------------------------------------------------------------
constexpr int DC_NT = 1024;
constexpr int DC_SEC = 256;   // threads from DC_SEC on work L lanes per root / per entry

// state of the merges of one level, NM: rows of the (sub)matrix at most
template <int NM> struct DcShared {
  double lam[NM];                 // eigenvalue of column g of the current eigenvector matrix
  double ds[NM], zs[NM];          // merged node: d and z sorted ascending by d
  int src[NM];                    // column of the sorted entry
  int nlo[NM];                    // lo of the merge node of index g at this level (-1: none)
  double dK[NM], zK[NM];          // kept entries (slots lo .. lo + K - 1)
  double z2[NM];                  // rho zK^2
  int kc[NM], ktype[NM];          // their columns; 0: top half only, 1: both halves, 2: bottom half only
  double dvl[NM];                 // deflated eigenvalues (slots lo + K .. hi - 1)
  int dcol[NM];                   // their columns
  int org[NM];                    // pole (absolute slot) the root of slot lo + j is measured from
  double tau[NM];                 // root = dK[org] + tau
  double zh[NM];                  // recomputed z
  int upos[NM], kcp[NM];          // row of kept entry i in the K x K matrix (first its index within
                                  // its type); column of row p
  double rc[NM], rs[NM];          // deflation rotations of a node (slots lo ..)
  int ra[NM], rb[NM];
  int nK[NM], nT1[NM], nT12[NM], nRot[NM];   // per node at slot lo
  double nRho[NM];
  unsigned long long nmd[NM], nmz[NM];       // per node: bits of max |d|, max |z| (non-negative)
  double floor;                   // least deflation threshold of any node
};

// node of index g at depth dd (recursive halving of [0, m), the lower half the smaller); false when it is a leaf (one
// or two rows)
__device__ __forceinline__ bool dc_node(int g, int dd, int m, int& lo, int& hi) {
  lo = 0;
  hi = m;
  for (int l = 0; l < dd; ++l) {
    if (hi - lo <= 2) return false;
    const int mid = lo + ((hi - lo) >> 1);
    if (g < mid) hi = mid;
    else lo = mid;
  }
  return dd == 0 || hi - lo > 2;
}

// levels of merges: halvings until no node has more than two rows
__device__ __forceinline__ int dc_depth(int m) {
  int d = 0;
  while ((2 << d) < m) ++d;
  return d;
}

// sums / products over the L aligned lanes that share a root, 8 or the wavefront (butterflies: the same bits in all of
// them)
template <int L>
__device__ __forceinline__ double sumL(double x) {
  static_assert(L == 8 || L == 64, "8 lanes or all");
  if constexpr (L == 64) return wave_sum(x);
  x += dpp_d<0xB1>(x);
  x += dpp_d<0x4E>(x);
  x += dpp_d<0x141>(x);
  return x;
}

template <int L>
__device__ __forceinline__ double prodL(double x) {
  if constexpr (L == 64) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) x *= __shfl_xor(x, o);
    return x;
  }
  x *= dpp_d<0xB1>(x);
  x *= dpp_d<0x4E>(x);
  x *= dpp_d<0x141>(x);
  return x;
}

// a / b to the accuracy of a division (b finite and nonzero)
__device__ __forceinline__ double div_nr(double a, double b) {
  const double r = rcp_nr(b), q = a * r;
  return fma(fma(-b, q, a), r, q);
}

// root e in (le, he) of c (djl - e)(djr - e) + s1 (djr - e) + s2 (djl - e) = 0 (the secular function
// modelled by its two nearest poles and a constant); false when none lies there
__device__ __forceinline__ bool dc_quad(double c, double djl, double djr, double s1, double s2, double le, double he,
                                        double& e) {
  // (quotients by the refined reciprocal: an iterate needs no correctly rounded division)
  const double qa = c, qb = -(c * (djl + djr) + s1 + s2), qc = c * djl * djr + s1 * djr + s2 * djl;
  if (qa == 0.0) {
    if (qb == 0.0) return false;
    e = -qc * rcp_nr(qb);
    return e > le && e < he;
  }
  const double D = qb * qb - 4.0 * qa * qc;
  double sq = 0.0;
  if (D > 1e-290) {
    const double y = __builtin_amdgcn_rsq(D);
    sq = D * fma(0.5 * y, fma(-D * y, y, 1.0), y);
  }
  const double qq = -0.5 * (qb + copysign(sq, qb));
  e = qq * rcp_nr(qa);
  if (e > le && e < he) return true;
  if (qq == 0.0) return false;
  e = qc * rcp_nr(qq);
  return e > le && e < he;
}

// root j (0 <= j < K) of 1 + rho sum_i zk_i^2 / (dk_i - lambda) = 0, dk ascending, L lanes (q = 0 .. L - 1) sharing the
// sums: lane q holds the terms q, q + L, ... (at most T) in registers.  Returns the pole o (index into dk) and
// lambda - dk[o].
template <int L, int T>
__device__ __forceinline__ void dc_secular(const double* dk, const double* z2, int K, int j, int q, int& o, double& t) {
  double d[T], w[T];   // a term that is not there: weight 0 at a distant pole
#pragma unroll
  for (int u = 0; u < T; ++u) {
    const int i = q + L * u, ic = min(i, K - 1);
    const double di = dk[ic], wi = z2[ic];
    d[u] = i < K ? di : 1e300;
    w[u] = i < K ? wi : 0.0;
  }
  double lo_t, hi_t;
  if (j < K - 1) {
    const double dj = dk[j], dn = dk[j + 1], wj = z2[j], wn = z2[j + 1];
    // the sign of the function midway picks the nearer pole; the midpoint is kept as an offset from d_j (rounded, it is off
    // by eps |d|, which between two close poles with equal weights decides the sign and puts the root outside the bracket)
    const double gap = dn - dj, hg = 0.5 * gap;
    double f = 0.0;
#pragma unroll
    for (int u = 0; u < T; ++u) f += w[u] * rcp_nr((d[u] - dj) - hg);
    f = 1.0 + sumL<L>(f);
    o = f > 0.0 ? j : j + 1;
    if (o == j) { lo_t = 0.0; hi_t = hg; }
    else { lo_t = -hg; hi_t = 0.0; }
    // first iterate: the two nearest poles exactly, the rest of the sum frozen at the midpoint
    const double djl = o == j ? 0.0 : -gap, djr = o == j ? gap : 0.0;
    const double rh = rcp_nr(hg), cc = f + wj * rh - wn * rh;
    double e;
    t = dc_quad(cc, djl, djr, wj, wn, lo_t, hi_t, e) ? e : 0.5 * (lo_t + hi_t);
  } else {
    double zz = 0.0;
#pragma unroll
    for (int u = 0; u < T; ++u) zz += w[u];
    o = j;
    lo_t = 0.0;
    hi_t = sumL<L>(zz);
    t = 0.5 * (lo_t + hi_t);
  }
  const double dorg = dk[o], dj = dk[j] - dorg, dj1 = j < K - 1 ? dk[j + 1] - dorg : 0.0;
#pragma unroll
  for (int u = 0; u < T; ++u) d[u] -= dorg;
  for (int it = 0; it < 80; ++it) {
    double f = 0.0, af = 0.0, psp = 0.0, php = 0.0;
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const double r = rcp_nr(d[u] - t), x = w[u] * r, y = x * r;
      f += x;
      af += fabs(x);
      const bool left = q + L * u <= j;
      psp += left ? y : 0.0;
      php += left ? 0.0 : y;
    }
    f = 1.0 + sumL<L>(f);
    af = sumL<L>(af);
    psp = sumL<L>(psp);
    php = sumL<L>(php);
    if (fabs(f) <= 16.0 * DBL_EPSILON * (1.0 + af) || hi_t - lo_t <= 2.0 * DBL_EPSILON * fmax(fabs(lo_t), fabs(hi_t)))
      break;
    if (f > 0.0) hi_t = t;
    else lo_t = t;
    const double djl = dj - t;
    const double s1 = djl * djl * psp;
    double tn = t;
    bool ok = false;
    if (j < K - 1) {
      const double djr = dj1 - t;
      const double s2 = djr * djr * php;
      const double c = f - djl * psp - djr * php;
      double e;
      if (dc_quad(c, djl, djr, s1, s2, lo_t - t, hi_t - t, e)) { tn = t + e; ok = true; }
    } else {
      const double c = f - djl * psp;
      if (c != 0.0) {
        const double e = djl + s1 * rcp_nr(c);
        if (e > lo_t - t && e < hi_t - t) { tn = t + e; ok = true; }
      }
    }
    if (!ok || !(tn > lo_t && tn < hi_t)) tn = 0.5 * (lo_t + hi_t);
    t = tn;
  }
}

// state of a merge node's deflation scan over its sorted entries: the kept entries so far (K, per type
// c0 top half only, c1 both halves (rotated), c2 bottom half only), the deflated ones (nd), the rotations
// (nr) and the pending entry (the last one not deflated, which a close successor may still rotate away)
struct DcScan {
  int K = 0, nd = 0, nr = 0, c0 = 0, c1 = 0, c2 = 0;
  bool have = false, prot = false;
  double dp = 0.0, zp = 0.0;
  int sp = 0;
};

// deflation threshold of the node at lo: 8 eps max(max |d|, rho max |z|), and no less than 1e-40 of the whole matrix (far
// below what the tridiagonalisation left): a rank-deficient matrix leaves nodes of rounding noise of noise, 1e-115 and
// smaller, where the squares in the secular function and the norms would leave the range of a double
template <class SH>
__device__ __forceinline__ double dc_tol(const SH& sh, int lo, double rho) {
  const double dmx = __longlong_as_double((long long)sh.nmd[lo]), zmx = __longlong_as_double((long long)sh.nmz[lo]);
  return fmax(8.0 * DBL_EPSILON * fmax(dmx, rho * zmx), sh.floor);
}

// keep entry (d, z, column src, rotated?) as kept entry number st.K
template <class SH>
__device__ __forceinline__ void dc_keep(SH& sh, int lo, int mid, double rho, double d, double z, int src,
                                        bool rot, DcScan& st) {
  const int ty = rot ? 1 : (src < mid ? 0 : 2);
  sh.dK[lo + st.K] = d;
  sh.zK[lo + st.K] = z;
  sh.z2[lo + st.K] = rho * z * z;
  sh.kc[lo + st.K] = src;
  sh.ktype[lo + st.K] = ty;
  sh.upos[lo + st.K] = ty == 0 ? st.c0 : (ty == 1 ? st.c1 : st.c2);
  st.c0 += ty == 0;
  st.c1 += ty == 1;
  st.c2 += ty == 2;
  ++st.K;
}

// sequential scan of the sorted entries from .. hi - 1 (one lane): small z deflates; a close pending /
// new pair is rotated (Givens on the two columns, recorded for the rows of Q) so that the pending entry
// deflates
template <class SH>
__device__ __forceinline__ void dc_scan_seq(SH& sh, int lo, int hi, int mid, double rho, double tol, int from, DcScan& st) {
  double dnx = sh.ds[from], znx = sh.zs[from];
  int snx = sh.src[from];
  for (int nj = from; nj < hi; ++nj) {
    const double dn = dnx, zn = znx;
    const int sn = snx;
    if (nj + 1 < hi) {   // the next entry's loads are in flight while this one is decided
      dnx = sh.ds[nj + 1];
      znx = sh.zs[nj + 1];
      snx = sh.src[nj + 1];
    }
    if (rho * fabs(zn) <= tol) {
      sh.dvl[hi - 1 - st.nd] = dn;
      sh.dcol[hi - 1 - st.nd] = sn;
      ++st.nd;
      continue;
    }
    if (st.have) {
      const double dt = dn - st.dp;
      if (fabs(dt) <= 2.0 * tol) {   // |dt c s| <= |dt| / 2: only close pairs can deflate
        const double tt = hypot(zn, st.zp);
        const double c = zn / tt, sr = -st.zp / tt;
        if (fabs(dt * c * sr) <= tol) {
          sh.ra[lo + st.nr] = st.sp;
          sh.rb[lo + st.nr] = sn;
          sh.rc[lo + st.nr] = c;
          sh.rs[lo + st.nr] = sr;
          ++st.nr;
          sh.dvl[hi - 1 - st.nd] = st.dp * c * c + dn * sr * sr;
          sh.dcol[hi - 1 - st.nd] = st.sp;
          ++st.nd;
          st.dp = st.dp * sr * sr + dn * c * c;
          st.zp = tt;
          st.sp = sn;
          st.prot = true;
          continue;
        }
      }
      dc_keep(sh, lo, mid, rho, st.dp, st.zp, st.sp, st.prot, st);
    }
    st.have = true;
    st.dp = dn;
    st.zp = zn;
    st.sp = sn;
    st.prot = false;
  }
}

template <class SH>
__device__ __forceinline__ void dc_scan_finish(SH& sh, int lo, int mid, double rho, DcScan& st) {
  if (st.have) dc_keep(sh, lo, mid, rho, st.dp, st.zp, st.sp, st.prot, st);
  sh.nK[lo] = st.K;
  sh.nT1[lo] = st.c0;
  sh.nT12[lo] = st.c0 + st.c1;
  sh.nRot[lo] = st.nr;
  sh.nRho[lo] = rho;
}

// the scan of the node [lo, hi) by one wavefront: chunks of 64 entries are decided by ballots as long as
// no entry of a chunk lies within 2 tol of its predecessor (then nothing rotates: every entry that is not
// deflated is kept, in order); from the first chunk with such a pair on, lane 0 scans sequentially
// from the state the chunks before it left (the same state the sequential scan would have reached)
template <class SH>
__device__ __forceinline__ void dc_scan_wave(SH& sh, const double* __restrict__ ev, int lo, int hi, int lane) {
  const int mid = lo + ((hi - lo) >> 1);
  const double rho = 2.0 * fabs(ev[mid - 1]);
  const double tol = dc_tol(sh, lo, rho);
  DcScan st;   // the same in every lane
  const unsigned long long lt = (1ull << lane) - 1ull;
  int h0 = lo;
  for (; h0 < hi; h0 += 64) {
    const int h = h0 + lane;
    const bool in = h < hi;
    const double dn = in ? sh.ds[h] : 0.0, zn = in ? sh.zs[h] : 0.0;
    const int sn = in ? sh.src[h] : 0;
    const bool defl = in && rho * fabs(zn) <= tol;
    const bool kept = in && !defl;
    const unsigned long long mk = __ballot(kept), md = __ballot(defl);
    const unsigned long long below = mk & lt;
    const int pl = below ? 63 - __clzll(below) : 0;
    const double dl = __shfl(dn, pl);
    const bool hasprev = below != 0 || st.have;
    const double dprev = below != 0 ? dl : st.dp;
    if (__ballot(kept && hasprev && fabs(dn - dprev) <= 2.0 * tol)) break;   // uniform
    if (mk) {
      const int last = 63 - __clzll(mk);
      if (st.have) {   // the pending entry of the chunks before: kept
        if (lane == 0) dc_keep(sh, lo, mid, rho, st.dp, st.zp, st.sp, false, st);
        else {
          const int ty = st.sp < mid ? 0 : 2;
          st.c0 += ty == 0;
          st.c2 += ty == 2;
          ++st.K;
        }
      }
      const bool top = sn < mid;
      const unsigned long long mk1 = mk & ~(1ull << last);   // kept now; the last one becomes pending
      const unsigned long long m0 = __ballot(kept && top) & mk1, m2 = __ballot(kept && !top) & mk1;
      if (kept && lane != last) {
        const int K = st.K + __popcll(mk1 & lt);
        sh.dK[lo + K] = dn;
        sh.zK[lo + K] = zn;
        sh.z2[lo + K] = rho * zn * zn;
        sh.kc[lo + K] = sn;
        sh.ktype[lo + K] = top ? 0 : 2;
        sh.upos[lo + K] = top ? st.c0 + __popcll(m0 & lt) : st.c2 + __popcll(m2 & lt);
      }
      st.K += __popcll(mk1);
      st.c0 += __popcll(m0);
      st.c2 += __popcll(m2);
      st.have = true;
      st.prot = false;
      st.dp = __shfl(dn, last);
      st.zp = __shfl(zn, last);
      st.sp = __shfl(sn, last);
    }
    if (defl) {
      const int e = hi - 1 - (st.nd + __popcll(md & lt));
      sh.dvl[e] = dn;
      sh.dcol[e] = sn;
    }
    st.nd += __popcll(md);
  }
  if (lane == 0) {
    if (h0 < hi) dc_scan_seq(sh, lo, hi, mid, rho, tol, h0, st);
    dc_scan_finish(sh, lo, mid, rho, st);
  }
}

// the roots of every merge of a level (threads DC_SEC.., L lanes per root, at most T terms each), then z from the roots
// (Lowner's formula) and the order of the kept columns, then the normalised vectors u_j into U (K x K per node, transposed:
// entry (row upos_i, column j) at U[lo + j + (lo + upos_i) LU]) and the new eigenvalues; three barriers
template <int L, int T, int NM>
__device__ __forceinline__ void dc_roots(DcShared<NM>& sh, double* U, int LU, int m, int tid) {
  const int g = (tid - DC_SEC) / L, q = (tid - DC_SEC) % L;
  const bool mine = tid >= DC_SEC && g < m && sh.nlo[g] >= 0;
  const int lo = mine ? sh.nlo[g] : 0, j = g - lo, K = mine ? sh.nK[lo] : 0;
  const bool root = mine && j < K;
  int o = 0;
  double t = 0.0;
  if (root) {
    dc_secular<L, T>(sh.dK + lo, sh.z2 + lo, K, j, q, o, t);
    if (q == 0) {
      sh.org[lo + j] = lo + o;
      sh.tau[lo + j] = t;
    }
  }
  __syncthreads();
  if (root) {
    const double* dk = sh.dK + lo;
    const double di = dk[j], rho = sh.nRho[lo];
    double p = 1.0;
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int i = q + L * u, ic = min(i, K - 1);
      const double lmd = (sh.dK[sh.org[lo + ic]] - di) + sh.tau[lo + ic];
      const double den = ic == K - 1 ? rho : dk[ic < j ? ic : ic + 1] - di;
      const double x = div_nr(lmd, den);
      p *= i < K ? x : 1.0;
    }
    p = prodL<L>(p);
    if (q == 0) {
      sh.zh[lo + j] = copysign(sqrt(fmax(p, 0.0)), sh.zK[lo + j]);
      const int ty = sh.ktype[lo + j];
      const int pos = sh.upos[lo + j] + (ty == 0 ? 0 : (ty == 1 ? sh.nT1[lo] : sh.nT12[lo]));
      sh.upos[lo + j] = pos;
      sh.kcp[lo + pos] = sh.kc[lo + j];
    }
  }
  __syncthreads();
  if (root) {
    const double dorg = sh.dK[lo + o];
    double s = 0.0, v[T];
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int i = q + L * u, ic = min(i, K - 1);
      const double x = div_nr(sh.zh[lo + ic], (sh.dK[lo + ic] - dorg) - t);
      v[u] = i < K ? x : 0.0;
      s = fma(v[u], v[u], s);
    }
    s = sumL<L>(s);
    const double rn = 1.0 / sqrt(s);
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int i = q + L * u;
      if (i < K) U[(lo + j) + (size_t)(lo + sh.upos[lo + i]) * LU] = v[u] * rn;
    }
    if (q == 0) sh.lam[lo + j] = dorg + t;
  } else if (mine && q == 0) {
    sh.lam[g] = sh.dvl[g];
  }
  if (tid < m) {
    sh.nmd[tid] = 0;
    sh.nmz[tid] = 0;
  }
  __syncthreads();
}

// the top merge as dc_top_kernel leaves it (after its deflation and rotations) for dc_sec_kernel, dc_zh_kernel
// and dc_final_kernel: the K kept poles (ascending), their z and rho z^2, their columns of Z, the deflated
// columns (slots K..m-1), and per root its pole, offset and recomputed z
struct DcTop {
  double *dK, *zK, *z2, *tau, *zh;
  int *kc, *dcol, *org, *K;
  double* rho;
};

// children's eigenpairs -> z, sorted d of every merge node of depth dd (DC_ZL lanes per index share its rank)
constexpr int DC_ZL = 4;
template <int NM>
__device__ __forceinline__ void dc_gather(DcShared<NM>& sh, const double* __restrict__ ev, int m, int dd, const double* Qin,
                                          int LD, int tid) {
  const int g = tid / DC_ZL, q = tid % DC_ZL;
  if (g < m) {
    int lo, hi;
    if (!dc_node(g, dd, m, lo, hi)) {
      if (q == 0) sh.nlo[g] = -1;
    } else {
      const int mid = lo + ((hi - lo) >> 1);
      const double be = ev[mid - 1];
      const double x = Qin[(g < mid ? mid - 1 : mid) + (size_t)g * LD];
      const double z = 0.70710678118654752440 * (g >= mid && be < 0.0 ? -x : x);
      // (a NaN counts as the largest value, so the ranks are a permutation whatever the input)
      const double lg = fmin(sh.lam[g], DBL_MAX);
      int rank = 0;
#pragma unroll 4
      for (int h = lo + q; h < hi; h += DC_ZL) {
        const double lh = fmin(sh.lam[h], DBL_MAX);
        rank += (lh < lg) || (lh == lg && h < g);
      }
      rank += __builtin_amdgcn_update_dpp(0, rank, 0xB1, 0xF, 0xF, true);
      rank += __builtin_amdgcn_update_dpp(0, rank, 0x4E, 0xF, 0xF, true);
      if (q == 0) {
        sh.nlo[g] = lo;
        sh.ds[lo + rank] = sh.lam[g];
        sh.zs[lo + rank] = z;
        sh.src[lo + rank] = g;
        atomicMax(&sh.nmd[lo], (unsigned long long)__double_as_longlong(fabs(lg)));
        atomicMax(&sh.nmz[lo], (unsigned long long)__double_as_longlong(fabs(z)));
      }
    }
  }
}

// the deflation rotations of its node on row r of Qin
template <int NM>
__device__ __forceinline__ void dc_rotate(const DcShared<NM>& sh, double* Qin, int LD, int m, int r) {
  if (r < m && sh.nlo[r] >= 0) {
    const int lo = sh.nlo[r], nr = sh.nRot[lo];
    for (int t = 0; t < nr; ++t) {
      const size_t ia = r + (size_t)sh.ra[lo + t] * LD, ib = r + (size_t)sh.rb[lo + t] * LD;
      const double x = Qin[ia], y = Qin[ib], c = sh.rc[lo + t], s = sh.rs[lo + t];
      Qin[ia] = c * x + s * y;
      Qin[ib] = -s * x + c * y;
    }
  }
}

// one level of merges: Qin holds the children's eigenvectors (block diagonal), Qout receives the
// merged ones (ld LO).
template <int L, int NM>
__device__ __forceinline__ void dc_level(DcShared<NM>& sh, const double* __restrict__ ev, int m, int dd, double* Qin, int LD,
                                         double* Qout, int LO, double* U, int LU, int tid) {
  dc_gather(sh, ev, m, dd, Qin, LD, tid);
  __syncthreads();
  // deflation: a wavefront per merge node while a level has at most 16 of them (ballots decide whole chunks
  // of 64 entries at once until a close pair needs the sequential scan), else one thread per node
  if (dd <= 4) {
    const int wave = tid >> 6, lane = tid & 63;
    if (wave < (1 << dd)) {
      int lo = 0, hi = m;
      for (int l = dd - 1; l >= 0; --l) {
        const int md = lo + ((hi - lo) >> 1);
        if ((wave >> l) & 1) lo = md;
        else hi = md;
      }
      if (hi - lo > 2) dc_scan_wave(sh, ev, lo, hi, lane);
    }
  } else if (tid < m && sh.nlo[tid] == tid) {
    int lo2, hi;
    dc_node(tid, dd, m, lo2, hi);
    DcScan st;
    const int mid = tid + ((hi - tid) >> 1);
    const double rho = 2.0 * fabs(ev[mid - 1]);
    dc_scan_seq(sh, tid, hi, mid, rho, dc_tol(sh, tid, rho), tid, st);
    dc_scan_finish(sh, tid, mid, rho, st);
  }
  __syncthreads();
  // deflation rotations on the rows of Qin (row-parallel); the secular roots, z from the roots, vectors
  if (tid < DC_SEC) dc_rotate(sh, Qin, LD, m, tid);
  const int smax = (m + (1 << dd) - 1) >> dd;   // the widest node of this level
  constexpr int T = NM / L, TH = (T + 1) / 2;
  if (smax <= L) dc_roots<L, 1>(sh, U, LU, m, tid);
  else if (smax <= 2 * L) dc_roots<L, 2>(sh, U, LU, m, tid);
  else if (smax <= 3 * L) dc_roots<L, 3>(sh, U, LU, m, tid);
  else if (smax <= TH * L) dc_roots<L, TH>(sh, U, LU, m, tid);
  else dc_roots<L, T>(sh, U, LU, m, tid);
  // Qout = Qin[:, kept] U, deflated columns copied: 16 x 16 output tiles on the FP64 matrix cores, one wavefront per
  // tile, the same number of tiles for every node of the level
  const int wave = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int tn = (smax + 15) >> 4, items = (tn * tn) << dd;
  for (int it = wave; it < items; it += DC_NT / 64) {
    const int k = it / (tn * tn), tl = it - k * tn * tn;
    int lo = 0, hi = m;
    for (int l = dd - 1; l >= 0; --l) {
      const int mid = lo + ((hi - lo) >> 1);
      if ((k >> l) & 1) lo = mid;
      else hi = mid;
    }
    const int s = hi - lo, r0 = lo + 16 * (tl % tn), t0 = 16 * (tl / tn);
    if (s <= 2 || r0 >= hi || t0 >= s) continue;   // a leaf, or no such tile in this node (uniform)
    const int K = sh.nK[lo], mid = lo + (s >> 1);
    // rows of the top half meet only top-half and rotated columns, the bottom half the others
    const int p0 = r0 >= mid ? sh.nT1[lo] : 0;
    const int p1 = t0 >= K ? 0 : (r0 + 15 < mid ? sh.nT12[lo] : K);
    const int ra = r0 + li;   // A-fragment row of this lane (A[li][lk])
    const int tb = t0 + li;   // B-fragment column of this lane (B[lk][li])
    // clamped addresses, no branches: rows and columns beyond the node only feed outputs that are not
    // stored, and the k-steps beyond p1 are zeroed through b
    const int rac = min(ra, hi - 1), tbc = min(tb, K - 1);
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    // four k-steps per pass: the column indices first (one LDS wait), then all eight operand loads in
    // flight before the first product
    for (int p = p0; p < p1; p += 16) {
      int kk[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) kk[u] = sh.kcp[lo + min(p + 4 * u + lk, p1 - 1)];
      double a[4], b[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        a[u] = Qin[rac + (size_t)kk[u] * LD];
        b[u] = U[(lo + tbc) + (size_t)(lo + min(p + 4 * u + lk, p1 - 1)) * LU];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], p + 4 * u + lk < p1 ? b[u] : 0.0, acc, 0, 0, 0);
    }
    // output lane layout of the 16 x 16 x 4 FP64 product: register q holds row lk + 4 q, column li
    const int src = tb >= K && tb < s ? sh.dcol[lo + tb] : 0;   // a deflated column is copied
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = r0 + lk + 4 * q;
      if (r < hi && tb < s) Qout[r + (size_t)(lo + tb) * LO] = tb < K ? acc[q] : Qin[r + (size_t)src * LD];
    }
  }
  __syncthreads();
}

// One half of the tridiagonal (d, e), rows [0, m / 2) or [m / 2, m) by block, torn off the other: its eigenvalues into lam
// and its eigenvectors into its columns of Qb (zero outside its rows).  NM: rows of a half at most; up to DC_QL of them
// the eigenvector matrices of the levels stay in LDS, above that they alternate between Qa and Qb.
constexpr int DC_QL = 72;
template <int L, int NM>
__global__ __launch_bounds__(DC_NT) void dc_kernel(const double* __restrict__ d, const double* __restrict__ e, int mtot,
                                                   double* __restrict__ Qag, double* __restrict__ Qbg,
                                                   double* __restrict__ lam_out, const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  constexpr bool QL = NM <= DC_QL;
  // pitch 16 mod 32 doubles: the columns of an operand read start in alternate halves of the banks
  constexpr int LQ = NM + (48 - NM % 32) % 32;
  __shared__ DcShared<NM> sh;
  __shared__ double Us[NM * LQ];
  __shared__ double Q0[QL ? NM * LQ : 1], Q1[QL ? NM * LQ : 1];
  const int tid = threadIdx.x;
  const int base = blockIdx.x ? mtot >> 1 : 0, m = (blockIdx.x ? mtot : mtot >> 1) - base;
  if (m < 1) return;
  // |T|: a wavefront's maximum of the bits of |d|, |e|
  if (tid < 64) {
    double x = 0.0;
    for (int i = tid; i < mtot; i += 64) x = fmax(x, fmax(fabs(d[i]), i + 1 < mtot ? fabs(e[i]) : 0.0));
    for (int o = 32; o > 0; o >>= 1) x = fmax(x, __shfl_xor(x, o));
    if (tid == 0) sh.floor = 1e-40 * x;
  }
  d += base;
  e += base;
  double* Zg = Qbg + base + (size_t)base * mtot;   // this half's block of Qb
  const int depth = dc_depth(m);
  // zeros outside the block
  {
    const int rows = mtot - m, r0 = blockIdx.x ? 0 : m;
    for (int idx = tid; idx < rows * m; idx += DC_NT) Qbg[r0 + idx % rows + (size_t)(base + idx / rows) * mtot] = 0.0;
  }
  // the levels alternate between two matrices, both starting as the leaves' vectors; the last one writes Zg (in LDS) or
  // ends there (in global memory)
  constexpr int LDC = LQ;
  const int LD = QL ? LDC : mtot;
  double* const Ya = Qag + base + (size_t)base * mtot;
  auto mat = [&](int par) -> double* {
    if constexpr (QL) return par ? Q1 : Q0;
    else return ((depth ^ par) & 1) ? Ya : Zg;   // level 0 (of depth levels) reads mat(0)
  };
  for (int idx = tid; idx < m * m; idx += DC_NT) {
    const int r = idx % m, c = idx / m;
    const double v = r == c ? 1.0 : 0.0;
    mat(0)[r + (size_t)c * LD] = v;
    if (depth > 0) mat(1)[r + (size_t)c * LD] = v;
  }
  __syncthreads();
  // leaves of one or two rows; every boundary between leaves is a tear, d_i -= |e_i| on both sides of it
  if (tid < m) {
    int lo = 0, hi = m;
    while (hi - lo > 2) {
      const int mid = lo + ((hi - lo) >> 1);
      if (tid < mid) hi = mid;
      else lo = mid;
    }
    if (tid == lo) {
      double a = d[lo] - (base + lo > 0 ? fabs(e[lo - 1]) : 0.0);
      if (hi - lo == 2) {
        const double b = e[lo], c = d[lo + 1] - (base + lo + 2 < mtot ? fabs(e[lo + 1]) : 0.0);
        double l0 = a, l1 = c;
        if (b != 0.0) {   // one Jacobi rotation
          const double ze = (c - a) / (2.0 * b), t = copysign(1.0, ze) / (fabs(ze) + sqrt(1.0 + ze * ze));
          const double cs = 1.0 / sqrt(1.0 + t * t), sn = cs * t;
          l0 = a - t * b;
          l1 = c + t * b;
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            double* Q = mat(k);
            if (k && depth == 0) break;
            Q[lo + (size_t)lo * LD] = cs;
            Q[lo + 1 + (size_t)lo * LD] = -sn;
            Q[lo + (size_t)(lo + 1) * LD] = sn;
            Q[lo + 1 + (size_t)(lo + 1) * LD] = cs;
          }
        }
        sh.lam[lo] = l0;
        sh.lam[lo + 1] = l1;
      } else {
        if (base + lo + 1 < mtot) a -= fabs(e[lo]);
        sh.lam[lo] = a;
      }
    }
    sh.nmd[tid] = 0;
    sh.nmz[tid] = 0;
  }
  __syncthreads();
  for (int l = 0; l < depth; ++l) {
    const int dd = depth - 1 - l;
    double* Qout = QL && dd == 0 ? Zg : mat((l + 1) & 1);
    dc_level<L>(sh, e, m, dd, mat(l & 1), LD, Qout, QL && dd == 0 ? mtot : LD, Us, LQ, tid);
  }
  if (QL && depth == 0 && tid < m * m) Zg[tid % m + (size_t)(tid / m) * mtot] = mat(0)[tid % m + (tid / m) * LD];
  if (tid < m) lam_out[base + tid] = sh.lam[tid];
}

// the deflation of the top merge of the two halves (eigenvalues lam, eigenvectors Qb)
__global__ __launch_bounds__(DC_NT) void dc_top_kernel(const double* __restrict__ e, int m, double* __restrict__ Qb, DcTop top,
                                                       double* __restrict__ lam, const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  __shared__ DcShared<JACOBI_MAX> sh;
  const int tid = threadIdx.x;
  if (m == 1) {   // Qb = 1, one deflated column
    if (tid == 0) {
      *top.K = 0;
      top.dcol[0] = 0;
    }
    return;
  }
  if (tid == 0) sh.floor = 0.0;   // the node is the whole matrix
  if (tid < m) {
    sh.lam[tid] = lam[tid];
    sh.nmd[tid] = 0;
    sh.nmz[tid] = 0;
  }
  __syncthreads();
  dc_gather(sh, e, m, 0, Qb, m, tid);
  __syncthreads();
  if (tid < 64) dc_scan_wave(sh, e, 0, m, tid);
  __syncthreads();
  dc_rotate(sh, Qb, m, m, tid);
  const int K = sh.nK[0];
  if (tid < m) {
    if (tid < K) {
      top.dK[tid] = sh.dK[tid];
      top.zK[tid] = sh.zK[tid];
      top.z2[tid] = sh.z2[tid];
      top.kc[tid] = sh.kc[tid];
    } else {
      top.dcol[tid] = sh.dcol[tid];
      lam[tid] = sh.dvl[tid];
    }
  }
  if (tid == 0) {
    *top.K = K;
    *top.rho = sh.nRho[0];
  }
}

// the top merge's secular roots, one wavefront per root (all 64 lanes share its sums): root j's pole and
// offset, and its eigenvalue
__global__ __launch_bounds__(64) void dc_sec_kernel(DcTop top, double* __restrict__ lam_out,
                                                    const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  const int j = blockIdx.x, lane = threadIdx.x;
  const int K = *top.K;
  if (j >= K) return;
  __shared__ double dk[JACOBI_MAX], z2[JACOBI_MAX];
  for (int i = lane; i < K; i += 64) {
    dk[i] = top.dK[i];
    z2[i] = top.z2[i];
  }
  __syncthreads();
  int o;
  double t;
  dc_secular<64, JACOBI_MAX / 64>(dk, z2, K, j, lane, o, t);
  if (lane == 0) {
    top.org[j] = o;
    top.tau[j] = t;
    lam_out[j] = dk[o] + t;
  }
}

// the top merge's z recomputed from its roots (Lowner's formula), one wavefront per entry
__global__ __launch_bounds__(64) void dc_zh_kernel(DcTop top, const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  const int i = blockIdx.x, lane = threadIdx.x;
  const int K = *top.K;
  if (i >= K) return;
  const double rho = *top.rho, di = top.dK[i];
  double p = 1.0;
  for (int jj = lane; jj < K; jj += 64) {
    const double lmd = (top.dK[top.org[jj]] - di) + top.tau[jj];
    const double den = jj == K - 1 ? rho : (jj < i ? top.dK[jj] - di : top.dK[jj + 1] - di);
    p *= div_nr(lmd, den);
  }
  p = prodL<64>(p);
  if (lane == 0) top.zh[i] = copysign(sqrt(fmax(p, 0.0)), top.zK[i]);
}

// W = Z M for the top merge, Z = Qb (the children's eigenvectors, deflation-rotated and back-transformed):
// column t < K of M holds the normalised eigenvector zhat_i / (d_i - lambda_t) of the merge on the rows kc_i,
// a deflated column t >= K is column dcol_t of Z.  A 16 x 16 tile of W per workgroup on the FP64 matrix
// cores, over the whole chip; each workgroup forms the norms of its 16 columns and the entries of M it needs.
__global__ __launch_bounds__(64) void dc_final_kernel(const double* __restrict__ Z, DcTop top, int m,
                                                      double* __restrict__ W, const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  __shared__ double dk[JACOBI_MAX], zh[JACOBI_MAX];
  __shared__ int kc[JACOBI_MAX];
  const int lane = threadIdx.x, li = lane & 15, lk = lane >> 4;
  const int r0 = 16 * blockIdx.x, t0 = 16 * blockIdx.y;
  const int K = *top.K;
  for (int i = lane; i < K; i += 64) {
    dk[i] = top.dK[i];
    zh[i] = top.zh[i];
    kc[i] = top.kc[i];
  }
  __syncthreads();
  // this lane's column t = t0 + li: its root's pole and offset, and its norm (four lanes per column)
  const int tb = t0 + li;
  const bool kept = tb < K;
  const double dorg = kept ? dk[top.org[tb]] : 0.0, tt = kept ? top.tau[tb] : 0.0;
  double sq = 0.0;
  if (kept)
    for (int i = lk; i < K; i += 4) {
      const double u = div_nr(zh[i], (dk[i] - dorg) - tt);
      sq += u * u;
    }
  sq += __shfl_xor(sq, 16);
  sq += __shfl_xor(sq, 32);
  const double rn = kept ? 1.0 / sqrt(sq) : 0.0;
  const int ra = r0 + li;
  const int rac = min(ra, m - 1);   // rows beyond m only feed outputs that are not stored
  d4 acc = {0.0, 0.0, 0.0, 0.0};
  for (int p = 0; p < K; p += 64) {
    double a[16], b[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int i = min(p + 4 * u + lk, K - 1);
      a[u] = Z[rac + (size_t)kc[i] * m];
      b[u] = div_nr(zh[i], (dk[i] - dorg) - tt) * rn;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 16; ++u)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], (kept && p + 4 * u + lk < K) ? b[u] : 0.0, acc, 0, 0, 0);
  }
  // register q holds row lk + 4 q, column li; deflated columns are copied
  const int src = kept ? 0 : (tb < m ? top.dcol[tb] : 0);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = r0 + lk + 4 * q;
    if (r < m && tb < m) W[r + (size_t)tb * m] = kept ? acc[q] : Z[r + (size_t)src * m];
  }
}


// Z <- H_0 H_1 ... H_(m-3) Z in place, one wavefront per column.  The reflectors are applied four at a
// time: with s_q = tau_q (u_q . z - sum_(p<q) s_p u_q . u_p) for the block's reflectors u_0..u_3 in the
// order of application, z - sum_q s_q u_q is the product of the four; the four products with z share one
// reduction, and the six among the u come from trd_gram_kernel (lanes 0..5 of one register per block).
// Each lane needs only its own entries of the reflectors (rows lane, lane + 64, lane + 128), so they are
// prefetched in chunks of 16 reflectors into registers, one chunk ahead (two register sets, the loop
// unrolled by two); the reflector count is padded to whole pairs of chunks with tau = 0.
constexpr int BK_Q = 16;

// the six products u_q . u_p (p < q) among each block of four reflectors, in the order the back-transformation
// uses them (u1.u0, u2.u0, u2.u1, u3.u0, u3.u1, u3.u2), once for all columns: one wavefront per block, over
// the padded reflector count (a padding reflector is column 0 again, finite, with tau = 0)
__global__ __launch_bounds__(64) void trd_gram_kernel(const double* __restrict__ Vh, int m, double* __restrict__ gram,
                                                      const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  const int b = blockIdx.x, lane = threadIdx.x;
  double u[4][3];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = m - 3 - (4 * b + q);
    const double* v = Vh + (size_t)(j >= 0 ? j : 0) * m;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int r = lane + 64 * k;
      const double x = v[r < m ? r : m - 1];
      u[q][k] = r < m ? x : 0.0;
    }
  }
  double d[6];
  int n = 0;
#pragma unroll
  for (int q = 1; q < 4; ++q)
#pragma unroll
    for (int p = 0; p < q; ++p, ++n) d[n] = u[q][0] * u[p][0] + u[q][1] * u[p][1] + u[q][2] * u[p][2];
  wave_sums<6>(d);
  if (lane < 6) {
    double x = d[0];
#pragma unroll
    for (int k = 1; k < 6; ++k) x = lane == k ? d[k] : x;
    gram[6 * b + lane] = x;
  }
}

__device__ __forceinline__ void back_load(const double* __restrict__ Vh, const double* __restrict__ tau,
                                          const double* __restrict__ gram, int m, int q0, int lane,
                                          double (&u)[BK_Q][3], double (&t)[BK_Q], double (&g)[BK_Q / 4]) {
  const int nblk = ((m - 2 + 2 * BK_Q - 1) / (2 * BK_Q)) * (BK_Q / 2);   // blocks trd_gram_kernel wrote
#pragma unroll
  for (int b = 0; b < BK_Q / 4; ++b)   // lane k: product k (a prefetch past the last block rereads it, unused)
    g[b] = gram[6 * min(q0 / 4 + b, nblk - 1) + (lane < 6 ? lane : 5)];
  // raw loads from clamped addresses (no select on a loaded value here, which would wait for it): a padding
  // reflector gets tau = 0, so whatever it holds has weight 0, and rows >= m are masked where they are used
#pragma unroll
  for (int i = 0; i < BK_Q; ++i) {
    const int j = m - 3 - (q0 + i);   // reflectors in the order of application
    const bool ok = j >= 0;
    const double tj = tau[ok ? j : 0];
    t[i] = ok ? tj : 0.0;
    const double* v = Vh + (size_t)(ok ? j : 0) * m;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int r = lane + 64 * k;
      u[i][k] = v[r < m ? r : m - 1];
    }
  }
}

__device__ __forceinline__ void back_apply(double (&z)[3], const double (&uraw)[BK_Q][3], const double (&t)[BK_Q],
                                           const double (&g)[BK_Q / 4], const bool (&rk)[3]) {
#pragma unroll
  for (int b = 0; b < BK_Q; b += 4) {
    double u[BK_Q][3];
#pragma unroll
    for (int q = b; q < b + 4; ++q)
#pragma unroll
      for (int k = 0; k < 3; ++k) u[q][k] = rk[k] ? uraw[q][k] : 0.0;
    double d[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) d[q] = u[b + q][0] * z[0] + u[b + q][1] * z[1] + u[b + q][2] * z[2];
    wave_sums<4>(d);
    const double gb = g[b / 4];
    const double g10 = lane_of(gb, 0), g20 = lane_of(gb, 1), g21 = lane_of(gb, 2), g30 = lane_of(gb, 3),
                 g31 = lane_of(gb, 4), g32 = lane_of(gb, 5);
    const double s0 = t[b] * d[0];
    const double s1 = t[b + 1] * (d[1] - s0 * g10);
    const double s2 = t[b + 2] * (d[2] - s0 * g20 - s1 * g21);
    const double s3 = t[b + 3] * (d[3] - s0 * g30 - s1 * g31 - s2 * g32);
#pragma unroll
    for (int k = 0; k < 3; ++k) z[k] -= s0 * u[b][k] + s1 * u[b + 1][k] + s2 * u[b + 2][k] + s3 * u[b + 3][k];
  }
}

// one wavefront per SIMD is all the grid has, so the scheduler may spend every register on the prefetch
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1))) void trd_back_kernel(
    const double* __restrict__ Vh, const double* __restrict__ tau, const double* __restrict__ gram, int m,
    double* __restrict__ Z, const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  const int c = blockIdx.x, lane = threadIdx.x;
  double* zc = Z + (size_t)c * m;
  double z[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) z[k] = lane + 64 * k < m ? zc[lane + 64 * k] : 0.0;
  const int nr = m - 2;
  const bool rk[3] = {lane < m, lane + 64 < m, lane + 128 < m};
  double ua[BK_Q][3], ta[BK_Q], ga[BK_Q / 4], ub[BK_Q][3], tb[BK_Q], gb[BK_Q / 4];
  back_load(Vh, tau, gram, m, 0, lane, ua, ta, ga);
  // whole pairs of chunks, no exit between a chunk's loads and their use (a conditional one would let the
  // compiler sink the loads past the other chunk's work)
  // (the scheduling barriers keep the machine scheduler from moving the loads down to their uses)
  for (int q = 0; q < nr; q += 2 * BK_Q) {
    back_load(Vh, tau, gram, m, q + BK_Q, lane, ub, tb, gb);
    __builtin_amdgcn_sched_barrier(0);
    back_apply(z, ua, ta, ga, rk);
    back_load(Vh, tau, gram, m, q + 2 * BK_Q, lane, ua, ta, ga);
    __builtin_amdgcn_sched_barrier(0);
    back_apply(z, ub, tb, gb, rk);
  }
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (lane + 64 * k < m) zc[lane + 64 * k] = z[k];
}

// Instances for m up to 48, 96, 144, 192 (us at m = 20 / 48 / 80 / 128 with the last one for all: 48 / 102 / 159 / 229;
// with these: 24 / 52 / 98 / 189)
void trd_launch(const double* H, int ldh, int m, double* d, double* e, double* Vh, double* tau, double* scale,
                const int* gate, hipStream_t s) {
  if (m <= 48) hipLaunchKernelGGL((trd_kernel<2, 3>), dim3(1), dim3(TD_NT), 0, s, H, ldh, m, d, e, Vh, tau, scale, gate);
  else if (m <= 96) hipLaunchKernelGGL((trd_kernel<3, 6>), dim3(1), dim3(TD_NT), 0, s, H, ldh, m, d, e, Vh, tau, scale, gate);
  else if (m <= 144) hipLaunchKernelGGL((trd_kernel<5, 9>), dim3(1), dim3(TD_NT), 0, s, H, ldh, m, d, e, Vh, tau, scale, gate);
  else hipLaunchKernelGGL((trd_kernel<6, 12>), dim3(1), dim3(TD_NT), 0, s, H, ldh, m, d, e, Vh, tau, scale, gate);
  TNAD_HIP_TRY(hipGetLastError());
}

// the work buffer: Vh, Qa, Qb (m x m each), d, e, tau, lambda (m each), the reflector block products, the scale
struct DcWork {
  double *Vh, *Qa, *Qb, *dv, *ev, *tau, *lam, *gram, *scale;
  DcTop top;
};

DcWork dc_work(double* w, int m) {
  const size_t mm = (size_t)m * m;
  DcWork d;
  d.Vh = w;
  d.Qa = d.Vh + mm;
  d.Qb = d.Qa + mm;
  d.dv = d.Qb + mm;
  d.ev = d.dv + m;
  d.tau = d.ev + m;
  d.lam = d.tau + m;
  d.gram = d.lam + m;   // 6 per block of four reflectors, the count padded to 32: at most 1.5 m + 44
  d.scale = d.gram + 2 * (size_t)m + 47;
  double* t = d.gram + 2 * (size_t)m + 48;   // the top merge: 5 m doubles, rho, then 3 m + 1 ints
  d.top.dK = t;
  d.top.zK = t + m;
  d.top.z2 = t + 2 * m;
  d.top.tau = t + 3 * m;
  d.top.zh = t + 4 * m;
  d.top.rho = t + 5 * m;
  int* ti = reinterpret_cast<int*>(t + 5 * m + 1);
  d.top.kc = ti;
  d.top.dcol = ti + m;
  d.top.org = ti + 2 * m;
  d.top.K = ti + 3 * m;
  return d;
}

// blocks of four reflectors that trd_back_kernel reads (m - 2 padded to a multiple of 32)
int dc_gram_blocks(int m) { return m > 2 ? ((m - 2 + 2 * BK_Q - 1) / (2 * BK_Q)) * (BK_Q / 2) : 0; }

// the divide and conquer: the merge tree below the top merge in a workgroup per half, the top merge's deflation in one, its
// roots and z over the whole chip
void dc_solve(const DcWork& w, int m, const int* gate, hipStream_t s) {
  const int half = (m + 1) / 2;
  if (half <= 48) hipLaunchKernelGGL((dc_kernel<8, 48>), dim3(2), dim3(DC_NT), 0, s, w.dv, w.ev, m, w.Qa, w.Qb, w.lam, gate);
  else if (half <= DC_QL) hipLaunchKernelGGL((dc_kernel<8, DC_QL>), dim3(2), dim3(DC_NT), 0, s, w.dv, w.ev, m, w.Qa, w.Qb, w.lam, gate);
  else hipLaunchKernelGGL((dc_kernel<8, 96>), dim3(2), dim3(DC_NT), 0, s, w.dv, w.ev, m, w.Qa, w.Qb, w.lam, gate);
  TNAD_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(dc_top_kernel, dim3(1), dim3(DC_NT), 0, s, w.ev, m, w.Qb, w.top, w.lam, gate);
  TNAD_HIP_TRY(hipGetLastError());
  if (m > 1) {
    hipLaunchKernelGGL(dc_sec_kernel, dim3(m), dim3(64), 0, s, w.top, w.lam, gate);
    TNAD_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(dc_zh_kernel, dim3(m), dim3(64), 0, s, w.top, gate);
    TNAD_HIP_TRY(hipGetLastError());
  }
}

// the eigenvectors: block products and back-transformation of the children's eigenvectors, then the top
// merge's product (into Qa)
void dc_vectors(const DcWork& w, int m, const int* gate, hipStream_t s) {
  if (m > 2) {
    hipLaunchKernelGGL(trd_gram_kernel, dim3(dc_gram_blocks(m)), dim3(64), 0, s, w.Vh, m, w.gram, gate);
    TNAD_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(trd_back_kernel, dim3(m), dim3(64), 0, s, w.Vh, w.tau, w.gram, m, w.Qb, gate);
    TNAD_HIP_TRY(hipGetLastError());
  }
  const int nt = (m + 15) / 16;
  hipLaunchKernelGGL(dc_final_kernel, dim3(nt, nt), dim3(64), 0, s, w.Qb, w.top, m, w.Qa, gate);
  TNAD_HIP_TRY(hipGetLastError());
}

}  // namespace

size_t syev_dc_work_doubles(int m) { return 3 * (size_t)m * m + 13 * (size_t)m + 56; }

void syev_dc(const double* H, int ldh, int m, double* evals, double* V, double* work, hipStream_t s,
             const int* gate) {
  if (m < 1 || m > JACOBI_MAX) throw Error(TNAD_ERR_ARG, "syev_dc: size out of range");
  const DcWork w = dc_work(work, m);
  trd_launch(H, ldh, m, w.dv, w.ev, w.Vh, w.tau, w.scale, gate, s);
  dc_solve(w, m, gate, s);
  dc_vectors(w, m, gate, s);
  sort_eigenpairs(w.lam, w.Qa, m, evals, V, gate, s, w.scale);
}

void syev_dc_time(const double* H, int m, int reps, double* work, hipStream_t s, float ms[3]) {
  if (m < 3 || m > JACOBI_MAX || reps < 1) throw Error(TNAD_ERR_ARG, "syev_dc_time: bad sizes");
  const DcWork w = dc_work(work, m);
  double* V = work + syev_dc_work_doubles(m);   // m x m sorted eigenvectors
  double* evals = V + (size_t)m * m;
  hipEvent_t e[4];
  for (auto& x : e) TNAD_HIP_TRY(hipEventCreate(&x));
  float acc[3] = {0.f, 0.f, 0.f};
  for (int r = 0; r <= reps; ++r) {   // the first run warms up
    TNAD_HIP_TRY(hipEventRecord(e[0], s));
    trd_launch(H, m, m, w.dv, w.ev, w.Vh, w.tau, w.scale, nullptr, s);
    TNAD_HIP_TRY(hipEventRecord(e[1], s));
    dc_solve(w, m, nullptr, s);
    TNAD_HIP_TRY(hipEventRecord(e[2], s));
    dc_vectors(w, m, nullptr, s);
    sort_eigenpairs(w.lam, w.Qa, m, evals, V, nullptr, s, w.scale);
    TNAD_HIP_TRY(hipEventRecord(e[3], s));
    TNAD_HIP_TRY(hipEventSynchronize(e[3]));
    if (r == 0) continue;
    for (int k = 0; k < 3; ++k) {
      float t = 0.f;
      TNAD_HIP_TRY(hipEventElapsedTime(&t, e[k], e[k + 1]));
      acc[k] += t;
    }
  }
  for (auto& x : e) (void)hipEventDestroy(x);
  for (int k = 0; k < 3; ++k) ms[k] = acc[k] / reps;
}

}  // namespace tnad
