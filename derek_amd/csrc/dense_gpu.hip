// FP64 dense subspace solvers on the GPU for batches of matrices.
//
// heev_gpu: lowest nev eigenpairs of a Hermitian n x n matrix.
//   1. Householder reduction to real tridiagonal form: while the trailing
//      matrix exceeds 128 columns, one multi-workgroup launch per column on the
//      matrix in global memory (L2 resident); then the last 128 columns in the
//      registers of one workgroup (matrix-core rank-2 updates, look-ahead
//      reflector, two barriers per column).  The reflectors overwrite the
//      eliminated columns.
//   2. Phases that make the sub-diagonal real and non-negative (a prefix
//      product over the workgroup).
//   3. Sturm-sequence multisection for the lowest nev eigenvalues, one
//      wavefront each (64 points per step).
//   4. Inverse iteration for the eigenvectors of the tridiagonal matrix with
//      partial-pivoting LU; eigenvalues closer than 1e-5 |T| form a cluster
//      whose vectors are computed by one thread in order and re-orthogonalised
//      (modified Gram-Schmidt) against the earlier members.
//   5. Back-transformation by the reflectors, one wavefront per vector.
// chol_inverse_gpu: inverse Cholesky factor of a unit-diagonal Hermitian
//   overlap, skipping every column whose remaining pivot is below tol (dependent
//   on earlier columns); many workgroups, one launch per panel of columns.
#include <cfloat>
#include <type_traits>

#include "dense_gpu.hpp"
#include "launch.hpp"

namespace derek {

constexpr int DT = 1024;  // threads per workgroup
constexpr int DW = DT / 64;

__device__ __forceinline__ double2 zmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 zconjmul(double2 a, double2 b) {  // conj(a) * b
  return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}

// One DPP move of a double (both 32-bit halves) with the given control and
// row mask; lanes without a source (or outside the mask) read 0.
template <int CTRL, int ROWS = 0xf> __device__ __forceinline__ double dpp_move(double x) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b & 0xffffffffull), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROWS, 0xf, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Sum over the 64 lanes of a wave (all lanes active), every lane gets it:
// quad butterflies, row shifts by 4 and 8 (lane 15 of each row holds the row
// sum), row broadcasts 15 and 31 (lane 63 holds the total), then a readlane.
// Cross-lane moves on the VALU instead of LDS permutes.
__device__ __forceinline__ double wave_sum(double x) {
  x += dpp_move<0xb1>(x);        // quad_perm [1,0,3,2]
  x += dpp_move<0x4e>(x);        // quad_perm [2,3,0,1]
  x += dpp_move<0x114>(x);       // row_shr:4
  x += dpp_move<0x118>(x);       // row_shr:8
  x += dpp_move<0x142, 0xa>(x);  // row_bcast:15 into rows 1 and 3
  x += dpp_move<0x143, 0xc>(x);  // row_bcast:31 into rows 2 and 3
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b & 0xffffffffull), 63);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), 63);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Maximum over the workgroup; every thread gets the result.
__device__ double block_max_all(double x, double* red) {
  for (int o = 32; o > 0; o >>= 1) x = fmax(x, __shfl_down(x, o, 64));
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wid] = x;
  __syncthreads();
  double t = red[0];
  for (int w = 1; w < DW; ++w) t = fmax(t, red[w]);
  return t;
}

// 1/q for q != 0: the hardware estimate refined by two Newton steps, fewer
// issue cycles than the division sequence (the Sturm recurrence below is
// bound by its wavefront's issue rate).  q is clamped to the finite range
// first, so an infinite q gives 0 as the division would.
__device__ __forceinline__ double recip_nr(double q) {
  const double qc = fmin(fmax(q, -DBL_MAX), DBL_MAX);
  double y = __builtin_amdgcn_rcp(qc);
  double e = fma(-qc, y, 1.0);
  y = fma(y, e, y);
  e = fma(-qc, y, 1.0);
  return fma(y, e, y);
}

// number of eigenvalues of the tridiagonal (d, e) smaller than x
__device__ int sturm_count(const double* d, const double* e2, int n, double x, double pivmin) {
  int c = 0;
  double q = d[0] - x;
  if (fabs(q) < pivmin) q = -pivmin;
  if (q < 0.0) ++c;
  for (int i = 1; i < n; ++i) {
    q = d[i] - x - e2[i - 1] * recip_nr(q);
    if (fabs(q) < pivmin) q = -pivmin;
    if (q < 0.0) ++c;
  }
  return c;
}

// Solve (T - lambda I) x = b by LU with partial pivoting; T has diagonal d and
// off-diagonal e.  u0/u1/u2/l/pv are scratch of length n; b is overwritten by x.
// LU factorisation with partial pivoting of T - lambda I (T symmetric
// tridiagonal: diagonal d, off-diagonal e), pivots below pivmin raised to it;
// U has the three diagonals (u0 holds the reciprocals of the pivots, so the
// solves multiply), L the multipliers l with row swaps pv.  The arrays are
// separate LDS regions (restrict), so the loads of the next row are issued
// while the recurrence runs in registers.
__device__ void tri_factor(const double* __restrict__ d, const double* __restrict__ e, int n, double lambda,
                           double pivmin, double* __restrict__ u0, double* __restrict__ u1, double* __restrict__ u2,
                           double* __restrict__ l, double* __restrict__ pv) {
  double cd = d[0] - lambda, cs = n > 1 ? e[0] : 0.0, cs2 = 0.0;
  for (int i = 0; i + 1 < n; ++i) {
    const double c = e[i];
    const double a1 = d[i + 1] - lambda;
    const double b1 = i + 2 < n ? e[i + 1] : 0.0;
    if (fabs(cd) >= fabs(c)) {
      const double piv = fabs(cd) < pivmin ? copysign(pivmin, cd == 0.0 ? 1.0 : cd) : cd;
      const double rp = recip_nr(piv);
      const double li = c * rp;
      u0[i] = rp;
      u1[i] = cs;
      u2[i] = cs2;
      l[i] = li;
      pv[i] = 0.0;
      cd = a1 - li * cs;
      cs = b1 - li * cs2;
      cs2 = 0.0;
    } else {
      const double rc = recip_nr(c);
      const double li = cd * rc;
      u0[i] = rc;
      u1[i] = a1;
      u2[i] = b1;
      l[i] = li;
      pv[i] = 1.0;
      cd = cs - li * a1;
      cs = cs2 - li * b1;
      cs2 = 0.0;
    }
  }
  u0[n - 1] = recip_nr(fabs(cd) < pivmin ? copysign(pivmin, cd == 0.0 ? 1.0 : cd) : cd);
}

// b <- (T - lambda I)^-1 b from tri_factor's factors; the values carried from
// row to row stay in registers and the next row's operands are loaded one
// step ahead, so each step waits only on its own arithmetic.
__device__ void tri_solve(int n, const double* __restrict__ u0, const double* __restrict__ u1,
                          const double* __restrict__ u2, const double* __restrict__ l, const double* __restrict__ pv,
                          double* __restrict__ b) {
  double bi = b[0];
  if (n > 1) {
    double nb = b[1], nl = l[0], np = pv[0];
    for (int i = 0; i + 1 < n; ++i) {
      double bn = nb;
      const double li = nl, pi = np;
      if (i + 2 < n) {
        nb = b[i + 2];
        nl = l[i + 1];
        np = pv[i + 1];
      }
      if (pi != 0.0) {
        const double t = bi;
        bi = bn;
        bn = t;
      }
      bn -= li * bi;
      b[i] = bi;
      bi = bn;
    }
  }
  double b1 = bi * u0[n - 1];  // b[i+1]
  b[n - 1] = b1;
  if (n < 2) return;
  double b0 = (b[n - 2] - u1[n - 2] * b1) * u0[n - 2];  // b[i+1] after the step below
  b[n - 2] = b0;
  if (n < 3) return;
  double cb = b[n - 3], c1 = u1[n - 3], c2 = u2[n - 3], cr = u0[n - 3];
  for (int i = n - 3; i >= 0; --i) {
    const double xb = cb, x1 = c1, x2 = c2, xr = cr;
    if (i > 0) {
      cb = b[i - 1];
      c1 = u1[i - 1];
      c2 = u2[i - 1];
      cr = u0[i - 1];
    }
    const double bi2 = (xb - x1 * b0 - x2 * b1) * xr;
    b[i] = bi2;
    b1 = b0;
    b0 = bi2;
  }
}

// Per-matrix workspace layout (doubles), see heev_work_doubles.
struct HeevWork {
  double2* sub;  // [n]  T(k+1,k) before the phase change
  double2* ph;   // [n]  phases
  double2* vb;   // [2n] reflector vectors of the wide reduction, double-buffered by k&1
  double2* uu;   // [2n] A v of the wide reduction, double-buffered by k&1
  double* d;     // [n]  diagonal
  double* e;     // [n]  |sub|
  double* lam;   // [nev]
  double* scal;  // [8]  wide reduction: (skip, 1/|v|, v0) per buffer
  double* xt;    // [n * nev] tridiagonal eigenvectors
  int* skip;     // [n]  1 if column k needed no reflector
  int* cstart;   // [nev + 1]
  int* ncl;      // [1]
  __device__ __host__ HeevWork(double* w, int n, int nev) {
    sub = reinterpret_cast<double2*>(w);
    ph = sub + n;
    vb = ph + n;
    uu = vb + 2 * n;
    d = reinterpret_cast<double*>(uu + 2 * n);
    e = d + n;
    lam = e + n;
    scal = lam + nev;
    xt = scal + 8;
    skip = reinterpret_cast<int*>(xt + (size_t)n * nev);
    cstart = skip + n;
    ncl = cstart + nev + 1;
  }
};

int64_t heev_work_doubles(int n, int nev) {
  // rounded to 256 bytes so every matrix of a batch starts aligned
  const int64_t w = 14 * (int64_t)n + nev + 8 + (int64_t)n * nev + (n + nev + 2 + 1) / 2 + 8;
  return (w + 31) / 32 * 32;
}

// ---- 1. Householder tridiagonalisation + phases
// Columns 0 .. n-129 (n > 128) take one multi-workgroup launch each
// (k_wide_step: the rank-2 update of column k's reflector, fused with the
// next reflector and u = A v for it); the trailing block of at most 128
// columns is loaded into registers and reduced by one workgroup per matrix
// (k_tridiag).

// e = |sub| and the phases ph[0] = 1, ph[k+1] = ph[k] f_k, f_k = sub_k/|sub_k|
// (1 where sub_k = 0), that make D^H T D real.  The phases are a prefix
// product of unit complex numbers: each thread takes four consecutive f_k
// (n <= 2048 = 4 TDT), the threads' products are scanned across the lanes of
// each wavefront and then across the wavefronts (s_wave: TDT / 64 entries).
constexpr int TDT = 512;  // threads of k_tridiag
__device__ void tri_phases(HeevWork& W, int n, double2* s_wave) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const double2 one = make_double2(1.0, 0.0);
  double2 f[4], q = one;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int k = 4 * tid + r;
    f[r] = one;
    if (k + 1 < n) {
      const double2 sk = W.sub[k];
      const double a = sqrt(sk.x * sk.x + sk.y * sk.y);
      W.e[k] = a;
      if (a > 0.0) f[r] = make_double2(sk.x / a, sk.y / a);
    }
    q = zmul(q, f[r]);
  }
  // inclusive scan of the thread products over the wavefront
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double2 t = make_double2(__shfl_up(q.x, o, 64), __shfl_up(q.y, o, 64));
    if (lane >= o) q = zmul(t, q);
  }
  if (lane == 63) s_wave[wid] = q;
  __syncthreads();
  double2 p = one;
  for (int w = 0; w < wid; ++w) p = zmul(p, s_wave[w]);
  double2 ex = make_double2(__shfl_up(q.x, 1, 64), __shfl_up(q.y, 1, 64));
  if (lane == 0) ex = one;
  p = zmul(p, ex);  // ph[4 tid]
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int k = 4 * tid + r;
    p = zmul(p, f[r]);
    if (k + 1 < n) W.ph[k + 1] = p;
  }
  if (tid == 0) {
    W.ph[0] = one;
    W.e[n - 1] = 0.0;
  }
}


// 1/sqrt(x) for x > 0 within a few ulps: the hardware estimate refined by two
// Newton steps, a shorter dependent chain than a square root and a division
__device__ __forceinline__ double rsqrt_nr(double x) {
  double y = __builtin_amdgcn_rsq(x);
  double e = fma(-x * y, y, 1.0);
  y = fma(0.5 * y, e, y);
  e = fma(-x * y, y, 1.0);
  return fma(0.5 * y, e, y);
}

__device__ __forceinline__ double read_lane(double x, int l) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b & 0xffffffffull), l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Householder scalars of column k from tail2 = sum_{i>k+1} |A(i,k)|^2 and
// x0 = A(k+1,k) (both wave-uniform): alpha = -(x0/|x0|) ||x|| (the new
// sub-diagonal), v0 = x0 - alpha and iv = 1/||v|| with
// ||v||^2 = 2 ||x|| (||x|| + |x0|); skip when x is already reduced, which the
// tail alone decides: in ||x||^2 - |x0|^2 entries below 1e-8 |x0| are lost.
// When rec is set the caller's lane records alpha and the skip flag.
__device__ __forceinline__ void tri_scalars(bool rec, int k, double tail2, double2 x0, HeevWork& W, int& skip,
                                            double& iv, double2& v0) {
  // without branches: the two square roots overlap
  const double a2 = x0.x * x0.x + x0.y * x0.y, xn2 = a2 + tail2;
  skip = tail2 <= 1e-300 ? 1 : 0;
  const double rx = rsqrt_nr(xn2), ra = rsqrt_nr(a2), xn = xn2 * rx;
  const bool nz = a2 > 0.0;
  const double ax0 = nz ? a2 * ra : 0.0;
  const double2 phs = make_double2(nz ? x0.x * ra : 1.0, nz ? x0.y * ra : 0.0);
  const double r = rsqrt_nr(2.0 * xn * (xn + ax0));
  const double2 alpha = skip ? x0 : make_double2(-phs.x * xn, -phs.y * xn);
  iv = skip ? 0.0 : r;
  v0 = make_double2(skip ? 0.0 : x0.x + phs.x * xn, skip ? 0.0 : x0.y + phs.y * xn);
  if (rec) {
    W.skip[k] = skip;
    W.sub[k] = alpha;
  }
}

// Reflector of column k from sum |A(i,k)|^2 (i > k+1) and x0 = A(k+1,k), both
// wave-uniform, for the multi-workgroup steps: every lane derives the
// scalars, lane 0 records them (with the scalars for the next launch).
__device__ __forceinline__ void wide_reflector_scalars(int lane, int k, double tail2, double2 x0, HeevWork& W,
                                                       int& skip, double& iv, double2& v0) {
  tri_scalars(lane == 0, k, tail2, x0, W, skip, iv, v0);
  if (lane == 0) {
    double* sc = W.scal + 4 * (k & 1);
    sc[0] = skip;
    sc[1] = iv;
    sc[2] = v0.x;
    sc[3] = v0.y;
  }
}

// Sum over the lanes l, l ^ 16, l ^ 32, l ^ 48, every lane gets it.
__device__ __forceinline__ double cross_row_sum(double x) {
  auto halves = [](double y, auto swap) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(y);
    const unsigned lo = (unsigned)(b & 0xffffffffull), hi = (unsigned)(b >> 32);
    const auto l = swap(lo), h = swap(hi);
    return __longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0])) +
           __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1]));
  };
  x = halves(x, [](unsigned w) { return __builtin_amdgcn_permlane16_swap(w, w, false, false); });
  return halves(x, [](unsigned w) { return __builtin_amdgcn_permlane32_swap(w, w, false, false); });
}

// Sum over the 16 lanes of a row, every lane gets it.
__device__ __forceinline__ double row_sum(double x) {
  x += dpp_move<0x128>(x);  // row_ror:8, 4, 2, 1
  x += dpp_move<0x124>(x);
  x += dpp_move<0x122>(x);
  return x + dpp_move<0x121>(x);
}
// Lane L of every row of 16 in all lanes of the row.
template <int L> __device__ __forceinline__ double row_bcast(double x) {
  return __longlong_as_double(__builtin_amdgcn_update_dpp(0ll, __double_as_longlong(x), 0x150 + L, 0xf, 0xf, true));
}

// Householder reduction of the trailing block A[k0:, k0:] (nb = n - k0 <= TNB
// rows and columns) in registers, one workgroup per matrix: the whole matrix
// for k0 = 0, or the tail after the multi-workgroup steps 0..k0-1.  Indices
// below are local to the block.  The block, both triangles, lies in 16 x 16
// accumulator tiles of the FP64 matrix cores: wavefront w holds columns
// 16 w + (lane & 15), tile t of it the rows 16 t + (lane >> 4) + 4 r.
// v, u and the next column go through LDS.  Per column c, with v in LDS:
//   1. u = A^H v = A v: a lane sums its column over its rows (v of the rows
//      is one LDS read per 64 rows, handed round the 16 columns by DPP), four
//      lanes share a column; the wavefronts' parts of gamma = v^H u to LDS;
//   2. A -= v (2u - 2 gamma v)^H + u (2v)^H, the rank-2 update of the
//      reflector, two matrix instructions per tile: (v, u) of the rows
//      against the columns' pair for the real part, against i times it for
//      the imaginary one.  One wavefront first updates column c+1 (a copy in
//      LDS) and forms its reflector.
// Two barriers per column; tiles left of and above column c+1 are skipped.
// v is zero outside rows c+1.. and u outside columns c+1.., so nothing else
// needs masks, and a column without a reflector is one with v = 0.
//
// Bound: the chain from one reflector to the next (two barriers, three
// reductions, the scalars of tri_scalars: 3100 cycles per column) and, on the
// first columns, the vector ALU in 1 and the matrix cores in 2 (6300 cycles).
// The block in LDS (98 columns at most, lower triangle) took 2.9 us per
// column, 32 us for 20 columns: this takes 2.0 and 24, and the 30 columns
// more save a launch of 5 us each (k_wide_step).  One matrix of 160 columns:
// 310 + 62 * 5.0 us -> 250 + 32 * 5.0 us.
constexpr int TNB = 128;       // rows and columns of the register block
constexpr int TW = TDT / 64;   // wavefronts, one per 16 columns

__global__ __launch_bounds__(TDT) void k_tridiag(double2* __restrict__ Aall, int lda_g, int64_t strideA, int n,
                                                int k0, int nev, double* __restrict__ work, int64_t strideWork) {
  typedef double d4 __attribute__((ext_vector_type(4)));
  static_assert(TNB == 16 * TW && TNB == 128, "a wavefront per 16 columns, two rows of the block per lane");
  __shared__ double2 s_vu[2][TNB][2];  // v (unit norm) and u of columns c and c + 1 (slot c & 1)
  __shared__ double s_col[2][2][TNB];  // column c + 1 (slot (c + 1) & 1; re, im) before the update of step c
  __shared__ double s_g[TW];           // the wavefronts' parts of v^H u
  __shared__ double2 s_ph[TW];
  const int nb = n - k0, nt = (nb + 15) / 16;
  const int mat = blockIdx.x;
  double2* Ag = Aall + mat * strideA + k0 + (int64_t)k0 * lda_g;
  HeevWork W(work + mat * strideWork, n, nev);
  const int tid = threadIdx.x, lane = tid & 63, ct = tid >> 6, l16 = lane & 15, lg = lane >> 4;
  const int j = 16 * ct + l16;  // this lane's column
  const int look = nt < TW ? TW - 1 : 0;  // the wavefront that forms the reflectors: one without columns, or soon
  d4 ar[TW], ai[TW];
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {  // from the lower triangle
      const int i = 16 * t + lg + 4 * r;
      double2 e = make_double2(0.0, 0.0);
      if (i < nb && j < nb) e = i >= j ? Ag[i + (int64_t)j * lda_g] : Ag[j + (int64_t)i * lda_g];
      ar[t][r] = e.x;
      ai[t][r] = i >= j ? e.y : -e.y;
    }
  // reflector of column c from its values x (rows lane and lane + 64, zero
  // outside c+1..nb-1): into s_vu and, for the back-transformation, column c
  auto reflector = [&](int c, const double2* x) {
    const int l = (c + 1) & 63;
    const bool hi = (c + 1) >> 6;  // row c + 1 is x[hi] of lane l
    const double q0 = x[0].x * x[0].x + x[0].y * x[0].y, q1 = x[1].x * x[1].x + x[1].y * x[1].y;
    const double part = wave_sum(lane == l ? (hi ? q0 : q1) : q0 + q1);
    const double2 y = hi ? x[1] : x[0];
    const double2 x0 = make_double2(read_lane(y.x, l), read_lane(y.y, l));
    int skip;
    double iv;
    double2 v0;
    tri_scalars(lane == 0, k0 + c, part, x0, W, skip, iv, v0);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int i = lane + 64 * q;
      const double2 a = i == c + 1 ? v0 : x[q];
      const double2 v = skip ? make_double2(0.0, 0.0) : make_double2(a.x * iv, a.y * iv);
      s_vu[c & 1][i][0] = v;
      if (i > c && i < nb) Ag[i + (int64_t)c * lda_g] = v;
    }
  };
  if (tid < TNB) {
    s_vu[0][tid][1] = s_vu[1][tid][1] = make_double2(0.0, 0.0);
    const double2 x = tid < nb && nb > 1 && tid >= 1 ? Ag[tid + lda_g] : make_double2(0.0, 0.0);
    s_col[1][0][tid] = x.x;
    s_col[1][1][tid] = x.y;
  }
  __syncthreads();  // columns 0 and 1 are read before the reflector overwrites column 0
  if (ct == look && nb >= 2) {
    double2 x[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int i = lane + 64 * q;
      x[q] = i >= 1 && i < nb ? Ag[i] : make_double2(0.0, 0.0);
    }
    if (nb > 2) {
      reflector(0, x);
    } else if (lane == 1) {
      W.sub[n - 2] = x[0];
      W.skip[n - 2] = 1;
    }
  }
  // the tiles are used here, before the loop: a wait for these loads inside it
  // would also wait for the reflectors' stores, once per column
#pragma unroll
  for (int t = 0; t < TW; ++t) asm volatile("" : "+v"(ar[t]), "+v"(ai[t]));
  __syncthreads();
  for (int c = 0; c + 2 < nb; ++c) {
    const int t0 = (c + 1) >> 4;  // first tile row and column still needed
    double2(*vu)[2] = s_vu[c & 1];
    if (ct >= t0 && ct < nt) {
      // v of this lane row's rows: lane 4 (t & 3) + r of half t >> 2 holds row 16 t + lg + 4 r
      const double2 vh[2] = {vu[4 * l16 + lg][0], vu[64 + 4 * l16 + lg][0]};
      const double2 vj = vu[j][0];
      double sr = 0.0, si = 0.0, tr = 0.0, ti = 0.0;
      auto rows = [&](auto tc, auto rc) {
        constexpr int t = decltype(tc)::value, r = decltype(rc)::value;
        const double vx = row_bcast<4 * (t & 3) + r>(vh[t >> 2].x), vy = row_bcast<4 * (t & 3) + r>(vh[t >> 2].y);
        sr += ar[t][r] * vx;
        si += ar[t][r] * vy;
        tr += ai[t][r] * vy;
        ti += ai[t][r] * vx;
      };
      auto tile = [&](auto tc) {
        if (decltype(tc)::value < t0 || decltype(tc)::value >= nt) return;
        rows(tc, std::integral_constant<int, 0>{});
        rows(tc, std::integral_constant<int, 1>{});
        rows(tc, std::integral_constant<int, 2>{});
        rows(tc, std::integral_constant<int, 3>{});
      };
      tile(std::integral_constant<int, 0>{});
      tile(std::integral_constant<int, 1>{});
      tile(std::integral_constant<int, 2>{});
      tile(std::integral_constant<int, 3>{});
      tile(std::integral_constant<int, 4>{});
      tile(std::integral_constant<int, 5>{});
      tile(std::integral_constant<int, 6>{});
      tile(std::integral_constant<int, 7>{});
      sr = cross_row_sum(sr + tr);
      si = cross_row_sum(si - ti);
      const double2 u = j > c ? make_double2(sr, si) : make_double2(0.0, 0.0);
      if (lg == 0) vu[j][1] = u;
      const double gp = row_sum(vj.x * u.x + vj.y * u.y);  // Re(conj(v_j) u_j)
      if (lane == 0) s_g[ct] = gp;
    } else if (lane == 0) {
      s_g[ct] = 0.0;
    }
    __syncthreads();
    const double g2 = row_sum(s_g[l16 & (TW - 1)]);  // 2 gamma: the row holds every part twice
    if (ct == look) {
      __builtin_amdgcn_s_setprio(3);  // ahead of the matrix instructions of its SIMD
      const int c1 = c + 1;
      const double2 vj = vu[c1][0], uj = vu[c1][1];
      const double2 wj = make_double2(2.0 * uj.x - g2 * vj.x, 2.0 * uj.y - g2 * vj.y);
      double2 x[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int i = lane + 64 * q;
        const double2 a = make_double2(s_col[c1 & 1][0][i], s_col[c1 & 1][1][i]), vi = vu[i][0], ui = vu[i][1];
        const double2 wi = make_double2(2.0 * ui.x - g2 * vi.x, 2.0 * ui.y - g2 * vi.y);
        const double2 p = zmul(vi, make_double2(wj.x, -wj.y)), s = zmul(wi, make_double2(vj.x, -vj.y));
        x[q] = i > c1 && i < nb ? make_double2(a.x - p.x - s.x, a.y - p.y - s.y) : make_double2(0.0, 0.0);
      }
      if (c1 + 2 < nb) {
        reflector(c1, x);
      } else {  // the last sub-diagonal element
        const double2 y = (c1 + 1) >> 6 ? x[1] : x[0];
        if (lane == ((c1 + 1) & 63)) {
          W.sub[n - 2] = y;
          W.skip[n - 2] = 1;
        }
      }
      __builtin_amdgcn_s_setprio(0);
    }
    if (ct >= t0 && ct < nt) {
      // operands, component k = lane >> 4: (v, u) of a row, negated; the
      // pair (2u - 2 gamma v, 2v) of the column and i times it
      const double2 vj = vu[j][0], uj = vu[j][1];
      const double2 q = lg < 2 ? make_double2(2.0 * (uj.x - g2 * vj.x), 2.0 * (uj.y - g2 * vj.y))
                               : make_double2(2.0 * vj.x, 2.0 * vj.y);
      const double b1 = lg & 1 ? q.y : q.x, b2 = lg & 1 ? q.x : -q.y;
      const double* rows = reinterpret_cast<const double*>(vu);
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        if (t < t0 || t >= nt) continue;
        const double a = -rows[4 * (16 * t + l16) + lg];
        ar[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b1, ar[t], 0, 0, 0);
        ai[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b2, ai[t], 0, 0, 0);
      }
      if (ct == (c + 2) >> 4) {
        double(*col)[TNB] = s_col[c & 1];
#pragma unroll
        for (int t = 0; t < TW; ++t) {
          if (t < t0 || t >= nt) continue;
          if (j == c + 2) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              col[0][16 * t + lg + 4 * r] = ar[t][r];
              col[1][16 * t + lg + 4 * r] = ai[t][r];
            }
          }
        }
      }
    }
    __syncthreads();
  }
  // the diagonal (rows before k0 were final after their own step)
  for (int i = tid; i < k0; i += TDT) W.d[i] = Aall[mat * strideA + i + (int64_t)i * lda_g].x;
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (t == ct && lg + 4 * r == l16 && j < nb) W.d[k0 + j] = ar[t][r];
  if (tid == 0) W.skip[n - 1] = 1;
  __syncthreads();
  // phases: T' = D^H T D real with off-diagonal |sub|
  tri_phases(W, n, s_ph);
}

// ---- 1'. wide tridiagonalisation (matrices of more than TNB columns): one
// launch per column, the trailing matrix spread over many workgroups (one
// wavefront per column).  k_wide_first and k_wide_gemv form reflector 0 and
// u_0 = A22 v_0; launch k (k_wide_step) applies the rank-2 update of step k
// and forms reflector k+1 and u_{k+1}.  Reflector k is kept in vb (buffer
// k&1, scaled to unit norm) with its scalars in scal; A's column k receives
// it for the back-transformation.
constexpr int WT = 256;       // threads per workgroup
constexpr int WC = WT / 64;   // columns per workgroup


// column k's reflector from its current values (one wavefront)
__device__ __forceinline__ void wide_reflector(const double2* __restrict__ A, int lda, int k, int n, HeevWork& W,
                                               int lane) {
  const double2* col = A + (int64_t)k * lda;
  double part = 0.0;
  for (int i = k + 2 + lane; i < n; i += 64) part += col[i].x * col[i].x + col[i].y * col[i].y;
  part = wave_sum(part);
  const double2 x0 = col[k + 1];
  int skip;
  double iv;
  double2 v0;
  wide_reflector_scalars(lane, k, part, x0, W, skip, iv, v0);
  double2* v = W.vb + (size_t)(k & 1) * n;
  for (int i = k + 1 + lane; i < n; i += 64) {
    const double2 a = i == k + 1 ? v0 : col[i];
    v[i] = make_double2(a.x * iv, a.y * iv);
  }
}

__global__ __launch_bounds__(64) void k_wide_first(double2* __restrict__ Aall, int lda, int64_t strideA, int n,
                                                   int nev, double* __restrict__ work, int64_t strideWork) {
  const int mat = blockIdx.x;
  HeevWork W(work + mat * strideWork, n, nev);
  wide_reflector(Aall + mat * strideA, lda, 0, n, W, threadIdx.x);
}

// u_i = sum_j conj(A(j,i)) v_j for the trailing columns i > k; the first
// workgroup also stores the reflector into column k.
__global__ __launch_bounds__(WT) void k_wide_gemv(double2* __restrict__ Aall, int lda, int64_t strideA, int n,
                                                  int nev, int k, double* __restrict__ work, int64_t strideWork) {
  const int mat = blockIdx.y;
  HeevWork W(work + mat * strideWork, n, nev);
  if (W.scal[4 * (k & 1)] != 0.0) return;  // no reflector for this column
  double2* A = Aall + mat * strideA;
  const double2* v = W.vb + (size_t)(k & 1) * n;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (blockIdx.x == 0 && wid == 0)
    for (int i = k + 1 + lane; i < n; i += 64) A[i + (int64_t)k * lda] = v[i];
  const int i = k + 1 + blockIdx.x * WC + wid;
  if (i >= n) return;
  const double2* col = A + (int64_t)i * lda;
  double sr = 0.0, si = 0.0;
  for (int j = k + 1 + lane; j < n; j += 64) {
    const double2 t = zconjmul(col[j], v[j]);
    sr += t.x;
    si += t.y;
  }
  sr = wave_sum(sr);
  si = wave_sum(si);
  if (lane == 0) W.uu[i] = make_double2(sr, si);
}

// Step k of the wide reduction in one launch.  Reflector k (vb[k&1], scal)
// and u_k = A22 v_k (uu[k&1]) come from the previous launch; with
// w = 2u - 2 (v^H u) v every wavefront applies A22 -= v w^H + w v^H to its
// column j.  Every workgroup also updates column k+1 on the fly and forms
// reflector k+1 from it in LDS (the column itself is not written back: its
// rows below k+1 become that reflector, and the other workgroups read its
// old values); the wavefront of each column j > k+1 then forms
// u_{k+1}(j) = (updated column j)^H v_{k+1} into uu[(k+1)&1], so the next
// step needs no separate product launch.  Workgroup 0 records
// reflector k+1 (vb, scal, skip, sub), the updated diagonal entry of column
// k+1, and reflector k into column k for the back-transformation.  On the
// last wide step (`last`) column k+1 is updated in place like the others,
// for the one-workgroup reduction that follows.
__global__ __launch_bounds__(WT) void k_wide_step(double2* __restrict__ Aall, int lda, int64_t strideA, int n,
                                                  int nev, int k, int last, double* __restrict__ work,
                                                  int64_t strideWork) {
  extern __shared__ __align__(16) unsigned char smem[];
  double2* vn = reinterpret_cast<double2*>(smem);  // [n] reflector k+1 (rows > k+1)
  const int mat = blockIdx.y;
  HeevWork W(work + mat * strideWork, n, nev);
  double2* A = Aall + mat * strideA;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  // the wavefront's column j and the thread's rows of column k+1 are loaded
  // before anything is stored (the stores into A below would otherwise keep
  // these loads, a second round trip, behind them)
  constexpr int PF = 4;  // rows per lane of column j held from entry (n - k - 1 <= 256)
  const int j = k + 1 + blockIdx.x * WC + wid;
  const bool colj = j < n && (last || j != k + 1);
  double2 pre[PF];
#pragma unroll
  for (int q = 0; q < PF; ++q) {
    const int i = k + 1 + lane + 64 * q;
    pre[q] = colj && i < n ? A[i + (int64_t)j * lda] : make_double2(0.0, 0.0);
  }
  const int i1 = k + 2 + (int)threadIdx.x;  // this thread's first row of column k+1
  const double2 c1pre = !last && i1 < n ? A[i1 + (int64_t)(k + 1) * lda] : make_double2(0.0, 0.0);
  const bool skip = W.scal[4 * (k & 1)] != 0.0;  // column k needed no reflector
  const double2* v = W.vb + (size_t)(k & 1) * n;
  const double2* u = W.uu + (size_t)(k & 1) * n;
  // v and u are read whether or not column k took a reflector (the values are
  // then unused), so these loads need not wait for the flag
  double gp = 0.0;
  for (int i = k + 1 + lane; i < n; i += 64) gp += zconjmul(v[i], u[i]).x;
  const double g2 = skip ? 0.0 : 2.0 * wave_sum(gp);
  auto wof = [=](int i) {
    const double2 vi = v[i], ui = u[i];
    return make_double2(2.0 * ui.x - g2 * vi.x, 2.0 * ui.y - g2 * vi.y);
  };
  // a - v_i conj(w_j) - w_i conj(v_j)
  auto upd = [](double2 a, double2 vi, double2 wi, double2 vj, double2 wj) {
    const double2 t1 = zmul(vi, make_double2(wj.x, -wj.y));
    const double2 t2 = zmul(wi, make_double2(vj.x, -vj.y));
    return make_double2(a.x - t1.x - t2.x, a.y - t1.y - t2.y);
  };
  if (blockIdx.x == 0 && wid == 0 && !skip)
    for (int i = k + 1 + lane; i < n; i += 64) A[i + (int64_t)k * lda] = v[i];
  // reflector k+1 from column k+1 after step k (rows > k+1), formed by the
  // whole workgroup: the unscaled values in vn, the norm from per-wavefront
  // partial sums; the scale and the first element enter the products below
  __shared__ double red[WC];
  int skip1 = 1;
  double iv1 = 0.0;
  double2 v01 = make_double2(0.0, 0.0);
  if (!last) {
    const double2* c1 = A + (int64_t)(k + 1) * lda;
    const double2 v1 = skip ? make_double2(0.0, 0.0) : v[k + 1];
    const double2 w1 = skip ? make_double2(0.0, 0.0) : wof(k + 1);
    double part = 0.0;
    for (int i = i1; i < n; i += WT) {  // thread 0 holds row k+2
      const double2 ci = i == i1 ? c1pre : c1[i];
      const double2 c = skip ? ci : upd(ci, v[i], wof(i), v1, w1);
      vn[i] = c;
      if (i > k + 2) part += c.x * c.x + c.y * c.y;
    }
    part = wave_sum(part);
    if (lane == 0) red[wid] = part;
    __syncthreads();
    part = 0.0;
    for (int q = 0; q < WC; ++q) part += red[q];
    // every thread derives the scalars; thread 0 of workgroup 0 records them
    wide_reflector_scalars(blockIdx.x == 0 && threadIdx.x == 0 ? 0 : 1, k + 1, part, vn[k + 2], W, skip1, iv1, v01);
    if (blockIdx.x == 0) {
      double2* vb1 = W.vb + (size_t)((k + 1) & 1) * n;
      for (int i = k + 2 + (int)threadIdx.x; i < n; i += WT) {
        const double2 c = i == k + 2 ? v01 : vn[i];
        vb1[i] = make_double2(c.x * iv1, c.y * iv1);
      }
      if (threadIdx.x == 0 && !skip) {
        double2* dkk = A + (k + 1) + (int64_t)(k + 1) * lda;
        *dkk = upd(*dkk, v1, w1, v1, w1);
      }
    }
  }
  if (!colj) return;
  double2* col = A + (int64_t)j * lda;
  const double2 vj = skip ? make_double2(0.0, 0.0) : v[j];
  const double2 wj = skip ? make_double2(0.0, 0.0) : wof(j);
  double sr = 0.0, si = 0.0;
  auto row = [&](int i, double2 a) {
    if (!skip) {
      a = upd(a, v[i], wof(i), vj, wj);
      col[i] = a;
    }
    if (!last && i > k + 1) {
      const double2 t = zconjmul(a, i == k + 2 ? v01 : vn[i]);
      sr += t.x;
      si += t.y;
    }
  };
#pragma unroll
  for (int q = 0; q < PF; ++q) {
    const int i = k + 1 + lane + 64 * q;
    if (i < n) row(i, pre[q]);
  }
  for (int i = k + 1 + lane + 64 * PF; i < n; i += 64) row(i, col[i]);
  if (!last) {
    sr = wave_sum(sr) * iv1;
    si = wave_sum(si) * iv1;
    if (lane == 0) W.uu[(size_t)((k + 1) & 1) * n + j] = make_double2(sr, si);
  }
}


// The same step for at most 64 PF trailing rows: a wavefront per column j with
// everything in registers, loaded at once: v, u, column k+1 and column j.
// Every wavefront forms reflector k+1 for itself; nothing goes through LDS and
// there are no barriers.  The wavefront of column k+1 records the reflector.
// Bound: one round trip of loads that miss the L2 of their XCD (the previous
// launch wrote them elsewhere), the chain of three reductions, and the launch.
// n = 600 (128 to 600 rows): 8.2 us a step with the workgroup's LDS copy,
// 4.6 here; n = 160: 5.0 and 3.8; four matrices of n = 600: 11.9 and 9.1.
template <int PF>
__global__ __launch_bounds__(WT) void k_wide_regs(double2* __restrict__ Aall, int lda, int64_t strideA, int n, int nev,
                                                  int k, int last, double* __restrict__ work, int64_t strideWork) {
  const int mat = blockIdx.y;
  HeevWork W(work + mat * strideWork, n, nev);
  double2* A = Aall + mat * strideA;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int k1 = k + 1, j = k1 + blockIdx.x * WC + wid;
  if (j >= n) return;
  const bool own = j == k1;  // records reflectors k and k+1
  const double2* vg = W.vb + (size_t)(k & 1) * n;
  const double2* ug = W.uu + (size_t)(k & 1) * n;
  double2* col = A + (int64_t)j * lda;
  double2 v[PF], w[PF], c[PF], a[PF];
#pragma unroll
  for (int q = 0; q < PF; ++q) {
    const int i = k1 + lane + 64 * q;
    v[q] = w[q] = c[q] = a[q] = make_double2(0.0, 0.0);
    if (i < n) {
      v[q] = vg[i];
      w[q] = ug[i];
      c[q] = A[i + (int64_t)k1 * lda];
      a[q] = col[i];
    }
  }
  double2 vj = vg[j], wj = ug[j];
  const bool skip = W.scal[4 * (k & 1)] != 0.0;  // column k needed no reflector: v = u = 0
  const double2 zero = make_double2(0.0, 0.0);
  if (skip) {
    vj = wj = zero;
#pragma unroll
    for (int q = 0; q < PF; ++q) v[q] = w[q] = zero;
  }
  double gp = 0.0;
#pragma unroll
  for (int q = 0; q < PF; ++q) gp += zconjmul(v[q], w[q]).x;
  const double g2 = 2.0 * wave_sum(gp);
  auto wof = [=](double2 vi, double2 ui) { return make_double2(2.0 * ui.x - g2 * vi.x, 2.0 * ui.y - g2 * vi.y); };
  // x - v_i conj(w_j) - w_i conj(v_j)
  auto upd = [](double2 x, double2 vi, double2 wi, double2 vl, double2 wl) {
    const double2 t1 = zmul(vi, make_double2(wl.x, -wl.y));
    const double2 t2 = zmul(wi, make_double2(vl.x, -vl.y));
    return make_double2(x.x - t1.x - t2.x, x.y - t1.y - t2.y);
  };
  wj = wof(vj, wj);
#pragma unroll
  for (int q = 0; q < PF; ++q) w[q] = wof(v[q], w[q]);
  if (own && !skip) {
#pragma unroll
    for (int q = 0; q < PF; ++q) {
      const int i = k1 + lane + 64 * q;
      if (i < n) A[i + (int64_t)k * lda] = v[q];
    }
  }
  int skip1 = 1;
  double iv1 = 0.0;
  if (!last) {
    // column k+1 below its diagonal (row k+1 is lane 0 of q = 0), its reflector
    const double2 v1 = make_double2(read_lane(v[0].x, 0), read_lane(v[0].y, 0));
    const double2 w1 = make_double2(read_lane(w[0].x, 0), read_lane(w[0].y, 0));
    double part = 0.0;
#pragma unroll
    for (int q = 0; q < PF; ++q) {
      c[q] = upd(c[q], v[q], w[q], v1, w1);
      if (q == 0 && lane == 0) {
        if (own && !skip) col[k1] = c[0];  // the diagonal entry
        c[0] = zero;
      }
      if (q > 0 || lane > 1) part += c[q].x * c[q].x + c[q].y * c[q].y;
    }
    part = wave_sum(part);
    const double2 x0 = make_double2(read_lane(c[0].x, 1), read_lane(c[0].y, 1));
    double2 v01;
    wide_reflector_scalars(own ? lane : 1, k1, part, x0, W, skip1, iv1, v01);
    if (lane == 1) c[0] = v01;
    if (own) {
      double2* vb1 = W.vb + (size_t)(k1 & 1) * n;
#pragma unroll
      for (int q = 0; q < PF; ++q) {
        const int i = k1 + lane + 64 * q;
        if (i > k1 && i < n) vb1[i] = make_double2(c[q].x * iv1, c[q].y * iv1);
      }
      return;
    }
  }
  double sr = 0.0, si = 0.0;
#pragma unroll
  for (int q = 0; q < PF; ++q) {
    const int i = k1 + lane + 64 * q;
    a[q] = upd(a[q], v[q], w[q], vj, wj);
    if (!skip && i < n) col[i] = a[q];
    const double2 t = zconjmul(a[q], c[q]);  // row k+1 of c is zero
    sr += t.x;
    si += t.y;
  }
  if (last) return;
  sr = wave_sum(sr) * iv1;
  si = wave_sum(si) * iv1;
  if (lane == 0) W.uu[(size_t)(k1 & 1) * n + j] = make_double2(sr, si);
}

// ---- 2. eigenvalues by multisection: one wavefront per eigenvalue; the 64
// lanes count eigenvalues below 64 interior points, so every step narrows the
// bracket 65-fold.  When the eigenvalues of a launch fit one round of the CUs,
// four wavefronts share an eigenvalue (256 points, 257-fold).  Then the
// clusters (one thread).
constexpr int BSW = 4;  // wavefronts (eigenvalues) per workgroup

// With `shared` set, the BSW wavefronts of a workgroup work on one eigenvalue
// together (64 BSW points per step, one wavefront per SIMD): for launches with
// few eigenvalues, where the CUs would otherwise idle.
__global__ __launch_bounds__(BSW * 64) void k_bisect(int n, int nev, int shared, double* __restrict__ work,
                                                    int64_t strideWork) {
  extern __shared__ __align__(16) unsigned char smem[];
  double* dd = reinterpret_cast<double*>(smem);  // [n]
  double* e2 = dd + n;                            // [n]
  const int mat = blockIdx.y;
  HeevWork W(work + mat * strideWork, n, nev);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double glo = 1e300, ghi = -1e300, emax = 0.0;
  for (int i = threadIdx.x; i < n; i += BSW * 64) {
    const double ei = W.e[i];
    dd[i] = W.d[i];
    e2[i] = ei * ei;
  }
  __syncthreads();
  // Gershgorin bounds (every wave computes them; they are cheap)
  for (int i = lane; i < n; i += 64) {
    const double r = (i > 0 ? sqrt(e2[i - 1]) : 0.0) + (i + 1 < n ? sqrt(e2[i]) : 0.0);
    glo = fmin(glo, dd[i] - r);
    ghi = fmax(ghi, dd[i] + r);
    if (i + 1 < n) emax = fmax(emax, e2[i]);
  }
  for (int o = 32; o > 0; o >>= 1) {
    glo = fmin(glo, __shfl_down(glo, o, 64));
    ghi = fmax(ghi, __shfl_down(ghi, o, 64));
    emax = fmax(emax, __shfl_down(emax, o, 64));
  }
  glo = __shfl(glo, 0, 64);
  ghi = __shfl(ghi, 0, 64);
  emax = __shfl(emax, 0, 64);
  const double tnorm = fmax(fabs(glo), fabs(ghi));
  const double pivmin = fmax(DBL_MIN * fmax(1.0, emax), 1e-300);
  const double span = ghi - glo;
  glo -= 2.0 * DBL_EPSILON * tnorm * n + 1e-300 + 1e-12 * span;
  ghi += 2.0 * DBL_EPSILON * tnorm * n + 1e-300 + 1e-12 * span;
  if (shared) {
    // invariant as below; point k (1..NP) sits at lo + (hi - lo) k / (NP + 1),
    // every thread recomputes the new bracket from the same formula
    __shared__ int s_p[BSW];
    constexpr int NP = BSW * 64;
    const int t = blockIdx.x;
    auto point = [](double lo, double hi, int k) {
      return fmin(fmax(lo + (hi - lo) * ((double)k / (double)(NP + 1)), lo), hi);
    };
    double lo = glo, hi = ghi;
    for (int it = 0; it < 64; ++it) {
      if (hi - lo <= 2.0 * DBL_EPSILON * fmax(fabs(lo), fabs(hi)) + pivmin) break;
      const int cnt = sturm_count(dd, e2, n, point(lo, hi, wid * 64 + lane + 1), pivmin);
      const uint64_t below = __ballot(cnt <= t);
      if (lane == 0) s_p[wid] = below ? wid * 64 + 64 - __clzll(below) : 0;
      __syncthreads();
      int p = 0;
#pragma unroll
      for (int w = 0; w < BSW; ++w) p = max(p, s_p[w]);
      __syncthreads();
      const double newlo = p > 0 ? point(lo, hi, p) : lo;
      const double newhi = p < NP ? point(lo, hi, p + 1) : hi;
      if (!(newlo > lo) && !(newhi < hi)) break;
      lo = newlo;
      hi = newhi;
    }
    if (threadIdx.x == 0) W.lam[t] = 0.5 * (lo + hi);
    return;
  }
  const int t = blockIdx.x * BSW + wid;
  if (t >= nev) return;
  // invariant: count(lo) <= t < count(hi); the points increase with the lane
  // and the Sturm count is monotone in x, so the lanes with count <= t form a
  // prefix 0..p: x_p is the new lo and x_(p+1) (or hi) the new hi
  double lo = glo, hi = ghi;
  for (int it = 0; it < 64; ++it) {
    if (hi - lo <= 2.0 * DBL_EPSILON * fmax(fabs(lo), fabs(hi)) + pivmin) break;
    const double x = fmin(fmax(lo + (hi - lo) * ((double)(lane + 1) / 65.0), lo), hi);
    const int cnt = sturm_count(dd, e2, n, x, pivmin);
    const uint64_t below = __ballot(cnt <= t);
    const int p = below ? 63 - __clzll(below) : -1;
    const double newlo = p >= 0 ? __shfl(x, p, 64) : lo;
    const double newhi = p < 63 ? __shfl(x, p + 1, 64) : hi;
    if (!(newlo > lo) && !(newhi < hi)) break;
    lo = newlo;
    hi = newhi;
  }
  if (lane == 0) W.lam[t] = 0.5 * (lo + hi);
}

// (d, e and the eigenvalues are staged in LDS, n + nev doubles, so that the
// one-thread scans run at LDS latency)
__global__ void k_clusters(int n, int nev, double* __restrict__ work, int64_t strideWork) {
  extern __shared__ __align__(16) unsigned char smem[];
  double* tn = reinterpret_cast<double*>(smem);  // [n] |d_i| + 2|e_i|
  double* lam = tn + n;                           // [nev]
  const int mat = blockIdx.x;
  HeevWork W(work + mat * strideWork, n, nev);
  for (int i = threadIdx.x; i < n; i += blockDim.x) tn[i] = fabs(W.d[i]) + 2.0 * (i + 1 < n ? fabs(W.e[i]) : 0.0);
  for (int t = threadIdx.x; t < nev; t += blockDim.x) lam[t] = W.lam[t];
  __syncthreads();
  if (threadIdx.x != 0) return;
  double tnorm = 0.0;
  for (int i = 0; i < n; ++i) tnorm = fmax(tnorm, tn[i]);
  // eigenvalues closer than 1e-5 |T| are computed in order and re-orthogonalised
  const double ortol = 1e-5 * fmax(tnorm, 1e-300);
  int nc = 0;
  for (int t = 0; t < nev; ++t)
    if (t == 0 || lam[t] - lam[t - 1] > ortol) W.cstart[nc++] = t;
  W.cstart[nc] = nev;
  *W.ncl = nc;
}

// ---- 3. inverse iteration: one thread per cluster, factors and vector in LDS
constexpr int IT = 64;  // threads per inverse-iteration workgroup

__global__ __launch_bounds__(IT) void k_inviter(int n, int nev, int cpw, double* __restrict__ work,
                                               int64_t strideWork) {
  extern __shared__ __align__(16) unsigned char smem[];
  double* dd = reinterpret_cast<double*>(smem);  // [n]
  double* ee = dd + n;                            // [n]
  const int mat = blockIdx.y;
  HeevWork W(work + mat * strideWork, n, nev);
  for (int i = threadIdx.x; i < n; i += IT) {
    dd[i] = W.d[i];
    ee[i] = W.e[i];
  }
  __syncthreads();
  const int c = blockIdx.x * cpw + threadIdx.x;
  if (threadIdx.x >= cpw || c >= *W.ncl) return;
  double* mine = ee + n + (size_t)threadIdx.x * (6 * n + 1);  // odd stride: the lanes' arrays on distinct banks
  double* u0 = mine;
  double* u1 = u0 + n;
  double* u2 = u1 + n;
  double* lv = u2 + n;
  double* pv = lv + n;
  double* x = pv + n;
  double emax = 0.0, tnorm = 0.0;
  for (int i = 0; i < n; ++i) {
    emax = fmax(emax, ee[i] * ee[i]);
    tnorm = fmax(tnorm, fabs(dd[i]) + 2.0 * ee[i]);
  }
  // no pivot below 1e-30 |T|: with 1e-300 (the pivot of a decoupled row at its
  // own eigenvalue) the solution's norm overflowed and the vector came out zero
  const double pivmin = fmax(fmax(DBL_MIN * fmax(1.0, emax), 1e-300), 1e-30 * tnorm);
  const int t0 = W.cstart[c], t1 = W.cstart[c + 1];
  double prev = -1e300;
  for (int t = t0; t < t1; ++t) {
    double lmb = W.lam[t];
    const double sep = 10.0 * DBL_EPSILON * fmax(tnorm, 1e-300);
    if (t > t0 && lmb - prev < sep) lmb = prev + sep;
    prev = lmb;
    uint64_t h = 0x9E3779B97F4A7C15ull * (uint64_t)(t + 1);
    for (int i = 0; i < n; ++i) {
      h ^= h >> 31;
      h *= 0xBF58476D1CE4E5B9ull;
      h ^= h >> 29;
      x[i] = ((double)(h >> 11) * (1.0 / 9007199254740992.0)) - 0.5;
    }
    tri_factor(dd, ee, n, lmb, pivmin, u0, u1, u2, lv, pv);
    for (int it = 0; it < 3; ++it) {
      tri_solve(n, u0, u1, u2, lv, pv, x);
      for (int q = t0; q < t; ++q) {  // orthogonalise against the earlier cluster members
        const double* y = W.xt + (size_t)q * n;
        double sdot = 0.0;
        for (int i = 0; i < n; ++i) sdot += y[i] * x[i];
        for (int i = 0; i < n; ++i) x[i] -= sdot * y[i];
      }
      double nr = 0.0;
      for (int i = 0; i < n; ++i) nr += x[i] * x[i];
      const double inr = nr > 0.0 ? 1.0 / sqrt(nr) : 0.0;
      for (int i = 0; i < n; ++i) x[i] *= inr;
    }
    double* out = W.xt + (size_t)t * n;
    for (int i = 0; i < n; ++i) out[i] = x[i];
  }
}

// ---- 4. back-transformation, one wavefront per eigenvector
// waves per back-transform workgroup: four, so that the eigenvectors spread
// over many CUs (a wave's reflector steps are bound by its own FP64 issue: 16
// waves per workgroup put 80 vectors on five CUs, 130 us at n = 160)
constexpr int BW = 4;

__global__ __launch_bounds__(BW * 64) void k_backtransform(const double2* __restrict__ Aall, int lda,
                                                          int64_t strideA, int n, int nev,
                                                          double* __restrict__ work, int64_t strideWork,
                                                          double* __restrict__ Wall, int64_t strideW,
                                                          double2* __restrict__ Zall, int ldz, int64_t strideZ) {
  const int mat = blockIdx.y;
  const double2* A = Aall + mat * strideA;
  HeevWork W(work + mat * strideWork, n, nev);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int t = blockIdx.x * BW + wid;
  if (t >= nev) return;
  double2* z = Zall + mat * strideZ + (int64_t)t * ldz;
  const double* xs = W.xt + (size_t)t * n;
  for (int i = lane; i < n; i += 64) z[i] = make_double2(W.ph[i].x * xs[i], W.ph[i].y * xs[i]);
  if (lane == 0) Wall[mat * strideW + t] = W.lam[t];
  for (int k = n - 3; k >= 0; --k) {
    if (W.skip[k]) continue;
    const double2* vk = A + (int64_t)k * lda;  // reflector in rows k+1..n-1
    double sr = 0.0, si = 0.0;
    for (int i = k + 1 + lane; i < n; i += 64) {
      const double2 p = zconjmul(vk[i], z[i]);
      sr += p.x;
      si += p.y;
    }
    sr = 2.0 * wave_sum(sr);
    si = 2.0 * wave_sum(si);
    for (int i = k + 1 + lane; i < n; i += 64) {
      const double2 p = zmul(vk[i], make_double2(sr, si));
      z[i] = make_double2(z[i].x - p.x, z[i].y - p.y);
    }
  }
}

// The same with the eigenvector in registers (rows lane + 64 q, q < NQ,
// n <= 64 NQ) and the reflector columns staged in LDS in panels of BTP
// columns: the workgroup loads the next panel (coalesced over rows) while its
// waves run the current one, and the skip flags sit in LDS, so no step waits
// on global memory.  LDS: 2 BTP n complex + n ints.
constexpr int BTP = 8;

template <int NQ>
__global__ __launch_bounds__(BW * 64) void k_backtransform_reg(const double2* __restrict__ Aall, int lda,
                                                              int64_t strideA, int n, int nev,
                                                              double* __restrict__ work, int64_t strideWork,
                                                              double* __restrict__ Wall, int64_t strideW,
                                                              double2* __restrict__ Zall, int ldz, int64_t strideZ) {
  extern __shared__ __align__(16) unsigned char smem[];
  double2* pan = reinterpret_cast<double2*>(smem);   // [2][BTP][n]
  int* skip = reinterpret_cast<int*>(pan + 2 * BTP * n);  // [n]
  const int mat = blockIdx.y;
  const double2* A = Aall + mat * strideA;
  HeevWork W(work + mat * strideWork, n, nev);
  constexpr int NT = BW * 64;
  constexpr int PL = (BTP * 64 * NQ + NT - 1) / NT;  // panel elements per thread (n <= 64 NQ)
  const int tid = threadIdx.x;
  for (int i = tid; i < n; i += NT) skip[i] = W.skip[i];
  // panel p holds columns k = n-3 - BTP p - c, c < BTP (rows > k, zero above)
  auto fetch = [&](int p, double2* r) {
#pragma unroll
    for (int e = 0; e < PL; ++e) {
      const int q = tid + e * NT, c = q / n, i = q - c * n, k = n - 3 - BTP * p - c;
      r[e] = (c < BTP && k >= 0 && i > k) ? A[i + (int64_t)k * lda] : make_double2(0.0, 0.0);
    }
  };
  auto store = [&](int p, const double2* r) {
    double2* b = pan + (size_t)(p & 1) * BTP * n;
#pragma unroll
    for (int e = 0; e < PL; ++e) {
      const int q = tid + e * NT;
      if (q < BTP * n) b[q] = r[e];
    }
  };
  double2 pre[PL];
  fetch(0, pre);
  store(0, pre);
  __syncthreads();
  const int lane = tid & 63, wid = tid >> 6;
  const int t = blockIdx.x * BW + wid;
  const bool act = t < nev;
  double2 z[NQ];
  if (act) {
    const double* xs = W.xt + (size_t)t * n;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int i = lane + 64 * q;
      z[q] = i < n ? make_double2(W.ph[i].x * xs[i], W.ph[i].y * xs[i]) : make_double2(0.0, 0.0);
    }
    if (lane == 0) Wall[mat * strideW + t] = W.lam[t];
  }
  const int np = n >= 3 ? (n - 3) / BTP + 1 : 0;
  for (int p = 0; p < np; ++p) {
    if (p + 1 < np) fetch(p + 1, pre);
    const double2* b = pan + (size_t)(p & 1) * BTP * n;
    if (act) {
      for (int c = 0; c < BTP; ++c) {
        const int k = n - 3 - BTP * p - c;
        if (k < 0) break;
        if (skip[k]) continue;
        const double2* col = b + (size_t)c * n;
        double2 v[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const int i = lane + 64 * q;
          v[q] = i < n ? col[i] : make_double2(0.0, 0.0);
        }
        double sr = 0.0, si = 0.0;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const double2 pr = zconjmul(v[q], z[q]);
          sr += pr.x;
          si += pr.y;
        }
        sr = 2.0 * wave_sum(sr);
        si = 2.0 * wave_sum(si);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const double2 pr = zmul(v[q], make_double2(sr, si));
          z[q] = make_double2(z[q].x - pr.x, z[q].y - pr.y);
        }
      }
    }
    if (p + 1 < np) store(p + 1, pre);
    __syncthreads();
  }
  if (act) {
    double2* zo = Zall + mat * strideZ + (int64_t)t * ldz;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int i = lane + 64 * q;
      if (i < n) zo[i] = z[q];
    }
  }
}

void heev_gpu(double2* A, int lda, int64_t strideA, int n, int nev, double* Wv, int64_t strideW, double2* Z, int ldz,
              int64_t strideZ, double* work, int64_t strideWork, int batch, hipStream_t s) {
  DEREK_REQUIRE(n >= 1 && nev >= 1 && nev <= n, "heev: need 1 <= nev <= n");
  DEREK_REQUIRE(n <= 2048, "heev: n must be <= 2048");
  {
    const int k0 = std::max(0, n - TNB);
    // steps 0..k0-1 with a multi-workgroup launch per column, then the rest in
    // one workgroup
    if (k0 > 0) {
      hipLaunchKernelGGL(k_wide_first, dim3(batch), dim3(64), 0, s, A, lda, strideA, n, nev, work, strideWork);
      hipLaunchKernelGGL(k_wide_gemv, dim3((unsigned)ceil_div(n - 1, WC), batch), dim3(WT), 0, s, A, lda, strideA, n,
                         nev, 0, work, strideWork);
      for (int k = 0; k < k0; ++k) {
        const dim3 grid((unsigned)ceil_div(n - k - 1, WC), batch);
        const int last = k == k0 - 1 ? 1 : 0, pf = (int)ceil_div(n - k - 1, 64);
        // in registers while a column and its three companions fit them
        if (pf > 10)
          hipLaunchKernelGGL(k_wide_step, grid, dim3(WT), sizeof(double2) * (size_t)n, s, A, lda, strideA, n, nev, k,
                             last, work, strideWork);
        else
          hipLaunchKernelGGL(pf > 7 ? k_wide_regs<10> : (pf > 4 ? k_wide_regs<7> : k_wide_regs<4>), grid, dim3(WT), 0,
                             s, A, lda, strideA, n, nev, k, last, work, strideWork);
      }
    }
    hipLaunchKernelGGL(k_tridiag, dim3(batch), dim3(TDT), 0, s, A, lda, strideA, n, k0, nev, work,
                       strideWork);
    DEREK_HIP(hipGetLastError());
  }
  {
    const size_t lds = sizeof(double) * 2 * (size_t)n;
    // one eigenvalue per workgroup while they fit one round of the CUs
    const int shared = (int64_t)nev * batch <= 256 ? 1 : 0;
    hipLaunchKernelGGL(k_bisect, dim3((unsigned)(shared ? nev : ceil_div(nev, BSW)), batch), dim3(BSW * 64), lds, s, n,
                       nev, shared, work, strideWork);
    DEREK_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_clusters, dim3(batch), dim3(64), sizeof(double) * ((size_t)n + nev), s, n, nev, work,
                       strideWork);
    DEREK_HIP(hipGetLastError());
  }
  {
    // clusters per workgroup: LDS holds d, e and 6 n + 1 doubles per cluster
    // thread, up to 156 KiB (at n = 600 that is five clusters per workgroup,
    // so the 300 clusters take one round of the CUs instead of two)
    constexpr size_t kInvLds = 156 * 1024;
    const int cpw =
        std::max(1, std::min(IT, (int)((kInvLds / sizeof(double) - 2 * (size_t)n) / (6 * (size_t)n + 1))));
    const size_t lds = sizeof(double) * (2 * (size_t)n + (6 * (size_t)n + 1) * cpw);
    DEREK_REQUIRE(lds <= kInvLds, "heev: inverse-iteration scratch exceeds the LDS budget");
    if (lds > 65536) allow_dynamic_lds(reinterpret_cast<const void*>(k_inviter), kInvLds);
    dim3 grid((unsigned)ceil_div(nev, cpw), batch);
    hipLaunchKernelGGL(k_inviter, grid, dim3(IT), lds, s, n, nev, cpw, work, strideWork);
    DEREK_HIP(hipGetLastError());
  }
  {
    dim3 grid((unsigned)ceil_div(nev, BW), batch);
    const size_t lds = sizeof(double2) * 2 * BTP * (size_t)n + sizeof(int) * (size_t)n;
#define BT_(NQ)                                                                                                  \
  do {                                                                                                           \
    if (lds > 65536) allow_dynamic_lds(reinterpret_cast<const void*>(k_backtransform_reg<NQ>), lds);             \
    hipLaunchKernelGGL(k_backtransform_reg<NQ>, grid, dim3(BW * 64), lds, s, A, lda, strideA, n, nev, work,      \
                       strideWork, Wv, strideW, Z, ldz, strideZ);                                                \
  } while (0)
    if (n <= 64) BT_(1);
    else if (n <= 128) BT_(2);
    else if (n <= 192) BT_(3);
    else if (n <= 256) BT_(4);
    else if (n <= 384) BT_(6);
    else if (n <= 512) BT_(8);
    else if (n <= 624) BT_(10);  // LDS: two 8-column panels of n rows, 260 n bytes <= 160 KiB
    else
      hipLaunchKernelGGL(k_backtransform, grid, dim3(BW * 64), 0, s, A, lda, strideA, n, nev, work, strideWork, Wv,
                         strideW, Z, ldz, strideZ);
#undef BT_
    DEREK_HIP(hipGetLastError());
  }
}

// ---------------------------------------------------------------- generalized problem pieces
// All matrices m x m, column-major, ld m; matrix kz of a batch at kz*m*m
// (blockIdx.y or blockIdx.x selects it).

// 1/sqrt of the diagonal entry i of S (0 for a zero column)
__device__ __forceinline__ double diag_scale(const double2* S, int m, int i) {
  const double d = S[i + (int64_t)i * m].x;
  return d > 0.0 ? 1.0 / sqrt(d) : 0.0;
}

// Lower triangle of W <- D (S + S^H)/2 D with D = 1/sqrt(diag S) (dsc), and
// Linv, LinvH <- 0
__global__ void k_chol_prep(const double2* __restrict__ Sall, int m, double* __restrict__ dscall,
                            double2* __restrict__ Wall, double2* __restrict__ Linvall,
                            double2* __restrict__ LinvHall) {
  const int64_t mm = (int64_t)m * m, o = blockIdx.y * mm;
  const double2* S = Sall + o;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < mm; q += (int64_t)gridDim.x * blockDim.x) {
    const int r = (int)(q % m), c = (int)(q / m);
    Linvall[o + q] = LinvHall[o + q] = make_double2(0.0, 0.0);
    if (r < c) continue;
    const double dr = diag_scale(S, m, r);
    if (r == c) {
      dscall[(int64_t)blockIdx.y * m + r] = dr;
      Wall[o + q] = make_double2(S[q].x * (dr * dr), 0.0);
    } else {
      const double f = 0.5 * dr * diag_scale(S, m, c);
      const double2 a = S[q], b = S[c + (int64_t)r * m];
      Wall[o + q] = make_double2((a.x + b.x) * f, (a.y - b.y) * f);
    }
  }
}

// Cholesky factor with dropped columns and its inverse, one launch per panel
// of CB columns: the factor L of the unit-diagonal W = L L^H, where column j
// is kept if its updated pivot exceeds tol and replaced by the identity
// column and row otherwise, is never stored; what the launches leave is
// Linv = L^-1 (and LinvH, its conjugate transpose), from the forward
// elimination of the identity carried along with the factorisation.
//
// A workgroup owns one CT x CT tile: a lower tile of the trailing W (right of
// and below the panel) or a tile (trailing rows, columns done so far) of the
// eliminated identity R.  Each one factors the CB x CB diagonal block of the
// panel for itself (one wavefront, a row per lane, pivots and columns by
// readlane), meanwhile another wavefront has loaded the tile's CT rows of the
// panel and either the CT rows of its columns (W tile) or the CT columns of
// the panel rows of R (R tile) and solves them against the block, one row or
// column per lane; then the tile takes its rank-CB update.  The panel columns
// of W and the panel rows of R are only read, X = L11^-1 R goes to Linv and
// LinvH, so no workgroup waits for another within a launch.
//
// Bound: the serial chain of a launch (launch, two loads, 16 pivots of about
// 400 cycles, a 16-step substitution).  The single-workgroup factorisation it
// replaces was bound by its one CU: 203 us at m = 160 and 4650 us at m = 600,
// plus 57 and 552 us for the inverse (one wavefront per column) and 13 and
// 139 us for the scaling (one workgroup).
constexpr int CB = 16, CT = 32, CNT = 256;

__global__ __launch_bounds__(CNT) void k_chol_panel(double2* __restrict__ Wall, double2* __restrict__ Rall,
                                                    double2* __restrict__ Linvall, double2* __restrict__ LinvHall,
                                                    int m, int p0, double tol, int nev, int* __restrict__ keepall,
                                                    int* __restrict__ naall, int* __restrict__ okall) {
  __shared__ double2 L11[CB][CB];      // rows of the panel's factor
  __shared__ double idiag[CB];         // 1 / L_jj, 0 where dropped
  __shared__ double2 La[CB][CT + 1];   // [panel column][tile row]
  __shared__ double2 Lb[CB][CT + 1];   // [panel column or row][tile column]
  const int64_t mm = (int64_t)m * m, o = blockIdx.y * mm;
  double2* W = Wall + o;
  double2* Rm = Rall + o;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int pn = min(CB, m - p0), p1 = p0 + pn;
  const int nt = (m - p1 + CT - 1) / CT;  // tile rows of the trailing part
  // tile: W tiles (bi, bj <= bi) first, then R tiles (bi, cb); with nothing
  // trailing only X is formed (tile row 0 without rows)
  int bi = 0, bj = blockIdx.x;
  const int nw = nt * (nt + 1) / 2;
  const bool wt = bj < nw;
  if (wt) {
    while (bj > bi) bj -= ++bi;
  } else {
    const int ncb = (p1 + CT - 1) / CT;
    bj -= nw;
    bi = bj / ncb;
    bj -= bi * ncb;
  }
  const int r0 = p1 + bi * CT, c0 = wt ? p1 + bj * CT : bj * CT, cend = wt ? m : p1;
  // this thread's tile elements: row tr, columns tc + 8 q
  const int tr = tid % CT, tc = tid / CT;
  double2* T = wt ? W : Rm;
  double2 t[CT * CT / CNT];
#pragma unroll
  for (int q = 0; q < CT * CT / CNT; ++q) {
    const int r = r0 + tr, c = c0 + tc + (CNT / CT) * q;
    // the panel's own columns of R have not been touched: zero
    t[q] = (r < m && c < cend && (wt || c < p0)) ? T[r + (int64_t)c * m] : make_double2(0.0, 0.0);
  }
  double2 x[CB];
  if (wid == 0) {
    // lanes 0..31: the tile's rows of the panel; 32..63: the rows of its
    // columns (W tile) or its columns of the panel's rows of R (R tile)
    const int h = lane / CT, l = lane % CT;
    const int row = (h == 0 ? r0 : c0) + l;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      double2 v = make_double2(0.0, 0.0);
      if (h == 0 || wt) {
        if (row < m && j < pn) v = W[row + (int64_t)(p0 + j) * m];
      } else if (j < pn) {
        if (row < p0) v = Rm[(p0 + j) + (int64_t)row * m];
        else if (row == p0 + j) v = make_double2(1.0, 0.0);
      }
      x[j] = v;
    }
  } else if (wid == 1) {
    double2 a[CB];
#pragma unroll
    for (int k = 0; k < CB; ++k)
      a[k] = (lane < pn && k <= lane) ? W[(p0 + lane) + (int64_t)(p0 + k) * m] : make_double2(0.0, 0.0);
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      const double d = read_lane(a[j].x, j);
      double idj = 0.0;
      if (j < pn && d > tol) {
        idj = rsqrt_nr(d);
        const double2 l = make_double2(a[j].x * idj, a[j].y * idj);
#pragma unroll
        for (int k = j + 1; k < CB; ++k) {
          const double kr = read_lane(l.x, k), ki = read_lane(l.y, k);
          a[k] = make_double2(a[k].x - (l.x * kr + l.y * ki), a[k].y - (l.y * kr - l.x * ki));
        }
        a[j] = l;
      } else {
        a[j] = make_double2(0.0, 0.0);
      }
      if (lane == 0) idiag[j] = idj;
    }
    if (lane < CB) {
#pragma unroll
      for (int k = 0; k < CB; ++k) L11[lane][k] = a[k];
    }
  }
  __syncthreads();
  if (wid == 0) {
    const int h = lane / CT, l = lane % CT;
    const bool left = h == 0 || wt;  // rows: x L11^H = w; columns: L11 x = r
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      double2 s = x[j];
#pragma unroll
      for (int k = 0; k < j; ++k) {
        const double2 b = L11[j][k];
        const double bi_ = left ? -b.y : b.y;  // x_k conj(L_jk) or L_jk x_k
        s = make_double2(s.x - (x[k].x * b.x - x[k].y * bi_), s.y - (x[k].x * bi_ + x[k].y * b.x));
      }
      const double id = idiag[j];
      x[j] = make_double2(s.x * id, s.y * id);
      // a dropped row of L is the identity row: x = e_j there
      if (!left && id == 0.0) x[j] = make_double2(c0 + l == p0 + j ? 1.0 : 0.0, 0.0);
    }
#pragma unroll
    for (int j = 0; j < CB; ++j) (h == 0 ? La : Lb)[j][l] = x[j];
    if (!wt && bi == 0 && h == 1 && c0 + l < p1) {
      const int c = c0 + l;
      double2* li = Linvall + o + (int64_t)c * m + p0;
      double2* lh = LinvHall + o + (int64_t)p0 * m + c;
#pragma unroll
      for (int j = 0; j < CB; ++j)
        if (j < pn) {
          li[j] = x[j];
          lh[(int64_t)j * m] = make_double2(x[j].x, -x[j].y);
        }
    }
  }
  __syncthreads();
  if (r0 < m) {
#pragma unroll
    for (int q = 0; q < CT * CT / CNT; ++q) {
      const int cc = tc + (CNT / CT) * q;
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        // W(r,c) -= L_rj conj(L_cj); R(r,c) -= L_rj X_jc.  An R tile uses the
        // dropped rows' X only through L_rj = 0.
        const double2 a = La[j][tr], b = Lb[j][cc];
        const double by = wt ? -b.y : b.y;
        t[q] = make_double2(t[q].x - (a.x * b.x - a.y * by), t[q].y - (a.x * by + a.y * b.x));
      }
      const int r = r0 + tr, c = c0 + cc;
      if (r < m && c < cend) T[r + (int64_t)c * m] = t[q];
    }
  }
  if (blockIdx.x == 0) {
    int* keep = keepall + (int64_t)blockIdx.y * m;
    if (tid < pn) keep[p0 + tid] = idiag[tid] != 0.0 ? 1 : 0;
    if (tid == 0) {
      int c = p0 == 0 ? 0 : naall[blockIdx.y];
      for (int j = 0; j < pn; ++j) c += idiag[j] != 0.0 ? 1 : 0;
      naall[blockIdx.y] = c;
      okall[blockIdx.y] = c >= nev ? 1 : 0;
    }
  }
}

// Hc = D (H + H^H)/2 D on the kept rows and columns, 0 elsewhere
__global__ void k_scale_mask(const double2* __restrict__ H, const double* __restrict__ dsc,
                             const int* __restrict__ keep, int m, double2* __restrict__ Hc) {
  const int64_t mm = (int64_t)m * m;
  const int kz = blockIdx.y;
  H += kz * mm;
  Hc += kz * mm;
  dsc += (int64_t)kz * m;
  keep += (int64_t)kz * m;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < mm; q += (int64_t)gridDim.x * blockDim.x) {
    const int r = (int)(q % m), c = (int)(q / m);
    const double f = (keep[r] && keep[c]) ? dsc[r] * dsc[c] * 0.5 : 0.0;
    const double2 a = H[q], b = H[c + (int64_t)r * m];
    Hc[q] = make_double2((a.x + b.x) * f, (a.y - b.y) * f);
  }
}

// Dropped diagonal entries of A <- 2 max_i sum_j |A_ij| + 1 (above every
// eigenvalue of the kept block), so the lowest eigenpairs are the kept ones.
// Row sums: R = min(m, DT) rows per pass over consecutive threads (coalesced
// column reads), the columns split over DT / R thread groups whose parts are
// added through LDS.
// Nothing to do, and nothing read, where every column was kept.
__global__ __launch_bounds__(DT) void k_big_diag(double2* __restrict__ Aall, const int* __restrict__ keepall,
                                                 const int* __restrict__ naall, int m) {
  if (naall[blockIdx.x] == m) return;
  __shared__ double red[DW];
  __shared__ double part[DT];
  const int kz = blockIdx.x;
  double2* A = Aall + (int64_t)kz * m * m;
  const int* keep = keepall + (int64_t)kz * m;
  const int R = min(m, DT), cg = DT / R;
  const int t = threadIdx.x % R, g = threadIdx.x / R;
  double rmax = 0.0;
  for (int i0 = 0; i0 < m; i0 += R) {
    const int i = i0 + t;
    double r = 0.0;
    if (g < cg && i < m) {
#pragma unroll 4
      for (int j = g; j < m; j += cg) {
        const double2 a = A[i + (int64_t)j * m];
        r += sqrt(a.x * a.x + a.y * a.y);
      }
    }
    if (g < cg) part[g * R + t] = r;
    __syncthreads();
    if (threadIdx.x < R && i0 + (int)threadIdx.x < m) {
      double sum = 0.0;
      for (int q = 0; q < cg; ++q) sum += part[q * R + threadIdx.x];
      rmax = fmax(rmax, sum);
    }
    __syncthreads();
  }
  const double big = 2.0 * block_max_all(rmax, red) + 1.0;
  for (int i = threadIdx.x; i < m; i += DT)
    if (!keep[i]) A[i + (int64_t)i * m] = make_double2(big, 0.0);
}

// U (m x nev) = D C on the kept rows, 0 on the dropped ones; where ok == 0
// the subspace step is void: U = [I; 0] and w keeps its previous values.
__global__ void k_expand(const double2* __restrict__ Call, const double* __restrict__ dscall,
                         const int* __restrict__ keepall, const int* __restrict__ okall, int m, int nev,
                         const double* __restrict__ wnew, double* __restrict__ w, double2* __restrict__ Uall) {
  const int kz = blockIdx.y;
  const int ok = okall[kz];
  const double2* C = Call + (int64_t)kz * m * m;
  const double* dsc = dscall + (int64_t)kz * m;
  const int* keep = keepall + (int64_t)kz * m;
  double2* U = Uall + (int64_t)kz * m * nev;
  const int64_t n = (int64_t)m * nev;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
    const int r = (int)(q % m), c = (int)(q / m);
    double2 v;
    if (ok) {
      const double f = keep[r] ? dsc[r] : 0.0;
      const double2 x = C[r + (int64_t)c * m];
      v = make_double2(x.x * f, x.y * f);
    } else {
      v = make_double2(r == c ? 1.0 : 0.0, 0.0);
    }
    U[q] = v;
  }
  if (blockIdx.x == 0 && ok)
    for (int c = threadIdx.x; c < nev; c += blockDim.x) w[(int64_t)kz * nev + c] = wnew[(int64_t)kz * nev + c];
}

// A <- (A + A^H)/2
__global__ void k_hermitize(double2* __restrict__ A, int m) {
  const int64_t mm = (int64_t)m * m;
  A += blockIdx.y * mm;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < mm; q += (int64_t)gridDim.x * blockDim.x) {
    const int r = (int)(q % m), c = (int)(q / m);
    if (r > c) continue;
    const double2 a = A[q], b = A[c + (int64_t)r * m];
    const double2 h = make_double2(0.5 * (a.x + b.x), 0.5 * (a.y - b.y));
    A[q] = r == c ? make_double2(h.x, 0.0) : h;
    if (r != c) A[c + (int64_t)r * m] = make_double2(h.x, -h.y);
  }
}

static dim3 mgrid(int m, int batch) {
  return dim3((unsigned)std::min<int64_t>(256, ceil_div((int64_t)m * m, 256)), (unsigned)batch);
}

void hermitize_gpu(double2* A, int m, int batch, hipStream_t s) {
  hipLaunchKernelGGL(k_hermitize, mgrid(m, batch), dim3(256), 0, s, A, m);
  DEREK_HIP(hipGetLastError());
}

void chol_inverse_gpu(const double2* S, int m, double tol, int nev, double2* Wm, double2* R, double2* Linv,
                      double2* LinvH, double* dsc, int* keep, int* na, int* ok, int batch, hipStream_t s) {
  DEREK_REQUIRE(m >= 1 && m <= 8192, "chol_inverse: matrix too large");
  hipLaunchKernelGGL(k_chol_prep, mgrid(m, batch), dim3(256), 0, s, S, m, dsc, Wm, Linv, LinvH);
  for (int p0 = 0; p0 < m; p0 += CB) {
    const int p1 = std::min(m, p0 + CB), nt = (int)ceil_div(m - p1, CT);
    const int tiles = nt * (nt + 1) / 2 + std::max(1, nt) * (int)ceil_div(p1, CT);
    hipLaunchKernelGGL(k_chol_panel, dim3(tiles, batch), dim3(CNT), 0, s, Wm, R, Linv, LinvH, m, p0, tol, nev, keep, na,
                       ok);
  }
  DEREK_HIP(hipGetLastError());
}

void scale_mask_gpu(const double2* H, const double* dsc, const int* keep, int m, double2* Hc, int batch,
                    hipStream_t s) {
  hipLaunchKernelGGL(k_scale_mask, mgrid(m, batch), dim3(256), 0, s, H, dsc, keep, m, Hc);
  DEREK_HIP(hipGetLastError());
}

void big_diag_gpu(double2* A, const int* keep, const int* na, int m, int batch, hipStream_t s) {
  hipLaunchKernelGGL(k_big_diag, dim3(batch), dim3(DT), 0, s, A, keep, na, m);
  DEREK_HIP(hipGetLastError());
}

void expand_gpu(const double2* C, const double* dsc, const int* keep, const int* ok, int m, int nev,
                const double* wnew, double* w, double2* U, int batch, hipStream_t s) {
  const int64_t n = (int64_t)m * nev;
  hipLaunchKernelGGL(k_expand, dim3((unsigned)std::min<int64_t>(256, ceil_div(n, 256)), batch), dim3(256), 0, s, C,
                     dsc, keep, ok, m, nev, wnew, w, U);
  DEREK_HIP(hipGetLastError());
}

}  // namespace derek
