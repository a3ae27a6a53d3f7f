// Tall-skinny complex GEMMs on the CDNA4 matrix cores, batched over k-points.
//
// Overlap  C = X^H Y  (X: npw x m, Y: npw x n, npw >> m, n): split-K over
// the plane-wave index; each workgroup owns a 64x64 tile of C and a chunk of
// rows of one k-point, stages 16-row slabs of X and Y through
// LDS and accumulates three real products per complex product (Gauss's
// method: 25% fewer matrix-core operations than the four-product form) with
// 16x16x4 MFMAs (f64, or f32 for complex64 data); the next slab is loaded
// into registers while the current one is multiplied.  A second kernel sums
// the chunk partials in a fixed order in FP64 (deterministic).
// Rotation Z = X U: each workgroup owns 64 rows x 64 columns of Z; U slabs
// (FP64, rounded to R) are staged through LDS, X is read straight into the
// MFMA A operand; three real products per complex product as well.
// Work items are dealt so that the workgroups that read the same rows (the
// tiles of one row chunk, the column blocks of one row block) run on one
// XCD, which then fetches those rows from HBM once into its L2.
//
// 16x16x4 MFMA operand layout (lane l of a 64-wide wave):
//   A (16x4): A[l%16][l/16]      B (4x16): B[l/16][l%16]
//   D (16x16), f64: register r holds D[l/16 + 4*r][l%16]
//   D (16x16), f32: register r holds D[4*(l/16) + r][l%16]
#include "launch.hpp"
#include "ov_geom.hpp"

namespace derek {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <typename R> struct Mfma;
template <> struct Mfma<double> {
  using acc = d4;
  __device__ static __forceinline__ d4 op(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <> struct Mfma<float> {
  using acc = f4;
  __device__ static __forceinline__ f4 op(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

constexpr int OV_PAD = 66;     // LDS row pitch
constexpr int kOvBlocks = 5;   // 16 x 16 blocks of C per wavefront at most (k_overlap_dealt)

constexpr int kXcds = 8;  // MI355X: 8 XCDs, each with its own L2

// Work item (0 .. total-1) of the workgroup with linear id L such that every
// XCD runs one contiguous range of items: the dispatcher deals workgroups to
// the XCDs round-robin, so id L runs on XCD L % 8 as its (L / 8)-th.
// Consecutive items share operand rows, which then stay in that XCD's L2.
__device__ __forceinline__ int64_t xcd_item(int64_t L, int64_t total) {
  const int64_t q = total / kXcds, r = total % kXcds;
  const int64_t x = L % kXcds, slot = L / kXcds;
  return x < r ? x * (q + 1) + slot : r * (q + 1) + (x - r) * q + slot;
}

// at least two waves per SIMD (register budget 256 per lane incl. accumulators)
template <typename R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_overlap(const cx_t<R>* __restrict__ X, int64_t ldx, int64_t sx,
                                                 const cx_t<R>* __restrict__ Y, int64_t ldy, int64_t sy,
                                                 const int* __restrict__ npwk, OvGeom g,
                                                 double2* __restrict__ part) {
  using M = Mfma<R>;
  using A4 = typename M::acc;
  using C = cx_t<R>;
  // slab operands for the three real products of the complex product
  // conj(x) y (Gauss):  P1 = xr yr,  P2 = xi yi,  P3 = (xr - xi)(yr + yi);
  // Re = P1 + P2,  Im = P3 - P1 + P2
  __shared__ R xr[OV_KS][OV_PAD], xi[OV_KS][OV_PAD], xs[OV_KS][OV_PAD];
  __shared__ R yr[OV_KS][OV_PAD], yi[OV_KS][OV_PAD], ys[OV_KS][OV_PAD];
  // work item: tile fastest, then row chunk, then k-point; the tiles of one
  // chunk share an XCD and read the same rows through its L2
  const int64_t w = xcd_item(blockIdx.x, gridDim.x);
  const int chunk = (int)((w / g.ntiles) % g.nchunk);
  const int kz = (int)(w / ((int64_t)g.ntiles * g.nchunk));
  X += kz * sx;
  Y += kz * sy;
  const int64_t npw = npwk ? (int64_t)npwk[kz] : g.npw;
  // tile coordinates
  int ti, tj;
  int t = (int)(w % g.ntiles);
  if (g.herm) {
    ti = 0;
    while (t >= g.tm - ti) { t -= g.tm - ti; ++ti; }
    tj = ti + t;
  } else {
    ti = t % g.tm;
    tj = t / g.tm;
  }
  const int i0 = ti * OV_T, j0 = tj * OV_T;
  const int64_t r0 = (int64_t)chunk * g.kch;
  const int64_t r1 = std::min<int64_t>(npw, r0 + g.kch);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wi = wave & 1, wj = wave >> 1;
  // 16 x 16 blocks wholly outside C (their operands are zero padding and
  // their results are never stored) skip the matrix cores; wave-uniform
  bool live[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) live[a][b] = i0 + wi * 32 + a * 16 < g.m && j0 + wj * 32 + b * 16 < g.n;
  A4 p1[2][2], p2[2][2], p3[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      p1[a][b] = A4{0, 0, 0, 0};
      p2[a][b] = A4{0, 0, 0, 0};
      p3[a][b] = A4{0, 0, 0, 0};
    }
  const int lrow = threadIdx.x & 15, lcol = threadIdx.x >> 4;  // 16 rows x 16 column groups
  // the next slab is loaded into registers while the current one is multiplied
  C px[4], py[4];
  auto gload = [&](int64_t k0) {
    const int64_t gr = k0 + lrow;
    const bool rok = gr < r1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = lcol + 16 * q;
      px[q] = (rok && i0 + c < g.m) ? X[(int64_t)(i0 + c) * ldx + gr] : cmk<C>(0, 0);
      py[q] = (rok && j0 + c < g.n) ? Y[(int64_t)(j0 + c) * ldy + gr] : cmk<C>(0, 0);
    }
  };
  if (r0 < r1) gload(r0);
  for (int64_t k0 = r0; k0 < r1; k0 += OV_KS) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = lcol + 16 * q;
      xr[lrow][c] = px[q].x;
      xi[lrow][c] = px[q].y;
      xs[lrow][c] = px[q].x - px[q].y;
      yr[lrow][c] = py[q].x;
      yi[lrow][c] = py[q].y;
      ys[lrow][c] = py[q].x + py[q].y;
    }
    __syncthreads();
    if (k0 + OV_KS < r1) gload(k0 + OV_KS);
#pragma unroll
    for (int kk = 0; kk < OV_KS / 4; ++kk) {
      const int k = kk * 4 + (lane >> 4);
      R ar[2], ai[2], as[2], br[2], bi[2], bs[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int ii = wi * 32 + a * 16 + (lane & 15);
        ar[a] = xr[k][ii];
        ai[a] = xi[k][ii];
        as[a] = xs[k][ii];
        const int jj = wj * 32 + a * 16 + (lane & 15);
        br[a] = yr[k][jj];
        bi[a] = yi[k][jj];
        bs[a] = ys[k][jj];
      }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          if (live[a][b]) {
            p1[a][b] = M::op(ar[a], br[b], p1[a][b]);
            p2[a][b] = M::op(ai[a], bi[b], p2[a][b]);
            p3[a][b] = M::op(as[a], bs[b], p3[a][b]);
          }
    }
    __syncthreads();
  }
  double2* P = part + ((int64_t)kz * g.nchunk + chunk) * g.m * g.n;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + wi * 32 + a * 16 + M::row(lane, r);
        const int j = j0 + wj * 32 + b * 16 + (lane & 15);
        const double q1 = (double)p1[a][b][r], q2 = (double)p2[a][b][r], q3 = (double)p3[a][b][r];
        if (i < g.m && j < g.n) P[(int64_t)j * g.m + i] = make_double2(q1 + q2, q3 - q1 + q2);
      }
}

// row groups of the wavefronts of a tile of nblk needed blocks
__host__ __device__ constexpr int ov_row_groups(int nblk) { return nblk <= 4 ? 4 : (nblk <= 2 * kOvBlocks ? 2 : 1); }

// Whether the tiles of an m x n overlap take the quarter layout: matrix-core
// steps per slab of the busiest wavefront against the dealt layout's, whose
// operands are single-use and cost more LDS reads per step.  They are compared
// summed over the tiles, or, while every workgroup has a CU to itself, by the
// tile that takes longest.  The dealt layout wins from a quarter fewer steps on,
// a third fewer where none of it comes from a diagonal.  Its time over the quarter
// layout's, FP64 / FP32, by the ratio of steps: 1: 1.13 / 1.20 (1503 x 160
// Hermitian, by the longest tile); 1.23: 1.09 / 1.05 (62669 x 200 x 100); 1.33:
// 1.06 / 0.92 (62669 x 128 Hermitian); 1.36: 0.91 / 0.96 (62669 x 200 Hermitian);
// 1.44: 1.09 / 1.04 (40000 x 160 x 80); 1.6: 0.94 / 1.04 (40000 x 80 x 40); 1.75:
// 0.84 / 0.93 (62669 x 160 Hermitian); 5.3: 0.68 / 0.78 (62669 x 20 Hermitian).
inline bool ov_quarter(int m, int n, bool herm, int64_t workgroups) {
  const int tm = (int)ceil_div(m, OV_T), tn = (int)ceil_div(n, OV_T);
  const bool alone = workgroups <= kOvCus;
  int64_t quarter = 0, dealt = 0;
  auto add = [alone](int64_t& t, int64_t x) { t = alone ? std::max(t, x) : t + x; };
  for (int ti = 0; ti < tm; ++ti)
    for (int tj = herm ? ti : 0; tj < tn; ++tj) {
      const int na = std::min(4, (int)ceil_div(m - ti * OV_T, 16)), nb = std::min(4, (int)ceil_div(n - tj * OV_T, 16));
      const int nblk = herm && ti == tj ? na * (na + 1) / 2 : na * nb, ks = ov_row_groups(nblk);
      add(quarter, std::min(2, na) * std::min(2, nb) * 4);
      add(dealt, ceil_div(nblk, 4 / ks) * (4 / ks));
    }
  return herm ? 3 * quarter <= 4 * dealt : 2 * quarter <= 3 * dealt;
}

// The same overlap with the 16 x 16 blocks that C needs (inside C; on a
// diagonal tile of a Hermitian result a <= b) dealt evenly to the wavefronts;
// with few of them the wavefronts also split each slab's rows (ksp groups,
// group kgrp takes every ksp-th step of four rows, the sums are added at the
// end).  A 24-column tile then keeps all four matrix cores busy where a
// quarter per wavefront leaves three idle.  Measured in FP64, per call: 20
// columns of 1503 rows 42 -> 10 us (with more row chunks); 48 columns of 17 x
// 17.5k rows 159 -> 109 us, now near the HBM time of the operands; 160 and 80
// columns of 62669 rows 212 -> 174 us.  Every operand is read from LDS for
// each use: full tiles (161214 x 600 x 300) ran 9 % slower than by quarters.
template <typename R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_overlap_dealt(const cx_t<R>* __restrict__ X, int64_t ldx, int64_t sx,
                                                 const cx_t<R>* __restrict__ Y, int64_t ldy, int64_t sy,
                                                 const int* __restrict__ npwk, OvGeom g,
                                                 double2* __restrict__ part) {
  using M = Mfma<R>;
  using A4 = typename M::acc;
  using C = cx_t<R>;
  // slab operands for the three real products of the complex product
  // conj(x) y (Gauss):  P1 = xr yr,  P2 = xi yi,  P3 = (xr - xi)(yr + yi);
  // Re = P1 + P2,  Im = P3 - P1 + P2
  __shared__ __align__(16) R sl[6][OV_KS][OV_PAD];
  auto xr = sl[0], xi = sl[1], xs = sl[2], yr = sl[3], yi = sl[4], ys = sl[5];
  // work item: tile fastest, then row chunk, then k-point; the tiles of one
  // chunk share an XCD and read the same rows through its L2
  const int64_t w = xcd_item(blockIdx.x, gridDim.x);
  const int chunk = (int)((w / g.ntiles) % g.nchunk);
  const int kz = (int)(w / ((int64_t)g.ntiles * g.nchunk));
  X += kz * sx;
  Y += kz * sy;
  const int64_t npw = npwk ? (int64_t)npwk[kz] : g.npw;
  // tile coordinates
  int ti, tj;
  int t = (int)(w % g.ntiles);
  if (g.herm) {
    ti = 0;
    while (t >= g.tm - ti) { t -= g.tm - ti; ++ti; }
    tj = ti + t;
  } else {
    ti = t % g.tm;
    tj = t / g.tm;
  }
  const int i0 = ti * OV_T, j0 = tj * OV_T;
  const int64_t r0 = (int64_t)chunk * g.kch;
  const int64_t r1 = std::min<int64_t>(npw, r0 + g.kch);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int na = min(OV_T / 16, (g.m - i0 + 15) / 16), nbk = min(OV_T / 16, (g.n - j0 + 15) / 16);
  const bool tri = g.herm && ti == tj;
  const int nblk = tri ? na * (na + 1) / 2 : na * nbk;
  const int ksp = ov_row_groups(nblk);
  const int wpg = 4 / ksp, kgrp = wave / wpg;
  const int per = (nblk + wpg - 1) / wpg;
  const int q0 = (wave % wpg) * per, nq = max(0, min(per, nblk - q0));
  constexpr int NQ = kOvBlocks;
  int ba[NQ], bb[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    int e = max(0, min(q0 + q, nblk - 1));
    if (tri) {
      int c = 0;
      while (e > c) e -= ++c;
      ba[q] = e * 16;
      bb[q] = c * 16;
    } else {
      ba[q] = (e % na) * 16;
      bb[q] = (e / na) * 16;
    }
  }
  A4 p1[NQ], p2[NQ], p3[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    p1[q] = A4{0, 0, 0, 0};
    p2[q] = A4{0, 0, 0, 0};
    p3[q] = A4{0, 0, 0, 0};
  }
  const int lrow = threadIdx.x & 15, lcol = threadIdx.x >> 4;  // 16 rows x 16 column groups
  // the next slab is loaded into registers while the current one is multiplied
  C px[4], py[4];
  auto gload = [&](int64_t k0) {
    const int64_t gr = k0 + lrow;
    const bool rok = gr < r1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = lcol + 16 * q;
      px[q] = (rok && i0 + c < g.m) ? X[(int64_t)(i0 + c) * ldx + gr] : cmk<C>(0, 0);
      py[q] = (rok && j0 + c < g.n) ? Y[(int64_t)(j0 + c) * ldy + gr] : cmk<C>(0, 0);
    }
  };
  if (r0 < r1) gload(r0);
  for (int64_t k0 = r0; k0 < r1; k0 += OV_KS) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = lcol + 16 * q;
      xr[lrow][c] = px[q].x;
      xi[lrow][c] = px[q].y;
      xs[lrow][c] = px[q].x - px[q].y;
      yr[lrow][c] = py[q].x;
      yi[lrow][c] = py[q].y;
      ys[lrow][c] = py[q].x + py[q].y;
    }
    __syncthreads();
    if (k0 + OV_KS < r1) gload(k0 + OV_KS);
    // the operands of the next block are read while the current one is multiplied
    R o[2][6];
    auto fetch = [&](int kk, int q, R* v) {
      const int k = kk * 4 + (lane >> 4), ii = ba[q] + (lane & 15), jj = bb[q] + (lane & 15);
      v[0] = xr[k][ii];
      v[1] = yr[k][jj];
      v[2] = xi[k][ii];
      v[3] = yi[k][jj];
      v[4] = xs[k][ii];
      v[5] = ys[k][jj];
    };
    for (int kk = kgrp; kk < OV_KS / 4; kk += ksp) {
      fetch(kk, 0, o[0]);
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        if (q < nq) {
          if (q + 1 < nq) fetch(kk, q + 1 < NQ ? q + 1 : q, o[(q + 1) & 1]);
          const R* v = o[q & 1];
          p1[q] = M::op(v[0], v[1], p1[q]);
          p2[q] = M::op(v[2], v[3], p2[q]);
          p3[q] = M::op(v[4], v[5], p3[q]);
        }
    }
    __syncthreads();
  }
  // the row groups' sums meet in LDS (the slab buffers), group 0 adds them
  double2* ex = reinterpret_cast<double2*>(&sl[0][0][0]);
  static_assert(sizeof(sl) >= 3 * 256 * sizeof(double2) && alignof(R) <= 16, "exchange of one block per wavefront");
  double2* P = part + ((int64_t)kz * g.nchunk + chunk) * g.m * g.n;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    double2 v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double q1 = (double)p1[q][r], q2 = (double)p2[q][r], q3 = (double)p3[q][r];
      v[r] = make_double2(q1 + q2, q3 - q1 + q2);
    }
    // one block of every wavefront at a time: 3 groups x 256 values at most
    // (ksp 4), 2 wavefronts x 256 (ksp 2)
    if (ksp > 1) {
      const int w0 = wave % wpg;
      if (kgrp > 0 && q < nq)
#pragma unroll
        for (int r = 0; r < 4; ++r) ex[(((kgrp - 1) * wpg + w0) * 4 + r) * 64 + lane] = v[r];
      __syncthreads();
      if (kgrp == 0 && q < nq)
        for (int h = 1; h < ksp; ++h)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const double2 u = ex[(((h - 1) * wpg + w0) * 4 + r) * 64 + lane];
            v[r] = make_double2(v[r].x + u.x, v[r].y + u.y);
          }
      __syncthreads();
    }
    if (kgrp == 0 && q < nq)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + ba[q] + M::row(lane, r), j = j0 + bb[q] + (lane & 15);
        if (i < g.m && j < g.n) P[(int64_t)j * g.m + i] = v[r];
      }
  }
}

// ---- complex64 data on the BF16 matrix cores --------------------------
// Each FP32 operand value v is split into NT bf16 terms t_0 + t_1 + ...,
// t_j = bf16(v - t_0 - ... - t_{j-1}) rounded to nearest even (each
// subtraction is exact in FP32).  A real product keeps the term products
// t_a s_b with a + b < NT: NT = 1 is plain BF16 (8 significant bits),
// NT = 2 three products (about 16 bits), NT = 3 six products (about FP32's
// 24).  Accumulation is FP32 on the matrix cores, chunk sums FP64 as above.
// The 16x16x32 BF16 MFMA takes 8 consecutive k per lane:
//   A (16x32): A[l%16][8*(l/16) + e]   B (32x16): B[8*(l/16) + e][l%16]
//   D as the f32 16x16x4 form (register r holds D[4*(l/16) + r][l%16]).
// Operands are split once, when their slab is staged into LDS ([column][k
// slot], slots contiguous, so a lane's 8 values are one 16-byte read).
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int BF_P = 6;    // LDS pitch of a column in bf8 units (96 bytes; measured 3 % faster than 80 or 64)

__device__ __forceinline__ f4 mfma_bf16(bf8 a, bf8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// out[t] = term t of the 8 values v (v is consumed)
template <int NT> __device__ __forceinline__ void bf_split(float (&v)[8], bf8 (&out)[NT]) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const __bf16 h = (__bf16)v[e];
      out[t][e] = h;
      if (t + 1 < NT) v[e] -= (float)h;
    }
}

// acc += sum over term pairs (a, b), a + b < NT, of A_a B_b
template <int NT> __device__ __forceinline__ f4 bf_products(const bf8 (&A)[NT], const bf8 (&B)[NT], f4 acc) {
#pragma unroll
  for (int s = NT - 1; s >= 0; --s)  // smallest terms first
#pragma unroll
    for (int a = 0; a <= s; ++a) acc = mfma_bf16(A[a], B[s - a], acc);
  return acc;
}

// Stage two complex values of one column as the three Gauss planes (re, im,
// re + sgn*im), each split into NT terms, into the adjacent k slots 2*slot
// and 2*slot + 1 of LDS column `col` (one 4-byte store per plane and term).
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
template <int NT, int TT>
__device__ __forceinline__ void bf_stage2(float2 v0, float2 v1, float sgn, bf8 (*L)[NT][TT][BF_P], int col, int slot) {
  float a[3][2] = {{v0.x, v1.x}, {v0.y, v1.y}, {v0.x + sgn * v0.y, v1.x + sgn * v1.y}};
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      bf2 h;
      h[0] = (__bf16)a[p][0];
      h[1] = (__bf16)a[p][1];
      reinterpret_cast<bf2*>(&L[p][t][col][0])[slot] = h;
      if (t + 1 < NT) {
        a[p][0] -= (float)h[0];
        a[p][1] -= (float)h[1];
      }
    }
}

// TT = 64: 4 wavefronts, each a 32 x 32 block of the tile; TT = 128: 8
// wavefronts, each 64 rows x 32 columns.  The larger tile reads every operand
// row half as often per matrix-core operation (fewer tiles share a row chunk)
// and splits and stages half as many values per product.
template <int TT> constexpr int kBfWaves = TT == 64 ? 4 : 8;
template <int NT, int TT>
__global__ __launch_bounds__(64 * kBfWaves<TT>) __attribute__((amdgpu_waves_per_eu(2))) void k_overlap_bf16(
    const float2* __restrict__ X, int64_t ldx, int64_t sx, const float2* __restrict__ Y, int64_t ldy, int64_t sy,
    const int* __restrict__ npwk, OvGeom g, double2* __restrict__ part) {
  static_assert(TT == 64 || TT == 128, "tile edge 64 or 128");
  constexpr int AB = TT / 32;  // 16-row blocks per wavefront
  // planes: conj(x) y = P1 + P2 + i (P3 - P1 + P2), P1 = xr yr, P2 = xi yi,
  // P3 = (xr - xi)(yr + yi)
  __shared__ bf8 lx[3][NT][TT][BF_P], ly[3][NT][TT][BF_P];
  const int64_t w = xcd_item(blockIdx.x, gridDim.x);
  const int chunk = (int)((w / g.ntiles) % g.nchunk);
  const int kz = (int)(w / ((int64_t)g.ntiles * g.nchunk));
  X += kz * sx;
  Y += kz * sy;
  const int64_t npw = npwk ? (int64_t)npwk[kz] : g.npw;
  int ti, tj;
  int t = (int)(w % g.ntiles);
  if (g.herm) {
    ti = 0;
    while (t >= g.tm - ti) { t -= g.tm - ti; ++ti; }
    tj = ti + t;
  } else {
    ti = t % g.tm;
    tj = t / g.tm;
  }
  const int i0 = ti * TT, j0 = tj * TT;
  const int64_t r0 = (int64_t)chunk * g.kch;
  const int64_t r1 = std::min<int64_t>(npw, r0 + g.kch);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wi = wave & 1, wj = wave >> 1;
  const int ri = wi * (TT / 2), cj = wj * 32;  // the wavefront's rows and columns in the tile
  // 16 x 16 blocks wholly outside C (their operands are zero padding and
  // their results are never stored) skip the matrix cores; wave-uniform
  bool live[AB][2];
#pragma unroll
  for (int a = 0; a < AB; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) live[a][b] = i0 + ri + a * 16 < g.m && j0 + cj + b * 16 < g.n;
  f4 p1[AB][2], p2[AB][2], p3[AB][2];
#pragma unroll
  for (int a = 0; a < AB; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      p1[a][b] = f4{0, 0, 0, 0};
      p2[a][b] = f4{0, 0, 0, 0};
      p3[a][b] = f4{0, 0, 0, 0};
    }
  // staging: wave w, pass q: tile column 16 w + 4 q + lane/16, slab rows
  // sr = lane%16 and sr + 16, so the lanes of a column read 128 contiguous
  // bytes.  The two rows go to the adjacent k slots 2 sr and 2 sr + 1; both
  // operands use the same slot order, so the sum over k is unchanged.
  const int sr = lane & 15;
  float2 px[4][2], py[4][2];
  auto gload = [&](int64_t k0) {
    const int64_t ga = k0 + sr, gb = k0 + sr + 16;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = 16 * wave + 4 * q + (lane >> 4);
      const bool xok = i0 + c < g.m, yok = j0 + c < g.n;
      const float2* xc = X + (int64_t)(xok ? i0 + c : 0) * ldx;
      const float2* yc = Y + (int64_t)(yok ? j0 + c : 0) * ldy;
      px[q][0] = (xok && ga < r1) ? xc[ga] : make_float2(0.f, 0.f);
      px[q][1] = (xok && gb < r1) ? xc[gb] : make_float2(0.f, 0.f);
      py[q][0] = (yok && ga < r1) ? yc[ga] : make_float2(0.f, 0.f);
      py[q][1] = (yok && gb < r1) ? yc[gb] : make_float2(0.f, 0.f);
    }
  };
  if (r0 < r1) gload(r0);
  const int kg = lane >> 4;
  for (int64_t k0 = r0; k0 < r1; k0 += BF_KS) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = 16 * wave + 4 * q + (lane >> 4);
      bf_stage2<NT, TT>(px[q][0], px[q][1], -1.f, lx, c, sr);
      bf_stage2<NT, TT>(py[q][0], py[q][1], 1.f, ly, c, sr);
    }
    __syncthreads();
    if (k0 + BF_KS < r1) gload(k0 + BF_KS);
    bf8 B[2][3][NT];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int jj = cj + b * 16 + (lane & 15);
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int q = 0; q < NT; ++q) B[b][p][q] = ly[p][q][jj][kg];
    }
#pragma unroll
    for (int a = 0; a < AB; ++a) {
      const int ii = ri + a * 16 + (lane & 15);
      bf8 A[3][NT];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int q = 0; q < NT; ++q) A[p][q] = lx[p][q][ii][kg];
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (live[a][b]) {
          p1[a][b] = bf_products<NT>(A[0], B[b][0], p1[a][b]);
          p2[a][b] = bf_products<NT>(A[1], B[b][1], p2[a][b]);
          p3[a][b] = bf_products<NT>(A[2], B[b][2], p3[a][b]);
        }
    }
    __syncthreads();
  }
  double2* P = part + ((int64_t)kz * g.nchunk + chunk) * g.m * g.n;
#pragma unroll
  for (int a = 0; a < AB; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + ri + a * 16 + Mfma<float>::row(lane, r);
        const int j = j0 + cj + b * 16 + (lane & 15);
        const double q1 = (double)p1[a][b][r], q2 = (double)p2[a][b][r], q3 = (double)p3[a][b][r];
        if (i < g.m && j < g.n) P[(int64_t)j * g.m + i] = make_double2(q1 + q2, q3 - q1 + q2);
      }
}

// ---- two-term BF16 products of interleaved complex values ----------------
// For large blocks the complex products are real ones of twice the depth: an
// operand column is its interleaved (re, im) sequence, split once into a high
// and a low bf16 term while its slab is staged, and
//   conj(x) y:  Re = (xr, xi) . (yr, yi),   Im = (xr, xi) . (yi, -yr)
//   x u:        Re = (xr, -xi) . (ur, ui),  Im = (xi, xr) . (ur, ui)
// so an operand's other form is a half-word rotation and a sign flip of
// registers.  Four real products per complex one, where the
// kernels above take Gauss's three: a third more matrix-core work, but two
// thirds of the LDS traffic and of the split's vector work, which is what
// bounded those (10-25 % matrix-core busy), two accumulators per block
// instead of three, and no cancellation between the products (error against
// the exact product 4.5e-6 of the largest element against 6.9e-6 at 3001
// rows).  A wavefront owns 64 x 64 of C or Z: 96 matrix-core instructions per
// 16 complex rows for 16 operand fragments read.
constexpr int CX_KS = 16;  // complex rows per slab: one 16x16x32 MFMA of interleaved values

typedef __bf16 bfp __attribute__((ext_vector_type(2)));
typedef float fp2 __attribute__((ext_vector_type(2)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

typedef unsigned int u2 __attribute__((ext_vector_type(2)));

// term t of the complex value with the FP32 bits (re, im) as one dword (re low, im high)
__device__ __forceinline__ void cx_split(unsigned re, unsigned im, unsigned (&t)[2]) {
  const fp2 f = {__builtin_bit_cast(float, re), __builtin_bit_cast(float, im)};
  const bfp h = __builtin_convertvector(f, bfp);
  const fp2 hf = __builtin_convertvector(h, fp2);
  const bfp l = __builtin_convertvector(f - hf, bfp);
  t[0] = __builtin_bit_cast(unsigned, h);
  t[1] = __builtin_bit_cast(unsigned, l);
}
// (re, im) -> (im, -re)
__device__ __forceinline__ u4 cx_swap(u4 v) {
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = __builtin_amdgcn_alignbit(v[e], v[e], 16) ^ 0x80000000u;
  return v;
}
__device__ __forceinline__ f4 cx_mfma(u4 a, u4 b, f4 c) {
  return mfma_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c);
}
// LDS slot (16 bytes: four complex values of one term) of column c, row group
// g of a slab; the XOR keeps the 16 lanes of an access on distinct banks
__device__ __forceinline__ int cx_slot(int c, int g) { return c * 4 + (g ^ ((c >> 2) & 3)); }

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_overlap_cx(
    const float2* __restrict__ X, int64_t ldx, int64_t sx, const float2* __restrict__ Y, int64_t ldy, int64_t sy,
    const int* __restrict__ npwk, OvGeom g, double2* __restrict__ part) {
  constexpr int TT = 128;
  __shared__ u4 lx[2][2][TT * 4], ly[2][2][TT * 4];  // [buffer][term][slot]
  const int64_t w = xcd_item(blockIdx.x, gridDim.x);
  const int chunk = (int)((w / g.ntiles) % g.nchunk);
  const int kz = (int)(w / ((int64_t)g.ntiles * g.nchunk));
  X += kz * sx;
  Y += kz * sy;
  const int64_t npw = npwk ? (int64_t)npwk[kz] : g.npw;
  int ti, tj;
  int t = (int)(w % g.ntiles);
  if (g.herm) {
    ti = 0;
    while (t >= g.tm - ti) { t -= g.tm - ti; ++ti; }
    tj = ti + t;
  } else {
    ti = t % g.tm;
    tj = t / g.tm;
  }
  const int i0 = ti * TT, j0 = tj * TT;
  const int64_t r0 = (int64_t)chunk * g.kch;
  const int64_t r1 = std::min<int64_t>(npw, r0 + g.kch);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ri = (wave & 1) * 64, cj = (wave >> 1) * 64;
  // 16-column blocks of this wavefront inside C; none below the diagonal of a
  // Hermitian result
  int na = max(0, min(4, (g.m - i0 - ri + 15) / 16)), nb = max(0, min(4, (g.n - j0 - cj + 15) / 16));
  if (g.herm && ti == tj && ri > cj) nb = 0;
  f4 re[4][4], im[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) re[a][b] = im[a][b] = f4{0, 0, 0, 0};
  // staging: pass q, column 32 q + thread / 8, rows 2 (thread % 8) and the
  // next, one 16-byte buffer load (columns past C: out of range, zero); only
  // the last slab of a chunk masks rows
  const int sc = threadIdx.x >> 3, sp = threadIdx.x & 7;
  const int64_t lastx = (int64_t)(min(TT, g.m - i0) - 1) * ldx, lasty = (int64_t)(min(TT, g.n - j0) - 1) * ldy;
  uint32_t ox[4], oy[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int c = 32 * q + sc;
    ox[q] = i0 + c < g.m ? (uint32_t)(c * ldx + 2 * sp) * 8u : kOob;
    oy[q] = j0 + c < g.n ? (uint32_t)(c * ldy + 2 * sp) * 8u : kOob;
  }
  u4 px[4], py[4];
  auto gload = [&](int64_t k0) {
    const int rows = (int)min((int64_t)CX_KS, r1 - k0) - 2 * sp;  // of this lane's two
    const auto rx = buf_rsrc(X + (int64_t)i0 * ldx + k0, (uint32_t)((lastx + r1 - k0) * 8));
    const auto ry = buf_rsrc(Y + (int64_t)j0 * ldy + k0, (uint32_t)((lasty + r1 - k0) * 8));
    if (r1 - k0 >= CX_KS) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        px[q] = __builtin_amdgcn_raw_buffer_load_b128(rx, (int)ox[q], 0, 0);
        py[q] = __builtin_amdgcn_raw_buffer_load_b128(ry, (int)oy[q], 0, 0);
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const u2 zero = {0u, 0u};
        const u2 x0 = rows > 0 ? __builtin_amdgcn_raw_buffer_load_b64(rx, (int)ox[q], 0, 0) : zero;
        const u2 x1 = rows > 1 ? __builtin_amdgcn_raw_buffer_load_b64(rx, (int)ox[q] + 8, 0, 0) : zero;
        const u2 y0 = rows > 0 ? __builtin_amdgcn_raw_buffer_load_b64(ry, (int)oy[q], 0, 0) : zero;
        const u2 y1 = rows > 1 ? __builtin_amdgcn_raw_buffer_load_b64(ry, (int)oy[q] + 8, 0, 0) : zero;
        px[q] = u4{x0[0], x0[1], x1[0], x1[1]};
        py[q] = u4{y0[0], y0[1], y1[0], y1[1]};
      }
    }
  };
  auto put = [&](u4 (&l)[2][TT * 4], int c, u4 v) {
    unsigned t0[2], t1[2];
    cx_split(v[0], v[1], t0);
    cx_split(v[2], v[3], t1);
#pragma unroll
    for (int q = 0; q < 2; ++q)
      reinterpret_cast<uint2*>(&l[q][cx_slot(c, sp >> 1)])[sp & 1] = make_uint2(t0[q], t1[q]);
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      put(lx[buf], 32 * q + sc, px[q]);
      put(ly[buf], 32 * q + sc, py[q]);
    }
  };
  const int lc = lane & 15, kg = lane >> 4;
  if (r0 < r1) {
    gload(r0);
    stage(0);
  }
  __syncthreads();
  int buf = 0;
  for (int64_t k0 = r0; k0 < r1; k0 += CX_KS, buf ^= 1) {
    const bool more = k0 + CX_KS < r1;
    if (more) gload(k0 + CX_KS);
    u4 A[4][2];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int q = 0; q < 2; ++q) A[a][q] = lx[buf][q][cx_slot(ri + a * 16 + lc, kg)];
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (b < nb) {
        u4 B[2], D[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          B[q] = ly[buf][q][cx_slot(cj + b * 16 + lc, kg)];
          D[q] = cx_swap(B[q]);
        }
        // smallest terms first
#pragma unroll
        for (int a = 0; a < 4; ++a)
          if (a < na) {
            re[a][b] = cx_mfma(A[a][0], B[1], re[a][b]);
            im[a][b] = cx_mfma(A[a][0], D[1], im[a][b]);
            re[a][b] = cx_mfma(A[a][1], B[0], re[a][b]);
            im[a][b] = cx_mfma(A[a][1], D[0], im[a][b]);
            re[a][b] = cx_mfma(A[a][0], B[0], re[a][b]);
            im[a][b] = cx_mfma(A[a][0], D[0], im[a][b]);
          }
      }
    if (more) stage(buf ^ 1);
    __syncthreads();
  }
  double2* P = part + ((int64_t)kz * g.nchunk + chunk) * g.m * g.n;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (a < na && b < nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = i0 + ri + a * 16 + Mfma<float>::row(lane, r), j = j0 + cj + b * 16 + lc;
          if (i < g.m && j < g.n) P[(int64_t)j * g.m + i] = make_double2((double)re[a][b][r], (double)im[a][b][r]);
        }
}

// Z = X U, 128 rows x 128 columns per workgroup, 64 x 64 per wavefront.  U is
// split once per call (k_rotate_split) into the LDS images of its slabs, 16
// rows x 128 columns in two terms, which each workgroup copies in 16-byte
// pieces; X's rows go straight into the A fragments (lane: one row, four
// columns of X).
constexpr int RC_ROWS = 128, RC_COLS = 128;
constexpr int RC_IMG = 2 * RC_COLS * 4;  // 16-byte slots of one slab image: [term][slot]

// image (column block, slab) of matrix kz at img + ((kz*ncb + block)*nslab + slab)*RC_IMG
__global__ __launch_bounds__(256) void k_rotate_split(const double2* __restrict__ U, int ldu, int64_t su, int m, int n,
                                                      u4* __restrict__ img) {
  const int nslab = gridDim.x, slab = blockIdx.x, cb = blockIdx.y;
  U += blockIdx.z * su;
  img += (((int64_t)blockIdx.z * gridDim.y + cb) * nslab + slab) * RC_IMG;
  for (int s = threadIdx.x; s < RC_COLS * 4; s += 256) {
    const int c = s >> 2, g = s & 3, col = cb * RC_COLS + c;
    u4 h, l;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = slab * CX_KS + 4 * g + e;
      const double2 v = (k < m && col < n) ? U[(int64_t)col * ldu + k] : make_double2(0.0, 0.0);
      unsigned t[2];
      cx_split(__builtin_bit_cast(unsigned, (float)v.x), __builtin_bit_cast(unsigned, (float)v.y), t);
      h[e] = t[0];
      l[e] = t[1];
    }
    img[cx_slot(c, g)] = h;
    img[RC_COLS * 4 + cx_slot(c, g)] = l;
  }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_rotate_cx(
    const float2* __restrict__ X, const float2* __restrict__ X2, int64_t ldx, int64_t sx, const u4* __restrict__ img,
    int m, int n, int64_t npw, const int* __restrict__ npwk, float2* __restrict__ Z, float2* __restrict__ Z2,
    int64_t ldz, int64_t sz) {
  __shared__ u4 lu[2][RC_IMG];
  const int ncb = (int)ceil_div(n, RC_COLS), nslab = (int)ceil_div(m, CX_KS);
  const int64_t nrb = ceil_div(npw, RC_ROWS);
  const int64_t w = xcd_item(blockIdx.x, gridDim.x);
  const int64_t rb = (w / ncb) % nrb;
  const int kz = (int)(w / (ncb * nrb));
  const int64_t nrow = npwk ? (int64_t)npwk[kz] : npw;
  if (rb * RC_ROWS >= nrow) return;
  X = (blockIdx.y ? X2 : X) + kz * sx;
  Z = (blockIdx.y ? Z2 : Z) + kz * sz;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cb = (int)(w % ncb), j0 = cb * RC_COLS;
  img += ((int64_t)kz * ncb + cb) * nslab * RC_IMG;
  const int64_t g0 = rb * RC_ROWS + wave * 32;
  const int lc = lane & 15, kg = lane >> 4;
  const int na = (int)max((int64_t)0, min((int64_t)2, (nrow - g0 + 15) / 16));
  const int nb = min(8, (n - j0 + 15) / 16);
  f4 re[2][8], im[2][8];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 8; ++b) re[a][b] = im[a][b] = f4{0, 0, 0, 0};
  // X: lane offsets of row lc of the wavefront's block, columns 4 kg + e.
  // Rows past the k-point's only reach rows of Z that are not stored; columns
  // past m read zero.
  uint32_t xo[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) xo[e] = (uint32_t)((4 * kg + e) * ldx + lc) * 8u;
  constexpr int UQ = RC_IMG / 256;
  u4 pu[UQ];
  u2 p0[2][4] = {}, p1[2][4] = {};
  auto uload = [&](int s) {
    const u4* is = img + (int64_t)s * RC_IMG + threadIdx.x;
#pragma unroll
    for (int q = 0; q < UQ; ++q) pu[q] = is[q * 256];
  };
  auto xload = [&](int s, u2 (&px)[2][4]) {
    if (na == 0 || s >= nslab) return;
    const int k0 = s * CX_KS;
    // in range: rows past the k-point's of all columns but the last, zero past that
    const auto rx = buf_rsrc(X + (int64_t)k0 * ldx + g0, (uint32_t)(((m - 1 - k0) * ldx + nrow - g0) * 8));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t o = k0 + 4 * kg + e < m ? xo[e] : kOob;
#pragma unroll
      for (int a = 0; a < 2; ++a) px[a][e] = __builtin_amdgcn_raw_buffer_load_b64(rx, (int)(o + a * 128), 0, 0);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int q = 0; q < UQ; ++q) lu[buf][q * 256 + threadIdx.x] = pu[q];
  };
  auto step = [&](int s, u2 (&px)[2][4]) {
    const int buf = s & 1;
    // (xr, -xi) for Re and (xi, xr) for Im against the same (ur, ui)
    u4 A[2][2], D[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        unsigned t[2];
        cx_split(px[a][e][0], px[a][e][1], t);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          A[a][q][e] = t[q] ^ 0x80000000u;
          D[a][q][e] = __builtin_amdgcn_alignbit(t[q], t[q], 16);
        }
      }
    const bool more = s + 1 < nslab;
    if (more) uload(s + 1);
    xload(s + 2, px);
#pragma unroll
    for (int b = 0; b < 8; ++b)
      if (b < nb) {
        u4 B[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) B[q] = lu[buf][q * RC_COLS * 4 + cx_slot(b * 16 + lc, kg)];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          re[a][b] = cx_mfma(A[a][0], B[1], re[a][b]);
          im[a][b] = cx_mfma(D[a][0], B[1], im[a][b]);
        }
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          re[a][b] = cx_mfma(A[a][1], B[0], re[a][b]);
          im[a][b] = cx_mfma(D[a][1], B[0], im[a][b]);
        }
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          re[a][b] = cx_mfma(A[a][0], B[0], re[a][b]);
          im[a][b] = cx_mfma(D[a][0], B[0], im[a][b]);
        }
      }
    if (more) stage(buf ^ 1);
    __syncthreads();
  };
  xload(0, p0);
  xload(1, p1);
  uload(0);
  stage(0);
  __syncthreads();
  for (int s = 0; s < nslab; s += 2) {
    step(s, p0);
    if (s + 1 < nslab) step(s + 1, p1);
  }
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int j = j0 + b * 16 + lc;
    if (j >= n) continue;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t gg = g0 + a * 16 + Mfma<float>::row(lane, r);
        if (gg < nrow) Z[(int64_t)j * ldz + gg] = make_float2(re[a][b][r], im[a][b][r]);
      }
  }
}

// resident 256-thread workgroups of `kern` on the current device (CUs x
// per-CU occupancy)
static int resident_slots(const void* kern, int threads) {
  int dev = 0;
  DEREK_HIP(hipGetDevice(&dev));
  hipDeviceProp_t p;
  DEREK_HIP(hipGetDeviceProperties(&p, dev));
  int per = 0;
  DEREK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, threads, 0));
  return std::max(1, per) * std::max(1, p.multiProcessorCount);
}
template <typename R> static int ov_slots() {
  static const int slots = resident_slots(reinterpret_cast<const void*>(k_overlap<R>), 256);
  return slots;
}
template <int NT, int TT> static int ov_slots_bf16() {
  static const int slots = resident_slots(reinterpret_cast<const void*>(k_overlap_bf16<NT, TT>), 64 * kBfWaves<TT>);
  return slots;
}

static int ov_slots_cx() {
  static const int slots = resident_slots(reinterpret_cast<const void*>(k_overlap_cx), 256);
  return slots;
}

// resident slots of every overlap kernel (FP64, FP32, BF16 with 1..3 terms
// on 64- and 128-wide tiles)
constexpr int kOvKernels = 8;
static void overlap_slots(int out[kOvKernels]) {
  out[0] = ov_slots<double>();
  out[1] = ov_slots<float>();
  out[2] = ov_slots_bf16<1, 64>();
  out[3] = ov_slots_bf16<2, 64>();
  out[4] = ov_slots_bf16<3, 64>();
  out[5] = ov_slots_bf16<1, 128>();
  out[6] = ov_slots_bf16<2, 128>();
  out[7] = ov_slots_cx();
}

int64_t overlap_work_elems(int m, int n, int64_t npw, int batch) {
  int slots[kOvKernels];
  overlap_slots(slots);
  return ov_work_elems(m, n, npw, batch, slots, kOvKernels);
}

int64_t engine_overlap_work_elems(int nb, int nk, int kc, int64_t npw) {
  int slots[kOvKernels];
  overlap_slots(slots);
  return ov_engine_work_elems(nb, nk, kc, npw, slots, kOvKernels);
}

// C[kz] = sum over chunks.  A workgroup takes RD_E consecutive elements;
// its RD_G thread groups each sum every RD_G-th chunk (in increasing
// order), and the group sums are added in group order through LDS, so the
// result does not depend on the launch.
constexpr int RD_E = 32, RD_G = 8;
__global__ __launch_bounds__(RD_E * RD_G) void k_overlap_reduce(const double2* __restrict__ part, OvGeom g,
                                                                double2* __restrict__ C, int ldc, int64_t sc) {
  __shared__ double2 red[RD_G][RD_E];
  const int kz = blockIdx.y;
  const int64_t mn = (int64_t)g.m * g.n;
  const double2* pk = part + (int64_t)kz * g.nchunk * mn;
  double2* Ck = C + kz * sc;
  const int el = threadIdx.x % RD_E, grp = threadIdx.x / RD_E;
  for (int64_t e0 = (int64_t)blockIdx.x * RD_E; e0 < mn; e0 += (int64_t)gridDim.x * RD_E) {
    const int64_t e = e0 + el;
    const int i = e < mn ? (int)(e % g.m) : 0, j = e < mn ? (int)(e / g.m) : 0;
    // Hermitian: only the upper triangle's partials are summed (read in
    // order, so the loads stay coalesced); each sum also gives its mirror
    // element, the conjugate (exactly Hermitian output, real diagonal)
    const bool ok = e < mn && !(g.herm && i > j);
    double sr = 0.0, si = 0.0;
    if (ok)
      for (int c = grp; c < g.nchunk; c += RD_G) {
        const double2 v = pk[(int64_t)c * mn + e];
        sr += v.x;
        si += v.y;
      }
    red[grp][el] = make_double2(sr, si);
    __syncthreads();
    if (grp == 0 && ok) {
      for (int q = 1; q < RD_G; ++q) {
        sr += red[q][el].x;
        si += red[q][el].y;
      }
      if (g.herm && i == j) si = 0.0;
      Ck[(int64_t)j * ldc + i] = make_double2(sr, si);
      if (g.herm && i < j) Ck[(int64_t)i * ldc + j] = make_double2(sr, -si);
    }
    __syncthreads();
  }
}

// Two-term overlaps whose tile edge is left to the size take k_overlap_cx
// once both sides exceed 64 columns and the rows keep every CU busy (8 x
// 161214 rows, 600 columns 9.1 -> 5.4 ms, 300 columns 2.7 -> 2.1 ms; 64 x
// 17529 rows, 96 columns 0.47 -> 0.30 ms, 48 columns 0.17 -> 0.21 ms; one
// k-point of 62669 rows, 160 columns 85 and 82 us, 320 columns 177 and 186
// us), the 64-wide k_overlap_bf16 otherwise.
bool overlap_wide(int m, int n, int64_t npw, int batch) {
  return std::min(m, n) > 64 && npw * batch >= 131072;
}

template <typename R>
void overlap(const cx_t<R>* X, int64_t ldx, int64_t sx, const cx_t<R>* Y, int64_t ldy, int64_t sy, int m, int n,
             int64_t npw, const int* npwk, double2* C, int ldc, int64_t sc, int batch, double2* work,
             int64_t work_cap, bool hermitian, hipStream_t s, int bf16_terms, int64_t max_chunks, int rounds,
             int tile) {
  DEREK_REQUIRE(m > 0 && n > 0 && batch > 0, "overlap: empty block");
  DEREK_REQUIRE(!hermitian || m == n, "overlap: hermitian needs a square result");
  DEREK_REQUIRE(bf16_terms == 0 || (std::is_same<R, float>::value && bf16_terms >= 1 && bf16_terms <= 3),
                "overlap: bf16 terms must be 0, or 1..3 for complex64 data");
  DEREK_REQUIRE(tile == 0 || tile == 64 || tile == 128, "overlap: tile must be 64 or 128 (0: by size)");
  // a tile's columns span less than 2 GiB (32-bit offsets)
  const bool cx = tile == 0 && bf16_terms == 2 && overlap_wide(m, n, npw, batch) &&
                  128 * std::max(ldx, ldy) * 8 < (int64_t)kOob;
  if (tile == 0) tile = 64;
  // the 128-wide tile exists for the BF16 kernels with 1 or 2 terms (three
  // terms of a 128-wide tile need 180 KB of LDS)
  const int tt = cx ? 128 : (bf16_terms && bf16_terms < 3 ? tile : 64);
  const int slots = cx                  ? ov_slots_cx()
                    : bf16_terms == 1   ? (tt == 128 ? ov_slots_bf16<1, 128>() : ov_slots_bf16<1, 64>())
                    : bf16_terms == 2   ? (tt == 128 ? ov_slots_bf16<2, 128>() : ov_slots_bf16<2, 64>())
                    : bf16_terms == 3   ? ov_slots_bf16<3, 64>()
                                        : ov_slots<R>();
  DEREK_REQUIRE(rounds == 1 || rounds == 2 || rounds == 4, "overlap: rounds must be 1, 2 or 4");
  OvGeom g = ov_geom(m, n, npw, hermitian, batch, slots, bf16_terms ? BF_KS : OV_KS, rounds, tt);
  ov_limit_chunks(g, max_chunks, bf16_terms ? BF_KS : OV_KS, batch, slots);
  DEREK_REQUIRE((int64_t)batch * g.nchunk * m * n <= work_cap, "overlap: partial-sum buffer too small");
  const int64_t items = (int64_t)g.ntiles * g.nchunk * batch;
  DEREK_REQUIRE(items < (int64_t)1 << 31, "overlap: too many workgroups");
  const dim3 grid((unsigned)items);
  if constexpr (std::is_same<R, float>::value) {
    const dim3 b64(64 * kBfWaves<64>), b128(64 * kBfWaves<128>);
    if (cx)
      hipLaunchKernelGGL(k_overlap_cx, grid, dim3(256), 0, s, X, ldx, sx, Y, ldy, sy, npwk, g, work);
    else if (bf16_terms == 1 && tt == 64)
      hipLaunchKernelGGL((k_overlap_bf16<1, 64>), grid, b64, 0, s, X, ldx, sx, Y, ldy, sy, npwk, g, work);
    else if (bf16_terms == 2 && tt == 64)
      hipLaunchKernelGGL((k_overlap_bf16<2, 64>), grid, b64, 0, s, X, ldx, sx, Y, ldy, sy, npwk, g, work);
    else if (bf16_terms == 3 && tt == 64)
      hipLaunchKernelGGL((k_overlap_bf16<3, 64>), grid, b64, 0, s, X, ldx, sx, Y, ldy, sy, npwk, g, work);
    else if (bf16_terms == 1)
      hipLaunchKernelGGL((k_overlap_bf16<1, 128>), grid, b128, 0, s, X, ldx, sx, Y, ldy, sy, npwk, g, work);
    else if (bf16_terms == 2)
      hipLaunchKernelGGL((k_overlap_bf16<2, 128>), grid, b128, 0, s, X, ldx, sx, Y, ldy, sy, npwk, g, work);
  }
  if (bf16_terms == 0 && ov_quarter(m, n, hermitian, items))
    hipLaunchKernelGGL(k_overlap<R>, grid, dim3(256), 0, s, X, ldx, sx, Y, ldy, sy, npwk, g, work);
  else if (bf16_terms == 0)
    hipLaunchKernelGGL(k_overlap_dealt<R>, grid, dim3(256), 0, s, X, ldx, sx, Y, ldy, sy, npwk, g, work);
  DEREK_HIP(hipGetLastError());
  const int64_t mn = (int64_t)m * n;
  hipLaunchKernelGGL(k_overlap_reduce, dim3((unsigned)std::min<int64_t>(4096, ceil_div(mn, RD_E)), batch),
                     dim3(RD_E * RD_G), 0, s, work, g, C, ldc, sc);
  DEREK_HIP(hipGetLastError());
}

constexpr int RT_ROWS = 64;
constexpr int RT_COLS = 64;
constexpr int RT_KS = 16;

template <typename R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_rotate(const cx_t<R>* __restrict__ X, const cx_t<R>* __restrict__ X2,
                                                int64_t ldx, int64_t sx, const double2* __restrict__ U, int ldu,
                                                int64_t su, int m, int n, int64_t npw, const int* __restrict__ npwk,
                                                cx_t<R>* __restrict__ Z, cx_t<R>* __restrict__ Z2, int64_t ldz,
                                                int64_t sz) {
  using M = Mfma<R>;
  using A4 = typename M::acc;
  using C = cx_t<R>;
  // three real products of x u (Gauss): P1 = xr ur, P2 = xi ui,
  // P3 = (xr + xi)(ur + ui);  Re = P1 - P2,  Im = P3 - P1 - P2
  __shared__ R ur[RT_KS][RT_COLS + 2], ui[RT_KS][RT_COLS + 2], us[RT_KS][RT_COLS + 2];
  // work item: column block fastest, then row block, then k-point; the
  // column blocks of one row block share an XCD and read its X rows through
  // that XCD's L2
  const int ncb = (int)ceil_div(n, RT_COLS);
  const int64_t nrb = ceil_div(npw, RT_ROWS);
  const int64_t w = xcd_item(blockIdx.x, gridDim.x);
  const int64_t rb = (w / ncb) % nrb;
  const int kz = (int)(w / (ncb * nrb));
  const int64_t nrow = npwk ? (int64_t)npwk[kz] : npw;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t g0 = rb * RT_ROWS + wave * 16;
  if (rb * RT_ROWS >= nrow) return;
  X = (blockIdx.y ? X2 : X) + kz * sx;
  U += kz * su;
  Z = (blockIdx.y ? Z2 : Z) + kz * sz;
  const int j0 = (int)(w % ncb) * RT_COLS;
  // 16-column blocks past n, and a wavefront whose 16 rows are all past the
  // k-point's plane waves, skip the matrix cores (wave-uniform)
  bool live[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) live[b] = j0 + b * 16 < n && rb * RT_ROWS + wave * 16 < nrow;
  const int64_t grow = g0 + (lane & 15);
  const bool rok = grow < nrow;
  A4 p1[4], p2[4], p3[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    p1[b] = A4{0, 0, 0, 0};
    p2[b] = A4{0, 0, 0, 0};
    p3[b] = A4{0, 0, 0, 0};
  }
  // next slab's U (staging thread -> (k = t%16, column group t/16)) and X
  // (A operand: row grow, k = 4 kk + lane/16) held in registers
  const int sk = threadIdx.x & 15, cg = threadIdx.x >> 4;
  double2 pu[4];
  C pxv[RT_KS / 4];
  auto gload = [&](int k0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = cg + 16 * q;
      pu[q] = (k0 + sk < m && j0 + c < n) ? U[(int64_t)(j0 + c) * ldu + k0 + sk] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int kk = 0; kk < RT_KS / 4; ++kk) {
      const int k = k0 + kk * 4 + (lane >> 4);
      pxv[kk] = (rok && k < m) ? X[(int64_t)k * ldx + grow] : cmk<C>(0, 0);
    }
  };
  gload(0);
  for (int k0 = 0; k0 < m; k0 += RT_KS) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = cg + 16 * q;
      const R vr = (R)pu[q].x, vi = (R)pu[q].y;
      ur[sk][c] = vr;
      ui[sk][c] = vi;
      us[sk][c] = vr + vi;
    }
    C xv[RT_KS / 4];
#pragma unroll
    for (int kk = 0; kk < RT_KS / 4; ++kk) xv[kk] = pxv[kk];
    __syncthreads();
    if (k0 + RT_KS < m) gload(k0 + RT_KS);
    R xs[RT_KS / 4];
#pragma unroll
    for (int kk = 0; kk < RT_KS / 4; ++kk) xs[kk] = xv[kk].x + xv[kk].y;
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (live[b]) {
        const int c = b * 16 + (lane & 15);
#pragma unroll
        for (int kk = 0; kk < RT_KS / 4; ++kk) {
          const int k = kk * 4 + (lane >> 4);
          p1[b] = M::op(xv[kk].x, ur[k][c], p1[b]);
          p2[b] = M::op(xv[kk].y, ui[k][c], p2[b]);
          p3[b] = M::op(xs[kk], us[k][c], p3[b]);
        }
      }
    __syncthreads();
  }
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int j = j0 + b * 16 + (lane & 15);
    if (j >= n) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t gg = rb * RT_ROWS + wave * 16 + M::row(lane, r);
      if (gg < nrow) Z[(int64_t)j * ldz + gg] = cmk<C>(p1[b][r] - p2[b][r], p3[b][r] - p1[b][r] - p2[b][r]);
    }
  }
}

// Z = X U with complex64 X on the BF16 matrix cores (terms as in
// k_overlap_bf16): U's slab (rounded to FP32, split) is staged in LDS, X's
// A operand (8 consecutive k of the lane's row) is split in registers.
template <int NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_rotate_bf16(
    const float2* __restrict__ X, const float2* __restrict__ X2, int64_t ldx, int64_t sx,
    const double2* __restrict__ U, int ldu, int64_t su, int m, int n, int64_t npw, const int* __restrict__ npwk,
    float2* __restrict__ Z, float2* __restrict__ Z2, int64_t ldz, int64_t sz) {
  // x u = P1 - P2 + i (P3 - P1 - P2), P1 = xr ur, P2 = xi ui, P3 = (xr + xi)(ur + ui)
  __shared__ bf8 lu[3][NT][64][BF_P];
  const int ncb = (int)ceil_div(n, RT_COLS);
  const int64_t nrb = ceil_div(npw, RT_ROWS);
  const int64_t w = xcd_item(blockIdx.x, gridDim.x);
  const int64_t rb = (w / ncb) % nrb;
  const int kz = (int)(w / (ncb * nrb));
  const int64_t nrow = npwk ? (int64_t)npwk[kz] : npw;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (rb * RT_ROWS >= nrow) return;
  X = (blockIdx.y ? X2 : X) + kz * sx;
  U += kz * su;
  Z = (blockIdx.y ? Z2 : Z) + kz * sz;
  const int j0 = (int)(w % ncb) * RT_COLS;
  // 16-column blocks past n, and a wavefront whose 16 rows are all past the
  // k-point's plane waves, skip the matrix cores (wave-uniform)
  bool live[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) live[b] = j0 + b * 16 < n && rb * RT_ROWS + wave * 16 < nrow;
  const int64_t grow = rb * RT_ROWS + wave * 16 + (lane & 15);
  const bool rok = grow < nrow;
  const int kg = lane >> 4;
  f4 p1[4], p2[4], p3[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    p1[b] = f4{0, 0, 0, 0};
    p2[b] = f4{0, 0, 0, 0};
    p3[b] = f4{0, 0, 0, 0};
  }
  // U staging: wave w, pass q: slab column 16 w + 4 q + lane/16, rows
  // sr = lane%16 and sr + 16 (consecutive lanes, consecutive rows) into the
  // k slots 2 sr, 2 sr + 1.  The A operand's element e (slot 8 kg + e) is
  // therefore X's column k0 + 4 kg + e/2 + 16 (e%2).
  const int sr = lane & 15;
  double2 pu[4][2];
  float2 pxv[8];
  auto gload = [&](int k0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = 16 * wave + 4 * q + (lane >> 4);
      const bool uok = j0 + c < n;
      const double2* uc = U + (int64_t)(uok ? j0 + c : 0) * ldu;
      pu[q][0] = (uok && k0 + sr < m) ? uc[k0 + sr] : make_double2(0.0, 0.0);
      pu[q][1] = (uok && k0 + sr + 16 < m) ? uc[k0 + sr + 16] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = k0 + 4 * kg + (e >> 1) + 16 * (e & 1);
      pxv[e] = (rok && k < m) ? X[(int64_t)k * ldx + grow] : make_float2(0.f, 0.f);
    }
  };
  gload(0);
  for (int k0 = 0; k0 < m; k0 += BF_KS) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = 16 * wave + 4 * q + (lane >> 4);
      bf_stage2<NT, 64>(make_float2((float)pu[q][0].x, (float)pu[q][0].y),
                    make_float2((float)pu[q][1].x, (float)pu[q][1].y), 1.f, lu, c, sr);
    }
    bf8 A[3][NT];
    {
      float r[8], i[8], q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        r[e] = pxv[e].x;
        i[e] = pxv[e].y;
        q[e] = pxv[e].x + pxv[e].y;
      }
      bf_split<NT>(r, A[0]);
      bf_split<NT>(i, A[1]);
      bf_split<NT>(q, A[2]);
    }
    __syncthreads();
    if (k0 + BF_KS < m) gload(k0 + BF_KS);
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (live[b]) {
        const int c = b * 16 + (lane & 15);
        bf8 B[3][NT];
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
          for (int q = 0; q < NT; ++q) B[p][q] = lu[p][q][c][kg];
        p1[b] = bf_products<NT>(A[0], B[0], p1[b]);
        p2[b] = bf_products<NT>(A[1], B[1], p2[b]);
        p3[b] = bf_products<NT>(A[2], B[2], p3[b]);
      }
    __syncthreads();
  }
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int j = j0 + b * 16 + (lane & 15);
    if (j >= n) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t gg = rb * RT_ROWS + wave * 16 + Mfma<float>::row(lane, r);
      if (gg < nrow) Z[(int64_t)j * ldz + gg] = make_float2(p1[b][r] - p2[b][r], p3[b][r] - p1[b][r] - p2[b][r]);
    }
  }
}

int64_t rotate_work_slots(int m, int n, int batch) {
  return ceil_div(m, CX_KS) * ceil_div(n, RC_COLS) * RC_IMG * batch;
}

template <typename R>
void rotate2(const cx_t<R>* X, const cx_t<R>* X2, int64_t ldx, int64_t sx, const double2* U, int ldu, int64_t su, int m,
             int n, int64_t npw, const int* npwk, cx_t<R>* Z, cx_t<R>* Z2, int64_t ldz, int64_t sz, int batch,
             hipStream_t s, int bf16_terms, void* work, int64_t work_slots) {
  DEREK_REQUIRE(m > 0 && n > 0 && batch > 0, "rotate: empty block");
  DEREK_REQUIRE(bf16_terms == 0 || (std::is_same<R, float>::value && bf16_terms >= 1 && bf16_terms <= 3),
                "rotate: bf16 terms must be 0, or 1..3 for complex64 data");
  const int64_t items = ceil_div(npw, RT_ROWS) * ceil_div(n, RT_COLS) * batch;
  DEREK_REQUIRE(items < (int64_t)1 << 31, "rotate: too many workgroups");
  const unsigned two = X2 ? 2 : 1;
  const dim3 grid((unsigned)items, two);
  if constexpr (std::is_same<R, float>::value) {
    // two terms: the 128-row workgroups once there is one per CU (600 -> 300
    // columns of 8 x 161214 rows 10.2 -> 5.3 ms, 48 -> 24 of 64 x 17529 0.248
    // -> 0.183 ms, 48 -> 24 of 40000 18.2 -> 17.6 us; with 125 workgroups, 80 ->
    // 40 of 4 x 4000 rows, 13 against 18 us), or four where the few columns of X
    // hardly pay the split's launch (32 -> 16 of 40000 rows 12.9 against 14.4 us,
    // of 62669 14.6 and 16.2, of 140000 25.8 and 25.9; 16 -> 8 of 140000 21.9 ->
    // 18.2), a buffer for the split U and 32-bit offsets
    const int64_t wide = ceil_div(npw, RC_ROWS) * ceil_div(n, RC_COLS) * batch;
    if (bf16_terms == 2 && wide * two >= (m > 32 ? 256 : 1024) && work && rotate_work_slots(m, n, batch) <= work_slots &&
        (int64_t)m * ldx * 8 < (int64_t)kOob) {
      u4* img = reinterpret_cast<u4*>(work);
      hipLaunchKernelGGL(k_rotate_split, dim3((unsigned)ceil_div(m, CX_KS), (unsigned)ceil_div(n, RC_COLS), batch),
                         dim3(256), 0, s, U, ldu, su, m, n, img);
      hipLaunchKernelGGL(k_rotate_cx, dim3((unsigned)wide, two), dim3(256), 0, s, X, X2, ldx, sx, img, m, n, npw, npwk, Z,
                         Z2, ldz, sz);
    } else if (bf16_terms == 1) {
      hipLaunchKernelGGL(k_rotate_bf16<1>, grid, dim3(256), 0, s, X, X2, ldx, sx, U, ldu, su, m, n, npw, npwk, Z, Z2, ldz,
                         sz);
    } else if (bf16_terms == 2) {
      hipLaunchKernelGGL(k_rotate_bf16<2>, grid, dim3(256), 0, s, X, X2, ldx, sx, U, ldu, su, m, n, npw, npwk, Z, Z2, ldz,
                         sz);
    } else if (bf16_terms == 3) {
      hipLaunchKernelGGL(k_rotate_bf16<3>, grid, dim3(256), 0, s, X, X2, ldx, sx, U, ldu, su, m, n, npw, npwk, Z, Z2, ldz,
                         sz);
    }
  }
  if (bf16_terms == 0)
    hipLaunchKernelGGL(k_rotate<R>, grid, dim3(256), 0, s, X, X2, ldx, sx, U, ldu, su, m, n, npw, npwk, Z, Z2, ldz, sz);
  DEREK_HIP(hipGetLastError());
}

template void overlap<double>(const double2*, int64_t, int64_t, const double2*, int64_t, int64_t, int, int, int64_t,
                              const int*, double2*, int, int64_t, int, double2*, int64_t, bool, hipStream_t, int,
                              int64_t, int, int);
template void overlap<float>(const float2*, int64_t, int64_t, const float2*, int64_t, int64_t, int, int, int64_t,
                             const int*, double2*, int, int64_t, int, double2*, int64_t, bool, hipStream_t, int,
                             int64_t, int, int);
template void rotate2<double>(const double2*, const double2*, int64_t, int64_t, const double2*, int, int64_t, int, int,
                              int64_t, const int*, double2*, double2*, int64_t, int64_t, int, hipStream_t, int, void*,
                              int64_t);
template void rotate2<float>(const float2*, const float2*, int64_t, int64_t, const double2*, int, int64_t, int, int,
                             int64_t, const int*, float2*, float2*, int64_t, int64_t, int, hipStream_t, int, void*,
                             int64_t);

}  // namespace derek
