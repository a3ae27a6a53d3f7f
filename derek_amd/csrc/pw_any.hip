// Two-stage register passes of the pruned FFT pipelines for any length
// n = r1 * r2, 1 <= r2 <= r1 <= 16 (84 of the 91 smooth lengths below 200;
// the lengths with kernels of their own are in pw_fft.hip).
//
// The radices are kernel arguments: every stage branches once, wave-uniformly,
// to the register DFT of its radix (fft.hpp: with_radix), so one kernel serves
// all lengths.  A transform is
//   stage 1, task j < r2:  v_r = in[j + r2 r] (r < r1), DFT_r1 -> slot k r2 + j
//   stage 2, task k < r1:  u_r = slot[k r2 + r] w^(k r), DFT_r2 -> index
//                          k + r1 m in slot k r2 + m
// and both stages write exactly the slots they read, so a single LDS buffer
// and one barrier per stage do, and the tasks of a stage are dealt to however
// many threads the workgroup has.  Forward transforms after an inverse one run
// the stages backwards (decimation in frequency).
//
// Q: the plane waves lie in the outer quarters of every axis (PwBatch::quarter,
// true for a sphere on a grid at least twice as fine as it needs).  The
// inverse transforms then take literal zeros for the digits that cannot hold
// input (this file and pw_fft.hip are compiled without signed zeros, so the
// additions fold away) and the forward ones drop the outputs that nobody
// reads: about a sixth of the arithmetic and half of the first loads and last
// stores, with the same values.  Measured together with the coprime register
// transforms (fft.hpp): the fused y/x pass on 144^3 complex64 2466 -> 2121 us,
// on 108^3 complex128 617 -> 543, on 72^3 complex64 324 -> 299; the x pass of
// 256 bands on 65^3 complex128 393 -> 352 us.
// The z passes bring each stick row once and wait for HBM (70 to 80 % of their
// cycles), so lengths in the code gain nothing over lengths as arguments:
// 72^3 complex64 43 and 47 us (inverse, forward) against 50 and 50 with
// compiled lengths, 144^3 418 and 552 against 428 and 534.
//
// Bound: HBM for the y and z passes, the vector ALU for the x pass in FP64.
// The Stockham kernels these replace (ping-pong LDS, one division per element,
// two or three passes over LDS per stage) took 2340 us for the x pass of 256
// complex128 items of a 65^3 grid.
#include "pw_any.hpp"

namespace derek {

namespace {

constexpr int AL = 16;   // columns of a workgroup of the y and x passes (256 bytes of complex128)
constexpr int AT = 256;  // most threads of a workgroup

// ---------------------------------------------------------------- z passes
// SL sticks per workgroup, stick fastest in LDS: element (slot, stick) at
// slot * pitch + stick.  The pitch is SL where the stick rows are z-major
// (consecutive lanes take consecutive sticks everywhere) and SL + 1 where a
// stick's line is contiguous in memory (consecutive lanes then walk z).
template <typename R, int SL> constexpr size_t any_z_lds(int n, bool zmajor) {
  return sizeof(cx_t<R>) * (size_t)n * (1 + (zmajor ? SL : SL + 1)) + sizeof(int) * (size_t)n;
}

// slot (times the pitch) of index z after the second stage
__device__ __forceinline__ void slot_table(int* slot, TwoStage q, int pitch) {
  for (int z = threadIdx.x; z < q.n; z += AT) slot[z] = ((z % q.r1) * q.r2 + z / q.r1) * pitch;
}

template <int SGN, int SL, bool Q, typename C>
__device__ __forceinline__ void any_z_stages(C* buf, const C* twl, TwoStage q, int pitch) {
  with_radix(q.r1, [&](auto rc) {
    constexpr int R1 = decltype(rc)::value;
    for (int t = threadIdx.x; t < SL * q.r2; t += AT) {
      const int l = t % SL, j = t / SL;
      const int step = q.r2 * pitch;
      C* p = buf + j * pitch + l;
      C v[R1];
#pragma unroll
      for (int r = 0; r < R1; ++r) v[r] = (!Q || SGN < 0 || quarter_has(r, R1)) ? p[r * step] : cmk<C>(0, 0);
      dftR<R1, SGN>(v, (const C*)nullptr, 0);
#pragma unroll
      for (int r = 0; r < R1; ++r) p[r * step] = v[r];
    }
  });
  __syncthreads();
  with_radix(q.r2, [&](auto rc) {
    constexpr int R2 = decltype(rc)::value;
    for (int t = threadIdx.x; t < SL * q.r1; t += AT) {
      const int l = t % SL, k = t / SL;
      C* p = buf + k * R2 * pitch + l;
      C u[R2];
#pragma unroll
      for (int r = 0; r < R2; ++r) u[r] = r ? cmul(p[r * pitch], twid<SGN>(twl, k * r)) : p[0];
      dftR<R2, SGN>(u, (const C*)nullptr, 0);
#pragma unroll
      for (int r = 0; r < R2; ++r)
        if (!Q || SGN > 0 || quarter_has(r, R2)) p[r * pitch] = u[r];
    }
  });
  __syncthreads();
}

// psi[b][perm[p]] -> S
template <typename R, bool ZM, int SL, bool Q>
__global__ __launch_bounds__(AT) void k_any_z_inv(PwBatch B, PwBlock<R> psi, TwoStage q, const cx_t<R>* __restrict__ tw,
                                                  cx_t<R>* __restrict__ S) {
  using C = cx_t<R>;
  constexpr int pitch = ZM ? SL : SL + 1;
  extern __shared__ __align__(16) unsigned char smem[];
  const PwMaps m = B.mt[B.k0 + blockIdx.z];
  const int s0 = blockIdx.x * SL;
  if (s0 >= m.nst) return;
  const int n = q.n, tid = threadIdx.x, band = blockIdx.y;
  C* twl = reinterpret_cast<C*>(smem);
  C* buf = twl + n;
  int* slot = reinterpret_cast<int*>(buf + (size_t)n * pitch);
  const int lines = min(SL, m.nst - s0);
  for (int t = tid; t < n; t += AT) twl[t] = tw[t];
  slot_table(slot, q, pitch);
  // the inputs that stage 1 reads: all, or the digits of the outer quarters
  const int lo = Q ? (q.r1 + 3) / 4 * q.r2 : n, hi = Q ? max(lo, 3 * q.r1 / 4 * q.r2) : n;
  for (int e = tid; e < lo * pitch; e += AT) buf[e] = cmk<C>(0, 0);
  for (int e = hi * pitch + tid; e < n * pitch; e += AT) buf[e] = cmk<C>(0, 0);
  __syncthreads();
  const int p0 = m.st_pw[s0], p1 = m.st_pw[s0 + lines];
  const C* pb = psi.p + blockIdx.z * psi.ks + (int64_t)band * psi.ld;
  for (int p = p0 + tid; p < p1; p += AT) buf[m.pw_z[p] * pitch + (m.pw_st[p] - s0)] = pb[m.perm[p]];
  __syncthreads();
  any_z_stages<+1, SL, Q>(buf, twl, q, pitch);
  const int64_t item = (int64_t)blockIdx.z * B.nbb + band;
  if constexpr (ZM) {
    const int l = tid % SL;
    C* dst = S + item * B.nst_cap * n + s0 + l;
    if (l < lines)
      for (int z = tid / SL; z < n; z += AT / SL) nt_store(dst + (int64_t)z * B.nst_cap, buf[slot[z] + l]);
  } else {
    C* dst = S + (item * B.nst_cap + s0) * n;
    for (int l = tid / 64; l < lines; l += AT / 64)
      for (int z = tid % 64; z < n; z += 64) nt_store(dst + (int64_t)l * n + z, buf[slot[z] + l]);
  }
}

// hpsi[b][perm[p]] = (z FFT of the stick)[pw_z[p]] + kin[perm[p]] psi[b][perm[p]]
template <typename R, bool ZM, int SL, bool Q>
__global__ __launch_bounds__(AT) void k_any_z_fwd(PwBatch B, const cx_t<R>* __restrict__ S, TwoStage q,
                                                  const cx_t<R>* __restrict__ tw, PwBlock<R> psi, PwBlock<R> hpsi) {
  using C = cx_t<R>;
  constexpr int pitch = ZM ? SL : SL + 1;
  extern __shared__ __align__(16) unsigned char smem[];
  const PwMaps m = B.mt[B.k0 + blockIdx.z];
  const int s0 = blockIdx.x * SL;
  if (s0 >= m.nst) return;
  const int n = q.n, tid = threadIdx.x, band = blockIdx.y;
  C* twl = reinterpret_cast<C*>(smem);
  C* buf = twl + n;
  int* slot = reinterpret_cast<int*>(buf + (size_t)n * pitch);
  const int lines = min(SL, m.nst - s0);
  for (int t = tid; t < n; t += AT) twl[t] = tw[t];
  slot_table(slot, q, pitch);
  const int64_t item = (int64_t)blockIdx.z * B.nbb + band;
  if constexpr (ZM) {
    const int l = tid % SL;
    const C* src = S + item * B.nst_cap * n + s0 + l;
    for (int z = tid / SL; z < n; z += AT / SL)
      buf[z * pitch + l] = l < lines ? nt_load(src + (int64_t)z * B.nst_cap) : cmk<C>(0, 0);
  } else {
    const C* src = S + (item * B.nst_cap + s0) * n;
    for (int l = tid / 64; l < SL; l += AT / 64)
      for (int z = tid % 64; z < n; z += 64)
        buf[z * pitch + l] = l < lines ? nt_load(src + (int64_t)l * n + z) : cmk<C>(0, 0);
  }
  __syncthreads();
  any_z_stages<-1, SL, Q>(buf, twl, q, pitch);
  const int p0 = m.st_pw[s0], p1 = m.st_pw[s0 + lines];
  const C* pb = psi.p + blockIdx.z * psi.ks + (int64_t)band * psi.ld;
  C* hb = hpsi.p + blockIdx.z * hpsi.ks + (int64_t)band * hpsi.ld;
  for (int p = p0 + tid; p < p1; p += AT) {
    const int g = m.perm[p];
    const C v = buf[slot[m.pw_z[p]] + (m.pw_st[p] - s0)];
    const C x = pb[g];
    const R t = (R)m.kin[g];
    hb[g] = cmk<C>(v.x + t * x.x, v.y + t * x.y);
  }
}

// ---------------------------------------------------------------- column passes
// AL neighbouring columns per workgroup, element (slot, column) at
// slot * AL + column.  Rows outside the sphere and lanes past the last column
// take the out-of-range buffer offset (loads give zero, stores are dropped).
template <typename C>
__device__ __forceinline__ void column_tables(C* twl, uint32_t* row, const C* __restrict__ tw, int n) {
  for (int t = threadIdx.x; t < n; t += blockDim.x) {
    twl[t] = tw[t];
    row[t] = kOob;
  }
}

// stage 1 of an inverse or forward transform: rows from a buffer resource
// (row[i]: byte offset of index i) into slots
template <int SGN, bool Q, typename C, int CP, typename Rs>
__device__ __forceinline__ void column_in(C* buf, const uint32_t* row, TwoStage q, const Rs& rs, int cols) {
  with_radix(q.r1, [&](auto rc) {
    constexpr int R1 = decltype(rc)::value;
    for (int t = threadIdx.x; t < AL * q.r2; t += blockDim.x) {
      const int l = t % AL, j = t / AL;
      const uint32_t lo = l < cols ? (uint32_t)l * (uint32_t)sizeof(C) : kOob;
      C v[R1];
#pragma unroll
      for (int r = 0; r < R1; ++r)
        v[r] = (!Q || quarter_has(r, R1)) ? buf_ld<C, CP>(rs, row[j + q.r2 * r] + lo) : cmk<C>(0, 0);
      dftR<R1, SGN>(v, (const C*)nullptr, 0);
      C* p = buf + j * AL + l;
#pragma unroll
      for (int r = 0; r < R1; ++r) p[r * q.r2 * AL] = v[r];
    }
  });
}

// stage 2: twiddles and DFT_r2 of task (k, column); op(k, l, u) takes the
// values of the indexes k + r1 m
template <int SGN, typename C, typename F>
__device__ __forceinline__ void column_out(const C* buf, const C* twl, TwoStage q, F&& op) {
  with_radix(q.r2, [&](auto rc) {
    constexpr int R2 = decltype(rc)::value;
    for (int t = threadIdx.x; t < AL * q.r1; t += blockDim.x) {
      const int l = t % AL, k = t / AL;
      const C* p = buf + k * R2 * AL + l;
      C u[R2];
#pragma unroll
      for (int r = 0; r < R2; ++r) u[r] = r ? cmul(p[r * AL], twid<SGN>(twl, k * r)) : p[0];
      dftR<R2, SGN>(u, (const C*)nullptr, 0);
      op(rc, k, l, u);
    }
  });
}

// y pass: SGN +1 sticks of plane a -> y rows of P, -1 y rows -> sticks
template <typename R, int SGN, bool Q>
__global__ __launch_bounds__(AT) void k_any_y(PwBatch B, cx_t<R>* __restrict__ S, cx_t<R>* __restrict__ P, int nz,
                                              int ztiles, int bpw, TwoStage q, const cx_t<R>* __restrict__ tw) {
  using C = cx_t<R>;
  extern __shared__ __align__(16) unsigned char smem[];
  const PwMaps m = B.mt[B.k0 + blockIdx.z];
  const int a = blockIdx.x / ztiles;
  if (a >= m.nax) return;
  const int n = q.n, tid = threadIdx.x;
  C* twl = reinterpret_cast<C*>(smem);
  C* buf = twl + n;
  uint32_t* st = reinterpret_cast<uint32_t*>(buf + (size_t)n * AL);  // stick lines of the plane
  uint32_t* yr = st + n;                                             // rows of the plane
  const int z0 = (blockIdx.x - a * ztiles) * AL, cols = min(AL, nz - z0);
  column_tables(twl, st, tw, n);
  for (int y = tid; y < n; y += blockDim.x) yr[y] = (uint32_t)(y * nz) * (uint32_t)sizeof(C);
  __syncthreads();
  for (int j = m.pl_st[a] + tid; j < m.pl_st[a + 1]; j += blockDim.x)
    st[m.st_y[j]] = (uint32_t)(j * nz) * (uint32_t)sizeof(C);
  __syncthreads();
  const uint32_t st_bytes = (uint32_t)(((int64_t)B.nst_cap * nz - z0) * (int64_t)sizeof(C));
  const uint32_t pl_bytes = (uint32_t)(((int64_t)n * nz - z0) * (int64_t)sizeof(C));
  const uint32_t* in = SGN > 0 ? st : yr;
  const uint32_t* out = SGN > 0 ? yr : st;
  const int bb0 = blockIdx.y * bpw, bb1 = min(B.nbb, bb0 + bpw);
  for (int band = bb0; band < bb1; ++band) {
    const int64_t item = (int64_t)blockIdx.z * B.nbb + band;
    const auto rst = buf_rsrc(S + item * B.nst_cap * nz + z0, st_bytes);
    const auto rpl = buf_rsrc(P + (item * B.nax_cap + a) * n * nz + z0, pl_bytes);
    column_in<SGN, Q && (SGN > 0), C, 0>(buf, in, q, SGN > 0 ? rst : rpl, cols);
    __syncthreads();
    const auto ro = SGN > 0 ? rpl : rst;
    column_out<SGN>(buf, twl, q, [&](auto rc, int k, int l, const C* u) {
      constexpr int R2 = decltype(rc)::value;
      const uint32_t lo = l < cols ? (uint32_t)l * (uint32_t)sizeof(C) : kOob;
#pragma unroll
      for (int i = 0; i < R2; ++i)
        if (!Q || SGN > 0 || quarter_has(i, R2)) buf_st<C>(ro, out[k + q.r1 * i] + lo, u[i]);
    });
    __syncthreads();
  }
}

// x pass: inverse of the active rows, * V * vscale, forward, active rows back
template <typename R, bool Q>
__global__ __launch_bounds__(AT) void k_any_x_vmul(PwBatch B, cx_t<R>* __restrict__ P, int64_t nyz, int bpw, TwoStage q,
                                                   const cx_t<R>* __restrict__ tw, const R* __restrict__ vloc,
                                                   R vscale) {
  using C = cx_t<R>;
  extern __shared__ __align__(16) unsigned char smem[];
  const PwMaps m = B.mt[B.k0 + blockIdx.z];
  const int n = q.n, tid = threadIdx.x;
  C* twl = reinterpret_cast<C*>(smem);
  C* buf = twl + n;
  R* vt = reinterpret_cast<R*>(buf + (size_t)n * AL);  // V * vscale in slot order
  uint32_t* row = reinterpret_cast<uint32_t*>(vt + (size_t)n * AL);
  const int64_t c0 = (int64_t)blockIdx.x * AL;
  const int cols = (int)min((int64_t)AL, nyz - c0);
  column_tables(twl, row, tw, n);
  for (int e = tid; e < n * AL; e += blockDim.x) {
    const int x = e / AL, l = e % AL;
    vt[((x % q.r1) * q.r2 + x / q.r1) * AL + l] = l < cols ? vloc[(int64_t)x * nyz + c0 + l] * vscale : (R)0;
  }
  __syncthreads();
  for (int a = tid; a < m.nax; a += blockDim.x) row[m.ax_x[a]] = (uint32_t)a * (uint32_t)nyz * (uint32_t)sizeof(C);
  __syncthreads();
  const uint32_t bytes = (uint32_t)((B.nax_cap * nyz - c0) * (int64_t)sizeof(C));
  const int bb0 = blockIdx.y * bpw, bb1 = min(B.nbb, bb0 + bpw);
  for (int band = bb0; band < bb1; ++band) {
    const auto rs = buf_rsrc(P + ((int64_t)blockIdx.z * B.nbb + band) * B.nax_cap * nyz + c0, bytes);
    column_in<+1, Q, C, kNt>(buf, row, q, rs, cols);
    __syncthreads();
    column_out<+1>(buf, twl, q, [&](auto rc, int k, int l, C* u) {
      constexpr int R2 = decltype(rc)::value;
      const R* v = vt + k * R2 * AL + l;
      C* p = buf + k * R2 * AL + l;
#pragma unroll
      for (int i = 0; i < R2; ++i) u[i] = cscale(u[i], v[i * AL]);
      dftR<R2, -1>(u, (const C*)nullptr, 0);
#pragma unroll
      for (int i = 0; i < R2; ++i) p[i * AL] = i ? cmul(u[i], twl[k * i]) : u[i];
    });
    __syncthreads();
    // last stage of the forward transform: index j + r2 k of task j
    with_radix(q.r1, [&](auto rc) {
      constexpr int R1 = decltype(rc)::value;
      for (int t = tid; t < AL * q.r2; t += blockDim.x) {
        const int l = t % AL, j = t / AL;
        const uint32_t lo = l < cols ? (uint32_t)l * (uint32_t)sizeof(C) : kOob;
        const C* p = buf + j * AL + l;
        C v[R1];
#pragma unroll
        for (int r = 0; r < R1; ++r) v[r] = p[r * q.r2 * AL];
        dftR<R1, -1>(v, (const C*)nullptr, 0);
#pragma unroll
        for (int r = 0; r < R1; ++r)
          if (!Q || quarter_has(r, R1)) buf_st<C, kNt>(rs, row[j + q.r2 * r] + lo, v[r]);
      }
    });
    __syncthreads();
  }
}

// x pass for the density: rho[x*nyz + c] = keep*rho + sum_items occ |inverse x|^2
template <typename R, bool Q>
__global__ __launch_bounds__(AT) void k_any_x_density(PwBatch B, const cx_t<R>* __restrict__ P, int64_t nyz, TwoStage q,
                                                      const cx_t<R>* __restrict__ tw, const double* __restrict__ occ,
                                                      int occ_ks, double* __restrict__ rho, int keep) {
  using C = cx_t<R>;
  extern __shared__ __align__(16) unsigned char smem[];
  const int n = q.n, tid = threadIdx.x;
  C* twl = reinterpret_cast<C*>(smem);
  C* buf = twl + n;
  double* acc = reinterpret_cast<double*>(buf + (size_t)n * AL);  // in slot order, one owner per element
  uint32_t* row = reinterpret_cast<uint32_t*>(acc + (size_t)n * AL);
  const int64_t c0 = (int64_t)blockIdx.x * AL;
  const int cols = (int)min((int64_t)AL, nyz - c0);
  for (int e = tid; e < n * AL; e += blockDim.x) acc[e] = 0.0;
  const uint32_t bytes = (uint32_t)((B.nax_cap * nyz - c0) * (int64_t)sizeof(C));
  for (int kz = 0; kz < B.nkc; ++kz) {
    const PwMaps m = B.mt[B.k0 + kz];
    __syncthreads();
    column_tables(twl, row, tw, n);
    __syncthreads();
    for (int a = tid; a < m.nax; a += blockDim.x) row[m.ax_x[a]] = (uint32_t)a * (uint32_t)nyz * (uint32_t)sizeof(C);
    __syncthreads();
    for (int band = 0; band < B.nbb; ++band) {
      const double w = occ[(int64_t)kz * occ_ks + band];
      if (w == 0.0) continue;  // uniform over the workgroup
      const auto rs = buf_rsrc(P + ((int64_t)kz * B.nbb + band) * B.nax_cap * nyz + c0, bytes);
      column_in<+1, Q, C, 0>(buf, row, q, rs, cols);
      __syncthreads();
      column_out<+1>(buf, twl, q, [&](auto rc, int k, int l, const C* u) {
        constexpr int R2 = decltype(rc)::value;
        double* p = acc + k * R2 * AL + l;
#pragma unroll
        for (int i = 0; i < R2; ++i) {
          const double re = (double)u[i].x, im = (double)u[i].y;
          p[i * AL] += w * (re * re + im * im);
        }
      });
      __syncthreads();
    }
  }
  __syncthreads();
  for (int e = tid; e < n * AL; e += blockDim.x) {
    const int x = e / AL, l = e % AL;
    if (l < cols) {
      double* r = rho + (int64_t)x * nyz + c0 + l;
      *r = (keep ? *r : 0.0) + acc[((x % q.r1) * q.r2 + x / q.r1) * AL + l];
    }
  }
}

// ---------------------------------------------------------------- launchers
// Threads of a column pass: the multiple of 64 with the least lane time over
// the stages (AL r2 tasks of radix r1 and AL r1 tasks of radix r2; an odd
// prime costs about twice a composite of its size), the larger on a tie.
int column_threads(TwoStage q) {
  auto cost = [](int r) {
    double c = 0.0;
    for (int p : {2, 3, 5, 7, 11, 13})
      for (int m = r; m % p == 0; m /= p) c += p < 7 ? (p + 1.0) : 1.5 * p;
    return r * (c + 2.0);
  };
  int best = 64;
  double least = 1e300;
  for (int nt = 64; nt <= AT; nt += 64) {
    const double t = nt * (ceil_div(AL * q.r2, nt) * cost(q.r1) + ceil_div(AL * q.r1, nt) * cost(q.r2));
    if (t <= least * 1.0001) {
      least = t;
      best = nt;
    }
  }
  return best;
}

constexpr size_t kLdsMax = 160 * 1024;

template <typename K> void allow_lds_any(K kern, size_t bytes) {
  if (bytes > 65536) allow_dynamic_lds(reinterpret_cast<const void*>(kern), bytes);
}

template <typename R, bool ZM, int SL>
bool z_inv_sl(const PwBatch& B, PwBlock<R> psi, const Axis<R>& az, cx_t<R>* S, TwoStage q, hipStream_t s) {
  const size_t lds = any_z_lds<R, SL>(q.n, ZM);
  if (lds > kLdsMax) return false;
  auto kern = B.quarter ? k_any_z_inv<R, ZM, SL, true> : k_any_z_inv<R, ZM, SL, false>;
  allow_lds_any(kern, lds);
  hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(B.nst_cap, SL), B.nbb, B.nkc), dim3(AT), lds, s, B, psi, q, az.tw, S);
  return true;
}

template <typename R, bool ZM, int SL>
bool z_fwd_sl(const PwBatch& B, const cx_t<R>* S, const Axis<R>& az, PwBlock<R> psi, PwBlock<R> hpsi, TwoStage q,
              hipStream_t s) {
  const size_t lds = any_z_lds<R, SL>(q.n, ZM);
  if (lds > kLdsMax) return false;
  auto kern = B.quarter ? k_any_z_fwd<R, ZM, SL, true> : k_any_z_fwd<R, ZM, SL, false>;
  allow_lds_any(kern, lds);
  hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(B.nst_cap, SL), B.nbb, B.nkc), dim3(AT), lds, s, B, S, q, az.tw, psi,
                     hpsi);
  return true;
}

template <typename R> int stick_block(const PwBatch& B) { return B.zsl ? B.zsl : (sizeof(R) == 8 ? 16 : 32); }

}  // namespace

template <typename R>
bool any_z_inv(const PwBatch& B, PwBlock<R> psi, const Axis<R>& az, cx_t<R>* S, bool zmajor, hipStream_t s) {
  const TwoStage q = two_stage(az.n);
  if (!q.r1) return false;
  if (stick_block<R>(B) == 32)
    return zmajor ? z_inv_sl<R, true, 32>(B, psi, az, S, q, s) : z_inv_sl<R, false, 32>(B, psi, az, S, q, s);
  return zmajor ? z_inv_sl<R, true, 16>(B, psi, az, S, q, s) : z_inv_sl<R, false, 16>(B, psi, az, S, q, s);
}

template <typename R>
bool any_z_fwd(const PwBatch& B, const cx_t<R>* S, const Axis<R>& az, PwBlock<R> psi, PwBlock<R> hpsi, bool zmajor,
               hipStream_t s) {
  const TwoStage q = two_stage(az.n);
  if (!q.r1) return false;
  if (stick_block<R>(B) == 32)
    return zmajor ? z_fwd_sl<R, true, 32>(B, S, az, psi, hpsi, q, s) : z_fwd_sl<R, false, 32>(B, S, az, psi, hpsi, q, s);
  return zmajor ? z_fwd_sl<R, true, 16>(B, S, az, psi, hpsi, q, s) : z_fwd_sl<R, false, 16>(B, S, az, psi, hpsi, q, s);
}

template <typename R>
bool any_y(const PwBatch& B, cx_t<R>* S, cx_t<R>* P, const Axis<R>& ay, int nz, int sign, int bands_per_wg,
           hipStream_t s) {
  const TwoStage q = two_stage(ay.n);
  const size_t lds = sizeof(cx_t<R>) * (size_t)q.n * (AL + 1) + 2 * sizeof(uint32_t) * (size_t)q.n;
  if (!q.r1 || lds > kLdsMax) return false;
  const int ztiles = (int)ceil_div(nz, AL);
  dim3 grid((unsigned)(B.nax_cap * ztiles), (unsigned)ceil_div(B.nbb, bands_per_wg), B.nkc);
  auto kern = sign > 0 ? (B.quarter ? k_any_y<R, +1, true> : k_any_y<R, +1, false>)
                       : (B.quarter ? k_any_y<R, -1, true> : k_any_y<R, -1, false>);
  allow_lds_any(kern, lds);
  hipLaunchKernelGGL(kern, grid, dim3(column_threads(q)), lds, s, B, S, P, nz, ztiles, bands_per_wg, q, ay.tw);
  return true;
}

template <typename R>
bool any_x_vmul(const PwBatch& B, cx_t<R>* P, const Axis<R>& ax, int64_t nyz, const R* vloc, R vscale,
                int bands_per_wg, hipStream_t s) {
  const TwoStage q = two_stage(ax.n);
  const size_t lds =
      (sizeof(cx_t<R>) * (AL + 1) + sizeof(R) * AL + sizeof(uint32_t)) * (size_t)q.n;
  if (!q.r1 || lds > kLdsMax) return false;
  dim3 grid((unsigned)ceil_div(nyz, AL), (unsigned)ceil_div(B.nbb, bands_per_wg), B.nkc);
  auto kern = B.quarter ? k_any_x_vmul<R, true> : k_any_x_vmul<R, false>;
  allow_lds_any(kern, lds);
  hipLaunchKernelGGL(kern, grid, dim3(column_threads(q)), lds, s, B, P, nyz, bands_per_wg, q, ax.tw, vloc, vscale);
  return true;
}

template <typename R>
bool any_x_density(const PwBatch& B, const cx_t<R>* P, const Axis<R>& ax, int64_t nyz, const double* occ, int occ_ks,
                   double* rho, int keep, hipStream_t s) {
  const TwoStage q = two_stage(ax.n);
  const size_t lds = (sizeof(cx_t<R>) * (AL + 1) + sizeof(double) * AL + sizeof(uint32_t)) * (size_t)q.n;
  if (!q.r1 || lds > kLdsMax) return false;
  auto kern = B.quarter ? k_any_x_density<R, true> : k_any_x_density<R, false>;
  allow_lds_any(kern, lds);
  hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(nyz, AL)), dim3(column_threads(q)), lds, s, B, P, nyz, q, ax.tw, occ,
                     occ_ks, rho, keep);
  return true;
}

#define INST(R)                                                                                                   \
  template bool any_z_inv<R>(const PwBatch&, PwBlock<R>, const Axis<R>&, cx_t<R>*, bool, hipStream_t);            \
  template bool any_z_fwd<R>(const PwBatch&, const cx_t<R>*, const Axis<R>&, PwBlock<R>, PwBlock<R>, bool,        \
                             hipStream_t);                                                                        \
  template bool any_y<R>(const PwBatch&, cx_t<R>*, cx_t<R>*, const Axis<R>&, int, int, int, hipStream_t);         \
  template bool any_x_vmul<R>(const PwBatch&, cx_t<R>*, const Axis<R>&, int64_t, const R*, R, int, hipStream_t);  \
  template bool any_x_density<R>(const PwBatch&, const cx_t<R>*, const Axis<R>&, int64_t, const double*, int,     \
                                 double*, int, hipStream_t);
INST(double)
INST(float)
#undef INST

}  // namespace derek
