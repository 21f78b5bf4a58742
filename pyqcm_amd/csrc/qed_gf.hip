// Green-function representations and the lattice k-sums on the device.
//
//  * Lehmann form: G_ab(z) = sum_m Q_am Q_bm / (z - e_m), batched over frequencies
//    (the reference's VDVH contraction, src_util/VDVH_kernel.cpp:28-48).
//  * Continued fractions evaluated bottom-up (src_ed/continued_fraction.cpp:52-57).
//  * CPT / VCA / CDMFT k-sums: for every (w, k) the n x n complex matrix
//    M = Gc(w)^-1 - V(k) is inverted (G_cpt = M^-1, src_qcm/CPT.cpp:76-86) or factorized
//    (log|det(V Gc - 1)| = log|det Gc| + log|det M|, src_qcm/lattice_model_instance.cpp:624-643).
//    A few lanes hold one matrix, some rows each; 8 to 64 matrices share a wave.
#include <cmath>
#include <complex>
#include <cstring>
#include <memory>
#include <mutex>
#include <type_traits>
#include <vector>

#include "../../include/qed.h"
#include "qed_common.hpp"
#include "qed_hostcopy.hpp"
#include "qed_linalg.hpp"

namespace qed {

namespace {

struct cplx {
  double re, im;
};
__device__ __forceinline__ cplx cmul(cplx a, cplx b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ cplx cadd(cplx a, cplx b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ cplx csub(cplx a, cplx b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ cplx cinv(cplx a) {
  double d = a.re * a.re + a.im * a.im;
  return {a.re / d, -a.im / d};
}
__device__ __forceinline__ double cabs2(cplx a) { return a.re * a.re + a.im * a.im; }

// ---- Lehmann G(z) --------------------------------------------------------------------
// one workgroup per frequency; thread t accumulates element (b, a) = (t % L, t / L)
__global__ __launch_bounds__(256) void k_qmatrix_gf(int L, int M, const double* __restrict__ e,
                                                    const double* __restrict__ Q,
                                                    const double* __restrict__ z,
                                                    double* __restrict__ G) {
  __shared__ double ur[256], ui[256];
  __shared__ double qs[256 * 16];
  const int iz = blockIdx.x;
  const double zr = z[2 * iz], zi = z[2 * iz + 1];
  const int t = threadIdx.x;
  const int b = t % L, a = t / L;
  const bool act = t < L * L;
  double gr = 0.0, gi = 0.0;
  for (int m0 = 0; m0 < M; m0 += 256) {
    const int mc = min(256, M - m0);
    __syncthreads();
    if (t < mc) {
      double dr = zr - e[m0 + t], di = zi;
      double d = dr * dr + di * di;
      ur[t] = dr / d;
      ui[t] = -di / d;
    }
    for (int i = t; i < mc * L && L <= 16; i += 256) qs[i] = Q[(size_t)m0 * L + i];
    __syncthreads();
    if (act) {
      for (int m = 0; m < mc; ++m) {
        double w = qs[m * L + a] * qs[m * L + b];
        gr += w * ur[m];
        gi += w * ui[m];
      }
    }
  }
  if (act) {
    G[((size_t)iz * L * L + (size_t)b + (size_t)a * L) * 2] += gr;
    G[((size_t)iz * L * L + (size_t)b + (size_t)a * L) * 2 + 1] += gi;
  }
}

__global__ void k_cf_eval(int n, const int* __restrict__ off, const int* __restrict__ depth,
                          const double* __restrict__ a, const double* __restrict__ b, int nz,
                          const double* __restrict__ z, double* __restrict__ out) {
  int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= n * nz) return;
  int f = id % n, iz = id / n;
  cplx zz{z[2 * iz], z[2 * iz + 1]};
  cplx G{0.0, 0.0};
  const double* aa = a + off[f];
  const double* bb = b + off[f];
  for (int i = depth[f] - 1; i >= 0; --i) {
    cplx den = csub(cplx{zz.re - aa[i], zz.im}, G);
    cplx inv = cinv(den);
    G = {bb[i] * inv.re, bb[i] * inv.im};
  }
  out[2 * (size_t)id] = G.re;
  out[2 * (size_t)id + 1] = G.im;
}

// ---- batched small complex matrices ---------------------------------------------------
//
// An n x n complex matrix (n <= 16, padded to N with an identity block) is held by LN
// lanes, R = N / LN rows in the registers of each: row i = q + LN s lives in lane q, slot s.
// Gauss-Jordan with partial pivoting, rows never moved: at step k the unused row with the
// largest |.|^2 in column k is the pivot; its lane writes it to LDS, every lane of the group
// reads it back and eliminates its own rows.
//
// An update is a product rounded once and then subtracted, six operations per element. Both
// terms of the product added to the accumulator in turn take four, but round twice at the
// accumulator's size: the error of an inverse is 1.09 to 1.10 times as large (n = 2 to 16,
// against long double; 4.6 ms instead of 6.0 for the map below). Scaling the pivot row
// or the row's factor by the pivot's inverse is the same for wide matrices; below 9 the
// scaled factor is 0.2 to 0.8% worse in an inverse, and costs no less (ROW).
//
// What bounds it: the 4 n^3 FP64 multiply-adds of the inversion (1.5 ms for the 8.4 million
// 12 x 12 matrices of a 128^2 k x 512 w map at 78.6 TFLOP/s) and the LDS broadcast of the
// pivot row, n 16-byte reads per step and wave. Few lanes with several rows each share one
// broadcast among more matrices: 4 lanes x 3 rows put 16 matrices in a wave, against 5 when
// every lane held one column and exchanged it by lane shuffles (n complex shuffles per step
// and 8 n selects per row exchange; that form took 23.8 ms for the map above, this one
// 6.0 ms, 19 TFLOP/s of 8 n^3 flops each). Small sums (4 x 4, 32^2 k x 20 w) are bound by their
// four launches: 98 us with 16 matrices in turn per group and 80 waves, 5.1 us with one.

struct KsumArgs {
  int n, nw, nk;        // nk: k points of this launch (k0: their first index of nk_all)
  int k0, nk_all;
  int chunk;            // matrices per group, one after the other
  int nchunk;           // chunks per k block (modes 0, 1) or per frequency (modes 2, 3)
  int part0, parts;     // first partial of this launch, partials per frequency (modes 2, 3)
  const double* ginv;   // nw x N x N complex (column-major per matrix): Gc(w)^-1
  const double* vk;     // nk x N x N complex: V(k)
  double* out;
  double* part;
};

__device__ __forceinline__ uint32_t larger(uint32_t v, uint32_t w) { return v > w ? v : w; }

// the maximum of v over the LN lanes of a group (LN = 1, 2, 4, 8; aligned groups)
template <int LN>
__device__ __forceinline__ uint32_t group_max(uint32_t v) {
  if constexpr (LN >= 2)  // quad_perm [1,0,3,2]
    v = larger(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true));
  if constexpr (LN >= 4)  // quad_perm [2,3,0,1]
    v = larger(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true));
  if constexpr (LN >= 8)  // row_half_mirror: lane i of eight <-> 7 - i
    v = larger(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true));
  return v;
}

__device__ __forceinline__ uint32_t mag_bits(cplx v) {  // monotone in |v|^2
  return (uint32_t)((uint64_t)__double_as_longlong(cabs2(v)) >> 32);
}

// The same for |v|^2 beyond the range of a double: its exponent in 13 bits, 14 of its mantissa
__device__ __forceinline__ uint32_t mag_bits_wide(cplx v) {
  const int e = __builtin_amdgcn_frexp_exp(fmax(fabs(v.re), fabs(v.im)));
  const double c2 = cabs2(cplx{ldexp(v.re, -e), ldexp(v.im, -e)});
  if (c2 == 0.0) return 0;
  const uint32_t mant = (uint32_t)((uint64_t)__double_as_longlong(__builtin_amdgcn_frexp_mant(c2)) >> 32) & 0xfffffu;
  return (uint32_t)(2 * e + __builtin_amdgcn_frexp_exp(c2) + 4096) << 19 | mant >> 6 << 5;
}

// a b with the product of the second terms rounded first
__device__ __forceinline__ cplx cmul_fma(cplx a, cplx b) {
  return {fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re)};
}

// log|det| as a product of |pivot|^2 kept in (0, 1) and a power of two
struct LogDet {
  double m = 1.0;
  int e = 0;
  __device__ __forceinline__ void mul(double c2) {
    const double p = m * __builtin_amdgcn_frexp_mant(c2);
    e += __builtin_amdgcn_frexp_exp(c2) + __builtin_amdgcn_frexp_exp(p);
    m = __builtin_amdgcn_frexp_mant(p);
  }
  __device__ __forceinline__ double value() const { return 0.5 * (log(m) + (double)e * M_LN2); }
};

// One elimination of the group's matrix. INV: the inverse in place, C = (P A)^-1 with the
// row that was the pivot of step k holding C[k][:], so that A^-1[k][p_j] = C[k][j]; the
// pivot rows p_j are the nibbles of perm and step[s] is the k of this lane's row s.
// Otherwise the rows below only (the determinant). buf: N double2 of LDS for the group.
// WIDE: pivots whose square leaves the range of a double (one inversion per frequency takes
// it, as an inverse on the host would; the sums over k do not).
template <int N, int LN, bool INV, bool WIDE = false>
__device__ __forceinline__ void eliminate(cplx (&a)[N / LN][N], int q, double2* buf, uint64_t& perm,
                                          int (&step)[N / LN], LogDet& ld, bool& zero) {
  constexpr int R = N / LN;
  constexpr bool ROW = N <= (INV ? 8 : 2);
  perm = 0;
#pragma unroll
  for (int s = 0; s < R; ++s) step[s] = -1;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    uint32_t key = 0;
#pragma unroll
    for (int s = 0; s < R; ++s) {
      const uint32_t mag = WIDE ? mag_bits_wide(a[s][k]) : mag_bits(a[s][k]);
      const uint32_t m = (mag & ~31u) | 16u | (uint32_t)(q + LN * s);
      key = larger(key, step[s] < 0 ? m : 0u);
    }
    key = group_max<LN>(key);
    const int p = (int)(key & 15u);
    perm |= (uint64_t)p << (4 * k);
#pragma unroll
    for (int s = 0; s < R; ++s) {
      if (p == q + LN * s) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
          if (!INV && j < k) continue;
          buf[j] = make_double2(a[s][j].re, a[s][j].im);
          a[s][j] = {0.0, 0.0};
        }
        step[s] = k;
      }
    }
    // the reads below see the pivot lane's writes: LDS accesses of a wave complete in
    // order, the fence keeps the compiler from reusing values of an earlier step
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    cplx rp[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (!INV && j < k) continue;
      const double2 t = buf[j];
      rp[j] = {t.x, t.y};
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    cplx pv = rp[k];
    int pe = 0;
    if constexpr (WIDE) {
      pe = __builtin_amdgcn_frexp_exp(fmax(fabs(pv.re), fabs(pv.im)));
      pv = {ldexp(pv.re, -pe), ldexp(pv.im, -pe)};
    }
    const double c2 = cabs2(pv);
    if (!INV) ld.mul(c2), ld.e += 2 * pe;
    else zero |= pv.re == 0.0 && pv.im == 0.0;
    cplx dinv{pv.re / c2, -pv.im / c2};
    if constexpr (WIDE) dinv = {ldexp(dinv.re, -pe), ldexp(dinv.im, -pe)};
    if constexpr (ROW) {
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (j != k && (INV || j > k)) rp[j] = cmul_fma(rp[j], dinv);
    }
#pragma unroll
    for (int s = 0; s < R; ++s) {
      cplx f = ROW ? a[s][k] : cmul_fma(a[s][k], dinv);
      if constexpr (INV) {  // the pivot row (cleared above) becomes the scaled row
        const cplx own = ROW ? cplx{-1.0, 0.0} : cplx{-dinv.re, -dinv.im};
        if (p == q + LN * s) f = own;
        const cplx c = ROW ? cmul_fma(f, dinv) : f;
        a[s][k] = {-c.re, -c.im};
      }
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (j != k && (INV || j > k)) a[s][j] = csub(a[s][j], cmul_fma(f, rp[j]));
    }
  }
}

// lanes per matrix for each padded dimension
template <int N>
constexpr int lanes_of() {
  return N == 16 ? 8 : N >= 4 ? 4 : N;
}

// V(k) = V0 + sum_t Vt e^(2 pi i k.n_t), padded to N x N with zeros; one block per 8 k points
template <int N>
__global__ __launch_bounds__(256) void k_vk(int n, int nterm, int nk, const double* __restrict__ V0,
                                            const double* __restrict__ Vt, const double* __restrict__ nv,
                                            const double* __restrict__ kk, double* __restrict__ vk) {
  constexpr int KB = 8, TB = 32;
  __shared__ double2 ph[KB][TB];
  const int kb = blockIdx.x * KB;
  constexpr int E = (KB * N * N + 255) / 256;
  cplx acc[E];
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int e = (threadIdx.x + 256 * u) % (N * N), i = e % N, j = e / N;
    acc[u] = {0.0, 0.0};
    if (i < n && j < n) acc[u] = {V0[2 * (i + j * n)], V0[2 * (i + j * n) + 1]};
  }
  for (int t0 = 0; t0 < nterm; t0 += TB) {
    const int tc = min(TB, nterm - t0);
    __syncthreads();
    for (int u = threadIdx.x; u < KB * TB; u += 256) {
      const int t = u % TB, kq = min(kb + u / TB, nk - 1);
      if (t < tc) {
        const double* v = nv + 3 * (t0 + t);
        double s, c;
        const double* k3 = kk + 3 * (size_t)kq;
        sincospi(2.0 * (k3[0] * v[0] + k3[1] * v[1] + k3[2] * v[2]), &s, &c);
        ph[u / TB][t] = make_double2(c, s);
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < E; ++u) {
      const int id = threadIdx.x + 256 * u;
      const int e = id % (N * N), i = e % N, j = e / N, kq = id / (N * N);
      if (kq >= KB || i >= n || j >= n) continue;
      for (int t = 0; t < tc; ++t) {
        const double* m = Vt + 2 * ((size_t)(t0 + t) * n * n + i + (size_t)j * n);
        const double2 p = ph[kq][t];
        acc[u] = cadd(acc[u], cmul(cplx{m[0], m[1]}, cplx{p.x, p.y}));
      }
    }
  }
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int id = threadIdx.x + 256 * u;
    const int kq = id / (N * N);
    if (kq >= KB || kb + kq >= nk) continue;
    reinterpret_cast<double2*>(vk)[(size_t)(kb + kq) * N * N + id % (N * N)] = make_double2(acc[u].re, acc[u].im);
  }
}

// Gc(w)^-1 padded with an identity block, log|det Gc(w)| and whether a pivot vanished
template <int N>
__global__ __launch_bounds__(64) void k_gc_inverse(int n, int nw, const double* __restrict__ Gc,
                                                   double* __restrict__ ginv, double* __restrict__ logdet,
                                                   int* __restrict__ singular) {
  constexpr int LN = lanes_of<N>(), R = N / LN, G = 64 / LN;
  __shared__ double2 buf[G][N + 1];
  const int g = threadIdx.x / LN, q = threadIdx.x % LN;
  const int w = min((int)blockIdx.x * G + g, nw - 1);
  const double2* src = reinterpret_cast<const double2*>(Gc) + (size_t)w * n * n;
  for (int pass = 0; pass < 2; ++pass) {
    cplx a[R][N];
#pragma unroll
    for (int s = 0; s < R; ++s)
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const int i = q + LN * s;
        a[s][j] = {i == j ? 1.0 : 0.0, 0.0};
        if (i < n && j < n) {
          const double2 v = src[i + j * n];
          a[s][j] = {v.x, v.y};
        }
      }
    uint64_t perm;
    int step[R];
    LogDet ld;
    bool zero = false;
    if (pass == 0) {
      if (!logdet) continue;
      eliminate<N, LN, false, true>(a, q, buf[g], perm, step, ld, zero);
      if (q == 0) logdet[w] = ld.value();
      continue;
    }
    eliminate<N, LN, true, true>(a, q, buf[g], perm, step, ld, zero);
    if (zero) *singular = 1;
    double2* o = reinterpret_cast<double2*>(ginv) + (size_t)w * N * N;
#pragma unroll
    for (int s = 0; s < R; ++s)
#pragma unroll
      for (int j = 0; j < N; ++j)
        o[step[s] + (size_t)((perm >> (4 * j)) & 15u) * N] = make_double2(a[s][j].re, a[s][j].im);
  }
}

// M(w, k) = Gc(w)^-1 - V(k) for the (w, k) of a launch. MODE 0: the inverses; 1: their
// traces; 2: their sum over k; 3: the sum over k of log|det|. A group takes `chunk`
// matrices in turn: one k point and a run of frequencies (modes 0, 1), or one frequency and
// a run of k blocks (modes 2, 3). Two waves per SIMD, for which the 12- and 16-wide forms
// spill 24 to 96 bytes per lane; the sum over k of wide matrices takes 40 KB of LDS and one wave.
template <int N, int MODE>
__global__ __launch_bounds__(64, MODE == 2 && N >= 12 ? 1 : 2) void k_ksum(KsumArgs A) {
  constexpr int LN = lanes_of<N>(), R = N / LN, G = 64 / LN;
  __shared__ double2 buf[G][N + 1];
  __shared__ double2 acc[MODE == 2 ? G : 1][MODE == 2 ? N * N + 1 : 1];
  const int g = threadIdx.x / LN, q = threadIdx.x % LN;
  const int b = blockIdx.x;
  const int nkb = (A.nk + G - 1) / G;
  const int fix = MODE < 2 ? b % nkb : b / A.nchunk;      // k block / frequency
  const int c0 = (MODE < 2 ? b / nkb : b % A.nchunk) * A.chunk;
  const int c1 = min(c0 + A.chunk, MODE < 2 ? A.nw : nkb);
  if constexpr (MODE == 2) {
    for (int e = q; e < N * N; e += LN) acc[g][e] = make_double2(0.0, 0.0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  LogDet ld;
  for (int c = c0; c < c1; ++c) {
    const int w = MODE < 2 ? c : fix;
    const int kr = (MODE < 2 ? fix : c) * G + g;
    const bool ok = kr < A.nk;
    const int kc = ok ? kr : A.nk - 1;
    const double2* gi = reinterpret_cast<const double2*>(A.ginv) + (size_t)w * N * N;
    const double2* vk = reinterpret_cast<const double2*>(A.vk) + (size_t)kc * N * N;
    cplx a[R][N];
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
      for (int s = 0; s < R; ++s) {
        const double2 x = gi[j * N + q + LN * s], v = vk[j * N + q + LN * s];
        a[s][j] = {x.x - v.x, x.y - v.y};
      }
    uint64_t perm;
    int step[R];
    bool zero = false;
    LogDet one;
    eliminate<N, LN, MODE != 3>(a, q, buf[g], perm, step, one, zero);
    if constexpr (MODE == 0) {
      double2* o = reinterpret_cast<double2*>(A.out) + ((size_t)w * A.nk_all + A.k0 + kc) * A.n * A.n;
#pragma unroll
      for (int s = 0; s < R; ++s)
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const int col = (int)((perm >> (4 * j)) & 15u);
          if (ok && step[s] < A.n && col < A.n) o[step[s] + col * A.n] = make_double2(a[s][j].re, a[s][j].im);
        }
    } else if constexpr (MODE == 1) {
      cplx d{0.0, 0.0};
#pragma unroll
      for (int s = 0; s < R; ++s)
#pragma unroll
        for (int j = 0; j < N; ++j)
          if (step[s] < A.n && (int)((perm >> (4 * j)) & 15u) == step[s]) d = cadd(d, a[s][j]);
#pragma unroll
      for (int o = 1; o < LN; o <<= 1) {
        d.re += __shfl_xor(d.re, o, 64);
        d.im += __shfl_xor(d.im, o, 64);
      }
      if (ok && q == 0)
        reinterpret_cast<double2*>(A.out)[(size_t)w * A.nk_all + A.k0 + kc] = make_double2(d.re, d.im);
    } else if constexpr (MODE == 2) {
      // element (step, p_j) has one owner in the group
      if (ok) {
#pragma unroll
        for (int s = 0; s < R; ++s)
#pragma unroll
          for (int j = 0; j < N; ++j) {
            double2* t = &acc[g][step[s] + (int)((perm >> (4 * j)) & 15u) * N];
            const double2 v = *t;
            *t = make_double2(v.x + a[s][j].re, v.y + a[s][j].im);
          }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    } else {
      if (ok) {
        ld.mul(one.m);
        ld.e += one.e;
      }
    }
  }
  if constexpr (MODE == 2) {
    double2* o = reinterpret_cast<double2*>(A.part) + ((size_t)fix * A.parts + A.part0 + b % A.nchunk) * N * N;
    for (int e = threadIdx.x; e < N * N; e += 64) {
      double2 t = make_double2(0.0, 0.0);
      for (int h = 0; h < G; ++h) {
        t.x += acc[h][e].x;
        t.y += acc[h][e].y;
      }
      o[e] = t;
    }
  }
  if constexpr (MODE == 3) {
    double v = q == 0 ? ld.value() : 0.0;
    v = wave_sum(v);
    if (threadIdx.x == 0) A.part[(size_t)fix * A.parts + A.part0 + b % A.nchunk] = v;
  }
}

// sums of the partials over the k chunks: out[w][i + j n] from parts x (N x N complex), or
// out[w] from parts (n = 0); one wave per output
__global__ __launch_bounds__(64) void k_ksum_reduce(int parts, int n, int N, const double* __restrict__ part,
                                                    double scale, double* __restrict__ out) {
  const int lane = threadIdx.x;
  if (n == 0) {
    double s = 0.0;
    for (int p = lane; p < parts; p += 64) s += part[(size_t)blockIdx.x * parts + p];
    s = wave_sum(s);
    if (lane == 0) out[blockIdx.x] = s * scale;
    return;
  }
  const int w = blockIdx.x / n, j = blockIdx.x % n;  // one column of one frequency
  const double2* src = reinterpret_cast<const double2*>(part) + (size_t)w * parts * N * N + (size_t)j * N;
  for (int i = 0; i < n; ++i) {
    double re = 0.0, im = 0.0;
    for (int p = lane; p < parts; p += 64) {
      const double2 v = src[(size_t)p * N * N + i];
      re += v.x;
      im += v.y;
    }
    re = wave_sum(re);
    im = wave_sum(im);
    if (lane == 0)
      reinterpret_cast<double2*>(out)[(size_t)w * n * n + (size_t)j * n + i] = make_double2(re * scale, im * scale);
  }
}

template <class T>
DevBuf up(const T* p, size_t n) {
  DevBuf b(std::max<size_t>(n, 1) * sizeof(T));
  if (n) QED_HIP(hipMemcpyAsync(b.p, p, n * sizeof(T), hipMemcpyHostToDevice, stream()));
  return b;
}

int padded_dim(int n) {
  if (n <= 2) return n;
  if (n <= 4) return 4;
  if (n <= 8) return 8;
  if (n <= 12) return 12;
  if (n <= 16) return 16;
  fail("lattice k-sum: cluster Green function dimension above 16 is not supported");
}

template <class F>
void with_dim(int N, F&& f) {
  switch (N) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    default: f(std::integral_constant<int, 16>{}); break;
  }
}

template <int N>
void launch_ksum(const KsumArgs& A, int mode, int blocks) {
  switch (mode) {
    case 0: k_ksum<N, 0><<<blocks, 64, 0, stream()>>>(A); break;
    case 1: k_ksum<N, 1><<<blocks, 64, 0, stream()>>>(A); break;
    case 2: k_ksum<N, 2><<<blocks, 64, 0, stream()>>>(A); break;
    default: k_ksum<N, 3><<<blocks, 64, 0, stream()>>>(A); break;
  }
}

// device time of the last CPT k-sum (HIP events on the library stream)
double& last_ksum_ms() {
  static double ms = 0.0;
  return ms;
}

// Device memory, pinned host memory and events of one k-sum call. Calls take a free one and
// give it back (concurrent calls have one each); at most kKeep are kept, and none with more
// than kKeepBytes of either memory, so that small calls allocate nothing.
struct KsumSpace {
  DevBuf dev;
  unsigned char* pin = nullptr;
  size_t pin_bytes = 0;
  hipEvent_t ev[2] = {nullptr, nullptr};
  KsumSpace() = default;
  KsumSpace(const KsumSpace&) = delete;
  ~KsumSpace() {
    if (pin) (void)hipHostFree(pin);
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
  }
  void reserve(size_t d, size_t p) {
    if (dev.bytes < d) dev.alloc(d);
    if (pin_bytes < p) {
      if (pin) (void)hipHostFree(pin);
      pin = nullptr;
      pin_bytes = 0;
      QED_HIP(hipHostMalloc((void**)&pin, p, hipHostMallocDefault));
      pin_bytes = p;
    }
    for (hipEvent_t& e : ev)
      if (!e) QED_HIP(hipEventCreate(&e));
  }
};

class KsumLease {
 public:
  KsumLease() {
    std::lock_guard<std::mutex> lk(mutex());
    if (!idle().empty()) {
      s_ = std::move(idle().back());
      idle().pop_back();
    } else {
      s_ = std::make_unique<KsumSpace>();
    }
  }
  ~KsumLease() {
    (void)hipStreamSynchronize(stream());  // also after a failure: nothing may still use the memory
    if (s_->dev.bytes > kKeepBytes || s_->pin_bytes > kKeepBytes) return;
    std::lock_guard<std::mutex> lk(mutex());
    if (idle().size() < kKeep) idle().push_back(std::move(s_));
  }
  KsumSpace* operator->() { return s_.get(); }

 private:
  static constexpr size_t kKeep = 4, kKeepBytes = size_t(64) << 20;
  static std::mutex& mutex() {
    static std::mutex m;
    return m;
  }
  static std::vector<std::unique_ptr<KsumSpace>>& idle() {  // never destroyed: the runtime may be gone by then
    static auto* v = new std::vector<std::unique_ptr<KsumSpace>>();
    return *v;
  }
  std::unique_ptr<KsumSpace> s_;
};

// Copies bytes from the device to caller memory through the pinned buffer, in pieces: while
// one piece is on its way the previous one is copied out, by several threads (128 MB: 2.8 ms,
// about 10 by one).
void copy_out(unsigned char* dst, const unsigned char* src_dev, size_t bytes, unsigned char* pin, size_t pin_bytes) {
  const size_t piece = pin_bytes / 2;
  auto send = [&](size_t i) {
    const size_t o = i * piece;
    if (o < bytes)
      QED_HIP(hipMemcpyAsync(pin + (i & 1) * piece, src_dev + o, std::min(piece, bytes - o), hipMemcpyDeviceToHost,
                             stream()));
  };
  send(0);
  for (size_t i = 0; i * piece < bytes; ++i) {
    QED_HIP(hipStreamSynchronize(stream()));
    send(i + 1);
    const size_t o = i * piece, len = std::min(piece, bytes - o);
    const unsigned char* from = pin + (i & 1) * piece;
    CopyHelpers::get().copy(dst + o, from, len);
  }
}

// The k-sums of mode 0 to 3 (see k_ksum) for host inputs: one upload, Gc^-1 and V(k) on the
// device, the sums, one download in the caller's layout.
void ksum(int n, int nw, const double* Gc, const double* V0, int nterm, const double* Vt, const double* nv, int nk,
          const double* k, int mode, double* out) {
  const int N = padded_dim(n), LN = N == 16 ? 8 : N >= 4 ? 4 : N, G = 64 / LN;
  const size_t n2 = 2 * (size_t)n * n, N2 = 2 * (size_t)N * N;  // doubles per matrix
  // V(k) of as many k points at a time as 256 MB hold
  const int kmax = (int)std::max<size_t>(G, std::min<size_t>(nk, (size_t(256) << 20) / (N2 * 8) / G * G));
  // Matrices per group: about 4096 waves (two per SIMD of 256 CUs, twice over), one matrix
  // each when there are fewer
  const long nkb_all = (nk + G - 1) / G;
  const long runs = mode < 2 ? nw : (kmax + G - 1) / G;
  const int chunk = (int)std::max<long>(1, std::min<long>(runs, nkb_all * nw / 4096));
  int parts = 0;
  for (int k0 = 0; k0 < nk; k0 += kmax)
    if (mode >= 2) parts += ((std::min(kmax, nk - k0) + G - 1) / G + chunk - 1) / chunk;
  const size_t nwk = (size_t)nw * nk;
  const size_t out_len = mode == 0 ? nwk * n2 : mode == 1 ? nwk * 2 : mode == 2 ? nw * n2 : (size_t)nw;
  // inputs in the order of the upload, then the device's own arrays (doubles)
  size_t off = 0;
  auto take = [&](size_t len) {
    const size_t o = off;
    off += (len + 31) & ~size_t(31);
    return o;
  };
  const size_t o_gc = take(nw * n2), o_v0 = take(n2), o_vt = take(nterm * n2), o_nv = take(3 * (size_t)nterm),
               o_k = take(3 * (size_t)nk), n_in = off;
  const size_t o_gi = take(nw * N2), o_vk = take(kmax * N2),
               o_part = take(mode == 2 ? nw * (size_t)parts * N2 : mode == 3 ? nw * (size_t)parts : 0),
               o_ld = take(nw + 1), o_out = take(out_len);
  // small results come down with log|det Gc| and the singular flag in one copy; large ones
  // after them, in pieces
  const size_t n_down = off - o_ld;
  const bool small = n_down * 8 <= (size_t(1) << 20);
  KsumLease L;
  const size_t piece = size_t(16) << 20;
  L->reserve(off * 8, std::max(n_in, small ? n_down : std::max<size_t>(nw + 1, 2 * piece / 8)) * 8);
  double* d = L->dev.as<double>();
  double* h = reinterpret_cast<double*>(L->pin);
  std::memcpy(h + o_gc, Gc, nw * n2 * 8);
  std::memcpy(h + o_v0, V0, n2 * 8);
  if (nterm > 0) {
    std::memcpy(h + o_vt, Vt, nterm * n2 * 8);
    std::memcpy(h + o_nv, nv, 3 * (size_t)nterm * 8);
  }
  std::memcpy(h + o_k, k, 3 * (size_t)nk * 8);
  hipStream_t st = stream();
  QED_HIP(hipMemcpyAsync(d, h, n_in * 8, hipMemcpyHostToDevice, st));
  double* ld = d + o_ld;
  int* singular = reinterpret_cast<int*>(ld + nw);
  QED_HIP(hipMemsetAsync(singular, 0, 8, st));
  QED_HIP(hipEventRecord(L->ev[0], st));
  with_dim(N, [&](auto dim) {
    constexpr int M = decltype(dim)::value;
    k_gc_inverse<M><<<(nw + G - 1) / G, 64, 0, st>>>(n, nw, d + o_gc, d + o_gi, mode == 3 ? ld : nullptr, singular);
    int part0 = 0;
    for (int k0 = 0; k0 < nk; k0 += kmax) {
      KsumArgs A{};
      A.n = n;
      A.nw = nw;
      A.nk = std::min(kmax, nk - k0);
      A.k0 = k0;
      A.nk_all = nk;
      A.chunk = chunk;
      const int nkb = (A.nk + G - 1) / G;
      A.nchunk = ((mode < 2 ? nw : nkb) + chunk - 1) / chunk;
      A.part0 = part0;
      A.parts = parts;
      A.ginv = d + o_gi;
      A.vk = d + o_vk;
      A.out = d + o_out;
      A.part = d + o_part;
      k_vk<M><<<(A.nk + 7) / 8, 256, 0, st>>>(n, nterm, A.nk, d + o_v0, d + o_vt, d + o_nv, d + o_k + 3 * (size_t)k0,
                                              d + o_vk);
      launch_ksum<M>(A, mode, (mode < 2 ? nkb : nw) * A.nchunk);
      if (mode >= 2) part0 += A.nchunk;
    }
  });
  if (mode == 2) k_ksum_reduce<<<nw * n, 64, 0, st>>>(parts, n, N, d + o_part, 1.0 / nk, d + o_out);
  if (mode == 3) k_ksum_reduce<<<nw, 64, 0, st>>>(parts, 0, 0, d + o_part, 1.0 / nk, d + o_out);
  QED_HIP(hipGetLastError());
  QED_HIP(hipEventRecord(L->ev[1], st));
  if (!small) touch_pages(reinterpret_cast<unsigned char*>(out), out_len * 8);  // while the kernels run
  QED_HIP(hipMemcpyAsync(h, ld, (small ? n_down : (size_t)nw + 1) * 8, hipMemcpyDeviceToHost, st));
  QED_HIP(hipStreamSynchronize(st));
  int bad = 0;
  std::memcpy(&bad, h + nw, sizeof(int));
  if (bad) fail("cluster Green function is singular at a requested frequency");
  if (small) {
    std::memcpy(out, h + (o_out - o_ld), out_len * 8);
    // log|det(V G - 1)| = log|det G| + log|det(G^-1 - V)|  (padding blocks contribute log 1 = 0)
    if (mode == 3)
      for (int w = 0; w < nw; ++w) out[w] += h[w];
  } else {
    std::vector<double> logdet(h, h + nw);
    copy_out(reinterpret_cast<unsigned char*>(out), reinterpret_cast<const unsigned char*>(d + o_out), out_len * 8,
             L->pin, 2 * piece);
    if (mode == 3)
      for (int w = 0; w < nw; ++w) out[w] += logdet[w];
  }
  float ms = 0.0f;
  QED_HIP(hipEventElapsedTime(&ms, L->ev[0], L->ev[1]));
  if (mode < 3) last_ksum_ms() = ms;
}

}  // namespace

}  // namespace qed

using namespace qed;

extern "C" {

int qed_qmatrix_gf(int L, int M, const double* e, const double* Q, int nz, const double* z, double* G) {
  return guard([&] {
    if (L <= 0 || nz <= 0) return;
    if (L > 16) fail("qmatrix_gf: at most 16 orbitals per block");
    DevBuf de = up(e, (size_t)M), dq = up(Q, (size_t)L * M), dz = up(z, (size_t)2 * nz);
    DevBuf dg = up(G, (size_t)2 * nz * L * L);
    if (M > 0) k_qmatrix_gf<<<nz, 256, 0, stream()>>>(L, M, de.as<double>(), dq.as<double>(), dz.as<double>(), dg.as<double>());
    QED_HIP(hipGetLastError());
    QED_HIP(hipMemcpyAsync(G, dg.p, (size_t)2 * nz * L * L * 8, hipMemcpyDeviceToHost, stream()));
    QED_HIP(hipStreamSynchronize(stream()));
  });
}

int qed_cf_eval(int n, const int* off, const int* depth, const double* a, const double* b, int nz,
                const double* z, double* out) {
  return guard([&] {
    if (n <= 0 || nz <= 0) return;
    size_t tot = 0;
    for (int f = 0; f < n; ++f) tot = std::max<size_t>(tot, (size_t)off[f] + depth[f]);
    DevBuf doff = up(off, n), ddep = up(depth, n), da = up(a, tot), db = up(b, tot), dz = up(z, 2 * (size_t)nz);
    DevBuf dout((size_t)2 * n * nz * 8);
    int tot_threads = n * nz;
    k_cf_eval<<<(tot_threads + 255) / 256, 256, 0, stream()>>>(n, doff.as<int>(), ddep.as<int>(), da.as<double>(),
                                                               db.as<double>(), nz, dz.as<double>(), dout.as<double>());
    QED_HIP(hipGetLastError());
    QED_HIP(hipMemcpyAsync(out, dout.p, (size_t)2 * n * nz * 8, hipMemcpyDeviceToHost, stream()));
    QED_HIP(hipStreamSynchronize(stream()));
  });
}

int qed_ksum_last_ms(double* ms) {
  *ms = last_ksum_ms();
  return 0;
}

int qed_cpt_batch(int n, int nw, const double* Gc, const double* V0, int nterm, const double* Vt,
                  const double* nv, int nk, const double* k, int mode, double* out) {
  return guard([&] {
    if (mode < 0 || mode > 2) fail("cpt_batch: mode must be 0, 1 or 2");
    if (n <= 0 || nw <= 0 || nk <= 0) return;
    ksum(n, nw, Gc, V0, nterm, Vt, nv, nk, k, mode, out);
  });
}

int qed_sef_batch(int n, int nw, const double* Gc, const double* V0, int nterm, const double* Vt,
                  const double* nv, int nk, const double* k, double* out) {
  return guard([&] {
    if (n <= 0 || nw <= 0 || nk <= 0) return;
    ksum(n, nw, Gc, V0, nterm, Vt, nv, nk, k, 3, out);
  });
}

}  // extern "C"
