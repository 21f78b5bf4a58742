// Krylov solvers on device vectors: BLAS-1 with wave64 shuffle reductions, Lanczos for
// the ground state (eigenvalue pass + eigenvector replay), the scalar Lanczos of the
// continued-fraction Green function and Freund's band Lanczos. The recurrence scalars
// (alpha, beta, the projected band matrix) and their small eigenproblems stay in FP64 on
// the host; every O(D) operation runs on the device.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>

#include "../../include/qed.h"
#include "qed_linalg.hpp"
#include "qed_sector.hpp"

namespace qed {

namespace {

constexpr int RB = 256;
constexpr int kMaxMulti = 64;
constexpr uint32_t kMaxBlocks = 2048;

struct PtrList {
  const double* p[kMaxMulti];
};
struct MutPtrList {
  double* p[kMaxMulti];
};

uint32_t red_blocks(uint64_t n) {
  uint64_t b = (n + (uint64_t)RB * 8 - 1) / ((uint64_t)RB * 8);
  return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(b, 1), kMaxBlocks);
}

// scratch for block partials and final scalars (library calls are serialized)
DevBuf& red_scratch() {
  static DevBuf b((size_t)kMaxBlocks * (kMaxMulti + 1) * sizeof(double) + 4096);
  return b;
}
std::vector<double>& host_scratch() {
  static std::vector<double> h;
  return h;
}

__global__ __launch_bounds__(RB) void k_multi_dot(const double* __restrict__ x, PtrList ys, int m,
                                                  uint64_t n, double* __restrict__ part) {
  __shared__ double sh[RB / 64];
  double acc[8];
  for (int base = 0; base < m; base += 8) {
    int cnt = min(8, m - base);
#pragma unroll
    for (int q = 0; q < 8; ++q) acc[q] = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * RB) {
      double xv = x[i];
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (q < cnt) acc[q] += xv * ys.p[base + q][i];
    }
    for (int q = 0; q < cnt; ++q) {
      double s = block_sum(acc[q], sh);
      if (threadIdx.x == 0) part[(size_t)(base + q) * gridDim.x + blockIdx.x] = s;
    }
  }
}

__global__ void k_finish(const double* __restrict__ part, int nb, int m, double* __restrict__ out) {
  __shared__ double sh[RB / 64];
  for (int j = 0; j < m; ++j) {
    double s = 0.0;
    for (int i = threadIdx.x; i < nb; i += RB) s += part[(size_t)j * nb + i];
    s = block_sum(s, sh);
    if (threadIdx.x == 0) out[j] = s;
  }
}

__global__ void k_axpy(double a, const double* __restrict__ x, double* __restrict__ y, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    y[i] += a * x[i];
}

__global__ void k_zero(double* __restrict__ x, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    x[i] = 0.0;
}

__global__ void k_scal(double a, double* __restrict__ x, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    x[i] *= a;
}

__global__ void k_scal2(double ar, double* __restrict__ r, double aq, double* __restrict__ q,
                        uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    r[i] *= ar;
    q[i] *= aq;
  }
}

// y += a x, partial sums of y^2
__global__ __launch_bounds__(RB) void k_axpy_nrm(double a, const double* __restrict__ x,
                                                 double* __restrict__ y, uint64_t n,
                                                 double* __restrict__ part) {
  __shared__ double sh[RB / 64];
  double acc = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * RB) {
    double v = y[i] + a * x[i];
    y[i] = v;
    acc += v * v;
  }
  double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// ---- Lanczos step (device scalars, LzStep) ----------------------------------------------
// w_{k+1} = y - alpha_k v_k with alpha_k = <w_k, y> / beta_{k-1}; the parts of |w_{k+1}|^2.
// Bound by its 24 bytes per element; each wave adds up the product's parts by itself, so
// that a step is two launches and no scalar kernel (at most kLzParts parts).
__global__ __launch_bounds__(RB) void k_lz_axpy_nrm(LzStep lz, int na, double* __restrict__ alpha,
                                                    double* __restrict__ beta, const double* __restrict__ x,
                                                    double* __restrict__ y, uint64_t n, double* __restrict__ part) {
  __shared__ double sh[RB / 64];
  const double b = lz.k == 0 ? 1.0 : sqrt(lz_sum(lz.pb, lz.nb));
  const double inv = lz_inv(b);
  const double al = lz_sum(lz.pa, na) * inv;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    alpha[lz.k % lz.ring] = al;
    if (lz.k > 0) beta[(lz.k - 1) % lz.ring] = b;
  }
  const double a = -al * inv;
  double acc = 0.0;
  const uint64_t n2 = n / 2;
  double2* __restrict__ y2 = reinterpret_cast<double2*>(y);
  const double2* __restrict__ x2 = reinterpret_cast<const double2*>(x);
  for (uint64_t i = (uint64_t)blockIdx.x * RB + threadIdx.x; i < n2; i += (uint64_t)gridDim.x * RB) {
    const double2 u = x2[i];
    double2 v = y2[i];
    v.x += a * u.x;
    v.y += a * u.y;
    y2[i] = v;
    acc += v.x * v.x + v.y * v.y;
  }
  if (n % 2 && blockIdx.x == 0 && threadIdx.x == 0) {
    const double v = y[n - 1] + a * x[n - 1];
    y[n - 1] = v;
    acc += v * v;
  }
  const double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// p[0] = sum of n values (more than kLzParts)
__global__ __launch_bounds__(1024) void k_lz_fold(double* __restrict__ p, int n) {
  __shared__ double sh[16];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) s += p[i];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) p[0] = s;
}

// beta_k of the last step of a chunk
__global__ __launch_bounds__(64) void k_lz_last(const double* __restrict__ pb, int nb, double* __restrict__ beta) {
  const double b = sqrt(lz_sum(pb, nb));
  if (threadIdx.x == 0) *beta = b;
}

// continued-fraction Lanczos step: (psi, q) <- (q / b, -b psi)
__global__ void k_swapscale(double b, double* __restrict__ psi, double* __restrict__ q, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    double t = psi[i];
    psi[i] = q[i] / b;
    q[i] = -b * t;
  }
}

// y -= sum_k c[k] xs[k]
__global__ void k_multi_axpy(PtrList xs, const double* __restrict__ c, int m, double* __restrict__ y,
                             uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    double v = y[i];
    for (int k = 0; k < m; ++k) v -= c[k] * xs.p[k][i];
    y[i] = v;
  }
}

// ys[k] -= c[k] x
__global__ void k_multi_axpy_rev(MutPtrList ys, const double* __restrict__ c, int m,
                                 const double* __restrict__ x, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    double xv = x[i];
    for (int k = 0; k < m; ++k) ys.p[k][i] -= c[k] * xv;
  }
}

// y += 0.5 x with 16-byte accesses: the read-modify-write stream the H.v is compared with
__global__ __launch_bounds__(256) void k_stream_rmw(const double2* __restrict__ x, double2* __restrict__ y,
                                                   uint64_t n2) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n2; i += (uint64_t)gridDim.x * 256) {
    const double2 a = x[i];
    double2 b = y[i];
    b.x += 0.5 * a.x;
    b.y += 0.5 * a.y;
    y[i] = b;
  }
}

uint32_t stream_blocks(uint64_t n) {
  uint64_t b = (n + 255) / 256;
  return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(b, 1), (uint64_t)device_cu_count() * 16);
}

}  // namespace

namespace {

// Normalized eigenvector of the lowest eigenvalue lam of the Lanczos tridiagonal: three
// steps of inverse iteration on (T - lam) with partial pivoting, one factorization
void tridiag_vector(const std::vector<double>& a, const std::vector<double>& b, double lam, std::vector<double>& vec) {
  const int n = (int)a.size();
  vec.assign(n, 1.0);
  double scale = 0.0;
  for (int i = 0; i < n; ++i) scale = std::max(scale, std::fabs(a[i]) + (i < n - 1 ? std::fabs(b[i]) : 0.0));
  const double shift = lam - 1e-14 * std::max(scale, 1.0);
  static thread_local std::vector<double> dm, du, du2, f;
  static thread_local std::vector<char> swapped;
  dm.resize(n);
  du.assign(b.begin(), b.begin() + (n - 1));
  du2.assign(n, 0.0);
  f.resize(n);
  swapped.assign(n, 0);
  for (int i = 0; i < n; ++i) dm[i] = a[i] - shift;
  for (int i = 0; i < n - 1; ++i) {
    const double dl = b[i];
    if (std::fabs(dm[i]) >= std::fabs(dl)) {
      if (dm[i] == 0.0) dm[i] = 1e-300;
      f[i] = dl / dm[i];
      dm[i + 1] -= f[i] * du[i];
    } else {
      swapped[i] = 1;
      f[i] = dm[i] / dl;
      dm[i] = dl;
      const double t = dm[i + 1];
      dm[i + 1] = du[i] - f[i] * t;
      if (i < n - 2) {
        du2[i] = du[i + 1];
        du[i + 1] = -f[i] * du2[i];
      }
      du[i] = t;
    }
  }
  if (dm[n - 1] == 0.0) dm[n - 1] = 1e-300;
  for (int it = 0; it < 3; ++it) {
    for (int i = 0; i < n - 1; ++i) {
      if (swapped[i]) std::swap(vec[i], vec[i + 1]);
      vec[i + 1] -= f[i] * vec[i];
    }
    vec[n - 1] /= dm[n - 1];
    if (n >= 2) vec[n - 2] = (vec[n - 2] - du[n - 2] * vec[n - 1]) / dm[n - 2];
    for (int i = n - 3; i >= 0; --i) vec[i] = (vec[i] - du[i] * vec[i + 1] - du2[i] * vec[i + 2]) / dm[i];
    double nrm = 0.0;
    for (double v : vec) nrm += v * v;
    nrm = std::sqrt(nrm);
    for (double& v : vec) v /= nrm;
  }
  // sign convention: first component positive (sign does not affect the Ritz residual)
  if (vec[0] < 0)
    for (double& v : vec) v = -v;
}

}  // namespace

// lowest eigenvalue of the Lanczos tridiagonal and its normalized eigenvector
// (QL eigenvalues, then inverse iteration for the vector)
void tridiag_lowest(const std::vector<double>& a, const std::vector<double>& b, double* e0,
                    std::vector<double>& vec) {
  const int n = (int)a.size();
  if (n == 1) {
    vec.assign(1, 1.0);
    *e0 = a[0];
    return;
  }
  std::vector<double> d(a), e(b.begin(), b.begin() + (n - 1));
  tridiag_eigen(n, d.data(), e.data(), nullptr);
  *e0 = d[0];
  tridiag_vector(a, b, d[0], vec);
}

namespace {

// The same for a matrix that grows by a row per call, started from the pair (lam, vec) of
// the last call: Rayleigh quotient iteration, accepted when it is stationary and a Sturm
// count finds no eigenvalue below. O(n) where the QL sweep is O(n^2), which took most of a
// small ground state (177 steps: 40 of 60 ms).
void tridiag_lowest_next(const std::vector<double>& a, const std::vector<double>& b, double* lam,
                         std::vector<double>& vec) {
  const int n = (int)a.size();
  if (n <= 16 || (int)vec.size() != n - 1) {
    tridiag_lowest(a, b, lam, vec);
    return;
  }
  static thread_local std::vector<double> x;
  x.assign(vec.begin(), vec.end());
  x.push_back(0.0);
  double scale = 1.0;
  for (int i = 0; i < n; ++i) scale = std::max(scale, std::fabs(a[i]) + std::fabs(b[i]));
  // the new row couples to the last component only: start from the first-order update
  x[n - 1] = b[n - 2] * x[n - 2] / (*lam - a[n - 1] != 0.0 ? *lam - a[n - 1] : scale);
  double rho = 0.0;
  bool ok = false;
  for (int it = 0; it < 6; ++it) {
    double nn = 0.0, num = 0.0;
    for (int i = 0; i < n; ++i) nn += x[i] * x[i];
    for (int i = 0; i < n; ++i) num += x[i] * (a[i] * x[i] + (i + 1 < n ? 2.0 * b[i] * x[i + 1] : 0.0));
    rho = num / nn;
    double res = 0.0;
    for (int i = 0; i < n; ++i) {
      const double r = (a[i] - rho) * x[i] + (i > 0 ? b[i - 1] * x[i - 1] : 0.0) + (i + 1 < n ? b[i] * x[i + 1] : 0.0);
      res += r * r;
    }
    // the quotient's error is of second order in the residual
    if (!(res <= nn * scale * scale)) break;
    if (res <= 1e-20 * nn * scale * scale) {
      ok = true;
      break;
    }
    static thread_local std::vector<double> next;
    tridiag_vector(a, b, rho, next);
    x = next;
  }
  if (ok) {  // negative pivots of T - (rho - delta): the eigenvalues below
    const double shift = rho - 1e-12 * scale;
    double q = a[0] - shift;
    for (int i = 0; ok && i < n; ++i) {
      if (i > 0) q = a[i] - shift - b[i - 1] * b[i - 1] / q;
      if (!(q > 0.0)) ok = false;
    }
  }
  if (!ok) {
    tridiag_lowest(a, b, lam, vec);
    return;
  }
  *lam = rho;
  tridiag_vector(a, b, rho, vec);
}

// The host side of a Lanczos run: pinned memory for the scalars of two chunks of steps, and
// an event for each.
struct LanczosHost {
  static constexpr size_t kDoubles = 4 * kLzRing;
  double* pin = nullptr;
  hipEvent_t done[2] = {nullptr, nullptr};
  LanczosHost() {
    try {
      QED_HIP(hipHostMalloc((void**)&pin, kDoubles * sizeof(double), hipHostMallocDefault));
      for (hipEvent_t& e : done) QED_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    } catch (...) {
      release();
      throw;
    }
  }
  LanczosHost(const LanczosHost&) = delete;
  ~LanczosHost() { release(); }

 private:
  void release() {
    if (pin) (void)hipHostFree(pin);
    for (hipEvent_t e : done)
      if (e) (void)hipEventDestroy(e);
  }
};

// made with the library for qed_lanczos_gs_noalloc, whose calls one lock serializes
LanczosHost* g_fixed_host = nullptr;

// One of them for the length of a run, from a small pool (one per concurrent run) and given
// back; or the fixed one.
class LanczosLease {
 public:
  explicit LanczosLease(bool fixed) : fixed_(fixed) {
    if (fixed_) {
      h_ = g_fixed_host;
      return;
    }
    std::lock_guard<std::mutex> lk(mutex());
    if (!idle().empty()) {
      h_ = idle().back();
      idle().pop_back();
    } else {
      h_ = new LanczosHost();
    }
  }
  LanczosLease(const LanczosLease&) = delete;
  ~LanczosLease() {
    (void)hipStreamSynchronize(stream());
    if (fixed_) return;
    std::lock_guard<std::mutex> lk(mutex());
    if (idle().size() < 8) idle().push_back(h_);
    else delete h_;
  }
  LanczosHost* operator->() { return h_; }

 private:
  static std::mutex& mutex() {
    static std::mutex m;
    return m;
  }
  static std::vector<LanczosHost*>& idle() {  // never destroyed: the runtime may be gone by then
    static auto* v = new std::vector<LanczosHost*>();
    return *v;
  }
  bool fixed_;
  LanczosHost* h_ = nullptr;
};

}  // namespace

void lanczos_host_init() {
  if (!g_fixed_host) g_fixed_host = new LanczosHost();
}

std::recursive_mutex& lib_mutex() {
  static std::recursive_mutex m;
  return m;
}

void multi_dot(const double* x, const double* const* ys, int m, uint64_t n, double* out) {
  if (m > kMaxMulti) fail("multi_dot: too many vectors");
  if (m == 0) return;
  if (n == 0) {
    std::fill(out, out + m, 0.0);
    return;
  }
  PtrList l{};
  for (int k = 0; k < m; ++k) l.p[k] = ys[k];
  uint32_t nb = red_blocks(n);
  double* part = red_scratch().as<double>();
  double* fin = part + (size_t)kMaxBlocks * kMaxMulti;
  k_multi_dot<<<nb, RB, 0, stream()>>>(x, l, m, n, part);
  k_finish<<<1, RB, 0, stream()>>>(part, nb, m, fin);
  QED_HIP(hipMemcpyAsync(out, fin, m * sizeof(double), hipMemcpyDeviceToHost, stream()));
  QED_HIP(hipStreamSynchronize(stream()));
}

double dot(const double* x, const double* y, uint64_t n) {
  double r;
  multi_dot(x, &y, 1, n, &r);
  return r;
}

double nrm2(const double* x, uint64_t n) { return std::sqrt(dot(x, x, n)); }

void axpy(double a, const double* x, double* y, uint64_t n) {
  if (n) k_axpy<<<stream_blocks(n), 256, 0, stream()>>>(a, x, y, n);
}
void scal(double a, double* x, uint64_t n) {
  if (n) k_scal<<<stream_blocks(n), 256, 0, stream()>>>(a, x, n);
}
void scal2(double ar, double* r, double aq, double* q, uint64_t n) {
  if (n) k_scal2<<<stream_blocks(n), 256, 0, stream()>>>(ar, r, aq, q, n);
}

double axpy_nrm2(double a, const double* x, double* y, uint64_t n) {
  uint32_t nb = red_blocks(n);
  double* part = red_scratch().as<double>();
  double* fin = part + (size_t)kMaxBlocks * kMaxMulti;
  k_axpy_nrm<<<nb, RB, 0, stream()>>>(a, x, y, n, part);
  k_finish<<<1, RB, 0, stream()>>>(part, nb, 1, fin);
  double s;
  QED_HIP(hipMemcpyAsync(&s, fin, sizeof(double), hipMemcpyDeviceToHost, stream()));
  QED_HIP(hipStreamSynchronize(stream()));
  return std::sqrt(s);
}

void multi_axpy(const double* c, const double* const* xs, int m, double* y, uint64_t n) {
  if (m == 0 || n == 0) return;
  if (m > kMaxMulti) fail("multi_axpy: too many vectors");
  PtrList l{};
  for (int k = 0; k < m; ++k) l.p[k] = xs[k];
  double* cd = red_scratch().as<double>() + (size_t)kMaxBlocks * kMaxMulti + 64;
  QED_HIP(hipMemcpyAsync(cd, c, m * sizeof(double), hipMemcpyHostToDevice, stream()));
  k_multi_axpy<<<stream_blocks(n), 256, 0, stream()>>>(l, cd, m, y, n);
  QED_HIP(hipStreamSynchronize(stream()));
}

void multi_axpy_rev(const double* c, const double* x, double* const* ys, int m, uint64_t n) {
  if (m == 0 || n == 0) return;
  if (m > kMaxMulti) fail("multi_axpy_rev: too many vectors");
  MutPtrList l{};
  for (int k = 0; k < m; ++k) l.p[k] = ys[k];
  double* cd = red_scratch().as<double>() + (size_t)kMaxBlocks * kMaxMulti + 64;
  QED_HIP(hipMemcpyAsync(cd, c, m * sizeof(double), hipMemcpyHostToDevice, stream()));
  k_multi_axpy_rev<<<stream_blocks(n), 256, 0, stream()>>>(l, cd, m, x, n);
  QED_HIP(hipStreamSynchronize(stream()));
}

namespace {

// The device side of a Lanczos run: the two vectors, the parts of the two reductions and
// the last kLzRing alpha and beta, in the caller's memory where given.
struct LanczosRun {
  const qed_sector& s;
  uint64_t n;
  DevBuf rb, qb, wb;
  double *r, *q, *pa, *pb[2], *alpha, *beta;
  int nb = 0;  // parts of the last |w|^2
  int k = 0;   // steps done

  LanczosRun(const qed_sector& sec, const LanczosWork* ws) : s(sec), n(sec.D) {
    if (ws) {
      r = ws->r;
      q = ws->q;
      pa = ws->red;
    } else {
      rb.alloc(n * 8);
      qb.alloc(n * 8);
      wb.alloc((kLzWork - kLzRows + lz_parts(s)) * 8);
      r = rb.as<double>();
      q = qb.as<double>();
      pa = wb.as<double>();
    }
    pb[0] = pa + lz_parts(s);
    pb[1] = pb[0] + kLzParts;
    alpha = pb[1] + kLzParts;
    beta = alpha + kLzRing;
  }
  void start(const double* psi) {
    if (n) {
      QED_HIP(hipMemcpyAsync(r, psi, n * 8, hipMemcpyDeviceToDevice, stream()));
      k_zero<<<stream_blocks(n), 256, 0, stream()>>>(q, n);
    }
    k = 0;
  }
  // one step: w in r, the next one in r afterwards
  void step() {
    LzStep L;
    L.kind = 1;
    L.k = k;
    L.pb = pb[(k + 1) & 1];
    L.nb = nb;
    L.beta = beta;
    L.ring = kLzRing;
    L.pa = pa;
    int na = hv_step(s, r, q, L);
    if (na > kLzParts) {
      k_lz_fold<<<1, 1024, 0, stream()>>>(pa, na);
      na = 1;
    }
    const uint32_t grid = (uint32_t)std::min<uint64_t>(std::max<uint64_t>((n + RB * 8 - 1) / (RB * 8), 1), kLzParts);
    k_lz_axpy_nrm<<<grid, RB, 0, stream()>>>(L, na, alpha, beta, r, q, n, pb[k & 1]);
    nb = (int)grid;
    std::swap(r, q);
    ++k;
  }
  // the alpha and beta of the last kLzRing steps into host memory (asynchronous)
  void fetch(double* h) {
    k_lz_last<<<1, 64, 0, stream()>>>(pb[(k + 1) & 1], nb, beta + (k - 1) % kLzRing);
    QED_HIP(hipMemcpyAsync(h, alpha, 2 * kLzRing * sizeof(double), hipMemcpyDeviceToHost, stream()));
    QED_HIP(hipGetLastError());
  }
};

}  // namespace

// The ground state by Lanczos. The recurrence runs on the device in chunks of steps, the
// scalars of a chunk come down with one copy, and the host applies the stopping test to
// each of its steps while the next chunk runs; steps beyond the converged one are dropped.
// The eigenvector is rebuilt by the same recurrence with the known scalars, one launch per
// step. Chunks are short where a step costs more than the round trip it saves (about 20 us):
// below 2^20 amplitudes a step takes 10 to 40 us, above 2^24 over 200 us.
void lanczos_gs(qed_sector& s, double accur, int max_iter, double* psi, double* E0, int* niter,
                std::vector<double>* alpha_out, std::vector<double>* beta_out, const LanczosWork* ws) {
  const uint64_t n = s.D;
  const int chunk = n <= (1u << 20) ? 8 : n <= (1u << 24) ? 2 : 1;
  std::vector<double> alpha, beta, evec;
  double e0 = 0.0;
  LanczosLease host(ws != nullptr);
  LanczosRun run(s, ws);
  run.start(psi);
  const bool ahead = chunk > 1;
  int launched = 0, tested = 0;  // steps
  int end[2] = {0, 0};           // steps done at the end of the two chunks in flight
  int slot = 0;
  bool converged = !(2.0 * accur > accur);  // as the loop of the scalar form: no step for such accur
  auto launch = [&] {
    // as many as there may be and one more, at which the limit is seen (the limit may be INT_MAX)
    const int left = max_iter - launched, c = left >= chunk ? chunk : std::max(1, left + 1);
    for (int i = 0; i < c; ++i) run.step();
    launched += c;
    run.fetch(host->pin + slot * 2 * kLzRing);
    QED_HIP(hipEventRecord(host->done[slot], stream()));
    end[slot] = launched;
    slot ^= 1;
  };
  while (!converged) {
    if (launched == tested) launch();
    if (ahead && launched <= max_iter && launched - tested <= chunk) launch();
    // the older chunk in flight
    const int o = launched > tested && end[slot] > tested ? slot : slot ^ 1;
    QED_HIP(hipEventSynchronize(host->done[o]));
    const double* h = host->pin + o * 2 * kLzRing;
    for (int k = tested; k < end[o] && !converged; ++k) {
      alpha.push_back(h[k % kLzRing]);
      beta.push_back(h[kLzRing + k % kLzRing]);
      tridiag_lowest_next(alpha, beta, &e0, evec);
      if ((int)alpha.size() > max_iter)
        fail("Lanczos procedure exceeded " + std::to_string(max_iter) + " iterations");
      converged = !(std::fabs(evec.back() * beta.back()) > accur);
    }
    tested = end[o];
  }
  if (!alpha.empty()) tridiag_lowest(alpha, beta, &e0, evec);
  *E0 = e0;
  *niter = (int)beta.size();
  if (alpha_out) *alpha_out = alpha;
  if (beta_out) *beta_out = beta;
  if (evec.empty()) return;
  // eigenvector: the recurrence again from the start vector
  run.start(psi);
  if (n) k_scal<<<stream_blocks(n), 256, 0, stream()>>>(evec[0], psi, n);
  for (size_t j = 1; j < evec.size(); ++j) {
    // w_j = (H w_{j-1}) / b1 - (b1 / b2) w_{j-2} - (alpha_{j-1} / b1) w_{j-1}, v_j = w_j / beta_{j-1}
    const double b1 = j >= 2 ? beta[j - 2] : 1.0, b2 = j >= 3 ? beta[j - 3] : 1.0;
    LzStep L;
    L.kind = 2;
    L.s0 = 1.0 / b1;
    L.s1 = j >= 2 ? -b1 * (1.0 / b2) : 0.0;
    L.s2 = alpha[j - 1] * (1.0 / b1);
    L.c = evec[j] / beta[j - 1];
    L.psi = psi;
    hv_step(s, run.r, run.q, L);
    std::swap(run.r, run.q);
  }
  QED_HIP(hipGetLastError());
  QED_HIP(hipStreamSynchronize(stream()));
}

// ---------------------------------------------------------------------------------------
// band Lanczos (Freund), device vectors, following src_ed/Hamiltonian/Lanczos.hpp:214-395

struct VecPool {
  uint64_t n;
  std::vector<std::unique_ptr<DevBuf>> owned;
  std::vector<double*> free_list;
  explicit VecPool(uint64_t n_) : n(n_) {}
  double* get() {
    if (!free_list.empty()) {
      double* p = free_list.back();
      free_list.pop_back();
      return p;
    }
    owned.emplace_back(new DevBuf(n * sizeof(double)));
    return owned.back()->as<double>();
  }
  void put(double* p) {
    if (p) free_list.push_back(p);
  }
};

int band_lanczos(qed_sector& s, const double* phi, int p0, int M0, int max_iter_BL, double accur_deflation,
                 double accur_band_lanczos, std::vector<double>& evals, std::vector<double>& Q, double min_gap) {
  const uint64_t n = s.D;
  if (n == 0 || p0 == 0) return 0;
  if (M0 <= 0) M0 = (int)(14 * p0 * std::log(1.0 * n));
  if (M0 <= 1) fail("band Lanczos: too few iterations requested");
  int pc = p0;
  if (M0 > max_iter_BL) M0 = max_iter_BL;
  int M0p = (M0 / p0 + 1) * p0;
  M0 = M0p - pc;
  VecPool pool(n);
  std::vector<double*> v(M0p + 1, nullptr);
  std::vector<const double*> ph(p0);
  for (int i = 0; i < p0; ++i) ph[i] = phi + (uint64_t)i * n;
  for (int i = 0; i < p0; ++i) {
    v[i] = pool.get();
    QED_HIP(hipMemcpyAsync(v[i], ph[i], n * 8, hipMemcpyDeviceToDevice, stream()));
  }
  std::vector<double> t((size_t)M0 * M0, 0.0), P((size_t)p0 * M0, 0.0);
  auto T = [&](int i, int j) -> double& { return t[(size_t)j * M0 + i]; };
  std::vector<int> defl(M0, 0), I;
  double ev_old = 1e12;
  int j = 0;
  std::vector<double> tmp(kMaxMulti);
  while (j < M0) {
    // norm of v[j] and its overlaps with the start vectors in one pass
    std::vector<const double*> ys(p0 + 1);
    ys[0] = v[j];
    for (int k = 0; k < p0; ++k) ys[k + 1] = ph[k];
    std::vector<double> dd(p0 + 1);
    multi_dot(v[j], ys.data(), p0 + 1, n, dd.data());
    double z = std::sqrt(std::max(dd[0], 0.0));
    if (z < accur_deflation) {
      if (j >= pc) {
        I.push_back(j - pc);
        defl[j - pc] = 1;
      }
      pc--;
      if (pc == 0) break;
      pool.put(v[j]);
      for (int k = j; k < j + pc; ++k) v[k] = v[k + 1];
      v[j + pc] = nullptr;
      continue;
    }
    scal(1.0 / z, v[j], n);
    if (j >= pc) T(j, j - pc) = z;
    for (int k = 0; k < p0; ++k) P[(size_t)j * p0 + k] = dd[k + 1] / z;
    // orthogonalize the pending block against v[j]
    int nk = 0;
    std::vector<const double*> blk;
    std::vector<double*> blk_mut;
    for (int k = j + 1; k < j + pc; ++k) {
      blk.push_back(v[k]);
      blk_mut.push_back(v[k]);
      ++nk;
    }
    if (nk) {
      std::vector<double> zz(nk);
      multi_dot(v[j], blk.data(), nk, n, zz.data());
      multi_axpy_rev(zz.data(), v[j], blk_mut.data(), nk, n);
      for (int q = 0; q < nk; ++q) {
        int k = j + 1 + q;
        if (k >= pc) T(j, k - pc) = zz[q];
      }
    }
    double* w = pool.get();
    QED_HIP(hipMemsetAsync(w, 0, n * 8, stream()));
    hv(s, v[j], w);
    int k0 = 0;
    if (j > pc) {
      k0 = j - pc;
      if (defl[k0 - 1] == 0) {
        pool.put(v[k0 - 1]);
        v[k0 - 1] = nullptr;
      }
    }
    {
      std::vector<const double*> xs;
      std::vector<double> cs;
      for (int k = k0; k < j; ++k) {
        T(k, j) = T(j, k);
        xs.push_back(v[k]);
        cs.push_back(T(k, j));
      }
      multi_axpy(cs.data(), xs.data(), (int)xs.size(), w, n);
    }
    for (int k : I) {
      double ww = dot(v[k], w, n);
      axpy(-ww, v[k], w, n);
      T(k, j) = ww;
    }
    double ww = dot(v[j], w, n);
    axpy(-ww, v[j], w, n);
    T(j, j) = ww;
    for (int k : I) T(j, k) = T(k, j);
    v[j + pc] = w;
    if (j >= 4 * p0 && j % p0 == 0) {
      std::vector<double> Hpr((size_t)j * j), evs(j);
      for (int c = 0; c < j; ++c)
        for (int r = 0; r < j; ++r) Hpr[(size_t)c * j + r] = T(r, c);
      sym_eigen(j, Hpr.data(), evs.data(), false);
      double test = std::fabs(evs[0] - ev_old);
      ev_old = evs[0];
      // no_degenerate_BL (src_ed/Hamiltonian/Lanczos.hpp:368-370)
      if (min_gap > 0.0 && j > 1 && evs[1] - evs[0] < min_gap)
        fail("band Lanczos: the gap between the first two eigenvalues is smaller than " + std::to_string(min_gap));
      if (test < accur_band_lanczos) break;
    }
    ++j;
  }
  QED_HIP(hipStreamSynchronize(stream()));
  if (j == 0) return 0;
  std::vector<double> Hpr((size_t)j * j);
  for (int c = 0; c < j; ++c)
    for (int r = c; r < j; ++r) Hpr[(size_t)r * j + c] = T(r, c);
  evals.assign(j, 0.0);
  // Q = P U  (p0 x j)
  Q.assign(P.begin(), P.begin() + (size_t)p0 * j);
  sym_eigen_project(j, Hpr.data(), evals.data(), p0, Q.data());
  return j;
}

void lanczos_green(qed_sector& s, const double* psi_in, double accur_cf, int max_iter,
                   std::vector<double>& a, std::vector<double>& b) {
  const uint64_t n = s.D;
  DevBuf pb(n * 8), qb(n * 8);
  double* psi = pb.as<double>();
  double* q = qb.as<double>();
  QED_HIP(hipMemcpyAsync(psi, psi_in, n * 8, hipMemcpyDeviceToDevice, stream()));
  QED_HIP(hipMemsetAsync(q, 0, n * 8, stream()));
  a.clear();
  b.assign(1, 1.0);
  double prod = 1.0;
  while (prod > accur_cf && std::fabs(b.back()) > accur_cf && (int)a.size() < max_iter) {
    if (!a.empty()) k_swapscale<<<stream_blocks(n), 256, 0, stream()>>>(b.back(), psi, q, n);
    hv(s, psi, q);
    double z = dot(psi, q, n);
    a.push_back(z);
    double zz = axpy_nrm2(-z, psi, q, n);
    b.push_back(zz);
    prod *= std::fabs(zz);
  }
}


// ---------------------------------------------------------------------------------------
// Davidson-Liu for the K lowest states (src_ed/Hamiltonian/Davidson.hpp:38-230)

namespace {

// out_k[i] = sum_p C[p + m k] in_p[i], k < K (outputs distinct from inputs)
constexpr int kDavMax = 24;  // basis vectors of the Davidson subspace (3 K, K <= 8)

// out[k][i] = sum_p C[p + m k] in[p][i] for k < nout, with every input of index i read
// before any output of it is written: the outputs may be some of the inputs
__global__ __launch_bounds__(256) void k_dav_transform(PtrList in, int m, MutPtrList out, int nout,
                                                       const double* __restrict__ C, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    double v[kDavMax];
#pragma unroll
    for (int p = 0; p < kDavMax; ++p) v[p] = p < m ? in.p[p][i] : 0.0;
    for (int k = 0; k < nout; ++k) {
      double acc = 0.0;
#pragma unroll
      for (int p = 0; p < kDavMax; ++p)
        if (p < m) acc += C[p + m * k] * v[p];
      out.p[k][i] = acc;
    }
  }
}

// the diagonal of H as the factorized format reports it (the interaction part)
__device__ __forceinline__ double diag_interaction(const HvView& v, uint64_t I) {
  const uint32_t iu = (uint32_t)(I % v.du), id = (uint32_t)(I / v.du);
  const uint32_t su = v.bup[iu], sd = v.bdn[id];
  if (v.hubbard_uniform) return v.hub_U * (double)__popc(su & sd & v.hub_sites);
  double e = 0.0;
  const uint64_t w = (uint64_t)sd | ((uint64_t)su << 32);
  for (int k = 0; k < v.n_int; ++k)
    if ((w & v.int_mask[k]) == v.int_mask[k]) e += v.int_val[k];
  return e;
}

// the diagonal Davidson reads: the factorized format's (interaction part, on the fly) or a
// stored one (the symmetry-adapted and mixed-number sectors: the true diagonal of H, as the
// reference's other formats report it)
struct DavDiag {
  HvView v;
  const double* d;  // stored diagonal, or null
  __device__ __forceinline__ double operator()(uint64_t I) const { return d ? d[I] : diag_interaction(v, I); }
};

// correction vector of one unconverged root: c = (H x - mu x) / (mu - d + tiny)
__global__ void k_dav_correction(DavDiag dg, const double* __restrict__ hx, const double* __restrict__ x, double mu,
                                 double tiny, double* __restrict__ c, uint64_t n) {
  for (uint64_t I = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; I < n;
       I += (uint64_t)gridDim.x * blockDim.x)
    c[I] = (hx[I] - mu * x[I]) / (-dg(I) + mu + tiny);
}

// the order of find_lowest (src_util/vector_num.hpp:242-264): ascending values, and among
// equal values the later index first
__device__ __forceinline__ bool dav_before(double va, uint64_t ia, double vb, uint64_t ib) {
  return va < vb || (va == vb && ia > ib);
}

// block partials of the first diagonal entry after (pv, pi) in that order (all entries
// when have_prev is 0); a block with no candidate reports +inf
__global__ __launch_bounds__(256) void k_dav_next_lowest(DavDiag dg, uint64_t n, int have_prev, double pv, uint64_t pi,
                                                         double* __restrict__ part_v, uint64_t* __restrict__ part_i) {
  __shared__ double sv[256];
  __shared__ uint64_t si[256];
  double bv = INFINITY;
  uint64_t bi = 0;
  for (uint64_t I = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; I < n;
       I += (uint64_t)gridDim.x * blockDim.x) {
    const double d = dg(I);
    if (have_prev && !dav_before(pv, pi, d, I)) continue;
    if (dav_before(d, I, bv, bi)) {
      bv = d;
      bi = I;
    }
  }
  sv[threadIdx.x] = bv;
  si[threadIdx.x] = bi;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w && dav_before(sv[threadIdx.x + w], si[threadIdx.x + w], sv[threadIdx.x], si[threadIdx.x])) {
      sv[threadIdx.x] = sv[threadIdx.x + w];
      si[threadIdx.x] = si[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part_v[blockIdx.x] = sv[0];
    part_i[blockIdx.x] = si[0];
  }
}

// the K lowest diagonal entries in find_lowest's order, one device pass per entry
std::vector<uint64_t> lowest_diagonal(const qed_sector& s, const DavDiag& dg, int K) {
  const uint64_t n = s.D;
  const uint32_t nb = (uint32_t)std::min<uint64_t>(kMaxBlocks, std::max<uint64_t>(1, (n + 255) / 256));
  DevBuf pv(nb * sizeof(double)), pi(nb * sizeof(uint64_t));
  std::vector<double> hv_(nb);
  std::vector<uint64_t> hi_(nb);
  std::vector<uint64_t> out;
  double lv = 0.0;
  uint64_t li = 0;
  for (int k = 0; k < K; ++k) {
    k_dav_next_lowest<<<nb, 256, 0, stream()>>>(dg, n, k > 0, lv, li, pv.as<double>(), pi.as<uint64_t>());
    QED_HIP(hipMemcpyAsync(hv_.data(), pv.p, nb * sizeof(double), hipMemcpyDeviceToHost, stream()));
    QED_HIP(hipMemcpyAsync(hi_.data(), pi.p, nb * sizeof(uint64_t), hipMemcpyDeviceToHost, stream()));
    QED_HIP(hipStreamSynchronize(stream()));
    double bv = INFINITY;
    uint64_t bi = 0;
    for (uint32_t b = 0; b < nb; ++b)
      if (std::isfinite(hv_[b]) && (bv == INFINITY || hv_[b] < bv || (hv_[b] == bv && hi_[b] > bi))) {
        bv = hv_[b];
        bi = hi_[b];
      }
    if (!std::isfinite(bv)) fail("Davidson: fewer diagonal entries than requested states");
    out.push_back(bi);
    lv = bv;
    li = bi;
  }
  return out;
}

// out = C-weighted combinations of `in` (see k_dav_transform); C is m x nout column-major
void dav_transform(const std::vector<double*>& in, const std::vector<double>& C, const std::vector<double*>& out,
                   uint64_t n) {
  const int m = (int)in.size(), nout = (int)out.size();
  if (m > kDavMax || nout > kDavMax) fail("Davidson: subspace too large");
  PtrList li{};
  MutPtrList lo{};
  for (int p = 0; p < m; ++p) li.p[p] = in[p];
  for (int k = 0; k < nout; ++k) lo.p[k] = out[k];
  double* cd = red_scratch().as<double>() + (size_t)kMaxBlocks * kMaxMulti + 64;
  QED_HIP(hipMemcpyAsync(cd, C.data(), C.size() * sizeof(double), hipMemcpyHostToDevice, stream()));
  k_dav_transform<<<stream_blocks(n), 256, 0, stream()>>>(li, m, lo, nout, cd, n);
  QED_HIP(hipStreamSynchronize(stream()));
}

}  // namespace

// Davidson-Liu for the K lowest states, following src_ed/Hamiltonian/Davidson.hpp:38-230
// (start vectors on the K lowest diagonal entries, at most 3K basis vectors, the new basis
// made of the Ritz vectors, the basis vectors of the unconverged roots and their
// preconditioned residuals, Gram-Schmidt), with a memory layout for large sectors: the
// products H b are not kept (each is formed in a scratch vector, reduced against the basis
// and dropped), the residuals H x - mu x are formed from a fresh product of the Ritz vector,
// and the basis is transformed in place. Device memory: the K output vectors (the first K
// basis slots) plus 2K further slots and two scratch vectors, 3K + 2 vectors in all (14 for
// K = 4) instead of the reference's ~9K. The diagonal (preconditioner and start vectors) is
// recomputed per entry on factorized sectors; symmetry-adapted and mixed-number sectors
// store it (one more vector), since their diagonal gathers over the orbit's hops.
void davidson(qed_sector& s, int K, double accur, int max_iter, std::vector<double>& val, double* xout,
              int* niter, bool verb) {
  const uint64_t n = s.D;
  const double tiny = 1e-14;
  if ((uint64_t)K > n) K = (int)n;
  if (K < 1) fail("Davidson: no state requested");
  const int J = (int)std::min<uint64_t>(3 * (uint64_t)K, n);
  if (J > kDavMax) fail("Davidson: at most " + std::to_string(kDavMax / 3) + " states");
  val.assign(K, 0.0);
  {
    size_t fr = 0, tot = 0;
    QED_HIP(hipMemGetInfo(&fr, &tot));
    const double need = (double)(J - K + 2 + (s.factorized() ? 0 : 1)) * n * 8;
    if (need > (double)fr)
      fail("Davidson: " + std::to_string(J - K + 2) + " work vectors of the sector need " +
           std::to_string(need / 1e9) + " GB of device memory, " + std::to_string(fr / 1e9) + " GB free");
  }
  std::vector<DevBuf> own;
  std::vector<double*> slot(J);
  for (int k = 0; k < K; ++k) slot[k] = xout + (uint64_t)k * n;
  for (int k = K; k < J; ++k) {
    own.emplace_back(n * 8);
    slot[k] = own.back().as<double>();
  }
  DevBuf tb(n * 8), ub(n * 8);
  double* t = tb.as<double>();
  double* u = ub.as<double>();
  const uint32_t sb = stream_blocks(n);

  if (verb)
    printf("\nDavidson method for %d vectors in sector (%d, %d), dim = %llu\n", K, s.nup, s.ndn,
           (unsigned long long)n);
  DevBuf dstore;
  DavDiag dg{s.factorized() ? view(s) : HvView{}, nullptr};
  if (!s.factorized()) {
    dstore.alloc(n * 8);
    k_zero<<<sb, 256, 0, stream()>>>(dstore.as<double>(), n);
    sector_diagonal(s, dstore.as<double>());
    dg.d = dstore.as<double>();
  }
  const std::vector<uint64_t> low = lowest_diagonal(s, dg, K);
  const double one = 1.0;
  for (int k = 0; k < K; ++k) {
    k_zero<<<sb, 256, 0, stream()>>>(slot[k], n);
    QED_HIP(hipMemcpyAsync(slot[k] + low[k], &one, 8, hipMemcpyHostToDevice, stream()));
  }
  int m = K;
  // bhb(i, j) = (H b_j)[low_i]
  std::vector<double> bhb((size_t)m * m);
  for (int j = 0; j < m; ++j) {
    k_zero<<<sb, 256, 0, stream()>>>(u, n);
    hv(s, slot[j], u);
    for (int i = 0; i < m; ++i)
      QED_HIP(hipMemcpyAsync(&bhb[(size_t)j * m + i], u + low[i], 8, hipMemcpyDeviceToHost, stream()));
  }
  QED_HIP(hipStreamSynchronize(stream()));

  int iter;
  for (iter = 0; iter < max_iter; ++iter) {
    std::vector<double> a(bhb), mu(m);
    sym_eigen(m, a.data(), mu.data(), true);  // column k of a: eigenvector k
    std::vector<double*> basis(slot.begin(), slot.begin() + m);
    // residual norms |H x_k - mu_k x_k| with x_k = sum_p a_pk b_p formed in t
    std::vector<int> unconv;
    double res_last = 0.0;
    for (int k = 0; k < K; ++k) {
      std::vector<double> ck(a.begin() + (size_t)k * m, a.begin() + (size_t)(k + 1) * m);
      dav_transform(basis, ck, {t}, n);
      k_zero<<<sb, 256, 0, stream()>>>(u, n);
      hv(s, t, u);
      res_last = axpy_nrm2(-mu[k], t, u, n);
      if (res_last > accur) unconv.push_back(k);
    }
    if (verb && iter % 10 == 0) {
      printf("--> iteration %d, evalue = %.12g,\tresidual = %.12g\n", iter, mu[0], res_last);
      fflush(stdout);
    }
    for (int k = 0; k < K; ++k) val[k] = mu[k];
    const int Q = (int)unconv.size();
    // the basis in place: slots 0..K-1 <- Ritz vectors, then the unconverged roots' own
    // basis vectors
    std::vector<double> C((size_t)m * (K + Q), 0.0);
    for (int k = 0; k < K; ++k)
      for (int p = 0; p < m; ++p) C[p + (size_t)m * k] = a[(size_t)k * m + p];
    for (int q = 0; q < Q; ++q) C[unconv[q] + (size_t)m * (K + q)] = 1.0;
    dav_transform(basis, C, std::vector<double*>(slot.begin(), slot.begin() + K + Q), n);
    if (Q == 0) break;
    // preconditioned residuals of the unconverged roots
    for (int q = 0; q < Q; ++q) {
      const int k = unconv[q];
      k_zero<<<sb, 256, 0, stream()>>>(u, n);
      hv(s, slot[k], u);
      k_dav_correction<<<sb, 256, 0, stream()>>>(dg, u, slot[k], mu[k], tiny, slot[K + Q + q], n);
    }
    // Gram-Schmidt in the reference's order (vectors below tiny are removed)
    std::vector<double*> b(slot.begin(), slot.begin() + K + 2 * Q);
    for (size_t i = 0; i < b.size(); ++i) {
      const double z = nrm2(b[i], n);
      if (z < tiny) {
        std::swap(b[i], b.back());
        b.pop_back();
        --i;
        continue;
      }
      scal(1.0 / z, b[i], n);
      const int cnt = (int)b.size() - (int)(i + 1);
      if (cnt > 0) {
        std::vector<const double*> ys(b.begin() + i + 1, b.end());
        std::vector<double> zz(cnt);
        multi_dot(b[i], ys.data(), cnt, n, zz.data());
        std::vector<double*> ym(b.begin() + i + 1, b.end());
        multi_axpy_rev(zz.data(), b[i], ym.data(), cnt, n);
      }
    }
    // keep the slots in basis order (a removed vector's slot moves to the end)
    {
      std::vector<double*> rest;
      for (double* p : slot)
        if (std::find(b.begin(), b.end(), p) == b.end()) rest.push_back(p);
      for (size_t i = 0; i < b.size(); ++i) slot[i] = b[i];
      for (size_t i = 0; i < rest.size(); ++i) slot[b.size() + i] = rest[i];
    }
    if ((int)b.size() == K) break;
    m = (int)b.size();
    // bhb(i, k) = <b_i, H b_k> for i >= k (the reference's pairing), one product at a time
    bhb.assign((size_t)m * m, 0.0);
    for (int k = 0; k < m; ++k) {
      k_zero<<<sb, 256, 0, stream()>>>(u, n);
      hv(s, slot[k], u);
      std::vector<const double*> ys(slot.begin() + k, slot.begin() + m);
      std::vector<double> zz(m - k);
      multi_dot(u, ys.data(), m - k, n, zz.data());
      for (int i = k; i < m; ++i) {
        bhb[(size_t)k * m + i] = zz[i - k];
        bhb[(size_t)i * m + k] = zz[i - k];
      }
    }
  }
  if (iter == max_iter) fail("Davidson method failed to converge!");
  *niter = iter;
  // the states are in the first K slots, which are the output vectors unless Gram-Schmidt
  // removed one of them: then exchange contents (through t) until each is in place
  for (int k = 0; k < K; ++k) {
    double* want = xout + (uint64_t)k * n;
    if (slot[k] == want) continue;
    const int j = (int)(std::find(slot.begin(), slot.end(), want) - slot.begin());
    QED_HIP(hipMemcpyAsync(t, want, n * 8, hipMemcpyDeviceToDevice, stream()));
    QED_HIP(hipMemcpyAsync(want, slot[k], n * 8, hipMemcpyDeviceToDevice, stream()));
    QED_HIP(hipMemcpyAsync(slot[k], t, n * 8, hipMemcpyDeviceToDevice, stream()));
    std::swap(slot[k], slot[j]);
  }
  QED_HIP(hipStreamSynchronize(stream()));
}

}  // namespace qed

using namespace qed;

// ---- the allocation-free Lanczos ground state --------------------------------------------
namespace {

// Device memory of qed_lanczos_gs_noalloc, one copy per GPU for the life of the process:
// the two recurrence vectors of a sector of at most kNoAllocMaxDim amplitudes, the BLAS-1
// parts and scalars of the steps (34.1 MB in all).
constexpr uint64_t kNoAllocMaxDim = 1ull << 21;
constexpr size_t kNoAllocDoubles = 2 * kNoAllocMaxDim + kLzWork;
static __device__ __align__(256) double scratch[kNoAllocDoubles];

constexpr int kMaxDevices = 64;
double* g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the current GPU, looked up on the first call there
// (the name is a host-side stand-in and must not be passed to a kernel). Caller holds the
// library mutex.
double* noalloc_scratch() {
  int dev = 0;
  QED_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) fail("qed_lanczos_gs_noalloc: device index out of range");
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    QED_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) fail("qed_lanczos_gs_noalloc: no device address for the scratch array");
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  return g_scratch_ptr[dev];
}

}  // namespace

extern "C" {

int qed_lanczos_gs(qed_sector* s, double accur, int max_iter, double* psi, double* E0, int* niter,
                   double* alpha, double* beta) {
  std::lock_guard<std::recursive_mutex> lk(lib_mutex());
  return guard([&] {
    std::vector<double> a, b;
    lanczos_gs(*s, accur, max_iter, psi, E0, niter, &a, &b);
    if (alpha) std::copy(a.begin(), a.end(), alpha);
    if (beta) std::copy(b.begin(), b.end(), beta);
  });
}

int qed_lanczos_gs_noalloc(qed_sector* s, double accur, int max_iter, double* psi, double* E0, int* niter,
                           double* alpha, double* beta) {
  std::lock_guard<std::recursive_mutex> lk(lib_mutex());
  return guard([&] {
    if (s->D > kNoAllocMaxDim)
      fail("qed_lanczos_gs_noalloc: sector dimension " + std::to_string(s->D) + " exceeds the scratch limit of " +
           std::to_string(kNoAllocMaxDim));
    double* base = noalloc_scratch();
    const LanczosWork ws{base, base + kNoAllocMaxDim, base + 2 * kNoAllocMaxDim};
    std::vector<double> a, b;
    lanczos_gs(*s, accur, max_iter, psi, E0, niter, &a, &b, &ws);
    if (alpha) std::copy(a.begin(), a.end(), alpha);
    if (beta) std::copy(b.begin(), b.end(), beta);
  });
}

// Measurement: average milliseconds per Lanczos step of the eigenvalue pass from psi
// (normalized), `steps` steps each (no stopping test), HIP events on the library stream:
// ms[0] the step of lanczos_gs (product with the scale and dot folded in, then axpy + norm),
// ms[1] the separate passes (scale, product, dot, axpy + norm), both with a host round trip
// per step.
int qed_lanczos_steps_timed(qed_sector* s, const double* psi, int steps, double* ms) {
  std::lock_guard<std::recursive_mutex> lk(lib_mutex());
  return guard([&] {
    const uint64_t n = s->D;
    LanczosRun run(*s, nullptr);
    double* r = run.r;
    double* q = run.q;
    hipEvent_t e0, e1;
    QED_HIP(hipEventCreate(&e0));
    QED_HIP(hipEventCreate(&e1));
    LanczosLease host(false);
    auto reset = [&] {
      run.start(psi);
      QED_HIP(hipStreamSynchronize(stream()));
    };
    reset();
    run.step();
    reset();
    {
      QED_HIP(hipEventRecord(e0, stream()));
      for (int k = 0; k < steps; ++k) {
        run.step();
        run.fetch(host->pin);
        QED_HIP(hipStreamSynchronize(stream()));
      }
      QED_HIP(hipEventRecord(e1, stream()));
      QED_HIP(hipEventSynchronize(e1));
      float t = 0.f;
      QED_HIP(hipEventElapsedTime(&t, e0, e1));
      ms[0] = t / std::max(1, steps);
    }
    reset();
    QED_HIP(hipEventRecord(e0, stream()));
    double bprev = 0.0;
    for (int k = 0; k < steps; ++k) {
      if (k > 0) scal2(1.0 / bprev, r, -bprev, q, n);
      hv(*s, r, q);
      std::swap(r, q);
      const double a = dot(q, r, n);
      bprev = axpy_nrm2(-a, q, r, n);
    }
    QED_HIP(hipEventRecord(e1, stream()));
    QED_HIP(hipEventSynchronize(e1));
    float t = 0.f;
    QED_HIP(hipEventElapsedTime(&t, e0, e1));
    ms[1] = t / std::max(1, steps);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
  });
}

int qed_lanczos_green(qed_sector* s, const double* psi, double accur_cf, int max_iter, double* a,
                      double* b, int* n) {
  std::lock_guard<std::recursive_mutex> lk(lib_mutex());
  return guard([&] {
    std::vector<double> av, bv;
    lanczos_green(*s, psi, accur_cf, max_iter, av, bv);
    std::copy(av.begin(), av.end(), a);
    std::copy(bv.begin(), bv.end(), b);
    *n = (int)av.size();
  });
}

int qed_band_lanczos(qed_sector* s, const double* phi, int p, int M0, int max_iter_BL,
                     double accur_deflation, double accur_band_lanczos, double* evals, double* Q,
                     int cap, int* M) {
  std::lock_guard<std::recursive_mutex> lk(lib_mutex());
  return guard([&] {
    std::vector<double> e, q;
    int m = band_lanczos(*s, phi, p, M0, max_iter_BL, accur_deflation, accur_band_lanczos, e, q);
    if (m > cap) fail("band Lanczos: output capacity too small");
    *M = m;
    std::copy(e.begin(), e.end(), evals);
    std::copy(q.begin(), q.end(), Q);
  });
}

int qed_davidson(qed_sector* s, int k, double accur, int max_iter, double* evals, double* psi,
                 int* niter) {
  std::lock_guard<std::recursive_mutex> lk(lib_mutex());
  return guard([&] {
    std::vector<double> e;
    davidson(*s, k, accur, max_iter, e, psi, niter, verbose_ed());
    std::copy(e.begin(), e.end(), evals);
  });
}

// Achievable read-modify-write bandwidth: reps launches of y += 0.5 x over n doubles (n
// even, 16-byte aligned vectors), timed with events; *ms = milliseconds per launch.
int qed_stream_rmw_timed(const double* x, double* y, uint64_t n, int reps, double* ms) {
  std::lock_guard<std::recursive_mutex> lk(lib_mutex());
  return guard([&] {
    if (n % 2) fail("stream: n must be even");
    const uint64_t n2 = n / 2;
    const uint32_t grid = (uint32_t)std::min<uint64_t>((n2 + 255) / 256, (uint64_t)device_cu_count() * 64);
    auto run = [&] {
      k_stream_rmw<<<grid, 256, 0, stream()>>>(reinterpret_cast<const double2*>(x), reinterpret_cast<double2*>(y), n2);
    };
    run();
    hipEvent_t e0, e1;
    QED_HIP(hipEventCreate(&e0));
    QED_HIP(hipEventCreate(&e1));
    QED_HIP(hipEventRecord(e0, stream()));
    for (int r = 0; r < std::max(1, reps); ++r) run();
    QED_HIP(hipEventRecord(e1, stream()));
    QED_HIP(hipEventSynchronize(e1));
    float t = 0.f;
    QED_HIP(hipEventElapsedTime(&t, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    QED_HIP(hipGetLastError());
    *ms = (double)t / std::max(1, reps);
  });
}

int qed_blas_dot(const double* x, const double* y, uint64_t n, double* out) {
  std::lock_guard<std::recursive_mutex> lk(lib_mutex());
  return guard([&] { *out = dot(x, y, n); });
}

int qed_util_tridiag_eigen(int n, double* d, const double* e, double* z) {
  return guard([&] { tridiag_eigen(n, d, e, z); });
}

int qed_util_sym_eigen(int n, double* a, double* w, int vectors) {
  return guard([&] { sym_eigen(n, a, w, vectors != 0); });
}

}  // extern "C"
