// Symmetry-adapted (mixed) basis of an Abelian point group for one (N_up, N_down) sector
// and one irreducible representation, and its Hamiltonian on the device.
//
// The group (src_ed/symmetry_group.cpp:183-352) is generated by commuting signed site
// permutations; with bath_irrep the bath orbitals are not permuted but carry a phase label
// per element. A basis state is the representative (smallest 64-bit state, up in the low
// word) of its orbit that survives the projection onto the irrep
// (Representative, src_ed/symmetry_group.cpp:428-454; ED_mixed_basis,
// src_ed/ED_basis.cpp:185-361). The Hamiltonian's elements follow HS_one_body_operator
// (src_ed/Operators/HS_one_body_operator.hpp:8-40): a hop from basis state I to a state
// whose representative is J carries the group phase of that representative, the fermionic
// sign and sqrt(length(I) / length(J)).
//
// Device layout: the factorized sector of the same (N_up, N_down) supplies the half bases,
// the hop tables (ELL) and the diagonal; one table over all its D factorized states holds,
// for each state, the index of its representative in the mixed basis and the sign of the
// group element that maps it there (or "vanishes"). The product is then a gather per
// basis state: its factorized hops, each looked up in that table. Only groups whose
// characters are real (generators of order <= 2) are built: the phases are then signs and
// the vectors stay real.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <vector>

#include "../../include/qed.h"
#include "qed_sector.hpp"

namespace qed {

namespace {

constexpr int kMaxGroup = 16;   // group elements
constexpr int kMaxOrb = 32;     // orbitals per spin
constexpr uint32_t kVanish = 0xffffffffu;
// codes of a sector with fewer than 2^27 basis states also carry log2 of the target's
// orbit length (bits 27-29; orbit lengths are powers of two for real groups), so that a
// hop needs no lookup of the target's length
constexpr uint32_t kPackedMax = 1u << 27;
constexpr uint32_t kIndexMask = kPackedMax - 1u;

// one group element as the device reads it: site images (i < L), the bath phase labels
// (i >= L, in units of 2 pi / g), and per site the sites above it that it puts below its
// image (the inversions whose parity is the fermionic sign of the permutation)
struct GroupElem {
  uint8_t img[kMaxOrb];
  uint8_t bath[kMaxOrb];
  uint32_t inv[kMaxOrb];
  int phi2;  // 2 phi(element, irrep): the irrep's phase in units of pi / g
};

struct GroupDev {
  GroupElem e[kMaxGroup];
  int g, L, N;
};

struct MixedTables {
  std::shared_ptr<qed_sector> base;  // the factorized sector of the same particle numbers
  DevBuf full_of;   // per basis state: its factorized index (u32)
  DevBuf len;       // per basis state: orbit length (u32)
  DevBuf code;      // per factorized state: basis index of its representative | sign << 31
                    // (packed: | log2 of its orbit length << 27)
  bool packed = false;
  std::vector<uint64_t> states;  // the basis as 64-bit states (up | down << 32), ascending
  int g = 1, irrep = 0;
  std::vector<std::vector<int>> elems;  // the group elements (site images, bath labels)
  std::vector<int> phi;                 // phi(a, b), g x g, units of 2 pi / g
};

// the image of one spin's bit string under element E and its phase (units of pi / g)
__device__ __forceinline__ uint32_t apply_word(const GroupElem& E, int L, int N, int g, uint32_t b, int* phase) {
  uint32_t bp = 0, par = 0;
  for (int i = 0; i < L; ++i)
    if (b >> i & 1u) {
      bp |= 1u << E.img[i];
      par += __popc(E.inv[i] & b);
    }
  for (int i = L; i < N; ++i)
    if (b >> i & 1u) {
      *phase += 2 * E.bath[i];
      bp |= 1u << i;
    }
  *phase += (int)(par & 1u) * g;
  return bp;
}

// Representative of state (up, dn): its 64-bit representative, phase and orbit length
// (0: the projection onto the irrep annihilates the state)
__device__ __forceinline__ void representative(const GroupDev& G, uint32_t up, uint32_t dn, uint64_t* rep, int* phase,
                                               int* length) {
  const uint64_t s = (uint64_t)up | ((uint64_t)dn << 32);
  int h = 1;
  uint64_t best = s;
  int bph = 0;
  for (int el = 1; el < G.g; ++el) {
    int ph = 0;
    const uint32_t u2 = apply_word(G.e[el], G.L, G.N, G.g, up, &ph);
    const uint32_t d2 = apply_word(G.e[el], G.L, G.N, G.g, dn, &ph);
    ph = (ph + G.e[el].phi2) % (2 * G.g);
    const uint64_t t = (uint64_t)u2 | ((uint64_t)d2 << 32);
    if (t == s) {
      ++h;
      if (ph != 0 && (2 * G.g) % ph == 0) {
        *rep = s;
        *phase = 0;
        *length = 0;
        return;
      }
    }
    if (t < best) {
      best = t;
      bph = ph;
    }
  }
  *rep = best;
  *phase = bph;
  *length = G.g / h;
}

// pass 1: for every factorized state, whether it is a basis state (its own representative)
__global__ void k_mixed_flags(GroupDev G, const uint32_t* __restrict__ bup, const uint32_t* __restrict__ bdn,
                              uint32_t du, uint64_t D, uint8_t* __restrict__ is_rep, uint8_t* __restrict__ len) {
  for (uint64_t f = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; f < D; f += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t up = bup[f % du], dn = bdn[f / du];
    uint64_t rep;
    int ph, length;
    representative(G, up, dn, &rep, &ph, &length);
    is_rep[f] = (length > 0 && rep == ((uint64_t)up | ((uint64_t)dn << 32))) ? 1 : 0;
    len[f] = (uint8_t)length;
  }
}

// pass 2: for every factorized state, the basis index of its representative and the sign
// (packed: and log2 of the orbit length, which is the representative's)
__global__ void k_mixed_codes(GroupDev G, const uint32_t* __restrict__ bup, const uint32_t* __restrict__ bdn,
                              uint32_t du, uint64_t D, int nup, int ndn, const uint32_t* __restrict__ binom,
                              const uint32_t* __restrict__ index_of, bool packed, uint32_t* __restrict__ code) {
  for (uint64_t f = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; f < D; f += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t up = bup[f % du], dn = bdn[f / du];
    uint64_t rep;
    int ph, length;
    representative(G, up, dn, &rep, &ph, &length);
    if (length == 0) {
      code[f] = kVanish;
      continue;
    }
    const uint64_t fr = (uint64_t)cns_rank((uint32_t)rep, binom) +
                        (uint64_t)du * cns_rank((uint32_t)(rep >> 32), binom);
    const uint32_t J = index_of[fr];
    // real characters: the phase is 0 or g (units of pi / g)
    const uint32_t lb = packed ? (uint32_t)(31 - __clz(length)) << 27 : 0u;
    code[f] = J == kVanish ? kVanish : (J | lb | (ph != 0 ? 0x80000000u : 0u));
    (void)nup;
    (void)ndn;
  }
}

// the basis index and orbit length of a code (not kVanish)
template <bool PACKED>
__device__ __forceinline__ uint32_t code_target(uint32_t c, const uint32_t* __restrict__ len, uint32_t* lenJ) {
  if (PACKED) {
    const uint32_t J = c & kIndexMask;
    *lenJ = 1u << ((c >> 27) & 7u);
    return J;
  }
  const uint32_t J = c & 0x7fffffffu;
  *lenJ = len[J];
  return J;
}

// y[I] += sum_J H[I, J] x[J], one thread per basis state: the diagonal of the factorized
// state, and every factorized hop of it mapped to its representative. A hop is a chain of
// three loads (table, code, x), and their latency and the vector units' address rate bound
// the kernel: kHops chains are in flight at a time, and the amplitudes are read from LDS.
// Packed orbit lengths are powers of two, so that sqrt(length(I) / length(J)) is one of 16
// values and not a division and a square root per hop. 2x7 sites, half filled, two mirrors
// (2,945,056 states): 329 us one hop at a time, 217 us by groups, 174 us with the
// amplitudes in LDS.
constexpr int kHops = 8;  // the tables' widths are multiples of it
// amplitudes (both spins) held in LDS, 4 KB: up to 127 bonds per spin, all pairs of 16
// orbitals; more are read from memory
constexpr uint32_t kLdsVals = 512;

template <bool PACKED>
__device__ __forceinline__ void hop_group(const uint32_t* e, const uint32_t* c, const double* vals,
                                          const uint32_t* __restrict__ len, const double* fac, uint32_t lin,
                                          const double* __restrict__ x, double& acc) {
  double xv[kHops], w[kHops];
#pragma unroll
  for (int q = 0; q < kHops; ++q) {
    uint32_t J = 0;
    w[q] = 0.0;
    if constexpr (PACKED) {
      J = c[q] == kVanish ? 0u : c[q] & kIndexMask;
      w[q] = fac[lin - ((c[q] >> 27) & 7u)];
    } else {
      J = c[q] == kVanish ? 0u : c[q] & 0x7fffffffu;
      w[q] = sqrt((double)lin / (double)len[J]);
    }
    xv[q] = x[J];
  }
#pragma unroll
  for (int q = 0; q < kHops; ++q) {
    const double a = vals[e[q] >> kEllTargetBits];
    const double t = a * w[q] * xv[q];
    if (a != 0.0 && c[q] != kVanish) acc += (c[q] >> 31) ? -t : t;
  }
}

template <bool PACKED, bool VLDS, int EP, class... Step>
__global__ __launch_bounds__(256) void k_hv_mixed(HvView v, const uint32_t* __restrict__ up_ell, uint32_t Wu,
                                                  const uint32_t* __restrict__ dn_ell, uint32_t Wd,
                                                  const uint32_t* __restrict__ full_of, const uint32_t* __restrict__ len,
                                                  const uint32_t* __restrict__ code, uint32_t n, uint32_t dn_nvals,
                                                  const double* __restrict__ x, double* __restrict__ y, Step... step) {
  const LzStep& lz = step_of<LzStep>(step...);
  constexpr uint32_t mask = (1u << kEllTargetBits) - 1u;
  __shared__ double fac[PACKED ? 16 : 1];  // fac[t] = sqrt(2^(t - 7))
  __shared__ double vals[VLDS ? kLdsVals : 1];
  if (PACKED && threadIdx.x < 16) fac[threadIdx.x] = sqrt((double)(1u << threadIdx.x) / 128.0);
  const double *uv = v.up_vals, *dv = v.dn_vals;
  if constexpr (VLDS) {  // up-spin amplitudes, then down-spin
    for (uint32_t i = threadIdx.x; i < v.up_nvals; i += 256) vals[i] = v.up_vals[i];
    for (uint32_t i = threadIdx.x; i < dn_nvals; i += 256) vals[v.up_nvals + i] = v.dn_vals[i];
    uv = vals;
    dv = vals + v.up_nvals;
  }
  __syncthreads();
  double2 sc = make_double2(0.0, 0.0);
  double dot = 0.0;
  if constexpr (EP != 0) sc = lz_scalars(lz);
  for (uint32_t I = blockIdx.x * blockDim.x + threadIdx.x; I < n; I += gridDim.x * blockDim.x) {
    const uint32_t f = full_of[I];
    const uint32_t iu = f % v.du, id = f / v.du;
    // packed: index of sqrt(length(I) / 1), from which a target's log2 is taken away
    const uint32_t lin = PACKED ? 7u + (31u - (uint32_t)__clz(len[I])) : len[I];
    double acc = (v.diag_up[iu] + v.diag_dn[id] + density_density(v, v.bup[iu], v.bdn[id])) * x[I];
    const uint32_t* crow = code + (uint64_t)v.du * id;
    for (uint32_t k = 0; k < Wu; k += kHops) {
      uint32_t e[kHops], c[kHops];
#pragma unroll
      for (int q = 0; q < kHops; ++q) e[q] = up_ell[(uint64_t)(k + q) * v.du + iu];
#pragma unroll
      for (int q = 0; q < kHops; ++q) c[q] = crow[e[q] & mask];
      hop_group<PACKED>(e, c, uv, len, fac, lin, x, acc);
    }
    const uint32_t dcnt = v.dn_ptr[id + 1] - v.dn_ptr[id];
    for (uint32_t k = 0; k < dcnt; k += kHops) {
      uint32_t e[kHops], c[kHops];
#pragma unroll
      for (int q = 0; q < kHops; ++q) e[q] = dn_ell[(uint64_t)id * Wd + k + q];
#pragma unroll
      for (int q = 0; q < kHops; ++q) c[q] = code[iu + (uint64_t)v.du * (e[q] & mask)];
      hop_group<PACKED>(e, c, dv, len, fac, lin, x, acc);
    }
    lz_update<EP>(lz, sc, acc, x[I], y + I, EP == 2 ? lz.psi + I : nullptr, dot);
  }
  if constexpr (EP == 1) {
    __shared__ double red[4];
    dot = block_sum(dot, red);
    if (threadIdx.x == 0) lz.pa[blockIdx.x] = dot;
  }
}

// d[I] += H[I, I]: the factorized state's diagonal and the hops that land on a member of
// the state's own orbit (their target's representative is I)
template <bool PACKED>
__global__ __launch_bounds__(256) void k_diag_mixed(HvView v, const uint32_t* __restrict__ up_ell, uint32_t Wu,
                                                    const uint32_t* __restrict__ dn_ell, uint32_t Wd,
                                                    const uint32_t* __restrict__ full_of, const uint32_t* __restrict__ len,
                                                    const uint32_t* __restrict__ code, uint32_t n, double* __restrict__ d) {
  constexpr uint32_t mask = (1u << kEllTargetBits) - 1u;
  for (uint32_t I = blockIdx.x * blockDim.x + threadIdx.x; I < n; I += gridDim.x * blockDim.x) {
    const uint32_t f = full_of[I];
    const uint32_t iu = f % v.du, id = f / v.du;
    double acc = v.diag_up[iu] + v.diag_dn[id] + density_density(v, v.bup[iu], v.bdn[id]);
    for (uint32_t k = 0; k < Wu; ++k) {
      const uint32_t e = up_ell[(uint64_t)k * v.du + iu];
      const double a = v.up_vals[e >> kEllTargetBits];
      if (a == 0.0) continue;
      const uint32_t c = code[(e & mask) + (uint64_t)v.du * id];
      if (c == kVanish) continue;
      uint32_t lj;
      if (code_target<PACKED>(c, len, &lj) != I) continue;
      acc += (c >> 31) ? -a : a;
    }
    for (uint32_t k = 0; k < Wd; ++k) {
      const uint32_t e = dn_ell[(uint64_t)id * Wd + k];
      const double a = v.dn_vals[e >> kEllTargetBits];
      if (a == 0.0) continue;
      const uint32_t c = code[iu + (uint64_t)v.du * (e & mask)];
      if (c == kVanish) continue;
      uint32_t lj;
      if (code_target<PACKED>(c, len, &lj) != I) continue;
      acc += (c >> 31) ? -a : a;
    }
    d[I] += acc;
  }
}

// Destroy of one orbital (src_ed/ED_basis.cpp:60-77) from a basis state of the source
// sector: the target basis index, the sign (group element and Jordan-Wigner parity of
// the 64-bit state's bits below the orbital), or false
struct MixedSide {
  const uint32_t* bup;   // half bases of the factorized sector
  const uint32_t* bdn;
  uint32_t du;
  const uint32_t* full_of;  // basis state -> factorized index
  const uint32_t* len;      // basis state -> orbit length
  const uint32_t* code;     // factorized state -> representative index | sign << 31
  bool packed;              // codes carry log2 of the orbit length
};

__device__ __forceinline__ bool destroy_one(const MixedSide& src, const MixedSide& dst, const uint32_t* binom,
                                            uint32_t I, int orb, int spin, uint32_t* J, bool* neg) {
  const uint32_t f = src.full_of[I];
  const uint32_t u = src.bup[f % src.du], d = src.bdn[f / src.du];
  const uint32_t bit = 1u << orb;
  uint32_t u2 = u, d2 = d;
  int par;
  if (spin == 0) {
    if (!(u & bit)) return false;
    u2 = u ^ bit;
    par = __popc(u & (bit - 1u));
  } else {
    if (!(d & bit)) return false;
    d2 = d ^ bit;
    par = __popc(u) + __popc(d & (bit - 1u));
  }
  const uint64_t f2 = (uint64_t)cns_rank(u2, binom) + (uint64_t)dst.du * cns_rank(d2, binom);
  const uint32_t c = dst.code[f2];
  if (c == kVanish) return false;
  *J = dst.packed ? (c & kIndexMask) : (c & 0x7fffffffu);
  *neg = ((c >> 31) != 0) != ((par & 1) != 0);
  return true;
}

// y += c_o x: the destruction operator of the symmetric orbital o (coefficients coef over
// the sites) from the source basis (x) to the target basis (y), from the source side as
// the reference builds it (destruction_operator.cpp:14-33), accumulated with atomics
__global__ void k_mixed_destroy(MixedSide src, MixedSide dst, const uint32_t* __restrict__ binom, uint32_t n_src,
                                int n_sites, const double* __restrict__ coef, int spin, const double* __restrict__ x,
                                double* __restrict__ y) {
  for (uint32_t I = blockIdx.x * blockDim.x + threadIdx.x; I < n_src; I += gridDim.x * blockDim.x) {
    const double xi = x[I];
    if (xi == 0.0) continue;
    const double li = (double)src.len[I];
    for (int a = 0; a < n_sites; ++a) {
      const double ca = coef[a];
      if (ca == 0.0) continue;
      uint32_t J;
      bool neg;
      if (!destroy_one(src, dst, binom, I, a, spin, &J, &neg)) continue;
      const double X = ca * sqrt(li / (double)dst.len[J]);
      atomicAdd(y + J, (neg ? -X : X) * xi);
    }
  }
}

// y += c^dagger_o x, the transpose of the destruction operator from the target (y, one
// more particle) to the source (x), built from the target side: a gather
__global__ void k_mixed_create(MixedSide tgt, MixedSide src, const uint32_t* __restrict__ binom, uint32_t n_tgt,
                               int n_sites, const double* __restrict__ coef, int spin, const double* __restrict__ x,
                               double* __restrict__ y) {
  for (uint32_t J = blockIdx.x * blockDim.x + threadIdx.x; J < n_tgt; J += gridDim.x * blockDim.x) {
    const double lj = (double)tgt.len[J];
    double acc = 0.0;
    for (int a = 0; a < n_sites; ++a) {
      const double ca = coef[a];
      if (ca == 0.0) continue;
      uint32_t I;
      bool neg;
      if (!destroy_one(tgt, src, binom, J, a, spin, &I, &neg)) continue;
      const double X = ca * sqrt(lj / (double)src.len[I]) * x[I];
      acc += neg ? -X : X;
    }
    y[J] += acc;
  }
}

// ---- the group on the host (src_ed/symmetry_group.cpp:36-100, 183-352) ---------------

struct HostGroup {
  int N = 0, L = 0, g = 1;
  std::vector<std::vector<int>> e;  // elements (N entries: site images, bath labels)
  std::vector<int> dims;            // orders of the generators
};

HostGroup build_group(int N, int n_sites, const std::vector<std::vector<int>>& gens_in, bool bath_irrep) {
  HostGroup G;
  G.N = N;
  std::vector<std::vector<int>> gens = gens_in;
  if (gens.empty()) {
    bath_irrep = false;
    gens.assign(1, std::vector<int>(N));
    for (int i = 0; i < N; ++i) gens[0][i] = i;
  }
  G.L = bath_irrep ? n_sites : N;
  const int L = G.L;
  auto identity = [&] {
    std::vector<int> v(N, 0);
    for (int i = 0; i < L; ++i) v[i] = i;
    return v;
  };
  auto product = [&](const std::vector<int>& x, const std::vector<int>& y, int g) {
    std::vector<int> v(N, 0);
    for (int i = 0; i < L; ++i) v[i] = x[y[i]];
    for (int i = L; i < N; ++i) v[i] = g ? (x[i] + y[i]) % g : 0;
    return v;
  };
  for (size_t k = 0; k < gens.size(); ++k) {
    if ((int)gens[k].size() != N) fail("generator " + std::to_string(k + 1) + " should have " + std::to_string(N) + " elements");
    std::vector<int> seen(L, 0);
    for (int i = 0; i < L; ++i) {
      if (gens[k][i] < 0 || gens[k][i] >= L || seen[gens[k][i]]) fail("generator " + std::to_string(k + 1) + " is not valid!");
      seen[gens[k][i]] = 1;
    }
  }
  for (size_t i = 0; i < gens.size(); ++i)
    for (size_t j = 0; j < i; ++j) {
      auto p1 = product(gens[i], gens[j], 1), p2 = product(gens[j], gens[i], 1);
      for (int q = 0; q < L; ++q)
        if (p1[q] != p2[q]) fail("generators " + std::to_string(i + 1) + " and " + std::to_string(j + 1) + " do not commute!");
    }
  for (const auto& gen : gens) {
    auto p = identity();
    int length = 1;
    while (true) {
      p = product(p, gen, 1);
      bool id = true;
      for (int i = 0; i < L; ++i) id = id && p[i] == i;
      if (id) break;
      ++length;
    }
    G.dims.push_back(length);
    G.g *= length;
  }
  for (int d : G.dims)
    if (d > 2) fail("symmetry groups with complex characters (a generator of order > 2) are not supported by this solver");
  if (G.g > kMaxGroup) fail("symmetry group larger than " + std::to_string(kMaxGroup) + " elements");
  for (int i = 0; i < G.g; ++i) {
    auto p = identity();
    int lab = i;
    for (size_t j = 0; j < gens.size(); ++j) {
      const int dj = lab % G.dims[j];
      lab /= G.dims[j];
      for (int l = 0; l < dj; ++l) p = product(p, gens[j], G.g);
    }
    if (i != 0) {
      bool id = true;
      for (int q = 0; q < L; ++q) id = id && p[q] == q;
      for (int q = L; q < N; ++q) id = id && p[q] == 0;
      if (id) fail("The identity is generated as a non trivial element");
    }
    for (int q = L; q < N; ++q)
      if (p[q] < 0 || p[q] >= G.g) fail("element " + std::to_string(i + 1) + " is not valid!");
    G.e.push_back(p);
  }
  return G;
}

// phi(a, b) = sum_j a_j b_j g / dim_j mod g (the Index product, src_ed/index.hpp:80-86)
int group_phi(const HostGroup& G, int a, int b) {
  int s = 0;
  for (size_t j = 0; j < G.dims.size(); ++j) {
    const int da = a % G.dims[j], db = b % G.dims[j];
    a /= G.dims[j];
    b /= G.dims[j];
    s += (da * db * G.g) / G.dims[j];
  }
  return s % G.g;
}

GroupDev device_group(const HostGroup& G, int irrep) {
  GroupDev D;
  std::memset(&D, 0, sizeof(D));
  D.g = G.g;
  D.L = G.L;
  D.N = G.N;
  for (int el = 0; el < G.g; ++el) {
    GroupElem& E = D.e[el];
    for (int i = 0; i < G.L; ++i) {
      E.img[i] = (uint8_t)G.e[el][i];
      uint32_t m = 0;
      for (int j = i + 1; j < G.L; ++j)
        if (G.e[el][i] > G.e[el][j]) m |= 1u << j;
      E.inv[i] = m;
    }
    for (int i = G.L; i < G.N; ++i) E.bath[i] = (uint8_t)G.e[el][i];
    E.phi2 = 2 * group_phi(G, el, irrep);
  }
  return D;
}

uint32_t grid_for(uint64_t n) { return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(1, (n + 255) / 256), 8192); }

}  // namespace

MixedSide side(const qed_sector& s) {
  auto T = std::static_pointer_cast<MixedTables>(s.mixed);
  const qed_sector& b = *T->base;
  return MixedSide{b.bup.as<uint32_t>(), b.bdn.as<uint32_t>(), b.du, T->full_of.as<uint32_t>(), T->len.as<uint32_t>(),
                   T->code.as<uint32_t>(), T->packed};
}

GroupTables group_tables(int N, int n_sites, const std::vector<std::vector<int>>& gens, bool bath_irrep) {
  if (N <= 0 || N > kMaxOrb) fail("number of orbitals out of range");
  if (n_sites < 0 || n_sites > N) fail("number of sites out of range");
  const HostGroup G = build_group(N, n_sites, gens, bath_irrep);
  GroupTables T;
  T.g = G.g;
  T.elements = G.e;
  T.phi.resize((size_t)G.g * G.g);
  for (int a = 0; a < G.g; ++a)
    for (int b = 0; b < G.g; ++b) T.phi[(size_t)a * G.g + b] = group_phi(G, a, b);
  return T;
}

template <int EP, class... Step>
static int launch_mixed(const qed_sector& s, const double* x, double* y, const Step&... step) {
  auto T = std::static_pointer_cast<MixedTables>(s.mixed);
  const qed_sector& b = *T->base;
  const uint32_t n = (uint32_t)s.D, grid = grid_for(n);
  if (n == 0) return 0;
  const bool vl = b.up_nvals + b.dn_nvals <= kLdsVals;
  auto k = T->packed ? (vl ? k_hv_mixed<true, true, EP, Step...> : k_hv_mixed<true, false, EP, Step...>)
                     : (vl ? k_hv_mixed<false, true, EP, Step...> : k_hv_mixed<false, false, EP, Step...>);
  k<<<grid, 256, 0, stream()>>>(view(b), b.up_ell.as<uint32_t>(), b.up_w, b.dn_ell.as<uint32_t>(), b.dn_w,
                                T->full_of.as<uint32_t>(), T->len.as<uint32_t>(), T->code.as<uint32_t>(), n, b.dn_nvals,
                                x, y, step...);
  QED_HIP(hipGetLastError());
  return (int)grid;
}

void hv_mixed(const qed_sector& s, const double* x, double* y) { launch_mixed<0>(s, x, y); }

int hv_step_mixed(const qed_sector& s, const double* x, double* y, const LzStep& L) {
  return L.kind == 1 ? launch_mixed<1>(s, x, y, L) : launch_mixed<2>(s, x, y, L);
}

void sector_diagonal(const qed_sector& s, double* d) {
  if (s.general) {
    diag_general(s, d);
    return;
  }
  if (!s.mixed) fail("sector_diagonal: a symmetry-adapted or mixed-number sector is expected");
  auto T = std::static_pointer_cast<MixedTables>(s.mixed);
  const qed_sector& b = *T->base;
  const uint32_t n = (uint32_t)s.D;
  if (n == 0) return;
  if (T->packed)
    k_diag_mixed<true><<<grid_for(n), 256, 0, stream()>>>(view(b), b.up_ell.as<uint32_t>(), b.up_w,
                                                         b.dn_ell.as<uint32_t>(), b.dn_w, T->full_of.as<uint32_t>(),
                                                         T->len.as<uint32_t>(), T->code.as<uint32_t>(), n, d);
  else
    k_diag_mixed<false><<<grid_for(n), 256, 0, stream()>>>(view(b), b.up_ell.as<uint32_t>(), b.up_w,
                                                          b.dn_ell.as<uint32_t>(), b.dn_w, T->full_of.as<uint32_t>(),
                                                          T->len.as<uint32_t>(), T->code.as<uint32_t>(), n, d);
  QED_HIP(hipGetLastError());
}

}  // namespace qed

using namespace qed;

extern "C" {

int qed_mixed_sector_create(int L, int n_up, int n_dn, int n_ops, const int* types, const double* coefs,
                            const int* nels, const int* er, const int* ec, const double* ev, int n_sites, int n_gen,
                            const int* gens, int bath_irrep, int irrep, qed_sector** out) {
  std::lock_guard<std::recursive_mutex> lk(lib_mutex());
  return guard([&] {
    *out = nullptr;
    if (L <= 0 || L > kMaxOrb) fail("number of orbitals out of range");
    if (n_sites < 0 || n_sites > L) fail("number of sites out of range");
    std::vector<std::vector<int>> gv(n_gen, std::vector<int>(L));
    for (int k = 0; k < n_gen; ++k)
      for (int i = 0; i < L; ++i) gv[k][i] = gens[(size_t)k * L + i];
    const HostGroup G = build_group(L, n_sites, gv, bath_irrep != 0);
    if (irrep < 0 || irrep >= G.g) fail("irreducible representation " + std::to_string(irrep) + " out of range");
    qed_sector* basep = nullptr;
    if (qed_sector_create(L, n_up, n_dn, n_ops, types, coefs, nels, er, ec, ev, &basep) != 0)
      fail(qed_last_error());
    std::shared_ptr<qed_sector> base(basep, [](qed_sector* p) { qed_sector_destroy(p); });
    const uint64_t D = base->D;
    if (D >= (1ull << 31)) fail("sector too large for the symmetry-adapted basis (2^31 factorized states)");
    if (base->du > (1u << kEllTargetBits) || base->dd > (1u << kEllTargetBits)) fail("half basis too large");
    auto T = std::make_shared<MixedTables>();
    T->base = base;
    T->g = G.g;
    T->irrep = irrep;
    T->elems = G.e;
    T->phi.resize((size_t)G.g * G.g);
    for (int a = 0; a < G.g; ++a)
      for (int b2 = 0; b2 < G.g; ++b2) T->phi[(size_t)a * G.g + b2] = group_phi(G, a, b2);
    const GroupDev GD = device_group(G, irrep);
    // pass 1: the representatives among the factorized states, in factorized order (which
    // is the order of the 64-bit states: down word first, then up word)
    DevBuf flags(std::max<uint64_t>(1, D)), lens(std::max<uint64_t>(1, D));
    k_mixed_flags<<<grid_for(D), 256, 0, stream()>>>(GD, base->bup.as<uint32_t>(), base->bdn.as<uint32_t>(), base->du, D,
                                                     flags.as<uint8_t>(), lens.as<uint8_t>());
    QED_HIP(hipGetLastError());
    std::vector<uint8_t> hf(D), hl(D);
    QED_HIP(hipMemcpyAsync(hf.data(), flags.p, D, hipMemcpyDeviceToHost, stream()));
    QED_HIP(hipMemcpyAsync(hl.data(), lens.p, D, hipMemcpyDeviceToHost, stream()));
    std::vector<uint32_t> hbu(base->du), hbd(base->dd);
    QED_HIP(hipMemcpyAsync(hbu.data(), base->bup.p, base->du * 4, hipMemcpyDeviceToHost, stream()));
    QED_HIP(hipMemcpyAsync(hbd.data(), base->bdn.p, base->dd * 4, hipMemcpyDeviceToHost, stream()));
    QED_HIP(hipStreamSynchronize(stream()));
    std::vector<uint32_t> index_of(D, kVanish), full_of, len;
    for (uint64_t f = 0; f < D; ++f)
      if (hf[f]) {
        index_of[f] = (uint32_t)full_of.size();
        full_of.push_back((uint32_t)f);
        len.push_back(hl[f]);
        T->states.push_back((uint64_t)hbu[f % base->du] | ((uint64_t)hbd[f / base->du] << 32));
      }
    DevBuf didx(std::max<uint64_t>(1, D) * 4);
    QED_HIP(hipMemcpyAsync(didx.p, index_of.data(), D * 4, hipMemcpyHostToDevice, stream()));
    T->code.alloc(std::max<uint64_t>(1, D) * 4);
    T->packed = full_of.size() < kPackedMax;
    k_mixed_codes<<<grid_for(D), 256, 0, stream()>>>(GD, base->bup.as<uint32_t>(), base->bdn.as<uint32_t>(), base->du, D,
                                                     n_up, n_dn, binom_dev(), didx.as<uint32_t>(), T->packed,
                                                     T->code.as<uint32_t>());
    QED_HIP(hipGetLastError());
    const size_t n = full_of.size();
    T->full_of.alloc(std::max<size_t>(1, n) * 4);
    T->len.alloc(std::max<size_t>(1, n) * 4);
    if (n) {
      QED_HIP(hipMemcpyAsync(T->full_of.p, full_of.data(), n * 4, hipMemcpyHostToDevice, stream()));
      QED_HIP(hipMemcpyAsync(T->len.p, len.data(), n * 4, hipMemcpyHostToDevice, stream()));
    }
    QED_HIP(hipStreamSynchronize(stream()));
    auto s = std::make_unique<qed_sector>();
    s->L = L;
    s->nup = n_up;
    s->ndn = n_dn;
    s->D = n;
    s->mixed = T;
    *out = s.release();
  });
}

int qed_mixed_apply_c(const qed_sector* src, const qed_sector* tgt, int spin, int pm, int n_sites,
                      const double* coef, const double* x, double* y) {
  std::lock_guard<std::recursive_mutex> lk(lib_mutex());
  return guard([&] {
    if (!src->mixed || !tgt->mixed) fail("qed_mixed_apply_c: both sectors must be symmetry-adapted");
    if (spin != 0 && spin != 1) fail("qed_mixed_apply_c: spin must be 0 or 1");
    if (n_sites < 0 || n_sites > src->L) fail("qed_mixed_apply_c: too many sites");
    const int dn = (spin == 0) ? 1 : 0;
    if (pm < 0 ? (tgt->nup != src->nup - dn || tgt->ndn != src->ndn - (1 - dn))
               : (tgt->nup != src->nup + dn || tgt->ndn != src->ndn + (1 - dn)))
      fail("qed_mixed_apply_c: the target sector does not match the operator");
    DevBuf cd((size_t)std::max(1, n_sites) * 8);
    if (n_sites) QED_HIP(hipMemcpyAsync(cd.p, coef, (size_t)n_sites * 8, hipMemcpyHostToDevice, stream()));
    if (pm < 0) {
      if (src->D)
        k_mixed_destroy<<<grid_for(src->D), 256, 0, stream()>>>(side(*src), side(*tgt), binom_dev(), (uint32_t)src->D,
                                                                n_sites, cd.as<double>(), spin, x, y);
    } else {
      if (tgt->D)
        k_mixed_create<<<grid_for(tgt->D), 256, 0, stream()>>>(side(*tgt), side(*src), binom_dev(), (uint32_t)tgt->D,
                                                               n_sites, cd.as<double>(), spin, x, y);
    }
    QED_HIP(hipGetLastError());
    QED_HIP(hipStreamSynchronize(stream()));
  });
}

int qed_mixed_group(const qed_sector* s, int* g, int* elements, int* phi) {
  return guard([&] {
    if (!s->mixed) fail("not a symmetry-adapted sector");
    auto T = std::static_pointer_cast<MixedTables>(s->mixed);
    *g = T->g;
    if (elements)
      for (int i = 0; i < T->g; ++i)
        for (int q = 0; q < s->L; ++q) elements[i * s->L + q] = T->elems[i][q];
    if (phi)
      for (int i = 0; i < T->g * T->g; ++i) phi[i] = T->phi[i];
  });
}

int qed_mixed_basis(const qed_sector* s, uint64_t* states, uint64_t* n) {
  return guard([&] {
    if (!s->mixed) fail("not a symmetry-adapted sector");
    auto T = std::static_pointer_cast<MixedTables>(s->mixed);
    *n = T->states.size();
    if (states) std::copy(T->states.begin(), T->states.end(), states);
  });
}

}  // extern "C"
