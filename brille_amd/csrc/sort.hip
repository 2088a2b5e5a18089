// Mode sorting on the device: the permutation table of DualInterpolator::sort
// (src/interpolatordual.hpp:398-434) built from the filled payload.
//
// 1. Pairs: every ordered pair of distinct vertices that share a cube node or a
//    tetrahedron (PolyTrellis::collect_keys, src/trellis_poly_parallel.tpp:487-524),
//    as per-vertex neighbour lists: count, scan, place, then sort and
//    de-duplicate each list (a vertex has a few dozen entries).  The keys
//    i * V + j come out sorted, i major.
// 2. The easy pairs, in one kernel (k_pair_easy): when the least cost of every
//    row of the pair's B x B cost matrix (DualInterpolator::cost_matrix,
//    src/interpolatordual.hpp:384-396) lies in a column of its own and leads
//    its row by more than rounding, that column-per-row assignment is the
//    optimum.  The matrix is never stored.
// 3. The other pairs, listed: their cost matrices entry by entry in the
//    reference's element order (Interpolator::add_cost,
//    src/interpolator_cost.tpp:21-58), the same row-minimum test on the exact
//    costs, then the exact linear assignment by successive shortest augmenting
//    paths, one wave per pair with the columns spread over the lanes (the LDS
//    holds the potentials, the Dijkstra distances and the matching).
// The assignment goes to key (i, j), its inverse to (j, i)
// (src/interpolatordual.hpp:422-432); identity assignments share permutation 0.
#include <algorithm>
#include <cmath>
#include <vector>

#include "grid_state.hpp"
#include "launch_pieces.hpp"

namespace brille_amd {

namespace {

constexpr int SORT_BLOCK = 64;  // one wave per pair
constexpr uint64_t kSortKeep = 128ull << 20;  // bytes of work space a sort may leave with the handle

// ---- pairs ----------------------------------------------------------------

// thread t: position t % 8 of cube t / 8, then position of a tetrahedron;
// PASS 0 counts each ordered pair at its first vertex, PASS 1 places the
// second vertex in the first's list (cursor = the count array, cleared)
template <int PASS>
__global__ __launch_bounds__(256) void k_pair_emit(const uint32_t* cube_v, uint64_t n_cubes, const uint32_t* tet_v,
                                                   uint64_t n_tets, uint32_t* __restrict__ cnt,
                                                   const uint32_t* __restrict__ off, uint32_t* __restrict__ adj) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t nc = 8 * n_cubes;
  const uint32_t* u;
  uint32_t k, a;
  if (t < nc) {
    u = cube_v + 8 * (t >> 3);
    k = 8;
    a = (uint32_t)(t & 7u);
  } else if (t < nc + 4 * n_tets) {
    u = tet_v + 4 * ((t - nc) >> 2);
    k = 4;
    a = (uint32_t)((t - nc) & 3u);
  } else {
    return;
  }
  const uint32_t va = u[a];
  for (uint32_t b = 0; b < k; ++b) {
    const uint32_t vb = u[b];
    if (b == a || vb == va) continue;
    if (PASS == 0) atomicAdd(&cnt[va], 1u);
    else adj[off[va] + atomicAdd(&cnt[va], 1u)] = vb;
  }
}

// Each list of the vertices [v0, V) sorted and de-duplicated in place, one wave per vertex;
// uniq[v] = its length, fwd[v] = its entries beyond v.  Lists of up to kListMax
// entries go through the wave's LDS slice (a bitonic sort over the next power
// of two: an insertion sort by one thread in memory took 1.1 ms for the 121 200
// lists of the hexagonal grid of 318 472 nodes, this 0.06 ms); longer ones are
// sorted by one lane.
constexpr uint32_t kListMax = 512;
__global__ __launch_bounds__(256) void k_pair_unique(uint64_t v0, uint64_t V, const uint32_t* __restrict__ off,
                                                     const uint32_t* __restrict__ cnt, uint32_t* __restrict__ adj,
                                                     uint32_t* __restrict__ uniq, uint32_t* __restrict__ fwd) {
  __shared__ uint32_t s_list[4][kListMax];
  const uint64_t v = v0 + (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (v >= V) return;  // wave-uniform; no block-wide barrier follows
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t* a = adj + off[v];
  const uint32_t n = cnt[v];
  uint32_t m = 0, beyond = 0;
  if (n <= kListMax) {
    uint32_t* l = s_list[threadIdx.x >> 6];
    uint32_t size = 64;
    while (size < n) size <<= 1;
    for (uint32_t i = lane; i < size; i += 64) l[i] = i < n ? a[i] : 0xFFFFFFFFu;
    wave_lds_fence();
    for (uint32_t k = 2; k <= size; k <<= 1)
      for (uint32_t j = k >> 1; j > 0; j >>= 1) {
        for (uint32_t i = lane; i < size; i += 64) {
          const uint32_t o = i ^ j;
          if (o > i) {
            const uint32_t x = l[i], y = l[o];
            if ((x > y) == ((i & k) == 0)) {
              l[i] = y;
              l[o] = x;
            }
          }
        }
        wave_lds_fence();
      }
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {
      const uint32_t i = i0 + lane;
      const uint32_t x = i < n ? l[i] : 0u;
      const bool keep = i < n && (i == 0 || l[i - 1] != x);
      const unsigned long long mask = __ballot(keep);
      if (keep) a[m + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = x;
      m += (uint32_t)__popcll(mask);
      beyond += (uint32_t)__popcll(__ballot(keep && x > (uint32_t)v));
    }
  } else if (lane == 0) {
    for (uint32_t i = 1; i < n; ++i) {
      const uint32_t x = a[i];
      uint32_t j = i;
      while (j > 0 && a[j - 1] > x) {
        a[j] = a[j - 1];
        --j;
      }
      a[j] = x;
    }
    for (uint32_t i = 0; i < n; ++i)
      if (m == 0 || a[i] != a[m - 1]) {
        a[m++] = a[i];
        beyond += a[m - 1] > (uint32_t)v ? 1u : 0u;
      }
  }
  if (lane == 0) {
    uniq[v] = m;
    fwd[v] = beyond;
  }
}

// One wave per vertex, from v0 on: its keys i * V + j in list order, the
// neighbour j of each key, and its forward pairs (j > i, the end of the sorted
// list) with the key each came from.
__global__ __launch_bounds__(256) void k_pair_keys(uint64_t v0, uint64_t V, const uint32_t* __restrict__ off,
                                                   const uint32_t* __restrict__ adj, const uint32_t* __restrict__ koff,
                                                   const uint32_t* __restrict__ poff, uint64_t* __restrict__ keys,
                                                   uint32_t* __restrict__ nbr, uint32_t* __restrict__ pi,
                                                   uint32_t* __restrict__ pj, uint32_t* __restrict__ pk) {
  const uint64_t v = v0 + (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (v >= V) return;
  const uint32_t* a = adj + off[v];
  const uint32_t k0 = koff[v], n = koff[v + 1] - k0, p0 = poff[v], nf = poff[v + 1] - p0;
  for (uint32_t k = threadIdx.x & 63u; k < n; k += 64) {
    const uint32_t j = a[k];
    keys[k0 + k] = v * V + j;
    nbr[k0 + k] = j;
    if (k >= n - nf) {
      const uint32_t p = p0 + (k - (n - nf));
      pi[p] = (uint32_t)v;
      pj[p] = j;
      pk[p] = k0 + k;
    }
  }
}

// rev[p]: the position of key (j, i) for the forward pair p = (i, j) (the
// lists are symmetric), by binary search in j's list
__global__ __launch_bounds__(256) void k_pair_rev(uint64_t n_pairs, const uint32_t* __restrict__ pi,
                                                  const uint32_t* __restrict__ pj, const uint32_t* __restrict__ nbr,
                                                  const uint32_t* __restrict__ koff, uint32_t* __restrict__ rev) {
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n_pairs) return;
  const uint32_t i = pi[p], j = pj[p];
  uint32_t lo = koff[j], hi = koff[j + 1];
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (nbr[mid] < i) lo = mid + 1;
    else hi = mid;
  }
  rev[p] = (lo < koff[j + 1] && nbr[lo] == i) ? lo : 0xFFFFFFFFu;
}

// ---- costs ----------------------------------------------------------------

// approx_float::scalar(|c|, 1) with its default tolerances (relative
// 1e4 x DBL_EPSILON, absolute 5e-15), then the clamp of |c| to one
// (src/utilities.tpp:263-275, 369-373); false when |c| exceeds one by more
__device__ __forceinline__ bool clamp_cos(double& c) {
  double act = fabs(c);
  const double x = fabs(act - 1.0);
  const bool near = x <= 5.0e-15 + (2.220446049250313e-16 * 10000.0) * fabs(act + 1.0) || x < 2.2250738585072014e-308;
  if (near && act > 1) {
    c /= act;
    act = fabs(c);
  }
  return act <= 1;
}

// utils::vector_angle of real vectors  src/utilities.tpp:249-278
template <typename Real>
__device__ double vec_angle_r(uint32_t n, const Real* A, const Real* B, bool& ok) {
  double AA = 0, BB = 0, AB = 0;
  for (uint32_t i = 0; i < n; ++i) {
    const double a = (double)A[i], b = (double)B[i];
    AA += a * a;
    BB += b * b;
    AB += a * b;
  }
  const double nA = sqrt(AA), nB = sqrt(BB);
  double c = (nA != 0 && nB != 0) ? AB / (nA * nB) : ((nA != 0 || nB != 0) ? 0.0 : 1.0);
  if (!clamp_cos(c)) ok = false;
  return acos(c);
}

template <typename Real>
__device__ double vec_dist_r(uint32_t n, const Real* a, const Real* b) {
  double s = 0;
  for (uint32_t i = 0; i < n; ++i) {
    const double d = (double)a[i] - (double)b[i];
    s += d * d;
  }
  return sqrt(s);
}

// the vector cost of real vectors  src/interpolator.hpp:256-293
template <typename Real>
__device__ double vecfun_r(int t, uint32_t n, const Real* a, const Real* b, bool& ok) {
  switch (t) {
    case 1: return vec_dist_r(n, a, b);
    case 2: {
      double h = 0;
      for (uint32_t i = 0; i < n; ++i) h += (double)a[i] * (double)b[i];
      return 1 - h;
    }
    case 3:
    case 4: return vec_angle_r(n, a, b, ok);
    default: {
      const double s = sin(vec_angle_r(n, a, b, ok));
      return s * s;
    }
  }
}

// The second vertex's vector elements after multiplication by the antiphase
// (er, ei): element z of phased = (er + i ei) (br + i bi), as
// utils::inplace_antiphase forms it (src/utilities.tpp:589-593).
template <typename Real>
struct Phased {
  const Real* b;
  double er, ei;
  __device__ double re(uint32_t z) const { return er * (double)b[2 * z] - ei * (double)b[2 * z + 1]; }
  __device__ double im(uint32_t z) const { return er * (double)b[2 * z + 1] + ei * (double)b[2 * z]; }
};

// hermitian_product of a (complex) and phased b from element z0, n elements
template <typename Real>
__device__ void herm_ab(uint32_t z0, uint32_t n, const Real* a, const Phased<Real>& b, double& hr, double& hi) {
  hr = 0;
  hi = 0;
  for (uint32_t i = z0; i < z0 + n; ++i) {
    const double ar = (double)a[2 * i], ai = (double)a[2 * i + 1], br = b.re(i), bi = b.im(i);
    hr += ar * br + ai * bi;
    hi += ar * bi - ai * br;
  }
}

// the vector cost of complex vectors, a against phased b, elements [z0, z0 + n)
// src/interpolator.hpp:256-293 with src/utilities.tpp:280-417
template <typename Real>
__device__ double vecfun_c(int t, uint32_t z0, uint32_t n, const Real* a, const Phased<Real>& b, bool& ok) {
  if (t == 1) {
    double s = 0;
    for (uint32_t i = z0; i < z0 + n; ++i) {
      const double dr = (double)a[2 * i] - b.re(i), di = (double)a[2 * i + 1] - b.im(i);
      s += dr * dr + di * di;
    }
    return sqrt(s);
  }
  if (t == 2) {
    double hr, hi;
    herm_ab(z0, n, a, b, hr, hi);
    return 1 - (hr * hr + hi * hi);
  }
  if (t == 3) {  // euclidean_angle
    double AB = 0, nA = 0, nB = 0;
    for (uint32_t i = z0; i < z0 + n; ++i) {
      const double ar = (double)a[2 * i], ai = (double)a[2 * i + 1], br = b.re(i), bi = b.im(i);
      AB += ar * br + ai * bi;
      nA += ar * ar + ai * ai;
      nB += br * br + bi * bi;
    }
    nA = sqrt(nA);
    nB = sqrt(nB);
    double c = (nA != 0 && nB != 0) ? AB / (nA * nB) : ((nA != 0 || nB != 0) ? 0.0 : 1.0);
    if (!clamp_cos(c)) ok = false;
    return acos(c);
  }
  // hermitian_angle: |a^H b| over the norms
  double hr, hi;
  herm_ab(z0, n, a, b, hr, hi);
  const double nAB = sqrt(hr * hr + hi * hi);
  double aa = 0, bb = 0;
  for (uint32_t i = z0; i < z0 + n; ++i) {
    const double ar = (double)a[2 * i], ai = (double)a[2 * i + 1];
    aa += ar * ar + ai * ai;
  }
  for (uint32_t i = z0; i < z0 + n; ++i) {
    const double br = b.re(i), bi = b.im(i);
    bb += br * br + bi * bi;
  }
  const double nA = sqrt(aa), nB = sqrt(bb);
  double c = (nA != 0 && nB != 0) ? nAB / (nA * nB) : ((nA != 0 || nB != 0) ? 0.0 : 1.0);
  if (!clamp_cos(c)) ok = false;
  const double th = acos(c);
  if (t == 4) return th;
  const double s = sin(th);
  return s * s;
}

struct CostArgs {
  uint32_t B, sv, sc, stride;
  uint32_t ev[3], ec[3];
  int32_t vs, vv, cs, cv;  // scalar / vector cost kinds of values and vectors
  double vw[3], cw[3];
};

// cost of mode a of row block x0 against mode b of row block x1: the values'
// term (no phase) then the vectors' term (after the antiphase), each
// weights[0] s + weights[1] v + weights[2] m, added in that order to zero
// (DualInterpolator::cost_matrix, src/interpolatordual.hpp:384-396)
template <typename Real>
__device__ double pair_cost(const CostArgs& c, const Real* x0, const Real* x1, bool& ok) {
  double cost = 0;
  if (c.sv) {
    const Real* a = x0 + 2 * c.sc;
    const Real* b = x1 + 2 * c.sc;
    const uint32_t mo = c.ev[0] + c.ev[1];
    double s = 0, v = 0, m = 0;
    if (c.ev[0])
      for (uint32_t z = 0; z < c.ev[0]; ++z) s += fabs((double)a[z] - (double)b[z]);
    if (c.ev[1]) v = vecfun_r(c.vv, c.ev[1], a + c.ev[0], b + c.ev[0], ok);
    if (c.ev[2])
      for (uint32_t q = 0; q < c.ev[2] / 9; ++q) m += vec_dist_r(9, a + mo + 9 * q, b + mo + 9 * q);
    cost += c.vw[0] * s + c.vw[1] * v + c.vw[2] * m;
  }
  if (c.sc) {
    // antiphase of the whole span  src/utilities.tpp:567-577
    double rd = 0, id = 0;
    for (uint32_t z = 0; z < c.sc; ++z) {
      const double ar = (double)x0[2 * z], ai = (double)x0[2 * z + 1], br = (double)x1[2 * z], bi = (double)x1[2 * z + 1];
      rd += ar * br + ai * bi;
      id += ar * bi - ai * br;
    }
    const double th = -1.0 * atan2(id, rd);
    const Phased<Real> ph{x1, 1.0 * cos(th), 1.0 * sin(th)};
    const uint32_t mo = c.ec[0] + c.ec[1];
    double s = 0, v = 0, m = 0;
    if (c.ec[0])
      for (uint32_t z = 0; z < c.ec[0]; ++z) {
        const double dr = (double)x0[2 * z] - ph.re(z), di = (double)x0[2 * z + 1] - ph.im(z);
        s += sqrt(dr * dr + di * di);
      }
    if (c.ec[1]) v = vecfun_c(c.cv, c.ec[0], c.ec[1], x0, ph, ok);
    if (c.ec[2])
      for (uint32_t q = 0; q < c.ec[2] / 9; ++q) m += vecfun_c(1, mo + 9 * q, 9, x0, ph, ok);
    cost += c.cw[0] * s + c.cw[1] * v + c.cw[2] * m;
  }
  return cost;
}

// (value, column) pairs: the smaller value, the lower column on ties
__device__ __forceinline__ void wave_argmin(double& v, uint32_t& j) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const double ov = __shfl_xor(v, o);
    const uint32_t oj = __shfl_xor(j, o);
    if (ov < v || (ov == v && oj < j)) {
      v = ov;
      j = oj;
    }
  }
}

// The easy pairs, a lane per (pair, mode a of the first vertex): the lane walks
// the second vertex's modes and keeps the least cost of its row and the runner-
// up.  For Gamma-like vectors (SC complex vector elements, the default cost
// sin^2 of the Hermitian angle) the cost needs no phase and no angle:
// sin^2 = 1 - |a.b|^2 / (|a|^2 |b|^2), some eighty operations against seven
// hundred, whose value agrees with the literal one to rounding (~1e-14 of the
// terms); a row whose lead is within kLead of that scale, a norm near zero or
// near overflow, or a value that is not finite sends the pair to the literal
// costs.  Memory: the rows
// alone (one wave reads each pair's from the cache); 1.4e6 pairs of 6 modes,
// FP64: 4.1 ms for the stored matrices and their row minima, 0.3 ms here.
// asg[p * B + a]: the column of row a; hard[p], moved[p]: 0 or 1.
constexpr double kLead = 1e-9;
template <typename Real, int SC>
__global__ __launch_bounds__(256) void k_pair_easy(CostArgs c, const Real* __restrict__ rows,
                                                   const uint32_t* __restrict__ pi, const uint32_t* __restrict__ pj,
                                                   const uint32_t* __restrict__ rev, uint64_t n_pairs,
                                                   uint16_t* __restrict__ asg, uint32_t* __restrict__ hard,
                                                   uint32_t* __restrict__ moved) {
  __shared__ uint32_t s_col[256], s_flag[256];  // column of each row; per pair: bit 0 hard, bit 1 moved
  const uint32_t B = c.B, per = 256 / B, tid = threadIdx.x;
  const uint32_t lp = tid / B, a = tid - lp * B;
  const uint64_t p = (uint64_t)blockIdx.x * per + lp;
  const bool on = lp < per && p < n_pairs;
  s_flag[tid] = 0;
  __syncthreads();
  uint32_t col = 0;
  if (on) {
    const Real* ra = rows + ((uint64_t)pi[p] * B + a) * c.stride;
    const Real* rb = rows + (uint64_t)pj[p] * B * c.stride;
    double x[2 * SC], aa = 0;
#pragma unroll
    for (int k = 0; k < 2 * SC; ++k) {
      x[k] = (double)ra[k];
      aa += x[k] * x[k];
    }
    double best = __builtin_huge_val(), second = __builtin_huge_val();
    bool fine = aa > 1e-140 && aa < 1e140;
    for (uint32_t b = 0; b < B; ++b, rb += c.stride) {
      double s = 0, hr = 0, hi = 0, bb = 0;
      for (uint32_t z = 0; z < c.ev[0]; ++z) s += fabs((double)ra[2 * SC + z] - (double)rb[2 * SC + z]);
#pragma unroll
      for (int k = 0; k < SC; ++k) {
        const double br = (double)rb[2 * k], bi = (double)rb[2 * k + 1];
        hr += x[2 * k] * br + x[2 * k + 1] * bi;
        hi += x[2 * k] * bi - x[2 * k + 1] * br;
        bb += br * br + bi * bi;
      }
      const double cost = c.vw[0] * s + c.cw[1] * (1.0 - (hr * hr + hi * hi) / (aa * bb));
      // (norms whose products neither overflow nor underflow; false for NaN)
      fine = fine && bb > 1e-140 && bb < 1e140 && fabs(cost) < 1e300;
      if (cost < best) {
        second = best;
        best = cost;
        col = b;
      } else if (cost < second) {
        second = cost;
      }
    }
    if (!(fine && second - best > kLead * (fabs(c.cw[1]) + fabs(best)))) atomicOr(&s_flag[lp], 1u);
    if (col != a) atomicOr(&s_flag[lp], 2u);
  }
  s_col[tid] = col;
  __syncthreads();
  if (on) {
    for (uint32_t k = 0; k < a; ++k)
      if (s_col[tid - a + k] == col) {
        atomicOr(&s_flag[lp], 1u);
        break;
      }
    asg[p * B + a] = (uint16_t)col;
  }
  __syncthreads();
  if (on && a == 0) {
    const uint32_t f = s_flag[lp];
    const bool h = (f & 1u) || rev[p] == 0xFFFFFFFFu;
    hard[p] = h ? 1u : 0u;
    moved[p] = !h && (f & 2u) ? 1u : 0u;
  }
}

__global__ __launch_bounds__(256) void k_fill_words(uint32_t* __restrict__ a, uint64_t n, uint32_t v) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

// list[off[p]] = p for the flagged pairs (off: exclusive scan of the flags)
__global__ __launch_bounds__(256) void k_pair_list(uint64_t n_pairs, const uint32_t* __restrict__ off,
                                                   uint32_t* __restrict__ list) {
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n_pairs && off[p + 1] != off[p]) list[off[p]] = (uint32_t)p;
}

// The cost matrices of the listed pairs [h0, h0 + nh): one lane per entry
// (pair, a, b), so every lane of every wave computes (B x B entries per pair).
template <typename Real>
__global__ __launch_bounds__(256) void k_pair_costs(CostArgs c, const Real* rows, const uint32_t* __restrict__ pi,
                                                    const uint32_t* __restrict__ pj, const uint32_t* __restrict__ list,
                                                    uint64_t h0, uint64_t nh, double* __restrict__ C,
                                                    uint32_t* __restrict__ bad) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t B = c.B, BB = B * B;
  if (t >= nh * BB) return;
  const uint64_t q = t / BB;
  const uint32_t e = (uint32_t)(t - q * BB);
  const uint32_t a = e / B, b = e - a * B;
  const uint32_t p = list[h0 + q];
  const uint64_t i = pi[p], j = pj[p];
  bool ok = true;
  C[t] = pair_cost(c, rows + (i * B + a) * c.stride, rows + (j * B + b) * c.stride, ok);
  if (!ok) atomicOr(bad, 1u);
}

// The row minima of the stored matrices, one thread per listed pair: when the
// first minimum of every row lies in a different column, that assignment is
// exactly what the augmenting-path solver below returns (each row's search
// then ends at its first minimum, a free column).  The others stay in todo (todo[q] =
// 1) for the solver.  Matrices of more than 64 columns all go to the solver.
__global__ __launch_bounds__(256) void k_pair_fast(const double* __restrict__ Cg, uint32_t B,
                                                   const uint32_t* __restrict__ list, uint64_t h0, uint64_t nh,
                                                   const uint32_t* __restrict__ rev, uint16_t* __restrict__ asg,
                                                   uint32_t* __restrict__ moved, uint32_t* __restrict__ todo) {
  const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nh) return;
  const uint64_t p = list[h0 + q];
  todo[q] = 1;
  if (B > 64 || rev[p] == 0xFFFFFFFFu) return;
  const double* C = Cg + q * B * B;
  unsigned long long taken = 0;
  bool shift = false;
  for (uint32_t a = 0; a < B; ++a) {
    double best = __builtin_huge_val();
    uint32_t bc = 0xFFFFFFFFu;
    for (uint32_t b = 0; b < B; ++b) {
      const double c = C[(uint64_t)a * B + b];
      if (c < best) {
        best = c;
        bc = b;
      }
    }
    if (bc == 0xFFFFFFFFu || (taken >> bc) & 1ull) return;
    taken |= 1ull << bc;
    shift = shift || bc != a;
    asg[p * B + a] = (uint16_t)bc;
  }
  todo[q] = 0;
  moved[p] = shift ? 1u : 0u;
}

// One wave per listed pair of [h0, h0 + nh) still to do (grid-stride): the exact
// assignment of its cost matrix (copied to LDS when it fits, read from C
// otherwise).  LDS: potentials u, v, distances minv ((B + 1) doubles each),
// matching p, predecessors way and scanned flags ((B + 1) words each), then the
// matrix.
__global__ __launch_bounds__(SORT_BLOCK) void k_pair_lap(const double* __restrict__ Cg, uint32_t B,
                                                         const uint32_t* __restrict__ list, uint64_t h0, uint64_t nh,
                                                         const uint32_t* __restrict__ todo, int cost_in_lds,
                                                         const uint32_t* __restrict__ rev,
                                                         uint16_t* __restrict__ asg, uint32_t* __restrict__ moved,
                                                         uint32_t* __restrict__ bad) {
  extern __shared__ double lds[];
  const uint32_t lane = threadIdx.x;
  double* u = lds;
  double* v = u + (B + 1);
  double* minv = v + (B + 1);
  int32_t* p = reinterpret_cast<int32_t*>(minv + (B + 1));
  int32_t* way = p + (B + 1);
  int32_t* used = way + (B + 1);
  double* Cl = lds + 3 * (B + 1) + (3 * (B + 1) + 1) / 2;
  const double INF = __builtin_huge_val();
  const uint32_t BB = B * B;
  for (uint64_t q0 = blockIdx.x; q0 < nh; q0 += gridDim.x) {
    if (!todo[q0]) continue;
    const double* C = Cg + q0 * BB;
    if (cost_in_lds) {
      for (uint32_t e = lane; e < BB; e += SORT_BLOCK) Cl[e] = C[e];
      C = Cl;
    }
    const uint64_t pair = list[h0 + q0];
    const bool has_rev = rev[pair] != 0xFFFFFFFFu;  // always, the lists being symmetric
    for (uint32_t q = lane; q <= B; q += SORT_BLOCK) {
      u[q] = 0;
      v[q] = 0;
      p[q] = 0;
      way[q] = 0;
    }
    __syncthreads();
    // successive shortest augmenting paths, rows 1..B; a cost matrix with
    // NaNs leaves no column to take, and the pair is abandoned
    bool stuck = false;
    for (uint32_t row = 1; row <= B && !stuck; ++row) {
      for (uint32_t q = lane; q <= B; q += SORT_BLOCK) {
        minv[q] = INF;
        used[q] = 0;
      }
      if (lane == 0) p[0] = (int32_t)row;
      __syncthreads();
      uint32_t j0 = 0;
      while (true) {
        if (lane == 0) used[j0] = 1;
        __syncthreads();
        const uint32_t i0 = (uint32_t)p[j0];
        double best = INF;
        uint32_t bj = 0xFFFFFFFFu;
        for (uint32_t q = 1 + lane; q <= B; q += SORT_BLOCK) {
          if (used[q]) continue;
          const double cur = C[(uint64_t)(i0 - 1) * B + (q - 1)] - u[i0] - v[q];
          if (cur < minv[q]) {
            minv[q] = cur;
            way[q] = (int32_t)j0;
          }
          if (minv[q] < best) {
            best = minv[q];
            bj = q;
          }
        }
        wave_argmin(best, bj);
        if (bj == 0xFFFFFFFFu) {  // wave-uniform
          stuck = true;
          break;
        }
        const double delta = best;
        __syncthreads();
        for (uint32_t q = lane; q <= B; q += SORT_BLOCK) {
          if (used[q]) {
            u[p[q]] += delta;
            v[q] -= delta;
          } else {
            minv[q] -= delta;
          }
        }
        __syncthreads();
        j0 = bj;
        if (p[j0] == 0) break;
      }
      if (lane == 0 && !stuck) {
        do {
          const uint32_t j1 = (uint32_t)way[j0];
          p[j0] = p[j1];
          j0 = j1;
        } while (j0);
      }
      __syncthreads();
    }
    if (stuck || !has_rev) {
      if (lane == 0) {
        atomicOr(bad, 1u);
        moved[pair] = 0;
      }
      __syncthreads();
      continue;
    }
    bool shift = false;
    for (uint32_t q = 1 + lane; q <= B; q += SORT_BLOCK) {
      asg[pair * B + (uint32_t)(p[q] - 1)] = (uint16_t)(q - 1);
      shift = shift || (uint32_t)(p[q] - 1) != q - 1;
    }
    shift = __any(shift);
    if (lane == 0) moved[pair] = shift ? 1u : 0u;
    __syncthreads();  // the LDS is reused by the next pair
  }
}

// The table: pair p's assignment and its inverse at permutations 1 + 2 off[p]
// and the next (off: exclusive scan of the moved flags), a lane per (pair, row);
// both keys point there, or to permutation 0 where nothing moved.
__global__ __launch_bounds__(256) void k_perm_write(uint64_t n_pairs, uint32_t B, const uint16_t* __restrict__ asg,
                                                    const uint32_t* __restrict__ off, const uint32_t* __restrict__ pk,
                                                    const uint32_t* __restrict__ rev,
                                                    uint32_t* __restrict__ perm_index, uint32_t* __restrict__ perms) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t p = t / B;
  if (p >= n_pairs) return;
  const uint32_t a = (uint32_t)(t - p * B);
  const bool shift = off[p + 1] != off[p];
  const uint64_t slot = shift ? 1 + 2 * (uint64_t)off[p] : 0;
  if (shift) {
    const uint32_t b = asg[t];
    perms[slot * B + a] = b;
    perms[(slot + 1) * B + b] = a;
  }
  if (a == 0) {
    perm_index[pk[p]] = (uint32_t)slot;
    if (rev[p] != 0xFFFFFFFFu) perm_index[rev[p]] = shift ? (uint32_t)slot + 1 : 0u;
  }
}

__global__ void k_identity_perm(uint32_t* perms, uint32_t B) {
  for (uint32_t q = threadIdx.x; q < B; q += blockDim.x) perms[q] = q;
}

// vkey[i]: the first key of vertex i (keys sorted, i * V + j)
__global__ __launch_bounds__(256) void k_vertex_keys(uint64_t V, const uint64_t* __restrict__ keys, uint64_t n_keys,
                                                     uint32_t* __restrict__ vkey) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i > V) return;
  uint64_t lo = 0, hi = n_keys;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (keys[mid] < i * V) lo = mid + 1;
    else hi = mid;
  }
  vkey[i] = (uint32_t)lo;
}

// out[t]: the permutation of block slot t against its block's slot-0 vertex
__global__ __launch_bounds__(256) void k_cell_perms(GridConst g, DataConst d, uint64_t n_cube_slots, uint64_t n_slots,
                                                    uint32_t* __restrict__ out) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_slots) return;
  if (t < n_cube_slots) {
    const uint32_t* v = g.cube_v + 8 * (t >> 3);
    out[t] = perm_find(d, v[7], v[7 - (int)(t & 7u)]);
  } else {
    const uint32_t* v = g.tet_v + 4 * ((t - n_cube_slots) >> 2);
    out[t] = perm_find(d, v[0], v[(t - n_cube_slots) & 3u]);
  }
}

struct DevBuf {
  std::vector<void*> held;
  ~DevBuf() {
    for (void* p : held) (void)hipFree(p);
  }
  template <typename T>
  T* get(size_t n) {
    void* p = nullptr;
    if (hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(T)) != hipSuccess) return nullptr;
    held.push_back(p);
    return static_cast<T*>(p);
  }
  void release(void* p) {
    held.erase(std::remove(held.begin(), held.end(), p), held.end());
  }
};

}  // namespace

// launches k_pair_easy where the payload and the cost kinds allow it (false: no)
static bool launch_easy(const brille_grid* G, const CostArgs& c, const uint32_t* pi, const uint32_t* pj,
                        const uint32_t* rev, uint64_t n_pairs, uint16_t* asg, uint32_t* hard, uint32_t* moved,
                        hipStream_t s) {
  const DataConst& d = G->d;
  const bool vectors = c.ec[0] == 0 && c.ec[2] == 0 && (c.cv < 1 || c.cv > 4);
  if (d.B > 64 || c.ev[1] || c.ev[2] || !vectors) return false;
  // (the literal sum has the terms of absent elements too: an infinite weight of
  // one is a NaN there)
  for (int q = 0; q < 3; ++q)
    if (!std::isfinite(c.vw[q]) || !std::isfinite(c.cw[q])) return false;
  auto go = [&](auto k64, auto k32) {
    in_pieces(n_pairs, 256 / d.B, [&](uint64_t p, uint64_t n, unsigned blocks) {
      if (d.rows64)
        hipLaunchKernelGGL(k64, dim3(blocks), dim3(256), 0, s, c, d.rows64, pi + p, pj + p, rev + p, n, asg + p * d.B, hard + p, moved + p);
      else
        hipLaunchKernelGGL(k32, dim3(blocks), dim3(256), 0, s, c, d.rows32, pi + p, pj + p, rev + p, n, asg + p * d.B, hard + p, moved + p);
    });
    return true;
  };
  switch (c.sc) {
    case 3: return go(k_pair_easy<double, 3>, k_pair_easy<float, 3>);
    case 6: return go(k_pair_easy<double, 6>, k_pair_easy<float, 6>);
    case 9: return go(k_pair_easy<double, 9>, k_pair_easy<float, 9>);
    case 12: return go(k_pair_easy<double, 12>, k_pair_easy<float, 12>);
    default: return false;
  }
}

int install_permutations(brille_grid* G, std::vector<void*>& allocs, hipStream_t s) {
  DataConst& d = G->d;
  d.vkey = nullptr;
  d.cell_perm = nullptr;
  if (d.n_keys == 0) return BRILLE_OK;
  void* p = nullptr;
  if (d.n_keys < 0xFFFFFFFFull) {
    if (hipMalloc(&p, (d.V + 1) * sizeof(uint32_t)) != hipSuccess)
      return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the permutation lookup");
    allocs.push_back(p);
    uint32_t* vkey = static_cast<uint32_t*>(p);
    hipLaunchKernelGGL(k_vertex_keys, dim3((unsigned)((d.V + 256) / 256)), dim3(256), 0, s, d.V, d.keys, d.n_keys, vkey);
    d.vkey = vkey;
  }
  const uint64_t cubes = 8 * G->n_cubes, slots = cubes + 4 * G->n_tets;
  if (d.has_blocks && slots) {
    if (hipMalloc(&p, slots * sizeof(uint32_t)) != hipSuccess)
      return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the permutation lookup");
    allocs.push_back(p);
    uint32_t* cell = static_cast<uint32_t*>(p);
    hipLaunchKernelGGL(k_cell_perms, dim3((unsigned)((slots + 255) / 256)), dim3(256), 0, s, G->g, d, cubes, slots, cell);
    d.cell_perm = cell;
  }
  if (hipGetLastError() != hipSuccess) return fail(BRILLE_ERR_DEVICE, "permutation lookup launch failed");
  // later calls read the lookup from any stream
  if (hipStreamSynchronize(s) != hipSuccess) return fail(BRILLE_ERR_DEVICE, "permutation lookup failed");
  return BRILLE_OK;
}
}  // namespace brille_amd

using namespace brille_amd;

extern "C" int brille_grid_sort(brille_grid* G, const brille_cost_info* values_cost,
                                const brille_cost_info* vectors_cost) {
  BRILLE_LOCK_GRID(G);
  if (!G) return fail(BRILLE_ERR_INVALID_ARGUMENT, "null grid");
  if (!G->filled) return fail(BRILLE_ERR_NOT_FILLED, "The interpolation data must be filled before sorting.");
  DataConst& d = G->d;
  const brille_cost_info dflt{0, 0, {1.0, 1.0, 1.0}};
  const brille_cost_info& vc = values_cost ? *values_cost : dflt;
  const brille_cost_info& cc = vectors_cost ? *vectors_cost : dflt;
  if (d.B == 0 || d.V == 0) return BRILLE_OK;
  if (d.B > 4096) return fail(BRILLE_ERR_UNSUPPORTED, "sorting supports at most 4096 branches");
  if (d.V > 0xFFFFFFFFull) return fail(BRILLE_ERR_UNSUPPORTED, "sorting supports at most 2^32 - 1 vertices");
  const uint64_t V = d.V;
  const hipStream_t s = 0;
  // earlier work may still use the handle's work space and the tables replaced
  // below
  if (hipDeviceSynchronize() != hipSuccess) return fail(BRILLE_ERR_DEVICE, "device error before sorting");
  DevBuf buf;
  const uint64_t units = 8 * G->n_cubes + 4 * G->n_tets;
  const uint64_t most = 56 * G->n_cubes + 12 * G->n_tets;  // ordered pairs emitted, at most
  if (most > 0xFFFFFFFFull) return fail(BRILLE_ERR_UNSUPPORTED, "sorting supports at most 2^32 - 1 vertex pairs");
  const uint64_t scan_words = (V + 1 + 4095) / 4096 + 1;
  // lists, offsets and scans in one allocation
  uint32_t* ws0 = buf.get<uint32_t>(5 * (V + 1) + scan_words + 4 + most);
  if (!ws0) return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the sort work space");
  uint32_t* cnt = ws0;
  uint32_t* off = cnt + (V + 1);
  uint32_t* koff = off + (V + 1);
  uint32_t* poff = koff + (V + 1);
  uint32_t* cursor = poff + (V + 1);
  uint32_t* part = cursor + (V + 1);
  uint32_t* counter = part + scan_words;
  uint32_t* adj = counter + 4;
  zero_words(ws0, (uint32_t)(5 * (V + 1) + scan_words + 4), s);
  const unsigned ub = (unsigned)((units + 255) / 256);
  if (units) hipLaunchKernelGGL(k_pair_emit<0>, dim3(ub), dim3(256), 0, s, G->g.cube_v, G->n_cubes, G->g.tet_v, G->n_tets, cnt, off, nullptr);
  if (hipMemcpyAsync(off, cnt, (V + 1) * 4, hipMemcpyDeviceToDevice, s) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "hipMemcpyAsync failed");
  if (int rc = exclusive_scan_u32(off, V + 1, part, s); rc != BRILLE_OK) return rc;
  if (units) hipLaunchKernelGGL(k_pair_emit<1>, dim3(ub), dim3(256), 0, s, G->g.cube_v, G->n_cubes, G->g.tet_v, G->n_tets, cursor, off, adj);
  in_pieces(V, 4, [&](uint64_t v0, uint64_t, unsigned blocks) {
    hipLaunchKernelGGL(k_pair_unique, dim3(blocks), dim3(256), 0, s, v0, V, off, cnt, adj, koff, poff);
  });
  if (int rc = exclusive_scan_u32(koff, V + 1, part, s); rc != BRILLE_OK) return rc;
  if (int rc = exclusive_scan_u32(poff, V + 1, part, s); rc != BRILLE_OK) return rc;
  uint32_t n32[2] = {0, 0};
  if (hipMemcpyAsync(&n32[0], koff + V, 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipMemcpyAsync(&n32[1], poff + V, 4, hipMemcpyDeviceToHost, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "reading the pair counts failed");
  const uint64_t n_keys = n32[0], n_pairs = n32[1];
  // the new table: keys and per-key permutation index here, the permutations
  // once their number is known
  uint64_t* keys = buf.get<uint64_t>(n_keys);
  uint32_t* pidx = buf.get<uint32_t>(n_keys);
  if (!keys || !pidx) return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the permutation table");
  // the rest of the work space is the binned pipeline's, grown when it is
  // smaller (its calls and this one hold the handle's lock in turn, and the
  // device was synchronised above): allocating and freeing as much anew took a
  // third of a sort of 1.4e6 pairs.  Beyond kSortKeep bytes the handle does not
  // keep it.
  const uint64_t hwords = (n_pairs + 1 + 4095) / 4096 + 1;
  const uint64_t words = n_keys + 4 * n_pairs + 3 * (n_pairs + 1) + hwords;
  const uint64_t ws_bytes = words * 4 + n_pairs * d.B * 2 + 16;
  uint32_t* nbr = nullptr;
  if (ws_bytes > std::max<uint64_t>(kSortKeep, G->bin_ws_bytes)) {
    nbr = reinterpret_cast<uint32_t*>(buf.get<char>(ws_bytes));
    if (!nbr) return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the sort work space");
  } else {
    if (int rc = ensure_work_space(G, ws_bytes); rc != BRILLE_OK) return rc;
    nbr = static_cast<uint32_t*>(G->bin_ws);
  }
  uint32_t* pi = nbr + n_keys;
  uint32_t* pj = pi + n_pairs;
  uint32_t* pk = pj + n_pairs;
  uint32_t* rev = pk + n_pairs;
  uint32_t* hard = rev + n_pairs;          // flags, then their exclusive scan
  uint32_t* moved = hard + (n_pairs + 1);  // flags, then their exclusive scan
  uint32_t* keep = moved + (n_pairs + 1);  // the moved flags, kept while hard pairs are left
  uint32_t* hpart = keep + (n_pairs + 1);
  uint16_t* asg = reinterpret_cast<uint16_t*>(hpart + hwords);
  in_pieces(V, 4, [&](uint64_t v0, uint64_t, unsigned blocks) {
    hipLaunchKernelGGL(k_pair_keys, dim3(blocks), dim3(256), 0, s, v0, V, off, adj, koff, poff, keys, nbr, pi, pj, pk);
  });
  CostArgs ca{};
  ca.B = d.B;
  ca.sv = d.sv;
  ca.sc = d.sc;
  for (int q = 0; q < 3; ++q) {
    ca.ev[q] = d.ev[q];
    ca.ec[q] = d.ec[q];
    ca.vw[q] = vc.weights[q];
    ca.cw[q] = cc.weights[q];
  }
  ca.vs = vc.scalar_cost;
  ca.vv = vc.vector_cost;
  ca.cs = cc.scalar_cost;
  ca.cv = cc.vector_cost;
  ca.stride = d.rows64 ? d.stride64 : d.stride32;
  const unsigned pb = (unsigned)((n_pairs + 255) / 256);
  uint32_t n_hard = 0, n_moved = 0;
  // exclusive scan of n_pairs flags (one word more: the total)
  auto scan_flags = [&](uint32_t* a) {
    zero_words(a + n_pairs, 1, s);
    return exclusive_scan_u32(a, n_pairs + 1, hpart, s);
  };
  if (n_pairs) {
    hipLaunchKernelGGL(k_pair_rev, dim3(pb), dim3(256), 0, s, n_pairs, pi, pj, nbr, koff, rev);
    const bool easy = launch_easy(G, ca, pi, pj, rev, n_pairs, asg, hard, keep, s);
    if (!easy) {
      hipLaunchKernelGGL(k_fill_words, dim3(pb), dim3(256), 0, s, hard, n_pairs, 1u);
      hipLaunchKernelGGL(k_fill_words, dim3(pb), dim3(256), 0, s, keep, n_pairs, 0u);
    }
    if (int rc = scan_flags(hard); rc != BRILLE_OK) return rc;
    auto scan_moved = [&]() -> int {
      if (hipMemcpyAsync(moved, keep, n_pairs * 4, hipMemcpyDeviceToDevice, s) != hipSuccess)
        return fail(BRILLE_ERR_DEVICE, "hipMemcpyAsync failed");
      if (int rc = scan_flags(moved); rc != BRILLE_OK) return rc;
      if (hipMemcpyAsync(&n_moved, moved + n_pairs, 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
          hipMemcpyAsync(&n_hard, hard + n_pairs, 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
          hipStreamSynchronize(s) != hipSuccess)
        return fail(BRILLE_ERR_DEVICE, "sort failed");
      return BRILLE_OK;
    };
    if (int rc = scan_moved(); rc != BRILLE_OK) return rc;
    if (n_hard) {
      // listed pairs in chunks whose cost matrices take at most 512 MB
      const uint64_t BB = (uint64_t)d.B * d.B;
      const uint64_t chunk = std::max<uint64_t>(1, std::min<uint64_t>(n_hard, (512ull << 20) / (BB * 8)));
      double* cost = buf.get<double>(chunk * BB);
      uint32_t* list = buf.get<uint32_t>(n_hard);
      uint32_t* todo = buf.get<uint32_t>(chunk);
      if (!cost || !list || !todo) return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the cost matrices");
      hipLaunchKernelGGL(k_pair_list, dim3(pb), dim3(256), 0, s, n_pairs, hard, list);
      const size_t lds_state = 3 * (d.B + 1) * sizeof(double) + ((3 * (d.B + 1) + 1) / 2) * sizeof(double);
      const int cost_in_lds = lds_state + BB * sizeof(double) <= 48 * 1024 ? 1 : 0;
      const size_t lds = lds_state + (cost_in_lds ? BB * sizeof(double) : 0);
      const unsigned lap_blocks = (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(chunk, (uint64_t)std::max(G->n_cu, 1u) * 32));
      for (uint64_t h0 = 0; h0 < n_hard; h0 += chunk) {
        const uint64_t nh = std::min<uint64_t>(chunk, n_hard - h0);
        const unsigned cb = (unsigned)((nh * BB + 255) / 256), qb = (unsigned)((nh + 255) / 256);
        if (d.rows64)
          hipLaunchKernelGGL(k_pair_costs<double>, dim3(cb), dim3(256), 0, s, ca, d.rows64, pi, pj, list, h0, nh, cost, counter + 1);
        else
          hipLaunchKernelGGL(k_pair_costs<float>, dim3(cb), dim3(256), 0, s, ca, d.rows32, pi, pj, list, h0, nh, cost, counter + 1);
        hipLaunchKernelGGL(k_pair_fast, dim3(qb), dim3(256), 0, s, (const double*)cost, d.B, list, h0, nh, rev, asg, keep,
                           todo);
        hipLaunchKernelGGL(k_pair_lap, dim3(lap_blocks), dim3(SORT_BLOCK), lds, s, (const double*)cost, d.B, list, h0, nh,
                           todo, cost_in_lds, rev, asg, keep, counter + 1);
      }
      if (int rc = scan_moved(); rc != BRILLE_OK) return rc;
    }
  }
  const uint32_t n_perms = 1 + 2 * n_moved;
  uint32_t* perms_fit = buf.get<uint32_t>((uint64_t)n_perms * d.B);
  if (!perms_fit) return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the permutation table");
  hipLaunchKernelGGL(k_identity_perm, dim3(1), dim3(256), 0, s, perms_fit, d.B);
  // (whole pairs in each launch, a lane per pair and row)
  const uint64_t most_pairs = kMostBlocks * 256 / d.B;
  for (uint64_t p = 0; p < n_pairs; p += most_pairs) {
    const uint64_t n = std::min(most_pairs, n_pairs - p);
    hipLaunchKernelGGL(k_perm_write, dim3((unsigned)((n * d.B + 255) / 256)), dim3(256), 0, s, n, d.B, asg + p * d.B,
                       moved + p, pk + p, rev + p, pidx, perms_fit);
  }
  if (hipGetLastError() != hipSuccess) return fail(BRILLE_ERR_DEVICE, "sort launch failed");
  uint32_t hc[2] = {0, 0};
  if (hipMemcpyAsync(hc, counter, 8, hipMemcpyDeviceToHost, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "sort failed");
  if (hc[1]) return fail(BRILLE_ERR_NUMERIC, "Complex Hermitian angle cos(theta) > 1 while sorting");
  // install: the previous sorted table goes, and the tables derived from the
  // payload and the permutations with it (the calls queued before this one have
  // ended, and others wait for the handle's lock); a fill-given table stays in
  // the payload allocations until the next fill, and so do tables whose
  // addresses a graph has recorded
  for (std::vector<void*>* old : {&G->sort_allocs, &G->derived_allocs}) {
    if (G->recorded) G->data_allocs.insert(G->data_allocs.end(), old->begin(), old->end());
    else
      for (void* p : *old) (void)hipFree(p);
    old->clear();
  }
  G->recorded = false;
  G->untabled[0] = G->untabled[1] = 0;
  G->tables_pending = false;
  for (void* p : {(void*)keys, (void*)pidx, (void*)perms_fit}) {
    buf.release(p);
    G->sort_allocs.push_back(p);
  }
  d.n_keys = n_keys;
  d.keys = keys;
  d.perm_index = pidx;
  d.perms = perms_fit;
  d.vkey = nullptr;
  d.cell_perm = nullptr;
  G->n_perms = n_perms;
  d.cube_rows32 = nullptr;
  d.cube_rows64 = nullptr;
  d.wide_fac32 = nullptr;
  d.wide_fac64 = nullptr;
  ++G->fill_gen;
  return install_permutations(G, G->sort_allocs, s);
}

extern "C" int brille_grid_permutations(const brille_grid* G, uint64_t* n_keys, uint32_t* n_perms, uint64_t* keys,
                                        uint32_t* perm_index, uint32_t* perms) {
  BRILLE_LOCK_GRID(G);
  if (!G) return fail(BRILLE_ERR_INVALID_ARGUMENT, "null grid");
  if (!G->filled) return fail(BRILLE_ERR_NOT_FILLED, "The interpolation data must be filled first.");
  const DataConst& d = G->d;
  if (n_keys) *n_keys = d.n_keys;
  if (n_perms) *n_perms = d.n_keys ? G->n_perms : 0;
  if (keys && d.n_keys && hipMemcpy(keys, d.keys, d.n_keys * 8, hipMemcpyDeviceToHost) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "hipMemcpy failed");
  if (perm_index && d.n_keys && hipMemcpy(perm_index, d.perm_index, d.n_keys * 4, hipMemcpyDeviceToHost) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "hipMemcpy failed");
  if (perms && d.n_keys && hipMemcpy(perms, d.perms, (uint64_t)G->n_perms * d.B * 4, hipMemcpyDeviceToHost) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "hipMemcpy failed");
  return BRILLE_OK;
}
