// Binned ir_interpolate_at for large calls.
//
// With Q spread over the whole zone, the eight payload rows a point gathers
// are unrelated to those of its neighbours in the input, and on a payload
// larger than the L2 nearly every row comes from HBM.  This pipeline first
// orders the points by trellis node range, so that the points one tile sums
// share their vertices and the rows hit in cache:
//   k_bin_fold     stage (a) + node subscript, one lane per point; a 32-byte
//                  FoldRec and a 4-byte key per point in input order and a
//                  per-block histogram of node-range buckets (failed points
//                  get the last bucket);
//   k_scan_*       exclusive scan of the block histograms (bucket-major);
//   k_bin_scatter  each block moves its keys and input indices to its reserved
//                  slots of each bucket;
//   k_bucket_perm  input indices in node order, bucket by bucket;
//   k_bin_sums     the rest of stage (b) and stages (c1, c2) on node-ordered
//                  tiles, reading FoldRecs and writing output rows at the
//                  input index.
// Within a bucket the order is whatever the LDS atomics give; every point is
// computed independently, so the outputs do not depend on it.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <vector>

#include "grid_state.hpp"

namespace brille_amd {

constexpr int BIN_BLOCK = 256;
constexpr int BIN_PPT = 8;                            // points per thread in the bucketing kernels
constexpr uint32_t BIN_SPAN = BIN_BLOCK * BIN_PPT;   // points per bucketing block
constexpr uint64_t BIN_CHUNK = 1ull << 24;           // points per pass of the pipeline
constexpr uint32_t SCAN_SEG = 4096;                   // elements per scan block (256 x 16)

// point-group operations the binned sums keep a Gamma frame for
constexpr uint32_t kMaxOps = 48;

struct FoldRec {
  double q[3];
  uint32_t node;
  uint32_t meta;  // rot | invrot << 8 | status << 16 | kMetaPoly
};
// the point is on the proposal list: it folded into a polyhedron node of at
// least kPropMinCand tetrahedra (in smaller nodes the exact scan costs no
// more than verifying a proposal, and the network is not run)
constexpr uint32_t kMetaPoly = 1u << 24;
// the same flag on the node words the node-order pass reads (node indices
// stay below 2^31, which the launch checks) and on the perm entries it
// writes (positions within a pass stay below 2^31)
constexpr uint32_t kNodePoly = 1u << 31;
constexpr uint32_t kPermPoly = 1u << 31;
constexpr uint32_t kPropMinCand = 8;
__device__ __forceinline__ uint32_t meta_status(uint32_t meta) { return (meta >> 16) & 255u; }
// what the bucketing moves of a point: its node | kNodePoly (kNoKey: it failed)
// and its input index within the pass.  The record stays where the fold wrote
// it: moving 40 bytes of it cost more than the sums' reading it by index does
// (1e7 points of 2 atoms FP32: bucketing 0.465 -> 0.225 ms, sums 1.75 -> 1.84;
// FP64, 3e6: 0.124 -> 0.077, sums unchanged; a record padded to 64 bytes to
// write whole granules was slower, 0.585).
struct SortKey {
  uint32_t key, index;
};
constexpr uint32_t kNoKey = 0xFFFFFFFFu;  // no node index: those stay below 2^31 - 1

__device__ __forceinline__ uint32_t bucket_of(uint32_t key, uint32_t nb, uint64_t n_nodes) {
  return key == kNoKey ? nb : (uint32_t)(((uint64_t)(key & ~kNodePoly) * nb) / n_nodes);
}

// mark_poly: flag (kMetaPoly) the points for the learned proposal, those
// that folded into polyhedron nodes of at least kPropMinCand tetrahedra; the
// node-order pass lists them
// Six waves per SIMD (a few spilled registers) hide more of the FP64 latency
// than the four that 124 VGPRs allow: 9 % less time.
template <bool Fast>
__global__ __launch_bounds__(BIN_BLOCK) __attribute__((amdgpu_waves_per_eu(6))) void k_bin_fold(GridConst g, const double* Q, uint32_t n, int fold,
                                                        FoldRec* __restrict__ rec, uint32_t* __restrict__ key,
                                                        uint32_t* __restrict__ hist,
                                                        uint32_t nblk, uint32_t nb,
                                                        ErrRec* __restrict__ err, uint64_t base, int mark_poly) {
  extern __shared__ uint32_t h[];  // nb + 1 counters
  for (uint32_t k = threadIdx.x; k <= nb; k += BIN_BLOCK) h[k] = 0;
  __syncthreads();
  const uint32_t b0 = blockIdx.x * BIN_SPAN;
  for (int i = 0; i < BIN_PPT; ++i) {
    const uint32_t p = b0 + i * BIN_BLOCK + threadIdx.x;
    if (p < n) {
      double Qp[3] = {Q[3 * (uint64_t)p], Q[3 * (uint64_t)p + 1], Q[3 * (uint64_t)p + 2]};
      Located L;
      fold_node<Fast>(g, Qp, fold, L);
      if (L.status != BRILLE_PT_OK) report_point(err, base + p, L.status);
      bool poly = false;
      if (mark_poly && L.status == BRILLE_PT_OK && g.node_type[L.node] == BRILLE_NODE_POLY) {
        const uint32_t pi = g.node_index[L.node];
        poly = g.poly_off[pi + 1] - g.poly_off[pi] >= kPropMinCand;
      }
      FoldRec r;
      r.q[0] = L.q[0]; r.q[1] = L.q[1]; r.q[2] = L.q[2];
      r.node = L.node;
      r.meta = (L.rot & 255u) | ((L.invrot & 255u) << 8) | ((uint32_t)L.status << 16) | (poly ? kMetaPoly : 0u);
      rec[p] = r;
      const uint32_t kp = L.status != BRILLE_PT_OK ? kNoKey : poly ? L.node | kNodePoly : L.node;
      key[p] = kp;
      atomicAdd(&h[bucket_of(kp, nb, g.n_nodes)], 1u);
    }
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k <= nb; k += BIN_BLOCK) hist[(uint64_t)k * nblk + blockIdx.x] = h[k];
}

// exclusive scan of 256 values held one per thread; returns the thread's
// exclusive prefix, *total gets the sum
template <int NT = BIN_BLOCK>
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* total) {
  __shared__ uint32_t wsum[NT / 64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t y = __shfl_up(x, o, 64);
    if (lane >= (uint32_t)o) x += y;
  }
  if (lane == 63) wsum[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    if ((uint32_t)w < wave) before += wsum[w];
    all += wsum[w];
  }
  __syncthreads();
  *total = all;
  return before + x - v;
}

__global__ __launch_bounds__(BIN_BLOCK) void k_scan_reduce(const uint32_t* a, uint64_t m, uint32_t* part) {
  const uint64_t s0 = (uint64_t)blockIdx.x * SCAN_SEG;
  uint32_t v = 0;
  for (uint32_t j = 0; j < SCAN_SEG / BIN_BLOCK; ++j) {
    const uint64_t i = s0 + (uint64_t)threadIdx.x * (SCAN_SEG / BIN_BLOCK) + j;
    if (i < m) v += a[i];
  }
  uint32_t total;
  (void)block_exclusive_scan(v, &total);
  if (threadIdx.x == 0) part[blockIdx.x] = total;
}

// one block: exclusive scan of the segment sums in place
__global__ __launch_bounds__(BIN_BLOCK) void k_scan_top(uint32_t* part, uint32_t np) {
  const uint32_t per = (np + BIN_BLOCK - 1) / BIN_BLOCK;
  const uint32_t i0 = threadIdx.x * per;
  uint32_t v = 0;
  for (uint32_t j = 0; j < per; ++j)
    if (i0 + j < np) v += part[i0 + j];
  uint32_t total;
  uint32_t run = block_exclusive_scan(v, &total);
  for (uint32_t j = 0; j < per; ++j)
    if (i0 + j < np) {
      const uint32_t t = part[i0 + j];
      part[i0 + j] = run;
      run += t;
    }
}

__global__ __launch_bounds__(BIN_BLOCK) void k_scan_apply(uint32_t* a, uint64_t m, const uint32_t* part) {
  constexpr uint32_t PER = SCAN_SEG / BIN_BLOCK;
  const uint64_t i0 = (uint64_t)blockIdx.x * SCAN_SEG + (uint64_t)threadIdx.x * PER;
  uint32_t v[PER];
  uint32_t s = 0;
#pragma unroll
  for (uint32_t j = 0; j < PER; ++j) {
    v[j] = i0 + j < m ? a[i0 + j] : 0u;
    s += v[j];
  }
  uint32_t total;
  uint32_t run = block_exclusive_scan(s, &total) + part[blockIdx.x];
#pragma unroll
  for (uint32_t j = 0; j < PER; ++j) {
    if (i0 + j < m) a[i0 + j] = run;
    run += v[j];
  }
}

__global__ __launch_bounds__(BIN_BLOCK) void k_bin_scatter(const uint32_t* key, uint32_t n, const uint32_t* off,
                                                           uint32_t nblk, uint32_t nb, uint64_t n_nodes,
                                                           SortKey* out) {
  extern __shared__ uint32_t s[];  // base[nb + 1], count[nb + 1]
  uint32_t* base = s;
  uint32_t* cnt = s + nb + 1;
  for (uint32_t k = threadIdx.x; k <= nb; k += BIN_BLOCK) {
    base[k] = off[(uint64_t)k * nblk + blockIdx.x];
    cnt[k] = 0;
  }
  __syncthreads();
  const uint32_t b0 = blockIdx.x * BIN_SPAN;
  uint32_t kk[BIN_PPT];  // requested before any is placed
#pragma unroll
  for (int i = 0; i < BIN_PPT; ++i) {
    const uint32_t p = b0 + i * BIN_BLOCK + threadIdx.x;
    if (p < n) kk[i] = key[p];
  }
#pragma unroll
  for (int i = 0; i < BIN_PPT; ++i) {
    const uint32_t p = b0 + i * BIN_BLOCK + threadIdx.x;
    if (p < n) {
      const uint32_t k = bucket_of(kk[i], nb, n_nodes);
      out[base[k] + atomicAdd(&cnt[k], 1u)] = SortKey{kk[i], p};
    }
  }
}

// Node order inside each bucket: one block per bucket counts its points per
// trellis node in LDS and writes perm, the input indices of the bucket's points
// in node order, so that the points of one cube are summed together and its
// rows are read from L1.  Within a node the order is whatever the LDS atomics
// give (the points are independent).  Buckets spanning more than kPermNodes
// nodes, and the failed-point bucket, keep their order.  Each entry carries
// the record's proposal flag (kPermPoly, from kNodePoly).
constexpr uint32_t kPermNodes = 4096;
constexpr int PERM_BLOCK = 1024;
__global__ __launch_bounds__(PERM_BLOCK) void k_bucket_perm(const SortKey* sk, uint32_t m, const uint32_t* off,
                                                           uint32_t nblk, uint32_t nb, uint64_t n_nodes,
                                                           uint32_t* perm) {
  __shared__ uint32_t cnt[kPermNodes];
  const uint32_t b = blockIdx.x;
  const uint32_t s0 = off[(uint64_t)b * nblk];
  const uint32_t s1 = b + 1 <= nb ? off[(uint64_t)(b + 1) * nblk] : m;
  const uint64_t lo = ((uint64_t)b * n_nodes + nb - 1) / nb;
  const uint64_t hi = b < nb ? ((uint64_t)(b + 1) * n_nodes + nb - 1) / nb : lo;
  const uint32_t nn = (uint32_t)(hi - lo);
  if (b == nb || nn == 0 || nn > kPermNodes) {
    for (uint32_t i = s0 + threadIdx.x; i < s1; i += PERM_BLOCK)
      perm[i] = sk[i].index | (sk[i].key == kNoKey ? 0u : sk[i].key & kNodePoly);
    return;
  }
  for (uint32_t k = threadIdx.x; k < nn; k += PERM_BLOCK) cnt[k] = 0;
  __syncthreads();
  for (uint32_t i = s0 + threadIdx.x; i < s1; i += PERM_BLOCK) atomicAdd(&cnt[(sk[i].key & ~kNodePoly) - (uint32_t)lo], 1u);
  __syncthreads();
  // exclusive scan of cnt[0, nn): each thread a contiguous run, then the runs
  const uint32_t per = (nn + PERM_BLOCK - 1) / PERM_BLOCK;
  const uint32_t k0 = threadIdx.x * per, k1 = k0 + per < nn ? k0 + per : nn;
  uint32_t run = 0;
  for (uint32_t k = k0; k < k1; ++k) run += cnt[k];
  uint32_t total;
  uint32_t acc = s0 + block_exclusive_scan<PERM_BLOCK>(run, &total);
  for (uint32_t k = k0; k < k1; ++k) {
    const uint32_t c = cnt[k];
    cnt[k] = acc;
    acc += c;
  }
  __syncthreads();
  for (uint32_t i = s0 + threadIdx.x; i < s1; i += PERM_BLOCK) {
    const SortKey e = sk[i];
    perm[atomicAdd(&cnt[(e.key & ~kNodePoly) - (uint32_t)lo], 1u)] = e.index | (e.key & kNodePoly);
  }
}

// The flagged records (kPermPoly) of perm, listed in perm order: each block
// compacts its 4096 consecutive entries in LDS and appends them with one
// atomic, so the list runs in node order within each block's share.
constexpr int LIST_PPT = 16;
constexpr uint32_t LIST_SPAN = BIN_BLOCK * LIST_PPT;
__global__ __launch_bounds__(BIN_BLOCK) void k_poly_list(const uint32_t* perm, uint32_t m, uint32_t* __restrict__ list,
                                                        uint32_t* __restrict__ count) {
  __shared__ uint32_t s_list[LIST_SPAN];
  __shared__ uint32_t s_n, s_at;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint64_t b0 = (uint64_t)blockIdx.x * LIST_SPAN;
  // each wave a contiguous quarter of the span, 64 entries at a time, so the
  // LDS list keeps perm order within each wave's quarter
  __shared__ uint32_t s_wn[BIN_BLOCK / 64];
  uint32_t local = 0;
  // pass 1: count per wave
  const uint64_t w0 = b0 + (uint64_t)wave * (LIST_SPAN / (BIN_BLOCK / 64));
  for (uint32_t k = 0; k < LIST_SPAN / BIN_BLOCK; ++k) {
    const uint64_t j = w0 + (uint64_t)k * 64u + lane;
    const bool poly = j < m && (perm[j] & kPermPoly) != 0u;
    local += (uint32_t)__popcll(__ballot(poly));
  }
  if (lane == 0) s_wn[wave] = local;
  __syncthreads();
  uint32_t at = 0;
  for (uint32_t w = 0; w < wave; ++w) at += s_wn[w];
  // pass 2: place, in order within the wave's quarter
  for (uint32_t k = 0; k < LIST_SPAN / BIN_BLOCK; ++k) {
    const uint64_t j = w0 + (uint64_t)k * 64u + lane;
    const uint32_t e = j < m ? perm[j] : 0u;
    const bool poly = (e & kPermPoly) != 0u;
    const unsigned long long mask = __ballot(poly);
    if (poly) s_list[at + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = e & ~kPermPoly;
    at += (uint32_t)__popcll(mask);
  }
  if (threadIdx.x == BIN_BLOCK - 1) s_n = at;  // the last wave ends at the block's total
  __syncthreads();
  if (threadIdx.x == 0) s_at = s_n ? atomicAdd(count, s_n) : 0u;
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < s_n; k += BIN_BLOCK) list[s_at + k] = s_list[k];
}

// The learned proposal for the listed records: each wave takes 16 list
// entries at a time (mostly of one node, so the candidate rows the chunk
// reads are mostly the same rows), stages their features and candidate
// ranges in its LDS slice, runs the network and writes the proposed
// tetrahedron to the record's hint.  Grid-stride over the list, whose length
// is read on the device.
__global__ __launch_bounds__(256) void k_bin_propose(GridConst g, ProposalConst pc, const FoldRec* recs, uint32_t* hint,
                                                     const uint32_t* list, const uint32_t* count) {
  // chunks of 16 listed points per wave, four waves per block, grid-stride
  // over the list; blocks past the list's end leave before copying weights
  const uint32_t n = *count;
  if (blockIdx.x * 64u >= n) return;
  __shared__ float s_feat[4][48];
  __shared__ uint32_t s_t0[4][16], s_nc[4][16], s_out[4][16];
  // the first two layers' weights, from LDS copies
  __shared__ float s_w1[3 * kPropH], s_b1[kPropH], s_b2[kPropH];
  __shared__ __attribute__((aligned(16))) uint16_t s_w2[kPropH * kPropH];
  for (uint32_t i = threadIdx.x; i < 3 * kPropH; i += 256) s_w1[i] = pc.W1[i];
  for (uint32_t i = threadIdx.x; i < kPropH; i += 256) {
    s_b1[i] = pc.b1[i];
    s_b2[i] = pc.b2[i];
  }
  for (uint32_t i = threadIdx.x; i < kPropH * kPropH / 8; i += 256)
    reinterpret_cast<uint4*>(s_w2)[i] = reinterpret_cast<const uint4*>(pc.W2)[i];
  __syncthreads();
  const PropWeights<LdsF, LdsH> W{(LdsF)s_w1, (LdsF)s_b1, (LdsF)s_b2, (LdsH)s_w2};
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  // wave-uniform loop; no block-wide barrier follows
  for (uint32_t c0 = (blockIdx.x * 4u + wave) * 16u; c0 < n; c0 += gridDim.x * 64u) {
  const uint32_t k = n - c0 < 16u ? n - c0 : 16u;
  uint32_t rec = 0;
  if (lane < k) {
    rec = list[c0 + lane];
    const FoldRec& r = recs[rec];
    const double q[3] = {r.q[0], r.q[1], r.q[2]};
    const uint32_t nd = r.node;
    double x[3];
    mat_vec(x, g.outer_to_xyz, q);
    float f[3];
    prop_features(g, x, nd, f);
    s_feat[wave][3 * lane] = f[0];
    s_feat[wave][3 * lane + 1] = f[1];
    s_feat[wave][3 * lane + 2] = f[2];
    const uint32_t pi = g.node_index[nd];
    const uint32_t a = g.poly_off[pi];
    s_t0[wave][lane] = a;
    s_nc[wave][lane] = g.poly_off[pi + 1] - a;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  propose16_inline(pc, W, s_feat[wave], s_t0[wave], s_nc[wave], k, s_out[wave]);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (lane < k) hint[rec] = s_out[wave][lane];
  // the next chunk overwrites this wave's LDS slices
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// XCD-aware tile order: the hardware hands consecutive blocks to the eight
// XCDs in turn, each with its own L2.  Block b runs on XCD b % 8, so giving XCD
// x the contiguous tiles [start(x), start(x) + count(x)) keeps a bucket's
// records and rows in one L2 instead of fetching them into all eight.  The
// map is a bijection for any grid size.
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t xcd_tile(uint32_t b, uint32_t nb) {
  const uint32_t q = nb / kXcds, r = nb % kXcds;
  const uint32_t x = b % kXcds, i = b / kXcds;
  return x * q + (x < r ? x : r) + i;
}

// points a block of the sums holds: the atom-major wide sums run as fast with 64
// as with 128 or 256 (24 atoms, 300 007 points of 72 modes FP32 5.2 ms), which
// leaves the LDS to the records being assembled
constexpr uint32_t sums_points(int L, int SC) { return L == LAYOUT_WIDE && wide_atom_major(SC) ? 64u : (uint32_t)TILE; }

// waves per SIMD asked of the compiler: the atom-major wide sums run best at
// four (FP32) and two (FP64), a few registers below what it would take for
// the antiphases of the rare points without a table block, and so do the narrow
// Gamma sums, whose one-lane-per-unit sums of those points would take up to
// twice the registers of the rest.  (Two atoms FP64 at three waves: 112 bytes
// of scratch in the walk, 3 000 017 points 1.03 -> 1.92 ms.)
template <typename Real, int L, int SC>
constexpr int sums_waves() {
  if (L == LAYOUT_WIDE && wide_atom_major(SC)) return sizeof(Real) == 4 ? 4 : 2;
  if (L == LAYOUT_GAMMA) return sizeof(Real) == 4 ? 4 : 2;
  return 1;
}
template <typename Real, int L, int SC, int SV, bool Prop>
__global__ __launch_bounds__(TILE) __attribute__((amdgpu_waves_per_eu(sums_waves<Real, L, SC>())))
void k_bin_sums(GridConst g, DataConst d, ProposalConst pc, const FoldRec* recs, const uint32_t* hint,
                                                    const uint32_t* perm, uint32_t n, void* __restrict__ vals,
                                                    void* __restrict__ vecs, brille_aux_out aux,
                                                    ErrRec* __restrict__ err, uint64_t base, uint32_t tile_pts) {
  using C = typename Cplx<Real>::T;
  constexpr int WSL = wide_bin_slots<Real>();
  using S = TileShape<L, SC, TILE, Real, WSL>;
  constexpr bool kWide = L == LAYOUT_WIDE;
  constexpr uint32_t TP = sums_points(L, SC);
  __shared__ PointRec<Real> s_rec[TP];
  // wide rows: the phase table of the node-ordered Gamma sums instead
  constexpr uint32_t kPh =
      kWide ? (wide_atom_major(SC) ? kWideAtomPhaseBytes : kWidePhaseBytes) / sizeof(C) : TILE * S::NPH;
  __shared__ C s_ph[kPh];
  __shared__ Real s_wrot[kWide ? 9 * kMaxOps : 1];
  __shared__ uint8_t s_wdst[kWide ? kWideAtoms * kMaxOps : 1];
  // Gamma layout: one frame per point-group operation instead of one per
  // point (12 KB less LDS in FP32, 20 KB in FP64)
  constexpr bool kOpFrames = L == LAYOUT_GAMMA;
  __shared__ double s_q[kWide ? S::NQ / TILE * TP : kOpFrames ? 1 : S::NQ];
  __shared__ GammaFrame<Real> s_frames[kOpFrames ? kMaxOps : 1];
  if (kOpFrames && threadIdx.x < g.G) fill_frame<Real, SC>(g, d, threadIdx.x, s_frames[threadIdx.x]);
  __shared__ uint32_t s_out[TP];
  // wide rows' slices, or the atom lanes' records
  constexpr bool kAtoms = kWide && wide_atom_major(SC);
  constexpr uint32_t kWalk = kOpFrames ? TILE / 64 * walk_slice<Real>() / sizeof(C)
                             : kAtoms  ? TILE / 64 * wide_walk_slice<Real>(WSL)
                                       : 1;
  __shared__ __attribute__((aligned(16))) C s_wide[(uint32_t)S::NW > kWalk ? S::NW : kWalk];
  __shared__ uint32_t s_tried, s_verified;
  if (Prop && threadIdx.x == 0) {
    s_tried = 0;
    s_verified = 0;
  }
  // wide rows take fewer points per block in passes of few points (tile_pts of
  // the TP a block's LDS holds); the others always TP
  const uint32_t tile_n = kWide ? tile_pts : TP;
  const uint32_t tile0 = xcd_tile(blockIdx.x, gridDim.x) * tile_n;
  const uint32_t tid = threadIdx.x;
  const uint32_t p = tile0 + tid;
  // wide rows: blockIdx.y picks a group of modes (gridDim.y groups; the
  // first one reports the points' errors and aux outputs)
  const bool lead = blockIdx.y == 0;
  uint32_t per_group = (d.B + gridDim.y - 1) / gridDim.y;
  if (L == LAYOUT_WIDE && wide_atom_major(SC)) {  // whole passes of the atom-major walk
    const uint32_t mpw = wide_pass_modes(d.sc, sizeof(C));
    per_group = (per_group + mpw - 1) / mpw * mpw;
  }
  const uint32_t b_lo = blockIdx.y * per_group, b_hi = b_lo + per_group;
  const bool want_phase = d.vec_rot == BRILLE_ROT_GAMMA && d.ec[1] > 0;
  const uint32_t n_atoms = d.ec[1] / 3u;
  const bool ph_in_lds = L == LAYOUT_GAMMA || (want_phase && n_atoms <= 4);
  WideGammaLds<Real> wg;
  if (kWide && want_phase) {
    wg.ph = s_ph;
    wg.rot = s_wrot;
    wg.dst = s_wdst;
    wg.cap = kPh;
    wide_gamma_ops<Real, TILE>(g, d, wg);
  }
  __shared__ uint32_t s_wave_tab[TILE / 64];
  if (Prop) __syncthreads();
  const bool live = tid < tile_n && p < n;
  FoldRec sr;
  uint32_t index = 0, tet_hint = kNoTet;
  Located P;
  P.status = BRILLE_PT_OK;
  P.cube = kNoCube;
  if (live) {
    const uint32_t e = perm[p];
    index = e & ~kPermPoly;
    sr = recs[index];
    if (Prop) tet_hint = (e & kPermPoly) ? hint[index] : kNoTet;
    P.q[0] = sr.q[0]; P.q[1] = sr.q[1]; P.q[2] = sr.q[2];
    P.tau[0] = P.tau[1] = P.tau[2] = 0;
    P.node = sr.node;
    P.rot = sr.meta & 255u;
    P.invrot = (sr.meta >> 8) & 255u;
    P.status = (int)meta_status(sr.meta);
    P.tet = kNoTet;
    P.nslot = 0;
    P.nkept = 0;
    if (P.status == BRILLE_PT_OK) {
      if constexpr (Prop) {
        bool verified = false;
        node_slots(g, P, tet_hint, pc.margin, &verified);
        if (tet_hint != kNoTet) {
          atomicAdd(&s_tried, 1u);
          if (verified) atomicAdd(&s_verified, 1u);
        }
      } else {
        node_slots(g, P);
      }
      // failed fold-ins were reported by k_bin_fold
      if (P.status != BRILLE_PT_OK && lead) report_point(err, base + index, P.status);
    }
  }
  // Stable partition of the tile: points the cube factor table serves first,
  // so that few waves of the sums mix the two kinds of point.
  // (a GammaTable that is not one to one keeps to the sums of one lane per unit)
  const bool table = ((L == LAYOUT_GAMMA && d.gamma_maps) || L == LAYOUT_SCALAR) && cube_rows<Real>(d) != nullptr;
  const bool tab = table && live && P.status == BRILLE_PT_OK && table_row(d, P) != kNoCube;
  const uint32_t lane = tid & 63u, wave = tid >> 6;
  const unsigned long long bal = __ballot(tab);
  const uint32_t rank = (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
  if (lane == 0) s_wave_tab[wave] = (uint32_t)__popcll(bal);
  __syncthreads();
  uint32_t before = 0, n_tab = 0;
#pragma unroll
  for (uint32_t w = 0; w < TILE / 64; ++w) {
    const uint32_t c = s_wave_tab[w];
    before += w < wave ? c : 0u;
    n_tab += c;
  }
  const uint32_t slot = tab ? before + rank : n_tab + (tid - before - rank);
  if (tid < TP) {
    PointRec<Real>& r = s_rec[slot];
    r.nslot = 0;
    if (live) {
      s_out[slot] = index;
      if (P.status == BRILLE_PT_OK)
        store_record<Real, L, SC>(g, d, P, r, s_ph, s_q, slot, ph_in_lds, n_atoms, !kOpFrames);
      if (lead) write_aux(aux, index, P);
    }
  }
  __syncthreads();
  if (Prop && lead && threadIdx.x == 0 && s_tried) {
    atomicAdd(&pc.stats[0], (unsigned long long)s_tried);
    atomicAdd(&pc.stats[1], (unsigned long long)s_verified);
  }
  const uint32_t npts = n - tile0 < tile_n ? n - tile0 : tile_n;
  const uint32_t* pm = nullptr;
  if (d.n_keys) {  // the row table's rows are permuted already
    tile_perms<TILE>(d, s_rec, n_tab, npts, s_perms);
    __syncthreads();
    pm = s_perms;
  }
  // the one-lane-per-unit sums see only the points the table does not serve:
  // fewer rows in flight keep the registers for occupancy
  constexpr int GRP = sizeof(Real) == 4 ? 2 : 1;
  tile_sums<Real, true, L, SC, SV, TILE, GRP, WSL>(g, d, s_rec, s_ph, s_q, s_out, 0, npts, ph_in_lds, vals, vecs, s_wide,
                                              table, n_tab, kOpFrames ? s_frames : nullptr, true, wg, b_lo, b_hi, pm);
}

// The row table: thread t = (block row, mode b) phases the row of a cube's or
// tetrahedron's slot-x vertex against the row of its slot-0 vertex with the
// sums' own functions, so a point summed from the table gets the same bits.
template <typename Real, int SC>
__global__ __launch_bounds__(256) void k_table_rows(GridConst g, DataConst d, uint64_t n_cube_units,
                                                    uint64_t n_units, Real* out) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_units) return;
  uint32_t pv, sv;
  uint32_t b;
  if (t < n_cube_units) {
    const uint64_t cx = t / d.B;
    b = (uint32_t)(t - cx * d.B);
    const uint32_t* v = g.cube_v + 8 * (cx >> 3);
    pv = v[7];
    sv = v[7 - (int)(cx & 7u)];
  } else {
    const uint64_t tx = (t - n_cube_units) / d.B;
    b = (uint32_t)(t - n_cube_units - tx * d.B);
    const uint32_t* v = g.tet_v + 4 * (tx >> 2);
    pv = v[0];
    sv = v[tx & 3u];
  }
  const Real* base = payload_rows<Real>(d);
  const uint64_t stride = payload_stride<Real>(d);
  Real pr[2 * SC];
  load_row<Real, 2 * SC>(pr, base + ((uint64_t)pv * d.B + b) * stride);
  const uint32_t bs = d.cell_perm ? perm_mode(d, d.cell_perm[t / d.B], b) : b;
  const Real* src = base + ((uint64_t)sv * d.B + bs) * stride;
  Real row[2 * SC];
  load_row<Real, 2 * SC>(row, src);
  const typename Cplx<Real>::T e = slot_antiphase<Real, SC>(pr, row);
  Real* dst = out + t * stride;
  for (int k = 0; k < SC; ++k) phase_elem<Real>(e, row[2 * k], row[2 * k + 1], &dst[2 * k], &dst[2 * k + 1]);
  for (uint32_t k = 2 * SC; k < stride; ++k) dst[k] = src[k];  // values and zero padding
}

// The wide factor table: wave w = (block row, mode b) computes the antiphases
// of a cube's eight or a tetrahedron's four slot rows against its slot-0 row
// with the sums' own wave-wide function (same lanes, same reductions), so a
// point summed from the table gets the same bits.
template <typename Real>
__global__ __launch_bounds__(256) void k_wide_factors(GridConst g, DataConst d, uint64_t n_cube_units,
                                                      uint64_t n_units, typename Cplx<Real>::T* out) {
  using C = typename Cplx<Real>::T;
  const uint64_t t = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= n_units) return;  // wave-uniform
  const uint32_t l = threadIdx.x & 63u;
  const uint32_t sc = d.sc;
  const bool h0 = l < sc, h1 = l + 64u < sc;
  uint32_t v[8], ns, b;
  uint64_t trow;
  if (t < n_cube_units) {
    const uint64_t c = t / d.B;
    b = (uint32_t)(t - c * d.B);
#pragma unroll
    for (int x = 0; x < 8; ++x) v[x] = g.cube_v[8 * c + 7 - x];
    ns = 8;
    trow = c * 8 * d.B;
  } else {
    const uint64_t tt = (t - n_cube_units) / d.B;
    b = (uint32_t)(t - n_cube_units - tt * d.B);
#pragma unroll
    for (int x = 0; x < 8; ++x) v[x] = g.tet_v[4 * tt + (x < 4 ? x : 0)];
    ns = 4;
    trow = d.tab_tet_row + tt * 4 * d.B;
  }
  const C zero = Elem<C>::zero();
  C v0[8], v1[8], e[8];
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    const uint32_t bx =
        d.cell_perm && (uint32_t)x < ns ? perm_mode(d, d.cell_perm[trow / d.B + x], b) : b;
    const C* rc = reinterpret_cast<const C*>(row_at<Real>(d, v[x], bx));
    v0[x] = h0 ? rc[l] : zero;
    v1[x] = h1 ? rc[l + 64] : zero;
  }
  wide_antiphases<Real, 8>(v0[0], v1[0], v0, v1, e, sc);
  if (l == 0) {
#pragma unroll
    for (int x = 0; x < 8; ++x)
      if ((uint32_t)x < ns) out[trow + (uint64_t)x * d.B + b] = e[x];
  }
}

// The same for Gamma rows summed atom-major: a wave forms the factors of the
// mpw modes of one pass of a block (wide_atom_antiphases, as the sums do).
template <typename Real>
__global__ __launch_bounds__(256) void k_wide_atom_factors(GridConst g, DataConst d, uint64_t n_cube_units,
                                                           uint64_t n_units, typename Cplx<Real>::T* out) {
  using C = typename Cplx<Real>::T;
  constexpr int SL = wide_bin_slots<Real>();
  __shared__ C s_lds[4 * wide_atom_slice<Real>(SL)];
  const uint64_t t = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= n_units) return;  // wave-uniform; no block-wide barrier follows
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t na = d.sc / 3u, mpw = 64u / na, passes = (d.B + mpw - 1) / mpw;
  const uint32_t m = lane / na, a = lane - m * na;
  const bool cube = t < n_cube_units;
  const uint64_t u = cube ? t : t - n_cube_units;
  const uint64_t c = u / passes;
  const uint32_t b = (uint32_t)(u - c * passes) * mpw + m;
  const bool on = m < mpw && b < d.B;
  const uint32_t ns = cube ? 8u : 4u;
  const uint64_t trow = cube ? c * 8 * d.B : d.tab_tet_row + c * 4 * d.B;
  C v[8][3], e[8];
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    const bool use = on && x < (int)ns;
    const uint32_t vert = cube ? g.cube_v[8 * c + 7 - x] : g.tet_v[4 * c + (x & 3)];
    const uint32_t bx = use && d.cell_perm ? perm_mode(d, d.cell_perm[trow / d.B + x], b) : (on ? b : 0u);
    const C* rc = reinterpret_cast<const C*>(row_at<Real>(d, vert, bx)) + 3u * a;
#pragma unroll
    for (int i = 0; i < 3; ++i) v[x][i] = use ? rc[i] : Elem<C>::zero();
  }
  wide_atom_antiphases<Real, SL>(v[0], v, ns, na, mpw, m, e, s_lds + (threadIdx.x >> 6) * wide_atom_slice<Real>(SL));
  if (on && a == 0) {
#pragma unroll
    for (int x = 0; x < 8; ++x)
      if ((uint32_t)x < ns) out[trow + (uint64_t)x * d.B + b] = e[x];
  }
}

using SumsKernel = void (*)(GridConst, DataConst, ProposalConst, const FoldRec*, const uint32_t*, const uint32_t*, uint32_t, void*,
                           void*, brille_aux_out, ErrRec*, uint64_t, uint32_t);

template <typename Real>
static SumsKernel pick_sums(const DataConst& d, bool prop) {
  const int L = payload_layout(d);
  if (prop) {
    // the learned proposal is instantiated for the two-atom Gamma payload and the general layout
    if (L == LAYOUT_GAMMA && d.sv == 1 && d.sc == 6) return k_bin_sums<Real, LAYOUT_GAMMA, 6, 1, true>;
    return k_bin_sums<Real, LAYOUT_GENERIC, 0, 0, true>;
  }
  if (L == LAYOUT_GAMMA && d.sv == 1) {
    switch (d.sc) {
      case 3: return k_bin_sums<Real, LAYOUT_GAMMA, 3, 1, false>;
      case 6: return k_bin_sums<Real, LAYOUT_GAMMA, 6, 1, false>;
      case 9: return k_bin_sums<Real, LAYOUT_GAMMA, 9, 1, false>;
      case 12: return k_bin_sums<Real, LAYOUT_GAMMA, 12, 1, false>;
      default: break;
    }
  }
  if (L == LAYOUT_SCALAR && d.sv == 1) {
    switch (d.sc) {
      case 1: return k_bin_sums<Real, LAYOUT_SCALAR, 1, 1, false>;
      case 2: return k_bin_sums<Real, LAYOUT_SCALAR, 2, 1, false>;
      case 3: return k_bin_sums<Real, LAYOUT_SCALAR, 3, 1, false>;
      case 4: return k_bin_sums<Real, LAYOUT_SCALAR, 4, 1, false>;
      default: break;
    }
  }
  if (wide_by_atom(d))
    return d.gamma_maps ? k_bin_sums<Real, LAYOUT_WIDE, kWideAtom, 0, false> : k_bin_sums<Real, LAYOUT_WIDE, kWideLoose, 0, false>;
  if (wide_rows(d, sizeof(Real) == 4 ? BRILLE_FP32 : BRILLE_FP64)) return k_bin_sums<Real, LAYOUT_WIDE, kWideAll, 0, false>;
  return k_bin_sums<Real, LAYOUT_GENERIC, 0, 0, false>;
}

// Points per block and mode groups (blockIdx.y) of the sums of a pass of m
// points.  Wide rows put a tile's modes in sequence on its four waves, so a
// pass of few points would leave most CUs idle: its tiles shrink until the
// pass has about eight blocks per CU or kLeastWideTile points are left (below
// that the runs of one table block are cut), then the modes split over blocks
// (each group repeats phase 1 and its points' Gamma phases).  The atom-major
// sums take eight mode passes per block, two per wave, however many the points:
// blocks of a whole tile's modes ran for milliseconds, four at a time on a CU,
// and left most of them idle at the end (72 modes FP32, 300 007 points: all 36
// passes in a block 6.6 ms, 16 5.4, 8 5.1, 6 (two of four waves idle in the
// second round) 5.8, 4 5.1, 2 5.6); fewer where even these leave under ten
// blocks per CU (10 001 points: eight 0.50 ms, four 0.47; 3 001: eight 0.30,
// two 0.26).  Other kernels pick_sums selects (the proposal's among them): TILE
// points, one group.
constexpr uint32_t kLeastWideTile = 32;
static void sum_split(const brille_grid* G, uint32_t m, bool prop, int precision, uint32_t* tile, uint32_t* groups) {
  *tile = TILE;
  *groups = 1;
  const DataConst& d = G->d;
  if (prop || !wide_rows(d, precision)) return;
  const bool atoms = wide_by_atom(d);
  if (atoms) *tile = sums_points(LAYOUT_WIDE, kWideAtom);
  const uint64_t want = 8ull * std::max<uint32_t>(G->n_cu, 1);
  while (*tile > kLeastWideTile && (m + *tile - 1) / *tile < want) *tile >>= 1;
  const uint64_t tiles = std::max<uint64_t>((m + *tile - 1) / *tile, 1);
  if (!atoms) {
    *groups = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(want / tiles, (d.B + 3) / 4));
    return;
  }
  const uint32_t mpw = wide_pass_modes(d.sc, precision == BRILLE_FP32 ? 8u : 16u);
  const uint32_t passes = (d.B + mpw - 1) / mpw;
  uint32_t per = 8;
  while (per > 2 && tiles * ((passes + per - 1) / per) < 5 * want / 4) per >>= 1;
  *groups = std::max<uint32_t>((passes + per - 1) / per, 1);
}

// SC of the one-pass sums kernel pick_sums selects, or 0 for the general ones
int onepass_sc(const DataConst& d) {
  const int L = payload_layout(d);
  if (d.sv != 1) return 0;
  if (L == LAYOUT_GAMMA && (d.sc == 3 || d.sc == 6 || d.sc == 9 || d.sc == 12)) return (int)d.sc;
  if (L == LAYOUT_SCALAR && d.sc >= 1 && d.sc <= 4) return (int)d.sc;
  return 0;
}

template <typename Real>
static uint64_t payload_stride_host(const DataConst& d) {
  return sizeof(Real) == 8 ? d.stride64 : d.stride32;
}

// The build of a table is queued on one stream and its address published at
// once, so that the call that builds it need not wait on the host (two atoms
// FP64, 3 000 017 points: first call 2090 us, 2170 with a wait).  Where the call
// returns without a wait, calls on other streams wait for an event (end_binned).
static int end_build(brille_grid* G) {
  if (hipGetLastError() != hipSuccess) return fail(BRILLE_ERR_DEVICE, "building a derived table failed");
  G->tables_touched = true;
  return BRILLE_OK;
}

int await_tables(brille_grid* G, hipStream_t s) {
  if (!G->tables_pending) return BRILLE_OK;
  if (!recording(s)) {
    if (hipStreamWaitEvent(s, G->tables_built, 0) != hipSuccess)
      return fail(BRILLE_ERR_DEVICE, "waiting for the derived tables failed");
    return BRILLE_OK;
  }
  // (a graph cannot wait for an event from outside it)
  if (hipEventSynchronize(G->tables_built) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "waiting for the derived tables failed");
  G->tables_pending = false;
  return BRILLE_OK;
}

template <typename Real>
static int build_cube_rows(brille_grid* G, hipStream_t s, const Real** out) {
  const DataConst& d = G->d;
  const uint64_t cube_units = G->n_cubes * 8 * d.B;
  const uint64_t units = cube_units + G->n_tets * 4 * d.B;
  void* p = nullptr;
  if (hipMalloc(&p, units * payload_stride_host<Real>(d) * sizeof(Real)) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the cube row table");
  G->derived_allocs.push_back(p);
  Real* t = static_cast<Real*>(p);
  const dim3 grid((unsigned)((units + 255) / 256));
  switch (onepass_sc(d)) {
    case 1: hipLaunchKernelGGL((k_table_rows<Real, 1>), grid, dim3(256), 0, s, G->g, d, cube_units, units, t); break;
    case 2: hipLaunchKernelGGL((k_table_rows<Real, 2>), grid, dim3(256), 0, s, G->g, d, cube_units, units, t); break;
    case 3: hipLaunchKernelGGL((k_table_rows<Real, 3>), grid, dim3(256), 0, s, G->g, d, cube_units, units, t); break;
    case 4: hipLaunchKernelGGL((k_table_rows<Real, 4>), grid, dim3(256), 0, s, G->g, d, cube_units, units, t); break;
    case 6: hipLaunchKernelGGL((k_table_rows<Real, 6>), grid, dim3(256), 0, s, G->g, d, cube_units, units, t); break;
    case 9: hipLaunchKernelGGL((k_table_rows<Real, 9>), grid, dim3(256), 0, s, G->g, d, cube_units, units, t); break;
    case 12: hipLaunchKernelGGL((k_table_rows<Real, 12>), grid, dim3(256), 0, s, G->g, d, cube_units, units, t); break;
    default: return fail(BRILLE_ERR_UNSUPPORTED, "no cube row kernel for this payload");
  }
  if (int rc = end_build(G); rc != BRILLE_OK) return rc;
  *out = t;
  return BRILLE_OK;
}

template <typename Real>
static int build_wide_factors(brille_grid* G, hipStream_t s, const typename Cplx<Real>::T** out) {
  using C = typename Cplx<Real>::T;
  const DataConst& d = G->d;
  const bool atom = wide_by_atom(d);
  const uint64_t mpw = 64u / (d.sc / 3u);
  const uint64_t per = atom ? (d.B + mpw - 1) / mpw : d.B;  // waves per block
  const uint64_t cube_units = G->n_cubes * per;
  const uint64_t units = cube_units + G->n_tets * per;
  void* p = nullptr;
  if (hipMalloc(&p, (G->n_cubes * 8 + G->n_tets * 4) * d.B * sizeof(C)) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the wide factor table");
  G->derived_allocs.push_back(p);
  C* t = static_cast<C*>(p);
  if (atom)
    hipLaunchKernelGGL((k_wide_atom_factors<Real>), dim3((unsigned)((units + 3) / 4)), dim3(256), 0, s, G->g, d,
                       cube_units, units, t);
  else
    hipLaunchKernelGGL((k_wide_factors<Real>), dim3((unsigned)((units + 3) / 4)), dim3(256), 0, s, G->g, d, cube_units,
                       units, t);
  if (int rc = end_build(G); rc != BRILLE_OK) return rc;
  *out = t;
  return BRILLE_OK;
}

// Bytes of the payload's derived table of a precision: the antiphased rows (8 per
// cube, 4 per tetrahedron and mode) for the one-pass layouts, the antiphase
// factors alone for wide rows.  The general layout, grids without cells and
// tables beyond kCubeRowsMax go without (0), and their sums compute every
// antiphase on the fly.
constexpr uint64_t kCubeRowsMax = (4ull << 30) - 1;  // the sums address the table with 32-bit offsets
static uint64_t table_bytes(const brille_grid* G, int precision) {
  const DataConst& d = G->d;
  if (!d.has_blocks) return 0;
  const bool f32 = precision == BRILLE_FP32;
  const uint64_t row = wide_rows(d, precision) ? (f32 ? 8 : 16)
                       : onepass_sc(d) == 0   ? 0
                       : f32                  ? d.stride32 * 4ull
                                              : d.stride64 * 8ull;
  const uint64_t bytes = (G->n_cubes * 8 + G->n_tets * 4) * d.B * row;
  return bytes > kCubeRowsMax ? 0 : bytes;
}

// the derived table of a precision exists (or the payload has none)
static bool has_table(const DataConst& d, int precision) {
  if (wide_rows(d, precision)) return precision == BRILLE_FP32 ? d.wide_fac32 != nullptr : d.wide_fac64 != nullptr;
  if (onepass_sc(d) == 0) return true;
  return precision == BRILLE_FP32 ? d.cube_rows32 != nullptr : d.cube_rows64 != nullptr;
}

// Builds that table once (freed with the payload, or when a sort replaces the
// permutations it follows), on a stream that has waited for any other build of
// the handle's (await_tables).
int ensure_cube_rows(brille_grid* G, int precision, hipStream_t s) {
  DataConst& d = G->d;
  if (table_bytes(G, precision) == 0 || has_table(d, precision)) return BRILLE_OK;
  const bool wide = wide_rows(d, precision);
  if (precision == BRILLE_FP32)
    return wide ? build_wide_factors<float>(G, s, &d.wide_fac32) : build_cube_rows<float>(G, s, &d.cube_rows32);
  return wide ? build_wide_factors<double>(G, s, &d.wide_fac64) : build_cube_rows<double>(G, s, &d.cube_rows64);
}

// Buckets of at most kNodesPerBucket trellis nodes: k_bucket_perm orders each
// bucket by node in LDS (kPermNodes counters), so the buckets only have to be
// few enough that a bucketing block (BIN_SPAN points) puts runs of keys into
// each: the scatter writes a block's keys of one bucket as one run, and short
// runs cost partial-line writes.  A grid of few nodes
// still gets kMinBuckets of them (at most one per node): k_bucket_perm runs a
// block per bucket, and sixteen blocks left the chip idle (1e7 points of a
// 360-node grid: bucketing 1.24 ms with 16).
constexpr uint32_t kNodesPerBucket = kPermNodes;
constexpr uint32_t kMinBuckets = 256;
static uint32_t bucket_count(const brille_grid* G) {
  const uint64_t n_nodes = std::max<uint64_t>(G->g.n_nodes, 1);
  uint32_t nb = kMinBuckets;
  while (nb < 2048 && (uint64_t)nb * kNodesPerBucket < n_nodes) nb <<= 1;
  return (uint32_t)std::min<uint64_t>(nb, n_nodes);
}

// AUTO's choice between the fused tile kernel and the binned pipeline, on the
// complex elements summed (n B sc) of Gamma rows.  The pipeline's fixed cost is
// nine launches; its sums read antiphased rows and reuse them over a node's
// points.  Measured with the tables built, tile against binned (us):
//   2 atoms FP32: 300 007 points 140 / 160, 600 011 256 / 218 (46 MB payload
//     330 / 328); FP64: 100 003 128 / 125, 200 003 239 / 160 (93 MB: 299 / 286)
//   4 atoms FP32: 60 013 138 / 150, 100 003 235 / 152; FP64: 60 013 157 / 155
//   10 atoms FP32: 10 007 129 / 130, 30 001 270 / 164; FP64: 3001 96 / 130
//   24 atoms FP32: 3001 263 / 261, 10 001 796 / 482; FP64: 1001 290 / 233
// (a lower line for wide FP32 rows gained 3 % at 3001 points of a coarser grid
// and cost the table's 0.4 ms on each first call).
// With fewer than two points a cell the narrow rows are reused too little
// (4 atoms FP64, 49 583 points of 34 973 cells: 213 / 236).  A table that is not
// there yet: see table_due.
// Rows of one to four scalars are so short that bucketing them costs more than
// it saves until a call sums many: payloads of 12 to 420 MB, tile / binned (us),
//   FP64: 1 element 2 000 003 points 598 / 546 (1 000 003: 310 / 343), 2 elements
//     1 000 003 492 / 405 (600 011: 305 / 317), on a grid of a million cells
//     578 / 707 (2 000 003: 1107 / 1044); 4 elements 300 007 336 / 330
//   FP32: 1 element 4 000 037 810 / 754 (2 000 003: 415 / 431), 2 elements
//     2 000 003 596 / 512 (1 000 003: 311 / 320), 4 elements 1 000 003 493 / 400
//     (600 011: 307 / 313), on the million cells 576 / 694 (2 000 003: 1107 / 1026)
// Longer rows, which the general sums read twice, take the pipeline like any
// other: 8 elements FP64, 49 MB, 300 007 points 3656 / 991.
// A call whose work space is not ordered after its other users' (`shared`
// false: allocation-free calls, and calls that a graph records, which may not
// build the table either) is binned only on payloads beyond the L2 and from
// 2^18 points on.
bool binned_applies(const brille_grid* G, const LaunchArgs& a, int kernel, int precision, bool shared) {
  if (kernel == BRILLE_KERNEL_PLAIN || kernel == BRILLE_KERNEL_TILE) return false;
  const brille_aux_out& x = a.aux;
  // the records carry no tau; the sums keep a Gamma frame per point-group
  // operation (a crystallographic point group has at most 48)
  if (x.tau || G->g.G > kMaxOps) return false;
  if (a.use_proposal || kernel == BRILLE_KERNEL_BINNED) return true;
  if (x.ir_q || x.rot || x.invrot || x.node || x.tet || x.n_iw || x.iw_index || x.iw_weight || x.status)
    return false;
  if (G->g.n_nodes >= kNodePoly) return false;  // the pipeline refuses such grids, the fused kernel takes them
  const DataConst& d = G->d;
  const uint64_t payload = (uint64_t)d.V * d.B * d.stride32 * 4;
  const uint64_t work = a.n * d.B * d.sc, cells = G->n_cubes + G->n_tets / 2;
  // large calls on payloads that do not fit the L2 of one XCD
  if (a.n >= (1ull << 18) && payload > (8ull << 20)) {
    const bool short_rows = payload_layout(d) == LAYOUT_SCALAR && onepass_sc(d) != 0;
    if (!short_rows || payload > (512ull << 20)) return true;
    if (precision == BRILLE_FP32) return work >= 26000000ull && a.n >= cells;
    return d.sc >= 4 ? work >= 7000000ull : work >= 14000000ull && 2 * a.n >= cells;
  }
  if (!shared || payload_layout(d) != LAYOUT_GAMMA || !(wide_rows(d, precision) || onepass_sc(d))) return false;
  if (wide_rows(d, precision)) return work >= (precision == BRILLE_FP32 ? 20000000ull : 4000000ull);
  return a.n >= 2 * cells && work >= (precision == BRILLE_FP32 ? 13000000ull : 7000000ull);
}

// Whether an ordinary call of n points may build the table it is to be summed
// from.  Building costs what the fused kernel takes for so many points a cell:
// narrow rows FP64 14, FP32 24, wide rows 1.5 and 2.5 (a first call of 4 atoms
// FP64, 10 757 cells, 99 166 points, 9 a cell: 431 us against 362 fused, 18 a
// cell 480 against 720; 2 atoms FP32, 20 a cell 249 against 188, 40 a cell 320
// against 353; 24 atoms FP64, 1 a cell 1738 against 1633, 2 a cell 1952 against
// 3129).  A call of so many builds it at once; shorter ones take the fused
// kernel until they have come to so many since the last fill or sort, so that
// a payload used for a call or two never pays for its table.
bool table_due(brille_grid* G, uint64_t n, int precision) {
  if (has_table(G->d, precision)) return true;
  if (table_bytes(G, precision) == 0) return false;
  uint64_t& points = G->untabled[precision == BRILLE_FP32];
  points += n;
  const bool f32 = precision == BRILLE_FP32;
  const uint64_t halves = wide_rows(G->d, precision) ? (f32 ? 5 : 3) : (f32 ? 48 : 28);
  return 2 * points >= halves * (G->n_cubes + G->n_tets / 2);
}

__global__ void k_zero_words(uint32_t* p, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

void zero_words(void* p, uint32_t n, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_zero_words, dim3((n + 255) / 256), dim3(256), 0, s, static_cast<uint32_t*>(p), n);
}

int exclusive_scan_u32(uint32_t* a, uint64_t m, uint32_t* part, hipStream_t s) {
  if (m == 0) return BRILLE_OK;
  const uint64_t np = (m + SCAN_SEG - 1) / SCAN_SEG;
  if (np > 256ull * 1024) return fail(BRILLE_ERR_UNSUPPORTED, "scan too long");
  hipLaunchKernelGGL(k_scan_reduce, dim3((unsigned)np), dim3(BIN_BLOCK), 0, s, a, m, part);
  hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(BIN_BLOCK), 0, s, part, (uint32_t)np);
  hipLaunchKernelGGL(k_scan_apply, dim3((unsigned)np), dim3(BIN_BLOCK), 0, s, a, m, part);
  if (hipGetLastError() != hipSuccess) return fail(BRILLE_ERR_DEVICE, "scan launch failed");
  return BRILLE_OK;
}

static void free_work_space(brille_grid* G) {
  if (G->bin_ws) (void)hipFree(G->bin_ws);
  G->bin_ws = nullptr;
  G->bin_ws_bytes = 0;
}

int ensure_work_space(brille_grid* G, uint64_t bytes) {
  if (G->bin_ws_bytes >= bytes) return BRILLE_OK;
  free_work_space(G);
  if (hipMalloc(&G->bin_ws, bytes) != hipSuccess) return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the work space");
  G->bin_ws_bytes = bytes;
  return BRILLE_OK;
}

void free_binned(brille_grid* G) {
  free_work_space(G);
  if (G->rec_ws) (void)hipFree(G->rec_ws);
  for (void* p : G->rec_old) (void)hipFree(p);
  for (auto& e : G->bin_ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  for (hipEvent_t* e : {&G->bin_used, &G->tables_built}) {
    if (*e) (void)hipEventDestroy(*e);
    *e = nullptr;
  }
  if (G->bin_side) (void)hipStreamDestroy(G->bin_side);
  G->bin_side = nullptr;
}

// the side stream and events of the two-stage pipeline, made on first use
// (default priority) and kept with the grid
static int ensure_side_stream(brille_grid* G) {
  if (G->bin_side) return BRILLE_OK;
  for (auto& e : G->bin_ev)
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess)
      return fail(BRILLE_ERR_DEVICE, "hipEventCreate failed");
  if (hipStreamCreateWithFlags(&G->bin_side, hipStreamNonBlocking) != hipSuccess) {
    G->bin_side = nullptr;
    return fail(BRILLE_ERR_DEVICE, "hipStreamCreate failed for the binned pipeline");
  }
  return BRILLE_OK;
}

// One half of the work space: the buffers of one pass.
struct PassBuffers {
  FoldRec* rec;
  SortKey* srt;
  uint32_t* key;   // shares perm's memory (read before perm is written)
  uint32_t* hint;  // shares srt's (written after srt is read)
  uint32_t *hist, *part, *plist, *pcount, *perm;
};

// A call's passes (BIN_CHUNK points each) run as a two-stage pipeline when
// there are several: the preparation of pass k + 1 (fold, scans, scatter,
// node order, proposal) on the grid's side stream while the sums of pass k run
// on the call's stream, each pass with its own half of the work space.  The
// fold is bound by FP64 issue and the sums by their scattered stores, and one
// fold wave per SIMD fits beside four sums waves, so the two overlap.  The
// call stream waits for each preparation before its sums, the side stream for
// the sums that last used a half, and the side stream starts after what the
// call stream held before the call: the call is ordered on `s` like a single
// kernel.
//
// stage_ms (nullable): adds the milliseconds of fold, bucket (scans, scatter,
// node order, proposal) and sums over all passes, each from events on the
// stream that ran it (with several passes the stages overlap, so they add up
// to more than the call)
// Byte offsets of one pass's buffers (a half of the work space) for passes of
// `chunk` points.
struct PassLayout {
  uint64_t rec, srt, hist, part, list, perm, cnt, half;
  uint64_t scan_blocks;  // segments of the histogram scan (k_scan_top handles at most 256 Ki)
};
static PassLayout pass_layout(uint64_t chunk, uint32_t nb) {
  const uint32_t nblk_max = (uint32_t)((chunk + BIN_SPAN - 1) / BIN_SPAN);
  const uint64_t m_max = (uint64_t)(nb + 1) * nblk_max;
  const uint64_t np_max = (m_max + SCAN_SEG - 1) / SCAN_SEG;
  auto al = [](uint64_t b) { return (b + 255) & ~uint64_t(255); };
  PassLayout L;
  L.rec = 0;
  L.srt = al(chunk * sizeof(FoldRec));
  L.hist = L.srt + al(chunk * sizeof(SortKey));
  L.part = L.hist + al(m_max * 4);
  L.list = L.part + al(np_max * 4);
  L.perm = L.list + al(chunk * 4);
  L.cnt = L.perm + al(chunk * 4);
  L.half = L.cnt + 256;
  L.scan_blocks = np_max;
  return L;
}

uint64_t binned_pass_bytes(const brille_grid* G, uint64_t chunk) { return pass_layout(chunk, bucket_count(G)).half; }

// The largest pass (a power of two, at most BIN_CHUNK points) whose buffers fit `bytes`.
uint64_t binned_pass_for(const brille_grid* G, uint64_t bytes) {
  uint64_t c = BIN_CHUNK;
  while (c > BIN_SPAN && binned_pass_bytes(G, c) > bytes) c >>= 1;
  return binned_pass_bytes(G, c) <= bytes ? c : 0;
}

// the passes of a call of n points
struct Passes {
  uint64_t chunk;  // points of each
  int halves;      // buffers: one, or two that take turns
  uint64_t bytes;  // of work space
};
static Passes passes_of(const brille_grid* G, uint64_t n) {
  Passes p;
  p.chunk = std::min<uint64_t>(n, BIN_CHUNK);
  p.halves = n > p.chunk ? 2 : 1;
  p.bytes = binned_pass_bytes(G, p.chunk) * (uint64_t)p.halves;
  return p;
}

// whether a graph can record a binned call of n points without an allocation
bool binned_recordable(const brille_grid* G, uint64_t n) {
  const Passes p = passes_of(G, n);
  return std::max(G->rec_ws_bytes, G->bin_ws_bytes) >= p.bytes && (p.halves == 1 || G->bin_side);
}

bool recording(hipStream_t s) {
  if (!s) return false;  // the null stream cannot
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return st != hipStreamCaptureStatusNone;
}

// The handle's lock covers the enqueueing of an unchecked call alone, so such
// calls on two streams would meet in the work space: each waits for the event
// the one before it recorded.  (A call that records a graph cannot wait for an
// event from outside it, nor leave one; one that the host waits for leaves
// nothing to wait for, which spares a call of 50 us some 10 of them.)
static int begin_work_space(brille_grid* G, hipStream_t s) {
  if (G->bin_pending && hipStreamWaitEvent(s, G->bin_used, 0) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "waiting for the work space failed");
  G->bin_touched = true;
  return BRILLE_OK;
}
void end_binned(brille_grid* G, hipStream_t s, bool waited) {
  // records *e after what the stream holds, or waits for it here
  auto leave = [s](hipEvent_t* e) {
    if (!*e && hipEventCreateWithFlags(e, hipEventDisableTiming) != hipSuccess) *e = nullptr;
    if (*e && hipEventRecord(*e, s) == hipSuccess) return true;
    (void)hipGetLastError();
    (void)hipStreamSynchronize(s);
    return false;
  };
  // (a call waits for what is pending before it adds to it)
  if (waited) G->tables_pending = false;
  else if (G->tables_touched) G->tables_pending = leave(&G->tables_built);
  if (G->bin_touched) G->bin_pending = !waited && leave(&G->bin_used);
  G->tables_touched = G->bin_touched = false;
}

// The work space of a call that a graph records.  The graph keeps the address,
// so the memory is never freed before the handle, and no call that runs at once
// works in it: a replay may run beside any of those.  It is the handle's
// present work space where that is large enough (the next call gets another).
// All recorded calls share it, one graph's in their order; replays of two
// graphs of one handle must not overlap.
static int recorded_work_space(brille_grid* G, uint64_t bytes) {
  if (G->rec_ws_bytes >= bytes) return BRILLE_OK;
  void* ws = nullptr;
  uint64_t held = bytes;
  if (G->bin_ws_bytes >= bytes) {
    // its last user is done before a replay can start
    if (G->bin_pending && hipEventSynchronize(G->bin_used) != hipSuccess)
      return fail(BRILLE_ERR_DEVICE, "waiting for the work space failed");
    G->bin_pending = false;
    ws = G->bin_ws;
    held = G->bin_ws_bytes;
    G->bin_ws = nullptr;
    G->bin_ws_bytes = 0;
  } else if (hipMalloc(&ws, bytes) != hipSuccess) {
    return fail(BRILLE_ERR_DEVICE, "hipMalloc failed for the work space");
  }
  if (G->rec_ws) G->rec_old.push_back(G->rec_ws);
  G->rec_ws = ws;
  G->rec_ws_bytes = held;
  return BRILLE_OK;
}

int prepare_binned(brille_grid* G, uint64_t n, int precision, hipStream_t s) {
  const bool rec = recording(s);
  // (a table built while a graph records would be complete only after a replay)
  if (!rec)
    if (int rc = ensure_cube_rows(G, precision, s); rc != BRILLE_OK) return rc;
  if (n == 0) return BRILLE_OK;
  const Passes p = passes_of(G, n);
  if (int rc = rec ? recorded_work_space(G, p.bytes) : ensure_work_space(G, p.bytes); rc != BRILLE_OK) return rc;
  return p.halves > 1 ? ensure_side_stream(G) : BRILLE_OK;
}

int launch_binned(brille_grid* G, const LaunchArgs& a, int precision, hipStream_t s, float* stage_ms) {
  if (a.n == 0) return BRILLE_OK;
  const Passes p = passes_of(G, a.n);
  if (recording(s)) return run_binned_passes(G, a, precision, s, stage_ms, G->rec_ws, p.chunk, p.halves);
  if (int rc = begin_work_space(G, s); rc != BRILLE_OK) return rc;
  return run_binned_passes(G, a, precision, s, stage_ms, G->bin_ws, p.chunk, p.halves);
}

// The pipeline over work space `ws` in passes of `chunk` points; with two
// halves the preparation of the next pass overlaps the sums (side stream
// and events of the grid), with one everything runs on `s` in order.
int run_binned_passes(brille_grid* G, const LaunchArgs& a, int precision, hipStream_t s, float* stage_ms, void* ws_base,
                      uint64_t chunk, int halves) {
  if (a.n == 0) return BRILLE_OK;
  const uint64_t passes = (a.n + chunk - 1) / chunk;
  const uint32_t nb = bucket_count(G);
  const PassLayout Lo = pass_layout(chunk, nb);
  if (Lo.scan_blocks > 256ull * 1024) return fail(BRILLE_ERR_INVALID_ARGUMENT, "binned pass too large");
  if (G->g.n_nodes >= kNodePoly) return fail(BRILLE_ERR_INVALID_ARGUMENT, "the binned kernel takes grids of fewer than 2^31 nodes");
  const uint64_t o_rec = Lo.rec, o_srt = Lo.srt, o_hist = Lo.hist, o_part = Lo.part, o_list = Lo.list,
                 o_perm = Lo.perm, o_cnt = Lo.cnt, half = Lo.half;
  const bool prop = a.use_proposal != 0;
  PassBuffers buf[2];
  for (int h = 0; h < halves; ++h) {
    char* ws = static_cast<char*>(ws_base) + h * half;
    PassBuffers& b = buf[h];
    b.rec = reinterpret_cast<FoldRec*>(ws + o_rec);
    b.srt = reinterpret_cast<SortKey*>(ws + o_srt);
    b.hint = reinterpret_cast<uint32_t*>(ws + o_srt);
    b.key = reinterpret_cast<uint32_t*>(ws + o_perm);
    b.hist = reinterpret_cast<uint32_t*>(ws + o_hist);
    b.part = reinterpret_cast<uint32_t*>(ws + o_part);
    b.plist = reinterpret_cast<uint32_t*>(ws + o_list);
    b.pcount = reinterpret_cast<uint32_t*>(ws + o_cnt);
    b.perm = reinterpret_cast<uint32_t*>(ws + o_perm);
  }
  // timing: five events per pass (fold start, fold end, bucket end on the
  // preparing stream; sums start and end on the call stream)
  std::vector<hipEvent_t> tev;
  auto destroy_tev = [&tev]() {
    for (auto e : tev)
      if (e) (void)hipEventDestroy(e);
  };
  if (stage_ms) {
    tev.assign(passes * 5, nullptr);
    for (auto& e : tev)
      if (hipEventCreate(&e) != hipSuccess) {
        destroy_tev();
        return fail(BRILLE_ERR_DEVICE, "hipEventCreate failed");
      }
  }
  auto mark = [&](uint64_t k, int j, hipStream_t st) {
    if (stage_ms) (void)hipEventRecord(tev[k * 5 + j], st);
  };
  const SumsKernel sums = precision == BRILLE_FP32 ? pick_sums<float>(G->d, prop) : pick_sums<double>(G->d, prop);
  const size_t rs = precision == BRILLE_FP32 ? 4 : 8;
  const size_t vb = (size_t)G->d.B * G->d.sv * rs, cb = (size_t)G->d.B * G->d.sc * 2 * rs;
  const size_t lds1 = (size_t)(nb + 1) * 4;
  hipStream_t side = halves > 1 ? G->bin_side : s;
  enum { EV_IN = 0, EV_PREP = 1, EV_DONE = 3 };  // G->bin_ev: call start, prepared[2], summed[2]
  if (halves > 1) {
    (void)hipEventRecord(G->bin_ev[EV_IN], s);
    (void)hipStreamWaitEvent(side, G->bin_ev[EV_IN], 0);
  }
  for (uint64_t k = 0; k < passes; ++k) {
    const uint64_t c0 = k * chunk;
    const int h = (int)(k & 1u) % halves;
    const PassBuffers& b = buf[h];
    const uint32_t m = (uint32_t)std::min<uint64_t>(chunk, a.n - c0);
    const uint32_t nblk = (m + BIN_SPAN - 1) / BIN_SPAN;
    const uint64_t M = (uint64_t)(nb + 1) * nblk;
    const uint32_t np = (uint32_t)((M + SCAN_SEG - 1) / SCAN_SEG);
    // preparation of pass k on the side stream, once the sums of pass k - 2
    // no longer read this half
    if (halves > 1 && k >= 2) (void)hipStreamWaitEvent(side, G->bin_ev[EV_DONE + h], 0);
    if (prop) zero_words(b.pcount, 1, side);
    mark(k, 0, side);
    hipLaunchKernelGGL(k_bin_fold<true>, dim3(nblk), dim3(BIN_BLOCK), lds1, side, G->g, a.Q + 3 * c0, m, a.fold,
                       b.rec, b.key, b.hist, nblk, nb, a.err, a.base + c0, prop ? 1 : 0);
    mark(k, 1, side);
    hipLaunchKernelGGL(k_scan_reduce, dim3(np), dim3(BIN_BLOCK), 0, side, b.hist, M, b.part);
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(BIN_BLOCK), 0, side, b.part, np);
    hipLaunchKernelGGL(k_scan_apply, dim3(np), dim3(BIN_BLOCK), 0, side, b.hist, M, b.part);
    hipLaunchKernelGGL(k_bin_scatter, dim3(nblk), dim3(BIN_BLOCK), 2 * lds1, side, b.key, m, b.hist, nblk, nb,
                       G->g.n_nodes, b.srt);
    hipLaunchKernelGGL(k_bucket_perm, dim3(nb + 1), dim3(PERM_BLOCK), 0, side, b.srt, m, b.hist, nblk, nb,
                       G->g.n_nodes, b.perm);
    if (prop) {
      hipLaunchKernelGGL(k_poly_list, dim3((m + LIST_SPAN - 1) / LIST_SPAN), dim3(BIN_BLOCK), 0, side, b.perm, m,
                         b.plist, b.pcount);
      hipLaunchKernelGGL(k_bin_propose, dim3(std::min<uint32_t>((m + 63) / 64, std::max<uint32_t>(G->n_cu, 1) * 4)),
                         dim3(256), 0, side, G->g, a.prop, b.rec, b.hint, b.plist, b.pcount);
    }
    mark(k, 2, side);
    if (halves > 1) {
      (void)hipEventRecord(G->bin_ev[EV_PREP + h], side);
      (void)hipStreamWaitEvent(s, G->bin_ev[EV_PREP + h], 0);
    }
    // sums of pass k on the call stream
    mark(k, 3, s);
    uint32_t tile_pts, groups;
    sum_split(G, m, prop, precision, &tile_pts, &groups);
    const dim3 sgrid((m + tile_pts - 1) / tile_pts, groups);
    hipLaunchKernelGGL(sums, sgrid, dim3(TILE), G->d.n_keys ? 32u * TILE : 0u, s, G->g, G->d, a.prop, b.rec, b.hint, b.perm, m,
                       static_cast<char*>(a.vals) + c0 * vb, static_cast<char*>(a.vecs) + c0 * cb,
                       offset_aux(a.aux, c0), a.err, a.base + c0, tile_pts);
    mark(k, 4, s);
    if (halves > 1) (void)hipEventRecord(G->bin_ev[EV_DONE + h], s);
  }
  if (stage_ms) {
    (void)hipEventSynchronize(tev[(passes - 1) * 5 + 4]);
    for (uint64_t k = 0; k < passes; ++k) {
      const int from[3] = {0, 1, 3}, to[3] = {1, 2, 4};
      for (int j = 0; j < 3; ++j) {
        float ms = 0;
        (void)hipEventElapsedTime(&ms, tev[k * 5 + from[j]], tev[k * 5 + to[j]]);
        stage_ms[j] += ms;
      }
    }
    destroy_tev();
  }
  if (hipGetLastError() != hipSuccess) return fail(BRILLE_ERR_DEVICE, "binned launch failed");
  return BRILLE_OK;
}

}  // namespace brille_amd
