// Launch logic behind brille_ir_interpolate_at: validation, staging of host
// buffers, kernel selection, error reduction and event timing.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "fast_tables.hpp"
#include "grid_state.hpp"
#include "launch_pieces.hpp"

using namespace brille_amd;

namespace brille_amd {

#define HIP_TRY(expr)                                                                                            \
  do {                                                                                                           \
    hipError_t e_ = (expr);                                                                                      \
    if (e_ != hipSuccess) return fail(BRILLE_ERR_DEVICE, std::string(#expr ": ") + hipGetErrorString(e_));       \
  } while (0)

__global__ void k_err_init2(ErrRec* e) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    e->first_bad = ~0ull;
    e->count = 0ull;
  }
}

void free_staging(brille_grid* G) {
  if (G->stage) (void)hipFree(G->stage);
  G->stage = nullptr;
  G->stage_bytes = 0;
  if (G->pin) (void)hipHostFree(G->pin);
  G->pin = nullptr;
  G->pin_bytes = 0;
  for (hipEvent_t& e : G->pin_ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
}

// Pinned memory of at least `bytes` for the handle's host-memory calls, kept
// for the next; false where it cannot be had (the calls then copy pageable).
static bool ensure_pin(brille_grid* G, size_t bytes) {
  if (G->pin_bytes >= bytes) return true;
  if (G->pin) (void)hipHostFree(G->pin);
  G->pin = nullptr;
  G->pin_bytes = 0;
  if (hipHostMalloc(&G->pin, bytes, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    G->pin = nullptr;
    return false;
  }
  G->pin_bytes = bytes;
  return true;
}

// One result on its way to the caller's memory.
struct OutPiece {
  char* host;
  const char* dev;
  size_t bytes;
};

// Results in device memory to the caller's pageable memory, on stream s; waits.
// What bounds it: a fresh array's pages are mapped and zeroed as they are first
// written, 14 GB/s for one thread, against 57 GB/s of the link.  Chunks of
// kPinChunk bytes come to a ring of pinned slots and go on to their place by
// up to kPinWorkers threads, each of which sends its freed slot the next chunk.
// Whole calls of 100 003 points of 6 modes and 2 atoms FP64 (62 MB), pageable
// copies 6.0 ms: one thread 4.7, three 2.5, six 2.3 in 1 MB chunks; four threads
// 2.0 in 2 MB chunks (eight the same), 2.0 in 4 MB, 2.2 in 8 MB, 3.2 in 512 KB
// (each chunk costs about 10 us of launches and waits).  Below one and a quarter
// chunks' bytes per thread the caller's thread works with fewer or none (by the
// number of chunks the dozen arrays of a call with every aux output, 4.5 to 6 MB,
// started threads that cost more than they copied: 20 011 points of 6 scalars
// FP32 506 us against 478 of pageable copies, 463 with one thread); where a
// thread or the ring cannot be had, the rest do the work.
constexpr uint64_t kPinWorkers = 4;
// bytes of a host-memory call up to which the kernels use pinned memory directly
constexpr size_t kDirectBytes = 4ull << 20;
static int copy_out(brille_grid* G, const std::vector<OutPiece>& out, hipStream_t s) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  std::vector<OutPiece> chunks;
  for (const OutPiece& p : out)
    for (size_t o = 0; o < p.bytes; o += kPinChunk)
      chunks.push_back({p.host + o, p.dev + o, std::min(kPinChunk, p.bytes - o)});
  bool ring = ensure_pin(G, kPinSlots * kPinChunk);
  for (hipEvent_t& e : G->pin_ev)
    if (ring && !e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      e = nullptr;
      ring = false;
    }
  if (!ring) {
    for (const OutPiece& p : out) HIP_TRY(hipMemcpyAsync(p.host, p.dev, p.bytes, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return BRILLE_OK;
  }
  char* pin = static_cast<char*>(G->pin);
  std::atomic<uint64_t> next{0};
  std::atomic<uint64_t> sent[kPinSlots];  // 1 + the chunk a slot was last sent
  std::atomic<int> error{(int)hipSuccess};
  auto send = [&](uint64_t k) {
    const int slot = (int)(k % kPinSlots);
    hipError_t e = hipMemcpyAsync(pin + slot * kPinChunk, chunks[k].dev, chunks[k].bytes, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipEventRecord(G->pin_ev[slot], s);
    if (e != hipSuccess) error = (int)e;
    sent[slot] = k + 1;
  };
  for (auto& x : sent) x = 0;
  for (uint64_t k = 0; k < chunks.size() && k < (uint64_t)kPinSlots; ++k) send(k);
  auto work = [&] {
    for (uint64_t k; (k = next.fetch_add(1)) < chunks.size();) {
      const int slot = (int)(k % kPinSlots);
      // chunk k - kPinSlots was taken before and its worker sends this one
      while (sent[slot] != k + 1 && error == (int)hipSuccess) std::this_thread::yield();
      if (error != (int)hipSuccess) return;
      const hipError_t e = hipEventSynchronize(G->pin_ev[slot]);
      if (e != hipSuccess) {
        error = (int)e;
        return;
      }
      std::memcpy(chunks[k].host, pin + slot * kPinChunk, chunks[k].bytes);
      if (k + kPinSlots < chunks.size()) send(k + kPinSlots);
    }
  };
  std::vector<std::thread> helpers;
  helpers.reserve(kPinWorkers);
  const uint64_t hw = std::max(1u, std::thread::hardware_concurrency());
  uint64_t bytes = 0;
  for (const OutPiece& p : out) bytes += p.bytes;
  const uint64_t n_help = std::min({kPinWorkers, bytes / (kPinChunk + kPinChunk / 4), hw});
  for (uint64_t i = 1; i < n_help; ++i) {
    try {
      helpers.emplace_back([&] {
        if (hipSetDevice(dev) == hipSuccess) work();
      });
    } catch (const std::exception&) {
      break;
    }
  }
  work();
  for (std::thread& t : helpers) t.join();
  HIP_TRY(hipStreamSynchronize(s));
  if (error != (int)hipSuccess)
    return fail(BRILLE_ERR_DEVICE, std::string("copying results: ") + hipGetErrorString((hipError_t)error.load()));
  return BRILLE_OK;
}

__global__ void k_report(const ErrRec* err, const unsigned long long* stats, CallReport* out) {
  out->err = *err;
  out->tried = stats ? stats[0] : 0ull;
  out->verified = stats ? stats[1] : 0ull;
}

// A kernel writes the record to pinned memory, one wait instead of a pageable
// copy's two (257 points of 6 scalar modes: whole call 54 -> 47 us).
int read_report(brille_grid* G, hipStream_t s, CallReport* out) {
  if (G->report) {
    hipLaunchKernelGGL(k_report, dim3(1), dim3(1), 0, s, G->err, G->prop_stats, G->report);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));
    *out = *G->report;
    return BRILLE_OK;
  }
  out->tried = out->verified = 0;
  if (G->prop_stats) HIP_TRY(hipMemcpyAsync(&out->tried, G->prop_stats, 16, hipMemcpyDeviceToHost, s));
  HIP_TRY(hipMemcpyAsync(&out->err, G->err, sizeof(ErrRec), hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  return BRILLE_OK;
}

// Interpolator::rotate_in_place dispatch  src/interpolator.hpp:387-428
int check_rotation_modes(const brille_grid* G) {
  const DataConst& d = G->d;
  auto one = [&](int rot, int lu, bool cplx, bool has_vm, const char* what) -> int {
    switch (lu) {
      case BRILLE_LU_REAL_LATTICE:
        if (rot == BRILLE_ROT_VECTOR || rot == BRILLE_ROT_PSEUDOVECTOR) return BRILLE_OK;
        if (rot == BRILLE_ROT_GAMMA) {
          if (!cplx) return fail(BRILLE_ERR_ROTATION, "RotatesLike == Gamma requires complex valued data!");
          return BRILLE_OK;
        }
        return fail(BRILLE_ERR_ROTATION, "Impossible RotatesLike value!");
      case BRILLE_LU_RECIPROCAL_LATTICE:
        if (rot == BRILLE_ROT_VECTOR) return BRILLE_OK;
        break;
      case BRILLE_LU_ANGSTROM:
        if (rot == BRILLE_ROT_GAMMA) {
          if (!cplx) return fail(BRILLE_ERR_ROTATION, "RotatesLike == Gamma requires complex valued data!");
          return BRILLE_OK;
        }
        break;
      default:
        break;
    }
    (void)has_vm;
    return fail(BRILLE_ERR_ROTATION, std::string("LengthUnit, RotatesLike combination not implemented (") + what + ")");
  };
  int rc = one(d.val_rot, d.val_lu, false, d.ev[1] + d.ev[2] > 0, "values");
  if (rc != BRILLE_OK) return rc;
  rc = one(d.vec_rot, d.vec_lu, true, d.ec[1] + d.ec[2] > 0, "vectors");
  if (rc != BRILLE_OK) return rc;
  if (d.vec_rot == BRILLE_ROT_GAMMA && d.ec[1] + d.ec[2] > 0) {
    if (!d.F0) return fail(BRILLE_ERR_ROTATION, "Gamma rotation requires a GammaTable");
    if (d.ec[1] / 3u != d.n_atoms)
      return fail(BRILLE_ERR_ROTATION, "the eigenvectors must hold one 3-vector per GammaTable atom");
    if (d.ec[2] > 0) return fail(BRILLE_ERR_UNSUPPORTED, "Gamma transformation of 3N x 3N tensors is not supported");
    if (d.vec_lu == BRILLE_LU_ANGSTROM && !d.cart_rot) return fail(BRILLE_ERR_ROTATION, "Cartesian Gamma rotation needs Cartesian matrices");
  }
  return BRILLE_OK;
}

// brille_grid_fill_ex may keep one precision of the payload only
int check_payload_precision(const brille_grid* G, int precision) {
  if (precision == BRILLE_FP64 && !G->d.rows64)
    return fail(BRILLE_ERR_INVALID_ARGUMENT, "the payload was filled without its FP64 rows");
  if (precision == BRILLE_FP32 && !G->d.rows32)
    return fail(BRILLE_ERR_INVALID_ARGUMENT, "the payload was filled without its FP32 rows");
  return BRILLE_OK;
}

using TileKernel = void (*)(GridConst, DataConst, LaunchArgs);

// which specialised phase 2 the payload admits
int payload_layout(const DataConst& d) {
  const bool scalar_values = d.ev[1] == 0 && d.ev[2] == 0;
  if (!scalar_values) return LAYOUT_GENERIC;
  if (d.ec[1] == 0 && d.ec[2] == 0) return LAYOUT_SCALAR;
  if (d.ec[0] == 0 && d.ec[2] == 0 && d.vec_rot == BRILLE_ROT_GAMMA &&
      (d.vec_lu == BRILLE_LU_REAL_LATTICE || d.vec_lu == BRILLE_LU_ANGSTROM))
    return LAYOUT_GAMMA;
  return LAYOUT_GENERIC;
}

// wide Gamma rows of at most one value per atom: the sums go atom-major
static bool by_atom(const DataConst& d) { return payload_layout(d) == LAYOUT_GAMMA && d.sv <= d.sc / 3u; }

// Gamma or scalar payloads whose rows are too long for one lane (more than 12
// and at most kWideMax complex elements, at most 64 values): one wave per row.
// With a PermutationTable the FP64 rows of up to kSortedLaneMax elements that are
// not summed atom by atom keep to the general sums, a lane per row, which leave
// fewer of a wave's lanes without an element (20 scalars of 6 modes, 300 007
// points binned: 342 vertices 4.49 ms a wave per row, 1.14 a lane, 14 513 vertices
// 3.09 / 1.64; 48 elements there 3.11 / 4.11; FP32, 20 elements: binned 1.58 /
// 1.22, fused 3.24 / 6.64).
constexpr uint32_t kSortedLaneMax = 24;
bool wide_rows(const DataConst& d, int precision) {
  const int L = payload_layout(d);
  if (!(L == LAYOUT_GAMMA || L == LAYOUT_SCALAR) || d.sc <= 12 || d.sc > kWideMax || d.sv > 64) return false;
  return d.n_keys == 0 || precision == BRILLE_FP32 || d.sc > kSortedLaneMax || by_atom(d);
}
bool wide_by_atom(const DataConst& d) { return wide_rows(d, BRILLE_FP32) && by_atom(d); }

// The instantiated specialisations: Gamma payloads of 1-4 atoms and scalar
// payloads of 1-4 complex elements, each with one value per mode; anything
// else runs the general phase 2.
template <typename Real>
static TileKernel pick_tuned(const DataConst& d) {
  const int L = payload_layout(d);
  if (L == LAYOUT_GAMMA && d.sv == 1) {
    switch (d.sc) {
      case 3: return k_ir_interpolate<Real, true, LAYOUT_GAMMA, 3, 1>;
      case 6: return k_ir_interpolate<Real, true, LAYOUT_GAMMA, 6, 1>;
      case 9: return k_ir_interpolate<Real, true, LAYOUT_GAMMA, 9, 1>;
      case 12: return k_ir_interpolate<Real, true, LAYOUT_GAMMA, 12, 1>;
      default: break;
    }
  }
  if (L == LAYOUT_SCALAR && d.sv == 1) {
    switch (d.sc) {
      case 1: return k_ir_interpolate<Real, true, LAYOUT_SCALAR, 1, 1>;
      case 2: return k_ir_interpolate<Real, true, LAYOUT_SCALAR, 2, 1>;
      case 3: return k_ir_interpolate<Real, true, LAYOUT_SCALAR, 3, 1>;
      case 4: return k_ir_interpolate<Real, true, LAYOUT_SCALAR, 4, 1>;
      default: break;
    }
  }
  if (wide_by_atom(d)) return k_ir_interpolate<Real, true, LAYOUT_WIDE, kWideAtom, 0>;
  if (wide_rows(d, sizeof(Real) == 4 ? BRILLE_FP32 : BRILLE_FP64)) return k_ir_interpolate<Real, true, LAYOUT_WIDE, kWideAll, 0>;
  return k_ir_interpolate<Real, true, LAYOUT_GENERIC, 0, 0>;
}

// Points per block and mode groups of a fused launch.  A block of TILE points
// walks them in sequence (narrow rows: TILE lanes take (point, mode) units;
// wide rows: four waves take (point, modes) units), so a call of few points
// gets smaller tiles.
//   narrow rows: down to one block per CU, as long as a tile has more units
//     than lanes (a second round of blocks repeats phase 1's latency: FP64 hex
//     grid of 6 modes, 20 011 points: 81 us in 256-point tiles, 56 us in 64,
//     72 us in 32);
//   wide rows: to eight blocks per CU, which spreads the tail, as long as a
//     block's waves have three units each (3 001 points of 72 modes: 17.8 ms in
//     256-point tiles, 0.25 ms in single points; 3 001 points of 24 modes: 88
//     us in single points, 50 us in fours); when single points still leave CUs
//     idle, the modes split too, to three blocks per CU (301 points of 72
//     modes: 64 us whole, 50 us in two groups, 68 us in six, each of which
//     repeats phase 1).
static void tile_split(const brille_grid* G, uint64_t n, int precision, bool fast, uint32_t* tile, uint32_t* groups) {
  const DataConst& d = G->d;
  const uint64_t cu = std::max<uint32_t>(G->n_cu, 1);
  uint32_t t = TILE;
  *groups = 1;
  if (fast && wide_rows(d, precision)) {
    const uint32_t mpw = wide_by_atom(d) ? 64u / (d.sc / 3u) : 1u;
    const uint32_t passes = (d.B + mpw - 1) / mpw;
    t = tile_capacity(LAYOUT_WIDE);
    while (t > 1 && (n + t - 1) / t < 8 * cu && (t >> 1) * passes >= 12) t >>= 1;
    const uint64_t blocks = (n + t - 1) / t;
    if (t == 1) *groups = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((d.B + 3) / 4, 3 * cu / blocks));
  } else {
    while (t > 32 && (n + t - 1) / t < cu && t * d.B > (uint32_t)TILE) t >>= 1;
  }
  *tile = t;
}

// plain: the literal FP64 restatement; tuned: fast fold-in and specialised sums
static void launch_sel(const brille_grid* G, LaunchArgs a, int precision, bool fast, hipStream_t s) {
  uint32_t groups;
  tile_split(G, a.n, precision, fast, &a.tile, &groups);
  TileKernel k;
  if (precision == BRILLE_FP32) k = fast ? pick_tuned<float>(G->d) : k_ir_interpolate<float, false, LAYOUT_GENERIC, 0, 0>;
  else k = fast ? pick_tuned<double>(G->d) : k_ir_interpolate<double, false, LAYOUT_GENERIC, 0, 0>;
  const size_t rs = precision == BRILLE_FP32 ? 4 : 8;
  in_pieces(a.n, a.tile, [&](uint64_t c0, uint64_t count, unsigned blocks) {
    LaunchArgs c = a;
    c.Q = a.Q + 3 * c0;
    c.n = count;
    c.base = a.base + c0;
    c.vals = static_cast<char*>(a.vals) + c0 * G->d.B * G->d.sv * rs;
    c.vecs = static_cast<char*>(a.vecs) + c0 * G->d.B * G->d.sc * 2 * rs;
    c.aux = offset_aux(a.aux, c0);
    hipLaunchKernelGGL(k, dim3(blocks, groups), dim3(TILE), G->d.n_keys ? 32u * a.tile : 0u, s, G->g, G->d, c);
  });
}

void launch_tile(const brille_grid* G, const LaunchArgs& a, int precision, bool fast, hipStream_t s) {
  launch_sel(G, a, precision, fast, s);
}

// A graph records an AUTO call as the fused kernel, which holds nothing of the
// handle's that another call writes; a large one as the pipeline if an earlier
// call has left a work space it can take over.
static bool takes_pipeline(const brille_grid* G, const LaunchArgs& a, const brille_run_opts& o, hipStream_t s) {
  if (!binned_applies(G, a, o.kernel, o.precision)) return false;
  if (o.kernel == BRILLE_KERNEL_BINNED || a.use_proposal || !recording(s)) return true;
  return binned_applies(G, a, o.kernel, o.precision, false) && binned_recordable(G, a.n);
}

// Whether the call runs in the pipeline, which is then ready for it.  A call that
// only AUTO gave to it needs none of the memory the pipeline allocates: where
// that cannot be had, the fused kernel serves it.
static int choose_pipeline(brille_grid* G, const LaunchArgs& a, const brille_run_opts& o, hipStream_t s, bool* binned) {
  *binned = takes_pipeline(G, a, o, s);
  if (!*binned) return BRILLE_OK;
  const bool asked = o.kernel == BRILLE_KERNEL_BINNED || a.use_proposal;
  if (!asked && !binned_applies(G, a, o.kernel, o.precision, false) && !table_due(G, a.n, o.precision)) {
    *binned = false;
    return BRILLE_OK;
  }
  const int rc = prepare_binned(G, a.n, o.precision, s);
  if (rc == BRILLE_OK || asked) return rc;
  (void)hipGetLastError();
  *binned = false;
  return BRILLE_OK;
}

// every kernel of one call on device buffers
static int dispatch(brille_grid* G, const LaunchArgs& a, const brille_run_opts& o, hipStream_t s) {
  bool binned;
  if (int rc = choose_pipeline(G, a, o, s, &binned); rc != BRILLE_OK) return rc;
  if (binned) return launch_binned(G, a, o.precision, s, nullptr);
  launch_sel(G, a, o.precision, o.kernel != BRILLE_KERNEL_PLAIN, s);
  return BRILLE_OK;
}

int report_point_error(const ErrRec& e, const double* Q, uint64_t n, bool host_mem) {
  const uint64_t idx = e.first_bad & ((1ull << kErrStatusShift) - 1ull);
  const int st = (int)(e.first_bad >> kErrStatusShift);
  double row[3];
  const double* rp = nullptr;
  if (idx < n) {
    if (host_mem) rp = Q + 3 * idx;
    else if (hipMemcpy(row, Q + 3 * idx, sizeof(row), hipMemcpyDeviceToHost) == hipSuccess) rp = row;
  }
  char buf[200];
  std::string q = "#" + std::to_string(idx);
  if (rp) {
    std::snprintf(buf, sizeof(buf), "[%.17g, %.17g, %.17g]", rp[0], rp[1], rp[2]);
    q = buf;
  }
  switch (st) {
    case BRILLE_PT_OUTSIDE_BZ:
      return fail(BRILLE_ERR_OUTSIDE_BZ, "Not all points inside Brillouin zone (first: Q = " + q + ")");
    case BRILLE_PT_OUTSIDE_IR:
      return fail(BRILLE_ERR_OUTSIDE_IR, "Q = " + q + " is outside of the irreducible BrillouinZone");
    case BRILLE_PT_NULL_NODE:
      return fail(BRILLE_ERR_NULL_NODE, "Attempting to access null node for point " + q);
    default: {
      std::string m = "interpolate_at failed to find " + std::to_string(e.count) + " point";
      m += e.count > 1 ? "s." : ".";
      return fail(BRILLE_ERR_NOT_FOUND, m);
    }
  }
}

int run_interpolate(brille_grid* G, const double* Q, uint64_t n, const brille_run_opts* opts_in, void* values_out,
                    void* vectors_out, const brille_aux_out* aux_in, hipStream_t s, brille_kernel_times* times,
                    uint32_t iters, int fold) {
  if (!G) return fail(BRILLE_ERR_INVALID_ARGUMENT, "null grid");
  if (!G->filled) return fail(BRILLE_ERR_NOT_FILLED, "The interpolation data must be filled before interpolating.");
  if (G->g.n_nodes == 0) return fail(BRILLE_ERR_INVALID_ARGUMENT, "this handle holds no trellis");
  brille_run_opts opts{};
  opts.check = 1;
  if (opts_in) opts = *opts_in;
  if (opts.precision != BRILLE_FP64 && opts.precision != BRILLE_FP32)
    return fail(BRILLE_ERR_INVALID_ARGUMENT, "unknown precision");
  int rc = check_rotation_modes(G);
  if (rc != BRILLE_OK) return rc;
  if (rc = check_payload_precision(G, opts.precision); rc != BRILLE_OK) return rc;
  if (n == 0) return BRILLE_OK;
  if (!Q || !values_out || !vectors_out) return fail(BRILLE_ERR_INVALID_ARGUMENT, "null input or output pointer");
  if (opts.use_proposal && !G->prop_trained)
    return fail(BRILLE_ERR_INVALID_ARGUMENT, "use_proposal requires a trained proposal (brille_proposal_train)");
  if (opts.use_proposal && (opts.kernel == BRILLE_KERNEL_PLAIN || opts.kernel == BRILLE_KERNEL_TILE))
    return fail(BRILLE_ERR_INVALID_ARGUMENT, "the learned proposal runs in the binned pipeline (kernel AUTO, TUNED or BINNED)");
  if (opts.use_proposal && aux_in && aux_in->tau)
    return fail(BRILLE_ERR_INVALID_ARGUMENT, "the binned pipeline does not report tau");
  const bool fast = opts.kernel != BRILLE_KERNEL_PLAIN;
  const size_t rs = opts.precision == BRILLE_FP32 ? 4 : 8;
  const size_t vbytes = (size_t)G->d.B * G->d.sv * rs;
  const size_t cbytes = (size_t)G->d.B * G->d.sc * 2 * rs;
  brille_aux_out aux{};
  if (aux_in) aux = *aux_in;
  LaunchArgs a{};
  a.fold = opts.no_move ? FOLD_NONE : fold;
  a.use_proposal = opts.use_proposal;
  a.prop = G->prop;
  if (opts.use_proposal) zero_words(G->prop_stats, 4, s);  // tried, verified (two 64-bit counters)
  a.err = G->err;
  CallReport rep{};
  struct End {  // however the call returns
    brille_grid* G;
    hipStream_t s;
    bool waited = false;
    ~End() { end_binned(G, s, waited); }
  } end{G, s};
  auto finish_call = [&] {
    const int r = read_report(G, s, &rep);
    end.waited = r == BRILLE_OK;
    if (r == BRILLE_OK && opts.use_proposal) {
      G->last_tried = rep.tried;
      G->last_hits = rep.verified;
    }
    return r;
  };
  if (rc = await_tables(G, s); rc != BRILLE_OK) return rc;
  if (opts.memory == BRILLE_MEM_DEVICE) {
    if (!opts.check && !times && recording(s)) G->recorded = true;
    a.Q = Q;
    a.n = n;
    a.base = 0;
    a.vals = values_out;
    a.vecs = vectors_out;
    a.aux = aux;
    hipLaunchKernelGGL(k_err_init2, dim3(1), dim3(1), 0, s, G->err);
    if (times) {
      std::memset(times, 0, sizeof(*times));
      const uint32_t it_n = std::max(iters, 1u);
      bool binned;
      if (rc = choose_pipeline(G, a, opts, s, &binned); rc != BRILLE_OK) return rc;
      if (binned) {
        // stages from events on the streams that ran them; the call from
        // events on `s` around all of it
        float st[3] = {0.f, 0.f, 0.f};
        hipEvent_t e0, e1;
        HIP_TRY(hipEventCreate(&e0));
        HIP_TRY(hipEventCreate(&e1));
        HIP_TRY(hipEventRecord(e0, s));
        for (uint32_t it = 0; it < it_n && rc == BRILLE_OK; ++it) rc = launch_binned(G, a, opts.precision, s, st);
        if (rc == BRILLE_OK) {
          HIP_TRY(hipEventRecord(e1, s));
          HIP_TRY(hipEventSynchronize(e1));
          float ms = 0;
          HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
          times->total_ms = ms / (float)it_n;
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        if (rc != BRILLE_OK) return rc;
        const char* nm[3] = {"k_bin_fold", opts.use_proposal ? "k_bin_bucket+propose" : "k_bin_bucket", "k_bin_sums"};
        times->n_kernels = 3;
        for (int k = 0; k < 3; ++k) {
          std::snprintf(times->names[k], sizeof(times->names[k]), "%s", nm[k]);
          times->ms[k] = st[k] / (float)it_n;
        }
      } else {
        hipEvent_t e0, e1;
        HIP_TRY(hipEventCreate(&e0));
        HIP_TRY(hipEventCreate(&e1));
        HIP_TRY(hipEventRecord(e0, s));
        for (uint32_t it = 0; it < it_n; ++it) launch_sel(G, a, opts.precision, fast, s);
        HIP_TRY(hipEventRecord(e1, s));
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipEventSynchronize(e1));
        float ms = 0;
        HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        times->n_kernels = 1;
        std::snprintf(times->names[0], sizeof(times->names[0]), "k_ir_interpolate");
        times->ms[0] = ms / (float)it_n;
        times->total_ms = times->ms[0];
      }
    } else {
      rc = dispatch(G, a, opts, s);
      if (rc != BRILLE_OK) return rc;
    }
    HIP_TRY(hipGetLastError());
    const bool check = opts.check || times;
    if (!check && !opts.use_proposal) return BRILLE_OK;
    rc = finish_call();
    if (rc != BRILLE_OK || !check) return rc;
    if (rep.err.count) return report_point_error(rep.err, Q, n, false);
    return BRILLE_OK;
  }
  // host memory: stream through device staging in chunks
  const uint64_t chunk = std::min<uint64_t>(n, 1ull << 20);
  struct Slot { void* host; size_t per; size_t off; };
  std::vector<Slot> slots;
  size_t off = 0;
  auto add = [&](void* h, size_t per) {
    slots.push_back({h, per, off});
    off += (per * chunk + 255) & ~size_t(255);
  };
  add(const_cast<double*>(Q), 3 * sizeof(double));
  add(values_out, vbytes);
  add(vectors_out, cbytes);
  void** auxp[10] = {(void**)&aux.ir_q, (void**)&aux.tau, (void**)&aux.rot, (void**)&aux.invrot, (void**)&aux.node,
                     (void**)&aux.tet, (void**)&aux.n_iw, (void**)&aux.iw_index, (void**)&aux.iw_weight,
                     (void**)&aux.status};
  const size_t auxper[10] = {24, 12, 4, 4, 4, 4, 1, 32, 64, 1};
  for (int i = 0; i < 10; ++i)
    if (*auxp[i]) add(*auxp[i], auxper[i]);
  // A small call's kernels read Q from and write results to pinned memory
  // themselves, one wait instead of a copy and wait per array (6 modes of 2
  // atoms FP64: 101 points 84 -> 48 us, 1 001 points, 0.6 MB, 125 -> 70 us, 6 001
  // points, 3.7 MB, 304 -> 247 us).  The general sums, which read back what they
  // wrote, and the larger calls go through device memory.
  const bool direct = off <= kDirectBytes && fast && !opts.use_proposal && (wide_rows(G->d, opts.precision) || onepass_sc(G->d)) &&
                      ensure_pin(G, kDirectBytes);
  if (!direct && G->stage_bytes < off) {
    if (G->stage) (void)hipFree(G->stage);
    G->stage = nullptr;
    G->stage_bytes = 0;
    HIP_TRY(hipMalloc(&G->stage, off));
    G->stage_bytes = off;
  }
  char* st = static_cast<char*>(direct ? G->pin : G->stage);
  hipLaunchKernelGGL(k_err_init2, dim3(1), dim3(1), 0, s, G->err);
  for (uint64_t c0 = 0; c0 < n; c0 += chunk) {
    const uint64_t m = std::min(chunk, n - c0);
    if (direct) std::memcpy(st + slots[0].off, Q + 3 * c0, m * 3 * sizeof(double));
    else HIP_TRY(hipMemcpyAsync(st + slots[0].off, Q + 3 * c0, m * 3 * sizeof(double), hipMemcpyHostToDevice, s));
    a.Q = reinterpret_cast<const double*>(st + slots[0].off);
    a.n = m;
    a.base = c0;
    a.vals = st + slots[1].off;
    a.vecs = st + slots[2].off;
    brille_aux_out da{};
    size_t k = 3;
    void** dauxp[10] = {(void**)&da.ir_q, (void**)&da.tau, (void**)&da.rot, (void**)&da.invrot, (void**)&da.node,
                        (void**)&da.tet, (void**)&da.n_iw, (void**)&da.iw_index, (void**)&da.iw_weight,
                        (void**)&da.status};
    for (int i = 0; i < 10; ++i)
      if (*auxp[i]) *dauxp[i] = st + slots[k++].off;
    a.aux = da;
    rc = dispatch(G, a, opts, s);
    if (rc != BRILLE_OK) {
      (void)hipStreamSynchronize(s);  // what was launched may still write to the buffers kept for the next call
      return rc;
    }
    HIP_TRY(hipGetLastError());
    if (c0 + m == n && direct) rc = finish_call();
    std::vector<OutPiece> out;
    for (size_t i = 1; i < slots.size(); ++i)
      out.push_back({static_cast<char*>(slots[i].host) + c0 * slots[i].per, st + slots[i].off, m * slots[i].per});
    if (direct)
      for (const OutPiece& p : out) std::memcpy(p.host, p.dev, p.bytes);
    else rc = copy_out(G, out, s);
    if (rc != BRILLE_OK) return rc;
  }
  if (!direct) rc = finish_call();
  if (rc != BRILLE_OK) return rc;
  if (rep.err.count) return report_point_error(rep.err, Q, n, true);
  return BRILLE_OK;
}

// *differ gets a bit for every cube whose vertices do not all have exactly
// vertex 0's or vertex 7's coordinate along each axis, in CubeNode order
__global__ __launch_bounds__(256) void k_cube_corners(GridConst g, uint64_t n_cubes, uint32_t* differ) {
  const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_cubes) return;
  const uint32_t* v = g.cube_v + 8 * c;
  const double* v0 = g.verts + 3 * (uint64_t)v[0];
  const double* v7 = g.verts + 3 * (uint64_t)v[7];
  bool same = true;
#pragma unroll
  for (int i = 1; i < 7; ++i) {
    const double* p = g.verts + 3 * (uint64_t)v[i];
    same = same && __double_as_longlong(p[0]) == __double_as_longlong(kCubeX[i] ? v7[0] : v0[0]) &&
           __double_as_longlong(p[1]) == __double_as_longlong(kCubeY[i] ? v7[1] : v0[1]) &&
           __double_as_longlong(p[2]) == __double_as_longlong(kCubeZ[i] ? v7[2] : v0[2]);
  }
  if (!same) *differ = 1u;
}

// FP32 affine forms of the barycentric weights of every tetrahedron (16 floats
// each, see GridConst::tet_bary).  The forms are rounded to FP32 and evaluated
// with x rounded to FP32 and three fused multiply-adds, an error of at most
// about 8 x 2^-24 (|f| . reach + |c|) for points within `reach` of the origin;
// a tetrahedron where that exceeds a tenth of kBarySkip, or that is so flat
// that the exact weights themselves could lose that much, gets zeros.
__global__ __launch_bounds__(256) void k_tet_bary(GridConst g, uint64_t n_tets, double reach, float* out) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_tets) return;
  double p[4][3];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int k = 0; k < 3; ++k) p[j][k] = g.verts[3 * (uint64_t)g.tet_v[4 * t + j] + k];
  constexpr double kMost = 0.1 * kBarySkip;
  const double vol6 = 6.0 * g.tet_vol[t];
  bool fine = 512.0 * DBL_EPSILON * reach * reach * reach < kMost * vol6;
  float f[16];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    // weight j (pseudo_orient3d with x in place of vertex j, over vol6) vanishes
    // on the opposite face and is 1 at vertex j: its slope is the face's
    // normal over the height
    const double *a = p[(j + 1) & 3], *b = p[(j + 2) & 3], *c = p[(j + 3) & 3];
    double u[3], v[3], w[3], n[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      u[k] = b[k] - a[k];
      v[k] = c[k] - a[k];
      w[k] = p[j][k] - a[k];
    }
    n[0] = u[1] * v[2] - u[2] * v[1];
    n[1] = u[2] * v[0] - u[0] * v[2];
    n[2] = u[0] * v[1] - u[1] * v[0];
    const double h = n[0] * w[0] + n[1] * w[1] + n[2] * w[2];  // +-6 V
    double off = 0, err = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      n[k] /= h;
      off -= n[k] * a[k];
      err += fabs(n[k]) * reach;
      f[4 * j + k] = (float)n[k];
    }
    f[4 * j + 3] = (float)off;
    // |h| is 6 V by either formula, or the forms are not the exact test's weights
    fine = fine && fabs(fabs(h) - vol6) < 1e-6 * vol6 && 8.0 * 5.9604644775390625e-08 * (err + fabs(off)) < kMost;
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) out[16 * t + k] = fine ? f[k] : 0.0f;
}

// the location tables derived from the cells: GridConst::cubes_aligned, tet_bary
static int build_cell_tables(const brille_grid_desc* d, brille_grid* G) {
  GridConst& g = G->g;
  g.cubes_aligned = 0;
  g.tet_bary = nullptr;
  const bool corners = d->n_cubes && G->report;
  if (corners) {
    G->report->differ = 0;
    hipLaunchKernelGGL(k_cube_corners, dim3((unsigned)((d->n_cubes + 255) / 256)), dim3(256), 0, nullptr, g, d->n_cubes,
                       &G->report->differ);
  }
  if (d->n_tets) {
    double reach = 0;
    for (int k = 0; k < 3; ++k)
      if (d->n_knots[k])
        reach = std::max(reach, std::max(std::abs(d->knots[k][0]), std::abs(d->knots[k][d->n_knots[k] - 1])));
    void* forms = nullptr;
    if (hipMalloc(&forms, 16 * d->n_tets * sizeof(float)) != hipSuccess) return fail(BRILLE_ERR_DEVICE, "hipMalloc failed");
    G->grid_allocs.push_back(forms);
    hipLaunchKernelGGL(k_tet_bary, dim3((unsigned)((d->n_tets + 255) / 256)), dim3(256), 0, nullptr, g, d->n_tets, reach,
                       static_cast<float*>(forms));
    g.tet_bary = static_cast<const float*>(forms);
  }
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess)
    return fail(BRILLE_ERR_DEVICE, "making the cell tables failed");
  if (corners) g.cubes_aligned = G->report->differ ? 0 : 1;
  return BRILLE_OK;
}

// Affine forms of the zone-face orientation tests and the seed orbit of the
// wedge (see fast_fold.hpp).  pseudo_orient3d(a,b,c,x) in a lattice with
// reciprocal volume V equals V det[a-x, b-x, c-x] on the components, i.e.
// V det[a,b,c] - x . V (a x b + b x c + c x a).
int build_fast_tables(const brille_grid_desc* d, brille_grid* G) {
  GridConst& g = G->g;
  FastTables ft = compute_fast_tables(d);
  g.aff_margin = ft.aff_margin;
  auto up = [&](const std::vector<double>& v, const double** dst) -> int {
    void* p = nullptr;
    if (hipMalloc(&p, v.size() * sizeof(double)) != hipSuccess) return fail(BRILLE_ERR_DEVICE, "hipMalloc failed");
    G->grid_allocs.push_back(p);
    if (hipMemcpy(p, v.data(), v.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess)
      return fail(BRILLE_ERR_DEVICE, "hipMemcpy failed");
    *dst = static_cast<const double*>(p);
    return BRILLE_OK;
  };
  int rc = up(ft.prim_aff, &g.prim_aff);
  if (rc == BRILLE_OK) rc = up(ft.outer_aff, &g.outer_aff);
  if (rc != BRILLE_OK) return rc;
  if (ft.has_orbit) {
    rc = up(ft.orbit, &g.orbit);
    if (rc != BRILLE_OK) return rc;
    g.orbit_margin = ft.orbit_margin;
  } else {
    g.has_seed = 0;
  }
  return build_cell_tables(d, G);
}


}  // namespace brille_amd

extern "C" {

int brille_time_ir_interpolate_at(brille_grid* G, const double* Q, uint64_t n, const brille_run_opts* opts,
                                  void* values_out, void* vectors_out, uint32_t iters, void* stream,
                                  brille_kernel_times* times) {
  BRILLE_LOCK_GRID(G);
  if (!times) return fail(BRILLE_ERR_INVALID_ARGUMENT, "null times");
  if (opts && opts->memory != BRILLE_MEM_DEVICE) return fail(BRILLE_ERR_INVALID_ARGUMENT, "timing needs device memory");
  return run_interpolate(G, Q, n, opts, values_out, vectors_out, nullptr, static_cast<hipStream_t>(stream), times, iters);
}


}  // extern "C"
