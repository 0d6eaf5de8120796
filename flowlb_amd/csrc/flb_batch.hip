// flb_batch.hip -- many independent single-phase culverts of uneven sizes in
// one kernel launch per step.  No reference counterpart: FlowLB runs one domain
// per process.
//
// Every instance keeps the single-domain layout (nine population planes, flags,
// fields, publication buffers; rows padded to a pitch of 64 cells so that each
// wavefront row segment starts on a 256-byte boundary) at its own offset of
// shared allocations.  The work of a step is a packed list of tiles --
// (instance, row, x-tile) -- over all instances, interleaved row by row.  Two
// launch modes:
//   * one launch per step, a block per tile or a grid-stride walk, runs of
//     steps replayed from hipGraphs captured for an even number of steps;
//   * persistent: one cooperative launch runs a chunk of steps, its resident
//     blocks walking the tile list and meeting at a grid barrier between
//     steps.
// The odd steps take the tile list's bands last to first (a second copy of
// the list), so that a step starts on what the Infinity Cache still holds of
// the previous one.  An autotuner times block sizes, grid sizes and both modes
// on the actual instance set and keeps the fastest.
#include <algorithm>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include <hip/hip_cooperative_groups.h>

#include "flb_cell.h"
#include "flb_cost.h"
#include "flb_internal.h"
#include "flb_march.h"

namespace flb {

struct Tile {
  uint32_t inst;
  uint32_t row;
  uint32_t tx;
  uint32_t pad;
};

// One step over `tiles`, the list in this step's order (the odd steps get the
// second copy).
template <class S, int ODD, bool MOM>
__global__ void __launch_bounds__(1024) k_batch_step(const Tile* __restrict__ tiles, uint32_t ntiles,
                                                      const Params* __restrict__ inst) {
  uint32_t k = blockIdx.x;
  if (k >= ntiles) return;
  Tile t = tiles[k];
  // A grid-stride block loads its next tile's descriptor while it evaluates
  // this one (with a block per tile there is no next: the same line again).
  for (;;) {
    const uint32_t kn = k + gridDim.x;
    const bool more = kn < ntiles;
    const Tile tn = tiles[more ? kn : k];
    const Params& p = inst[t.inst];
    const uint32_t x = t.tx * blockDim.x + threadIdx.x;
    if (x < p.nx) {
      const Cell c{x, t.row, x + t.row * p.pitch, true};
      stream_collide_cell<S, ODD, false, MOM, false>(p, c);
    }
    if (!more) break;
    k = kn;
    t = tn;
  }
}

// Persistent mode: `nsteps` steps from parity odd0 in one cooperative launch
// (every block resident, so the grid barrier between steps completes); the
// readback fields are not written (the last step of a call runs as a plain
// launch).  Every block reaches every barrier.
template <class S>
__global__ void __launch_bounds__(1024) k_batch_persistent(const Tile* __restrict__ tiles,
                                                            uint32_t ntiles,
                                                            const Params* __restrict__ inst,
                                                            uint32_t nsteps, uint32_t odd0) {
  cooperative_groups::grid_group grid = cooperative_groups::this_grid();
  for (uint32_t s = 0; s < nsteps; ++s) {
    const bool odd = ((odd0 + s) & 1u) != 0;
    const Tile* const list = tiles + (odd ? ntiles : 0u);  // the odd steps' order
    for (uint32_t k = blockIdx.x; k < ntiles; k += gridDim.x) {
      const Tile t = list[k];
      const Params& p = inst[t.inst];
      const uint32_t x = t.tx * blockDim.x + threadIdx.x;
      if (x < p.nx) {
        const Cell c{x, t.row, x + t.row * p.pitch, true};
        if (odd) stream_collide_cell<S, 1, false, false, false>(p, c);
        else stream_collide_cell<S, 0, false, false, false>(p, c);
      }
    }
    if (s + 1 < nsteps) grid.sync();
  }
}

// A block of a multi-step pass over the batch: rows [ya, yb) of up to
// kMarchWaves strips of an instance, or (io) of one strip with inlet or outlet
// columns, split by rows between the wavefronts, as in k_march.
struct MarchBlock {
  static constexpr uint32_t kNone = ~0u;
  uint32_t inst, ya, yb, io;
  uint32_t strip[kMarchWaves];  // kNone: no strip
};

// inst: the instances with the populations the pass reads, out: those it writes.
template <class S, int T, int MODEL>
__global__ void __launch_bounds__(64 * kMarchWaves)
__attribute__((amdgpu_waves_per_eu(march_occupancy<S, MODEL>())))
k_batch_march(const MarchBlock* __restrict__ blocks, const Params* __restrict__ inst,
              const Params* __restrict__ out, int odd, int moments) {
  const MarchBlock* const d = blocks + blockIdx.x;
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(threadIdx.x / 64u));
  const uint32_t i = d->inst;
  if (i == MarchBlock::kNone) return;
  // What the pass uses of the instance, held in scalar registers.
  const Params& q = inst[i];
  Params p{};
  p.nx = q.nx;
  p.ny = q.ny;
  p.pitch = q.pitch;
  p.N = q.N;
  p.Np = q.Np;
  p.inv_tau = q.inv_tau;
  p.tau = q.tau;
  p.trt_minus = q.trt_minus;
  p.fx = q.fx;
  p.fy = q.fy;
  p.use_force = q.use_force;
  p.flags = q.flags;
  p.rho = q.rho;
  p.u = q.u;
  March a{};
  a.f_in = q.f;
  a.f_out = out[i].f;
  a.pub_rho_in = q.pub_rho[odd ^ 1];
  a.pub_u_in = q.pub_u[odd ^ 1];
  a.pub_rho_out = q.pub_rho[odd];
  a.pub_u_out = q.pub_u[odd];
  // A program cannot reach an instance's fields, so these hold the same values.
  a.own_rho = a.pub_rho_in;
  a.own_u = a.pub_u_in;
  a.odd = odd;
  a.moments = moments;
  if (d->io) {
    const uint32_t rows = (d->yb - d->ya + uint32_t(kMarchWaves) - 1u) / uint32_t(kMarchWaves);
    const uint32_t ya = d->ya + wave * rows, yb = min(ya + rows, d->yb);
    if (ya < yb) march_rows<S, T, MODEL, true>(p, a, d->strip[0], ya, yb);
    return;
  }
  const uint32_t strip = d->strip[wave];
  if (strip != MarchBlock::kNone) march_rows<S, T, MODEL, false>(p, a, strip, d->ya, d->yb);
}

// Populations of instance i to / from nx * ny host-ordered float planes
// (unshifted), through the pitched device planes.
template <class S>
__global__ void k_batch_to_f32(const Params* inst, uint32_t i, float* out) {
  const Params& p = inst[i];
  for (uint64_t n = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; n < p.NL;
       n += uint64_t(gridDim.x) * blockDim.x) {
    const typename S::T* f = static_cast<const typename S::T*>(p.f);
    const uint64_t y = n / p.nx, d = n + y * (p.pitch - p.nx);
    for (int q = 0; q < 9; q++) out[q * p.NL + n] = S::load(f + q * p.Np, d) + wgt(q);
  }
}

template <class S>
__global__ void k_batch_from_f32(const Params* inst, uint32_t i, const float* in) {
  const Params& p = inst[i];
  for (uint64_t n = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; n < p.NL;
       n += uint64_t(gridDim.x) * blockDim.x) {
    typename S::T* f = static_cast<typename S::T*>(p.f);
    const uint64_t y = n / p.nx, d = n + y * (p.pitch - p.nx);
    for (int q = 0; q < 9; q++) S::store(f + q * p.Np, d, in[q * p.NL + n]);
  }
}

using BatchFn = void (*)(const Tile*, uint32_t, const Params*);
template <class S>
BatchFn batch_fn(int odd, bool mom) {
  if (mom) return odd ? k_batch_step<S, 1, true> : k_batch_step<S, 0, true>;
  return odd ? k_batch_step<S, 1, false> : k_batch_step<S, 0, false>;
}
BatchFn get_batch(int storage, int odd, bool mom) {
  switch (storage) {
    case 1: return batch_fn<StoreF16S>(odd, mom);
    case 2: return batch_fn<StoreBF16S>(odd, mom);
    default: return batch_fn<StoreF32>(odd, mom);
  }
}
using BatchMarchFn = void (*)(const MarchBlock*, const Params*, const Params*, int, int);
template <class S, int T>
BatchMarchFn batch_march_fn(bool forced) {
  return forced ? k_batch_march<S, T, kMarchGeneral> : k_batch_march<S, T, kMarchPlain>;
}
template <class S>
BatchMarchFn batch_march_steps(int steps, bool forced) {
  switch (steps) {
    case 2: return batch_march_fn<S, 2>(forced);
    case 3: return batch_march_fn<S, 3>(forced);
    default: return batch_march_fn<S, 4>(forced);
  }
}
BatchMarchFn get_batch_march(int storage, int steps, bool forced) {
  switch (storage) {
    case 1: return batch_march_steps<StoreF16S>(steps, forced);
    case 2: return batch_march_steps<StoreBF16S>(steps, forced);
    default: return batch_march_steps<StoreF32>(steps, forced);
  }
}
using PersistFn = void (*)(const Tile*, uint32_t, const Params*, uint32_t, uint32_t);
PersistFn get_persistent(int storage) {
  switch (storage) {
    case 1: return k_batch_persistent<StoreF16S>;
    case 2: return k_batch_persistent<StoreBF16S>;
    default: return k_batch_persistent<StoreF32>;
  }
}

}  // namespace flb

struct flb_batch : flb::Kept {
  int storage = 0;
  int block_x = 256;
  int grid = 0;            // blocks of the grid-stride launch
  int graph_chunk = 100;   // steps per captured graph (even), 0 = no graphs
  int mode = FLB_BATCH_LAUNCH;
  int order = FLB_BATCH_ORDER_ROWS;
  int persist_per_cu = 0;  // persistent mode: resident blocks per CU
  int persist_chunk = 100; // persistent mode: steps per cooperative launch
  int ncu = 256;
  hipStream_t stream = nullptr;
  flb::Staging staging;
  std::vector<flb::Params> host_inst;
  // The instances' parameters, four sets of count: bit 0 of the set says which
  // of the two population arrays they name, bit 1 whether the publication
  // buffers are exchanged (a pass of an even number of steps leaves what it
  // published at the other parity).  inst is the current set.
  flb::Params* inst_sets = nullptr;
  flb::Params* inst = nullptr;
  int set = 0;
  // Blocks of the multi-step passes by number of steps; no passes if shape.steps is 0.
  flb::MarchBlock* march[flb::kMarchMax + 1] = {};
  uint32_t march_blocks[flb::kMarchMax + 1] = {};
  flb::MarchShape shape{0, 0};
  flb::MarchShape rule_shape{0, 0};  // march_shape's choice
  bool any_shape = false;            // set by flb_test_batch_pass_shape: taken always
  // Runs of several steps: by flb_cost.h, or what flb_batch_autotune measured.
  enum Way { kEstimated, kSingle, kPasses } way = kEstimated;
  flb::StepModel model{};            // flb_cost.h
  flb::PassRows pass_rows[flb::kMarchMax + 1];
  double mb = 0.0;                   // populations, megabytes
  std::vector<std::vector<uint8_t>> io;  // per instance, its columns with inlet or outlet cells
  bool forced = false;
  flb::Tile* tiles = nullptr;
  uint32_t ntiles = 0;
  std::vector<void*> owned;
  void* pops[2] = {nullptr, nullptr};  // the population arrays; the second for the passes
  hipGraphExec_t graph[4] = {};  // by the set it starts from
  int graph_set[4] = {};         // the set it ends at
  uint64_t t = 0;
  std::string err;
  bool give_back() override;
};

namespace {

#define BAT_HIP(b, call)                                                                   \
  do {                                                                                     \
    hipError_t e_ = (call);                                                                \
    if (e_ != hipSuccess) {                                                                \
      (b)->err = std::string(#call) + ": " + hipGetErrorString(e_);                        \
      return FLB_ERR_DEVICE;                                                               \
    }                                                                                      \
  } while (0)

template <class T>
int balloc(flb_batch* b, T** p, size_t count) {
  void* v = nullptr;
  if (flb::device_malloc(&v, std::max<size_t>(count, 1) * sizeof(T), b->device, b) != hipSuccess) {
    b->err = "hipMalloc of " + std::to_string(count * sizeof(T)) + " bytes failed";
    return FLB_ERR_MEMORY;
  }
  b->owned.push_back(v);
  *p = static_cast<T*>(v);
  return FLB_OK;
}

template <class T>
void release(flb_batch* b, T** p) {
  if (!*p) return;
  (void)hipFree(*p);
  b->owned.erase(std::remove(b->owned.begin(), b->owned.end(), static_cast<void*>(*p)), b->owned.end());
  *p = nullptr;
}

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Tile list for block size bx in the batch's tile order:
//   FLB_BATCH_ORDER_ROWS      instances interleaved row by row (consecutive
//                             tiles come from different instances);
//   FLB_BATCH_ORDER_INSTANCE  instance after instance, each row-major;
//   FLB_BATCH_ORDER_BANDS     instance after instance, each in bands of 32
//                             rows walked column by column (the single-domain
//                             kernels' block order).
int build_tiles(flb_batch* b, int bx) {
  std::vector<flb::Tile> tl;
  const uint32_t n = uint32_t(b->host_inst.size());
  if (b->order == FLB_BATCH_ORDER_ROWS) {
    uint32_t max_rows = 0;
    for (const auto& p : b->host_inst) max_rows = std::max(max_rows, p.ny);
    for (uint32_t r = 0; r < max_rows; ++r)
      for (uint32_t i = 0; i < n; ++i) {
        const auto& p = b->host_inst[i];
        if (r >= p.ny) continue;
        const uint32_t tx = (p.nx + bx - 1) / bx;
        for (uint32_t k = 0; k < tx; ++k) tl.push_back(flb::Tile{i, r, k, 0});
      }
  } else {
    constexpr uint32_t kBand = 32;
    for (uint32_t i = 0; i < n; ++i) {
      const auto& p = b->host_inst[i];
      const uint32_t tx = (p.nx + bx - 1) / bx;
      if (b->order == FLB_BATCH_ORDER_INSTANCE) {
        for (uint32_t r = 0; r < p.ny; ++r)
          for (uint32_t k = 0; k < tx; ++k) tl.push_back(flb::Tile{i, r, k, 0});
      } else {
        // In a full band the tile at list position q runs on XCD q mod 8 (one
        // block per tile, or a grid-stride walk over a multiple of 8 blocks) and
        // takes row (q mod 8) * 4 + j / 8 of its column (j its place in the
        // column): each XCD gets four adjacent rows, as in the single-domain
        // band order, so that row-neighbour reads stay in one L2.
        for (uint32_t r0 = 0; r0 < p.ny; r0 += kBand) {
          const uint32_t h = std::min(p.ny - r0, kBand);
          for (uint32_t k = 0; k < tx; ++k) {
            const uint32_t base = uint32_t(tl.size());
            for (uint32_t j = 0; j < h; ++j) {
              const uint32_t r = h == kBand ? r0 + ((base + j) % 8u) * 4u + j / 8u : r0 + j;
              tl.push_back(flb::Tile{i, r, k, 0});
            }
          }
        }
      }
    }
  }
  release(b, &b->tiles);
  // The odd steps take the list's bands (runs of tiles of one instance and one
  // 32-row band) last to first, each band's tiles in their order, so that a
  // step starts on the tiles the previous one wrote last, which are still in
  // the Infinity Cache.  Both orders go into one allocation, the odd one second.
  std::vector<flb::Tile> both(tl);
  both.reserve(2 * tl.size());
  std::vector<std::pair<size_t, size_t>> runs;  // [begin, end) of each band run
  for (size_t a = 0; a < tl.size();) {
    size_t e = a + 1;
    while (e < tl.size() && tl[e].inst == tl[a].inst && tl[e].row / 32 == tl[a].row / 32) ++e;
    runs.emplace_back(a, e);
    a = e;
  }
  for (size_t r = runs.size(); r-- > 0;)
    both.insert(both.end(), tl.begin() + ptrdiff_t(runs[r].first), tl.begin() + ptrdiff_t(runs[r].second));
  int rc = balloc(b, &b->tiles, both.size());
  if (rc) return rc;
  BAT_HIP(b, hipMemcpy(b->tiles, both.data(), both.size() * sizeof(flb::Tile), hipMemcpyHostToDevice));
  b->ntiles = uint32_t(tl.size());
  b->block_x = bx;
  return FLB_OK;
}

void drop_graph(flb_batch* b) {
  for (hipGraphExec_t& g : b->graph) {
    if (g) (void)hipGraphExecDestroy(g);
    g = nullptr;
  }
}

void use_set(flb_batch* b, int set) {
  b->set = set;
  b->inst = b->inst_sets + size_t(set) * b->host_inst.size();
}

// Block list of the passes of T steps: the inlet/outlet strips first (they take
// longest), the others in an order that gives each XCD (block index mod 8)
// consecutive groups of strips.
int build_march(flb_batch* b, int T) {
  constexpr uint32_t G = flb::kMarchWaves;
  std::vector<flb::MarchBlock> first, rest;
  std::vector<uint32_t> order;
  b->pass_rows[T] = flb::PassRows{};
  for (uint32_t i = 0; i < b->host_inst.size(); ++i) {
    const flb::Params& p = b->host_inst[i];
    const uint32_t nio = flb::march_strips(p.nx, T, b->io[i], order);
    b->pass_rows[T].add(uint32_t(order.size()) - nio, nio, p.ny, T, b->shape.rows,
                        (b->shape.rows + G - 1) / G, true);
    for (uint32_t ya = 0; ya < p.ny; ya += b->shape.rows) {
      flb::MarchBlock d{};
      d.inst = i;
      d.ya = ya;
      d.yb = std::min(ya + b->shape.rows, p.ny);
      d.io = 1;
      for (uint32_t k = 0; k < nio; ++k) {
        d.strip[0] = order[k];
        first.push_back(d);
      }
      d.io = 0;
      for (uint32_t k = nio; k < order.size(); k += G) {
        for (uint32_t w = 0; w < G; ++w)
          d.strip[w] = k + w < order.size() ? order[k + w] : flb::MarchBlock::kNone;
        rest.push_back(d);
      }
    }
  }
  const size_t per = (rest.size() + 7) / 8;
  flb::MarchBlock none{};
  none.inst = flb::MarchBlock::kNone;
  for (size_t q = 0; q < 8 * per; ++q) {
    const size_t w = (q % 8) * per + q / 8;
    first.push_back(w < rest.size() ? rest[w] : none);
  }
  release(b, &b->march[T]);
  int rc = balloc(b, &b->march[T], first.size());
  if (rc) return rc;
  const size_t bytes = first.size() * sizeof(flb::MarchBlock);
  BAT_HIP(b, b->staging.to_device(b->stream, b->march[T], first.data(), bytes, bytes, 1));
  b->march_blocks[T] = uint32_t(first.size());
  return FLB_OK;
}

// Shape of the passes and their block lists.
int set_shape(flb_batch* b, flb::MarchShape shape) {
  b->shape = shape;
  if (!shape.steps) return FLB_OK;
  int rc = FLB_OK;
  for (int T = flb::kMarchMin; T <= flb::kMarchMax && !rc; ++T) rc = build_march(b, T);
  if (rc) b->shape = flb::MarchShape{0, 0};
  return rc;
}

// The second population array, the four sets of parameters and the block lists
// of the passes; single steps only where an instance does not fit the passes'
// rules or the array would take more than a quarter of the memory left.
int prepare_march(flb_batch* b, const flb_instance* in, size_t f_bytes) {
  const size_t count = b->host_inst.size();
  b->io.resize(count);
  uint64_t strip_rows = 0;
  bool fits = true;
  const uint32_t cols = flb::march_columns(flb::kMarchMax);
  for (size_t i = 0; i < count && fits; ++i) {
    fits = flb::march_columns_io(in[i].flags, in[i].nx, in[i].ny, b->io[i]);
    strip_rows += uint64_t((in[i].nx + cols - 1) / cols) * in[i].ny;
    b->forced = b->forced || in[i].use_force;
  }
  size_t left = 0, total = 0;
  void* alt = nullptr;
  if (fits && (hipMemGetInfo(&left, &total) != hipSuccess || f_bytes > left / 4 ||
               hipMalloc(&alt, f_bytes) != hipSuccess)) {
    (void)hipGetLastError();
    alt = nullptr;
  }
  b->pops[1] = alt;
  const uint8_t* const base = static_cast<const uint8_t*>(b->host_inst[0].f);
  std::vector<flb::Params> sets;
  sets.reserve(4 * count);
  for (int s = 0; s < 4; ++s)
    for (flb::Params p : b->host_inst) {
      if ((s & 1) && alt)
        p.f = static_cast<uint8_t*>(alt) + (static_cast<const uint8_t*>(p.f) - base);
      if (s & 2) {
        std::swap(p.pub_rho[0], p.pub_rho[1]);
        std::swap(p.pub_u[0], p.pub_u[1]);
      }
      sets.push_back(p);
    }
  const size_t bytes = sets.size() * sizeof(flb::Params);
  BAT_HIP(b, b->staging.to_device(b->stream, b->inst_sets, sets.data(), bytes, bytes, 1));
  if (!alt) return FLB_OK;
  b->model.storage = b->storage;
  b->model.force = b->forced;
  b->model.kernel = b->forced ? flb::kMarchGeneral : flb::kMarchPlain;
  b->mb = 1e-6 * double(f_bytes);
  b->rule_shape = flb::march_shape(b->ncu, strip_rows, b->storage == 0 ? 4 : 2, false);
  if (set_shape(b, b->rule_shape)) b->rule_shape = flb::MarchShape{0, 0};  // no room: single steps
  return FLB_OK;
}

int launch_step(flb_batch* b, int odd, bool mom) {
  const uint32_t grid = b->grid > 0 ? uint32_t(b->grid) : b->ntiles;  // 0: a block per tile
  hipLaunchKernelGGL(flb::get_batch(b->storage, odd, mom), dim3(grid), dim3(b->block_x), 0,
                     b->stream, b->tiles + (odd ? b->ntiles : 0u), b->ntiles, b->inst);
  BAT_HIP(b, hipGetLastError());
  return FLB_OK;
}

// A pass of T steps from time parity odd; moves on to the set it leaves.
int launch_march(flb_batch* b, int T, int odd, bool mom) {
  const flb::Params* const out = b->inst_sets + size_t(b->set ^ 1) * b->host_inst.size();
  hipLaunchKernelGGL(flb::get_batch_march(b->storage, T, b->forced), dim3(b->march_blocks[T]),
                     dim3(64 * flb::kMarchWaves), 0, b->stream, b->march[T], b->inst, out, odd,
                     int(mom));
  BAT_HIP(b, hipGetLastError());
  use_set(b, b->set ^ (T % 2 == 0 ? 3 : 1));
  return FLB_OK;
}

// Whether to take a pass of T steps: where it takes less time than T single steps
// in the batch's tile order (flb_cost.h).
bool pass_pays(const flb_batch* b, int T) {
  if (b->way == flb_batch::kSingle) return false;
  return b->any_shape || (b->way == flb_batch::kPasses && T == b->shape.steps) ||
         flb::faster(flb::pass_time(b->model, T, b->pass_rows[T], b->mb, b->ncu),
                     flb::batch_single_time(b->model, b->mb, b->order == FLB_BATCH_ORDER_ROWS));
}

// The next steps of a run with `left` to go: a pass, or a single step.
int advance(flb_batch* b, uint64_t t, uint64_t left, bool mom, int* done) {
  int T = flb::march_steps_next(left, b->shape.steps);
  if (T && !(pass_pays(b, b->shape.steps) && pass_pays(b, T))) T = 0;
  *done = T ? T : 1;
  const bool last = mom && left == uint64_t(*done);
  return T ? launch_march(b, T, int(t & 1), last) : launch_step(b, int(t & 1), last);
}

}  // namespace

// The population array that the current set does not name.
bool flb_batch::give_back() {
  if (!pops[1] || !pops[0]) return false;
  (void)hipStreamSynchronize(stream);
  drop_graph(this);
  shape = rule_shape = flb::MarchShape{0, 0};
  void*& other = pops[(set & 1) ^ 1];
  (void)hipFree(other);
  other = nullptr;
  return true;
}

namespace {

// Resident blocks per CU the persistent kernel can have at block size bx.
int persistent_capacity(flb_batch* b, int bx, int* per_cu) {
  int n = 0;
  BAT_HIP(b, hipOccupancyMaxActiveBlocksPerMultiprocessor(
                 &n, reinterpret_cast<const void*>(flb::get_persistent(b->storage)), bx, 0));
  *per_cu = n;
  return FLB_OK;
}

// One cooperative launch of nsteps steps starting at parity odd0.  The runtime
// rejects a grid that cannot be resident at once, so the barrier always
// completes.
int launch_persistent(flb_batch* b, uint32_t nsteps, uint32_t odd0) {
  const uint32_t grid = uint32_t(b->persist_per_cu * b->ncu);
  const flb::Tile* tiles = b->tiles;
  uint32_t ntiles = b->ntiles;
  const flb::Params* inst = b->inst;
  void* args[] = {&tiles, &ntiles, &inst, &nsteps, &odd0};
  BAT_HIP(b, hipLaunchCooperativeKernel(reinterpret_cast<const void*>(flb::get_persistent(b->storage)),
                                        dim3(grid), dim3(b->block_x), args, 0, b->stream));
  return FLB_OK;
}

// Graph of graph_chunk steps starting at an even t from the current set.
int ensure_graph(flb_batch* b) {
  const int from = b->set;
  if (b->graph[from] || b->graph_chunk <= 0) return FLB_OK;
  hipGraph_t g = nullptr;
  BAT_HIP(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  int rc = FLB_OK, done = 0;
  for (int s = 0; s < b->graph_chunk && !rc; s += done)
    rc = advance(b, uint64_t(s), uint64_t(b->graph_chunk - s), false, &done);
  hipError_t e = hipStreamEndCapture(b->stream, &g);
  b->graph_set[from] = b->set;
  use_set(b, from);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  BAT_HIP(b, e);
  e = hipGraphInstantiate(&b->graph[from], g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  BAT_HIP(b, e);
  return FLB_OK;
}

}  // namespace

extern "C" {

const char* flb_batch_last_error(const flb_batch* b) { return b ? b->err.c_str() : ""; }

void flb_batch_destroy(flb_batch* b) {
  if (!b) return;
  flb::forget(b);
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  drop_graph(b);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  for (void* v : b->owned) (void)hipFree(v);
  for (void* v : b->pops)
    if (v) (void)hipFree(v);
  delete b;
}

int flb_batch_create(const flb_instance* in, uint32_t count, int32_t storage, int32_t device,
                     flb_batch** out) {
  if (!out) return FLB_ERR_ARGUMENT;
  *out = nullptr;
  if (!in || count == 0 || storage < 0 || storage > 2) return FLB_ERR_ARGUMENT;
  for (uint32_t i = 0; i < count; ++i) {
    const flb_instance& s = in[i];
    if (!s.flags || s.nx < 2 || s.ny < 2 || !(s.tau > 0.5f)) return FLB_ERR_ARGUMENT;
    const size_t N = size_t(s.nx) * s.ny;
    if (s.flags[N - 1] & FLB_INLET) return FLB_ERR_ARGUMENT;
    // Planes addressed through 32-bit offsets and buffer descriptors.
    if (flb::plane_stride(align_up(s.nx, 64) * s.ny, 4) * 4 >= (1ull << 32)) return FLB_ERR_ARGUMENT;
    if ((s.flags[0] & FLB_OUTLET) && !(s.flags[0] & FLB_INLET)) return FLB_ERR_ARGUMENT;
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
    (void)hipGetLastError();
    return FLB_ERR_DEVICE;
  }
  if (device < 0 || device >= ndev) return FLB_ERR_ARGUMENT;
  if (hipSetDevice(device) != hipSuccess) return FLB_ERR_DEVICE;
  flb_batch* b = new flb_batch();
  b->storage = storage;
  b->device = device;
  auto bail = [&](int rc) {
    flb_batch_destroy(b);
    return rc;
  };
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) b->ncu = prop.multiProcessorCount;
  size_t largest = 0;  // velocities
  for (uint32_t i = 0; i < count; ++i)
    largest = std::max(largest, 2 * sizeof(float) * in[i].nx * in[i].ny);
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess ||
      b->staging.init(largest) != hipSuccess)
    return bail(FLB_ERR_DEVICE);
  const size_t eb = storage == 0 ? 4 : 2;
  // Offsets of every instance in the shared allocations (elements).
  // Rows of every instance padded to a pitch of 64 cells.
  std::vector<size_t> off_f(count), off_c(count);
  size_t tot_f = 0, tot_c = 0;
  for (uint32_t i = 0; i < count; ++i) {
    const size_t Nd = align_up(in[i].nx, 64) * in[i].ny;
    off_f[i] = tot_f;
    tot_f += 9 * flb::plane_stride(Nd, uint32_t(eb));
    off_c[i] = tot_c;
    tot_c += align_up(Nd, 64);
  }
  uint8_t* f = nullptr;
  uint8_t* flags = nullptr;
  float *rho = nullptr, *u = nullptr, *pr0 = nullptr, *pr1 = nullptr, *pu0 = nullptr, *pu1 = nullptr;
  int rc;
  if ((rc = balloc(b, &f, tot_f * eb)) || (rc = balloc(b, &flags, tot_c)) ||
      (rc = balloc(b, &rho, tot_c)) || (rc = balloc(b, &u, 2 * tot_c)) ||
      (rc = balloc(b, &pr0, tot_c)) || (rc = balloc(b, &pr1, tot_c)) ||
      (rc = balloc(b, &pu0, 2 * tot_c)) || (rc = balloc(b, &pu1, 2 * tot_c)) ||
      (rc = balloc(b, &b->inst_sets, 4 * size_t(count))))
    return bail(rc);
  b->pops[0] = f;
  b->owned.erase(b->owned.begin());  // f, the first
  float* staging = nullptr;
  size_t max_n = 0;
  for (uint32_t i = 0; i < count; ++i) max_n = std::max(max_n, size_t(in[i].nx) * in[i].ny);
  if (flb::device_malloc(reinterpret_cast<void**>(&staging), 9 * max_n * sizeof(float), device, b) !=
      hipSuccess)
    return bail(FLB_ERR_MEMORY);
  b->host_inst.resize(count);
  use_set(b, 0);
  std::vector<float> fs, hr, hu;
  for (uint32_t i = 0; i < count && !rc; ++i) {
    const flb_instance& s = in[i];
    const size_t N = size_t(s.nx) * s.ny;
    flb::Params& p = b->host_inst[i];
    p = flb::Params{};
    p.nx = s.nx;
    p.ny = s.ny;
    p.pitch = uint32_t(align_up(s.nx, 64));
    p.N = size_t(p.pitch) * s.ny;  // device plane of a cell field
    p.NL = N;                      // host plane
    p.Np = flb::plane_stride(p.N, uint32_t(eb));
    flb::set_relaxation(p, 1.0f / s.tau);
    p.use_force = s.use_force;
    p.fx = s.use_force ? s.fx : 0.0f;
    p.fy = s.use_force ? s.fy : 0.0f;
    p.f = f + off_f[i] * eb;
    p.flags = flags + off_c[i];
    p.rho = rho + off_c[i];
    p.u = u + 2 * off_c[i];
    p.pub_rho[0] = pr0 + off_c[i];
    p.pub_rho[1] = pr1 + off_c[i];
    p.pub_u[0] = pu0 + 2 * off_c[i];
    p.pub_u[1] = pu1 + 2 * off_c[i];
    hr.assign(N, 1.0f);
    hu.assign(2 * N, 0.0f);
    if (s.rho0) std::memcpy(hr.data(), s.rho0, N * sizeof(float));
    if (s.u0) std::memcpy(hu.data(), s.u0, 2 * N * sizeof(float));
    flb::host_initial_populations(s.nx, s.ny, s.rho0, s.u0, fs);
    // Host planes of nx * ny cells into pitched device planes (a device plane
    // is exactly ny rows of pitch cells, so `planes` planes are planes * ny rows).
    auto in2d = [&](void* dst, const void* src, size_t elem, int planes) {
      return b->staging.to_device(b->stream, dst, src, p.pitch * elem, s.nx * elem,
                                  size_t(s.ny) * planes);
    };
    hipError_t e = in2d(p.flags, s.flags, 1, 1);
    if (e == hipSuccess) e = in2d(p.rho, hr.data(), 4, 1);
    if (e == hipSuccess) e = in2d(p.u, hu.data(), 4, 2);
    for (int k = 0; k < 2 && e == hipSuccess; ++k) {
      e = in2d(p.pub_rho[k], hr.data(), 4, 1);
      if (e == hipSuccess) e = in2d(p.pub_u[k], hu.data(), 4, 2);
    }
    if (e == hipSuccess)
      e = b->staging.to_device(b->stream, staging, fs.data(), 9 * N * 4, 9 * N * 4, 1);
    if (e == hipSuccess) e = hipMemcpy(b->inst + i, &p, sizeof(p), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
      void (*conv)(const flb::Params*, uint32_t, const float*) =
          storage == 1 ? flb::k_batch_from_f32<flb::StoreF16S>
                       : (storage == 2 ? flb::k_batch_from_f32<flb::StoreBF16S>
                                       : flb::k_batch_from_f32<flb::StoreF32>);
      hipLaunchKernelGGL(conv, dim3(512), dim3(256), 0, b->stream, b->inst, i, staging);
      e = hipGetLastError();
      if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
    }
    if (e != hipSuccess) {
      b->err = std::string("batch upload: ") + hipGetErrorString(e);
      rc = FLB_ERR_DEVICE;
    }
  }
  (void)hipFree(staging);
  if (rc) return bail(rc);
  if ((rc = prepare_march(b, in, tot_f * eb))) return bail(rc);
  b->grid = 8 * b->ncu;
  if ((rc = build_tiles(b, 256))) return bail(rc);
  flb::keep(b);
  *out = b;
  return FLB_OK;
}

int flb_batch_configure(flb_batch* b, int32_t block_x, int32_t grid, int32_t graph_chunk) {
  if (!b) return FLB_ERR_ARGUMENT;
  const std::lock_guard<std::recursive_mutex> lock(b->in_use);
  if (block_x % 64 || block_x < 64 || block_x > 1024 || grid < 0 || graph_chunk < 0 ||
      graph_chunk % 2)
    return FLB_ERR_ARGUMENT;
  drop_graph(b);
  b->way = flb_batch::kEstimated;
  b->mode = FLB_BATCH_LAUNCH;
  b->grid = grid;
  b->graph_chunk = graph_chunk;
  if (block_x != b->block_x) return build_tiles(b, block_x);
  return FLB_OK;
}

int flb_batch_set_order(flb_batch* b, int32_t order) {
  if (!b || order < FLB_BATCH_ORDER_ROWS || order > FLB_BATCH_ORDER_BANDS) return FLB_ERR_ARGUMENT;
  const std::lock_guard<std::recursive_mutex> lock(b->in_use);
  if (order == b->order) return FLB_OK;
  drop_graph(b);
  b->way = flb_batch::kEstimated;
  b->order = order;
  return build_tiles(b, b->block_x);
}

int flb_batch_configure_persistent(flb_batch* b, int32_t block_x, int32_t blocks_per_cu,
                                   int32_t chunk) {
  if (!b) return FLB_ERR_ARGUMENT;
  const std::lock_guard<std::recursive_mutex> lock(b->in_use);
  if (block_x % 64 || block_x < 64 || block_x > 1024 || blocks_per_cu < 1 || chunk < 1)
    return FLB_ERR_ARGUMENT;
  int cap = 0, rc;
  if ((rc = persistent_capacity(b, block_x, &cap))) return rc;
  if (blocks_per_cu > cap) {
    b->err = "persistent batch: " + std::to_string(blocks_per_cu) + " blocks of " +
             std::to_string(block_x) + " threads per CU cannot be resident (at most " +
             std::to_string(cap) + ")";
    return FLB_ERR_ARGUMENT;
  }
  drop_graph(b);
  if (block_x != b->block_x && (rc = build_tiles(b, block_x))) return rc;
  b->way = flb_batch::kEstimated;
  b->mode = FLB_BATCH_PERSISTENT;
  b->persist_per_cu = blocks_per_cu;
  b->persist_chunk = chunk;
  return FLB_OK;
}

int flb_batch_step(flb_batch* b, uint64_t nsteps) {
  if (!b) return FLB_ERR_ARGUMENT;
  const std::lock_guard<std::recursive_mutex> lock(b->in_use);
  int rc = FLB_OK;
  uint64_t left = nsteps;
  while (left > 0 && !rc) {
    if (b->mode == FLB_BATCH_PERSISTENT && left > 1) {
      // The last step of the call runs as a plain launch and writes the fields.
      const uint64_t k = std::min<uint64_t>(left - 1, uint64_t(b->persist_chunk));
      rc = launch_persistent(b, uint32_t(k), uint32_t(b->t & 1));
      b->t += k;
      left -= k;
      continue;
    }
    // Graph replays need an even start; the last step writes the readback fields.
    if (b->graph_chunk > 0 && (b->t & 1) == 0 && left > uint64_t(b->graph_chunk)) {
      if ((rc = ensure_graph(b))) break;
      BAT_HIP(b, hipGraphLaunch(b->graph[b->set], b->stream));
      use_set(b, b->graph_set[b->set]);
      b->t += uint64_t(b->graph_chunk);
      left -= uint64_t(b->graph_chunk);
    } else {
      int done = 0;
      rc = advance(b, b->t, left, true, &done);
      b->t += uint64_t(done);
      left -= uint64_t(done);
    }
  }
  return rc;
}

int flb_test_batch_pass_shape(flb_batch* b, int32_t steps, uint32_t rows) {
  if (!b) return FLB_ERR_ARGUMENT;
  const std::lock_guard<std::recursive_mutex> lock(b->in_use);
  if (!b->rule_shape.steps || steps == 1 || steps > flb::kMarchMax || (steps > 1 && rows == 0))
    return FLB_ERR_ARGUMENT;
  BAT_HIP(b, hipStreamSynchronize(b->stream));
  drop_graph(b);
  b->any_shape = steps >= 0;
  return set_shape(b, steps < 0 ? b->rule_shape : flb::MarchShape{steps, rows});
}

int flb_batch_sync(flb_batch* b) {
  if (!b) return FLB_ERR_ARGUMENT;
  BAT_HIP(b, hipStreamSynchronize(b->stream));
  return FLB_OK;
}

int flb_batch_step_timed(flb_batch* b, uint64_t nsteps, float* ms) {
  if (!b) return FLB_ERR_ARGUMENT;
  hipEvent_t e0, e1;
  BAT_HIP(b, hipEventCreate(&e0));
  BAT_HIP(b, hipEventCreate(&e1));
  BAT_HIP(b, hipEventRecord(e0, b->stream));
  int rc = flb_batch_step(b, nsteps);
  BAT_HIP(b, hipEventRecord(e1, b->stream));
  BAT_HIP(b, hipEventSynchronize(e1));
  float v = 0.0f;
  BAT_HIP(b, hipEventElapsedTime(&v, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (ms) *ms = v;
  return rc;
}

// For each tile order, times block sizes {64, 128, 256, 512} x {4, 16, 64
// blocks per CU, one block per tile} with one launch per step, and the
// persistent kernel at block sizes {256, 512} with 1, 2 or 4 resident blocks
// per CU (as far as they fit), over `steps` steps each (the state advances); then
// the passes, which none of these settings change, and keeps the fastest.
// best_grid reports blocks of the launch (0: one per tile); a persistent
// winner reports -(blocks per CU).  Where the passes win, the settings are the
// fastest ones of the single steps that are left: calls of one step.
int flb_batch_autotune(flb_batch* b, uint32_t steps, int32_t* best_block, int32_t* best_grid,
                       float* best_ms) {
  if (!b || steps == 0) return FLB_ERR_ARGUMENT;
  const std::lock_guard<std::recursive_mutex> lock(b->in_use);
  const int blocks[4] = {64, 128, 256, 512};
  const int per_cu[4] = {4, 16, 64, 0};
  const int chunk = b->graph_chunk;
  struct Setting {
    float ms = 1e30f;
    int block, grid, order;
    bool persistent = false;
  } best, launched;
  best.block = launched.block = b->block_x;
  best.grid = launched.grid = b->grid;
  best.order = launched.order = b->order;
  int rc = FLB_OK;
  auto time_it = [&](flb_batch::Way way, float* ms) -> int {
    b->way = way;
    int r = flb_batch_step(b, 2);  // warm
    if (!r) r = flb_batch_step_timed(b, steps, ms);
    return r;
  };
  for (int order : {FLB_BATCH_ORDER_ROWS, FLB_BATCH_ORDER_INSTANCE, FLB_BATCH_ORDER_BANDS}) {
    if ((rc = flb_batch_set_order(b, order))) return rc;
    for (int bx : blocks)
      for (int pc : per_cu) {
        if ((rc = flb_batch_configure(b, bx, pc * b->ncu, 0))) return rc;
        float ms = 0.0f;
        if ((rc = time_it(flb_batch::kSingle, &ms))) return rc;
        if (ms < launched.ms) launched = Setting{ms, bx, pc * b->ncu, order, false};
      }
    for (int bx : {256, 512})
      for (int pc : {1, 2, 4}) {
        int cap = 0;
        if ((rc = persistent_capacity(b, bx, &cap))) return rc;
        if (pc > cap) continue;
        if ((rc = flb_batch_configure_persistent(b, bx, pc, int(steps)))) return rc;
        float ms = 0.0f;
        if ((rc = time_it(flb_batch::kSingle, &ms))) return rc;
        if (ms < best.ms) best = Setting{ms, bx, pc, order, true};
      }
  }
  if (launched.ms <= best.ms) best = launched;
  flb_batch::Way way = flb_batch::kSingle;
  if (b->shape.steps && steps > 1) {
    if ((rc = flb_batch_set_order(b, launched.order)) ||
        (rc = flb_batch_configure(b, launched.block, launched.grid, 0)))
      return rc;
    float ms = 0.0f;
    if ((rc = time_it(flb_batch::kPasses, &ms))) return rc;
    if (ms < best.ms) {
      best = launched;
      best.ms = ms;
      way = flb_batch::kPasses;
    }
  }
  if ((rc = flb_batch_set_order(b, best.order))) return rc;
  if (best.persistent) {
    if ((rc = flb_batch_configure_persistent(b, best.block, best.grid, chunk > 0 ? chunk : 100))) return rc;
  } else if ((rc = flb_batch_configure(b, best.block, best.grid, chunk))) {
    return rc;
  }
  // Timed by calls of one step, the tuning says nothing of longer runs.
  b->way = steps > 1 ? way : flb_batch::kEstimated;
  if (best_block) *best_block = best.block;
  if (best_grid) *best_grid = best.persistent ? -best.grid : best.grid;
  if (best_ms) *best_ms = best.ms / float(steps);
  return FLB_OK;
}

int flb_batch_read(flb_batch* b, uint32_t i, float* u, float* rho) {
  if (!b || i >= b->host_inst.size()) return FLB_ERR_ARGUMENT;
  const flb::Params& p = b->host_inst[i];
  const size_t row = p.nx * sizeof(float), dp = p.pitch * sizeof(float);
  if (u) BAT_HIP(b, b->staging.to_host(b->stream, u, p.u, dp, row, 2 * size_t(p.ny)));
  if (rho) BAT_HIP(b, b->staging.to_host(b->stream, rho, p.rho, dp, row, p.ny));
  if (!u && !rho) BAT_HIP(b, hipStreamSynchronize(b->stream));
  return FLB_OK;
}

int flb_batch_read_populations(flb_batch* b, uint32_t i, float* f) {
  if (!b || !f || i >= b->host_inst.size()) return FLB_ERR_ARGUMENT;
  const flb::Params& p = b->host_inst[i];
  float* tmp = nullptr;
  BAT_HIP(b, flb::device_malloc(reinterpret_cast<void**>(&tmp), 9 * p.NL * sizeof(float), b->device, nullptr));
  void (*conv)(const flb::Params*, uint32_t, float*) =
      b->storage == 1 ? flb::k_batch_to_f32<flb::StoreF16S>
                      : (b->storage == 2 ? flb::k_batch_to_f32<flb::StoreBF16S>
                                         : flb::k_batch_to_f32<flb::StoreF32>);
  hipLaunchKernelGGL(conv, dim3(512), dim3(256), 0, b->stream, b->inst, i, tmp);
  hipError_t e = hipGetLastError();
  const size_t bytes = 9 * p.NL * sizeof(float);
  if (e == hipSuccess) e = b->staging.to_host(b->stream, f, tmp, bytes, bytes, 1);
  (void)hipFree(tmp);
  BAT_HIP(b, e);
  return FLB_OK;
}

uint64_t flb_batch_time(const flb_batch* b) { return b ? b->t : 0; }

int32_t flb_batch_order(const flb_batch* b) { return b ? b->order : -1; }

int flb_batch_info(const flb_batch* b, int32_t* block_x, int32_t* grid, int32_t* graph_chunk,
                   uint32_t* ntiles) {
  if (!b) return FLB_ERR_ARGUMENT;
  const bool pers = b->mode == FLB_BATCH_PERSISTENT;
  if (block_x) *block_x = b->block_x;
  if (grid) *grid = pers ? -b->persist_per_cu : b->grid;
  if (graph_chunk) *graph_chunk = pers ? b->persist_chunk : b->graph_chunk;
  if (ntiles) *ntiles = b->ntiles;
  return FLB_OK;
}

}  // extern "C"
