// flb_march.hip -- the multi-step pass (flb_march.h) over a single-phase
// domain: one wavefront per block, blocks of an XCD on adjacent strips.
#include "flb_march.h"
#include "flb_internal.h"

namespace flb {

// A block is kMarchWaves wavefronts.  The first io_strips * chunks blocks take a
// chunk of an inlet/outlet strip each, split by rows between their wavefronts
// (such a strip costs two to three times the others: with whole chunks these
// wavefronts ended last, alone).  The others take a chunk of kMarchWaves adjacent
// strips, which stay within a row of each other (a barrier per row), so that
// the lines two strips share are read and written while they are in the L2.
// Block b runs on XCD b mod 8; one XCD's blocks take consecutive groups of strips.
template <class S, int T, int MODEL>
__global__ void __launch_bounds__(64 * kMarchWaves)
__attribute__((amdgpu_waves_per_eu(march_occupancy<S, MODEL>())))
k_march(const Params p, const March a) {
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(threadIdx.x / 64u));
  const uint32_t io_blocks = a.io_strips * a.chunks;
  if (blockIdx.x < io_blocks) {
    const uint32_t chunk = blockIdx.x / a.io_strips;
    const uint32_t ya = chunk * a.rows + wave * a.io_rows;
    const uint32_t end = min((chunk + 1u) * a.rows, p.ny);
    const uint32_t yb = min(ya + a.io_rows, end);
    if (ya < yb) march_rows<S, T, MODEL, true>(p, a, a.order[blockIdx.x - chunk * a.io_strips], ya, yb);
    return;
  }
  const uint32_t b = blockIdx.x - io_blocks, per = (gridDim.x - io_blocks) / 8u;
  const uint32_t w = (b % 8u) * per + b / 8u;
  const uint32_t chunk = div_by(w, a.groups, a.group_magic);
  const uint32_t k = a.io_strips + (w - chunk * a.groups) * uint32_t(kMarchWaves) + wave;
  const uint32_t ya = chunk * a.rows, yb = min(ya + a.rows, p.ny);
  if (ya < yb && k < a.strips) march_rows<S, T, MODEL, false>(p, a, a.order[k], ya, yb);
}

namespace {
template <class S, int T>
MarchFn march_fn(int model) {
  switch (model) {
    case kMarchPlain: return k_march<S, T, kMarchPlain>;
    case kMarchForced: return k_march<S, T, kMarchForced>;
    case kMarchUnforced: return k_march<S, T, kMarchUnforced>;
    default: return k_march<S, T, kMarchGeneral>;
  }
}
template <class S>
MarchFn march_steps(int steps, int model) {
  switch (steps) {
    case 2: return march_fn<S, 2>(model);
    case 3: return march_fn<S, 3>(model);
    case 4: return march_fn<S, 4>(model);
    default: return nullptr;
  }
}
}  // namespace

MarchFn get_march(int storage, int steps, int model) {
  switch (storage) {
    case 1: return march_steps<StoreF16S>(steps, model);
    case 2: return march_steps<StoreBF16S>(steps, model);
    case 3: return march_steps<StoreF64>(steps, model);
    default: return march_steps<StoreF32>(steps, model);
  }
}

}  // namespace flb
