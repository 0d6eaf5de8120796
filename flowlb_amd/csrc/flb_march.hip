// flb_march.hip -- the multi-step pass (flb_march.h) over a single-phase domain.
#include "flb_march.h"
#include "flb_internal.h"

namespace flb {

template <class S, int T, int MODEL, bool TRACE>
__global__ void __launch_bounds__(64 * kMarchWaves)
__attribute__((amdgpu_waves_per_eu(march_occupancy<S, MODEL>())))
k_march(const Params p, const March a) {
  const MarchWork w = march_work(a.grid, p.ny);
  if (w.ya >= w.yb) return;
  if (w.io) march_rows<S, T, MODEL, true, TRACE>(p, a, w.strip, w.ya, w.yb);
  else march_rows<S, T, MODEL, false, TRACE>(p, a, w.strip, w.ya, w.yb);
}

namespace {
template <class S, int T>
MarchFn march_fn(int model, bool trace) {
  if constexpr (S::kBytes >= 4) {  // drag and the trace: FP32 and FP64 storage
    if (trace) return k_march<S, T, kMarchDrag, true>;
    if (model == kMarchDrag) return k_march<S, T, kMarchDrag, false>;
  }
  switch (model) {
    case kMarchPlain: return k_march<S, T, kMarchPlain, false>;
    case kMarchForced: return k_march<S, T, kMarchForced, false>;
    case kMarchUnforced: return k_march<S, T, kMarchUnforced, false>;
    default: return k_march<S, T, kMarchGeneral, false>;
  }
}
template <class S>
MarchFn march_steps(int steps, int model, bool trace) {
  switch (steps) {
    case 2: return march_fn<S, 2>(model, trace);
    case 3: return march_fn<S, 3>(model, trace);
    case 4: return march_fn<S, 4>(model, trace);
    default: return nullptr;
  }
}
}  // namespace

MarchFn get_march(int storage, int steps, int model, bool trace) {
  switch (storage) {
    case 1: return march_steps<StoreF16S>(steps, model, trace);
    case 2: return march_steps<StoreBF16S>(steps, model, trace);
    case 3: return march_steps<StoreF64>(steps, model, trace);
    default: return march_steps<StoreF32>(steps, model, trace);
  }
}

}  // namespace flb
