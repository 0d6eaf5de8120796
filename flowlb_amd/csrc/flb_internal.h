// flb_internal.h -- handle layout and helpers shared by the translation units
// of libflbcore.so (not part of the public ABI).
#pragma once

#include <atomic>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/flb_core.h"
#include "flb_device.h"

namespace flb {
// Stride between population planes, in elements of elem_bytes: the plane
// rounded up to 8 KiB, plus 4 KiB.  A wavefront reads and writes the same
// offset of nine planes; with planes a multiple of 8 KiB apart (any
// power-of-two grid) those nine streams meet on the same HBM channels.  The
// nine-plane esoteric pattern in 16-bit at 8192 x 2048 moved 5.88 TB/s
// unpadded and 6.32-6.39 TB/s with the planes 4-6 KiB past a multiple of 8 KiB
// (FP32 moved 5.3-5.45 TB/s either way).  The stride stays a multiple of 256
// bytes, so every plane starts 256-byte aligned.
inline uint64_t plane_stride(uint64_t cells, uint32_t elem_bytes) {
  const uint64_t bytes = (cells * elem_bytes + 8191u) / 8192u * 8192u + 4096u;
  return bytes / elem_bytes;
}

using KernelFn = void (*)(const Params);
using MassFn = void (*)(const Params, double*);
using ConvOutFn = void (*)(const Params, float*);
using ConvInFn = void (*)(const Params, const float*);
using ConvOut64Fn = void (*)(const Params, double*);
using ConvIn64Fn = void (*)(const Params, const double*);
using HistFn = void (*)(const Params, unsigned long long*);
KernelFn get_stream_collide(int storage, int odd, bool fs, bool mom);
KernelFn get_stream_collide_dense(int storage, int odd, bool mom);
KernelFn get_stream_collide_surface(int storage, int odd, bool mom);
KernelFn get_stream_collide_all(int storage, int odd, bool mom);  // nullptr for FP64
KernelFn get_fs1(int storage, int odd);
KernelFn get_fs_update(int storage, int odd, uint32_t nx, uint32_t ny);
KernelFn get_stream_collide_trace(int storage, int odd, bool mom);  // FP32 or FP64
MassFn get_pop_mass(int storage);
MassFn get_fs_mass(int storage);
ConvOutFn get_pop_to_f32(int storage);
ConvOut64Fn get_pop_to_f64(int storage);
ConvInFn get_f32_to_pop(int storage);
ConvIn64Fn get_f64_to_pop(int storage);
HistFn get_flag_hist();

// The multi-step pass (flb_march.h): `steps` in [kMarchMin, kMarchMax].
struct March;
struct MarchGrid;
using MarchFn = void (*)(const Params, const March);
constexpr int kMarchMin = 2, kMarchMax = 4;
// Shape of the passes of a run of steps: steps per pass and rows per chunk.
struct MarchShape {
  int steps;
  uint32_t rows;
};
MarchShape march_shape(int cus, uint64_t strip_rows, int elem_bytes, bool heavy);
// Steps of the next pass of a run with `left` steps to go; 0: a single step.
inline int march_steps_next(uint64_t left, int most) {
  if (left < 2 || most < kMarchMin) return 0;
  return int(left == uint64_t(most) + 1 ? (left + 1) / 2 : (left < uint64_t(most) ? left : most));
}
// Strips of a domain of nx columns for passes of `steps` steps, those whose 64
// columns hold a column marked in io (inlet or outlet cells) first; returns
// the number of these.
uint32_t march_strips(uint32_t nx, int steps, const std::vector<uint8_t>& io,
                      std::vector<uint32_t>& order);
// Columns with an inlet or outlet cell; false where passes are not used: an
// inlet cell in the last column or an outlet cell in the first one reads the
// linear neighbour in another row, and a pass needs as many rows as steps.
bool march_columns_io(const uint8_t* flags, uint32_t nx, uint32_t ny, std::vector<uint8_t>& io);
// trace: record the trace (SRT with or without drag; FP32 and FP64).
MarchFn get_march(int storage, int steps, int model, bool trace);
}  // namespace flb

namespace flb {
// Pinned buffers a handle's copies to and from pageable memory go through (two,
// so that one is filled while the other is copied): one for the largest field from
// the start, so that short readbacks never allocate, the other by the first copy
// of more than 8 MiB; freed with the handle.  A strided copy to or from pageable memory is done
// row by row by the runtime, 7 us each: 7.2 ms for 1000 rows of 8 KB against 0.25 ms
// through the buffers (54 GB/s over the bus, 70 GB/s for the host's copy).
//
// The runtime copies by itself (direct) where that is the faster way:
//  - memory the HIP runtime knows, as a caller's pinned buffers, needs no second copy:
//    u and rho of 1024 x 512 cells 0.13 ms, through the buffers 0.34 (as a strided
//    copy also where the rows have no padding: 64 x 16 18 us, as a plain one 25);
//  - contiguous copies of middling size, which the runtime stages as well: to the
//    host 8 KiB 23 us, 16 by the buffers, 32 KiB 30 / 35, 590 KB 48 / 55, 1.2 MB 92 / 90,
//    19 MB 1100 / 840; to the device, with what the caller does before, 150 KB 36 / 42,
//    9.4 MB 527 / 600, 38 MB 9320 / 9320.
// One copy at a time, as all calls on a handle.
struct Staging {
  static constexpr size_t kBytes = 8u << 20;
  static constexpr size_t kSmall = 16u << 10;        // direct above, to the host
  static constexpr size_t kLargeIn = 1u << 20;       // direct below, to the host
  static constexpr size_t kLargeOut = 2 * kBytes;    // direct up to, to the device
  void* buf[2] = {nullptr, nullptr};
  size_t size = 0;
  hipEvent_t done[2] = {nullptr, nullptr};
  Staging() = default;
  Staging(const Staging&) = delete;
  Staging& operator=(const Staging&) = delete;
  ~Staging();
  // With the handle's device current.  bytes: the largest field to be copied (each
  // pinned allocation takes 0.2 to 0.6 ms).
  hipError_t init(size_t bytes);
  // `rows` rows of row_bytes: contiguous on the host, `pitch` bytes apart on
  // the device.  Returns when the host memory may be used.
  hipError_t to_host(hipStream_t s, void* host, const void* dev, size_t pitch, size_t row_bytes,
                     size_t rows);
  hipError_t to_device(hipStream_t s, void* dev, const void* host, size_t pitch, size_t row_bytes,
                       size_t rows);

 private:
  bool reserve(size_t bytes);
  void release();
  static bool known(const void* host);  // to the runtime
};
}  // namespace flb

namespace flb {
// Device memory that a handle or batch holds for speed alone: the second population
// array, the buffers of the last gradient.  Where an allocation of the library
// finds no room, the others on that device give theirs back (device_malloc), so
// that what fits without such memory still fits.  Any thread may ask for it: calls
// that use it hold in_use, and who uses it keeps it.
struct Kept {
  std::recursive_mutex in_use;
  int device = 0;
  std::atomic<size_t> idle{0};  // bytes held between calls (Workspace)
  // With in_use held.  Waits for the work on the memory; returns whether any was freed.
  virtual bool give_back() = 0;

 protected:
  ~Kept() = default;
};
void keep(Kept* k);    // from now on others may ask
void forget(Kept* k);  // from now on they do not; waits for one who is asking
size_t idle_elsewhere(const Kept* self);  // on self's device
// hipMalloc; without room, after the others on the device, and owner unless its
// calling thread holds in_use (self), gave back what they keep.
hipError_t device_malloc(void** p, size_t bytes, int device, const Kept* self);

// Device buffers a handle keeps between calls that need the same ones
// (objective, gradient), by slot.  Allocating and freeing 2 GB takes 0.6 ms, and
// now and then 60 to 200 ms.  After each call trim() gives back what exceeds a
// thirty-second of the device's memory (9 GB of 288) for all handles together.
struct Workspace {
  enum Slot { kCheckpoints, kState, kTrace, kTraceOnce, kAdjoint, kAdjointAlt, kDensity, kVelocity,
              kAlpha, kSums, kColumn, kSlots };
  void* ptr[kSlots] = {};
  size_t size[kSlots] = {};
  Kept* owner = nullptr;
  Workspace() = default;
  Workspace(const Workspace&) = delete;
  Workspace& operator=(const Workspace&) = delete;
  ~Workspace() { trim(0); }
  // A buffer of at least `count` elements, nullptr if there is no memory.
  template <class T>
  T* get(Slot s, size_t count) {
    const size_t bytes = (count ? count : 1) * sizeof(T);
    if (size[s] < bytes) {
      drop(s);
      if (device_malloc(&ptr[s], bytes, owner->device, owner) != hipSuccess) {
        ptr[s] = nullptr;
        return nullptr;
      }
      size[s] = bytes;
    }
    return static_cast<T*>(ptr[s]);
  }
  void drop(Slot s) {
    if (ptr[s]) (void)hipFree(ptr[s]);
    ptr[s] = nullptr;
    size[s] = 0;
  }
  size_t held() const {
    size_t n = 0;
    for (size_t b : size) n += b;
    return n;
  }
  // Frees the largest buffers until at most `most` bytes are held.
  void trim(size_t most) {
    while (held() > most) {
      int big = 0;
      for (int s = 1; s < kSlots; ++s)
        if (size[s] > size[big]) big = s;
      drop(Slot(big));
    }
    if (owner) owner->idle = held();
  }
};
}  // namespace flb

struct flb_handle : flb::Kept {
  flb_options opt{};
  flb::Workspace work;
  flb::Staging staging;
  uint32_t nx = 0, ny = 0;
  uint32_t pitch = 0;  // row stride of the device planes (cells)
  uint64_t N = 0;      // cells, nx * ny (host arrays)
  uint64_t Nd = 0;     // device plane of a cell field, pitch * ny
  uint64_t Np = 0;     // population plane stride (elements), plane_stride(Nd, elem_bytes)
  int elem_bytes = 4;   // bytes per stored population
  int field_bytes = 4;  // bytes per element of the cell fields (8 for FP64)
  hipStream_t stream = nullptr;
  void* f = nullptr;  // with f_alt not in `owned`: passes exchange the two
  // Single phase, the multi-step pass (flb_march.h): second population array
  // (null where the pass is not used) and, per number of steps, the strips with
  // those that hold an inlet or outlet column first and the number of these.
  void* f_alt = nullptr;
  uint32_t* march_order[flb::kMarchMax + 1] = {};
  uint32_t march_io[flb::kMarchMax + 1] = {};
  // Shapes set by flb_test_pass_shape; steps < 0: by march_shape, adjoint_shape.
  flb::MarchShape pass_shape{-1, 0}, reverse_shape{-1, 0};
  uint8_t* flags[2] = {nullptr, nullptr};
  int cur = 0;
  float* rho = nullptr;
  float* u = nullptr;
  float* pub_rho[2] = {nullptr, nullptr};
  float* pub_u[2] = {nullptr, nullptr};
  float* mass = nullptr;
  float* excess[2] = {nullptr, nullptr};  // shares by step parity (index cur: read)
  float* phi = nullptr;
  float* rec = nullptr;
  uint32_t* tile_work = nullptr;  // free surface: per-tile work words (Params::tile_work)
  uint32_t* tile_pub = nullptr;   // free surface: chunks holding an inlet/outlet publisher
  uint32_t work_x = 0, tile_rows = 0;
  // Free-surface pass-1 lists by step parity (Params::fs1_list), their
  // lengths (4 words per parity) and the update's per-tile skip marks.
  uint32_t* fs1_list[2] = {nullptr, nullptr};
  uint32_t* counts = nullptr;
  uint32_t* tile_list = nullptr;  // tiles the update of this step evaluates
  uint32_t* tile_body = nullptr;  // tiles stream-collide updates (bodies of fluid)
  uint32_t* tile_counts = nullptr;  // its length, by step parity
  // Stream-collide launch window: the box of chunks with stream-collide work
  // (device, by step parity) and its copy in mapped host memory (box, step).
  uint32_t* box = nullptr;
  unsigned long long* box_host = nullptr;      // host view
  unsigned long long* box_host_dev = nullptr;  // its device address (Params::box_host)
  bool seam_y_closed = false, seam_x_closed = false;  // a wall row / column on the edge
  // flb_step keeps at most 2 kGroup steps queued, so that the box the host
  // sizes a launch from is at most a few steps old: it records an event after
  // every kGroup-th step (ring of kRing) and, starting a group, waits for the
  // event two groups back.
  static constexpr int kGroup = 4;
  static constexpr int kRing = 4;
  static constexpr int kInFlight = 2 * kGroup;  // queued steps at most
  hipEvent_t in_flight[kRing] = {};
  int cus = 256;  // compute units of the device (grid size of the list-driven pass 1)
  float* alpha = nullptr;     // Brinkman solid fraction (allocated on first use)
  float* rho_init = nullptr;  // rho0 and u0 as given to flb_create
  float* u_init = nullptr;
  double* partial = nullptr;
  // Device address of the file-scope histogram scratch on this handle's GPU
  // (flb_flag_histogram_noalloc); not owned.
  unsigned long long* hist_scratch = nullptr;
  hipError_t hist_scratch_err = hipSuccess;
  size_t partial_len = 0;
  uint64_t t = 0;
  float inv_tau = 0.0f;
  std::vector<void*> owned;
  std::string err;

  flb_handle() { work.owner = this; }
  bool give_back() override;
};


namespace flb {
// Helpers defined in flb_core.hip.
int set_error(flb_handle* h, int code, const std::string& msg);
Params make_params(const flb_handle* h, int bx);
int handle_block_x(const flb_handle* h);
// A pass of T steps.  trace: as March::trace, with the window bits and the
// buffer for the discharge of `column` (nullptr: no trace).
struct MarchTrace {
  void* trace;
  double* discharge;
  uint32_t column, window;
};
int enqueue_march_ex(flb_handle* h, int T, bool moments, const MarchTrace* trace);
MarchGrid march_grid(const flb_handle* h, int T, uint32_t rows, uint32_t io_rows);
MarchShape adjoint_shape(const flb_handle* h);  // of the adjoint's passes
int march_most(const flb_handle* h);  // steps per pass of a long run, 0: no passes
// Copies `planes` planes of cells of `elem` bytes between a host array
// (planes of nx * ny, row-major) and a pitched device array (planes of Nd),
// on the handle's stream, and waits for the copy.
int copy_cells_in(flb_handle* h, void* dev, const void* host, size_t elem, int planes);
int copy_cells_out(flb_handle* h, void* host, const void* dev, size_t elem, int planes);
// Shifted initial populations feq(rho0, u0) in the odd-step slot pattern.
void host_initial_populations(uint32_t nx, uint32_t ny, const float* rho0, const float* u0,
                              std::vector<float>& fs);
}  // namespace flb

// For tests and measurements, on handles whose domain fits the passes: the steps
// (0: single steps only; 2 to 4, in reverse 2 or 3) and rows per chunk of the
// passes in place of the rules' choice; steps < 0 returns to the rules.
extern "C" {
int flb_test_pass_shape(flb_handle* h, int32_t steps, uint32_t rows, int32_t reverse_steps,
                        uint32_t reverse_rows);
int flb_test_batch_pass_shape(struct flb_batch* b, int32_t steps, uint32_t rows);
}
