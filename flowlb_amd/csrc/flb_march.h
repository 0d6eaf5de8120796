// flb_march.h -- several lattice steps of a single-phase domain in one pass
// over memory (device code shared by flb_march.hip and flb_batch.hip).
//
// A wavefront owns a strip of columns, one column per lane, and marches up a
// chunk of rows.  In one iteration it loads the next row's populations and
// runs step 1 on that row, step 2 on the row below it, ... step T on the row
// T - 1 below, whose populations it stores.  What step s needs of step s - 1
// comes from registers: the populations along x of the row itself (kept one
// iteration), those moving up of the row below (kept two) and those moving down
// of the row above (just computed), each shifted by a lane for its x component
// (DPP wavefront shift).  No LDS; no wavefront waits for another's values.
//
// Dependencies reach one cell per step, so of the 64 columns a wavefront loads
// the 64 - 2 (T - 1) inner ones are its own, and it starts T - 1 rows below its
// chunk and ends T - 1 above.  Neighbouring wavefronts read those halos from
// the state before the pass, so the pass reads one population array and
// writes another.  The cells' results are those of T single steps, bit for
// bit: the same per-cell arithmetic in the same order, 16-bit storage rounded
// between the steps as a store and a load would, walls returning what they
// receive (what they leave in place in the in-place slot layout).
//
// What bounds it: a single step moves 18 values per cell (72 bytes in FP32) and is
// bound by memory on large grids and by the launch on small ones.  T = 4 steps in
// one pass move about a third of that and the vector units become the bound: about
// 110 instructions per step and row of 64 columns, 10 % of them for halo columns.
// A pass of four over 8192 x 2048 in FP32 reads 966 MB, 1.6 times the populations
// (22 rows for a chunk of 16, 64 columns for 58), and writes 628 MB.  Measured in
// one run, us per step, single steps / passes of one handle alone, and in brackets
// of three stepping side by side: 8192 x 2048 FP32 201 / 80 (5.0 TB/s of that traffic,
// 0.7 of the vector rate) [233 / 76], FP16S 119 / 65 [116 / 57], FP64 432 / 148 [480 /
// 153], 2001 x 401 FP64 with a force 18.7 / 12.3 [16.8 / 8.9], 1024 x 256 FP32 6.2 / 4.0
// [3.3 / 2.1], 512 x 128 FP32 4.9 / 3.5 [3.3 / 1.4].  Where single steps are the faster
// way they are taken: flb_cost.h.
#pragma once

#include "flb_cell.h"

namespace flb {

constexpr uint32_t kMarchLanes = 64;
constexpr int kMarchWaves = 4;  // wavefronts per block
constexpr uint32_t march_columns(int steps) { return kMarchLanes - 2u * uint32_t(steps - 1); }

// Blocks of a pass over a single domain.  The first io_strips * io_chunks blocks
// take rows of an inlet/outlet strip each, io_rows for each of their wavefronts
// (such a strip costs two to three times the others: with whole chunks these
// wavefronts ended last, alone).  The others take a chunk of kMarchWaves adjacent
// strips, which stay within a row of each other (a barrier per row), so that
// the lines two strips share are read and written while they are in the L2.
// Block b runs on XCD b mod 8; one XCD's blocks take consecutive groups of strips.
struct MarchGrid {
  uint32_t strips, io_strips;  // strips, and those whose 64 columns hold an inlet or outlet cell
  uint32_t chunks;             // chunks of rows
  uint32_t rows;               // rows per chunk
  uint32_t io_chunks;          // blocks per inlet/outlet strip
  uint32_t io_rows;            // rows a wavefront takes of such a strip
  uint32_t groups, group_magic;  // blocks per chunk of the other strips, div_magic of it
  uint32_t blocks;
  const uint32_t* order;       // strips, the io_strips ones first
};
struct MarchWork {
  uint32_t strip, ya, yb;  // nothing to do where ya >= yb
  bool io;
};
__device__ __forceinline__ MarchWork march_work(const MarchGrid& g, uint32_t ny) {
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(threadIdx.x / 64u));
  const uint32_t io_blocks = g.io_strips * g.io_chunks;
  MarchWork w{};
  if (blockIdx.x < io_blocks) {
    const uint32_t chunk = blockIdx.x / g.io_strips;
    w.io = true;
    w.strip = g.order[blockIdx.x - chunk * g.io_strips];
    w.ya = (chunk * uint32_t(kMarchWaves) + wave) * g.io_rows;
    w.yb = min(w.ya + g.io_rows, ny);
    return w;
  }
  const uint32_t b = blockIdx.x - io_blocks, per = (gridDim.x - io_blocks) / 8u;
  const uint32_t i = (b % 8u) * per + b / 8u;
  const uint32_t chunk = div_by(i, g.groups, g.group_magic);
  const uint32_t k = g.io_strips + (i - chunk * g.groups) * uint32_t(kMarchWaves) + wave;
  if (k >= g.strips) return w;
  w.strip = g.order[k];
  w.ya = chunk * g.rows;
  w.yb = min(w.ya + g.rows, ny);
  return w;
}

// One pass of T steps, from time t.
struct March {
  const void* f_in;   // populations at time t
  void* f_out;        // populations at time t + T
  // Densities and velocities published for inlet/outlet neighbours at the
  // step before the pass, and by its last step.
  const float* pub_rho_in;
  const float* pub_u_in;
  float* pub_rho_out;
  float* pub_u_out;
  // Where inlet cells find the velocity they prescribe and outlet cells the density
  // they keep: the readback fields of a handle, which its program may write to.  The
  // pass leaves those values as they are.
  const float* own_rho;
  const float* own_u;
  int32_t odd;        // t % 2
  int32_t moments;    // write the readback fields of the last step
  // TRACE: the trace of step t + k at trace + k * 3 N elements of R; and, where
  // bit k of window is set, rho u_x of the cells of `column` (0 for walls) at
  // discharge + k * ny, for the objective.
  void* trace;
  double* discharge;
  uint32_t column, window;
  MarchGrid grid;
};

// Value of the lane one to the left (lower x) / right.  The lanes at the ends
// receive zero; their columns are halo.
__device__ __forceinline__ float from_left(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float from_right(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ double from_left(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, int(uint32_t(b)), 0x138, 0xf, 0xf, true);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, int(uint32_t(b >> 32)), 0x138, 0xf, 0xf, true);
  return __builtin_bit_cast(double, uint64_t(hi) << 32 | lo);
}
__device__ __forceinline__ double from_right(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, int(uint32_t(b)), 0x130, 0xf, 0xf, true);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, int(uint32_t(b >> 32)), 0x130, 0xf, 0xf, true);
  return __builtin_bit_cast(double, uint64_t(hi) << 32 | lo);
}

__device__ __forceinline__ uint32_t left_flags(uint32_t fl) {
  return uint32_t(__builtin_amdgcn_update_dpp(0, int(fl), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ uint32_t right_flags(uint32_t fl) {
  return uint32_t(__builtin_amdgcn_update_dpp(0, int(fl), 0x130, 0xf, 0xf, true));
}

// In the flags a pass keeps of its rows (where the bit says nothing a pass uses):
// an inlet beside a wall it reads the density of, or an outlet beside a wall or an
// inlet it reads the velocity of.  Walls publish nothing and inlets no velocity;
// what the publication buffers were filled with stands there.
constexpr uint32_t kFilled = kFluid;

// A loaded value that is waited for here, in the branch that loads it: waited for
// where the branches meet, it would hold up every wavefront until the loads of the
// row ahead are in as well (1.5 % of a gradient of 1024 x 256).
template <class R>
__device__ __forceinline__ R arrived(R v) {
  asm volatile("" : "+v"(v));
  return v;
}

// How the pass holds populations between memory and the collision: in the
// arithmetic type, times kUnit.  FP16S keeps the stored scale (2^15), so that a
// conversion is all that loading, storing and rounding take.  Rounding goes in
// pairs, one conversion for two values on gfx950.
template <class S>
struct Held {
  using R = typename S::R;
  using E = typename S::T;
  static constexpr R kUnit = R(1);
  __device__ static R in(E v) { return S::decode(v); }
  __device__ static E out(R v) { return S::encode(v); }
  __device__ static void round(R* g) {}
};
template <>
struct Held<StoreF16S> {
  static constexpr float kUnit = 32768.0f;
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  __device__ static float in(_Float16 v) { return float(v); }
  // A value is rounded to FP32 before it is to FP16: the empty statement keeps
  // the compiler from fusing the collision's last multiply-add with the
  // conversion (v_fma_mixlo_f16), which rounds once.
  __device__ static void settle(float& v) { asm("" : "+v"(v)); }
  __device__ static _Float16 out(float v) {
    settle(v);
    return _Float16(v);
  }
  __device__ static void round(float* g) {
#pragma unroll
    for (int i = 0; i < 9; i++) settle(g[i]);
    g[0] = float(_Float16(g[0]));
#pragma unroll
    for (int i = 1; i < 9; i += 2) {
      const f16x2 h = __builtin_convertvector((f32x2{g[i], g[i + 1]}), f16x2);
      g[i] = float(h.x);
      g[i + 1] = float(h.y);
    }
  }
};
template <>
struct Held<StoreBF16S> {
  static constexpr float kUnit = 1.0f;
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  __device__ static float in(uint16_t v) { return StoreBF16S::decode(v); }
  __device__ static uint16_t out(float v) { return StoreBF16S::encode(v); }
  __device__ static void round(float* g) {
    g[0] = StoreBF16S::round(g[0]);
#pragma unroll
    for (int i = 1; i < 9; i += 2) {
      const bf16x2 h = __builtin_convertvector((f32x2{g[i], g[i + 1]}), bf16x2);
      const uint32_t b = __builtin_bit_cast(uint32_t, h);
      g[i] = __uint_as_float(b << 16);
      g[i + 1] = __uint_as_float(b & 0xffff0000u);
    }
  }
};

// Collision models compiled apart: plain SRT (no force, drag or subgrid
// model), SRT with a body force, any collision and subgrid model without force
// or drag, everything by the handle's options, and SRT with drag (TRACE too).
enum : int { kMarchPlain = 0, kMarchForced = 1, kMarchUnforced = 2, kMarchGeneral = 3,
             kMarchDrag = 4 };
// Wavefronts per SIMD the pass is compiled for (its registers: 128, 168, 256).  The
// interior path fits these with no scratch memory; the inlet/outlet path in the same
// kernel spills in passes of four in the plain model (10 to 14 registers in FP32 and
// 16-bit storage), with a force (24 to 26, and 8 to 12 in passes of three) and in FP64
// with drag or every option (10 to 22).  FP64 gains from four steps all the same
// (march_shape).
template <class S, int MODEL>
constexpr int march_occupancy() {
  return S::kBytes > 4 ? 2 : (MODEL >= kMarchUnforced ? 3 : 4);
}

// The density and velocity an inlet or outlet cell takes (stream_collide_cell): an
// inlet the published density of the cell at x + 1, of the step before, and the
// velocity it prescribes; an outlet the published velocity of the cell at x - 1 and
// the density it keeps.
template <class R>
struct IoValues {
  R rho, ux, uy;
};

// One step of one cell: g holds its incoming populations and receives the
// ones it emits; rho, ux, uy are set for cells that collide.
// `alpha` is the cell's solid fraction (kMarchDrag); tr receives its trace
// (stream_collide_cell).
template <class S, int MODEL, bool IO>
__device__ __forceinline__ void march_cell(const Params& p, uint8_t fl, uint32_t n, float alpha,
                                           const IoValues<typename S::R>& v, typename S::R* g,
                                           typename S::R& rho, typename S::R& ux,
                                           typename S::R& uy, typename S::R* tr) {
#pragma clang fp contract(off)
  using R = typename S::R;
  if (fl & (kGas | kWall)) {
#pragma unroll
    for (int i = 1; i < 9; i += 2) {
      const R t = g[i];
      g[i] = g[i + 1];
      g[i + 1] = t;
    }
    return;
  }
  constexpr R unit = Held<S>::kUnit;
  const uint8_t io = IO ? fl & (kInlet | kOutlet) : 0;
  R rho1, mx = R(0), my = R(0);
  if (IO && io) {
    rho = v.rho;
    rho1 = rho - R(1);
    ux = v.ux;
    uy = v.uy;
  } else {
    rho1 = g[0];
#pragma unroll
    for (int i = 1; i < 9; i++) rho1 += g[i];
    rho1 *= R(1) / unit;
    rho = R(1) + rho1;
    mx = (g[1] - g[2] + g[5] - g[6] + g[7] - g[8]) * (R(1) / unit);
    my = (g[3] - g[4] + g[5] - g[6] + g[8] - g[7]) * (R(1) / unit);
  }
  tr[0] = rho;
  tr[1] = io ? ux : mx;
  tr[2] = io ? uy : my;
  const Quotient<R> over_rho(rho);
  if (!io) {
    ux = over_rho(mx);
    uy = over_rho(my);
  }
  R fi[9], fe[9];
  bool forced = false;
  if (MODEL != kMarchPlain && MODEL != kMarchUnforced) {
    const bool brinkman = MODEL != kMarchForced && p.alpha && !io;
    if (MODEL == kMarchGeneral && brinkman) alpha = at(p.alpha, n);
    forced = apply_force<R>(p, MODEL == kMarchForced || p.use_force != 0, brinkman, R(alpha), rho,
                            over_rho, ux, uy, fi, unit);
  }
  equilibrium_shifted<R>(rho, rho1, ux, uy, fe, unit);
  const bool any = MODEL == kMarchUnforced || MODEL == kMarchGeneral;
  relax<R>(p, any ? p.collision : 0, any && p.smagorinsky != 0, io != 0, forced, over_rho, fe,
           fi, g, unit);
}

struct Fill { static constexpr bool value = false; };
struct Steady { static constexpr bool value = true; };

// The pass over one chunk of one strip: rows [ya, yb).
template <class S, int T, int MODEL, bool IO, bool TRACE = false>
__device__ __forceinline__ void march_rows(const Params& p, const March& a, uint32_t strip,
                                           uint32_t ya, uint32_t yb) {
  static_assert(T >= 2 && T <= 4, "a lane keeps the flags of the T rows in one word");
  using R = typename S::R;
  using E = typename S::T;
  constexpr int H = T - 1;  // halo
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t nx = p.nx, ny = p.ny, pitch = p.pitch;
  const uint32_t xs = strip * march_columns(T) + lane;  // column + H
  const bool own = lane >= H && lane < 64 - H && xs - H < nx;
  const uint32_t x = (xs + H * (nx - 1)) % nx;
  const uint32_t xr = x + 1 == nx ? 0u : x + 1, xl = x == 0 ? nx - 1 : x - 1;
  // Planes the first step loads from and the last one stores to (pairs i, i + 1
  // of opposite directions): at the cell, and at its neighbour in direction i.
  const bool odd = a.odd != 0, odd_last = odd != ((T & 1) == 0);
  const E* const fi = static_cast<const E*>(a.f_in);
  E* const fo = static_cast<E*>(a.f_out);
  const uint64_t Np = p.Np;
  auto up = [&](uint32_t y) { return y + 1 == ny ? 0u : y + 1; };
  auto down = [&](uint32_t y) { return y == 0 ? ny - 1 : y - 1; };

  const R* const pub_rho = fld<R>(const_cast<float*>(a.pub_rho_in));
  const R* const pub_u = fld<R>(const_cast<float*>(a.pub_u_in));
  const R* const own_rho = fld<R>(const_cast<float*>(a.own_rho));
  const R* const own_u = fld<R>(const_cast<float*>(a.own_u));
  E raw[9];
  uint8_t raw_fl;
  uint8_t next_fl = 0;  // IO: flags of the row after, which say what it loads
  float raw_alpha = 0.0f;
  IoValues<R> raw_io{};
  auto load_row = [&](uint32_t y) {
    const uint64_t rc = uint64_t(y) * pitch, ru = uint64_t(up(y)) * pitch,
                   rd = uint64_t(down(y)) * pitch;
    auto here = [&](int i) { return fi + (odd ? i : i + 1) * Np; };
    auto there = [&](int i) { return fi + (odd ? i + 1 : i) * Np; };
    raw[0] = at(fi + rc, x);
    raw[1] = at(here(1) + rc, x);
    raw[2] = at(there(1) + rc, xr);
    raw[3] = at(here(3) + rc, x);
    raw[4] = at(there(3) + ru, x);
    raw[5] = at(here(5) + rc, x);
    raw[6] = at(there(5) + ru, xr);
    raw[7] = at(here(7) + rc, x);
    raw[8] = at(there(7) + rd, xr);
    if (MODEL == kMarchDrag && p.alpha) raw_alpha = at(p.alpha + rc, x);
    if (IO) {
      raw_fl = next_fl;
      next_fl = at(p.flags + ru, x);
      if (raw_fl & kInlet) {
        raw_io.rho = at(pub_rho + rc, xr);
        raw_io.ux = at(own_u + rc, x);
        raw_io.uy = at(own_u + p.N + rc, x);
      } else if (raw_fl & kOutlet) {
        raw_io.rho = at(own_rho + rc, x);
        raw_io.ux = at(pub_u + rc, xl);
        raw_io.uy = at(pub_u + p.N + rc, xl);
      }
    } else {
      raw_fl = at(p.flags + rc, x);
    }
  };
  auto store_row = [&](uint32_t y, const R* g) {
    const uint64_t rc = uint64_t(y) * pitch, ru = uint64_t(up(y)) * pitch,
                   rd = uint64_t(down(y)) * pitch;
    auto here = [&](int i) { return fo + (odd_last ? i : i + 1) * Np; };
    auto there = [&](int i) { return fo + (odd_last ? i + 1 : i) * Np; };
    at(fo + rc, x) = Held<S>::out(g[0]);
    at(there(1) + rc, xr) = Held<S>::out(g[1]);
    at(here(1) + rc, x) = Held<S>::out(g[2]);
    at(there(3) + ru, x) = Held<S>::out(g[3]);
    at(here(3) + rc, x) = Held<S>::out(g[4]);
    at(there(5) + ru, xr) = Held<S>::out(g[5]);
    at(here(5) + rc, x) = Held<S>::out(g[6]);
    at(there(7) + rd, xr) = Held<S>::out(g[7]);
    at(here(7) + rc, x) = Held<S>::out(g[8]);
  };

  // Between step s and s + 1 (index s - 1), already shifted to the receiving
  // lane: populations 0, 1, 2 of the row s + 1 takes next; 3, 5, 8 of that row
  // and of the one below it.
  R flat[H][3], rise0[H][3], rise1[H][3];
  R pr[H], pu[H], pv[H];  // values published for inlet/outlet neighbours (IO)
#pragma unroll
  for (int s = 0; s < H; s++) {
#pragma unroll
    for (int k = 0; k < 3; k++) flat[s][k] = rise0[s][k] = rise1[s][k] = R(0);
    pr[s] = pu[s] = pv[s] = R(0);
  }
  uint32_t fls = 0;  // flags of the rows of steps 1 .. T, a byte each
  float alpha[T] = {};  // solid fractions of these rows (kMarchDrag)

  uint32_t y1 = ya >= uint32_t(H) ? ya - H : ya + ny - H;  // row of step 1 (ny >= T)
  if (IO) next_fl = at(p.flags + uint64_t(y1) * pitch, x);
  load_row(y1);
  const uint32_t iterations = yb - ya + 2 * H;
  const auto iterate = [&](uint32_t it, auto steady) {
    R g[9];
#pragma unroll
    for (int i = 0; i < 9; i++) g[i] = Held<S>::in(raw[i]);
    fls = fls << 8 | raw_fl;
    if (IO) {
      const uint32_t left = left_flags(raw_fl), right = right_flags(raw_fl);
      const bool filled = (raw_fl & kInlet) ? (right & (kGas | kWall))
                                            : (raw_fl & kOutlet) && (left & (kGas | kWall | kInlet));
      fls = (fls & ~uint32_t(kFilled)) | (filled ? kFilled : 0u);
    }
    if (MODEL == kMarchDrag) {
#pragma unroll
      for (int s = T - 1; s > 0; s--) alpha[s] = alpha[s - 1];
      alpha[0] = raw_alpha;
    }
    const IoValues<R> io_now = raw_io;
    const uint32_t y = y1;
    y1 = up(y1);
    load_row(y1);  // one row past the last is loaded and not used
    R rho = R(1), ux = R(0), uy = R(0);
    IoValues<R> kept = io_now;  // published by step s - 1 (IO)
    uint32_t ys = y;  // row of step s
#pragma unroll
    for (int s = 1; s <= T; s++) {
      if (decltype(steady)::value || it >= 2u * uint32_t(s - 1)) {
        const uint8_t fl = uint8_t(fls >> (8 * (s - 1)));
        const uint32_t n = ys * pitch + x;
        IoValues<R> v{};
        const bool solid = fl & (kGas | kWall);
        if (IO) {
          v = kept;
          if (s > 1) {
            const R next = from_right(v.rho), px = from_left(v.ux), py = from_left(v.uy);
            if (fl & kInlet) {
              v.rho = next;
              if (fl & kFilled) v.rho = arrived(at(pub_rho + uint64_t(ys) * pitch, xr));
            } else {
              v.ux = px;
              v.uy = py;
              if (fl & kFilled) {
                v.ux = arrived(at(pub_u + uint64_t(ys) * pitch, xl));
                v.uy = arrived(at(pub_u + p.N + uint64_t(ys) * pitch, xl));
              }
            }
          }
        }
        R tr[3];
        march_cell<S, MODEL, IO>(p, fl, n, alpha[s - 1], v, g, rho, ux, uy, tr);
        // The row is in the chunk (the halo rows are another wavefront's).
        if (TRACE && it - uint32_t(H + s - 1) < yb - ya && own) {
          if (!solid && a.trace) {
            R* const to = static_cast<R*>(a.trace) + uint64_t(s - 1) * 3u * p.N;
            at(to, n) = tr[0];
            at(to + p.N, n) = tr[1];
            at(to + 2 * p.N, n) = tr[2];
          }
          if ((a.window >> (s - 1) & 1u) && x == a.column)
            a.discharge[uint64_t(s - 1) * ny + ys] =
                solid ? 0.0 : double(rho) * double(IO && (fl & kInlet) ? tr[1] : ux);
        }
        if (s < T) {
          Held<S>::round(g);
        } else {
          if (own) {
            store_row(ys, g);
            if (a.moments && !solid) {
              if (!(IO && (fl & kInlet))) {
                at(fld<R>(p.u), n) = ux;
                at(fld<R>(p.u) + p.N, n) = uy;
              }
              at(fld<R>(p.rho), n) = rho;
            }
          }
          if (IO) {
            const uint32_t left = left_flags(fl), right = right_flags(fl);
            if (own && !solid && (left & kInlet)) at(fld<R>(a.pub_rho_out), n) = rho;
            if (own && !solid && (right & kOutlet) && !(fl & kInlet)) {
              at(fld<R>(a.pub_u_out), n) = ux;
              at(fld<R>(a.pub_u_out) + p.N, n) = uy;
            }
          }
        }
        if (s < T) {
          constexpr int last = H - 1;
          const int b = s - 1 < last ? s - 1 : last;
          // Incoming populations of step s + 1 on the row below, then this
          // row's into the registers.
          R in[9];
          in[0] = flat[b][0];
          in[1] = flat[b][1];
          in[2] = flat[b][2];
          in[3] = rise1[b][0];
          in[5] = rise1[b][1];
          in[8] = rise1[b][2];
          in[4] = g[4];
          in[6] = from_right(g[6]);
          in[7] = from_left(g[7]);
          flat[b][0] = g[0];
          flat[b][1] = from_left(g[1]);
          flat[b][2] = from_right(g[2]);
#pragma unroll
          for (int k = 0; k < 3; k++) rise1[b][k] = rise0[b][k];
          rise0[b][0] = g[3];
          rise0[b][1] = from_left(g[5]);
          rise0[b][2] = from_right(g[8]);
          if (IO) {
            kept.rho = pr[b];
            kept.ux = pu[b];
            kept.uy = pv[b];
            pr[b] = rho;
            pu[b] = (fl & kInlet) ? v.ux : ux;
            pv[b] = (fl & kInlet) ? v.uy : uy;
          }
#pragma unroll
          for (int i = 0; i < 9; i++) g[i] = in[i];
          ys = down(ys);
        }
      }
    }
    if (!IO) __builtin_amdgcn_s_barrier();  // a block's strips keep to the same row
  };
  // The first 2 H iterations fill the pipeline; from there every step runs.
  for (uint32_t it = 0; it < 2 * H; ++it) iterate(it, Fill{});
#pragma unroll 2
  for (uint32_t it = 2 * H; it < iterations; ++it) iterate(it, Steady{});
}

}  // namespace flb
