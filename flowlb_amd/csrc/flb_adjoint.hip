// flb_adjoint.hip -- hand-written discrete adjoint of the single-phase step
// (SRT, Guo forcing, Brinkman drag, velocity inlet, density outlet, implicit
// full-way bounce-back) for gradients of the time-averaged discharge through a
// column with respect to the Brinkman solid fraction and the inlet velocity.
// No reference counterpart: FlowLB has no adjoint.
//
// Reverse of one step, per cell and, where steps go singly, in place: the forward step of a cell
// loads nine slots and stores nine results into the same slot set (esoteric
// pull), so the adjoint kernel reads the adjoints of the stored results from
// the store slots and writes the adjoints of the loaded populations to the
// load slots.  The collision depends on the loaded populations only through
// rho and m = sum c_i f_i, so the forward recompute records three numbers per
// cell and step (the trace) instead of nine populations.
//
// Memory: the trace of every step (3 N values per step) is kept from the
// forward sweep for as many of the last checkpoint segments as fit in the
// trace budget (by default half the free device memory: on a 288 GB device
// the whole 2000-step, 1024 x 256 rollout, 6.3 GB); the earlier segments get a
// checkpoint of the populations and the inlet/outlet publication buffers every
// `ckpt` steps and are recomputed, with their trace, during the reverse sweep.
// The adjoint state (9 population planes, the adjoints of the published
// inlet/outlet values; the planes twice where the reverse steps go in passes)
// and its arithmetic are FP64: over 2000 reverse steps an
// FP32 adjoint lost about 2e-4 (relative) on cells with small gradients.  The
// trace is what the forward computed: FP32 for an FP32 handle, FP64 for an
// FP64 handle (FP64 forward and trace: the gradient of the FP64 discrete
// model).  The forward's float constants enter as their exact double values.
#include <algorithm>
#include <vector>

#include "flb_cell.h"
#include "flb_internal.h"
#include "flb_march.h"

namespace flb {

struct AdjParams {
  double* abar;         // adjoint populations, 9 planes of Np
  double* rbar[2];      // adjoint of published densities, by parity
  double* ubar[2];      // adjoint of published velocities, by parity
  double* galpha;       // dJ/dalpha accumulator (N), FP64 over all steps, or nullptr
  const void* trace;    // (rho, m_x, m_y) or inlet/outlet reads of this step, T
  const float* rho_init;
  const float* u_init;
  double* duin;         // dJ/du_inlet accumulator
  uint32_t column;
  int in_window;
  double qbar;          // 1 / number of averaged steps
};

// Equilibrium derivatives with respect to the velocity at x, with the weights
// of the forward arithmetic T (float weights for FP32, exact ones for FP64).
template <class T>
__device__ __forceinline__ double feq_dx(double rho, double ux, double uy, int i) {
  const double ex = double(cx(i)), cu = ex * ux + double(cy(i)) * uy;
  return double(wgt_r<T>(i)) * rho * (3.0 * ex + 9.0 * cu * ex - 3.0 * ux);
}

// Weighted moments of nine adjoint values.  The collision's derivatives contract
// them with polynomials of the velocities c_i of degree two at most, so six
// moments replace three sums over the nine directions (equilibrium, and its two
// velocity derivatives) and four more with a force: about 500 FP64 instructions
// per cell became 130.
struct Moments {
  double s, x, y, xx, yy, xy;
};
template <class T>
__device__ __forceinline__ Moments moments(const double* v) {
#pragma clang fp contract(on)
  const double w0 = double(wgt_r<T>(0)), w1 = double(wgt_r<T>(1)), w5 = double(wgt_r<T>(5));
  const double h = v[1] + v[2], k = v[3] + v[4], p = v[5] + v[6], m = v[7] + v[8];
  const double d = p + m;
  Moments r;
  r.s = w0 * v[0] + w1 * (h + k) + w5 * d;
  r.x = w1 * (v[1] - v[2]) + w5 * ((v[5] - v[6]) + (v[7] - v[8]));
  r.y = w1 * (v[3] - v[4]) + w5 * ((v[5] - v[6]) + (v[8] - v[7]));
  r.xx = w1 * h + w5 * d;
  r.yy = w1 * k + w5 * d;
  r.xy = w5 * (p - m);
  return r;
}

// Adjoint of feq(rho, u) from the moments of the adjoints of its nine values.
__device__ __forceinline__ void feq_adjoint(const Moments& m, double rho, double ux, double uy,
                                            double& rb, double& ubx, double& uby) {
#pragma clang fp contract(on)
  const double qx = ux * m.xx + uy * m.xy, qy = ux * m.xy + uy * m.yy;
  rb = m.s * (1.0 - 1.5 * (ux * ux + uy * uy)) + 3.0 * (ux * m.x + uy * m.y) +
       4.5 * (ux * qx + uy * qy);
  ubx = rho * (3.0 * (m.x - ux * m.s) + 9.0 * qx);
  uby = rho * (3.0 * (m.y - uy * m.s) + 9.0 * qy);
}

// 1 / v for a density or 1 + alpha / 2, to within a unit in the last place: the
// hardware's estimate and two Newton steps, half the instructions of a division,
// which rounds correctly and scales operands near the ends of the range.
__device__ __forceinline__ double reciprocal(double v) {
  double r = __builtin_amdgcn_rcp(v);
  r = fma(r, fma(-v, r, 1.0), r);
  return fma(r, fma(-v, r, 1.0), r);
}
__device__ __forceinline__ double drag_scale(double al) { return reciprocal(fma(0.5, al, 1.0)); }

// Reverse of one cell's step.  v: adjoints of the populations it emitted;
// rb, ubx, uby: adjoints of its density and velocity as published (0 where none);
// al: its solid fraction, sa = drag_scale(al); t0, t1, t2: its trace.  gb:
// adjoints of the populations it received; ab: of its solid fraction.  For an inlet or outlet cell (io) gb is zero and rb, ubx,
// uby become the adjoints of the density and velocity it read.  `in_window`:
// the objective takes the discharge here at this step.  Contractions are the
// source's, not the optimiser's: the single step and the passes agree bit for bit.
template <class T>
__device__ __forceinline__ void adjoint_cell(const Params& p, bool io, double al, double sa,
                                             double t0, double t1, double t2, bool in_window,
                                             double qbar, const double* v, double* gb, double& rb,
                                             double& ubx, double& uby, double& ab) {
#pragma clang fp contract(on)
  const double Fx = p.use_force ? p.fx : 0.0f, Fy = p.use_force ? p.fy : 0.0f;
  const Moments m = moments<T>(v);
  double r, x, y;
  const double rho = t0, inv = reciprocal(rho);
  if (io) {
    // populations = feq(rho, u_read + F/(2 rho)): no dependence on the loaded ones
    const double ux = t1 + 0.5 * inv * Fx, uy = t2 + 0.5 * inv * Fy;
    feq_adjoint(m, rho, ux, uy, r, x, y);
    ubx += x;
    uby += y;
    rb += r - (ubx * Fx + uby * Fy) * 0.5 * inv * inv;
#pragma unroll
    for (int i = 0; i < 9; i++) gb[i] = 0.0;
    ab = 0.0;
    return;
  }
  const double si = sa * inv;
  const double ux = (t1 + 0.5 * Fx) * si, uy = (t2 + 0.5 * Fy) * si;
  // The forward's SRT weights are float constants (also in FP64).
  const double om = p.inv_tau, omc = 1.0f - p.inv_tau, tl = 1.0f - 0.5f * p.inv_tau;
  feq_adjoint(m, rho, ux, uy, r, x, y);
  rb += om * r;
  ubx += om * x;
  uby += om * y;
  ab = 0.0;
  if (p.use_force || p.alpha) {
    const double k3 = double(0.33333334f), f = 9.0 * tl;
    const double Gx = Fx - al * rho * ux, Gy = Fy - al * rho * uy;
    ubx += f * (Gx * m.xx + Gy * m.xy - k3 * Gx * m.s);
    uby += f * (Gx * m.xy + Gy * m.yy - k3 * Gy * m.s);
    const double Gbx = f * (ux * m.xx + uy * m.xy + k3 * (m.x - ux * m.s));
    const double Gby = f * (ux * m.xy + uy * m.yy + k3 * (m.y - uy * m.s));
    const double uG = ux * Gbx + uy * Gby;
    ubx += -al * rho * Gbx;
    uby += -al * rho * Gby;
    rb += -al * uG;
    ab = -rho * uG;
  }
  if (in_window) {  // J += qbar * rho * u_x
    rb += qbar * ux;
    ubx += qbar * rho;
  }
  const double mbx = ubx * si, mby = uby * si, ubu = ubx * ux + uby * uy;
  rb += -ubu * inv;
  ab += -0.5 * sa * ubu;
#pragma unroll
  for (int i = 0; i < 9; i++) gb[i] = omc * v[i] + (rb + along(i, mbx, mby));
}

__device__ __forceinline__ uint32_t cell_neighbour(const Params& p, uint32_t x, uint32_t y, int i) {
  const uint32_t nx = p.nx, ny = p.ny;
  uint32_t xx = x, yy = y;
  if (cx(i) == 1) xx = x + 1 == nx ? 0 : x + 1;
  if (cx(i) == -1) xx = x == 0 ? nx - 1 : x - 1;
  if (cy(i) == 1) yy = y + 1 == ny ? 0 : y + 1;
  if (cy(i) == -1) yy = y == 0 ? ny - 1 : y - 1;
  return xx + yy * p.pitch;
}

// Slot (plane, cell) where the forward step of parity ODD stores population i.
template <int ODD>
__device__ __forceinline__ uint64_t store_index(const Params& p, uint32_t n, const uint32_t* nb,
                                                int i) {
  if (i == 0) return n;
  if (i & 1) return (ODD ? i + 1 : i) * p.Np + nb[i];
  return (ODD ? i - 1 : i) * p.Np + n;
}
// Slot where it loads population i.
template <int ODD>
__device__ __forceinline__ uint64_t load_index(const Params& p, uint32_t n, const uint32_t* nb,
                                               int i) {
  if (i == 0) return n;
  if (i & 1) return (ODD ? i : i + 1) * p.Np + n;
  return (ODD ? i : i - 1) * p.Np + nb[i - 1];
}

__device__ __forceinline__ void block_add(double v, double* target) {
  __shared__ double lds[16];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) lds[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int k = 0; k < int(blockDim.x >> 6); k++) s += lds[k];
    if (s != 0.0) atomicAdd(target, s);
  }
}

template <class T, int ODD>
__global__ void __launch_bounds__(256) k_adjoint_step(const Params p, const AdjParams a) {
  uint32_t tx, y;
  block_tile(blockIdx.x, p.tiles_x, p.ny, p.band_magic, p.last_magic, tx, y);
  const uint32_t x = tx * blockDim.x + threadIdx.x;
  double duin = 0.0;
  if (x < p.nx) {
    const uint32_t n = x + y * p.pitch;
    const uint64_t N = p.N;
    const uint8_t fl = p.flags[n];
    if (!(fl & (kGas | kWall))) {
      uint32_t nb[9];
      nb[0] = n;
#pragma unroll
      for (int i = 1; i < 9; i++) nb[i] = cell_neighbour(p, x, y, i);
      double v[9];
#pragma unroll
      for (int i = 0; i < 9; i++) v[i] = a.abar[store_index<ODD>(p, n, nb, i)];
      const Linear lin = linear_neighbours(p, x, y, n);
      const uint8_t fl_prev = p.flags[lin.prev];  // unconditional: one round trip
      const uint8_t fl_next = p.flags[lin.next];
      const bool pub_r = lin.has_prev && (fl_prev & kInlet);
      const bool pub_v = lin.has_next && (fl_next & kOutlet) && !(fl & kInlet);
      double rb = 0.0, ubx = 0.0, uby = 0.0;
      if (pub_r) {
        rb = a.rbar[ODD][n];
        a.rbar[ODD][n] = 0.0;
      }
      if (pub_v) {
        ubx = a.ubar[ODD][n];
        uby = a.ubar[ODD][N + n];
        a.ubar[ODD][n] = 0.0;
        a.ubar[ODD][N + n] = 0.0;
      }
      const T* const tr = static_cast<const T*>(a.trace);
      const uint8_t io = fl & (kInlet | kOutlet);
      double gb[9], ab;
      const double al = p.alpha ? p.alpha[n] : 0.0f;
      adjoint_cell<T>(p, io != 0, al, drag_scale(al), tr[n], tr[N + n], tr[2 * N + n],
                      a.in_window && x == a.column, a.qbar, v, gb, rb, ubx, uby, ab);
      if (io & kInlet) {
        a.rbar[ODD ^ 1][lin.next] += rb;
        duin = ubx;
      } else if (io) {
        a.ubar[ODD ^ 1][lin.prev] += ubx;
        a.ubar[ODD ^ 1][N + lin.prev] += uby;
      } else if (a.galpha) {
        a.galpha[n] += ab;
      }
#pragma unroll
      for (int i = 0; i < 9; i++) a.abar[load_index<ODD>(p, n, nb, i)] = gb[i];
    }
  }
  block_add(duin, a.duin);
}

// Reverse of K steps, from the one at time t down to t - K + 1, in one pass over
// the adjoint state: the forward pass (march_rows) mirrored.  A wavefront owns
// 64 - 2 (K - 1) columns of a strip and marches up its chunk of rows; the reverse
// of step t - s takes the row below that of step t - s + 1.  Since a population i
// that cell n emits is received at n + c_i, the adjoint cell n needs is the one
// of the cell it sent to: those above come from the row just done, those
// beside from one iteration ago, those below from two.  A wall, which emits what
// it received in the opposite direction, exchanges the adjoints.  A single step
// moves 196 bytes per cell, 144 of them the adjoint populations, which a pass of
// three moves once; 1024 x 256, FP32: 9.8 us per step one by one, 6.0 in passes
// (140 FP64 instructions of about 200 per step-row, halo rows included: the
// vector units bind, except on grids beyond the caches).
struct AdjMarch {
  const double* in;   // adjoint populations after step t
  double* out;        // before step t - K + 1
  // Adjoints of the densities and velocities published at step t, and those
  // at step t - K.  Cells no inlet or outlet reads hold zero.
  const double* rb_in;
  const double* ub_in;
  double* rb_out;
  double* ub_out;
  double* galpha;
  double* duin;
  const void* trace;  // of step t; that of step t - s is 3 s N values before it
  int32_t odd;        // t % 2
  uint32_t column, window;  // bit s of window: step t - s is averaged
  double qbar;
  MarchGrid grid;
};

template <class T, int K, bool IO>
__device__ __forceinline__ void adjoint_rows(const Params& p, const AdjMarch& a, uint32_t strip,
                                             uint32_t ya, uint32_t yb) {
  constexpr int H = K - 1;  // halo
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t nx = p.nx, ny = p.ny, pitch = p.pitch;
  const uint32_t xs = strip * march_columns(K) + lane;  // column + H
  const bool own = lane >= H && lane < 64 - H && xs - H < nx;
  const uint32_t x = (xs + H * (nx - 1)) % nx;
  const uint32_t xr = x + 1 == nx ? 0u : x + 1;
  const bool odd = a.odd != 0, odd_last = odd != ((K & 1) == 0);
  const uint64_t Np = p.Np;
  auto up = [&](uint32_t y) { return y + 1 == ny ? 0u : y + 1; };
  auto down = [&](uint32_t y) { return y == 0 ? ny - 1 : y - 1; };

  double raw[9], raw_ga = 0.0, raw_rb = 0.0, raw_ub = 0.0, raw_vb = 0.0;
  T raw_tr[K][3];
  uint8_t raw_fl;
  float raw_al = 0.0f;
  auto load_row = [&](uint32_t y) {
    const uint64_t rc = uint64_t(y) * pitch, ru = uint64_t(up(y)) * pitch,
                   rd = uint64_t(down(y)) * pitch;
    auto here = [&](int i) { return a.in + (odd ? i : i + 1) * Np; };
    auto there = [&](int i) { return a.in + (odd ? i + 1 : i) * Np; };
    raw[0] = at(a.in + rc, x);
    raw[1] = at(there(1) + rc, xr);
    raw[2] = at(here(1) + rc, x);
    raw[3] = at(there(3) + ru, x);
    raw[4] = at(here(3) + rc, x);
    raw[5] = at(there(5) + ru, xr);
    raw[6] = at(here(5) + rc, x);
    raw[7] = at(there(7) + rd, xr);
    raw[8] = at(here(7) + rc, x);
    raw_fl = at(p.flags + rc, x);
    if (p.alpha) raw_al = at(p.alpha + rc, x);
    if (a.galpha) raw_ga = at(a.galpha + rc, x);
    if (IO) {
      raw_rb = at(a.rb_in + rc, x);
      raw_ub = at(a.ub_in + rc, x);
      raw_vb = at(a.ub_in + p.N + rc, x);
    }
    uint32_t ys = y;  // each step's row of the next iteration
#pragma unroll
    for (int s = 0; s < K; s++) {
      const T* const tr = static_cast<const T*>(a.trace) - uint64_t(s) * 3u * p.N +
                          uint64_t(ys) * pitch;
#pragma unroll
      for (int k = 0; k < 3; k++) raw_tr[s][k] = at(tr + k * p.N, x);
      ys = down(ys);
    }
  };
  auto store_row = [&](uint32_t y, const double* g) {
    const uint64_t rc = uint64_t(y) * pitch, ru = uint64_t(up(y)) * pitch,
                   rd = uint64_t(down(y)) * pitch;
    auto here = [&](int i) { return a.out + (odd_last ? i : i + 1) * Np; };
    auto there = [&](int i) { return a.out + (odd_last ? i + 1 : i) * Np; };
    at(a.out + rc, x) = g[0];
    at(here(1) + rc, x) = g[1];
    at(there(1) + rc, xr) = g[2];
    at(here(3) + rc, x) = g[3];
    at(there(3) + ru, x) = g[4];
    at(here(5) + rc, x) = g[5];
    at(there(5) + ru, xr) = g[6];
    at(here(7) + rc, x) = g[7];
    at(there(7) + rd, xr) = g[8];
  };

  // Between two steps (index of the first), already shifted to the lane that
  // takes them: 0, 1, 2 of the row the second takes next; 4, 6, 7 of that row
  // and of the one below it; the published values' adjoints of that row (IO).
  double flat[H][3] = {}, fall0[H][3] = {}, fall1[H][3] = {};
  double pr[H] = {}, pu[H] = {}, pv[H] = {};
  uint32_t fls = 0;
  float al[K] = {};  // solid fractions of the rows under way
  double sa[K] = {};  // drag_scale of them
  double ga[K] = {};  // dJ/dalpha
  double duin = 0.0;

  uint32_t y1 = ya >= uint32_t(H) ? ya - H : ya + ny - H;
  load_row(y1);
  const uint32_t iterations = yb - ya + 2 * H;
  const auto iterate = [&](uint32_t it, auto steady) {
    double g[9];
#pragma unroll
    for (int i = 0; i < 9; i++) g[i] = raw[i];
    fls = fls << 8 | raw_fl;
#pragma unroll
    for (int s = K - 1; s > 0; s--) {
      al[s] = al[s - 1];
      sa[s] = sa[s - 1];
      ga[s] = ga[s - 1];
    }
    al[0] = raw_al;
    sa[0] = drag_scale(raw_al);
    ga[0] = raw_ga;
    double rb = raw_rb, ubx = raw_ub, uby = raw_vb;
    T tr[K][3];
#pragma unroll
    for (int s = 0; s < K; s++)
#pragma unroll
      for (int k = 0; k < 3; k++) tr[s][k] = raw_tr[s][k];
    uint32_t ys = y1;
    y1 = up(y1);
    load_row(y1);  // one row past the last is loaded and not used
#pragma unroll
    for (int s = 0; s < K; s++) {
      if (decltype(steady)::value || it >= 2u * uint32_t(s)) {
        const uint8_t fl = uint8_t(fls >> (8 * s));
        const bool solid = fl & (kGas | kWall);
        const uint8_t io = IO ? fl & (kInlet | kOutlet) : 0;
        if (solid) {
#pragma unroll
          for (int i = 1; i < 9; i += 2) {
            const double t = g[i];
            g[i] = g[i + 1];
            g[i + 1] = t;
          }
        } else {
          if (!IO) rb = ubx = uby = 0.0;
          if (IO && (fl & kInlet)) ubx = uby = 0.0;
          double gb[9], ab;
          adjoint_cell<T>(p, io != 0, al[s], sa[s], tr[s][0], tr[s][1], tr[s][2],
                          (a.window >> s & 1u) && x == a.column, a.qbar, g, gb, rb, ubx, uby, ab);
#pragma unroll
          for (int i = 0; i < 9; i++) g[i] = gb[i];
          if (!io) ga[s] += ab;
        }
        const bool inlet = IO && !solid && (fl & kInlet);
        const bool outlet = IO && !solid && !inlet && (fl & kOutlet);
        // The row is in the chunk (the halo rows are another wavefront's).
        if (inlet && own && it - uint32_t(H + s) < yb - ya) duin += ubx;
        if (s < K - 1) {
          constexpr int last = K > 1 ? H - 1 : 0;
          const int b = s < last ? s : last;
          double v[9];
          v[0] = flat[b][0];
          v[1] = flat[b][1];
          v[2] = flat[b][2];
          v[4] = fall1[b][0];
          v[6] = fall1[b][1];
          v[7] = fall1[b][2];
          v[3] = g[3];
          v[5] = from_right(g[5]);
          v[8] = from_left(g[8]);
          flat[b][0] = g[0];
          flat[b][1] = from_right(g[1]);
          flat[b][2] = from_left(g[2]);
#pragma unroll
          for (int k = 0; k < 3; k++) fall1[b][k] = fall0[b][k];
          fall0[b][0] = g[4];
          fall0[b][1] = from_left(g[6]);
          fall0[b][2] = from_right(g[7]);
          if (IO) {
            const double r = from_left(inlet ? rb : 0.0);
            const double q = from_right(outlet ? ubx : 0.0), w = from_right(outlet ? uby : 0.0);
            rb = pr[b];
            ubx = pu[b];
            uby = pv[b];
            pr[b] = r;
            pu[b] = q;
            pv[b] = w;
          }
#pragma unroll
          for (int i = 0; i < 9; i++) g[i] = v[i];
          ys = down(ys);
        } else if (own) {
          const uint64_t rc = uint64_t(ys) * pitch;
          store_row(ys, g);
          if (a.galpha && !solid && !io) at(a.galpha + rc, x) = ga[s];
          if (inlet) at(a.rb_out + rc, x + 1) = rb;
          if (outlet) {
            at(a.ub_out + rc, x - 1) = ubx;
            at(a.ub_out + p.N + rc, x - 1) = uby;
          }
        }
      }
    }
    if (!IO) __builtin_amdgcn_s_barrier();  // a block's strips keep to the same row
  };
  for (uint32_t it = 0; it < 2 * H; ++it) iterate(it, Fill{});
#pragma unroll 2
  for (uint32_t it = 2 * H; it < iterations; ++it) iterate(it, Steady{});
  if (IO) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) duin += __shfl_down(duin, o, 64);
    if (lane == 0 && duin != 0.0) atomicAdd(a.duin, duin);
  }
}

template <class T, int K>
__global__ void __launch_bounds__(64 * kMarchWaves) __attribute__((amdgpu_waves_per_eu(2)))
k_adjoint_march(const Params p, const AdjMarch a) {
  const MarchWork w = march_work(a.grid, p.ny);
  if (w.ya >= w.yb) return;
  if (w.io) adjoint_rows<T, K, true>(p, a, w.strip, w.ya, w.yb);
  else adjoint_rows<T, K, false>(p, a, w.strip, w.ya, w.yb);
}

// The initial populations of inlet cells, feq(rho0, u0) stored with the odd
// pattern, depend on the inlet velocity.  The set-up evaluates them in double
// with exact weights for every storage format.
__global__ void __launch_bounds__(256) k_adjoint_inlet_init(const Params p, const AdjParams a) {
  uint32_t tx, y;
  block_tile(blockIdx.x, p.tiles_x, p.ny, p.band_magic, p.last_magic, tx, y);
  const uint32_t x = tx * blockDim.x + threadIdx.x;
  double acc = 0.0;
  if (x < p.nx) {
    const uint32_t n = x + y * p.pitch;
    const uint8_t fl = p.flags[n];
    if ((fl & kInlet) && !(fl & (kGas | kWall))) {
      uint32_t nb[9];
      nb[0] = n;
#pragma unroll
      for (int i = 1; i < 9; i++) nb[i] = cell_neighbour(p, x, y, i);
#pragma unroll
      for (int i = 0; i < 9; i++)
        acc += a.abar[store_index<1>(p, n, nb, i)] *
               feq_dx<double>(a.rho_init[n], a.u_init[n], a.u_init[p.N + n], i);
    }
  }
  block_add(acc, a.duin);
}

// Discharge through a column: sum of rho * u_x over its non-wall cells, from the
// readback fields of the last step, accumulated as scale * Q into acc[0].
template <class R>
__global__ void __launch_bounds__(256) k_discharge(const Params p, uint32_t column, double scale,
                                                   double* acc) {
  __shared__ double lds[4];
  double s = 0.0;
  for (uint32_t y = threadIdx.x; y < p.ny; y += blockDim.x) {
    const uint32_t n = column + y * p.pitch;
    if (!(p.flags[n] & (kWall | kGas))) s += double(fld<R>(p.rho)[n]) * double(fld<R>(p.u)[n]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) acc[0] = fma(scale, lds[0] + lds[1] + lds[2] + lds[3], acc[0]);
}

// The same of `steps` steps recorded by passes, ny values each: the sums of
// k_discharge in its order, and the steps in theirs, so that neither the length
// of the passes nor that of the segments changes a bit.
constexpr uint32_t kDischargeSteps = 256;
__global__ void __launch_bounds__(1024) k_discharge_rows(const double* rows, uint32_t steps,
                                                         uint32_t ny, double scale, double* acc) {
  __shared__ double q[kDischargeSteps];
  const uint32_t lane = threadIdx.x & 63u;
  for (uint32_t k = threadIdx.x >> 6; k < steps; k += blockDim.x >> 6) {
    const double* const r = rows + uint64_t(k) * ny;
    double sum[4];
#pragma unroll
    for (uint32_t w = 0; w < 4; w++) {
      double s = 0.0;
      for (uint32_t y = w * 64u + lane; y < ny; y += 256u) s += r[y];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
      sum[w] = s;
    }
    if (lane == 0) q[k] = sum[0] + sum[1] + sum[2] + sum[3];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = acc[0];
    for (uint32_t k = 0; k < steps; k++) s = fma(scale, q[k], s);
    acc[0] = s;
  }
}

}  // namespace flb

namespace {

#define ADJ_HIP(h, call)                                                                   \
  do {                                                                                     \
    hipError_t e_ = (call);                                                                \
    if (e_ != hipSuccess)                                                                  \
      return flb::set_error((h), FLB_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

// Bounds what the handles of a device keep of their buffers after a call, a
// thirty-second of its memory together (9 GB of 288; a gradient of 2000 steps of 1024 x
// 256 takes 6.3 GB in FP32).
struct TrimWork {
  flb_handle* h;
  ~TrimWork() {
    size_t left = 0, total = 0;
    if (hipMemGetInfo(&left, &total) != hipSuccess) {
      (void)hipGetLastError();
      total = 0;
    }
    const size_t most = total / 32, others = flb::idle_elsewhere(h);
    h->work.trim(most > others ? most - others : 0);
  }
};

// Copies the step state (populations and the inlet/outlet publication buffers,
// plus the readback fields when with_fields) between the handle and buf.
// Layout of buf (device planes of Nd cells, bytes): f (9 Np populations) |
// pub_rho[0] | pub_rho[1] (N each) | pub_u[0] | pub_u[1] (2N each) | rho (N) |
// u (2N), the fields in the handle's field type.
size_t state_bytes(const flb_handle* h, bool with_fields) {
  return 9 * h->Np * h->elem_bytes + (6 * h->Nd + (with_fields ? 3 * h->Nd : 0)) * h->field_bytes;
}
int copy_state(flb_handle* h, uint8_t* buf, bool to_handle, bool with_fields) {
  const size_t N = h->Nd * h->field_bytes, o = 9 * h->Np * h->elem_bytes;
  struct Part {
    void* dev;
    size_t off, bytes;
  } parts[7] = {{h->f, 0, o},
                {h->pub_rho[0], o, N},
                {h->pub_rho[1], o + N, N},
                {h->pub_u[0], o + 2 * N, 2 * N},
                {h->pub_u[1], o + 4 * N, 2 * N},
                {h->rho, o + 6 * N, N},
                {h->u, o + 7 * N, 2 * N}};
  const int count = with_fields ? 7 : 5;
  for (int k = 0; k < count; ++k) {
    void* a = to_handle ? parts[k].dev : static_cast<void*>(buf + parts[k].off);
    const void* b = to_handle ? static_cast<const void*>(buf + parts[k].off) : parts[k].dev;
    ADJ_HIP(h, hipMemcpyAsync(a, b, parts[k].bytes, hipMemcpyDeviceToDevice, h->stream));
  }
  return FLB_OK;
}

int check_adjoint_state(flb_handle* h, const flb_adjoint_spec* sp) {
  if (!h || !sp) return FLB_ERR_ARGUMENT;
  if (h->opt.problem != FLB_MONOFLUID || h->opt.collision != FLB_SRT || h->opt.smagorinsky ||
      (h->opt.storage != FLB_STORAGE_FP32 && h->opt.storage != FLB_STORAGE_FP64))
    return flb::set_error(h, FLB_ERR_UNSUPPORTED,
                          "adjoint needs a monofluid SRT handle with FP32 or FP64 storage and no "
                          "subgrid model");
  if (h->t != 0) return flb::set_error(h, FLB_ERR_STATE, "adjoint runs from the initial state (t = 0)");
  if (sp->nsteps == 0 || sp->t1 < sp->t0 || sp->t1 >= sp->nsteps || sp->column >= h->nx ||
      sp->ckpt == 0)
    return flb::set_error(h, FLB_ERR_ARGUMENT, "invalid adjoint window");
  return FLB_OK;
}

using flb::kDischargeSteps;

using AdjMarchFn = void (*)(const flb::Params, const flb::AdjMarch);
AdjMarchFn adjoint_march(bool fp64, int steps) {
  if (fp64) return steps == 2 ? flb::k_adjoint_march<double, 2> : flb::k_adjoint_march<double, 3>;
  return steps == 2 ? flb::k_adjoint_march<float, 2> : flb::k_adjoint_march<float, 3>;
}

// Forward steps [t, t+count) with the objective accumulated into d_j; with a
// trace buffer, step t + k records its trace at trace + k * 3 N values.  In
// passes of several steps where the handle has them: the averaged steps record
// the column's discharge, summed every kDischargeSteps steps and at the end,
// which takes the place of a reduction of one block after each step.  600 steps of
// 1024 x 256 in FP32 with the trace: 4.31 ms step by step, 3.29 ms (the trace's
// 1.9 GB take 0.4 ms at the rate of a copy; the rest is the passes' arithmetic
// on a domain of one wavefront per SIMD).
int run_forward(flb_handle* h, uint64_t count, const flb_adjoint_spec* sp, double qscale,
                double* d_j, uint8_t* trace = nullptr) {
  const bool fp64 = h->opt.storage == FLB_STORAGE_FP64;
  const int bx = flb::handle_block_x(h);
  const int most = flb::march_most(h);
  double* q = nullptr;
  if (most && d_j) {
    q = h->work.get<double>(flb::Workspace::kColumn, uint64_t(kDischargeSteps) * h->ny);
    if (!q) return flb::set_error(h, FLB_ERR_MEMORY, "discharge of the averaged steps");
  }
  uint64_t held = 0;  // steps in q
  auto flush = [&]() -> int {
    if (held)
      hipLaunchKernelGGL(flb::k_discharge_rows, dim3(1), dim3(1024), 0, h->stream, q,
                         uint32_t(held), h->ny, qscale, d_j);
    held = 0;
    ADJ_HIP(h, hipGetLastError());
    return FLB_OK;
  };
  int rc = FLB_OK;
  for (uint64_t k = 0; k < count && !rc;) {
    const uint64_t t = h->t;
    uint8_t* const to = trace ? trace + k * 3 * h->Nd * h->field_bytes : nullptr;
    const bool win = d_j && t >= sp->t0 && t <= sp->t1;
    // A pass lies in the averaged steps as a whole or not at all.
    uint64_t left = count - k;
    if (d_j && t < sp->t0) left = std::min(left, sp->t0 - t);
    if (win) left = std::min(left, sp->t1 + 1 - t);
    const int T = most ? flb::march_steps_next(left, most) : 0;
    if (T && (trace || win)) {
      if (win && held + uint64_t(T) > kDischargeSteps && (rc = flush())) break;
      flb::MarchTrace m{};
      m.trace = to;
      m.discharge = win ? q + held * h->ny : nullptr;
      m.column = sp->column;
      m.window = win ? (1u << T) - 1u : 0u;
      if (win) held += uint64_t(T);
      rc = flb::enqueue_march_ex(h, T, false, &m);
      k += uint64_t(T);
      continue;
    }
    if (T) {
      rc = flb::enqueue_march_ex(h, T, false, nullptr);
      k += uint64_t(T);
      continue;
    }
    flb::Params p = flb::make_params(h, bx);
    p.trace = reinterpret_cast<float*>(to);
    hipLaunchKernelGGL(trace ? flb::get_stream_collide_trace(h->opt.storage, int(t & 1), win)
                             : flb::get_stream_collide(h->opt.storage, int(t & 1), false, win),
                       dim3(p.nblocks), dim3(bx), 0, h->stream, p);
    ADJ_HIP(h, hipGetLastError());
    if (win) {
      if ((rc = flush())) break;
      hipLaunchKernelGGL(fp64 ? flb::k_discharge<double> : flb::k_discharge<float>, dim3(1),
                         dim3(256), 0, h->stream, p, sp->column, qscale, d_j);
      ADJ_HIP(h, hipGetLastError());
    }
    h->t += 1;
    ++k;
  }
  return rc ? rc : flush();
}

}  // namespace

extern "C" {

int flb_set_brinkman(flb_handle* h, const float* alpha) {
  if (!h) return FLB_ERR_ARGUMENT;
  if (!alpha) {
    h->alpha = nullptr;  // buffer stays owned by the handle
    return FLB_OK;
  }
  if (h->opt.problem != FLB_MONOFLUID)
    return flb::set_error(h, FLB_ERR_UNSUPPORTED, "Brinkman drag needs a monofluid handle");
  if (!h->alpha) {
    void* v = nullptr;
    ADJ_HIP(h, flb::device_malloc(&v, h->Nd * sizeof(float), h->device, nullptr));
    h->owned.push_back(v);
    h->alpha = static_cast<float*>(v);
    ADJ_HIP(h, hipMemsetAsync(v, 0, h->Nd * sizeof(float), h->stream));
  }
  return flb::copy_cells_in(h, h->alpha, alpha, sizeof(float), 1);
}

int flb_objective(flb_handle* h, const flb_adjoint_spec* sp, double* J) {
  int rc = check_adjoint_state(h, sp);
  if (rc) return rc;
  const std::lock_guard<std::recursive_mutex> lock(h->in_use);
  using W = flb::Workspace;
  TrimWork trim{h};
  uint8_t* saved = nullptr;
  double* d_j = nullptr;
  auto buffers = [&]() {
    return (saved = h->work.get<uint8_t>(W::kState, state_bytes(h, true))) &&
           (d_j = h->work.get<double>(W::kSums, 2));
  };
  if (!buffers()) {
    h->work.trim(0);  // buffers of an earlier call may be what is in the way
    if (!buffers()) return flb::set_error(h, FLB_ERR_MEMORY, "objective buffers");
  }
  if ((rc = copy_state(h, saved, false, true))) return rc;
  ADJ_HIP(h, hipMemsetAsync(d_j, 0, sizeof(double), h->stream));
  rc = run_forward(h, sp->nsteps, sp, 1.0 / double(sp->t1 - sp->t0 + 1), d_j);
  const int rc2 = copy_state(h, saved, true, true);
  h->t = 0;
  if (rc) return rc;
  if (rc2) return rc2;
  double j = 0.0;
  ADJ_HIP(h, hipMemcpyAsync(&j, d_j, sizeof(double), hipMemcpyDeviceToHost, h->stream));
  ADJ_HIP(h, hipStreamSynchronize(h->stream));
  if (J) *J = j;
  return FLB_OK;
}

int flb_adjoint(flb_handle* h, const flb_adjoint_spec* sp, double* J, float* dj_dalpha,
                double* dj_duin, float* phase_ms) {
  int rc = check_adjoint_state(h, sp);
  if (rc) return rc;
  const std::lock_guard<std::recursive_mutex> lock(h->in_use);
  const size_t N = h->Nd, Np = h->Np;  // device planes
  const uint64_t K = sp->ckpt, T = sp->nsteps;
  const uint64_t nseg = (T + K - 1) / K;
  const size_t ck_bytes = state_bytes(h, false);
  const size_t seg_bytes = size_t(std::min<uint64_t>(K, T)) * 3 * N * h->field_bytes;
  const bool fp64 = h->opt.storage == FLB_STORAGE_FP64;
  // Segments whose trace stays resident from the forward sweep: the last
  // `resident` ones, as many as the budget holds.
  size_t budget = sp->trace_budget_bytes;
  if (budget == 0) {
    size_t free_b = 0, total_b = 0;
    ADJ_HIP(h, hipMemGetInfo(&free_b, &total_b));
    // What handles keep between calls counts as free.
    budget = (free_b + h->work.held() + flb::idle_elsewhere(h)) / 2;
  } else if (h->work.size[flb::Workspace::kTrace] > budget) {
    h->work.drop(flb::Workspace::kTrace);  // an earlier call's, larger than this one allows
  }
  const uint64_t resident = std::min<uint64_t>(nseg, budget / seg_bytes);
  const uint64_t first_res = nseg - resident;  // segments [0, first_res) are recomputed
  using W = flb::Workspace;
  TrimWork trim{h};
  uint8_t *ckpt = nullptr, *fields0 = nullptr, *trace_res = nullptr, *trace_tmp = nullptr;
  double *abar = nullptr, *abar_alt = nullptr, *rbar = nullptr, *ubar = nullptr, *galpha = nullptr, *d_acc = nullptr;
  auto buffers = [&]() {
    flb::Workspace& w = h->work;
    return (!first_res || ((ckpt = w.get<uint8_t>(W::kCheckpoints, first_res * ck_bytes)) &&
                           (trace_tmp = w.get<uint8_t>(W::kTraceOnce, seg_bytes)))) &&
           (!resident || (trace_res = w.get<uint8_t>(W::kTrace, resident * seg_bytes))) &&
           (fields0 = w.get<uint8_t>(W::kState, state_bytes(h, true))) &&
           (abar = w.get<double>(W::kAdjoint, 9 * Np)) &&
           (rbar = w.get<double>(W::kDensity, 2 * N)) &&
           (ubar = w.get<double>(W::kVelocity, 4 * N)) &&
           (!h->alpha || (galpha = w.get<double>(W::kAlpha, N))) &&
           (d_acc = w.get<double>(W::kSums, 2));  // J, dJ/du_in
  };
  if (!buffers()) {
    h->work.trim(0);  // buffers of an earlier call may be what is in the way
    if (!buffers())
      return flb::set_error(h, FLB_ERR_MEMORY, "adjoint buffers (checkpoints, trace, adjoint state)");
  }
  // Passes need a second adjoint state; without room for it, single steps.
  flb::MarchShape shape = flb::adjoint_shape(h);
  if (std::min(K, T) < 2 || !h->f_alt) shape.steps = 0;
  if (shape.steps && !(abar_alt = h->work.get<double>(W::kAdjointAlt, 9 * Np))) shape.steps = 0;
  auto seg_trace = [&](uint64_t s) {
    return s >= first_res ? trace_res + (s - first_res) * seg_bytes : trace_tmp;
  };

  if ((rc = copy_state(h, fields0, false, true))) return rc;
  ADJ_HIP(h, hipMemsetAsync(d_acc, 0, 2 * sizeof(double), h->stream));
  hipEvent_t ev[4];
  for (auto& e : ev) ADJ_HIP(h, hipEventCreate(&e));
  ADJ_HIP(h, hipEventRecord(ev[0], h->stream));

  // Forward sweep: the objective, checkpoints of the segments to recompute,
  // the trace of the resident ones.
  const double qs = 1.0 / double(sp->t1 - sp->t0 + 1);
  for (uint64_t s = 0; s < nseg && !rc; ++s) {
    const uint64_t count = std::min(K, T - s * K);
    if (s < first_res) {
      if ((rc = copy_state(h, ckpt + s * ck_bytes, false, false))) break;
      rc = run_forward(h, count, sp, qs, d_acc);
    } else {
      rc = run_forward(h, count, sp, qs, d_acc, seg_trace(s));
    }
  }
  ADJ_HIP(h, hipEventRecord(ev[1], h->stream));

  // Reverse sweep, one checkpoint segment at a time.
  ADJ_HIP(h, hipMemsetAsync(abar, 0, 9 * Np * sizeof(double), h->stream));
  ADJ_HIP(h, hipMemsetAsync(rbar, 0, 2 * N * sizeof(double), h->stream));
  ADJ_HIP(h, hipMemsetAsync(ubar, 0, 4 * N * sizeof(double), h->stream));
  if (galpha) ADJ_HIP(h, hipMemsetAsync(galpha, 0, N * sizeof(double), h->stream));
  const int abx = 256;
  float recompute_ms = 0.0f;
  double *rb[2] = {rbar, rbar + N}, *ub[2] = {ubar, ubar + 2 * N};  // by parity
  bool stale = false;  // the other parity's hold values a pass has used
  for (uint64_t s = nseg; s-- > 0 && !rc;) {
    const uint64_t ts = s * K, te = std::min(ts + K, T);
    uint8_t* trace = seg_trace(s);
    if (s < first_res) {
      if ((rc = copy_state(h, ckpt + s * ck_bytes, true, false))) break;
      h->t = ts;
      ADJ_HIP(h, hipEventRecord(ev[2], h->stream));
      if ((rc = run_forward(h, te - ts, sp, qs, nullptr, trace))) break;
      ADJ_HIP(h, hipEventRecord(ev[3], h->stream));
    }
    for (uint64_t t = te; t-- > ts;) {
      const uint8_t* const tr = trace + (t - ts) * 3 * N * h->field_bytes;
      flb::Params p = flb::make_params(h, abx);
      const int steps = shape.steps ? flb::march_steps_next(t + 1 - ts, shape.steps) : 0;
      if (steps) {
        const int par = int(t & 1), to = par ^ (steps & 1);
        // Published values' adjoints go to the parity of the step below the pass;
        // an even pass would write what it reads, so the buffers change places.
        if (!(steps & 1)) {
          std::swap(rb[0], rb[1]);
          std::swap(ub[0], ub[1]);
        }
        flb::AdjMarch a{};
        a.in = abar;
        a.out = abar_alt;
        a.rb_in = rb[steps & 1 ? par : par ^ 1];
        a.ub_in = ub[steps & 1 ? par : par ^ 1];
        a.rb_out = rb[to];
        a.ub_out = ub[to];
        a.galpha = galpha;
        a.duin = d_acc + 1;
        a.trace = tr;
        a.odd = par;
        a.column = sp->column;
        for (int k = 0; k < steps; ++k)
          if (t - k >= sp->t0 && t - k <= sp->t1) a.window |= 1u << k;
        a.qbar = qs;
        a.grid = flb::march_grid(h, steps, shape.rows, (shape.rows + 1) / 2);
        hipLaunchKernelGGL(adjoint_march(fp64, steps), dim3(a.grid.blocks),
                           dim3(64 * flb::kMarchWaves), 0, h->stream, p, a);
        ADJ_HIP(h, hipGetLastError());
        std::swap(abar, abar_alt);
        stale = true;
        t -= uint64_t(steps - 1);
        continue;
      }
      if (stale) {  // a single step adds to what it publishes for the step below
        const int to = int(t & 1) ^ 1;
        ADJ_HIP(h, hipMemsetAsync(rb[to], 0, N * sizeof(double), h->stream));
        ADJ_HIP(h, hipMemsetAsync(ub[to], 0, 2 * N * sizeof(double), h->stream));
        stale = false;
      }
      flb::AdjParams a{};
      a.abar = abar;
      for (int k = 0; k < 2; ++k) {
        a.rbar[k] = rb[k];
        a.ubar[k] = ub[k];
      }
      a.galpha = galpha;
      a.trace = tr;
      a.duin = d_acc + 1;
      a.column = sp->column;
      a.in_window = t >= sp->t0 && t <= sp->t1;
      a.qbar = qs;
      const auto kernel = fp64 ? ((t & 1) ? flb::k_adjoint_step<double, 1> : flb::k_adjoint_step<double, 0>)
                               : ((t & 1) ? flb::k_adjoint_step<float, 1> : flb::k_adjoint_step<float, 0>);
      hipLaunchKernelGGL(kernel, dim3(p.nblocks), dim3(abx), 0, h->stream, p, a);
      ADJ_HIP(h, hipGetLastError());
    }
    if (s < first_res) {
      ADJ_HIP(h, hipEventSynchronize(ev[3]));
      float ms = 0.0f;
      ADJ_HIP(h, hipEventElapsedTime(&ms, ev[2], ev[3]));
      recompute_ms += ms;
    }
  }
  if (!rc) {
    flb::Params p = flb::make_params(h, abx);
    flb::AdjParams a{};
    a.abar = abar;
    a.rho_init = h->rho_init;
    a.u_init = h->u_init;
    a.duin = d_acc + 1;
    hipLaunchKernelGGL(flb::k_adjoint_inlet_init, dim3(p.nblocks), dim3(abx), 0, h->stream, p, a);
    ADJ_HIP(h, hipGetLastError());
  }
  // Leave the handle in its initial state.
  hipEvent_t end;
  ADJ_HIP(h, hipEventCreate(&end));
  const int rc_restore = copy_state(h, fields0, true, true);
  if (!rc) rc = rc_restore;
  ADJ_HIP(h, hipEventRecord(end, h->stream));
  h->t = 0;
  double acc[2] = {0.0, 0.0};
  ADJ_HIP(h, hipMemcpyAsync(acc, d_acc, 2 * sizeof(double), hipMemcpyDeviceToHost, h->stream));
  ADJ_HIP(h, hipStreamSynchronize(h->stream));
  if (dj_dalpha && galpha && !rc) {
    std::vector<double> g(h->N);
    rc = flb::copy_cells_out(h, g.data(), galpha, sizeof(double), 1);
    for (size_t n = 0; n < h->N && !rc; ++n) dj_dalpha[n] = float(g[n]);
  }
  if (phase_ms) {
    float fwd = 0.0f, tot = 0.0f;
    ADJ_HIP(h, hipEventElapsedTime(&fwd, ev[0], ev[1]));
    ADJ_HIP(h, hipEventElapsedTime(&tot, ev[0], end));
    phase_ms[0] = fwd;                   // forward sweep (checkpoints or trace)
    phase_ms[1] = recompute_ms;          // forward recompute of non-resident segments
    phase_ms[2] = tot - fwd - recompute_ms;  // reverse sweep and restore
  }
  for (auto& e : ev) (void)hipEventDestroy(e);
  (void)hipEventDestroy(end);
  if (rc) return rc;
  if (dj_dalpha && !galpha)
    for (size_t n = 0; n < h->N; ++n) dj_dalpha[n] = 0.0f;
  if (J) *J = acc[0];
  if (dj_duin) *dj_duin = acc[1];
  return FLB_OK;
}

}  // extern "C"
