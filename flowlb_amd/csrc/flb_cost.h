// flb_cost.h -- whether a pass of several steps (flb_march.h) takes less time than
// single steps (host code; no device or HIP types).
//
// A pass moves a third of the bytes of its steps but is bound by the vector units
// or by the chain of rows of one wavefront, and pays for halo rows and columns; a
// single step is bound by the launch on small domains, by the L2 or the Infinity
// Cache on middling ones and by memory on large ones.  Plain SRT gains from 1.2 to
// 2.9 times nearly everywhere.  It is the other way round where a cell costs many
// instructions or the values are small (2048 x 512, us per step, single / passes: FP16S
// TRT with the subgrid model 11.8 / 14.1, with TRT-Guo forcing too 13.1 / 17.2, drag
// 11.7 / 13.5; FP32 TRT-Guo with the subgrid model 14.1 / 16.5) and in part where most
// strips hold inlet or outlet cells, a row of which takes up to 1.9 times the others
// (an outlet along the top, FP32: 2048 x 512 12.0 / 14.7, 4096 x 1024 37.7 / 43.4, but
// 8192 x 2048 199 / 158).
//
// Two times count, which can differ either way: of a run by itself, and per run of
// several handles' runs side by side, which fill each other's idle wavefronts and
// push each other's populations out of the caches (5001 x 1001 BF16S TRT with the subgrid
// model: 41 / 37 alone, 40 / 31 side by side).  Both are estimated, and what is faster
// by the geometric mean of the two ratios is taken.
//
// The constants are fits to 7000 timed domains and 2000 batches (64 to 8192 columns, 16
// to 8192 rows, 12 models, four storages; inlet and outlet columns, an outlet along
// the top, periodic).  The estimates are off by 5 to 9 % (single steps), 9 % (passes
// alone) and 12 % (side by side).  Of 1810 domains, always taking passes was slower than
// single steps by more than a tenth in 334 alone and in 235 side by side; the rule is in
// 101 and 21, and slower than passes by as much in 16 and 20.
#pragma once

#include <algorithm>
#include <cstdint>

namespace flb {

// What a step computes in each cell.
struct StepModel {
  int storage;  // FLB_STORAGE_*
  bool force, drag, trt, guo /* TRT with forcing terms */, smagorinsky;
  int kernel;   // the compiled model (kMarchPlain ...)
};

// Rows of a pass, each counted once for every step.
struct PassRows {
  double chain = 0, io_chain = 0;  // of one wavefront, of an interior and an inlet/outlet strip
  double all = 0, io_all = 0;      // of all wavefronts
  // Adds a domain of ny rows: its strips, and the rows a wavefront has of each.  A
  // batch shares out an inlet/outlet strip chunk by chunk (chunked).
  void add(uint32_t interior, uint32_t io, uint32_t ny, int steps, uint32_t rows, uint32_t io_rows,
           bool chunked = false) {
    const double halo = steps - 1, r = steps * (rows + halo), q = steps * (io_rows + halo);
    if (interior) chain = std::max(chain, r);
    if (io) io_chain = std::max(io_chain, q);
    const uint32_t chunks = (ny + rows - 1) / rows;
    all += r * interior * chunks;
    io_all += q * io * (chunked ? chunks * ((rows + io_rows - 1) / io_rows) : (ny + io_rows - 1) / io_rows);
  }
};

// us a wavefront takes for such a row, alone on its SIMD: the sum of what the model
// has; of an inlet/outlet strip, io[kernel] times that.
struct RowCost {
  double plain, force, trt, smagorinsky, drag, guo;
  double mixed;          // the subgrid model in the kernel that takes every option
  double io[5];
  double shared, among;  // of it, where a SIMD has several wavefronts; of several handles
                         // (FP64 wavefronts get in each other's way)
  double start;          // us a pass takes before and after its rows
};
inline const RowCost& row_cost(int storage) {
  static const RowCost fp32{.24, .04, .06, .13, .10, .11, .05, {1.55, 1.9, 1.2, 1.2, 1.25}, .88, .70, 6.7};
  static const RowCost fp16{.285, .055, .04, .12, .165, .10, .03, {1.2, 1.4, 1.2, 1.15, 1.2}, .90, .67, 6.0};
  static const RowCost bf16{.285, .055, .04, .12, .165, .10, .03, {1.2, 2.0, 1.2, 1.15, 1.2}, .90, .67, 6.0};
  static const RowCost fp64{.28, .055, .085, .125, .115, .11, .045, {1.2, 1.2, 1.15, 1.3, 1.2}, 1.42, 1.2, 7.5};
  return storage == 0 ? fp32 : (storage == 1 ? fp16 : (storage == 2 ? bf16 : fp64));
}

// us per step: of a run alone, and side by side with others.
struct StepTime {
  double alone, among;
};
inline bool faster(const StepTime& a, const StepTime& b) {
  return a.alone * a.among < b.alone * b.among;
}

// A pass of `steps` over populations of `mb` megabytes.
inline StepTime pass_time(const StepModel& m, int steps, const PassRows& r, double mb, int cus) {
  constexpr int kGeneral = 3;  // kMarchGeneral
  const RowCost& c = row_cost(m.storage);
  const double row = c.plain + m.force * c.force + m.trt * c.trt + m.smagorinsky * c.smagorinsky +
                     m.drag * c.drag + m.guo * c.guo + (m.kernel == kGeneral && m.smagorinsky) * c.mixed;
  const double io = row * c.io[m.kernel];
  const double chain = std::max(r.chain * row, r.io_chain * io);
  const double simd = (r.all * row + r.io_all * io) / (4.0 * cus), busy = c.shared * simd;
  // The larger of the two, and a part of the other.
  const double rows = c.start + std::max(chain, busy) + 0.35 * std::min(chain, busy);
  // Both population arrays once, from memory where they do not fit the Infinity
  // Cache (256 MB), alone or with two other handles'.
  const double bytes = mb * (2 * mb > 256 ? .5 : .3), others = mb * (6 * mb > 256 ? .5 : .3);
  // A short pass (what a call's end leaves) writes the fields for few steps.
  const double per = (steps == 2 ? 1.08 : 1.0) / steps;
  return {std::max(rows, bytes) * per, std::max({5.0, 2.6 + c.among * simd, others}) * per};
}

// A single step of one domain.  same_xcd: the blocks in an odd step's last band of
// rows are a multiple of 8, so that every row stays on its XCD and finds its
// populations in that L2 (the last band comes first in odd steps).
inline StepTime single_time(const StepModel& m, double mb, bool same_xcd) {
  const bool half = m.storage == 1 || m.storage == 2, fp64 = m.storage == 3;
  const double l2 = half ? .31 : .14;  // us per MB
  double t = mb < 32 ? std::max(4.9, 4.5 + l2 * mb) : 0.0;
  if (mb >= 20) t = std::max(t, half ? 4.6 + .31 * mb : (fp64 ? 3.2 + .235 * mb : 2.4 + .245 * mb));
  if (mb > 256) t = std::max(t, (half ? .39 : (fp64 ? .30 : .33)) * mb);
  if (!same_xcd)
    t = std::max(t, std::min(4.2 + (half ? .6 : (fp64 ? .47 : .5)) * mb, half ? 13.5 : 11.5));
  double side = std::max(3.4, half ? 1.9 + .325 * mb : 2.2 + .21 * mb);
  if (3 * mb > 225) side = std::max(side, (half ? .41 : .345) * mb);  // three handles' populations
  const double factor = 1.0 + .04 * (m.force + m.smagorinsky + m.drag) + .02 * m.trt;
  // 16-bit values in quantity: the instructions count as well.
  const double more = half && mb > 40 ? .08 * (m.force + m.smagorinsky + m.drag) + .02 * m.trt + .06 * m.guo : 0.0;
  return {t * (factor + more), side * factor};
}

// A single step of a batch, whose tiles are interleaved row by row (rows) or taken
// instance after instance.
inline StepTime batch_single_time(const StepModel& m, double mb, bool rows) {
  const bool half = m.storage == 1 || m.storage == 2;
  const double t = half ? (rows ? 4.1 + .46 * mb : 4.5 + .36 * mb)
                        : (rows ? 3.7 + .325 * mb : 4.0 + .29 * mb);
  const double side = half ? (rows ? 1.6 + .35 * mb : 1.0 + .385 * mb) : .34 * mb;
  const double factor = m.force ? 1.06 : 1.0;
  return {std::max(4.0, t) * factor, std::max(3.3, side) * factor};
}

}  // namespace flb
