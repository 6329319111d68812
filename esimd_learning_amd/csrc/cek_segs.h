// cek_segs.h -- the table of weight matrices ("segments") that one GEMV
// launch covers, shared by the GEMV kernels (cek_gemv.hip) and the
// weight-streaming kernel (cek_stream.hip).
#pragma once

#include "cek_common.h"

namespace cek {

constexpr int kCUs = 256;  // MI355X compute units, for the launch-balance rules
constexpr int MAX_SEGS = 8;

// Weight matrices sharing one x; gstart[i] = first workgroup of segment i.
struct GemvSegs {
  const uint8_t* w[MAX_SEGS];
  const void* s[MAX_SEGS];
  uint16_t* y[MAX_SEGS];
  int n[MAX_SEGS];
  int gstart[MAX_SEGS + 1];
  int count;
  const float* xs;  // per-row activation scales [M] when x holds e4m3 codes
};

struct SegRef {
  const uint8_t* w;
  const void* s;
  uint16_t* y;
  int n, group;
};

__device__ inline SegRef find_seg(const GemvSegs& sg, int b) {
  int i = 0;
#pragma unroll
  for (int j = 1; j < MAX_SEGS; ++j)
    if (j < sg.count && b >= sg.gstart[j]) i = j;
  return SegRef{sg.w[i], sg.s[i], sg.y[i], sg.n[i], b - sg.gstart[i]};
}

// Append matrix i of `from` to `to`.
inline void seg_push(GemvSegs& to, const GemvSegs& from, int i) {
  to.w[to.count] = from.w[i];
  to.s[to.count] = from.s[i];
  to.y[to.count] = from.y[i];
  to.n[to.count] = from.n[i];
  ++to.count;
}

// Fill gstart for `rows_per_wg` output rows per workgroup; returns the grid.
inline int seg_grid(GemvSegs& sg, int rows_per_wg) {
  int g = 0;
  for (int i = 0; i < sg.count; ++i) {
    sg.gstart[i] = g;
    g += (sg.n[i] + rows_per_wg - 1) / rows_per_wg;
  }
  for (int i = sg.count; i <= MAX_SEGS; ++i) sg.gstart[i] = g;
  return g;
}

// The weight-streaming kernel (cek_stream.hip): up to 64 rows, K % 64 == 0,
// 16-byte aligned x and weights; CEK_ERR_UNSUPPORTED for what it does not take.
constexpr int64_t kStreamMaxK = 1 << 24;
int launch_stream(const void* x, const GemvSegs& sg, int skind, int64_t M, int64_t K, int io_dtype, int fp8_fmt,
                  hipStream_t st);

// LDS writes of this wave done, then a workgroup barrier -- without the
// vmcnt(0) a fenced __syncthreads adds, which would drain the loads of the
// stages in flight.  The "memory" clobber keeps LDS accesses (and the
// activation loads, which are therefore not __restrict__) on their side.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace cek
