// cek_stream.hip -- weight-streaming product of a few activation rows with
// fp8 weights, gfx950: y[m, n] = Out((sum_k x[m, k] * dq(W[n, k])) * scale[n])
// for 3 <= M <= 64 rows and any K (a multiple of 64).
//
// What bounds it: the weights have to be read from HBM once, and every CU
// reads all M activation rows (from L2) for its share of the weight rows; at
// M >= 32 the activations are most of what a CU moves.  Both go to LDS by
// direct-to-LDS loads (1 KB contiguous per instruction: 4 weight rows x 256
// bytes or 2 activation rows x 512), the form the CU's load path takes at its
// full rate, issued by loader waves that do nothing else: two for the
// weights, two or four for the activations, so that no stream's in-order
// vmcnt waits wait for the other's loads, through rings as deep as LDS holds.
// Eight consumer waves each take an eighth of a stage's K values over all MB x
// NT 16 x 16 blocks (every LDS byte is read once) and meet in LDS at the end;
// their only memory operations in the loop are LDS reads.  One barrier per
// stage.  e4m3 activations: up to 16 rows decoded to fp16 like the weights
// (both exactly) and multiplied there, since the fp8 MFMA's sums are not
// rounded as fp32 ones are: 1.5e-5 of the result (2-norm; 6.7% of the fp16
// outputs differ from the correctly rounded product) against 1e-7 (0.1%); above
// 16 rows by the fp8 MFMA, as in every other kernel for them.  What a launch
// takes is about 4.8 us (the launch, the first bytes,
// the stages' barriers, the epilogue) plus a CU's bytes at 90 per ns for the
// activations and 25-30 for the weights.  Measured on MI355X, weights from
// HBM, against the kernels that served these shapes before (us): M = 48, K =
// 4096, N = 6144 47.7 (128 x 128 tiles) -> 12.4, N = 28672 51.7 -> 33.3; M = 32, K
// = 4096, N = 14336 36.7 -> 15.2; M = 8, K = 2560, N = 20480 23.2 (operand loads
// straight from global memory) -> 12.5; M = 4, K = 10240, N = 2560 11.1
// (v_dot2) -> 8.4.
// What did not pay: one workgroup per CU for small M (M = 8, K = 2560, N =
// 20480 12.4 -> 16.6 us: the rings of the second one cover the first one's
// fill and epilogue); a deeper weight ring beside a shallow activation ring
// (within 2%); run-time loads per stage (M = 48 12.4 -> 17.7 us: the waits
// become a branch tree).
#include <algorithm>
#include <type_traits>

#include "cek_segs.h"

namespace cek {

constexpr int kStreamConsumers = 8;  // waves that multiply
constexpr int kStreamMaxRows = 64;   // weight rows of a workgroup
constexpr int kStreamNarrowRows = 24;    // the same, for the narrow form (launch_stream)
constexpr int kStreamRotateRows = 8192;  // rows from which on a matrix has its K stages rotated
constexpr int kStreamScaleBytes = kStreamMaxRows * 4 + 64 * 4;

// One configuration: AR activation rows held in LDS, RW weight rows per
// workgroup, KW K values per consumer wave and stage.
template <bool XF8, int AR, int RW, int KW>
struct StreamCfg {
  static constexpr int KS = KW * kStreamConsumers;    // K values of a stage
  static constexpr int ARB = KS * (XF8 ? 1 : 2);      // activation bytes per row and stage
  static constexpr int MB = (AR + 15) / 16, NT = (RW + 15) / 16;
  static constexpr int WL = 2, AL = AR >= 64 ? 4 : 2; // loader waves
  static constexpr int THREADS = 64 * (kStreamConsumers + WL + AL);
  static constexpr int LDSB = AR <= 16 && RW * KS <= 12288 ? 81920 : 163840;  // two workgroups per CU, or one
  static constexpr int RING = LDSB - kStreamScaleBytes;   // bytes of both rings
  static constexpr int ASZ = AR * ARB, WSZ = RW * KS;
  static constexpr int ALOADS = ASZ / 1024, WLOADS = WSZ / 1024;
  static constexpr int AM = (ALOADS + AL - 1) / AL, WM = (WLOADS + WL - 1) / WL;  // per loader wave and stage
  // Both rings hold the same number of stages: the CU's load path returns
  // data in order, so an activation load waits behind the weight loads issued
  // before it and needs as long a lead.
  static constexpr int R0 = RING / (ASZ + WSZ), R1 = R0 > 24 ? 24 : R0;
  static constexpr int PER = AM > WM ? AM : WM, R = R1 > 62 / PER + 1 ? 62 / PER + 1 : R1;
  static_assert(ASZ % 1024 == 0 && WSZ % 1024 == 0, "1 KB loads");
  static_assert(R >= 2 && (R - 1) * PER <= 63 && R * (ASZ + WSZ) <= RING, "rings");
};

// One loader wave (`who` of WAVES): streams the S stages of a matrix through
// a ring of RING LDS slots, ROWS rows x RB bytes per stage.  A slot holds the
// stage's rows one after another in 16-byte units, unit u of row r at
// u ^ (r & 15) (the sixteen rows of an MFMA fragment read then fall in
// sixteen different bank groups); load j fills the slot's bytes [1024 j,
// 1024 j + 1024), each lane fetching the unit that belongs at its place.
// Rows past rmax read row rmax, units past the row its last one (neither is
// used).  It takes part in the S stage barriers: before barrier i stage i has
// landed; after it the slot of stage i - 1 is free and takes stage
// i - 1 + RING.  Every wait count is an immediate (a run-time count cost a
// branch tree of ~300 cycles per stage).
template <int RB, int ROWS, int RING, int WAVES>
__device__ __forceinline__ void stream_load(uint8_t* slots, int rmax, uint32_t row_bytes, int S, int k_first,
                                            __amdgpu_buffer_rsrc_t rsrc, int who, int lane) {
  constexpr int UPR = RB / 16, LOADS = ROWS * RB / 1024, MINE = (LOADS + WAVES - 1) / WAVES, SLOT = ROWS * RB;
  uint32_t vo[MINE], ku[MINE];
#pragma unroll
  for (int m = 0; m < MINE; ++m) {
    const int q = 64 * min(who + WAVES * m, LOADS - 1) + lane, row = q / UPR;
    ku[m] = 16u * (uint32_t)((q % UPR) ^ (row & 15));
    vo[m] = (uint32_t)min(row, rmax) * row_bytes;
  }
  auto issue = [&](int s, int slot) {
    uint8_t* dst = slots + slot * SLOT;
    const uint32_t k0 = (uint32_t)(s + k_first >= S ? s + k_first - S : s + k_first) * RB;
    const bool tail = k0 + RB > row_bytes;
#pragma unroll
    for (int m = 0; m < MINE; ++m) {
      uint32_t k = k0 + ku[m];
      if (tail) k = min(k, row_bytes - 16u);
#if defined(__HIP_DEVICE_COMPILE__)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(dst + 1024 * min(who + WAVES * m, LOADS - 1)), 16,
                                               vo[m] + k, 0, 0, 0);
#endif
    }
  };
#pragma unroll
  for (int s = 0; s < RING; ++s)
    if (s < S) issue(s, s);
  if (S >= RING) {
    wait_vmcnt<(RING - 1) * MINE>();
    bare_barrier();
    int slot = 0;
    for (int s = RING; s < S; ++s) {  // before the barrier of stage s + 1 - RING
      wait_vmcnt<(RING - 2) * MINE>();
      bare_barrier();
      issue(s, slot);
      slot = slot + 1 == RING ? 0 : slot + 1;
    }
  }
  // the last stages, S - 1 - r: r stages after them in flight
  auto drain = [&](auto self, auto rc) {
    constexpr int r = decltype(rc)::value;
    if (S >= RING ? r < RING - 1 : r < S) {
      wait_vmcnt<r * MINE>();
      bare_barrier();
    }
    if constexpr (r > 0) self(self, std::integral_constant<int, r - 1>{});
  };
  drain(drain, std::integral_constant<int, RING - 1>{});
}

template <typename T, int FMT, bool XF8, int AR, int RW, int KW>
__global__ __launch_bounds__((StreamCfg<XF8, AR, RW, KW>::THREADS), (StreamCfg<XF8, AR, RW, KW>::LDSB > 81920 ? 3 : 6))
void stream_kernel(const uint8_t* __restrict__ x, GemvSegs sg, int skind, int M, int K, int bf16_out) {
  using C = StreamCfg<XF8, AR, RW, KW>;
  constexpr int KS = C::KS, ARB = C::ARB, MB = C::MB, NT = C::NT, R = C::R;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[C::LDSB];
  uint32_t* const sw = reinterpret_cast<uint32_t*>(smem + C::RING);             // weight scales (raw bits) [RW]
  float* const sx = reinterpret_cast<float*>(smem + C::RING) + kStreamMaxRows;  // activation scales [M]
  uint8_t* const wslots = smem + R * C::ASZ;
  const SegRef sr = find_seg(sg, blockIdx.x);
  const int N = sr.n, n0 = sr.group * RW;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int S = (K + KS - 1) / KS;
  const int k_first = N >= kStreamRotateRows ? (int)((unsigned)(sr.group >> 3) % (unsigned)S) : 0;

  f4 acc[MB][NT];
#pragma unroll
  for (int b = 0; b < MB; ++b)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[b][t] = f4{0.f, 0.f, 0.f, 0.f};

  if (wave >= kStreamConsumers + C::WL) {
    const uint32_t xb = (uint32_t)K * (XF8 ? 1 : 2);
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(x), 0, (int)((uint32_t)M * xb), 0x00020000);
    stream_load<ARB, AR, R, C::AL>(smem, M - 1, xb, S, k_first, r, wave - kStreamConsumers - C::WL, lane);
  } else if (wave >= kStreamConsumers) {
    const int rows = min(RW, N - n0);
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(sr.w + (size_t)n0 * K), 0, (int)((uint32_t)rows * (uint32_t)K), 0x00020000);
    stream_load<KS, RW, R, C::WL>(wslots, rows - 1, (uint32_t)K, S, k_first, r, wave - kStreamConsumers, lane);
  } else {
    // the scales, for the epilogue (published by the first barrier)
    if (wave == 0 && lane < RW) sw[lane] = load_scale_bits(sr.s, skind, min(n0 + lane, N - 1));
    if constexpr (XF8) {
      if (wave == 1 && lane < M) sx[lane] = sg.xs[lane];
    }
    // this lane's fragment places within a slot: NU 16-byte activation units
    // per row from unit 4 NU wave + NU g on (w8a16: KW / 4 values; e4m3: KW / 4
    // codes), the weights' K values likewise (rows past the slot's repeat its
    // last one)
    constexpr int NU = ARB / kStreamConsumers / 64;  // units per lane: 1, or 2 for 64 16-bit values per wave
    constexpr int WB = KW / 4;                       // weight bytes per lane: 8 or 16
    int ao[MB][NU], wo[NT];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int row = min(16 * b + r16, AR - 1);
#pragma unroll
      for (int u = 0; u < NU; ++u) ao[b][u] = row * ARB + 16 * ((4 * NU * wave + NU * g + u) ^ (row & 15));
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int row = min(16 * t + r16, RW - 1), byte = wave * KW + g * WB;
      wo[t] = row * KS + 16 * ((byte >> 4) ^ (row & 15)) + (byte & 15);
    }
    const uint8_t* pa = smem;
    const uint8_t* pw = wslots;
    int ks = k_first;
    for (int i = 0; i < S; ++i) {
      lds_barrier();  // stage i has landed; this wave's reads of stage i - 1 are done
      if (ks * KS + wave * KW < K) {
        u4 af[MB][NU];
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
          for (int u = 0; u < NU; ++u) af[b][u] = *reinterpret_cast<const u4*>(pa + ao[b][u]);
        [[maybe_unused]] u4 alo, ahi;
        if constexpr (XF8 && AR <= 16) decode16<F16, CEK_E4M3>(af[0][0], alo, ahi);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          if constexpr (XF8 && AR <= 16) {
            u4 lo, hi;
            decode16<F16, CEK_E4M3>(*reinterpret_cast<const u4*>(pw + wo[t]), lo, hi);
            acc[0][t] = mfma16x16x32<F16>(alo, lo, acc[0][t]);
            acc[0][t] = mfma16x16x32<F16>(ahi, hi, acc[0][t]);
          } else if constexpr (XF8) {
            typedef long l2 __attribute__((ext_vector_type(2)));
            const l2 wv = *reinterpret_cast<const l2*>(pw + wo[t]);
#pragma unroll
            for (int b = 0; b < MB; ++b) {
              const l2 av = __builtin_bit_cast(l2, af[b][0]);
              acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(av[0], wv[0], acc[b][t], 0, 0, 0);
              acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(av[1], wv[1], acc[b][t], 0, 0, 0);
            }
          } else if constexpr (WB == 8) {
            const uint2 wv = *reinterpret_cast<const uint2*>(pw + wo[t]);
            const u4 wd = decode8<T, FMT>(wv.x, wv.y);
#pragma unroll
            for (int b = 0; b < MB; ++b) acc[b][t] = mfma16x16x32<T>(af[b][0], wd, acc[b][t]);
          } else {
            u4 lo, hi;
            decode16<T, FMT>(*reinterpret_cast<const u4*>(pw + wo[t]), lo, hi);
#pragma unroll
            for (int b = 0; b < MB; ++b) {
              acc[b][t] = mfma16x16x32<T>(af[b][0], lo, acc[b][t]);
              acc[b][t] = mfma16x16x32<T>(af[b][NU - 1], hi, acc[b][t]);
            }
          }
        }
      }
      ks = ks + 1 == S ? 0 : ks + 1;
      pa = pa + C::ASZ == smem + R * C::ASZ ? smem : pa + C::ASZ;
      pw = pw + C::WSZ == wslots + R * C::WSZ ? wslots : pw + C::WSZ;
    }
  }

  // The eight waves' sums meet in LDS, GB blocks at a time, added in wave
  // order; D row 4 (lane >> 4) + v of a block is activation row m, column
  // lane & 15 the weight row.
  constexpr int BL = MB * NT, GB0 = C::RING / (kStreamConsumers * 1024), GB = GB0 < BL ? GB0 : BL;
  f4* const red = reinterpret_cast<f4*>(smem);  // [8][GB][64]
#pragma unroll
  for (int b0 = 0; b0 < BL; b0 += GB) {
    lds_barrier();  // the slots, or the blocks before, are done with
    if (wave < kStreamConsumers) {
#pragma unroll
      for (int j = 0; j < GB; ++j)
        if (b0 + j < BL) red[(wave * GB + j) * 64 + lane] = acc[(b0 + j) / NT][(b0 + j) % NT];
    }
    lds_barrier();
    for (int q = threadIdx.x; q < GB * 64; q += C::THREADS) {
      const int blk = b0 + q / 64, n = 16 * (blk % NT) + (q & 15), m0 = 16 * (blk / NT) + 4 * ((q & 63) >> 4);
      if (blk >= BL || n >= RW || n0 + n >= N || m0 >= M) continue;
      f4 c = red[q];
#pragma unroll
      for (int w = 1; w < kStreamConsumers; ++w) c += red[w * GB * 64 + q];
      const float sc = scale_value(sw[n], skind);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (m0 + v >= M) continue;
        const float o = f32_round(c[v] * (XF8 ? sc * sx[m0 + v] : sc));
        sr.y[(size_t)(m0 + v) * N + n0 + n] = bf16_out ? BF16::from_f32(o) : F16::from_f32(o);
      }
    }
  }
}

constexpr int kStreamRows[] = {8, 12, 16, 24, 32, 40, 48, 56, 64};

// Weight rows per workgroup: the count with the least work for the busiest
// CU.  Its workgroups each cost their weight rows and the activation rows (at
// 0.3-0.4 of a weight row each: 90 against 30 bytes per ns and CU measured),
// and every one after the first something by itself: 0.3 us where a CU holds two
// at a time, and where it holds one the filling and draining of the rings
// between two of them (2.7 us, or with e4m3 activations as long as the weight
// rows take if that is less; 1.5 us above 16 rows).  Without the first of these,
// up to 16 rows took workgroups of 8-16 weight rows for wide matrices (us,
// before -> now: M = 3, K = 5376, N = 26240 47.5 -> 27.7; M = 5, K = 1024, N =
// 28672 12.4 -> 9.1; e4m3 activations, M = 5, K = 1024, N = 26240 18.2 -> 9.9).  Over
// 2800 shapes of 3-16 rows the pick is 1% (geometric mean) above the fastest
// count.  Measured on MI355X, us: M = 4, K = 10240, N = 2560 8 / 12 / 16 rows
// 10.9 / 8.5 / 9.0; M = 16, K = 4096, N = 14336 32 / 56 rows 15.0 / 13.6; M = 8, K
// = 2560, N = 20480 40 / 48 rows 12.4 / 12.9; M = 5, K = 1024, N = 32768 32 / 48 /
// 64 rows 9.9 / 9.7 / 11.0; M = 48, K = 4096, N = 6144 24 / 32 rows 12.3 / 12.9.
static int stream_rows(int M, int64_t N, int K, bool xf8, int max_rows) {
  int best = 8;
  int64_t cost = INT64_MAX;
  const int64_t act = (M > 16 ? 3 : 4) * (xf8 ? (M + 1) / 2 : M);
  for (int r : kStreamRows) {
    if (r > max_rows) break;
    if (r == 8 && N >= kStreamRotateRows) continue;  // (never the fastest there)
    const int64_t per_cu = ((N + r - 1) / r + kCUs - 1) / kCUs;
    const bool pair = M <= 16 && r <= (xf8 ? 24 : 48);  // two workgroups per CU
    int64_t next = pair ? 100000 : (M > 16 ? 450000 : 800000);
    if (!pair && xf8 && M <= 16) next = std::min(next, (int64_t)8 * r * K);
    const int64_t c = per_cu * (10 * r + act) * K + (per_cu - 1) * next;
    if (c <= cost) {
      cost = c;
      best = r;
    }
  }
  return best;
}

template <typename T, int FMT, bool XF8>
static int launch_stream_t(const uint8_t* x, GemvSegs& sg, int skind, int M, int K, bool bf16_out, int rw, bool narrow,
                           hipStream_t st) {
  const dim3 grid((unsigned)seg_grid(sg, rw));
#define CEK_ST(AR, RW, KW)                                                                        \
  do {                                                                                            \
    stream_kernel<T, FMT, XF8, AR, RW, KW><<<grid, StreamCfg<XF8, AR, RW, KW>::THREADS, 0, st>>>( \
        x, sg, skind, M, K, bf16_out);                                                    \
    return check_launch();                                                                        \
  } while (0)
#define CEK_ST_ROWS(AR)                             \
  do {                                              \
    constexpr int kw = XF8 ? 64 : 32;               \
    if constexpr (!XF8 && (AR) <= 8) {              \
      if (narrow) {                                 \
        switch (rw) {                               \
          case 8: CEK_ST(AR, 8, 64);                \
          case 12: CEK_ST(AR, 12, 64);              \
          case 16: CEK_ST(AR, 16, 64);              \
          case 24: CEK_ST(AR, 24, 64);              \
          default: return CEK_ERR_UNSUPPORTED;      \
        }                                           \
      }                                             \
    }                                               \
    if constexpr (XF8 || (AR) > 8) {                \
      if (rw == 8) CEK_ST(AR, 8, kw);               \
    }                                               \
    switch (rw) {                                   \
      case 12: CEK_ST(AR, 12, kw);                  \
      case 16: CEK_ST(AR, 16, kw);                  \
      case 24: CEK_ST(AR, 24, kw);                  \
      case 32: CEK_ST(AR, 32, kw);                  \
      case 40: CEK_ST(AR, 40, kw);                  \
      case 48: CEK_ST(AR, 48, kw);                  \
      case 56: CEK_ST(AR, 56, kw);                  \
      case 64: CEK_ST(AR, 64, kw);                  \
      default: return CEK_ERR_UNSUPPORTED;          \
    }                                               \
  } while (0)
  if (M <= 4) CEK_ST_ROWS(4);
  else if (M <= 8) CEK_ST_ROWS(8);
  else if (M <= 16) CEK_ST_ROWS(16);
  else if (M <= 24) CEK_ST_ROWS(24);
  else if (M <= 32) CEK_ST_ROWS(32);
  else if (M <= 48) CEK_ST_ROWS(48);
  else CEK_ST_ROWS(64);
#undef CEK_ST
#undef CEK_ST_ROWS
}

// x: fp16 / bf16 [M, K] (io_dtype), or e4m3 codes with sg.xs set (io_dtype:
// the output type); x and the weights 16-byte aligned.  M <= 64, K % 64 == 0;
// CEK_ERR_UNSUPPORTED otherwise.  An output's sum order must not depend on
// which matrices share the launch, so what it depends on is set per matrix:
//  * 8192 rows or more: workgroup g starts at K stage (g / 8) mod S (g / 8: its
//    place on its XCD), so that workgroups streaming at the same time read
//    different columns of their rows and HBM's channels share the load (M =
//    16, K = 4096, N = 16384: 17.3 -> 14.6 us).  g counts workgroups of the rows
//    that stream_rows gives the matrix alone: matrices that agree in it share a
//    launch, and the other ones of their K per stage join it, whatever its rows;
//  * up to 8 rows of 16-bit activations and fewer than 8192 weight rows (narrow,
//    at most 24 rows per workgroup): 64 K values per wave and stage instead of
//    32, half the barriers (M = 4, K = 10240, N = 2560 9.2 -> 8.5 us, N = 512 9.4
//    -> 7.1; N = 6144 within 3%): a launch of their own.
// Three matrices of 9000 rows, M = 4, K = 2560 27.9 us in a launch each -> 15.8;
// 5120 + 1024 + 1024 rows, M = 5 10.1 us in two launches -> 6.4.
int launch_stream(const void* x, const GemvSegs& sg, int skind, int64_t M, int64_t K, int io_dtype, int fp8_fmt,
                  hipStream_t st) {
  if (M < 1 || M > 64 || K < 64 || K > kStreamMaxK || K % 64 != 0) return CEK_ERR_UNSUPPORTED;
  const uint8_t* xp = static_cast<const uint8_t*>(x);
  const int m = (int)M, k = (int)K;
  const bool bf = io_dtype == CEK_BF16, xf8 = sg.xs != nullptr;
  auto launch = [&](GemvSegs& part, bool narrow, int rw) {
    if (part.count == 0) return (int)CEK_OK;
    if (rw == 0) {
      int64_t N = 0;
      for (int i = 0; i < part.count; ++i) N += part.n[i];
      rw = stream_rows(m, N, k, xf8, narrow ? kStreamNarrowRows : kStreamMaxRows);
    }
    if (xf8) return launch_stream_t<F16, CEK_E4M3, true>(xp, part, skind, m, k, bf, rw, narrow, st);
    if (!bf) {
      if (fp8_fmt == CEK_E4M3) return launch_stream_t<F16, CEK_E4M3, false>(xp, part, skind, m, k, bf, rw, narrow, st);
      return launch_stream_t<F16, CEK_E5M2, false>(xp, part, skind, m, k, bf, rw, narrow, st);
    }
    if (fp8_fmt == CEK_E4M3) return launch_stream_t<BF16, CEK_E4M3, false>(xp, part, skind, m, k, bf, rw, narrow, st);
    return launch_stream_t<BF16, CEK_E5M2, false>(xp, part, skind, m, k, bf, rw, narrow, st);
  };
  GemvSegs narrow{}, wide{};  // wide: with the first group of rotated matrices
  narrow.xs = wide.xs = sg.xs;
  int rows[MAX_SEGS];  // of a rotated matrix not yet launched, else 0
  for (int i = 0; i < sg.count; ++i) {
    rows[i] = sg.n[i] >= kStreamRotateRows ? stream_rows(m, sg.n[i], k, xf8, kStreamMaxRows) : 0;
    if (!rows[i]) seg_push(!xf8 && M <= 8 ? narrow : wide, sg, i);
  }
  for (int i = 0; i < sg.count; ++i) {
    const int rw = rows[i];
    if (!rw) continue;
    for (int j = i; j < sg.count; ++j)
      if (rows[j] == rw) {
        seg_push(wide, sg, j);
        rows[j] = 0;
      }
    const int rc = launch(wide, false, rw);
    if (rc != CEK_OK) return rc;
    wide.count = 0;
  }
  const int rc = launch(wide, false, 0);
  return rc != CEK_OK ? rc : launch(narrow, true, 0);
}

}  // namespace cek
