// cek_norm.hip -- fused residual-add + RMSNorm (+ per-token e4m3 quant), and
// standalone per-token e4m3 quantisation, gfx950.
//
// Reference algorithm (csrc/xpu/esimd_kernels/fused_add_rms_norm_batched.h):
//   pass 1 (:30-50)  r' = f16(h + r) stored; sum_sq over the unrounded fp32 sum
//   (:52-53)         inv = rsqrt(sum_sq / H + eps)
//   pass 2 (:55-62)  h  = f16(r' * inv * w)
// The reference runs one work-item per row; here one 256-thread workgroup
// owns a row: each thread keeps UPT 8-element units of the row in registers
// between the passes, so the row is read once and written once.
//
// The quantising variant rounds the normed row to the activation type, takes
// amax over those rounded values, and quantises them exactly as
// per_token_quant_kernel does, with the same launch shape and reduction
// order as the plain norm kernel.  The fused result is therefore bit-identical
// to the unfused pair (norm kernel, then quant kernel).
#include "cek_rowops.h"

namespace cek {

constexpr int NORM_THREADS = 256;

// Workgroup-wide sum / max for NORM_THREADS threads (4 waves).
__device__ inline float block_sum(float v, float* sh) { return wg4_sum(v, sh); }
__device__ inline float block_max(float v, float* sh) {
  v = wave_max(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  float t = fmaxf(fmaxf(sh[0], sh[1]), fmaxf(sh[2], sh[3]));
  __syncthreads();
  return t;
}


// Vector path: H % 8 == 0, 16-byte aligned rows, H <= 8 * NORM_THREADS * UPT.
template <typename T, int UPT, bool QUANT, bool EARLY>
__global__ __launch_bounds__(NORM_THREADS) void add_rmsnorm_kernel(
    const uint16_t* hidden, const uint16_t* residual, uint16_t* hidden_out, uint16_t* residual_out,
    const uint16_t* __restrict__ weight, int H, float eps, uint8_t* __restrict__ q, float* __restrict__ qscale) {
  __shared__ float sh[4];
  const int row = blockIdx.x;
  const int units = H >> 3;
  const uint16_t* hr = hidden + (size_t)row * H;
  const uint16_t* rr = residual + (size_t)row * H;
  uint16_t* ho = hidden_out + (size_t)row * H;
  uint16_t* ro = residual_out + (size_t)row * H;

  // EARLY (up to 512 rows of more than one unit a thread, where the chain of
  // latencies is what a launch takes, and always when quantising): all loads, the
  // norm weight's too, go out before the first sum (64 rows of 5120 3.35 -> 3.03
  // us, quantising 4.46 -> 3.91; 2048 rows of 5120 quantising 17.7 -> 14.3).  Without
  // quantising, more rows are up to 5% faster with a unit's loads beside its sum
  // (1024 rows of 5120 6.45 against 6.78 us): other rows' waves cover them.
  u4 hv[UPT], rv[UPT], wv[UPT];
  if constexpr (EARLY) {
#pragma unroll
    for (int j = 0; j < UPT; ++j) {
      const int u = min((int)threadIdx.x + j * NORM_THREADS, units - 1);
      hv[j] = load_u4(hr + u * 8);
      rv[j] = load_u4(rr + u * 8);
    }
#pragma unroll
    for (int j = 0; j < UPT; ++j) wv[j] = load_u4(weight + min((int)threadIdx.x + j * NORM_THREADS, units - 1) * 8);
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < UPT; ++j) {
    const int u = threadIdx.x + j * NORM_THREADS;
    if (u < units) {
      if constexpr (!EARLY) {
        hv[j] = load_u4(hr + u * 8);
        rv[j] = load_u4(rr + u * 8);
      }
      const u4 o = addnorm_pass1<T>(hv[j], rv[j], ss);
      rv[j] = o;
      *reinterpret_cast<u4*>(ro + u * 8) = o;
    }
  }
  ss = block_sum(ss, sh);
  const float inv = rsqrtf(ss / (float)H + eps);

  float amax = 0.f;
  u4 nv[UPT];
#pragma unroll
  for (int j = 0; j < UPT; ++j) {
    const int u = threadIdx.x + j * NORM_THREADS;
    if (u < units) {
      if constexpr (!EARLY) wv[j] = load_u4(weight + u * 8);
      const u4 o = addnorm_pass2<T>(rv[j], wv[j], inv);
      if (QUANT) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          amax = fmaxf(amax, fmaxf(fabsf(T::to_f32(o[e] & 0xFFFF)), fabsf(T::to_f32(o[e] >> 16))));
        nv[j] = o;
      } else {
        *reinterpret_cast<u4*>(ho + u * 8) = o;
      }
    }
  }
  if (!QUANT) return;

  amax = block_max(amax, sh);
  const float s = quant_scale(amax);
  const QuantDiv qd = quant_div(s);
  if (threadIdx.x == 0) qscale[row] = s;
  uint8_t* qr = q + (size_t)row * H;
#pragma unroll
  for (int j = 0; j < UPT; ++j) {
    const int u = threadIdx.x + j * NORM_THREADS;
    if (u < units) {
      uint32_t c[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t a = nv[j][2 * e], b = nv[j][2 * e + 1];
        c[e] = f32x4_to_e4m3x4(quant_clamp(T::to_f32(a & 0xFFFF), qd), quant_clamp(T::to_f32(a >> 16), qd),
                               quant_clamp(T::to_f32(b & 0xFFFF), qd), quant_clamp(T::to_f32(b >> 16), qd));
      }
      *reinterpret_cast<uint2*>(qr + u * 8) = make_uint2(c[0], c[1]);
    }
  }
}

// Scalar path for any H / alignment: three passes over global memory.
template <typename T, bool QUANT>
__global__ __launch_bounds__(NORM_THREADS) void add_rmsnorm_generic_kernel(
    const uint16_t* hidden, const uint16_t* residual, uint16_t* hidden_out, uint16_t* residual_out,
    const uint16_t* __restrict__ weight, int H, float eps, uint8_t* __restrict__ q, float* __restrict__ qscale) {
  __shared__ float sh[4];
  const int row = blockIdx.x;
  const uint16_t* hr = hidden + (size_t)row * H;
  const uint16_t* rr = residual + (size_t)row * H;
  uint16_t* ho = hidden_out + (size_t)row * H;
  uint16_t* ro = residual_out + (size_t)row * H;
  float ss = 0.f;
  for (int i = threadIdx.x; i < H; i += NORM_THREADS) {
    float a = T::to_f32(hr[i]) + T::to_f32(rr[i]);
    ss = fmaf(a, a, ss);
    ro[i] = T::from_f32(a);  // re-read below by this same thread only
  }
  ss = block_sum(ss, sh);
  const float inv = rsqrtf(ss / (float)H + eps);
  float amax = 0.f;
  for (int i = threadIdx.x; i < H; i += NORM_THREADS) {
    uint16_t b = T::from_f32(f32_round(T::to_f32(ro[i]) * inv * T::to_f32(weight[i])));
    if (QUANT) amax = fmaxf(amax, fabsf(T::to_f32(b)));
    else ho[i] = b;
  }
  if (!QUANT) return;
  amax = block_max(amax, sh);
  const float s = quant_scale(amax);
  const QuantDiv qd = quant_div(s);
  if (threadIdx.x == 0) qscale[row] = s;
  for (int i = threadIdx.x; i < H; i += NORM_THREADS) {
    uint16_t b = T::from_f32(f32_round(T::to_f32(ro[i]) * inv * T::to_f32(weight[i])));
    q[(size_t)row * H + i] = (uint8_t)f32_to_e4m3(quant_clamp(T::to_f32(b), qd));
  }
}

// Per-token quantisation of a [rows, H] activation matrix: rows that the
// register form below does not take (unaligned, or longer than 32768).
template <typename T>
__global__ __launch_bounds__(NORM_THREADS) void per_token_quant_kernel(
    const uint16_t* __restrict__ x, int H, uint8_t* __restrict__ q, float* __restrict__ qscale, int vec) {
  __shared__ float sh[4];
  const int row = blockIdx.x;
  const uint16_t* xr = x + (size_t)row * H;
  uint8_t* qr = q + (size_t)row * H;
  float amax = 0.f;
  if (vec) {
    for (int u = threadIdx.x; u < (H >> 3); u += NORM_THREADS) {
      u4 v = load_u4(xr + u * 8);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        amax = fmaxf(amax, fmaxf(fabsf(T::to_f32(v[e] & 0xFFFF)), fabsf(T::to_f32(v[e] >> 16))));
    }
  } else {
    for (int i = threadIdx.x; i < H; i += NORM_THREADS) amax = fmaxf(amax, fabsf(T::to_f32(xr[i])));
  }
  amax = block_max(amax, sh);
  const float s = quant_scale(amax);
  const QuantDiv qd = quant_div(s);
  if (threadIdx.x == 0) qscale[row] = s;
  if (vec) {
    for (int u = threadIdx.x; u < (H >> 3); u += NORM_THREADS) {
      u4 v = load_u4(xr + u * 8);
      uint32_t c[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t a = v[2 * e], b = v[2 * e + 1];
        c[e] = f32x4_to_e4m3x4(quant_clamp(T::to_f32(a & 0xFFFF), qd), quant_clamp(T::to_f32(a >> 16), qd),
                               quant_clamp(T::to_f32(b & 0xFFFF), qd), quant_clamp(T::to_f32(b >> 16), qd));
      }
      *reinterpret_cast<uint2*>(qr + u * 8) = make_uint2(c[0], c[1]);
    }
  } else {
    for (int i = threadIdx.x; i < H; i += NORM_THREADS)
      qr[i] = (uint8_t)f32_to_e4m3(quant_clamp(T::to_f32(xr[i]), qd));
  }
}

// The same with the row held in registers between the maximum and the codes
// (read once): H % 8 == 0, 16-byte aligned rows, H <= 8 NT UPT.  The maximum does
// not depend on the thread layout, so neither do scale and codes.  What bounds
// it: HBM for many rows (2048 rows of 14336: 28.6 us reading twice with a
// divide per element -> 20.4; 23.4 with 1024 threads a row), the chain load,
// reduction, store for few, so a long row takes up to 1024 threads (64 rows of
// 14336 7.1 -> 3.9 us, 4 of 24576 8.7 -> 4.3).
template <typename T, int NT, int UPT>
__global__ __launch_bounds__(NT) void per_token_quant_row_kernel(const uint16_t* __restrict__ x, int H,
                                                                 uint8_t* __restrict__ q, float* __restrict__ qscale) {
  __shared__ float sh[NT / 64];
  const int row = blockIdx.x, units = H >> 3;
  const uint16_t* xr = x + (size_t)row * H;
  uint8_t* qr = q + (size_t)row * H;
  u4 v[UPT];
#pragma unroll
  for (int j = 0; j < UPT; ++j) v[j] = load_u4(xr + min((int)threadIdx.x + j * NT, units - 1) * 8);
  float amax = 0.f;  // (units past the row repeat its last one)
#pragma unroll
  for (int j = 0; j < UPT; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      amax = fmaxf(amax, fmaxf(fabsf(T::to_f32(v[j][e] & 0xFFFF)), fabsf(T::to_f32(v[j][e] >> 16))));
  amax = wave_max(amax);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = amax;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) amax = fmaxf(amax, sh[w]);
  const float s = quant_scale(amax);
  const QuantDiv qd = quant_div(s);
  if (threadIdx.x == 0) qscale[row] = s;
#pragma unroll
  for (int j = 0; j < UPT; ++j) {
    const int u = threadIdx.x + j * NT;
    if (u < units) {
      uint32_t c[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t a = v[j][2 * e], b = v[j][2 * e + 1];
        c[e] = f32x4_to_e4m3x4(quant_clamp(T::to_f32(a & 0xFFFF), qd), quant_clamp(T::to_f32(a >> 16), qd),
                               quant_clamp(T::to_f32(b & 0xFFFF), qd), quant_clamp(T::to_f32(b >> 16), qd));
      }
      *reinterpret_cast<uint2*>(qr + u * 8) = make_uint2(c[0], c[1]);
    }
  }
}

template <typename T>
static void launch_quant_t(const uint16_t* x, int64_t rows, int H, uint8_t* q, float* s, bool vec, hipStream_t st) {
  const dim3 grid((unsigned)rows);
  const int units = H / 8;
  // many rows: few threads per row, so that a CU holds many rows in flight;
  // few rows: many threads, for the latency of a long row
  const bool many = rows >= 512;
#define CEK_Q(NT, UPT) per_token_quant_row_kernel<T, NT, UPT><<<grid, NT, 0, st>>>(x, H, q, s)
  if (vec && units <= 256) CEK_Q(256, 1);
  else if (vec && units <= 512) CEK_Q(256, 2);
  else if (vec && units <= 1024) { if (many) CEK_Q(256, 4); else CEK_Q(512, 2); }
  else if (vec && units <= 2048) { if (many) CEK_Q(256, 8); else CEK_Q(1024, 2); }
  else if (vec && units <= 4096) { if (many) CEK_Q(512, 8); else CEK_Q(1024, 4); }
  else per_token_quant_kernel<T><<<grid, NORM_THREADS, 0, st>>>(x, H, q, s, vec);
#undef CEK_Q
}

template <typename T, bool QUANT>
static int launch_norm_t(const void* hidden, const void* residual, void* hidden_out, void* residual_out,
                         const void* weight, int rows, int H, float eps, uint8_t* q, float* qs, hipStream_t st) {
  const uint16_t* h = static_cast<const uint16_t*>(hidden);
  const uint16_t* r = static_cast<const uint16_t*>(residual);
  uint16_t* ho = static_cast<uint16_t*>(hidden_out);
  uint16_t* ro = static_cast<uint16_t*>(residual_out);
  const uint16_t* w = static_cast<const uint16_t*>(weight);
  const int units = H / 8;
  const bool vec = H % 8 == 0 && aligned(hidden, 16) && aligned(residual, 16) && aligned(weight, 16) &&
                   aligned(residual_out, 16) && (QUANT ? aligned(q, 8) : aligned(hidden_out, 16));
  const int upt = (units + NORM_THREADS - 1) / NORM_THREADS;
  dim3 grid(rows);
#define CEK_NORM_K(UPT, EARLY) \
  add_rmsnorm_kernel<T, UPT, QUANT, EARLY><<<grid, NORM_THREADS, 0, st>>>(h, r, ho, ro, w, H, eps, q, qs)
#define CEK_NORM(UPT)                                                                        \
  do {                                                                                       \
    if (QUANT || (UPT > 1 && rows <= 512)) CEK_NORM_K(UPT, (QUANT || UPT > 1));              \
    else CEK_NORM_K(UPT, QUANT);                                                             \
  } while (0)
  if (vec && upt <= 1) CEK_NORM(1);
  else if (vec && upt <= 2) CEK_NORM(2);
  else if (vec && upt <= 3) CEK_NORM(3);
  else if (vec && upt <= 4) CEK_NORM(4);
  else if (vec && upt <= 8) CEK_NORM(8);
#undef CEK_NORM
#undef CEK_NORM_K
  else add_rmsnorm_generic_kernel<T, QUANT><<<grid, NORM_THREADS, 0, st>>>(h, r, ho, ro, w, H, eps, q, qs);
  return check_launch();
}

}  // namespace cek

using namespace cek;

static int norm_args_ok(const void* h, const void* r, const void* w, int64_t rows, int64_t H) {
  if (rows < 0 || H <= 0 || rows > INT32_MAX || H > INT32_MAX / 2) return CEK_ERR_INVALID;
  if (rows > 0 && (!h || !r || !w)) return CEK_ERR_INVALID;
  return CEK_OK;
}

extern "C" int cek_add_rms_norm_out(const void* hidden, const void* residual, const void* weight, void* residual_out,
                                    void* hidden_out, int64_t rows, int64_t H, float eps, int io_dtype, uint8_t* q,
                                    float* scale, void* stream) {
  int rc = norm_args_ok(hidden, residual, weight, rows, H);
  if (rc) return rc;
  if (rows == 0) return CEK_OK;
  if (!residual_out || (q ? !scale : !hidden_out)) return CEK_ERR_INVALID;
  hipStream_t st = (hipStream_t)stream;
  const int r = (int)rows, h = (int)H;
  void* ho = q ? residual_out : hidden_out;  // (never stored by the quantising form)
  if (io_dtype == CEK_F16) {
    if (q) return launch_norm_t<F16, true>(hidden, residual, ho, residual_out, weight, r, h, eps, q, scale, st);
    return launch_norm_t<F16, false>(hidden, residual, ho, residual_out, weight, r, h, eps, nullptr, nullptr, st);
  }
  if (io_dtype == CEK_BF16) {
    if (q) return launch_norm_t<BF16, true>(hidden, residual, ho, residual_out, weight, r, h, eps, q, scale, st);
    return launch_norm_t<BF16, false>(hidden, residual, ho, residual_out, weight, r, h, eps, nullptr, nullptr, st);
  }
  return CEK_ERR_INVALID;
}

extern "C" int cek_fused_add_rms_norm(void* hidden, void* residual, const void* weight,
                                      int64_t rows, int64_t H, float eps, int io_dtype, void* stream) {
  return cek_add_rms_norm_out(hidden, residual, weight, residual, hidden, rows, H, eps, io_dtype, nullptr, nullptr,
                              stream);
}

extern "C" int cek_fused_add_rms_norm_quant_fp8(const void* hidden, void* residual, const void* weight,
                                                int64_t rows, int64_t H, float eps, int io_dtype,
                                                uint8_t* q, float* scale, void* stream) {
  if (!q || !scale) {  // (no rows: nothing to write them to)
    const int rc = norm_args_ok(hidden, residual, weight, rows, H);
    return rc ? rc : (rows == 0 ? CEK_OK : CEK_ERR_INVALID);
  }
  return cek_add_rms_norm_out(hidden, residual, weight, residual, nullptr, rows, H, eps, io_dtype, q, scale, stream);
}

extern "C" int cek_per_token_quant_fp8(const void* x, int64_t rows, int64_t H, int io_dtype,
                                       uint8_t* q, float* scale, void* stream) {
  if (rows < 0 || H <= 0 || rows > INT32_MAX || H > INT32_MAX / 2) return CEK_ERR_INVALID;
  if (rows == 0) return CEK_OK;
  if (!x || !q || !scale) return CEK_ERR_INVALID;
  hipStream_t st = (hipStream_t)stream;
  const bool vec = H % 8 == 0 && aligned(x, 16) && aligned(q, 8);
  const uint16_t* xp = static_cast<const uint16_t*>(x);
  if (io_dtype == CEK_F16) launch_quant_t<F16>(xp, rows, (int)H, q, scale, vec, st);
  else if (io_dtype == CEK_BF16) launch_quant_t<BF16>(xp, rows, (int)H, q, scale, vec, st);
  else return CEK_ERR_INVALID;
  return check_launch();
}
