// Residual-add + LayerNorm / RMSNorm, forward and backward, for gfx950.
//
//   v = x (+ residual when prenorm)           accumulated in fp32
//   LayerNorm: y = (v - mean) * rsqrt(var + eps) * w + b     (two-pass biased variance)
//   RMSNorm:   y = v * rsqrt(mean(v^2) + eps) * w + b
//   post-norm: y += residual
//
// One wavefront normalises one row and keeps the row in registers, so x and
// the residual are read from HBM exactly once and y / residual_out are written
// once; row statistics (mean, rstd) can be saved for the backward pass.
// Rows longer than the register budget (64 lanes * 32 values) fall back to a
// re-reading variant.
//
// Backward: a persistent grid walks rows; each wavefront produces dx (and
// dresidual) for its rows and accumulates dw/db columns in registers; per-wave
// partials are written once and folded by a second kernel in a fixed order.
#include "common.hpp"

#include <mutex>

#include <type_traits>

namespace ssm {

constexpr int LN_THREADS = 256;
constexpr int LN_WAVES = LN_THREADS / WAVE;

struct NormParams {
  const void *x, *res, *dy, *gro;   // gro: bwd, gradient of residual_out or NULL
  const float *w, *b;
  void *y, *res_out, *dx, *dres;
  float *mean, *rstd;       // per row; fwd: optional outputs, bwd: required inputs (mean unused for RMS)
  float *partial;           // bwd: [nwaves_total][2][hidden]
  int rows, hidden;
  int x_dtype, res_dtype, res_out_dtype, gro_dtype;
  int is_rms, prenorm;
  int has_db;                       // bwd: the second half of a partial is asked for
  int past_caches;                  // typed kernels: how to read what is not read again (NORM_CACHED)
  float eps;
};

// Calls up to these sizes leave what they read to the caches; larger ones read past them what is not read again (a backward
// everything, a forward its residual: x is what a backward reads again): the space is better spent on what is written, for
// those who read that.  Forward and backward (the forward keeps rstd), by elements, bf16 with a float32 residual and gradient
// through it, us without / with (replayed as graphs): 2048 x 768 16.8 / 17.4, 2048 x 2560 38.1 / 38.7, 4 x 2048 x 768 42.7 /
// 42.0, 8 x 2048 x 768 72.8 / 73.4 (72.0 / 69.4 one behind the other), 16 x 2048 x 768 149 / 145.5 (147 / 139); what is written
// past them: slower.  A forward alone, by bytes, where they are more than the last-level cache holds: 75 MB 13.8 / 15.9, 252 MB
// 44.0 / 44.8, 302 MB 54.6 / 53.7, float32 403 MB 71.8 / 63.1.
constexpr size_t NORM_CACHED = (size_t)5632 << 10, NORM_CACHED_BYTES = (size_t)268 << 20;

__device__ __forceinline__ void store_f32_as(void *p, int dtype, size_t i, float v) {
  if (dtype == SSM_F32) reinterpret_cast<float *>(p)[i] = v;
  else if (dtype == SSM_BF16) reinterpret_cast<bf16_t *>(p)[i] = from_f32<bf16_t>(v);
  else reinterpret_cast<f16_t *>(p)[i] = from_f32<f16_t>(v);
}

// Row element j of lane `lane`, trip `k`: column = (k * 64 + lane) * VEC + i.
template <int VEC>
__device__ __forceinline__ void load_cols(const void *p, int dtype, size_t base, int col, int hidden, bool vec_ok,
                                          float (&v)[VEC]) {
  if (vec_ok && col + VEC <= hidden) {
    if (dtype == SSM_F32) {
      Pack<float, VEC> r = *reinterpret_cast<const Pack<float, VEC> *>(reinterpret_cast<const float *>(p) + base + col);
#pragma unroll
      for (int i = 0; i < VEC; ++i) v[i] = r.v[i];
    } else if (dtype == SSM_BF16) {
      Pack<bf16_t, VEC> r = *reinterpret_cast<const Pack<bf16_t, VEC> *>(reinterpret_cast<const bf16_t *>(p) + base + col);
#pragma unroll
      for (int i = 0; i < VEC; ++i) v[i] = to_f32(r.v[i]);
    } else {
      Pack<f16_t, VEC> r = *reinterpret_cast<const Pack<f16_t, VEC> *>(reinterpret_cast<const f16_t *>(p) + base + col);
#pragma unroll
      for (int i = 0; i < VEC; ++i) v[i] = to_f32(r.v[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) v[i] = (col + i < hidden) ? load_as_f32(p, dtype, base + col + i) : 0.0f;
  }
}

template <int VEC>
__device__ __forceinline__ void store_cols(void *p, int dtype, size_t base, int col, int hidden, bool vec_ok,
                                           const float (&v)[VEC]) {
  if (vec_ok && col + VEC <= hidden) {
    if (dtype == SSM_F32) {
      Pack<float, VEC> r;
#pragma unroll
      for (int i = 0; i < VEC; ++i) r.v[i] = v[i];
      *reinterpret_cast<Pack<float, VEC> *>(reinterpret_cast<float *>(p) + base + col) = r;
    } else if (dtype == SSM_BF16) {
      Pack<bf16_t, VEC> r;
#pragma unroll
      for (int i = 0; i < VEC; ++i) r.v[i] = from_f32<bf16_t>(v[i]);
      *reinterpret_cast<Pack<bf16_t, VEC> *>(reinterpret_cast<bf16_t *>(p) + base + col) = r;
    } else {
      Pack<f16_t, VEC> r;
#pragma unroll
      for (int i = 0; i < VEC; ++i) r.v[i] = from_f32<f16_t>(v[i]);
      *reinterpret_cast<Pack<f16_t, VEC> *>(reinterpret_cast<f16_t *>(p) + base + col) = r;
    }
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      if (col + i < hidden) store_f32_as(p, dtype, base + col + i, v[i]);
  }
}

// ------------------------------------------------------------------ forward

// A row is held in registers by one wavefront (WG = false: TRIPS * 64 * VEC >= hidden) or, for long rows, by
// the whole workgroup (WG = true: TRIPS * 256 * VEC >= hidden; sums over the row go through LDS).  VEC = 4
// keeps every access <= 16 bytes for all dtypes.
template <bool WG>
__device__ __forceinline__ float row_sum(float v, float *red) {
  v = wave_sum(v);
  if constexpr (WG) {
    const int wave = threadIdx.x >> 6;
    __syncthreads();                                   // the slots may still be read from the sum before
    if ((threadIdx.x & 63) == 0) red[wave] = v;
    __syncthreads();
    v = 0.0f;
#pragma unroll
    for (int w = 0; w < LN_WAVES; ++w) v += red[w];
  }
  return v;
}

template <int TRIPS, bool WG>
__global__ __launch_bounds__(LN_THREADS) void norm_fwd_kernel(const NormParams p, int vec_ok) {
  constexpr int VEC = 4;
  constexpr int OWNERS = WG ? LN_THREADS : WAVE;       // threads that share a row
  __shared__ float red[LN_WAVES];
  const int wave = threadIdx.x >> 6, lane = WG ? (int)threadIdx.x : (int)(threadIdx.x & 63);
  const int row = WG ? (int)blockIdx.x : (int)(blockIdx.x * LN_WAVES + wave);
  if (row >= p.rows) return;                           // whole workgroups in WG mode
  const int H = p.hidden;
  const size_t base = (size_t)row * H;
  const bool vok = vec_ok != 0;
  float v[TRIPS][VEC], r[TRIPS][VEC];
  float sum = 0.0f;
#pragma unroll
  for (int k = 0; k < TRIPS; ++k) {
    const int col = (k * OWNERS + lane) * VEC;
    load_cols<VEC>(p.x, p.x_dtype, base, col, H, vok, v[k]);
    if (p.res) {
      load_cols<VEC>(p.res, p.res_dtype, base, col, H, vok, r[k]);
      if (p.prenorm) {
#pragma unroll
        for (int i = 0; i < VEC; ++i) v[k][i] += r[k][i];
      }
    }
#pragma unroll
    for (int i = 0; i < VEC; ++i) sum += v[k][i];
    if (p.res_out) store_cols<VEC>(p.res_out, p.res_out_dtype, base, col, H, vok, v[k]);
  }
  const float inv_h = 1.0f / (float)H;
  float mean = 0.0f;
  if (!p.is_rms) mean = row_sum<WG>(sum, red) * inv_h;
  float sq = 0.0f;
#pragma unroll
  for (int k = 0; k < TRIPS; ++k) {
    const int col = (k * OWNERS + lane) * VEC;
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      const float c = (col + i < H) ? v[k][i] - mean : 0.0f;
      sq = __builtin_fmaf(c, c, sq);
    }
  }
  const float rstd = 1.0f / sqrtf(row_sum<WG>(sq, red) * inv_h + p.eps);
  if (lane == 0) {
    if (p.mean) p.mean[row] = mean;
    if (p.rstd) p.rstd[row] = rstd;
  }
#pragma unroll
  for (int k = 0; k < TRIPS; ++k) {
    const int col = (k * OWNERS + lane) * VEC;
    if (col >= H) continue;
    float wv[VEC], bv[VEC], out[VEC];
    load_cols<VEC>(p.w, SSM_F32, 0, col, H, vok, wv);
    if (p.b) load_cols<VEC>(p.b, SSM_F32, 0, col, H, vok, bv);
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      float o = (v[k][i] - mean) * rstd * wv[i];
      if (p.b) o += bv[i];
      if (p.res && !p.prenorm) o += r[k][i];
      out[i] = o;
    }
    store_cols<VEC>(p.y, p.x_dtype, base, col, H, vok, out);
  }
}

// The one-wavefront-per-row kernel with the element types known at compile time (XT: x and y; RT: residual
// and residual_out) for rows of a multiple of four columns with 16-byte aligned tensors.  Every read is
// unconditional - column indices are clamped into the row, an absent residual or bias reads a stand-in of
// the same type whose value is dropped - so a wavefront's reads are in flight together instead of one
// behind the other, which is what a call on a handful of rows (a decoding step) waits for.
// Large calls (NORM_CACHED) read the residual past the caches.
template <typename T, int VEC>
__device__ __forceinline__ void ld_pack(const void *p, size_t i, float (&v)[VEC]) {
  const Pack<T, VEC> raw = *reinterpret_cast<const Pack<T, VEC> *>(reinterpret_cast<const T *>(p) + i);
#pragma unroll
  for (int j = 0; j < VEC; ++j) v[j] = to_f32(raw.v[j]);
}
template <typename T, int VEC>
__device__ __forceinline__ void st_pack(void *p, size_t i, const float (&v)[VEC]) {
  Pack<T, VEC> raw;
#pragma unroll
  for (int j = 0; j < VEC; ++j) raw.v[j] = from_f32<T>(v[j]);
  *reinterpret_cast<Pack<T, VEC> *>(reinterpret_cast<T *>(p) + i) = raw;
}

template <typename T, int VEC>
__device__ __forceinline__ void ld_once(const void *p, size_t i, float (&v)[VEC]) {
  const Pack<T, VEC> raw = load_once(reinterpret_cast<const Pack<T, VEC> *>(reinterpret_cast<const T *>(p) + i));
#pragma unroll
  for (int j = 0; j < VEC; ++j) v[j] = to_f32(raw.v[j]);
}
template <int TRIPS, bool WG, typename XT, typename RT, bool PAST>
__global__ __launch_bounds__(LN_THREADS) void norm_fwd_typed_kernel(const NormParams p) {
  constexpr int VEC = 4;
  constexpr int OWNERS = WG ? LN_THREADS : WAVE;       // threads that share a row
  __shared__ float red[LN_WAVES];
  const int wave = threadIdx.x >> 6, lane = WG ? (int)threadIdx.x : (int)(threadIdx.x & 63);
  const int row = WG ? (int)blockIdx.x : (int)(blockIdx.x * LN_WAVES + wave);
  if (row >= p.rows) return;                           // whole workgroups in WG mode
  const int H = p.hidden;
  const size_t base = (size_t)row * H;
  const bool has_res = p.res != nullptr, has_b = p.b != nullptr;
  // stand-ins of the right element type: residual_out (type RT) or, without one, x (then RT = XT)
  const void *resp = has_res ? p.res : (p.res_out ? (const void *)p.res_out : p.x);
  const float *bp = has_b ? p.b : p.w;
  float v[TRIPS][VEC], r[TRIPS][VEC];
  float sum = 0.0f;
#pragma unroll
  for (int k = 0; k < TRIPS; ++k) {
    const int colc = min((k * OWNERS + lane) * VEC, H - VEC);
    ld_pack<XT, VEC>(p.x, base + colc, v[k]);
  }
  if (has_res) {                 // one test in front of all of a row's residual reads, none between them
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) {
      const int colc = min((k * OWNERS + lane) * VEC, H - VEC);
      if constexpr (PAST) ld_once<RT, VEC>(resp, base + colc, r[k]);
      else ld_pack<RT, VEC>(resp, base + colc, r[k]);
    }
  } else {
#pragma unroll
    for (int k = 0; k < TRIPS; ++k)
#pragma unroll
      for (int i = 0; i < VEC; ++i) r[k][i] = 0.0f;
  }
#pragma unroll
  for (int k = 0; k < TRIPS; ++k) {
    const int col = (k * OWNERS + lane) * VEC;
    const bool live = col < H;
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      if (p.prenorm) v[k][i] += r[k][i];
      if (!live) v[k][i] = 0.0f;
      sum += v[k][i];
    }
    if (p.res_out && live) st_pack<RT, VEC>(p.res_out, base + col, v[k]);
  }
  float wv[TRIPS][VEC], bv[TRIPS][VEC];
#pragma unroll
  for (int k = 0; k < TRIPS; ++k) {
    const int colc = min((k * OWNERS + lane) * VEC, H - VEC);
    ld_pack<float, VEC>(p.w, colc, wv[k]);
    ld_pack<float, VEC>(bp, colc, bv[k]);
  }
  const float inv_h = 1.0f / (float)H;
  float mean = 0.0f;
  if (!p.is_rms) mean = row_sum<WG>(sum, red) * inv_h;
  float sq = 0.0f;
#pragma unroll
  for (int k = 0; k < TRIPS; ++k) {
    const bool live = (k * OWNERS + lane) * VEC < H;
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      const float c = live ? v[k][i] - mean : 0.0f;
      sq = __builtin_fmaf(c, c, sq);
    }
  }
  const float rstd = 1.0f / sqrtf(row_sum<WG>(sq, red) * inv_h + p.eps);
  if (lane == 0) {
    if (p.mean) p.mean[row] = mean;
    if (p.rstd) p.rstd[row] = rstd;
  }
#pragma unroll
  for (int k = 0; k < TRIPS; ++k) {
    const int col = (k * OWNERS + lane) * VEC;
    float out[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      float o = (v[k][i] - mean) * rstd * wv[k][i];
      if (has_b) o += bv[k][i];
      if (has_res && !p.prenorm) o += r[k][i];
      out[i] = o;
    }
    if (col < H) st_pack<XT, VEC>(p.y, base + col, out);
  }
}

template <typename XT, typename RT, bool PAST>
static void launch_norm_fwd_typed_as(const NormParams &p, int per_lane, unsigned grid, hipStream_t s) {
  const dim3 b(LN_THREADS);
  if (per_lane <= 4) hipLaunchKernelGGL((norm_fwd_typed_kernel<1, false, XT, RT, PAST>), dim3(grid), b, 0, s, p);
  else if (per_lane <= 8) hipLaunchKernelGGL((norm_fwd_typed_kernel<2, false, XT, RT, PAST>), dim3(grid), b, 0, s, p);
  else if (per_lane <= 12) hipLaunchKernelGGL((norm_fwd_typed_kernel<3, false, XT, RT, PAST>), dim3(grid), b, 0, s, p);
  else if (per_lane <= 16) hipLaunchKernelGGL((norm_fwd_typed_kernel<4, false, XT, RT, PAST>), dim3(grid), b, 0, s, p);
  // (a trip that holds no column still reads one: rows of 1280, 1536 and 1792 columns get trip counts of their own)
  else if (per_lane <= 20) hipLaunchKernelGGL((norm_fwd_typed_kernel<5, false, XT, RT, PAST>), dim3(grid), b, 0, s, p);
  else if (per_lane <= 24) hipLaunchKernelGGL((norm_fwd_typed_kernel<6, false, XT, RT, PAST>), dim3(grid), b, 0, s, p);
  else if (per_lane <= 28) hipLaunchKernelGGL((norm_fwd_typed_kernel<7, false, XT, RT, PAST>), dim3(grid), b, 0, s, p);
  else if (per_lane <= 32) hipLaunchKernelGGL((norm_fwd_typed_kernel<8, false, XT, RT, PAST>), dim3(grid), b, 0, s, p);
  else if (p.hidden <= 4096) hipLaunchKernelGGL((norm_fwd_typed_kernel<4, true, XT, RT, PAST>), dim3(p.rows), b, 0, s, p);
  else if (p.hidden <= 5120) hipLaunchKernelGGL((norm_fwd_typed_kernel<5, true, XT, RT, PAST>), dim3(p.rows), b, 0, s, p);
  else if (p.hidden <= 6144) hipLaunchKernelGGL((norm_fwd_typed_kernel<6, true, XT, RT, PAST>), dim3(p.rows), b, 0, s, p);
  else if (p.hidden <= 8192) hipLaunchKernelGGL((norm_fwd_typed_kernel<8, true, XT, RT, PAST>), dim3(p.rows), b, 0, s, p);
  else hipLaunchKernelGGL((norm_fwd_typed_kernel<16, true, XT, RT, PAST>), dim3(p.rows), b, 0, s, p);
}
template <typename XT, typename RT>
static void launch_norm_fwd_typed(const NormParams &p, int per_lane, unsigned grid, hipStream_t s) {
  if (p.past_caches && p.res) launch_norm_fwd_typed_as<XT, RT, true>(p, per_lane, grid, s);
  else launch_norm_fwd_typed_as<XT, RT, false>(p, per_lane, grid, s);
}

// True when the call was taken by a typed kernel.
static bool norm_fwd_typed(const NormParams &p, int per_lane, unsigned grid, hipStream_t s) {
  if (p.hidden > 16384 || p.hidden < 4) return false;
  // residual and residual_out must agree on one type, float32 or that of x
  int rt = -1;
  if (p.res) rt = p.res_dtype;
  if (p.res_out) {
    if (rt >= 0 && p.res_out_dtype != rt) return false;
    rt = p.res_out_dtype;
  }
  if (rt < 0) rt = p.x_dtype;
  if (rt != SSM_F32 && rt != p.x_dtype) return false;
  const bool rf = rt == SSM_F32;
  if (p.x_dtype == SSM_BF16) rf ? launch_norm_fwd_typed<bf16_t, float>(p, per_lane, grid, s) : launch_norm_fwd_typed<bf16_t, bf16_t>(p, per_lane, grid, s);
  else if (p.x_dtype == SSM_F16) rf ? launch_norm_fwd_typed<f16_t, float>(p, per_lane, grid, s) : launch_norm_fwd_typed<f16_t, f16_t>(p, per_lane, grid, s);
  else launch_norm_fwd_typed<float, float>(p, per_lane, grid, s);
  return true;
}

// Any hidden size: three sweeps over the row from memory.
__global__ __launch_bounds__(LN_THREADS) void norm_fwd_long_kernel(const NormParams p) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row = blockIdx.x * LN_WAVES + wave;
  if (row >= p.rows) return;
  const int H = p.hidden;
  const size_t base = (size_t)row * H;
  auto val = [&](int c) -> float {
    float v = load_as_f32(p.x, p.x_dtype, base + c);
    if (p.res && p.prenorm) v += load_as_f32(p.res, p.res_dtype, base + c);
    return v;
  };
  float sum = 0.0f;
  for (int c = lane; c < H; c += WAVE) sum += val(c);
  const float inv_h = 1.0f / (float)H;
  const float mean = p.is_rms ? 0.0f : wave_sum(sum) * inv_h;
  float sq = 0.0f;
  for (int c = lane; c < H; c += WAVE) {
    const float d = val(c) - mean;
    sq = __builtin_fmaf(d, d, sq);
  }
  const float rstd = 1.0f / sqrtf(wave_sum(sq) * inv_h + p.eps);
  if (lane == 0) {
    if (p.mean) p.mean[row] = mean;
    if (p.rstd) p.rstd[row] = rstd;
  }
  for (int c = lane; c < H; c += WAVE) {
    const float v = val(c);
    if (p.res_out) store_f32_as(p.res_out, p.res_out_dtype, base + c, v);
    float o = (v - mean) * rstd * p.w[c];
    if (p.b) o += p.b[c];
    if (p.res && !p.prenorm) o += load_as_f32(p.res, p.res_dtype, base + c);
    store_f32_as(p.y, p.x_dtype, base + c, o);
  }
}

// ----------------------------------------------------------------- backward

// The words of a pack as they stand here: what is made of them further on is made there, not kept from before.
template <typename T, int VEC>
__device__ __forceinline__ void pin_pack(Pack<T, VEC> &v) {
  static_assert(sizeof(v) % 4 == 0);
  unsigned w[sizeof(v) / 4];
  __builtin_memcpy(w, &v, sizeof(v));
#pragma unroll
  for (unsigned &x : w) asm volatile("" : "+v"(x));
  __builtin_memcpy(&v, w, sizeof(v));
}

// Each wave handles rows wave_global, wave_global + nwaves, ...; columns are
// owned by (lane, trip) exactly as in the forward kernel.
// XT = void: element types looked up at run time.  Otherwise x, dy, dx have type XT, residual and dresidual
// type RT, rows are a multiple of four columns long and aligned, and all reads of a row are unconditional
// (clamped columns, a stand-in for an absent residual), i.e. in flight together.
//
// GRO (typed form): the gradient that arrives through residual_out = x (+ residual), of type RT, is added to dx and
// dresidual while they are in registers.  The pass is bound by memory; added in launches of its own, that gradient
// cost a (16 x 2048 x 768) bf16 step with a float32 residual 106 us beside the 66 of this kernel.
//
// Bound by memory: 16 x 2048 x 768, bf16 with a float32 residual and gradient through it, 400 MB, 74 us.  Before, 98 with
// 50 for the forward's 300 MB, now 63: what the backward no longer leaves in the caches the forward has to write out itself;
// together they are at the rate of a large copy.
// Rows of 16-bit elements alone (no gradient through residual_out) put too few bytes in flight: they ask for the next row before
// this one is worked on (a float32 residual beside them would spill), read no residual where there is none, and
// store the sums in vectors, those of the bias only where there is one.  8192 x 1536 bf16 24.0 -> 19.0 us, 2048 x 4096 19.8 -> 13.8,
// 1707 x 4864 22.1 -> 14.4, 1600 x 8192 35.2 -> 29.3, 2000 x 704 6.7 -> 5.7 (the reads ahead alone: 21.5, 17.3, 18.6, 33.4, 6.4).
// The grid is held to the workgroups that the registers let onto the chip at once (with four to a CU for any width, the
// fourth of three ran alone), and the registers are few: words as they came, 32-bit offsets from a scalar row, no value kept
// that can be formed again.  Forward and backward, 4096 rows of 4096 columns 107 -> 95 us, of 8192 223 -> 197.
constexpr int norm_bwd_resident(int trips, bool gro) {                   // workgroups to a CU of a typed kernel
  return trips <= 2 ? 4 : trips == 3 ? (gro ? 3 : 4) : trips == 4 ? (gro ? 2 : 3) : trips == 5 ? 2 : trips == 6 ? (gro ? 1 : 2) : 1;
}
template <int TRIPS, bool WG, typename XT = void, typename RT = void, bool GRO = false>
__global__ __launch_bounds__(LN_THREADS) __attribute__((amdgpu_waves_per_eu(std::is_void<XT>::value ? 1 : norm_bwd_resident(TRIPS, GRO))))
void norm_bwd_kernel(const NormParams p, int vec_ok) {
  constexpr int VEC = 4;
  constexpr bool TYPED = !std::is_void<XT>::value;
  using xt = typename std::conditional<TYPED, XT, float>::type;
  using rt = typename std::conditional<TYPED, RT, float>::type;
  constexpr int OWNERS = WG ? LN_THREADS : WAVE;       // threads that share a row
  __shared__ float red[LN_WAVES];
  const int wave = wave_id_uniform(), lane = WG ? (int)threadIdx.x : (int)(threadIdx.x & 63);
  const int nwaves = WG ? (int)gridDim.x : (int)(gridDim.x * LN_WAVES);      // row owners in the grid
  const int gw = WG ? (int)blockIdx.x : (int)(blockIdx.x * LN_WAVES + wave);
  const int H = p.hidden;
  const bool vok = vec_ok != 0;
  const float inv_h = 1.0f / (float)H;
  float dw[TRIPS][VEC], db[TRIPS][VEC], wv[TRIPS][VEC];
#pragma unroll
  for (int k = 0; k < TRIPS; ++k) {
    const int col = (k * OWNERS + lane) * VEC;
    if constexpr (TYPED) ld_pack<float, VEC>(p.w, min(col, H - VEC), wv[k]);
    else load_cols<VEC>(p.w, SSM_F32, 0, col, H, vok, wv[k]);
#pragma unroll
    for (int i = 0; i < VEC; ++i) dw[k][i] = db[k][i] = 0.0f;
  }
  const bool has_add = p.res && p.prenorm;
  // typed reads of a residual that is absent (or not added: post-norm) go to memory of the same element type
  // and extent and are dropped: the residual itself if there is one, else dresidual, else gro or x (then RT = XT)
  const void *resp = p.res ? p.res : (p.dres ? (const void *)p.dres : (GRO ? p.gro : p.x));
  const float *meanp = p.is_rms ? p.rstd : p.mean;
  struct Raw {
    Pack<xt, VEC> x[TRIPS], dy[TRIPS];
    Pack<rt, VEC> r[TRIPS], g[TRIPS];
    float mean, rstd;
  };
  const auto request = [&](int row, Raw &o) {
    const size_t base = (size_t)row * H;
    o.mean = meanp[row];
    o.rstd = p.rstd[row];
    if constexpr (TYPED) {
      const auto read = [&](auto past) {
        const auto get = [&](const auto *q) {
          if constexpr (past.value) return load_once(q);
          else return *q;
        };
        const auto column = [&](int k) { return (unsigned)min((k * OWNERS + lane) * VEC, H - VEC); };
#pragma unroll
        for (int k = 0; k < TRIPS; ++k) {
          o.x[k] = get(at_bytes<const Pack<xt, VEC>>(reinterpret_cast<const xt *>(p.x) + base, column(k) * (unsigned)sizeof(xt)));
          o.dy[k] = get(at_bytes<const Pack<xt, VEC>>(reinterpret_cast<const xt *>(p.dy) + base, column(k) * (unsigned)sizeof(xt)));
          if constexpr (GRO) {
            o.r[k] = get(at_bytes<const Pack<rt, VEC>>(reinterpret_cast<const rt *>(resp) + base, column(k) * (unsigned)sizeof(rt)));
            o.g[k] = get(at_bytes<const Pack<rt, VEC>>(reinterpret_cast<const rt *>(p.gro) + base, column(k) * (unsigned)sizeof(rt)));
          }
        }
        if (!GRO && has_add) {                                 // one test in front of all of them
#pragma unroll
          for (int k = 0; k < TRIPS; ++k)
            o.r[k] = get(at_bytes<const Pack<rt, VEC>>(reinterpret_cast<const rt *>(resp) + base, column(k) * (unsigned)sizeof(rt)));
        }
      };
      if (p.past_caches) read(std::true_type{});
      else read(std::false_type{});
    }
  };
  constexpr bool AHEAD = TYPED && !GRO && sizeof(rt) == 2;
  Raw cur, next;
  if (AHEAD && gw < p.rows) request(gw, cur);
  for (int row = gw; row < p.rows; row += nwaves) {
    const size_t base = (size_t)row * H;
    if (!AHEAD) request(row, cur);
    else if (row + nwaves < p.rows) request(row + nwaves, next);
    const float mean = p.is_rms ? 0.0f : cur.mean, rstd = cur.rstd;
    float xh[TRIPS][VEC], g[TRIPS][VEC], dyv[TRIPS][VEC], gin[TRIPS][VEC];
    float s1 = 0.0f, s2 = 0.0f;     // sum g*xhat, sum g
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) {
      const int col = (k * OWNERS + lane) * VEC;
      float v[VEC];
      if constexpr (TYPED) {
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
          v[i] = to_f32(cur.x[k].v[i]);
          if (has_add) v[i] += to_f32(cur.r[k].v[i]);
          dyv[k][i] = to_f32(cur.dy[k].v[i]);
        }
      } else {
        load_cols<VEC>(p.x, p.x_dtype, base, col, H, vok, v);
        if (has_add) {
          float r[VEC];
          load_cols<VEC>(p.res, p.res_dtype, base, col, H, vok, r);
#pragma unroll
          for (int i = 0; i < VEC; ++i) v[i] += r[i];
        }
        load_cols<VEC>(p.dy, p.x_dtype, base, col, H, vok, dyv[k]);
      }
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        const bool in = col + i < H;
        xh[k][i] = in ? (v[i] - mean) * rstd : 0.0f;
        g[k][i] = in ? dyv[k][i] * wv[k][i] : 0.0f;
        s1 = __builtin_fmaf(g[k][i], xh[k][i], s1);
        s2 += g[k][i];
        dw[k][i] = __builtin_fmaf(dyv[k][i], xh[k][i], dw[k][i]);
        db[k][i] += dyv[k][i];
      }
    }
    const float c1 = row_sum<WG>(s1, red) * inv_h;
    const float c2 = p.is_rms ? 0.0f : row_sum<WG>(s2, red) * inv_h;
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) {
      const int col = (k * OWNERS + lane) * VEC;
      if (col >= H) continue;
      float dxv[VEC];
      if constexpr (TYPED) {
        pin_pack(cur.dy[k]);
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
          dyv[k][i] = to_f32(cur.dy[k].v[i]);
          g[k][i] = dyv[k][i] * wv[k][i];
          if constexpr (GRO) gin[k][i] = to_f32(cur.g[k].v[i]);
        }
      }
#pragma unroll
      for (int i = 0; i < VEC; ++i) dxv[i] = (g[k][i] - c2 - xh[k][i] * c1) * rstd;
      if constexpr (!TYPED) {
        if (p.gro) load_cols<VEC>(p.gro, p.gro_dtype, base, col, H, vok, gin[k]);
      }
      if (TYPED ? GRO : p.gro != nullptr) {
#pragma unroll
        for (int i = 0; i < VEC; ++i) dxv[i] += gin[k][i];
      }
      if constexpr (TYPED) {
        st_pack<xt, VEC>(reinterpret_cast<xt *>(p.dx) + base, (unsigned)col, dxv);
        if (p.dres) st_pack<rt, VEC>(reinterpret_cast<rt *>(p.dres) + base, (unsigned)col, p.prenorm ? dxv : dyv[k]);
      } else {
        store_cols<VEC>(p.dx, p.x_dtype, base, col, H, vok, dxv);
        if (p.dres) store_cols<VEC>(p.dres, p.res_dtype, base, col, H, vok, p.prenorm ? dxv : dyv[k]);
      }
    }
    if (AHEAD) cur = next;
  }
  typedef float four_t __attribute__((ext_vector_type(4), aligned(4)));
  const auto put = [&](float *to, int col, const float (&v)[VEC]) {
    if constexpr (TYPED) {
      if (col < H) *reinterpret_cast<four_t *>(to + col) = four_t{v[0], v[1], v[2], v[3]};
    } else {
#pragma unroll
      for (int i = 0; i < VEC; ++i)
        if (col + i < H) to[col + i] = v[i];
    }
  };
  if constexpr (WG) {                                  // every thread owns its columns: the partial is complete
    float *pw = p.partial + (size_t)blockIdx.x * 2 * H;
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) put(pw, (k * OWNERS + lane) * VEC, dw[k]);
    if (p.has_db) {
#pragma unroll
      for (int k = 0; k < TRIPS; ++k) put(pw + H, (k * OWNERS + lane) * VEC, db[k]);
    }
    return;
  }
  // one partial per workgroup: waves 1.. hand their column sums to wave 0 through LDS (fixed order)
  __shared__ float wsum[LN_WAVES - 1][2][WG ? 1 : TRIPS * WAVE * VEC];
  if (wave > 0) {
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) {
      const int col = (k * OWNERS + lane) * VEC;
      *reinterpret_cast<float4 *>(&wsum[wave - 1][0][col]) = make_float4(dw[k][0], dw[k][1], dw[k][2], dw[k][3]);
      *reinterpret_cast<float4 *>(&wsum[wave - 1][1][col]) = make_float4(db[k][0], db[k][1], db[k][2], db[k][3]);
    }
  }
  __syncthreads();
  if (wave == 0) {
    float *pw = p.partial + (size_t)blockIdx.x * 2 * H;
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) {
      const int col = (k * OWNERS + lane) * VEC;
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
#pragma unroll
        for (int w = 0; w < LN_WAVES - 1; ++w) {
          dw[k][i] += wsum[w][0][col + i];
          db[k][i] += wsum[w][1][col + i];
        }
      }
      put(pw, col, dw[k]);
      if (p.has_db) put(pw + H, col, db[k]);
    }
  }
}

__global__ __launch_bounds__(LN_THREADS) void norm_bwd_long_kernel(const NormParams p) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nwaves = gridDim.x * LN_WAVES;
  const int gw = blockIdx.x * LN_WAVES + wave;
  const int H = p.hidden;
  const float inv_h = 1.0f / (float)H;
  float *pw = p.partial + (size_t)gw * 2 * H;
  for (int c = lane; c < 2 * H; c += WAVE) pw[c] = 0.0f;
  for (int row = gw; row < p.rows; row += nwaves) {
    const size_t base = (size_t)row * H;
    const float mean = p.is_rms ? 0.0f : p.mean[row];
    const float rstd = p.rstd[row];
    auto xhat = [&](int c) -> float {
      float v = load_as_f32(p.x, p.x_dtype, base + c);
      if (p.res && p.prenorm) v += load_as_f32(p.res, p.res_dtype, base + c);
      return (v - mean) * rstd;
    };
    float s1 = 0.0f, s2 = 0.0f;
    for (int c = lane; c < H; c += WAVE) {
      const float dy = load_as_f32(p.dy, p.x_dtype, base + c);
      const float gg = dy * p.w[c];
      const float xh = xhat(c);
      s1 = __builtin_fmaf(gg, xh, s1);
      s2 += gg;
      pw[c] = __builtin_fmaf(dy, xh, pw[c]);
      pw[H + c] += dy;
    }
    const float c1 = wave_sum(s1) * inv_h;
    const float c2 = p.is_rms ? 0.0f : wave_sum(s2) * inv_h;
    for (int c = lane; c < H; c += WAVE) {
      const float dy = load_as_f32(p.dy, p.x_dtype, base + c);
      float dxv = (dy * p.w[c] - c2 - xhat(c) * c1) * rstd;
      if (p.gro) dxv += load_as_f32(p.gro, p.gro_dtype, base + c);
      store_f32_as(p.dx, p.x_dtype, base + c, dxv);
      if (p.dres) store_f32_as(p.dres, p.res_dtype, base + c, p.prenorm ? dxv : dy);
    }
  }
}

// dw[c] = sum_w partial[w][0][c], db[c] = sum_w partial[w][1][c].  A workgroup takes 16 columns; its 1024
// threads are 16 columns x 64 slices of the partials, summed in a fixed order (slice by slice, then over slices).
// Bound by latency: few workgroups (hidden / 16) that each walk up to 1024 partials, so the walk is cut to at most
// two rounds of reads, and the second half of a partial is left alone where there is no bias.
// 1024 partials of 768 columns 6.5 -> 4.8 us, of 1536 6.8 -> 4.3 us (before: 256 threads, 16 slices, both halves read).
constexpr int FOLD_COLS = 16, FOLD_THREADS = 1024, FOLD_SLICES = FOLD_THREADS / FOLD_COLS;

template <bool BIAS>
__global__ __launch_bounds__(FOLD_THREADS) void norm_bwd_fold_kernel(const float *partial, float *dw, float *db,
                                                                     int nparts, int hidden) {
  constexpr int SUMS = BIAS ? 2 : 1;
  __shared__ float part[SUMS][FOLD_SLICES][FOLD_COLS];
  const int cl = threadIdx.x % FOLD_COLS, sl = threadIdx.x / FOLD_COLS;
  const int c = blockIdx.x * FOLD_COLS + cl;
  float sum[SUMS] = {};
  if (c < hidden) {
    // eight partials at a time: their reads are in flight together, the additions keep their order
    int w = sl;
    for (; w + 7 * FOLD_SLICES < nparts; w += 8 * FOLD_SLICES) {
      float v[SUMS][8];
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int q = 0; q < SUMS; ++q) v[q][k] = partial[((size_t)(w + k * FOLD_SLICES) * 2 + q) * hidden + c];
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int q = 0; q < SUMS; ++q) sum[q] += v[q][k];
    }
    for (; w < nparts; w += FOLD_SLICES)
#pragma unroll
      for (int q = 0; q < SUMS; ++q) sum[q] += partial[((size_t)w * 2 + q) * hidden + c];
  }
#pragma unroll
  for (int q = 0; q < SUMS; ++q) part[q][sl][cl] = sum[q];
  __syncthreads();
  // the first wave: four lanes a column, a quarter of the slices each
  if (threadIdx.x < WAVE) {
#pragma unroll
    for (int q = 0; q < SUMS; ++q) {
      float t = 0.0f;
#pragma unroll
      for (int j = 0; j < FOLD_SLICES / 4; ++j) t += part[q][4 * j + sl][cl];
      t += __shfl_xor(t, FOLD_COLS, WAVE);
      t += __shfl_xor(t, 2 * FOLD_COLS, WAVE);
      if (sl == 0 && c < hidden) (q ? db : dw)[c] = t;
    }
  }
}

static int norm_bwd_grid(int rows) {
  // persistent: at most 4 workgroups per CU on a 256-CU part, never more waves than rows
  const int want = (rows + LN_WAVES - 1) / LN_WAVES;
  return want < 1024 ? (want < 1 ? 1 : want) : 1024;
}

static int norm_check(const char *who, const void *x, const float *w, const void *y, int rows, int hidden,
                      int x_dtype, const void *res, int res_dtype) {
  SSM_REQUIRE(x && w && y, SSM_ERR_NULL_POINTER, "%s: x, weight and output are required", who);
  SSM_REQUIRE(rows > 0 && hidden > 0, SSM_ERR_BAD_SHAPE, "%s: rows=%d hidden=%d must be positive", who, rows, hidden);
  SSM_REQUIRE(valid_dtype(x_dtype) && (!res || valid_dtype(res_dtype)), SSM_ERR_BAD_DTYPE,
              "%s: x_dtype=%d residual_dtype=%d", who, x_dtype, res_dtype);
  SSM_REQUIRE((size_t)rows * hidden < ((size_t)1 << 40), SSM_ERR_TOO_LARGE, "%s: tensor too large", who);
  return SSM_OK;
}

}  // namespace ssm

extern "C" int ssm_norm_fwd(const ssm_norm_fwd_args *a, void *hip_stream) {
  using namespace ssm;
  SSM_REQUIRE(a != nullptr, SSM_ERR_NULL_POINTER, "ssm_norm_fwd: args is NULL");
  int rc = norm_check("ssm_norm_fwd", a->x, a->weight, a->y, a->rows, a->hidden, a->x_dtype, a->residual,
                      a->residual_dtype);
  if (rc != SSM_OK) return rc;
  if (a->residual_out)
    SSM_REQUIRE(valid_dtype(a->residual_out_dtype), SSM_ERR_BAD_DTYPE, "ssm_norm_fwd: residual_out_dtype=%d",
                a->residual_out_dtype);
  NormParams p{};
  p.x = a->x; p.res = a->residual; p.w = a->weight; p.b = a->bias; p.y = a->y; p.res_out = a->residual_out;
  p.mean = a->mean; p.rstd = a->rstd;
  p.rows = a->rows; p.hidden = a->hidden;
  p.x_dtype = a->x_dtype; p.res_dtype = a->residual_dtype; p.res_out_dtype = a->residual_out_dtype;
  const size_t each = 2 * (a->x_dtype == SSM_F32 ? 4 : 2) + (a->residual ? (a->residual_dtype == SSM_F32 ? 4 : 2) : 0) +
                      (a->residual_out ? (a->residual_out_dtype == SSM_F32 ? 4 : 2) : 0);        // bytes moved
  p.past_caches = a->rstd ? (size_t)a->rows * a->hidden > NORM_CACHED : (size_t)a->rows * a->hidden * each > NORM_CACHED_BYTES;
  p.is_rms = a->is_rms ? 1 : 0; p.prenorm = a->prenorm ? 1 : 0; p.eps = a->eps;
  const int vec_ok = a->hidden % 4 == 0 && aligned_to(a->x, 16) && aligned_to(a->y, 16) &&
                     aligned_to(a->weight, 16) && (!a->bias || aligned_to(a->bias, 16)) &&
                     (!a->residual || aligned_to(a->residual, 16)) &&
                     (!a->residual_out || aligned_to(a->residual_out, 16));
  hipStream_t s = reinterpret_cast<hipStream_t>(hip_stream);
  const unsigned grid = (unsigned)((a->rows + LN_WAVES - 1) / LN_WAVES);
  const int per_lane = (a->hidden + WAVE - 1) / WAVE;
  if (vec_ok && norm_fwd_typed(p, per_lane, grid, s)) {
    SSM_CHECK_LAUNCH("ssm_norm_fwd");
    return SSM_OK;
  }
  if (per_lane <= 4) hipLaunchKernelGGL((norm_fwd_kernel<1, false>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (per_lane <= 8) hipLaunchKernelGGL((norm_fwd_kernel<2, false>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (per_lane <= 12) hipLaunchKernelGGL((norm_fwd_kernel<3, false>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (per_lane <= 16) hipLaunchKernelGGL((norm_fwd_kernel<4, false>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (per_lane <= 32) hipLaunchKernelGGL((norm_fwd_kernel<8, false>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (a->hidden <= 4096) hipLaunchKernelGGL((norm_fwd_kernel<4, true>), dim3(a->rows), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (a->hidden <= 8192) hipLaunchKernelGGL((norm_fwd_kernel<8, true>), dim3(a->rows), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (a->hidden <= 16384) hipLaunchKernelGGL((norm_fwd_kernel<16, true>), dim3(a->rows), dim3(LN_THREADS), 0, s, p, vec_ok);
  else hipLaunchKernelGGL(norm_fwd_long_kernel, dim3(grid), dim3(LN_THREADS), 0, s, p);
  SSM_CHECK_LAUNCH("ssm_norm_fwd");
  return SSM_OK;
}

namespace ssm {
// The typed kernels; the workgroups launched, at most `grid`.
template <int TRIPS, bool WG, typename XT, typename RT, bool GRO>
static int launch_norm_bwd_trips(const NormParams &p, int grid, hipStream_t s) {
  const int resident = 256 * norm_bwd_resident(TRIPS, GRO), g = grid < resident ? grid : resident;
  hipLaunchKernelGGL((norm_bwd_kernel<TRIPS, WG, XT, RT, GRO>), dim3(g), dim3(LN_THREADS), 0, s, p, 1);
  return g;
}
template <typename XT, typename RT, bool GRO>
static int launch_norm_bwd_gro(const NormParams &p, int hidden, int grid, hipStream_t s) {
  const int per_lane = (hidden + WAVE - 1) / WAVE;
  if (per_lane <= 4) return launch_norm_bwd_trips<1, false, XT, RT, GRO>(p, grid, s);
  if (per_lane <= 8) return launch_norm_bwd_trips<2, false, XT, RT, GRO>(p, grid, s);
  if (per_lane <= 12) return launch_norm_bwd_trips<3, false, XT, RT, GRO>(p, grid, s);
  if (hidden <= 1024) return launch_norm_bwd_trips<1, true, XT, RT, GRO>(p, grid, s);
  if (hidden <= 2048) return launch_norm_bwd_trips<2, true, XT, RT, GRO>(p, grid, s);
  // a thread's registers grow with the trips it is compiled for: the widths of common models (2560, 5120) get
  // their own count rather than the next power of two
  if (hidden <= 3072) return launch_norm_bwd_trips<3, true, XT, RT, GRO>(p, grid, s);
  if (hidden <= 4096) return launch_norm_bwd_trips<4, true, XT, RT, GRO>(p, grid, s);
  if (hidden <= 5120) return launch_norm_bwd_trips<5, true, XT, RT, GRO>(p, grid, s);
  if (hidden <= 6144) return launch_norm_bwd_trips<6, true, XT, RT, GRO>(p, grid, s);
  return launch_norm_bwd_trips<8, true, XT, RT, GRO>(p, grid, s);
}
template <typename XT, typename RT>
static int launch_norm_bwd_typed(const NormParams &p, int hidden, int grid, hipStream_t s) {
  return p.gro ? launch_norm_bwd_gro<XT, RT, true>(p, hidden, grid, s) : launch_norm_bwd_gro<XT, RT, false>(p, hidden, grid, s);
}
}  // namespace ssm

extern "C" size_t ssm_norm_bwd_workspace_bytes(int rows, int hidden) {
  if (rows <= 0 || hidden <= 0) return 0;
  return (size_t)ssm::norm_bwd_grid(rows) * ssm::LN_WAVES * 2 * (size_t)hidden * sizeof(float);
}

namespace ssm {

// Partial column sums one call writes before the fold reads them: one per workgroup, or one per wave for rows
// beyond 8192 columns.
static size_t norm_bwd_partials(int rows, int hidden) {
  const size_t grid = (size_t)norm_bwd_grid(rows);
  return hidden <= 8192 ? grid : grid * LN_WAVES;
}

static int norm_bwd_check(const char *who, const ssm_norm_bwd_args *a) {
  SSM_REQUIRE(a != nullptr, SSM_ERR_NULL_POINTER, "%s: args is NULL", who);
  int rc = norm_check(who, a->x, a->weight, a->dx, a->rows, a->hidden, a->x_dtype, a->residual, a->residual_dtype);
  if (rc != SSM_OK) return rc;
  SSM_REQUIRE(a->dy && a->rstd && a->dweight && (a->is_rms || a->mean), SSM_ERR_NULL_POINTER,
              "%s: dy, rstd, dweight (and mean for LayerNorm) are required", who);
  SSM_REQUIRE(!a->dresidual || a->residual, SSM_ERR_NULL_POINTER, "%s: dresidual needs residual", who);
  SSM_REQUIRE(!a->grad_residual_out || valid_dtype(a->grad_residual_out_dtype), SSM_ERR_BAD_DTYPE,
              "%s: grad_residual_out_dtype=%d", who, a->grad_residual_out_dtype);
  return SSM_OK;
}

// The launches of the backward pass; `partial` holds norm_bwd_partials() x 2 x hidden floats.
static int norm_bwd_launch(const ssm_norm_bwd_args *a, float *partial, void *hip_stream) {
  NormParams p{};
  p.x = a->x; p.res = a->residual; p.dy = a->dy; p.w = a->weight; p.dx = a->dx; p.dres = a->dresidual;
  p.mean = const_cast<float *>(a->mean); p.rstd = const_cast<float *>(a->rstd);
  p.partial = partial;
  p.rows = a->rows; p.hidden = a->hidden;
  p.x_dtype = a->x_dtype; p.res_dtype = a->residual_dtype;
  p.gro = a->grad_residual_out; p.gro_dtype = a->grad_residual_out_dtype;
  p.past_caches = (size_t)a->rows * a->hidden > NORM_CACHED;
  p.has_db = a->dbias != nullptr;
  p.is_rms = a->is_rms ? 1 : 0; p.prenorm = a->prenorm ? 1 : 0;
  const int vec_ok = a->hidden % 4 == 0 && aligned_to(a->x, 16) && aligned_to(a->dy, 16) && aligned_to(a->dx, 16) &&
                     aligned_to(a->weight, 16) && (!a->residual || aligned_to(a->residual, 16)) &&
                     (!a->dresidual || aligned_to(a->dresidual, 16)) &&
                     (!a->grad_residual_out || aligned_to(a->grad_residual_out, 16));
  hipStream_t s = reinterpret_cast<hipStream_t>(hip_stream);
  int grid = norm_bwd_grid(a->rows);
  const int per_lane = (a->hidden + WAVE - 1) / WAVE;
  // typed kernels: one element type RT (float32 or that of x) for residual, dresidual and grad_residual_out
  const int rt = (a->residual || a->dresidual) ? a->residual_dtype : p.gro ? p.gro_dtype : a->x_dtype;
  if (vec_ok && a->hidden >= 4 && a->hidden <= 8192 && (rt == SSM_F32 || rt == a->x_dtype) && (!p.gro || p.gro_dtype == rt)) {
    const bool rf = rt == SSM_F32;
    if (a->x_dtype == SSM_BF16) grid = rf ? launch_norm_bwd_typed<bf16_t, float>(p, a->hidden, grid, s) : launch_norm_bwd_typed<bf16_t, bf16_t>(p, a->hidden, grid, s);
    else if (a->x_dtype == SSM_F16) grid = rf ? launch_norm_bwd_typed<f16_t, float>(p, a->hidden, grid, s) : launch_norm_bwd_typed<f16_t, f16_t>(p, a->hidden, grid, s);
    else grid = launch_norm_bwd_typed<float, float>(p, a->hidden, grid, s);
  }
  else if (per_lane <= 4) hipLaunchKernelGGL((norm_bwd_kernel<1, false>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (per_lane <= 8) hipLaunchKernelGGL((norm_bwd_kernel<2, false>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (per_lane <= 12) hipLaunchKernelGGL((norm_bwd_kernel<3, false>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (a->hidden <= 1024) hipLaunchKernelGGL((norm_bwd_kernel<1, true>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (a->hidden <= 2048) hipLaunchKernelGGL((norm_bwd_kernel<2, true>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (a->hidden <= 4096) hipLaunchKernelGGL((norm_bwd_kernel<4, true>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else if (a->hidden <= 8192) hipLaunchKernelGGL((norm_bwd_kernel<8, true>), dim3(grid), dim3(LN_THREADS), 0, s, p, vec_ok);
  else hipLaunchKernelGGL(norm_bwd_long_kernel, dim3(grid), dim3(LN_THREADS), 0, s, p);
  SSM_CHECK_LAUNCH("ssm_norm_bwd");
  const int nparts = a->hidden <= 8192 ? grid : grid * LN_WAVES;   // the long-row kernel writes one per wave
  const dim3 fold((a->hidden + FOLD_COLS - 1) / FOLD_COLS);
  if (a->dbias) hipLaunchKernelGGL(norm_bwd_fold_kernel<true>, fold, dim3(FOLD_THREADS), 0, s, p.partial, a->dweight, a->dbias, nparts, a->hidden);
  else hipLaunchKernelGGL(norm_bwd_fold_kernel<false>, fold, dim3(FOLD_THREADS), 0, s, p.partial, a->dweight, nullptr, nparts, a->hidden);
  SSM_CHECK_LAUNCH("ssm_norm_bwd(fold)");
  return SSM_OK;
}

// Device memory for the partial sums of ssm_norm_bwd_static: part of the code object, so every GPU that the
// library runs on holds its own copy from load to process end.  The name is a host-side handle only; the
// address on the current device comes from hipGetSymbolAddress and is kept per device.
constexpr size_t NORM_BWD_STATIC_FLOATS = SSM_NORM_BWD_STATIC_BYTES / sizeof(float);
static __device__ __align__(256) float scratch[NORM_BWD_STATIC_FLOATS];

constexpr int MAX_DEVICES = 64;
static std::mutex scratch_lock;
static float *scratch_on_device[MAX_DEVICES];

static int norm_bwd_scratch(float **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
    set_error("ssm_norm_bwd_static: no usable current device (%s)", e == hipSuccess ? "index out of range" : hipGetErrorString(e));
    return SSM_ERR_LAUNCH;
  }
  std::lock_guard<std::mutex> guard(scratch_lock);
  if (!scratch_on_device[dev]) {
    void *ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      (void)hipGetLastError();
      set_error("ssm_norm_bwd_static: hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(e));
      return SSM_ERR_LAUNCH;
    }
    scratch_on_device[dev] = reinterpret_cast<float *>(ptr);
  }
  *out = scratch_on_device[dev];
  return SSM_OK;
}

}  // namespace ssm

extern "C" int ssm_norm_bwd(const ssm_norm_bwd_args *a, void *hip_stream) {
  using namespace ssm;
  const int rc = norm_bwd_check("ssm_norm_bwd", a);
  if (rc != SSM_OK) return rc;
  SSM_REQUIRE(a->workspace && a->workspace_bytes >= ssm_norm_bwd_workspace_bytes(a->rows, a->hidden),
              SSM_ERR_WORKSPACE, "ssm_norm_bwd: workspace of %zu bytes required",
              ssm_norm_bwd_workspace_bytes(a->rows, a->hidden));
  return norm_bwd_launch(a, reinterpret_cast<float *>(a->workspace), hip_stream);
}

extern "C" int ssm_norm_bwd_static(const ssm_norm_bwd_args *a, void *hip_stream) {
  using namespace ssm;
  int rc = norm_bwd_check("ssm_norm_bwd_static", a);
  if (rc != SSM_OK) return rc;
  const size_t need = norm_bwd_partials(a->rows, a->hidden) * 2 * (size_t)a->hidden;
  SSM_REQUIRE(need <= NORM_BWD_STATIC_FLOATS, SSM_ERR_TOO_LARGE,
              "ssm_norm_bwd_static: rows=%d hidden=%d need %zu bytes of partial sums, the built-in buffer holds %zu; "
              "use ssm_norm_bwd with a workspace", a->rows, a->hidden, need * sizeof(float),
              (size_t)SSM_NORM_BWD_STATIC_BYTES);
  float *partial = nullptr;
  rc = norm_bwd_scratch(&partial);
  if (rc != SSM_OK) return rc;
  return norm_bwd_launch(a, partial, hip_stream);
}
