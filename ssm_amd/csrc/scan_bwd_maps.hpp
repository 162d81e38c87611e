// Selective scan, backward: what crosses the borders of 512-step chunks, found up front, so that the chunks of a call of
// few rows can run side by side instead of one after the other.  Included by scan_bwd.hip.
//
// Per row and state a chunk is an affine map: the adjoint q that enters from the right leaves at the left as P q + S.
// With s_t the sum of the steps up to and with t, P = exp2(A2 s_end) and S = sum_t exp2(A2 s_t) g_t C_t: the running sum of
// the steps is the same for all states, and no scan over the lanes is left, only a wave sum per state.  The kernels
// that walk the chunks compose the maps between the row's end and their chunk themselves (compose_maps).
// A sixth of the backward's arithmetic per step.  A workgroup takes one chunk of eight rows, which share the slab of C in
// LDS (where groups are whole blocks of eight channels; otherwise every wave reads its own): with a row's chunks in one workgroup instead, every wave reading C from memory, that traffic bound the kernel.
#pragma once
#include "scan_bwd_fast.hpp"

namespace ssm {

constexpr int MAPS_WAVES = 8;

// SLAB: a C that blocks of eight channels share, staged in LDS; otherwise it is read per row, from memory
// (a group per channel) or as one value per state (CONST_BC).
template <typename io_t, typename bc_t, bool SLAB, bool CONST_BC, bool RAGGED>
__global__ __launch_bounds__(WAVE *MAPS_WAVES)
void scan_maps_kernel(const ScanBwdParams p, float2 *maps) {
  constexpr int K = FAST_T / WAVE, T = FAST_T;
  __shared__ __align__(16) float slab[SLAB ? FAST_N * FAST_T : 4];
  const int wave = wave_id_uniform();
  const int lane = lane_id();
  const int L = p.len, N = p.nstate;
  const int nchunks = (L + T - 1) / T;
  const int c = (int)(blockIdx.x % nchunks);
  const size_t row = (size_t)(blockIdx.x / nchunks) * MAPS_WAVES + wave;
  const bool in_grid = row < (size_t)p.batch * p.dim;        // (always with a slab: eight rows of one batch entry)
  const int b = in_grid ? (int)(row / p.dim) : 0, d = in_grid ? (int)(row % p.dim) : 0;
  const int t = c * T + lane * K;
  const bool tail = (c + 1) * T > L;
  const bc_t *G = reinterpret_cast<const bc_t *>(p.Cp);
  size_t groom = 0;
  float G_lanes = 0.0f;
  if constexpr (CONST_BC) {
    if (lane < N) G_lanes = load_as_f32(p.Cp, p.bc_dtype, (p.c_kind == SSM_PROJ_BDN ? (size_t)b * p.dim + d : (size_t)d) * N + lane);
  } else {
    const size_t g = (size_t)b * p.c_groups + d / (p.dim / p.c_groups);
    G += g * N * L;
    groom = ((size_t)p.batch * p.c_groups - g) * N * L;
  }
  const size_t rd = in_grid ? row : 0;
  const size_t at = rd * L, room = ((size_t)p.batch * p.dim - rd) * L;
  const Pack<io_t, K> dr = load_steps<RAGGED, io_t, K>(reinterpret_cast<const io_t *>(p.delta) + at, t, L, tail, room);
  const Pack<io_t, K> xr = load_steps<RAGGED, io_t, K>(reinterpret_cast<const io_t *>(p.dout) + at, t, L, tail, room);
  Pack<io_t, K> zr;
  if (p.z) zr = load_steps<RAGGED, io_t, K>(reinterpret_cast<const io_t *>(p.z) + at, t, L, tail, room);
  if constexpr (SLAB) {
    fast_stage<bc_t, WAVE, RAGGED>(slab, G, L, c * T, N, WAVE * MAPS_WAVES, groom);
    __syncthreads();
  }
  if (!in_grid) return;                                      // no barrier below
  Pack<bc_t, K> graw;
  if constexpr (!SLAB && !CONST_BC) graw = load_steps<RAGGED, bc_t, K>(G, t, L, tail, groom);
  const float A2_lanes = lane < N ? p.A[(size_t)d * N + lane] * LOG2E : 0.0f;
  const float bias = p.bias ? p.bias[d] : 0.0f;
  float sum[K], x[K], dsum = 0.0f;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const bool in = t + (RAGGED ? i : 0) < L;
    const float v = to_f32(dr.v[i]) + bias;
    dsum += in ? (p.softplus ? fast_softplus(v) : v) : 0.0f;
    sum[i] = dsum;
    x[i] = in ? to_f32(xr.v[i]) : 0.0f;
    if (p.z) {
      const float zz = to_f32(zr.v[i]);
      x[i] *= zz * rcp_hw(1.0f + exp2_hw(-LOG2E * zz));
    }
  }
  const float upto = wave_inclusive_sum(dsum), before = wave_prev(upto, 0.0f);
  const float total = wave_read_lane(upto, WAVE - 1);
#pragma unroll
  for (int i = 0; i < K; ++i) sum[i] += before;
  float S_lanes = 0.0f;
#pragma unroll 2
  for (int n = 0; n < N; ++n) {
    const float A2 = wave_read_lane(A2_lanes, n);
    float gq[K];
    if constexpr (SLAB) {
#pragma unroll
      for (int q = 0; q < K / 4; ++q) {
        const float4 v = *reinterpret_cast<const float4 *>(slab + n * T + q * (WAVE * 4) + lane * 4);
        gq[4 * q] = v.x; gq[4 * q + 1] = v.y; gq[4 * q + 2] = v.z; gq[4 * q + 3] = v.w;
      }
    } else if constexpr (CONST_BC) {
      const float gn = wave_read_lane(G_lanes, n);
#pragma unroll
      for (int i = 0; i < K; ++i) gq[i] = gn;
    } else {
#pragma unroll
      for (int i = 0; i < K; ++i) gq[i] = to_f32(graw.v[i]);
      const size_t next = (size_t)min(n + 1, N - 1) * L;     // the next state's, before this one's arithmetic
      graw = load_steps<RAGGED, bc_t, K>(G + next, t, L, tail, groom - next);
    }
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < K; ++i) s = __builtin_fmaf(exp2_hw(sum[i] * A2), x[i] * gq[i], s);
    s = wave_sum(s);
    S_lanes = lane == n ? s : S_lanes;
  }
  if (lane < N) maps[(row * nchunks + c) * (size_t)N + lane] = make_float2(exp2_hw(total * A2_lanes), S_lanes);
}

template <typename io_t, typename bc_t, bool SLAB, bool CONST_BC>
static int launch_scan_maps_as(const ScanBwdParams &p, float2 *maps, hipStream_t s) {
  const size_t blocks = ((size_t)p.batch * p.dim + MAPS_WAVES - 1) / MAPS_WAVES * ((p.len + FAST_T - 1) / FAST_T);
  const dim3 grid((unsigned)blocks), block(WAVE * MAPS_WAVES);
  if (p.ragged) hipLaunchKernelGGL((scan_maps_kernel<io_t, bc_t, SLAB, CONST_BC, true>), grid, block, 0, s, p, maps);
  else hipLaunchKernelGGL((scan_maps_kernel<io_t, bc_t, SLAB, CONST_BC, false>), grid, block, 0, s, p, maps);
  SSM_CHECK_LAUNCH("selective scan (maps of the chunks)");
  return SSM_OK;
}

}  // namespace ssm
