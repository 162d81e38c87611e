// Diagonal chunked scan: the time axis of a call with few channels cut into segments that run side by side.
// Included by dscan.hip and dscan_bwd.hip, whose one-pass kernels give a workgroup 64 or 128 channels for all of time: at
// 2 x 2048 steps x 1024 float32 channels that is 32 workgroups on 256 CUs.
//
// Per channel a segment is an affine map.  Forward, the state s leaves it as P s + S; backward, mu = lambda a, the adjoint
// times its decay, leaves at the left as P mu + M.  This kernel finds the maps: a workgroup owns one segment of its
// channels, each of its 16 waves folds a sixteenth of the steps (no wave waits for another until the 16 folds
// meet in LDS once), and the one-pass kernels compose the maps between the sequence's end and their segment themselves.
// It reads X, dt and B (dy, dt, C and the gate) once more, which caches or a mostly idle memory serve.
#pragma once
#include "common.hpp"

namespace ssm {

constexpr int DM_WAVES = 16, DM_STEPS = 8;        // steps whose reads are in flight together

struct DscanMapParams {
  const void *drive, *dt, *proj, *z;        // X, B forward; dy, C and the gate (or NULL) backward
  const float *A;
  const int *lengths;
  float2 *maps;                             // (B, nseg, HP)
  int batch, len, heads, width;             // width: channels of a head
  int proj_dtype, a_stride_p;
  long long proj_stride_b;                  // PARAMS: element stride of the projection over the batch
  int seg_len, nseg;                        // steps per segment
};

template <typename io_t, int VEC, bool BWD, bool HAS_Z, bool PARAMS>
__global__ __launch_bounds__(WAVE *DM_WAVES) void dscan_maps_kernel(const DscanMapParams p) {
  static_assert(sizeof(io_t) * VEC == 4, "a lane's vector is one register");
  constexpr int AV = PARAMS ? VEC : 1;            // decays per lane
  __shared__ float2 folds[DM_WAVES][VEC][WAVE];
  const int wave = wave_id_uniform(), lane = lane_id();
  const int HP = p.heads * p.width;
  // (channels past the last one of a last workgroup that is not full stand for it: the same values to the same places)
  const unsigned ch = min(((unsigned)blockIdx.x * WAVE + lane) * VEC, (unsigned)HP - VEC);
  const int b = blockIdx.y, seg = blockIdx.z;
  const int h = (int)ch / p.width;
  const int L = p.len;
  const int valid = p.lengths ? min(max(p.lengths[b], 0), L) : L;
  float A2[AV], Gc[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    if (v < AV) A2[v] = p.A[p.a_stride_p ? (size_t)ch + v : (size_t)h] * LOG2E;
    Gc[v] = PARAMS ? load_as_f32(p.proj, p.proj_dtype, (size_t)b * p.proj_stride_b + ch + v) : 0.0f;
  }
  const size_t row0 = (size_t)b * L;
  const io_t *X = reinterpret_cast<const io_t *>(p.drive) + row0 * HP;
  const io_t *G = reinterpret_cast<const io_t *>(PARAMS ? p.drive : p.proj) + row0 * HP;
  const io_t *Z = reinterpret_cast<const io_t *>(HAS_Z ? p.z : p.drive) + row0 * HP;
  const float *DT = reinterpret_cast<const float *>(p.dt) + row0 * p.heads;
  // the wave's steps: whole groups, so that a group's reads go out together
  const int share = (p.seg_len + DM_WAVES * DM_STEPS - 1) / (DM_WAVES * DM_STEPS) * DM_STEPS;
  const int begin = seg * p.seg_len + wave * share;
  const int end = min(min(begin + share, (seg + 1) * p.seg_len), valid);
  float prod[AV], s[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) s[v] = 0.0f;
#pragma unroll
  for (int v = 0; v < AV; ++v) prod[v] = 1.0f;
  for (int k = 0; k < share; k += DM_STEPS) {
    const int t0 = BWD ? begin + share - DM_STEPS - k : begin + k;
    if (t0 >= end) continue;                      // uniform over the wave
    float dt[DM_STEPS];
    Word<io_t> x[DM_STEPS], g[DM_STEPS], z[DM_STEPS];
#pragma unroll
    for (int j = 0; j < DM_STEPS; ++j) {
      const unsigned row = (unsigned)min(t0 + j, L - 1);
      const unsigned at = (row * (unsigned)HP + ch) * (unsigned)sizeof(io_t);
      dt[j] = *at_bytes<const float>(DT, (row * (unsigned)p.heads + (unsigned)h) * 4u);
      x[j] = Word<io_t>{*at_bytes<const unsigned>(X, at)};
      if (!PARAMS) g[j] = Word<io_t>{*at_bytes<const unsigned>(G, at)};
      if (HAS_Z) z[j] = Word<io_t>{*at_bytes<const unsigned>(Z, at)};
    }
#pragma unroll
    for (int i = 0; i < DM_STEPS; ++i) {
      const int j = BWD ? DM_STEPS - 1 - i : i;
      const bool live = t0 + j < end;             // a dead step is the identity
      const float d = live ? dt[j] : 0.0f;
      x[j].mask(live);
      if (!PARAMS) g[j].mask(live);
      float a[AV];
#pragma unroll
      for (int v = 0; v < AV; ++v) {
        a[v] = exp2_hw(d * A2[v]);
        prod[v] *= a[v];
      }
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const float gv = PARAMS ? Gc[v] : g[j].elem(v);
        float xv = x[j].elem(v);
        if (HAS_Z) xv *= silu_f32(z[j].elem(v));
        s[v] = BWD ? a[v % AV] * __builtin_fmaf(live ? xv : 0.0f, gv, s[v]) : __builtin_fmaf(a[v % AV], s[v], d * gv * xv);
      }
    }
  }
#pragma unroll
  for (int v = 0; v < VEC; ++v) folds[wave][v][lane] = make_float2(prod[v % AV], s[v]);
  __syncthreads();
  if (wave < VEC) {                               // wave v composes channel v's folds
    float P = 1.0f, S = 0.0f;
#pragma unroll
    for (int w = 0; w < DM_WAVES; ++w) {
      const float2 f = folds[BWD ? DM_WAVES - 1 - w : w][wave][lane];
      S = __builtin_fmaf(f.x, S, f.y);
      P *= f.x;
    }
    p.maps[((size_t)b * p.nseg + seg) * HP + ch + wave] = make_float2(P, S);
  }
}

// A channel's value through the maps of `count` segments, `step` elements apart.
__device__ __forceinline__ float dscan_compose(const float2 *m, int count, ptrdiff_t step, float v) {
  for (int k = 0; k < count; k += 8) {
    float2 f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = m[(ptrdiff_t)min(k + j, count - 1) * step];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (k + j < count) v = __builtin_fmaf(f[j].x, v, f[j].y);
  }
  return v;
}

template <typename io_t, int VEC, bool BWD, bool PARAMS>
static void launch_dscan_maps(const DscanMapParams &p, hipStream_t s) {
  const dim3 grid((unsigned)(((size_t)p.heads * p.width + WAVE * VEC - 1) / (WAVE * VEC)), (unsigned)p.batch, (unsigned)p.nseg), block(WAVE * DM_WAVES);
  if constexpr (BWD) {
    if (p.z) {
      hipLaunchKernelGGL((dscan_maps_kernel<io_t, VEC, true, true, PARAMS>), grid, block, 0, s, p);
      return;
    }
  }
  hipLaunchKernelGGL((dscan_maps_kernel<io_t, VEC, BWD, false, PARAMS>), grid, block, 0, s, p);
}

// Segments of a walk of `rounds` rounds by `wgs` workgroups, in rounds per segment.  A workgroup fills a CU, a round takes
// it `us`, starting a workgroup about two; the maps are a launch of `launch` us and a `share` of the walk's own work.
static int dscan_rounds_per_segment(size_t wgs, int rounds, double us, double launch, double share) {
  int best_per = rounds;
  double best = 0.0;
  for (int most = 1; most <= 32 && most <= rounds; ++most) {          // at most so many segments, equal but for the last
    const int per = (rounds + most - 1) / most, n = (rounds + per - 1) / per;
    const double turns = (double)((wgs * n + 255) / 256);
    const double cost = turns * (2.0 + us * per) + (n > 1 ? launch + share * us * rounds * (double)wgs / 256 : 0.0);
    if (most == 1 || cost < 0.97 * best) {
      best = cost;
      best_per = per;
    }
  }
  return best_per;
}

}  // namespace ssm
