// Selective scan, forward: few rows, several chunks of time each.  Included by scan_fwd_fast.hpp.
//
// With one row per wave, a call of 512 rows puts two waves on every other SIMD and lets each walk its chunks one after
// the other.  Here the chunks of a row run side by side: a workgroup owns one row, wave w its w-th chunk of 512 steps
// (lanes and arithmetic as in scan_fwd_rowbc_kernel, projections read straight from memory).  What crosses chunks is one
// affine map per state.  A chunk's decay follows from the sum of its steps alone and is known for all states at once; its
// contribution is the last lane's result of the lane scan with nothing carried in.  The waves leave both in LDS, meet at
// one barrier per pair of states (two buffers), and each composes the maps of the chunks before its own into the state
// that enters it, which a lane picks up through its own decay from the chunk's start -- one more exponential per lane and
// state instead of a second walk.
// More chunks than waves (8): the workgroup takes them 8 at a time, the state between them in lanes of every wave.
//
// Bound: latency and issue at one to four waves per SIMD.  1 x 512 x 2048, 16 states, float32: see the rule in
// scan_fwd.hip for what it measured.
#pragma once

namespace ssm {

constexpr int SPLIT_MAX_WAVES = 8;

// A lane's run: aligned whole runs by load_steps, runs of any start by row_run (and row_end where a row ends).
template <bool RAGGED, typename T, int K>
__device__ __forceinline__ Pack<T, K> lane_run(const T *row, int t, int len) {
  if constexpr (RAGGED) return row_run<T, K>(row, t, len);
  else return load_steps<false, T, K>(row, t, len, false, 0);
}

template <typename io_t, typename bc_t, bool CONST_BC, bool RAGGED>
__global__ __launch_bounds__(WAVE *SPLIT_MAX_WAVES)
void scan_fwd_split_kernel(const ScanFwdParams p) {
  constexpr int K = FAST_T / WAVE, T = FAST_T;
  __shared__ float decay[SPLIT_MAX_WAVES][FAST_N];          // of every chunk, per state
  __shared__ float add[2][SPLIT_MAX_WAVES][2];              // of every chunk, for the pair of states at hand
  const int waves = (int)(blockDim.x >> 6);
  const int wave = wave_id_uniform();
  const int lane = lane_id();
  const size_t row = blockIdx.x;
  const int b = (int)(row / p.dim), d = (int)(row % p.dim);
  const int L = p.len, N = p.nstate;
  const bc_t *Bg = reinterpret_cast<const bc_t *>(p.Bp), *Cg = reinterpret_cast<const bc_t *>(p.Cp);
  float B_lanes = 0.0f, C_lanes = 0.0f;
  if constexpr (CONST_BC) {
    if (lane < N) {
      B_lanes = load_as_f32(p.Bp, p.bc_dtype, (p.b_kind == SSM_PROJ_BDN ? row : (size_t)d) * N + lane);
      C_lanes = load_as_f32(p.Cp, p.bc_dtype, (p.c_kind == SSM_PROJ_BDN ? row : (size_t)d) * N + lane);
    }
  } else {
    const size_t bg = (size_t)b * p.b_groups + d / (p.dim / p.b_groups), cg = (size_t)b * p.c_groups + d / (p.dim / p.c_groups);
    Bg += bg * N * L;
    Cg += cg * N * L;
  }
  const io_t *U = reinterpret_cast<const io_t *>(p.u) + row * L, *DT = reinterpret_cast<const io_t *>(p.delta) + row * L;
  const io_t *Z = reinterpret_cast<const io_t *>(p.z) + row * L;
  io_t *Y = reinterpret_cast<io_t *>(p.out) + row * L;
  const float A2_lanes = lane < N ? p.A[(size_t)d * N + lane] * LOG2E : 0.0f;
  const float Dk = p.Dk ? p.Dk[d] : 0.0f, bias = p.bias ? p.bias[d] : 0.0f;
  const int nchunks = (L + T - 1) / T;
  float carry_lanes = 0.0f;                                  // lane n: state entering the chunks at hand, the same in every wave

  for (int c0 = 0; c0 < nchunks; c0 += waves) {
    const int c = c0 + wave;                                 // beyond the end: a wave of identity maps
    const int t = c * T + lane * K;
    const bool tail = (c + 1) * T > L;
    // A run's 32-bit offset counts from the chunk's first step, or from the row's last run where the chunk lies beyond the end.
    const int origin = RAGGED ? min(c * T, L - K) : 0;
    const auto run_of = [&](const auto *row) {
      return lane_run<RAGGED, std::remove_const_t<std::remove_pointer_t<decltype(row)>>, K>(row + origin, t - origin, L - origin);
    };
    Pack<bc_t, K> braw[2], craw[2];
    auto fetch = [&](int n) {
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const size_t at = (size_t)min(n + w, N - 1) * L;
        braw[w] = run_of(Bg + at);
        craw[w] = run_of(Cg + at);
      }
    };
    if constexpr (!CONST_BC) fetch(0);
    Pack<io_t, K> ur = run_of(U), dr = run_of(DT), zr;
    if (p.z) zr = run_of(Z);
    if (RAGGED && tail) {
      row_end(t, L, ur);
      row_end(t, L, dr);
    }
    float dl[K], du[K], y[K], dsum = 0.0f;
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const float x = to_f32(dr.v[i]) + bias, uu = to_f32(ur.v[i]);
      dl[i] = t + (RAGGED ? i : 0) < L ? (p.softplus ? fast_softplus(x) : x) : 0.0f;
      du[i] = dl[i] * uu;
      y[i] = Dk * uu;
      dsum += dl[i];
    }
    const float upto = wave_inclusive_sum(dsum), before = wave_prev(upto, 0.0f);
    const float total = wave_read_lane(upto, WAVE - 1);
    __syncthreads();                                         // the chunks before are through with `decay`
    if (lane < N) decay[wave][lane] = exp2_hw(total * A2_lanes);
    float Hin_lanes = 0.0f;

    for (int n = 0, buf = 0; n < N; n += 2, buf ^= 1) {
      float a[2][K], bx[2][K], cq[2][K], h[2], Pw[2], A2[2];
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        A2[w] = wave_read_lane(A2_lanes, n + w);             // a state past the last one: lane N and beyond hold zero
        float bq[K];
        if constexpr (CONST_BC) {
          const float bn = wave_read_lane(B_lanes, n + w), cn = wave_read_lane(C_lanes, n + w);
#pragma unroll
          for (int i = 0; i < K; ++i) { bq[i] = bn; cq[w][i] = cn; }
        } else {
          if (RAGGED && tail) {
            row_end(t, L, braw[w]);
            row_end(t, L, craw[w]);
          }
#pragma unroll
          for (int i = 0; i < K; ++i) { bq[i] = to_f32(braw[w].v[i]); cq[w][i] = to_f32(craw[w].v[i]); }
        }
        Pw[w] = dsum * A2[w];
#pragma unroll
        for (int i = 0; i < K; ++i) a[w][i] = dl[i] * A2[w];
        exp2_run(a[w], Pw[w]);
#pragma unroll
        for (int i = 0; i < K; ++i) {
          bx[w][i] = du[i] * bq[i];
          h[w] = i == 0 ? bx[w][0] : __builtin_fmaf(a[w][i], h[w], bx[w][i]);
        }
      }
      if constexpr (!CONST_BC) fetch(n + 2);                 // requested before this pair is finished
      wave_scan_affine_x2(Pw[0], h[0], Pw[1], h[1]);
      if (lane == WAVE - 1) {
        add[buf][wave][0] = h[0];
        add[buf][wave][1] = h[1];
      }
      __syncthreads();
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        if (n + w >= N) break;
        float H = wave_read_lane(carry_lanes, n + w), Hin = H;
        for (int v = 0; v < waves; ++v) {
          Hin = v == wave ? H : Hin;
          H = __builtin_fmaf(decay[v][n + w], H, add[buf][v][w]);
        }
        carry_lanes = lane == n + w ? H : carry_lanes;
        Hin_lanes = lane == n + w ? Hin : Hin_lanes;
        float hs = __builtin_fmaf(exp2_hw(before * A2[w]), Hin, wave_prev(h[w], 0.0f));
#pragma unroll
        for (int i = 0; i < K; ++i) {
          hs = __builtin_fmaf(a[w][i], hs, bx[w][i]);
          y[i] = __builtin_fmaf(hs, cq[w][i], y[i]);
        }
      }
    }

    if (p.chunk_states && c < nchunks && lane < N) p.chunk_states[(row * nchunks + c) * (size_t)N + lane] = Hin_lanes;
    if (p.z) {
      if (RAGGED && tail) row_end(t, L, zr);
#pragma unroll
      for (int i = 0; i < K; ++i) {
        const float zz = to_f32(zr.v[i]);
        y[i] *= zz * rcp_hw(1.0f + exp2_hw(-LOG2E * zz));
      }
    }
    Pack<io_t, K> o;
#pragma unroll
    for (int i = 0; i < K; ++i) o.v[i] = from_f32<io_t>(y[i]);
    store_steps<RAGGED, io_t, K>(Y, t, L, o);
  }
  if (p.last && wave == 0 && lane < N) reinterpret_cast<io_t *>(p.last)[row * N + lane] = from_f32<io_t>(carry_lanes);
}

template <typename io_t, typename bc_t, bool CONST_BC>
static int launch_scan_fwd_split(const ScanFwdParams &p, hipStream_t stream) {
  const int nchunks = (p.len + FAST_T - 1) / FAST_T;
  // as many waves as a workgroup may have, or just enough for equal turns
  const int turns = (nchunks + SPLIT_MAX_WAVES - 1) / SPLIT_MAX_WAVES, waves = (nchunks + turns - 1) / turns;
  const dim3 grid((unsigned)((size_t)p.batch * p.dim)), block(WAVE * waves);
#define SSM_K(R) scan_fwd_split_kernel<io_t, bc_t, CONST_BC, R>
  SSM_RAGGED_LAUNCH(p, SSM_K, grid, block, 0, stream);
#undef SSM_K
  SSM_CHECK_LAUNCH("ssm_scan_fwd");
  return SSM_OK;
}

}  // namespace ssm
