// Selective scan, forward: any number of channels to a workgroup.  Included by scan_fwd_fast.hpp.
//
// The walk of scan_fwd_fast.hpp (chunks of 512 steps, 32 lanes of 16 steps, two slabs of B and C in LDS, three waves a SIMD),
// but a workgroup of twelve waves takes as many channels of a group as the host says, not a multiple of what its waves hold:
// wave w takes rows w, w + 12, ..., so that what is left over spreads over the SIMDs.  A call then is as many equal
// workgroups as there are CUs, whatever its number of channels (a group's last one may have fewer).
// A wave works on one row at a time: both halves of the wave hold the same 512 steps, each with half of the states.  What is
// formed per step (step sizes, gate, output) is formed by the half that owns the step and handed across with
// v_permlane32_swap; the sums for y meet the same way.  A row's A and the state it carries live in LDS, touched by its own
// wave only.  The next row and the next chunk's slab are requested as soon as the present row is in float32, the gate one
// state before it is needed.  Rows of any length and start: a run is one access at its own address, a row's end is put right
// in registers.  K = 8: the same for rows of at most 256 steps, with half the run.
//
// Bound: vector issue at three waves a SIMD, 115 instructions per state and run; below twelve rows on a CU the chain of one
// wave, about 5 us a chunk.  us, with the workgroups of 8, 24 or 48 channels before / so: 8 x 1536 x 2048 float32 142 / 127, 2047
// steps 146 / 124, bf16 2047 steps 123 / 113; 8 x 1152 x 2048 bf16 125 / 86; 8 x 640 x 2048 83 / 55; 4 x 1872 x 1750 f16 132 / 82;
// 8 x 384 x 2048 57 / 36; 3 x 640 x 1021 float32 21.8 / 18.4; 8 x 1536 x 250 bf16 (the general kernel before) 33 / 22.
#pragma once

namespace ssm {

constexpr int ROWS_WAVES = 12;
constexpr int ROWS_MAX = 96;             // channels a workgroup takes at most
constexpr int ROWS_MIN = 12;             // groups of fewer channels are not worth their slab
constexpr int ROWS_VARIANT = 11120;

// Values of the two halves of a wave: lo takes what lanes 0..31 hold, hi what lanes 32..63 hold, in every lane's own
// position of its half.
__device__ __forceinline__ void both_halves(float v, float &lo, float &hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  lo = __uint_as_float(r[0]);
  hi = __uint_as_float(r[1]);
}
// Sums over the two halves: lanes 0..31 get that of a, lanes 32..63 that of b.
__device__ __forceinline__ float sum_halves(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <typename io_t, typename bc_t, int K>
__global__ __launch_bounds__(WAVE *ROWS_WAVES) __attribute__((amdgpu_waves_per_eu(3, 3)))
void scan_fwd_rows_kernel(const ScanFwdParams p) {
  constexpr int LPR = WAVE / 2, T = LPR * K, THREADS = WAVE * ROWS_WAVES;
  constexpr int SLABS = T == FAST_T ? 2 : 1;               // shorter runs are for rows of one chunk
  constexpr int PER_ROW = T / (WAVE * 4);                  // waves, or instructions, to a row of the slab
  constexpr int KO = K / 2;              // steps a lane owns
  constexpr bool IN_REGISTERS = sizeof(bc_t) == 2;
  extern __shared__ __align__(16) float tiles[];           // B [16][T], C [16][T], twice; A and carried state [rows][16]
  float *A2s = tiles + SLABS * 2 * FAST_N * T, *Hs = A2s + p.rows_per_wg * FAST_N;

  const int wave = wave_id_uniform();
  const int lane = lane_id(), sl = lane & (LPR - 1), sub = lane / LPR;
  const int lane_t = sl * K + sub * KO;                    // the first of the lane's own steps of a chunk
  const int per_span = (p.span + p.rows_per_wg - 1) / p.rows_per_wg, per_batch = per_span * (p.dim / p.span);
  const int b = (int)blockIdx.x / per_batch, blk = (int)blockIdx.x % per_batch;
  const int first = blk % per_span * p.rows_per_wg;
  const int d0 = blk / per_span * p.span + first, count = min(p.rows_per_wg, p.span - first);
  const int L = p.len, N = p.nstate;
  const bc_t *Bg = reinterpret_cast<const bc_t *>(p.Bp) + ((size_t)b * p.b_groups + d0 / (p.dim / p.b_groups)) * N * L;
  const bc_t *Cg = reinterpret_cast<const bc_t *>(p.Cp) + ((size_t)b * p.c_groups + d0 / (p.dim / p.c_groups)) * N * L;
  const int nchunks = (L + T - 1) / T;
  const int n_half = (N + 1) / 2, n_mine = sub * n_half;   // states a half of the wave walks, the first of them

  const io_t *U = reinterpret_cast<const io_t *>(p.u), *DT = reinterpret_cast<const io_t *>(p.delta);
  const io_t *Z = reinterpret_cast<const io_t *>(p.z);
  Pack<io_t, KO> ur, dr;
  auto request = [&](int r, int c) {
    const size_t at = ((size_t)b * p.dim + d0 + r) * L;
    ur = row_run<io_t, KO>(U + at, c * T + lane_t, L);
    dr = row_run<io_t, KO>(DT + at, c * T + lane_t, L);
  };
  if (wave < count) request(wave, 0);

  // The slab of a chunk.  16-bit projections are requested early in the chunk before and wait in 12 registers: two waves
  // share a row of B or C, a lane takes four steps of it and of every sixth row.  Float32 goes to its place in LDS by
  // itself: an instruction takes two of the four vectors of every lane's run.
  constexpr int EVERY = IN_REGISTERS ? ROWS_WAVES / PER_ROW : ROWS_WAVES, GROUPS = IN_REGISTERS ? (2 * FAST_N + EVERY - 1) / EVERY : 1;
  const int mine = IN_REGISTERS ? wave / PER_ROW : wave, all = IN_REGISTERS ? 2 * N : PER_ROW * 2 * N;
  auto row_at = [&](int j) { const int m = IN_REGISTERS ? j : j / PER_ROW; return m < N ? Bg + (size_t)m * L : Cg + (size_t)(m - N) * L; };
  auto place_at = [&](int c, int j) {
    const int m = IN_REGISTERS ? j : j / PER_ROW;
    return ((SLABS == 2 ? c & 1 : 0) * 2 * FAST_N + (m < N ? m : m - N + FAST_N)) * T + (IN_REGISTERS ? 0 : j % PER_ROW * (WAVE * 4));
  };
  auto step_at = [&](int j) { return IN_REGISTERS ? wave % PER_ROW * (WAVE * 4) + lane * 4 : sl * K + j % PER_ROW * 8 + sub * 4; };
  auto lane_at = [&](int j) { return IN_REGISTERS ? step_at(j) % K * LPR + step_at(j) / K * 4 : lane * 4; };
  Pack<bc_t, 4> slab[GROUPS];
  auto request_slab = [&](int c) {
    if constexpr (IN_REGISTERS) {
#pragma unroll
      for (int k = 0; k < GROUPS; ++k)
        if (mine + k * EVERY < all) slab[k] = row_run<bc_t, 4>(row_at(mine + k * EVERY), c * T + step_at(0), L);
    } else {
      const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float *)tiles;
      for (int j = mine; j < all; j += EVERY)
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds + 4u * (unsigned)place_at(c, j)),
                     "v"((unsigned)min(c * T + step_at(j), L - 4) * 4u), "s"(row_at(j)) : "memory");
    }
  };
  auto place_slab = [&](int c) {
    const bool tail = c * T + T > L;
    if constexpr (IN_REGISTERS) {
#pragma unroll
      for (int k = 0; k < GROUPS; ++k) {
        const int j = mine + k * EVERY;
        if (j >= all) break;
        if (tail) row_end(c * T + step_at(j), L, slab[k]);
        *reinterpret_cast<float4 *>(tiles + place_at(c, j) + lane_at(j)) =
            make_float4(to_f32(slab[k].v[0]), to_f32(slab[k].v[1]), to_f32(slab[k].v[2]), to_f32(slab[k].v[3]));
      }
    } else if (tail) {                   // (it has arrived)
      for (int j = mine; j < all; j += EVERY)
        if (c * T + step_at(j) + 4 > L) {
          Pack<bc_t, 4> *at = reinterpret_cast<Pack<bc_t, 4> *>(tiles + place_at(c, j) + lane_at(j)), v = *at;
          row_end(c * T + step_at(j), L, v);
          *at = v;
        }
    }
  };
  auto slab_arrived = [] {
    if constexpr (!IN_REGISTERS) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  request_slab(0);
  for (int e = threadIdx.x; e < count * FAST_N; e += THREADS) {
    A2s[e] = e % FAST_N < N ? p.A[(size_t)(d0 + e / FAST_N) * N + e % FAST_N] * LOG2E : 0.0f;
    Hs[e] = 0.0f;
  }
  if (N % 2)                             // the state that the second half has none of
    for (int e = threadIdx.x; e < 2 * SLABS * T; e += THREADS) tiles[(e / T * FAST_N + N) * T + e % T] = 0.0f;
  slab_arrived();
  place_slab(0);

  for (int c = 0; c < nchunks; ++c) {
    const int t0 = c * T;
    const bool tail = t0 + T > L;
    __syncthreads();                     // slab c is complete; every wave is done with slab c - 1 (written over below)
    const float *Bs = tiles + (SLABS == 2 ? c & 1 : 0) * 2 * FAST_N * T + n_mine * T + sl * 4, *Cs = Bs + FAST_N * T;

    for (int r = wave; r < count; r += ROWS_WAVES) {
      const int d = d0 + r;
      const size_t row = (size_t)b * p.dim + d;
      const float *A2r = A2s + r * FAST_N + n_mine;
      float *Hr = Hs + r * FAST_N + n_mine;
      if (p.chunk_states && lane < N) p.chunk_states[(row * nchunks + c) * (size_t)N + lane] = Hs[r * FAST_N + lane];
      float dl[K], du[K], y[K];
      {
        const float bias = p.bias ? p.bias[d] : 0.0f, Dk = p.Dk ? p.Dk[d] : 0.0f;
        float v[KO];
        if (tail) {
          row_end(t0 + lane_t, L, ur);
          row_end(t0 + lane_t, L, dr);
        }
#pragma unroll
        for (int i = 0; i < KO; ++i) v[i] = to_f32(dr.v[i]) + bias;
        if (p.softplus) {
#pragma unroll
          for (int i = 0; i < KO; ++i) v[i] = fast_softplus(v[i]);
        }
        if (tail) {                      // steps past the end: the identity map
#pragma unroll
          for (int i = 0; i < KO; ++i) v[i] = t0 + lane_t + i < L ? v[i] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < KO; ++i) {
          const float uu = to_f32(ur.v[i]);
          y[i] = sub ? 0.0f : Dk * uu;   // counted once, by the half that owns the step: picked, since 0 * u is NaN where u is not
          y[KO + i] = sub ? Dk * uu : 0.0f;   // finite, and would reach the other half's step, eight earlier or later
          both_halves(v[i], dl[i], dl[KO + i]);
          both_halves(v[i] * uu, du[i], du[KO + i]);
        }
      }
      float dsum = 0.0f;
#pragma unroll
      for (int i = 0; i < K; ++i) dsum += dl[i];
      if (r == wave && c + 1 < nchunks) request_slab(c + 1);
      {
        const bool again = r + ROWS_WAVES < count;
        if (again || c + 1 < nchunks) request(again ? r + ROWS_WAVES : wave, again ? c : c + 1);
      }

      auto process = [&](int n) {
        float a[K], bx[K], h;
        float4 v[K / 4];
        // the slab reads of this state are requested before anything else, so that they return while the exponentials run
#pragma unroll
        for (int q = 0; q < K / 4; ++q) v[q] = *reinterpret_cast<const float4 *>(Bs + n * T + q * (LPR * 4));
        const float A2 = A2r[n], H = Hr[n];
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < K; ++i) a[i] = dl[i] * A2;
        float P = dsum * A2;
        exp2_run(a, P);
#pragma unroll
        for (int q = 0; q < K / 4; ++q) {
          const float bq[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int i = q * 4 + j;
            bx[i] = du[i] * bq[j];
            h = i == 0 ? bx[0] : __builtin_fmaf(a[i], h, bx[i]);
          }
        }
        // the first lane of a row absorbs the state carried in from the previous chunk
        h = __builtin_fmaf(P, sl == 0 ? H : 0.0f, h);
#pragma unroll
        for (int q = 0; q < K / 4; ++q) v[q] = *reinterpret_cast<const float4 *>(Cs + n * T + q * (LPR * 4));
        half_scan_affine_x1(P, h);
        // h is the row state at the end of each lane's run; a lane starts from its predecessor's
        float hs = wave_prev(h, H);
        hs = sl == 0 ? H : hs;
        if (sl == LPR - 1) Hr[n] = h;
#pragma unroll
        for (int q = 0; q < K / 4; ++q) {
          const float cq[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int i = q * 4 + j;
            hs = __builtin_fmaf(a[i], hs, bx[i]);
            y[i] = __builtin_fmaf(hs, cq[j], y[i]);
          }
        }
      };
      // The SIMD serves its oldest wave first: the order of its three waves is turned round from state to state, which keeps
      // them out of step with each other (one in its exponentials while another replays).
      int rank = wave >> 2;
      for (int n = 0; n < n_half - 1; ++n) {
        if (rank == 0) __builtin_amdgcn_s_setprio(0);
        else if (rank == 1) __builtin_amdgcn_s_setprio(1);
        else __builtin_amdgcn_s_setprio(2);
        rank = rank == 2 ? 0 : rank + 1;
        process(n);
      }
      Pack<io_t, KO> zr;
      if (p.z) zr = row_run<io_t, KO>(Z + row * L, t0 + lane_t, L);
      if (N % 2) {                       // the half that has no such state walks zeros, whatever the row holds
#pragma unroll
        for (int i = 0; i < K; ++i) {
          dl[i] = n_mine + n_half > N ? 0.0f : dl[i];
          du[i] = n_mine + n_half > N ? 0.0f : du[i];
        }
        dsum = n_mine + n_half > N ? 0.0f : dsum;
      }
      process(n_half - 1);

      float o[KO];
#pragma unroll
      for (int i = 0; i < KO; ++i) o[i] = sum_halves(y[i], y[KO + i]);
      if (p.z) {
        if (tail) row_end(t0 + lane_t, L, zr);
#pragma unroll
        for (int i = 0; i < KO; ++i) {
          const float zz = to_f32(zr.v[i]);
          o[i] *= zz * rcp_hw(1.0f + exp2_hw(-LOG2E * zz));
        }
      }
      slab_arrived();                    // (asked behind the store, it would wait for the store)
      Pack<io_t, KO> out;
#pragma unroll
      for (int i = 0; i < KO; ++i) out.v[i] = from_f32<io_t>(o[i]);
      store_steps<true, io_t, KO>(reinterpret_cast<io_t *>(p.out) + row * L, t0 + lane_t, L, out);
    }
    if (c + 1 < nchunks) {
      if (wave >= count) {               // a wave without rows
        request_slab(c + 1);
        slab_arrived();
      }
      place_slab(c + 1);
    }
  }

  if (p.last) {
    __syncthreads();
    for (int e = threadIdx.x; e < count * N; e += THREADS)
      reinterpret_cast<io_t *>(p.last)[((size_t)b * p.dim + d0) * N + e] = from_f32<io_t>(Hs[e / N * FAST_N + e % N]);
  }
}

template <typename io_t, typename bc_t, int K>
static int launch_scan_fwd_rows_as(const ScanFwdParams &p, hipStream_t stream) {
  const size_t lds = ((K == 16 ? 4 : 2) * FAST_N * (WAVE / 2 * K) + 2 * (size_t)p.rows_per_wg * FAST_N) * sizeof(float);
  auto kernel = scan_fwd_rows_kernel<io_t, bc_t, K>;
  if (allow_dynamic_lds(kernel, lds) != hipSuccess) {
    (void)hipGetLastError();
    set_error("ssm_scan_fwd: cannot reserve %zu bytes of LDS", lds);
    return SSM_ERR_LAUNCH;
  }
  const size_t grid = (size_t)p.batch * (p.dim / p.span) * ((p.span + p.rows_per_wg - 1) / p.rows_per_wg);
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(WAVE * ROWS_WAVES), lds, stream, p);
  SSM_CHECK_LAUNCH("ssm_scan_fwd");
  return SSM_OK;
}

template <typename io_t, typename bc_t>
static int launch_scan_fwd_rows(const ScanFwdParams &p, hipStream_t s) {
  return p.len <= FAST_T / 2 ? launch_scan_fwd_rows_as<io_t, bc_t, 8>(p, s) : launch_scan_fwd_rows_as<io_t, bc_t, 16>(p, s);
}

}  // namespace ssm
