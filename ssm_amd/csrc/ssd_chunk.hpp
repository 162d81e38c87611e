// The SSD of 16-bit calls with the chunks side by side, forward and backward: one workgroup per (batch, chunk, head).
//
//   states: what a chunk adds to the state,             S_c = sum_s exp(cs_Q - cs_s) dt_s x_s (x) B_s
//   carry:  the state entering each chunk,              H_{c+1} = exp(cs_Q) H_c + S_c
//   scan:   y_l = exp(cs_l) C_l.H_c + sum_{s<=l} (C_l.B_s) exp(cs_l - cs_s) dt_s x_s
//
// and, for the gradients, the same three with the adjoint in the place of x: dS_c = sum_l exp(cs_l) dy_l (x) C_l, passed
// from the last chunk to the first, and u_s = exp(cs_Q - cs_s) B_s.G_c + sum_{l>=s} (C_l.B_s) exp(cs_l - cs_s) dy_l
// with dx_s = dt_s u_s + D dy_s.
//
// What chunks add travels in float32, the states entering them in the element type (as operands; the recurrence is in
// float32, and what a backward needs of them in float32 travels beside them), both in fragment order: [p / 32][n / 16][lane][8], lane = p % 32 + 32 (n % 16 / 8), the order
// in which a wave holds 32 x 16 of them as a matrix operand.  A wave's accumulators of S^T are written as whole KiB that
// way, the pass is element by element in any order, and the scan reads operands without a transposition.
//
// The 64 channels of a chunk's rows are staged once, transposed, in LDS ([p][s], 16-byte pieces XOR-swizzled by p: no
// bank conflicts on either side); the fragments of B, C and C.B come from L2, shared by the heads of a group, whose
// workgroups are numbered onto one XCD.  What bounds these kernels is the traffic of x, z, y and the states: the matrix
// products take about 1 us of a CU per workgroup, a decay factor per element of C.B another.
//
// A growing head (A > 0): decays between steps of a chunk are bounded by 1, the factors on carried states are not (as in
// ssd_walk.hip); the gradients are those of that function.
#pragma once
#include "ssd_common.hpp"

#include <algorithm>

namespace ssm {

template <typename E, int C> struct Row { static_assert(sizeof(E) == 2); E v[C]; } __attribute__((aligned(2 * C)));

// (batch, chunk, head) of a workgroup and what follows from it.
struct ChunkUnit {
  int b, c, h, g, rows;          // rows: steps of this chunk
  size_t row0, step0, unit, state;
  __device__ __forceinline__ ChunkUnit(unsigned vid, int len, int heads, int groups, int nchunks, int Q, int N) {
    h = (int)(vid % heads);
    const unsigned bc = vid / heads;
    c = (int)(bc % nchunks);
    b = (int)(bc / nchunks);
    g = h / (heads / groups);
    rows = min(Q, len - c * Q);
    row0 = (size_t)b * len + (size_t)c * Q;                       // of (B, L, ...)
    step0 = (((size_t)b * heads + h) * nchunks + c) * Q;          // of (B, H, nc, Q)
    unit = (size_t)bc * groups + g;                               // of the fragments
    state = (size_t)vid * (SSD_P * N);                            // of (B, nc, H, 64 N)
  }
};

// Eight rows x Q / 32 channels per thread of the 256: channel group tid % TPR, rows 8 (tid / TPR) ...
template <int Q> struct Staging {
  static constexpr int CPT = Q / 32, TPR = 64 / CPT, QMASK = Q >= 128 ? 15 : Q / 8 - 1;
};

template <typename E, int Q>
__device__ __forceinline__ void stage_transposed(E *xT, int tid, const V8<E> (&col)[Q / 32]) {
  using S = Staging<Q>;
  const int cg = tid % S::TPR, rg = tid / S::TPR;
#pragma unroll
  for (int i = 0; i < S::CPT; ++i) {
    const int p = cg * S::CPT + i;
    *reinterpret_cast<V8<E> *>(xT + p * Q + ((rg ^ (p & S::QMASK)) << 3)) = col[i];
  }
}
// Operand fragment of channels 32 pt .. and steps 16 ks ..
template <typename E, int Q>
__device__ __forceinline__ V8<E> staged_frag(const E *xT, int pt, int ks, int m, int g2) {
  return load_frag_e<E>(xT + (32 * pt + m) * Q + (((2 * ks + g2) ^ (m & Staging<Q>::QMASK)) << 3));
}

__device__ __forceinline__ void load8(const float *p, float (&v)[8]) {
  const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// ---------------------------------------------------------------------- states

struct SsdStatesParams {
  const void *x;                 // forward: x;  backward: dout
  const void *z;                 // backward: the gate, or null
  void *dy;                      // backward: dout silu(z) in the element type
  const void *frag;              // forward: Btblk;  backward: Ctblk
  const float *dA2, *dtv;
  float *states;
  int len, heads, groups, nchunks;
};

// 8 x2 float32 tiles per workgroup, 16 steps of two products per wave; 33 KB of LDS.
template <typename E, int Q, int N, bool BWD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void ssd_states_kernel(const SsdStatesParams p) {
  __shared__ __align__(16) E xT[SSD_P * Q];
  using S = Staging<Q>;
  constexpr int KS = Q >> 4, KN = N >> 4, NT = N >> 5, PW = NT >= 4 ? 2 : 1, AHEAD = BWD || KS < 8 ? 4 : 8;
  const ChunkUnit u(xcd_order(blockIdx.x, gridDim.x), p.len, p.heads, p.groups, p.nchunks, Q, N);
  const int wave = wave_id_uniform(), lane = lane_id(), tid = (int)threadIdx.x;
  const int m = lane & 31, g2 = lane >> 5;
  const int nt = PW == 2 ? wave : wave & 1, pt0 = PW == 2 ? 0 : wave >> 1;
  const int cg = tid % S::TPR, rg = tid / S::TPR;
  const unsigned pitch = (unsigned)p.heads * SSD_P * 2;                // bytes between rows
  const size_t at = (u.row0 * p.heads + u.h) * SSD_P;
  unsigned off[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) off[r] = (unsigned)min(8 * rg + r, u.rows - 1) * pitch + cg * S::CPT * 2;
  typedef Row<E, S::CPT> row_t;
  row_t raw[8], gate[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) raw[r] = *at_bytes<const row_t>(reinterpret_cast<const E *>(p.x) + at, off[r]);
  if (BWD && p.z) {
#pragma unroll
    for (int r = 0; r < 8; ++r) gate[r] = *at_bytes<const row_t>(reinterpret_cast<const E *>(p.z) + at, off[r]);
  }
  float w[8];
  load8(p.dA2 + u.step0 + 8 * rg, w);
  if (BWD) {
#pragma unroll
    for (int r = 0; r < 8; ++r) w[r] = 8 * rg + r < u.rows ? exp2_hw(w[r]) : 0.0f;
  } else {
    float dt[8];
    load8(p.dtv + u.step0 + 8 * rg, dt);
    const float end = p.dA2[u.step0 + Q - 1];
#pragma unroll
    for (int r = 0; r < 8; ++r) w[r] = dt[r] * exp2_hw(fminf(end - w[r], 0.0f));
  }
  if (BWD && p.z) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
#pragma unroll
      for (int i = 0; i < S::CPT; ++i) raw[r].v[i] = (E)((float)raw[r].v[i] * silu_f32((float)gate[r].v[i]));
    }
  }
  if (BWD && p.dy) {
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (8 * rg + r < u.rows) *at_bytes<row_t>(reinterpret_cast<E *>(p.dy) + at, off[r]) = raw[r];
  }
  const E *frag = reinterpret_cast<const E *>(p.frag) + (u.unit * KS * NT + nt) * SSD_FRAG + lane * 8;
  V8<E> f[AHEAD];
#pragma unroll
  for (int k = 0; k < AHEAD; ++k) f[k] = load_frag_e<E>(frag + k * NT * SSD_FRAG);
  V8<E> col[S::CPT];
#pragma unroll
  for (int i = 0; i < S::CPT; ++i) {
#pragma unroll
    for (int r = 0; r < 8; ++r) col[i][r] = (E)((float)raw[r].v[i] * w[r]);
  }
  stage_transposed<E, Q>(xT, tid, col);
  __syncthreads();
  f32x16_t acc[PW];
#pragma unroll
  for (int pt = 0; pt < PW; ++pt) acc[pt] = (f32x16_t){0};
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
    for (int pt = 0; pt < PW; ++pt) acc[pt] = mma(f[ks % AHEAD], staged_frag<E, Q>(xT, pt0 + pt, ks, m, g2), acc[pt]);
    if (ks + AHEAD < KS) f[ks % AHEAD] = load_frag_e<E>(frag + (ks + AHEAD) * NT * SSD_FRAG);
  }
  float *out = p.states + u.state;
#pragma unroll
  for (int pt = 0; pt < PW; ++pt) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<float4 *>(out + ((pt0 + pt) * KN + 2 * nt + (q >> 1)) * SSD_FRAG + (m + 32 * (q & 1)) * 8 + 4 * g2) =
          make_float4(acc[pt][4 * q], acc[pt][4 * q + 1], acc[pt][4 * q + 2], acc[pt][4 * q + 3]);
  }
}

// ---------------------------------------------------------------------- carry

struct SsdCarryParams {
  const float *added;            // (B, nc, H, dim) in fragment order: what each chunk adds
  void *states;                  // (B, nc, H, dim): the state entering each chunk, element type, fragment order
  uint16_t *low;                 // KEEP: the rest of those states' float32 (split_f32).  REV: H's, read
  const float *dA2;              // (B, H, nc, Q)
  const float *first;            // (B, H, P, N): the state before the first chunk (after the last one), or null
  float *last;                   // (B, H, P, N) or null
  const void *entering;          // REV: the forward's states H
  void *turned, *h_turned;       // REV: G and H as rows of 64 channels, (B, nc, H, N, 64): what ssd_dbc_dt_kernel reads
  float *through;                // REV: (B, H, nc, dim / 256) partial sums of exp(cs_Q) <G, H>
  int heads, nchunks, chunk, nstate;
  int runs;                      // REV: runs of chunks, a workgroup each; it carries the state through those in front of its own as well
};

// A float32 as its bfloat16, rounded to nearest, and the 16 bits that complete it: the operands of the matrix products and
// the number they were rounded from, in the bytes of the latter.  Below half a bfloat16 step the low bits stand above the
// rounded number, past it below; exactly half (either may be meant) moves by one float32 step towards the rounded one.
__device__ __forceinline__ void split_f32(float v, uint16_t &high, uint16_t &low) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  unsigned h = u >> 16, l = u & 0xffff;
  if (l == 0x8000) l = h & 1 ? 0x8001 : 0x7fff;
  if ((u & 0x7fffffff) > 0x7f800000) { h |= 0x40; l = 0; }               // NaN
  high = (uint16_t)(h + (l > 0x8000));
  low = (uint16_t)l;
}
__device__ __forceinline__ float join_f32(uint16_t high, uint16_t low) {
  return __builtin_bit_cast(float, ((unsigned)high << 16) + low - (low > 0x8000 ? 0x10000u : 0u));
}

// The 4 x 4 16-bit values of a quad of lanes, a row of four in each, turned: lane q takes column q.
__device__ __forceinline__ uint2 quad_turn(uint2 v) {
  const int q = lane_id() & 3;
  const unsigned got = __builtin_amdgcn_update_dpp(0, q & 2 ? v.x : v.y, 0x4e, 0xf, 0xf, true);      // lanes 2 3 0 1
  const unsigned a = q & 2 ? got : v.x, b = q & 2 ? v.y : got, pick = q & 1 ? 0x03020706u : 0x05040100u;
  const unsigned a1 = __builtin_amdgcn_update_dpp(0, a, 0xb1, 0xf, 0xf, true);                       // lanes 1 0 3 2
  const unsigned b1 = __builtin_amdgcn_update_dpp(0, b, 0xb1, 0xf, 0xf, true);
  return make_uint2(__builtin_amdgcn_perm(a1, a, pick), __builtin_amdgcn_perm(b1, b, pick));
}

// A thread carries 4 states of one channel over the chunks of its run; a quad of lanes holds four neighbouring channels, which
// turn their 4 x 4 among themselves for the copies with channels innermost that the backward stores, of G and of H.  The reads of
// eight chunks are in flight together.  Bound: memory where the calls are large (backwards 14 bytes a state and chunk: at 4 x
// 2048 steps, 24 heads, 128 states 88 MB in 19.3 us; forwards 10 us), one wave's chain from chunk to chunk where they are
// small.  With the 4 x 4 of a backward in one thread a quarter of the waves had four times the instructions each: there 22.0 us,
// at 1 x 3456, 34 heads 27.2 (now 16.2), 1 x 7040, 19 heads, 64 states, chunks of 128 87 (now 20), 1 x 569, 62 heads 8.9 (now 4.9).
template <typename E, bool REV, bool KEEP>                   // KEEP: for a backward
__global__ __launch_bounds__(256) void ssd_carry_kernel(const SsdCarryParams p) {
  constexpr int AHEAD = 8, PASS = 16;
  const int N = p.nstate, dim = SSD_P * N, per = dim >> 10, kn = N >> 4;
  // the workgroups with the most chunks in front of theirs start first
  const unsigned units = gridDim.x / (unsigned)(REV ? p.runs : 1), vid = REV ? blockIdx.x % units : blockIdx.x;
  const int run_at = REV ? p.runs - 1 - (int)(blockIdx.x / units) : 0;
  const int begin = REV ? (int)((long long)run_at * p.nchunks / p.runs) : 0;
  const int stop = REV ? (int)((long long)(run_at + 1) * p.nchunks / p.runs) : p.nchunks;
  const int part = (int)(vid % per), tid = part * 256 + (int)threadIdx.x;
  const size_t bh = vid / per;
  const int h = (int)(bh % p.heads);
  const size_t b = bh / p.heads;
  // element j of lane fl of fragment frag
  const int q = tid & 3, frag = tid >> 7, j = REV ? tid & 4 : (tid & 1) * 4, fl = REV ? (tid >> 3 & 15) * 4 + q : tid >> 1 & 63;
  const int e = frag * SSD_FRAG + fl * 8 + j, ch = 32 * (frag / kn) + (fl & 31), n = 16 * (frag % kn) + 8 * (fl >> 5) + j;
  const int turned = (n + q) * SSD_P + ch - q;
  const size_t user = (bh * SSD_P + ch) * N + n;
  const size_t pitch = (size_t)p.heads * dim, at = (b * p.nchunks * p.heads + h) * dim;
  const float *end = p.dA2 + bh * p.nchunks * p.chunk + p.chunk - 1;
  const auto chunk_of = [&](int i) { return REV ? p.nchunks - 1 - i : i; };
  float run[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) run[k] = p.first ? p.first[user + k] : 0.0f;
  const auto pass = [&](float f, const float4 &v) {
    const float add[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int s = 0; s < 4; ++s) run[s] = __builtin_fmaf(run[s], f, add[s]);
  };
  for (int i0 = 0; REV && i0 < begin; i0 += PASS) {
    float4 v[PASS];
    float a[PASS];
#pragma unroll
    for (int k = 0; k < PASS; ++k) {
      const int c = chunk_of(min(i0 + k, begin - 1));
      v[k] = *reinterpret_cast<const float4 *>(p.added + at + c * pitch + e);
      a[k] = end[(size_t)c * p.chunk];
    }
#pragma unroll
    for (int k = 0; k < PASS; ++k)
      if (i0 + k < begin) pass(exp2_hw(a[k]), v[k]);
  }
  for (int i0 = begin; i0 < stop; i0 += AHEAD) {
    float4 v[AHEAD];
    uint2 high[AHEAD], low[AHEAD];
    float a[AHEAD];
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) {
      const int c = chunk_of(min(i0 + k, stop - 1));
      const size_t o = at + c * pitch + e;
      v[k] = *reinterpret_cast<const float4 *>(p.added + o);
      if constexpr (REV) {
        high[k] = *reinterpret_cast<const uint2 *>(reinterpret_cast<const uint16_t *>(p.entering) + o);
        low[k] = *reinterpret_cast<const uint2 *>(p.low + o);
      }
      a[k] = end[(size_t)c * p.chunk];
    }
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) {
      const int i = i0 + k, c = chunk_of(i);
      if (i < stop) {
        const size_t o = at + c * pitch;
        const float f = exp2_hw(a[k]);
        if constexpr (!REV && KEEP) {
          Pack<uint16_t, 4> hi, lo;
#pragma unroll
          for (int s = 0; s < 4; ++s) split_f32(run[s], hi.v[s], lo.v[s]);
          *reinterpret_cast<Pack<uint16_t, 4> *>(reinterpret_cast<uint16_t *>(p.states) + o + e) = hi;
          *reinterpret_cast<Pack<uint16_t, 4> *>(p.low + o + e) = lo;
        } else {
          store4_e<E>(reinterpret_cast<E *>(p.states) + o + e, run);
        }
        if constexpr (REV) {
          const auto rounded = [](float lo, float hi) {
            return (unsigned)__builtin_bit_cast(uint16_t, (E)lo) | (unsigned)__builtin_bit_cast(uint16_t, (E)hi) << 16;
          };
          *reinterpret_cast<uint2 *>(reinterpret_cast<E *>(p.turned) + o + turned) = quad_turn(make_uint2(rounded(run[0], run[1]), rounded(run[2], run[3])));
          *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(p.h_turned) + o + turned) = quad_turn(high[k]);
          const unsigned hs[4] = {high[k].x & 0xffff, high[k].x >> 16, high[k].y & 0xffff, high[k].y >> 16};
          const unsigned ls[4] = {low[k].x & 0xffff, low[k].x >> 16, low[k].y & 0xffff, low[k].y >> 16};
          float through = 0.0f;
#pragma unroll
          for (int s = 0; s < 4; ++s) through = __builtin_fmaf(run[s], join_f32((uint16_t)hs[s], (uint16_t)ls[s]), through);
          through = wave_sum(through) * f;
          if (lane_id() == 0) p.through[(bh * p.nchunks + c) * (dim >> 8) + part * 4 + (threadIdx.x >> 6)] = through;
        }
        pass(f, v[k]);
      }
    }
  }
  if (p.last && stop == p.nchunks)
    *reinterpret_cast<float4 *>(p.last + user) = make_float4(run[0], run[1], run[2], run[3]);
}

// A backward's workgroup writes the states of a run of chunks; where there are fewer than one workgroup to two CUs the chunks
// are cut into several runs of at least 8, each of which reads what the chunks in front of it add once more and forms the
// same numbers.  1 x 4200 steps, 9 heads, 64 states, chunks of 128: 15.7 us in one run, 12.6 in four (11.6 in eight); 1 x 7040, 19 heads
// 23.2, 21.2 in three (20.0 in six).  More runs gained nothing more there and cost up to twice the time where chunks are few; the
// forward, which reads and writes less, gained nothing from any.
inline int carry_units(const SsdDims &d) { return d.batch * d.heads * (SSD_P * d.nstate / 1024); }
inline int carry_runs(const SsdDims &d) { return std::max(1, std::min(d.nchunks / 8, 256 / carry_units(d))); }

// ---------------------------------------------------------------------- scan

enum { SCAN_Y, SCAN_DZ, SCAN_DX };

struct SsdChunkScanParams {
  const void *op;                // rows of the in-chunk product: x, or dy for SCAN_DX
  const void *blk;               // fragments of C.B (transposed for SCAN_DX)
  const void *carry;             // fragments of C (of B for SCAN_DX)
  const void *states;            // H entering the chunks (G leaving them for SCAN_DX), element type, fragment order
  const float *dA2, *dtv, *Dk;
  const void *x, *dy, *z, *dout; // (B, L, H, 64) rows the last step reads
  void *out;                     // y, dz (or null) or dx
  float *sum0, *sum1;            // (B, H, nc, Q): SCAN_DZ <dy, y before skip>;  SCAN_DX <x, u> and <round(dt x), u>
  float *dD;                     // SCAN_DZ: (B, nc, H) sums of dy x, or null
  float *carried;                // SCAN_DZ: (B, H, nc) sums of <dy, what the state entering the chunk adds to y>
  int len, heads, groups, nchunks, d_per_p;
  int has_first;                 // a state enters the first chunk (leaves the last)
};

// Row blocks of 32 steps: a wave takes blocks NLB - 1 - i and i (NLB + 1 of the blocks on and below the diagonal
// whatever i is), both halves of the channels where there are four such pairs, else one half.  The decays multiply the
// elements of C.B in registers, in front of their product: on the diagonal one exp2 per element, below it
//   exp(cs_l - cs_s) = exp(cs_l - cs[end of the block before l's]) exp(.. - cs[end of s's block]) exp(.. - cs_s),
// a factor of each side from a table and a scalar per block (every factor at most 1).  With an exp2 per element
// everywhere the scan took 208 us at 4 x 4096 steps and 80 heads, so 199.  The accumulators (lane = step, registers =
// channels) go through LDS to whole rows for the last step: skip and gate, or dz and the row sums, or dx and its sums.
// SCAN_Y takes the step into that factor, so that x itself is the operand and each product is rounded once.
// SCAN_DZ and SCAN_DX take it into the staged x, and form the same rounded numbers C.B x decay: the difference of their
// row sums needs both to multiply the same block.
// SCAN_DZ forms dy from dout and z, which it reads for dz anyway, where reading the states kernel's dy back made it
// wait for a fourth tensor: 39.5 us before, 36.5 now (2 x 2048 steps, 24 heads, bfloat16).
template <typename E, int Q, int N, bool GRAD> struct ScanLds {
  // the carried state is through before the staged rows take its place
  __align__(16) E tile[SSD_P * (Q > N ? Q : N)];
  __align__(16) float dAs[Q];
  __align__(16) float Ps[Q], Rs[Q];                           // decay from the block before to a step, from a step to the end of its block
  __align__(16) float l2s[GRAD ? 4 : Q];                      // log2 dt
  float halves[Q < 256 && GRAD ? 4 * Q : 8];                  // row sums of half rows; or sums per wave
};

template <typename E, int Q, int N, int MODE, bool HAS_Z>
__device__ __forceinline__ void chunk_scan(const SsdChunkScanParams &p, unsigned vid, ScanLds<E, Q, N, MODE != SCAN_Y> &lds) {
  using S = Staging<Q>;
  constexpr int NLB = Q >> 5, KS = Q >> 4, KN = N >> 4, NPAIR = NLB / 2, PW = NPAIR >= 4 ? 2 : 1;
  E *tile = lds.tile, *xT = tile, *hs = tile;
  float *dAs = lds.dAs, *Ps = lds.Ps, *Rs = lds.Rs, *l2s = lds.l2s, *halves = lds.halves;
  const ChunkUnit u(vid, p.len, p.heads, p.groups, p.nchunks, Q, N);
  const int wave = wave_id_uniform(), lane = lane_id(), tid = (int)threadIdx.x;
  const int m = lane & 31, g2 = lane >> 5;
  const int pair = PW == 2 ? wave : wave >> 1, pt0 = PW == 2 ? 0 : wave & 1;
  const bool active = pair < NPAIR;
  const int rbs[2] = {NLB - 1 - pair, pair};
  const bool carried = MODE == SCAN_DX ? (u.c < p.nchunks - 1 || p.has_first) : (u.c > 0 || p.has_first);
  const int cg = tid % S::TPR, rg = tid / S::TPR;
  const unsigned pitch = (unsigned)p.heads * SSD_P * 2;                // bytes between rows
  const size_t at = (u.row0 * p.heads + u.h) * SSD_P;

  // ---- stage the rows and the carried state
  typedef Row<E, S::CPT> row_t;
  row_t raw[8];
#pragma unroll
  for (int r = 0; r < 8; ++r)
    raw[r] = *at_bytes<const row_t>(reinterpret_cast<const E *>(p.op) + at, (unsigned)min(8 * rg + r, u.rows - 1) * pitch + cg * S::CPT * 2);
  float w[8];
  if (MODE == SCAN_DZ) load8(p.dtv + u.step0 + 8 * rg, w);      // zero past the end
  // The blocks of this wave in the order of use: those below the diagonal of the first row block (nA of them), of the
  // second, then the two on the diagonal, second row block first: NLB + 1 steps whatever the wave, unrolled, so that
  // fragments can be requested AHEAD steps before their use without a register ever being copied.
  constexpr int AHEAD = MODE == SCAN_Y ? 4 : 2;
  const int nA = MODE == SCAN_DX ? NLB - 1 - rbs[0] : rbs[0];
  const E *bf = reinterpret_cast<const E *>(p.blk) + u.unit * NLB * KS * SSD_FRAG + lane * 8;
  V8<E> ring[AHEAD][2];
  const auto row_of = [&](int t) { return t < nA || t == NLB ? rbs[0] : rbs[1]; };
  const auto other_of = [&](int t) {
    return t >= NLB - 1 ? row_of(t) : (MODE == SCAN_DX ? row_of(t) + 1 : 0) + (t < nA ? t : t - nA);
  };
  const auto request = [&](int t) {
    const E *f = bf + (row_of(t) * KS + 2 * other_of(t)) * SSD_FRAG;
    ring[t % AHEAD][0] = load_frag_e<E>(f);
    ring[t % AHEAD][1] = load_frag_e<E>(f + SSD_FRAG);
  };
  // fragments of the carried product, CAHEAD of its KN steps ahead
  constexpr int CAHEAD = MODE == SCAN_Y ? (KN < 8 ? KN : 8) : 4;
  V8<E> fc[2][CAHEAD];
  const E *cf = reinterpret_cast<const E *>(p.carry) + u.unit * NLB * KN * SSD_FRAG + lane * 8;
  const auto request_carry = [&](int k) {
    fc[0][k % CAHEAD] = load_frag_e<E>(cf + (rbs[0] * KN + k) * SSD_FRAG);
    fc[1][k % CAHEAD] = load_frag_e<E>(cf + (rbs[1] * KN + k) * SSD_FRAG);
  };
  if (active && carried) {
#pragma unroll
    for (int k = 0; k < CAHEAD; ++k) request_carry(k);
  }
  if (tid < Q) {
    const float cs = p.dA2[u.step0 + tid];
    dAs[tid] = cs;
    const float before = tid < 32 ? 0.0f : p.dA2[u.step0 + (tid & ~31) - 1];
    Ps[tid] = exp2_hw(fminf(cs - before, 0.0f));
    float r = exp2_hw(fminf(__shfl(cs, lane | 31, WAVE) - cs, 0.0f));
    if (MODE == SCAN_Y) {
      const float dt = p.dtv[u.step0 + tid];
      r *= dt;
      l2s[tid] = log2_hw(dt);                                   // dt = 0: -inf, a weight of zero
    }
    Rs[tid] = r;
  }
  if (carried) {
    const E *st = reinterpret_cast<const E *>(p.states) + u.state;
#pragma unroll
    for (int i = 0; i < SSD_P * N / 2048; ++i)
      *reinterpret_cast<V8<E> *>(hs + (i * 256 + tid) * 8) = load_frag_e<E>(st + (i * 256 + tid) * 8);
  }
  __syncthreads();

  // ---- the carried state
  float carried_dy = 0.0f;
  f32x16_t acc[2][PW];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int pt = 0; pt < PW; ++pt) acc[i][pt] = (f32x16_t){0};
  }
  if (active && carried) {
#pragma unroll
    for (int k = 0; k < KN; ++k) {
#pragma unroll
      for (int pt = 0; pt < PW; ++pt) {
        const V8<E> h = load_frag_e<E>(hs + ((pt0 + pt) * KN + k) * SSD_FRAG + lane * 8);
        acc[0][pt] = mma(h, fc[0][k % CAHEAD], acc[0][pt]);
        acc[1][pt] = mma(h, fc[1][k % CAHEAD], acc[1][pt]);
      }
      if (k + CAHEAD < KN) request_carry(k + CAHEAD);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float own = dAs[32 * rbs[i] + m];
      const float f = exp2_hw(MODE == SCAN_DX ? fminf(dAs[Q - 1] - own, 0.0f) : own);
#pragma unroll
      for (int pt = 0; pt < PW; ++pt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][pt][r] *= f;
        if (MODE == SCAN_DZ) {
          const unsigned row = (unsigned)min(32 * rbs[i] + m, u.rows - 1) * pitch + (32 * (pt0 + pt) + 4 * g2) * 2;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float d[4];
            load4_e<E>(at_bytes<const E>(reinterpret_cast<const E *>(p.dy) + at, row + 16 * q), d);
#pragma unroll
            for (int j = 0; j < 4; ++j) carried_dy = __builtin_fmaf(d[j], acc[i][pt][4 * q + j], carried_dy);
          }
        }
      }
    }
    if (MODE == SCAN_DZ) asm volatile("" : "+v"(carried_dy));
  }
  if (active) {
#pragma unroll
    for (int t = 0; t < AHEAD && t <= NLB; ++t) request(t);
  }
  if (carried) __syncthreads();
  V8<E> col[S::CPT];
#pragma unroll
  for (int i = 0; i < S::CPT; ++i) {
#pragma unroll
    for (int r = 0; r < 8; ++r)
      col[i][r] = MODE == SCAN_DZ ? (E)((float)raw[r].v[i] * w[r])
                                  : MODE == SCAN_Y || 8 * rg + r < u.rows ? raw[r].v[i] : (E)0.0f;
  }
  stage_transposed<E, Q>(xT, tid, col);
  __syncthreads();

  const float head_D = p.Dk && !p.d_per_p ? p.Dk[u.h] : 0.0f;
  if (active) {
    // ---- the chunk's own steps
    const auto step = [&](int t, f32x16_t (&to)[PW], auto diagonal) {
      const int rb = row_of(t), ob = other_of(t);
      const int lb = MODE == SCAN_DX ? ob : rb, sb = MODE == SCAN_DX ? rb : ob;
      const float own = dAs[32 * rb + m];
      float lane_f = 0.0f;
      if (!diagonal.value)
        lane_f = (MODE == SCAN_DX ? Rs : Ps)[32 * rb + m] * exp2_hw(fminf(dAs[32 * lb - 1] - dAs[32 * sb + 31], 0.0f));
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        float d[8], v[8];
        const V8<E> f = ring[t % AHEAD][kk];
        const int o = 32 * ob + 16 * kk + 8 * g2;
        if constexpr (diagonal.value) {
          load8(dAs + o, d);
          if constexpr (MODE == SCAN_Y) {
            // dt_s exp(min(cs_l - cs_s, 0)) as one exponential: min(a, 0) + b = min(a + b, b)
            float l2[8];
            load8(l2s + o, l2);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              // a skip factor per head joins the diagonal: CB dt + D at s = l, rounded as one number
              const float skip = 16 * kk + 8 * g2 + j == m ? head_D : 0.0f;
              v[j] = __builtin_fmaf((float)f[j], exp2_hw(fminf(own + (l2[j] - d[j]), l2[j])), skip);
            }
          } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = (float)f[j] * exp2_hw(fminf(MODE == SCAN_DX ? d[j] - own : own - d[j], 0.0f));
          }
        } else {
          load8((MODE == SCAN_DX ? Ps : Rs) + o, d);
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = (float)f[j] * d[j] * lane_f;
        }
        const V8<E> wv = pack8_e<E>(v);
#pragma unroll
        for (int pt = 0; pt < PW; ++pt) to[pt] = mma(staged_frag<E, Q>(xT, pt0 + pt, 2 * ob + kk, m, g2), wv, to[pt]);
      }
      if (t + AHEAD <= NLB) request(t + AHEAD);
    };
    const auto swap = [&]() {
#pragma unroll
      for (int pt = 0; pt < PW; ++pt) {
        const f32x16_t v = acc[0][pt];
        acc[0][pt] = acc[1][pt];
        acc[1][pt] = v;
      }
    };
#pragma unroll
    for (int t = 0; t < NLB - 1; ++t) {
      if (t == nA) swap();
      step(t, acc[0], std::false_type{});
    }
    if (nA == NLB - 1) swap();             // acc[0] now belongs to the second row block
    step(NLB - 1, acc[0], std::true_type{});
    step(NLB, acc[1], std::true_type{});
  }
  __syncthreads();                       // the staged rows are through: their place turns accumulators into rows

  // ---- whole rows: a lane holds 8 channels of a row.  What a row block reads from memory is requested in front of the
  // work on the block before it.
  constexpr int LPR = 4 * PW, RPP = 64 / LPR, PASSES = 32 / RPP, SMASK = 8 * PW - 1;      // lanes per row, rows per pass
  constexpr bool Z = HAS_Z && MODE != SCAN_DX;
  float *stg = reinterpret_cast<float *>(tile) + wave * (32 * 32 * PW);
  const int c8 = lane % LPR, ch = 32 * pt0 + 8 * c8;
  const bool skip_rows = MODE == SCAN_Y && p.Dk && p.d_per_p;
  float D8[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) D8[j] = MODE != SCAN_Y ? head_D : skip_rows ? p.Dk[u.h * SSD_P + ch + j] : 0.0f;
  constexpr int AT_ONCE = MODE == SCAN_Y ? PASSES : MODE == SCAN_DZ ? (PASSES + 3) / 4 : PASSES / 2, GROUPS = PASSES / AT_ONCE;      // what the registers hold
  V8<E> rx[AT_ONCE], rdy[AT_ONCE], rz[AT_ONCE], rgo[AT_ONCE];
  float rdt[AT_ONCE];
  const auto request_rows = [&](int rb, int first) {
#pragma unroll
    for (int pass = 0; pass < AT_ONCE; ++pass) {
      const int l = 32 * rb + (first + pass) * RPP + lane / LPR;
      const unsigned ra = (unsigned)min(l, u.rows - 1) * pitch + ch * 2;
      if (MODE != SCAN_Y || skip_rows) rx[pass] = *at_bytes<const V8<E>>(reinterpret_cast<const E *>(p.x) + at, ra);
      if (MODE == SCAN_DX || (MODE == SCAN_DZ && !Z)) rdy[pass] = *at_bytes<const V8<E>>(reinterpret_cast<const E *>(p.dy) + at, ra);
      if (Z) rz[pass] = *at_bytes<const V8<E>>(reinterpret_cast<const E *>(p.z) + at, ra);
      if (Z && MODE == SCAN_DZ) rgo[pass] = *at_bytes<const V8<E>>(reinterpret_cast<const E *>(p.dout) + at, ra);
      if (MODE == SCAN_DX) rdt[pass] = p.dtv[u.step0 + l];
    }
  };
  float dyx = 0.0f;
  if (active) {
    request_rows(rbs[1], 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int pt = 0; pt < PW; ++pt) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4 *>(stg + m * 32 * PW + (((8 * pt + 2 * q + g2) ^ (m & SMASK)) << 2)) =
              make_float4(acc[i][pt][4 * q], acc[i][pt][4 * q + 1], acc[i][pt][4 * q + 2], acc[i][pt][4 * q + 3]);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int grp = 0; grp < GROUPS; ++grp) {
        V8<E> res[AT_ONCE];
        float s0[AT_ONCE], s1[AT_ONCE];
#pragma unroll
        for (int pass = 0; pass < AT_ONCE; ++pass) {
          const int lr = (grp * AT_ONCE + pass) * RPP + lane / LPR;
          const bool live = 32 * rbs[1 - i] + lr < u.rows;
          const float4 a0 = *reinterpret_cast<const float4 *>(stg + lr * 32 * PW + (((2 * c8) ^ (lr & SMASK)) << 2));
          const float4 a1 = *reinterpret_cast<const float4 *>(stg + lr * 32 * PW + (((2 * c8 + 1) ^ (lr & SMASK)) << 2));
          float v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
          const V8<E> x = rx[pass], dy = rdy[pass], z = rz[pass], go = rgo[pass];
          s0[pass] = 0.0f;
          s1[pass] = 0.0f;
          if (MODE == SCAN_Y) {
            if (skip_rows) {
#pragma unroll
              for (int j = 0; j < 8; ++j) v[j] = __builtin_fmaf(D8[j], (float)x[j], v[j]);
            }
            if (Z) {
#pragma unroll
              for (int j = 0; j < 8; ++j) v[j] *= silu_f32((float)z[j]);
            }
          } else if (MODE == SCAN_DZ) {
            float dyx_row = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const float xf = (float)x[j];
              if (Z) {
                const float zf = (float)z[j], sg = sigmoid_f32(zf), gf = (float)go[j], dyf = gf * (zf * sg);
                s0[pass] = __builtin_fmaf((float)(E)dyf, v[j], s0[pass]);       // dy as the states kernel rounds it
                dyx_row = __builtin_fmaf(dyf, xf, dyx_row);
                v[j] = gf * __builtin_fmaf(D8[j], xf, v[j]) * (sg * __builtin_fmaf(zf, 1.0f - sg, 1.0f));
              } else {
                s0[pass] = __builtin_fmaf((float)dy[j], v[j], s0[pass]);
                dyx_row = __builtin_fmaf((float)dy[j], xf, dyx_row);
              }
            }
            dyx += live ? dyx_row : 0.0f;
            asm volatile("" : "+v"(dyx));        // formed here: left to the compiler, all its terms wait for the end of the kernel
          } else {
            const float dt = rdt[pass];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const float xf = (float)x[j];
              s0[pass] = __builtin_fmaf(xf, v[j], s0[pass]);
              s1[pass] = __builtin_fmaf((float)(E)(xf * dt), v[j], s1[pass]);
              v[j] = __builtin_fmaf(dt, v[j], D8[j] * (float)dy[j]);
            }
          }
          res[pass] = pack8_e<E>(v);
          s0[pass] = live ? s0[pass] : 0.0f;
          s1[pass] = live ? s1[pass] : 0.0f;
        }
        if (grp + 1 < GROUPS) request_rows(rbs[1 - i], (grp + 1) * AT_ONCE);
        else if (i == 0) request_rows(rbs[0], 0);
#pragma unroll
        for (int pass = 0; pass < AT_ONCE; ++pass) {
          const int l = 32 * rbs[1 - i] + (grp * AT_ONCE + pass) * RPP + lane / LPR;
          if ((MODE != SCAN_DZ || Z) && l < u.rows)
            *at_bytes<V8<E>>(reinterpret_cast<E *>(p.out) + at, (unsigned)l * pitch + ch * 2) = res[pass];
          if (MODE == SCAN_Y) continue;
          if (PW == 2) {
            const float t0 = lane_run_sum_last<8>(s0[pass]), t1 = MODE == SCAN_DX ? lane_run_sum_last<8>(s1[pass]) : 0.0f;
            if (c8 == 7) {
              p.sum0[u.step0 + l] = t0;
              if (MODE == SCAN_DX) p.sum1[u.step0 + l] = t1;
            }
          } else {
            float t0 = s0[pass], t1 = s1[pass];
            t0 += dpp_move<DPP_ROW_SHR1, 0xf>(0.0f, t0);
            t0 += dpp_move<DPP_ROW_SHR2, 0xf>(0.0f, t0);
            t1 += dpp_move<DPP_ROW_SHR1, 0xf>(0.0f, t1);
            t1 += dpp_move<DPP_ROW_SHR2, 0xf>(0.0f, t1);
            if (c8 == 3) {
              halves[pt0 * Q + l] = t0;
              if (MODE == SCAN_DX) halves[(2 + pt0) * Q + l] = t1;
            }
          }
        }
      }
    }
  }
  if (MODE == SCAN_Y) return;
  if (PW == 1) {
    __syncthreads();
    if (tid < Q) {
      p.sum0[u.step0 + tid] = halves[tid] + halves[Q + tid];
      if (MODE == SCAN_DX) p.sum1[u.step0 + tid] = halves[2 * Q + tid] + halves[3 * Q + tid];
    }
  }
  if (MODE == SCAN_DZ) {
    const float t0 = wave_sum(dyx), t1 = wave_sum(carried_dy);
    __syncthreads();
    if (lane == 0) {
      halves[wave] = t0;
      halves[4 + wave] = t1;
    }
    __syncthreads();
    if (tid == 0 && p.dD) p.dD[(size_t)(u.b * p.nchunks + u.c) * p.heads + u.h] = (halves[0] + halves[1]) + (halves[2] + halves[3]);
    if (tid == 0) p.carried[u.step0 / Q] = (halves[4] + halves[5]) + (halves[6] + halves[7]);
  }
}

template <typename E, int Q, int N, bool HAS_Z>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void ssd_chunk_scan_kernel(const SsdChunkScanParams p) {
  __shared__ ScanLds<E, Q, N, false> lds;
  chunk_scan<E, Q, N, SCAN_Y, HAS_Z>(p, xcd_order(blockIdx.x, gridDim.x), lds);
}

// Both scans of a backward in one launch, neighbouring workgroups a unit's dz and dx: neither needs the other, and calls whose units do
// not fill the chip take little more time for both than for one.  3 x 896 steps, 18 heads, 128 states, chunks of 256: 23.3 us, in
// two launches 17.5 and 13.7; 1 x 7040, 19 heads, 64 states, chunks of 128 36.5, so 24.5 and 19.9; 4 x 2048, 24 heads 66 either way.
template <typename E, int Q, int N, bool HAS_Z>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void ssd_grad_scans_kernel(const SsdChunkScanParams dz, const SsdChunkScanParams dx) {
  __shared__ ScanLds<E, Q, N, true> lds;
  const unsigned vid = xcd_order(blockIdx.x, gridDim.x);
  if (vid & 1) chunk_scan<E, Q, N, SCAN_DX, false>(dx, vid >> 1, lds);
  else chunk_scan<E, Q, N, SCAN_DZ, HAS_Z>(dz, vid >> 1, lds);
}

}  // namespace ssm
