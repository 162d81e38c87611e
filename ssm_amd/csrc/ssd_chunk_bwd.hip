// Backward of the side-by-side SSD (ssd_chunk.hpp) for bfloat16 calls:
//
//   states  dy = dout silu(z), rounded and kept; what each chunk adds to the adjoint state
//   carry   the adjoint state leaving each chunk, last to first, and what of <G, H> goes through each chunk
//   scans   y again for dz and its row sums;  u for dx and its row sums
//   dbc     dB and dC, every head of a group in one workgroup; and in the same launch
//   dt      the chain behind ddt, and the partial sums of dA, dD and the bias; one more launch adds those up
//
// What the forward prepared (steps, running sums, operand fragments, the states entering the chunks) is read, not formed again.
#include "ssd_chunk.hpp"

namespace ssm {

typedef __bf16 elem_t;

// ---------------------------------------------------------------------- dB, dC

// Inside a chunk dB and dC follow from one matrix, summed over the heads h of the group,
//   M[l,s] = sum_h dt_s exp(cs_l - cs_s) <dy_l, x_s>   (s <= l),      dC_l = sum_s M[l,s] B_s,   dB_s = sum_l M[l,s] C_l,
// and across chunk boundaries dC_l += sum_h exp(cs_l) dy_l.H_c,   dB_s += sum_h dt_s exp(cs_Q - cs_s) x_s.G_c.
struct SsdDbcParams {
  const elem_t *x, *dy;          // (B, L, H, 64)
  const elem_t *H, *G;           // states entering / adjoint states leaving the chunks, (B, nc, H, N, 64)
  const float *dA2, *dtv;
  const void *Btblk, *Ctblk;
  elem_t *dB, *dC;               // (B, L, G, N)
  int len, heads, groups, nchunks, units;      // units = batch * nchunks * groups
};

// A workgroup takes 64 rows of dC (or of dB) of one (batch, chunk, group) and walks the heads: the 64 own rows, all rows they
// meet (s <= l, or l >= s) and the state of the next head are on their way from L2 to registers while those of this head, in
// LDS, are multiplied (one barrier per head).  Wave w has the own tile w & 1 and, of the tiles it meets, every eighth (every
// fourth in shorter chunks); M stays in its accumulators, in float32, over all heads and is rounded once, for the product
// with B or C.  Rows are read whole (128 bytes a row) and turned into fragments by LDS, 16-byte pieces XOR-swizzled by pairs
// of rows: two rows are all banks.
// The 64-row cut keeps the reads at 2.5 times the tensors (32 rows: 4.5 times) with 8 such workgroups per chunk.
// Bound: the chain from one barrier to the next, one workgroup to a CU: fragments, four dependent products, weights, rows
// to LDS.  At 4 x 2048 steps, 24 heads, 128 states, chunks of 256 it takes 48.5 us; its loads without the arithmetic take
// 36, the arithmetic without the loads 43.  Before, 58.6: 8 waves hid less of the chain (57 with everything else as it is
// now), a swizzle by single rows left every read two to a bank (50.3), and 64-bit addresses, masks in scalars and both sides
// in one body took the registers that 16 waves do not have.  Tiles of a chunk's two ends paired, so that every workgroup
// meets as many: 48.7 here, 1.5 % more of a training step at three times the batch.
template <int Q> constexpr int DBC_WAVES = Q >= 256 ? 16 : 8;
template <int Q, int N, bool for_b>
__device__ __forceinline__ void dbc_rows(const SsdDbcParams &p, unsigned block, unsigned char *smem) {
  typedef V8<elem_t> v8;
  typedef const __attribute__((address_space(1))) char *global_bytes;
  typedef const __attribute__((address_space(1))) v8 *global_v8;
  typedef const __attribute__((address_space(1))) float *global_f32;
  constexpr int KS = Q >> 4, NT = N >> 5, NR = Q >> 6, QMASK = Staging<Q>::QMASK;
  constexpr int TILE = 64 * 64, BUF = (1 + NR) * TILE + N * 64;        // own rows, met rows, state
  constexpr int MW = DBC_WAVES<Q> / 2, MT = (2 * NR + MW - 1) / MW;      // waves an own tile has, tiles it meets in each
  constexpr int RPP = 8 * DBC_WAVES<Q>, MET = (64 * NR + RPP - 1) / RPP, ST = (N + RPP - 1) / RPP;     // rows read at a time
  elem_t *bufs = reinterpret_cast<elem_t *>(smem);                     // [2][BUF]
  float *steps = reinterpret_cast<float *>(smem + 2 * BUF * sizeof(elem_t));     // [2][4][Q]: running sum, log2 dt, P, R
  const int wave = wave_id_uniform(), lane = lane_id(), tid = (int)threadIdx.x;
  const int m = lane & 31, g2 = lane >> 5, ot = wave & 1, mw = wave >> 1;
  // the workgroups that meet the most rows start first
  const unsigned rank = block / (2u * p.units), rest = block % (2u * p.units);
  const unsigned unit = rest >> 1;
  const int r = for_b ? (int)rank : NR - 1 - (int)rank;
  const int meets = (int)(NR - rank);                                  // blocks of 64 rows
  const int g = (int)(unit % p.groups), bc = (int)(unit / p.groups), c = bc % p.nchunks, b = bc / p.nchunks;
  const int per = p.heads / p.groups, h0 = g * per;
  const int rows = min(Q, p.len - c * Q);
  if (64 * r >= rows) return;
  const size_t pitch = (size_t)p.heads * SSD_P;
  const size_t row0 = ((size_t)b * p.len + (size_t)c * Q) * pitch + h0 * SSD_P;
  const elem_t *own_src = (for_b ? p.x : p.dy) + row0, *met_src = (for_b ? p.dy : p.x) + row0;
  const elem_t *st_src = (for_b ? p.G : p.H) + ((size_t)bc * p.heads + h0) * (SSD_P * N);
  const size_t step0 = (((size_t)b * p.heads + h0) * p.nchunks + c) * Q, step_pitch = (size_t)p.nchunks * Q;
  const int met0 = for_b ? 64 * r : 0;                                 // first met row

  // ---- one head's operands, global -> registers -> LDS
  const int lr = tid >> 3, piece = tid & 7;                            // row of those read at a time, 16-byte piece
  const unsigned own_at = ((unsigned)min(64 * r + lr, rows - 1) * (unsigned)pitch + piece * 8) * 2;      // bytes
  unsigned met_at[MET];
#pragma unroll
  for (int k = 0; k < MET; ++k) met_at[k] = ((unsigned)min(met0 + RPP * k + lr, rows - 1) * (unsigned)pitch + piece * 8) * 2;
  v8 own_r, met_r[MET], st_r[ST];
  float cs_r = 0.0f, dt_r = 0.0f, cs_b = 0.0f;
  const auto fetch = [&](int h) {
    // scalar bases, formed anew for each head: a lane keeps 32-bit offsets alone
    global_bytes own_h = (global_bytes)(own_src + h * SSD_P), met_h = (global_bytes)(met_src + h * SSD_P);
    global_bytes st_h = (global_bytes)(st_src + (size_t)h * (SSD_P * N));
    global_bytes cs_h = (global_bytes)(p.dA2 + step0 + h * step_pitch), dt_h = (global_bytes)(p.dtv + step0 + h * step_pitch);
    asm volatile("" : "+s"(own_h), "+s"(met_h), "+s"(st_h), "+s"(cs_h), "+s"(dt_h));
    if (lr < 64) own_r = *(global_v8)(own_h + own_at);
#pragma unroll
    for (int k = 0; k < MET; ++k)
      if (RPP * k + lr < 64 * meets) met_r[k] = *(global_v8)(met_h + met_at[k]);
#pragma unroll
    for (int k = 0; k < ST; ++k)
      if (RPP * k + lr < N) st_r[k] = *(global_v8)(st_h + (RPP * k * 128 + (unsigned)tid * 16));
    if (tid < Q) {
      cs_r = *(global_f32)(cs_h + (unsigned)tid * 4);
      dt_r = *(global_f32)(dt_h + (unsigned)tid * 4);
      if (wave) cs_b = *(global_f32)(cs_h + (256 * wave - 4));
    }
  };
  const auto put = [&](int at) {
    elem_t *own = bufs + at * BUF, *met = own + TILE, *st = met + NR * TILE;
    if (lr < 64) *reinterpret_cast<v8 *>(own + lr * 64 + ((piece ^ (lr >> 1 & 7)) << 3)) = own_r;
#pragma unroll
    for (int k = 0; k < MET; ++k)
      if (RPP * k + lr < 64 * meets) *reinterpret_cast<v8 *>(met + (RPP * k + lr) * 64 + ((piece ^ (lr >> 1 & 7)) << 3)) = met_r[k];
#pragma unroll
    for (int k = 0; k < ST; ++k)
      if (RPP * k + lr < N) *reinterpret_cast<v8 *>(st + (RPP * k + lr) * 64 + ((piece ^ (lr >> 1 & 7)) << 3)) = st_r[k];
    if (tid < Q) {
      // decays from the block of 32 before to a step, and (times dt) from a step to the end of its block
      float *t = steps + 4 * at * Q + tid;
      const float before = __shfl(cs_r, 31, WAVE);
      t[0] = cs_r;
      t[Q] = log2_hw(dt_r);                                            // dt = 0: -inf, a weight of zero
      t[2 * Q] = exp2_hw(fminf(cs_r - (lane & 32 ? before : cs_b), 0.0f));
      t[3 * Q] = dt_r * exp2_hw(fminf(__shfl(cs_r, lane | 31, WAVE) - cs_r, 0.0f));
    }
  };
  const auto frag = [&](const elem_t *tile, int kp) { return load_frag_e<elem_t>(tile + (m * 64 + (((2 * kp + g2) ^ (m >> 1 & 7)) << 3))); };

  const auto load4 = [](const float *from, float (&v)[4]) {
    const float4 t = *reinterpret_cast<const float4 *>(from);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
  };
  f32x16_t M[MT], out = {0};
#pragma unroll
  for (int i = 0; i < MT; ++i) M[i] = (f32x16_t){0};
  const int own_row = 64 * r + 32 * ot + m;                            // of the chunk
  fetch(0);
  put(0);
  __syncthreads();
  for (int h = 0; h < per; ++h) {
    const int at = h & 1;
    if (h + 1 < per) fetch(h + 1);
    const elem_t *own = bufs + at * BUF, *met = own + TILE, *st = met + NR * TILE;
    const float *cs = steps + 4 * at * Q, *l2 = cs + Q, *P = l2 + Q, *R = P + Q;
    const float cs_own = cs[own_row], l2_own = l2[own_row];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int t = mw + MW * i, tile = (met0 >> 5) + t, mine = 2 * r + ot;
      if (t < 2 * meets && (for_b ? tile >= mine : tile <= mine)) {
        f32x16_t d = {0};
#pragma unroll
        for (int kp = 0; kp < 4; ++kp) d = mma(frag(met + 32 * t * 64, kp), frag(own + 32 * ot * 64, kp), d);
        // off the diagonal a factor per own row, a scalar per pair of blocks and a factor per met row (ssd_chunk.hpp)
        const int lb = for_b ? tile : mine, sb = for_b ? mine : tile;
        float f = 0.0f;
        int own_lane = m;
        asm volatile("" : "+v"(own_lane));                               // its 16 comparisons stay here: the scalars are few
        if (tile != mine) f = (for_b ? R : P)[own_row] * exp2_hw(fminf(cs[32 * lb - 1] - cs[32 * sb + 31], 0.0f));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = 32 * tile + 8 * q + 4 * g2;
          float w[4];
          if (tile == mine) {
            load4(cs + row, w);
            float l[4];
            if (!for_b) load4(l2 + row, l);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              // dt_s exp(min(cs_l - cs_s, 0)) as one exponential
              w[j] = for_b ? exp2_hw(fminf(w[j] - cs_own, 0.0f) + l2_own) : exp2_hw(fminf(cs_own - w[j], 0.0f) + l[j]);
              const int at = 8 * q + 4 * g2 + j;
              w[j] = (for_b ? at >= own_lane : at <= own_lane) ? w[j] : 0.0f;
            }
          } else {
            load4((for_b ? P : R) + row, w);
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] *= f;
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) M[i][4 * q + j] = __builtin_fmaf(w[j], d[4 * q + j], M[i][4 * q + j]);
        }
      }
    }
    if (mw < NT) {
      f32x16_t d = {0};
      int again = 32 * ot * 64;
      asm volatile("" : "+s"(again));                                    // read a second time, not kept in registers
#pragma unroll
      for (int kp = 0; kp < 4; ++kp) d = mma(frag(st + 32 * mw * 64, kp), frag(own + again, kp), d);
      const float w = for_b ? exp2_hw(fminf(cs[Q - 1] - cs_own, 0.0f) + l2_own) : exp2_hw(cs_own);
#pragma unroll
      for (int j = 0; j < 16; ++j) out[j] = __builtin_fmaf(w, d[j], out[j]);
    }
    if (h + 1 < per) put(at ^ 1);
    __syncthreads();
  }
  // ---- M, rounded, as an operand (rows = own, columns = met), times the columns of B (of C)
  elem_t *Ms = bufs;                                                   // [64][Q]
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int t = mw + MW * i, row = 32 * ot + m;
    if (t < 2 * meets) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float v[4] = {M[i][4 * q], M[i][4 * q + 1], M[i][4 * q + 2], M[i][4 * q + 3]};
        store4_e<elem_t>(Ms + row * Q + (((4 * t + q) ^ (row & QMASK)) << 3) + 4 * g2, v);
      }
    }
  }
  __syncthreads();
  if (mw >= NT) return;
  const elem_t *bt = reinterpret_cast<const elem_t *>(for_b ? p.Ctblk : p.Btblk) + (((size_t)unit * KS + (met0 >> 4)) * NT + mw) * SSD_FRAG + lane * 8;
  for (int ks = 0; ks < 4 * meets; ++ks) {
    const int row = 32 * ot + m;
    out = mma(load_frag_e<elem_t>(bt + ks * NT * SSD_FRAG),
              load_frag_e<elem_t>(Ms + row * Q + (((2 * ks + g2) ^ (row & QMASK)) << 3)), out);
  }
  if (own_row < rows) {
    elem_t *dst = (for_b ? p.dB : p.dC) + (((size_t)b * p.len + (size_t)c * Q + own_row) * p.groups + g) * N + 32 * mw + 4 * g2;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float v[4] = {out[4 * q], out[4 * q + 1], out[4 * q + 2], out[4 * q + 3]};
      store4_e<elem_t>(dst + 8 * q, v);
    }
  }
}

// ---------------------------------------------------------------------- dt

// With q_t = a_t <G_t, H_{t-1}>:  ddt_t = A q_t + <x_t, u_t>,  dA = sum dt_t q_t.  Inside a chunk q follows from row sums of the
// two scans, q_{t+1} = q_t + <dt_t x_t, u_t> - <dy_t, y_t>.  At a chunk's first step it is
//   exp(cs_Q) <G_c, H_c> + sum_l <dy_l, exp(cs_l) C_l.H_c>,
// the sum taken over the very terms that <dy_l, y_l> holds: what their 16-bit operands are off by leaves q again with each
// row it came from.  (From <G, H> at the boundary alone, the difference stayed in q over the whole chunk, long after the
// state had forgotten it, and was most of the error: in the 2-norm against float64, over 12 calls of 300 to 4096 steps, dA
// is off by 0.06 to 0.25 % and the bias by 0.2 to 0.5 %, where they were by 0.2 to 5 % and 0.7 to 3.6 %.)  <G, H> itself
// takes both in float32.
struct SsdDtParams {
  const float *s2, *xu, *s1;     // (B, H, nc, Q)
  const float *dtv;
  const float *through;          // (B, H, nc, parts) partial sums of exp(cs_Q) <G, H>
  const float *carried;          // (B, H, nc)
  const void *dt_raw;            // (B, L, H)
  const float *A, *bias;
  void *ddt;                     // (B, L, H)
  float *dA, *dbias;             // (B, nc, H) partial sums
  int len, heads, nchunks, parts, dt_dtype, softplus;
  float dt_min, dt_max;
};

// A workgroup takes a chunk of as many heads as it has waves, a wave one of them, each lane Q / 64 neighbouring steps.
template <int Q>
__device__ __forceinline__ void dt_rows(const SsdDtParams &p, unsigned block, unsigned char *smem) {
  constexpr int PER = Q / 64, DT_HEADS = DBC_WAVES<Q>, PITCH = Q + 1;
  float *tile = reinterpret_cast<float *>(smem);                       // [DT_HEADS][PITCH]
  const int hgroups = (p.heads + DT_HEADS - 1) / DT_HEADS;
  const int hg = (int)(block % hgroups), bc = (int)(block / hgroups), c = bc % p.nchunks, b = bc / p.nchunks;
  const int h0 = hg * DT_HEADS, rows = min(Q, p.len - c * Q);
  const size_t base = ((size_t)b * p.len + (size_t)c * Q) * p.heads + h0;
  const int hh = (int)threadIdx.x % DT_HEADS, l0 = (int)threadIdx.x / DT_HEADS;
  for (int l = l0; l < Q; l += 64)
    tile[hh * PITCH + l] = h0 + hh < p.heads && l < rows ? load_as_f32(p.dt_raw, p.dt_dtype, base + (size_t)l * p.heads + hh) : 0.0f;
  __syncthreads();
  const int wave = wave_id_uniform(), lane = lane_id();
  const int h = h0 + wave;
  float *row = tile + wave * PITCH;
  if (h < p.heads) {
    const size_t unit = ((size_t)b * p.heads + h) * p.nchunks + c, at = unit * Q + lane * PER;
    float s1[PER], s2[PER], xu[PER], dt[PER], d[PER], tot = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      s1[i] = p.s1[at + i];
      s2[i] = p.s2[at + i];
      xu[i] = p.xu[at + i];
      dt[i] = p.dtv[at + i];
    }
    const float a0 = p.carried[unit] + wave_sum(lane < p.parts ? p.through[unit * p.parts + lane] : 0.0f);
    const float A = p.A[h], bias = p.bias ? p.bias[h] : 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      d[i] = tot;
      tot += s1[i] - s2[i];
    }
    const float before = a0 + wave_prev(wave_inclusive_sum(tot), 0.0f);
    float dA = 0.0f, db = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int l = lane * PER + i;
      const float q = before + d[i];
      const float raw = row[l] + bias;
      const float v = p.softplus ? softplus_f32(raw) : raw;
      const float chain = v >= p.dt_min && v <= p.dt_max ? (p.softplus ? sigmoid_f32(raw) : 1.0f) : 0.0f;
      const float g = l < rows ? __builtin_fmaf(A, q, xu[i]) * chain : 0.0f;
      dA = l < rows ? __builtin_fmaf(dt[i], q, dA) : dA;
      db += g;
      row[l] = g;
    }
    dA = wave_sum(dA);
    db = wave_sum(db);
    if (lane == 0) {
      p.dA[(size_t)bc * p.heads + h] = dA;
      p.dbias[(size_t)bc * p.heads + h] = db;
    }
  }
  __syncthreads();
  if (h0 + hh < p.heads)
    for (int l = l0; l < rows; l += 64) store_any(p.ddt, p.dt_dtype, base + (size_t)l * p.heads + hh, tile[hh * PITCH + l]);
}

// Both in one launch: the workgroups of dt, of which there are few and short ones, start first, and those of dbc that meet the fewest rows
// wait for their CUs.  At 4 x 2048 steps, 24 heads, 128 states, chunks of 256 52.6 us, in two launches 51.7 and 7.1; 2 x 2048, 48 heads, 64
// states 43.3, so 43.1 and 7.0.
template <int Q> constexpr unsigned dt_blocks(const SsdDims &d) {
  return (unsigned)(d.batch * d.nchunks * ((d.heads + DBC_WAVES<Q> - 1) / DBC_WAVES<Q>));
}
template <int Q, int N>
__global__ __launch_bounds__(64 * DBC_WAVES<Q>) void ssd_dbc_dt_kernel(const SsdDbcParams p, const SsdDtParams t, unsigned first) {
  extern __shared__ __align__(16) unsigned char smem[];
  if (blockIdx.x < first) return dt_rows<Q>(t, blockIdx.x, smem);
  const unsigned block = blockIdx.x - first;
  if (block & 1) dbc_rows<Q, N, true>(p, block, smem);
  else dbc_rows<Q, N, false>(p, block, smem);
}

// ---------------------------------------------------------------------- host

struct BwdLayout {
  size_t dy, added, states, turned, h_turned, s2, xu, s1, through, carried, dA, dbias, dD, total;
};

static BwdLayout bwd_layout(const SsdDims &d) {
  BwdLayout f;
  const size_t units = (size_t)d.batch * d.nchunks * d.heads;
  size_t at = 0;
  const auto take = [&](size_t bytes) { const size_t v = at; at += ssd_align_up(bytes); return v; };
  f.dy = take((size_t)d.batch * d.len * d.heads * SSD_P * 2);
  f.added = take(units * SSD_P * d.nstate * 4);
  f.states = take(units * SSD_P * d.nstate * 2);
  f.turned = take(units * SSD_P * d.nstate * 2);
  f.h_turned = take(units * SSD_P * d.nstate * 2);
  f.s2 = take(units * d.chunk * 4);
  f.xu = take(units * d.chunk * 4);
  f.s1 = take(units * d.chunk * 4);
  f.through = take(units * (SSD_P * d.nstate / 256) * 4);
  f.carried = take(units * 4);
  f.dA = take(units * 4);
  f.dbias = take(units * 4);
  f.dD = take(units * 4);
  f.total = at;
  return f;
}

static SsdDims plain_dims(const ssm_ssd_dims &s) {
  SsdDims d;
  d.batch = s.batch; d.len = s.seqlen; d.heads = s.heads; d.hdim = s.headdim; d.groups = s.groups;
  d.nstate = s.nstate; d.chunk = s.chunk; d.nchunks = (s.seqlen + s.chunk - 1) / s.chunk;
  return d;
}

static bool bwd_shape_ok(const ssm_ssd_dims *s, int io_dtype) {
  if (!s || io_dtype != SSM_BF16 || !ssm_ssd_combined_supported(s, io_dtype)) return false;
  const SsdDims d = plain_dims(*s);
  // a chunk's rows are addressed by 32-bit offsets
  return (size_t)d.batch * d.nchunks * d.heads < ((size_t)1 << 26) && (size_t)d.chunk * d.heads * SSD_P < ((size_t)1 << 31);
}

template <int Q, int N>
static int backward_launches(const SsdStatesParams &st, const SsdCarryParams &ca, const SsdChunkScanParams &dz,
                             const SsdChunkScanParams &dx, const SsdDbcParams &bc, const SsdDtParams &dt, const SsdDims &d,
                             hipStream_t s) {
  const dim3 units((unsigned)(d.batch * d.nchunks * d.heads)), block(256);
  constexpr size_t dbc_lds = 2 * ((1 + Q / 64) * 64 * 64 + N * 64) * sizeof(elem_t) + 8 * Q * sizeof(float);
  static_assert(dbc_lds >= DBC_WAVES<Q> * (Q + 1) * sizeof(float));
  if (allow_dynamic_lds(ssd_dbc_dt_kernel<Q, N>, dbc_lds) != hipSuccess) {
    set_error("ssm_ssd_combined_bwd: cannot reserve %zu bytes of LDS", dbc_lds);
    return SSM_ERR_LAUNCH;
  }
  hipLaunchKernelGGL((ssd_states_kernel<elem_t, Q, N, true>), units, block, 0, s, st);
  hipLaunchKernelGGL((ssd_carry_kernel<elem_t, true, true>), dim3((unsigned)(carry_units(d) * ca.runs)), block, 0, s, ca);
  const dim3 both(2 * units.x);
  if (dz.z) hipLaunchKernelGGL((ssd_grad_scans_kernel<elem_t, Q, N, true>), both, block, 0, s, dz, dx);
  else hipLaunchKernelGGL((ssd_grad_scans_kernel<elem_t, Q, N, false>), both, block, 0, s, dz, dx);
  const unsigned first = dt_blocks<Q>(d), all = first + 2u * bc.units * (Q / 64);
  hipLaunchKernelGGL((ssd_dbc_dt_kernel<Q, N>), dim3(all), dim3(64 * DBC_WAVES<Q>), dbc_lds, s, bc, dt, first);
  return SSM_OK;
}

}  // namespace ssm

extern "C" int ssm_ssd_combined_bwd_supported(const ssm_ssd_dims *dims, int io_dtype) { return ssm::bwd_shape_ok(dims, io_dtype) ? 1 : 0; }

extern "C" size_t ssm_ssd_combined_bwd_workspace_bytes(const ssm_ssd_dims *dims) {
  return ssm::bwd_shape_ok(dims, SSM_BF16) ? ssm::bwd_layout(ssm::plain_dims(*dims)).total : 0;
}

extern "C" int ssm_ssd_combined_bwd(const ssm_ssd_combined_bwd_args *a, void *hip_stream) {
  using namespace ssm;
  SSM_REQUIRE(a && a->fwd.x && a->fwd.dt && a->fwd.A && a->fwd.workspace && a->dout && a->dx && a->dB && a->dC && a->ddt && a->dA,
              SSM_ERR_NULL_POINTER, "ssm_ssd_combined_bwd: x, dt, A, the forward's workspace, dout, dx, dB, dC, ddt and dA are required");
  const ssm_ssd_combined_args &f = a->fwd;
  SSM_REQUIRE(bwd_shape_ok(&f.dims, f.io_dtype) && !f.seq_idx && !f.d_per_p && f.keep_for_backward, SSM_ERR_BAD_SHAPE,
              "ssm_ssd_combined_bwd: needs a bf16 forward run with keep_for_backward, a shape ssm_ssd_combined_bwd_supported accepts, "
              "no seq_idx and no per-channel Dskip");
  SSM_REQUIRE(valid_dtype(f.dt_dtype), SSM_ERR_BAD_DTYPE, "ssm_ssd_combined_bwd: dt_dtype=%d", f.dt_dtype);
  const SsdDims d = plain_dims(f.dims);
  const SsdWorkLayout kept = ssd_work_layout(d, true, true);
  const BwdLayout lay = bwd_layout(d);
  SSM_REQUIRE(f.workspace_bytes >= kept.total && a->workspace && a->workspace_bytes >= lay.total, SSM_ERR_WORKSPACE,
              "ssm_ssd_combined_bwd: workspaces of %zu (kept) and %zu bytes required", kept.total, lay.total);
  SSM_REQUIRE((f.z != nullptr) == (a->dz != nullptr), SSM_ERR_NULL_POINTER, "ssm_ssd_combined_bwd: dz is given exactly with z");
  SSM_REQUIRE(aligned_to(f.x, 16) && aligned_to(a->dout, 16) && (!f.z || aligned_to(f.z, 16)) && aligned_to(a->dx, 16) &&
                  (!a->dz || aligned_to(a->dz, 16)) && aligned_to(a->dB, 8) && aligned_to(a->dC, 8) && aligned_to(f.workspace, 256) &&
                  aligned_to(a->workspace, 256) && (!a->dinitial_states || aligned_to(a->dinitial_states, 16)),
              SSM_ERR_ALIGNMENT, "ssm_ssd_combined_bwd: tensors must be 16-byte aligned (workspaces 256)");
  hipStream_t s = reinterpret_cast<hipStream_t>(hip_stream);
  const unsigned char *kw = reinterpret_cast<const unsigned char *>(f.workspace);
  unsigned char *ws = reinterpret_cast<unsigned char *>(a->workspace);
  const float *dA2 = reinterpret_cast<const float *>(kw + kept.dA2), *dtv = reinterpret_cast<const float *>(kw + kept.dt_out);
  const auto f32 = [&](size_t off) { return reinterpret_cast<float *>(ws + off); };

  SsdStatesParams st{};
  st.x = a->dout; st.z = f.z; st.dy = ws + lay.dy; st.frag = kw + kept.Ctblk; st.dA2 = dA2; st.dtv = dtv; st.states = f32(lay.added);
  st.len = d.len; st.heads = d.heads; st.groups = d.groups; st.nchunks = d.nchunks;
  SsdCarryParams ca{};
  ca.runs = carry_runs(d);
  ca.added = f32(lay.added); ca.states = ws + lay.states; ca.turned = ws + lay.turned; ca.dA2 = dA2; ca.first = a->dfinal; ca.last = a->dinitial_states; ca.entering = kw + kept.states; ca.through = f32(lay.through);
  ca.low = const_cast<uint16_t *>(reinterpret_cast<const uint16_t *>(kw + kept.states_low)); ca.h_turned = ws + lay.h_turned;
  ca.heads = d.heads; ca.nchunks = d.nchunks; ca.chunk = d.chunk; ca.nstate = d.nstate;
  SsdChunkScanParams dz{};
  dz.op = f.x; dz.blk = kw + kept.CBblk; dz.carry = kw + kept.Cblk; dz.states = kw + kept.states; dz.dA2 = dA2; dz.dtv = dtv; dz.Dk = f.Dskip;
  dz.x = f.x; dz.dy = ws + lay.dy; dz.z = f.z; dz.dout = a->dout; dz.out = a->dz; dz.sum0 = f32(lay.s2);
  dz.carried = f32(lay.carried); dz.dD = f.Dskip ? f32(lay.dD) : nullptr; dz.len = d.len; dz.heads = d.heads; dz.groups = d.groups; dz.nchunks = d.nchunks;
  dz.has_first = f.initial_states != nullptr;
  SsdChunkScanParams dx = dz;
  dx.op = ws + lay.dy; dx.blk = kw + kept.CBtblk; dx.carry = kw + kept.Bblk; dx.states = ws + lay.states; dx.z = nullptr; dx.out = a->dx;
  dx.sum0 = f32(lay.xu); dx.sum1 = f32(lay.s1); dx.dD = nullptr; dx.has_first = a->dfinal != nullptr;
  SsdDbcParams bc{};
  bc.x = reinterpret_cast<const elem_t *>(f.x); bc.dy = reinterpret_cast<const elem_t *>(ws + lay.dy); bc.H = reinterpret_cast<const elem_t *>(ws + lay.h_turned); bc.G = reinterpret_cast<const elem_t *>(ws + lay.turned);
  bc.dA2 = dA2; bc.dtv = dtv; bc.Btblk = kw + kept.Btblk; bc.Ctblk = kw + kept.Ctblk;
  bc.dB = reinterpret_cast<elem_t *>(a->dB); bc.dC = reinterpret_cast<elem_t *>(a->dC);
  bc.len = d.len; bc.heads = d.heads; bc.groups = d.groups; bc.nchunks = d.nchunks; bc.units = d.batch * d.nchunks * d.groups;
  SsdDtParams dt{};
  dt.s2 = f32(lay.s2); dt.xu = f32(lay.xu); dt.s1 = f32(lay.s1); dt.dtv = dtv; dt.through = f32(lay.through); dt.carried = f32(lay.carried); dt.dt_raw = f.dt;
  dt.A = f.A; dt.bias = f.dt_bias; dt.ddt = a->ddt; dt.dA = f32(lay.dA); dt.dbias = f32(lay.dbias);
  dt.len = d.len; dt.heads = d.heads; dt.nchunks = d.nchunks; dt.parts = SSD_P * d.nstate / 256; dt.dt_dtype = f.dt_dtype;
  dt.softplus = f.dt_softplus ? 1 : 0; dt.dt_min = f.dt_min; dt.dt_max = f.dt_max;

  int rc = SSM_OK;
#define SSM_CHUNK_BACKWARD(QQ, NN) \
  if (d.chunk == QQ && d.nstate == NN) rc = backward_launches<QQ, NN>(st, ca, dz, dx, bc, dt, d, s);
  SSM_CHUNK_BACKWARD(256, 128) SSM_CHUNK_BACKWARD(128, 128) SSM_CHUNK_BACKWARD(64, 128)
  SSM_CHUNK_BACKWARD(256, 64) SSM_CHUNK_BACKWARD(128, 64) SSM_CHUNK_BACKWARD(64, 64)
#undef SSM_CHUNK_BACKWARD
  if (rc != SSM_OK) return rc;
  FoldJobs jobs{};
  const int parts = d.batch * d.nchunks;
  jobs.add(f32(lay.dA), a->dA, 1, parts, (size_t)d.heads, SSM_F32);
  if (a->ddt_bias) jobs.add(f32(lay.dbias), a->ddt_bias, 1, parts, (size_t)d.heads, SSM_F32);
  if (a->dD && f.Dskip) jobs.add(f32(lay.dD), a->dD, 1, parts, (size_t)d.heads, SSM_F32);
  launch_fold_jobs(jobs, s);
  SSM_CHECK_LAUNCH("ssm_ssd_combined_bwd");
  return SSM_OK;
}
