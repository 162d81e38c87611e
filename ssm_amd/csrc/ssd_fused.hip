// The matrix-core forward of 16-bit Mamba-2 SSD calls: the launch that prepares what its kernels read besides x and z, and
// the entry point.  What follows the preparation is one walk over the sequence (ssd_walk.hip) or the call's chunks side by
// side (ssd_chunk.hip).
//
// Requires bf16 or fp16 tensors (the kernels are compiled per element type), P = 64, Q in {64, 128, 256}, N in {64, 128}.
#include "ssd_common.hpp"
#include "ssd_walk.hpp"
#include <algorithm>
#include <type_traits>

namespace ssm {

constexpr int FU_P = SSD_P;
constexpr int FRAG = SSD_FRAG;

template <typename E> using V4 = __attribute__((__vector_size__(4 * sizeof(E)))) E;

__device__ __forceinline__ void wave_lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// ---------------------------------------------------------------------- prep
// One launch prepares everything that the walk, or the kernels of the chunks side by side, read besides x and z; the
// workgroups (256 threads) take one of three roles by their index:
//
//  dt:   one workgroup per (b, c, 4 heads).  The (Q x 4) slab of dt is read row by
//        row (16 contiguous bytes per step) into LDS transposed to [head][step];
//        then one wave per head forms dt' = clamp(softplus(dt + bias)) and the
//        running sum of dt' A (stored scaled by log2 e, the unit of the kernels'
//        exponentials).  For the walk the sums start anew every 32 steps (prep_walk_dt_role).
//  pack: one workgroup per 32 steps of one (b, c, g): their rows of B and C go into LDS once, as 16-byte loads of whole
//        rows, and come out as operand fragments, transposed ones by ds_read_b64_tr_b16.  Fragment (lane, j) of a
//        32 x 16 block: row 32 rb + lane % 32, column 16 kb + 8 (lane / 32) + j.
//          Cblk [(b,c,g)][lb][kn]  from C  (rows = time, columns = state)
//          Btblk[(b,c,g)][ks][nt]  from B  (rows = state, columns = time)
//        and, where a backward will follow, Bblk and Ctblk with B and C in each other's place.
//  CB:   one wave per 32 x 32 block on or below the diagonal of C B^T of a chunk: both sets of rows as whole rows
//        through a wave-private LDS tile, MFMA over the state dimension, and through the tile again into
//          CBblk[(b,c,g)][lb][ks]  (rows = l, columns = s),
//        with zeros above the diagonal inside the diagonal blocks; for a backward also its transpose,
//          CBtblk[(b,c,g)][sb][kl]  (rows = s, columns = l).
// Steps past the end of a last chunk that is no whole one: size zero, rows of B and C zero.
// What bounds it is latency, and the lines that a load touches: with fragments read straight from the rows (a load touches 32
// of them, or two bytes of each of eight), a wave each, 4 x 2048 steps, 24 heads, everything a backward needs, took 14.4 us
// where this takes 8.9; 4 x 4096 steps, 80 heads, for the walk, 14.3 and 8.2; 3 x 4288, 11 heads 12.7 and 7.8; 1 x 3001, 24 heads
// 6.0 and 4.9.
// The walk takes the pack role with chunks of 32 steps, the first wave of each workgroup also the block of C B^T, and a
// fragment of C with its states in the order in which an accumulator's registers hold rows: (lane, j) = state 16 kn +
// 4 (lane / 32) + j, 8 further for j >= 4.  It is a kernel of its own: blocks of C B^T take 100 registers, without them 64 leave
// room for all of its workgroups at once (8.2 us against 10.2).
constexpr int PD_HEADS = 4, PW_HEADS = 32;     // heads of a workgroup of either dt role
struct SsdPrepParams {
  SsdCumsumParams cs;
  float *dA2;
  const void *Cm, *Bm;                   // element type of the call
  void *Cblk, *Btblk, *CBblk;
  void *Bblk, *Ctblk, *CBtblk;           // what the backward reads besides, or null
  unsigned n_dt, n_pack;                 // workgroups of the first two roles
  const int *seq_idx;                    // (B, L) sequence ids of a packed batch, or null
  float *steps, *ends;                   // what the walk takes from dt (SsdWalkParams); null: the chunks side by side
  size_t b_row, c_row;                   // elements between the (G, N) blocks of consecutive steps in Bm / Cm
};

// Packed sequences: the first step of a sequence gets an extra decay of 2^-64 (a jump in the running sum),
// so that nothing of the sequences before it - state or in-chunk terms - reaches it or the steps after it:
// exp2(cs_l - cs_s) then carries that factor whenever a boundary lies in (s, l].  The steps of one sequence
// see the same jumps on both sides of the difference; with every step a boundary the sum reaches 2^14 in a chunk of 256,
// where float32 still resolves 1e-3 of the exponent, and 2^11 in a block of the walk.  (Three boundaries in a block are more
// than the decays of one that factors: heads of such calls go element by element.)
constexpr float SEQ_JUMP_LN = -64.0f * 0.69314718056f;

// dt' = clamp(softplus(dt + bias)), and what a step adds to the running sum of dt' A beyond its product: the jump into a
// sequence at step t of batch row b.
__device__ __forceinline__ float prep_step(const SsdCumsumParams &p, float x) {
  if (p.softplus) x = softplus_f32(x);
  return fminf(fmaxf(x, p.dt_min), p.dt_max);
}
__device__ __forceinline__ float sequence_jump(const SsdPrepParams &pp, int b, size_t t) {
  const int *sid = pp.seq_idx + (size_t)b * pp.cs.d.len;
  return (t == 0 ? sid[0] != 0 : sid[t] != sid[t - 1]) ? SEQ_JUMP_LN : 0.0f;
}

__device__ __forceinline__ void prep_dt_role(const SsdPrepParams &pp, unsigned wg, float *lds) {
  float (*tile)[256 + 1] = reinterpret_cast<float (*)[256 + 1]>(lds);
  const SsdCumsumParams &p = pp.cs;
  const SsdDims &d = p.d;
  const int Q = d.chunk;
  const unsigned hgroups = (unsigned)(d.heads + PD_HEADS - 1) / PD_HEADS, rest = wg / hgroups;
  const int h0 = (int)(wg - rest * hgroups) * PD_HEADS, b = (int)(rest / (unsigned)d.nchunks), c = (int)rest - b * d.nchunks;
  const int wave = wave_id_uniform(), lane = lane_id(), h = h0 + wave;        // a wave a head
  const float A = p.A[min(h, d.heads - 1)], bias = p.bias ? p.bias[min(h, d.heads - 1)] : 0.0f;
#pragma unroll 4
  for (int e = threadIdx.x; e < Q * PD_HEADS; e += 256) {
    const int l = e / PD_HEADS, hh = e % PD_HEADS;
    float v = 0.0f;
    if (h0 + hh < d.heads && c * Q + l < d.len)
      v = load_as_f32(p.dt, p.dt_dtype, ((size_t)b * d.len + (size_t)c * Q + l) * d.heads + h0 + hh);
    tile[hh][l] = v;
  }
  __syncthreads();
  if (h >= d.heads) return;
  const int per = (Q + 63) >> 6;
  const int rows = min(Q, d.len - c * Q);          // steps past the end have size zero
  float v[4], run[4];
  float tot = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int l = lane * per + i;
    const bool live = i < per && l < rows;
    v[i] = live ? prep_step(p, tile[wave][l] + bias) : 0.0f;
    tot = __builtin_fmaf(v[i], A, tot);
    if (pp.seq_idx && live) tot += sequence_jump(pp, b, (size_t)c * Q + l);
    run[i] = tot;
  }
  const float excl = wave_inclusive_sum(tot) - tot;
  const size_t out = (((size_t)b * d.heads + h) * d.nchunks + c) * (size_t)Q;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int l = lane * per + i;
    if (i < per && l < Q) {
      p.dt_out[out + l] = v[i];
      pp.dA2[out + l] = (excl + run[i]) * LOG2E;
    }
  }
}

// 64 steps of 32 heads of dt, from (row, h0) on, into LDS as [head][65]; past the last step or head some other value.  A
// thread's reads are in flight together: the type is looked up once, not in front of each of them.
template <typename T>
__device__ __forceinline__ void stage_walk_dt(const void *dt, size_t row, int steps, int h0, int heads, float *tile) {
  T raw[PW_HEADS / 4];
  const int hh = (int)threadIdx.x % PW_HEADS, l0 = (int)threadIdx.x / PW_HEADS;
  const T *from = reinterpret_cast<const T *>(dt) + row * heads + min(h0 + hh, heads - 1);
#pragma unroll
  for (int i = 0; i < PW_HEADS / 4; ++i) raw[i] = from[(size_t)min(l0 + 8 * i, steps - 1) * heads];
#pragma unroll
  for (int i = 0; i < PW_HEADS / 4; ++i) tile[hh * 65 + l0 + 8 * i] = to_f32(raw[i]);
}

// For the walk: two blocks of 32 heads, whose 64 bytes of a row are read together.
// Bound by latency: 80 heads of 512 steps 4.8 us for the launch, 24 heads of 256 5.3 (8.5 and 6.8 with the reads of dt, A and
// bias one behind the other).
template <bool FACTORS>
__device__ __forceinline__ void prep_walk_dt_role(const SsdPrepParams &pp, unsigned wg, float *lds) {
  float (*tile)[64 + 1] = reinterpret_cast<float (*)[64 + 1]>(lds);
  const SsdCumsumParams &p = pp.cs;
  const SsdDims &d = p.d;
  const unsigned turns = (unsigned)ssd_walk_turns(d.nchunks), hgroups = (unsigned)(d.heads + PW_HEADS - 1) / PW_HEADS, rest = wg / hgroups;
  const int h0 = (int)(wg - rest * hgroups) * PW_HEADS, b = (int)(rest / (turns >> 1)), unit = (int)(rest - b * (turns >> 1));
  const int l0 = 64 * unit;
  const int wave = wave_id_uniform(), lane = lane_id();
  // lane k: what this wave's k-th head multiplies and adds
  const int lane_h = min(h0 + 4 * (lane % (PW_HEADS / 4)) + wave, d.heads - 1);
  const float A_lanes = p.A[lane_h], bias_lanes = p.bias ? p.bias[lane_h] : 0.0f;
  if (l0 < d.len) {
    const size_t row = (size_t)b * d.len + l0;
    if (p.dt_dtype == SSM_F32) stage_walk_dt<float>(p.dt, row, d.len - l0, h0, d.heads, lds);
    else if (p.dt_dtype == SSM_BF16) stage_walk_dt<bf16_t>(p.dt, row, d.len - l0, h0, d.heads, lds);
    else stage_walk_dt<f16_t>(p.dt, row, d.len - l0, h0, d.heads, lds);
  }
  __syncthreads();
  const bool live = l0 + lane < d.len;               // steps past the end have size zero
  const float jump = pp.seq_idx && live ? sequence_jump(pp, b, (size_t)l0 + lane) : 0.0f;
#pragma unroll 2
  for (int k = 0; k < PW_HEADS / 4; ++k) {
    const int hh = 4 * k + wave, h = h0 + hh;
    if (h >= d.heads) return;
    const float v = live ? prep_step(p, tile[hh][lane] + wave_read_lane(bias_lanes, k)) : 0.0f;
    const float cs = half_wave_inclusive_sum(__builtin_fmaf(v, wave_read_lane(A_lanes, k), jump)) * LOG2E;
    const float end = lane < SSD_WALK_BLOCK ? wave_read_lane(cs, SSD_WALK_BLOCK - 1) : wave_read_lane(cs, 2 * SSD_WALK_BLOCK - 1);
    const size_t at = ((size_t)b * d.heads + h) * turns + 2 * unit;           // block
    reinterpret_cast<float2 *>(pp.steps)[at * SSD_WALK_BLOCK + lane] = make_float2(FACTORS && walk_factors(end) ? cs - 0.5f * end : cs, v);
    if (lane % SSD_WALK_BLOCK == SSD_WALK_BLOCK - 1) pp.ends[at + lane / SSD_WALK_BLOCK] = end;
  }
}

// A 32 x 32 block of C B^T from the fragments of its rows, through `lds` (32 x 33), to CBblk and its transpose's place.
template <typename E, int KN>
__device__ __forceinline__ void prep_cb_block(const SsdPrepParams &pp, size_t unit, int lb, int sb, const V8<E> (&cf)[KN], const V8<E> (&bf)[KN], float *lds) {
  const int lane = lane_id(), m = lane & 31, g2 = lane >> 5, NLB = pp.cs.d.chunk >> 5, KS = pp.cs.d.chunk >> 4;
  f32x16_t acc = {0};
#pragma unroll
  for (int i = 0; i < KN; ++i) acc = mma(cf[i], bf[i], acc);
  float (*tile)[33] = reinterpret_cast<float (*)[33]>(lds);
#pragma unroll
  for (int r = 0; r < 16; ++r) tile[crow(r, g2)][m] = acc[r];
  wave_lds_sync();
  E *out = reinterpret_cast<E *>(pp.CBblk) + ((unit * NLB + lb) * KS + 2 * sb) * FRAG + lane * 8;
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int sl = 16 * kk + 8 * g2 + j;
      v[j] = (sb < lb || sl <= m) ? tile[m][sl] : 0.0f;
    }
    *reinterpret_cast<V8<E> *>(out + kk * FRAG) = pack8_e<E>(v);
  }
  if (!pp.CBtblk) return;
  E *out_t = reinterpret_cast<E *>(pp.CBtblk) + ((unit * NLB + sb) * KS + 2 * lb) * FRAG + lane * 8;
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int ll = 16 * kk + 8 * g2 + j;
      v[j] = (sb < lb || m <= ll) ? tile[ll][m] : 0.0f;
    }
    *reinterpret_cast<V8<E> *>(out_t + kk * FRAG) = pack8_e<E>(v);
  }
}

// What the pack role keeps of 32 steps of B and C in LDS: their rows, 16-byte pieces XOR-swizzled by the row.
template <int KN> struct PackTile {
  static constexpr int PIECES = 2 * KN, ROW = 16 * PIECES, BYTES = 32 * ROW;
  static __device__ __forceinline__ int at(int row, int piece) { return row * ROW + ((piece ^ (row & (PIECES - 1))) << 4); }
};
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short i16x4_t;

template <typename E, int KN, bool WALK>
__device__ __forceinline__ void prep_pack_role(const SsdPrepParams &pp, unsigned wg, unsigned char *lds) {
  using Tile = PackTile<KN>;
  const SsdDims &d = pp.cs.d;
  const int wave = wave_id_uniform(), lane = lane_id(), tid = (int)threadIdx.x;
  constexpr int N = 16 * KN, NT = N >> 5, EACH = 32 * Tile::PIECES / 256;
  const int Q = d.chunk, NLB = Q >> 5, len = d.len;
  const unsigned unit = wg / (unsigned)NLB, bc = unit / (unsigned)d.groups;
  const int lb = (int)(wg - unit * NLB), g = (int)(unit - bc * d.groups), b = (int)(bc / (unsigned)d.nchunks), c = (int)bc - b * d.nchunks;
  const int t0 = c * Q + 32 * lb;
  V8<E> raw[2][EACH];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const size_t stride = k ? pp.c_row : pp.b_row;
    const E *src = reinterpret_cast<const E *>(k ? pp.Cm : pp.Bm) + (size_t)b * len * stride + (size_t)g * N;
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int e = tid + 256 * i;
      raw[k][i] = load_frag_e<E>(src + (size_t)min(t0 + e / Tile::PIECES, len - 1) * stride + 8 * (e % Tile::PIECES));
    }
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int e = tid + 256 * i, row = e / Tile::PIECES;
      *reinterpret_cast<V8<E> *>(lds + k * Tile::BYTES + Tile::at(row, e % Tile::PIECES)) = t0 + row < len ? raw[k][i] : V8<E>{};
    }
  }
  __syncthreads();
  const int m = lane & 31, g2 = lane >> 5, k16 = lane & 15;
  const size_t base = (size_t)unit * NLB * KN;
  const auto put = [&](void *dst, int inner, const V8<E> &v) { *reinterpret_cast<V8<E> *>(reinterpret_cast<E *>(dst) + (base + inner) * FRAG + lane * 8) = v; };
  const auto rows = [&](const unsigned char *tile, void *dst, int i) {
    put(dst, lb * KN + i, load_frag_e<E>(tile + Tile::at(m, 2 * i + g2)));
  };
  const auto columns = [&](const unsigned char *tile, void *dst, int i) {
    typedef __attribute__((address_space(3))) i16x4_t *ptr;
    const int ks = i / NT, nt = i % NT, row = 16 * ks + 8 * g2 + (k16 >> 2), piece = 4 * nt + 2 * (lane >> 4 & 1) + ((k16 & 3) >> 1);
    struct { i16x4_t a, b; } r = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(tile + Tile::at(row, piece) + (k16 & 1) * 8)),
                                  __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(tile + Tile::at(row + 4, piece) + (k16 & 1) * 8))};
    put(dst, (2 * lb + ks) * NT + nt, __builtin_bit_cast(V8<E>, r));
  };
  const unsigned char *tb = lds, *tc = lds + Tile::BYTES;
#pragma unroll
  for (int i0 = 0; i0 < KN; i0 += 4) {
    const int i = i0 + wave;
    columns(tb, pp.Btblk, i);
    if constexpr (WALK) {
      const V4<E> lo = *reinterpret_cast<const V4<E> *>(tc + Tile::at(m, 2 * i) + 8 * g2), hi = *reinterpret_cast<const V4<E> *>(tc + Tile::at(m, 2 * i + 1) + 8 * g2);
      put(pp.Cblk, i, V8<E>{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
    } else {
      rows(tc, pp.Cblk, i);
    }
    if (!WALK && pp.Bblk) {
      rows(tb, pp.Bblk, i);
      columns(tc, pp.Ctblk, i);
    }
  }
  if (WALK && wave == 0) {
    V8<E> cf[KN], bf[KN];
#pragma unroll
    for (int i = 0; i < KN; ++i) {
      cf[i] = load_frag_e<E>(tc + Tile::at(m, 2 * i + g2));
      bf[i] = load_frag_e<E>(tb + Tile::at(m, 2 * i + g2));
    }
    prep_cb_block<E, KN>(pp, unit, 0, 0, cf, bf, reinterpret_cast<float *>(lds + 2 * Tile::BYTES));
  }
}

template <typename E, int KN>
__device__ __forceinline__ void prep_cb_role(const SsdPrepParams &pp, unsigned wg, unsigned char *lds) {
  using Tile = PackTile<KN>;
  const SsdDims &d = pp.cs.d;
  const int wave = wave_id_uniform(), lane = lane_id();
  constexpr int N = 16 * KN;
  const int Q = d.chunk, groups = d.groups;
  const int NLB = Q >> 5, KS = Q >> 4;
  const unsigned per_unit = (unsigned)NLB * (NLB + 1) / 2;
  const unsigned units = (unsigned)d.batch * d.nchunks * groups;
  const unsigned blk = wg * 4 + wave, unit32 = blk / per_unit;
  if (unit32 >= units) return;
  const size_t unit = unit32;
  const int idx = (int)(blk - unit32 * per_unit);
  int lb = 0;
  while ((lb + 1) * (lb + 2) / 2 <= idx) ++lb;
  const int sb = idx - lb * (lb + 1) / 2;
  const unsigned bc = unit32 / (unsigned)groups, b = bc / (unsigned)d.nchunks;
  const int g = (int)(unit32 - bc * groups), c = (int)(bc - b * d.nchunks);
  const size_t row0 = (size_t)b * d.len;                  // rows past the end stand for the last one: they meet only zeros
  const int m = lane & 31, g2 = lane >> 5, r0 = lane / Tile::PIECES, piece = lane % Tile::PIECES;
  const E *C = reinterpret_cast<const E *>(pp.Cm) + row0 * pp.c_row + (size_t)g * N + 8 * piece;
  const E *B = reinterpret_cast<const E *>(pp.Bm) + row0 * pp.b_row + (size_t)g * N + 8 * piece;
  unsigned char *tile = lds + wave * std::max(Tile::BYTES, 32 * 33 * 4);
  V8<E> craw[KN], braw[KN], cf[KN], bf[KN];
#pragma unroll
  for (int i = 0; i < KN; ++i) craw[i] = load_frag_e<E>(C + (size_t)min(c * Q + 32 * lb + r0 + 32 / KN * i, d.len - 1) * pp.c_row);
#pragma unroll
  for (int i = 0; i < KN; ++i) braw[i] = load_frag_e<E>(B + (size_t)min(c * Q + 32 * sb + r0 + 32 / KN * i, d.len - 1) * pp.b_row);
#pragma unroll
  for (int i = 0; i < KN; ++i) *reinterpret_cast<V8<E> *>(tile + Tile::at(r0 + 32 / KN * i, piece)) = craw[i];
  wave_lds_sync();
#pragma unroll
  for (int i = 0; i < KN; ++i) cf[i] = load_frag_e<E>(tile + Tile::at(m, 2 * i + g2));
  wave_lds_sync();
#pragma unroll
  for (int i = 0; i < KN; ++i) *reinterpret_cast<V8<E> *>(tile + Tile::at(r0 + 32 / KN * i, piece)) = braw[i];
  wave_lds_sync();
#pragma unroll
  for (int i = 0; i < KN; ++i) bf[i] = load_frag_e<E>(tile + Tile::at(m, 2 * i + g2));
  wave_lds_sync();
  prep_cb_block<E, KN>(pp, unit, lb, sb, cf, bf, reinterpret_cast<float *>(tile));
}

// Bytes of LDS: of dt 32 x 65 or 4 x 257 floats; of the pack role the rows of B and C and for the walk a tile of float32; of
// the blocks of C B^T a tile per wave.
constexpr int prep_lds_bytes(int KN, bool walk) {
  return walk ? 2 * 32 * 32 * KN + 32 * 33 * 4 : 4 * std::max(32 * 32 * KN, 32 * 33 * 4);
}

template <typename E, int KN, bool WALK>
__global__ __launch_bounds__(256) void ssd_fused_prep_kernel(const SsdPrepParams pp) {
  extern __shared__ __align__(16) unsigned char prep_lds[];
  const unsigned wg = blockIdx.x;
  // neighbours in a role, which read the same lines, on one XCD
  if (wg < pp.n_dt) {
    float *lds = reinterpret_cast<float *>(prep_lds);
    if constexpr (WALK) prep_walk_dt_role<std::is_same<E, __bf16>::value>(pp, xcd_order(wg, pp.n_dt), lds);
    else prep_dt_role(pp, xcd_order(wg, pp.n_dt), lds);
  } else if (WALK || wg < pp.n_dt + pp.n_pack) {
    prep_pack_role<E, KN, WALK>(pp, xcd_order(wg - pp.n_dt, pp.n_pack), prep_lds);
  } else if constexpr (!WALK) {
    prep_cb_role<E, KN>(pp, xcd_order(wg - pp.n_dt - pp.n_pack, gridDim.x - pp.n_dt - pp.n_pack), prep_lds);
  }
}

template <bool WALK>
static void launch_prep(const SsdPrepParams &pp, dim3 grid, size_t lds, bool f16, int nstate, hipStream_t s) {
  if (nstate == 128) {
    if (f16) hipLaunchKernelGGL((ssd_fused_prep_kernel<_Float16, 8, WALK>), grid, dim3(256), lds, s, pp);
    else hipLaunchKernelGGL((ssd_fused_prep_kernel<__bf16, 8, WALK>), grid, dim3(256), lds, s, pp);
  } else {
    if (f16) hipLaunchKernelGGL((ssd_fused_prep_kernel<_Float16, 4, WALK>), grid, dim3(256), lds, s, pp);
    else hipLaunchKernelGGL((ssd_fused_prep_kernel<__bf16, 4, WALK>), grid, dim3(256), lds, s, pp);
  }
}

static bool fused_shape_ok(const SsdDims &d) {
  const bool q_ok = d.chunk == 64 || d.chunk == 128 || d.chunk == 256;
  const bool n_ok = d.nstate == 64 || d.nstate == 128;
  if (!(q_ok && n_ok && d.hdim == FU_P && d.heads % d.groups == 0)) return false;
  // 32-bit byte offsets: inside one batch row of x, z and y, inside the per-step arrays and inside the fragment copies
  const size_t lim = (size_t)1 << 31;
  const SsdWorkLayout f = ssd_work_layout(d, false, true);
  return (size_t)d.nchunks * d.chunk * d.heads * FU_P * 2 < lim && f.Cblk - f.dt_out + (size_t)d.nchunks * d.chunk * 4 < lim &&
         f.Bblk - f.Cblk < lim;
}

}  // namespace ssm

static int fused_dims(const char *who, const ssm_ssd_dims *s, ssm::SsdDims &d) {
  using namespace ssm;
  SSM_REQUIRE(s, SSM_ERR_NULL_POINTER, "%s: dims is required", who);
  SSM_REQUIRE(s->batch > 0 && s->seqlen > 0 && s->heads > 0 && s->headdim > 0 && s->groups > 0 && s->nstate > 0 &&
                  s->chunk > 0,
              SSM_ERR_BAD_SHAPE, "%s: all of batch, seqlen, heads, headdim, groups, nstate, chunk must be positive", who);
  SSM_REQUIRE(s->heads % s->groups == 0, SSM_ERR_BAD_SHAPE, "%s: groups=%d must divide heads=%d", who, s->groups,
              s->heads);
  d.batch = s->batch; d.len = s->seqlen; d.heads = s->heads; d.hdim = s->headdim; d.groups = s->groups;
  d.nstate = s->nstate; d.chunk = s->chunk; d.nchunks = (s->seqlen + s->chunk - 1) / s->chunk;
  SSM_REQUIRE((size_t)d.batch * d.len * d.heads * d.hdim < ((size_t)1 << 40), SSM_ERR_TOO_LARGE, "%s: tensor too large",
              who);
  return SSM_OK;
}

extern "C" int ssm_ssd_combined_supported(const ssm_ssd_dims *dims, int io_dtype) {
  ssm::SsdDims d;
  if (fused_dims("ssm_ssd_combined_supported", dims, d) != SSM_OK) return 0;
  return (io_dtype == SSM_BF16 || io_dtype == SSM_F16) && ssm::fused_shape_ok(d) ? 1 : 0;
}

extern "C" size_t ssm_ssd_combined_workspace_bytes(const ssm_ssd_dims *dims) {
  ssm::SsdDims d;
  if (fused_dims("ssm_ssd_combined_workspace_bytes", dims, d) != SSM_OK) return 0;
#ifdef SSM_TEST_HOOKS
  return std::max(ssm::ssd_work_layout(d, false, true).total, ssm::ssd_work_layout(d, false, false).total);
#else
  return ssm::ssd_work_layout(d, false, ssm::ssd_side_by_side(d)).total;
#endif
}

extern "C" size_t ssm_ssd_combined_keep_bytes(const ssm_ssd_dims *dims) {
  ssm::SsdDims d;
  if (fused_dims("ssm_ssd_combined_keep_bytes", dims, d) != SSM_OK) return 0;
  return ssm::ssd_work_layout(d, true, true).total;
}

extern "C" size_t ssm_ssd_combined_scratch_bytes(const ssm_ssd_dims *dims) {
  ssm::SsdDims d;
  if (fused_dims("ssm_ssd_combined_scratch_bytes", dims, d) != SSM_OK) return 0;
  return ssm::ssd_added_bytes(d);
}

extern "C" int ssm_ssd_combined_fwd(const ssm_ssd_combined_args *a, void *hip_stream) {
  using namespace ssm;
  SSM_REQUIRE(a && a->x && a->dt && a->A && a->Bm && a->Cm && a->y, SSM_ERR_NULL_POINTER,
              "ssm_ssd_combined_fwd: x, dt, A, Bm, Cm and y are required");
  SSM_CHECK_RESERVED("ssm_ssd_combined_fwd", a);
  SsdDims d;
  int rc = fused_dims("ssm_ssd_combined_fwd", &a->dims, d);
  if (rc != SSM_OK) return rc;
  SSM_REQUIRE(a->io_dtype == SSM_BF16 || a->io_dtype == SSM_F16, SSM_ERR_BAD_DTYPE,
              "ssm_ssd_combined_fwd: x, z, y, Bm and Cm must be bf16 or fp16 (one type for all)");
  SSM_REQUIRE(valid_dtype(a->dt_dtype), SSM_ERR_BAD_DTYPE, "ssm_ssd_combined_fwd: dt_dtype=%d", a->dt_dtype);
  SSM_REQUIRE(fused_shape_ok(d), SSM_ERR_BAD_SHAPE,
              "ssm_ssd_combined_fwd: needs headdim 64, chunk in {64,128,256} and nstate in {64,128} "
              "(got headdim=%d chunk=%d nstate=%d)",
              d.hdim, d.chunk, d.nstate);
  const bool keep = a->keep_for_backward != 0;
  const bool side_by_side = keep || (SSM_RESERVED(a) ? SSM_RESERVED(a) == 2 : ssd_side_by_side(d));
  const SsdWorkLayout lay = ssd_work_layout(d, keep, side_by_side);
  SSM_REQUIRE(a->workspace && a->workspace_bytes >= lay.total, SSM_ERR_WORKSPACE,
              "ssm_ssd_combined_fwd: workspace of %zu bytes required", lay.total);
  SSM_REQUIRE(!keep || (a->scratch && a->scratch_bytes >= ssd_added_bytes(d) && aligned_to(a->scratch, 256)), SSM_ERR_WORKSPACE,
              "ssm_ssd_combined_fwd: keep_for_backward needs a scratch of %zu bytes, 256-byte aligned", ssd_added_bytes(d));
  SSM_REQUIRE(aligned_to(a->x, 16) && aligned_to(a->y, 16) && (!a->z || aligned_to(a->z, 16)) && aligned_to(a->Bm, 16) &&
                  aligned_to(a->Cm, 16) && aligned_to(a->workspace, 256) &&
                  (!a->Dskip || aligned_to(a->Dskip, a->d_per_p ? 16 : 4)) && (!a->final_states || aligned_to(a->final_states, 16)) &&
                  (!a->initial_states || aligned_to(a->initial_states, 4)),
              SSM_ERR_ALIGNMENT, "ssm_ssd_combined_fwd: tensors must be 16-byte aligned (workspace 256; a per-head Dskip 4)");
  hipStream_t s = reinterpret_cast<hipStream_t>(hip_stream);
  unsigned char *ws = reinterpret_cast<unsigned char *>(a->workspace);

  // the walk's blocks stand for chunks in the preparation
  SsdDims units = d;
  if (!side_by_side) {
    units.chunk = SSD_WALK_BLOCK;
    units.nchunks = ssd_walk_blocks(d.len);
  }
  const size_t bcg = (size_t)d.batch * units.nchunks * d.groups;
  const int NLB = units.chunk >> 5;
  SsdPrepParams pp{};
  SsdCumsumParams &cp = pp.cs;
  cp.dt = a->dt; cp.A = a->A; cp.bias = a->dt_bias;
  cp.dA_cs = nullptr;
  if (side_by_side) {
    cp.dt_out = reinterpret_cast<float *>(ws + lay.dt_out);
    pp.dA2 = reinterpret_cast<float *>(ws + lay.dA2);
  } else {
    pp.steps = reinterpret_cast<float *>(ws + lay.steps);
    pp.ends = reinterpret_cast<float *>(ws + lay.ends);
  }
  cp.d = units; cp.dt_dtype = a->dt_dtype; cp.softplus = a->dt_softplus ? 1 : 0; cp.dt_min = a->dt_min; cp.dt_max = a->dt_max;
  pp.Cm = a->Cm; pp.Bm = a->Bm;
  const size_t dense_row = (size_t)d.groups * d.nstate;
  SSM_REQUIRE(a->b_row_stride >= 0 && a->c_row_stride >= 0 && (a->b_row_stride == 0 || (size_t)a->b_row_stride >= dense_row) &&
                  (a->c_row_stride == 0 || (size_t)a->c_row_stride >= dense_row) && a->b_row_stride % 8 == 0 && a->c_row_stride % 8 == 0,
              SSM_ERR_BAD_SHAPE, "ssm_ssd_combined_fwd: b_row_stride=%lld c_row_stride=%lld must be 0 or at least groups * nstate=%zu, in multiples of 8",
              (long long)a->b_row_stride, (long long)a->c_row_stride, dense_row);
  pp.b_row = a->b_row_stride ? (size_t)a->b_row_stride : dense_row;
  pp.c_row = a->c_row_stride ? (size_t)a->c_row_stride : dense_row;
  void *Cblk = ws + lay.Cblk, *Btblk = ws + lay.Btblk;
  pp.Cblk = Cblk; pp.Btblk = Btblk; pp.CBblk = ws + lay.CBblk;
  if (keep) { pp.Bblk = ws + lay.Bblk; pp.Ctblk = ws + lay.Ctblk; pp.CBtblk = ws + lay.CBtblk; }
  const size_t n_dt = side_by_side ? (size_t)d.batch * d.nchunks * ((d.heads + PD_HEADS - 1) / PD_HEADS)
                                   : (size_t)d.batch * (ssd_walk_turns(units.nchunks) / 2) * ((d.heads + PW_HEADS - 1) / PW_HEADS);
  const size_t n_pack = bcg * NLB;
  const size_t n_cb = side_by_side ? (bcg * (NLB * (NLB + 1) / 2) + 3) / 4 : 0;
  SSM_REQUIRE(n_dt + n_pack + n_cb < ((size_t)1 << 29), SSM_ERR_TOO_LARGE, "ssm_ssd_combined_fwd: too many workgroups");
  pp.n_dt = (unsigned)n_dt; pp.n_pack = (unsigned)n_pack;
  pp.seq_idx = a->seq_idx;
  const bool f16 = a->io_dtype == SSM_F16;
  const dim3 prep_grid((unsigned)(n_dt + n_pack + n_cb));
  const size_t prep_lds = (size_t)prep_lds_bytes(d.nstate >> 4, !side_by_side);
  if (side_by_side) launch_prep<false>(pp, prep_grid, prep_lds, f16, d.nstate, s);
  else launch_prep<true>(pp, prep_grid, prep_lds, f16, d.nstate, s);
  SSM_CHECK_LAUNCH("ssm_ssd_combined_fwd(prep)");
  note_mfma_launch(side_by_side ? 16 : 8);
  if (side_by_side) return ssd_chunk_forward(*a, d, lay, s);

  SsdWalkParams wp{};
  wp.x = a->x; wp.z = a->z; wp.y = a->y;
  wp.steps = pp.steps; wp.ends = pp.ends; wp.Cblk = Cblk; wp.CBblk = ws + lay.CBblk; wp.Btblk = Btblk;
  wp.Dk = a->Dskip; wp.init = a->initial_states; wp.A = a->A; wp.final_states = a->final_states;
  wp.batch = d.batch; wp.len = d.len; wp.heads = d.heads; wp.groups = d.groups;
  wp.nblocks = units.nchunks; wp.turns = ssd_walk_turns(units.nchunks); wp.chunk_blocks = d.chunk / SSD_WALK_BLOCK;
  return ssd_walk_forward(wp, !a->Dskip ? 0 : (a->d_per_p ? 2 : 1), f16, d.nstate, s);
}
