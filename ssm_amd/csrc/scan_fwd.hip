// C-ABI entry point of the forward selective scan: argument validation and
// kernel selection.  The kernels live in scan_fwd_kernel.hpp and are
// instantiated per activation dtype in scan_fwd_{f32,bf16,f16}.hip.
#include "scan_fwd_fast.hpp"

#include <numeric>

namespace ssm {

extern template int scan_fwd_dispatch<float>(const ScanFwdParams &, int, int, hipStream_t);
extern template int scan_fwd_dispatch<bf16_t>(const ScanFwdParams &, int, int, hipStream_t);
extern template int scan_fwd_dispatch<f16_t>(const ScanFwdParams &, int, int, hipStream_t);

extern template int scan_fwd_fast_dispatch<float, float>(const ScanFwdParams &, int, hipStream_t);
extern template int scan_fwd_fast_dispatch<bf16_t, bf16_t>(const ScanFwdParams &, int, hipStream_t);
extern template int scan_fwd_fast_dispatch<bf16_t, float>(const ScanFwdParams &, int, hipStream_t);
extern template int scan_fwd_fast_dispatch<f16_t, f16_t>(const ScanFwdParams &, int, hipStream_t);
extern template int scan_fwd_fast_dispatch<f16_t, float>(const ScanFwdParams &, int, hipStream_t);

// Rows up to which the chunks of a row run side by side in one workgroup (scan_fwd_split.hpp) rather than in turn, us at
// 16 states, side by side / in turn (grouped: scan_fwd_rows.hpp):
//   grouped, runs aligned, bf16: 1024 x 504 8.8 / 11.0, 2048 x 504 11.0 / 12.2, 1280 x 1024 15.5 / 17.6, 1536 x 1024 18.5 / 17.5,
//   1536 x 2048 27.6 / 29.6, 1280 x 4096 50.5 / 53.9, 1280 x 8192 95 / 102, 1536 x 8192 112 / 103; six chunks, whose waves share a
//   CU badly, 768 x 3072 29.4 / 35.7, 1024 x 3072 47 / 37.
//   float32: 1536 x 504 11.0 / 11.3, 2048 x 504 11.8 / 11.5, 1536 x 1024 16.2 / 17.1, 2048 x 1024 23.4 / 17.7, 1024 x 2048 25.3 / 25.3,
//   512 x 4096 34.7 / 43.9, 768 x 4096 51 / 44, 512 x 8192 67 / 83, 768 x 8192 99 / 83.
//   Every wave reads B and C itself there, and runs of odd rows at a lower rate: bf16 768 x 1021 14.2 / 16.1, 1280 x 1021 20.9 /
//   18.3, 1024 x 2045 26.3 / 27.5, 768 x 8111 80 / 90, 1024 x 8111 99 / 91; float32 1024 x 1021 16.0 / 16.0, 768 x 2045 21.3 / 25.3,
//   1024 x 2045 31.1 / 26.6, 512 x 8111 71 / 84, 768 x 8111 104 / 85.
//   Few channels to a group (a row per wave in turn): 1024 x 2048 float32 71 / 48, bf16 29 / 27, 1536 x 2048 38.5 / 37.9.
//   Constant projections: 256 x 2048 18.4 / 10.2, 512 x 8192 68 / 43, 512 x 1024 10.6 / 10.9, 1024 x 4096 41 / 43.
// (A single chunk has none beside it: up to those rows such a call goes a row to a wave, of which the x 504 figures are.)
// Over 1200 random grouped calls (1 to 8 x 12 to 2560 channels, 256 to 6000 steps, 1 to 16 states) what is chosen here and below
// took 1.9 % more in the mean than the fastest of the kernels that could have been, 6 % or less in nine calls of ten, 17 % in 99 of
// 100, 42 % at worst (2 x 402 x 2176 bf16: 39.8 side by side, 28.1 a row to a wave in turn).
static bool scan_fwd_splits(size_t rows, int len, bool varying, bool grouped, bool half, bool ragged) {
  const int chunks = (len + FAST_T - 1) / FAST_T;
  if (!varying) return chunks > 1 && rows <= (chunks > 2 ? 512 : 384);
  if (!grouped) return chunks > 1 && rows <= (ragged ? 512 : half ? 1536 : 1024);
  if (len <= FAST_T / 2 || (ragged && chunks == 1)) return false;      // ragged: 864 x 403 f16 13.4 / 11.1
  if (ragged) return rows <= (chunks <= 2 ? 896 : half ? (chunks <= 4 ? 1024 : 768) : (chunks <= 4 ? 832 : 512));
  if (chunks == 1) return rows <= (half ? 2048 : 1536);
  if (!half) return rows <= (chunks <= 2 ? 1536 : chunks <= 4 ? 1280 : 576);
  const int turns = (chunks + SPLIT_MAX_WAVES - 1) / SPLIT_MAX_WAVES, waves = (chunks + turns - 1) / turns;
  return rows <= (chunks <= 2 ? 1440 : chunks <= 4 ? 1536 : waves > 4 && waves < 8 ? 896 : 1280);
}

// Channels to a workgroup of scan_fwd_rows.hpp: those of the cheapest number of rounds of 256 workgroups.  A chunk costs a
// workgroup 6.2 us for every twelve rows, 4.0, 5.0 or 6.2 for the last four, eight or twelve, and 0.9 (4 chunks of bf16 with 4, 8,
// 12, 16, 24, 36, 48 rows on every CU: 27, 31, 36, 53, 61, 86, 111 us); the start of a workgroup another 3.
static int scan_fwd_rows_per_wg(int batch, int spans, int span, int chunks) {
  const size_t units = (size_t)batch * spans;
  const size_t least = (units * ((span + ROWS_MAX - 1) / ROWS_MAX) + 255) / 256;
  const double part[4] = {0.0, 4.0, 5.0, 6.2};
  double best = 0.0;
  int pick = 0;
  for (size_t k = least; k < least + 4; ++k) {
    const size_t blocks = k * 256 / units;                   // workgroups that a span may have
    const int rows = blocks <= 1 ? span : (int)((span + blocks - 1) / blocks);
    if (rows > ROWS_MAX) continue;
    const size_t rounds = (units * ((span + rows - 1) / rows) + 255) / 256;
    const double cost = (double)rounds * (3.0 + chunks * (0.9 + 6.2 * (rows / 12) + part[(rows % 12 + 3) / 4]));
    if (!pick || cost < best) {
      best = cost;
      pick = rows;
    }
    if (rows <= 4) break;
  }
  return pick ? pick : ROWS_MAX;
}

static bool valid_kind(int k) { return k == SSM_PROJ_DN || k == SSM_PROJ_BDN || k == SSM_PROJ_BGNL; }

}  // namespace ssm

extern "C" int ssm_scan_chunk_len(void) { return 512; }

#ifdef SSM_TEST_HOOKS
extern "C" int ssm_scan_fwd_rows_per_workgroup(int batch, int dim, int seqlen, int b_groups, int c_groups) {
  const int span = std::gcd(dim / b_groups, dim / c_groups);
  return ssm::scan_fwd_rows_per_wg(batch, dim / span, span, (seqlen + ssm::FAST_T - 1) / ssm::FAST_T);
}
#endif

extern "C" int ssm_scan_fwd(const ssm_scan_fwd_args *a, void *hip_stream) {
  using namespace ssm;
  SSM_REQUIRE(a != nullptr, SSM_ERR_NULL_POINTER, "ssm_scan_fwd: args is NULL");
  SSM_REQUIRE(a->u && a->delta && a->A && a->Bproj && a->Cproj && a->out, SSM_ERR_NULL_POINTER,
              "ssm_scan_fwd: u, delta, A, Bproj, Cproj and out are required");
  SSM_REQUIRE(a->batch > 0 && a->dim > 0 && a->seqlen > 0 && a->nstate > 0, SSM_ERR_BAD_SHAPE,
              "ssm_scan_fwd: batch=%d dim=%d seqlen=%d nstate=%d must all be positive", a->batch, a->dim,
              a->seqlen, a->nstate);
  SSM_REQUIRE(a->nstate <= SCAN_MAX_N, SSM_ERR_TOO_LARGE, "ssm_scan_fwd: nstate=%d exceeds %d", a->nstate,
              SCAN_MAX_N);
  SSM_REQUIRE(valid_dtype(a->io_dtype) && valid_dtype(a->bc_dtype), SSM_ERR_BAD_DTYPE,
              "ssm_scan_fwd: io_dtype=%d bc_dtype=%d", a->io_dtype, a->bc_dtype);
  SSM_REQUIRE(valid_kind(a->b_kind) && valid_kind(a->c_kind), SSM_ERR_BAD_KIND, "ssm_scan_fwd: b_kind=%d c_kind=%d",
              a->b_kind, a->c_kind);
  const bool bvary = a->b_kind == SSM_PROJ_BGNL, cvary = a->c_kind == SSM_PROJ_BGNL;
  if (bvary)
    SSM_REQUIRE(a->b_groups > 0 && a->dim % a->b_groups == 0, SSM_ERR_BAD_SHAPE,
                "ssm_scan_fwd: b_groups=%d must divide dim=%d", a->b_groups, a->dim);
  if (cvary)
    SSM_REQUIRE(a->c_groups > 0 && a->dim % a->c_groups == 0, SSM_ERR_BAD_SHAPE,
                "ssm_scan_fwd: c_groups=%d must divide dim=%d", a->c_groups, a->dim);
  const size_t rows_total = (size_t)a->batch * a->dim;
  SSM_REQUIRE(rows_total * (size_t)a->seqlen < ((size_t)1 << 40) && rows_total < ((size_t)1 << 31),
              SSM_ERR_TOO_LARGE, "ssm_scan_fwd: tensor too large");
  const int es = dtype_size(a->io_dtype), bs = dtype_size(a->bc_dtype);
  SSM_REQUIRE(aligned_to(a->u, es) && aligned_to(a->delta, es) && aligned_to(a->out, es) &&
                  (!a->z || aligned_to(a->z, es)) && (!a->last_state || aligned_to(a->last_state, es)) &&
                  aligned_to(a->Bproj, bs) && aligned_to(a->Cproj, bs) && aligned_to(a->A, 4) &&
                  (!a->Dskip || aligned_to(a->Dskip, 4)) && (!a->dt_bias || aligned_to(a->dt_bias, 4)),
              SSM_ERR_ALIGNMENT, "ssm_scan_fwd: a pointer is not aligned to its element size");

  ScanFwdParams p;
  p.u = a->u; p.delta = a->delta; p.z = a->z; p.Bp = a->Bproj; p.Cp = a->Cproj;
  p.A = a->A; p.Dk = a->Dskip; p.bias = a->dt_bias; p.out = a->out; p.last = a->last_state;
  p.chunk_states = a->chunk_states;
  p.batch = a->batch; p.dim = a->dim; p.len = a->seqlen; p.nstate = a->nstate;
  p.bc_dtype = a->bc_dtype;
  p.b_kind = a->b_kind; p.c_kind = a->c_kind;
  p.b_groups = bvary ? a->b_groups : 1; p.c_groups = cvary ? a->c_groups : 1;
  p.softplus = a->delta_softplus ? 1 : 0;
  p.vec_ok = ((size_t)a->seqlen * es) % 16 == 0 && aligned_to(a->u, 16) && aligned_to(a->delta, 16) &&
             aligned_to(a->out, 16) && (!a->z || aligned_to(a->z, 16));
  p.bc_vec_ok = a->seqlen % 4 == 0 && aligned_to(a->Bproj, 4 * bs) && aligned_to(a->Cproj, 4 * bs);

  // channels per workgroup: all must read the same B group and the same C group
  const int per_b = bvary ? a->dim / a->b_groups : a->dim;
  const int per_c = cvary ? a->dim / a->c_groups : a->dim;
  int rows = SCAN_MAX_WAVES;
  while (rows > 1 && (per_b % rows != 0 || per_c % rows != 0)) --rows;      // any divisor, not only powers of two

  // Two channels per wave (tune 1616) pay off once the grid still fills every CU twice.
  const bool pair_ok = bvary && cvary && a->nstate <= 16 && per_b % 16 == 0 && per_c % 16 == 0;
  SSM_CHECK_RESERVED("ssm_scan_fwd", a);
  int tune = SSM_RESERVED(a);               // 0 = automatic
  hipStream_t stream = reinterpret_cast<hipStream_t>(hip_stream);

  // The specialised kernels: time-varying B and C of one element type (that of the activations, or fp32), at most
  // 16 states.  A selector of 100000 + v asks for variant v.
  const bool aligned = p.vec_ok && a->seqlen < (1 << 29) && (!bvary || aligned_to(a->Bproj, 4 * bs)) && (!cvary || aligned_to(a->Cproj, 4 * bs));
  const bool fast_ok = bvary && cvary && a->nstate <= FAST_N && (a->bc_dtype == a->io_dtype || a->bc_dtype == SSM_F32);
  const bool const_ok = !bvary && !cvary && a->nstate <= FAST_N;
  const bool whole8 = (const_ok ? p.vec_ok && a->seqlen < (1 << 29) : aligned) && a->seqlen % 8 == 0;    // runs of 8 steps
  const bool whole16 = aligned && a->seqlen % 16 == 0;
  p.ragged = !whole8;
  const bool in_turn = tune >= 200000;      // a selector of 200000 + v: variant v, a row's chunks in turn however few the rows are
  if (in_turn) tune -= 100000;
  const bool half = a->io_dtype != SSM_F32;
  p.span = std::gcd(per_b, per_c);          // channels that share a group of B and one of C
  const int spans = a->dim / p.span, nchunks = (a->seqlen + FAST_T - 1) / FAST_T;
  p.split = !in_turn && scan_fwd_splits(rows_total, a->seqlen, !const_ok, p.span >= ROWS_MIN, half, p.ragged);
  if (tune == 0 && fast_ok) {
    int pick = 0;
    // (rows of at most 256 steps and few states: the general kernel, 3 x 1024 x 64 bf16 with 5 states 7.2 us against 8.5)
    if (p.span >= ROWS_MIN && a->seqlen >= 4 && a->seqlen < (1 << 28) && (a->seqlen > FAST_T / 2 || a->nstate > 8)) {
      // Any number of channels to a workgroup, but where
      //   few states leave little but the reads.  16-bit, aligned runs: a row to a wave, at most 9 states 0.82 of the time over 165
      //   random calls, 10 states 0.99, 12 1.03 (float32 1.02 to 1.14).  16-bit runs of any start: workgroups of 8 channels, at most
      //   4 states 0.91 over 44 calls of up to 4096 rows and three chunks (one state: any number of chunks), more rows 1.0.  Float32: 24
      //   channels on every CU 88 to 103 us against 102 to 109 (8 x 1536 x 2048), or workgroups of 8 (3 x 1072 x 640, one state, 9.6 / 12.4);
      //   two rows to a wave at once come out even (aligned 16-bit rows, 48 channels to a workgroup on every CU in every round:
      //   109.6 us against 111.0 at the headline shape);
      //   a single chunk would take a second turn for its last rows, or has no more than 8 on a CU: workgroups of 8 channels, two
      //   to a CU (aligned: 2 x 1984 x 448 f16 16.3 / 19.0, 8 x 384 x 448 bf16, 12 on a CU, 15.4 / 13.9, 8 x 256 x 448 10.4 / 12.2).
      pick = p.split ? 31041 : ROWS_VARIANT;
      const int even = half ? 48 : 24;
      const size_t wgs = rows_total / even;
      if (!p.split && a->seqlen > FAST_T / 2) {
        if (half && whole8 && aligned_to(a->Bproj, 16) && aligned_to(a->Cproj, 16) && a->nstate <= 9) pick = 31041;
        else if (half && !whole8 && p.span % 8 == 0 && a->nstate <= 4 && rows_total <= 4096 && (nchunks <= 3 || a->nstate == 1)) pick = 11082;
        else if (whole16 && p.span % even == 0 && wgs >= 256 && (half ? wgs % 256 == 0 : a->nstate <= 8)) pick = half ? 22123 : 12121;
        else if (whole16 && p.span % 8 == 0 && ((!half && a->nstate <= 2 && nchunks <= 4) ||
                                                (nchunks == 1 && rows_total <= 4096 && (rows_total <= 2048 || rows_total > 3072)))) pick = 11082;
      }
    } else if (per_b % 8 == 0 && per_c % 8 == 0 && a->seqlen > 256) {
      pick = p.split ? 31041 : 11082;
    } else if (a->seqlen > 256 || (per_b == 1 && per_c == 1)) {
      // groups of fewer than 8 channels (down to one per channel): nothing to share, a row per wave, which reads its runs of
      // B and C as 16-byte vectors.  (Rows of at most 256 steps fill half a chunk there: the general kernel, which has chunks of
      // 256, keeps them unless every channel has its own projections: 58 against 26 us, of 195 steps 119 against 63.)
      pick = 31041;
    }
    if (nchunks == 1) p.split = 0;          // nothing is beside a row's one chunk: 2 x 777 x 320 f16 10.0 us without what they exchange, 11.2 with
    if (pick == 31041) p.ragged = !(whole8 && aligned_to(a->Bproj, 16) && aligned_to(a->Cproj, 16));
    else if (pick != ROWS_VARIANT) p.ragged = !whole16;
    p.rows_per_wg = pick == ROWS_VARIANT ? scan_fwd_rows_per_wg(a->batch, spans, p.span, nchunks) : 0;
    if (pick) tune = 100000 + pick;
  }
  // Projections constant in time, (D, N) or (B, D, N): a row per wave with B and C in lanes (variant 31042).
  if ((tune == 0 && const_ok && a->seqlen > 256) || tune == 100000 + 31042) {
    SSM_REQUIRE(const_ok, SSM_ERR_BAD_KIND, "ssm_scan_fwd: selector %d needs constant projections and at most %d states",
                tune, FAST_N);
    switch (a->io_dtype) {
      case SSM_F32: return scan_fwd_fast_dispatch<float, float>(p, 31042, stream);
      case SSM_BF16: return scan_fwd_fast_dispatch<bf16_t, float>(p, 31042, stream);
      default: return scan_fwd_fast_dispatch<f16_t, float>(p, 31042, stream);
    }
  }
  if (tune >= 100000) {
    SSM_REQUIRE(fast_ok, SSM_ERR_BAD_KIND, "ssm_scan_fwd: selector %d needs the shape of the specialised kernel", tune);
    const int v = tune - 100000, per_wg = scan_fwd_fast_rows(v);
    SSM_REQUIRE(per_wg > 0 && per_b % per_wg == 0 && per_c % per_wg == 0, SSM_ERR_BAD_KIND,
                "ssm_scan_fwd: variant %d takes %d channels per workgroup, which must divide a group", v, per_wg);
    if (SSM_RESERVED(a)) {
      SSM_REQUIRE(per_wg == 1 || whole16, SSM_ERR_BAD_KIND, "ssm_scan_fwd: selector %d is for aligned rows of whole 16-step runs", tune);
      SSM_REQUIRE(v == 31041 || (a->seqlen >= 4 && a->seqlen < (1 << 28)), SSM_ERR_BAD_SHAPE,
                  "ssm_scan_fwd: selector %d is for rows of 4 to 2^28 - 1 steps", tune);
      p.rows_per_wg = v == ROWS_VARIANT ? scan_fwd_rows_per_wg(a->batch, spans, p.span, nchunks) : per_wg;
    }
    const bool bc32 = a->bc_dtype == SSM_F32;
    switch (a->io_dtype) {
      case SSM_F32: return scan_fwd_fast_dispatch<float, float>(p, v, stream);
      case SSM_BF16: return bc32 ? scan_fwd_fast_dispatch<bf16_t, float>(p, v, stream)
                                 : scan_fwd_fast_dispatch<bf16_t, bf16_t>(p, v, stream);
      default: return bc32 ? scan_fwd_fast_dispatch<f16_t, float>(p, v, stream)
                           : scan_fwd_fast_dispatch<f16_t, f16_t>(p, v, stream);
    }
  }
  if (tune == 0) {
    if (a->seqlen <= 256 && !a->chunk_states) tune = 408;
    else tune = a->nstate > 8 ? 816 : 808;
    if (tune != 408 && pair_ok) {
      // Several channels per wave share one staged B/C slab.  Two workgroups of 8 waves are resident per CU;
      // take the number of channels per wave whose grid leaves the fewest of those 512 places idle in its
      // last round (at B=8, D=1536: 3 -> 512 workgroups, one full round; 2 -> 768, the second round half empty).
      const int cand[4] = {3, 2, 4, 6};
      double best = 0.0;
      for (int i = 0; i < 4; ++i) {
        const int per_wg = cand[i] * SCAN_MAX_WAVES;
        if (per_b % per_wg != 0 || per_c % per_wg != 0) continue;
        const size_t wgs = (size_t)a->batch * a->dim / per_wg;
        if (wgs < 512) continue;
        const size_t rounds = (wgs + 511) / 512;
        const double fill = (double)wgs / (double)(rounds * 512);
        if (fill > best + 1e-9) {
          best = fill;
          tune = cand[i] * 800 + 16;
        }
      }
    }
  }
  if (tune == 1616 || tune == 2416 || tune == 3216 || tune == 4816) {        // 2, 3, 4, 6 channels per wave
    const int r = tune / 100;
    if (pair_ok && per_b % r == 0 && per_c % r == 0) rows = r;
    else tune = 816;
  }
  const int steps_per_lane = tune >= 1616 ? 8 : tune / 100;
  if (a->chunk_states)
    SSM_REQUIRE(steps_per_lane * WAVE == ssm_scan_chunk_len(), SSM_ERR_BAD_KIND,
                "ssm_scan_fwd: chunk_states needs a tiling of %d steps per chunk (selectors 808, 816 or 1616)",
                ssm_scan_chunk_len());
  switch (a->io_dtype) {
    case SSM_F32: return scan_fwd_dispatch<float>(p, tune, rows, stream);
    case SSM_BF16: return scan_fwd_dispatch<bf16_t>(p, tune, rows, stream);
    default: return scan_fwd_dispatch<f16_t>(p, tune, rows, stream);
  }
}
