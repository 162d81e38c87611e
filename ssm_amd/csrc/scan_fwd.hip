// C-ABI entry point of the forward selective scan: argument validation and
// kernel selection.  The kernels live in scan_fwd_kernel.hpp and are
// instantiated per activation dtype in scan_fwd_{f32,bf16,f16}.hip.
#include "scan_fwd_fast.hpp"

namespace ssm {

extern template int scan_fwd_dispatch<float>(const ScanFwdParams &, int, int, hipStream_t);
extern template int scan_fwd_dispatch<bf16_t>(const ScanFwdParams &, int, int, hipStream_t);
extern template int scan_fwd_dispatch<f16_t>(const ScanFwdParams &, int, int, hipStream_t);

extern template int scan_fwd_fast_dispatch<float, float>(const ScanFwdParams &, int, hipStream_t);
extern template int scan_fwd_fast_dispatch<bf16_t, bf16_t>(const ScanFwdParams &, int, hipStream_t);
extern template int scan_fwd_fast_dispatch<bf16_t, float>(const ScanFwdParams &, int, hipStream_t);
extern template int scan_fwd_fast_dispatch<f16_t, f16_t>(const ScanFwdParams &, int, hipStream_t);
extern template int scan_fwd_fast_dispatch<f16_t, float>(const ScanFwdParams &, int, hipStream_t);

// Rows up to which the chunks of a row run side by side in one workgroup (scan_fwd_split.hpp) rather than in turn; us at
// 16 states in turn / side by side:
//   grouped, float32, 512 x 2048 31.7 / 15.0, 768 x 8192 109 / 93, 1024 x 2048 30.7 / 25.7, 1024 x 4096 58 / 67,
//   1280 x 2048 32 / 29.9, 1536 x 1024 18.1 / 16.7, 1536 x 2048 32.8 / 33.7;
//   bf16 512 x 2048 32.2 / 13.8, 1280 x 1024 16.6 / 14.3, 1280 x 8192 104 / 93.5, 3 x 512 x 1024 21.2 / 19.6, x 2048 29.0 /
//   27.7, x 4096 63.0 / 61.8, x 8192 118 / 117; with 4 states x 4096 31.5 / 27.0, x 8192 56 / 49.
//   float32 of few states, whose rows two waves do not share (below): 1024 x 4096, 1 state 25.5 / 23.0.
//   Every wave reads B and C itself there, and runs of odd rows at a lower rate: float32 512 x 2047 33 / 23, 768 x 2047
//   33 / 42, bf16 768 x 2047 32 / 27, 768 x 1021 18.6 / 19.5, 768 x 3000 48 / 67.
//   Few channels to a group (a row per wave in turn): 1024 x 2048 float32 71 / 48, bf16 29 / 27, 1536 x 2048 38.5 / 37.9.
//   Constant projections: 256 x 2048 18.4 / 10.2, 512 x 8192 68 / 43, 512 x 1024 10.6 / 10.9, 1024 x 4096 41 / 43.
static bool scan_fwd_splits(size_t rows, int len, bool varying, bool grouped, bool half, bool ragged, bool few) {
  if (len <= FAST_T) return false;
  if (!varying) return rows <= (len > 2 * FAST_T ? 512 : 384);
  const bool to_four = len > 2 * FAST_T && len <= 4 * FAST_T;       // chunks
  if (ragged) return rows <= (grouped && half && to_four ? 768 : 512);
  if (!grouped) return rows <= (half ? 1536 : 1024);
  if (half) return rows <= 1536;
  return rows <= (len <= 2 * FAST_T ? 1536 : len <= 4 * FAST_T ? 1280 : few ? 1024 : 768);
}

static bool valid_kind(int k) { return k == SSM_PROJ_DN || k == SSM_PROJ_BDN || k == SSM_PROJ_BGNL; }

}  // namespace ssm

extern "C" int ssm_scan_chunk_len(void) { return 512; }

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
  // 16 states.  Rows that are not aligned whole 16-step runs take their RAGGED form.  A selector of 100000 + v asks for
  // variant v.
  const bool whole_rows = p.vec_ok && a->seqlen % 16 == 0 && a->seqlen < (1 << 29) && (!bvary || aligned_to(a->Bproj, 4 * bs)) &&
                          (!cvary || aligned_to(a->Cproj, 4 * bs));
  const bool fast_ok = bvary && cvary && a->nstate <= FAST_N && (a->bc_dtype == a->io_dtype || a->bc_dtype == SSM_F32);
  const bool const_ok = !bvary && !cvary && a->nstate <= FAST_N;
  p.ragged = const_ok ? !(p.vec_ok && a->seqlen % 8 == 0 && a->seqlen < (1 << 29)) : !whole_rows;
  const bool in_turn = tune >= 200000;      // a selector of 200000 + v: variant v, a row's chunks in turn however few the rows are
  if (in_turn) tune -= 100000;
  const bool half = a->io_dtype != SSM_F32, few = a->nstate <= 4;
  p.split = !in_turn && scan_fwd_splits(rows_total, a->seqlen, !const_ok, per_b % 8 == 0 && per_c % 8 == 0, half, p.ragged, few);
  // Rows of at most 256 steps fill half a chunk there; the general kernel, which has chunks of 256, keeps them (6720 rows of
  // 256 bf16 20 us against 33) unless every channel has its own projections: 58 against 26 us, of 195 119 against 63.
  if (tune == 0 && fast_ok && (a->seqlen > 256 || (per_b == 1 && per_c == 1))) {
    // The variant whose workgroups (48, 24 or 8 channels of one group) still give every CU its share:
    // two rows per wave with 16-step runs and two slabs where 256 such workgroups exist, else 8-step runs at six waves
    // per SIMD, else the smallest workgroup.
    const size_t total = (size_t)a->batch * a->dim;
    // float32 activations: the 8-step runs at six waves per SIMD come out ahead (142.9 against 149.6 us at the
    // headline shape, where twice the bytes per step leave more to wait for); 16-bit: the 16-step runs (120.5 / 133.3)
    const int pref16[3] = {22123, 12121, 11082}, pref32[3] = {12121, 22123, 11082};
    const int *pref = a->io_dtype == SSM_F32 ? pref32 : pref16;
    int pick = p.split ? 31041 : 0;
    for (int i = 0; i < 3 && !pick; ++i) {
      const int per_wg = scan_fwd_fast_rows(pref[i]);
      if (per_b % per_wg == 0 && per_c % per_wg == 0 && (total / per_wg >= 256 || i == 2)) pick = pref[i];
    }
    // its rows by two waves each where that leaves a CU no more than one such workgroup, there are chunks to walk (1920 rows of
    // 16 states, us with one / two, 1024 steps 19.1 / 18.8, 2048 40.4 / 33.6, 8192 139 / 112, bf16 17.0 / 16.8, 32.1 / 29.3,
    // 129 / 106) and states enough that halving them is worth forming a row's steps twice: 2 x 640 x 1030 float32 with 1, 4, 8,
    // 16 states 13.4 / 14.7, 16.1 / 17.3, 21.5 / 21.3, 32.1 / 29.5, bf16 (runs of any start) 12.2 / 14.9, 14.9 / 17.4, 20.0 /
    // 21.4, 29.9 / 29.2; 4 states, aligned, 2 x 640 x 4096 31.8 / 32.8, 3 x 512 x 4096 34.8 / 33.6, 2 x 640 x 8192 68.9 / 63.5
    const bool halves = p.ragged ? a->nstate > (half ? 8 : 4) : a->nstate > 4 || (a->nstate > 2 && total * a->seqlen >= (size_t)6 << 20);
    if (pick == 11082 && total <= 2048 && a->seqlen > 2 * FAST_T && halves) pick = 11162;
    // groups of fewer than 8 channels (down to one per channel): nothing to share, a row per wave, which reads its runs of
    // B and C as 16-byte vectors
    if (!pick) pick = 31041;
    if (pick == 31041 && !(aligned_to(a->Bproj, 16) && aligned_to(a->Cproj, 16) && ((size_t)a->seqlen * bs) % 16 == 0)) p.ragged = 1;
    tune = 100000 + pick;
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
    SSM_REQUIRE(!p.ragged || !SSM_RESERVED(a) || per_wg == 1, SSM_ERR_BAD_KIND,
                "ssm_scan_fwd: selector %d is for aligned rows of whole 16-step runs", tune);
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
