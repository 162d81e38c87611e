// Forward launches of the side-by-side SSD (ssd_chunk.hpp).
#include "ssd_chunk.hpp"

namespace ssm {

// One walk over the sequence (the state never leaves the chip; a workgroup per head, or per two, so few heads leave CUs idle)
// or the chunks side by side (states through memory, twice x)?  Both times in us, heads counted over the batch.  The walk
// takes a time per block of 32 steps that grows with the heads that share memory, and above 256 heads, two to a workgroup,
// faster; 512 fill the chip.  The workgroups of the other way (one per chunk and head) take a fixed share of the chip each.
// Fitted to both routes at 210 sizes (24 to 640 heads, 256 to 8192 steps, each chunk length and state size):
//   heads, 4096 steps, 128 states:       24         64         96         128        160        256        320        400
//   walk / side by side, chunks of 256: 109 / 41   110 / 67   114 / 97   118 / 125  120 / 152  146 / 244  192 / 289  211 / 356
// Up to two chunks the walk is always the faster one (24 heads, 512 steps: 21 / 24).
bool ssd_side_by_side(const SsdDims &d) {
  // the walk's offsets from the start of a head have 32 bits, some blocks past its end included
  if ((size_t)(d.len + 512) * d.heads * SSD_P * 2 >= (size_t)1 << 31) return true;
  static const double unit_us[3][2] = {{0.0167, 0.0264}, {0.0262, 0.0355}, {0.0421, 0.0536}};   // chunks of 64, 128, 256 steps; 64, 128 states
  const bool large = d.nstate > 64;
  const auto block_us = [&](int64_t n) {
    if (n == 0) return 0.0;
    if (n <= 256) return large ? 0.77 + 0.0012 * (double)n : 0.62 + 0.0010 * (double)n;
    return large ? 0.68 + 0.0024 * (double)n : 0.55 + 0.0020 * (double)n;
  };
  const int64_t heads = (int64_t)d.batch * d.heads;
  const double walk = 7.5 + ssd_walk_turns(ssd_walk_blocks(d.len)) * ((double)(heads / 512) * block_us(512) + block_us(heads % 512));
  return d.nchunks > 2 && walk > 16.0 + unit_us[d.chunk > 128 ? 2 : d.chunk > 64][large] * (double)heads * d.nchunks;
}

template <typename E, int Q, int N>
static void forward_launches(const SsdStatesParams &st, const SsdCarryParams &ca, const SsdChunkScanParams &sc, const SsdDims &d,
                             hipStream_t s) {
  const dim3 units((unsigned)(d.batch * d.nchunks * d.heads)), block(256);
  hipLaunchKernelGGL((ssd_states_kernel<E, Q, N, false>), units, block, 0, s, st);
  const unsigned carriers = (unsigned)(d.batch * d.heads) * (SSD_P * N / 1024);
  bool kept = false;
  if constexpr (std::is_same<E, __bf16>::value) {
    kept = ca.low != nullptr;
    if (kept) hipLaunchKernelGGL((ssd_carry_kernel<E, false, true>), dim3(carriers), block, 0, s, ca);
  }
  if (!kept) hipLaunchKernelGGL((ssd_carry_kernel<E, false, false>), dim3(carriers), block, 0, s, ca);
  if (sc.z) hipLaunchKernelGGL((ssd_chunk_scan_kernel<E, Q, N, SCAN_Y, true>), units, block, 0, s, sc);
  else hipLaunchKernelGGL((ssd_chunk_scan_kernel<E, Q, N, SCAN_Y, false>), units, block, 0, s, sc);
}

int ssd_chunk_forward(const ssm_ssd_combined_args &a, const SsdDims &d, const SsdWorkLayout &lay, hipStream_t s) {
  SSM_REQUIRE((size_t)d.batch * d.nchunks * d.heads < ((size_t)1 << 26), SSM_ERR_TOO_LARGE, "ssm_ssd_combined_fwd: too many workgroups");
  unsigned char *ws = reinterpret_cast<unsigned char *>(a.workspace);
  float *added = a.keep_for_backward ? reinterpret_cast<float *>(a.scratch) : reinterpret_cast<float *>(ws + lay.added);
  const float *dA2 = reinterpret_cast<const float *>(ws + lay.dA2), *dtv = reinterpret_cast<const float *>(ws + lay.dt_out);
  SsdStatesParams st{};
  st.x = a.x; st.frag = ws + lay.Btblk; st.dA2 = dA2; st.dtv = dtv; st.states = added;
  st.len = d.len; st.heads = d.heads; st.groups = d.groups; st.nchunks = d.nchunks;
  SsdCarryParams ca{};
  if (a.keep_for_backward && a.io_dtype == SSM_BF16) ca.low = reinterpret_cast<uint16_t *>(ws + lay.states_low);
  ca.added = added; ca.states = ws + lay.states; ca.dA2 = dA2; ca.first = a.initial_states; ca.last = a.final_states;
  ca.heads = d.heads; ca.nchunks = d.nchunks; ca.chunk = d.chunk; ca.nstate = d.nstate;
  SsdChunkScanParams sc{};
  sc.op = a.x; sc.blk = ws + lay.CBblk; sc.carry = ws + lay.Cblk; sc.states = ws + lay.states; sc.dA2 = dA2; sc.dtv = dtv;
  sc.Dk = a.Dskip; sc.x = a.x; sc.z = a.z; sc.out = a.y; sc.len = d.len; sc.heads = d.heads; sc.groups = d.groups;
  sc.nchunks = d.nchunks; sc.d_per_p = a.d_per_p ? 1 : 0; sc.has_first = a.initial_states != nullptr;
#define SSM_CHUNK_FORWARD(E, QQ, NN) \
  if (d.chunk == QQ && d.nstate == NN) forward_launches<E, QQ, NN>(st, ca, sc, d, s);
#define SSM_CHUNK_FORWARD_ALL(E)                                                                       \
  SSM_CHUNK_FORWARD(E, 256, 128) SSM_CHUNK_FORWARD(E, 128, 128) SSM_CHUNK_FORWARD(E, 64, 128)          \
  SSM_CHUNK_FORWARD(E, 256, 64) SSM_CHUNK_FORWARD(E, 128, 64) SSM_CHUNK_FORWARD(E, 64, 64)
  if (a.io_dtype == SSM_F16) { SSM_CHUNK_FORWARD_ALL(_Float16) }
  else { SSM_CHUNK_FORWARD_ALL(__bf16) }
#undef SSM_CHUNK_FORWARD_ALL
#undef SSM_CHUNK_FORWARD
  SSM_CHECK_LAUNCH("ssm_ssd_combined_fwd");
  return SSM_OK;
}

}  // namespace ssm
