// Forward launches of the side-by-side SSD (ssd_chunk.hpp).
#include "ssd_chunk.hpp"

namespace ssm {

// Chunks one after the other (the state never leaves the chip; 32 channels per workgroup, so few heads leave CUs idle) or
// side by side (states through memory, twice x)?  Both times in us as measured on one MI355X, heads counted over the batch:
// a chunk of the walk takes a fixed time plus what its workgroups add to each other (768 are resident at once), a unit of
// the other way a fixed share of the chip, and its two further launches 10 us.
//   batch x heads x steps, 256-step chunks, 128 states:   1 x 80 x 8192   4 x 40 x 4096   4 x 80 x 4096   4 x 80 x 512
//   walk / side by side:                                     266 / 148       193 / 153       272 / 285       33 / 47
//   128-step chunks:                                                         228 / 209       291 / 402
bool ssd_side_by_side(const SsdDims &d) {
  const double heads = (double)d.batch * d.heads, nc = d.nchunks;
  const bool long_chunk = d.chunk > 128, wide = d.nstate > 64;
  const double chunk_us = long_chunk ? (wide ? 6.5 : 6.0) : (wide ? 4.1 : 3.7);
  const double head_us = long_chunk ? (wide ? 0.033 : 0.028) : (wide ? 0.0134 : 0.0122);
  const double unit_us = long_chunk ? (wide ? 0.052 : 0.042) : (wide ? 0.0375 : 0.0258);
  const double rounds = (double)((2 * d.batch * (int64_t)d.heads + 767) / 768);
  return d.nchunks > 1 && nc * (chunk_us * rounds + head_us * heads) > 10.0 + unit_us * heads * nc;
}

template <typename E, int Q, int N>
static void forward_launches(const SsdStatesParams &st, const SsdCarryParams &ca, const SsdChunkScanParams &sc, const SsdDims &d,
                             hipStream_t s) {
  const dim3 units((unsigned)(d.batch * d.nchunks * d.heads)), block(256);
  hipLaunchKernelGGL((ssd_states_kernel<E, Q, N, false>), units, block, 0, s, st);
  const unsigned carriers = (unsigned)(d.batch * d.heads) * (SSD_P * N / 1024);
  if (ca.turned) hipLaunchKernelGGL((ssd_carry_kernel<E, false, true>), dim3(carriers / 4), block, 0, s, ca);
  else hipLaunchKernelGGL((ssd_carry_kernel<E, false, false>), dim3(carriers), block, 0, s, ca);
  if (sc.z) hipLaunchKernelGGL((ssd_chunk_scan_kernel<E, Q, N, SCAN_Y, true>), units, block, 0, s, sc);
  else hipLaunchKernelGGL((ssd_chunk_scan_kernel<E, Q, N, SCAN_Y, false>), units, block, 0, s, sc);
}

int ssd_chunk_forward(const ssm_ssd_combined_args &a, const SsdDims &d, const SsdWorkLayout &lay, hipStream_t s) {
  SSM_REQUIRE((size_t)d.batch * d.nchunks * d.heads < ((size_t)1 << 26), SSM_ERR_TOO_LARGE, "ssm_ssd_combined_fwd: too many workgroups");
  unsigned char *ws = reinterpret_cast<unsigned char *>(a.workspace);
  float *added = reinterpret_cast<float *>(ws + lay.added);
  const float *dA2 = reinterpret_cast<const float *>(ws + lay.dA2), *dtv = reinterpret_cast<const float *>(ws + lay.dt_out);
  SsdStatesParams st{};
  st.x = a.x; st.frag = ws + lay.Btblk; st.dA2 = dA2; st.dtv = dtv; st.states = added;
  st.len = d.len; st.heads = d.heads; st.groups = d.groups; st.nchunks = d.nchunks;
  SsdCarryParams ca{};
  if (a.keep_for_backward) ca.turned = ws + lay.turned;
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
