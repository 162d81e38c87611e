// Forward launches of the side-by-side SSD (ssd_chunk.hpp).
#include "ssd_chunk.hpp"
#include <algorithm>

namespace ssm {

// One walk over the sequence (the state never leaves the chip; a workgroup per head, or per two, so few heads leave CUs idle)
// or the chunks side by side (states through memory, twice x)?  Both times in us, heads counted over the batch.  The walk
// takes a time per block of 32 steps that grows with the heads that share memory, and above 256 heads, two to a workgroup,
// faster; 512 fill the chip.  The workgroups of the other way (one per chunk and head) share it, a little better while they
// all fit.  Fitted to both routes, replayed as graphs, at 350 sizes (8 to 400 heads, 256 to 4096 steps), and looked at again at
// 390 (16 to 400 heads, 768 to 4096 steps, every chunk and state size) in either element type, one line for both: the route
// taken is the faster one or within 5 % of it but at three of them in bfloat16 (11, 10 and 7 %), on average 0.1 % off.
//   heads, 4096 steps, 128 states:       24         48         80         112        128        160        256        400
//   walk / side by side, chunks of 256: 107 / 38   106 / 53   105 / 85   109 / 110  110 / 130  117 / 150  138 / 241  197 / 341
//   float16                             113 / 39   113 / 55   116 / 87   118 / 112  123 / 131  124 / 151  146 / 243  215 / 357
// Up to two chunks the walk is always the faster one (24 heads, 512 steps: 20.8 / 23.7).
// Side by side a group beyond the first has C.B of its own for whole chunks, the walk for blocks of 32 steps: `group` is what
// that costs more for each block of each group, fitted at 420 sizes of 1 to 128 groups, 600 to 4096 steps, and looked at again
// at 700 others: within 5 % of the faster route at all but seven, the worst 11 % off.  Without it 52 %: 4096 steps, 128 states,
// chunks of 256, 100 groups of one head 256 / 401, 48 of one 162 / 170, 24 of one 136 / 92, 8 of ten 117 / 98.
bool ssd_side_by_side(const SsdDims &d) {
  // the walk's offsets from the start of a head have 32 bits, some blocks past its end included
  if ((size_t)(d.len + 512) * d.heads * SSD_P * 2 >= (size_t)1 << 31) return true;
  struct Chunks { double start, each, more, from, group; };  // `more` for each workgroup after the first `from`
  static const Chunks chunks[3][2] = {{{16.0, 0.0135, 0.0060, 2300.0, 0.0003}, {20.0, 0.0175, 0.0116, 1600.0, 0.0018}},      // of 64 steps; 64, 128 states
                                      {{16.0, 0.0195, 0.0075, 1280.0, 0.0020}, {18.0, 0.0255, 0.0120, 1280.0, 0.0060}},
                                      {{20.5, 0.0295, 0.0145, 640.0, 0.0060}, {22.5, 0.0385, 0.0150, 640.0, 0.0098}}};
  const bool large = d.nstate > 64;
  const auto block_us = [&](int64_t n) {
    if (n == 0) return 0.0;
    const double share = std::max(0.0, (double)n - 192.0);
    if (n <= 256) return large ? 0.775 + 0.0005 * (double)n + 0.0018 * share : 0.62 + 0.0005 * (double)n + 0.0012 * share;
    return large ? 0.77 + 0.0016 * (double)n : 0.72 + 0.0012 * (double)n;
  };
  const int64_t heads = (int64_t)d.batch * d.heads;
  const double start = heads > 256 ? (large ? 12.7 : 10.0) : large ? 8.7 : 7.7;
  const double walk = start + ssd_walk_turns(ssd_walk_blocks(d.len)) * ((double)(heads / 512) * block_us(512) + block_us(heads % 512));
  const Chunks &c = chunks[d.chunk > 128 ? 2 : d.chunk > 64][large];
  const double units = (double)heads * d.nchunks, group_blocks = (double)d.batch * (d.groups - 1) * ssd_walk_blocks(d.len);
  return d.nchunks > 2 && walk > c.start + c.each * units + c.more * std::max(0.0, units - c.from) + c.group * group_blocks;
}

template <typename E, int Q, int N>
static void forward_launches(const SsdStatesParams &st, const SsdCarryParams &ca, const SsdChunkScanParams &sc, const SsdDims &d,
                             hipStream_t s) {
  const dim3 units((unsigned)(d.batch * d.nchunks * d.heads)), block(256);
  hipLaunchKernelGGL((ssd_states_kernel<E, Q, N, false>), units, block, 0, s, st);
  const unsigned carriers = (unsigned)carry_units(d);
  bool kept = false;
  if constexpr (std::is_same<E, __bf16>::value) {
    kept = ca.low != nullptr;
    if (kept) hipLaunchKernelGGL((ssd_carry_kernel<E, false, true>), dim3(carriers), block, 0, s, ca);
  }
  if (!kept) hipLaunchKernelGGL((ssd_carry_kernel<E, false, false>), dim3(carriers), block, 0, s, ca);
  if (sc.z) hipLaunchKernelGGL((ssd_chunk_scan_kernel<E, Q, N, true>), units, block, 0, s, sc);
  else hipLaunchKernelGGL((ssd_chunk_scan_kernel<E, Q, N, false>), units, block, 0, s, sc);
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
