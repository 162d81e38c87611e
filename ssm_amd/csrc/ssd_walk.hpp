// What the one-pass SSD forward (ssd_walk.hip) is called with.
#pragma once
#include "ssd_common.hpp"

namespace ssm {

// Whether the decays of a block factor (bfloat16 calls; ssd_walk.hip), by its running sum at its end in powers of two.
constexpr float SSD_WALK_RANGE = 160.0f;
__device__ __forceinline__ bool walk_factors(float end) { return end <= 0.0f && end >= -SSD_WALK_RANGE; }

struct SsdWalkParams {                  // x, z, y and the fragment copies hold the call's 16-bit element type
  const void *x, *z;
  void *y;
  const float *steps;                   // (B, H, turns, 32, 2): cs (running sum of dt A log2(e) since the block's first step), less half of the block's where it factors, and dt
  const float *ends;                    // (B, H, turns): cs at the block's last step
  const void *Cblk, *Btblk, *CBblk;     // fragments of blocks of 32 steps
  const float *Dk, *init, *A;
  float *final_states;
  int batch, len, heads, groups, nblocks;
  int sets;                             // workgroups of one or two heads (set by ssd_walk_forward)
  int turns;                            // nblocks in whole turns through a ring of four
  int chunk_blocks;                     // blocks in a chunk of the call (what a growing head's factors go by)
  bool in_place;                        // y over x or z (set by ssd_walk_forward)
};

int ssd_walk_forward(SsdWalkParams p, int dmode, bool f16, int nstate, hipStream_t s);

}  // namespace ssm
