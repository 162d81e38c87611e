/*
 * ssm_amd_testing.h - what a -DSSM_TEST_HOOKS build of the library adds to ssm_amd.h.
 *
 * The shipped library (libssm_amd.so) picks its kernels by shape and dtype alone and rejects a non-zero
 * `reserved` field.  The test suite also needs to run a chosen kernel where the library would pick another
 * (to compare two implementations of one operator on the same inputs) and to learn which kernel a call
 * took.  A second build of the same sources with -DSSM_TEST_HOOKS (libssm_amd_testhooks.so) reads the
 * `reserved` fields as the selectors below and exports three more functions.  Nothing here has a counterpart
 * in the reference and nothing here is part of the backend's interface.
 *
 *   ssm_scan_fwd_args.reserved        0 = automatic; 100 * steps-per-lane + states-per-LDS-pass (408, 808, 816);
 *                                     1616, 2416, 3216, 4816 = 816 with two, three, four, six channels per wave;
 *                                     100000 + v = variant v of the kernel for grouped time-varying projections
 *                                     (131041: the row-per-wave kernel; 131042: that for projections constant in time;
 *                                     111120: the kernel for any number of channels to a workgroup; 113082, 111162, 122121,
 *                                     121081: that with 24, 8, 48, 16);
 *                                     200000 + v = the same with a row's chunks one after the other however few rows
 *   ssm_scan_bwd_args.reserved        1 = the general kernel also where a wave-per-row kernel applies (grouped
 *                                     projections, projections of their own per channel, or projections that are
 *                                     constant in time);
 *                                     2 = the wave-per-row kernel with its bounded wait for a neighbouring wave
 *                                     cut to nothing, so that every wave takes the give-up path (dB and dC
 *                                     come back as NaN; the kernel ends normally);
 *                                     3 = a row's chunks one after the other also where they would run side by side
 *   ssm_dscan_bwd_args.reserved       non-zero = the general two-kernel path also where the one-pass kernel applies
 *   ssm_ssd_bmm_args.reserved,
 *   ssm_ssd_chunk_state_args.reserved,
 *   ssm_ssd_chunk_scan_args.reserved  non-zero = the one-thread-per-output kernel instead of a matrix-core kernel
 *   ssm_ssd_combined_args.reserved    1 = one pass over the sequence, 2 = the chunks side by side (a call with
 *                                     keep_for_backward runs side by side whatever it says);
 *                                     ssm_ssd_combined_workspace_bytes() of this build covers either
 */
#ifndef SSM_AMD_TESTING_H
#define SSM_AMD_TESTING_H

#include "ssm_amd.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Which of the calls made by this thread since the last query ran a bf16 / fp16 matrix-core kernel:
 * bit 0 bmm_chunk, bit 1 chunk_state, bit 2 chunk_scan, bit 3 ssm_ssd_combined_fwd in one pass over the sequence,
 * bit 4 the same with its chunks side by side.
 * Resets on read. */
int ssm_ssd_mfma_launches(void);

/* Channels that a call with time-varying projections gives to a workgroup where its rows go many to a workgroup: the forward's
 * kernel for any number of channels, the backward's wave-per-row kernel (0: the call's shape is not for that). */
int ssm_scan_fwd_rows_per_workgroup(int batch, int dim, int seqlen, int b_groups, int c_groups);
int ssm_scan_bwd_rows_per_workgroup(int batch, int dim, int seqlen, int nstate, int b_groups, int c_groups);

#ifdef __cplusplus
}
#endif
#endif /* SSM_AMD_TESTING_H */
