"""ctypes binding of ``libssm_amd.so`` (the C ABI declared in include/ssm_amd.h).

The shared library is built ahead of time by ``python -m ssm_amd.build`` and is
loaded from ``ssm_amd/lib``.  There is no fallback: if the library is missing
or a call returns a non-zero status, an exception is raised.
"""

from __future__ import annotations

import ctypes as C
import importlib.util
import threading
import warnings
from pathlib import Path
from typing import Optional

import torch

import os

# SSM_AMD_LIB points the binding at another build of the same C ABI.
LIB_PATH = Path(os.environ.get("SSM_AMD_LIB") or
                Path(__file__).resolve().parent / "lib" / "libssm_amd.so")
ABI_VERSION = 11

SSM_F32, SSM_BF16, SSM_F16 = 0, 1, 2
PROJ_DN, PROJ_BDN, PROJ_BGNL = 0, 1, 2

_DTYPE_ENUM = {torch.float32: SSM_F32, torch.bfloat16: SSM_BF16, torch.float16: SSM_F16}

_vp, _i32, _f32, _i64 = C.c_void_p, C.c_int32, C.c_float, C.c_int64


class BackendUnavailable(RuntimeError):
    """The HIP library could not be loaded."""


class KernelError(RuntimeError):
    """A C-ABI entry point returned a failure status."""


class ScanFwdArgs(C.Structure):
    _fields_ = [
        ("u", _vp), ("delta", _vp), ("z", _vp), ("A", _vp), ("Bproj", _vp), ("Cproj", _vp),
        ("Dskip", _vp), ("dt_bias", _vp), ("out", _vp), ("last_state", _vp), ("chunk_states", _vp),
        ("batch", _i32), ("dim", _i32), ("seqlen", _i32), ("nstate", _i32),
        ("io_dtype", _i32), ("bc_dtype", _i32), ("b_kind", _i32), ("c_kind", _i32),
        ("b_groups", _i32), ("c_groups", _i32), ("delta_softplus", _i32), ("reserved", _i32),
    ]


class ScanBwdArgs(C.Structure):
    _fields_ = [
        ("u", _vp), ("delta", _vp), ("z", _vp), ("dout", _vp), ("A", _vp), ("Bproj", _vp), ("Cproj", _vp),
        ("Dskip", _vp), ("dt_bias", _vp), ("dlast_state", _vp), ("chunk_states", _vp),
        ("du", _vp), ("ddelta", _vp), ("dz", _vp), ("dA", _vp), ("dB", _vp), ("dC", _vp), ("dD", _vp),
        ("ddt_bias", _vp), ("workspace", _vp), ("workspace_bytes", C.c_size_t),
        ("batch", _i32), ("dim", _i32), ("seqlen", _i32), ("nstate", _i32),
        ("io_dtype", _i32), ("bc_dtype", _i32), ("b_kind", _i32), ("c_kind", _i32),
        ("b_groups", _i32), ("c_groups", _i32), ("delta_softplus", _i32), ("reserved", _i32), ("dbc_dtype", _i32),
    ]


class StateStepArgs(C.Structure):
    _fields_ = [
        ("state", _vp), ("x", _vp), ("dt", _vp), ("z", _vp), ("A", _vp), ("Bproj", _vp), ("Cproj", _vp),
        ("Dskip", _vp), ("dt_bias", _vp), ("out", _vp),
        ("batch", _i32), ("dim", _i32), ("nstate", _i32),
        ("state_dtype", _i32), ("io_dtype", _i32), ("bc_dtype", _i32),
        ("b_kind", _i32), ("c_kind", _i32), ("b_groups", _i32), ("c_groups", _i32),
        ("dt_softplus", _i32),
        ("z_batch_stride", C.c_int64), ("b_batch_stride", C.c_int64), ("c_batch_stride", C.c_int64),
    ]


class StateStepBwdArgs(C.Structure):
    _fields_ = [
        ("grad_out", _vp), ("grad_state", _vp), ("state", _vp), ("x", _vp), ("dt", _vp), ("z", _vp), ("A", _vp),
        ("Bproj", _vp), ("Cproj", _vp), ("Dskip", _vp), ("dt_bias", _vp),
        ("dstate", _vp), ("dx", _vp), ("ddt", _vp), ("dz", _vp), ("dA", _vp), ("dB", _vp), ("dC", _vp),
        ("dD", _vp), ("ddt_bias", _vp), ("workspace", _vp), ("workspace_bytes", C.c_size_t),
        ("batch", _i32), ("dim", _i32), ("nstate", _i32),
        ("state_dtype", _i32), ("io_dtype", _i32), ("bc_dtype", _i32),
        ("b_kind", _i32), ("c_kind", _i32), ("b_groups", _i32), ("c_groups", _i32),
        ("dt_softplus", _i32),
    ]


class DecodeStepArgs(C.Structure):
    _fields_ = [("step", StateStepArgs), ("conv_state", _vp), ("conv_weight", _vp), ("conv_bias", _vp),
                ("conv_out", _vp), ("conv_width", _i32), ("conv_activation", _i32)]


CHUNK_HP, CHUNK_BHP, CHUNK_BLHP = 0, 1, 2


class DscanFwdArgs(C.Structure):
    _fields_ = [
        ("X", _vp), ("dt", _vp), ("A", _vp), ("Bproj", _vp), ("Cproj", _vp), ("Dskip", _vp), ("z", _vp),
        ("initial_states", _vp), ("seq_lens", _vp), ("Y", _vp), ("workspace", _vp),
        ("workspace_bytes", C.c_size_t),
        ("batch", _i32), ("seqlen", _i32), ("heads", _i32), ("proj", _i32),
        ("x_dtype", _i32), ("dt_dtype", _i32), ("bc_dtype", _i32), ("z_dtype", _i32), ("init_dtype", _i32),
        ("b_kind", _i32), ("c_kind", _i32), ("a_per_p", _i32), ("d_per_p", _i32), ("z_per_p", _i32),
        ("round_states", _vp),
    ]


class DscanBwdArgs(C.Structure):
    _fields_ = [
        ("grad_y", _vp), ("X", _vp), ("dt", _vp), ("A", _vp), ("Bproj", _vp), ("Cproj", _vp), ("Dskip", _vp),
        ("z", _vp), ("initial_states", _vp), ("seq_lens", _vp),
        ("dX", _vp), ("ddt", _vp), ("dA", _vp), ("dB", _vp), ("dC", _vp), ("dD", _vp), ("dz", _vp),
        ("dinitial_states", _vp), ("workspace", _vp), ("workspace_bytes", C.c_size_t),
        ("batch", _i32), ("seqlen", _i32), ("heads", _i32), ("proj", _i32),
        ("x_dtype", _i32), ("dt_dtype", _i32), ("bc_dtype", _i32), ("z_dtype", _i32), ("init_dtype", _i32),
        ("b_kind", _i32), ("c_kind", _i32), ("a_per_p", _i32), ("d_per_p", _i32), ("z_per_p", _i32),
        ("grads_in_io_dtype", _i32), ("reserved", _i32), ("round_states", _vp),
    ]


class SsdDims(C.Structure):
    _fields_ = [("batch", _i32), ("seqlen", _i32), ("heads", _i32), ("headdim", _i32), ("groups", _i32),
                ("nstate", _i32), ("chunk", _i32)]


class SsdCumsumArgs(C.Structure):
    _fields_ = [("dt", _vp), ("A", _vp), ("dt_bias", _vp), ("dA_cumsum", _vp), ("dt_out", _vp),
                ("dims", SsdDims), ("dt_dtype", _i32), ("dt_softplus", _i32), ("dt_min", _f32), ("dt_max", _f32)]


class SsdBmmArgs(C.Structure):
    _fields_ = [("a", _vp), ("b", _vp), ("seq_idx", _vp), ("out", _vp),
                ("batch", _i32), ("seqlen", _i32), ("groups", _i32), ("kdim", _i32), ("chunk", _i32),
                ("in_dtype", _i32), ("out_dtype", _i32), ("causal", _i32), ("reserved", _i32)]


class SsdChunkStateArgs(C.Structure):
    _fields_ = [("Bm", _vp), ("x", _vp), ("dt", _vp), ("dA_cumsum", _vp), ("states", _vp),
                ("workspace", _vp), ("workspace_bytes", C.c_size_t), ("dims", SsdDims),
                ("x_dtype", _i32), ("b_dtype", _i32), ("states_dtype", _i32), ("reserved", _i32),
                ("seq_idx", _vp), ("x_row_scale", _vp), ("x_time_reversed", _i32)]


class SsdStatePassingArgs(C.Structure):
    _fields_ = [("states", _vp), ("dA_chunk_last", _vp), ("initial_states", _vp), ("states_out", _vp),
                ("final_states", _vp), ("batch", _i32), ("nchunks", _i32), ("heads", _i32), ("dim", _i32),
                ("states_dtype", _i32), ("seqlen", _i32), ("chunk", _i32), ("seq_idx", _vp)]


class SsdChunkScanArgs(C.Structure):
    _fields_ = [("CB", _vp), ("Cm", _vp), ("x", _vp), ("z", _vp), ("prev_states", _vp), ("dt", _vp),
                ("dA_cumsum", _vp), ("Dskip", _vp), ("y", _vp), ("dims", SsdDims),
                ("x_dtype", _i32), ("c_dtype", _i32), ("cb_dtype", _i32), ("states_dtype", _i32),
                ("z_dtype", _i32), ("d_per_p", _i32), ("reserved", _i32), ("seq_idx", _vp),
                ("y_f32", _i32), ("x_row_scale", _vp), ("dx_x", _vp), ("dx_dt", _vp), ("dx_Dskip", _vp), ("dx_out", _vp),
                ("dx_xu", _vp), ("dx_s1", _vp), ("dx_d_per_p", _i32), ("dx_out_f32", _i32), ("dx_round_dtx", _i32),
                ("x_time_reversed", _i32)]


class SsdChunkStateVarlenArgs(C.Structure):
    _fields_ = [("Bm", _vp), ("x", _vp), ("dt", _vp), ("dA_cumsum", _vp), ("chunk_states", _vp),
                ("cu_seqlens", _vp), ("states", _vp), ("dims", SsdDims), ("nseq", _i32),
                ("x_dtype", _i32), ("b_dtype", _i32), ("states_dtype", _i32)]


class Mamba2DecodeArgs(C.Structure):
    _fields_ = [("zxbcdt", _vp), ("conv_state", _vp), ("conv_weight", _vp), ("conv_bias", _vp), ("xbc", _vp),
                ("ssm_state", _vp), ("A", _vp), ("Dskip", _vp), ("dt_bias", _vp), ("y", _vp),
                ("batch", _i32), ("heads", _i32), ("headdim", _i32), ("groups", _i32), ("nstate", _i32),
                ("conv_width", _i32), ("io_dtype", _i32), ("d_per_p", _i32), ("dt_softplus", _i32), ("gate", _i32)]


class Conv1dUpdateArgs(C.Structure):
    _fields_ = [("x", _vp), ("conv_state", _vp), ("weight", _vp), ("bias", _vp), ("out", _vp),
                ("x_row_stride", C.c_int64), ("batch", _i32), ("channels", _i32), ("width", _i32),
                ("io_dtype", _i32), ("activation", _i32)]


class SsdCombinedArgs(C.Structure):
    _fields_ = [("x", _vp), ("dt", _vp), ("A", _vp), ("dt_bias", _vp), ("Bm", _vp), ("Cm", _vp), ("Dskip", _vp),
                ("z", _vp), ("initial_states", _vp), ("y", _vp), ("final_states", _vp), ("workspace", _vp),
                ("workspace_bytes", C.c_size_t), ("dims", SsdDims), ("io_dtype", _i32), ("dt_dtype", _i32),
                ("dt_softplus", _i32), ("d_per_p", _i32), ("dt_min", C.c_float), ("dt_max", C.c_float),
                ("seq_idx", _vp), ("b_row_stride", _i64), ("c_row_stride", _i64), ("keep_for_backward", _i32),
                ("reserved", _i32), ("scratch", _vp), ("scratch_bytes", C.c_size_t)]


class SsdCombinedBwdArgs(C.Structure):
    _fields_ = [("fwd", SsdCombinedArgs), ("dout", _vp), ("dfinal", _vp), ("dx", _vp), ("dz", _vp), ("dB", _vp), ("dC", _vp),
                ("ddt", _vp), ("dA", _vp), ("dD", _vp), ("ddt_bias", _vp), ("dinitial_states", _vp), ("workspace", _vp),
                ("workspace_bytes", C.c_size_t)]


class SsdBwdGateArgs(C.Structure):
    _fields_ = [("dout", _vp), ("z", _vp), ("x", _vp), ("ypre", _vp), ("Dskip", _vp), ("dy", _vp), ("dy_rev", _vp),
                ("dz", _vp), ("s2", _vp), ("dyx", _vp), ("batch", _i32), ("seqlen", _i32), ("heads", _i32),
                ("headdim", _i32), ("io_dtype", _i32), ("dy_dtype", _i32), ("d_per_p", _i32), ("w_dy", _vp),
                ("w_x", _vp), ("dy_w", _vp), ("x_w", _vp), ("dz_in_io_dtype", _i32)]


class SsdBwdDxArgs(C.Structure):
    _fields_ = [("dout", _vp), ("z", _vp), ("x", _vp), ("u_rev", _vp), ("dt", _vp), ("Dskip", _vp), ("dx", _vp),
                ("xu", _vp), ("s1", _vp), ("batch", _i32), ("seqlen", _i32), ("heads", _i32), ("headdim", _i32),
                ("io_dtype", _i32), ("d_per_p", _i32), ("round_bf16", _i32), ("dx_in_io_dtype", _i32)]


class SsdBwdDbArgs(C.Structure):
    _fields_ = [("v_rev", _vp), ("dt", _vp), ("dB", _vp), ("batch", _i32), ("seqlen", _i32), ("heads", _i32),
                ("groups", _i32), ("nstate", _i32)]


class SsdBwdDcbArgs(C.Structure):
    _fields_ = [("dy", _vp), ("x", _vp), ("dt", _vp), ("dA_cumsum", _vp), ("dCB", _vp), ("batch", _i32),
                ("seqlen", _i32), ("heads", _i32), ("headdim", _i32), ("groups", _i32), ("chunk", _i32)]


class SsdBwdStatesArgs(C.Structure):
    _fields_ = [("entering_fwd", _vp), ("entering_rev", _vp), ("fwd_bf16", _vp), ("rev_bf16", _vp), ("anchor", _vp),
                ("batch", _i32), ("nchunks", _i32), ("heads", _i32), ("dim", _i32)]


class SsdScaleRowsArgs(C.Structure):
    _fields_ = [("x", _vp), ("w", _vp), ("out", _vp), ("rows", C.c_int64), ("cols", _i32), ("x_dtype", _i32),
                ("out_dtype", _i32)]


class SsdBwdPrepArgs(C.Structure):
    _fields_ = [("dt", _vp), ("A", _vp), ("dt_bias", _vp), ("dA_cumsum", _vp), ("dt_out", _vp), ("dA_cumsum_rev", _vp),
                ("dt_rows", _vp), ("w_dy", _vp), ("w_x", _vp), ("batch", _i32), ("seqlen", _i32), ("heads", _i32),
                ("chunk", _i32), ("dt_dtype", _i32), ("dt_softplus", _i32), ("dt_min", C.c_float), ("dt_max", C.c_float)]


class SsdBwdDtArgs(C.Structure):
    _fields_ = [("s1", _vp), ("s2", _vp), ("xu", _vp), ("dt", _vp), ("dt_raw", _vp), ("A", _vp), ("dt_bias", _vp),
                ("q0", _vp), ("anchor", _vp), ("first_step", _vp), ("ddt", _vp), ("dA_part", _vp), ("dbias_part", _vp),
                ("batch", _i32), ("seqlen", _i32), ("heads", _i32), ("chunk", _i32), ("dt_dtype", _i32),
                ("dt_softplus", _i32), ("dt_min", C.c_float), ("dt_max", C.c_float)]


LAYOUT_BCL, LAYOUT_BLC, LAYOUT_ROWS_TO_BCL = 0, 1, 2
ACT_IDENTITY, ACT_SILU = 0, 1


class Conv1dFwdArgs(C.Structure):
    _fields_ = [
        ("x", _vp), ("weight", _vp), ("bias", _vp), ("y", _vp),
        ("batch", _i32), ("channels", _i32), ("seqlen", _i32), ("width", _i32),
        ("io_dtype", _i32), ("layout", _i32), ("activation", _i32), ("pad0", _i32),
        ("x_batch_stride", C.c_int64), ("x_row_stride", C.c_int64),
    ]


class Conv1dBwdArgs(C.Structure):
    _fields_ = [
        ("x", _vp), ("dout", _vp), ("weight", _vp), ("bias", _vp), ("dx", _vp), ("dweight", _vp),
        ("dbias", _vp), ("workspace", _vp), ("workspace_bytes", C.c_size_t),
        ("batch", _i32), ("channels", _i32), ("seqlen", _i32), ("width", _i32),
        ("io_dtype", _i32), ("layout", _i32), ("activation", _i32), ("pad0", _i32),
        ("x_batch_stride", C.c_int64), ("x_row_stride", C.c_int64),
    ]


class RowsToBclArgs(C.Structure):
    _fields_ = [
        ("src", _vp), ("dst", _vp), ("src_batch_stride", C.c_int64), ("src_row_stride", C.c_int64),
        ("batch", _i32), ("channels", _i32), ("seqlen", _i32), ("element_size", _i32),
    ]


class NormFwdArgs(C.Structure):
    _fields_ = [
        ("x", _vp), ("residual", _vp), ("weight", _vp), ("bias", _vp), ("y", _vp), ("residual_out", _vp),
        ("mean", _vp), ("rstd", _vp),
        ("rows", _i32), ("hidden", _i32),
        ("x_dtype", _i32), ("residual_dtype", _i32), ("residual_out_dtype", _i32),
        ("is_rms", _i32), ("prenorm", _i32), ("eps", _f32),
    ]


class NormBwdArgs(C.Structure):
    _fields_ = [
        ("x", _vp), ("residual", _vp), ("dy", _vp), ("weight", _vp), ("mean", _vp), ("rstd", _vp),
        ("dx", _vp), ("dresidual", _vp), ("dweight", _vp), ("dbias", _vp),
        ("workspace", _vp), ("workspace_bytes", C.c_size_t),
        ("rows", _i32), ("hidden", _i32), ("x_dtype", _i32), ("residual_dtype", _i32),
        ("is_rms", _i32), ("prenorm", _i32), ("grad_residual_out", _vp), ("grad_residual_out_dtype", _i32),
    ]


# name -> argument struct (every entry point is ``int f(const args*, void* stream)``)
_pd, _f64 = C.c_void_p, C.c_double


class F64ScanArgs(C.Structure):
    _fields_ = [
        ("u", _pd), ("delta", _pd), ("z", _pd), ("A", _pd), ("Bproj", _pd), ("Cproj", _pd), ("Dskip", _pd),
        ("dt_bias", _pd), ("out", _pd), ("last_state", _pd), ("b_stride", _i64 * 4), ("c_stride", _i64 * 4),
        ("dout", _pd), ("dlast_state", _pd), ("states", _pd), ("ypre", _pd), ("du", _pd), ("ddelta", _pd),
        ("dz", _pd), ("dA_rows", _pd), ("dB", _pd), ("dC", _pd), ("dD_rows", _pd), ("dbias_rows", _pd),
        ("batch", _i32), ("dim", _i32), ("seqlen", _i32), ("nstate", _i32), ("delta_softplus", _i32),
    ]


class F64StepArgs(C.Structure):
    _fields_ = [
        ("state", _pd), ("x", _pd), ("dt", _pd), ("z", _pd), ("A", _pd), ("Bproj", _pd), ("Cproj", _pd),
        ("Dskip", _pd), ("dt_bias", _pd), ("out", _pd), ("b_stride", _i64 * 3), ("c_stride", _i64 * 3),
        ("dout", _pd), ("dstate_new", _pd), ("dstate", _pd), ("dx", _pd), ("ddt", _pd), ("dz", _pd),
        ("dA_rows", _pd), ("dB", _pd), ("dC", _pd), ("dD_rows", _pd),
        ("batch", _i32), ("dim", _i32), ("nstate", _i32), ("dt_softplus", _i32),
    ]


class F64DscanArgs(C.Structure):
    _fields_ = [
        ("X", _pd), ("dt", _pd), ("A", _pd), ("Bproj", _pd), ("Cproj", _pd), ("Dskip", _pd), ("z", _pd),
        ("init", _pd), ("lengths", _pd), ("Y", _pd),
        ("b_stride", _i64 * 4), ("c_stride", _i64 * 4), ("z_stride", _i64 * 4),
        ("dY", _pd), ("states", _pd), ("dX", _pd), ("ddt_rows", _pd), ("dB", _pd), ("dC", _pd), ("dz", _pd),
        ("dA_rows", _pd), ("dD_rows", _pd), ("dinit", _pd),
        ("batch", _i32), ("seqlen", _i32), ("heads", _i32), ("hdim", _i32),
    ]


class F64ConvArgs(C.Structure):
    _fields_ = [
        ("x", _pd), ("weight", _pd), ("bias", _pd), ("y", _pd), ("x_stride", _i64 * 3), ("y_stride", _i64 * 3),
        ("dy", _pd), ("dx", _pd), ("dy_stride", _i64 * 3), ("dx_stride", _i64 * 3), ("dpre", _pd), ("dw", _pd),
        ("db", _pd),
        ("batch", _i32), ("channels", _i32), ("seqlen", _i32), ("width", _i32), ("activation", _i32),
    ]


class F64NormArgs(C.Structure):
    _fields_ = [
        ("x", _pd), ("residual", _pd), ("weight", _pd), ("bias", _pd), ("y", _pd), ("residual_out", _pd),
        ("mean", _pd), ("rstd", _pd), ("dy", _pd), ("dx", _pd), ("dresidual", _pd), ("dw", _pd), ("db", _pd),
        ("rows", _i64), ("hidden", _i32), ("is_rms", _i32), ("prenorm", _i32), ("eps", _f64),
    ]


ENTRY_POINTS = {
    "ssm_scan_fwd": ScanFwdArgs,
    "ssm_scan_bwd": ScanBwdArgs,
    "ssm_state_step": StateStepArgs,
    "ssm_state_step_bwd": StateStepBwdArgs,
    "ssm_decode_step": DecodeStepArgs,
    "ssm_mamba2_decode_step": Mamba2DecodeArgs,
    "ssm_dscan_fwd": DscanFwdArgs,
    "ssm_dscan_bwd": DscanBwdArgs,
    "ssm_ssd_chunk_cumsum": SsdCumsumArgs,
    "ssm_ssd_bmm_chunk": SsdBmmArgs,
    "ssm_ssd_chunk_state": SsdChunkStateArgs,
    "ssm_ssd_state_passing": SsdStatePassingArgs,
    "ssm_ssd_chunk_scan": SsdChunkScanArgs,
    "ssm_ssd_chunk_state_varlen": SsdChunkStateVarlenArgs,
    "ssm_ssd_combined_fwd": SsdCombinedArgs,
    "ssm_ssd_bwd_gate": SsdBwdGateArgs,
    "ssm_ssd_bwd_dx": SsdBwdDxArgs,
    "ssm_ssd_bwd_db": SsdBwdDbArgs,
    "ssm_ssd_bwd_dcb": SsdBwdDcbArgs,
    "ssm_ssd_bwd_states": SsdBwdStatesArgs,
    "ssm_ssd_scale_rows": SsdScaleRowsArgs,
    "ssm_ssd_bwd_dt": SsdBwdDtArgs,
    "ssm_ssd_bwd_prep": SsdBwdPrepArgs,
    "ssm_conv1d_fwd": Conv1dFwdArgs,
    "ssm_conv1d_bwd": Conv1dBwdArgs,
    "ssm_conv1d_update": Conv1dUpdateArgs,
    "ssm_rows_to_bcl": RowsToBclArgs,
    "ssm_norm_fwd": NormFwdArgs,
    "ssm_norm_bwd": NormBwdArgs,
    "ssm_norm_bwd_static": NormBwdArgs,
    "ssm_f64_scan_fwd": F64ScanArgs,
    "ssm_f64_scan_bwd": F64ScanArgs,
    "ssm_f64_state_step": F64StepArgs,
    "ssm_f64_state_step_bwd": F64StepArgs,
    "ssm_f64_dscan_fwd": F64DscanArgs,
    "ssm_f64_dscan_bwd": F64DscanArgs,
    "ssm_f64_conv_fwd": F64ConvArgs,
    "ssm_f64_conv_bwd": F64ConvArgs,
    "ssm_f64_norm_fwd": F64NormArgs,
    "ssm_f64_norm_bwd": F64NormArgs,
}
# name -> (restype, argtypes) of the remaining exported functions
PLAIN_SYMBOLS = {
    "ssm_amd_abi_version": (C.c_int, []),
    "ssm_amd_status_string": (C.c_char_p, [C.c_int]),
    "ssm_amd_last_error": (C.c_char_p, []),
    "ssm_scan_chunk_len": (C.c_int, []),
    "ssm_scan_bwd_workspace_bytes": (C.c_size_t, [C.c_int] * 8),
    "ssm_scan_bwd_per_row_workspace_bytes": (C.c_size_t, [C.POINTER(ScanBwdArgs)]),
    "ssm_scan_bwd_full_workspace_bytes": (C.c_size_t, [C.POINTER(ScanBwdArgs)]),
    "ssm_state_step_bwd_workspace_bytes": (C.c_size_t, [C.c_int] * 3),
    "ssm_dscan_fwd_workspace_bytes": (C.c_size_t, [C.c_int] * 4),
    "ssm_dscan_bwd_workspace_bytes": (C.c_size_t, [C.c_int] * 4),
    "ssm_dscan_fwd_one_pass": (C.c_int, [C.POINTER(DscanFwdArgs)]),
    "ssm_ssd_chunk_state_workspace_bytes": (C.c_size_t, [C.POINTER(SsdDims)]),
    "ssm_ssd_combined_supported": (C.c_int, [C.POINTER(SsdDims), C.c_int]),
    "ssm_ssd_combined_workspace_bytes": (C.c_size_t, [C.POINTER(SsdDims)]),
    "ssm_ssd_combined_keep_bytes": (C.c_size_t, [C.POINTER(SsdDims)]),
    "ssm_ssd_combined_scratch_bytes": (C.c_size_t, [C.POINTER(SsdDims)]),
    "ssm_ssd_combined_bwd": (C.c_int, [C.POINTER(SsdCombinedBwdArgs), C.c_void_p]),
    "ssm_ssd_combined_bwd_supported": (C.c_int, [C.POINTER(SsdDims), C.c_int]),
    "ssm_ssd_combined_bwd_workspace_bytes": (C.c_size_t, [C.POINTER(SsdDims)]),
    "ssm_conv1d_bwd_workspace_bytes": (C.c_size_t, [C.c_int, C.c_int, C.c_int]),
    "ssm_norm_bwd_workspace_bytes": (C.c_size_t, [C.c_int, C.c_int]),
}

# exported by the test-hooks build only (include/ssm_amd_testing.h)
HOOKS_SYMBOLS = {
    "ssm_ssd_mfma_launches": (C.c_int, []),
    "ssm_scan_fwd_rows_per_workgroup": (C.c_int, [C.c_int] * 5),
    "ssm_scan_bwd_rows_per_workgroup": (C.c_int, [C.c_int] * 6),
}
HOOKS_LIB_PATH = LIB_PATH.with_name("libssm_amd_testhooks.so")

# The native host path of repeated calls (csrc/host/host.cpp), an extension module beside the library.
HOST_PATH = Path(__file__).resolve().parent / "lib" / "_host.so"


class _HostMissing:
    """Stands in for the module where it cannot be loaded: knows no form, so that every call takes the checks of the Python
    side to the same kernels (SSD training: the backward made of passes of the forward's kernels)."""

    def bind(self, handle, error):
        pass

    def __getattr__(self, name):
        if name.startswith("_"):
            raise AttributeError(name)
        return lambda *call: None


def _load_host(path=HOST_PATH):
    try:
        spec = importlib.util.spec_from_file_location("_host", path)
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        return mod
    except (ImportError, OSError) as exc:
        warnings.warn(f"{path.name} cannot be loaded, calls take 10 to 100 us longer on the host ({exc}); build it with "
                      "`python -m ssm_amd.build`", RuntimeWarning, stacklevel=2)
        return _HostMissing()


host = _load_host()

_lock = threading.Lock()
_libs: dict = {}                     # hooks? -> CDLL
_load_errors: dict = {}              # hooks? -> Exception
_hooks_active = 0                    # depth of test_hooks_build() contexts


def _bind(path: Path, hooks: bool) -> C.CDLL:
    if not path.exists():
        raise FileNotFoundError(f"{path} not found: build it with `python -m ssm_amd.build`")
    lib = C.CDLL(str(path))
    plain = dict(PLAIN_SYMBOLS, **HOOKS_SYMBOLS) if hooks else PLAIN_SYMBOLS
    for name, (res, argt) in plain.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = argt
    got = lib.ssm_amd_abi_version()
    if got != ABI_VERSION:
        raise RuntimeError(f"{path.name} ABI {got}, binding expects {ABI_VERSION}")
    for name, struct in ENTRY_POINTS.items():
        fn = getattr(lib, name)
        fn.restype = C.c_int
        fn.argtypes = [C.POINTER(struct), _vp]
    return lib


def _load(hooks: bool) -> C.CDLL:
    lib = _libs.get(hooks)
    if lib is not None:
        return lib
    with _lock:
        if hooks in _libs:
            return _libs[hooks]
        if hooks in _load_errors:
            raise BackendUnavailable(str(_load_errors[hooks]))
        try:
            lib = _bind(HOOKS_LIB_PATH if hooks else LIB_PATH, hooks)
            if hooks == (_hooks_active > 0):
                host.bind(lib._handle, KernelError)
            _libs[hooks] = lib
        except Exception as exc:  # remembered: a broken install stays broken
            _load_errors[hooks] = exc
            raise BackendUnavailable(str(exc)) from exc
    return _libs[hooks]


def load() -> C.CDLL:
    """The shipped library, loaded once; raises :class:`BackendUnavailable` if impossible.  Inside
    :func:`test_hooks_build` the test-hooks build stands in for it."""
    return _load(_hooks_active > 0)


def load_test_hooks() -> C.CDLL:
    """The ``-DSSM_TEST_HOOKS`` build of the same sources (``include/ssm_amd_testing.h``): reads the argument
    structs' ``reserved`` fields as kernel selectors and exports ``ssm_ssd_mfma_launches``."""
    return _load(True)


class test_hooks_build:
    """Context manager for the test suite: every call inside goes to the test-hooks build, so that
    ``load().ssm_ssd_mfma_launches()`` reports the kernels those calls took."""
    __test__ = False

    def __enter__(self):
        global _hooks_active
        lib = load_test_hooks()
        _hooks_active += 1
        host.bind(lib._handle, KernelError)
        return lib

    def __exit__(self, *exc):
        global _hooks_active
        _hooks_active -= 1
        host.bind(load()._handle, KernelError)
        return False


def available() -> bool:
    try:
        load()
        return True
    except BackendUnavailable:
        return False


def dtype_enum(dt: torch.dtype) -> int:
    try:
        return _DTYPE_ENUM[dt]
    except KeyError:
        raise ValueError(f"unsupported dtype {dt}: the HIP backend handles float32, bfloat16 and float16")


def ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


def stream_handle(device: torch.device) -> int:
    """The raw HIP stream that torch currently launches on for ``device``."""
    index = device.index
    if index is None:
        index = torch.cuda.current_device()
    return torch._C._cuda_getCurrentRawStream(index)


def call(name: str, args: C.Structure, device: torch.device) -> None:
    """Invoke an entry point on the current stream of ``device``; a contract
    violation reported by the library surfaces as ``ValueError`` (as the
    reference's compiled backends do, src/ssm/ops/__init__.py:1244-1252)."""
    # a kernel selector in the struct only means something to the test-hooks build
    lib = load_test_hooks() if getattr(args, "reserved", 0) else load()
    fn = getattr(lib, name)
    index = device.index
    if index is None or index == torch.cuda.current_device():
        status = fn(C.byref(args), stream_handle(device))        # the usual case: no device switch to pay for
    else:
        with torch.cuda.device(device):
            status = fn(C.byref(args), stream_handle(device))
    if status != 0:
        detail = lib.ssm_amd_last_error().decode() or lib.ssm_amd_status_string(status).decode()
        if status == -7:
            raise KernelError(f"{name}: {detail}")
        raise ValueError(f"{name}: {detail}")
