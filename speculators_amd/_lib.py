"""Binding of ``libspx_hip.so``: the native module ``_spx_native`` (``csrc/binding.cpp``) for the calls of this
package, ctypes signatures of the same entry points for programs that use the C ABI directly.

There is no CPU or PyTorch fallback: if the library is not built, or a call is
made with tensors that are not on a HIP device, the call raises.
"""

from __future__ import annotations

import ctypes
import os
from ctypes import c_char_p, c_float, c_int, c_int32, c_int64, c_void_p

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("SPX_LIB_PATH") or os.path.join(_HERE, "libspx_hip.so")

_P, _I64, _I, _F = c_void_p, c_int64, c_int, c_float

_I32 = c_int32

# name -> argument types (return type int unless listed in RESTYPES); mirrors include/spx.h
SIGNATURES: dict[str, list] = {
    "spx_vocab_gather": [_P, _I64, _P, _P, _I64, _I64, _I64, _I64, _I, _P],
    "spx_fused_vocab_loss_fwd": [_I, _P, _I64, _P, _I64, _I64, _I64, _I, _P, _P, _P, _P, _P, _P, _I,
                                 _P],
    "spx_fused_vocab_loss_bwd": [_I, _P, _I64, _P, _I64, _I64, _I64, _I, _P, _P, _P, _P, _P, _P, _P,
                                 _I64, _P],
    "spx_fused_vocab_loss_bwd_packed": [_I, _P, _I64, _P, _I64, _I64, _I64, _I, _P, _P, _P, _P, _P, _P, _P,
                                        _P, _I64, _P],
    "spx_ttt_step_reduce": [_P, _P, _P, _P, _I, _P, _I, _I64, _F, _P, _P, _P],
    "spx_ttt_row_lo": [_P, _I, _I64, _I64, _P, _P],
    "spx_ttt_attn_workspace_bytes": [_I64, _I32, _I32, _I32, _I32],
    "spx_ttt_attn_fwd": [_P, _I64, _P, _I64, _P, _I64, _P, _I64, _I32, _I32, _I32, _I32, _F, _P, _P,
                         _P, _I64, _P],
    "spx_ttt_attn_bwd": [_P, _I64, _P, _I64, _P, _I64, _P, _P, _P, _P, _I64, _I32, _I32, _I32, _I32,
                         _F, _P, _I64, _P, _I64, _P, _I64, _P, _I64, _P],
}
SIGNATURES["spx_ttt_attn_bwd_accumulate"] = SIGNATURES["spx_ttt_attn_bwd"]
SIGNATURES["spx_vocab_loss_step_fwd"] = [_I, _P, _I64, _P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I, _P, _P, _P,
                                         _P, _P, _P, _I, _P, _I, _P, _I, _P, _P]
SIGNATURES["spx_ttt_step_mean"] = [_P, _P, _I, _I64, _F, _P, _P, _P, _P]
SIGNATURES["spx_ttt_step_total"] = [_P, _P, _P, _P, _I, _P, _I, _I64, _F, _P, _F, _P, _P, _P, _P, _P]
SIGNATURES["spx_block_total"] = [_P, _P, _P, _P, _I, _P, _F, _I, _I64, _I32, _F, _P, _P, _P, _P, _P]
SIGNATURES["spx_dflash_inputs"] = [_P, _P, _I64, _I32, _I64, _I64, _P, _P, _P, _I, _I, _P, _P, _P, _P, _P]
SIGNATURES["spx_dflash_inputs_checked"] = [*SIGNATURES["spx_dflash_inputs"], _P]
SIGNATURES["spx_ttt_step_terms"] = [_I32, _P, _P, _P, _I, _I64, _F, _P, _P, _P, _P, _P, _P]
SIGNATURES["spx_mask_row_map"] = [_P, _I, _I64, _P, _P, _P, _P]
SIGNATURES["spx_mask_row_lists"] = [_P, _I, _I64, _P, _P, _P, _P, _P]
SIGNATURES["spx_loss_steps_mask"] = [_P, _I, _I64, _I32, _P, _P, _P, _P, _P, _P, _P, _P]
SIGNATURES["spx_loss_steps_pass"] = [_I, _I32, _P, _P, _I64, _P, _I64, _P, _I64, _I64, _I32, _I32, _I32, _I32, _P, _I, _P, _P,
                                     _P, _P, _P, _P, _P, _P, _P, _P, _P, _I64, _P]
SIGNATURES["spx_loss_steps_partials"] = [_I64, _I32, _I32]
SIGNATURES["spx_loss_steps_total"] = [_P, _P, _P, _I, _P, _I, _I64, _I32, _F, _I32, _P, _P, _P, _P, _P, _P, _P, _P, _P]
SIGNATURES["spx_row_tokens"] = [_P, _I64, _P, _I64, _I64, _I64, _I, _P, _P]
SIGNATURES["spx_span_attn_fwd"] = [_P, _I64, _P, _I64, _P, _I64, _P, _P, _I64, _I32, _I32, _I32, _F, _P, _P,
                                   _P, _I64, _P]
SIGNATURES["spx_span_attn_bwd"] = [_P, _I64, _P, _I64, _P, _I64, _P, _P, _P, _P, _P, _I64, _I32, _I32, _I32,
                                   _F, _P, _I64, _P, _I64, _P, _I64, _P, _I64, _P]
SIGNATURES["spx_ttt_attn_fwd_static_max_bytes"] = []
SIGNATURES["spx_ttt_attn_fwd_static"] = [_P, _I64, _P, _I64, _P, _I64, _P, _I64, _I32, _I32, _I32, _I32, _F,
                                         _P, _P, _P]
SIGNATURES["spx_dflash_row_ranges"] = [_P, _I, _I64, _P, _I, _I64, _I32, _I64, _I32, _P, _P, _P, _P, _P, _P]
SIGNATURES["spx_dflash_attn_workspace_bytes"] = [_I64, _I64, _I32, _I32, _I32, _I32]
SIGNATURES["spx_dflash_attn_fwd"] = [_P, _I64, _P, _I64, _P, _I64, _P, _P, _P, _P, _I64, _I64, _I32,
                                     _I32, _I32, _F, _P, _P, _P, _I64, _P]
SIGNATURES["spx_dflash_attn_bwd"] = [_P, _I64, _P, _I64, _P, _I64, _P, _P, _P, _P, _P, _P, _P, _I64,
                                     _I64, _I32, _I32, _I32, _F, _P, _I64, _P, _I64, _P, _I64, _P,
                                     _I64, _P]
SIGNATURES["spx_rmsnorm_fwd"] = [_P, _I64, _P, _P, _I64, _P, _I64, _I64, _F, _P]
SIGNATURES["spx_rmsnorm_pair_fwd"] = [_P, _I64, _P, _P, _I64, _P, _P, _I64, _P, _I64, _I64, _F, _P]
SIGNATURES["spx_rmsnorm_pair_bwd_partial"] = [_P, _I64, _P, _P, _I64, _P, _P, _I64, _P, _I64, _P, _P, _P, _I64, _P,
                                              _I32, _P, _I32, _I64, _I64, _P]
SIGNATURES["spx_rope_qkv"] = [_P, _I64, _P, _I64, _P, _I64, _P, _I64, _P, _P, _I64, _I32, _I32, _I32, _I32, _I32,
                              _I64, _F, _P]
SIGNATURES["spx_cat_bf16"] = [_P, _P, _P, _I32, _P, _P]
SIGNATURES["spx_head_norm_rope"] = [_P, _I64, _P, _I64, _P, _I64, _P, _P, _P, _P, _I64, _I32, _I32, _I32, _I64, _F, _F, _P]
SIGNATURES["spx_head_norm_rope_bwd"] = [_P, _I64, _P, _I64, _P, _I64, _P, _P, _P, _P, _P, _I64, _P, _I32, _I64, _I32, _I32,
                                        _I32, _I64, _F, _P]
SIGNATURES["spx_head_norm_rope_sets"] = [_P, _I32, _P, _I32, _I64, _F, _P]
SIGNATURES["spx_head_norm_rope_bwd_sets"] = [_P, _I32, _P, _I32, _I64, _F, _P]
SIGNATURES["spx_rmsnorm_bwd_slots"] = [_I64, _I64]
SIGNATURES["spx_rmsnorm_bwd"] = [_P, _I64, _P, _P, _I64, _P, _P, _I64, _P, _P, _I64, _I64, _P]
SIGNATURES["spx_add_rmsnorm_fwd"] = [_P, _I64, _P, _I64, _P, _I64, _P, _P, _I64, _P, _I64, _I64, _F, _P]
SIGNATURES["spx_add_rmsnorm_bwd"] = [_P, _I64, _P, _P, _I64, _P, _I64, _P, _P, _I64, _P, _P, _I64, _I64, _P]
SIGNATURES["spx_add_rmsnorm_fwd_parts"] = [_P, _I64, _P, _I32, _P, _I64, _P, _P, _I64, _P, _I64, _I64, _F, _P]
SIGNATURES["spx_rmsnorm_bwd_parts"] = [_P, _I64, _P, _P, _I32, _P, _I64, _P, _P, _I64, _P, _I32, _I64, _I64, _P]
SIGNATURES["spx_rmsnorm_bwd_partial"] = [_P, _I64, _P, _P, _I64, _P, _I64, _P, _P, _I64, _P, _I32, _I64, _I64, _P]
SIGNATURES["spx_rmsnorm_dweight"] = [_P, _I64, _I64, _P, _P]
SIGNATURES["spx_rmsnorm_dweights"] = [_P, _P, _P, _P, _P, _I32, _P]
SIGNATURES["spx_rope_relayout"] = [_P, _I64, _P, _P, _P, _I64, _I64, _I32, _I32, _I32, _I32, _I64, _P]
SIGNATURES["spx_swiglu_rows_fwd"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _P]
SIGNATURES["spx_swiglu_rows_bwd"] = [_P, _I64, _P, _I64, _P, _I64, _P, _I64, _P, _I64, _I64, _I64, _P]
SIGNATURES["spx_swiglu_fwd"] = [_P, _P, _P, _I64, _P]
SIGNATURES["spx_swiglu_bwd"] = [_P, _P, _P, _P, _P, _I64, _P]
SIGNATURES["spx_label_ce_fwd"] = [_P, _I64, _P, _I64, _I64, _I, _I64, _P, _P, _P, _P]
SIGNATURES["spx_label_ce_from_lse"] = [_P, _I64, _P, _I64, _I64, _I, _I64, _P, _P, _P]
SIGNATURES["spx_label_ce_fwd_grad"] = [_P, _I64, _P, _I64, _I64, _I64, _P, _P, _P, _P, _P, _I64, _P]
SIGNATURES["spx_label_ce_bwd"] = [_P, _I64, _P, _P, _P, _I64, _I64, _I, _I64, _P, _I64, _P]
SIGNATURES["spx_label_ce_bwd_packed"] = [_P, _I64, _P, _P, _P, _I64, _I64, _I, _I64, _P, _P, _I64, _P]
SIGNATURES["spx_pack_batch"] = [_P, _I, _I64, _I64, _I64, _P, _P, _I, _P, _P, _P, _I64, _I64, _I,
                                _P, _P, _P, _P, _P, _P, _P]
SIGNATURES["spx_gemm_bf16_nt"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _P]
SIGNATURES["spx_pack_row_map"] = [_P, _P, _I64, _I64, _P, _P, _P]
SIGNATURES["spx_unpack_rows"] = [_P, _I64, _P, _I64, _I64, _I64, _P, _I64, _P]
SIGNATURES["spx_unpack_rows_graded"] = [_P, _I64, _P, _P, _P, _F, _I64, _I64, _I64, _P, _I64, _P]
SIGNATURES["spx_unpack_rows_scaled"] = [_P, _I64, _P, _P, _I64, _I64, _I64, _P, _I64, _P]
SIGNATURES["spx_vocab_loss_step_fwd_grad"] = [_I, _P, _I64, _P, _I64, _I64, _I64, _P, _P, _P, _P, _P, _P, _I,
                                              _P, _I, _P, _I, _P, _P, _P, _I64, _P]
SIGNATURES["spx_vocab_loss_terms_fwd_grad"] = [_I32, _P, _P, _I64, _P, _I64, _I64, _I64, _P, _P, _P, _P, _P, _I, _P, _I, _P,
                                               _I, _P, _P, _P, _I64, _P]
SIGNATURES["spx_gemm_bf16_nt_tail"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _I32, _P, _I64, _P]
SIGNATURES["spx_gemm_tail_workspace_bytes"] = []
SIGNATURES["spx_gemm_bf16_nt_stats"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _P, _P, _P, _I64, _P]
SIGNATURES["spx_gemm_stats_workspace_bytes"] = [_I64, _I64]
SIGNATURES["spx_gemm_bf16_nt_rows"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _P, _P]
SIGNATURES["spx_gemm_bf16_nt_rows_split"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _P, _I32, _P, _I64, _P]
SIGNATURES["spx_gemm_bf16_rows_graded"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _P, _P, _P, _P, _F, _I32, _I32, _P,
                                           _I64, _P]
SIGNATURES["spx_gemm_bf16_tn"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _I, _P]
SIGNATURES["spx_gemm_bf16_tn_auto"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _I, _I, _P, _I64, _P]
SIGNATURES["spx_gemm_tn_parts"] = [_I64, _I64, _I64]
SIGNATURES["spx_gemm_tn_us"] = [_I64, _I64, _I64]
SIGNATURES["spx_gemm_bf16_tn_list"] = [_P, _I, _I, _P, _I64, _P]
SIGNATURES["spx_gemm_tn_list_us"] = [_P, _I, _I]
SIGNATURES["spx_gemm_tn_list_workspace_bytes"] = [_P, _I, _I]
SIGNATURES["spx_gemm_tn_tile"] = [_I64, _I64, _I64]
SIGNATURES["spx_gemm_tn_workspace_bytes"] = [_I64, _I64, _I64]
SIGNATURES["spx_gemm_bf16_tn_f32"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _I, _P]
SIGNATURES["spx_rope_relayout_partial"] = [_P, _I64, _I32, _P, _P, _P, _I64, _I64, _I32, _I32, _I32, _I32, _I32,
                                           _I64, _F, _P]
SIGNATURES["spx_sigmoid_gate_fwd"] = [_P, _I64, _P, _I64, _I32, _P, _I64, _I64, _I32, _I32, _P]
SIGNATURES["spx_sigmoid_gate_bwd"] = [_P, _I64, _P, _I64, _I32, _P, _I64, _P, _I64, _P, _I64, _I32, _I64, _I32,
                                      _I32, _P]
SIGNATURES["spx_gemm_grouped_workspace_bytes"] = [_I64, _I64]
SIGNATURES["spx_gemm_split_workspace_bytes"] = [_I64, _I64, _I32]
SIGNATURES["spx_gemm_bf16_nt_grouped"] = [_P, _I64, _P, _I64, _I64, _P, _I64, _I64, _I64, _I64, _P, _I64, _P,
                                          _I64, _P]
SIGNATURES["spx_gemm_bf16_nn_grouped"] = SIGNATURES["spx_gemm_bf16_nt_grouped"]
SIGNATURES["spx_gemm_bf16_tn_grouped"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _I64, _P, _I64, _I, _I,
                                          _P]
SIGNATURES["spx_gemm_bf16_tn_grouped_multi"] = [_P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _I64, _I64, _P, _I64,
                                                _I, _I, _P]
SIGNATURES["spx_gemm_bf16_grouped_picked"] = [_I, _P, _I64, _P, _I64, _P, _I64, _I64, _P, _I64, _I64, _I64, _I64, _P, _I64, _P,
                                              _I64, _I, _P]
SIGNATURES["spx_gemm_bf16_tn_grouped_picked"] = [_P, _I64, _P, _I64, _P, _I64, _I, _P, _I64, _I64, _I64, _I64, _I64, _P, _I64,
                                                 _I, _I, _P]
SIGNATURES["spx_transpose_bf16"] = [_P, _I64, _I64, _P, _I64, _I64, _I64, _I64, _I64, _P]
SIGNATURES["spx_moe_gather_rows"] = [_P, _I64, _I64, _P, _P, _P, _I64, _I64, _I64, _P]
SIGNATURES["spx_moe_combine_rows"] = [_P, _I64, _I64, _P, _P, _P, _I64, _I64, _I32, _I64, _P]
SIGNATURES["spx_moe_pair_dot"] = [_P, _I64, _P, _I64, _I64, _P, _P, _I64, _I32, _I64, _P]
SIGNATURES["spx_moe_swiglu_bwd"] = [_P, _I64, _P, _P, _P, _I64, _P, _I64, _P, _I64, _P, _I, _I64, _I64, _P]
SIGNATURES["spx_moe_sort_workspace_bytes"] = [_I64, _I64]
SIGNATURES["spx_moe_sort_pairs"] = [_P, _I64, _I32, _I64, _P, _P, _P, _P, _P, _I64, _P]
SIGNATURES["spx_gemm_auto_workspace_bytes"] = [_I, _I64, _I64, _I64, _I32]
SIGNATURES["spx_gemm_auto_us"] = [_I, _I64, _I64, _I64, _I32]
SIGNATURES["spx_gemm_auto_tile"] = [_I, _I64, _I64, _I64, _I32]
SIGNATURES["spx_gemm_graded_workspace_bytes"] = [_I64, _I64, _I64, _I32, _I32]
SIGNATURES["spx_gemm_graded_parts"] = [_I64, _I64, _I64, _I32, _I32, _I64, _I64]
SIGNATURES["spx_gemm_bf16_auto_parts"] = [_I, _P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _I32, _P, _I64, _P, _P]
SIGNATURES["spx_gemm_pair_takes"] = [_I, _I64, _I64, _I64, _I64, _I32]
SIGNATURES["spx_gemm_bf16_pair"] = [_I, _P, _I64, _P, _P, _I64, _P, _I64, _I64, _I64, _I64, _I32, _P, _I64, _P, _P]
SIGNATURES["spx_gemm_bf16_auto"] = [_I, _P, _I64, _P, _I64, _P, _I64, _I64, _I64, _I64, _P, _I32, _P, _I64, _P]
SIGNATURES["spx_stage_upload"] = [_P, _I64, _P, _P, _I64, _I32, _P]
RESTYPES = {"spx_gemm_auto_workspace_bytes": c_int64, "spx_gemm_graded_workspace_bytes": c_int64, "spx_gemm_tn_workspace_bytes": c_int64, "spx_gemm_auto_us": c_float, "spx_gemm_tn_us": c_float, "spx_gemm_tn_list_us": c_float, "spx_gemm_tn_list_workspace_bytes": c_int64, "spx_moe_sort_workspace_bytes": c_int64, "spx_loss_steps_partials": c_int64, "spx_gemm_grouped_workspace_bytes": c_int64, "spx_gemm_tail_workspace_bytes": c_int64, "spx_gemm_stats_workspace_bytes": c_int64, "spx_gemm_split_workspace_bytes": c_int64, "spx_ttt_attn_workspace_bytes": c_int64, "spx_ttt_attn_fwd_static_max_bytes": c_int64, "spx_dflash_attn_workspace_bytes": c_int64,
            "spx_rmsnorm_bwd_slots": c_int64}

_lib = None


class StageSegment(ctypes.Structure):
    """``spx_stage_segment``"""

    _fields_ = [("src", c_void_p), ("dst", c_void_p), ("offset", c_int64), ("bytes", c_int64), ("fd", c_int32)]


class SpxError(RuntimeError):
    pass


def load() -> ctypes.CDLL:
    """Load the shared library (once).  Raises if it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise SpxError(
            f"{LIB_PATH} is missing: build it with `make -C speculators_amd/csrc` "
            "(or __graft_entry__.build()); there is no fallback path"
        )
    lib = ctypes.CDLL(LIB_PATH)
    lib.spx_version.restype = c_int
    lib.spx_version.argtypes = []
    lib.spx_last_error.restype = c_char_p
    lib.spx_last_error.argtypes = []
    for name, argtypes in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = RESTYPES.get(name, c_int)
        fn.argtypes = argtypes
    _lib = lib
    return lib


_native = None


def native():
    """The binding module (``csrc/binding.cpp``): every entry point as a function that takes integers,
    floats, None and HIP tensors (where C takes a pointer) and raises ``SpxError`` on a failed status."""
    global _native
    if _native is None:
        load()  # (first: the module then binds to this build of the library, whatever its path)
        try:
            from . import _spx_native as mod
        except ImportError as exc:
            raise SpxError("speculators_amd/_spx_native.so is missing: build it with "
                           "`make -C speculators_amd/csrc`; there is no fallback path") from exc
        mod.set_error(SpxError)
        _native = mod
    return _native


def call(name: str, *args) -> None:
    getattr(_native or native(), name)(*args)


def ptr(t: torch.Tensor | None):
    """Device pointer of a tensor (None -> NULL).  Refuses host tensors."""
    if t is None:
        return None
    if not t.is_cuda:
        raise SpxError("libspx_hip works on HIP device tensors only (got a CPU tensor)")
    return t.data_ptr()


def stream_ptr(device=None):
    """The current stream of a device (an address; None for a host device, whose tensors no call takes)."""
    if isinstance(device, torch.device):
        if device.type != "cuda":
            return None
        index = device.index
    else:
        index = device
    if index is None:
        index = torch.cuda.current_device()
    return torch._C._cuda_getCurrentRawStream(index)


_zeros: dict = {}


def zero(device, dtype=torch.float32) -> torch.Tensor:
    """A one-element zero, kept per device: the memory behind empty gradient markers.  Never written."""
    key = (device, dtype)
    z = _zeros.get(key)
    if z is None:
        z = _zeros[key] = torch.zeros(1, device=device, dtype=dtype)
    return z


DTYPE_CODE = {torch.bfloat16: 0, torch.float32: 1}
KIND_CODE = {
    torch.bool: 0, torch.uint8: 0, torch.int8: 0, torch.int32: 1, torch.int64: 2,
    torch.float32: 3, torch.bfloat16: 4,
}


def dtype_code(t: torch.Tensor) -> int:
    try:
        return DTYPE_CODE[t.dtype]
    except KeyError:
        raise SpxError(f"unsupported dtype {t.dtype}: bf16 and f32 only") from None


def kind_code(t: torch.Tensor) -> int:
    try:
        return KIND_CODE[t.dtype]
    except KeyError:
        raise SpxError(f"unsupported mask dtype {t.dtype}") from None
