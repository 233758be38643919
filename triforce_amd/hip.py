"""ctypes binding of the C ABIs: libtriforce_hip.so (include/triforce_hip.h, ``lib``) and the libraries of the batch-served model
families - libtriforce_tile.so (include/triforce_tile.h, ``tile_lib``), libtriforce_latent.so (include/triforce_latent.h,
``latent_lib``), libtriforce_hybrid.so (include/triforce_hybrid.h, ``hybrid_lib``).

There is deliberately NO fallback: if the shared library is missing or a symbol is absent the
import of any op raises.  Build it with ``python -m triforce_amd.build`` (hipcc, gfx950).
"""
import ctypes
import os

from .build import HYBRID_LIB_PATH, LATENT_LIB_PATH, LIB_PATH, TILE_LIB_PATH

_c = ctypes
_vp, _i32, _i64, _f32 = _c.c_void_p, _c.c_int, _c.c_int64, _c.c_float

# name -> (restype, argtypes); mirrors include/triforce_hip.h one to one
SIGNATURES = {
    "tf_abi_version": (_i32, []),
    "tf_attn_decode_ws_floats": (_i64, [_i32, _i32, _i32, _i32]),
    "tf_attn_decode_pick_nsplit": (_i32, [_i32, _i32]),
    "tf_attn_decode": (_i32, [_vp, _vp, _vp, _vp, _i64, _i64, _i32, _i32, _vp, _i32, _i32, _f32, _i32, _vp, _i64, _vp]),
    "tf_attn_decode_fused": (_i32, [_vp, _vp, _vp, _vp, _i64, _i64, _i32, _i32, _vp, _i32, _i32, _f32, _i32, _vp, _i64, _vp,
                                    _vp]),
    "tf_attn_decode_act": (_i32, [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i32, _i32, _vp, _i32, _i32, _f32, _i32, _vp,
                                  _i64, _vp, _vp]),
    "tf_attn_tune": (_i32, [_i32, _i32]),
    "tf_attn_block_ws_floats": (_i64, [_i32, _i32, _i32]),
    "tf_attn_block_pick_nsplit": (_i32, [_i32, _i32, _i32]),
    "tf_attn_prefill_pick_nsplit": (_i32, [_i32, _i32, _i32]),
    "tf_attn_prefill_ws_floats": (_i64, [_i32, _i32, _i32, _i32]),
    "tf_attn_prefill": (_i32, [_vp, _vp, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _i32, _vp, _i64, _vp]),
    "tf_attn_block": (_i32, [_vp, _vp, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _i32, _vp, _i64, _vp, _i32,
                             _i32, _i32, _vp]),
    "tf_attn_rope_on_read": (_i32, [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _i32, _f32, _vp]),
    "tf_retrieval_score": (_i32, [_vp, _i64, _i64, _vp, _vp, _i32, _i32, _i32, _i32, _vp]),
    "tf_retrieval_topk": (_i32, [_vp, _vp, _i32, _i32, _i32, _vp]),
    "tf_retrieval_gather": (_i32, [_vp, _vp, _i64, _i64, _vp, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _i32, _vp]),
    "tf_kv_copy_rows": (_i32, [_vp, _i64, _i64, _i64, _vp, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _vp]),
    "tf_kv_shift_rows": (_i32, [_vp, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _vp]),
    "tf_kv_copy_rows_pair": (_i32, [_vp, _vp, _i64, _i64, _i64, _vp, _vp, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _i32,
                                    _i32, _vp]),
    "tf_kv_shift_rows_pair": (_i32, [_vp, _vp, _i64, _i64, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _vp]),
    "tf_kv_gather_rows": (_i32, [_vp, _vp, _i64, _i64, _i64, _i32, _vp, _i32, _i32, _i32, _i32, _vp]),
    "tf_tree_accept": (_i32, [_vp, _vp, _vp, _vp, _vp, _vp, _i32, _f32, _vp, _vp]),
    "tf_sample_without_replacement": (_i32, [_vp, _vp, _vp, _i32, _i32, _i32, _f32, _vp]),
    "tf_rows_gemm_plan": (_i64, [_i32, _i32, _i32, _c.POINTER(_c.c_int32), _c.POINTER(_c.c_int32)]),
    "tf_rows_gemm": (_i32, [_vp, _i64, _vp, _vp, _i64, _vp, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _vp]),
    "tf_rmsnorm": (_i32, [_vp, _vp, _vp, _vp, _vp, _i32, _i32, _f32, _vp]),
    "tf_rope_append": (_i32, [_vp, _i64, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i32, _vp, _i32, _i32, _i32, _i32, _vp]),
    "tf_silu_mul": (_i32, [_vp, _vp, _i32, _i32, _vp]),
    "tf_embed_rows": (_i32, [_vp, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _vp]),
    "tf_set_tokens": (_i32, [_vp, _i32, _vp, _i32, _i64, _vp, _i32, _i64, _vp, _vp, _i32, _vp]),
    "tf_skinny_gemm": (_i32, [_vp, _vp, _i64, _vp, _i64, _i32, _i32, _i32, _i32, _vp]),
    "tf_skinny_gemm_ex": (_i32, [_vp, _vp, _i64, _vp, _f32, _vp, _vp, _i64, _vp, _vp, _i64, _i32, _i32, _i32, _i32, _vp]),
    "tf_skinny_gemm_swiglu_ex": (_i32, [_vp, _vp, _vp, _i64, _vp, _f32, _vp, _vp, _i64, _i32, _i32, _i32, _vp]),
    "tf_skinny_qkv_rope": (_i32, [_vp, _vp, _i64, _vp, _f32, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i32, _vp,
                                  _i32, _i32, _i32, _i32, _i32, _vp]),
    "tf_skinny_gemm_swiglu": (_i32, [_vp, _vp, _vp, _i64, _vp, _i64, _i32, _i32, _i32, _vp]),
    "tf_skinny_gemm_act": (_i32, [_vp, _vp, _i64, _i64, _vp, _f32, _vp, _vp, _i64, _i64, _vp, _vp, _i64, _i64, _i32, _i32,
                                  _i32, _i32, _vp]),
    "tf_skinny_gemm_swiglu_act": (_i32, [_vp, _vp, _vp, _i64, _i64, _vp, _f32, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _vp]),
    "tf_skinny_qkv_rope_act": (_i32, [_vp, _vp, _i64, _i64, _vp, _f32, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i32,
                                      _vp, _i32, _i32, _i32, _i32, _i32, _vp]),
    "tf_wide_gemm_takes": (_i32, [_i32, _i32, _i32]),
    "tf_wide_gemm_act": (_i32, [_vp, _vp, _i64, _i64, _vp, _f32, _vp, _vp, _i64, _i64, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _i32, _vp]),
    "tf_wide_gemm_swiglu_act": (_i32, [_vp, _vp, _i64, _i64, _vp, _f32, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _vp]),
    "tf_wide_qkv_rope_act": (_i32, [_vp, _vp, _i64, _i64, _vp, _f32, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i32, _vp, _i32, _i32, _i32,
                                    _i32, _i32, _vp]),
    "tf_skinny_gemm_swiglu_n8": (_i32, [_vp, _vp, _vp, _i64, _i64, _vp, _f32, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _vp]),
    "tf_skinny_qkv_rope_n8": (_i32, [_vp, _vp, _i64, _i64, _vp, _f32, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i32,
                                     _vp, _i32, _i32, _i32, _i32, _i32, _vp]),
    "tf_sg_tune": (_i32, [_i32, _i32]),
    "tf_sg_workspace": (_i32, [_vp, _i64]),
    "tf_topp_probs": (_i32, [_vp, _vp, _i32, _i32, _f32, _f32, _vp]),
    "tf_sample_inverse_cdf": (_i32, [_vp, _vp, _vp, _i32, _vp]),
    "tf_accept_chain": (_i32, [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _i64, _vp, _vp]),
    "tf_middle_accept": (_i32, [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _vp, _vp]),
    "tf_mid_record_tokens": (_i32, [_vp, _vp, _i32, _i32, _vp]),
    "tf_sample_inverse_cdf_cur": (_i32, [_vp, _vp, _vp, _i32, _vp, _i32, _vp]),
    "tf_middle_accept_cur": (_i32, [_vp, _vp, _vp, _i32, _vp, _vp, _i32, _i32, _i32, _vp, _vp]),
    "tf_accept_chain_step": (_i32, [_vp, _vp, _vp, _i32, _vp, _vp, _i32, _i32, _i32, _i64, _i64, _vp, _i32,
                                    _vp, _i32, _vp, _vp, _i32, _vp, _i32, _vp, _vp, _i32, _vp, _vp]),
    "tf_accept_chain_cur": (_i32, [_vp, _vp, _vp, _vp, _vp, _i32, _i32, _i32, _i64, _vp, _vp]),
    "tf_kv_h2d_async": (_i32, [_vp, _i64, _vp, _i64, _i64, _i32, _vp]),
    "tf_kv_d2h_async": (_i32, [_vp, _i64, _vp, _i64, _i64, _i32, _vp]),
    "tf_ar_flags_bytes": (_i32, []),
    "tf_ar_ipc_handle_bytes": (_i32, []),
    "tf_ar_alloc": (_i32, [_i64, _vp]),
    "tf_ar_free": (_i32, [_vp]),
    "tf_ar_get_ipc_handle": (_i32, [_vp, _vp]),
    "tf_ar_open_ipc_handle": (_i32, [_vp, _vp]),
    "tf_ar_close_ipc_handle": (_i32, [_vp]),
    "tf_allreduce_oneshot": (_i32, [_vp, _vp, _i32, _i32, _vp, _i64, _vp]),
    "tf_allreduce_oneshot_add": (_i32, [_vp, _vp, _i32, _i32, _vp, _vp, _i64, _vp]),
    "tf_allreduce_oneshot_add_ss": (_i32, [_vp, _vp, _i32, _i32, _vp, _vp, _i64, _i32, _vp, _vp]),
    "tf_allreduce_oneshot_alt": (_i32, [_vp, _vp, _i32, _i32, _vp, _vp, _i64, _i32, _vp, _i64, _i32, _vp]),
    "tf_allreduce_oneshot_act": (_i32, [_vp, _vp, _i32, _i32, _vp, _vp, _i64, _i32, _i32, _vp, _i64, _i32, _vp]),
    "tf_ar_litmus_stage": (_i32, [_vp, _i64, _i32, _vp, _vp]),
    "tf_ar_litmus_check": (_i32, [_vp, _i64, _i32, _vp, _vp, _vp]),
    "tf_xchg_ctl_bytes": (_i64, []),
    "tf_skinny_gemm_xchg": (_i32, [_vp, _vp, _i64, _i64, _vp, _vp, _i32, _i32, _i64, _vp, _i64, _i64, _vp, _i64, _i64, _vp,
                                   _i32, _i32, _i32, _vp]),
    "tf_xchg_error": (_i32, [_vp]),
    "tf_xchg_set_error": (_i32, [_vp, _i32, _vp, _i32]),
    "tf_xchg_tune": (_i32, [_i32, _i32]),
    "tf_xchg_reset": (_i32, [_vp]),
    "tf_ar_error": (_i32, [_vp]),
    "tf_ar_epoch": (_i64, [_vp]),
    "tf_ar_set_error_mirror": (_i32, [_vp, _vp]),
    "tf_ar_inject_error": (_i32, [_vp, _i32]),
}

TF_DRAFT_MAX_LAYERS = 8


class TfDraftModel(_c.Structure):
    """include/triforce_hip.h: TfDraftModel (device pointers of the 68M draft model's weights)."""
    _fields_ = ([("embed", _vp)] + [(n, _vp * TF_DRAFT_MAX_LAYERS) for n in
                                    ("ln1", "wqkv", "wo", "ln2", "wgate", "wup", "wdown")]
                + [("norm", _vp), ("lm_head", _vp), ("cos", _vp), ("sin", _vp)]
                + [(n, _i32) for n in ("layers", "hidden", "heads", "head_dim", "inter", "vocab")]
                + [("eps", _f32), ("scale", _f32)])


class TfDraftCache(_c.Structure):
    _fields_ = [("k", _vp * TF_DRAFT_MAX_LAYERS), ("v", _vp * TF_DRAFT_MAX_LAYERS), ("stride_t", _i64), ("stride_h", _i64)]


SIGNATURES["tf_draft_forward_ws_bytes"] = (_i64, [_c.POINTER(TfDraftModel), _i32])
SIGNATURES["tf_draft_forward_68m"] = (_i32, [_c.POINTER(TfDraftModel), _c.POINTER(TfDraftCache), _vp, _i32, _i32, _i32, _vp,
                                             _vp, _f32, _f32, _vp, _i64, _vp])
SIGNATURES["tf_topp_multi_ctl_bytes"] = (_i64, [])
SIGNATURES["tf_topp_multi_ws_bytes"] = (_i64, [_i32, _i32])
SIGNATURES["tf_topp_probs_multi"] = (_i32, [_vp, _vp, _vp, _i32, _i32, _f32, _f32, _vp, _vp, _i64, _vp])
SIGNATURES["tf_topp_multi_tune"] = (_i32, [_i32, _i32])
SIGNATURES["tf_topp_multi_error"] = (_i32, [_vp])
SIGNATURES["tf_topp_multi_reset"] = (_i32, [_vp])
SIGNATURES["tf_draft_persist_ctl_bytes"] = (_i64, [])
SIGNATURES["tf_draft_persist_ws_bytes"] = (_i64, [_c.POINTER(TfDraftModel)])
SIGNATURES["tf_draft_persist_supported"] = (_i32, [_c.POINTER(TfDraftModel), _i32, _i32])
SIGNATURES["tf_draft_forward_68m_persist"] = (_i32, [_c.POINTER(TfDraftModel), _c.POINTER(TfDraftCache), _vp, _i32, _i32, _i32,
                                                     _vp, _vp, _f32, _f32, _vp, _i64, _vp, _vp])
SIGNATURES["tf_draft_persist_tune"] = (_i32, [_i32, _i32])
SIGNATURES["tf_draft_persist_stamps"] = (_i32, [_vp])
SIGNATURES["tf_draft_persist_error"] = (_i32, [_vp])
SIGNATURES["tf_draft_persist_reset"] = (_i32, [_vp, _vp, _i32])

ABI_VERSION = 1
_lib = None

# ---- libtriforce_tile.so (include/triforce_tile.h) ------------------------------------------------------------------
TFL_PAGE = 64
TFL_MAX_ENTRIES = 64
TFL_EPI = {n: i for i, n in enumerate(("f32", "in", "query", "latent", "gated", "residual", "token", "glu"))}


class TflDecodePrep(_c.Structure):
    """include/triforce_tile.h: TflDecodePrep."""
    _fields_ = [(n, _vp) for n in ("len", "table", "pos", "slot", "klen")] + [(n, _i32) for n in ("table_ld", "table_cols", "rows")]


class TflGemm(_c.Structure):
    """include/triforce_tile.h: TflGemm."""
    _fields_ = ([(n, _vp) for n in ("wp", "x", "norm_w", "ss_in", "out_t", "out_t2", "out_f", "ss_out", "gate", "tok_table", "ids",
                                    "pos", "cos", "sin", "kv_raw", "kv_norm_w", "cache", "slot")]
                + [(n, _i64) for n in ("ld_x", "x_oct", "x_group", "ld_t", "t_oct", "ld_f", "ld_gate", "ld_tok", "ld_kv")]
                + [(n, _i32) for n in ("rows", "n", "k", "groups", "n_real", "k_real", "n_raw", "n_scaled", "ss_n", "ss_ld", "H", "N", "R", "C",
                                       "half", "c_real", "max_pos", "cache_rows", "vocab")]
                + [("eps", _f32), ("chunk_major", _i32), ("n_also", _i32), ("also", _vp)])


TILE_SIGNATURES = {
    "tfl_tile_abi_version": (_i32, []),
    "tfl_gemm": (_i32, [_c.POINTER(TflGemm), _i32, _i32, _vp]),
    "tfl_gemm_carry": (_i32, [_c.POINTER(TflGemm), _c.POINTER(TflGemm), _vp]),
    "tfl_split_gemm_ws_floats": (_i64, [_i32, _i32, _i32, _i32]),
    "tfl_split_gemm": (_i32, [_vp, _vp, _i64, _vp, _i64, _vp, _i64, _i32, _i32, _i32, _i32, _vp]),
    "tfl_rows_gemm_plan": (_i64, [_i32, _i32, _i32, _c.POINTER(_c.c_int32), _c.POINTER(_c.c_int32)]),
    "tfl_rows_gemm": (_i32, [_vp, _i64, _vp, _vp, _i64, _vp, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _vp]),
    "tfl_set_pages": (_i32, [_vp, _i32, _i32, _i32, _c.POINTER(_c.c_int32), _i32, _vp]),
    "tfl_decode_prep": (_i32, [_vp, _vp, _i32, _i32, _vp, _vp, _vp, _i32, _vp]),
}
TILE_ABI_VERSION = 3
_tile = None

# ---- libtriforce_latent.so (include/triforce_latent.h) ------------------------------------------------------------------
class TflFinish(_c.Structure):
    """include/triforce_latent.h: TflFinish."""
    _fields_ = [(n, _vp) for n in ("y", "y_w", "step", "norm_w", "x", "x_out")] + [("ld_y", _i64), ("width", _i32), ("width_real", _i32), ("eps", _f32)]


LATENT_SIGNATURES = {
    "tfl_token_side_ws_floats": (_i64, [_i32, _i32]),
    "tfl_token_side": (_i32, [_vp, _vp, _vp, _i64, _i64, _vp, _i64, _vp, _i32, _vp, _i64, _vp, _i64, _i32, _i32, _i32, _i32, _i32, _vp]),
    "tfl_finish_gemm_takes": (_i32, [_i32] * 6),
    "tfl_finish_gemm": (_i32, [_c.POINTER(TflFinish), _c.POINTER(TflGemm), _i32, _vp]),
    "tfl_abi_version": (_i32, []),
    "tfl_finish": (_i32, [_vp, _vp, _i32, _vp, _i32, _i64, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _f32, _i32, _vp]),
    "tfl_residual": (_i32, [_vp, _vp, _vp, _i64, _i32, _vp]),
    "tfl_token_gate": (_i32, [_vp, _i64, _vp, _i64, _vp, _i32, _vp, _i32, _i32, _i32, _i32, _vp]),
    "tfl_prepare": (_i32, [_vp, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp, _vp, _f32, _vp, _vp, _i32, _i32, _vp, _vp,
                           _vp, _i32, _vp, _vp, _vp, _i64, _i32, _i32, _vp]),
    "tfl_gather_rows": (_i32, [_vp, _i32, _vp, _vp, _i32, _i32, _i32, _vp]),
    "tfl_attn_prefill": (_i32, [_vp, _vp, _vp, _vp, _i32, _i32, _vp, _vp, _vp, _i32, _i32, _vp, _i64, _vp, _i64, _i32, _i32, _i32,
                                _i32, _i32, _i32, _i32, _f32, _i32, _vp]),
    "tfl_attn_decode_ws_floats": (_i64, [_i32, _i32, _i32, _i32]),
    "tfl_attn_decode_splits": (_i32, [_i32, _i32, _i32, _i32, _i32, _i32]),
    "tfl_attn_decode_pick_nsplit": (_i32, [_i32, _i32, _i32]),
    "tfl_attn_beside_plan": (_i32, [_i32, _i32, _i32, _i32, _i64, _i32, _i32] + 3 * [_c.POINTER(_c.c_int32)]),
    "tfl_attn_beside_plan_of": (_i32, [_i32, _i32, _i32, _i32, _i64, _i64, _i32, _i32] + 3 * [_c.POINTER(_c.c_int32)]),
    "tfl_attn_decode_beside_parts": (_i32, [_vp, _vp, _i32, _vp, _i32, _vp, _vp, _vp, _i64, _i32, _i32, _f32, _i32, _i32, _i32, _c.POINTER(TflGemm), _vp]),
    "tfl_finish_first": (_i32, [_vp, _vp, _i32, _vp, _vp, _vp, _vp, _i64, _i64, _i32, _i32, _i32, _f32, _c.POINTER(TflDecodePrep), _i32, _vp]),
    "tfl_beside_parts": (_i32, [_i32, _i32, _i32, _i32, _i64, _i64, _i32, _i32, _c.POINTER(_c.c_int32), _c.POINTER(_c.c_int32)]),
    "tfl_latent_carry": (_i32, [_i32, _i32, _i32, _i32, _i64, _i64, _i32, _i32]),
    "tfl_latent_value": (_i32, [_vp, _i64, _i32, _c.POINTER(TflGemm), _vp]),
    "tfl_attn_decode_beside": (_i32, [_vp, _vp, _i32, _vp, _i32, _vp, _vp, _vp, _i64, _i32, _i32, _f32, _i32, _i32, _i32, _c.POINTER(TflGemm), _vp]),
    "tfl_attn_decode": (_i32, [_vp, _vp, _i32, _vp, _i32, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _i32, _f32, _i32, _i32, _vp]),
}
LATENT_ABI_VERSION = 2
_latent = None


# ---- libtriforce_hybrid.so (include/triforce_hybrid.h) ------------------------------------------------------------------
class TfhRecurrence(_c.Structure):
    """include/triforce_hybrid.h: TfhRecurrence."""
    _fields_ = ([(n, _vp) for n in ("q", "k", "v", "gcum", "dt", "nega", "skip", "gate", "state", "part", "decay", "out", "seq", "seg", "span")]
                + [(n, _i64) for n in ("ld_q", "ld_k", "ld_v", "ld_gate", "ld_out")]
                + [(n, _i32) for n in ("nseq", "nseg", "max_segs", "tokens", "seats", "H", "per_group", "N", "V")]
                + [("q_scale", _f32)])


class TfhAttnStep(_c.Structure):
    """include/triforce_hybrid.h: TfhAttnStep."""
    _fields_ = ([(n, _vp) for n in ("q_norm", "k_norm", "cos", "sin", "cache", "table", "ws")] + [("n_pages", _i64)]
                + [(n, _i32) for n in ("q_off", "k_off", "v_off", "gate_off", "half", "max_pos", "table_ld", "H", "G", "D", "D_real", "V",
                                       "chunk", "nsplit")]
                + [(n, _f32) for n in ("scale", "out_scale")])


class TfhRecStep(_c.Structure):
    """include/triforce_hybrid.h: TfhRecStep."""
    _fields_ = ([(n, _vp) for n in ("conv_w", "conv_b", "ring", "dt_bias", "nega", "skip", "a2", "a2_b", "norm_w", "state", "seat", "out")]
                + [(n, _i32) for n in ("x_off", "dt_off", "gate_off", "q_off", "k_off", "v_off", "a_off", "taps", "channels", "rank", "seats",
                                       "H", "per_group", "N", "V", "V_real", "norm_groups")]
                + [(n, _f32) for n in ("inv_tau", "q_scale", "out_scale")])


class TfhConnect(_c.Structure):
    """include/triforce_hybrid.h: TfhConnect."""
    _fields_ = ([(n, _vp) for n in ("y", "out", "mix", "in", "norm_w", "x", "x_out")] + [("ld_y", _i64)]
                + [(n, _i32) for n in ("streams", "width", "width_real")] + [("eps", _f32)])


HYBRID_SIGNATURES = {
    "tfh_connect_gemm_takes": (_i32, [_i32] * 6),
    "tfh_connect_first": (_i32, [_vp, _vp, _i32, _vp, _vp, _vp, _vp, _i32, _vp, _i64, _i64, _i32, _i32, _i32, _f32, _c.POINTER(TflDecodePrep), _i32, _vp]),
    "tfh_streams_gemm_takes": (_i32, [_i32] * 4),
    "tfh_streams_gemm": (_i32, [_c.POINTER(TfhConnect), _c.POINTER(TflGemm), _vp]),
    "tfh_scaled_gemm_takes": (_i32, [_i32] * 3),
    "tfh_scaled_gemm": (_i32, [_c.POINTER(TflGemm), _i32, _vp]),
    "tfh_connect_gemm": (_i32, [_c.POINTER(TfhConnect), _c.POINTER(TflGemm), _i32, _vp]),
    "tfh_abi_version": (_i32, []),
    "tfh_connect": (_i32, [_vp, _vp, _i32, _vp, _vp, _i32, _i64, _vp, _vp, _vp, _vp, _vp, _i32, _i32, _vp, _i64, _i64, _i32, _i32, _i32,
                           _f32, _i32, _vp]),
    "tfh_qkv_prepare": (_i32, [_vp, _i64, _i32, _i32, _i32, _vp, _vp, _vp, _vp, _i32, _i32, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _i32,
                               _i32, _i32, _f32, _i32, _vp]),
    "tfh_attn_prefill": (_i32, [_vp, _i64, _vp, _i64, _vp, _i32, _vp, _i32, _i32, _vp, _i64, _vp, _i64, _i32, _i32, _i32, _i32, _i32, _i32,
                                _f32, _f32, _i32, _vp]),
    "tfh_conv_prepare": (_i32, [_vp, _i64, _i32, _i32, _vp, _vp, _i32, _i32, _vp, _i32, _vp, _i32, _vp, _vp, _vp, _i32, _i32, _i32, _i32,
                                _vp]),
    "tfh_decay_prepare": (_i32, [_vp, _i64, _vp, _f32, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _vp]),
    "tfh_recurrence": (_i32, [_c.POINTER(TfhRecurrence), _i32, _vp]),
    "tfh_group_norm": (_i32, [_vp, _i64, _vp, _i64, _i32, _vp, _i32, _vp, _i64, _i64, _i32, _i32, _i32, _i32, _i32, _f32, _f32, _i32, _vp]),
    "tfh_glu": (_i32, [_vp, _vp, _i32, _i32, _i32, _vp]),
    "tfh_attn_step_ws_floats": (_i64, [_i32, _i32, _i32, _i32]),
    "tfh_attn_step_splits": (_i32, [_i32, _i32, _i32, _i32, _i32, _i32, _i32]),
    "tfh_attn_step_pick_nsplit": (_i32, [_i32, _i32, _i32, _i32]),
    "tfh_step": (_i32, [_c.POINTER(TfhAttnStep), _c.POINTER(TfhRecStep), _vp, _i64, _vp, _i32, _f32, _i32, _vp]),
    "tfh_step_out": (_i32, [_c.POINTER(TfhAttnStep), _c.POINTER(TfhRecStep), _vp, _i64, _vp, _i64, _i64, _i32, _f32, _i32, _vp]),
}
HYBRID_ABI_VERSION = 1
_hybrid = None


class TriforceHipError(RuntimeError):
    pass


def _preload_torch_hip_runtime():
    """PyTorch-ROCm ships its own libamdhip64.so.7.  Our library must bind to THAT runtime instance (the one
    that owns torch's device context and streams): load it first so the dynamic linker reuses it for our
    NEEDED libamdhip64.so.7 instead of opening the system copy as a second, uninitialised runtime
    (symptom: every launch fails with hipErrorNoDevice)."""
    import torch  # noqa: F401  (imports libtorch_hip -> torch/lib/libamdhip64.so)
    cand = os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so")
    if os.path.exists(cand):
        ctypes.CDLL(cand, mode=ctypes.RTLD_GLOBAL)


def _load(path, signatures, version_fn, version):
    """Open a library and bind its entry points; raises (never falls back) when anything is missing."""
    _preload_torch_hip_runtime()
    if not os.path.exists(path):
        raise TriforceHipError(
            f"{path} not found: the HIP extension is required (python -m triforce_amd.build); "
            "there is no CPU fallback")
    L = ctypes.CDLL(path)
    for name, (res, args) in signatures.items():
        try:
            fn = getattr(L, name)
        except AttributeError as e:
            raise TriforceHipError(f"{path} does not export {name}") from e
        fn.restype, fn.argtypes = res, args
    have = getattr(L, version_fn)()
    if have != version:
        raise TriforceHipError(f"ABI mismatch: library {have} != binding {version}")
    return L


def lib():
    """The core library."""
    global _lib
    if _lib is None:                                               # TRIFORCE_HIP_LIB: tuning builds (triforce_amd.build.build_variant)
        _lib = _load(os.environ.get("TRIFORCE_HIP_LIB", LIB_PATH), SIGNATURES, "tf_abi_version", ABI_VERSION)
    return _lib


def tile_lib():
    """The library the batch-served families share."""
    global _tile
    if _tile is None:
        _tile = _load(TILE_LIB_PATH, TILE_SIGNATURES, "tfl_tile_abi_version", TILE_ABI_VERSION)
    return _tile


def latent_lib():
    """The latent-attention library."""
    global _latent
    if _latent is None:
        _latent = _load(LATENT_LIB_PATH, LATENT_SIGNATURES, "tfl_abi_version", LATENT_ABI_VERSION)
    return _latent


def hybrid_lib():
    """The library of chunked attention, linear recurrences and residual streams."""
    global _hybrid
    if _hybrid is None:
        _hybrid = _load(HYBRID_LIB_PATH, HYBRID_SIGNATURES, "tfh_abi_version", HYBRID_ABI_VERSION)
    return _hybrid


def check(rc, what):
    if rc != 0:
        kind = {-22: "TF_EINVAL", -28: "TF_ENOSPC", -34: "TF_ERANGE"}.get(rc, f"hipError {rc}" if rc > 0 else str(rc))
        raise TriforceHipError(f"{what} failed: {kind}")
