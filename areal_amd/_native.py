"""ctypes binding of ``libareal_amd.so`` (the C ABI declared in ``include/areal_amd.h``).

The library is loaded from the package directory.  There is no fallback: if it
is missing or a call returns a non-zero status, an exception is raised.
"""
from __future__ import annotations

import ctypes as C
import threading
from pathlib import Path

LIB_PATH = Path(__file__).resolve().parent / "libareal_amd.so"
HOST_PATH = LIB_PATH.with_name("_host.so")

AA_OK = 0
AA_ERR_INVALID_ARGUMENT = 1
AA_LMHEAD_COUNT_ON_DEVICE = -1  # a kept_per_chunk entry: the device counts the rows itself
AA_ERR_UNSUPPORTED = 2
AA_ERR_LAUNCH = 3
AA_BF16, AA_F16, AA_F32 = 0, 1, 2

RS_LEVEL = {"token": 0, "sequence": 1}
RS_ACTION = {"mask": 0, "clamp": 1}
RS_METRIC = {"ratio": 0, "kl_k1": 1, "kl_k2": 2, "kl_k3": 3}
RS_AGG = {"sum": 0, "mean": 1, "max": 2}


class NativeLibraryError(RuntimeError):
    """The HIP library is missing, incomplete, or a call into it failed."""


class PpoParams(C.Structure):
    """``aa_ppo_params``"""

    _fields_ = [
        ("clip_lo", C.c_float),
        ("clip_hi", C.c_float),
        ("c_clip", C.c_float),
        ("has_c_clip", C.c_int32),
        ("has_behave_weight", C.c_int32),
        ("loss_kind", C.c_int32),
        ("sapo_tau_pos", C.c_float),
        ("sapo_tau_neg", C.c_float),
    ]


class RsParams(C.Structure):
    """``aa_rs_params``"""

    _fields_ = [
        ("enabled", C.c_int32),
        ("level", C.c_int32),
        ("action", C.c_int32),
        ("metric", C.c_int32),
        ("agg", C.c_int32),
        ("has_lower", C.c_int32),
        ("upper", C.c_float),
        ("lower", C.c_float),
    ]


class LossScale(C.Structure):
    """``aa_loss_scale``"""

    _fields_ = [
        ("factor", C.c_void_p),
        ("total", C.c_void_p),
        ("value", C.c_float),
        ("total_value", C.c_float),
        ("per_valid_token", C.c_int32),
    ]


STEP_WORK_BYTES = 4096  # AA_STEP_WORK_BYTES


class PpoStep(C.Structure):
    """``aa_ppo_step``"""

    _fields_ = [
        ("T", C.c_int64),
        ("T_active", C.c_int64),
        ("prox_logp", C.c_void_p),
        ("old_logp", C.c_void_p),
        ("adv", C.c_void_p),
        ("mask", C.c_void_p),
        ("cu_seqlens", C.c_void_p),
        ("n_segments", C.c_int64),
        ("params", PpoParams),
        ("rs", RsParams),
        ("scale", LossScale),
        ("logp", C.c_void_p),
        ("entropy", C.c_void_p),
        ("vmax", C.c_void_p),
        ("vmin", C.c_void_p),
        ("stat_loss", C.c_void_p),
        ("ratio", C.c_void_p),
        ("flags", C.c_void_p),
        ("approx_kl", C.c_void_p),
        ("clip_mask", C.c_void_p),
        ("dual_clip_mask", C.c_void_p),
        ("behave_mask", C.c_void_p),
        ("behave_kl", C.c_void_p),
        ("mask_out", C.c_void_p),
        ("behave_w", C.c_void_p),
        ("counts", C.c_void_p),
        ("counts_given", C.c_int32),
        ("loss", C.c_void_p),
        ("host_counts", C.c_void_p),
        ("host_tag", C.c_int32),
        ("work", C.c_void_p),
    ]


class NormParams(C.Structure):
    """``aa_norm_params``"""

    _fields_ = [
        ("mean_level", C.c_int32),
        ("mean_leave1out", C.c_int32),
        ("std_level", C.c_int32),
        ("std_unbiased", C.c_int32),
        ("eps", C.c_float),
        ("group_size", C.c_int64),
    ]


class AdvantageStep(C.Structure):
    """``aa_advantage_step``"""

    _fields_ = [
        ("bs", C.c_int64),
        ("L", C.c_int64),
        ("loss_mask", C.c_void_p),
        ("loss_mask_bytes", C.c_int32),
        ("roll_logp", C.c_int32),
        ("logp", C.c_void_p),
        ("ref_logp", C.c_void_p),
        ("attention_mask", C.c_void_p),
        ("seqlens", C.c_void_p),
        ("reward_score", C.c_void_p),
        ("values", C.c_void_p),
        ("kl_ctl", C.c_float),
        ("discount", C.c_float),
        ("gae_lambda", C.c_float),
        ("kl_estimator", C.c_int32),
        ("mask_no_eos_with_zero", C.c_int32),
        ("norm", C.POINTER(NormParams)),
        ("mask_out", C.c_void_p),
        ("logp_out", C.c_void_p),
        ("kl_rewards", C.c_void_p),
        ("rewards", C.c_void_p),
        ("advantages", C.c_void_p),
        ("returns", C.c_void_p),
        ("scratch", C.c_void_p),
        ("scratch_bytes", C.c_int64),
        ("work", C.c_void_p),
    ]


SCORE_GROUP = 64  # AA_SCORE_GROUP


class ScoreStep(C.Structure):
    """``aa_score_step``"""

    _fields_ = [
        ("rewards", C.c_void_p),
        ("bias", C.c_float),
        ("scaling", C.c_float),
        ("clip", C.c_float),
        ("norm", C.POINTER(NormParams)),
    ]


_p = C.c_void_p
_i64 = C.c_int64
_f = C.c_float
_i = C.c_int
_d = C.c_double

# name -> (restype, argtypes); must list every function of include/areal_amd.h
SIGNATURES = {
    "aa_version": (_i, []),
    "aa_layout": (C.c_uint64, []),
    "aa_status_string": (C.c_char_p, [_i]),
    "aa_logits_fwd": (_i, [_p, _i, _i64, _i64, _i64, _p, _f, _p, _p, _p, _p, _p, _p, _p]),
    "aa_logits_bwd": (_i, [_p, _i, _i64, _i64, _i64, _p, _f, _p, _p, _p, _p, _i64, _p, _p]),
    "aa_logits_ppo_fused": (
        _i,
        [_p, _i, _i64, _i64, _i64, _p, _f, _i64, _p, _p, _p, _p, C.POINTER(PpoParams), _p, _p,
         _p, _p, _p, _p, _p, _p, _p, _p, _p, _p],
    ),
    "aa_logits_ppo_step": (_i, [C.POINTER(PpoStep), _p, _i, _i64, _i64, _p, _f, _p, _p]),
    "aa_ppo_loss_step": (_i, [C.POINTER(PpoStep), _p, _i, _i, _p, _p]),
    "aa_lmhead_ppo_step": (_i, [C.POINTER(PpoStep), _p, _p, _i64, _i64, _p, _f, _p, _i, _p, _p, _i, _p, _i64, _p]),
    "aa_vocab_partials_combine": (_i, [_p, _p, _p, _i, _i64, _p, _p, _p, _p, _p]),
    "aa_logits_pairs_fwd": (_i, [_p, _i, _i64, _i64, _i64, _p, _p, _i64, _f, _p, _p, _p, _p, _p]),
    "aa_logits_pairs_scatter": (_i, [_p, _i, _i64, _i64, _i64, _p, _p, _i64, _p, _f, _p]),
    "aa_rejection_sampling": (_i, [_p, _p, _p, _i64, _p, _i64, _i, _i, _i, _i, _f, _f, _i, _p, _p, _p, _p]),
    "aa_count_nonzero_u8": (_i, [_p, _i64, _p, _p]),
    "aa_ppo_loss": (_i, [_p, _p, _p, _p, _p, _i64, _p, _i64, _i, C.POINTER(PpoParams), _p, _p, _p, _p, _p, _p]),
    "aa_masked_sum": (_i, [_p, _p, _i64, _p, _p, _p, _p]),
    "aa_ppo_stat_outputs": (_i, [_p, _p, _p, _p, _p, _p, _i64, _p, _p, _p, _p, _p, _p]),
    "aa_scale_inplace": (_i, [_p, _i, _i64, _p, _p]),
    "aa_scale_rows_inplace": (_i, [_p, _i, _i64, _i64, _i64, _p, _p]),
    "aa_lmhead_workspace_bytes": (_i64, [_i64, _i64, _i64]),
    "aa_lmhead_fwd_workspace_bytes": (_i64, [_i64, _i64, _i64]),
    "aa_lmhead_fwd_stats_workspace_bytes": (_i64, [_i64, _i64, _i64]),
    "aa_lmhead_prepare": (_i, []),
    "aa_lmhead_fwd": (_i, [_p, _p, _i64, _i64, _i64, _p, _f, _p, _p, _p, _p, _p, _p, _p, _i64, _p]),
    "aa_lmhead_chunk_tokens": (_i64, []),
    "aa_lmhead_fwd_static": (_i, [_p, _p, _i64, _i64, _i64, _p, _f, _p, _p, _p, _p, _p]),
    "aa_lmhead_fwd_static_scratch_bytes": (_i64, []),
    "aa_lmhead_fwd_static_max_vocab": (_i64, []),
    "aa_lmhead_bwd": (_i, [_p, _p, _i64, _i64, _i64, _p, _f, _p, _p, _p, _p, _p, _p, _p, _p, _i, _p, _i64, _p]),
    "aa_lmhead_carry_workspace_bytes": (_i64, [_i64, _i64, _i64]),
    "aa_lmhead_panel_pitch": (_i64, [_i64]),
    "aa_lmhead_fwd_carry": (_i, [_p, _p, _i64, _i64, _i64, _p, _f, _p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _p, _i64, _p]),
    "aa_lmhead_bwd_carry": (_i, [_p, _p, _i64, _i64, _i64, _p, _f, _p, _p, _p, _p, _p, _p, _i64, _p, _p, _i, _p, _i64, _p]),
    "aa_lmhead_ppo_fused": (
        _i,
        [_p, _p, _i64, _i64, _i64, _p, _f, _i64, _p, _p, _p, _p, C.POINTER(PpoParams), _p, _p, _p, _i,
         _p, _p, _p, _p, _p, _p, _p, _p, _p, _i, _p, _i64, _p],
    ),
    "aa_sapo_loss": (_i, [_p, _p, _p, _p, _i64, _p, _i64, _i, _f, _f, _p, _p, _p, _p, _p, _p]),
    "aa_critic_loss": (_i, [_p, _p, _p, _p, _i64, _f, _i, _p, _p, _p, _p, _p]),
    "aa_prox_logp_approx": (_i, [_p, _p, _p, _i64, _i, _i, _p, _p]),
    "aa_masked_normalization_scratch_bytes": (_i64, [_i64, _i64]),
    "aa_masked_normalization": (_i, [_p, _p, _i64, _i64, _i, _d, _p, _p, _i64, _p]),
    "aa_kl_estimate": (_i, [_p, _p, _i64, _i, _i, _p, _p]),
    "aa_overlong_penalty": (_i, [_p, _p, _i64, _i64, _i, _f, _i64, _p]),
    "aa_kd_terms": (_i, [_p, _p, _p, _p, _i64, _i, _p, _p, _p]),
    "aa_sft_sequence_stats": (_i, [_p, _p, _i64, _p, _i64, _p, _p, _p, _p, _p]),
    "aa_sft_loss": (_i, [_p, _p, _i64, _p, _i64, _p, _p, _p, _p, _p, _p, _p, _p, _p]),
    "aa_dpo_seq_sums": (_i, [_p, _p, _p, _p, _i64, _i64, _p, _p, _p, _p]),
    "aa_dpo_seq_sums_bwd": (_i, [_p, _p, _p, _p, _i64, _i64, _p, _p]),
    "aa_dpo_preference_loss": (_i, [_p, _i64, _d, _i, _p, _p, _p]),
    "aa_dpo_pair_loss": (_i, [_p, _p, _p, _p, _i64, _d, _i, _p, _p, _p, _p, _p, _p, _p, _p]),
    "aa_logging_stats_scratch_bytes": (_i64, [_i64]),
    "aa_logging_stats": (_i, [_p, _p, _p, _p, _p, _i64, _i, _i, _i, _p, _p, _i64, _p]),
    "aa_logging_stats_table": (_i, [_p, _p, _p, _p, _p, _i64, _i, _i, _i, _p, _p, _i64, _p, _p]),
    "aa_moments_table_scratch_bytes": (_i64, [_i, _i64]),
    "aa_moments_table": (_i, [C.POINTER(_p), C.POINTER(_p), C.c_uint32, _i, _i64, _p, _p, _i64, _p, _p]),
    "aa_rw_pair_loss": (_i, [_p, _i64, _p, _i64, _p, _p, _p, _p, _p, _p, _p, _p]),
    "aa_m2po_workspace_bytes": (_i64, [_i64]),
    "aa_m2po_mask": (_i, [_p, _p, _p, _i64, _f, _p, _p, _p, _i64, _p]),
    "aa_reward_scores": (_i, [_p, _i64, _f, _f, _f, C.POINTER(NormParams), _p, _p]),
    "aa_advantages_scratch_bytes": (_i64, [_i64]),
    "aa_advantages": (_i, [C.POINTER(AdvantageStep), _p]),
    "aa_advantages_scored": (_i, [C.POINTER(AdvantageStep), C.POINTER(ScoreStep), _p]),
    "aa_kl_rewards": (_i, [_p, _p, _p, _p, _p, _i64, _i64, _f, _i, _i, _p, _p, _p]),
    "aa_gae": (_i, [_p, _p, _p, _p, _i64, _i64, _f, _f, _p, _p, _p]),
    "aa_normalize_scratch_bytes": (_i64, [_i64, _i64, _i64]),
    "aa_normalize": (_i, [_p, _p, _i64, _i64, C.POINTER(NormParams), _p, _p, _i64, _p]),
    "aa_masked_moments": (_i, [C.POINTER(C.c_void_p), _i, _p, _i64, _p, _p]),
    "aa_segment_copy": (_i, [_p, _p, _i64, _p, _p, _p, _i64, _i64, _p]),
    "aa_copy_bytes": (_i, [_p, _p, _i64, _p]),
    "aa_mfma_only_loop": (_i, [_i, _i, _i, _i, _p, _p]),
    "aa_hbm_stream_probe": (_i, [_i, _i, _p, _p, _i64, _i, _p]),
}

_SHARED_STRUCTS = (PpoParams, RsParams, LossScale, PpoStep, NormParams, AdvantageStep, ScoreStep)


def _layout(structs=_SHARED_STRUCTS) -> int:
    """The number of ``csrc/layout.h`` for the structs as they are written down here."""
    h = 0xCBF29CE484222325

    def mix(name: str, size: int, place: int) -> None:
        nonlocal h
        for n in (*name.encode(), size, place):
            h = (h ^ n) * 0x100000001B3 % 2**64

    for struct in structs:
        mix(struct.__doc__.strip("`"), C.sizeof(struct), 0)
        for name, *_ in struct._fields_:
            field = getattr(struct, name)
            mix(name, field.size, field.offset)
    return h


def _check_layout(path: Path, found: int | None) -> None:
    """Three binaries fill in and read the same structs; one of another header would write past them without a word."""
    if found != _layout():
        raise NativeLibraryError(f"{path} was built from another include/areal_amd.h than this package: build both libraries "
                                 "with `python -m areal_amd.build`")


_lib = None
_lock = threading.Lock()


def load() -> C.CDLL:
    """Load the shared library once and bind the signatures."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not LIB_PATH.exists():
            raise NativeLibraryError(
                f"{LIB_PATH} not found: build it with `python -m areal_amd.build` "
                "(there is no CPU or PyTorch fallback for these ops)"
            )
        try:
            lib = C.CDLL(str(LIB_PATH))
        except OSError as e:  # missing ROCm runtime etc.
            raise NativeLibraryError(f"cannot load {LIB_PATH}: {e}") from e
        for name, (res, args) in SIGNATURES.items():
            try:
                fn = getattr(lib, name)
            except AttributeError as e:
                raise NativeLibraryError(f"{LIB_PATH} does not export {name}") from e
            fn.restype = res
            fn.argtypes = args
        _check_layout(LIB_PATH, lib.aa_layout())
        _lib = lib
    return _lib


def host():
    """The native host side of the steps (``csrc/host.cpp``), behind the library that it calls."""
    if _host is None:
        load()
        _load_host()
    return _host


_host = None


def _load_host() -> None:
    global _host
    try:
        from . import _host as module
    except ImportError as e:
        raise NativeLibraryError(f"cannot load {HOST_PATH}: build it with `python -m areal_amd.build` ({e})") from e
    _check_layout(HOST_PATH, getattr(module, "layout", None))
    _host = module


def check(status: int, what: str) -> None:
    if status != AA_OK:
        msg = load().aa_status_string(status).decode()
        raise NativeLibraryError(f"{what} failed: {msg} (status {status})")
