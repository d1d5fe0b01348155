"""ctypes binding of liblfm25_hip.so (the C ABI declared in include/lfm25_hip.h).

By default torch is imported first so the library binds to the HIP runtime
torch already loaded (both carry the soname libamdhip64.so.7); device pointers
from torch tensors and the library's kernels then share one runtime and one
context. Torch-free callers (hip.py, bench.py) load it on its own.

There is no fallback: if the library is missing, every operation raises.
"""

from __future__ import annotations

import ctypes
from pathlib import Path

HERE = Path(__file__).resolve().parent
LIBRARY_PATH = HERE / "liblfm25_hip.so"

LFM25_OK, LFM25_EINVAL, LFM25_EDEVICE = 0, 1, 2
EXEC_STAGED, EXEC_PERSISTENT = 0, 1
CTL_POSITION, CTL_TOKEN, CTL_STATUS = 0, 1, 2

_p = ctypes.c_void_p
_i32 = ctypes.c_int32
_i64p = ctypes.POINTER(ctypes.c_int64)
_size = ctypes.c_size_t


class Decoder(ctypes.Structure):
    """lfm25_decoder (include/lfm25_hip.h)."""

    _fields_ = [
        ("weights", _p), ("embedding", _p), ("rope", _p), ("conv_state", _p),
        ("key_cache", _p), ("value_cache", _p), ("workspace", _p),
        ("capacity", _i32), ("vocab", _i32),
    ]


class Batch(ctypes.Structure):
    """lfm25_batch (include/lfm25_hip.h)."""

    _fields_ = [
        ("weights", _p), ("embedding", _p), ("rope", _p), ("conv_state", _p),
        ("key_cache", _p), ("value_cache", _p), ("workspace", _p),
        ("sequences", _i32), ("capacity", _i32), ("vocab", _i32),
    ]


class W8Model(ctypes.Structure):
    """lfm25_w8_model (include/lfm25_hip.h): the w8g32 projections and table."""

    _fields_ = [("layers", _p), ("table", _p), ("table_scales", _p)]


BATCH_MAX_ROWS = 64
PROMPT_MAX_ROWS = 4096
LAYER_CONV, LAYER_ATTN = 0, 1


class Layer(ctypes.Structure):
    """lfm25_layer (include/lfm25_hip.h): one decoder layer's tensors."""

    _fields_ = [
        ("kind", _i32), ("op_norm", _p), ("mixer", _p), ("conv_weight", _p), ("conv_state_in", _p),
        ("conv_state_out", _p), ("q_norm", _p), ("k_norm", _p), ("key_cache", _p), ("value_cache", _p),
        ("rope", _p), ("capacity", _i32), ("out", _p), ("ffn_norm", _p), ("w1", _p), ("w3", _p), ("w2", _p),
    ]


class PkLayer(ctypes.Structure):
    """lfm25_pk_layer (include/lfm25_hip.h)."""

    _fields_ = [(n, _p) for n in (
        "ln", "ff1_w1", "ff1_w2", "qkv", "qkv_bias", "att_delta", "pos", "out", "pw1", "dw", "dw_b", "pw2",
        "ff2_w1", "ff2_w2")]

# name -> (restype, argtypes)
SIGNATURES = {
    "lfm25_version": (ctypes.c_int, []),
    "lfm25_last_error": (ctypes.c_char_p, []),
    "lfm25_init": (ctypes.c_int, []),
    "lfm25_rms_norm": (ctypes.c_int, [_p, _p, _p, _i32, _p]),
    "lfm25_bf16_bf16_gemv": (ctypes.c_int, [_p, _p, _p, _i32, _i32, _p]),
    "lfm25_bf16_f32_gemv": (ctypes.c_int, [_p, _p, _p, _i32, _i32, _p]),
    "lfm25_norm_bf16_gemv": (ctypes.c_int, [_p, _p, _p, _i32, _i32, _p]),
    "lfm25_w8_gemv": (ctypes.c_int, [_p, _p, _p, _p, _i32, _i32, _i32, _p]),
    "lfm25_f32_to_bf16": (ctypes.c_int, [_p, _p, _i32, _p]),
    "lfm25_bf16_add": (ctypes.c_int, [_p, _p, _p, _i32, _p]),
    "lfm25_silu_gate": (ctypes.c_int, [_p, _p, _p, _i32, _p]),
    "lfm25_conv_gate": (ctypes.c_int, [_p, _p, _p, _p, _p]),
    "lfm25_conv_gate_packed_state": (ctypes.c_int, [_p, _p, _p, _p, _p]),
    "lfm25_attention_norm_rope": (ctypes.c_int, [_p, _p, _p]),
    "lfm25_attention_context": (ctypes.c_int, [_p, _p, _p, _i32, _p]),
    "lfm25_attention_append_cache": (ctypes.c_int, [_p, _p, _p, _i32, _p]),
    "lfm25_layer_workspace_bytes": (_size, []),
    "lfm25_recurrent_block": (ctypes.c_int, [_p, _p, _p, _p, _p, _p, _p, _p]),
    "lfm25_attention_prefix": (ctypes.c_int, [_p, _p, _p, _p, _i32, _p]),
    "lfm25_attention_context_cache": (ctypes.c_int, [_p, _p, _p, _p, _i32, _p, _p]),
    "lfm25_attention_tail": (ctypes.c_int, [_p, _p, _p, _p, _p]),
    "lfm25_attention_first_context": (ctypes.c_int, [_p, _p, _p, _p]),
    "lfm25_attention_fixed": (ctypes.c_int, [_p, _p, _p, _p, _i32, _i32, _p, _p]),
    "lfm25_pack_block_input": (ctypes.c_int, [_p, _p, _p, _p]),
    "lfm25_pack_conv": (ctypes.c_int, [_p, _p, _p, _p]),
    "lfm25_pack_attention_tail": (ctypes.c_int, [_p, _p, _p, _p]),
    "lfm25_concat_hidden_pair": (ctypes.c_int, [_p, _p, _p, _p]),
    "lfm25_split_hidden_pair": (ctypes.c_int, [_p, _p, _p, _p]),
    "lfm25_pack_recurrent_pair": (ctypes.c_int, [_p, _p, _p, _p]),
    "lfm25_bf16_f32_matmul": (ctypes.c_int, [_p, _p, _p, _i32, _i32, _i32, _p]),
    "lfm25_argmax_workspace_bytes": (_size, [_i32]),
    "lfm25_argmax": (ctypes.c_int, [_p, _i32, _p, _p, _p]),
    "lfm25_fused_vocab": (ctypes.c_int, [_p, _p, _p, _p, _p, _i32, _p, _p]),
    "lfm25_fused_vocab_static": (ctypes.c_int, [_p, _p, _p, _p, _p, _i32, _p]),
    "lfm25_embedding_gather": (ctypes.c_int, [_p, _p, _p, _i32, _p, _p]),
    "lfm25_weights_elems": (_size, []),
    "lfm25_weights_offsets": (_i32, [_i64p, _i32]),
    "lfm25_decoder_workspace_bytes": (_size, []),
    "lfm25_decode_layer": (ctypes.c_int, [ctypes.POINTER(Layer), _p, _p, _i32, _p, _p]),
    "lfm25_decoder_reset": (ctypes.c_int, [ctypes.POINTER(Decoder), _p]),
    "lfm25_decode": (ctypes.c_int, [ctypes.POINTER(Decoder), _p, _i32, _i32, _p, _i32, _p]),
    "lfm25_decode_exchange": (_i32, []),
    "lfm25_w8_layers_bytes": (_size, []),
    "lfm25_w8_layers_offsets": (_i32, [_i64p, _i32]),
    "lfm25_decode_w8": (ctypes.c_int, [ctypes.POINTER(Decoder), ctypes.POINTER(W8Model), _p, _i32, _i32, _p, _p]),
    "lfm25_batch_workspace_bytes": (_size, []),
    "lfm25_batch_pass": (ctypes.c_int, [ctypes.POINTER(Batch), _p, _i32, _i32, _p, _p, _p]),
    "lfm25_prompt_workspace_bytes": (_size, [_i32]),
    "lfm25_prompt_pass": (ctypes.c_int, [ctypes.POINTER(Batch), _p, _p, _i32, _p, _p, _p, _p]),
    "lfm25_batch_decode": (ctypes.c_int, [ctypes.POINTER(Batch), _p, _p, _i32, _p, _p]),
    "lfm25_batch_decode_hidden": (ctypes.c_int, [ctypes.POINTER(Batch), _p, _p, _i32, _p, _p, _p]),
    "lfm25_batch_linear": (ctypes.c_int, [_p, _p, _p, _i32, _i32, _i32, _p]),
    "lfm25_pk_gemm": (ctypes.c_int, [_p, _i32, _p, _i32, _p, _p, _i32, _i32, _i32, _i32, _i32, _i32, _p, _p]),
    "lfm25_pk_layer_norm": (ctypes.c_int, [_p, _p, ctypes.c_float, _p, _p, _p, _p, _i32, _p, _i32, _p]),
    "lfm25_pk_attention": (ctypes.c_int, [_p, _p, _p, _p, _i32, _i32, _i32, _p]),
    "lfm25_pk_conv": (ctypes.c_int, [_p, _p, _p, _p, _i32, _i32, _i32, _p]),
    "lfm25_pk_workspace_bytes": (_size, [_i32, _i32]),
    "lfm25_pk_encoder": (ctypes.c_int, [ctypes.POINTER(PkLayer), _i32, _p, _i32, _i32, _i32, _p, _p]),
}

_lib = None


def load(bind_torch: bool = True) -> ctypes.CDLL:
    """Load (once) and return the library; raises if it has not been built.

    With bind_torch (the default) torch is imported first so that tensors and
    the library share torch's HIP runtime; torch-free callers (hip.py) pass
    False and the library loads libamdhip64.so.7 through its runpath."""
    global _lib
    if _lib is not None:
        return _lib
    if bind_torch:
        try:
            import torch  # noqa: F401  (binds the HIP runtime torch ships)
        except ImportError:
            pass
    if not LIBRARY_PATH.exists():
        raise RuntimeError(
            f"{LIBRARY_PATH} is missing: build the gfx950 HIP library first "
            "(python ryzenai-npu-lab_amd/build.py)")
    lib = ctypes.CDLL(str(LIBRARY_PATH))
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    _lib = lib
    return lib


def check(rc: int, what: str) -> None:
    if rc == LFM25_OK:
        return
    msg = (load().lfm25_last_error() or b"").decode(errors="replace")
    if rc == LFM25_EINVAL:
        raise ValueError(f"{what}: {msg}")
    raise RuntimeError(f"{what}: {msg}")


_functions = {}  # name -> the library's function, from its first call on


def call(name: str, *args) -> None:
    fn = _functions.get(name)
    if fn is None:
        fn = _functions[name] = getattr(load(), name)
    rc = fn(*args)
    if rc != LFM25_OK:
        check(rc, name)
