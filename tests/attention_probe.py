"""Weights that show one stage of the prompt pass alone (not collected by
pytest). Token t's embedding is 32 in dimension 512 + t and 0 elsewhere, so
its RMSNorm is the same vector and every projection of it is one column, exact
whatever the order of the sums. All layers but the chosen ones are zero. What
the stage leaves in dimensions 0 .. 511 of the residual stream is read back
from the values of a later attention layer, whose v_proj picks those
dimensions: at values below 2^-5 the norm's scale there stays within 2^-9 of
1, so the BF16 values come through unchanged."""

from __future__ import annotations

import numpy as np

from oracle import lfm25 as O

HIDDEN, HEADS, KV_HEADS, DIM = 1024, 16, 8, 64
PICK = 512          # residual dimensions that are read back
TOKENS = 256


def bits(x) -> np.ndarray:
    return O.bf16_bits(np.asarray(x, np.float32))


def bf(x) -> np.ndarray:
    return O.f32(bits(x))


def checkpoint(lab) -> dict:
    ck = {}
    for name, shape in lab.weights.all_tensors(TOKENS):
        norm = name.endswith(lab.weights.NORMS) or name == "model.embedding_norm.weight"
        ck[name] = np.full(shape, 0x3F80 if norm else 0, np.uint16)
    for t in range(TOKENS):
        ck["model.embed_tokens.weight"][t, 512 + t] = 0x4200  # 32
    return ck


def columns(rows: np.ndarray) -> np.ndarray:
    """The weight [n, 1024] that gives token t the projection rows[t] (n values)."""
    w = np.zeros((rows.shape[1], HIDDEN), np.uint16)
    w[:, 512:512 + len(rows)] = bits(rows / 32).T
    return w


def read_back(ck: dict, layer: int) -> None:
    """Attention layer `layer` keeps dimensions 0 .. 511 as its values."""
    w = np.zeros((KV_HEADS * DIM, HIDDEN), np.uint16)
    w[np.arange(PICK), np.arange(PICK)] = bits(1.0)
    ck[f"model.layers.{layer}.self_attn.v_proj.weight"] = w


def picked() -> np.ndarray:
    """Context entries that out_proj puts into dimensions 0 .. 511: every
    other dimension of every head."""
    return np.arange(0, HEADS * DIM, 2)


def attention_checkpoint(lab, q, k, v, q_gamma, k_gamma) -> dict:
    """q [T, 16, 64], k, v [T, 8, 64] per token id through the attention of
    layer 2 (attention layer 0), read back from layer 4 (attention layer 1)."""
    ck = checkpoint(lab)
    p = "model.layers.2.self_attn."
    for name, x in (("q", q), ("k", k), ("v", v)):
        ck[p + name + "_proj.weight"] = columns(x.reshape(len(x), -1))
    ck[p + "q_layernorm.weight"], ck[p + "k_layernorm.weight"] = bits(q_gamma), bits(k_gamma)
    out = np.zeros((HIDDEN, HIDDEN), np.uint16)
    out[np.arange(PICK), picked()] = bits(1.0)
    ck[p + "out_proj.weight"] = out
    read_back(ck, 4)
    return ck


def norm_rope(x, gamma, positions) -> np.ndarray:
    """QK norm and RoPE of x [P, heads, 64] at `positions`."""
    cos, sin = O.rope_table(positions)
    return np.stack([O.norm_rope(x[i], bf(gamma), cos[i], sin[i]) for i in range(len(x))])
