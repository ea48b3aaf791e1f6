"""Which score and value kernels a call takes. The value kernel (the summing waves of
k_attn.hip, or k_values_many with two or four column tiles) is decided by expected times, the
score kernel (k_scores_many or the others) by rows and tokens: shapes on both sides of the
lines, bit for bit against the oracle. Single heads, groups of 4 and 8, 64 / 128 / 192 columns,
latent rows of 256 and 512 and of 16 and 48 heads; chains and trees of few and of many tokens,
from empty and after a context; and the device loop's padded steps of 21 tokens. The outputs
have no tolerance: every sum's order is fixed."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import oracle_py as O
from hearth_amd import _native, container
from hearth_amd.engine import Engine
from test_gpu_spec_loop import _prompt, _same

pytestmark = pytest.mark.gpu

BASE = dataclasses.replace(container.TINY, n_layers=2, d_model=256, n_experts=4, top_k=2, expert_ffn=128, vocab=512)
SINGLE = dataclasses.replace(BASE, n_heads=32, n_kv_heads=32, head_dim=128)
H64 = dataclasses.replace(BASE, n_heads=32, n_kv_heads=8, head_dim=64)
H192 = dataclasses.replace(BASE, n_heads=32, n_kv_heads=4, head_dim=192)
LATENT256 = dataclasses.replace(container.TINY_MLA_NOQ, d_model=256, n_experts=4, top_k=2, expert_ffn=128, vocab=512,
                                n_heads=32, n_kv_heads=32)
LATENT512 = dataclasses.replace(container.TINY_DSV3, n_layers=2, d_model=256, n_experts=8, n_group=2, topk_group=1, top_k=2,
                                expert_ffn=128, shared_ffn=128, dense_ffn=128, vocab=512, n_heads=48, n_kv_heads=48,
                                kv_lora=512)
LATENT16 = dataclasses.replace(LATENT512, n_heads=16, n_kv_heads=16)
ROPE32 = dataclasses.replace(LATENT256, n_heads=16, n_kv_heads=16, kv_lora=512)   # the RoPE term a pass of its own


def _bits(x):
    return np.ascontiguousarray(x, dtype=np.float32).view(np.uint32)


# chains one after another, then trees (each from the chains' end). Four column tiles: LATENT512
# from 50 tokens on; two: SINGLE from 17 on, the 200 tokens of H64, 500 of H192 and 129 of
# LATENT256; the summing waves: the others
@pytest.mark.parametrize("shape,lens,trees", [(SINGLE, (17, 33, 64, 2, 130), (21, 70)), (H64, (100, 40, 200, 9), (33, 129)),
                                              (H192, (31, 500, 20), (100,)), (LATENT256, (24, 48, 129, 3), (40, 90)),
                                              (LATENT512, (13, 260, 50, 18), (21, 64)), (LATENT16, (1, 2, 3, 40, 1), (2, 3)),
                                              (ROPE32, (1, 3, 20, 1), (4,))],
                         ids=["single", "h64", "h192", "latent256", "latent512", "latent16", "rope32"])
def test_value_sums(tmp_path, shape, lens, trees):
    O.gpu_numerics()
    path = container.make_tiny(tmp_path / "m.hearth", _native.quantize, seed=23, shape=shape)
    cap = sum(lens) + max(trees)
    toks = container.uniform_ints(9, cap, shape.vocab).astype(np.int32)
    m = O.Model(path, cap=cap, threads=8)
    with Engine(path, max_seq=cap, max_batch=512) as e:
        at = 0
        for n in lens:
            got, want = e.eval(toks[at:at + n], all_logits=True), m.eval(toks[at:at + n])
            assert np.array_equal(_bits(got), _bits(want)), f"{n} tokens at {at}"
            at += n
        for n in trees:
            back = 1 + container.uniform_ints(n, n, 5).astype(np.int64)
            parent = np.array([-1] + [max(0, i - int(back[i])) for i in range(1, n)], dtype=np.int32)
            got, want = e.verify_tree(toks[at:at + n], parent), m.eval_tree(toks[at:at + n], parent)
            assert np.array_equal(_bits(got), _bits(want)), f"tree of {n} at {at}"


def test_padded_steps_of_the_device_loop(tmp_path):
    """21-token steps with fewer live tokens, through the many-row kernels"""
    path = container.make_tiny(tmp_path / "m.hearth", _native.quantize, seed=23, shape=SINGLE)
    with Engine(path, max_seq=256) as e:
        _same(e, _prompt(e.vocab_size), 48, (), "ngram", 20, 2)
