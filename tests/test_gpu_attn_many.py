"""The attention of many rows (k_attn_many.hip) at the edges of its tiles, bit for bit
against the oracle: 64-row workgroups and 16-row tiles of one or several tokens, 16-slot
score tiles, 32-slot value tiles, chains from empty (rows of very different lengths) and
after a context, trees whose paths leave out most of the step's slots, groups of 1, 5 and 8
heads, 64 / 128 / 256 columns, and the latent attention's 512 columns with the RoPE term.
The outputs have no tolerance: the order of every sum is fixed."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import oracle_py as O
from hearth_amd import _native, container
from hearth_amd.engine import Engine

pytestmark = pytest.mark.gpu

ONE = dataclasses.replace(container.TINY, n_layers=2, d_model=256, n_experts=4, top_k=2, expert_ffn=128, vocab=512)
G8 = dataclasses.replace(ONE, n_heads=64, n_kv_heads=8, head_dim=128)
G5 = dataclasses.replace(ONE, n_heads=20, n_kv_heads=4, head_dim=64)
G1 = dataclasses.replace(ONE, n_heads=32, n_kv_heads=32, head_dim=256)
LATENT = dataclasses.replace(container.TINY_DSV3, n_layers=2, d_model=256, n_experts=8, n_group=2, topk_group=1, top_k=2,
                             expert_ffn=128, shared_ffn=128, dense_ffn=128, vocab=512, n_heads=64, n_kv_heads=64,
                             kv_lora=512)


def _parents(n, seed):
    back = 1 + container.uniform_ints(seed, n, 9).astype(np.int64)
    return np.array([-1] + [max(0, i - int(back[i])) for i in range(1, n)], dtype=np.int32)


# chain lengths one after another, then the nodes of a tree after them
@pytest.mark.parametrize("shape,lens,tree", [(G8, (300, 1, 259), 257), (G8, (33,), 9), (G5, (13, 30, 64), 77),
                                             (G1, (260, 63), 258), (LATENT, (65, 9, 1), 70)],
                         ids=["group8", "group8_few", "group5", "group1", "latent"])
def test_chains_and_trees(tmp_path, shape, lens, tree):
    O.gpu_numerics()
    path = container.make_tiny(tmp_path / "m.hearth", _native.quantize, seed=13, shape=shape)
    toks = container.uniform_ints(6, sum(lens) + tree, shape.vocab).astype(np.int32)
    parent = _parents(tree, 8)
    m = O.Model(path, cap=sum(lens) + tree)
    with Engine(path, max_seq=sum(lens) + tree, max_batch=512) as e:
        at = 0
        for n in lens:
            got, want = e.eval(toks[at:at + n], all_logits=True), np.asarray(m.eval(toks[at:at + n]))
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"{n} tokens at {at}"
            at += n
        got, want = e.verify_tree(toks[at:], parent), np.asarray(m.eval_tree(toks[at:], parent))
        assert np.array_equal(np.asarray(got).view(np.uint32), want.view(np.uint32)), f"tree of {tree} at {at}"
