"""The chunked int8 products (k_mm.hip: more than 16 tokens, and experts whose token blocks
do not fit the few-token kernel's LDS) at the edges of their tiles, bit for bit against the
oracle: 16- and 32-token tiles, 64-row groups, K chunks of 8 blocks (one block, one whole
chunk, a chunk and one block), odd block counts (a padding block follows), slots of 0, 1 and
many passes. The outputs have no tolerance: the fold's order is fixed."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import oracle_py as O
from hearth_amd import _native, container
from hearth_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [3, 4])
@pytest.mark.parametrize("rows,cols,T", [(16, 64, 17), (65, 512, 32), (130, 576, 33), (64, 1088, 48), (8200, 128, 130)])
def test_dense_products(dtype, rows, cols, T):
    """8200 rows x 130 tokens take two token tiles a workgroup, the others one"""
    rng = np.random.default_rng(rows + cols + T)
    q = _native.quantize(dtype, rng.standard_normal((rows, cols)).astype(np.float32))
    X = rng.standard_normal((T, cols)).astype(np.float32) * np.exp(rng.normal(0, 4, (T, 1))).astype(np.float32)
    assert np.array_equal(_native.matmul(dtype, q, rows, cols, X).view(np.uint32),
                          O.matmul(dtype, q, rows, cols, X).view(np.uint32))


# 9 blocks of K for gate/up, 3 for down (both odd); few experts, so slots of several passes
MOE = dataclasses.replace(container.TINY, n_layers=2, d_model=576, n_experts=6, top_k=2, expert_ffn=192, vocab=512)
# a gate/up input too wide for the few-token kernel: the chunked one from one token on
WIDE = dataclasses.replace(container.TINY, n_layers=1, d_model=4160, n_experts=8, top_k=2, expert_ffn=128, vocab=256)
MLA = dataclasses.replace(container.TINY_DSV3, n_layers=2)


@pytest.mark.parametrize("shape,lens", [(MOE, (17, 40, 130)), (WIDE, (1, 9, 16, 33)), (MLA, (17, 33, 70))],
                         ids=["odd_blocks", "wide", "per_head"])
def test_routed_and_per_head_products(tmp_path, shape, lens):
    O.gpu_numerics()
    path = container.make_tiny(tmp_path / "m.hearth", _native.quantize, seed=11, shape=shape)
    toks = container.uniform_ints(5, sum(lens), shape.vocab).astype(np.int32)
    m = O.Model(path, cap=sum(lens))
    want = np.asarray(m.eval(toks))
    with Engine(path, max_seq=sum(lens), max_batch=512) as e:
        at = 0
        for n in lens:
            got = e.eval(toks[at:at + n], all_logits=True)
            assert np.array_equal(got.view(np.uint32), want[at:at + n].view(np.uint32)), f"{n} tokens at {at}"
            at += n
