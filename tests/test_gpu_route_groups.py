"""Grouped routing at the edges of its key layout, bit for bit against the oracle: more
experts than one key a lane and than four, groups of one expert (no second best), groups
that do not divide the wave."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import oracle_py as O
from hearth_amd import _native, container
from hearth_amd.engine import Engine

pytestmark = pytest.mark.gpu

SMALL = dataclasses.replace(container.TINY_DSV3_GQA, n_layers=2, d_model=256, expert_ffn=64, shared_ffn=64, dense_ffn=64,
                            vocab=512)


@pytest.mark.parametrize("experts,groups,keep,k", [(16, 16, 4, 4), (48, 3, 2, 5), (256, 8, 4, 8), (320, 10, 3, 8)])
def test_routes(tmp_path, experts, groups, keep, k):
    O.gpu_numerics()
    shape = dataclasses.replace(SMALL, n_experts=experts, n_group=groups, topk_group=keep, top_k=k)
    path = container.make_tiny(tmp_path / "m.hearth", _native.quantize, seed=5, shape=shape)
    toks = container.uniform_ints(9, 21, shape.vocab).astype(np.int32)
    want, routes = O.Model(path, cap=32).eval(toks, routes=True)
    with Engine(path, max_seq=32) as e:
        tr = tmp_path / "r.hrtr"
        e.trace_start(tr)
        got = e.eval(toks, all_logits=True)
        e.trace_stop()
    ids = np.frombuffer(tr.read_bytes()[24:], dtype="<u2").reshape(routes.shape).astype(np.int32)
    assert np.array_equal(ids, routes)
    assert np.array_equal(got.view(np.uint32), np.asarray(want).view(np.uint32))
