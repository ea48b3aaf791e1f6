"""The expert products of few tokens where the slots are of both dtypes or K is too wide for
the resident kernel, bit for bit against the oracle: Q4 and Q8 experts in one layer (a launch
per dtype up to 4 tokens, the chunked kernels from 5 on), gate/up of K = 4160 and down of K =
4224 (split over K up to 4 tokens, chunked from 5 on), odd block counts. The outputs have no
tolerance: the fold's order is fixed."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import oracle_py as O
from hearth_amd import _native, container
from hearth_amd.engine import Engine

pytestmark = pytest.mark.gpu

NARROW = dataclasses.replace(container.TINY, n_layers=2, d_model=576, n_experts=6, top_k=2, expert_ffn=320, vocab=512)
BLOCKS = dataclasses.replace(NARROW, d_model=512, expert_ffn=256)     # gate/up quantizes its rows
WIDE_IN = dataclasses.replace(container.TINY, n_layers=1, d_model=4160, n_experts=4, top_k=2, expert_ffn=192, vocab=256)
WIDE_OUT = dataclasses.replace(container.TINY, n_layers=1, d_model=320, n_experts=4, top_k=2, expert_ffn=4224, vocab=256)


@pytest.mark.parametrize("q8", ["odd", "all"])
@pytest.mark.parametrize("shape", [NARROW, BLOCKS, WIDE_IN, WIDE_OUT], ids=["narrow", "blocks", "wide_in", "wide_out"])
def test_few_token_experts(tmp_path, monkeypatch, shape, q8):
    """q8: which experts' slabs are Q8 (the others Q4)"""
    add = container.ContainerWriter.add_expert

    def add_some_q8(self, layer, e, dtype, slab):
        if q8 == "all" or e % 2:
            D, F = shape.d_model, shape.expert_ffn
            nb, *offs = container.slab_layout(container.Q8, D, F)
            b = bytearray(nb)
            for i, (off, (rows, cols)) in enumerate(zip(offs, ((F, D), (F, D), (D, F)))):
                w = container.normal(1000 * layer + 10 * e + i, rows * cols, 0.02).reshape(rows, cols)
                w = _native.quantize(container.Q8, w)
                b[off:off + len(w)] = w
            dtype, slab = container.Q8, bytes(b)
        add(self, layer, e, dtype, slab)

    monkeypatch.setattr(container.ContainerWriter, "add_expert", add_some_q8)
    O.gpu_numerics()
    path = container.make_tiny(tmp_path / "m.hearth", _native.quantize, seed=17, shape=shape)
    lens = (1, 2, 3, 4, 5, 16, 17)
    toks = container.uniform_ints(7, sum(lens), shape.vocab).astype(np.int32)
    want = np.asarray(O.Model(path, cap=sum(lens)).eval(toks))
    with Engine(path, max_seq=sum(lens)) as e:
        at = 0
        for n in lens:
            got = e.eval(toks[at:at + n], all_logits=True)
            assert np.array_equal(got.view(np.uint32), want[at:at + n].view(np.uint32)), f"{n} tokens at {at}"
            at += n
