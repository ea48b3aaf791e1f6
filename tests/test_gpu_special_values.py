"""Products at the ends of the float range through the attention's matrix-unit kernels
(k_scores_many, k_values_many, k_mla_qlat): a v_mfma with a zero accumulator has to give what
one multiplication gives, subnormals kept, infinities and NaN as they come, and nothing of a
slot that a row leaves out. Prefill, tree and single tokens, so that the kernels of few rows
take part, bit for bit against the oracle (the subnormal models) or against each other."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

import oracle_py as O
from hearth_amd import _native, container
from hearth_amd.engine import Engine

GQA = dataclasses.replace(container.TINY, n_layers=1, d_model=256, n_heads=32, n_kv_heads=32, head_dim=128, n_experts=4,
                          top_k=2, expert_ffn=128, vocab=512, qkv_bias=1)
LATENT = dataclasses.replace(container.TINY_DSV3, n_layers=1, n_dense=0, d_model=256, n_experts=8, n_group=2, topk_group=1,
                             top_k=2, expert_ffn=128, shared_ffn=128, vocab=512, n_heads=32, n_kv_heads=32, kv_lora=512,
                             nope=192)


def _model(monkeypatch, path, shape, tensors, **meta):
    """make_tiny with `tensors` (name in layer 0, or global -> f(old float32 values); "zeros" for
    a quantized matrix) and metadata keys replaced"""
    add, old_meta = container.ContainerWriter.add, container._meta

    def patched(self, name, dtype, shp, data):
        f = tensors.get(name.removeprefix("blk.0."))
        if f == "zeros":
            data = _native.quantize(dtype, np.zeros(shp, dtype=np.float32))
        elif f is not None:
            data = np.asarray(f(np.frombuffer(data, dtype=np.float32)), dtype=np.float32).tobytes()
        add(self, name, dtype, shp, data)

    with monkeypatch.context() as mp:
        mp.setattr(container.ContainerWriter, "add", patched)
        mp.setattr(container, "_meta", lambda s, src: {**old_meta(s, src), **meta})
        return container.make_tiny(path, _native.quantize, seed=29, shape=shape)


def _v_bias(old):
    """values whose products with a probability of 1 / 100 are subnormal, zeros of both signs"""
    u = container.uniforms(5, old.size) * 2 - 1
    v = (6e-37 * u).astype(np.float32)
    v[::17], v[1::17], v[2::17] = 0.0, -0.0, 1e-44
    return v


def _with(index, value):
    def f(old):
        new = old.copy()
        new[index] = value
        return new
    return f


def _scaled(s):
    return lambda old: old * np.float32(s)


# hidden rows of 1e-39 to 1e-36, brought to 1 by the norms; the experts' input is zero, so that
# the attention's subnormal-sized output is what the logits show
SUBNORMAL_GQA = (GQA, dict(attn_norm=_scaled(1e36), ffn_norm=_scaled(0), out_norm=_scaled(1e36), attn_q_norm=_scaled(1e-20),
                           attn_k_norm=_scaled(1e-19), attn_v="zeros", attn_v_bias=_v_bias), dict(attn_scale=2e38, emb_scale=1e-37))
# absorbed queries from products of 1e-39
SUBNORMAL_LATENT = (LATENT, dict(attn_q_a_norm=_scaled(3e-37)), dict(attn_scale=3e36))
MODELS = {"subnormal": SUBNORMAL_GQA, "subnormal_latent": SUBNORMAL_LATENT}
# value columns that overflow, are infinite or NaN, score terms that overflow: what a norm or
# a quantized block makes of them hides them from the logits, so the attention's own output is read
UNBOUNDED = {
    "overflow_v": dict(attn_v_bias=_with(slice(3, None, 64), np.finfo(np.float32).max)),
    "inf_v": dict(attn_v_bias=_with([5, 200], [np.inf, -np.inf])),
    "nan_v": dict(attn_v_bias=_with(130, np.nan)),
    "inf_scores": dict(attn_q_norm=_with(9, 1e25), attn_k_norm=_with(9, 2e13)),
}
LENS, TREE = (1, 1, 40, 100, 1), 70


def _inputs(shape):
    toks = container.uniform_ints(3, sum(LENS) + TREE, shape.vocab).astype(np.int32)
    back = 1 + container.uniform_ints(4, TREE, 7).astype(np.int64)
    return toks, np.array([-1] + [max(0, i - int(back[i])) for i in range(1, TREE)], dtype=np.int32)


def _bits(x):
    return np.ascontiguousarray(x, dtype=np.float32).view(np.uint32)


def _oracle(path, shape):
    toks, parent = _inputs(shape)
    m = O.Model(path, cap=toks.size)
    chain = m.eval(toks[:sum(LENS)])
    return np.concatenate([chain, m.eval_tree(toks[sum(LENS):], parent)])


@pytest.mark.parametrize("name", sorted(MODELS))
def test_flushed_subnormals_would_show(tmp_path, monkeypatch, name):
    """the models' logits change when the oracle's subnormals are flushed to zero"""
    O.gpu_numerics()
    shape, tensors, meta = MODELS[name]
    path = _model(monkeypatch, tmp_path / "m.hearth", shape, tensors, **meta)
    toks = _inputs(shape)[0][:16]
    want = O.Model(path, cap=toks.size).eval(toks)
    if not torch.set_flush_denormal(True):
        pytest.skip("this CPU does not flush subnormals")
    try:
        flushed = O.Model(path, cap=toks.size).eval(toks)
    finally:
        torch.set_flush_denormal(False)
    assert np.isfinite(want).all() and (_bits(want) != _bits(flushed)).mean() > 0.5


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(MODELS))
def test_special_values(tmp_path, monkeypatch, name):
    O.gpu_numerics()
    shape, tensors, meta = MODELS[name]
    path = _model(monkeypatch, tmp_path / "m.hearth", shape, tensors, **meta)
    want = _oracle(path, shape)
    toks, parent = _inputs(shape)
    with Engine(path, max_seq=toks.size, max_batch=512) as e:
        at = 0
        for n in LENS:
            got = e.eval(toks[at:at + n], all_logits=True)
            assert np.array_equal(_bits(got), _bits(want[at:at + n])), f"{n} tokens at {at}"
            at += n
        got = e.verify_tree(toks[at:], parent)
        assert np.array_equal(_bits(got), _bits(want[at:])), f"tree of {TREE}"


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(UNBOUNDED))
def test_unbounded_values(tmp_path, monkeypatch, name):
    """a chunk and a tree against their tokens one at a time (the kernels of few rows)"""
    path = _model(monkeypatch, tmp_path / "m.hearth", GQA, UNBOUNDED[name])
    n, width = 100, GQA.n_heads * GQA.head_dim
    toks = container.uniform_ints(3, n + TREE, GQA.vocab).astype(np.int32)
    parent = _inputs(GQA)[1]
    monkeypatch.setenv("HEARTH_DEBUG_DUMP", str(tmp_path))
    dump = tmp_path / "l0_att.bin"

    def att():
        a = np.fromfile(dump, dtype=np.float32).reshape(-1, width)
        dump.unlink()
        return a

    def same(a, b):
        nan = np.isnan(b)
        return np.array_equal(nan, np.isnan(a)) and np.array_equal(_bits(a)[~nan], _bits(b)[~nan])

    with Engine(path, max_seq=n + TREE, max_batch=512) as e:
        e.eval(toks[:n])
        chunk = att()
        e.verify_tree(toks[n:n + TREE], parent)
        tree = att()
        e.rewind(0)
        for t in toks[:n]:
            e.eval([t])
        assert same(chunk, att()), "chunk"
        node, path_toks = TREE - 1, []
        while node >= 0:
            path_toks.append(node)
            node = int(parent[node])
        path_toks.reverse()
        for i in path_toks:
            e.eval([toks[n + i]])
        assert same(tree[path_toks], att()), "tree path"
    special, total = int((~np.isfinite(chunk)).sum()), chunk.size
    assert 0 < special < total, (special, total)
