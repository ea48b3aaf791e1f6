"""The work that users of the verify engine have it do, as measurable cases.

Every case drives one open Engine through its public calls (eval, verify_greedy,
verify_sample, rewind) on a synthetic container of container.make_tiny / make_shaped:

    decode   eval of one token: plain generation
    chain    verify_greedy of the last token and n - 1 drafts in a line
    tree     verify_greedy of a draft tree of n nodes
    sample   verify_sample of a chain (temperature 0.8, top-p 0.95, point-mass drafts)
    prefill  eval of n prompt tokens, the last token's logits

after a context of `ctx` prefilled tokens. A case is {model, layers, vocab, op, n, ctx,
attn}. Models: "tiny" (4 layers of width 512), "qwen3" (the Qwen3-30B-A3B widths) and
"dsv3" (the DeepSeek-V3 widths: multi-head latent attention, groups, a shared expert, the
first layer dense). `layers` cuts the depth and `vocab` the vocabulary, so that most cases
are a short stack of blocks whose time is the blocks' own; one case is the whole model.

Weights come from a fixed seed, as a user's model file does; prompts, drafts and uniforms
come from the case's seed.
"""
from __future__ import annotations

import dataclasses
import math
import os
import struct
import tempfile
from pathlib import Path

import numpy as np
import torch

from hearth_amd import _native, container
from hearth_amd.engine import Engine, chain_uniforms, make_sampler

SHAPES = {"tiny": container.TINY, "qwen3": container.QWEN3_30B_A3B,
          "dsv3": dataclasses.replace(container.DEEPSEEK_V3, n_dense=1)}
FULL_VOCAB = container.QWEN3_30B_A3B.vocab
BLOCK_VOCAB = 8192      # block stacks: a small head, so that the layers are what is timed


def _case(name, model, layers, vocab, op, n, ctx, attn="canonical"):
    c = dict(model=model, layers=layers, vocab=vocab, op=op, n=n, ctx=ctx, attn=attn)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one token of a small model early in a reply: the shortest call there is
        _case("tiny_decode", "tiny", 4, 4096, "decode", 1, 40),
        # the parity configuration: k = 4 drafts on the small model, an odd context
        _case("tiny_chain_k4", "tiny", 4, 4096, "chain", 5, 131),
        # plain generation after a long prompt
        _case("decode_ctx4096", "qwen3", 8, BLOCK_VOCAB, "decode", 1, 4095),
        # a verify step early in a chat: most steps of short conversations
        _case("chain_k8_ctx500", "qwen3", 8, BLOCK_VOCAB, "chain", 9, 500),
        # the benchmark's step as a whole model, every row's logits returned
        _case("chain_k8_ctx4096_model", "qwen3", 48, FULL_VOCAB, "chain", 9, 4095),
        # the same blocks in the opt-in chunked attention order
        _case("chain_k8_ctx4096_chunked", "qwen3", 8, BLOCK_VOCAB, "chain", 9, 4095, "chunked"),
        # the 4 x 4 x 4 draft tree at its context
        _case("tree_85_ctx2048", "qwen3", 8, BLOCK_VOCAB, "tree", 85, 2047),
        # sampled generation with drafts over the full vocabulary
        _case("sample_k8_ctx1000", "qwen3", 4, FULL_VOCAB, "sample", 9, 1000),
        # a prompt of one batch, from empty
        _case("prefill_512", "qwen3", 8, BLOCK_VOCAB, "prefill", 512, 0),
        # the second half of a long prompt, four batches, the last one ragged
        _case("prefill_2000_at_2048", "qwen3", 8, BLOCK_VOCAB, "prefill", 2000, 2048),
        # a verify step of the latent-attention model
        _case("mla_chain_k8_ctx4096", "dsv3", 3, BLOCK_VOCAB, "chain", 9, 4095),
        # a prompt of the latent-attention model, an odd length
        _case("mla_prefill_301", "dsv3", 3, BLOCK_VOCAB, "prefill", 301, 0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["decode", "chain", "chain", "tree", "sample", "prefill"])
    model = rng.choice(["tiny", "qwen3", "qwen3", "dsv3"])
    if op == "sample":
        return _case(None, "qwen3", 4, FULL_VOCAB, op, rng.randint(2, 13), _log(rng, 40, 4095))
    layers, vocab = {"tiny": (4, 4096), "qwen3": (8, BLOCK_VOCAB), "dsv3": (3, BLOCK_VOCAB)}[model]
    top = 900 if model == "tiny" else 4095
    attn = "chunked" if model != "dsv3" and op in ("chain", "decode") and rng.random() < 0.2 else "canonical"
    if op == "decode":
        return _case(None, model, layers, vocab, op, 1, _log(rng, 16, top), attn)
    if op == "chain":
        return _case(None, model, layers, vocab, op, rng.randint(2, 16), _log(rng, 16, top), attn)
    if op == "tree":
        return _case(None, model, layers, vocab, op, rng.randint(5, 40 if model == "dsv3" else 100),
                     _log(rng, 16, min(top, 2047)))
    if model == "dsv3":
        return _case(None, model, layers, vocab, op, _log(rng, 20, 301), 0)
    return _case(None, model, layers, vocab, op, _log(rng, 20, min(top, 1900)), 0 if rng.random() < 0.5 else
                 rng.randint(1, min(top, 2048) // (16 if model == "tiny" else 1)))


# ---------------------------------------------------------------- the cases' inputs

def _shape(case):
    s = SHAPES[case["model"]]
    return dataclasses.replace(s, n_layers=case["layers"], vocab=case["vocab"], max_seq=max(s.max_seq, 1024))


def _container(case) -> Path:
    """The model file, written once."""
    d = Path(tempfile.gettempdir()) / f"hearth_cases_{os.getuid()}"
    d.mkdir(exist_ok=True)
    p = d / f"{case['model']}_L{case['layers']}_V{case['vocab']}.hearth"
    if not p.is_file():
        tmp = p.with_suffix(f".tmp{os.getpid()}")
        if case["model"] == "tiny":
            container.make_tiny(tmp, _native.quantize, seed=3, shape=_shape(case))
        else:
            container.make_shaped(tmp, _shape(case), seed=3)
        os.replace(tmp, p)
    return p


def _tree_parents(n):
    """Breadth-first parents of a tree whose inner nodes have four children."""
    return np.array([-1] + [(i - 1) // 4 for i in range(1, n)], dtype=np.int32)


def _inputs(case, seed):
    """prompt [ctx], the step's own random tokens [n] and uniforms."""
    V = case["vocab"]
    toks = container.uniform_ints(seed * 2 + 11, case["ctx"] + case["n"], V).astype(np.int32)
    return toks[:case["ctx"]], toks[case["ctx"]:], container.uniforms(seed * 2 + 12, 2 * case["n"])


def prepare(case, seed):
    path = _container(case)
    prompt, toks, u = _inputs(case, seed)
    n, ctx = case["n"], case["ctx"]
    eng = Engine(path, max_seq=ctx + n + 32, max_batch=512, attn=case["attn"])
    if ctx:
        eng.eval(prompt)
    state = dict(engine=eng, op=case["op"], ctx=ctx, tokens=toks, parent=None)
    if case["op"] in ("chain", "tree", "sample"):
        # drafts that the model partly accepts: its own greedy continuation, from a third
        # of the way on the random tokens
        parent = _tree_parents(n) if case["op"] == "tree" else np.arange(-1, n - 1, dtype=np.int32)
        toks, node = toks.copy(), 0
        for depth in range(1, max(2, n // 3)):
            child = np.flatnonzero(parent == node)
            if not len(child):
                break
            toks[child[-1]] = int(np.argmax(eng.eval([int(toks[node])])))
            node = int(child[-1])
        eng.rewind(ctx)
        state.update(tokens=toks, parent=parent if case["op"] == "tree" else None)
    if case["op"] == "sample":
        state.update(sampler=make_sampler(temperature=0.8, top_p=0.95), u=chain_uniforms(u[:n], n - 1))
    return state


def run(state):
    eng, op = state["engine"], state["op"]
    eng.rewind(state["ctx"])
    if op in ("decode", "prefill"):
        return dict(logits=eng.eval(state["tokens"]))
    if op == "sample":
        path, final, logits = eng.verify_sample(state["tokens"], None, state["sampler"], u=state["u"], want_logits=True)
    else:
        path, final, logits = eng.verify_greedy(state["tokens"], state["parent"], want_logits=True)
    return dict(path=np.array(path, dtype=np.int64), final=final, logits=logits)


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    s, n, ctx = _shape(case), case["n"], case["ctx"]
    D, H, E, K, F, V = s.d_model, s.n_heads, s.n_experts, s.top_k, s.expert_ffn, s.vocab
    q8, q4 = 66 / 64, 34 / 64
    if s.attn_kind == 1:
        attn = D * s.q_lora + s.q_lora * H * (s.nope + s.rope_qk) + D * (s.kv_lora + s.rope_qk) + \
            s.kv_lora * H * (s.nope + s.v_head) + H * s.v_head * D
        kv_row, per_row = s.kv_lora + s.rope_qk, H * (2 * s.kv_lora + s.rope_qk)
    else:
        attn = D * s.head_dim * (2 * H + 2 * s.n_kv_heads)
        kv_row, per_row = 2 * s.n_kv_heads * s.head_dim, 2 * H * s.head_dim
    rows = n * (n + 1) / 2 if case["op"] != "tree" else n * math.log(max(n, 2), 4)
    expert = 3 * D * F
    n_moe = s.n_layers - s.n_dense
    distinct = E * (1.0 - (1.0 - K / E) ** n)
    head = V * D
    head_rows = n if case["op"] in ("chain", "tree", "sample") else 1
    dense = 3 * D * s.dense_ffn * s.n_dense + 3 * D * s.shared_ffn * n_moe
    per_step = s.n_layers * attn + dense
    nbytes = q8 * (per_step + head) + n_moe * (distinct * expert * q4 + 4 * E * D) + \
        4 * s.n_layers * kv_row * (ctx + n) + 4 * V * head_rows
    macs = n * per_step + head_rows * head + n_moe * n * (K * expert + E * D) + s.n_layers * per_row * (n * ctx + rows)
    return {"bytes": float(nbytes), "flops": 2.0 * macs}


def tolerance(case):
    """The engine's numerics fix the order of every rounding (block sums in int32, folds in
    block order, 16-lane dot products, sequential value sums), so that a batch equals its
    tokens evaluated one at a time: another correct implementation gives the same bits."""
    return "exact"


# ---------------------------------------------------------------- the same in 64 bits

class _File:
    """Tensors of a .hearth container as float64 on the GPU."""

    def __init__(self, path):
        self.raw = np.memmap(path, dtype=np.uint8, mode="r")
        _, _, _, _, tdir, nt, edir, ne, _, _ = struct.unpack("<IIQQQQQQII", self.raw[:64].tobytes())
        self.tensors, self.experts = {}, []
        for i in range(nt):
            e = self.raw[tdir + 128 * i:tdir + 128 * (i + 1)].tobytes()
            dt, nd, s0, s1, _, _, off, nb, _ = struct.unpack("<II4IQQQ", e[80:])
            self.tensors[e[:80].rstrip(b"\0").decode()] = (dt, (s0, s1)[:nd], off, nb)
        for i in range(ne):
            self.experts.append(struct.unpack("<QQIIQ", self.raw[edir + 32 * i:edir + 32 * (i + 1)].tobytes())[0])
        self.kept = {}

    def _bytes(self, off, nb):
        return torch.from_numpy(np.array(self.raw[off:off + nb])).cuda()

    def matrix(self, off, rows, cols, bits):
        """rows x cols of blocks of 64: a binary16 scale, then int8s, or nibbles + 8."""
        if (off, rows) not in self.kept:
            w = 2 + (64 if bits == 8 else 32)
            b = self._bytes(off, rows * cols // 64 * w).view(-1, w)
            d = b[:, :2].contiguous().view(torch.float16).double()
            q = b[:, 2:].contiguous()
            q = q.view(torch.int8).double() if bits == 8 else torch.cat([q & 15, q >> 4], 1).double() - 8.0
            self.kept[off, rows] = (q * d).view(rows, cols)
        return self.kept[off, rows]

    def __call__(self, name):
        dt, shape, off, nb = self.tensors[name]
        if dt == container.F32:
            return self._bytes(off, nb).view(torch.float32).double().view(*shape)
        return self.matrix(off, shape[0], shape[1], 8)


def _q(x):
    """Activations as the engine's int8 blocks of 64 hold them: codes are x / (amax / 127)
    rounded, formed in 32 bits as the format says."""
    b = x.view(*x.shape[:-1], -1, 64)
    f = b.float()
    d = f.abs().amax(-1, keepdim=True) / 127.0
    r = torch.round(f * torch.where(d > 0, 1.0 / d, torch.zeros_like(d))).clamp(-127, 127)
    return (r.double() * (b.abs().amax(-1, keepdim=True) / 127.0)).view(x.shape)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w


def _rms_embedding(h):
    """The first norm (unit weights), in 32 bits and the engine's order of summation: the
    synthetic embeddings are integers times one scale, so that many of their int8 codes are
    ties, which the last bit of the norm decides."""
    a = h.float().cpu().numpy()
    lanes = np.zeros((len(a), 16), dtype=np.float32)
    for i in range(0, a.shape[1], 16):
        lanes = lanes + a[:, i:i + 16] * a[:, i:i + 16]
    for k in (8, 4, 2, 1):
        lanes = lanes[:, :k] + lanes[:, k:2 * k]
    r = np.float32(1.0) / np.sqrt(lanes / np.float32(a.shape[1]) + np.float32(1e-6))
    return torch.from_numpy(a * r).to(h.device).double()


def _rope(x, pos, inv, style):
    """x [n][heads][dim], pos [n]"""
    th = pos.double()[:, None, None] * inv
    c, s = torch.cos(th), torch.sin(th)
    if style:
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _ffn(x, g, u, d):
    xq = _q(x)
    a = xq @ g.T
    return _q(a / (1.0 + torch.exp(-a)) * (xq @ u.T)) @ d.T


def _moe(f, s, layer, x):
    p = f"blk.{layer}."
    score = x @ f(p + "moe_router").T
    score = torch.sigmoid(score) if s.score_fn else torch.softmax(score, -1)
    sel = score + f(p + "moe_router_bias") if s.score_bias else score
    if s.n_group > 1:
        g = sel.view(len(x), s.n_group, -1)
        keep = torch.topk(torch.topk(g, 2, -1).values.sum(-1), s.topk_group, -1).indices
        mask = torch.zeros(len(x), s.n_group, device=x.device, dtype=torch.bool).scatter_(1, keep, True)
        sel = torch.where(mask[..., None], g, torch.zeros_like(g)).view(len(x), -1)
    ids = torch.topk(sel, s.top_k, -1).indices
    w = torch.gather(score, 1, ids)
    if s.norm_topk:
        w = w / (w.sum(-1, keepdim=True) + 1e-20)
    w = w * s.routed_scale
    D, F = s.d_model, s.expert_ffn
    ou = -(-F * (D // 64) * 34 // 64) * 64              # gate at 0, up and down at multiples of 64 bytes
    og, od = 0, -(-(ou + F * (D // 64) * 34) // 64) * 64
    slabs = sorted({f.experts[layer * s.n_experts + e] for e in range(s.n_experts)})
    which = torch.tensor([slabs.index(f.experts[layer * s.n_experts + e]) for e in range(s.n_experts)], device=x.device)
    out = torch.zeros_like(x)
    for i, off in enumerate(slabs):
        t, j = torch.nonzero(which[ids] == i, as_tuple=True)
        if len(t):
            y = _ffn(x[t], f.matrix(off + og, F, D, 4), f.matrix(off + ou, F, D, 4), f.matrix(off + od, D, F, 4))
            out.index_add_(0, t, y * w[t, j][:, None])
    if s.shared_ffn:
        out = out + _ffn(x, f(p + "shexp_gate"), f(p + "shexp_up"), f(p + "shexp_down"))
    return out


def _attend(q, k, v, see, scale):
    """q [n][H][a], k [m][G][a], v [m][G][b], see [n][m]: [n][H][b], a few heads at a time"""
    n, H, _ = q.shape
    r = H // k.shape[1]
    out = torch.empty(n, H, v.shape[2], device=q.device, dtype=q.dtype)
    for h in range(H):
        sc = (q[:, h] @ k[:, h // r].T) * scale
        out[:, h] = torch.softmax(sc.masked_fill(~see, -math.inf), -1) @ v[:, h // r]
    return out


def _attention(f, s, layer, x, pos, see, kv, inv):
    """x [n][D] at positions pos; kv holds the rows so far (appended to); see [n][all rows]"""
    p, n, H = f"blk.{layer}.", len(x), s.n_heads
    xq = _q(x)
    if s.attn_kind == 1:
        qa = _rms(xq @ f(p + "attn_q_a").T, f(p + "attn_q_a_norm"))
        q = (_q(qa) @ f(p + "attn_q_b").T).view(n, H, -1)
        kva = xq @ f(p + "attn_kv_a").T
        c = _rms(kva[:, :s.kv_lora], f(p + "attn_kv_a_norm"))
        pe = _rope(kva[:, None, s.kv_lora:], pos, inv, s.rope_style)[:, 0]
        b = f(p + "attn_kv_b").view(H, s.nope + s.v_head, s.kv_lora)
        ql = torch.einsum("nha,hac->nhc", q[..., :s.nope], b[:, :s.nope])
        q = torch.cat([ql, _rope(q[..., s.nope:], pos, inv, s.rope_style)], -1)
        kv.append((torch.cat([c, pe], -1)[:, None], c[:, None]))
    else:
        q = (xq @ f(p + "attn_q").T).view(n, H, -1)
        k = (xq @ f(p + "attn_k").T).view(n, s.n_kv_heads, -1)
        v = (xq @ f(p + "attn_v").T).view(n, s.n_kv_heads, -1)
        q, k = _rms(q, f(p + "attn_q_norm")), _rms(k, f(p + "attn_k_norm"))
        q, k = _rope(q, pos, inv, s.rope_style), _rope(k, pos, inv, s.rope_style)
        kv.append((k, v))
    width = s.nope + s.rope_qk if s.attn_kind == 1 else s.head_dim
    o = _attend(q, torch.cat([a for a, _ in kv]), torch.cat([a for _, a in kv]), see, 1.0 / math.sqrt(width))
    if s.attn_kind == 1:
        o = torch.einsum("nhc,hvc->nhv", _q(o), b[:, s.nope:])
    return _q(o.reshape(n, -1)) @ f(p + "attn_o").T


def exact(case, seed):
    if case["layers"] > 8:
        return None     # the whole model's prompt takes minutes in 64 bits
    if case["model"] == "dsv3":
        # no such value: int8 codes and routes are steps, and with 256 experts behind grouped
        # sigmoid scores one code that falls the other way soon sends tokens to other experts
        # (the logits of a context differ by 20%, those of a lone token by 3e-7)
        return None
    s, f = _shape(case), _File(_container(case))
    state = prepare(case, seed)
    tokens, parent = state["tokens"], state["parent"]
    state["engine"].close()
    prompt = _inputs(case, seed)[0]
    n, ctx = case["n"], case["ctx"]
    parent = np.arange(-1, n - 1) if parent is None else parent
    depth, anc = np.zeros(n, dtype=np.int64), np.eye(n, dtype=bool)
    for i in range(1, n):
        depth[i], anc[i] = depth[parent[i]] + 1, anc[i] | anc[parent[i]]
    toks = torch.from_numpy(np.concatenate([prompt, tokens]).astype(np.int64)).cuda()
    pos = torch.from_numpy(np.concatenate([np.arange(ctx), ctx + depth])).cuda()
    see = torch.ones(ctx + n, ctx + n, dtype=torch.bool, device="cuda").tril()
    see[ctx:, ctx:] = torch.from_numpy(anc).cuda()
    inv = f("rope_inv_freq")
    h = f("tok_embd")[toks]
    for layer in range(s.n_layers):
        kv, done = [], []
        for a in range(0, len(h), 1024):
            b = min(len(h), a + 1024)
            x = h[a:b]
            y = _rms(x, f(f"blk.{layer}.attn_norm")) if layer else _rms_embedding(x)
            x = x + _attention(f, s, layer, y, pos[a:b], see[a:b, :b], kv, inv)
            y = _rms(x, f(f"blk.{layer}.ffn_norm"))
            done.append(x + (_moe(f, s, layer, y) if layer >= s.n_dense else _ffn(y, *(
                f(f"blk.{layer}.ffn_{m}") for m in ("gate", "up", "down")))))
        h = torch.cat(done)
    if case["op"] in ("decode", "prefill"):
        return dict(logits=_q(_rms(h[-1:], f("out_norm")))[0] @ f("lm_head").T)
    return dict(path=None, final=None, logits=_q(_rms(h[ctx:], f("out_norm"))) @ f("lm_head").T)
