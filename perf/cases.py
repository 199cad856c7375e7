"""The calls whose speed this package stands for, as data.

Every case goes through the public entry points (``qknorm_attention`` and its autograd, the positional drop-in
``QKNormFlashAttnFunc``, ``MultiHeadSelfAttention`` with a ``KVCache``), with the operands a model has in hand at that
moment.  ``kind`` selects what a user does:

* ``train``    forward + backward of the attention of one layer, as a training step calls it.
* ``prefill``  forward alone, no gradient: a whole prompt (Sq == Sk) or the next chunk of a long one (Sq < Sk, the
  chunk's queries sit at the end of the keys).
* ``decode``   one generated token per sequence against a cache of Sk keys.
* ``generate`` the same through the attention module with its cache: projections, gate, cache append and all.

``module`` operands are what the attention module hands over (strided views of one projection output, rotary
embedding, per-head gate, value residual, one scale vector, ``b seq head d`` output); ``plain`` operands are contiguous
``[B, H, S, D]`` tensors with a scale vector per side; ``flat`` ones the ``[(h b), S, d]`` tensors of the drop-in.
"""

from __future__ import annotations

import math

import torch

from sample_efficient_gpt_amd import KVCache, MultiHeadSelfAttention, QKNormFlashAttnFunc, qknorm_attention

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, kind, operands, B, H, Hkv, Sq, Sk, D, dtype="bf16", qk_norm=True, gate=False, residual=False):
    c = {"kind": kind, "operands": operands, "B": B, "H": H, "Hkv": Hkv, "Sq": Sq, "Sk": Sk, "D": D, "dtype": dtype,
         "qk_norm": qk_norm, "gate": gate, "residual": residual}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the pre-training step of the IMU-1 model: 8 sequences of 2048 tokens, 18 query / 6 kv heads
        _case("train_2k", "train", "plain", 8, 18, 6, 2048, 2048, 64),
        # its long-context stage: two sequences of 8192, gate and value residual on
        _case("train_8k_extras", "train", "plain", 2, 18, 6, 8192, 8192, 64, gate=True, residual=True),
        # a wider-head model at 4096 tokens
        _case("train_4k_d128", "train", "plain", 4, 16, 4, 4096, 4096, 128),
        # the call the module makes, at a length that is no multiple of anything (unpacked documents)
        _case("train_module_999", "train", "module", 8, 18, 6, 999, 999, 64, gate=True, residual=True),
        # one short sequence: fine-tuning and debugging, where the card is far from full
        _case("train_short", "train", "flat", 1, 18, 6, 512, 512, 64),
        # evaluation / prompt processing of a batch, forward alone
        _case("prefill_2k", "prefill", "plain", 8, 18, 6, 2048, 2048, 64),
        # the next 256-token chunk of one long prompt, against the keys already cached
        _case("prefill_chunk", "prefill", "module", 1, 18, 6, 256, 8192, 64, gate=True),
        # generation, one sequence, through the module: the latency of a token
        _case("generate_b1", "generate", "module", 1, 18, 6, 1, 4096, 64, gate=True),
        # batched generation against long caches: the bandwidth of the cache
        _case("decode_b32", "decode", "module", 32, 18, 6, 1, 8192, 64, gate=True),
        # the same with wide heads, a smaller batch and an odd length
        _case("decode_b8_d128", "decode", "module", 8, 16, 4, 1, 5001, 128),
        # float32: the forward of a small model, as a checkpoint is verified
        _case("fp32_forward", "prefill", "plain", 2, 4, 4, 256, 256, 64, dtype="fp32"),
        # float32: a training step of a small model
        _case("fp32_train", "train", "plain", 2, 8, 4, 1000, 1000, 64, dtype="fp32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "prefill", "prefill", "decode", "decode", "generate", "fp32"])
    H, Hkv, D = rng.choice([(18, 6, 64), (18, 6, 64), (16, 4, 128), (8, 8, 64), (16, 4, 64)])
    gate, residual = rng.random() < 0.5, rng.random() < 0.4
    qk_norm = rng.random() < 0.85
    if kind == "fp32":
        H, Hkv, D = rng.choice([(4, 4, 64), (8, 4, 64), (6, 2, 32), (4, 2, 128)])
        S = _log(rng, 64, 1000)
        B = rng.randint(1, max(1, min(8, 16_000_000 * 64 // (H * S * S * D))))
        kind = rng.choice(["train", "prefill"])
        return _case("", kind, rng.choice(["plain", "module"]), B, H, Hkv, S, S, D, "fp32", qk_norm, gate, residual)
    if kind == "train":
        S = _log(rng, 256, 8192)
        B = rng.randint(1, max(1, min(24, 2 * 18 * 8192 * 8192 * 64 // (2 * H * S * S * D))))
        operands = rng.choice(["plain", "module", "flat"])
        if operands == "flat":
            qk_norm = True
        return _case("", kind, operands, B, H, Hkv, S, S, D, "bf16", qk_norm, gate, residual)
    if kind == "prefill":
        Sk = _log(rng, 128, 8192)
        Sq = Sk if rng.random() < 0.5 else min(Sk, _log(rng, 32, 1024))
        B = rng.randint(1, max(1, min(16, 2 * 18 * 8192 * 8192 * 64 // (H * Sq * Sk * D))))
        return _case("", kind, rng.choice(["plain", "module"]), B, H, Hkv, Sq, Sk, D, "bf16", qk_norm, gate, residual)
    if kind == "decode":
        Sk = _log(rng, 200, 16000)
        B = min(_log(rng, 1, 64), max(1, 64 * 6 * 8192 * 64 // (Hkv * Sk * D)))
        return _case("", kind, "module", B, H, Hkv, 1, Sk, D, "bf16", qk_norm, gate, residual)
    Sk = _log(rng, 64, 8192)
    B = _log(rng, 1, 16)
    return _case("", kind, "module", B, H, Hkv, 1, Sk, D, "bf16", True, gate, False)


class _State:
    """What a program holds before the call."""


def _rope(length, D, dev):
    ang = torch.outer(torch.arange(length, device=dev), 10_000.0 ** (-2 * torch.arange(0, D // 2, device=dev) / D))
    return ang.cos().float(), ang.sin().float()


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = _DTYPES[case["dtype"]]
    B, H, Hkv, Sq, Sk, D = (case[k] for k in ("B", "H", "Hkv", "Sq", "Sk", "D"))
    n = lambda *s: torch.randn(*s, generator=gen, device=dev, dtype=torch.float32)
    st = _State()
    st.case = case

    if case["kind"] == "generate":
        m = MultiHeadSelfAttention(H * D, H, Hkv, max_seq_len=Sk, qknorm=True, gating="per-head" if case["gate"] else False,
                                   device=dev, dtype=dt)
        with torch.no_grad():
            for prm in m.parameters():
                if prm.dim() == 2:
                    prm.copy_(n(*prm.shape) / math.sqrt(prm.shape[1]))
        st.module, st.cache = m, KVCache(capacity=Sk)
        st.cache.append(n(B, Hkv, Sk - 1, D).to(dt), n(B, Hkv, Sk - 1, D).to(dt))  # the tokens before this one
        st.x = n(B, 1, H * D).to(dt)
        return st

    train = case["kind"] == "train"
    vec = lambda k: (1.0 + 0.02 * n(k)).requires_grad_(train)
    st.kw = {}
    if case["operands"] == "module":
        past = Sk - Sq
        proj = n(B, Sq, (H + 2 * Hkv) * D).to(dt).requires_grad_(train)
        st.q, k, v = (t.unflatten(-1, (-1, D)).permute(0, 2, 1, 3) for t in proj.split([H * D, Hkv * D, Hkv * D], dim=-1))
        if past:  # keys and values come out of the cache: a prefix of a buffer that is longer than they are
            buf = lambda: n(B, Hkv, Sk + 128, D).to(dt)[:, :, :Sk]
            st.k, st.v = buf(), buf()
            v_first = buf() if case["residual"] else None
        else:
            st.k, st.v = k, v
            v_first = n(B, Sk, Hkv, D).to(dt).permute(0, 2, 1, 3) if case["residual"] else None
        st.g = (vec(D), None)
        st.wrt = [proj]
        cos, sin = _rope(Sk, D, dev)
        st.kw.update(rope_cos=cos, rope_sin=sin, q_start=past, rope_q_pos0=past, out_bshd=True)
        st.d_o = n(B, Sq, H, D).to(dt).permute(0, 2, 1, 3) if train else None
    elif case["operands"] == "flat":
        st.q, st.k, st.v = (n(h * B, s, D).to(dt).requires_grad_(train) for h, s in ((H, Sq), (Hkv, Sk), (Hkv, Sk)))
        v_first = n(Hkv * B, Sk, D).to(dt) if case["residual"] else None
        st.g = (vec(D), None)
        st.wrt = [st.q, st.k, st.v]
        st.d_o = n(H * B, Sq, D).to(dt) if train else None
    else:
        st.q, st.k, st.v = (n(B, h, s, D).to(dt).requires_grad_(train) for h, s in ((H, Sq), (Hkv, Sk), (Hkv, Sk)))
        v_first = n(B, Hkv, Sk, D).to(dt) if case["residual"] else None
        st.g = (vec(D), vec(D))
        st.wrt = [st.q, st.k, st.v]
        st.kw["q_start"] = Sk - Sq
        st.d_o = n(B, H, Sq, D).to(dt) if train else None
    st.kw["qk_norm"] = case["qk_norm"]
    st.wrt += [g for g in st.g if g is not None]
    if case["residual"]:
        lam = 0.3 + 0.4 * torch.rand(1, generator=gen, device=dev)
        st.kw["v_first"] = v_first.requires_grad_(train)
        st.kw["vr_coef"] = torch.cat([lam, 1.0 - lam]).requires_grad_(train)
        st.wrt += [st.kw["v_first"], st.kw["vr_coef"]]
    if case["gate"]:
        st.kw["gate_logits"] = n(B, Sq, H).to(dt).requires_grad_(train)
        st.wrt.append(st.kw["gate_logits"])
    if not train:
        st.wrt = []
    return st


def _attend(st):
    if st.case["operands"] == "flat":
        kw = st.kw
        return QKNormFlashAttnFunc.apply(st.q, st.k, st.v, st.g[0], True, 0, None, kw.get("v_first"), kw.get("vr_coef"),
                                         kw.get("gate_logits"), 2.0, st.case["Hkv"])
    return qknorm_attention(st.q, st.k, st.v, st.g[0], st.g[1], **st.kw)


def run(st):
    kind = st.case["kind"]
    if kind == "train":
        y = _attend(st)
        return [y.detach(), *torch.autograd.grad(y, st.wrt, st.d_o)]
    with torch.no_grad():
        if kind == "generate":
            st.cache.length = st.case["Sk"] - 1  # the same token again: what it appended is written over
            return st.module(st.x, kv_cache=st.cache)[0]
        return _attend(st)


def work(case):
    B, H, Hkv, Sq, Sk, D = (case[k] for k in ("B", "H", "Hkv", "Sq", "Sk", "D"))
    elem = 4 if case["dtype"] == "fp32" else 2
    pairs = B * H * (Sq * (Sk - Sq) + Sq * (Sq + 1) / 2)  # (query, visible key) pairs
    q, kv = B * H * Sq * D * elem, B * Hkv * Sk * D * elem
    gate = B * Sq * H * elem if case["gate"] else 0
    first = kv if case["residual"] else 0
    flops = 4.0 * pairs * D
    nbytes = 2.0 * q + 2 * kv + first + gate
    if case["kind"] == "train":  # backward: q, k, v, y, dy in, their gradients out
        flops += 10.0 * pairs * D
        nbytes += 4.0 * q + 4 * kv + 2 * first + 2 * gate
    if case["kind"] == "generate":
        d = H * D
        weights = d * (H + 2 * Hkv) * D + d * d + (d * H if case["gate"] else 0)
        flops += 2.0 * B * weights
        nbytes += elem * weights
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Four times the distance to the same computation in float64.  Seen in bf16, in norm: 3.7e-3 (y), 4.7e-3 (dq, dk, dv,
    # dg), 7.3e-3 (the two sums of vr_coef's gradient); at the worst element 0.02 (y of a long cache), 0.11 (y), 0.39 (dq
    # with a gate).  In fp32: 1e-6 (dk, dv) and 2e-5.  The gradient of a SCALAR gain is no output of any case: it is a
    # sum that all but cancels, 0.6 away from float64 whatever the kernel.
    if case["dtype"] == "fp32":
        return {"rel": 5e-6, "max": 1e-4}
    if case["kind"] == "train":
        return {"rel": 3e-2 if case["residual"] else 2e-2, "max": 0.9}
    return {"rel": 1.5e-2, "max": 0.1 if case["kind"] == "decode" else 0.4}
