"""CPU-only checks of the drop-in boundary: the C-ABI library loads, exports what the header declares,
validates arguments before any launch, and the Python front end keeps the reference's signature."""

import ctypes as C
import inspect
import os
import re

import pytest
import torch

from sample_efficient_gpt_amd import QKNormFlashAttnFunc, SelfDotProductAttnQKNorm, TritonFlashAttnQKNormFunc, _lib
from sample_efficient_gpt_amd import CONFIGS, make_inputs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "segpt_attn.h")


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def _declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return re.findall(r"^\s*(?:const\s+)?[A-Za-z_][\w\s\*]*?\b(segpt_\w+)\s*\(", text, flags=re.M)


def test_library_exports_every_declared_symbol(lib):
    declared = _declared_functions()
    assert set(declared) == set(_lib.EXPORTED_SYMBOLS), declared
    for name in declared:
        assert getattr(lib, name) is not None
    assert lib.segpt_abi_version() == _lib.SEGPT_ABI_VERSION


def test_header_constants_match_binding():
    text = open(HEADER).read()
    consts = dict(re.findall(r"#define\s+(SEGPT_\w+)\s+(-?\d+)", text))
    assert int(consts["SEGPT_ABI_VERSION"]) == _lib.SEGPT_ABI_VERSION
    assert int(consts["SEGPT_DTYPE_BF16"]) == _lib.SEGPT_DTYPE_BF16
    assert int(consts["SEGPT_DTYPE_FP32"]) == _lib.SEGPT_DTYPE_FP32
    for name in ("SEGPT_FLAG_KV_PREPARED", "SEGPT_FLAG_RUNNING_MAX", "SEGPT_FLAG_DECODE", "SEGPT_FLAG_NO_NORM", "SEGPT_WS_KV", "SEGPT_WS_BWD"):
        assert int(consts[name]) == getattr(_lib, name), name
    stages = lambda prefix: [k for k, _ in sorted(((k, int(v)) for k, v in consts.items() if k.startswith(prefix)), key=lambda kv: kv[1])]
    assert [s.rsplit("_", 1)[1].lower() for s in stages("SEGPT_FWD_STAGE_")] == list(_lib.FWD_STAGES)
    assert [s.rsplit("_", 1)[1].lower() for s in stages("SEGPT_BWD_STAGE_")] == list(_lib.BWD_STAGES)
    # every error code has its own text
    texts = {_lib.strerror(int(v)) for k, v in consts.items() if k.startswith("SEGPT_E_")}
    assert len(texts) == len([k for k in consts if k.startswith("SEGPT_E_")])
    assert _lib.strerror(0) == "ok" and "HIP" in _lib.strerror(700)


def _valid_params(dtype=_lib.SEGPT_DTYPE_BF16, D=64):
    """Params with plausible (fake, never dereferenced) device addresses: validation happens on the host."""
    p = _lib.new_params()
    p.dtype = dtype
    p.B, p.H, p.Hkv, p.Sq, p.Sk, p.D = 2, 6, 2, 128, 128, D
    p.causal, p.q_start, p.gq_numel, p.gk_numel = 1, 0, D, 0
    p.eps, p.sm_scale, p.gate_scale = 1e-6, 0.125, 2.0
    fake = 0x10000
    for name in ("q", "o", "d_o", "dq"):
        setattr(p, name, _lib.Tensor4(fake, 6 * 128 * D, 128 * D, D))
    for name in ("k", "v", "dk", "dv"):
        setattr(p, name, _lib.Tensor4(fake, 2 * 128 * D, 128 * D, D))
    p.lse = p.g_q = p.dg_q = fake
    p.kv_workspace, p.kv_workspace_bytes = 0x40000, 1 << 30
    return p


def test_argument_errors_are_reported_before_any_launch(lib):
    # no GPU in this process: every call below must return from host-side validation
    assert lib.segpt_attn_fwd(None, None) == -1
    p = _valid_params()
    p.struct_bytes = 8
    assert lib.segpt_attn_fwd(p, None) == -2
    p = _valid_params(); p.dtype = 7
    assert lib.segpt_attn_fwd(p, None) == -3
    p = _valid_params(); p.Hkv = 4
    assert lib.segpt_attn_fwd(p, None) == -4
    p = _valid_params(); p.Sq = 0
    assert lib.segpt_attn_fwd(p, None) == -4
    p = _valid_params(); p.gq_numel = 3
    assert lib.segpt_attn_fwd(p, None) == -4
    p = _valid_params(D=48)
    assert lib.segpt_attn_fwd(p, None) == -5
    p = _valid_params(dtype=_lib.SEGPT_DTYPE_BF16, D=32)
    assert lib.segpt_attn_fwd(p, None) == -5
    p = _valid_params(); p.q.stride_s = 60
    assert lib.segpt_attn_fwd(p, None) == -6
    p = _valid_params(); p.k.stride_h = 7
    assert lib.segpt_attn_fwd(p, None) == -6
    # a bf16 row stride whose 256-row tile offsets would not fit 32 bits (the tile loads address rows that way)
    p = _valid_params(); p.q.stride_s = 1 << 23
    assert lib.segpt_attn_fwd(p, None) == -6
    # an OUTPUT view must not alias itself (a broadcast or overlapping view would make workgroups race)
    p = _valid_params(); p.o.stride_h = 0
    assert lib.segpt_attn_fwd(p, None) == -6
    p = _valid_params(); p.o.stride_b = 128 * 64  # batches overlap the heads
    assert lib.segpt_attn_fwd(p, None) == -6
    p = _valid_params(); p.workspace, p.workspace_bytes = 0x20000, 1 << 30
    p.dq.stride_b = 0
    assert lib.segpt_attn_bwd(p, None) == -6
    p = _valid_params(); p.workspace, p.workspace_bytes = 0x20000, 1 << 30
    p.dk = _lib.Tensor4(0x10000, 2 * 128 * 64, 64, 64)  # heads interleaved at the row pitch: rows collide
    assert lib.segpt_attn_bwd(p, None) == -6
    # the entry point with the library's own scratch validates the same way and needs no kv_workspace
    assert lib.segpt_attn_fwd_noalloc(None, None) == -1
    p = _valid_params(); p.kv_workspace, p.kv_workspace_bytes = None, 0; p.q.stride_s = 60
    assert lib.segpt_attn_fwd_noalloc(p, None) == -6
    p = _valid_params(); p.B, p.Sk = 4096, 4096  # 4096 * 2 * 4096 * 64 * 2 B of normalised keys
    assert lib.segpt_attn_fwd_noalloc(p, None) == _lib.SEGPT_E_SCRATCH_LIMIT
    p = _valid_params(); p.q_start = -1
    assert lib.segpt_attn_fwd(p, None) == -9
    p = _valid_params(); p.v.ptr = 0x10004
    assert lib.segpt_attn_fwd(p, None) == -10
    p = _valid_params(); p.q.ptr = None
    assert lib.segpt_attn_fwd(p, None) == -1
    p = _valid_params(); p.v_first = _lib.Tensor4(0x10000, 2 * 128 * 64, 128 * 64, 64)  # v_first without vr_coef
    assert lib.segpt_attn_fwd(p, None) == -8
    p = _valid_params(); p.kv_workspace = None
    assert lib.segpt_attn_fwd(p, None) == -7  # bf16 needs the key/value workspace
    p = _valid_params(); p.kv_workspace_bytes = lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_KV) - 1
    assert lib.segpt_attn_fwd(p, None) == -7
    p = _valid_params(); p.kv_workspace = 0x40010
    assert lib.segpt_attn_fwd(p, None) == -10
    assert lib.segpt_attn_fwd_stage(_valid_params(), 2, None) == -11
    assert lib.segpt_attn_bwd_stage(_valid_params(), 4, None) == -11
    # rotary tables: both or neither, aligned, long enough for the positions, bf16 only
    p = _valid_params(); p.rope_cos = 0x50000
    assert lib.segpt_attn_fwd(p, None) == -12
    p = _valid_params(); p.rope_cos, p.rope_sin, p.rope_len = 0x50000, 0x60000, 127  # Sq = Sk = 128 rows
    assert lib.segpt_attn_fwd(p, None) == -12
    p.rope_len, p.rope_q_pos0 = 128, 1
    assert lib.segpt_attn_fwd(p, None) == -12
    p.rope_q_pos0, p.rope_sin = 0, 0x60004
    assert lib.segpt_attn_fwd(p, None) == -12
    p = _valid_params(dtype=_lib.SEGPT_DTYPE_FP32); p.rope_cos, p.rope_sin, p.rope_len = 0x50000, 0x60000, p.Sk - 1
    assert lib.segpt_attn_fwd(p, None) == -12  # the fp32 path takes the tables too, under the same checks
    # backward-only checks
    p = _valid_params()
    assert lib.segpt_attn_bwd(p, None) == -7  # no workspace
    need = lib.segpt_attn_workspace_bytes(p, 1)
    p.workspace, p.workspace_bytes = 0x20000, need - 1
    assert lib.segpt_attn_bwd(p, None) == -7
    p = _valid_params(); p.dg_q = None
    assert lib.segpt_attn_bwd(p, None) == -1
    p = _valid_params(); p.gate = _lib.Tensor3(0x10000, 128 * 6, 6, 1)
    p.workspace, p.workspace_bytes = 0x20000, 1 << 30
    assert lib.segpt_attn_bwd(p, None) == -8  # gate without dgate slot


def test_workspace_bytes(lib):
    p = _valid_params()
    kv = lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_KV)
    assert kv >= 2 * 2 * 128 * 64 * 2 and kv % 256 == 0  # normalised keys [B,Hkv,Sk,D] bf16
    p.v_first = _lib.Tensor4(0x10000, 2 * 128 * 64, 128 * 64, 64)
    assert lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_KV) >= 2 * kv  # + mixed values
    assert lib.segpt_attn_workspace_bytes(_valid_params(dtype=_lib.SEGPT_DTYPE_FP32), _lib.SEGPT_WS_KV) == 0
    assert lib.segpt_attn_workspace_bytes(p, 2) == 0
    p = _valid_params()
    base = lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_BWD)
    rows = 2 * 6 * 128
    assert base >= rows * 4 and base % 256 == 0
    p.gate = _lib.Tensor3(0x10000, 128 * 6, 6, 1)
    assert lib.segpt_attn_workspace_bytes(p, 1) == base  # gate scale 2: the gate factor travels in the row statistics
    p.gate_scale = -1.0
    assert lib.segpt_attn_workspace_bytes(p, 1) == base + rows * 64 * 2  # a gate scale <= 0: + gated dO copy
    p32 = _valid_params(dtype=_lib.SEGPT_DTYPE_FP32)
    base32 = lib.segpt_attn_workspace_bytes(p32, 1)
    p32.gate = _lib.Tensor3(0x10000, 128 * 6, 6, 1)
    assert lib.segpt_attn_workspace_bytes(p32, 1) == base32 + rows * 64 * 4  # fp32 path: always
    bad = _valid_params(); bad.struct_bytes = 4
    assert lib.segpt_attn_workspace_bytes(bad, 1) == 0


def test_params_struct_matches_header_field_order():
    text = open(HEADER).read()
    body = text[text.index("typedef struct segpt_attn_params {"): text.index("} segpt_attn_params;")]
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    names = []
    for decl in body.split(";"):
        decl = decl.strip()
        decl = decl.split("{")[-1].strip()
        if not decl:
            continue
        first, *rest = decl.split(",")
        names.append(re.findall(r"(\w+)\s*$", first.strip())[0])
        names += [r.strip().lstrip("*") for r in rest]
    assert names == [f[0] for f in _lib.AttnParams._fields_]


def test_function_signature_is_the_reference_one():
    # reference: forward(ctx, Q, K, V, gain, is_causal=True, q_start=0)  (triton_flash_attn_qknorm.py:264-272)
    sig = inspect.signature(QKNormFlashAttnFunc.forward)
    names = list(sig.parameters)
    assert names[:7] == ["ctx", "Q", "K", "V", "gain", "is_causal", "q_start"]
    assert sig.parameters["is_causal"].default is True and sig.parameters["q_start"].default == 0
    for extra in names[7:]:
        assert sig.parameters[extra].default is not inspect.Parameter.empty  # extras are optional
    assert issubclass(QKNormFlashAttnFunc, torch.autograd.Function)
    # the reference's own name: same positional signature, but its defaults are the reference KERNEL's formula
    # (eps = 1e-8 / d on the mean, logits gain * cos; triton_flash_attn_qknorm.py:67-91), resolved at call time
    assert issubclass(TritonFlashAttnQKNormFunc, QKNormFlashAttnFunc)
    ref_sig = inspect.signature(TritonFlashAttnQKNormFunc.forward)
    assert list(ref_sig.parameters) == names
    assert ref_sig.parameters["eps"].default is None and ref_sig.parameters["sm_scale"].default is None
    assert sig.parameters["eps"].default == 1e-6 and sig.parameters["sm_scale"].default is None


def test_function_asserts_like_the_reference_on_host_tensors():
    Q = torch.randn(2, 16, 64)
    with pytest.raises(AssertionError):  # `assert Q.is_cuda and Q.is_contiguous()`, :273
        QKNormFlashAttnFunc.apply(Q, Q, Q, torch.ones(1))


def test_module_interface():
    m = SelfDotProductAttnQKNorm(64)
    sd = m.state_dict()
    assert list(sd) == ["gain"] and sd["gain"].shape == (1,) and sd["gain"].dtype == torch.float32 and float(sd["gain"]) == 1.0
    sig = inspect.signature(m.forward)
    assert list(sig.parameters) == ["Q", "K", "V", "is_causal", "q_start"]


def test_generation_step_leaves_replaced_layers_alone(monkeypatch):
    """The native step multiplies by the weights itself, so a layer whose call is anything else has none to give."""
    import torch.nn as nn
    import torch.nn.functional as F

    from sample_efficient_gpt_amd import module as M

    plain = lambda: M._Linear(8, 8)
    layer = plain()
    assert M._weight_of(layer) is layer.linear.weight and not M._linear_replaced()
    for where, other in ((nn.Linear, lambda self, x: 2 * x), (nn.Linear, print), (M._Linear, lambda self, x: 2 * x), (F, lambda x, w, b=None: 2 * x)):
        with monkeypatch.context() as m:
            m.setattr(where, "linear" if where is F else "forward", other)
            assert M._linear_replaced(), where
    assert not M._linear_replaced()
    for spoil in (lambda l: l.register_forward_hook(print), lambda l: l.linear.register_forward_pre_hook(print), lambda l: setattr(l, "forward", print),
                  lambda l: setattr(l.linear, "forward", print), lambda l: setattr(l.linear, "bias", nn.Parameter(l.linear.weight[0].detach())),
                  lambda l: nn.utils.parametrizations.weight_norm(l.linear)):
        layer = plain()
        spoil(layer)
        assert M._weight_of(layer) is None


def test_linear_rows_rejects_bad_arguments_before_any_launch(lib):
    """segpt_linear_rows returns its error codes without a device."""
    def call(M=2, K=64, x=256, xs=64, n_segments=1, w=512, ws=64, out=1024, n=5, width=5, sm=5, sh=0, struct_bytes=None):
        p = _lib.LinearRowsParams()
        p.struct_bytes = C.sizeof(p) if struct_bytes is None else struct_bytes
        p.M, p.K, p.n_segments, p.x, p.x_stride = M, K, n_segments, x, xs
        for i in range(4):
            p.seg[i] = _lib.LinearSegment(w, ws, out, sm, sh, n, width)
        return lib.segpt_linear_rows(p, None)

    codes = {k: int(v) for k, v in re.findall(r"#define\s+SEGPT_E_(\w+)\s+\(?(-?\d+)", open(HEADER).read())}
    assert lib.segpt_linear_rows(None, None) == codes["NULL"]
    assert call(struct_bytes=8) == codes["STRUCT"]
    for bad in (dict(M=0), dict(M=17), dict(K=0), dict(K=48), dict(n_segments=0), dict(n_segments=5), dict(n=0), dict(n=(1 << 24) + 1), dict(width=0)):
        assert call(**bad) == codes["SHAPE"], bad
    for bad in (dict(x=None), dict(w=None), dict(out=None)):
        assert call(**bad) == codes["NULL"], bad
    for bad in (dict(x=264), dict(w=520)):
        assert call(**bad) == codes["ALIGN"], bad
    for bad in (dict(xs=63), dict(xs=68), dict(ws=32), dict(ws=68), dict(sm=-1), dict(sh=-1)):
        assert call(**bad) == codes["STRIDE"], bad


def test_kv_append_rejects_bad_arguments_before_any_launch(lib):
    """segpt_kv_append returns its error codes without a device."""
    t = lambda ptr=256, sb=4096, sh=1024, ss=64: _lib.Tensor4(ptr, sb, sh, ss)
    call = lambda dtype=_lib.SEGPT_DTYPE_BF16, B=2, Hkv=4, S=8, D=64, k=t(), v=t(), kt=t(), vt=t(): lib.segpt_kv_append(dtype, B, Hkv, S, D, k, v, kt, vt, None)
    codes = dict(re.findall(r"#define\s+(SEGPT_E_\w+)\s+\(?(-?\d+)", open(HEADER).read()))
    want = lambda name: int(codes["SEGPT_E_" + name])
    assert call(k=t(ptr=0)) == want("NULL") and call(vt=t(ptr=0)) == want("NULL")
    assert call(dtype=7) == want("DTYPE") and call(S=0) == want("SHAPE") and call(Hkv=40000) == want("SHAPE")
    assert call(S=1 << 29) == want("SHAPE")                      # more 16-byte pieces than an int counts
    assert call(D=60) == want("STRIDE") and call(v=t(ss=66)) == want("STRIDE") and call(kt=t(ptr=264)) == want("ALIGN")
    assert call(kt=t(sh=64, ss=64)) == want("STRIDE")            # a destination whose rows overlap


@pytest.mark.parametrize("D", [64, 128])
def test_decode_partials_fit_the_scratch_of_a_split(lib, D):
    """The split-key forward asks for at most 32 rows of partials per 128 keys and (batch, kv head) pair and per pair of one
    resident round: a workspace sized without SEGPT_FLAG_DECODE (the normalised keys) holds them from 256 keys on, and the
    entry point without a workspace takes every call it could take."""
    round_ = 768 if D == 64 else 256
    for B, H, Hkv, Sq in ((1, 1, 1, 1), (1, 18, 6, 1), (3, 12, 4, 2), (1, 8, 8, 9), (2, 8, 4, 16), (5, 32, 1, 1), (64, 18, 6, 1), (1, 32, 32, 32), (300, 16, 4, 8)):
        for Sk in (1, 31, 128, 129, 1000, 4096, 70000):
            p = _lib.new_params()
            p.dtype, p.B, p.H, p.Hkv, p.Sq, p.Sk, p.D, p.causal, p.q_start = _lib.SEGPT_DTYPE_BF16, B, H, Hkv, Sq, Sk, D, 1, max(0, Sk - Sq)
            keys = lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_KV)
            p.flags = _lib.SEGPT_FLAG_DECODE
            part = lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_KV)
            pairs = B * Hkv
            splits = min(-(-round_ // pairs), -(-Sk // 128), 512)
            assert 0 < part <= -(-pairs * splits * 32 * (D + 2) * 4 // 256) * 256, (B, H, Hkv, Sq, Sk)
            assert Sk < 256 or part <= keys, (B, H, Hkv, Sq, Sk)


def test_fp32_backward_needs_partials_only_where_there_are_several(lib):
    """dK and dV of a key tile come in one part per query head of the group and share of the query tiles; a single part is formed in
    contiguous dk and dv and needs no workspace beside the row statistics and the scale-gradient partials (one row of D per 32
    query rows)."""
    B, D = 16, 64

    def ws(H, Hkv, S, bshd=False):
        p = _lib.new_params()
        p.dtype, p.B, p.H, p.Hkv, p.Sq, p.Sk, p.D, p.causal = _lib.SEGPT_DTYPE_FP32, B, H, Hkv, S, S, D, 1
        p.dk = p.dv = _lib.Tensor4(4096, S * Hkv * D, *((D, Hkv * D) if bshd else (S * D, D)))
        return lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_BWD)

    kv = lambda H, S: 2 * B * H * S * D * 4  # dK and dV of H heads
    small = lambda H, S: B * H * S * 4 + B * H * -(-S // 32) * D * 4
    for H, S in ((8, 2048), (4, 128), (1, 100)):
        assert ws(H, H, S) < small(H, S) + kv(H, S) // 16, (H, S)
    assert ws(8, 8, 2048, bshd=True) >= small(8, 2048) + kv(8, 2048)  # the parts are [B, H, S, D]
    assert ws(8, 4, 2048) >= small(8, 2048) + kv(8, 2048)
    assert ws(1, 1, 256) >= small(1, 256) + 2 * kv(1, 256)  # two shares: the launch does not fill the card


def test_fp32_split_scratch(lib):
    """SEGPT_FLAG_F32_SPLIT: sizes (0 where the other kernels are taken: short calls, forwards of a query or two against a long cache), what the
    flag asks of kv_workspace, and no effect without it or on bf16."""

    def params(Sq, Sk, D=64, **kw):
        p = _valid_params(dtype=_lib.SEGPT_DTYPE_FP32, D=D)
        p.Sq, p.Sk, p.flags = Sq, Sk, _lib.SEGPT_FLAG_F32_SPLIT
        p.workspace, p.workspace_bytes = 0x20000, 1 << 40
        for name in ("q", "o", "d_o", "dq"):
            setattr(p, name, _lib.Tensor4(0x10000, 6 * Sq * D, Sq * D, D))
        for name in ("k", "v", "dk", "dv"):
            setattr(p, name, _lib.Tensor4(0x10000, 2 * Sk * D, Sk * D, D))
        return p

    up = lambda n: -(-n // 256) * 256
    size = lambda p: [lib.segpt_attn_workspace_bytes(p, w) for w in (_lib.SEGPT_WS_F32_FWD, _lib.SEGPT_WS_F32_BWD)]
    for D in (32, 64, 128):
        few = size(params(1, 8192, D))
        assert few[0] == 0 and (few[1] > 0) == (D == 128)  # the backward is the faster one at head_dim 128, whatever the queries
        kv, q = 2 * 2 * 32, 2 * 6 * 32  # tiles of 32 rows of K and of Q: three bf16 numbers an element, two flags; lse and delta of the queries
        assert size(params(1000, 1000, D)) == [up(kv * (2 * 32 * D * 6 + 8)), up(kv * (3 * 32 * D * 6 + 8) + q * (4 * 32 * D * 6 + 8 + 64 * 4))]
    assert size(params(128, 128)) == [0, 0]
    # head_dim 128: short keys are not worth the forward's pre-pass in launches of fewer than 512 workgroups
    heads = lambda n, S, D: (lambda p: (setattr(p, "H", n), setattr(p, "Hkv", n), setattr(p, "B", 1), size(p))[-1])(params(S, S, D))
    assert heads(32, 256, 128)[0] == 0 and heads(32, 256, 128)[1] > 0
    assert heads(8, 256, 128)[0] == 0 and heads(64, 256, 128)[0] > 0 and heads(32, 416, 128)[0] > 0 and heads(8, 320, 128)[0] > 0
    # one or two kv heads under very many query tiles are left to the fp32 instructions in the backward
    group = lambda n, S, D: (lambda p: (setattr(p, "H", n), setattr(p, "Hkv", 1), setattr(p, "B", 1), size(p))[-1])(params(S, S, D))
    assert group(16, 4096, 64)[1] > 0 and group(16, 6000, 64)[1] == 0 and group(16, 6000, 64)[0] > 0 and group(16, 6000, 128)[1] > 0
    # the forward's lines at the other head sizes
    assert heads(128, 256, 32)[0] == 0 and heads(128, 448, 32)[0] > 0 and heads(320, 256, 32)[0] > 0
    assert heads(16, 512, 64)[0] == 0 and heads(8, 512, 64)[0] > 0 and heads(17, 768, 64)[0] > 0
    p = _valid_params(); p.Sq = p.Sk = 1000
    assert size(p) == [0, 0]
    # the other workspace follows the flag: no delta, no copy of a gated dO, parts of dK and dV per kv head and not per query head
    ws = lambda p: lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_BWD)
    p, rows, kv_rows = params(1000, 1000), 2 * 6 * 1000, 2 * 2 * 1000
    p.gate = _lib.Tensor3(0x10000, 6000, 6, 1)
    with_flag = ws(p)
    p.flags = 0
    assert with_flag < 2 * 4 * kv_rows * 64 * 4 + (1 << 20) and ws(p) > with_flag + rows * 65 * 4
    for call, i in ((lib.segpt_attn_fwd, 0), (lib.segpt_attn_bwd, 1)):
        p = params(1000, 1000); p.kv_workspace, p.kv_workspace_bytes = None, 0
        assert call(p, None) == -7
        p = params(1000, 1000); p.kv_workspace_bytes = size(p)[i] - 1
        assert call(p, None) == -7
        p = params(1000, 1000); p.kv_workspace, p.kv_workspace_bytes = 0x40010, 1 << 40
        assert call(p, None) == -10


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libsegpt_attn.so"))
    with pytest.raises(RuntimeError, match="no fallback"):
        _lib.load()


def test_missing_binding_fails_loudly(monkeypatch, tmp_path):
    from sample_efficient_gpt_amd import _native

    monkeypatch.setattr(_native, "_module", None)
    monkeypatch.setattr(_native, "MODULE_PATH", str(tmp_path / "_segpt_torch.so"))
    with pytest.raises(RuntimeError, match="no fallback"):
        _native.load()


def test_input_generators_are_seeded_and_shaped():
    c = CONFIGS[1]
    a, b = make_inputs(c), make_inputs(c)
    assert all(torch.equal(a[k], b[k]) for k in a)
    assert a["q"].shape == (2, 4, 256, 64) and a["q"].dtype == torch.float32 and a["g_q"].shape == (64,)
    c4 = CONFIGS[4].scaled(S=64)
    x = make_inputs(c4)
    assert x["gate_logits"].shape == (2, 64, 18) and x["v_first"].shape == (2, 6, 64, 64)
    lam = float(x["vr_coef"][0])
    assert 0.3 <= lam <= 0.7 and abs(float(x["vr_coef"].sum()) - 1) < 1e-6
    assert CONFIGS[3].flops() == 7 * 8 * 18 * 2048 * 2048 * 64 and CONFIGS[2].flops() == 2 * 8 * 18 * 2048 * 2048 * 64


def test_library_op_is_registered_with_a_shape_only_implementation():
    """torch.ops.segpt.qknorm_attention: schema, fake (meta) forward and backward shapes, no kernel involved."""
    from sample_efficient_gpt_amd import qknorm_attention_op
    from torch._subclasses.fake_tensor import FakeTensorMode

    assert hasattr(torch.ops.segpt, "qknorm_attention") and hasattr(torch.ops.segpt, "qknorm_attention_backward")
    mk = lambda *s, dt=torch.bfloat16: torch.empty(*s, dtype=dt, device="meta", requires_grad=True)
    q, k, v, g = mk(2, 6, 96, 64), mk(2, 2, 96, 64), mk(2, 2, 96, 64), mk(64, dt=torch.float32)
    y, lse = qknorm_attention_op(q, k, v, g, None, return_lse=True)
    assert y.shape == q.shape and y.dtype == q.dtype and lse.shape == (2, 6, 96) and lse.dtype == torch.float32
    y.sum().backward()
    assert q.grad.shape == q.shape and k.grad.shape == k.shape and v.grad.shape == v.shape and g.grad.shape == g.shape
    with FakeTensorMode():  # what torch.compile sees: device tensors without storage
        dev = lambda *s, dt=torch.bfloat16: torch.empty(*s, dtype=dt, device="cuda")
        out = torch.ops.segpt.qknorm_attention(dev(1, 4, 50, 128), dev(1, 2, 70, 128), dev(1, 2, 70, 128), dev(1, dt=torch.float32),
                                               None, dev(1, 2, 70, 128), dev(2, dt=torch.float32), dev(1, 50, 4), 2.0, 1e-6, 0.1, True, 20, None, None, -1, 0, True, False, False)
        assert out[0].shape == (1, 4, 50, 128) and out[1].shape == (1, 4, 50)
        assert out[2].numel() == 2 * (2 * 70 * 128 * 2 + 255) // 256 * 256 or out[2].numel() >= 2 * 2 * 70 * 128 * 2


def test_plain_c_program_uses_the_library(tmp_path):
    """The boundary is a C ABI: a C99 program (gcc, no HIP or torch headers) includes the header, links the
    shared library and calls the entry points that need no GPU; its view of the struct matches the binding's."""
    import shutil
    import subprocess

    from sample_efficient_gpt_amd import _lib

    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("gcc not found")
    lib_path = _lib.LIB_PATH if hasattr(_lib, "LIB_PATH") else os.path.join(os.path.dirname(_lib.__file__), "libsegpt_attn.so")
    src = tmp_path / "t.c"
    src.write_text(r'''
#include <stdio.h>
#include <string.h>
#include "segpt_attn.h"
int main(void) {
  segpt_attn_params p;
  memset(&p, 0, sizeof p);
  p.struct_bytes = (int)sizeof p;
  p.dtype = SEGPT_DTYPE_BF16; p.B = 2; p.H = 6; p.Hkv = 2; p.Sq = 100; p.Sk = 100; p.D = 64;
  printf("%d %zu %zu %zu %d %s\n", segpt_abi_version(), sizeof p, segpt_attn_workspace_bytes(&p, SEGPT_WS_KV),
         segpt_attn_workspace_bytes(&p, SEGPT_WS_BWD), segpt_attn_fwd(&p, NULL), segpt_strerror(SEGPT_E_HEAD_DIM));
  return 0;
}
''')
    exe = tmp_path / "t"
    inc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(_lib.__file__))), "include")
    subprocess.run([gcc, "-std=c99", "-Wall", "-Wextra", "-Werror", "-pedantic", f"-I{inc}", str(src), "-o", str(exe), lib_path,
                    f"-Wl,-rpath,{os.path.dirname(lib_path)}", "-Wl,-rpath,/opt/rocm/lib"], check=True)
    out = subprocess.run([str(exe)], check=True, stdout=subprocess.PIPE, text=True).stdout.split(maxsplit=5)
    lib = _lib.load()
    p = _lib.new_params()
    p.dtype, p.B, p.H, p.Hkv, p.Sq, p.Sk, p.D = _lib.SEGPT_DTYPE_BF16, 2, 6, 2, 100, 100, 64
    assert int(out[0]) == lib.segpt_abi_version()
    assert int(out[1]) == C.sizeof(p)
    assert int(out[2]) == lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_KV) == (2 * 2 * 100 * 64 * 2 + 255) // 256 * 256
    assert int(out[3]) == lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_BWD)
    assert int(out[4]) < 0  # argument error (no tensors bound), reported before any launch
    assert "head_dim" in out[5]
