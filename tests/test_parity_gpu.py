"""GPU parity: HIP kernels (through the C ABI) vs the CPU oracle on identical seeded inputs.

bf16: |err| <= 2e-2 + 1e-2*|ref| against the fp64 oracle on the same bf16 bits; fp32: 1e-5 (abs and rel).
"""

import math

import pytest
import torch

from oracle import qknorm_attn_oracle as orc
from sample_efficient_gpt_amd import (CONFIGS, FlashAttnFunc, KVCache, MultiHeadSelfAttention, QKNormFlashAttnFunc,
                                      SelfDotProductAttnQKNorm, TritonFlashAttnQKNormFunc, make_inputs, qknorm_attention, qknorm_attention_op)
from tests.parity_util import compare, decode_rounding_model, gen, run_gpu, run_oracle, scalar_gain_scale, value_residual_scale

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


def _case(device, dtype, B, H, Hkv, Sq, Sk, D, *, backward=True, seed=0, gen_kw=None, outliers=None, _x=None, **kw):
    x = gen(B, H, Hkv, Sq, Sk, D, dtype, seed=seed, **(gen_kw or {})) if _x is None else _x
    print(f"case dtype={dtype} B={B} H={H} Hkv={Hkv} Sq={Sq} Sk={Sk} D={D} bwd={backward} gen={gen_kw} "
          f"kw={ {k: v for k, v in kw.items() if k != 'rope'} } rope={'rope' in kw}", flush=True)
    got = run_gpu(x, device, backward=backward, **kw)
    ref = run_oracle(x, backward=backward, **kw)
    scales = {}
    if backward and x["g_q"].numel() == 1:
        scales.update(scalar_gain_scale(x, **kw))
    if backward and x.get("vr_coef") is not None:
        scales.update(value_residual_scale(x, ref))
    if dtype == BF16 and backward:
        _fp32_proof(device, x, ref, kw)
    try:
        return compare(got, ref, dtype, scales=scales or None)
    except AssertionError:
        if outliers is None:
            raise
        # Allowance for isolated elements: granted only to a case whose mathematics the fp32 kernels have just
        # reproduced at 1e-5 on the same inputs (_fp32_proof above), so that what is left is bf16 rounding noise.
        print("strict bound exceeded; fp32 kernels agree with the oracle at 1e-5 on this case: applying the outlier allowance", flush=True)
        return compare(got, ref, dtype, scales=scales or None, outliers=outliers)


def _fp32_proof(device, x, ref, kw, backward=True):
    """The bf16 comparisons use magnitude yardsticks for gradients that are sums over every row (and, in the sweep,
    an allowance for isolated elements).  They are only meaningful if the slack they grant is bf16 rounding noise and
    not a wrong formula, so every such case also runs the fp32 kernels on the SAME inputs (the bf16 values, widened)
    and asserts 1e-5 against the same oracle result, every output and gradient, element-wise for the tensors and
    relative to the largest entry for the summed parameter gradients."""
    x32 = {n: (t.float() if torch.is_tensor(t) and t.dtype == BF16 else t) for n, t in x.items()}
    got32 = run_gpu(x32, device, backward=backward, **kw)
    compare(got32, ref, F32, label="fp32 kernels on the same inputs: ")


# ------------------------------------------------------------------ fp32 path (1e-5)


def test_cfg1_fp32_forward(gpu_device):
    c = CONFIGS[1]
    x = make_inputs(c)
    print("cfg1 fp32 forward", flush=True)
    got = run_gpu(x, gpu_device, backward=False, eps=c.eps, sm_scale=c.sm_scale)
    ref = run_oracle(x, backward=False, eps=c.eps, sm_scale=c.sm_scale)
    errs = compare(got, ref, F32)
    print("cfg1 max abs err", errs)


@pytest.mark.parametrize(
    "B,H,Hkv,Sq,Sk,D,kw,gen_kw",
    [
        (2, 4, 4, 256, 256, 64, {}, {}),
        (1, 6, 2, 100, 100, 64, {}, {"extras": True}),
        (2, 4, 2, 77, 77, 32, {}, {"scalar_gain": True, "no_gk": True}),
        (1, 4, 1, 130, 130, 128, {}, {}),
        (1, 2, 2, 48, 80, 64, {"causal": False}, {}),
        (1, 3, 3, 40, 104, 64, {"q_start": 64}, {"extras": True}),
        (1, 2, 1, 64, 64, 64, {"eps": 1e-8 / 64, "sm_scale": 1 / 64}, {"scalar_gain": True, "no_gk": True}),
        (1, 4, 2, 200, 200, 64, {"gate_scale": 2.0}, {"extras": True, "scalar_gain": True}),  # scalar q gain + vector k scale
        (1, 2, 1, 200, 130, 64, {}, {}),   # causal with more queries than keys: rows >= 130 see every key
    ],
)
def test_fp32_fwd_bwd(gpu_device, B, H, Hkv, Sq, Sk, D, kw, gen_kw):
    _case(gpu_device, F32, B, H, Hkv, Sq, Sk, D, gen_kw=gen_kw, **kw)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize(
    "B,H,Hkv,Sq,Sk,kw,gen_kw",
    [
        (1, 1, 1, 1, 1, {}, {}),                                  # three of the four waves own no tile
        (1, 2, 1, 31, 33, {"q_start": 2}, {"extras": True}),      # one row short of / past a 32-row tile
        (2, 2, 2, 32, 129, {"causal": False}, {}),                # the fifth tile goes to wave 0 again
        (1, 9, 3, 97, 97, {}, {"extras": True}),                  # every query tile its own split, some splits empty
        (5, 16, 4, 289, 289, {}, {}),                             # more than 1024 work items: the plain order
        (1, 2, 1, 5, 300, {"causal": True}, {}),                  # keys that no query sees: zero gradients
    ],
)
def test_fp32_tile_edges(gpu_device, B, H, Hkv, Sq, Sk, D, kw, gen_kw):
    """The 32-row tiles of the fp32 kernels, the four-way split of the streamed rows and the splits of dK/dV, same
    1e-5 as above."""
    _case(gpu_device, F32, B, H, Hkv, Sq, Sk, D, gen_kw=gen_kw, seed=71, **kw)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize(
    "B,H,Hkv,Sq,Sk,kw,gen_kw",
    [
        (2, 4, 2, 769, 769, {}, {}),                                                      # one row past 24 tiles
        (1, 8, 8, 895, 895, {"rope": True, "gate_scale": -1.5}, {"extras": True}),         # one short of 28; one head a group
        (2, 9, 3, 640, 833, {"q_start": 193, "rope": True}, {"extras": True, "scalar_gain": True}),
        (2, 6, 2, 545, 801, {"causal": False}, {"scalar_gain": True, "no_gk": True}),
        (1, 8, 2, 830, 790, {}, {}),                                                      # queries that see every key
        (2, 4, 1, 800, 800, {"qk_norm": False}, {"scalar_gain": True, "no_gk": True}),
        (4, 8, 2, 200, 900, {"q_start": 3}, {}),                                          # keys that no query sees
        (5, 9, 3, 769, 769, {}, {}),  # more than 1024 workgroups, (batch, kv head) pairs that are no multiple of the XCDs
        (1, 44, 1, 770, 770, {}, {}),  # the same with one pair for all XCDs
        (3, 10, 5, 1100, 1100, {}, {}),  # dK/dV: 525 workgroups would take one part each, two where they walk more than an L2 holds
        (4, 8, 4, 1025, 1025, {}, {"extras": True}),  # one part of dK and dV for two heads a group, formed in place
        (1, 27, 3, 1290, 1290, {}, {}),  # three pairs: two and one at a time; dK/dV between 512 and 1024 workgroups, more than an L2 streamed
    ],
)
def test_fp32_split_edges(gpu_device, B, H, Hkv, Sq, Sk, D, kw, gen_kw):
    """Calls long enough for the three-way bf16 splits (operands as sums of three bf16 numbers on the bf16 matrix pipe): tile edges,
    shares of the query tiles over the heads of a group, both orders of the workgroups; the same 1e-5."""
    from sample_efficient_gpt_amd import _lib

    p = _lib.new_params()
    p.dtype, p.B, p.H, p.Hkv, p.Sq, p.Sk, p.D = _lib.SEGPT_DTYPE_FP32, B, H, Hkv, Sq, Sk, D
    for which in (_lib.SEGPT_WS_F32_FWD, _lib.SEGPT_WS_F32_BWD):
        assert _lib.load().segpt_attn_workspace_bytes(p, which) > 0
    kw = dict(kw)
    if kw.pop("rope", False):
        kw["rope"] = orc.rope_tables(1000, 10000.0, D)
    print(f"split edges B={B} H={H} Hkv={Hkv} Sq={Sq} Sk={Sk} D={D}", flush=True)
    _case(gpu_device, F32, B, H, Hkv, Sq, Sk, D, gen_kw=gen_kw, seed=72, **kw)


@pytest.mark.parametrize("B,H,Hkv,S,D,extras", [(1, 4, 2, 401, 64, True), (4, 12, 4, 300, 32, False), (4, 8, 4, 1024, 64, False), (4, 8, 4, 1025, 64, True),
                                               (1, 5, 5, 2700, 64, False), (1, 4, 1, 3700, 32, True)])
def test_fp32_split_backward_in_one_launch_is_its_stages(gpu_device, B, H, Hkv, S, D, extras):
    """dQ and dK/dV of a whole backward share a launch up to 1024 workgroups each (the third case; the fourth has more) while what dQ streams
    fits an L2 (the last two do not); the stages run one by one.  Both are within 8 units of 2^-24 of float64 in norm (test_fp32_split_is_no_less_accurate), so within 16 of each other."""
    from sample_efficient_gpt_amd import _lib
    from sample_efficient_gpt_amd.plan import AttnPlan

    x = gen(B, H, Hkv, S, S, D, F32, seed=51, extras=extras)
    plan = AttnPlan({n: None if t is None else t.to(gpu_device) for n, t in x.items()})
    need = plan.lib.segpt_attn_workspace_bytes(plan.p, _lib.SEGPT_WS_F32_BWD)
    assert need > 0
    plan.forward()
    scratch = torch.empty(need, dtype=torch.uint8, device=gpu_device)
    plan.p.kv_workspace, plan.p.kv_workspace_bytes = scratch.data_ptr(), need
    plan.base_flags |= _lib.SEGPT_FLAG_F32_SPLIT
    grads = [t for t in (plan.dq, plan.dk, plan.dv, plan.dg_q, plan.dg_k, plan.dv_first, plan.dgate) if t is not None]
    plan.backward()
    whole = [t.clone() for t in grads]
    for t in grads:
        t.fill_(float("nan"))
    for stage in range(4):
        plan.backward_stage(stage)
    for w, t in zip(whole, grads):
        assert (w.double() - t.double()).norm() <= 16 * 2.0**-24 * w.double().norm()


@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_split_is_no_less_accurate(gpu_device, D):
    """Distance to float64 in norm, in units of 2^-24, of y, dq, dk, dv of a call that the splits take.  With the fp32 matrix instruction
    it was 3.31, 6.36, 7.60, 6.09 at its largest over the three head sizes, the bounds; with the splits 2.64, 5.74, 6.09, 4.82."""
    rng = torch.Generator().manual_seed(D)
    S = 770
    ops = [torch.randn(2, h, S, D, generator=rng) for h in (4, 2, 2)]
    dy, one = torch.randn(2, 4, S, D, generator=rng), torch.ones(1)
    wide = [t.double().requires_grad_(True) for t in ops]
    y64 = orc.attention_forward(*wide, one.double(), qk_norm=True)[0]
    leaves = [t.to(gpu_device).requires_grad_(True) for t in ops]
    y = qknorm_attention(*leaves, one.to(gpu_device))
    got = [y, *torch.autograd.grad(y, leaves, dy.to(gpu_device))]
    ref = [y64, *torch.autograd.grad(y64, wide, dy.double())]
    err = [((a.detach().cpu().double() - b).norm() / b.norm()).item() * 2**24 for a, b in zip(got, ref)]
    print("units of 2^-24:", " ".join(f"{e:.2f}" for e in err), flush=True)
    assert all(e <= bound for e, bound in zip(err, (3.31, 6.36, 7.60, 6.09)))


@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_split_against_the_instructions_on_the_same_inputs(gpu_device, D):
    """The same per head size, against the fp32 instructions on the same inputs: the distances to float64 of y, dq, dk and dv, added up over
    three draws and lengths, are no larger (0.7 to 0.95 of theirs)."""
    sums = torch.zeros(2, 4)
    for seed, S in ((1, 770), (2, 830), (3, 1001)):
        x = gen(1, 8, 4, S, S, D, F32, seed=seed, scalar_gain=True, no_gk=True)
        ref = run_oracle(x)
        for row, outs in zip(sums, _fp32_both_ways(x, gpu_device)):
            row += torch.tensor([(a.double() - ref[n]).norm() / ref[n].norm() * 2**24 for a, n in zip(outs, ("y", "dq", "dk", "dv"))])
    print("units of 2^-24, three bf16 numbers and fp32 instructions:", (sums / 3).tolist(), flush=True)
    assert bool((sums[0] <= sums[1]).all())


def test_fp32_without_room_for_the_split_operands(gpu_device):
    """Where the scratch of the three-bf16 kernels does not fit, a step that fits without it runs with the fp32 instructions instead of out of
    memory; against a plan that never asks for the scratch, at 1e-5."""
    from sample_efficient_gpt_amd import _lib
    from sample_efficient_gpt_amd.plan import AttnPlan

    x = {n: None if t is None else t.to(gpu_device) for n, t in gen(4, 8, 2, 2048, 2048, 64, F32, seed=66).items()}
    plan = AttnPlan(x)
    plan.forward()
    plan.backward()
    want = [t.clone() for t in (plan.y, plan.dq, plan.dk, plan.dv)]
    need = plan.lib.segpt_attn_workspace_bytes(plan.p, _lib.SEGPT_WS_F32_BWD)
    step = 2 * x["q"].nbytes + 2 * x["k"].nbytes + plan.ws.numel()  # y, dq, dk, dv, workspace
    assert need > 100 << 20 and step < 90 << 20
    del plan
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(gpu_device).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(gpu_device) + step + (24 << 20)) / total, gpu_device)
        leaves = [x[n].requires_grad_(True) for n in ("q", "k", "v")]
        y = qknorm_attention(*leaves, x["g_q"], x["g_k"])
        got = [y.detach(), *torch.autograd.grad(y, leaves, x["d_o"])]
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu_device)
    for a, b in zip(got, want):
        assert torch.allclose(a, b, atol=1e-5, rtol=1e-5)


def _fp32_both_ways(x, device):
    """y, dq, dk, dv with the three-bf16 kernels (the call as users make it) and with the fp32 instructions (without the flag)."""
    from sample_efficient_gpt_amd import _lib
    from sample_efficient_gpt_amd.plan import AttnPlan

    plan = AttnPlan({n: None if t is None else t.to(device) for n, t in x.items()})
    for which in (_lib.SEGPT_WS_F32_FWD, _lib.SEGPT_WS_F32_BWD):
        assert plan.lib.segpt_attn_workspace_bytes(plan.p, which) > 0
    plan.forward()
    plan.backward()
    torch.cuda.synchronize()
    got = run_gpu(x, device)
    return [got[n] for n in ("y", "dq", "dk", "dv")], [t.cpu() for t in (plan.y, plan.dq, plan.dk, plan.dv)]


def _within(a, b, units):
    """Distance in norm of the finite values, in units of 2^-24; the others have to agree."""
    fa, fb = torch.isfinite(a), torch.isfinite(b)
    assert torch.equal(fa, fb) and torch.equal(a.isinf(), b.isinf()) and torch.equal(a[a.isinf()], b[b.isinf()])
    a, b = a.double()[fa], b.double()[fb]
    assert (a - b).norm() <= units * 2.0**-24 * b.norm()


@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_split_values_beyond_bf16s_range(gpu_device, D):
    """Infinities and finite values above bf16's largest number in v and dO: infinite, NaN and finite results stand where the fp32
    instructions have them.  Both are within 8 units of 2^-24 of float64 (test_fp32_split_is_no_less_accurate), so within 16 of each other."""
    base = gen(1, 8, 4, 800, 800, D, F32, seed=67, scalar_gain=True, no_gk=True)

    def run(name, row, value):
        x = dict(base, **{name: base[name].clone()})
        x[name][0, 1, row, 3] = value
        print(f"{name}[{row}] = {value}, D={D}", flush=True)
        return _fp32_both_ways(x, gpu_device)

    new, old = run("v", 500, float("inf"))
    assert new[0].isinf().sum() == 2 * 300 and new[0].isnan().sum() == old[0].isnan().sum()
    for a, b in zip(new, old):
        _within(a, b, 16)
    for row in (0, 400):
        new, old = run("d_o", row, float("-inf"))
        assert new[3].isinf().any()
        for a, b in zip(new, old):
            _within(a, b, 16)
    # query 0 sees key 0 alone: its row of y is v's, and dv gets dO's times the other probabilities
    for value in (3.4e38, -3.3962e38):
        new, old = run("v", 0, value)
        assert torch.isfinite(new[0]).all() and new[0][0, 2, 0, 3] == torch.tensor(value)
        _within(new[0], old[0], 16)
        new, old = run("d_o", 0, value)
        assert torch.isfinite(new[3]).all()
        _within(new[3], old[3], 16)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_split_small_values(gpu_device, D):
    """The calls are linear in v (y) and in dO (dq, dk, dv): scaled by 2^-112 (1e-34) they give the same numbers times 2^-112, within the 16
    units of two results that are 8 from float64 each; products that end among the subnormal numbers lose up to 2^-150, 2^-38 of a result of
    ordinary size, 0.05 units for 800 of them.  With some rows scaled and others not, in one tile and in a tile of their own, every row
    of y and dq scales with its own operand (the values of its keys, its dO) alone."""
    x = gen(1, 8, 4, 800, 800, D, F32, seed=68, scalar_gain=True, no_gk=True)
    f = 2.0**-112
    (y, dq, dk, dv), _ = _fp32_both_ways(x, gpu_device)
    print(f"small values, D={D}", flush=True)
    small_y = _fp32_both_ways(dict(x, v=x["v"] * f), gpu_device)[0][0]
    small = _fp32_both_ways(dict(x, d_o=x["d_o"] * f), gpu_device)[0][1:]
    for a, b in zip((small_y, *small), (y, dq, dk, dv)):
        _within(a.double() / f, b.double(), 16)
    scale = torch.ones(800, 1)
    scale[100:101] = scale[320:352] = scale[700:750] = f
    got = _fp32_both_ways(dict(x, d_o=x["d_o"] * scale), gpu_device)[0]
    _within(got[1].double() / scale.double(), dq.double(), 16)
    scale = torch.where(torch.arange(800).unsqueeze(1) < 40, f, 1.0)  # queries 0 .. 39 see small values alone
    got, old = _fp32_both_ways(dict(x, v=x["v"] * scale), gpu_device)
    _within(got[0][:, :, :40].double() / f, y[:, :, :40].double(), 16)
    for a, b in zip(got, old):
        _within(a, b, 16)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_split_small_probabilities(gpu_device, D):
    """Keys that every query ignores: with logits 78 below the others' (112.5 in base 2) their probabilities are 2^-114 to 2^-122, and their
    rows of dv and dk have the accuracy that the logits allow: five roundings of them (the scale vector's three, Qhat's, the sum's) are
    5 * 112.5 * ln 2 * 2^-24 = 2.3e-5 of a probability.  Unscaled, the parts of the smallest ones are off by 2^-12."""
    x = gen(1, 8, 4, 800, 800, D, F32, seed=69, scalar_gain=True, no_gk=True)
    x["q"] *= 0.05
    x["q"][..., 0] = 1.0
    x["k"][..., 0] = 0.0
    ignored = torch.arange(0, 800, 3)[1:]
    x["k"][:, :, ignored, 0] = -78.0 * D**0.5 / 1.3
    print(f"small probabilities, D={D}", flush=True)
    got, ref = run_gpu(x, gpu_device, qk_norm=False), run_oracle(x, qk_norm=False)
    late = ignored[(ignored > 400) & (ignored < 700)]
    assert 2.0**-126 < ref["dv"][:, :, late].abs().max() < 2.0**-110
    for n in ("dk", "dv"):
        for rows in (late, late + 1):
            a, b = got[n][:, :, rows, 1:].double(), ref[n][:, :, rows, 1:]  # column 0 of dk is the sum of dS, which all but cancels
            assert (a - b).norm() <= 5 * 112.5 * math.log(2) * 2.0**-24 * b.norm(), n


@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_rows_whose_mean_square_leaves_the_normal_range(gpu_device, D):
    """A key whose sum of squares overflows has the normaliser 0, like a key of zeros, and poisons nobody; keys so small
    that their mean square is subnormal (eps = 0) are normalised like any others."""
    x = gen(1, 2, 1, 70, 70, D, F32, seed=65)
    row = lambda k, j, f: torch.cat([k[:, :, :j], k[:, :, j:j + 1] * f, k[:, :, j + 1:]], 2)
    print(f"huge key, D={D}", flush=True)
    got = run_gpu(dict(x, k=row(x["k"], 33, 1e25)), gpu_device)
    ref = run_oracle(dict(x, k=row(x["k"], 33, 0.0)))
    compare(got, ref, F32, names=["y", "lse", "dq", "dv", "dg_q", "dg_k"])
    assert (got["dk"][:, :, 33] == 0).all()
    keep = [j for j in range(70) if j != 33]
    compare({"dk": got["dk"][:, :, keep]}, {"dk": ref["dk"][:, :, keep]}, F32)
    print(f"tiny keys, D={D}", flush=True)
    small = dict(x, k=x["k"] * torch.where(torch.arange(70) % 3 == 0, 1e-20, 1.0).reshape(1, 1, 70, 1))
    got, ref = (f(small, backward=False, eps=0.0) for f in (lambda x, **kw: run_gpu(x, gpu_device, **kw), run_oracle))
    # a square of 1e-40 is rounded to a multiple of 2^-149, 0.7e-5 of it, and so is their mean: up to 0.7e-5 on the key and,
    # logits of up to about 5, 4e-5 on a probability
    for n in ("y", "lse"):
        assert (got[n].double() - ref[n].reshape(got[n].shape)).abs().max() < 1e-4, n


@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_forward_rounding_does_not_grow_with_the_head_size(gpu_device, D):
    """Scores are sums of D products; added up one after the other their error grows with D and y's distance to float64
    was 2.9e-7 in norm for a call of this length at head_dim 128.  Bound: four roundings of half a unit in the last place
    (2^-24 each); seen 1.3e-7, 1.4e-7, 1.5e-7 at head_dim 32, 64, 128."""
    rng = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(3, h, 212, D, generator=rng) for h in (4, 2, 2))
    one = torch.ones(1)
    ref = orc.attention_forward(q.double(), k.double(), v.double(), one.double(), qk_norm=False)[0]
    with torch.no_grad():
        y = qknorm_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), one.to(gpu_device), qk_norm=False)
    assert (y.cpu().double() - ref).norm() <= 4 * 2.0**-24 * ref.norm()


@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_dq_rounding_does_not_grow_with_the_head_size(gpu_device, D):
    """dq's scores and its products with dO are sums of D products as well: two sums each put it 6.2 units of 2^-24 from float64 in
    norm for a call of this length at head_dim 128.  Bound: 5.7, what plain FMA loops with four sums a row reached (5.6)."""
    rng = torch.Generator().manual_seed(D)
    ops = torch.randn(3, 4, 212, D, generator=rng), torch.randn(3, 2, 212, D, generator=rng), torch.randn(3, 2, 212, D, generator=rng)
    dy = torch.randn(3, 4, 212, D, generator=rng)
    one = torch.ones(1)
    wide = [t.double().requires_grad_(True) for t in ops]
    ref, = torch.autograd.grad(orc.attention_forward(*wide, one.double(), qk_norm=False)[0], wide[0], dy.double())
    q, k, v = (t.to(gpu_device).requires_grad_(True) for t in ops)
    dq, = torch.autograd.grad(qknorm_attention(q, k, v, one.to(gpu_device), qk_norm=False), q, dy.to(gpu_device))
    assert (dq.cpu().double() - ref).norm() <= 5.7 * 2.0**-24 * ref.norm()


@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_backward_rounds_the_row_statistic_once(gpu_device, D):
    """All keys have one and the same large score (46 to 60, exact in every order of summation): row i's probabilities are 1/(i+1),
    and what the backward makes of them shows the error of exp(score - lse) alone.  Bound, relative: lse below 64 is stored to half
    a unit, 2^-19; the two constants ln 2 and log2 e miss 1 by 1.1e-8, 7e-7 at 64; exponential, logarithm and products 3e-7.
    With lse * log2 e rounded as well it was up to 2.6e-6 more (5.1e-6 on these inputs)."""
    n, S = 64, 32
    eye = torch.eye(S, device=gpu_device)
    q, k, v, dy = (torch.zeros(n, 1, S, D, device=gpu_device) for _ in range(4))
    q[..., 0] = 46.0 + 14.0 * torch.arange(n, device=gpu_device).reshape(n, 1, 1) / n
    k[..., :S] = eye
    k[..., 0] = 1.0
    sign = 1.0 - 2.0 * (torch.arange(S, device=gpu_device) % 2)
    v[..., :S] = sign.unsqueeze(1)
    dy[..., :S] = eye
    for t in (q, k, v):
        t.requires_grad_(True)
    y = qknorm_attention(q, k, v, torch.ones(1, device=gpu_device), sm_scale=1.0, qk_norm=False)
    dq, dv = (t.double() for t in torch.autograd.grad(y, [q, v], dy))
    p = torch.tril(torch.ones(S, S, dtype=torch.float64, device=gpu_device)) / torch.arange(1, S + 1, device=gpu_device).unsqueeze(1)
    ds = p * (sign - (p * sign).sum(-1, keepdim=True))  # dp_ij = sign_j
    bound = 2.0**-19 + 7e-7 + 3e-7
    assert bool(((dv[..., :S].transpose(2, 3) - p).abs() <= bound * p).all())
    # from the second row on (the first has p (dp - delta) = 0); delta carries y's rounding, 2e-7
    assert bool(((dq[:, :, 1:, 1:S] - ds[1:, 1:]).abs() <= bound * ds[1:, 1:].abs() + 2e-7 * p[1:, 1:]).all())


# ------------------------------------------------------------------ bf16 MFMA path


@pytest.mark.parametrize(
    "B,H,Hkv,Sq,Sk,D,kw,gen_kw",
    [
        (1, 1, 1, 64, 64, 64, {}, {}),
        (1, 1, 1, 256, 256, 64, {}, {}),
        (2, 6, 2, 512, 512, 64, {}, {}),
        (1, 3, 1, 300, 300, 64, {}, {}),          # ragged: not a multiple of any tile
        (1, 2, 2, 77, 77, 64, {}, {"scalar_gain": True, "no_gk": True}),
        (2, 6, 2, 384, 384, 64, {"gate_scale": 1.0}, {"extras": True}),
        (1, 4, 2, 200, 200, 64, {"gate_scale": 2.0}, {"extras": True, "scalar_gain": True}),
        (1, 2, 1, 256, 256, 128, {}, {}),
        (1, 4, 1, 333, 333, 128, {}, {"extras": True, "head_scales": True}),
        (1, 2, 2, 96, 200, 64, {"causal": False}, {}),
        (1, 2, 1, 130, 130, 128, {"causal": False}, {}),
        (1, 3, 3, 72, 200, 64, {"q_start": 128}, {}),
        (1, 2, 1, 1, 257, 64, {"q_start": 256}, {}),   # decode step: one query against a 257-key cache
        (8, 2, 1, 128, 128, 64, {}, {}),              # B*Hkv multiple of 8: XCD-pinned workgroup order
        (3, 6, 3, 300, 300, 64, {}, {}),              # 9 pairs: 8 pinned + 1 spread, 6 left-over workgroups padded to 8
        (9, 2, 1, 128, 128, 64, {"gate_scale": 2.0}, {"extras": True}),   # 9 pairs, one tile: 2 left-over workgroups + 6 idle
        (5, 4, 4, 200, 200, 128, {}, {}),             # 20 pairs at head_dim 128: 16 pinned + 4 spread
        (1, 2, 2, 128, 128, 64, {"eps": 1e-8 / 64, "sm_scale": 1 / 64}, {"scalar_gain": True, "no_gk": True}),
        (2, 4, 2, 300, 130, 64, {}, {}),               # causal with more queries than keys: rows >= 130 see every key
        (1, 2, 1, 257, 64, 128, {}, {"extras": True}),
        (1, 2, 1, 100, 400, 64, {"gate_scale": 2.0}, {"extras": True}),  # key tiles beyond every query: dK/dV workgroups without a loop
        (1, 2, 2, 60, 300, 128, {}, {}),
    ],
)
def test_bf16_fwd_bwd(gpu_device, B, H, Hkv, Sq, Sk, D, kw, gen_kw):
    _case(gpu_device, BF16, B, H, Hkv, Sq, Sk, D, gen_kw=gen_kw, **kw)


@pytest.mark.parametrize("S", [768, 896, 1152])
def test_bf16_reference_training_contexts(gpu_device, S):
    """The context lengths of the reference's training curriculum (configs/imu1_base.yaml:56,80,105) with the IMU-1 head
    layout (GQA 3:1, head_dim 64), gate + value residual as the model runs them: 768 and 896 are multiples of the
    128-row workgroup tile, 1152 is nine tiles (an odd count for the paired 64-row stages)."""
    _case(gpu_device, BF16, 2, 6, 2, S, S, 64, seed=S, gen_kw={"extras": True}, gate_scale=2.0)


@pytest.mark.parametrize("D", [64, 128])
def test_bf16_gate_factor_through_the_row_statistics(gpu_device, D):
    """The dK/dV kernel receives a positive gate factor f inside the two row statistics (-lse2 + log2 f, -delta / f)
    and streams the caller's dO.  Gate logits over the whole range of the sigmoid: saturated on (f = gate_scale),
    ordinary, so negative that f is 1e-20 (still carried), and so negative that it underflows (the row is switched
    off: its contributions to dk, dv, dq, dgate are below 1e-30 in the oracle too)."""
    x = gen(2, 6, 2, 300, 300, D, BF16, extras=True, seed=5)
    z = x["gate_logits"]
    S = z.shape[1]
    z[:, 0::7] = 30.0
    z[:, 3::7] = -46.0
    z[:, 5::7] = -90.0
    z[:, 6::7] = -200.0
    z[1, S // 2:] = -200.0  # whole query tiles switched off
    _case(gpu_device, BF16, 2, 6, 2, 300, 300, D, gate_scale=2.0, _x=x)
    got = run_gpu(x, gpu_device, gate_scale=2.0)
    for n, t in got.items():
        assert torch.isfinite(t.float()).all(), n


@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D,kw", [
    (1, 3, 1, 33, 65, 64, {"q_start": 32}),                # one key in the last workgroup, second key wave beyond the end
    (2, 3, 1, 161, 97, 64, {"causal": False}),             # three key blocks: the last workgroup holds one
    (2, 2, 1, 64, 290, 128, {"q_start": 226}),             # the last 64-key tile is 34 rows
    (4, 64, 64, 96, 200, 64, {"q_start": 104}),            # 512 128-key workgroups, short: not split
    (3, 86, 86, 70, 190, 64, {"causal": False}),           # more than 512
    (2, 65, 65, 130, 250, 128, {"q_start": 120}),          # head_dim 128, just more than 256: not split
])
def test_bf16_dkdv_workgroup_shapes(gpu_device, B, H, Hkv, Sq, Sk, D, kw):
    """dK/dV with 64-key workgroups whose waves split the queries (launches that do not fill the card) and with 128-key
    ones, at the ragged ends of both, with gate, value residual and rotary embedding."""
    _case(gpu_device, BF16, B, H, Hkv, Sq, Sk, D, seed=61, gen_kw={"extras": True}, rope=orc.rope_tables(max(Sq, Sk), 10000.0, D), **kw)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,kw", [
    (4, 66, 66, 33, 40, {"q_start": 7}),        # one streamed tile, requested over and over; its second block has one query
    (4, 66, 66, 70, 100, {"causal": False}),    # two, the last of six rows
    (3, 174, 87, 64, 64, {}),                   # two heads, one tile each, nothing but diagonal
    (2, 198, 66, 97, 300, {}),                  # six; the later key tiles see one query or none
    (3, 90, 90, 200, 140, {"causal": False}),   # four, and a last key tile of 12 rows
])
def test_bf16_dkdv_pipeline_ends(gpu_device, B, H, Hkv, Sq, Sk, D, kw):
    """dK/dV of launches that fill the card (128-key workgroups) at the shortest streams and at ragged ends; at head_dim 128 the
    loop runs two blocks ahead of itself and requests a tile in every iteration (at head_dim 64 it takes longer streams: the next test).
    Outliers: a launch that fills the card has millions of entries, and dk of a row that few queries see is a sum of few terms
    with roundings of 2^-9 each against a result that cancels; over the 198-head case dk is 3.7e-3 from float64 in norm and
    one entry of 2.5 million is 0.043 away where the elementwise bound says 0.04 (both to all digits also with the products
    in the order of tiles, head by head).  One in a million may be up to twice the bound away."""
    assert B * Hkv * (-(-Sk // 128)) > 256
    _case(gpu_device, BF16, B, H, Hkv, Sq, Sk, D, seed=63, outliers=(1e-6, 2.0), rope=orc.rope_tables(max(Sq, Sk), 10000.0, D), **kw)


def test_bf16_dkdv_pipeline_ends_many_heads_a_group(gpu_device):
    """The same at head_dim 64, whose laid-out loop takes streams of 48 tiles and more: one tile of every head, its second block of one
    query; a second key tile of one row (outliers: as above).  More such ends stand with the single batches below: where 24
    heads of a group add up, the bf16 roundings of P and dS (2^-9 each, some thousand of them) pass the elementwise
    bound against float64 in either form of the loop."""
    B, H, Hkv, Sq, Sk = 3, 86 * 48, 86, 33, 129
    assert B * Hkv * (-(-Sk // 128)) > 512 and H // Hkv * (-(-Sq // 64)) >= 48
    _case(gpu_device, BF16, B, H, Hkv, Sq, Sk, 64, seed=67, outliers=(1e-6, 2.0), rope=orc.rope_tables(max(Sq, Sk), 10000.0, 64), q_start=96)


@pytest.mark.parametrize("use_rope", [False, True])
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,kw", [
    (2, 66, 22, 60, 40, {"causal": False}),      # one streamed tile, its second block of eight keys
    (2, 66, 66, 20, 129, {"q_start": 109}),      # three, the last of one key
    (3, 46, 23, 33, 33, {}),                     # the second row wave has one row, the others none
    (2, 33, 33, 150, 150, {}),                   # two query tiles, the second of 22 rows
    (2, 33, 33, 256, 330, {"q_start": 74}),      # waves that need one block of their last tile, or none of it
])
def test_bf16_dq_pipeline_ends(gpu_device, B, H, Hkv, Sq, Sk, kw, use_rope):
    """dQ at head_dim 128 with 128-row workgroups, whose pipeline runs two blocks ahead of itself and requests a tile in every
    iteration, at the shortest streams and at ragged ends (outliers: as for dK/dV above)."""
    assert B * H * (-(-Sq // 128)) > 128
    if use_rope:
        kw = dict(kw, rope=orc.rope_tables(max(Sq, Sk), 10000.0, 128))
    _case(gpu_device, BF16, B, H, Hkv, Sq, Sk, 128, seed=64, outliers=(1e-6, 2.0), **kw)


@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,kw,extras,use_rope", [
    (11, 18, 6, 999, 999, {}, True, True),                   # dK/dV pipelined at its shortest stream (48 tiles), dQ not
    (9, 12, 4, 1030, 2050, {"q_start": 1020}, False, True),  # both, queries at the end of the keys
    (6, 18, 6, 2017, 2017, {}, True, False),                 # both, ragged
    (5, 24, 6, 777, 2300, {"causal": False}, False, False),  # both, no mask but the ends
    (4, 24 * 43, 43, 66, 257, {}, False, True),              # dK/dV: 24 short heads, the last tile of two queries; the third key tile sees no query
    (3, 48 * 58, 58, 60, 300, {"q_start": 240}, True, True), # 48 heads of one tile; a third key tile that only sees its last block
])
def test_bf16_backward_pipelines_against_single_batches(gpu_device, B, H, Hkv, Sq, Sk, kw, extras, use_rope):
    """head_dim 64: a launch long and large enough for the backward loops that are laid out instruction by instruction, against
    its batches one by one, whose launches take the compiler's loops.  Scores, P and dS are the same bits; dK, dV and T are
    fp32 sums of them in another order (at most 7000 terms: 7000 x 2^-24 of their magnitudes' sum), rounded to bf16 once: equal but
    for roundings that fall the other way, one unit in the last place (2^-7 of a value's power of two) each, and few of them."""
    assert B * Hkv * (-(-Sk // 128)) > 512 and H // Hkv * (-(-Sq // 64)) >= 48
    x = gen(B, H, Hkv, Sq, Sk, 64, BF16, extras=extras, seed=65)
    if use_rope:
        kw = dict(kw, rope=orc.rope_tables(max(Sq, Sk), 10000.0, 64))
    got = run_gpu(x, gpu_device, **kw)
    per_batch = [n for n in ("q", "k", "v", "d_o", "v_first", "gate_logits") if x.get(n) is not None]
    for i in (0, B - 1):
        one = run_gpu(dict(x, **{n: x[n][i:i + 1] for n in per_batch}), gpu_device, **kw)
        for n in ("dq", "dk", "dv") + (("dv_first", "dgate_logits") if extras else ()):
            a, b = got[n][i].float(), one[n][0].float()
            scale = torch.maximum(b.abs(), b.square().mean().sqrt())
            assert ((a - b).abs() <= 2.0 ** -7 * scale).all(), (n, float(((a - b).abs() / scale).max()))
            assert (a - b).norm() <= 1e-3 * b.norm(), (n, float((a - b).norm() / b.norm()))


@pytest.mark.parametrize("option", ["gated copy", "rows switched off", "no norm"])
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D,q_start", [(9, 12, 4, 1030, 2050, 64, 1020), (9, 8, 4, 1000, 1000, 128, 0)])
def test_bf16_backward_pipelines_options_against_single_batches(gpu_device, B, H, Hkv, Sq, Sk, D, q_start, option):
    """The laid-out loops on what else they stream: a copy of the gradient that the dQ kernel writes (gate scale not positive), rows whose
    gate factor vanishes (their -lse is -inf), scores of any size (no normaliser).  Against single batches, with the bounds
    of the test above."""
    assert B * Hkv * (-(-Sk // 128)) > 512 // (D // 64) and B * H * (-(-Sq // 128)) > 384
    x = gen(B, H, Hkv, Sq, Sk, D, BF16, extras=option != "no norm", seed=68)
    kw = {"q_start": q_start, "rope": orc.rope_tables(Sk, 10000.0, D)}
    if option == "gated copy": kw["gate_scale"] = -1.5
    if option == "rows switched off": x["gate_logits"][:, ::3] = -200.0
    if option == "no norm": kw["qk_norm"] = False
    got = run_gpu(x, gpu_device, **kw)
    per_batch = [n for n in ("q", "k", "v", "d_o", "v_first", "gate_logits") if x.get(n) is not None]
    for i in (0, B - 1):
        one = run_gpu(dict(x, **{n: x[n][i:i + 1] for n in per_batch}), gpu_device, **kw)
        for n in ("dq", "dk", "dv") + (("dv_first", "dgate_logits") if "gate_logits" in per_batch else ()):
            a, b = got[n][i].float(), one[n][0].float()
            scale = torch.maximum(b.abs(), b.square().mean().sqrt())
            assert ((a - b).abs() <= 2.0 ** -7 * scale).all(), (n, float(((a - b).abs() / scale).max()))
            assert (a - b).norm() <= 1e-3 * b.norm(), (n, float((a - b).norm() / b.norm()))


@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D,q_start,gate_scale,layout", [
    (9, 12, 4, 1030, 2050, 64, 1020, None, "b seq head d"),  # dQ and dK/dV
    (9, 12, 4, 1030, 2050, 64, 1020, -1.5, "b seq head d"),  # ... which streams a copy of the gradient
    (43, 96, 6, 190, 190, 64, 0, None, "b seq head d"),      # dK/dV, short heads
    (43, 96, 6, 190, 190, 64, 0, None, "rows far apart"),
    (30, 8, 4, 300, 300, 128, 0, None, "b seq head d"),
    (30, 8, 4, 300, 300, 128, 0, None, "rows far apart"),
    (30, 8, 4, 300, 300, 128, 0, -1.5, "rows far apart"),
])
def test_bf16_backward_pipelines_with_strided_operands(gpu_device, B, H, Hkv, Sq, Sk, D, q_start, gate_scale, layout):
    """The laid-out loops walk the heads and tiles of a gradient, and the tiles of v, that have strides of their own: the same bits
    as with contiguous ones.  Far apart: the largest row stride that is accepted (3 to 5 GB an operand)."""
    assert B * Hkv * (-(-Sk // 128)) > 512 // (D // 64) and (D == 128 or H // Hkv * (-(-Sq // 64)) >= 48)
    far = 2**23 - 8
    x = gen(B, H, Hkv, Sq, Sk, D, BF16, extras=gate_scale is not None, seed=69)
    x = {n: t.to(gpu_device) for n, t in x.items() if t is not None}
    kw = {"q_start": q_start}
    if gate_scale is not None:
        kw.update(gate_scale=gate_scale, gate_logits=x["gate_logits"])

    def placed(t):
        b, h, s, d = t.shape
        if layout == "b seq head d":
            return t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
        out = torch.empty(s * far, dtype=t.dtype, device=t.device).as_strided((b, h, s, d), (h * d, d, far, 1))
        return out.copy_(t)

    def grads(place):
        q, k = x["q"].clone().requires_grad_(), x["k"].clone().requires_grad_()
        v = place(x["v"]).requires_grad_()
        y = qknorm_attention(q, k, v, x["g_q"], x["g_k"], **kw)
        return torch.autograd.grad(y, [q, k, v], place(x["d_o"]))

    for n, a, b in zip(("dq", "dk", "dv"), grads(placed), grads(lambda t: t)):
        assert torch.equal(a, b), n
    torch.cuda.empty_cache()


@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D,q_start", [
    (11, 18, 6, 999, 999, 64, 0),        # launches that take the laid-out dK/dV loop
    (9, 12, 4, 1030, 2050, 64, 1020),    # ... the diagonal off the tiles' edges
    (9, 8, 4, 1000, 1000, 128, 0),
    (8, 8, 4, 500, 1100, 128, 600),
    (4, 18, 6, 999, 999, 64, 0),         # ... and the compiler's
])
def test_bf16_non_finite_rows_stay_with_the_keys_they_see(gpu_device, B, H, Hkv, Sq, Sk, D, q_start):
    """One query row of every batch with a gradient or a query that is not finite: dk and dv of the keys behind the 32-key block in
    which the row's 32-query block ends are the same bits as without it, as are the other heads' and dq's other rows."""
    x = gen(B, H, Hkv, Sq, Sk, D, BF16, seed=66)
    bad = {n: x[n].clone() for n in ("q", "d_o")}
    rows = [(5, 40, 70, 100, 127, 128, 300, 400)[b % 8] for b in range(B)]
    for b, i in enumerate(rows):
        if b % 2: bad["q"][b, b % H, i] = math.nan
        else: bad["d_o"][b, b % H, i] = math.inf
    ref, got = (run_gpu(t, gpu_device, q_start=q_start) for t in (x, dict(x, **bad)))
    for b, i in enumerate(rows):
        h, g = b % H, b % H // (H // Hkv)
        first = 32 * ((i // 32 * 32 + 31 + q_start) // 32) + 32  # first key that must not notice
        for n in ("dk", "dv"):
            assert not got[n][b, g, : i + q_start + 1].float().isfinite().any(-1).any(), (n, b)
            assert torch.equal(got[n][b, g, first:], ref[n][b, g, first:]), (n, b, i)
            others = [o for o in range(Hkv) if o != g]
            assert torch.equal(got[n][b, others], ref[n][b, others]), (n, b)
        keep = torch.ones(H, Sq, dtype=torch.bool)
        keep[h, i] = False
        assert torch.equal(got["dq"][b][keep], ref["dq"][b][keep]), b


@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D,kw,gen_kw,use_rope", [
    (1, 2, 1, 65, 65, 64, {}, {"extras": True}, True),                         # one row in the last workgroup, its second wave beyond the end
    (1, 2, 2, 31, 130, 64, {"q_start": 99}, {"extras": True}, False),          # fewer rows than one wave owns
    (2, 2, 1, 97, 33, 64, {"causal": False}, {}, True),                        # the second wave of a pair has one key
    (1, 1, 1, 70, 20, 128, {"causal": False}, {"extras": True}, True),         # ... or none
    (2, 3, 1, 129, 229, 128, {"q_start": 100}, {"extras": True}, False),
    # the launches with thousands of rows at head_dim 128 go without a gate: its gradient (1 - sigma) sum_d y dy sees the
    # bf16 rounding of y, rms 2^-9 / sqrt(3) sqrt(128) |y| |dy| = 0.013 for a row of one key, and 16128 such rows reach 4 rms
    (3, 42, 42, 128, 130, 128, {"q_start": 2}, {}, True),                      # 126 workgroups of 128 rows: the last shape below the line
    (3, 43, 43, 130, 100, 128, {"causal": False}, {}, True),                   # 258: above it
    (4, 97, 97, 65, 70, 64, {"q_start": 5}, {"extras": True}, True),           # 388: forward and dQ above it
])
def test_bf16_forward_and_dq_workgroup_shapes(gpu_device, B, H, Hkv, Sq, Sk, D, kw, gen_kw, use_rope):
    """Forward and dQ with 64-row workgroups whose waves split the key blocks of a tile (launches that do not fill the
    card) and with 128-row ones, at the ragged ends of both."""
    if use_rope:
        kw = dict(kw, rope=orc.rope_tables(max(Sq, Sk), 10000.0, D))
    _case(gpu_device, BF16, B, H, Hkv, Sq, Sk, D, seed=62, gen_kw=gen_kw, **kw)


@pytest.mark.parametrize("D,gain", [(64, 7.0), (128, 5.0)])
def test_bf16_forward_parts_with_scales_beyond_the_bound(gpu_device, D, gain):
    """Scale vectors too large for the fixed softmax reference (known on the device only): the two waves of a pair then keep a
    running one each, and the early rows' second wave sees no key at all.  y against the float64 model that rounds where the
    kernels do, at the ordinary tolerance; lse against the launch whose waves each see all keys: a row sum adds bf16 probabilities
    (8 significant bits), each rounded by up to 2^-8 of itself against either launch's own reference, 2^-7 between the two."""
    import tests.parity_util as pu
    from sample_efficient_gpt_amd import _lib
    from sample_efficient_gpt_amd.plan import AttnPlan

    x = gen(1, 2, 1, 150, 150, D, BF16, seed=63)
    x["g_q"] = x["g_q"] * gain
    assert float((x["g_q"] * x["g_k"]).abs().max()) * D**0.5 * 1.4427 * 1.02 > 64.0
    flat = lambda t, r=1: t.repeat_interleave(r, dim=1).flatten(0, 1)
    model = pu.kernel_rounding_model(flat(x["q"]), flat(x["k"], 2), flat(x["v"], 2), x["g_q"].double() * x["g_k"].double(), flat(x["d_o"]),
                                     eps=1e-6, sm_scale=D**-0.5, causal=True, q_start=0)["y"]
    plan = AttnPlan({n: (t.to(gpu_device) if t is not None else None) for n, t in x.items()}, backward=False)
    print(f"scales beyond the bound, D={D}", flush=True)
    plan.forward()
    parts = {"y": plan.y.cpu(), "lse": plan.lse.cpu()}
    plan.forward(flags=_lib.SEGPT_FLAG_RUNNING_MAX)  # always 128-row workgroups
    whole = {"y": plan.y.cpu(), "lse": plan.lse.cpu()}
    for got in (parts, whole):
        err = (got["y"].double().flatten(0, 1) - model).abs()
        assert bool((err <= 2e-2 + 1e-2 * model.abs()).all()), float(err.max())
    assert not torch.equal(parts["lse"], whole["lse"])  # two different launches
    assert (parts["lse"] - whole["lse"]).abs().max() < 2.0**-7


def test_bf16_gate_scale_not_positive_takes_the_gated_copy(gpu_device):
    """A gate scale <= 0 has no logarithm: the dQ kernel then leaves a gate-scaled copy of dO for the dK/dV kernel
    (the workspace grows by that tensor)."""
    from sample_efficient_gpt_amd import _lib
    from sample_efficient_gpt_amd.function import _fill_common
    x = gen(1, 4, 2, 200, 200, 64, BF16, extras=True, seed=6)
    _case(gpu_device, BF16, 1, 4, 2, 200, 200, 64, gate_scale=-1.5, _x=x)
    _case(gpu_device, BF16, 1, 4, 2, 200, 200, 64, gate_scale=0.0, _x=x)
    lib = _lib.load()
    sizes = {}
    for gs in (2.0, -1.5):
        p = _lib.new_params()
        t = {n: x[n] for n in ("q", "k", "v", "v_first", "gate_logits")}
        y = torch.empty_like(t["q"])
        lse = torch.empty(t["q"].shape[:3], dtype=torch.float32)
        _fill_common(p, t["q"], t["k"], t["v"], y, lse, x["g_q"].float(), x["g_k"].float(), t["v_first"], x["vr_coef"].float(),
                     t["gate_logits"], gs, 1e-6, 0.125, True, 0)
        sizes[gs] = lib.segpt_attn_workspace_bytes(p, _lib.SEGPT_WS_BWD)
    assert sizes[-1.5] - sizes[2.0] == 1 * 4 * 200 * 64 * 2 + (-(1 * 4 * 200 * 64 * 2) % 256), sizes


def _slice_inputs(c, x, b, g):
    rep = c.H // c.Hkv
    hs = slice(g * rep, (g + 1) * rep)
    xs = {"q": x["q"][b:b + 1, hs], "k": x["k"][b:b + 1, g:g + 1], "v": x["v"][b:b + 1, g:g + 1],
          "d_o": x["d_o"][b:b + 1, hs], "g_q": x["g_q"], "g_k": x["g_k"]}
    if c.extras:
        xs.update(gate_logits=x["gate_logits"][b:b + 1, :, hs], v_first=x["v_first"][b:b + 1, g:g + 1], vr_coef=x["vr_coef"])
    return xs, hs


REDUCED_GRADS = ("dg_q", "dg_k", "dvr_coef")


def _slice_check(device, c, pairs, odtype=torch.float64):
    """Full-size run on the GPU; oracle on single (batch, kv-group) slices (they are independent units).
    Tensors: the full run's slice against the oracle's.  Parameter gradients that sum over every row
    (dg_q, dg_k, dvr_coef): (i) a GPU run on the slice alone against the oracle's slice result, (ii) the full run's
    value against the sum of GPU runs over ALL (batch, kv-group) slices (the reduction is additive over them), so
    that a wrong partial, a dropped workgroup or a wrong second-stage reduce at full size fails."""
    x = make_inputs(c)
    kw = dict(eps=c.eps, sm_scale=c.sm_scale)
    if c.extras:
        kw["gate_scale"] = c.gate_scale
    print(f"full-size {c.name}", flush=True)
    got = run_gpu(x, device, backward=c.backward, **kw)
    worst = {}
    for b, g in pairs:
        xs, hs = _slice_inputs(c, x, b, g)
        ref = run_oracle(xs, backward=c.backward, odtype=odtype, **kw)
        gs = {"y": got["y"][b:b + 1, hs], "lse": got["lse"][b:b + 1, hs]}
        names = ["y", "lse"]
        if c.backward:
            gs.update(dq=got["dq"][b:b + 1, hs], dk=got["dk"][b:b + 1, g:g + 1], dv=got["dv"][b:b + 1, g:g + 1])
            names += ["dq", "dk", "dv"]
            if c.extras:
                gs.update(dv_first=got["dv_first"][b:b + 1, g:g + 1], dgate_logits=got["dgate_logits"][b:b + 1, :, hs])
                names += ["dv_first", "dgate_logits"]
        errs = compare(gs, ref, c.dtype, names=names, label=f"{c.name}[b={b},g={g}] ")
        if c.backward:  # (i) the summed parameter gradients of this slice, GPU alone on the slice vs the oracle
            alone = run_gpu(xs, device, **kw)
            red = [n for n in REDUCED_GRADS if n in ref]
            scales = value_residual_scale(xs, ref) if c.extras else None
            errs.update(compare(alone, ref, c.dtype, names=red, label=f"{c.name}[b={b},g={g}] slice alone ", scales=scales))
        for n, e in errs.items():
            worst[n] = max(worst.get(n, 0.0), e)
    print(c.name, "worst max-abs errors over slices:", {k: f"{v:.2e}" for k, v in worst.items()}, flush=True)
    if c.backward:  # (ii) additivity over every (batch, kv-group) slice
        red = [n for n in REDUCED_GRADS if n in got]
        acc = {n: torch.zeros_like(got[n], dtype=torch.float64) for n in red}
        mag = {n: torch.zeros_like(got[n], dtype=torch.float64) for n in red}
        for b in range(c.B):
            for g in range(c.Hkv):
                part = run_gpu(_slice_inputs(c, x, b, g)[0], device, **kw)
                for n in red:
                    acc[n] += part[n].double()
                    mag[n] += part[n].double().abs()
        for n in red:
            # both sides are fp32 sums of the same per-workgroup partials in different orders: only fp32 summation
            # noise separates them (1e-4 of the summed magnitudes is ~100x that noise and ~100x below the bf16 budget)
            err = (got[n].double() - acc[n]).abs()
            assert bool((err <= 1e-5 + 1e-4 * mag[n]).all()), f"{c.name} {n}: full run {got[n]} vs sum of slices {acc[n]}"
            print(f"{c.name} {n}: full run vs sum over {c.B * c.Hkv} slices, max abs diff {float(err.max()):.3e}", flush=True)
    return x, got, kw


def test_cfg2_imu1_forward_full_size(gpu_device):
    _slice_check(gpu_device, CONFIGS[2], [(0, 0), (7, 5), (3, 2)])


def test_cfg3_imu1_fwd_bwd_full_size(gpu_device):
    _slice_check(gpu_device, CONFIGS[3], [(0, 0), (7, 5)])


@pytest.mark.parametrize("cfg", [3, 4, 5])
def test_full_size_exact_properties(gpu_device, cfg):
    """Size-independent properties at the full benchmark shapes (IMU-1; S=8192 with gate and value residual;
    head_dim 128), all bit-exact: (1) scaling v (and v_first) or dO by a power of two scales what is linear in
    them and leaves the rest alone; (2) causality: changing tokens >= t leaves the outputs and dq of rows < t
    alone, changing queries / dO of rows < t leaves dk, dv of rows >= t alone; (3) the batch entries are
    independent: reversing the batch reverses the results."""
    c = CONFIGS[cfg]
    x = make_inputs(c)
    kw = dict(eps=c.eps, sm_scale=c.sm_scale)
    if c.extras:
        kw["gate_scale"] = c.gate_scale
    print(f"cfg{cfg} exact properties", flush=True)
    base = run_gpu(x, gpu_device, **kw)
    per_token = ["q", "k", "v", "d_o"] + (["v_first"] if c.extras else [])
    dvs = ["dv"] + (["dv_first"] if c.extras else [])

    def eq(a, b):
        a, b = a.float(), b.float()
        if torch.equal(a, b):
            return True
        idx = (a != b).nonzero()  # say where, before the assertion fires
        print(f"  mismatch: {idx.shape[0]} of {a.numel()} elements, first {idx[0].tolist()} last {idx[-1].tolist()}, "
              f"max |diff| {float((a - b).abs().max()):.3e}", flush=True)
        return False

    # (1a) v, v_first -> 2 v, 2 v_first
    x2 = dict(x, v=x["v"] * 2)
    if c.extras:
        x2["v_first"] = x["v_first"] * 2
    got = run_gpu(x2, gpu_device, **kw)
    assert eq(got["y"], base["y"] * 2) and eq(got["lse"], base["lse"])
    assert eq(got["dq"], base["dq"] * 2) and eq(got["dk"], base["dk"] * 2)
    for n in dvs:
        assert eq(got[n], base[n]), n
    assert eq(got["dg_q"], base["dg_q"] * 2)
    # (1b) dO -> dO / 4
    got = run_gpu(dict(x, d_o=x["d_o"] * 0.25), gpu_device, **kw)
    assert eq(got["y"], base["y"])
    for n in ["dq", "dk", "dg_q", "dg_k"] + dvs + (["dgate_logits", "dvr_coef"] if c.extras else []):
        assert eq(got[n], base[n] * 0.25), n
    # (2a) new q, k, v, dO (and gate logits) from token t on
    t = c.S // 2 + 87
    g = torch.Generator().manual_seed(77)
    xp = dict(x)
    for n in per_token:
        xp[n] = x[n].clone()
        xp[n][:, :, t:] = torch.randn(x[n][:, :, t:].shape, generator=g).to(x[n].dtype)
    if c.extras:
        xp["gate_logits"] = x["gate_logits"].clone()
        xp["gate_logits"][:, t:] = torch.randn(x["gate_logits"][:, t:].shape, generator=g).to(x["gate_logits"].dtype)
    got = run_gpu(xp, gpu_device, **kw)
    for n in ("y", "lse", "dq"):
        assert eq(got[n][:, :, :t], base[n][:, :, :t]), n
        assert not torch.equal(got[n][:, :, t:], base[n][:, :, t:]), n
    # (2b) new q, dO before token t
    xp = dict(x)
    for n in ("q", "d_o"):
        xp[n] = x[n].clone()
        xp[n][:, :, :t] = torch.randn(x[n][:, :, :t].shape, generator=g).to(x[n].dtype)
    got = run_gpu(xp, gpu_device, **kw)
    for n in ["dk"] + dvs:
        assert eq(got[n][:, :, t:], base[n][:, :, t:]), n
        assert not torch.equal(got[n][:, :, :t], base[n][:, :, :t]), n
    # (3) reversed batch
    flipped = {n: (v.flip(0) if n in per_token + ["gate_logits"] else v) for n, v in x.items()}
    got = run_gpu(flipped, gpu_device, **kw)
    for n in ["y", "lse", "dq", "dk"] + dvs:
        assert eq(got[n].flip(0), base[n]), n
    assert torch.allclose(got["dg_q"], base["dg_q"], atol=2e-2, rtol=1e-2)


def test_cfg4_long_context_extras_full_size(gpu_device):
    # both batches, the first and a later kv group
    _slice_check(gpu_device, CONFIGS[4], [(0, 0), (1, 3)], odtype=torch.float32)


def test_cfg5_wide_head_full_size(gpu_device):
    _slice_check(gpu_device, CONFIGS[5], [(0, 0), (3, 3)])


def test_running_maximum_path(gpu_device):
    """The forward has two softmax paths: raw exp2 when the QK-norm bound on the logits allows it, and a lazily
    raised running maximum otherwise.  (a) Forced onto the second path, ordinary inputs must meet the same
    tolerance against the oracle and agree with the first path; (b) gains large enough to leave the bound
    (sm_scale*log2e*D*max|g|*1.02 ~ 68 > 64) select it by themselves."""
    from sample_efficient_gpt_amd import _lib
    from sample_efficient_gpt_amd.plan import AttnPlan

    x = gen(2, 4, 2, 320, 320, 64, BF16, seed=11)
    ref = run_oracle(x, backward=False)
    plan = AttnPlan({n: (t.to(gpu_device) if t is not None else None) for n, t in x.items()}, backward=False)
    print("forced running-maximum path", flush=True)
    plan.forward()
    fast = {"y": plan.y.cpu(), "lse": plan.lse.cpu()}
    plan.forward(flags=_lib.SEGPT_FLAG_RUNNING_MAX)
    slow = {"y": plan.y.cpu(), "lse": plan.lse.cpu()}
    compare(fast, ref, BF16)
    compare(slow, ref, BF16)
    assert torch.allclose(fast["y"].float(), slow["y"].float(), atol=4e-3, rtol=8e-3)  # one bf16 ulp of each other
    # the row sum adds bf16-rounded probabilities, which round differently under a shifted reference point
    assert torch.allclose(fast["lse"], slow["lse"], atol=4e-3, rtol=0)

    x["g_q"] = x["g_q"] * 2.4
    x["g_k"] = x["g_k"] * 2.4
    assert float((x["g_q"] * x["g_k"]).abs().max()) * 0.125 * 1.4427 * 64 * 1.02 > 64.0
    print("large-gain case", flush=True)
    got = run_gpu(x, gpu_device, backward=False)
    ref = run_oracle(x, backward=False)
    # the bf16 rounding of Qhat and Khat perturbs a logit in proportion to the gain product (5.8x the ordinary
    # case here), and P = exp(logit) inherits it: the absolute part of the tolerance is scaled accordingly
    _fp32_proof(gpu_device, x, ref, {}, backward=False)  # the fp32 kernels meet 1e-5 on these inputs: the slack below is rounding
    err = (got["y"].double() - ref["y"]).abs()
    assert bool((err <= 5.8 * 2e-2 + 1e-2 * ref["y"].abs()).all()), float(err.max())
    # the same claim made precise: against the float64 model that rounds Qhat, Khat and P where the kernels do, the
    # output meets the ORDINARY tolerance (the model with the roundings switched off is the oracle)
    import tests.parity_util as pu

    rep = x["q"].shape[1] // x["k"].shape[1]
    flat = lambda t, r=1: t.repeat_interleave(r, dim=1).flatten(0, 1)
    margs = (flat(x["q"]), flat(x["k"], rep), flat(x["v"], rep), x["g_q"].double() * x["g_k"].double(), torch.zeros_like(flat(x["q"])))
    mkw = dict(eps=1e-6, sm_scale=0.125, causal=True, q_start=0)
    keep = pu.bf16_round
    try:
        pu.bf16_round = lambda t: t
        exact_y = pu.kernel_rounding_model(*margs, **mkw)["y"]
    finally:
        pu.bf16_round = keep
    assert float((exact_y - ref["y"].flatten(0, 1)).abs().max()) <= 1e-9
    model_y = pu.kernel_rounding_model(*margs, **mkw)["y"]
    err_m = (got["y"].double().flatten(0, 1) - model_y).abs()
    print(f"  large gain: max abs err {float(err.max()):.2e} vs the oracle, {float(err_m.max()):.2e} vs the rounding model", flush=True)
    assert bool((err_m <= 2e-2 + 1e-2 * model_y.abs()).all()), float(err_m.max())
    assert torch.allclose(got["lse"].double(), ref["lse"], atol=5.8 * 2e-2, rtol=1e-2)


def test_plan_reuses_forward_kv_workspace_and_stages_match(gpu_device):
    """C-ABI plan: backward with SEGPT_FLAG_KV_PREPARED (forward's normalised keys) == backward that runs its
    own pre-pass == the stage-by-stage entry points, bit for bit; a forward without a kv workspace is refused."""
    from sample_efficient_gpt_amd import _lib
    from sample_efficient_gpt_amd.plan import AttnPlan

    x = gen(2, 6, 2, 300, 300, 64, BF16, extras=True, seed=5)
    xd = {n: (t.to(gpu_device) if t is not None else None) for n, t in x.items()}
    plan = AttnPlan(xd, gate_scale=2.0)
    outs = ("y", "lse", "dq", "dk", "dv", "dv_first", "dgate", "dg_q", "dg_k", "dcoef")
    snap = lambda: {n: getattr(plan, n).clone() for n in outs}
    plan.forward(); plan.backward(kv_prepared=True)
    a = snap()
    plan.kv_ws.zero_()  # a backward without the flag must rebuild the workspace itself
    plan.backward(kv_prepared=False)
    b = snap()
    plan.kv_ws.zero_()
    for n in outs:
        getattr(plan, n).zero_()
    for st in range(len(_lib.FWD_STAGES)):
        plan.forward_stage(st)
    for st in range(len(_lib.BWD_STAGES)):
        plan.backward_stage(st)
    c = snap()
    torch.cuda.synchronize()
    for n in outs:
        assert torch.equal(a[n], b[n]), n
        assert torch.equal(a[n], c[n]), n
    ref = run_oracle(x, gate_scale=2.0)
    compare({"y": a["y"].cpu(), "lse": a["lse"].cpu(), "dq": a["dq"].cpu(), "dk": a["dk"].cpu(), "dv": a["dv"].cpu()},
            ref, BF16, names=["y", "lse", "dq", "dk", "dv"])
    plan.p.kv_workspace = None
    with pytest.raises(_lib.SegptError):
        plan.forward()


def test_library_op_compiled_and_checkpointed_matches_eager(gpu_device):
    """torch.ops.segpt.qknorm_attention under torch.compile (aot_eager: the op stays one opaque node) and under
    non-reentrant activation checkpointing gives bit-identical outputs and gradients to the autograd Function."""
    from torch.utils.checkpoint import checkpoint

    from sample_efficient_gpt_amd import qknorm_attention_op

    x = gen(2, 6, 2, 160, 160, 64, BF16, extras=True, seed=21)
    names = ["q", "k", "v", "g_q", "g_k", "v_first", "vr_coef", "gate_logits"]

    def run(fn):
        t = {n: x[n].to(gpu_device).requires_grad_(True) for n in names}
        y = fn(t["q"], t["k"], t["v"], t["g_q"], t["g_k"], v_first=t["v_first"], vr_coef=t["vr_coef"], gate_logits=t["gate_logits"])
        y.backward(x["d_o"].to(gpu_device))
        return [y.detach()] + [t[n].grad for n in names]

    print("library op: eager / compiled / checkpointed", flush=True)
    ref = run(qknorm_attention)
    eager = run(qknorm_attention_op)
    compiled = run(torch.compile(qknorm_attention_op, backend="aot_eager", fullgraph=True))
    ckpt = run(lambda *a, **kw: checkpoint(qknorm_attention_op, *a, use_reentrant=False, **kw))
    torch.cuda.synchronize()
    for other in (eager, compiled, ckpt):
        for a, b in zip(ref, other):
            assert torch.equal(a, b)
    torch.library.opcheck(torch.ops.segpt.qknorm_attention,
                          tuple(x[n].to(gpu_device) for n in names) + (2.0, 1e-6, 0.125, True, 0, None, None, -1, 0, True, False, False),
                          test_utils=("test_schema", "test_faketensor"))
    # every optional operand absent: the backward op then returns several empty placeholders, which must be
    # distinct tensors (returns of a custom op may not alias one another)
    def run_min(fn):
        t = {n: x[n].to(gpu_device).requires_grad_(True) for n in ("q", "k", "v", "g_q")}
        y = fn(t["q"], t["k"], t["v"], t["g_q"], None)
        y.backward(x["d_o"].to(gpu_device))
        return [y.detach()] + [t[n].grad for n in ("q", "k", "v", "g_q")]

    for a, b in zip(run_min(qknorm_attention), run_min(qknorm_attention_op)):
        assert torch.equal(a, b)


def test_positional_dropin_functions_under_torch_compile(gpu_device):
    """The positional drop-ins (`QKNormFlashAttnFunc.apply`, `FlashAttnFunc.apply`) called from a compiled function:
    their `apply` records the caller's grad mode in Python, which the compiler may only run by breaking the graph
    around the call (no fullgraph here); outputs and gradients must equal the eager call bit for bit, for a call
    that is followed by a backward and for one under no_grad."""
    H, B, S, d = 4, 2, 136, 64
    g = torch.Generator().manual_seed(33)
    mk = lambda: torch.randn(H * B, S, d, generator=g).to(BF16).to(gpu_device)
    Q, K, V, dO = mk(), mk(), mk(), mk()
    gain = torch.full((1,), 1.1, device=gpu_device)

    def f_norm(q, k, v, gn):
        return QKNormFlashAttnFunc.apply(q * 1, k, v, gn, True, 0)

    def f_plain(q, k, v):
        return FlashAttnFunc.apply(q * 1, k, v, 0, True)

    def run(fn, *args):
        leaves = [a.detach().clone().requires_grad_(True) for a in args]
        y = fn(*leaves)
        y.backward(dO)
        return [y.detach()] + [l.grad for l in leaves]

    for fn, args in ((f_norm, (Q, K, V, gain)), (f_plain, (Q, K, V))):
        ref = run(fn, *args)
        got = run(torch.compile(fn, backend="aot_eager"), *args)
        for a, b in zip(ref, got):
            assert torch.equal(a, b)
        with torch.no_grad():
            assert torch.equal(fn(*args), torch.compile(fn, backend="aot_eager")(*args))
    # a nested apply leaves the outer call's decision in place
    QKNormFlashAttnFunc._tls.inference = True
    try:
        with torch.no_grad():
            FlashAttnFunc.apply(Q, K, V, 0, True)
        assert QKNormFlashAttnFunc._inference() is True
    finally:
        QKNormFlashAttnFunc._tls.inference = False


def test_native_node_on_other_threads_and_streams(gpu_device):
    """The op and its native autograd node from two Python threads, each on a stream of its own, with the backward run
    after a retained graph's first one: every result equals the default stream's bit for bit; lse takes no gradient and
    a library error in the forward is the package's exception class."""
    import threading

    from sample_efficient_gpt_amd import _lib

    x = gen(2, 6, 2, 160, 160, 64, BF16, extras=True, seed=51)
    names = ["q", "k", "v", "g_q", "g_k", "v_first", "vr_coef", "gate_logits"]

    def run(out, stream):
        with torch.cuda.stream(stream):
            t = {n: x[n].to(gpu_device).requires_grad_(True) for n in names}
            y = qknorm_attention(t["q"], t["k"], t["v"], t["g_q"], t["g_k"], v_first=t["v_first"], vr_coef=t["vr_coef"], gate_logits=t["gate_logits"])
            d_o = x["d_o"].to(gpu_device)
            first = torch.autograd.grad(y, [t[n] for n in names], d_o, retain_graph=True)
            again = torch.autograd.grad(y, [t[n] for n in names], d_o)
            out.extend([y.detach(), *first, *again])
        stream.synchronize()

    ref, a, b = [], [], []
    run(ref, torch.cuda.default_stream())
    threads = [threading.Thread(target=run, args=(o, torch.cuda.Stream())) for o in (a, b)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(a) == len(b) == len(ref) == 1 + 2 * len(names)
    for got in (a, b):
        for i, (r, g) in enumerate(zip(ref, got)):
            assert torch.equal(r, g), i
    q = x["q"].to(gpu_device).requires_grad_(True)
    k, v, g = (x[n].to(gpu_device) for n in ("k", "v", "g_q"))
    y, lse = qknorm_attention(q, k, v, g, return_lse=True)
    assert not lse.requires_grad and torch.autograd.grad((y * 0.0).sum() + q.sum() * 0.0, q)[0].abs().max() == 0
    with pytest.raises(_lib.SegptError):
        qknorm_attention(q[..., :32], k[..., :32], v[..., :32], torch.ones(1, device=gpu_device))


def test_native_node_keeps_what_python_callers_see(gpu_device):
    """What an autograd function in Python gives its callers holds for the native node: an undefined output gradient counts
    as zero, torch's exceptions and the package's own keep their types in both directions, what a saved-tensor hook
    raises reaches the caller, forward-mode tangents and function transforms are refused whether or not a gradient is
    recorded, and operand combinations that do not add up are refused before any launch."""
    import torch.autograd.forward_ad as fwAD
    from torch.utils._python_dispatch import TorchDispatchMode

    from sample_efficient_gpt_amd import _lib

    x = gen(1, 6, 2, 96, 96, 64, BF16, seed=52)
    dev = {n: x[n].to(gpu_device) for n in ("q", "k", "v", "g_q", "d_o")}
    call = lambda **kw: qknorm_attention(*(kw.get(n, dev[n]) for n in ("q", "k", "v", "g_q")))

    class Drops(torch.autograd.Function):
        @staticmethod
        def forward(ctx, t):
            return t.clone()

        @staticmethod
        def backward(ctx, g):
            return None

    q = dev["q"].clone().requires_grad_(True)
    g = torch.autograd.grad(Drops.apply(call(q=q)), q, dev["d_o"])[0]
    assert g.shape == q.shape and g.abs().max() == 0

    odd = torch.empty(q.numel() + 1, dtype=BF16, device=gpu_device)[1:].view(q.shape)  # rows that are not 16-byte aligned
    with pytest.raises(_lib.SegptError, match="segpt_attn_bwd"):
        torch.autograd.grad(call(q=q), q, odd)

    class Stop(Exception):
        pass

    def refuse(t):
        raise Stop("hook")

    with pytest.raises(Stop), torch.autograd.graph.saved_tensors_hooks(refuse, lambda t: t):
        call(q=q)

    for qq in (q, dev["q"]):
        with fwAD.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
            call(q=fwAD.make_dual(qq, torch.ones_like(qq)))
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda t: call(q=t))(dev["q"][None])

    seen = []

    class Look(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with torch.no_grad(), Look():
        y = qknorm_attention_op(dev["q"], dev["k"], dev["v"], dev["g_q"])
    assert torch.ops.segpt.qknorm_attention.default in seen and torch.equal(y, call())

    Q, K = (t.transpose(0, 1).reshape(-1, 96, 64).contiguous() for t in (dev["q"], dev["k"]))
    gate = torch.zeros(1, 96, 4, dtype=BF16, device=gpu_device)  # six rows are not a multiple of its four heads
    with pytest.raises((AssertionError, RuntimeError)):
        QKNormFlashAttnFunc.apply(Q, Q, Q, dev["g_q"], True, 0, None, None, None, gate)
    with pytest.raises((AssertionError, RuntimeError, ValueError, IndexError)):
        QKNormFlashAttnFunc.apply(Q[:2], K, K, dev["g_q"], True, 0, None, K[0], torch.ones(2, device=gpu_device), None, 2.0, 2)

    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(1e-4)
    try:
        with pytest.raises(torch.OutOfMemoryError), torch.no_grad():
            big = dev["q"].expand(400, -1, -1, -1)
            qknorm_attention(big, dev["k"].expand(400, -1, -1, -1), dev["v"].expand(400, -1, -1, -1), dev["g_q"])
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


def _traced_callers(x, device):
    """name -> (operands of a layout from a generated case, caller of three tensors)"""
    g = x["g_q"].to(device)
    rope = dict(zip(("rope_cos", "rope_sin"), (t.float().to(device) for t in orc.rope_tables(x["k"].shape[2], 10000.0, x["q"].shape[3]))))
    gate = x["gate_logits"].to(device)
    canon = lambda s: [s[n].to(device) for n in ("q", "k", "v")]
    flat = lambda s: [s[n].transpose(0, 1).reshape(-1, *s[n].shape[2:]).contiguous().to(device) for n in ("q", "k", "v")]
    Hkv = x["k"].shape[1]

    def cached(q, k, v):
        keys, values = KVCache().append(k, v)
        return qknorm_attention(q, keys, values, g)

    return {
        "function": (canon, lambda q, k, v: qknorm_attention(q, k, v, g, gate_logits=gate, out_bshd=True, **rope)),
        "operator": (canon, lambda q, k, v: qknorm_attention_op(q, k, v, g, **rope)),
        "cache": (canon, cached),
        "flat": (flat, lambda q, k, v: QKNormFlashAttnFunc.apply(q, k, v, g, True, 0, None, None, None, gate, 2.0, Hkv)),
        "reference formula": (flat, lambda q, k, v: TritonFlashAttnQKNormFunc.apply(q, k, v, g, True, 0, None, None, None, None, 2.0, Hkv)),
        "plain": (flat, lambda q, k, v: FlashAttnFunc.apply(q, k, v, 0, True, Hkv)),
    }


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("name", ["function", "operator", "cache", "flat", "reference formula", "plain"])
@pytest.mark.filterwarnings("ignore")
def test_traced_callers_compute_when_replayed(gpu_device, name, grad):
    """torch.jit.trace records operators, so what it records has to be one: a trace taken on one set of inputs gives the eager
    result on another."""
    a, b = (gen(2, 4, 2, 40, 40, 64, BF16, seed=s, extras=True) for s in (3, 4))
    layout, caller = _traced_callers(a, gpu_device)[name]
    first, second = ([t.requires_grad_(grad) for t in layout(x)] for x in (a, b))
    traced = torch.jit.trace(caller, tuple(first), check_trace=False)
    assert torch.equal(traced(*second), caller(*second))
    if grad and name != "cache":
        d = torch.randn_like(caller(*second))
        for got, want in zip(torch.autograd.grad(traced(*second), second, d), torch.autograd.grad(caller(*second), second, d)):
            assert torch.equal(got, want)


@pytest.mark.parametrize("caller", [qknorm_attention_op, qknorm_attention])
def test_rotary_tables_are_saved_variables(gpu_device, caller):
    """Tables written in place between forward and backward would give the gradients of another function: the backward
    notices, as for every other operand, and tables pass through saved-tensor hooks."""
    x = gen(1, 2, 1, 33, 33, 64, BF16, seed=5)
    q, k, v, g, d_o = (x[n].to(gpu_device) for n in ("q", "k", "v", "g_q", "d_o"))
    q.requires_grad_(True)
    for dtype in (F32, torch.float64):  # fp64 tables are converted for the kernels; the caller's are what is watched
        cos, sin = (t.to(gpu_device, dtype) for t in orc.rope_tables(33, 10000.0, 64))
        y = caller(q, k, v, g, rope_cos=cos, rope_sin=sin)
        ref, = torch.autograd.grad(y, q, d_o, retain_graph=True)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(gpu_device)):
            moved = caller(q, k, v, g, rope_cos=cos, rope_sin=sin)
        assert torch.equal(torch.autograd.grad(moved, q, d_o)[0], ref)
        sin.mul_(0.5)
        with pytest.raises(RuntimeError, match="inplace"):
            torch.autograd.grad(y, q, d_o)


@pytest.mark.parametrize("caller", [qknorm_attention_op, qknorm_attention])
def test_second_derivatives_are_refused(gpu_device, caller):
    """First derivatives with create_graph=True are the ordinary ones; going back through them raises instead of leaving the
    attention's terms out of a gradient penalty."""
    x = gen(1, 2, 1, 33, 33, 64, BF16, seed=5)
    q, k, v, g, d_o = (x[n].to(gpu_device) for n in ("q", "k", "v", "g_q", "d_o"))
    wrt = [t.requires_grad_(True) for t in (q, v, g)]
    plain = torch.autograd.grad(caller(q, k, v, g), wrt, d_o)
    first = torch.autograd.grad(caller(q, k, v, g), wrt, d_o, create_graph=True)
    for a, b in zip(plain, first):
        assert torch.equal(a, b) and not a.requires_grad
    for d in first:
        with pytest.raises(RuntimeError, match="derivative|autograd formula"):
            (d.float().pow(2).sum() + q.float().pow(2).sum()).backward(retain_graph=True)
        with pytest.raises(RuntimeError, match="derivative|autograd formula"):
            torch.autograd.grad(d.float().sum(), q, retain_graph=True, allow_unused=True)
    only_dy = d_o.clone().requires_grad_(True)  # linear in dy, but that is a derivative too
    first, = torch.autograd.grad(caller(q, k, v, g), q, only_dy, create_graph=True)
    with pytest.raises(RuntimeError, match="derivative|autograd formula"):
        torch.autograd.grad(first.float().sum(), only_dy)


# ------------------------------------------------------------------ rotary embedding fused into the loads


@pytest.mark.parametrize(
    "B,H,Hkv,Sq,Sk,D,kw,gen_kw",
    [
        (2, 6, 2, 300, 300, 64, {}, {}),
        (1, 4, 2, 200, 200, 64, {"gate_scale": 2.0}, {"extras": True, "scalar_gain": True}),
        (1, 4, 1, 160, 160, 128, {}, {}),
        (1, 3, 3, 72, 200, 64, {"q_start": 128}, {}),                      # queries at positions 128.. (attention.py:191-195)
        (1, 2, 1, 96, 96, 64, {"rope_q_pos0": 40, "rope_k_pos0": 40}, {}),  # explicit positions
        (1, 2, 2, 80, 140, 64, {"causal": False}, {}),
        # the dQ kernel's two-phase start-up with one, two and three key tiles in all (its second phase requests up to
        # three), and a last query block of 5 rows (the staged table blocks repeat the last row)
        (2, 2, 1, 40, 40, 64, {"gate_scale": 2.0}, {"extras": True}),
        (1, 4, 2, 100, 100, 64, {}, {}),
        (1, 2, 2, 133, 133, 64, {"gate_scale": 2.0}, {"extras": True}),
        (1, 4, 1, 333, 333, 128, {"gate_scale": 2.0}, {"extras": True}),
        # key tiles beyond every query (causal, fewer queries than keys, no offset): the dK/dV workgroups of those
        # tiles stream nothing and go straight to the epilogue's row blocks; their dk, dv are zero
        (1, 2, 1, 100, 400, 64, {"gate_scale": 2.0}, {"extras": True}),
        (1, 2, 1, 70, 300, 128, {}, {}),
    ],
)
def test_bf16_fused_rope(gpu_device, B, H, Hkv, Sq, Sk, D, kw, gen_kw):
    """q, k are the unrotated projections; the kernels rotate them in their loads (forward, pre-pass, dQ
    prologue) and rotate dq, dk back in their epilogues.  Oracle: rope.py's rotation, then the family forward,
    gradients by autograd (fp64)."""
    cos, sin = orc.rope_tables(512, 10000.0, D)
    _case(gpu_device, BF16, B, H, Hkv, Sq, Sk, D, gen_kw=gen_kw, seed=31, rope=(cos, sin), **kw)


@pytest.mark.parametrize("D", [64, 128])
def test_bf16_fused_rope_tables_of_exactly_the_needed_length(gpu_device, D):
    """Tables with exactly as many rows as there are positions (the staged table blocks of the last, partial query
    block must stay inside them), with positions offset into the tables for q."""
    Sq, Sk = 77, 205
    cos, sin = orc.rope_tables(Sk, 10000.0, D)
    _case(gpu_device, BF16, 1, 4, 2, Sq, Sk, D, gen_kw={"extras": True}, seed=33, rope=(cos, sin), gate_scale=2.0, q_start=Sk - Sq)


def test_fused_rope_equals_rotating_first_and_rejects_bad_tables(gpu_device):
    from sample_efficient_gpt_amd import _lib

    x = gen(1, 4, 2, 256, 256, 64, BF16, seed=33)
    cos, sin = orc.rope_tables(256, 10000.0, 64)
    fused = run_gpu(x, gpu_device, backward=False, rope=(cos, sin))
    # rotate on the host in fp32 and round to bf16 (what the reference's caller hands its kernel)
    xr = dict(x, q=orc.apply_rope(x["q"].float(), cos, sin).to(BF16), k=orc.apply_rope(x["k"].float(), cos, sin).to(BF16))
    twostep = run_gpu(xr, gpu_device, backward=False)
    assert torch.allclose(fused["y"].float(), twostep["y"].float(), atol=2e-2, rtol=1e-2)
    assert torch.allclose(fused["lse"], twostep["lse"], atol=2e-2, rtol=1e-2)
    short = orc.rope_tables(100, 10000.0, 64)
    with pytest.raises(_lib.SegptError):  # table shorter than the positions it must serve
        run_gpu(x, gpu_device, backward=False, rope=short)


@pytest.mark.parametrize(
    "B,H,Hkv,Sq,Sk,D,kw,gen_kw",
    [
        (2, 4, 2, 130, 130, 64, {}, {}),
        (1, 6, 2, 100, 100, 64, {}, {"extras": True}),
        (1, 2, 1, 77, 77, 32, {}, {"scalar_gain": True, "no_gk": True}),
        (1, 4, 1, 70, 70, 128, {}, {}),
        (1, 3, 3, 40, 104, 64, {"q_start": 64}, {}),                      # query positions start at q_start
        (1, 2, 2, 48, 80, 64, {"causal": False, "rope_q_pos0": 11, "rope_k_pos0": 3}, {}),
        (1, 2, 1, 64, 64, 64, {"qk_norm": False}, {"scalar_gain": True, "no_gk": True}),
    ],
)
def test_fp32_fused_rope(gpu_device, B, H, Hkv, Sq, Sk, D, kw, gen_kw):
    """The rotary embedding on the fp32 parity path: forward, dq and dk (gradients with respect to the UNROTATED
    rows) against the oracle at 1e-5 -- pins the pair indexing and the table rows far tighter than bf16 can."""
    _case(gpu_device, F32, B, H, Hkv, Sq, Sk, D, gen_kw=gen_kw, rope=orc.rope_tables(160, 10000.0, D), **kw)


# ------------------------------------------------------------------ decode-shaped calls (split-key kernels)


@pytest.mark.parametrize(
    "B,H,Hkv,Sq,Sk,D,kw,gen_kw,use_rope",
    [
        (1, 18, 6, 1, 2048, 64, {"q_start": 2047}, {}, False),          # one new token against a 2048-key cache
        (2, 6, 2, 1, 1000, 64, {"q_start": 999}, {}, True),             # ragged cache length, rotary positions
        (1, 6, 2, 4, 777, 64, {"q_start": 773}, {"extras": True}, True),  # 4 new tokens, gate + value residual
        (1, 8, 1, 3, 300, 64, {"q_start": 297}, {"scalar_gain": True, "no_gk": True}, False),  # 24 rows per kv head
        (3, 4, 4, 1, 129, 128, {"q_start": 128}, {}, True),
        (1, 4, 2, 2, 640, 128, {"causal": False}, {}, False),
        (16, 6, 2, 1, 4096, 64, {"q_start": 4095}, {}, False),          # many groups: few splits each
        (1, 32, 1, 1, 513, 64, {"q_start": 512}, {}, False),            # exactly 32 query rows per kv head
        (2, 4, 2, 2, 500, 64, {"q_start": 10}, {}, True),               # only the first 12 keys are visible
        (1, 4, 2, 1, 5, 64, {"q_start": 4}, {}, False),                 # cache shorter than one key block
        (1, 2, 2, 1, 1, 64, {"q_start": 0}, {}, True),                  # the very first token: one key
    ],
)
def test_decode_path_matches_oracle_and_training_kernel(gpu_device, B, H, Hkv, Sq, Sk, D, kw, gen_kw, use_rope):
    """Forward-only calls with H/Hkv * Sq <= 32 take the split-key decode kernels (through the C ABI, flag
    SEGPT_FLAG_DECODE set by the front end when nothing requires grad); same tolerance against the oracle, and
    agreement with the training kernel on the same inputs."""
    x = gen(B, H, Hkv, Sq, Sk, D, BF16, seed=41, **gen_kw)
    if use_rope:
        kw = dict(kw, rope=orc.rope_tables(Sk + 8, 10000.0, D))
    print(f"decode case B={B} H={H} Hkv={Hkv} Sq={Sq} Sk={Sk} D={D} kw={ {k: v for k, v in kw.items() if k != 'rope'} } rope={use_rope}", flush=True)
    ref = run_oracle(x, backward=False, **kw)
    with torch.no_grad():
        dec = run_gpu(x, gpu_device, backward=False, **kw)          # inference: decode kernels
    compare(dec, ref, BF16)
    xg = dict(x)
    trn = run_gpu(xg, gpu_device, backward=True, **kw)                # needs grad: training kernels
    compare({n: trn[n] for n in ("y", "lse")}, ref, BF16)
    assert torch.allclose(dec["y"].float(), trn["y"].float(), atol=2e-2, rtol=1e-2)
    assert torch.allclose(dec["lse"], trn["lse"], atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("extras,use_rope,qk_norm", [(False, True, True), (True, True, True), (True, False, False)])
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk", [
    (1, 2, 1, 1, 31),      # one partial block; three waves of the workgroup idle
    (1, 10, 5, 2, 65),     # the second workgroup has one live wave; two blocks and a third of one key
    (3, 3, 1, 1, 448),     # 14 blocks over 2-block splits, whole tiles only
    (2, 32, 4, 4, 2085),   # 32 query rows, 66 blocks, last split shorter
    (30, 4, 4, 1, 1001),   # 30 workgroups in three rounds at most: unequal blocks per split
])
def test_decode_split_edges(gpu_device, B, H, Hkv, Sq, Sk, D, extras, use_rope, qk_norm):
    """Tile and split edges of the decode kernels (32-key blocks, four (batch, kv head) pairs per workgroup); values
    scaled per head without QK-norm so that the running maximum moves."""
    x = gen(B, H, Hkv, Sq, Sk, D, BF16, seed=43, extras=extras, head_scales=not qk_norm)
    kw = {"q_start": Sk - Sq, "qk_norm": qk_norm}
    if use_rope:
        kw["rope"] = orc.rope_tables(Sk, 10000.0, D)
    ref = run_oracle(x, backward=False, **kw)
    with torch.no_grad():
        compare(run_gpu(x, gpu_device, backward=False, **kw), ref, BF16)


def _decode_distance(device, x, use_rope):
    """Norm-wise distance of a decode-shaped call to the model of its roundings (chunks as decode_plan() cuts them)."""
    (B, H, Sq, D), (Hkv, Sk) = x["q"].shape, x["k"].shape[1:3]
    splits = min(-(-(768 if D == 64 else 256) // (B * Hkv)), -(-Sk // 128))
    chunk = -(-(-(-Sk // splits)) // 128) * 128
    rope = orc.rope_tables(Sk, 10000.0, D) if use_rope else None
    model = decode_rounding_model(x, q_start=Sk - Sq, chunk=chunk, streams=4, rope=rope)
    with torch.no_grad():
        y = run_gpu(x, device, backward=False, q_start=Sk - Sq, **({"rope": rope} if use_rope else {}))["y"].double()
    return float((y - model).norm() / model.norm())


@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D,use_rope", [
    (2, 6, 2, 1, 700, 64, True),       # one block per stream, the last streams empty
    (70, 18, 6, 1, 900, 64, False),    # three or four blocks per stream
    (20, 16, 4, 1, 1333, 128, True),
    (3, 8, 4, 2, 2100, 128, False),
    (2, 8, 8, 32, 1500, 64, True),     # 9 to 32 query rows per kv head: streams merged inside a workgroup
    (100, 4, 2, 5, 700, 64, False),
    (2, 12, 4, 3, 1000, 128, True),
    (40, 10, 5, 8, 1100, 128, False),
])
def test_decode_rounds_keys_and_probabilities_like_the_training_kernels(gpu_device, B, H, Hkv, Sq, Sk, D, use_rope):
    """Normalised keys as bf16, probabilities against the running maximum of their stream.  Bound: what is left is fp32 against
    float64 in front of a rounding.  A score off by 2^-20 flips the rounding of one probability in 2^12 by 2^-8, 6e-5 in
    norm; y off by 1e-5 flips one value in 400 by 2^-8, 2e-4 (seen 0 to 2.6e-4; another reference or raw keys 3.7e-3)."""
    print(f"decode rounding B={B} H={H} Hkv={Hkv} Sq={Sq} Sk={Sk} D={D} rope={use_rope}", flush=True)
    assert _decode_distance(gpu_device, gen(B, H, Hkv, Sq, Sk, D, BF16, seed=81), use_rope) < 1e-3


@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D,use_rope", [(2, 6, 2, 1, 700, 64, True), (70, 18, 6, 1, 900, 64, False), (20, 16, 4, 1, 1333, 128, True),
                                                      (2, 12, 4, 3, 1000, 64, True), (40, 10, 5, 8, 1100, 128, False)])
def test_decode_mixes_a_value_residual_before_it_rounds(gpu_device, B, H, Hkv, Sq, Sk, D, use_rope):
    """Coefficients of opposite sign on nearly equal values (a first layer's v_first is its own v; the coefficients are learned):
    V' = c1 v + c2 v_first is a small difference, and its rounding error has to be relative to it.  Bound as above (seen
    0 to 2.2e-4; the two parts rounded one by one 4e-2)."""
    x = gen(B, H, Hkv, Sq, Sk, D, BF16, seed=82, extras=True)
    x["vr_coef"], x["v_first"] = torch.tensor([0.9, -0.85]), x["v"].clone()
    print(f"decode value residual B={B} H={H} Hkv={Hkv} Sq={Sq} Sk={Sk} D={D} rope={use_rope}", flush=True)
    assert _decode_distance(gpu_device, x, use_rope) < 1e-3


@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D,kw,gen_kw,use_rope", [
    (1, 2, 1, 70, 2500, 64, {"q_start": 2430}, {"extras": True}, True),                       # one ragged query tile, last share ragged
    (2, 3, 3, 130, 1100, 128, {"q_start": 970}, {}, False),                                   # two query tiles, the second of 2 rows
    (1, 2, 1, 1500, 1500, 64, {}, {"extras": True}, False),                                   # early tiles fit one share, later ones do not
    (1, 2, 1, 1500, 1500, 128, {"qk_norm": False}, {"head_scales": True}, True),              # shares whose keys some rows do not see
    (1, 8, 2, 257, 2113, 64, {"q_start": 1856, "qk_norm": False}, {"head_scales": True}, False),
    (1, 4, 2, 200, 1900, 64, {"causal": False}, {}, False),
    (1, 1, 1, 70, 5000, 64, {"q_start": 4930}, {"extras": True}, False),                      # 20 shares: more than a lane requests up front
    (1, 1, 1, 70, 5000, 128, {"q_start": 4930}, {}, False),                                   # 40
    (1, 4, 4, 2100, 8192, 64, {"q_start": 6092}, {"extras": True}, False),                    # 8400 rows: one lane takes all 5 shares of its columns
])
def test_forward_only_split_keys(gpu_device, B, H, Hkv, Sq, Sk, D, kw, gen_kw, use_rope):
    """Forward-only calls with few query tiles share out the keys of a tile (partials in the kv workspace, merged by a
    second kernel): against the oracle, and against the unsplit kernel that a call with gradients runs."""
    from sample_efficient_gpt_amd import _lib
    from sample_efficient_gpt_amd.plan import AttnPlan

    x = gen(B, H, Hkv, Sq, Sk, D, BF16, seed=47, **gen_kw)
    if use_rope:
        kw = dict(kw, rope=orc.rope_tables(Sk, 10000.0, D))
    ref = run_oracle(x, backward=False, **kw)
    with torch.no_grad():
        split = run_gpu(x, gpu_device, backward=False, **kw)
    compare(split, ref, BF16)
    whole = run_gpu(x, gpu_device, backward=True, **kw)
    # the same scores; with a running maximum the probabilities are rounded to bf16 against another reference, each by at
    # most 2^-9 of itself on either side, so the logarithms of their sums differ by at most 2^-8
    assert torch.allclose(split["lse"], whole["lse"], atol=2.0**-8 if kw.get("qk_norm") is False else 1e-4, rtol=0)
    plan = AttnPlan({n: None if t is None else t.to(gpu_device) for n, t in x.items() if n != "gate_logits"}, causal=kw.get("causal", True),
                    q_start=kw.get("q_start", 0), backward=False)

    def kv_bytes(flags):
        plan.p.flags = flags
        return plan.lib.segpt_attn_workspace_bytes(plan.p, _lib.SEGPT_WS_KV)

    assert kv_bytes(_lib.SEGPT_FLAG_DECODE) > kv_bytes(0), "no room for partials is asked for: the call is not split"


# ------------------------------------------------------------------ attention without QK-norm (SEGPT_FLAG_NO_NORM)


@pytest.mark.parametrize(
    "dtype,B,H,Hkv,Sq,Sk,D,kw,gen_kw",
    [
        (F32, 2, 4, 2, 130, 130, 64, {}, {"scalar_gain": True, "no_gk": True}),
        (F32, 1, 3, 3, 40, 104, 128, {"q_start": 64}, {"extras": True}),
        (BF16, 2, 6, 2, 384, 384, 64, {}, {"scalar_gain": True, "no_gk": True}),
        (BF16, 1, 3, 1, 300, 300, 64, {}, {}),                           # the scale vectors still apply
        (BF16, 1, 4, 2, 200, 200, 64, {"gate_scale": 2.0}, {"extras": True}),
        (BF16, 1, 2, 1, 256, 256, 128, {}, {"head_scales": True}),       # rows of different norms: logits up to +-20
        (BF16, 1, 2, 2, 96, 200, 64, {"causal": False}, {}),
        (BF16, 1, 3, 3, 72, 200, 64, {"q_start": 128}, {}),
    ],
)
def test_plain_attention_fwd_bwd(gpu_device, dtype, B, H, Hkv, Sq, Sk, D, kw, gen_kw):
    """qk_norm=False: normalisers fixed at 1, against the oracle's family with the same switch (itself pinned
    against SDPA).  head_scales makes the row norms differ, so a normaliser left in by mistake would show."""
    _case(gpu_device, dtype, B, H, Hkv, Sq, Sk, D, gen_kw=gen_kw, qk_norm=False, **kw)


def test_plain_dropin_matches_sdpa_restatement(gpu_device):
    """FlashAttnFunc.apply(Q, K, V, q_start, is_causal) -- the reference's TritonFlashAttnFunc call shape
    (attention.py:240) -- against the brute-force softmax restatement and its autograd gradients; GQA-native
    K/V equal the expanded call; the library op reaches the same kernels."""
    B, H, Hkv, S, D = 2, 6, 2, 320, 64
    x = gen(B, H, Hkv, S, S, D, BF16, seed=17, head_scales=True)
    x["q"] = (x["q"].float() * 0.7).to(BF16)
    Q, K, V, dO = _flat(x["q"], H), _flat(x["k"], Hkv), _flat(x["v"], Hkv), _flat(x["d_o"], H)
    Kx, Vx = (orc.expand_kv_flat(t, Hkv, H).contiguous() for t in (K, V))
    Qr, Kr, Vr = (t.detach().clone().double().requires_grad_(True) for t in (Q, Kx, Vx))
    ref_out = orc.plain_flash_variant(Qr, Kr, Vr, 0, True)
    ref_out.backward(dO.double())
    d = gpu_device
    Qd, Kd, Vd = (t.detach().clone().to(d).requires_grad_(True) for t in (Q, Kx, Vx))
    out = FlashAttnFunc.apply(Qd, Kd, Vd, 0, True)
    assert out.shape == Q.shape and out.dtype == Q.dtype
    out.backward(dO.to(d))
    got = {"y": out.detach().cpu(), "dq": Qd.grad.cpu(), "dk": Kd.grad.cpu(), "dv": Vd.grad.cpu()}
    ref = {"y": ref_out.detach(), "dq": Qr.grad, "dk": Kr.grad, "dv": Vr.grad}
    print("plain drop-in max abs err", compare(got, ref, BF16), flush=True)
    # un-expanded GQA tensors: same output bits, dK/dV are the group sums
    Qn, Kn, Vn = (t.detach().clone().to(d).requires_grad_(True) for t in (Q, K, V))
    o_nat = FlashAttnFunc.apply(Qn, Kn, Vn, 0, True, Hkv)
    assert torch.equal(o_nat, out)
    o_nat.backward(dO.to(d))
    rep = H // Hkv
    dk_sum = ref["dk"].reshape(Hkv, rep, B, S, D).sum(1).reshape(Hkv * B, S, D)
    compare({"dk": Kn.grad.cpu()}, {"dk": dk_sum}, BF16)
    # decode-time call shape: q_start = past length, forward only (split-key kernels)
    with torch.no_grad():
        tail = FlashAttnFunc.apply(Q[:, 317:].contiguous().to(d), K.to(d), V.to(d), 317, True, Hkv)
    compare({"y": tail.cpu()}, {"y": ref_out.detach()[:, 317:]}, BF16)
    # the registered op with qk_norm=False
    q4 = x["q"].to(d)
    y_op = qknorm_attention_op(q4, x["k"].to(d), x["v"].to(d), torch.ones(1, device=d), None, qk_norm=False)
    assert torch.equal(orc.flatten_heads(y_op.cpu()), out.detach().cpu())


def test_backward_is_deterministic(gpu_device):
    x = gen(2, 6, 2, 512, 512, 64, BF16, extras=True, seed=4)
    a = run_gpu(x, gpu_device)
    b = run_gpu(x, gpu_device)
    for n in a:
        assert torch.equal(a[n], b[n]), n


# ------------------------------------------------------------------ the reference's call signature


def _flat(x, H):
    return orc.flatten_heads(x).contiguous()


def test_dropin_matches_live_module_variant_a(gpu_device):
    """Positional call exactly as the reference makes it (expanded K/V, scalar gain): compare with the
    restatement of the live module, attention.py:43-80, incl. its bf16 rounding points."""
    B, H, Hkv, S, D = 2, 6, 2, 320, 64
    x = gen(B, H, Hkv, S, S, D, BF16, scalar_gain=True, no_gk=True, seed=7)
    Q = _flat(x["q"], H)
    K = orc.expand_kv_flat(_flat(x["k"], Hkv), Hkv, H).contiguous()
    V = orc.expand_kv_flat(_flat(x["v"], Hkv), Hkv, H).contiguous()
    gain = x["g_q"]
    dO = _flat(x["d_o"], H)
    # reference side (CPU): bf16 module forward; gradients from the fp32 evaluation of the same formula
    ref_out = orc.live_module_variant_a(Q, K, V, gain)
    Qr, Kr, Vr, gr = (t.detach().clone().float().requires_grad_(True) for t in (Q, K, V, gain))
    orc.live_module_variant_a(Qr, Kr, Vr, gr).backward(dO.float())
    Qd, Kd, Vd, gd = (t.detach().clone().to(gpu_device).requires_grad_(True) for t in (Q, K, V, gain))
    out = QKNormFlashAttnFunc.apply(Qd, Kd, Vd, gd, True, 0)
    assert out.shape == Q.shape and out.dtype == Q.dtype
    out.backward(dO.to(gpu_device))
    got = {"y": out.detach().cpu(), "dq": Qd.grad.cpu(), "dk": Kd.grad.cpu(), "dv": Vd.grad.cpu(), "dg": gd.grad.cpu()}
    ref = {"y": ref_out, "dq": Qr.grad, "dk": Kr.grad, "dv": Vr.grad, "dg": gr.grad}
    assert gd.grad.shape == gain.shape and gd.grad.dtype == gain.dtype
    xs = dict(x, g_k=None)
    compare(got, ref, BF16, scales={"dg": scalar_gain_scale(xs)["dg_q"]})


def test_dropin_gqa_native_equals_expanded_and_2d_inputs(gpu_device):
    B, H, Hkv, S, D = 2, 6, 2, 192, 64
    x = gen(B, H, Hkv, S, S, D, BF16, scalar_gain=True, no_gk=True, seed=8)
    Q, K, V = _flat(x["q"], H), _flat(x["k"], Hkv), _flat(x["v"], Hkv)
    Kx, Vx = (orc.expand_kv_flat(t, Hkv, H).contiguous() for t in (K, V))
    d = gpu_device
    g = x["g_q"].to(d)
    o_exp = QKNormFlashAttnFunc.apply(Q.to(d), Kx.to(d), Vx.to(d), g)
    o_nat = QKNormFlashAttnFunc.apply(Q.to(d), K.to(d), V.to(d), g, True, 0, None, None, None, None, 2.0, Hkv)
    assert torch.equal(o_exp, o_nat)
    o2 = QKNormFlashAttnFunc.apply(Q[0].to(d), Kx[0].to(d), Vx[0].to(d), g)
    assert o2.shape == (1, S, D) and torch.equal(o2[0], o_exp[0])


def test_dropin_rejects_bad_inputs(gpu_device):
    d = gpu_device
    Q = torch.randn(2, 64, 64, device=d, dtype=BF16)
    g = torch.ones(1, device=d)
    with pytest.raises(AssertionError):
        QKNormFlashAttnFunc.apply(Q.transpose(0, 1), Q, Q, g)       # not contiguous
    with pytest.raises(AssertionError):
        QKNormFlashAttnFunc.apply(Q.cpu(), Q.cpu(), Q.cpu(), g)     # not on the device
    with pytest.raises(TypeError):
        QKNormFlashAttnFunc.apply(Q.half(), Q.half(), Q.half(), g)  # unsupported dtype
    with pytest.raises(RuntimeError, match="head_dim"):
        QKNormFlashAttnFunc.apply(Q[..., :48].contiguous(), Q[..., :48].contiguous(), Q[..., :48].contiguous(), g)


def test_fused_triton_formula_is_reachable_variant_b(gpu_device):
    """eps = 1e-8/d, sm_scale = 1/d reproduces the fused Triton kernel's own logits (gain*cos)."""
    S, D = 128, 64
    x = gen(3, 1, 1, S, S, D, F32, scalar_gain=True, no_gk=True, seed=9)
    Q, K, V = (x[n][:, 0].contiguous() for n in ("q", "k", "v"))
    O_ref, L_ref = orc.fused_kernel_variant_b(Q.double(), K.double(), V.double(), x["g_q"].double())
    eps, sc = orc.family_params("B", D)
    d = gpu_device
    out = QKNormFlashAttnFunc.apply(Q.to(d), K.to(d), V.to(d), x["g_q"].to(d), True, 0, None, None, None, None, 2.0, None, eps, sc)
    compare({"y": out.cpu()}, {"y": O_ref}, F32)


def test_reference_named_function_defaults_to_the_reference_kernel_formula(gpu_device):
    """`TritonFlashAttnQKNormFunc.apply(Q, K, V, gain)` with NO further arguments computes what the reference class of
    that name computes (triton_flash_attn_qknorm.py:67-91: L2 normaliser with 1e-8 on the sum, logits gain*cos), not
    the live module's 1/sqrt(d)-scaled RMS form; forward and the gradients of Q, K, V and the gain."""
    from sample_efficient_gpt_amd import TritonFlashAttnQKNormFunc

    S, D = 96, 64
    x = gen(2, 1, 1, S, S, D, F32, scalar_gain=True, no_gk=True, seed=19)
    Q, K, V, dO = (x[n][:, 0].contiguous() for n in ("q", "k", "v", "d_o"))
    ref_in = [t.double().requires_grad_(True) for t in (Q, K, V, x["g_q"])]
    O_ref, _ = orc.fused_kernel_variant_b(*ref_in)
    O_ref.backward(dO.double())
    d = gpu_device
    dev_in = [t.to(d).requires_grad_(True) for t in (Q, K, V, x["g_q"])]
    out = TritonFlashAttnQKNormFunc.apply(*dev_in)
    out.backward(dO.to(d))
    compare({"y": out.detach().cpu(), "dq": dev_in[0].grad.cpu(), "dk": dev_in[1].grad.cpu(), "dv": dev_in[2].grad.cpu(),
             "dg_q": dev_in[3].grad.cpu()},
            {"y": O_ref.detach(), "dq": ref_in[0].grad, "dk": ref_in[1].grad, "dv": ref_in[2].grad, "dg_q": ref_in[3].grad}, F32)
    # and it differs from the live-module defaults of QKNormFlashAttnFunc (logits sqrt(d) times larger there)
    live = QKNormFlashAttnFunc.apply(*(t.detach() for t in dev_in))
    assert float((live.cpu().double() - O_ref.detach()).abs().max()) > 1e-2


@pytest.mark.parametrize("D,d_big", [(64, 0), (64, 15), (64, 16), (64, 31), (64, 32), (64, 47), (64, 63),
                                     (128, 0), (128, 63), (128, 64), (128, 100), (128, 127)])
def test_bf16_forward_sees_a_single_large_scale_entry(gpu_device, D, d_big):
    """The bf16 forward drops the running maximum when max_d |g_q g_k| bounds the logits inside the exponent range;
    that maximum is a wave-wide reduction over the scale vector.  One entry of g_q is made large enough (logits of
    +-320 in natural units, 2^461 as a raw exponent) that the forward must keep the running maximum, whichever
    lane and DPP row holds the entry: queries and keys are dominated by that dimension, so a forward that missed
    the entry would overflow to inf / NaN.  Checked here: the output is finite and every row is a convex
    combination of value rows (|y| <= max |v|); parity at such logits is the variant-C test's business."""
    torch.manual_seed(5)
    B, H, S = 1, 2, 160
    q = 0.01 * torch.randn(B, H, S, D)
    k = 0.01 * torch.randn(B, H, S, D)
    q[..., d_big] = 1.0
    k[..., d_big] = torch.where(torch.rand(B, H, S) < 0.5, -1.0, 1.0)
    v = torch.randn(B, H, S, D)
    g = torch.full((D,), 0.5)
    g[d_big] = 40.0
    print(f"large scale entry D={D} at {d_big}", flush=True)
    dev = lambda t: t.to(BF16).to(gpu_device)
    y = qknorm_attention(dev(q), dev(k), dev(v), g.to(gpu_device), None, eps=1e-6, sm_scale=D ** -0.5)
    y = y.float().cpu()
    assert torch.isfinite(y).all(), "the forward took the no-maximum path with logits outside the exponent range"
    assert float(y.abs().max()) <= float(v.to(BF16).float().abs().max()) * 1.01


@pytest.mark.parametrize("dtype,S,Sk,q_start,causal", [(F32, 96, 96, 0, True), (F32, 40, 104, 64, True), (F32, 50, 70, 0, False),
                                                      (BF16, 128, 128, 0, True), (BF16, 72, 200, 128, True)])
def test_cpu_patch_formula_variant_c(gpu_device, dtype, S, Sk, q_start, causal):
    """The reference's CPU patch (convert_imu1_checkpoint.py:73-89: RMS normaliser with eps 1e-8, NO 1/sqrt(d), so
    logits are gain*d*cos, up to +-64 at head_dim 64) is the family at (eps, sm_scale) = (1e-8, 1): the HIP kernels with
    those parameters against `cpu_patch_variant_c`, forward and every gradient, q_start and non-causal included.
    fp32 at 1e-5.  The logit bound leaves the raw-exponent range, so the bf16 forward takes its running-maximum
    path.  A bf16 logit carries the 2^-9 rounding of both normalised operands times its magnitude, sqrt(d) = 8 times
    the live module's, which no kernel working on bf16 operands can avoid; the bf16 leg therefore compares with a
    float64 model of the kernels' mathematics that rounds where they round (pinned to the oracle with the roundings
    switched off) at the ordinary bf16 tolerance.  The reference itself runs this formula on the CPU in fp32 only."""
    D, n = 64, 3
    x = gen(n, 1, 1, S, Sk, D, dtype, no_gk=True, seed=23)
    gain = torch.tensor([1.0])
    Q, K, V, dO = (x[k][:, 0].contiguous() for k in ("q", "k", "v", "d_o"))
    ref_in = [t.double().requires_grad_(True) for t in (Q, K, V, gain)]
    O_ref = orc.cpu_patch_variant_c(*ref_in, causal, q_start)
    O_ref.backward(dO.double())
    ref = {"y": O_ref.detach(), "dq": ref_in[0].grad, "dk": ref_in[1].grad, "dv": ref_in[2].grad, "dg_q": ref_in[3].grad}
    eps, sc = orc.family_params("C", D)
    assert (eps, sc) == (1e-8, 1.0)

    def run(dt):
        dev_in = [t.to(dt).to(gpu_device).requires_grad_(True) for t in (Q, K, V)] + [gain.to(gpu_device).requires_grad_(True)]
        out = QKNormFlashAttnFunc.apply(*dev_in, causal, q_start, None, None, None, None, 2.0, None, eps, sc)
        out.backward(dO.to(dt).to(gpu_device))
        return {"y": out.detach().cpu(), "dq": dev_in[0].grad.cpu(), "dk": dev_in[1].grad.cpu(), "dv": dev_in[2].grad.cpu(),
                "dg_q": dev_in[3].grad.cpu()}

    print(f"variant C {dtype} S={S} Sk={Sk} q_start={q_start} causal={causal}", flush=True)
    # yardstick of the scalar gain's gradient (a sum over d of per-dimension gradients that cancel)
    dgs = float(orc.attention_backward_autograd(
        x["q"].double(), x["k"].double(), x["v"].double(), torch.ones(D, dtype=torch.float64), None, x["d_o"].double(),
        eps=eps, sm_scale=sc, causal=causal, q_start=q_start)["dg_q"].abs().sum())

    def check(got, atol, rtol, what):
        for name, r in ref.items():
            g = got[name].double().reshape(r.shape)
            scale = max(float(r.abs().max()), dgs) if name == "dg_q" else float(r.abs().max())
            err = float((g - r).abs().max())
            print(f"  {what} {name}: max abs err {err:.2e} (largest entry {float(r.abs().max()):.2e})", flush=True)
            assert err <= atol + rtol * scale, f"{what} {name}: max abs err {err:.3e} > {atol + rtol * scale:.3e}"

    # fp32: 1e-5, norm-wise (relative to the tensor's largest entry).  Element-wise 1e-5 is not attainable in fp32
    # arithmetic here: one fp32 ulp of a logit of magnitude 64 is 7.6e-6, which alone moves exp(logit) by 7.6e-6 relative,
    # and the gradients sum thousands of such terms against entries of size 20.
    check(run(F32), 1e-5, 1e-5, "fp32")
    if dtype == BF16:
        # bf16: the comparison target is derived per case.  `kernel_rounding_model` is the same mathematics in float64 with
        # a bf16 rounding wherever the kernels hold a bf16 value; with the roundings switched off it must BE the oracle
        # (that pins it), with them on the kernels have to meet the ORDINARY bf16 tolerance against it, and its own
        # distance to the oracle, i.e. what operand rounding costs at logits of +-64, is reported (it is what the
        # earlier blanket allowance of 8x stood for).
        import tests.parity_util as pu

        args = (Q, K, V, gain.double(), dO)
        kw = dict(eps=eps, sm_scale=sc, causal=causal, q_start=q_start)
        keep = pu.bf16_round
        try:
            pu.bf16_round = lambda t: t
            exact = pu.kernel_rounding_model(*args, **kw)
        finally:
            pu.bf16_round = keep
        for name in ("y", "dq", "dk", "dv"):
            assert float((exact[name] - ref[name]).abs().max()) <= 1e-9 * max(1.0, float(ref[name].abs().max())), name
        assert abs(float(exact["dg"].sum() - ref["dg_q"])) <= 1e-9 * max(1.0, dgs)
        model = pu.kernel_rounding_model(*args, **kw)
        model["dg_q"] = model.pop("dg").sum().reshape(ref["dg_q"].shape)
        got = run(BF16)
        for name, r in model.items():
            g = got[name].double().reshape(r.shape)
            err = (g - r).abs()
            # y and dv element-wise; dq, dk norm-wise like the fp32 leg above: delta is taken from the bf16-rounded
            # output, whose rounding residue (modelled in size, not entry by entry) enters them times the logit scale
            scale = max(float(r.abs().max()), dgs) if name == "dg_q" else (r.abs() if name in ("y", "dv") else float(r.abs().max()))
            drift = float((r - ref[name]).abs().max())
            print(f"  bf16 {name}: max abs err vs the rounding model {float(err.max()):.2e}; the model is {drift:.2e} from the oracle "
                  f"(largest entry {float(ref[name].abs().max()):.2e})", flush=True)
            assert bool((err <= 2e-2 + 1e-2 * scale).all()), f"bf16 {name}: max abs err {float(err.max()):.3e} vs the rounding model"
            assert drift <= 8 * (2e-2 + 1e-2 * float(ref[name].abs().max())), name  # operand rounding stays what it was known to be


def test_module_state_dict_and_forward(gpu_device):
    m = SelfDotProductAttnQKNorm(64).to(gpu_device)
    assert list(m.state_dict().keys()) == ["gain"] and m.gain.shape == (1,) and m.gain.dtype == torch.float32
    x = gen(1, 4, 4, 96, 96, 64, BF16, seed=10)
    Q, K, V = (_flat(x[n], 4).to(gpu_device) for n in ("q", "k", "v"))
    out = m(Q, K, V, True, q_start=0)
    ref = orc.live_module_variant_a(Q.cpu(), K.cpu(), V.cpu(), torch.ones(1))
    compare({"y": out.cpu()}, {"y": ref}, BF16)


def test_strided_projection_views(gpu_device):
    """q/k/v taken as strided slices of one `[b, S, (H+2Hkv)*D]` projection output (no copies)."""
    B, H, Hkv, S, D = 2, 6, 2, 160, 64
    x = gen(B, H, Hkv, S, S, D, BF16, seed=11)
    W = (H + 2 * Hkv) * D
    proj = torch.empty(B, S, W, dtype=BF16)
    proj[..., : H * D] = x["q"].permute(0, 2, 1, 3).reshape(B, S, H * D)
    proj[..., H * D: (H + Hkv) * D] = x["k"].permute(0, 2, 1, 3).reshape(B, S, Hkv * D)
    proj[..., (H + Hkv) * D:] = x["v"].permute(0, 2, 1, 3).reshape(B, S, Hkv * D)
    pd = proj.to(gpu_device)
    q = pd[..., : H * D].view(B, S, H, D).permute(0, 2, 1, 3)
    k = pd[..., H * D: (H + Hkv) * D].view(B, S, Hkv, D).permute(0, 2, 1, 3)
    v = pd[..., (H + Hkv) * D:].view(B, S, Hkv, D).permute(0, 2, 1, 3)
    y = qknorm_attention(q, k, v, x["g_q"].to(gpu_device), x["g_k"].to(gpu_device))
    ref = run_oracle(x, backward=False)
    compare({"y": y.cpu()}, ref, BF16, names=["y"])


# ------------------------------------------------------------------ the whole attention module around one kernel call


def _module_and_oracle_weights(device, dtype, d_model, H, Hkv, qknorm, value_residual, gating, seed):
    torch.manual_seed(seed)
    m = MultiHeadSelfAttention(d_model, H, Hkv, max_seq_len=1024, qknorm=qknorm, value_residual=value_residual, gating=gating)
    with torch.no_grad():
        if qknorm:
            m.sdpa_qknorm.gain.fill_(1.3)
        if value_residual:
            m.alpha1.fill_(0.8); m.alpha2.fill_(0.5); m.scale.fill_(1.1)
    for name in ("qkv", "out", "attn_gate"):
        if hasattr(m, name):
            getattr(m, name).to(dtype)
    m = m.to(device)
    w = {n: t.detach().cpu().double().requires_grad_(True) for n, t in m.state_dict().items()}
    rope = (m.rope.cos.detach().cpu().double(), m.rope.sin.detach().cpu().double())
    return m, w, rope


def _weight_close(got, ref, dtype, name, yardstick=None):
    """Weight gradients are sums over every token: tolerance relative to the largest entry (norm-wise).
    A scalar parameter's gradient is ONE sum over every element of the layer, so the rounding noise of
    the summands does not shrink with the (cancelling) total: for those the relative part refers to
    `yardstick`, the sum of the magnitudes of the partial gradients the scalar is the total of.  The fp32 cases
    pin the same gradients at 1e-5 of that yardstick (measured: the output projection, computed by torch's fp32 GEMM
    on both sides, agrees with the fp64 oracle to 5e-6 at matmul precision "highest", the default)."""
    tol = {BF16: (2e-2, 1e-2), F32: (1e-5, 1e-5)}[dtype]
    err = (got.double() - ref).abs().max()
    scale = ref.abs().max() if yardstick is None else max(float(ref.abs().max()), yardstick)
    bound = tol[0] + tol[1] * scale
    assert err <= bound, f"{name}: max abs err {float(err):.3e} > {float(bound):.3e} (ref max {float(ref.abs().max()):.3e})"


@pytest.mark.parametrize(
    "dtype,H,Hkv,d,S,qknorm,value_residual,gating,use_v1",
    [
        (F32, 4, 2, 64, 100, True, True, "per-head", True),
        (F32, 2, 2, 32, 70, False, False, False, False),
        (BF16, 6, 2, 64, 256, True, True, "per-head", True),      # the IMU-1 layer shape in small
        (BF16, 6, 2, 64, 200, True, True, "per-head", False),     # first layer: v1 is None
        (BF16, 4, 4, 64, 130, True, False, "per-head-hd", False),
        (BF16, 4, 1, 128, 96, False, False, "elementwise", False),
        (BF16, 4, 2, 64, 160, True, False, False, False),
    ],
)
def test_mhsa_module_matches_oracle(gpu_device, dtype, H, Hkv, d, S, qknorm, value_residual, gating, use_v1):
    """MultiHeadSelfAttention (projection -> ONE fused kernel call -> output projection) against the oracle's
    step-by-step restatement of attention.py:175-267 on the same weights: outputs, the value tensor handed to
    later layers, and the gradients of x, v1 and every parameter."""
    b, d_model = 2, H * d
    m, w, rope = _module_and_oracle_weights(gpu_device, dtype, d_model, H, Hkv, qknorm, value_residual, gating, seed=3)
    g = torch.Generator().manual_seed(4)
    x = torch.randn(b, S, d_model, generator=g).to(dtype)
    d_out = torch.randn(b, S, d_model, generator=g).to(dtype)
    v1 = torch.randn(H // Hkv * 0 + Hkv * b, S, d, generator=g).to(dtype) if use_v1 else None   # [(hkv b), S, d]
    print(f"mhsa case {dtype} H={H} Hkv={Hkv} d={d} S={S} qknorm={qknorm} vr={value_residual} gating={gating} v1={use_v1}", flush=True)
    # oracle (fp64 on the same bits); v1 in the reference's expanded layout
    xr = x.double().requires_grad_(True)
    v1r = None if v1 is None else v1.double().requires_grad_(True)
    v1x = None if v1 is None else orc.expand_kv_flat(v1r, Hkv, H)
    ref_out, ref_V = orc.mhsa_forward(xr, w, n_heads=H, n_kv_heads=Hkv, qknorm=qknorm, gating=gating, v1=v1x, rope=rope)
    ref_out.backward(d_out.double())
    # product
    xd = x.to(gpu_device).requires_grad_(True)
    v1d = None if v1 is None else v1.to(gpu_device).requires_grad_(True)
    if use_v1:  # a layer that is handed v1 returns no V by default (only the first layer's is ever used)
        assert m(xd.detach(), v1=v1d.detach())[1] is None
        m.always_return_values = True
    out, V = m(xd, v1=v1d)
    assert out.shape == (b, S, d_model) and V.shape == (b, Hkv, S, d)
    out.backward(d_out.to(gpu_device))
    torch.cuda.synchronize()
    tol = dict(atol=2e-2, rtol=1e-2) if dtype == BF16 else dict(atol=1e-5, rtol=1e-5)
    assert torch.allclose(out.detach().cpu().double(), ref_out.detach(), **tol), (out.detach().cpu().double() - ref_out.detach()).abs().max()
    ref_V_native = orc.unflatten_heads(ref_V.detach(), H)[:, :: H // Hkv]
    assert torch.allclose(V.detach().cpu().double(), ref_V_native, **tol)
    _weight_close(xd.grad.cpu(), xr.grad, dtype, "dx")
    if v1 is not None:
        _weight_close(v1d.grad.cpu(), v1r.grad, dtype, "dv1")
    # yardsticks of the scalar parameters: the gain as a vector of equal entries gives its per-dimension
    # gradients; alpha1 / alpha2 / scale act through (c1, c2), whose gradients are sums over (batch, kv head)
    yard = {}
    if True:  # both dtypes: in fp32 the same sums carry fp32 rounding noise of the same structure, at 1e-5
        wv = {n: t.detach().clone().requires_grad_(True) for n, t in w.items()}
        if qknorm:
            wv["sdpa_qknorm.gain"] = w["sdpa_qknorm.gain"].detach().expand(d).clone().requires_grad_(True)
        pieces = {}
        if value_residual:  # one (alpha1, alpha2, scale) copy per flattened value row
            for n in ("alpha1", "alpha2", "scale"):
                pieces[n] = w[n].detach().expand(H * b, 1, 1).clone().requires_grad_(True)
                wv[n] = pieces[n]
        o2, _ = orc.mhsa_forward(x.double(), wv, n_heads=H, n_kv_heads=Hkv, qknorm=qknorm, gating=gating,
                                 v1=None if v1 is None else orc.expand_kv_flat(v1.double(), Hkv, H), rope=rope)
        o2.backward(d_out.double())
        if qknorm:
            yard["sdpa_qknorm.gain"] = float(wv["sdpa_qknorm.gain"].grad.abs().sum())
        for n, t in pieces.items():
            yard[n] = float(t.grad.abs().sum())
        print("scalar-parameter yardsticks", yard, flush=True)
    for n, p in m.named_parameters():
        _weight_close(p.grad.cpu(), w[n].grad, dtype, n, yard.get(n))


def test_mhsa_module_cached_step_takes_the_decode_kernels(gpu_device):
    """Under no_grad (the reference generates under inference_mode, transformer.py:160) a cached single-token step
    of the module reaches the split-key decode kernels: its attention output is bit-identical to a direct
    qknorm_attention call on the same operands without grad (which sets SEGPT_FLAG_DECODE) and NOT to the training
    kernels' result (same call with an input that requires grad); with grad mode on, the module takes the
    training kernels."""
    H, Hkv, d, S0 = 6, 2, 64, 333
    b, d_model = 2, H * d
    m, _, _ = _module_and_oracle_weights(gpu_device, BF16, d_model, H, Hkv, True, True, "per-head", seed=21)
    g = torch.Generator().manual_seed(22)
    x = torch.randn(b, S0 + 1, d_model, generator=g).to(BF16).to(gpu_device)
    captured = {}
    lin = m.out.linear
    hook = lin.register_forward_hook(lambda mod, inp, out: captured.__setitem__("attn_cat", inp[0].detach().clone()))

    def direct(cache, xt, requires_grad):
        """The kernel call the module makes for token xt, rebuilt outside it."""
        proj = m.qkv(xt)
        q = proj[..., : H * d].unflatten(-1, (H, d)).permute(0, 2, 1, 3)
        n = torch.rsqrt(m.alpha1**2 + m.alpha2**2 + 1e-8)
        coef = torch.cat([m.scale * m.alpha1 * n, m.scale * m.alpha2 * n]).float().detach()
        q = q.detach().requires_grad_(requires_grad)
        y = qknorm_attention(q, cache.keys, cache.values, m.sdpa_qknorm.gain.detach(), None, v_first=cache.values, vr_coef=coef,
                             gate_logits=m.attn_gate(xt), gate_scale=2.0, q_start=cache.length - 1, rope_cos=m.rope.cos,
                             rope_sin=m.rope.sin, rope_q_pos0=cache.length - 1, out_bshd=True)
        return y.detach().permute(0, 2, 1, 3).reshape(b, 1, H * d)

    with torch.no_grad():
        cache = KVCache()
        m(x[:, :S0], kv_cache=cache)
        m(x[:, S0:], kv_cache=cache)
        mod_nograd = captured["attn_cat"]
        dec = direct(cache, x[:, S0:], requires_grad=False)
    trn = direct(cache, x[:, S0:], requires_grad=True)   # grad mode on and an input that wants a gradient: training kernels
    cache2 = KVCache()
    with torch.no_grad():
        m(x[:, :S0], kv_cache=cache2)
    m(x[:, S0:], kv_cache=cache2)                         # grad mode on, parameters require grad: training kernels
    mod_grad = captured["attn_cat"]
    hook.remove()
    same = lambda a, c: torch.equal(a.view(torch.int16), c.view(torch.int16))
    assert same(mod_nograd, dec), "the module's no_grad cached step is not the decode kernels' result"
    assert same(mod_grad, trn), "the module's cached step with grad mode on is not the training kernels' result"
    assert not same(dec, trn), "decode and training kernels agree bit for bit here: the test cannot tell them apart"
    assert torch.allclose(dec.float(), trn.float(), atol=2e-2, rtol=1e-2)


def test_mhsa_module_generation_with_cache(gpu_device):
    """Prefill + single-token steps through KVCache (raw, un-expanded keys; under no_grad the steps run the
    split-key decode kernels, see test_mhsa_module_cached_step_takes_the_decode_kernels) reproduce one full causal
    pass and the oracle's cached run; the value tensor handed to later layers is mixed for the new rows only and
    still equals the full pass's."""
    H, Hkv, d, S0, S = 6, 2, 64, 150, 154
    b, d_model = 2, H * d
    m, w, rope = _module_and_oracle_weights(gpu_device, BF16, d_model, H, Hkv, True, True, "per-head", seed=9)
    x = torch.randn(b, S, d_model, generator=torch.Generator().manual_seed(12)).to(BF16)
    xd = x.to(gpu_device)
    with torch.no_grad():
        full, V_full = m(xd)
        cache = KVCache()
        outs = [m(xd[:, :S0], kv_cache=cache)[0]]
        for t in range(S0, S):
            o, V_t = m(xd[:, t : t + 1], kv_cache=cache)
            outs.append(o)
    assert cache.length == S and cache.keys.shape == (b, Hkv, S, d)
    steps = torch.cat(outs, dim=1)
    assert torch.allclose(steps.float(), full.float(), atol=2e-2, rtol=1e-2)
    assert torch.allclose(V_t.float(), V_full.float(), atol=1e-2, rtol=1e-2)
    wd = {n: t.detach() for n, t in w.items()}
    ref, _ = orc.mhsa_forward(x.double(), wd, n_heads=H, n_kv_heads=Hkv, qknorm=True, gating="per-head", rope=rope)
    assert torch.allclose(steps.cpu().double(), ref, atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("dtype,D", [(BF16, 64), (BF16, 128), (F32, 32), (F32, 64)])
def test_kv_cache_append_is_the_two_copies(gpu_device, dtype, D):
    """KVCache.append in one launch: a prompt, single rows, a run that makes the buffers grow and an odd run, from strided views
    of a projection, hold exactly what was appended; what the launch does not take (rows off 16 bytes, a tensor that records
    gradients) goes the old way; the views of earlier steps notice that their buffer was written."""
    B, Hkv = 3, 5
    cache, want_k, want_v = KVCache(capacity=70), [], []
    for i, S in enumerate((37, 1, 1, 64, 129, 1)):
        proj = torch.randn(B, S, 3 * Hkv * D + 8, device=gpu_device, dtype=dtype)
        lo = 1 if i == 4 else 0  # the fifth run: rows that start at an odd element
        k, v = (proj[..., lo + j * Hkv * D : lo + (j + 1) * Hkv * D].unflatten(-1, (Hkv, D)).permute(0, 2, 1, 3) for j in (1, 2))
        before = cache._kbuf._version if cache._kbuf is not None else None
        grown = cache.length + S > (0 if cache._kbuf is None else cache._kbuf.shape[2])
        with torch.no_grad():
            keys, values = cache.append(k, v)
        want_k.append(k); want_v.append(v)
        assert torch.equal(keys, torch.cat(want_k, dim=2)) and torch.equal(values, torch.cat(want_v, dim=2)), i
        assert keys.data_ptr() == cache._kbuf.data_ptr() and cache.length == keys.shape[2]
        assert grown or cache._kbuf._version > before
    k = torch.randn(B, Hkv, 2, D, device=gpu_device, dtype=dtype, requires_grad=True)
    keys, _ = cache.append(k, k.detach())
    assert keys.requires_grad and torch.equal(keys[:, :, -2:], k)


@pytest.mark.parametrize("M,K,ns", [(1, 32, (1,)), (2, 288, (16, 15)), (15, 1152, (1152, 384, 384, 18)), (16, 2048, (17, 64)), (3, 2080, (33,))])
def test_linear_rows(gpu_device, M, K, ns):
    """segpt_linear_rows at the edges of its tiles (rows, columns, steps shared out unevenly over the waves, more than one batch
    of them) and with heads scattered over a larger buffer.  Bound: one rounding to bf16 of a sum whose fp32 additions err by
    2^-24 of the summed magnitudes each, at most K / 32 / 8 * 2 + 8 of them in a row."""
    import ctypes

    from sample_efficient_gpt_amd import _lib
    g = torch.Generator().manual_seed(M + K)
    n = lambda *s: torch.randn(*s, generator=g).to(BF16).to(gpu_device)
    x = n(M, K + 8)[:, :K]
    p = _lib.LinearRowsParams()
    p.struct_bytes, p.M, p.K, p.n_segments, p.x, p.x_stride = ctypes.sizeof(p), M, K, len(ns), x.data_ptr(), x.stride(0)
    ws, outs = [n(c, K) for c in ns], []
    for i, c in enumerate(ns):
        width = 16 if c % 16 == 0 else c
        outs.append(torch.full((M, c // width, 3, width), 7.0, dtype=BF16, device=gpu_device))
        p.seg[i] = _lib.LinearSegment(ws[i].data_ptr(), K, outs[i][:, :, 1].data_ptr(), outs[i].stride(0), outs[i].stride(1), c, width)
    print(f"linear_rows M={M} K={K} ns={ns}", flush=True)
    assert _lib.load().segpt_linear_rows(p, torch.cuda.current_stream(gpu_device).cuda_stream) == 0
    torch.cuda.synchronize()
    for w, o in zip(ws, outs):
        want = x.double() @ w.double().T
        slack = (x.double().abs() @ w.double().abs().T) * (K / 128 + 8) * 2.0**-24
        assert bool(((o[:, :, 1].reshape(M, -1).double() - want).abs() <= want.abs() * 2.0**-8 + slack).all())
        assert bool((o[:, :, 0] == 7).all()) and bool((o[:, :, 2] == 7).all())


@pytest.mark.parametrize("b,H,Hkv,d,gating,qknorm", [(1, 18, 6, 64, "per-head", True), (3, 6, 2, 64, False, True), (16, 4, 4, 128, "per-head", False)])
def test_mhsa_module_generation_step_is_the_separate_calls(gpu_device, b, H, Hkv, d, gating, qknorm):
    """A cached token as one native call against the same module whose layers are called one by one (a hook on a layer asks
    for that): the same new rows of the cache and outputs but for the order of the projections' sums, the earlier rows
    untouched, and every caller that has to see the layers still does."""
    S0, d_model = 70, H * d
    m, _, _ = _module_and_oracle_weights(gpu_device, BF16, d_model, H, Hkv, qknorm, False, gating, seed=31)
    x = torch.randn(b, S0 + 2, d_model, generator=torch.Generator().manual_seed(32)).to(BF16).to(gpu_device)
    seen, native = [], _record_generation_steps(m)

    def run(hooked):
        cache = KVCache(capacity=S0 + 2)
        with torch.no_grad():
            m(x[:, :S0], kv_cache=cache)
            prompt = cache.keys.clone(), cache.values.clone()
            hook = m.qkv.linear.register_forward_hook(lambda *_: seen.append(1)) if hooked else None
            version = cache._kbuf._version
            outs = [m(x[:, t : t + 1], kv_cache=cache) for t in (S0, S0 + 1)]
            assert cache._kbuf._version > version
            if hooked:
                hook.remove()
        assert cache.length == S0 + 2 and cache.keys.shape == (b, Hkv, S0 + 2, d)
        assert torch.equal(cache.keys[:, :, :S0], prompt[0]) and torch.equal(cache.values[:, :, :S0], prompt[1])
        assert all(v.data_ptr() == cache._vbuf.data_ptr() and v.shape[2] == S0 + 1 + i for i, (_, v) in enumerate(outs))
        return torch.cat([o for o, _ in outs], 1), cache

    print(f"generation step b={b} H={H} d={d}", flush=True)
    y, cache = run(False)
    assert native == [True, True] and not seen  # both tokens were native steps
    want, want_cache = run(True)
    assert len(seen) == 2 and native == [True, True, False, False]
    with torch.no_grad(), pytest.MonkeyPatch.context() as patch:  # a layer that is replaced for all is called too
        patch.setattr(torch.nn.Linear, "forward", lambda self, t: torch.zeros(*t.shape[:-1], self.out_features, dtype=t.dtype, device=t.device))
        other = KVCache(capacity=2)
        other.append(cache.keys[:, :, :1].contiguous(), cache.values[:, :, :1].contiguous())
        assert not m(x[:, :1], kv_cache=other)[0].any() and not other.keys[:, :, 1].any()
    for a, r in ((cache.keys, want_cache.keys), (cache.values, want_cache.values)):
        assert torch.allclose(a.float(), r.float(), rtol=2.0**-7, atol=1e-5)  # neighbouring bf16 values
    assert torch.allclose(y.float(), want.float(), atol=2e-2, rtol=1e-2)
    real = _native_module().generation_step
    args = lambda xt, length: (xt, m.qkv.linear.weight, m.out.linear.weight, m.attn_gate.linear.weight if gating else None, torch.ones(1, device=gpu_device),
                               m.rope.cos, m.rope.sin, cache._kbuf, cache._vbuf, length, H, Hkv, 4, 1e-6, 2.0)
    token = x[:, :1].clone()
    with torch.no_grad():
        # accepted as it stands; what follows differs from it in one argument each
        row = cache._kbuf[:, :, 0].clone(), cache._vbuf[:, :, 0].clone()
        assert real(*args(token, 0)) is not None
        cache._kbuf[:, :, 0], cache._vbuf[:, :, 0] = row
        before = cache._kbuf.clone()
        assert real(*args(token, cache._kbuf.shape[2])) is None                       # the buffers are full
        assert real(*args(x[:, :2], 0)) is None and real(*args(token.float(), 0)) is None
        with torch.autocast("cuda", dtype=torch.float16):
            assert real(*args(token, 0)) is None
        assert torch.equal(cache._kbuf.view(torch.int16), before.view(torch.int16))
    assert real(*args(token.requires_grad_(), 0)) is None


def test_generation_step_asks_for_the_prompts_attention(gpu_device, monkeypatch):
    """eps and gate scale have one place: changed there, prompt and token change alike (the last row of a prompt is the token behind its
    other rows, within two roundings to bf16 of the projections)."""
    from sample_efficient_gpt_amd import module

    monkeypatch.setattr(module, "_EPS", 0.5)
    monkeypatch.setattr(module, "_GATE_SCALE", 3.0)
    H, Hkv, d, S = 6, 2, 64, 40
    m, _, _ = _module_and_oracle_weights(gpu_device, BF16, H * d, H, Hkv, True, False, "per-head", seed=43)
    x = torch.randn(2, S, H * d, generator=torch.Generator().manual_seed(44)).to(BF16).to(gpu_device)
    native, cache = _record_generation_steps(m), KVCache()
    with torch.no_grad():
        whole = m(x)[0][:, -1:]
        m(x[:, :-1], kv_cache=cache)
        token = m(x[:, -1:], kv_cache=cache)[0]
        monkeypatch.undo()
        before = m(x)[0][:, -1:]
    assert native == [True]
    assert (token - whole).float().norm() <= 0.01 * whole.float().norm() < 0.1 * (before - whole).float().norm()


def _record_generation_steps(m):
    """Whether each cached token that `m` is given takes the native step."""
    steps, real = [], m._generation_step

    def record(*args):
        step = real(*args)
        steps.append(step is not None)
        return step

    m._generation_step = record
    return steps


def _native_module():
    from sample_efficient_gpt_amd import _native
    return _native.load()


def test_generation_step_in_a_graph(gpu_device):
    """A captured step replayed with new tokens and eager work in between equals the eager step bit for bit."""
    H, Hkv, d, S0 = 6, 2, 64, 200
    m, _, _ = _module_and_oracle_weights(gpu_device, BF16, H * d, H, Hkv, True, False, "per-head", seed=41)
    x = torch.randn(2, S0 + 1, H * d, generator=torch.Generator().manual_seed(42)).to(BF16).to(gpu_device)
    cache, token, native = KVCache(capacity=S0 + 1), x[:, S0:].clone(), _record_generation_steps(m)

    def step():
        cache.length = S0
        return m(token, kv_cache=cache)[0]

    with torch.no_grad():
        m(x[:, :S0], kv_cache=cache)
        step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = step()
        assert native == [True, True]
        for i in range(4):
            token.copy_(torch.randn(token.shape, generator=torch.Generator().manual_seed(i)).to(BF16))
            eager = step().clone()
            row = cache.keys[:, :, S0].clone()
            cache._kbuf[:, :, S0].zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, eager) and torch.equal(cache._kbuf[:, :, S0], row), i


def test_mhsa_module_prefill_with_grad_then_cached_steps_without(gpu_device):
    """A prefill that runs with gradients enabled (its mixed values are not kept in the cache) followed by
    generation steps under no_grad: the first cached step mixes every row the cache is still missing, and the value
    tensor handed on equals the full pass's."""
    H, Hkv, d, S0, S = 6, 2, 64, 70, 73
    b, d_model = 1, H * d
    m, w, rope = _module_and_oracle_weights(gpu_device, BF16, d_model, H, Hkv, True, True, "per-head", seed=19)
    xd = torch.randn(b, S, d_model, generator=torch.Generator().manual_seed(21)).to(BF16).to(gpu_device)
    with torch.no_grad():
        full, V_full = m(xd)
    cache = KVCache()
    outs = [m(xd[:, :S0], kv_cache=cache)[0].detach()]  # grad mode on: the module's parameters require grad
    assert cache.mixed_length == 0
    with torch.no_grad():
        for t in range(S0, S):
            o, V_t = m(xd[:, t : t + 1], kv_cache=cache)
            outs.append(o)
            assert cache.mixed_length == t + 1
    assert torch.allclose(torch.cat(outs, dim=1).float(), full.float(), atol=2e-2, rtol=1e-2)
    assert torch.allclose(V_t.float(), V_full.float(), atol=1e-2, rtol=1e-2)
    with pytest.raises(ValueError):
        cache.append_mixed(V_t[:, :, :2])


# ------------------------------------------------------------------ HIP graph capture of a forward + backward pair


def test_graph_replays_match_eager_step(gpu_device):
    """A captured forward + backward (the library allocates, copies and clears nothing per call) replayed
    several times, with eager work and new inputs between the replays: every replay is bit-identical to the
    eager step on the same inputs."""
    from sample_efficient_gpt_amd.plan import AttnPlan

    c = CONFIGS[4].scaled(B=1, S=640)  # gate + value residual: every kernel and the reduce stage take part
    x = make_inputs(c, device=gpu_device)
    plan = AttnPlan(x, eps=c.eps, sm_scale=c.sm_scale, gate_scale=c.gate_scale)
    outs = [plan.y, plan.lse, plan.dq, plan.dk, plan.dv, plan.dv_first, plan.dgate, plan.dg_q, plan.dg_k, plan.dcoef]

    def eager():
        plan.forward()
        plan.backward(kv_prepared=True)
        torch.cuda.synchronize()
        return [t.clone() for t in outs]

    ref0 = eager()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.forward()
        plan.backward(kv_prepared=True)
    gen_ = torch.Generator(device=gpu_device).manual_seed(5)
    for it in range(4):
        if it:  # new inputs in the bound buffers (eager kernels between the replays)
            for n in ("q", "k", "v", "d_o"):
                x[n].copy_(torch.randn(x[n].shape, generator=gen_, device=gpu_device).to(x[n].dtype))
        ref = eager() if it else ref0
        for t in outs:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(outs, ref):
            assert torch.equal(a, b), f"replay {it} differs from the eager step"


# ------------------------------------------------------------------ seeded sweep over shapes and options


def _sweep_cases(n, seed):
    import random

    rnd = random.Random(seed)
    cases = []
    for i in range(n):
        dtype = BF16 if rnd.random() < 0.7 else F32
        D = rnd.choice([64, 64, 128] if dtype == BF16 else [32, 64, 128])
        Hkv = rnd.choice([1, 2, 3])
        H = Hkv * rnd.choice([1, 2, 3, 4])
        B = rnd.choice([1, 2, 3])
        causal = rnd.random() < 0.8
        Sq = rnd.choice([1, 2, 31, 32, 33, 63, 64, 65, 100, 127, 128, 129, 191, 200, 257, 320])
        extra_k = rnd.choice([0, 0, 1, 37, 64, 150])     # keys before the first query (a cache)
        Sk = Sq + extra_k if causal else rnd.choice([1, 17, 64, 65, 130, 260])
        kw = {"causal": causal}
        if causal and extra_k:
            kw["q_start"] = extra_k
        gen_kw = {"extras": rnd.random() < 0.4, "scalar_gain": rnd.random() < 0.3, "no_gk": rnd.random() < 0.3}
        if gen_kw["extras"]:
            kw["gate_scale"] = rnd.choice([1.0, 2.0])
        if rnd.random() < 0.3:
            kw["qk_norm"] = False
        use_rope = rnd.random() < 0.4
        backward = rnd.random() < 0.75
        cases.append((i, dtype, B, H, Hkv, Sq, Sk, D, kw, gen_kw, use_rope, backward))
    return cases


@pytest.mark.parametrize("case", _sweep_cases(48, seed=2024), ids=lambda c: f"sweep{c[0]}")
def test_seeded_sweep(gpu_device, case):
    """Ragged lengths around every tile size, caches of odd lengths, GQA ratios, every optional operand, both
    dtypes, forward-only (decode kernels where the shape allows) and forward + backward.  Here
    one element in 10^4 of a tensor may exceed the tolerance, by at most a factor 2: with gate_scale 2, a value
    residual and head_dim 128 the dS entries of the first rows reach +-10 and a couple of dk entries of the
    first keys collect rounding errors of 4e-2 (the fp32 kernels agree with the oracle to 6e-6 on that case)."""
    i, dtype, B, H, Hkv, Sq, Sk, D, kw, gen_kw, use_rope, backward = case
    if use_rope:
        kw = dict(kw, rope=orc.rope_tables(Sk + Sq + 8, 10000.0, D))
    _case(gpu_device, dtype, B, H, Hkv, Sq, Sk, D, backward=backward, seed=500 + i, gen_kw=gen_kw, outliers=(1e-4, 2.0), **kw)


def test_mhsa_module_compiles_to_one_graph(gpu_device):
    """torch.compile(fullgraph=True) traces the whole module (projection, the registered attention op as one
    opaque node, gate / output projection) without a graph break; outputs and every gradient equal the eager
    module's bit for bit.  Also under non-reentrant checkpointing, as the reference wraps its layers
    (transformer.py:123-132)."""
    from torch.utils.checkpoint import checkpoint

    H, Hkv, d, S, b = 6, 2, 64, 192, 2
    m, _, _ = _module_and_oracle_weights(gpu_device, BF16, H * d, H, Hkv, True, True, "per-head", seed=13)
    m.always_return_values = True  # the layer is handed v1 here and its own V is compared too
    g = torch.Generator().manual_seed(14)
    x = torch.randn(b, S, H * d, generator=g).to(BF16).to(gpu_device)
    v1 = torch.randn(Hkv * b, S, d, generator=g).to(BF16).to(gpu_device)
    d_out = torch.randn(b, S, H * d, generator=g).to(BF16).to(gpu_device)

    def run(fn):
        m.zero_grad(set_to_none=True)
        xi, vi = x.clone().requires_grad_(True), v1.clone().requires_grad_(True)
        out, V = fn(xi, vi)
        out.backward(d_out)
        return [out.detach(), V.detach(), xi.grad, vi.grad] + [p.grad.clone() for p in m.parameters()]

    print("module: eager / compiled / checkpointed", flush=True)
    ref = run(lambda a, c: m(a, v1=c))
    mc = torch.compile(m, backend="aot_eager", fullgraph=True)
    compiled = run(lambda a, c: mc(a, v1=c))
    ckpt = run(lambda a, c: checkpoint(lambda a_, c_: m(a_, v1=c_), a, c, use_reentrant=False))
    torch.cuda.synchronize()
    for other in (compiled, ckpt):
        for r, o in zip(ref, other):
            assert torch.equal(r, o)


def test_mhsa_module_compiles_with_the_default_backend(gpu_device):
    """`torch.compile(module)` with the DEFAULT backend (inductor), as the reference compiles its model
    (trainer.py:227-228 `model.compile()`): the attention op stays one opaque call into the HIP library while the
    code around it is generated; outputs and gradients equal the eager module's within the bf16 tolerance (inductor
    may fuse and reorder the elementwise code around the GEMMs, so bit equality is not asked for).  Skipped, with the
    reason, where inductor's own toolchain cannot run on the box."""
    H, Hkv, d, S, b = 6, 2, 64, 192, 2
    m, _, _ = _module_and_oracle_weights(gpu_device, BF16, H * d, H, Hkv, True, True, "per-head", seed=31)
    g = torch.Generator().manual_seed(32)
    x = torch.randn(b, S, H * d, generator=g).to(BF16).to(gpu_device)
    d_out = torch.randn(b, S, H * d, generator=g).to(BF16).to(gpu_device)

    def run(fn):
        m.zero_grad(set_to_none=True)
        xi = x.clone().requires_grad_(True)
        out, V = fn(xi)
        out.backward(d_out)
        torch.cuda.synchronize()
        return [out.detach().float(), V.detach().float(), xi.grad.float()] + [p.grad.float().clone() for p in m.parameters()]

    eager = run(m)
    try:
        compiled_m = torch.compile(m)  # default backend
        comp = run(compiled_m)
    except Exception as e:  # inductor needs a working triton / C++ toolchain at run time
        name = type(e).__name__
        if any(k in (name + str(e)) for k in ("BackendCompilerFailed", "InductorError", "triton", "Triton", "CppCompileError", "compiler")):
            pytest.skip(f"inductor cannot compile on this box: {name}: {str(e)[:300]}")
        raise
    for a, c in zip(eager, comp):
        scale = float(a.abs().max())
        assert torch.allclose(c, a, atol=2e-2 + 1e-2 * scale * 0, rtol=1e-2) or float((c - a).abs().max()) <= 2e-2 + 1e-2 * scale, \
            f"compiled vs eager: max abs diff {float((c - a).abs().max()):.3e} (scale {scale:.3e})"


def test_compiled_module_without_grad_takes_the_inference_route(gpu_device):
    """Under no_grad the compiled module (aot_eager: the registered op stays one opaque node, its `inference` argument is
    decided while tracing, in the caller's grad mode) equals the eager module bit for bit, for a prefill-shaped call and
    for a decode-shaped one (few query rows against many keys: the split-key kernels)."""
    H, Hkv, d, b = 6, 2, 64, 2
    m, _, _ = _module_and_oracle_weights(gpu_device, BF16, H * d, H, Hkv, True, True, "per-head", seed=41)
    g = torch.Generator().manual_seed(42)
    x = torch.randn(b, 200, H * d, generator=g).to(BF16).to(gpu_device)
    cm = torch.compile(m, backend="aot_eager")
    with torch.no_grad():
        e_out, e_V = m(x)
        c_out, c_V = cm(x)
        assert torch.equal(e_out, c_out) and torch.equal(e_V, c_V)
        # decode-shaped: one new token against a 333-key cache, through the op directly (the cache object is host state)
        q = torch.randn(b, H, 1, d, generator=g).to(BF16).to(gpu_device)
        k = torch.randn(b, Hkv, 333, d, generator=g).to(BF16).to(gpu_device)
        v = torch.randn(b, Hkv, 333, d, generator=g).to(BF16).to(gpu_device)
        f = lambda q, k, v: qknorm_attention_op(q, k, v, m.sdpa_qknorm.gain, None, q_start=332)
        assert torch.equal(f(q, k, v), torch.compile(f, backend="aot_eager", fullgraph=True)(q, k, v))
        assert torch.equal(f(q, k, v), qknorm_attention(q, k, v, m.sdpa_qknorm.gain, None, q_start=332))


def test_dropin_with_every_trailing_positional_equals_canonical_call(gpu_device):
    """The flattened drop-in with k_gain, v_first, vr_coef, gate_logits, gate_scale, n_kv_heads, eps, sm_scale and
    the rope tables against the canonical-layout call on the same data: same kernels, so outputs and every
    gradient (in the order of the positionals) agree bit for bit."""
    B, H, Hkv, S, D = 2, 6, 2, 200, 64
    x = gen(B, H, Hkv, S, S, D, BF16, extras=True, seed=31)
    d = gpu_device
    cos, sin = (t.float().to(d) for t in orc.rope_tables(S, 10000.0, D))
    names = ["q", "k", "v", "g_q", "g_k", "v_first", "vr_coef", "gate_logits"]
    t = {n: x[n].to(d).requires_grad_(True) for n in names}
    y = qknorm_attention(t["q"], t["k"], t["v"], t["g_q"], t["g_k"], v_first=t["v_first"], vr_coef=t["vr_coef"],
                         gate_logits=t["gate_logits"], gate_scale=2.0, eps=1e-5, sm_scale=0.11, rope_cos=cos, rope_sin=sin)
    y.backward(x["d_o"].to(d))
    flat = lambda a, h: orc.flatten_heads(a).contiguous()
    f = {"Q": flat(x["q"], H), "K": flat(x["k"], Hkv), "V": flat(x["v"], Hkv), "VF": flat(x["v_first"], Hkv)}
    f = {n: a.to(d).requires_grad_(True) for n, a in f.items()}
    p = {n: x[n].to(d).requires_grad_(True) for n in ("g_q", "g_k", "vr_coef", "gate_logits")}
    O = QKNormFlashAttnFunc.apply(f["Q"], f["K"], f["V"], p["g_q"], True, 0, p["g_k"], f["VF"], p["vr_coef"], p["gate_logits"],
                                  2.0, Hkv, 1e-5, 0.11, cos, sin)
    O.backward(flat(x["d_o"], H).to(d))
    torch.cuda.synchronize()
    assert torch.equal(O, flat(y.detach(), H))
    assert torch.equal(f["Q"].grad, flat(t["q"].grad, H)) and torch.equal(f["K"].grad, flat(t["k"].grad, Hkv))
    assert torch.equal(f["V"].grad, flat(t["v"].grad, Hkv)) and torch.equal(f["VF"].grad, flat(t["v_first"].grad, Hkv))
    for n in ("g_q", "g_k", "vr_coef", "gate_logits"):
        assert torch.equal(p[n].grad, t[n].grad), n


@pytest.mark.parametrize("B,S,steps", [(8, 2048, 100), (21, 768, 300), (42, 384, 300)])
def test_full_size_steps_repeat_bit_for_bit(gpu_device, B, S, steps):
    """Forward + backward steps at the IMU-1 size, and at two of the reference's shorter training contexts with the
    same number of tokens, on one set of buffers: every output of every step equals the first step's bit for bit
    (no atomics, fixed reduction orders, no stray LDS traffic, and no tile read before it has landed: short
    contexts have the most workgroup start-ups per step, which is where a missing wait in the tile pipeline
    showed, in 8 % of the steps at S = 768)."""
    from sample_efficient_gpt_amd.plan import AttnPlan

    c = CONFIGS[3].scaled(B=B, S=S)
    x = make_inputs(c, device=gpu_device)
    plan = AttnPlan(x, eps=c.eps, sm_scale=c.sm_scale)
    outs = [plan.y, plan.lse, plan.dq, plan.dk, plan.dv, plan.dg_q, plan.dg_k]
    plan.forward()
    plan.backward(kv_prepared=True)
    torch.cuda.synchronize()
    ref = [t.clone() for t in outs]
    print(f"repeatability B={B} S={S}", flush=True)
    for it in range(steps):
        for t in outs[:5]:
            t.zero_()
        plan.forward()
        plan.backward(kv_prepared=True)
        for name, a, b in zip(("y", "lse", "dq", "dk", "dv", "dg_q", "dg_k"), outs, ref):
            assert torch.equal(a, b), f"step {it}: {name} differs from the first step"


@pytest.mark.parametrize("B,S,steps", [(8, 2048, 50), (21, 768, 200), (3, 1100, 200)])
def test_module_shaped_steps_repeat_bit_for_bit(gpu_device, B, S, steps):
    """The same on the call the attention module makes (strided views of one projection buffer, rotary embedding,
    scalar gain, gate, value residual): its kernels have start-up and epilogue phases of their own (the dQ kernel's
    two-phase start-up with the rotary table blocks, the row blocks behind the loops of dQ and dK/dV, the gate
    factor inside the row statistics); S = 1100 leaves a last query block of 76 rows."""
    import bench
    from sample_efficient_gpt_amd.plan import AttnPlan

    c = CONFIGS[3].scaled(extras=True, B=B, S=S)
    x, rope = bench.module_shaped_inputs(c, gpu_device)
    plan = AttnPlan(x, eps=c.eps, sm_scale=c.sm_scale, gate_scale=2.0, backward=True, rope_cos=rope[0], rope_sin=rope[1],
                    rope_q_pos0=0, rope_k_pos0=0)
    names = ("y", "lse", "dq", "dk", "dv", "dv_first", "dgate", "dg_q", "dcoef")
    outs = [getattr(plan, n) for n in names]
    plan.forward()
    plan.backward(kv_prepared=True)
    torch.cuda.synchronize()
    ref = [t.clone() for t in outs]
    print(f"module-shaped repeatability B={B} S={S}", flush=True)
    for it in range(steps):
        for t in outs[:7]:
            t.zero_()
        plan.forward()
        plan.backward(kv_prepared=True)
        for name, a, b in zip(names, outs, ref):
            assert torch.equal(a, b), f"step {it}: {name} differs from the first step"


def test_empty_batch_and_no_query_rows(gpu_device):
    """B = 0 and Sq = 0: empty outputs, zero gradients, nothing launched (like torch's SDPA on empty inputs)."""
    d = gpu_device
    g = torch.ones(64, device=d, requires_grad=True)
    for shape_q, shape_k in (((0, 4, 16, 64), (0, 2, 16, 64)), ((2, 4, 0, 64), (2, 2, 16, 64))):
        q = torch.empty(shape_q, dtype=BF16, device=d, requires_grad=True)
        k = torch.randn(shape_k, device=d).to(BF16).requires_grad_(True)
        v = torch.randn(shape_k, device=d).to(BF16).requires_grad_(True)
        y, lse = qknorm_attention(q, k, v, g, None, return_lse=True, causal=shape_q[2] != 0)
        assert y.shape == shape_q and lse.shape == shape_q[:3]
        y.sum().backward()
        assert q.grad.shape == shape_q and torch.count_nonzero(k.grad) == 0 and torch.count_nonzero(v.grad) == 0
        assert torch.count_nonzero(g.grad) == 0
        g.grad = None
    out = FlashAttnFunc.apply(torch.empty(0, 8, 64, dtype=BF16, device=d), torch.empty(0, 8, 64, dtype=BF16, device=d),
                              torch.empty(0, 8, 64, dtype=BF16, device=d))
    assert out.shape == (0, 8, 64)
