"""The C++ host path of the operator against the Python one: same kernels, same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # B, S, N, H, D, mask, bias, per_head, gated, dtype
    (1, 1, 1, 1, 8, None, None, False, False, torch.bfloat16),
    (2, 3, 33, 2, 32, "f64", "f16", False, False, torch.bfloat16),      # operands of foreign dtypes, widened
    (2, 3, 40, 2, 16, "one", "shared", True, False, torch.float16),     # broadcast over the batch and the rows
    (1, 4, 200, 3, 64, "bool", "strided", True, True, torch.bfloat16),
    (2, 2, 24, 2, 128, "int", "same", False, True, torch.float32),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_both_host_paths_give_the_same_bits(gpu_device, case, monkeypatch):
    import evoformer_triton_amd.evoformer as E
    B, S, N, H, D, mask, bias, per_head, gated, dt = case
    g = torch.Generator().manual_seed(3)
    q, k, v, gate, dO = (torch.randn((B, S, N, H, D), generator=g).to(dt).to(gpu_device) for _ in range(5))
    keep = torch.rand((1 if mask == "one" else B, 1 if mask == "one" else S, 1, 1, N), generator=g) < 0.8
    keep[..., 0] = True
    m = None if mask is None else {"bool": keep, "int": keep.long(), "f64": torch.where(keep, 0.25, -1e9).double(),
                                   "one": torch.where(keep, 0.5, -1e9)}[mask].to(gpu_device)
    b = None
    if bias is not None:
        b = torch.randn((1 if bias == "shared" else B, 1, H, N, N * (2 if bias == "strided" else 1)), generator=g)
        b = b.to(torch.float16 if bias == "f16" else dt).to(gpu_device)
        b = b[..., ::2] if bias == "strided" else b
    fmask = m is not None and m.is_floating_point()

    def run():
        leaves = [t.detach().clone().requires_grad_() for t in (q, k, v)] + ([gate.detach().clone().requires_grad_()] if gated else [])
        bb = None if b is None else b.detach().requires_grad_()
        mm = m.detach().requires_grad_() if fmask else m
        o = E.evoformer_attention(*leaves[:3], mm, bb, layout="ds4sci" if per_head else "reference", gate=leaves[3] if gated else None)
        return [o, *torch.autograd.grad(o, leaves + ([] if bb is None else [bb]) + ([mm] if fmask else []), dO)]

    got = run()
    monkeypatch.setattr(E, "_native", lambda *a: None)
    want = run()
    for a, w in zip(got, want):
        assert a.shape == w.shape and a.dtype == w.dtype and torch.equal(a, w)


def test_the_native_node_is_once_differentiable(gpu_device):
    import evoformer_triton_amd.evoformer as E
    q = torch.randn((1, 2, 32, 2, 32), device=gpu_device).requires_grad_()
    o = E.EvoformerAttention.apply(q, q, q, None, None)
    (dq,) = torch.autograd.grad(o, q, torch.ones_like(o), create_graph=True)
    with pytest.raises(RuntimeError, match="once_differentiable"):
        dq.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(o, q, torch.ones_like(o))
        torch.autograd.grad(o, q, torch.ones_like(o))


def test_what_the_native_path_does_not_take(gpu_device):
    """Head dims that need padding go the Python way; invalid arguments keep their errors."""
    import evoformer_triton_amd.evoformer as E
    q = torch.randn((1, 2, 32, 2, 24), device=gpu_device, dtype=torch.bfloat16).requires_grad_()
    o = E.EvoformerAttention.apply(q, q, q)
    assert o.shape == q.shape and torch.isfinite(torch.autograd.grad(o, q, torch.ones_like(o))[0]).all()
    p = torch.randn((1, 2, 32, 2, 32), device=gpu_device, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="res_mask"):
        E.EvoformerAttention.apply(p, p, p, torch.zeros(1, 2, 1, 1, 31, device=gpu_device), None)
    with pytest.raises(ValueError, match="pair_bias"):
        E.EvoformerAttention.apply(p, p, p, None, torch.zeros(1, 1, 3, 32, 32, device=gpu_device))
    with pytest.raises(RuntimeError, match="same device"):
        E.EvoformerAttention.apply(p, p, p, torch.zeros(1, 2, 1, 1, 32), None)


def _gpu_block(dev):
    from evoformer_triton_amd.block import GatedAttentionBlock
    torch.manual_seed(4)
    blk = GatedAttentionBlock(64, 32, 4, c_z=64).to(dev).to(torch.bfloat16)
    m = torch.randn(1, 3, 40, 64, device=dev).to(torch.bfloat16)
    z = torch.randn(1, 40, 40, 64, device=dev).to(torch.bfloat16)
    return blk, m, z


def _attention_operands(dev):
    g = torch.Generator().manual_seed(5)
    q = [torch.randn((1, 3, 40, 4, 32), generator=g).to(torch.bfloat16).to(dev) for _ in range(4)]
    return q, torch.randn((1, 3, 1, 1, 40), generator=g).to(dev), torch.randn((1, 1, 4, 40, 40), generator=g).to(torch.bfloat16).to(dev)


@pytest.mark.parametrize("which", ["q", "v", "mask", "bias", "gate"])
def test_a_forward_mode_tangent_is_refused_by_the_attention(gpu_device, which):
    import evoformer_triton_amd.evoformer as E
    from torch.autograd import forward_ad
    (q, k, v, gate), mask, bias = _attention_operands(gpu_device)
    args = {"q": q, "k": k, "v": v, "mask": mask, "bias": bias, "gate": gate}
    with forward_ad.dual_level():
        args[which] = forward_ad.make_dual(args[which], torch.ones_like(args[which]))
        with pytest.raises(NotImplementedError, match="jvp|forward mode"):
            E.evoformer_attention(args["q"], args["k"], args["v"], args["mask"], args["bias"], gate=args["gate"] if which == "gate" else None)


def test_a_forward_mode_tangent_is_refused_by_the_block_and_its_slots(gpu_device):
    import evoformer_triton_amd.evoformer as E
    from torch.autograd import forward_ad
    blk, m, z = _gpu_block(gpu_device)
    dual = lambda t: forward_ad.make_dual(t.detach(), torch.ones_like(t))
    with forward_ad.dual_level():
        for args in ((dual(m), z), (m, dual(z))):
            with pytest.raises(NotImplementedError, match="jvp|forward mode"):
                blk(*args)
        for name in ("linear_q.weight", "linear_g.bias", "linear_o.weight", "linear_o.bias", "linear_z.weight"):
            with pytest.raises(NotImplementedError, match="jvp|forward mode"):
                torch.func.functional_call(blk, {name: dual(blk.get_parameter(name))}, (m, z))
        P = torch.randn((1, 3, 40, 3, 2, 32), device=gpu_device).to(torch.bfloat16)
        with pytest.raises(NotImplementedError, match="forward mode"):
            E.slot_attention(dual(P))


def test_traced_calls_compute_on_replay(gpu_device):
    """torch.jit's tracer has to see operators that launch: a module traced through calls that it cannot look into returns
    memory that nobody wrote."""
    import evoformer_triton_amd.evoformer as E
    (q, k, v, gate), mask, bias = _attention_operands(gpu_device)
    P = torch.stack([q, k, v, gate], 3).contiguous()
    blk, m, z = _gpu_block(gpu_device)
    keep = torch.ones(m.shape[:3], device=gpu_device)
    calls = {
        "flat": (lambda q, k, v, bias: E.EvoformerAttention.apply(q, k, v, mask, bias), (q, k, v, bias)),
        "per head": (lambda q, k, v, bias: E.DS4Sci_EvoformerAttention(q, k, v, [mask, bias]), (q, k, v, bias)),
        "gated": (lambda q, k, v, gate: E.evoformer_attention(q, k, v, mask, bias, gate=gate), (q, k, v, gate)),
        "slots": (lambda P: E.slot_attention(P, mask, bias, gated=True)[0], (P,)),
        "block": (blk, (m, z, keep)),
    }
    for name, (call, args) in calls.items():
        traced = torch.jit.trace(call, args, check_trace=False)
        new = tuple(t.flip(-1).contiguous() for t in args)
        with torch.no_grad():
            got, want = traced(*new).float(), call(*new).float()
        # (the block and its slots go another way under the tracer: their results differ by roundings to bf16)
        assert torch.isfinite(got).all() and (got - want).norm() <= 1e-2 * want.norm(), name
        assert "^" in str(traced.graph) or "^" in str(traced.inlined_graph), name


def test_the_flags_reach_the_slots_and_the_block(gpu_device, monkeypatch):
    """`FLAGS` selects kernels for every call: with the plain fp32-arithmetic kernels the results differ by roundings."""
    import evoformer_triton_amd.evoformer as E
    from evoformer_triton_amd import _lib
    (q, k, v, gate), mask, bias = _attention_operands(gpu_device)
    P = torch.stack([q, k, v, gate], 3).contiguous()
    blk, m, z = _gpu_block(gpu_device)

    def run():
        p, mm = P.detach().requires_grad_(), m.detach().requires_grad_()
        out, _ = E.slot_attention(p, mask, bias, gated=True)
        y = blk(mm, z)
        return [out, *torch.autograd.grad(out, p, torch.ones_like(out)), y, *torch.autograd.grad(y, mm, torch.ones_like(y))]

    got = run()
    monkeypatch.setattr(E, "FLAGS", _lib.EVO_FLAG_FORCE_GENERIC)
    want = run()
    for a, b in zip(got, want):
        assert not torch.equal(a, b) and (a.float() - b.float()).norm() <= 2e-2 * b.float().norm()
    ref = E.evoformer_attention(q, k, v, mask, bias, layout="ds4sci", gate=gate)
    assert torch.equal(want[0], ref)
