"""Hooks on saved tensors (torch.autograd.graph.save_on_cpu and the like) hand the backward copies, dense where the caller's mask
and bias were views of wider tensors and where an output was a slot of a buffer: the gradients are those without hooks."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _views(B, S, N, H, dt, dev, g):
    """A mask and a bias whose rows lie apart."""
    mask = torch.randn((B, S + 1, 1, 1, 2 * N), generator=g).to(dev)[:, :S, :, :, :N]
    bias = torch.randn((B, 1, H, N, N + 8), generator=g).to(dt).to(dev)[..., :N]
    assert not bias.is_contiguous() and (S == 1 or not mask.is_contiguous())
    return mask, bias


def _same(run):
    want = run()
    with torch.autograd.graph.save_on_cpu():
        got = run()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("case", [(1, 3, 40, 2, 32, "reference", False, torch.bfloat16), (2, 6, 136, 2, 16, "ds4sci", True, torch.float16),
                                  (1, 1, 72, 4, 64, "reference", False, torch.bfloat16),       # the caller's rows, dBias as formed
                                  (1, 3, 40, 2, 24, "reference", True, torch.bfloat16),        # padded: the path in Python
                                  (1, 2, 33, 2, 32, "ds4sci", False, torch.float32)], ids=str)
def test_attention(gpu_device, case):
    import evoformer_triton_amd.evoformer as E
    B, S, N, H, D, layout, gated, dt = case
    g = torch.Generator().manual_seed(47)
    q, k, v, gate, dO = (torch.randn((B, S, N, H, D), generator=g).to(dt).to(gpu_device) for _ in range(5))
    mask, bias = _views(B, S, N, H, dt, gpu_device, g)

    def run():
        leaves = [t.detach().requires_grad_() for t in (q, k, v, mask, bias)] + ([gate.detach().requires_grad_()] if gated else [])
        o = E.evoformer_attention(*leaves[:5], layout=layout, gate=leaves[5] if gated else None)
        return torch.autograd.grad(o, leaves, dO)

    _same(run)


@pytest.mark.parametrize("gated", [True, False])
def test_slots(gpu_device, gated):
    import evoformer_triton_amd.evoformer as E
    g = torch.Generator().manual_seed(48)
    P = torch.randn((1, 3, 40, 4 if gated else 3, 2, 32), generator=g).to(torch.bfloat16).to(gpu_device)
    mask, bias = _views(1, 3, 40, 2, torch.bfloat16, gpu_device, g)

    def run():
        p, b = P.detach().requires_grad_(), bias.detach().requires_grad_()
        out, _ = E.slot_attention(p, mask, b, gated=gated)
        return torch.autograd.grad(out, [p, b], torch.ones_like(out))

    _same(run)


@pytest.mark.parametrize("native", [True, False], ids=["one_node", "layers"])
def test_block(gpu_device, native):
    from evoformer_triton_amd.block import GatedAttentionBlock
    torch.manual_seed(4)
    blk = GatedAttentionBlock(64, 32, 4, c_z=64).to(gpu_device).to(torch.bfloat16)
    if not native:
        blk._native = lambda *a: None
    m = torch.randn(2, 5, 72, 64, device=gpu_device).to(torch.bfloat16).requires_grad_()
    z = torch.randn(2, 72, 72, 64, device=gpu_device).to(torch.bfloat16).requires_grad_()
    leaves = [m, z, *blk.parameters()]
    _same(lambda: torch.autograd.grad(blk(m, z, None), leaves, torch.ones_like(m)))
