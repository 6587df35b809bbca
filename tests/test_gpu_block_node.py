"""The block as one call and one autograd node (csrc/host.cpp): the layer-by-layer form's bits, whatever is asked for."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _block(dev, gating, c_z, seed=4):
    from evoformer_triton_amd.block import GatedAttentionBlock
    torch.manual_seed(seed)
    blk = GatedAttentionBlock(64, 32, 4, c_z=c_z, gating=gating).to(dev).to(torch.bfloat16)
    m = torch.randn(2, 5, 72, 64, device=dev).to(torch.bfloat16).requires_grad_()
    z = torch.randn(2, 72, 72, c_z, device=dev).to(torch.bfloat16).requires_grad_() if c_z else None
    keep = torch.rand(2, 5, 72, device=dev) < 0.9
    return blk, m, z, keep, torch.randn(2, 5, 72, 64, device=dev).to(torch.bfloat16)


@pytest.mark.parametrize("gating,c_z,mask", [(True, 64, "float"), (False, 128, "bool"), (True, None, None)])
def test_one_node_gives_the_layers_bits(gpu_device, gating, c_z, mask):
    blk, m, z, keep, dout = _block(gpu_device, gating, c_z)
    keep = None if mask is None else keep.float() if mask == "float" else keep
    leaves = [t for t in (m, z) if t is not None] + list(blk.parameters())
    y = blk(m, z, keep)
    assert y.grad_fn.name() == "GatedAttentionBlockBackward"
    got = torch.autograd.grad(y, leaves, dout, retain_graph=True)
    again = torch.autograd.grad(y, leaves, dout)
    blk._native = lambda *a: None
    want_y = blk(m, z, keep)
    want = torch.autograd.grad(want_y, leaves, dout)
    assert torch.equal(y, want_y)
    for a, b, c in zip(got, again, want):
        assert torch.equal(a, c) and torch.equal(b, c)
    del blk._native
    for i in range(len(leaves)):      # one gradient at a time (without the bias' another kernel forms dQ)
        one, = torch.autograd.grad(blk(m, z, keep), [leaves[i]], dout)
        assert (one.float() - want[i].float()).norm() <= 1e-2 * want[i].float().norm() + 1e-3 * want[i].numel() ** 0.5, i


def test_calls_that_the_node_does_not_take_go_the_layers_way(gpu_device):
    blk, m, z, keep, _ = _block(gpu_device, True, 64)
    y = blk(m, z, keep)
    soft = keep.float().requires_grad_()
    for other in (blk(m, z, soft), blk(m.detach().transpose(1, 2).contiguous().transpose(1, 2), z, keep)):
        assert "GatedAttentionBlock" not in other.grad_fn.name() and torch.equal(other, y)
