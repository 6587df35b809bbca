"""The pair bias kernels (csrc/pair_bias.hip) at the edges of their tiles, against the separate steps in fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # B, N, C, H, affine, dtype
    (1, 1, 64, 1, True, torch.bfloat16),
    (1, 5, 128, 8, True, torch.float16),          # a wave's 32 rows not filled
    (2, 11, 128, 4, False, torch.bfloat16),       # batches meet inside a wave
    (3, 12, 64, 16, True, torch.bfloat16),
    (1, 67, 256, 5, True, torch.bfloat16),
    (1, 263, 128, 8, True, torch.bfloat16),       # more rows than the backward has workgroups for in one turn
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_pair_bias_matches_the_separate_steps(gpu_device, case):
    from evoformer_triton_amd import _lib
    B, N, C, H, affine, dt = case
    g = torch.Generator().manual_seed(29)
    z, dout = torch.randn((B, N, N, C), generator=g), torch.randn((B, 1, H, N, N), generator=g)
    w = torch.randn((H, C), generator=g) * C ** -0.5
    lw, lb = (1.0 + 0.3 * torch.randn((C,), generator=g), 0.3 * torch.randn((C,), generator=g)) if affine else (None, None)
    leaves = [None if t is None else t.to(dt).to(gpu_device).requires_grad_() for t in (z, lw, lb, w)]
    out = _lib.host().pair_bias(leaves[0], leaves[1], leaves[2], 1e-5, leaves[3])
    assert out is not None and tuple(out.shape) == (B, 1, H, N, N)
    out.backward(dout.to(dt).to(gpu_device))
    ref = [None if t is None else t.to(dt).float().requires_grad_() for t in (z, lw, lb, w)]
    y = torch.nn.functional.layer_norm(ref[0], (C,), ref[1], ref[2], 1e-5)
    want = torch.nn.functional.linear(y, ref[3]).permute(0, 3, 1, 2).unsqueeze(1)
    want.backward(dout.to(dt).float())
    for name, a, b in [("out", out, want)] + [(n, a.grad, b.grad) for n, a, b in zip(("z", "ln_weight", "ln_bias", "weight"), leaves, ref) if a is not None]:
        d = a.detach().float().cpu() - b.detach()
        assert torch.isfinite(d).all() and d.norm() <= 1e-2 * b.detach().norm() + 1e-4 * b.numel() ** 0.5, (name, (d.norm() / b.detach().norm()).item())
    # only some gradients wanted
    part = torch.autograd.grad(_lib.host().pair_bias(leaves[0], leaves[1], leaves[2], 1e-5, leaves[3]), [leaves[3]], dout.to(dt).to(gpu_device))[0]
    assert torch.equal(part, leaves[3].grad)
