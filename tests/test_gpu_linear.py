"""The Linear kernels (csrc/linear.hip) at the edges of their tiles, against products in fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # rows, k, weights, outputs per weight, bias, dtype
    (1, 64, 1, 64, True, torch.bfloat16),
    (127, 128, 2, 64, False, torch.float16),         # outputs that do not fill a tile
    (129, 192, 3, 64, True, torch.bfloat16),         # a tile of one row; 192 of a 128-wide tile
    (300, 256, 4, 128, True, torch.bfloat16),        # slices of the weight gradient whose last stage is partial
    (5000, 320, 1, 448, True, torch.float16),
    (129, 4096, 1, 64, True, torch.bfloat16),        # a contraction of 64 stages, the most that y and dx are given here ..
    (129, 4160, 2, 64, False, torch.bfloat16),       # .. and of 65: the library's product for y, ..
    (129, 128, 1, 4160, True, torch.bfloat16),       # .. for dx, ..
    (300, 1024, 2, 2112, True, torch.bfloat16),      # .. and for a weight gradient too wide to keep in fp32 per slice
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_linear_kernels_match_fp32_products(gpu_device, case):
    from evoformer_triton_amd import _lib
    rows, k, nw, n, with_bias, dt = case
    g = torch.Generator().manual_seed(31)
    x, dy = torch.randn((rows, k), generator=g).to(dt), torch.randn((rows, nw * n), generator=g).to(dt)
    ws = [(torch.randn((n, k), generator=g) * k ** -0.5).to(dt) for _ in range(nw)]
    b = torch.randn((n,), generator=g).to(dt) if with_bias else None
    ref = [t.float().requires_grad_() for t in [x, *ws] + ([b] if with_bias else [])]
    want = torch.cat([torch.nn.functional.linear(ref[0], w, ref[-1] if with_bias and i == nw - 1 else None) for i, w in enumerate(ref[1:1 + nw])], -1)
    want_g = torch.autograd.grad(want, ref, dy.float())
    leaves = [t.to(gpu_device).requires_grad_() for t in [x, *ws] + ([b] if with_bias else [])]
    bias = leaves[-1] if with_bias else None
    calls = [lambda: _lib.host().stacked_projection(leaves[0], bias, leaves[1:1 + nw])]
    if nw == 1:   # the same as a single layer, its input gradient written into rows that lie apart
        place = torch.zeros((rows, k + 8), dtype=dt, device=gpu_device)
        calls.append(lambda: _lib.host().linear(leaves[0], leaves[1], bias, place[:, :k] if k % 8 == 0 else None))
    for call in calls:
        y = call()
        got = torch.autograd.grad(y, leaves, dy.to(gpu_device))
        for name, a, w in [("y", y, want)] + [(str(i), a, w) for i, (a, w) in enumerate(zip(got, want_g))]:
            d = a.detach().float().cpu() - w.detach()
            assert torch.isfinite(d).all() and d.norm() <= 1e-2 * w.detach().norm() + 1e-5 * w.numel() ** 0.5, (name, (d.norm() / w.detach().norm()).item())
    if nw == 1:
        assert not place[:, k:].any().item()
