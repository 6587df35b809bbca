"""LayerNorm (csrc/layernorm.hip): every number of lanes per row it is built for, rows that do not fill their lanes, and several rows per group."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("rows,pieces", [(1, 1), (257, 2), (1025, 3), (300, 4), (9, 7), (50, 16), (70, 17), (16399, 32), (40, 64), (5, 65), (4, 200)])
def test_rows_match_64_bits(gpu_device, rows, pieces, dtype):
    from evoformer_triton_amd.block import _LayerNorm
    cols = pieces * (16 // dtype.itemsize)   # a row's 16-byte pieces
    g = torch.Generator().manual_seed(11)
    x, dy = ((torch.randn((rows, cols), generator=g) + 0.3).to(dtype).to(gpu_device) for _ in range(2))
    w, b = ((1.0 + 0.2 * torch.randn(cols, generator=g)).to(dtype).to(gpu_device) for _ in range(2))
    leaves = [t.requires_grad_() for t in (x, w, b)]
    y = _LayerNorm.apply(*leaves, 1e-5)
    got = (y, *torch.autograd.grad(y, leaves, dy))
    ref = [t.detach().double().requires_grad_() for t in leaves]
    y64 = torch.nn.functional.layer_norm(ref[0], (cols,), ref[1], ref[2], 1e-5)
    want = (y64, *torch.autograd.grad(y64, ref, dy.double()))
    # y and dx, of a row alone: their own rounding (u), and some sums of `cols` terms in fp32, each within 2^-24 (1 + sqrt(cols) / 4) of the sum of the sizes of its terms
    # (16 lanes' partial sums and more, random signs: a plain chain's bound is cols).  mean, 1 / std and xhat carry four such roundings, dx's two sums one each;
    # sizes: |xhat| + |mean| / std of a row for xhat, |dy w| (1 + |xhat|) / std for dx.  dw and db: `rows` such terms.
    u, f = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23, 2.0 ** -24
    x64, dy64, w64 = ref[0].detach(), dy.double(), ref[1].detach()
    mu, std = x64.mean(1, keepdim=True), (x64.var(1, keepdim=True, unbiased=False) + 1e-5).sqrt()
    xhat = ((x64 - mu) / std).abs()
    row = 4 * (1 + cols ** 0.5 / 4) * f * (1 + mu.abs() / std) * (1 + xhat)
    g64 = (dy64 * w64).abs()
    bounds = {"y": row * w64.abs() + f * y64.abs(), "dx": 4 * row * (g64 + g64.mean(1, keepdim=True) + xhat * (g64 * xhat).mean(1, keepdim=True)) / std,
              "dw": ((dy64.abs() * (row + f * rows ** 0.5 * xhat)).sum(0)), "db": f * rows ** 0.5 * dy64.abs().sum(0)}
    for name, a, c in zip(("y", "dx", "dw", "db"), got, want):
        off = (a.double() - c).abs()
        assert (off <= u * c.abs() + bounds[name]).all(), (name, (off / (u * c.abs() + bounds[name])).max().item())


def test_weight_gradients_in_fp32_come_from_1024_partial_sums(gpu_device):
    """With half as many each is a sum of twice as many rows one after the other, and further from 64 bits: read from what the call leaves in its workspace."""
    import ctypes
    from evoformer_triton_amd import _lib
    lib, rows, cols = _lib.load(), 8192, 256
    x, dy = (torch.randn((rows, cols), device=gpu_device) for _ in range(2))
    mean, rstd, dw, db = x.mean(1), 1.0 / x.std(1), torch.empty(cols, device=gpu_device), torch.empty(cols, device=gpu_device)
    n = lib.evoattn_layernorm_bwd_workspace_bytes(rows, cols, _lib.EVO_F32)
    ws = torch.full((n // 4,), float("nan"), device=gpu_device)
    assert lib.evoattn_layernorm_bwd(dy.data_ptr(), x.data_ptr(), None, mean.data_ptr(), rstd.data_ptr(), None, dw.data_ptr(), db.data_ptr(), ws.data_ptr(), n, rows, cols,
                                     _lib.EVO_F32, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    assert torch.isfinite(ws).sum().item() == 1024 * 2 * cols and torch.isfinite(dw).all()
