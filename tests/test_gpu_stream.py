"""The kernels whose rows stream through LDS (csrc/mfma_stream.hip, head dims from 32 on) at the edges of their stages, against eager in fp32."""
import pytest
import torch

from oracle import eager

pytestmark = pytest.mark.gpu

CASES = [  # B, S, N, H, D, mask, bias, layout, gated, dtype
    (1, 1, 1, 1, 64, None, "q", "reference", False, torch.bfloat16),
    (1, 6, 31, 2, 128, "bool", "q", "ds4sci", False, torch.float16),
    (2, 5, 64, 1, 64, "dead", "f32", "reference", False, torch.bfloat16),
    (1, 9, 65, 2, 128, "soft", "f32", "reference", True, torch.bfloat16),
    (1, 70, 96, 1, 128, "bool", "q", "reference", False, torch.bfloat16),        # several chunks of rows
    (1, 2, 128, 3, 64, "soft", None, "ds4sci", True, torch.float16),
    (1, 17, 129, 2, 64, "jump", "q", "reference", False, torch.bfloat16),        # the maximum lies far above the first tile's
    (4, 1, 200, 16, 64, "bool", "f32", "reference", False, torch.bfloat16),      # the caller's bias rows, dBias written as formed
    (1, 3, 257, 2, 128, "jump", "f32", "ds4sci", False, torch.float16),
    (4, 1, 320, 16, 128, "bool", "q", "reference", False, torch.bfloat16),
    (1, 5, 1, 2, 32, "dead", None, "reference", False, torch.float16),
    (1, 40, 33, 2, 32, "soft", "q", "reference", True, torch.bfloat16),          # a second tile of one key
    (1, 33, 193, 1, 32, "jump", "q", "ds4sci", False, torch.bfloat16),
    (1, 3, 232, 1, 32, "dead", "q", "reference", False, torch.float16),          # too few S rows for a resident bias
    (1, 70, 232, 8, 32, "bool", "q", "reference", False, torch.bfloat16),
    (1, 6, 264, 2, 32, "soft", "f32", "reference", True, torch.bfloat16),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_stream_kernels_match_eager(gpu_device, case):
    import evoformer_triton_amd.evoformer as E
    B, S, N, H, D, mask, bias, layout, gated, dt = case
    g = torch.Generator().manual_seed(23)
    Q, K, V, G, dO = ((torch.randn((B, S, N, H, D), generator=g) * 0.7).to(dt) for _ in range(5))
    keep = torch.rand((B, S, 1, 1, N), generator=g) < 0.85
    keep[..., 0] = True
    if mask == "dead":
        keep[0, 1] = False
    m = keep if mask in ("bool", "dead") else torch.randn((B, S, 1, 1, N), generator=g) if mask == "soft" else None
    b = None if bias is None else torch.randn((B, 1, H, N, N), generator=g) * 0.5
    if mask == "jump":
        b[..., N // 2:] += 30.0
    b = None if b is None else b.to(torch.float32 if bias == "f32" else dt)
    fmask = mask == "soft"
    ref = eager.attention_fwd_bwd(Q, K, V, m, b, dO, layout=layout, compute_dtype=torch.float32, gate=G if gated else None)
    dev = gpu_device
    q, k, v, gg = (t.to(dev).requires_grad_() for t in (Q, K, V, G))
    bb = None if b is None else b.to(dev).requires_grad_()
    mm = None if m is None else (m.to(dev).requires_grad_() if fmask else m.to(dev))
    o = E.evoformer_attention(q, k, v, mm, bb, layout=layout, gate=gg if gated else None)
    o.backward(dO.to(dev))
    got = {"Og" if gated else "O": o, "dQ": q.grad, "dK": k.grad, "dV": v.grad}
    if bb is not None:
        got["dBias"] = bb.grad
    if fmask:
        got["dMask"] = mm.grad
    if gated:
        got["dGate"] = gg.grad
    for name, t in got.items():
        want = ref[name].float()
        d = t.detach().float().cpu() - want
        assert torch.isfinite(d).all(), name
        assert d.norm() <= 1.5e-2 * want.norm() + 1e-4 * want.numel() ** 0.5, (name, (d.norm() / want.norm()).item())
