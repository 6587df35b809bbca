"""The forward whose waves split a row's keys (csrc/mfma_stream.hip, calls without a backward), against eager in fp32."""
import pytest
import torch

from oracle import eager

pytestmark = pytest.mark.gpu

CASES = [  # B, N, H, D, mask, bias, layout, gated, dtype
    (1, 1, 1, 32, None, "q", "reference", False, torch.bfloat16),
    (2, 31, 3, 64, "bool", "f32", "reference", False, torch.float16),
    (3, 33, 2, 128, "dead", "q", "ds4sci", False, torch.bfloat16),         # a wave with one key, two with none
    (1, 128, 16, 64, "bool", "f32", "reference", False, torch.bfloat16),
    (1, 129, 4, 32, "soft", "q", "ds4sci", True, torch.float16),
    (2, 250, 4, 64, "dead", "f32", "reference", True, torch.bfloat16),     # rows that no four-wide load fits
    (1, 516, 2, 128, "jump", "f32", "ds4sci", False, torch.bfloat16),
    (1, 700, 5, 32, "soft16", None, "reference", False, torch.bfloat16),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_split_forward_matches_eager(gpu_device, case):
    import evoformer_triton_amd.evoformer as E
    B, N, H, D, mask, bias, layout, gated, dt = case
    g = torch.Generator().manual_seed(37)
    Q, K, V, G = ((torch.randn((B, 1, N, H, D), generator=g) * 0.7).to(dt) for _ in range(4))
    keep = torch.rand((B, 1, 1, 1, N), generator=g) < 0.85
    keep[..., 0] = True
    if mask == "dead":
        keep[0] = False
    m = keep if mask in ("bool", "dead") else torch.randn((B, 1, 1, 1, N), generator=g) if mask in ("soft", "soft16") else None
    m = m.to(dt) if mask == "soft16" else m
    b = None if bias is None else torch.randn((B, 1, H, N, N), generator=g) * 0.5
    if mask == "jump":
        b[..., N // 2:] += 30.0
    b = None if b is None else b.to(torch.float32 if bias == "f32" else dt)
    name = "Og" if gated else "O"
    want = eager.attention_fwd_bwd(Q, K, V, m, b, torch.zeros_like(Q), layout=layout, compute_dtype=torch.float32, gate=G if gated else None)[name].float()
    dev = gpu_device
    args = [t if t is None else t.to(dev) for t in (Q, K, V, m, b)]
    with torch.no_grad():
        o = E.evoformer_attention(*args, layout=layout, gate=G.to(dev) if gated else None)
    d = o.float().cpu() - want
    assert torch.isfinite(d).all() and d.norm() <= 1e-2 * want.norm() + 1e-4 * want.numel() ** 0.5, (d.norm() / want.norm()).item()
