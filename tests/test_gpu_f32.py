"""The fp32 matrix-instruction kernels (csrc/f32.hip) against the eager formula in fp64, at the edges of their tiles."""
import pytest
import torch

from oracle import eager

pytestmark = pytest.mark.gpu

CASES = [  # B, S, N, H, D, mask, bias, layout, gated
    (1, 1, 1, 1, 8, None, "row", "reference", False),
    (2, 3, 31, 2, 16, "bool", "row", "ds4sci", False),
    (1, 2, 32, 3, 32, "dead", "row", "reference", False),       # a row with every key dropped
    (1, 5, 33, 2, 32, "neginf", "row", "ds4sci", True),
    (1, 4, 64, 2, 64, "soft", None, "reference", False),
    (2, 2, 65, 1, 128, "soft", "one", "ds4sci", False),          # one bias for the batch
    (1, 40, 97, 2, 8, "bool", "row", "reference", False),        # chunks of rows that do not divide S
    (1, 3, 128, 2, 32, "deadadd", "row", "ds4sci", True),
    (1, 2, 129, 2, 16, "soft", "row", "reference", False),
    (1, 2, 300, 1, 32, "bool", "odd", "ds4sci", False),          # bias rows at an odd address
    (1, 1, 520, 2, 64, None, None, "reference", False),
    (1, 2, 200, 1, 128, "bool", "row", "reference", True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_f32_kernels_match_the_formula(gpu_device, case):
    import ctypes
    import evoformer_triton_amd.evoformer as E
    from evoformer_triton_amd import _lib
    B, S, N, H, D, mask, bias, layout, gated = case
    g = torch.Generator().manual_seed(17)
    Q, K, V, G, dO = (torch.randn((B, S, N, H, D), generator=g) for _ in range(5))
    keep = torch.rand((B, S, 1, 1, N), generator=g) < 0.8
    keep[..., 0] = True
    if mask in ("dead", "deadadd"):
        keep[0, 0] = False
    m = {None: None, "bool": keep, "dead": keep, "soft": torch.randn((B, S, 1, 1, N), generator=g), "neginf": torch.where(keep, 0.0, -float("inf")),
         "deadadd": torch.where(keep, 0.0, -1e9)}[mask]
    b = None if bias is None else torch.randn((1 if bias == "one" else B, 1, H, N, N), generator=g)
    fmask = m is not None and m.dtype != torch.bool
    wide = torch.float32 if mask == "deadadd" else torch.float64     # (in fp64 scores next to -1e9 would keep what fp32 rounds away)
    f64 = lambda t: t if t is None or t.dtype == torch.bool else t.to(wide)
    ref = eager.attention_fwd_bwd(f64(Q), f64(K), f64(V), f64(m), None if b is None else f64(b).expand(B, 1, H, N, N), f64(dO), layout=layout,
                                  compute_dtype=wide, gate=f64(G) if gated else None)
    dev = gpu_device
    q, k, v = (t.to(dev).requires_grad_() for t in (Q, K, V))
    bb = None
    if b is not None:
        bb = b.to(dev)
        if bias == "odd":
            buf = torch.empty(b.numel() + 1, device=dev)
            buf[1:] = bb.reshape(-1)
            bb = buf[1:].view(b.shape)
        bb = bb.detach().requires_grad_()
    mm = None if m is None else (m.to(dev).requires_grad_() if fmask else m.to(dev))
    gg = G.to(dev).requires_grad_() if gated else None
    o = E.evoformer_attention(q, k, v, mm, bb, layout=layout, gate=gg)
    o.backward(dO.to(dev))
    got = {"Og" if gated else "O": o, "dQ": q.grad, "dK": k.grad, "dV": v.grad}
    if bb is not None:
        got["dBias"] = bb.grad
        if bias == "one":
            ref["dBias"] = ref["dBias"].sum(0, keepdim=True)
    if fmask:
        got["dMask"] = mm.grad
    if gated:
        got["dGate"] = gg.grad
    for name, t in got.items():
        want = ref[name].double()
        err = (t.detach().double().cpu() - want).abs().max().item()
        assert err <= 1e-5 * max(1.0, want.abs().max().item()), (name, err)
    p = E._params(q.detach(), k.detach(), v.detach(), None, _lib.EVO_MASK_NONE, (0, 0), None, _lib.EVO_NONE, (0, 0, 0), o.detach(), o.detach(), layout)
    assert _lib.load().evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_FWD) == b"f32_fwd"
