"""The backward of one S row at head dim 64, dQ with dBias and dK/dV in one launch (csrc/mfma_stream.hip), at the edges of its blocks of 128 queries and
keys, stages of 64 rows and tiles of 32, against eager in fp32."""
import ctypes

import pytest
import torch

from oracle import eager

pytestmark = pytest.mark.gpu

CASES = [  # B, N, H, mask, bias, layout, dtype
    (32, 4, 1, "bool", "f32", "reference", torch.bfloat16),      # the smallest: one block of each kind per problem, four rows of it
    (16, 64, 2, "dead", "f32", "ds4sci", torch.float16),         # one whole stage
    (11, 68, 3, "soft", "q", "reference", torch.bfloat16),       # a second stage of four rows
    (2, 128, 16, "dead_added", "f32", "reference", torch.bfloat16),
    (4, 132, 5, "dead", "f32", "reference", torch.bfloat16),     # a second block of four rows
    (2, 256, 8, "dead", "q", "ds4sci", torch.float16),
    (3, 292, 4, "bool", "f32", "ds4sci", torch.bfloat16),        # an odd number of tiles
    (1, 516, 8, None, "f32", "reference", torch.float16),
    (2, 1000, 3, "dead_added", "q", "reference", torch.bfloat16),
    (32, 5, 1, "dead", "f32", "reference", torch.bfloat16),      # rows that end within a group of four: one entry of it,
    (16, 31, 2, "bool", "f32", "ds4sci", torch.float16),         # three in a tile's last group,
    (8, 33, 4, "soft", "f32", "reference", torch.bfloat16),      # a tile of one key,
    (3, 250, 8, "dead_added", "f32", "reference", torch.bfloat16),
    (2, 517, 5, "dead", "f32", "ds4sci", torch.bfloat16),
    (4, 1023, 17, "bool", "f32", "reference", torch.float16),    # 544 workgroups of each kind
    (4, 1023, 16, "bool", "f32", "reference", torch.bfloat16),   # 512: two launches
    (3, 724, 32, "bool", "f32", "reference", torch.bfloat16),    # more workgroups than the chip takes at a time
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_single_row_backward_matches_eager(gpu_device, case):
    import evoformer_triton_amd.evoformer as E
    from evoformer_triton_amd import _lib
    B, N, H, mask, bias, layout, dt = case
    g = torch.Generator().manual_seed(31)
    Q, K, V, dO = ((torch.randn((B, 1, N, H, 64), generator=g) * 0.7).to(dt) for _ in range(4))
    keep = torch.rand((B, 1, 1, 1, N), generator=g) < 0.85
    keep[..., 0] = True
    if mask in ("dead", "dead_added"):
        keep[1] = False
    m = {None: None, "bool": keep, "dead": keep, "dead_added": torch.where(keep, 0.0, -1e9), "soft": torch.randn((B, 1, 1, 1, N), generator=g)}[mask]
    b = (torch.randn((B, 1, H, N, N), generator=g) * 0.5).to(torch.float32 if bias == "f32" else dt)
    xs = [None if t is None else t.to(gpu_device) for t in (Q, K, V, m, b, dO)]
    ref = eager.attention_fwd_bwd(*xs, layout=layout, compute_dtype=torch.float32, s_chunk=16)
    q, k, v = (t.detach().clone().requires_grad_() for t in xs[:3])
    bb = xs[4].detach().clone().requires_grad_()
    mz, mk, mstr = E._prep_mask(xs[3], B, 1, N, q.device)
    bz, bdt, bstr = E._prep_bias(xs[4], B, H, N, dt, q.device)
    p = E._params(q, k, v, mz, mk, mstr, bz, bdt, bstr, q, bz, layout)
    p.dout = p.dq = p.dk = p.dv = p.dbias = p.q
    kernels = _lib.load().evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD)
    assert kernels == b"mfma_dq_wide,mfma_dkdv" + (b"" if (B, N, H) == (4, 1023, 16) else b"(one launch)"), kernels   # (that one: a full round of each kernel)
    o = E.evoformer_attention(q, k, v, xs[3], bb, layout=layout)
    o.backward(xs[5])
    # P, dS, the scaled Q, O (in delta) and the results are each rounded by at most 2^-9 of their size, and the errors of the probabilities that
    # come of the scaled Q are of that order too: 5 * 2^-9, as relative 2-norms
    for name, t in {"O": o, "dQ": q.grad, "dK": k.grad, "dV": v.grad, "dBias": bb.grad}.items():
        want = ref[name].float()
        d = t.detach().float() - want
        assert torch.isfinite(d).all(), name
        assert d.norm() <= 1e-2 * want.norm(), (name, (d.norm() / want.norm()).item())


@pytest.mark.parametrize("gated,dbias", [(False, False), (True, True), (True, False)])
@pytest.mark.parametrize("case", [(32, 5, 1, "dead", torch.bfloat16), (2, 193, 8, "bool", torch.float16), (1, 129, 16, "dead_added", torch.bfloat16),
                                  (3, 385, 8, None, torch.bfloat16), (1, 1022, 5, "bool", torch.float16)], ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_rows_read_in_place_without_dbias_and_gated(gpu_device, case, gated, dbias):
    """Rows that end within a group of four are read in place whether dBias is wanted or not, and with an output gate, whose pass writes delta."""
    import evoformer_triton_amd.evoformer as E
    from evoformer_triton_amd import _lib
    B, N, H, mask, dt = case
    g = torch.Generator().manual_seed(43)
    q, k, v, gate, dO = ((torch.randn((B, 1, N, H, 64), generator=g) * 0.7).to(dt).to(gpu_device) for _ in range(5))
    keep = torch.rand((B, 1, 1, 1, N), generator=g) < 0.85
    keep[..., 0] = True
    if mask in ("dead", "dead_added") and B > 1:
        keep[1] = False
    m = None if mask is None else (torch.where(keep, 0.0, -1e9) if mask == "dead_added" else keep).to(gpu_device)
    b = (torch.randn((B, 1, H, N, N), generator=g) * 0.5).to(gpu_device)
    ref = eager.attention_fwd_bwd(q, k, v, m, b, dO, layout="ds4sci", compute_dtype=torch.float32, s_chunk=None if gated else 16, gate=gate if gated else None)
    leaves = [t.detach().clone().requires_grad_() for t in (q, k, v)] + ([b.detach().clone().requires_grad_()] if dbias else [])
    gg = gate.detach().clone().requires_grad_() if gated else None
    bb = leaves[3] if dbias else b
    mz, mk, mstr = E._prep_mask(m, B, 1, N, q.device)
    bz, bdt, bstr = E._prep_bias(b, B, H, N, dt, q.device)
    p = E._params(q, k, v, mz, mk, mstr, bz, bdt, bstr, q, bz, "ds4sci")
    p.dout = p.dq = p.dk = p.dv = p.q
    if dbias:
        p.dbias = p.q
    if gated:
        p.gate = p.o_gated = p.dgate = p.q
    kernels = _lib.load().evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD)
    assert kernels == b"mfma_dq_wide,mfma_dkdv(one launch)", kernels
    o = E.evoformer_attention(*leaves[:3], m, bb, layout="ds4sci", gate=gg)
    o.backward(dO)
    got = {"Og" if gated else "O": o, "dQ": leaves[0].grad, "dK": leaves[1].grad, "dV": leaves[2].grad}
    if dbias:
        got["dBias"] = bb.grad
    if gated:
        got["dGate"] = gg.grad
    # as above; the gate adds one rounding of dO sigmoid(g), and delta and dgate come of the rounded gated output: 2 * 2^-9 more, as relative 2-norms
    for name, t in got.items():
        want = ref[name].float()
        d = t.detach().float() - want
        assert torch.isfinite(d).all(), name
        assert d.norm() <= 1.4e-2 * want.norm(), (name, (d.norm() / want.norm()).item())
