"""dQ, dK and dV from one kernel (csrc/mfma_bwd_fused.hip, mfma_bwd_fused8.hip) at the edges of its tiles, groups, stages and blocks of keys, against eager
in fp32."""
import ctypes

import pytest
import torch

from oracle import eager

pytestmark = pytest.mark.gpu

CASES = [  # B, S, N, H, D, mask, bias, layout, dtype, dBias
    (1, 48, 96, 8, 32, "bool", "q", "reference", torch.bfloat16, False),
    (2, 48, 127, 4, 32, "soft", "f32", "ds4sci", torch.float16, False),
    (1, 64, 128, 6, 32, "dead", "q", "reference", torch.bfloat16, False),
    (1, 96, 129, 4, 32, "dead", "f32", "reference", torch.bfloat16, False),     # a group of one query; three tiles of keys per wave
    (1, 192, 192, 2, 32, None, None, "ds4sci", torch.bfloat16, False),
    (2, 96, 193, 2, 32, "bool", "q", "reference", torch.float16, False),
    (1, 128, 251, 3, 32, "soft", "q", "ds4sci", torch.bfloat16, False),
    (1, 96, 256, 4, 32, "jump", "q", "reference", torch.bfloat16, False),
    (1, 96, 256, 4, 32, "dead", "q", "ds4sci", torch.float16, False),
    (2, 96, 250, 2, 32, "dead_added", "f32", "reference", torch.bfloat16, False),
    (1, 200, 257, 2, 32, "dead", "q", "reference", torch.bfloat16, False),      # a second block of keys, a last one of one key
    (1, 768, 264, 1, 32, "bool", "f32", "ds4sci", torch.float16, False),        # more problems than workgroups
    (1, 193, 384, 2, 32, "dead_added", "q", "reference", torch.bfloat16, False),
    (1, 128, 516, 3, 32, "soft", "q", "reference", torch.bfloat16, False),      # three blocks
    (1, 1024, 321, 1, 32, "dead", "q", "reference", torch.bfloat16, True),
    (2, 224, 385, 1, 32, "dead_added", "f32", "ds4sci", torch.float16, True),
    (1, 224, 516, 2, 32, "bool", "q", "reference", torch.bfloat16, True),
    # a last stage of one group of queries, with delta read by the dBias kernel
    (1, 224, 385, 2, 32, "dead", "q", "reference", torch.bfloat16, True),
    (1, 448, 449, 1, 32, "soft", "q", "ds4sci", torch.float16, True),
    (1, 128, 352, 8, 32, "bool", "f32", "reference", torch.bfloat16, True),
    (1, 256, 288, 3, 8, "dead", "q", "reference", torch.bfloat16, True),
    (1, 256, 513, 1, 8, "soft", "f32", "ds4sci", torch.float16, True),
    (1, 96, 96, 8, 8, "bool", "q", "reference", torch.bfloat16, False),
    (2, 48, 129, 4, 8, "dead", "f32", "ds4sci", torch.float16, False),         # a last group of one query, a last tile of one key
    (1, 128, 193, 4, 8, "jump", "q", "reference", torch.bfloat16, False),
    (1, 300, 257, 2, 8, "dead_added", "q", "ds4sci", torch.bfloat16, False),
    (1, 96, 384, 8, 8, "dead", "q", "reference", torch.bfloat16, True),        # the widest block
    (1, 256, 385, 3, 8, "soft", "q", "reference", torch.float16, True),        # two blocks of keys
    (1, 128, 300, 6, 8, None, "f32", "ds4sci", torch.bfloat16, True),
    (1, 600, 1000, 1, 8, "dead", None, "reference", torch.bfloat16, False),    # three blocks, keys past the padded mask; more problems than workgroups
    (1, 256, 545, 1, 8, "dead_added", "q", "reference", torch.bfloat16, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_fused_backward_matches_eager(gpu_device, case):
    import evoformer_triton_amd.evoformer as E
    from evoformer_triton_amd import _lib
    B, S, N, H, D, mask, bias, layout, dt, dbias = case
    g = torch.Generator().manual_seed(29)
    Q, K, V, dO = ((torch.randn((B, S, N, H, D), generator=g) * 0.7).to(dt) for _ in range(4))
    keep = torch.rand((B, S, 1, 1, N), generator=g) < 0.85
    keep[..., 0] = True
    if mask in ("dead", "dead_added"):
        keep[0, 1] = False
    m = None
    if mask in ("bool", "dead"):
        m = keep
    elif mask == "dead_added":
        m = torch.where(keep, 0.0, -1e9)
    elif mask == "soft":
        m = torch.randn((B, S, 1, 1, N), generator=g)
    b = None if bias is None else torch.randn((B, 1, H, N, N), generator=g) * 0.5
    if mask == "jump":
        b[..., N // 2:] += 30.0
    b = None if b is None else b.to(torch.float32 if bias == "f32" else dt)
    dev = gpu_device
    xs = [None if t is None else t.to(dev) for t in (Q, K, V, m, b, dO)]
    ref = eager.attention_fwd_bwd(*xs, layout=layout, compute_dtype=torch.float32, s_chunk=16)
    q, k, v = (t.detach().clone().requires_grad_() for t in xs[:3])
    bb = None if b is None else xs[4].detach().clone().requires_grad_(dbias)
    o = E.evoformer_attention(q, k, v, xs[3], bb, layout=layout)
    o.backward(xs[5])
    got = {"O": o, "dQ": q.grad, "dK": k.grad, "dV": v.grad}
    if dbias:
        got["dBias"] = bb.grad
    lib = _lib.load()
    mz, mk, mstr = E._prep_mask(xs[3], B, S, N, q.device)
    bz, bdt, bstr = E._prep_bias(xs[4], B, H, N, q.dtype, q.device)
    p = E._params(q, k, v, mz, mk, mstr, bz, bdt, bstr, o, torch.empty((B, H, S, N), device=dev), layout)
    if dbias:
        p.dbias, p.dbias_dtype = bz.data_ptr(), E._DTYPES[bz.dtype]
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD).decode().startswith("mfma_bwd_fused")
    # P, dS, the scaled Q, O (in delta) and the results are each rounded by at most 2^-9 of their size, and the errors of the probabilities that
    # come of the scaled Q are of that order too: 5 * 2^-9, as relative 2-norms
    for name, t in got.items():
        want = ref[name].float()
        d = t.detach().float() - want
        assert torch.isfinite(d).all(), name
        assert d.norm() <= 1e-2 * want.norm(), (name, (d.norm() / want.norm()).item())
