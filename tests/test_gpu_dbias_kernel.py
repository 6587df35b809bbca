"""dBias from the kernel of its own whose bias stays resident (csrc/mfma_stream.hip, stream_dbias; csrc/mfma_stream8.hip) at the edges of its blocks of queries and
keys and of its chunks of S rows, against eager in fp32."""
import ctypes

import pytest
import torch

from oracle import eager

pytestmark = pytest.mark.gpu

CASES = [  # B, S, N, H, D, mask, bias dtype, dtype
    (1, 8, 513, 2, 32, "dead", "q", torch.bfloat16),            # a last block of one query and one key
    (2, 9, 545, 1, 32, "bool", "f32", torch.float16),           # a last block of 33 keys: one tile and one key; two batches
    (1, 67, 640, 1, 32, "dead_added", "q", torch.float16),      # whole blocks; a last chunk that is shorter
    (1, 8, 1120, 1, 32, None, "f32", torch.bfloat16),           # chunks of one row
    (1, 9, 513, 2, 8, "dead", "q", torch.bfloat16),
    (2, 8, 609, 1, 8, "bool", "f32", torch.float16),
    (1, 67, 640, 1, 8, "dead_added", "q", torch.bfloat16),
    (1, 16, 129, 2, 64, "dead", "f32", torch.bfloat16),
    (2, 17, 161, 1, 64, "dead_added", "q", torch.float16),
    (1, 5, 129, 16, 128, "dead", "q", torch.bfloat16),
    (1, 8, 161, 8, 128, "bool", "f32", torch.float16),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_dbias_kernel_matches_eager(gpu_device, case):
    import evoformer_triton_amd.evoformer as E
    from evoformer_triton_amd import _lib
    B, S, N, H, D, mask, bias, dt = case
    g = torch.Generator().manual_seed(31)
    Q, K, V, dO = ((torch.randn((B, S, N, H, D), generator=g) * 0.7).to(dt) for _ in range(4))
    keep = torch.rand((B, S, 1, 1, N), generator=g) < 0.85
    keep[..., 0] = True
    if mask in ("dead", "dead_added"):
        keep[0, 1] = False
    m = None if mask is None else torch.where(keep, 0.0, -1e9) if mask == "dead_added" else keep
    b = (torch.randn((B, 1, H, N, N), generator=g) * 0.5).to(torch.float32 if bias == "f32" else dt)
    dev = gpu_device
    q, k, v, do, m, b = (None if t is None else t.to(dev) for t in (Q, K, V, dO, m, b))
    q.requires_grad_()
    ref = eager.attention_fwd_bwd(q.detach(), k, v, m, b, do, layout="reference", compute_dtype=torch.float32, s_chunk=16)
    b = b.detach().clone().requires_grad_()
    o = E.evoformer_attention(q, k, v, m, b, layout="reference")
    o.backward(do)
    mz, mk, mstr = E._prep_mask(m, B, S, N, q.device)
    bz, bdt, bstr = E._prep_bias(b.detach(), B, H, N, q.dtype, q.device)
    p = E._params(q, k, v, mz, mk, mstr, bz, bdt, bstr, o, torch.empty((B, H, S, N), device=dev), "reference")
    p.dbias, p.dbias_dtype = bz.data_ptr(), E._DTYPES[bz.dtype]
    assert b"+mfma_dbias" in _lib.load().evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD)
    # the scaled Q, O (in delta) and a 16-bit dBias are each rounded by at most 2^-9 of their size, and the errors of P and of dP - delta that come of it
    # are of that order too: 5 * 2^-9, as relative 2-norms
    want = ref["dBias"].float()
    d = b.grad.float() - want
    assert torch.isfinite(d).all()
    assert d.norm() <= 1e-2 * want.norm(), (d.norm() / want.norm()).item()
