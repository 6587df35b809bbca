"""dBias asked for without a bias through the C ABI: the sum of dS over the S rows, against eager in fp32 with a bias of zeros."""
import ctypes

import pytest
import torch

from oracle import eager

pytestmark = pytest.mark.gpu

CASES = [  # B, S, N, H, D, layout, dtype; with a bias dQ, dK and dV would come from one kernel
    (1, 256, 384, 4, 32, "reference", torch.bfloat16),
    (1, 384, 705, 1, 32, "ds4sci", torch.float16),
    (1, 256, 1030, 2, 32, "reference", torch.bfloat16),
    (1, 96, 384, 8, 8, "reference", torch.bfloat16),
    (2, 64, 600, 2, 8, "ds4sci", torch.float16),
    (8, 1, 130, 4, 8, "reference", torch.bfloat16),          # one S row, where dBias is dS itself
    (4, 1, 300, 8, 16, "ds4sci", torch.float16),
    (2, 1, 512, 8, 32, "reference", torch.bfloat16),
    (4, 1, 257, 8, 64, "ds4sci", torch.bfloat16),
    (2, 1, 512, 4, 128, "reference", torch.float16),
    (1, 1, 2100, 2, 32, "reference", torch.bfloat16),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_dbias_without_a_bias(gpu_device, case):
    import evoformer_triton_amd.evoformer as E
    from evoformer_triton_amd import _lib
    B, S, N, H, D, layout, dt = case
    g = torch.Generator().manual_seed(41)
    q, k, v, do = ((torch.randn((B, S, N, H, D), generator=g) * 0.7).to(dt).to(gpu_device) for _ in range(4))
    keep = torch.rand((B, S, 1, 1, N), generator=g) < 0.85
    keep[..., 0] = True
    m = keep.to(gpu_device)
    zero = torch.zeros((B, 1, H, N, N), device=gpu_device)
    ref = eager.attention_fwd_bwd(q, k, v, m, zero, do, layout=layout, compute_dtype=torch.float32, s_chunk=16)

    lib = _lib.load()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    mz, mk, mstr = E._prep_mask(m, B, S, N, q.device)
    bz, bdt, bstr = E._prep_bias(None, B, H, N, q.dtype, q.device)
    o, lse = torch.empty_like(q), torch.empty((B, H, S, N), device=q.device)
    p = E._params(q, k, v, mz, mk, mstr, bz, bdt, bstr, o, lse, layout)
    dq, dk, dv = (torch.empty_like(q) for _ in range(3))
    dbias = torch.full((B, H, N, N), float("nan"), device=q.device)
    p.dout, p.dq, p.dk, p.dv = do.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr()
    p.dbias, p.dbias_dtype = dbias.data_ptr(), _lib.EVO_F32
    prep = torch.empty(max(1, lib.evoattn_prep_bytes(ctypes.byref(p))), dtype=torch.uint8, device=q.device)
    ws = torch.empty(lib.evoattn_bwd_workspace_bytes(ctypes.byref(p)), dtype=torch.uint8, device=q.device)
    p.prep, p.prep_bytes, p.workspace, p.workspace_bytes = prep.data_ptr(), prep.numel(), ws.data_ptr(), ws.numel()
    names = lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD)
    assert all(x not in names for x in (b"fused", b"mfma_dbias", b"mfma_dq_wide")), names
    assert lib.evoattn_fwd(ctypes.byref(p), st) == 0
    assert lib.evoattn_bwd(ctypes.byref(p), st) == 0
    # P, dS, the scaled Q, O (in delta) and the results are each rounded by at most 2^-9 of their size, and the errors of the probabilities that
    # come of the scaled Q are of that order too: 5 * 2^-9, as relative 2-norms
    for name, t in {"O": o, "dQ": dq, "dK": dk, "dV": dv, "dBias": dbias.view(B, 1, H, N, N)}.items():
        want = ref[name].float()
        d = t.float() - want
        assert torch.isfinite(d).all(), name
        assert d.norm() <= 1e-2 * want.norm(), (name, (d.norm() / want.norm()).item())
