"""The forward that takes two S rows at a time (csrc/mfma_stream.hip, stream_fwd_pair; csrc/mfma_stream8.hip, stream_fwd8) at the edges of its stages, tiles and pairs, against eager in fp32
and against the kernel that takes one row."""
import ctypes

import pytest
import torch

from oracle import eager

pytestmark = pytest.mark.gpu

CASES = [  # B, S, N, H, D, mask, bias, layout, dtype
    (1, 193, 193, 8, 32, "dead", "q", "reference", torch.bfloat16),          # a last pair of one row; a last tile of one key
    (2, 97, 224, 8, 32, "dead_added", "f32", "reference", torch.float16),    # the same in two batches, each with a bias of its own
    (1, 256, 257, 4, 32, "bool", "q", "ds4sci", torch.bfloat16),           # a last query block and a last stage of one
    (1, 258, 300, 4, 32, "jump", "q", "reference", torch.float16),           # scores that outgrow the first tile's maximum
    (3, 171, 288, 2, 32, "dead", "f32", "ds4sci", torch.bfloat16),
    (1, 300, 513, 3, 32, None, "q", "reference", torch.bfloat16),
    (1, 17, 130, 4, 8, "dead", "q", "reference", torch.bfloat16),      # a last pair of one row; a second stage and block of two
    (2, 16, 256, 2, 8, "dead_added", "q", "ds4sci", torch.float16),
    (1, 21, 193, 4, 8, "jump", "q", "reference", torch.float16),
    (3, 257, 33, 4, 8, "dead", "q", "reference", torch.bfloat16),      # two tiles, the second of one key
    (1, 401, 65, 8, 8, "jump", "f32", "reference", torch.bfloat16),    # three
    (2, 401, 97, 4, 8, "dead_added", "f32", "ds4sci", torch.float16),  # four, one stage
    (1, 257, 300, 4, 8, "bool", "f32", "ds4sci", torch.bfloat16),
    (1, 145, 513, 3, 8, None, "q", "reference", torch.bfloat16),       # a last stage of one key
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_forward_pairs_match_eager(gpu_device, case):
    import evoformer_triton_amd.evoformer as E
    from evoformer_triton_amd import _lib
    B, S, N, H, D, mask, bias, layout, dt = case
    g = torch.Generator().manual_seed(37)
    q, k, v = ((torch.randn((B, S, N, H, D), generator=g) * 0.7).to(dt).to(gpu_device) for _ in range(3))
    keep = torch.rand((B, S, 1, 1, N), generator=g) < 0.85
    keep[..., 0] = True
    if mask in ("dead", "dead_added"):   # the second row of a pair, the first one, both, and the last row
        for s in (1, 4, 10, 11, S - 1):
            keep[B - 1, s] = False
    m = None if mask in (None, "jump") else torch.where(keep, 0.0, -1e9) if mask == "dead_added" else keep
    b = torch.randn((B, 1, H, N, N), generator=g) * 0.5
    if mask == "jump":
        b[..., N // 2:] += 30.0
    b = b.to(torch.float32 if bias == "f32" else dt).to(gpu_device)
    m = None if m is None else m.to(gpu_device)
    want = eager.attention_fwd_bwd(q, k, v, m, b, torch.zeros_like(q), layout=layout, compute_dtype=torch.float32, s_chunk=32)["O"].float()

    lib = _lib.load()
    mz, mk, mstr = E._prep_mask(m, B, S, N, q.device)
    bz, bdt, bstr = E._prep_bias(b, B, H, N, q.dtype, q.device)
    got = {}
    for name, flags in (("pairs", 0), ("one", _lib.EVO_FLAG_PER_PROBLEM)):
        o, lse = torch.empty_like(q), torch.empty((B, H, S, N), device=q.device)
        p = E._params(q, k, v, mz, mk, mstr, bz, bdt, bstr, o, lse, layout)
        p.flags |= flags
        prep = torch.empty(lib.evoattn_prep_bytes(ctypes.byref(p)), dtype=torch.uint8, device=q.device)
        p.prep, p.prep_bytes = prep.data_ptr(), prep.numel()
        kernel = lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_FWD)
        assert (kernel == b"mfma_fwd_pair") == (name == "pairs"), kernel
        assert lib.evoattn_fwd(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        got[name] = (o.float(), lse)
    # the scaled Q, the probabilities and O are each rounded by at most 2^-9 of their size, and the scores' error that comes of the first moves the
    # probabilities by as much again: 4 * 2^-9, as relative 2-norms
    for name, (o, _) in got.items():
        d = o - want
        assert torch.isfinite(d).all(), name
        assert d.norm() <= 8e-3 * want.norm(), (name, (d.norm() / want.norm()).item())
    # the two kernels form the same scores and differ in the order of fp32 sums alone (N + 2 rounding steps of 2^-24 at most)
    a, c = got["pairs"][1], got["one"][1]
    assert ((a - c).abs() <= (N + 2) * 2.0 ** -24 * (1.0 + c.abs())).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N", [130, 160, 256])
def test_no_further_from_64_bits_than_the_kernel_over_a_chunk_of_rows(gpu_device, N, dt):
    """Head dim 8, 129 to 256 keys: O is divided by the sum of the probabilities as they are rounded, as that kernel does."""
    import evoformer_triton_amd.evoformer as E
    from evoformer_triton_amd import _lib
    B, S, H, D = 1, 64, 4, 8
    g = torch.Generator(device=gpu_device).manual_seed(5)
    q, k, v = (torch.randn((B, S, N, H, D), device=gpu_device, generator=g).to(dt) for _ in range(3))
    b = torch.randn((B, 1, H, N, N), device=gpu_device, generator=g).to(dt)
    heads = [t.double().permute(0, 3, 1, 2, 4).contiguous() for t in (q, k, v)]
    p64 = torch.softmax(torch.matmul(heads[0], heads[1].transpose(-1, -2).contiguous()) * D ** -0.5 + b.double().permute(0, 2, 1, 3, 4), -1)
    want = torch.matmul(p64, heads[2])
    lib = _lib.load()
    bz, bdt, bstr = E._prep_bias(b, B, H, N, dt, gpu_device)
    err = {}
    for name, flags in ((b"mfma_fwd_pair", 0), (b"mfma_fwd_ring", _lib.EVO_FLAG_DEBUG_FWD_BIAS_TILES)):
        o, lse = torch.empty_like(q), torch.empty((B, H, S, N), device=gpu_device)
        p = E._params(q, k, v, None, _lib.EVO_MASK_NONE, (0, 0), bz, bdt, bstr, o, lse, "ds4sci")
        p.flags |= flags
        prep = torch.empty(lib.evoattn_prep_bytes(ctypes.byref(p)), dtype=torch.uint8, device=gpu_device)
        p.prep, p.prep_bytes = prep.data_ptr(), prep.numel()
        assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_FWD) == name
        assert lib.evoattn_fwd(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        err[name] = ((o.double().permute(0, 3, 1, 2, 4) - want).norm() / want.norm()).item()
    # some 65000 independent roundings each: the two norms are known to well under 1 %
    assert err[b"mfma_fwd_pair"] <= 1.01 * err[b"mfma_fwd_ring"], err
