"""Bias entries of -inf or of the type's lowest value (what a program writes to keep two chains apart): whole key tiles of
them, in kept and in dropped rows, through each kernel that reads a bias, against eager in fp32."""
import pytest
import torch

from oracle import eager

pytestmark = pytest.mark.gpu

# A result is a sum of products rounded to 16 bits on its way: the tolerance of the other tests against eager in fp32.
REL = 1.5e-2


def _closed(kind, B, H, N, value, g):
    """A bias whose entries `kind` names are closed; every query keeps a key."""
    b = torch.randn((B, 1, H, N, N), generator=g) * 0.5
    if kind == "chains":
        b[..., : N // 2, N // 2:] = value
        b[..., N // 2:, : N // 2] = value
    elif kind == "first":                      # the first tiles of a row, of half of the queries
        b[..., N // 2:, : min(64, N - 1)] = value
    elif kind == "last":                       # the last key (a tile of one where N = 32 n + 1)
        b[..., N - 1] = value
    return b


def _check(dev, shape, kind, bias_dt, dt, lowest, mask, layout, grad):
    import evoformer_triton_amd.evoformer as E
    B, S, N, H, D = shape
    g = torch.Generator().manual_seed(41)
    Q, K, V, dO = ((torch.randn(shape, generator=g) * 0.7).to(dt) for _ in range(4))
    bdt = dt if bias_dt == "q" else torch.float32
    b = _closed(kind, B, H, N, torch.finfo(bdt).min if lowest else -float("inf"), g).to(bdt)
    m = None
    if mask == "dead":                         # a row with every key dropped: uniform over the keys, whatever the bias says
        m = torch.ones((B, S, 1, 1, N), dtype=torch.bool)
        m[:, S - 1] = False
    # (the oracle's own bias closed by a finite value: the same probabilities, and gradients that its autograd forms)
    want = eager.attention_fwd_bwd(Q, K, V, m, b.float().clamp_min(-1e30), dO, layout=layout, compute_dtype=torch.float32)
    q, k, v, bb = (t.to(dev).requires_grad_(grad) for t in (Q, K, V, b))
    o = E.evoformer_attention(q, k, v, None if m is None else m.to(dev), bb, layout=layout)
    got = {"O": o}
    if grad:
        o.backward(dO.to(dev))
        got.update(dQ=q.grad, dK=k.grad, dV=v.grad, dBias=bb.grad)
    for name, t in got.items():
        d = t.detach().float().cpu() - want[name]
        assert torch.isfinite(d).all(), name
        assert d.norm() <= REL * want[name].norm() + 1e-4 * d.numel() ** 0.5, (name, (d.norm() / want[name].norm()).item())


SPLIT = [  # single sequences without a backward: each wave has every fourth tile of 32 keys
    ((1, 1, 33, 2, 32), "last", "f", torch.bfloat16, False, None, "reference"),
    ((1, 1, 65, 3, 64), "last", "q", torch.float16, False, None, "ds4sci"),
    ((2, 1, 97, 2, 128), "last", "q", torch.bfloat16, True, None, "reference"),
    ((1, 1, 250, 4, 64), "chains", "f", torch.bfloat16, False, None, "reference"),
    ((1, 1, 256, 4, 32), "first", "q", torch.bfloat16, False, "dead", "reference"),
    ((1, 1, 130, 2, 128), "chains", "f", torch.float16, False, "dead", "reference"),
    ((1, 1, 128, 16, 64), "chains", "f", torch.bfloat16, True, "dead", "reference"),
]


@pytest.mark.parametrize("case", SPLIT, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_forward_that_splits_the_keys(gpu_device, case):
    _check(gpu_device, *case, grad=False)


STREAM = [  # rows that stream through LDS: the first step has 32 keys (head dim 32: 64)
    ((1, 6, 96, 2, 64), "chains", "q", torch.bfloat16, False, None, "reference"),
    ((1, 6, 130, 2, 128), "first", "f", torch.float16, False, None, "ds4sci"),
    ((1, 5, 65, 1, 64), "first", "f", torch.bfloat16, True, "dead", "reference"),
    ((2, 1, 200, 4, 128), "chains", "q", torch.bfloat16, True, None, "reference"),
    ((1, 6, 130, 2, 32), "chains", "f", torch.bfloat16, False, None, "reference"),
    ((1, 9, 300, 2, 32), "first", "q", torch.float16, True, None, "ds4sci"),
    ((1, 2, 1100, 1, 64), "last", "q", torch.bfloat16, False, None, "reference"),
]


@pytest.mark.parametrize("case", STREAM, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_kernels_whose_rows_stream(gpu_device, case):
    _check(gpu_device, *case, grad=True)


ONE_STEP = [  # kernels whose first step has 64 keys, and the plain ones, which go key by key
    ((1, 6, 130, 2, 8), "first", "f", torch.bfloat16, False, None, "reference"),
    ((1, 6, 96, 2, 16), "first", "q", torch.float16, False, None, "ds4sci"),
    ((1, 5, 300, 2, 16), "chains", "f", torch.bfloat16, True, None, "reference"),
    ((2, 1, 300, 4, 8), "chains", "q", torch.bfloat16, False, None, "reference"),
    ((1, 40, 200, 2, 8), "first", "f", torch.bfloat16, False, None, "reference"),       # fp32 tiles resident
]


@pytest.mark.parametrize("plain", [False, True], ids=["matrix_core", "plain"])
@pytest.mark.parametrize("case", ONE_STEP, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_kernels_with_a_step_of_64_keys_and_plain_ones(gpu_device, case, plain, monkeypatch):
    import evoformer_triton_amd.evoformer as E
    from evoformer_triton_amd import _lib
    monkeypatch.setattr(E, "FLAGS", _lib.EVO_FLAG_FORCE_GENERIC if plain else 0)
    _check(gpu_device, *case, grad=True)


TIMES_ZERO = [  # entries that a kernel multiplies by zero: the identity product of a resident bias, rows with every key dropped
    ((1, 40, 256, 2, 32), "chains", "q", torch.bfloat16, False, "dead", "reference"),
    ((1, 40, 200, 2, 16), "last", "q", torch.float16, False, None, "ds4sci"),
    ((1, 40, 250, 1, 8), "chains", "q", torch.bfloat16, True, "dead", "reference"),        # rows that pass through LDS
    ((1, 6, 130, 2, 64), "first", "q", torch.bfloat16, False, "dead", "reference"),
    ((1, 2, 256, 2, 32), "chains", "f", torch.bfloat16, False, "dead", "reference"),       # the caller's rows
    ((2, 1, 200, 2, 16), "chains", "q", torch.bfloat16, False, "dead", "ds4sci"),
    ((1, 64, 200, 2, 64), "chains", "q", torch.bfloat16, False, "dead", "reference"),      # dBias from a kernel of its own
    ((1, 64, 544, 1, 32), "chains", "q", torch.float16, False, "dead", "reference"),
    ((1, 24, 384, 2, 8), "chains", "q", torch.bfloat16, False, "dead", "reference"),
]


@pytest.mark.parametrize("grad", [False, True], ids=["forward", "step"])
@pytest.mark.parametrize("case", TIMES_ZERO, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_entries_that_meet_a_factor_of_zero(gpu_device, case, grad):
    _check(gpu_device, *case, grad=grad)


def test_a_gated_forward_with_a_resident_bias(gpu_device):
    import evoformer_triton_amd.evoformer as E
    g = torch.Generator().manual_seed(43)
    B, S, N, H, D = shape = (1, 40, 250, 2, 32)
    Q, K, V, G = ((torch.randn(shape, generator=g) * 0.7).to(torch.bfloat16) for _ in range(4))
    b = _closed("chains", B, H, N, -float("inf"), g).to(torch.bfloat16)
    want = eager.attention_fwd_bwd(Q, K, V, None, b.float().clamp_min(-1e30), torch.zeros_like(Q), compute_dtype=torch.float32, gate=G)["Og"]
    d = E.evoformer_attention(*(t.to(gpu_device) for t in (Q, K, V)), None, b.to(gpu_device), gate=G.to(gpu_device)).float().cpu() - want
    assert torch.isfinite(d).all() and d.norm() <= REL * want.norm()
