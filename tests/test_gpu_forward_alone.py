"""A forward without a backward at 129 to 256 keys reads the mask as the caller has it (csrc/mfma_fwd_ring.hip): the bits of the forward whose mask the
prep kernel has prepared, for every kind of mask, rows with every key masked, and mask rows that start anywhere."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # S, N, H, D, mask, dtype, layout, gated
    (5, 129, 2, 32, "bool", torch.bfloat16, "reference", False),
    (9, 160, 3, 16, "dead", torch.float16, "ds4sci", False),
    (33, 251, 8, 32, "dead_added", torch.float16, "ds4sci", True),
    (64, 256, 8, 32, "f32", torch.bfloat16, "reference", True),
    (7, 193, 2, 32, "neginf", torch.bfloat16, "ds4sci", False),
    (300, 130, 4, 32, "bool", torch.bfloat16, "ds4sci", True),       # several rows per workgroup, mask rows of 130 bytes
    (40, 255, 8, 8, "bool", torch.bfloat16, "ds4sci", True),
    (11, 200, 2, 32, None, torch.float16, "reference", False),
    (6, 256, 2, 16, "other16", torch.bfloat16, "reference", False),  # fp16 mask entries beside bf16 tensors
    (20, 131, 3, 32, "dead_f32", torch.bfloat16, "reference", True),
    (12, 224, 2, 32, "lowest", torch.float16, "ds4sci", False),
]


@pytest.mark.parametrize("bias", ["q", None])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_same_bits_as_with_a_backward(gpu_device, case, bias):
    from evoformer_triton_amd import evoformer_attention
    S, N, H, D, mask, dt, layout, gated = case
    g = torch.Generator().manual_seed(7)
    q, k, v, gate = (torch.randn((2, S, N, H, D), generator=g).to(dt).to(gpu_device) for _ in range(4))
    b = torch.randn((2, 1, H, N, N), generator=g).to(dt).to(gpu_device) if bias else None
    keep = torch.rand((2, S, 1, 1, N), generator=g) < 0.85
    keep[..., 0] = True
    if mask and mask.startswith("dead"):
        keep[0, S // 2] = keep[1, S - 1] = False
    soft = torch.randn((2, S, 1, 1, N), generator=g)
    lowest = torch.finfo(dt).min
    m = {None: None, "bool": keep, "dead": keep, "dead_added": torch.where(keep, 0.0, -1e9).to(torch.bfloat16), "dead_f32": torch.where(keep, 0.0, -1e9) + soft,
         "f32": soft, "neginf": torch.where(keep, soft, -float("inf")).to(dt), "other16": soft.half(), "lowest": torch.where(keep, 0.0, lowest).to(dt)}[mask]
    if m is not None:
        m = m.to(gpu_device)

    def call(grad):
        qq = q.clone().requires_grad_() if grad else q
        return evoformer_attention(qq, k, v, m, b, layout=layout, **({"gate": gate} if gated else {})).detach()

    with torch.no_grad():
        alone = call(False)
    both = call(True)
    assert torch.isfinite(both).all()
    assert torch.equal(alone, both)


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("bits", [0x7FC0, 0xFFC0, 0x7F81, 0xFF81], ids=hex)
@pytest.mark.parametrize("kind", ["f32", "bf16", "f16"])
def test_a_mask_entry_that_is_no_number_drops_its_key(gpu_device, kind, bits, gated):
    """Quiet and signalling, of either sign: the key gets the floor that a prepared mask gives it; a row of nothing else is a row with every key masked."""
    from evoformer_triton_amd import evoformer_attention
    g = torch.Generator().manual_seed(9)
    q, k, v, gate = (torch.randn((1, 7, 150, 2, 32), generator=g).to(torch.float16 if kind == "f16" else torch.bfloat16).to(gpu_device) for _ in range(4))
    m = torch.randn((1, 7, 1, 1, 150), generator=g)
    drop = torch.rand(m.shape, generator=g) < 0.2
    drop[..., 0] = False
    drop[0, 3] = True
    if kind == "f32":
        none = torch.tensor(bits << 16 | 1, dtype=torch.int64).to(torch.int32)
        m = torch.where(drop, none, m.view(torch.int32)).view(torch.float32)
    elif kind == "bf16":
        m = torch.where(drop, torch.tensor(bits).to(torch.int16), m.bfloat16().view(torch.int16)).view(torch.bfloat16)
    else:
        m = torch.where(drop, torch.tensor({0x7FC0: 0x7E00, 0xFFC0: 0xFE00, 0x7F81: 0x7C01, 0xFF81: 0xFC01}[bits]).to(torch.int16), m.half().view(torch.int16)).view(torch.float16)
    assert torch.isnan(m[drop]).all()
    m = m.to(gpu_device)
    out = []
    for grad in (False, True):
        qq = q.clone().requires_grad_(grad)
        out.append(evoformer_attention(qq, k, v, m, None, layout="ds4sci", **({"gate": gate} if gated else {})).detach())
    assert torch.isfinite(out[1]).all() and torch.equal(*out)
