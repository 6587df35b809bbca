"""The C-ABI library loads on a GPU-less host, exports every symbol include/evoattn.h
declares, and its host-side validation returns the documented codes.  No kernel runs."""
import ctypes
import os
import re

import pytest

from evoformer_triton_amd import _lib
from evoformer_triton_amd._lib import EvoAttnParams

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def declared_functions():
    text = open(os.path.join(ROOT, "include", "evoattn.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(evoattn_\w+)\s*\(", text)))


def test_every_declared_symbol_is_exported(lib):
    names = declared_functions()
    assert set(names) == set(_lib.EXPORTS)
    for n in names:
        assert hasattr(lib, n), n
    assert lib.evoattn_version() == 4


def test_the_library_reports_the_version_the_header_declares(lib):
    text = open(os.path.join(ROOT, "include", "evoattn.h")).read()
    declared = int(re.search(r"#define\s+EVOATTN_VERSION\s+(\d+)", text).group(1))
    assert lib.evoattn_version() == declared
    # (the build entry point checks the same after compiling; it must not carry a number of its own)
    entry = open(os.path.join(ROOT, "__graft_entry__.py")).read()
    assert not re.search(r"evoattn_version\(\)\s*==\s*\d", entry)


def test_struct_layout_matches_header():
    # 12 x 4-byte fields, 9 x int64, 14 pointers, one size_t, then prep pointer + size; no padding
    assert ctypes.sizeof(EvoAttnParams) == 12 * 4 + 9 * 8 + 14 * 8 + 8 + 16 + 3 * 8        # ... and the three gate pointers
    assert EvoAttnParams.stride_b.offset == 48 and EvoAttnParams.q.offset == 120


def good(B=1, S=4, N=64, H=2, D=32, dtype=_lib.EVO_BF16):
    p = EvoAttnParams()
    p.B, p.S, p.N, p.H, p.D = B, S, N, H, D
    p.dtype, p.bias_dtype, p.mask_kind, p.dbias_dtype = dtype, _lib.EVO_F32, _lib.EVO_MASK_F32, _lib.EVO_F32
    p.scale = D ** -0.5
    p.stride_b, p.stride_h, p.stride_s, p.stride_n = S * N * H * D, S * N * D, N * D, D
    p.bias_stride_b, p.bias_stride_h, p.bias_stride_row = H * N * N, N * N, N
    p.mask_stride_b, p.mask_stride_s = S * N, N
    fake = 0x10000  # never dereferenced by the host-side checks
    for f in ("q", "k", "v", "o", "lse", "bias", "mask", "dout", "dq", "dk", "dv", "dbias"):
        setattr(p, f, fake)
    p.workspace, p.workspace_bytes = fake, 1 << 30
    p.prep, p.prep_bytes = fake, 1 << 30
    return p


def test_check_accepts_a_valid_block(lib):
    p = good()
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == 0
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == 0
    assert lib.evoattn_path(ctypes.byref(p), _lib.EVO_PASS_FWD) == b"mfma"
    # rows so far apart that a problem's rows (and its padding up to the next 256) leave 32-bit byte offsets: the plain kernels
    p.stride_n = 1 << 22
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == 0
    assert lib.evoattn_path(ctypes.byref(p), _lib.EVO_PASS_FWD) == b"generic"
    assert lib.evoattn_path(ctypes.byref(p), _lib.EVO_PASS_BWD) == b"generic"


@pytest.mark.parametrize("mutate,code", [
    (lambda p: setattr(p, "N", 0), _lib.EVO_EINVAL),
    (lambda p: setattr(p, "q", None), _lib.EVO_EINVAL),
    (lambda p: setattr(p, "dtype", 7), _lib.EVO_EINVAL),
    (lambda p: setattr(p, "bias_dtype", _lib.EVO_F16), _lib.EVO_EINVAL),      # neither fp32 nor q's dtype
    (lambda p: setattr(p, "bias", None), _lib.EVO_EINVAL),                    # dtype says there is one
    (lambda p: setattr(p, "mask_kind", 9), _lib.EVO_EINVAL),
    (lambda p: setattr(p, "scale", float("nan")), _lib.EVO_EINVAL),
    (lambda p: setattr(p, "D", 24), _lib.EVO_EUNSUPPORTED),
    (lambda p: setattr(p, "stride_n", 16), _lib.EVO_EINVAL),                  # rows would overlap
    (lambda p: setattr(p, "q", 0x10001), _lib.EVO_EALIGN),
    (lambda p: setattr(p, "lse", 0x10002), _lib.EVO_EALIGN),
    (lambda p: setattr(p, "B", 1 << 30), _lib.EVO_EOVERFLOW),
])
def test_check_rejects(lib, mutate, code):
    p = good()
    mutate(p)
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == code
    assert lib.evoattn_fwd(ctypes.byref(p), None) == code      # rejected before any launch
    assert lib.evoattn_strerror(code)


def test_bwd_checks_workspace_and_outputs(lib):
    p = good()
    need = lib.evoattn_bwd_workspace_bytes(ctypes.byref(p))
    rows = 1 * 2 * 4 * 64
    assert need >= rows * 4 + 4 * 4 + 2 * 64 * 64 * 4          # delta + shift + >= one dBias partial
    p.workspace_bytes = need - 1
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == _lib.EVO_EWORKSPACE
    p.workspace_bytes = need
    p.workspace = 0x10010
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == _lib.EVO_EALIGN
    p = good()
    p.dq = None
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == _lib.EVO_EINVAL
    assert lib.evoattn_bwd(ctypes.byref(p), None) == _lib.EVO_EINVAL
    p = good()
    p.dbias_dtype = _lib.EVO_F16
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == _lib.EVO_EINVAL
    # without dbias / dmask the workspace shrinks
    p = good()
    p.dbias = None
    assert lib.evoattn_bwd_workspace_bytes(ctypes.byref(p)) < need
    assert lib.evoattn_bwd_workspace_bytes(None) == 0


def test_path_selection(lib):
    p = good(dtype=_lib.EVO_F32)
    assert lib.evoattn_path(ctypes.byref(p), 0) == b"generic"            # check mode
    p = good(D=128)
    assert lib.evoattn_path(ctypes.byref(p), 0) == b"mfma" and lib.evoattn_path(ctypes.byref(p), 1) == b"mfma"
    assert b"ring" not in lib.evoattn_kernels(ctypes.byref(p), 0) + lib.evoattn_kernels(ctypes.byref(p), 1)
    p = good(D=24)
    assert lib.evoattn_check(ctypes.byref(p), 0) == _lib.EVO_EUNSUPPORTED
    p = good()
    p.flags = _lib.EVO_FLAG_FORCE_GENERIC
    assert lib.evoattn_path(ctypes.byref(p), 0) == b"generic"
    p = good()
    p.q = 0x10008                                                          # 8-byte aligned only
    assert lib.evoattn_check(ctypes.byref(p), 0) == 0
    assert lib.evoattn_path(ctypes.byref(p), 0) == b"generic"
    p = good(N=4096)
    assert lib.evoattn_path(ctypes.byref(p), 0) == b"mfma"
    # the dBias sums of so long a row exceed the register file of the dQ kernels: a kernel of its own sums dBias,
    # for a bias in fp32 and in the dtype of q alike
    assert lib.evoattn_path(ctypes.byref(p), 1) == b"mfma"
    assert lib.evoattn_kernels(ctypes.byref(p), 1) == b"mfma_dq_wide+mfma_dbias,mfma_dkdv"
    p.bias_dtype = p.dbias_dtype = _lib.EVO_BF16
    assert lib.evoattn_path(ctypes.byref(p), 1) == b"mfma"
    assert lib.evoattn_kernels(ctypes.byref(p), 1) == b"mfma_dq_wide+mfma_dbias,mfma_dkdv"
    p = good(N=4096, D=128)                                                # (that kernel is not built for head dim 128)
    assert lib.evoattn_path(ctypes.byref(p), 1) == b"generic"
    p = good(N=4096)
    p.dbias = None
    assert lib.evoattn_path(ctypes.byref(p), 1) == b"mfma"


@pytest.mark.parametrize("shape", [(1, 384, 384, 4, 32), (1, 192, 705, 4, 32), (1, 64, 2048, 8, 32), (1, 1024, 384, 8, 8), (1, 256, 600, 8, 8)])
def test_dbias_without_a_bias_comes_with_dq(lib, shape):
    """The kernel that sums dBias by itself keeps the bias' tiles: without a bias there are none, and the dQ kernels sum dS."""
    p = good(*shape)
    assert b"+mfma_dbias" in lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD)
    p.bias, p.bias_dtype = None, _lib.EVO_NONE
    need = lib.evoattn_bwd_workspace_bytes(ctypes.byref(p))
    p.workspace_bytes = need
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == 0
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD).split(b",")[0] in (b"mfma_dq_ring", b"mfma_dq")
    B, S, N, H, D = shape
    assert need >= B * H * S * N * 4 + B * H * N * N * 4           # delta, at least one dBias partial
    p.dbias = None
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD) == b"mfma_bwd_fused"


@pytest.mark.parametrize("D", [8, 16, 32, 64, 128])
def test_dbias_of_one_row_without_a_bias(lib, D):
    """One S row: the dQ kernel that writes dBias as it goes does so beside a bias; without one the partial sums are kept."""
    p = good(4, 1, 512, 8, D)
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD).startswith(b"mfma_dq_wide")
    with_bias = lib.evoattn_bwd_workspace_bytes(ctypes.byref(p))
    p.bias, p.bias_dtype = None, _lib.EVO_NONE
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD).split(b",")[0] in (b"mfma_dq_ring", b"mfma_dq")
    assert lib.evoattn_bwd_workspace_bytes(ctypes.byref(p)) >= with_bias + 4 * 8 * 512 * 512 * 4
    p.N = 4096                                                             # (no such sums that long)
    p.stride_b, p.stride_h, p.stride_s = 4096 * 8 * D, 4096 * D, 4096 * D
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD) == b"generic"


@pytest.mark.parametrize("shape,wgs", [((1, 384, 384, 4, 32), 512), ((1, 96, 2048, 4, 32), 384), ((1, 32, 1024, 8, 8), 256), ((1, 1024, 400, 8, 8), 512), ((1, 1024, 384, 8, 8), 0)])
def test_dq_scratch_is_that_of_the_workgroups_that_run(lib, shape, wgs):
    """Several blocks of keys: a problem's dQ in fp32 for every workgroup, of which at most 512 run; with dBias in the place of its partial sums."""
    B, S, N, H, D = shape
    up = lambda n: (n + 255) // 256 * 256
    p = good(*shape)
    with_dbias = lib.evoattn_bwd_workspace_bytes(ctypes.byref(p))
    p.flags = _lib.EVO_FLAG_ONLY_DQ                                          # the dQ kernel of its own: no scratch
    partials = lib.evoattn_bwd_workspace_bytes(ctypes.byref(p))
    p.flags, p.dbias = 0, None
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD) == b"mfma_bwd_fused"
    plain = up(B * H * S * N * 4) + up(B * S * 4)
    assert lib.evoattn_bwd_workspace_bytes(ctypes.byref(p)) == plain + up(wgs * N * D * 4)
    assert with_dbias <= max(partials, plain + up(wgs * N * D * 4), plain + up(4 * 512 * 128 * 128 * 4))   # (as many partials as four rounds of workgroups have blocks)


def test_error_strings(lib):
    assert _lib.strerror(0) == "ok"
    assert "workspace" in _lib.strerror(_lib.EVO_EWORKSPACE)
    assert _lib.strerror(_lib.EVO_EHIP - 1)                                # a hipError_t string
    with pytest.raises(_lib.EvoAttnError) as ei:
        _lib.check(_lib.EVO_EALIGN, "evoattn_fwd")
    assert ei.value.code == _lib.EVO_EALIGN and "evoattn_fwd" in str(ei.value)


def header_flags():
    text = open(os.path.join(ROOT, "include", "evoattn.h")).read()
    return {name: int(val, 0) for name, val in re.findall(r"\b(EVO_FLAG_[A-Z_]+)\s*=\s*(0x[0-9a-fA-F]+|\d+)", text)}


def test_every_flag_bit_is_declared_in_the_header(lib):
    """The binding's flag constants are the header's, every flag literal a test passes is one of them,
    and a bit the header does not declare is rejected."""
    declared = header_flags()
    bound = {n: v for n, v in vars(_lib).items() if n.startswith("EVO_FLAG_")}
    assert bound == declared
    all_bits = 0
    for v in declared.values():
        assert v and v & (v - 1) == 0, "one bit per flag"
        all_bits |= v
    # no test spells a flag as a bare number
    for fn in os.listdir(os.path.join(ROOT, "tests")):
        if fn.endswith(".py") and fn != "test_abi.py":
            src = open(os.path.join(ROOT, "tests", fn)).read()
            assert not re.search(r"FLAGS\s*=\s*(0x[0-9a-fA-F]+|[1-9]\d*)\b", src), fn
            assert not re.search(r"flags\s*=\s*(0x[0-9a-fA-F]+|[1-9]\d*)\b", src), fn
    for bit in (0x20, 0x40, 0x4000, 1 << 30):
        assert not bit & all_bits
        p = good()
        p.flags = bit
        assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == _lib.EVO_EINVAL
    p = good()
    p.flags = all_bits & ~_lib.EVO_FLAG_GATE_DOUT_INPLACE
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == 0
    p.flags = _lib.EVO_FLAG_GATE_DOUT_INPLACE | _lib.EVO_FLAG_ONLY_DQ      # the gate would be applied twice
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == _lib.EVO_EINVAL
    p.flags = _lib.EVO_FLAG_GATE_DOUT_INPLACE
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == 0


def test_shift_threshold_is_the_header_constant():
    text = open(os.path.join(ROOT, "include", "evoattn.h")).read()
    m = re.search(r"#define\s+EVOATTN_SHIFT_THRESHOLD\s+\((-[0-9.e]+)f\)", text)
    assert m and float(m.group(1)) == -5.0e8
    common = open(os.path.join(ROOT, "evoformer_triton_amd", "csrc", "common.h")).read()
    assert "kShiftThreshold = EVOATTN_SHIFT_THRESHOLD" in common


def test_static_forward_rejects_oversized_problems_on_the_host(lib):
    """evoattn_fwd_static checks the size of the prepared operands against its built-in array
    before it touches the GPU."""
    p = good(S=8, N=2048, H=8)
    p.bias_dtype = _lib.EVO_BF16
    assert lib.evoattn_prep_bytes(ctypes.byref(p)) > _lib.EVOATTN_STATIC_PREP_BYTES
    assert lib.evoattn_fwd_static(ctypes.byref(p), None) == _lib.EVO_EWORKSPACE
    p = good()
    p.q = None
    assert lib.evoattn_fwd_static(ctypes.byref(p), None) == _lib.EVO_EINVAL
    text = open(os.path.join(ROOT, "include", "evoattn.h")).read()
    assert re.search(r"#define\s+EVOATTN_STATIC_PREP_BYTES\s+\(16u << 20\)", text)


def test_gate_validation_on_the_host(lib):
    """The gate's pointers are checked before any launch: the forward needs o_gated, the backward
    dgate and one more tensor of workspace, and the q-family has to be dense."""
    p = good()
    fake = 0x10000
    p.gate = fake
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == _lib.EVO_EINVAL        # no o_gated
    p.o_gated = fake
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == 0
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == _lib.EVO_EINVAL        # no dgate
    p.dgate = fake
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == 0
    # the gated output may stand alone (no ungated O is written, none is read); without a gate `o` is required
    keep, p.o = p.o, None
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == 0
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == 0
    p.o_gated = None
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == _lib.EVO_EINVAL
    p.o, p.o_gated = keep, fake
    q = good()
    q.o = None
    assert lib.evoattn_check(ctypes.byref(q), _lib.EVO_PASS_FWD) == _lib.EVO_EINVAL
    q = good()
    need_plain = lib.evoattn_bwd_workspace_bytes(ctypes.byref(q))
    assert lib.evoattn_bwd_workspace_bytes(ctypes.byref(p)) >= need_plain + 1 * 4 * 64 * 2 * 32 * 2   # + dO, bf16
    p.flags = _lib.EVO_FLAG_GATE_DOUT_INPLACE                                               # dO in the place of dout
    assert lib.evoattn_bwd_workspace_bytes(ctypes.byref(p)) == need_plain
    p.flags = 0
    p.gate = 0x10008
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == _lib.EVO_EALIGN
    p.gate = fake
    dense_ws = lib.evoattn_bwd_workspace_bytes(ctypes.byref(p))
    p.stride_s *= 2                                              # rows with gaps (a slot of a wider buffer): the workspace's dO has them too
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == 0
    assert lib.evoattn_bwd_workspace_bytes(ctypes.byref(p)) == dense_ws + 3 * 64 * 32 * 2              # three more gaps of a row's size
    p.stride_s *= 16                                             # sparser than a slot of 8
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == _lib.EVO_EUNSUPPORTED
    # the per-head layout of the same dense tensor is fine
    p = good()
    B, S, N, H, D = 1, 4, 64, 2, 32
    p.stride_b, p.stride_h, p.stride_s, p.stride_n = S * N * H * D, D, N * H * D, H * D
    p.gate = p.o_gated = fake
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == 0
    # strides that are no whole number of 16-byte pieces: the gate's kernels move rows in such pieces
    p = good()
    p.gate = p.o_gated = fake
    p.stride_n += 2
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == _lib.EVO_EALIGN
    p.gate = p.o_gated = None                                    # without a gate such rows go to the kernels that read element by element
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == 0
    # more heads than the gate's backward pass has LDS for
    p = good(H=257)
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == 0
    p.gate = p.o_gated = fake
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_FWD) == _lib.EVO_EUNSUPPORTED
    # gate outputs without a gate are a mistake
    p = good()
    p.dgate = fake
    assert lib.evoattn_check(ctypes.byref(p), _lib.EVO_PASS_BWD) == _lib.EVO_EINVAL


def test_header_is_plain_c_and_the_library_loads_from_c(tmp_path):
    """tests/abi_check.c, compiled as strict C99 against include/evoattn.h, loads the library with
    dlopen and exercises the host-side validation: the boundary holds without Python or torch."""
    import shutil
    import subprocess
    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("no C compiler")
    exe = tmp_path / "abi_check"
    src = os.path.join(ROOT, "tests", "abi_check.c")
    subprocess.check_call([gcc, "-std=c99", "-pedantic", "-Wall", "-Werror", "-D_POSIX_C_SOURCE=200809L",
                           "-I", os.path.join(ROOT, "include"), src, "-o", str(exe), "-ldl"])
    out = subprocess.run([str(exe), _lib.LIB_PATH], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    assert f"sizeof(EvoAttnParams) = {ctypes.sizeof(EvoAttnParams)}" in out.stdout


def test_layernorm_entry_points_validate_on_the_host(lib):
    """Argument errors of the LayerNorm entry points are found before anything is launched."""
    import ctypes
    buf = ctypes.create_string_buffer(4096 + 16)
    a = (ctypes.addressof(buf) + 15) & ~15
    fwd = lambda x=a, y=a, mean=a, rstd=a, rows=4, cols=64, dtype=_lib.EVO_BF16, eps=1e-5, gamma=None: \
        lib.evoattn_layernorm_fwd(x, gamma, None, y, mean, rstd, rows, cols, dtype, eps, None)
    assert fwd(x=None) == _lib.EVO_EINVAL and fwd(cols=0) == _lib.EVO_EINVAL and fwd(dtype=7) == _lib.EVO_EINVAL
    assert fwd(cols=12) == _lib.EVO_EALIGN and fwd(x=a + 2) == _lib.EVO_EALIGN and fwd(gamma=a + 4) == _lib.EVO_EALIGN
    assert fwd(cols=4096) == _lib.EVO_EUNSUPPORTED and fwd(cols=2048, dtype=_lib.EVO_F32) == _lib.EVO_EUNSUPPORTED
    assert fwd(rows=0) == 0                                   # no rows: nothing to launch
    assert lib.evoattn_layernorm_bwd_workspace_bytes(100, 256, _lib.EVO_BF16) == 1024 * 2 * 256 * 4
    assert lib.evoattn_layernorm_bwd_workspace_bytes(100, 12, _lib.EVO_BF16) == 0
    bwd = lambda dx=a, dgamma=None, ws=None, ws_bytes=0, cols=64: \
        lib.evoattn_layernorm_bwd(a, a, None, a, a, dx, dgamma, None, ws, ws_bytes, 4, cols, _lib.EVO_BF16, None)
    assert bwd(dx=None) == _lib.EVO_EINVAL                    # no output asked for
    assert bwd(dgamma=a) == _lib.EVO_EWORKSPACE and bwd(dgamma=a, ws=a, ws_bytes=100) == _lib.EVO_EWORKSPACE
    assert bwd(cols=20) == _lib.EVO_EALIGN
    assert lib.evoattn_colsum_workspace_bytes(100, 256, _lib.EVO_F16) == 1024 * 256 * 4
    assert lib.evoattn_colsum(None, 64, a, a, 1 << 30, 4, 64, _lib.EVO_BF16, None) == _lib.EVO_EINVAL
    assert lib.evoattn_colsum(a, 64, a, None, 0, 4, 64, _lib.EVO_BF16, None) == _lib.EVO_EWORKSPACE
    assert lib.evoattn_colsum(a, 12, a, a, 1 << 30, 4, 12, _lib.EVO_BF16, None) == _lib.EVO_EALIGN
    assert lib.evoattn_colsum(a, 32, a, a, 1 << 30, 4, 64, _lib.EVO_BF16, None) == _lib.EVO_EINVAL       # rows overlap
    assert lib.evoattn_colsum(a, 68, a, a, 1 << 30, 4, 64, _lib.EVO_BF16, None) == _lib.EVO_EALIGN


@pytest.mark.parametrize("shape,dbias,fused", [
    ((1, 73, 784, 8, 32), False, False), ((1, 96, 784, 8, 32), False, True),     # 784 keys are four blocks of 256, 584 problems a round and a bit
    ((1, 68, 602, 8, 32), False, False), ((1, 64, 602, 8, 32), False, True),
    ((2, 35, 1182, 8, 32), False, False), ((1, 64, 2048, 8, 32), False, True),
    ((1, 145, 824, 4, 32), True, False), ((1, 192, 824, 4, 32), True, True),
    ((4, 8, 384, 32, 32), True, False), ((1, 128, 384, 8, 32), True, True),      # partial sums of few S rows
    ((2, 24, 377, 16, 8), True, False), ((1, 96, 377, 8, 8), True, True),
    ((1, 958, 336, 1, 8), True, False), ((1, 480, 336, 2, 8), True, True),       # one head alone
    ((2, 18, 824, 8, 8), False, False), ((2, 16, 824, 8, 8), False, True),
    ((1, 137, 864, 2, 8), True, False), ((1, 256, 864, 2, 8), True, True),
])
def test_backward_of_padded_rows_and_few_rows(lib, shape, dbias, fused):
    """The kernel of dQ, dK and dV leaves calls alone whose keys, padded to whole blocks, or problems fill its rounds badly, and dBias of few S rows per head."""
    p = good(*shape)
    p.bias_dtype = p.dtype
    if not dbias:
        p.dbias = None
    assert (b"mfma_bwd_fused" in lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD)) == fused


@pytest.mark.parametrize("shape,bias,fwd,bwd", [
    ((1, 384, 384, 4, 32), "q", b"mfma_fwd_pair", b"mfma_bwd_fused+mfma_dbias"), ((1, 100, 384, 4, 32), "q", b"mfma_fwd", b"mfma_dq_ring,mfma_dkdv"),
    ((1, 1024, 384, 8, 8), "q", b"mfma_fwd_pair", b"mfma_bwd_fused+mfma_dbias"), ((1, 64, 200, 4, 8), "f32", b"mfma_fwd_ring", b"mfma_dq_ring,mfma_dkdv"),
    ((4, 1, 1024, 32, 64), "f32", b"mfma_fwd", b"mfma_dq_wide,mfma_dkdv(one launch)"), ((4, 1, 1023, 16, 64), "f32", b"mfma_fwd", b"mfma_dq_wide,mfma_dkdv"),
])
def test_kernel_names_tell_the_forms_apart(lib, shape, bias, fwd, bwd):
    p = good(*shape)
    p.bias_dtype = p.dtype if bias == "q" else _lib.EVO_F32
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_FWD) == fwd
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD) == bwd
    p.flags = _lib.EVO_FLAG_PER_PROBLEM
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_FWD) == b"mfma_fwd"


@pytest.mark.parametrize("shape,phases", [((1, 512, 256, 8, 32), 2), ((1, 384, 384, 4, 32), 1), ((1, 768, 768, 4, 32), 1), ((1, 1024, 384, 8, 8), 1),
                                          ((1, 200, 640, 5, 64), 2), ((4, 1, 1024, 32, 64), 1), ((1, 64, 512, 4, 128), 2)])
def test_the_benchmark_names_the_kernels_that_it_times(lib, shape, phases):
    """A phase's time is that of the kernels that the call with its flags launches, and the step launches the same ones."""
    import bench
    p = good(*shape)
    if shape[1] == 1:
        p.bias_dtype = _lib.EVO_F32
    got = bench.backward_phases(lib, p)
    assert p.flags == 0 and len(got) == phases
    for _, flags, kernels in got:
        p.flags = flags
        assert kernels in lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD).decode()
    p.flags = 0
    assert lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD).decode() == ",".join(kernels for _, _, kernels in got)


@pytest.mark.parametrize("shape,bias,pairs", [
    ((1, 197, 64, 16, 8), "f32", False), ((1, 197, 64, 16, 8), "q", True), ((1, 197, 65, 16, 8), "f32", True),
    ((1, 323, 128, 16, 8), "f32", False), ((1, 323, 96, 16, 8), "f32", True), ((1, 400, 128, 8, 8), "f32", True),
    ((2, 9, 576, 16, 8), "q", False), ((2, 9, 576, 16, 8), "f32", True), ((2, 12, 576, 16, 8), "q", True),
    ((4, 3, 823, 16, 8), "q", False), ((4, 5, 823, 16, 8), "q", True),
])
def test_forward_of_two_rows_where_it_pays(lib, shape, bias, pairs):
    p = good(*shape)
    p.bias_dtype = p.dtype if bias == "q" else _lib.EVO_F32
    p.flags = _lib.EVO_FLAG_DEBUG_BIAS_TILES if shape[1] <= 4 else 0
    assert (lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_FWD) == b"mfma_fwd_pair") == pairs


def test_flags_where_bias_rows_are_read_in_place(lib):
    """One S row of an odd length at head dim 64, fp32 bias: the flags that choose among dQ kernels split the one launch in two, and choose another
    kernel only together with the one that prepares tiles."""
    p = good(4, 1, 251, 8, 64)
    p.bias_dtype = _lib.EVO_F32

    def names(flags):
        p.flags = flags
        return lib.evoattn_kernels(ctypes.byref(p), _lib.EVO_PASS_BWD)
    assert names(0) == b"mfma_dq_wide,mfma_dkdv(one launch)"
    for flag in (_lib.EVO_FLAG_PER_PROBLEM, _lib.EVO_FLAG_DEBUG_NO_DQ_WIDE):
        assert names(flag) == b"mfma_dq_wide,mfma_dkdv"
        assert names(flag | _lib.EVO_FLAG_DEBUG_BIAS_TILES) == b"mfma_dq,mfma_dkdv"
