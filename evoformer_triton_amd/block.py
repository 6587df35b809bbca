"""The attention block either side of the kernels: projections in, gate and projection out.

The reference stops at the attention itself and returns O ungated (evoformer.py:735); in an
Evoformer block the steps around it are a LayerNorm, the Q/K/V and gate projections, the
pair-bias projection from the pair representation, sigmoid(gate) * O and the output
projection.  This module does those with this package's LayerNorm and Linear kernels (csrc/linear.hip;
fp32, large products and sizes that it does not take through the library's GEMMs, the weight
gradients summed over slices of the rows, which as single GEMMs would leave most of the chip
idle), and lays the results out so that the attention kernels read them as they fall:

  * in 16-bit on the GPU Q, K, V and the gate come out of one GEMM with the four weights stacked,
    as [B,S,N,4*H*D]; viewed as [B,S,N,4,H,D] each is a slot that the kernels take by its strides
    (per-head rows, a token's 4*H*D elements from the next token's): no permute, no copy, and the
    gradients come back in the same arrangement, so the projection's backward is one GEMM for the
    input and one for the weights (`evoformer._SlotAttention`);
  * elsewhere (fp32, under a tracer, head dims that need padding) they come out of the four
    Linear layers as [B,S,N,H*D], which viewed as [B,S,N,H,D] is the per-head ("ds4sci") layout;
  * the gate is applied in the forward kernel's epilogue and its gradient comes from the
    backward (`evoformer_attention(..., gate=g)`), so sigmoid(g) * O never makes a round trip
    of its own;
  * the gated output [B,S,N,H,D] viewed as [B,S,N,H*D] is the input of the output projection;
  * the pair bias Linear(LayerNorm(z)) comes from one kernel as [B,1,H,N,N] in the dtype of Q, so the attention kernels
    take it from 16-bit tiles; for shapes that kernel does not take, from the separate steps and a permute.
"""
from __future__ import annotations

from typing import Optional

import torch
from torch import nn

from . import _lib
from . import evoformer as _evoformer
from .evoformer import _DTYPES, _HEAD_DIMS, _SlotAttention, _alloc_bytes, _on_device, _ptr, _stream, evoformer_attention


def _row_slices(rows: int, n_out: int, n_in: int) -> int:
    """Slices of the rows a weight gradient is summed over.  The gradient of an [n_out, n_in] weight is
    one small matrix summed over all rows of the activations: as one library GEMM it has a handful of
    output tiles (four of 128 x 128 for 256 x 256) for a chip of 256 CUs.  Summed per slice of the rows
    as a batched GEMM and added up afterwards it fills the chip (32 768 rows, 256 x 256, bf16: 113 us as
    one GEMM, 33 us in 8 to 128 slices; 131 072 rows: 325 against 38 us in 128)."""
    tiles = -(-n_out // 128) * -(-n_in // 128)
    g = 1
    while g * tiles < 512 and rows % (2 * g) == 0 and rows // (2 * g) >= 256:
        g *= 2
    return g


def _weight_grad(dy2: torch.Tensor, x2: torch.Tensor) -> torch.Tensor:
    """dy2^T x2 ([rows, n_out], [rows, n_in] -> [n_out, n_in]) summed over slices of the rows."""
    rows, g = dy2.shape[0], _row_slices(dy2.shape[0], dy2.shape[1], x2.shape[1])
    if g == 1:
        return dy2.t() @ x2
    part = torch.bmm(dy2.view(g, rows // g, -1).transpose(1, 2), x2.view(g, rows // g, -1))
    return part.sum(0)          # (torch adds 16-bit inputs in fp32 and rounds the sum once)


def _bias_grad(dy2: torch.Tensor) -> torch.Tensor:
    """Column sums of dy2 [rows, n_out] (rows may lie further apart than n_out: some columns of a wider array):
    through the library's kernel (one pass at the rate of HBM, fp32 sums in a
    fixed order) where it takes the shape, else torch's."""
    rows, cols = dy2.shape
    if rows and not torch.compiler.is_compiling() and dy2.is_cuda and dy2.dtype in _DTYPES and dy2.stride(1) == 1 \
            and dy2.stride(0) >= cols and dy2.stride(0) % 8 == 0 and dy2.data_ptr() % 16 == 0:
        lib = _lib.load()
        nbytes = lib.evoattn_colsum_workspace_bytes(rows, cols, _DTYPES[dy2.dtype])
        if nbytes:
            with _on_device(dy2.device):
                out = torch.empty((cols,), device=dy2.device, dtype=dy2.dtype)
                ws = _alloc_bytes(nbytes, dy2.device)
                _lib.check(lib.evoattn_colsum(_ptr(dy2), dy2.stride(0), _ptr(out), _ptr(ws), ws.numel(), rows, cols, _DTYPES[dy2.dtype],
                                              _stream(dy2.device)), "evoattn_colsum")
            return out
    return dy2.sum(0)


class _Projections(torch.autograd.Function):
    """Several Linear layers of one input (Q, K, V and the gate of the normalised representation):
    forward(x, w0, b0, w1, b1, ...) -> (x w0^T + b0, x w1^T + b1, ...).  The gradient of the input
    accumulates inside the GEMMs (`addmm_`) instead of as additions of full-size tensors after
    them; the weight gradients are summed over slices of the rows (see _row_slices)."""

    @staticmethod
    def forward(ctx, x, *params):
        ws, bs = params[0::2], params[1::2]
        ctx.save_for_backward(x, *ws)
        ctx.has_bias = tuple(b is not None for b in bs)
        return tuple(torch.nn.functional.linear(x, w, b) for w, b in zip(ws, bs))

    @staticmethod
    def backward(ctx, *dys):
        x, *ws = ctx.saved_tensors
        x2 = x.reshape(-1, x.shape[-1])
        dx, grads = None, []
        for i, (w, dy) in enumerate(zip(ws, dys)):
            dy2 = dy.reshape(-1, dy.shape[-1])
            if ctx.needs_input_grad[0]:
                dx = dy2 @ w if dx is None else dx.addmm_(dy2, w)
            grads.append(_weight_grad(dy2, x2) if ctx.needs_input_grad[1 + 2 * i] else None)
            grads.append(_bias_grad(dy2) if ctx.has_bias[i] and ctx.needs_input_grad[2 + 2 * i] else None)
        return (None if dx is None else dx.view(x.shape), *grads)


class _Linear(torch.autograd.Function):
    """x W^T + b with the weight gradient summed over slices of the rows (see _row_slices); forward and
    input gradient are the library's GEMMs as torch.nn.functional.linear calls them.  What the compiler's tracer sees, and
    what a call reaches that the C++ node does not stand for (under vmap, func.grad and the like, which refuse it)."""

    @staticmethod
    def forward(ctx, x, weight, bias):
        ctx.save_for_backward(x, weight)
        ctx.has_bias = bias is not None
        # (as a matrix: for an input of more dimensions whose rows lie apart torch multiplies and then adds the
        # bias in a pass of its own)
        y = torch.nn.functional.linear(x.reshape(-1, x.shape[-1]), weight, bias)
        return y.view(*x.shape[:-1], weight.shape[0])

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        dy2, x2 = dy.reshape(-1, dy.shape[-1]), x.reshape(-1, x.shape[-1])
        dx = dw = db = None
        if ctx.needs_input_grad[0]:
            dx = (dy2 @ weight).view(x.shape)
        if ctx.needs_input_grad[1]:
            dw = _weight_grad(dy2, x2)
        if ctx.has_bias and ctx.needs_input_grad[2]:
            db = _bias_grad(dy2)
        return dx, dw, db


def _linear(layer: nn.Linear, x: torch.Tensor, dx_place: Optional[torch.Tensor] = None) -> torch.Tensor:
    # (the same in C++)
    y = None if torch.compiler.is_compiling() else _lib.host().linear(x, layer.weight, layer.bias, dx_place)
    return _Linear.apply(x, layer.weight, layer.bias) if y is None else y


class _StackedProjection:
    """The Q, K, V (and gate) projections of one input as a single GEMM with their weights stacked:
    apply(x, gate_bias, w0, w1, ...) -> x [w0; w1; ...]^T (+ gate_bias on the last layer's columns), shaped
    [..., n * out].  The input is read once instead of n times, its gradient is one GEMM over the whole
    gradient of the result (no additions of n partial gradients), and so is the weight gradient (summed over
    slices of the rows, see _row_slices), cut into the layers' pieces afterwards."""

    @staticmethod
    def apply(x, gate_bias, *weights):
        y = _lib.host().stacked_projection(x, gate_bias, weights)
        if y is not None:
            return y
        w = torch.cat(weights, 0)
        if gate_bias is not None:
            gate_bias = torch.cat([gate_bias.new_zeros(w.shape[0] - gate_bias.shape[0]), gate_bias])
        return _Linear.apply(x, w, gate_bias)


class _LayerNorm:
    """LayerNorm over the last dimension through the library's kernels (evoattn_layernorm_fwd / _bwd): x and y
    cross HBM once in the forward, x, dy and dx once in the backward; the gradients of weight and bias are summed
    in a fixed order.  None where those kernels do not take the call."""

    @staticmethod
    def apply(x, weight, bias, eps):
        return _lib.host().layer_norm(x, weight, bias, eps)


def _layer_norm(layer: nn.LayerNorm, x: torch.Tensor) -> torch.Tensor:
    # under the tracer, no rows, mixed dtypes, or a row length the kernels do not take: the framework's
    y = None if torch.compiler.is_compiling() else _LayerNorm.apply(x, layer.weight, layer.bias, layer.eps)
    return layer(x) if y is None else y


def _pair_bias(norm: nn.LayerNorm, layer: nn.Linear, z: torch.Tensor) -> Optional[torch.Tensor]:
    """Linear(LayerNorm(z)) permuted to [B,1,H,N,N] in one pass over z (csrc/pair_bias.hip), rounded where the separate steps
    round.  None where that kernel does not take the call."""
    if torch.compiler.is_compiling() or layer.bias is not None or z.dim() != 4:
        return None
    return _lib.host().pair_bias(z, norm.weight, norm.bias, norm.eps, layer.weight)


_NO_PARAMETERS = {"weight": None, "bias": None}
_UNBIASED = ("linear_q", "linear_k", "linear_v", "linear_z")


class GatedAttentionBlock(nn.Module):
    """Row-wise gated self-attention with pair bias (the MSA row attention of an Evoformer
    block).

    m    [B,S,N,c_m]   the representation attended over (S rows of N residues)
    z    [B,N,N,c_z]   optional pair representation; its projection to H channels is the bias
    mask [B,S,N]       optional, 1 = keep, 0 = drop the key (bool or float)
    ->   [B,S,N,c_m]
    """

    def __init__(self, c_m: int, c_hidden: int, no_heads: int, c_z: Optional[int] = None, gating: bool = True,
                 inf: float = 1e9):
        super().__init__()
        self.c_hidden, self.no_heads, self.inf = c_hidden, no_heads, inf
        hd = c_hidden * no_heads
        self.layer_norm_m = nn.LayerNorm(c_m)
        self.linear_q = nn.Linear(c_m, hd, bias=False)
        self.linear_k = nn.Linear(c_m, hd, bias=False)
        self.linear_v = nn.Linear(c_m, hd, bias=False)
        self.linear_g = nn.Linear(c_m, hd) if gating else None
        self.linear_o = nn.Linear(hd, c_m)
        if c_z is not None:
            self.layer_norm_z = nn.LayerNorm(c_z)
            self.linear_z = nn.Linear(c_z, no_heads, bias=False)
        else:
            self.layer_norm_z = self.linear_z = None

    def operands(self, m: torch.Tensor, z: Optional[torch.Tensor], mask: Optional[torch.Tensor], plain: bool = False):
        """Q, K, V, gate [B,S,N,H,D] (views of the projections), additive mask [B,S,1,1,N],
        bias [B,1,H,N,N].  `plain`: the framework's LayerNorm and Linear throughout (what
        `forward_eager` uses), else the library's LayerNorm kernels and the projections with
        their weight gradients summed over slices of the rows."""
        B, S, N, _ = m.shape
        H, D = self.no_heads, self.c_hidden
        norm = (lambda layer, t: layer(t)) if plain or not m.is_cuda else _layer_norm
        lin = (lambda layer, t: layer(t)) if plain else _linear
        x = norm(self.layer_norm_m, m)
        layers = [self.linear_q, self.linear_k, self.linear_v] + ([self.linear_g] if self.linear_g is not None else [])
        if plain:
            outs = [layer(x) for layer in layers]
        else:
            outs = _Projections.apply(x, *(t for layer in layers for t in (layer.weight, layer.bias)))
        q, k, v = (t.view(B, S, N, H, D) for t in outs[:3])
        g = outs[3].view(B, S, N, H, D) if self.linear_g is not None else None
        bias, add_mask = self._bias_and_mask(z, mask, q.dtype, (B, S, N), norm, lin)
        return q, k, v, g, add_mask, bias

    def _bias_and_mask(self, z, mask, dtype, shape, norm, lin):
        B, S, N = shape
        bias = add_mask = None
        if z is not None and self.linear_z is not None and norm is _layer_norm and lin is _linear and z.dtype == dtype:
            bias = _pair_bias(self.layer_norm_z, self.linear_z, z)
        if bias is None and z is not None and self.linear_z is not None:
            bias = lin(self.linear_z, norm(self.layer_norm_z, z)).permute(0, 3, 1, 2).unsqueeze(1).contiguous().to(dtype)
        if mask is not None:
            add_mask = (self.inf * (mask.to(torch.float32) - 1.0)).view(B, S, 1, 1, N)
        return bias, add_mask

    def _slots_ok(self, m: torch.Tensor) -> bool:
        """Whether Q, K, V and the gate can come from one GEMM and reach the kernels as slots of its result."""
        if not m.is_cuda or m.dtype not in (torch.bfloat16, torch.float16) or m.numel() == 0 or torch.compiler.is_compiling() \
                or torch.jit.is_tracing() or self.c_hidden not in _HEAD_DIMS:
            return False
        mods = self._modules
        layers = [mods["linear_q"], mods["linear_k"], mods["linear_v"], mods["linear_o"]] + ([mods["linear_g"]] if mods.get("linear_g") is not None else [])
        return all(l.weight.dtype == m.dtype for l in layers) and all(l.bias is None for l in layers[:3])

    def _native(self, m, z, mask):
        """The block as one call and one autograd node (csrc/host.cpp); None where it does not take the call.  (Layers are
        looked up as a module stores them: their attribute access alone takes 15 us of a 100 us forward.)"""
        mods, with_z = self._modules, z is not None and self._modules.get("linear_z") is not None
        inputs = [m, z if with_z else None]
        for name, used in (("layer_norm_m", True), ("linear_q", True), ("linear_k", True), ("linear_v", True), ("linear_g", mods.get("linear_g") is not None),
                           ("linear_o", True), ("layer_norm_z", with_z), ("linear_z", with_z)):
            own = mods[name]._parameters if used else _NO_PARAMETERS
            if "weight" not in own or "bias" not in own:
                return None     # (a layer whose weight is formed from something else)
            if name in _UNBIASED:
                if own["bias"] is not None:
                    return None
                inputs.append(own["weight"])
            else:
                inputs += (own["weight"], own["bias"])
        return _lib.host().block(inputs, mask, self.no_heads, mods["layer_norm_m"].eps, mods["layer_norm_z"].eps if with_z else 0.0, self.inf,
                                 _evoformer.FLAGS)

    def forward(self, m: torch.Tensor, z: Optional[torch.Tensor] = None, mask: Optional[torch.Tensor] = None):
        B, S, N, _ = m.shape
        if self._slots_ok(m):
            out = self._native(m, z, mask)
            if out is not None:
                return out
            H, D = self.no_heads, self.c_hidden
            gated = self.linear_g is not None
            x = _layer_norm(self.layer_norm_m, m)
            weights = [self.linear_q.weight, self.linear_k.weight, self.linear_v.weight] + ([self.linear_g.weight] if gated else [])
            P = _StackedProjection.apply(x, self.linear_g.bias if gated else None, *weights).view(B, S, N, len(weights), H, D)
            bias, add_mask = self._bias_and_mask(z, mask, m.dtype, (B, S, N), _layer_norm, _linear)
            o, grad_slot = _SlotAttention.apply(P, add_mask, bias, gated)
            return _linear(self.linear_o, o.reshape(B, S, N, H * D), grad_slot.view(B, S, N, H * D))
        q, k, v, g, add_mask, bias = self.operands(m, z, mask)
        o = evoformer_attention(q, k, v, add_mask, bias, layout="ds4sci", gate=g)
        return _linear(self.linear_o, o.reshape(B, S, N, self.no_heads * self.c_hidden))

    def forward_eager(self, m: torch.Tensor, z: Optional[torch.Tensor] = None, mask: Optional[torch.Tensor] = None):
        """The same block with plain torch operations (the formula of the reference's oracle,
        test.py:47-57, with the per-head view): what `forward` is tested against."""
        B, S, N, _ = m.shape
        q, k, v, g, add_mask, bias = self.operands(m, z, mask, plain=True)
        qh, kh, vh = (t.permute(0, 1, 3, 2, 4) for t in (q, k, v))              # [B,S,H,N,D]
        s = torch.matmul(qh * self.c_hidden ** -0.5, kh.transpose(-1, -2)).float()
        if bias is not None:
            s = s + bias.float()                                                 # [B,1,H,N,N] over S
        if add_mask is not None:
            s = s + add_mask.float()                                             # [B,S,1,1,N] over H and queries
        o = torch.matmul(torch.softmax(s, -1).to(q.dtype), vh).permute(0, 1, 3, 2, 4)   # [B,S,N,H,D]
        if g is not None:
            o = torch.sigmoid(g) * o
        return self.linear_o(o.reshape(B, S, N, self.no_heads * self.c_hidden))
