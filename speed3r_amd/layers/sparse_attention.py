"""``SparseFlashAttentionRope``: the reference's global sparse attention layer
(pi3/models/layers/sparse_attention.py:60-141) on the HIP kernels of this package.

Same constructor arguments, same parameter names (``qkv``, ``proj``, ``q_norm``, ``k_norm``, ``gate.0``) and the
same ``forward(x, attn_bias=None, xpos=None)``, so a reference checkpoint loads with ``load_state_dict``.
Differences, all on the host side of the operator boundary:

* for inference the projection, qk-norm, RoPE and the block means are one kernel (:func:`project`) and ``proj`` is another
  (:func:`linear`); where these are not built or do not pay, q, k, v are strided views of the packed projection (no
  ``.contiguous()`` copies), which one pass reads directly;
* the gated merge runs in the selection kernel's epilogue (or in its own kernel where that is not built), writing
  ``[B, N, C]`` for ``proj``;
* when a gradient is wanted (grad mode on and the input or a parameter requires grad) the layer runs as projections
  around one differentiable operator with a backward of kernels (bf16/fp16, head_dim 64, blocks of 64 or 16 tokens; see
  ``_forward_with_grad`` for the rest), the gradients of the projections' parameters by a kernel of their own;
* ``N`` need not be a multiple of the block: the last block pools its valid tokens, its keys beyond ``N`` are
  masked and its query rows beyond ``N`` do not exist (the reference raises for such ``N``);
* the top-k count, 32 in the reference, is a constructor argument.
"""
from __future__ import annotations

from typing import Optional

import torch
from torch import Tensor, nn

from ..sparse_attn import ops
from ..sparse_attn.flash_attention_topk import flash_attn_topk_func
from .pos_embed import RoPE2D, block_positions


def calls_forward_only(m: nn.Module, kind: type) -> bool:
    """Whether calling ``m`` runs ``kind.forward`` and nothing else: exactly of that type, ``forward`` not replaced, not
    compiled, no hooks of its own and no global ones.  A kernel may only then stand in for the call."""
    g = nn.modules.module
    return type(m) is kind and "forward" not in m.__dict__ and m._compiled_call_impl is None and not (
        m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks or g._global_forward_hooks
        or g._global_forward_pre_hooks or g._global_backward_hooks or g._global_backward_pre_hooks)


LINEAR_FORWARD = nn.Linear.forward   # what the kernels stand in for: not a forward that was put in its place for all layers


def sizes_are_known(x: Tensor) -> bool:
    """Whether the sizes of ``x`` may choose a path: not where a call is traced, compiled or exported for any sizes."""
    return type(x) is Tensor and not torch.compiler.is_compiling() and not torch._C._is_tracing()


# Calls with less work keep torch's products and the passes over them.  A layer of few rows is bound by the host: 400 to 1 020 tokens of
# 1024 channels take 162 us with those, 137 with the projection in one launch, 126 with both products here (2 016 tokens: 180 / 126).  Other
# widths, with those / here, 16-token blocks: 1 024 tokens of 128 channels 201 / 129, 512 of 768 177 / 130, 272 to 1 024 of 2048 199 / 178; the
# kernels alone 70 / 55, 76 / 68, 91 / 90 to 119 / 107.
def enough_work(x: Tensor) -> bool:
    return x.numel() >= max(1, min(1024 * x.shape[-1], 384 * 1024))


def linear_takes(m: nn.Linear, x: Tensor, gelu: Optional[bool] = None) -> bool:
    """Whether a kernel may stand in for ``m(x)``: an ordinary call for inference of a module that would run
    ``nn.Linear.forward`` and nothing else, on enough rows (asked first: few rows wait for the host) and, unless ``gelu`` is None,
    where ``ops.linear`` with it or without is the faster one."""
    return sizes_are_known(x) and enough_work(x) and type(m) is nn.Linear \
        and (gelu is None or ops.linear_pays(x.numel() // x.shape[-1], *m.weight.shape, gelu)) \
        and calls_forward_only(m, nn.Linear) and nn.Linear.forward is LINEAR_FORWARD and type(m.weight) is nn.Parameter \
        and x.shape[-1] == m.weight.shape[1] and not torch.is_autocast_enabled("cuda") and ops.unchanged_here(x) \
        and not (torch.is_grad_enabled() and (x.requires_grad or m.weight.requires_grad or (m.bias is not None and m.bias.requires_grad)))


def linear_trains(m: nn.Linear, x: Tensor) -> bool:
    """Whether ``ops.linear_autograd`` may stand in for ``m(x)``: an ordinary call, with or without autocast, in a 16-bit type, of
    a module that would run ``nn.Linear.forward`` and nothing else, on so many rows that the kernel for the weight's gradient
    is the faster one."""
    # (first: few rows wait for the host)
    if not torch.is_grad_enabled() or not sizes_are_known(x) or not ops.linear_wgrad_pays(x.numel() // max(x.shape[-1], 1)):
        return False
    dtype = torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else x.dtype
    return calls_forward_only(m, nn.Linear) and nn.Linear.forward is LINEAR_FORWARD and type(m.weight) is nn.Parameter and m.weight.requires_grad \
        and dtype in (torch.bfloat16, torch.float16) and x.shape[-1] == m.weight.shape[1] \
        and ops.linear_wgrad_takes(*m.weight.shape) \
        and ops.unchanged_here(x) \
        and all(t is None or t.dtype in (torch.float32, torch.bfloat16, torch.float16) for t in (x, m.weight, m.bias))


# The function in the place of F.linear costs the host up to 40 us a product under autocast, what its kernels save of the device counts where
# the step waits for the device.  Multiply-adds of a product from which that is so (and, of a layer under autocast, rows: with fewer the step
# waits for the host), us a step, torch's / here.  An MLP (its two products) under autocast: 4 160 rows of 1024 channels 384 / 470, 6 016 479 /
# 475, 8 320 663 / 557; 8 320 of 768 488 / 483; 12 032 of 512 424 / 341; without: 6 016 of 512 273 / 309, 8 320 301 / 229, 4 160 of 768 263 / 231,
# 2 048 of 1024 275 / 275.  A layer (its projection, which gives its other products their way too) under autocast: 8 064 rows of 1024 channels
# 1 022 / 1 017, 12 096 1 136 / 1 021, 16 128 1 366 / 1 135; 12 096 of 768 1 123 / 1 142, 24 192 1 708 / 1 415; 6 048 of 1536 1 046 / 1 157, 8 064
# 1 178 / 1 154, 12 096 1 701 / 1 482; without: 6 048 of 768 965 / 932, 4 032 of 1024 903 / 906, 6 048 895 / 832, 8 064 905 / 831, 12 096
# 1 085 / 879.
def training_pays(x: Tensor, m: nn.Module, layer: bool) -> bool:
    """Whether the gradients of ``m``'s parameters, those of an attention layer's projection or another product, are enough work
    for :func:`linear_with_grad` in the place of ``m(x)``."""
    if not sizes_are_known(x) or type(m) is not nn.Linear:
        return False
    work = x.numel() * m.weight.shape[0]
    if not torch.is_autocast_enabled("cuda"):
        return work >= (1e10 if layer else 8.5e9)
    if not layer:
        return work >= 2e10
    return work >= 6e10 or (work >= 3.5e10 and x.numel() >= 10000 * x.shape[-1])


def linear_with_grad(m: nn.Linear, x: Tensor) -> Tensor:
    """``m(x)`` in training: with a kernel for the parameters' gradients where :func:`linear_trains` says so."""
    return ops.linear_autograd(x, m.weight, m.bias) if linear_trains(m, x) else m(x)


def linear(m: nn.Linear, x: Tensor, gelu: bool = False, trains: Optional[bool] = None) -> Tensor:
    """``m(x)``, with ``gelu`` followed by ``F.gelu``: one kernel where :func:`linear_takes` says so, the product with a kernel for
    the parameters' gradients where :func:`linear_trains` does (and ``trains``, where it is given), else the modules."""
    if trains is not False and linear_trains(m, x):
        out = ops.linear_autograd(x, m.weight, m.bias)
        return nn.functional.gelu(out) if gelu else out
    if linear_takes(m, x, gelu):
        out = ops.linear(x, m.weight, m.bias, gelu)
        if out is not None:
            return out
    return nn.functional.gelu(m(x)) if gelu else m(x)


def project_args(attn: nn.Module, x: Tensor, pos: Optional[Tensor], n_pos: Optional[int], block: int, pooled: bool):
    """:func:`fused_qk_args` of a layer's projection with all that follows it row by row, or None where the kernel does not take the
    layer or does not stand in for its modules (then: ``linear`` and the passes over its result)."""
    # (asked before the tables are, which the passes over the projection ask for again and a rope of another kind looks at the positions for)
    if pos is None or not linear_takes(attn.qkv, x) or pos.is_floating_point() or x.dim() != 3 \
            or not ops.qkv_project_takes(x, attn.num_heads, block, pooled, isinstance(attn.q_norm, nn.LayerNorm)):
        return None
    fused = fused_qk_args(attn, x, pos, n_pos, takes=True)
    return fused if fused is not None and fused[0].shape == (*x.shape[:2], 2) else None


def project(attn: nn.Module, x: Tensor, fused, block: int, pooled: bool, gate=None):
    """The projection of an attention layer with what :func:`project_args` said, and the layer's gate (weight, bias) beside it
    (``ops.qkv_project``); None where there is nothing to say."""
    if fused is None:
        return None
    return ops.qkv_project(x, attn.qkv.weight, attn.qkv.bias, attn.num_heads, block, *fused[:3], *fused[4:], pooled=pooled, inv_freq=fused[3],
                           gate=gate, takes=True)


def norm_rope_fused_or_eager(t: Tensor, norm: nn.Module, rope, pos: Optional[Tensor], n_pos: Optional[int] = None) -> Tensor:
    """qk-norm, cast and RoPE of one ``[B,H,N,D]`` tensor (reference sparse_attention.py:103-110,120-124): one fused
    kernel where it is built -- a tensor on the GPU, head_dim 64, ``nn.Identity`` or an affine ``nn.LayerNorm`` of
    exactly that type, the package's RoPE2D or no rotation -- and the separate torch modules otherwise (any other norm
    module, a LayerNorm without affine parameters, another rope).  Same rounding points either way, except that the
    kernel takes the LayerNorm parameters in the tokens' dtype (fp32 parameters under autocast are rounded to it).
    ``n_pos``: number of rows of the kernel's cos/sin tables for THIS call (every coordinate in ``pos`` must be below it;
    the kernel clamps larger ones); default: the rope module's ``max_positions``, else ``pos.max() + 1`` (a device
    synchronisation)."""
    fused_norm = isinstance(norm, nn.Identity) or (type(norm) is nn.LayerNorm and norm.elementwise_affine)
    fused_rope = pos is None or isinstance(rope, RoPE2D)
    if t.is_cuda and t.shape[-1] == 64 and fused_norm and fused_rope and not (isinstance(norm, nn.Identity) and pos is None):
        cos = sin = None
        if pos is not None:
            rows = n_pos or rope.max_positions or int(pos.max()) + 1
            cos, sin = rope.tables(64, rows, t.device, t.dtype)
        ln = norm if isinstance(norm, nn.LayerNorm) else None
        out = ops.norm_rope(t, pos, cos, sin, ln.weight if ln is not None else None,
                            ln.bias if ln is not None else None, ln.eps if ln is not None else 0.0)
        if out is not None:
            return out
    t = norm(t).to(t.dtype)
    return rope(t, pos) if pos is not None else t


def fused_qk_args(attn: nn.Module, qkv: Tensor, pos: Optional[Tensor], n_pos: Optional[int] = None, training: bool = False,
                  takes: Optional[bool] = None):
    """``(pos, cos, sin, inv_freq, q_ln, k_ln, eps)`` for the kernels that take qk-norm and RoPE with the packed
    projection, or None where their conditions do not hold (those of ``norm_rope_fused_or_eager`` for both norms).
    ``takes``: whether the kernel takes ``qkv`` (default: a packed projection, ``ops.prepass_takes``).
    ``training``: in the place of the modules' own calls, which know no bound of the positions and must do nothing else."""
    def plain(norm):
        if training and not (calls_forward_only(norm, nn.Identity) or calls_forward_only(norm, nn.LayerNorm)):
            return False
        return isinstance(norm, nn.Identity) or (type(norm) is nn.LayerNorm and norm.elementwise_affine)
    same_kind = isinstance(attn.q_norm, nn.Identity) == isinstance(attn.k_norm, nn.Identity)
    if takes is None:
        takes = qkv.is_cuda and ops.prepass_takes(qkv, attn.num_heads)
    if not (takes and plain(attn.q_norm) and plain(attn.k_norm) and same_kind
            and (pos is None or (calls_forward_only(attn.rope, RoPE2D) if training else isinstance(attn.rope, RoPE2D)))):
        return None
    if training and pos is not None:   # (a rope module takes one set of positions for all sequences, fractional ones, and more)
        if pos.is_floating_point() or pos.shape not in (qkv.shape[:2] + (2,), (1, qkv.shape[1], 2)):
            return None
        pos = pos.expand(*qkv.shape[:2], 2)
    ln = isinstance(attn.q_norm, nn.LayerNorm)
    if ln and attn.q_norm.eps != attn.k_norm.eps:
        return None
    cos = sin = inv_freq = None
    if pos is not None:
        if not training and type(attn.rope).tables is not RoPE2D.tables and not (n_pos or attn.rope.max_positions):
            n_pos = int(pos.max()) + 1   # (the kernels' own angles are RoPE2D's: tables of another kind hold every position)
        cos, sin, inv_freq = attn.rope.fused_tables(64, n_pos, qkv.device, qkv.dtype, bounded=not training)
    return (pos, cos, sin, inv_freq, (attn.q_norm.weight, attn.q_norm.bias) if ln else None,
            (attn.k_norm.weight, attn.k_norm.bias) if ln else None, attn.q_norm.eps if ln else 0.0)


class SparseFlashAttentionRope(nn.Module):
    def __init__(
        self,
        dim: int,
        num_heads: int = 16,
        qkv_bias: bool = False,
        proj_bias: bool = True,
        attn_drop: float = 0.0,
        proj_drop: float = 0.0,
        qk_norm: bool = False,
        norm_layer=nn.LayerNorm,
        rope=None,
        block_size: int = 4,
        topk: int = 32,
    ) -> None:
        super().__init__()
        assert dim % num_heads == 0, "dim must be a multiple of num_heads"
        self.num_heads = num_heads
        head_dim = dim // num_heads
        self.scale = head_dim ** -0.5  # kept for parity with the reference; both operators default to it

        self.qkv = nn.Linear(dim, dim * 3, bias=qkv_bias)
        self.attn_drop = nn.Dropout(attn_drop)
        self.proj = nn.Linear(dim, dim, bias=proj_bias)
        self.proj_drop = nn.Dropout(proj_drop)
        self.q_norm = norm_layer(head_dim) if qk_norm else nn.Identity()
        self.k_norm = norm_layer(head_dim) if qk_norm else nn.Identity()
        self.rope = rope

        # gate: sigmoid(linear), weight 0 and bias (-1, +1) per head at initialisation
        gate_linear = nn.Linear(dim, num_heads * 2, bias=True)
        nn.init.zeros_(gate_linear.weight)
        with torch.no_grad():
            gate_linear.bias.copy_(torch.tensor([-1.0, 1.0]).repeat(num_heads))
        self.gate = nn.Sequential(gate_linear, nn.Sigmoid())
        self.block_size = block_size
        self.topk = topk
        self.keep_topk_idx = False   # debugging aid: keep the last forward's block indices in ``last_topk_idx``
        self.last_topk_idx = None
        self.last_prepass = None     # whether the last forward took q, k and the block means from one launch over the packed projection
        self.last_passes = None      # the launches that made these: 1 (a pass over the projection, or the projection's own kernel), 2 (block
                                     # means, then q and k) or 0 (kernels per tensor)
        self.last_path = None        # which route the last forward took: "fused-merge", "two-operators" or "autograd"

    def _norm_rope(self, t: Tensor, norm: nn.Module, pos: Optional[Tensor], n_pos: Optional[int] = None) -> Tensor:
        return norm_rope_fused_or_eager(t, norm, self.rope, pos, n_pos)

    def _plain_gate(self) -> bool:
        """Whether the gate is the plain pair of modules it was built as, whose calls run nothing but their ``forward``."""
        return calls_forward_only(self.gate, nn.Sequential) and len(self.gate) == 2 and calls_forward_only(self.gate[0], nn.Linear) \
            and calls_forward_only(self.gate[1], nn.Sigmoid)

    def _gate(self, x: Tensor) -> Tensor:
        """``self.gate(x)`` for inference: one kernel where it is plain, and outside of autocast."""
        if x.is_cuda and self._plain_gate() and not torch.is_autocast_enabled("cuda"):
            out = ops.gate(x, self.gate[0].weight, self.gate[0].bias)
            if out is not None:
                return out
        return self.gate(x)

    def _forward_with_grad(self, x: Tensor, xpos: Optional[Tensor], n_pos: Optional[int] = None) -> Tensor:
        """The same layer for training.  Between its projections it is one differentiable operator whose forward and
        backward are kernels (``ops.layer_core_autograd``; where only the gate is trained, the attention without gradients
        and the merge as a torch expression).  Where that is not built (another norm or rope module, blocks of
        128 or 256 tokens): a composition in which the two attention operators carry their own backward kernels and pooling,
        qk-norm/RoPE and the gated merge run as the torch expressions of the reference (sparse_attention.py:97-110,120-136),
        whose gradients autograd provides."""
        b, n, c = x.shape
        h = self.num_heads
        block = self.block_size ** 2
        product = linear_with_grad if training_pays(x, self.qkv, layer=True) else lambda m, t: m(t)
        if product is linear_with_grad and linear_trains(self.qkv, x) and self._plain_gate() and linear_trains(self.gate[0], x):
            x = ops.autocast_once(x)
            qkv = ops.linear_autograd(x, self.qkv.weight, self.qkv.bias)
            gate = torch.sigmoid(ops.linear_autograd(x, self.gate[0].weight, self.gate[0].bias))
        else:
            qkv, gate = product(self.qkv, x), self.gate(x)
        gate = gate.view(b, n, h, 2).permute(0, 2, 1, 3)                      # [B, H, N, 2]
        use_pos = xpos is not None and self.rope is not None
        fused = fused_qk_args(self, qkv, xpos if use_pos else None, n_pos, training=True)
        branches = None
        if fused is not None and self.topk in (1, 2, 4, 8, 16, 32, 64):
            pos, cos, sin, inv_freq, q_ln, k_ln, eps = fused
            core = ops.layer_core_autograd(qkv, gate, h, block, self.topk, pos, cos, sin, inv_freq, q_ln, k_ln, eps)
            if core is not None:
                *branches, idx = core
                if self.keep_topk_idx:
                    self.last_topk_idx = idx
                if len(branches) == 1:
                    return self.proj_drop(product(self.proj, branches[0]))
        o_c, o_s = branches if branches is not None else self._branches_with_grad(qkv, xpos if use_pos else None)
        blk = torch.arange(n, device=x.device) // block
        out = gate[..., 0:1] * o_c[:, :, blk] + gate[..., 1:2] * o_s           # [B, H, N, D]
        out = out.permute(0, 2, 1, 3).reshape(b, n, c)
        return self.proj_drop(product(self.proj, out))

    def _branches_with_grad(self, qkv: Tensor, xpos: Optional[Tensor]):
        """Outputs of the two attention branches as a composition of torch expressions around the attention operators."""
        b, n, c3 = qkv.shape
        h = self.num_heads
        d = c3 // (3 * h)
        block = self.block_size ** 2
        nc = -(-n // block)
        q, k, v = qkv.view(b, n, 3, h, d).permute(2, 0, 3, 1, 4).unbind(0)    # each [B, H, N, D]

        def pool(t):  # block means; a ragged tail block averages its valid tokens
            pad = nc * block - n
            tf = torch.nn.functional.pad(t, (0, 0, 0, pad)) if pad else t
            sums = tf.reshape(b, h, nc, block, d).float().sum(dim=3)
            counts = torch.full((nc, 1), float(block), device=t.device)
            if pad:
                counts[-1] = float(block - pad)
            return (sums / counts).to(t.dtype)

        def norm_rope(t, norm, pos):
            t = norm(t).to(t.dtype)
            return self.rope(t, pos) if pos is not None else t

        pos_c = block_positions(xpos, block) if xpos is not None else None
        q_c, k_c, v_c = pool(q), pool(k), pool(v)
        q_c, k_c = norm_rope(q_c, self.q_norm, pos_c), norm_rope(k_c, self.k_norm, pos_c)
        o_c, idx = flash_attn_topk_func(q_c, k_c, v_c, self.topk)
        if self.keep_topk_idx:
            self.last_topk_idx = idx
        q, k = norm_rope(q, self.q_norm, xpos), norm_rope(k, self.k_norm, xpos)
        return o_c, ops.select_attn_autograd(q, k, v, idx, block)

    def forward(self, x: Tensor, attn_bias=None, xpos: Optional[Tensor] = None, n_pos: Optional[int] = None) -> Tensor:
        """``n_pos`` (optional, beyond the reference's signature): an upper bound, exclusive, of the coordinates in
        ``xpos`` for this call; sizes the fused kernels' cos/sin tables without a device synchronisation and without
        touching state shared between calls.  Larger coordinates are clamped to it for inference; a training call gives
        them their own angles."""
        if torch.is_grad_enabled() and (x.requires_grad or any(p.requires_grad for p in self.parameters())):
            self.last_path = "autograd"
            return self._forward_with_grad(x, xpos, n_pos)
        b, n, c = x.shape
        h = self.num_heads
        d = c // h
        block = self.block_size ** 2

        use_pos = xpos is not None and self.rope is not None
        pos = xpos if use_pos else None
        # The projection and all that follows it row by row in one kernel, where that takes the layer.  Else one pass over the
        # packed projection: block means of the raw q, k, v, normalised and rotated at the block
        # positions (compressed branch), and norm + RoPE of the full-token q and k (selection branch), each input row read
        # once.  Where that kernel is not built (head_dim other than 64, another norm or rope module): pooling kernel, then
        # norm/RoPE per tensor.  16-token blocks take the pass in two launches: the block means first, so that the index
        # kernel, long for so many pooled tokens, starts while the full tokens are still to come.
        q = k = v = fused = qkv = None
        self.last_prepass, self.last_passes = False, 0
        gate = None
        projected = None
        if pos is not None and enough_work(x):
            args = project_args(self, x, pos, n_pos, block, True)
            gate_args = (self.gate[0].weight, self.gate[0].bias) if args is not None and self._plain_gate() else None
            if gate_args is not None and not self.keep_topk_idx:
                # all of the layer in one call where the kernels follow each other on this stream: 2 016 tokens of 1024 channels
                # wait for the host, 126 us with a call a kernel, 81 with one
                with_proj = linear_takes(self.proj, x, False)
                out = ops.attention_layer(x, (self.qkv.weight, self.qkv.bias), gate_args, (self.proj.weight, self.proj.bias) if with_proj else None,
                                          h, block, self.topk, *args[:3], *args[4:], args[3])
                if out is not None:
                    self.last_prepass, self.last_passes, self.last_path = True, 1, "fused-merge"
                    return self.proj_drop(out if with_proj else linear(self.proj, out))
            projected = project(self, x, args, block, True, gate_args)
        if projected is None:
            qkv = linear(self.qkv, x)                                  # [B, N, 3C], layout (qkv h d)
            fused = fused_qk_args(self, qkv, pos, n_pos)
        if projected is not None:
            q, k, v, q_c, k_c, v_c = projected[:6]
            gate = projected[6] if len(projected) > 6 else None
            self.last_prepass, self.last_passes = True, 1
        elif fused is not None and (pos is not None or fused[4] is not None):   # (else q and k are read in place)
            args = (pos, fused[1], fused[2], *fused[4:])
            self.last_prepass = block >= 32
            self.last_passes = 1 if self.last_prepass else 2
            if self.last_prepass:
                q, k, v, q_c, k_c, v_c = ops.qkv_prepass(qkv, h, block, *args, pooled="final", inv_freq=fused[3])
            else:
                q_c, k_c, v_c = ops.qkv_prepass(qkv, h, block, *args, tokens=False, pooled="final", inv_freq=fused[3])
        else:
            q_c, k_c, v_c = ops.pool_qkv_packed(qkv, h, block)
            pos_c = block_positions(xpos, block) if use_pos else None
            q_c, k_c = self._norm_rope(q_c, self.q_norm, pos_c, n_pos), self._norm_rope(k_c, self.k_norm, pos_c, n_pos)
        # the index kernel needs pooled q and k only and its result is first read by the selection kernel: where
        # it is a kernel of its own, and long enough, it runs on a second stream, beside the compressed attention (and the norm/RoPE of
        # the full tokens where they come after it)
        side = x.is_cuda and ops._indices_beside(q_c, self.topk)
        if side:
            idx, join = ops.topk_indices_on_side_stream(q_c, k_c, self.topk)
            o_c, _ = ops.compressed_attn_topk(q_c, k_c, v_c, None)
        else:
            o_c, idx = flash_attn_topk_func(q_c, k_c, v_c, self.topk)
        gate = (self._gate(x) if gate is None else gate).view(b, n, h, 2).permute(0, 2, 1, 3)   # [B, H, N, 2], strided view

        if q is None and fused is not None and (pos is not None or fused[4] is not None):
            q, k, v = ops.qkv_prepass(qkv, h, 64, *args, pooled=None, inv_freq=fused[3])
        elif q is None:  # selection branch on strided views of the projection; norm/RoPE make q, k contiguous
            q, k, v = qkv.view(b, n, 3, h, d).permute(2, 0, 3, 1, 4).unbind(0)   # each [B, H, N, D]
            q, k = self._norm_rope(q, self.q_norm, pos, n_pos), self._norm_rope(k, self.k_norm, pos, n_pos)
        if side:
            join()
        if self.keep_topk_idx:
            self.last_topk_idx = idx

        out = ops._select_attn_merge(q, k, v, idx, o_c, gate, block)
        self.last_path = "fused-merge"
        if out is None:
            self.last_path = "two-operators"
            out = ops.gated_merge(o_c, ops.select_attn(q, k, v, idx, block), gate, block)

        out = linear(self.proj, out)
        return self.proj_drop(out)
