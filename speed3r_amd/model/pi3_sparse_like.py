"""A Pi3_Sparse-style multi-view forward built around the package's sparse global attention layer.

Purpose: the end-to-end throughput figure (frames/s, share of time in the sparse attention) of the reference's
model family on random-initialised weights; it is not a weight-compatible re-implementation of the reference model.
Structure after pi3/models/pi3_sparse.py:74-321 (encoder -> alternating frame-local / global decoder -> point,
confidence and camera heads), pi3/models/layers/block.py:259-335 (pre-norm block with LayerScale),
pi3/models/layers/transformer_head.py (head decoders, linear pixel-shuffle head):

* patch encoder: ViT-L/14 with a class token and 4 register tokens (dim 1024, 24 blocks), dense attention per frame;
* decoder: ``dec_depth // 2`` pairs of [frame-local dense attention block, global sparse attention block]
  (dim 1024, 16 heads, MLP x4, qk-LayerNorm, LayerScale 0.01, RoPE2D base 100); the global block is
  ``speed3r_amd.layers.SparseFlashAttentionRope`` over all frames' tokens;
* tokens per frame: ``num_register`` register tokens followed by the patches in row-major order (the Pi3 teacher's
  layout, pi3/models/pi3.py:140-154), so 518x392 frames give 5 + 37*28 = 1041 tokens; the global attention sees the
  flat sequence in blocks of 64 tokens with the ragged-tail policy of the kernels;
* heads: three 5-block frame-local decoders on the concatenated outputs of the last local and global blocks, a linear
  pixel-shuffle head for local points and confidence, a small pose head.
* ``token_order="tile"`` with ``num_register=0, block_tokens=16, topk=32`` is the reference model's own token
  pipeline: no register tokens (pi3_sparse.py:163-169), positions from 0 (pos_embed.py:162-174), every frame's patches
  in 4 x 4-tile-major order through the decoder (pi3_sparse.py:29-45,228-229) and back in row-major order in front of
  the head decoders (:265-269), global attention over 16-token blocks = 4 x 4 patch tiles with the 32 best blocks
  (sparse_attention.py:73,98,112).  The patch grid must split into 4 x 4 tiles (frames of 56-pixel multiples).

The linear layers run on the package's kernel (GELU of the MLPs in its epilogue) for bf16/fp16 inference where their sizes
allow, else on library calls, as do the patch embedding and the pixel-shuffle heads; the frame-local dense attentions run on the package's
dense flash kernel (the one behind the compressed branch) for bf16/fp16 inference with head_dim 64, else on
scaled_dot_product_attention.
Inference only: call under ``torch.no_grad()`` with the module in one dtype (bf16).
"""
from __future__ import annotations

from functools import partial
from typing import Optional

import torch
import torch.nn.functional as F
from torch import Tensor, nn

from ..layers import RoPE2D, SparseFlashAttentionRope
from ..layers.sparse_attention import calls_forward_only, fused_qk_args, linear, norm_rope_fused_or_eager, project, project_args, training_pays
from ..sparse_attn import ops
from .token_order import tile_major, tile_major_inverse


def product(m: nn.Module, x: Tensor, gelu: bool = False, layer: bool = False) -> Tensor:
    """``linear``, in training where the product is enough work for it (``layer``: an attention layer's projection)."""
    return linear(m, x, gelu, trains=torch.is_grad_enabled() and training_pays(x, m, layer))


class Mlp(nn.Module):
    def __init__(self, dim: int, hidden: int) -> None:
        super().__init__()
        self.fc1 = nn.Linear(dim, hidden)
        self.fc2 = nn.Linear(hidden, dim)

    def forward(self, x: Tensor) -> Tensor:
        if torch.jit.is_scripting():
            return self.fc2(F.gelu(self.fc1(x)))
        else:   # (not compiled by TorchScript)
            return product(self.fc2, product(self.fc1, x, gelu=True))


class LayerScale(nn.Module):
    def __init__(self, dim: int, init_values: float) -> None:
        super().__init__()
        self.gamma = nn.Parameter(init_values * torch.ones(dim))

    def forward(self, x: Tensor) -> Tensor:
        return x * self.gamma

    def add_to(self, residual: Tensor, x: Tensor) -> Tensor:  # residual + gamma * x in one pass
        return torch.addcmul(residual, x, self.gamma)


def token_norm(norm: nn.LayerNorm, x: Tensor) -> Tensor:
    """The block norms: the package's one-pass kernel for inference on the GPU, the torch module otherwise."""
    if x.is_cuda and not torch.is_grad_enabled() and norm.elementwise_affine and x.dtype == norm.weight.dtype:
        y = ops.layer_norm(x, norm.weight, norm.bias, norm.eps)
        if y is not None:
            return y
    return norm(x)


def add_and_norm(x: Tensor, scale: nn.Module, branch: Tensor, norm: Optional[nn.LayerNorm]):
    """``(s, norm(s))`` of the residual sum ``s = x + scale(branch)``: one pass for inference on the GPU (``norm=None``:
    ``(s, None)``)."""
    scaled = isinstance(scale, LayerScale)
    plain = not scaled or (type(scale) is LayerScale and "add_to" not in vars(scale))
    if plain and norm is not None and x.is_cuda and not torch.is_grad_enabled() and norm.elementwise_affine and x.dtype == norm.weight.dtype:
        out = ops.add_layer_norm(x, branch, scale.gamma if scaled else None, norm.weight, norm.bias, norm.eps)
        if out is not None:
            return out
    s = scale.add_to(x, branch) if scaled else x + branch
    return s, token_norm(norm, s) if norm is not None else None


class DenseAttentionRope(nn.Module):
    """Dense attention inside each sequence of the batch (one frame), optional qk-norm and RoPE2D."""

    def __init__(self, dim, num_heads=16, qkv_bias=True, proj_bias=True, attn_drop=0.0, proj_drop=0.0, qk_norm=False,
                 norm_layer=nn.LayerNorm, rope=None) -> None:
        super().__init__()
        self.num_heads = num_heads
        head_dim = dim // num_heads
        self.qkv = nn.Linear(dim, dim * 3, bias=qkv_bias)
        self.proj = nn.Linear(dim, dim, bias=proj_bias)
        self.q_norm = norm_layer(head_dim) if qk_norm else nn.Identity()
        self.k_norm = norm_layer(head_dim) if qk_norm else nn.Identity()
        self.rope = rope

    def _norm_rope(self, t: Tensor, norm: nn.Module, pos: Optional[Tensor], n_pos: Optional[int] = None) -> Tensor:
        return norm_rope_fused_or_eager(t, norm, self.rope, pos, n_pos)

    def forward(self, x: Tensor, attn_bias=None, xpos: Optional[Tensor] = None, n_pos: Optional[int] = None) -> Tensor:
        b, n, c = x.shape
        h = self.num_heads
        pos = xpos if self.rope is not None else None
        projected = project(self, x, project_args(self, x, pos, n_pos, 64, False), 64, False) if not torch.is_grad_enabled() else None
        if projected is None:
            qkv = product(self.qkv, x, layer=True)
            fused = fused_qk_args(self, qkv, pos, n_pos) if not torch.is_grad_enabled() else None
            if fused is not None and (pos is not None or fused[4] is not None):   # one pass over the projection for q and k
                projected = ops.qkv_prepass(qkv, h, 64, *fused[:3], *fused[4:], pooled=None, inv_freq=fused[3])
        if projected is not None:
            q, k, v = projected
        else:
            q, k, v = qkv.view(b, n, 3, h, c // h).permute(2, 0, 3, 1, 4).unbind(0)
            q, k = self._norm_rope(q, self.q_norm, pos, n_pos), self._norm_rope(k, self.k_norm, pos, n_pos)
        if x.is_cuda and x.dtype in (torch.bfloat16, torch.float16) and c // h == 64 and not torch.is_grad_enabled():
            # the package's dense flash kernel (the compressed branch's attention), written straight into [B,N,H,D]
            o = torch.empty((b, n, h, c // h), dtype=x.dtype, device=x.device)
            ops.compressed_attn_topk(q, k, v, None, out=o.permute(0, 2, 1, 3))
            return product(self.proj, o.view(b, n, c), layer=True)
        o = F.scaled_dot_product_attention(q, k, v)
        return self.proj(o.transpose(1, 2).reshape(b, n, c))


class Block(nn.Module):
    def __init__(self, dim, num_heads, attn_class, mlp_ratio=4.0, init_values=None, qk_norm=False, rope=None, **attn_kw):
        super().__init__()
        self.norm1 = nn.LayerNorm(dim, eps=1e-6)
        self.attn = attn_class(dim, num_heads=num_heads, qkv_bias=True, proj_bias=True, qk_norm=qk_norm,
                               norm_layer=partial(nn.LayerNorm, eps=1e-6), rope=rope, **attn_kw)
        self.ls1 = LayerScale(dim, init_values) if init_values else nn.Identity()
        self.norm2 = nn.LayerNorm(dim, eps=1e-6)
        self.mlp = Mlp(dim, int(dim * mlp_ratio))
        self.ls2 = LayerScale(dim, init_values) if init_values else nn.Identity()

    def forward(self, x: Tensor, xpos: Optional[Tensor] = None, n_pos: Optional[int] = None) -> Tensor:
        return self._run(x, token_norm(self.norm1, x), None, xpos, n_pos)[0]

    def _run(self, x, normed, next_norm, xpos=None, n_pos=None):
        """The block on ``x`` with ``normed = norm1(x)`` at hand: its output and ``next_norm`` of that (None without)."""
        x, y = add_and_norm(x, self.ls1, self.attn(normed, xpos=xpos, n_pos=n_pos), self.norm2)
        return add_and_norm(x, self.ls2, self.mlp(y), next_norm)


def takes_normed(blk: nn.Module) -> bool:
    """Whether ``blk`` may be handed ``norm1`` of its input from the block before it: for inference, where calling the
    module would run ``Block.forward`` and nothing else."""
    return not torch.is_grad_enabled() and calls_forward_only(blk, Block)


def run_block(blk: nn.Module, x: Tensor, normed: Optional[Tensor], next_norm: Optional[nn.LayerNorm], **kw):
    """One block of a sequence: its output and, where it could be had in the pass over the residual sum, ``next_norm`` of
    that output (else None).  ``normed``: ``norm1(x)`` if the block before it gave it."""
    if takes_normed(blk):
        return blk._run(x, token_norm(blk.norm1, x) if normed is None else normed, next_norm, **kw)
    return blk(x, **kw), None


def run_blocks(blocks, x: Tensor, last_norm: Optional[nn.LayerNorm], **kw):
    """``blocks`` in sequence: the last one's output and ``last_norm`` of it (None without)."""
    y = None
    for blk, after in zip(blocks, [*list(blocks)[1:], None]):
        x, y = run_block(blk, x, y, last_norm if after is None else after.norm1 if takes_normed(after) else None, **kw)
    return x, token_norm(last_norm, x) if y is None and last_norm is not None else y


class PatchEncoder(nn.Module):
    """ViT patch encoder: class token + register tokens + patch tokens with a learned position embedding."""

    def __init__(self, dim=1024, depth=24, num_heads=16, patch=14, grid=(37, 28), num_register=4) -> None:
        super().__init__()
        self.patch = patch
        self.grid = grid
        self.patch_embed = nn.Conv2d(3, dim, kernel_size=patch, stride=patch)
        self.cls_token = nn.Parameter(torch.zeros(1, 1, dim))
        self.register_tokens = nn.Parameter(torch.zeros(1, num_register, dim))
        self.pos_embed = nn.Parameter(torch.randn(1, 1 + grid[0] * grid[1], dim) * 0.02)
        self.blocks = nn.ModuleList([Block(dim, num_heads, DenseAttentionRope, init_values=1e-5) for _ in range(depth)])
        self.norm = nn.LayerNorm(dim, eps=1e-6)

    def _pos(self, gh: int, gw: int) -> Tensor:
        if (gh, gw) == self.grid:
            return self.pos_embed
        cls, patch = self.pos_embed[:, :1], self.pos_embed[:, 1:]
        patch = patch.view(1, self.grid[0], self.grid[1], -1).permute(0, 3, 1, 2).float()
        patch = F.interpolate(patch, size=(gh, gw), mode="bicubic", align_corners=False).to(self.pos_embed.dtype)
        return torch.cat((cls, patch.permute(0, 2, 3, 1).reshape(1, gh * gw, -1)), dim=1)

    def forward(self, imgs: Tensor) -> Tensor:  # [F,3,H,W] -> patch tokens [F, gh*gw, dim]
        f, ch, hh, ww = imgs.shape
        p = self.patch
        gh, gw = hh // p, ww // p
        # kernel == stride: the convolution is one GEMM over the unfolded patches (same parameters as the Conv2d)
        x = imgs[:, :, :gh * p, :gw * p].reshape(f, ch, gh, p, gw, p).permute(0, 2, 4, 1, 3, 5).reshape(f, gh * gw, ch * p * p)
        x = F.linear(x, self.patch_embed.weight.reshape(self.patch_embed.out_channels, -1), self.patch_embed.bias)
        x = torch.cat((self.cls_token.expand(f, -1, -1), x), dim=1) + self._pos(gh, gw)
        x = torch.cat((x[:, :1], self.register_tokens.expand(f, -1, -1), x[:, 1:]), dim=1)
        return run_blocks(self.blocks, x, self.norm)[1][:, 1 + self.register_tokens.shape[1]:]


class HeadDecoder(nn.Module):
    def __init__(self, in_dim, out_dim, dim=1024, depth=5, num_heads=16, rope=None) -> None:
        super().__init__()
        self.project = nn.Linear(in_dim, dim)
        self.blocks = nn.ModuleList([Block(dim, num_heads, DenseAttentionRope, rope=rope) for _ in range(depth)])
        self.linear_out = nn.Linear(dim, out_dim)

    def forward(self, x: Tensor, xpos: Tensor, n_pos: Optional[int] = None) -> Tensor:
        return product(self.linear_out, run_blocks(self.blocks, product(self.project, x), None, xpos=xpos, n_pos=n_pos)[0])


class PixelShuffleHead(nn.Module):
    def __init__(self, patch: int, dim: int, out_dim: int) -> None:
        super().__init__()
        self.patch = patch
        self.proj = nn.Linear(dim, out_dim * patch * patch)

    def forward(self, tokens: Tensor, gh: int, gw: int) -> Tensor:  # [F, gh*gw, dim] -> [F, H, W, out]
        f = tokens.shape[0]
        feat = self.proj(tokens).transpose(-1, -2).reshape(f, -1, gh, gw)
        return F.pixel_shuffle(feat, self.patch).permute(0, 2, 3, 1)


class PoseHead(nn.Module):
    """Frame tokens -> 4x4 camera-to-world matrix (rotation from two 3-vectors by Gram-Schmidt, translation)."""

    def __init__(self, dim: int) -> None:
        super().__init__()
        self.mlp = nn.Sequential(nn.Linear(dim, dim), nn.GELU(), nn.Linear(dim, 9))

    def forward(self, tokens: Tensor) -> Tensor:  # [F, T, dim] -> [F, 4, 4]
        p = self.mlp(tokens.mean(dim=1)).float()
        a, b, t = p[:, 0:3], p[:, 3:6], p[:, 6:9]
        e1 = F.normalize(a + torch.tensor([1.0, 0.0, 0.0], device=p.device), dim=-1)
        b = b + torch.tensor([0.0, 1.0, 0.0], device=p.device)
        e2 = F.normalize(b - (e1 * b).sum(-1, keepdim=True) * e1, dim=-1)
        e3 = torch.cross(e1, e2, dim=-1)
        pose = torch.zeros((p.shape[0], 4, 4), device=p.device)
        pose[:, :3, :3] = torch.stack((e1, e2, e3), dim=-1)
        pose[:, :3, 3] = t
        pose[:, 3, 3] = 1.0
        return pose


class Pi3SparseLike(nn.Module):
    def __init__(self, dim=1024, enc_depth=24, dec_depth=36, num_heads=16, head_depth=5, patch=14, grid=(37, 28),
                 num_register=5, block_tokens=64, topk=16, rope_freq=100.0, token_order="row", tile=4) -> None:
        super().__init__()
        assert dec_depth % 2 == 0 and int(block_tokens ** 0.5) ** 2 == block_tokens
        assert token_order in ("row", "tile")
        assert token_order == "row" or num_register == 0, "the tile-major order has no place for register tokens"
        self.token_order = token_order
        self.tile = tile
        self.patch = patch
        self.encoder = PatchEncoder(dim, enc_depth, num_heads, patch, grid)
        self.rope = RoPE2D(freq=rope_freq, max_positions=max(grid) + 2)
        self.register_token = nn.Parameter(torch.randn(1, num_register, dim) * 1e-6)
        self.local_decoder = nn.ModuleList([
            Block(dim, num_heads, DenseAttentionRope, init_values=0.01, qk_norm=True, rope=self.rope)
            for _ in range(dec_depth // 2)])
        self.global_decoder = nn.ModuleList([
            Block(dim, num_heads, SparseFlashAttentionRope, init_values=0.01, qk_norm=True, rope=self.rope,
                  block_size=int(block_tokens ** 0.5), topk=topk)
            for _ in range(dec_depth // 2)])
        self.point_decoder = HeadDecoder(2 * dim, dim, dim, head_depth, num_heads, self.rope)
        self.conf_decoder = HeadDecoder(2 * dim, dim, dim, head_depth, num_heads, self.rope)
        self.camera_decoder = HeadDecoder(2 * dim, dim // 2, dim, head_depth, num_heads, self.rope)
        self.point_head = PixelShuffleHead(patch, dim, 3)
        self.conf_head = PixelShuffleHead(patch, dim, 1)
        self.camera_head = PoseHead(dim // 2)
        self.register_buffer("image_mean", torch.tensor([0.485, 0.456, 0.406]).view(1, 3, 1, 1))
        self.register_buffer("image_std", torch.tensor([0.229, 0.224, 0.225]).view(1, 3, 1, 1))

    def _positions(self, f: int, gh: int, gw: int, device) -> Tensor:
        yy, xx = torch.meshgrid(torch.arange(gh, device=device), torch.arange(gw, device=device), indexing="ij")
        patch = torch.stack((yy, xx), dim=-1).reshape(gh * gw, 2)
        if self.register_token.shape[1] == 0:                                     # the reference model: positions from 0
            return patch[None].expand(f, -1, -1).contiguous()
        reg = torch.zeros((self.register_token.shape[1], 2), dtype=patch.dtype, device=device)   # register tokens sit at (0, 0)
        return torch.cat((reg, patch + 1), dim=0)[None].expand(f, -1, -1).contiguous()

    def forward(self, imgs: Tensor, return_features: bool = False) -> dict:
        """imgs [B, F, 3, H, W] in [0,1] -> dict(points, local_points, conf, camera_poses); ``return_features`` adds the
        decoder output the heads read (last frame-local and last global block, concatenated) under "features"."""
        b, f, _, hh, ww = imgs.shape
        gh, gw = hh // self.patch, ww // self.patch
        # cos/sin tables of the fused norm/RoPE kernels sized for THIS call's grid (patch coordinates run up to gh, gw; the
        # kernels clamp positions beyond their table, so a table sized at construction would be wrong for larger
        # frames); handed down call by call, no state shared between calls changes
        n_pos = max(gh, gw) + 1
        x = ((imgs - self.image_mean) / self.image_std).reshape(b * f, 3, hh, ww).to(self.register_token.dtype)
        x = self.encoder(x)                                                        # [B*F, gh*gw, dim]
        x = torch.cat((self.register_token.expand(b * f, -1, -1), x), dim=1)       # [B*F, T, dim]
        t = x.shape[1]
        pos = self._positions(b * f, gh, gw, x.device)                             # [B*F, T, 2]
        tiled = self.token_order == "tile"
        if tiled:                                                                  # tokens and their positions, tile-major
            x, pos_dec = tile_major(x, gh, gw, self.tile), tile_major(pos, gh, gw, self.tile)
        else:
            pos_dec = pos
        local_out = normed = None
        blocks = [blk for pair in zip(self.local_decoder, self.global_decoder) for blk in pair]
        for i, blk in enumerate(blocks):
            # a global block sees the frames of a batch as one sequence
            shape, p = ((b * f, t, -1), pos_dec) if i % 2 == 0 else ((b, f * t, -1), pos_dec.reshape(b, f * t, 2))
            after = blocks[i + 1] if i + 1 < len(blocks) and takes_normed(blocks[i + 1]) else None
            x, normed = run_block(blk, x.reshape(shape), normed.reshape(shape) if normed is not None else None,
                                  after.norm1 if after is not None else None, xpos=p, n_pos=n_pos)
            local_out = x if i % 2 == 0 else local_out
        x = x.reshape(b * f, t, -1)
        feat = torch.cat((local_out, x), dim=-1)
        if tiled:                                                                  # the heads see row-major tokens again
            feat = tile_major_inverse(feat, gh, gw, self.tile)
        nreg = self.register_token.shape[1]
        pts = self.point_head(self.point_decoder(feat, pos, n_pos)[:, nreg:], gh, gw).float()
        conf = self.conf_head(self.conf_decoder(feat, pos, n_pos)[:, nreg:], gh, gw).float()
        poses = self.camera_head(self.camera_decoder(feat, pos, n_pos)).reshape(b, f, 4, 4)
        xy, z = pts.split([2, 1], dim=-1)
        z = torch.exp(z)
        local_points = torch.cat((xy * z, z), dim=-1).reshape(b, f, gh * self.patch, gw * self.patch, 3)
        homog = torch.cat((local_points, torch.ones_like(local_points[..., :1])), dim=-1)
        points = torch.einsum("bnij,bnhwj->bnhwi", poses, homog)[..., :3]
        out = dict(points=points, local_points=local_points,
                   conf=conf.reshape(b, f, gh * self.patch, gw * self.patch, 1), camera_poses=poses)
        if return_features:
            out["features"] = feat
        return out
