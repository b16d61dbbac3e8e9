"""The attention layer's inference in one call of the library: refused arguments (CPU), and the bits of its kernels called one by one (GPU)."""
import ctypes
from functools import partial

import pytest
import torch
from torch import nn

from speed3r_amd import _lib
from speed3r_amd.layers import RoPE2D, SparseFlashAttentionRope
from speed3r_amd.sparse_attn import ops

DEV = "cuda"


def test_refused_before_anything_is_launched():
    L = _lib.lib()
    one, far = ctypes.c_void_p(4096), ctypes.c_void_p(8192)   # (never dereferenced: every call here is refused)

    def call(x=one, gate=one, out=one, ws=far, size=1 << 40, k=16, proj=one, scale=0.125, **fields):
        a = _lib.PrepassArgs(positions=4096, cos_table=4096, sin_table=4096, q_norm_weight=4096, k_norm_weight=4096, N=2048, B=1, H=16, head_dim=64,
                             block=16, table_rows=37, dtype=_lib.S3R_BF16, pos_stride_b=4096, pos_stride_n=2)
        for name, value in fields.items():
            setattr(a, name, value)
        return L.s3r_attention_layer(x, one, None, gate, None, proj, None, out, ws, size, ctypes.byref(a), k, scale, None)

    for name in ("x", "gate", "out", "ws"):
        assert call(**{name: None}) == _lib.S3R_ERR_BAD_ARG
    assert call(N=0) == _lib.S3R_ERR_BAD_ARG and call(k=0) == _lib.S3R_ERR_BAD_ARG
    assert call(k=3) == _lib.S3R_ERR_UNSUPPORTED and call(k=64) == _lib.S3R_ERR_UNSUPPORTED and call(block=32) == _lib.S3R_ERR_UNSUPPORTED
    assert call(H=18) == _lib.S3R_ERR_UNSUPPORTED                                  # a gate that no kernel takes
    assert call(proj=ctypes.c_void_p(4104)) == _lib.S3R_ERR_UNSUPPORTED
    # what the index kernels would refuse behind the projection
    for scale in (0.0, -0.125, float("nan")):
        assert call(scale=scale) == _lib.S3R_ERR_UNSUPPORTED and b"s3r_attention_layer" in L.s3r_last_error()
    assert call(B=4096, N=256, size=1 << 50) == _lib.S3R_ERR_UNSUPPORTED and b"s3r_attention_layer" in L.s3r_last_error()
    need = L.s3r_attention_layer_workspace(1, 16, 2048, 16, 16, 1)
    assert need >= 4 * 2048 * 1024 * 2 and call(size=need - 1) == _lib.S3R_ERR_BAD_ARG
    assert call(ws=ctypes.c_void_p(8192 + 128)) == _lib.S3R_ERR_BAD_ARG and call(out=ctypes.c_void_p(4104)) == _lib.S3R_ERR_BAD_ARG
    assert call(head_dim=32) == _lib.S3R_ERR_UNSUPPORTED and call(positions=None) == _lib.S3R_ERR_BAD_ARG   # by the projection's own checks
    assert L.s3r_attention_layer_workspace(0, 16, 2048, 16, 16, 1) == 0


def _layer(heads, block, topk, dtype, proj_bias=True):
    torch.manual_seed(heads + block)
    with torch.device(DEV):
        m = SparseFlashAttentionRope(64 * heads, num_heads=heads, qkv_bias=True, proj_bias=proj_bias, qk_norm=True,
                                     norm_layer=partial(nn.LayerNorm, eps=1e-6), rope=RoPE2D(freq=100.0), block_size=block, topk=topk)
        nn.init.normal_(m.gate[0].weight, std=0.02)
    return m.to(dtype).eval()


# (sequences, tokens): gates that ride with the projection and that do not, ragged ends, several sequences, few and many blocks
@pytest.mark.gpu
@pytest.mark.parametrize("heads,block,topk,b,n,dtype,bias", [
    (16, 4, 32, 1, 2016, torch.bfloat16, True), (16, 8, 16, 1, 1041, torch.float16, True), (16, 4, 8, 2, 1024, torch.bfloat16, False),
    (4, 4, 4, 1, 4099, torch.bfloat16, True), (16, 8, 2, 1, 25212, torch.bfloat16, True), (8, 8, 1, 3, 1280, torch.float16, False)])
def test_one_call_has_the_bits_of_the_kernels_one_by_one(heads, block, topk, b, n, dtype, bias):
    m = _layer(heads, block, topk, dtype, bias)
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn((b, n, 64 * heads), generator=g, device=DEV).to(dtype)
    pos = torch.randint(0, 40, (b, n, 2), generator=g, device=DEV)
    calls = []
    real = ops.attention_layer
    try:
        ops.attention_layer = lambda *a: (calls.append(real(*a)), calls[-1])[1]
        with torch.no_grad():
            got = m(x, xpos=pos)
            m.keep_topk_idx = True                                               # (which takes the kernels one by one)
            want = m(x, xpos=pos)
    finally:
        ops.attention_layer = real
    assert len(calls) == 1 and calls[0] is not None and m.last_topk_idx is not None
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_a_projection_with_a_hook_is_called():
    m = _layer(16, 4, 16, torch.bfloat16)
    x = torch.randn((1, 2016, 1024), device=DEV).bfloat16()
    pos = torch.randint(0, 36, (1, 2016, 2), device=DEV)
    with torch.no_grad():
        plain = m(x, xpos=pos)
        seen = []
        m.proj.register_forward_hook(lambda mod, args, out: seen.append(args[0]))
        hooked = m(x, xpos=pos)
        assert len(seen) == 1 and (hooked - plain).abs().max() <= 4e-2 * plain.abs().max()   # the library's product on the merged branches
        m.gate[0].register_forward_hook(lambda mod, args, out: seen.append(args[0]))
        m(x, xpos=pos)
        assert len(seen) == 3


@pytest.mark.gpu
def test_one_call_replays_in_a_graph():
    m = _layer(16, 4, 32, torch.bfloat16)
    x = torch.randn((1, 2016, 1024), device=DEV).bfloat16()
    pos = torch.randint(0, 36, (1, 2016, 2), device=DEV)
    with torch.no_grad():
        m(x, xpos=pos, n_pos=36)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = m(x, xpos=pos, n_pos=36)
        for i in range(3):
            x.copy_(torch.randn(x.shape, device=DEV))
            want = m(x, xpos=pos, n_pos=36)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
