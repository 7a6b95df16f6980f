"""The ``out`` buffer of the operators: written in place where it stands apart from the operands, computed
beside them and copied where it shares their memory -- the bits of a call without ``out`` either way."""
import pytest
import torch

from tests import gen

OPS = {
    "dense": lambda M, q, k, v, out: M.dense_causal_attention(q, k, v, out),
    "a-shape": lambda M, q, k, v, out: M.ops.streaming_forward(q, k, v, 70, 500, out),
    "block-sparse": lambda M, q, k, v, out: M.block_sparse_attention(q, k, v, 9, out=out),
    "vertical-slash": lambda M, q, k, v, out: M.vertical_slash_prefill(q, k, v, 60, 300, out),
    "mixed": lambda M, q, k, v, out: M.minference_prefill_forward(q, k, v, {"layer_idx": 0, "out": out, "attn_forward_config": {
        "best_pattern": [{"0": ["vertical_and_slash", 60, 300, 1.0], "1": ["block_sparse", 100, 0, 1.0]}]}}),
}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("op", sorted(OPS))
def test_out_may_share_memory_with_the_operands(gpu, op, dtype):
    """q, k, v, one of them shifted by a row, and the fourth part of a [B, N, 4 H, D] projection as ``out``.  The
    scores rise past the fp32 range, so that bf16 walks are made twice."""
    import minference_amd as M
    n, H = 1500, 2
    q, k, v, _ = gen.planted_layer(n, H, H, seed=3, dtype=torch.bfloat16, decay_per_token=0.3)
    q, k, v = (t.to(dtype).to(gpu) for t in (q, k, v))
    want = OPS[op](M, q, k, v, None)
    separate = torch.empty_like(q)
    assert OPS[op](M, q, k, v, separate) is separate and torch.equal(separate, want)
    for i in range(3):
        x = [t.clone() for t in (q, k, v)]
        assert OPS[op](M, *x, x[i]) is x[i] and torch.equal(x[i], want), "qkv"[i]
        store = torch.empty(1, H, n + 1, 128, dtype=dtype, device=gpu)
        x = [t.clone() for t in (q, k, v)]
        store[:, :, 1:] = x[i]
        x[i] = store[:, :, 1:]
        assert torch.equal(OPS[op](M, *x, store[:, :, :n]), want), "qkv"[i]
    packed = torch.empty(1, n, 4 * H, 128, dtype=dtype, device=gpu).transpose(1, 2)
    parts = [packed[:, i * H:(i + 1) * H] for i in range(4)]
    for p, t in zip(parts, (q, k, v)):
        p.copy_(t)
    assert torch.equal(OPS[op](M, *parts), want)


def test_which_views_share_memory():
    from minference_amd.ops import _overlap
    x = torch.empty(2, 3, 10, 8)
    assert _overlap(x, x) and _overlap(x, x[1:, 2:, 9:, 7:]) and not _overlap(x[:1], x[1:]) and not _overlap(x[0, :, :4], x[1])
    assert _overlap(x[..., :4], x[..., 4:]) and not _overlap(x, torch.empty_like(x)) and not _overlap(x[:, :0], x)
    assert _overlap(x.transpose(1, 2)[:, 5:], x[0, 0, 9:]) and _overlap(x[:1, :1, :1].expand(2, 3, 10, 8), x[0, 0, 0])


@pytest.mark.gpu
@pytest.mark.parametrize("op", sorted(OPS))
def test_out_need_not_be_aligned(gpu, op):
    """A contiguous ``out`` that starts an element past a 16-byte boundary, and one whose rows are not whole
    16-byte vectors apart, take the bits of a call without."""
    import minference_amd as M
    n, H, d = 700, 2, 128
    q, k, v = (t.bfloat16().to(gpu) for t in gen.qkv(1, H, H, n, d, seed=4, scale=1.0))
    want = OPS[op](M, q, k, v, None)
    shifted = torch.zeros(q.numel() + 8, dtype=q.dtype, device=gpu)[1:1 + q.numel()].view(q.shape)
    padded = torch.zeros(1, H, n, d + 3, dtype=q.dtype, device=gpu)[..., :d]
    for out in (shifted, padded):
        assert OPS[op](M, q, k, v, out) is out and torch.equal(out, want)
