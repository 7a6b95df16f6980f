"""The vertical-slash layer in one call against its four stages called one by one.  From 257 to 16384 tokens (up to 4096,
512 heads) the layer's selections read the estimation's sums directly, in one kernel that makes the index builder's tables
behind them; elsewhere the kernels are the stages' own.  The sums are added in the same order and ties go to the lower
index in both, so the bits are the same."""
import pytest
import torch

from tests import gen

pytestmark = pytest.mark.gpu


def stages(q, k, v, nv, ns):
    import minference_amd as M
    n = q.shape[2]
    v_idx, s_idx = M.estimate_vertical_slash(q, k, nv, ns)
    seqlens = torch.full((q.shape[0],), n, dtype=torch.int32, device=q.device)
    index = M.convert_vertical_slash_indexes(seqlens, v_idx, s_idx, n, zero_fill=False)
    return M.vertical_slash_attention_from_index(q, k, v, *index)


@pytest.mark.parametrize("batch,hq,hk,n,d,dtype,nv,ns", [
    (1, 1, 1, 1, 128, torch.bfloat16, 1000, 6096), (1, 1, 1, 33, 64, torch.float16, 30, 800), (2, 4, 2, 65, 128, torch.bfloat16, 1, 1),
    (1, 4, 4, 700, 96, torch.bfloat16, 100, 750), (2, 2, 1, 2049, 64, torch.bfloat16, 500, 700), (1, 1, 1, 4097, 128, torch.float16, 500, 700),
    (1, 2, 1, 256, 128, torch.bfloat16, 100, 200), (1, 2, 1, 257, 128, torch.bfloat16, 257, 257), (1, 3, 3, 4096, 128, torch.bfloat16, 4096, 4096),
    (1, 2, 2, 8192, 64, torch.bfloat16, 3500, 100), (1, 2, 2, 8193, 128, torch.bfloat16, 1000, 6096), (2, 260, 4, 300, 64, torch.bfloat16, 30, 60),
    (1, 257, 1, 600, 64, torch.float16, 30, 128), (1, 256, 1, 4097, 64, torch.bfloat16, 30, 129), (1, 1, 1, 16384, 64, torch.bfloat16, 30, 16384),
    (1, 8, 2, 16384, 128, torch.bfloat16, 1000, 6096), (1, 4, 1, 16385, 128, torch.bfloat16, 3500, 100)])
def test_same_bits_as_the_stages(gpu, batch, hq, hk, n, d, dtype, nv, ns):
    import minference_amd as M
    print(f"case {batch} x {hq} / {hk} heads, {n} tokens, head_dim {d}, {dtype}, {nv} / {ns}", flush=True)
    q, k, v = (t.to(gpu, dtype) for t in gen.qkv(batch, hq, hk, n, d, seed=n, dtype=torch.float32, scale=1.0))
    want = stages(q, k, v, nv, ns)
    assert torch.equal(M.vertical_slash_prefill(q, k, v, nv, ns), want)
    t = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v)]
    out = torch.empty_like(t[0])
    assert M.vertical_slash_prefill(*t, nv, ns, out) is out and torch.equal(out, want)


def test_replays_from_a_graph(gpu):
    import minference_amd as M
    q, k, v = (t.to(gpu, torch.bfloat16) for t in gen.qkv(1, 2, 1, 3000, 128, seed=5, dtype=torch.float32, scale=1.0))
    f = lambda: M.vertical_slash_prefill(q, k, v, 100, 300)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        f()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = f()
    for _ in range(3):
        k.copy_(torch.randn_like(k.float()))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, f())
