"""fp32 tensors narrowed on the device: the same bits as the caller's own conversion to the 16-bit format the rule
names (fp16 when the largest |value| of q, k and v lies in [2^-10, 32768], else bf16), for padded head dims,
strided and unaligned tensors and an output buffer; outputs compared with torch.equal (one kernel, one plan)."""
import pytest
import torch

from tests import gen

pytestmark = pytest.mark.gpu


def _inputs(dev, n, hq, hk, d, scale=1.0):
    q, k, v = gen.qkv(2, hq, hk, n, d, seed=n + d, dtype=torch.float32, scale=scale)
    return q.to(dev), k.to(dev), v.to(dev)


@pytest.mark.parametrize("n,hq,hk,d", [(1, 1, 1, 64), (65, 2, 1, 128), (700, 4, 2, 96), (130, 3, 3, 20), (517, 2, 2, 256), (300, 2, 1, 66)])
@pytest.mark.parametrize("amax,dtype", [(None, torch.float16), (32768.0, torch.float16), (32769.0, torch.bfloat16), (1e30, torch.bfloat16), ("tiny", torch.bfloat16)])
def test_same_bits_as_the_callers_conversion(gpu, n, hq, hk, d, amax, dtype):
    import minference_amd as M
    q, k, v = _inputs(gpu, n, hq, hk, d)
    if amax == "tiny":
        q, k, v = (t * 2.0 ** -14 / 4 for t in (q, k, v))
    elif amax is not None:
        v[1, hk - 1, n - 1, d - 1] = -amax
    got = M.dense_causal_attention(q, k, v)
    want = M.dense_causal_attention(q.to(dtype), k.to(dtype), v.to(dtype)).float()
    assert got.dtype == torch.float32 and got.shape == q.shape and torch.equal(got, want)
    got = M.streaming_forward(q, k, v, 16, 100)
    assert torch.equal(got, M.streaming_forward(q.to(dtype), k.to(dtype), v.to(dtype), 16, 100).float())


def test_strided_unaligned_and_caller_owned_tensors(gpu):
    import minference_amd as M
    q, k, v = _inputs(gpu, 400, 4, 2, 128)
    want = M.dense_causal_attention(q.half(), k.half(), v.half()).float()
    t = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v)]
    assert torch.equal(M.dense_causal_attention(*t), want)
    flat = torch.empty(q.numel() + 1, device=gpu)
    shifted = flat[1:].view(q.shape)
    shifted.copy_(q)
    assert torch.equal(M.dense_causal_attention(shifted, k, v), want)
    for out in (torch.empty_like(q), torch.empty_like(t[0]), torch.empty_like(q, dtype=torch.float16)):
        assert M.dense_causal_attention(q, k, v, out) is out and torch.equal(out.float(), want)
    assert torch.equal(M.dense_causal_attention(q, k[:, :1].expand(2, 2, 400, 128), v),
                       M.dense_causal_attention(q.half(), k[:, :1].expand(2, 2, 400, 128).half(), v.half()).float())


@pytest.mark.parametrize("n", [1024, 1025, 2048, 2049, 3071, 4096, 4097])
@pytest.mark.parametrize("layout", ["rows", "tokens first", "gaps", "one row for all heads"])
def test_the_largest_value_is_found_wherever_it_lies(gpu, n, layout):
    """2 heads of 128 around the 65536 vectors of 8 that all threads read in one step and the 131072 of two; tensors that fill
    one stretch of memory and ones that do not; the one value that asks for bf16 first, last and in between."""
    import minference_amd as M
    g = torch.Generator(device=gpu).manual_seed(n)
    q, k, x = (torch.randn(1, 2, n, 128, device=gpu, generator=g) for _ in range(3))
    if layout == "tokens first":
        v = x.transpose(1, 2).contiguous().transpose(1, 2)
    elif layout == "gaps":
        v = torch.full((1, 2, n, 132), 1e9, device=gpu)[..., :128]      # (what lies in the gaps must not count)
        v.copy_(x)
    elif layout == "rows":
        v = x
    else:
        v = x[:, :1].expand(1, 2, n, 128)
    f = lambda: M.streaming_forward(q, k, v, 16, 100)
    want = lambda dtype: M.streaming_forward(q.to(dtype), k.to(dtype), v.to(dtype), 16, 100).float()
    assert torch.equal(f(), want(torch.float16))
    last = 0 if layout.startswith("one") else 1
    for h, t, d in ((0, 0, 0), (last, n - 1, 127), (last, n // 2, 64)):
        old = float(v[0, h, t, d])
        v[0, h, t, d] = 40000.0
        assert torch.equal(f(), want(torch.bfloat16)), (h, t, d)
        v[0, h, t, d] = old


@pytest.mark.parametrize("where", ["nowhere", "one channel", "all of q", "from the middle of k on", "first rows", "last row", "one wavefront of many steps",
                                   "a tail", "tiny", "tiny middle head", "zero middle head", "large middle row"])
def test_the_rows_looked_at_first_do_not_decide(gpu, where):
    """Seventeen steps of a workgroup (sixteen whole ones and a tail), and the middle head's rows, by some of which the first conversion
    goes: values that ask for bf16 in all of them, in other rows, in them alone, in the vector that several threads write past
    the end; rows that ask for bf16 in tensors that do not."""
    import minference_amd as M
    n = 16 * 1024 + 3
    g = torch.Generator(device=gpu).manual_seed(3)
    q, k, v = (torch.randn(1, 8, n, 128, device=gpu, generator=g) for _ in range(3))
    dtype = torch.float16 if where == "nowhere" else torch.bfloat16
    if where == "one channel":
        k[..., 5] *= 1e5
    elif where == "all of q":
        q *= 1e6
    elif where == "from the middle of k on":
        k[:, 4:] *= 1e6
    elif where == "first rows":
        v[:, 0, :3] = 1e5
    elif where == "last row":
        v[0, 7, n - 1, 127] = -1e30
    elif where == "one wavefront of many steps":
        q[0, 3, 7, 8:16] = float("inf")
        q[0, 7, 16000, 3] = 5e4
    elif where == "a tail":
        q[0, 7, n - 3:] = 4e4
        v[0, 7, n - 1] = 0
    elif where == "tiny":
        q, k, v = q * 1e-6, k * 1e-6, v * 1e-6
    elif where == "large middle row":
        k[0, 4, n // 2, 127] = 1e9
    elif where.endswith("middle head"):
        dtype = torch.float16
        for t in (q, k, v):
            t[0, 4] *= 1e-7 if where.startswith("tiny") else 0
    want = M.streaming_forward(q.to(dtype), k.to(dtype), v.to(dtype), 16, 100).float()
    for _ in range(2):
        assert torch.equal(M.streaming_forward(q, k, v, 16, 100).nan_to_num(7.0), want.nan_to_num(7.0))


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_values_that_are_no_numbers_choose_bf16(gpu, bad):
    import minference_amd as M
    q, k, v = _inputs(gpu, 100, 1, 1, 64)
    v[0, 0, 99, 3] = bad
    got = M.dense_causal_attention(q, k, v)
    want = M.dense_causal_attention(q.bfloat16(), k.bfloat16(), v.bfloat16()).float()
    assert torch.equal(got[1], want[1]) and torch.equal(got[0, 0, :64], want[0, 0, :64])


def test_a_call_on_fp32_tensors_does_not_wait_for_the_gpu(gpu):
    """Recorded into a graph (a host read would end the capture) and replayed on inputs of the other format."""
    import minference_amd as M
    q, k, v = _inputs(gpu, 600, 4, 2, 128)
    vi = torch.arange(0, 40, device=gpu).expand(2, 4, 40).contiguous()
    si = torch.arange(0, 150, device=gpu).expand(2, 4, 150).contiguous()
    f = lambda: M.vertical_slash_sparse_attention(q, k, v, vi, si)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        f()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = f()
    for scale in (1.0, 1e6, 1.0, 3.0):
        v.mul_(scale)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, f()), scale
