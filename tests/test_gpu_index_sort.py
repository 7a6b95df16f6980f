"""Index rows sorted by one workgroup each, against torch's sort (whole numbers: equal).  Sizes: one value, one
below / at / above a wavefront and the rows one instantiation takes, the longest row and one more (torch)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv,ns", [(1, 1), (63, 64), (65, 1023), (1024, 1025), (2048, 2049), (4097, 30), (700, 8193), (16384, 16383), (16385, 5)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_sorted_rows_equal_torchs(gpu, nv, ns, dtype):
    from minference_amd.ops import _sorted_indices
    g = torch.Generator(device=gpu).manual_seed(nv + ns)
    lowest, largest = -2 ** 31, 2 ** 31 - 1
    for lo, hi in ((0, 50), (0, 65536), (0, 131072), (-5, 300), (lowest, largest), (7, 8)):
        v = torch.randint(lo, hi, (2, 3, nv), generator=g, device=gpu, dtype=torch.int64).to(dtype)
        s = torch.randint(lo, hi, (2, 3, ns), generator=g, device=gpu, dtype=torch.int64).to(dtype)
        v[0, 0, -1], s[0, 0, 0] = hi, lo                # (the padding's own key among the values)
        s[1, 1, -1], v[1, 2, 0] = lo, lo
        vo, so = _sorted_indices(v, s, 2, 3)
        assert vo.dtype == so.dtype == torch.int32
        assert torch.equal(vo, v.to(torch.int32).sort(-1)[0]) and torch.equal(so, s.to(torch.int32).sort(-1, descending=True)[0]), (lo, hi)


def test_index_forms_of_the_operator(gpu):
    """Other integer types, expanded and strided index tensors, and values above 32 bits (truncated)."""
    from minference_amd.ops import _sorted_indices
    v = torch.randint(0, 200, (1, 1, 77), device=gpu)
    for t in (v.to(torch.int16), v.to(torch.uint8), v.to(torch.int32).expand(2, 4, 77), torch.stack([v, v], -1)[..., 0], v + 2 ** 40, v[0]):
        b, h = (2, 4) if t.shape[:2] == (2, 4) else (1, 1)
        vo, so = _sorted_indices(t, t, b, h)
        want = t.to(torch.int32).reshape(b, h, -1)
        assert torch.equal(vo, want.sort(-1)[0]) and torch.equal(so, want.sort(-1, descending=True)[0])


@pytest.mark.parametrize("n,nv,ns", [(64, 1, 1), (700, 128, 128), (700, 30, 129), (5000, 1024, 1025), (9000, 2049, 2048), (20001, 500, 8192), (20001, 500, 8193),
                                     (20001, 16384, 16384), (524160, 60, 300), (524224, 60, 300),       # (the bitmap shares LDS with the lists up to 524160)
                                     (524160, 16384, 16384), (524224, 300, 16384), (524160, 8193, 8192)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_index_of_unsorted_lists(gpu, n, nv, ns, dtype):
    """Sorting, tables and row blocks in one call against a call each; offsets beyond the context among them."""
    from minference_amd.index import _build
    from minference_amd.ops import _index_from_lists, _sorted_indices
    print(f"case {n} tokens, {nv} columns, {ns} slashes, {dtype}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(n + ns)
    v = torch.rand(2, 1, max(n, nv), generator=g, device=gpu).argsort(-1)[..., :nv].to(dtype)
    s = torch.rand(2, 1, max(n + 100, ns), generator=g, device=gpu).argsort(-1)[..., :ns].to(dtype)
    s[1, 0] = torch.arange(ns, device=gpu).flip(0).roll(ns // 3)
    s[:, :, ns // 2] = 0
    vs, ss = _sorted_indices(v, s, 2, 1)
    want, got = _build(None, vs, ss, n, zero_fill=False), _index_from_lists(v, s, 2, 1, n)
    for count, payload in ((0, 1), (2, 3)):
        assert torch.equal(got[count], want[count])
        there = torch.arange(want[payload].shape[-1], device=gpu) < want[count][..., None]
        assert torch.equal(got[payload][there], want[payload][there])
