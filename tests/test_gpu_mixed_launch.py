"""The pattern types of a layer in one attention launch against a launch for each: the same walks, so the same bits."""
import ctypes

import pytest
import torch

from tests import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("present", ["vba", "vb", "va", "ba", "v", "a"])
@pytest.mark.parametrize("n,d,dtype", [(9001, 128, torch.bfloat16), (8300, 64, torch.float16), (8257, 64, torch.bfloat16), (8448, 128, torch.float16), (1500, 128, torch.bfloat16)])
def test_same_bits_as_a_launch_per_type(gpu, n, d, dtype, present):
    """8 / 2 heads; the last size is split (and launched one after another)."""
    import minference_amd as M
    from minference_amd import _lib
    from minference_amd.ops import _Call
    print(f"case {n} tokens, head_dim {d}, {dtype}, parts {present}", flush=True)
    q, k, v = (t.to(gpu, dtype) for t in gen.qkv(1, 8, 2, n, d, seed=n, dtype=torch.float32, scale=1.0))
    heads = {"v": [0, 2, 3, 7], "b": [1, 6], "a": [4, 5]}
    slots = {x: torch.tensor(h, dtype=torch.int32, device=gpu) for x, h in heads.items()}
    group = lambda t, x: t[:, [h // 4 for h in heads[x]]].contiguous()
    rows, lib, keep = (n + 63) // 64, _lib.load(), []
    v_idx, s_idx = M.estimate_vertical_slash(q[:, heads["v"]].contiguous(), group(k, "v"), 100, 500)
    lens = torch.full((1,), n, dtype=torch.int32, device=gpu)
    index = M.convert_vertical_slash_indexes(lens, v_idx, s_idx, n, zero_fill=False)
    blocks = torch.sort(torch.rand(1, 2, rows, rows, device=gpu).argsort(-1)[..., :20].int(), dim=-1)[0].contiguous()
    blocks = torch.minimum(blocks, torch.arange(rows, device=gpu, dtype=torch.int32).view(1, 1, rows, 1)).contiguous()

    def run(one):
        c = _Call(q, k, v, out=torch.full_like(q, 7.0))
        assert c.o is c.out

        def part(x, op, a, b):
            if x not in present:
                return None
            c.select_heads(slots[x])
            c.scratch(op, a, b)
            keep.append(c._scratch)
            return _lib.QKVO.from_buffer_copy(c.struct)
        vs = part("v", _lib.MINF_OP_VERTICAL_SLASH, 100, 500)
        bs = part("b", _lib.MINF_OP_BLOCK_SPARSE, 0, 20)
        a = part("a", _lib.MINF_OP_ASHAPE, 64, 1000)
        ref = lambda s: None if s is None else ctypes.byref(s)
        st = _lib.stream_ptr(gpu)
        lists = [t.data_ptr() for t in index]
        if one:
            _lib.check(lib.minf_mixed_attn_fwd(ref(vs), *lists, rows, 500, 100, ref(bs), blocks.data_ptr(), rows, 20, ref(a), 64, 1000, st), "mixed")
        else:
            if vs is not None:
                _lib.check(lib.minf_vs_attn_fwd(ref(vs), *lists, rows, 500, 100, st), "vs")
            if bs is not None:
                _lib.check(lib.minf_bs_attn_fwd(ref(bs), blocks.data_ptr(), rows, 20, st), "bs")
            if a is not None:
                _lib.check(lib.minf_ashape_attn_fwd(ref(a), 64, 1000, st), "ashape")
        torch.cuda.synchronize()
        return c.o
    want, got = run(False), run(True)
    assert torch.equal(got, want)
    untouched = [h for x, hs in heads.items() if x not in present for h in hs]
    assert bool((got[:, untouched] == 7.0).all())
