"""Split walks (few row blocks, or a few walks far longer than the rest): segments of a walk on several
workgroups and the fold of their sums, against the fp32 masked-dense oracle.  Sizes: one step, exactly one
segment (8 steps), one step more, a ragged end, a lone row block in the last pair, rows past seqlen.
Tolerance: that of the tile engine (the fold adds fp32 roundings only)."""
import pytest
import torch

from oracle import oracle as O
from tests import gen
from tests.test_gpu_attention import check, expand, make, sdpa_causal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,dtype", [(128, torch.bfloat16), (64, torch.float16), (256, torch.bfloat16)])
@pytest.mark.parametrize("n,hq,hk,b", [(1, 1, 1, 1), (512, 2, 1, 1), (576, 1, 1, 2), (1300, 4, 2, 1)])
def test_split_walks_match_the_oracle(gpu, n, hq, hk, b, d, dtype):
    import minference_amd as M
    print(f"case split n={n} hq={hq} b={b} d={d} {dtype}", flush=True)
    q, k, v = make(b, hq, hk, n, n + d, dtype, d)
    qg, kg, vg, ke, ve = q.to(gpu), k.to(gpu), v.to(gpu), expand(k, hq), expand(v, hq)
    check(M.dense_causal_attention(qg, kg, vg), sdpa_causal(q, ke, ve), "dense")
    check(M.streaming_forward(qg, kg, vg, 70, 300), O.streaming_forward(q, ke, ve, 70, 300), "a-shape")
    if n > 1:
        check(M.tri_shape_forward(qg, kg, vg, 8, 130, 100), O.tri_shape_forward(q, ke, ve, 8, 130, 100), "tri-shape")
    if d <= 128:
        check(M.block_sparse_attention(qg, kg, vg, 1000), sdpa_causal(q, ke, ve), "block-sparse")
        v_idx, s_idx = M.estimate_vertical_slash(qg, kg, 40, 300)
        check(M.vertical_slash_sparse_attention(qg, kg, vg, v_idx, s_idx),
              O.vertical_slash_sparse_attention(q, ke, ve, v_idx.cpu(), s_idx.cpu()), "vertical-slash")


@pytest.mark.parametrize("n,hq", [(1300, 1), (1000, 40)])
@pytest.mark.parametrize("window", [129, 192, 193, 256, 320, 575, 640, 5000])
def test_short_stretches_of_unmasked_tiles_at_head_dim_64(gpu, n, hq, window):
    """Windows that leave a walk no, one, a few and more than eight tiles without a masked key, sinks beside them or
    before them, segments that begin and end among those tiles (one head) and whole walks (forty)."""
    import minference_amd as M
    q, k, v = make(1, hq, 1, n, window, torch.float16, 64)
    qg, kg, vg, one = q.to(gpu), k.to(gpu), v.to(gpu), (slice(None), slice(hq - 1, hq))
    for n_init in (0, 200):
        check(M.streaming_forward(qg, kg, vg, n_init, window)[one], O.streaming_forward(q[one], k, v, n_init, window), f"a-shape {n_init}")
        check(M.tri_shape_forward(qg, kg, vg, n_init, window, 150)[one], O.tri_shape_forward(q[one], k, v, n_init, window, 150), f"tri-shape {n_init}")
    check(M.dense_causal_attention(qg, kg, vg)[one], sdpa_causal(q[one], k, v), "dense")


@pytest.mark.parametrize("op,n,segments", [("ashape", 1024, 2), ("ashape", 2048, 4), ("ashape", 2100, 5), ("ashape", 4000, 8),
                                           ("ashape", 4200, 9), ("ashape", 8192, 16), ("dense", 16000, 6), ("tri", 9000, 18)])
def test_folds_of_every_number_of_segments(gpu, op, n, segments):
    """One head, walks of every earlier key (tri-shape: those of the last 128 rows): the fold takes the registers of four
    segments, holds the statistics of up to sixteen, adds eight at once.  Every such row against fp32."""
    import minference_amd as M
    from minference_amd import _lib
    q, k, v = (t.to(gpu) for t in make(1, 1, 1, n, n, torch.bfloat16))
    last = 128 if op == "tri" else 0
    sizes = {"ashape": (_lib.MINF_OP_ASHAPE, 0, n, 0), "dense": (_lib.MINF_OP_DENSE, 0, 0, 0), "tri": (_lib.MINF_OP_ASHAPE, 64, 128, last)}[op]
    nbytes = _lib.load().minf_attn_workspace_bytes(M.ops._Call(q, k, v).ref, *sizes)
    pairs = (n + 127) // 128 - ((n - last) // 128 if last else 0)
    assert nbytes == pairs * segments * (4 * 128 * 32 * 4 + 4 * 64 * 8)
    out = M.tri_shape_forward(q, k, v, 64, 128, last) if last else M.dense_causal_attention(q, k, v) if op == "dense" else \
        M.streaming_forward(q, k, v, 0, n)
    qf, kf, vf = (t[0, 0].float() for t in (q, k, v))
    for r0 in range(n - last if last else 0, n, 1000):
        rows = torch.arange(r0, min(r0 + 1000, n), device=gpu)
        p = (qf[rows] @ kf.T) * 128 ** -0.5
        p.masked_fill_(torch.arange(n, device=gpu)[None] > rows[:, None], float("-inf"))
        check(out[0, 0, rows], (torch.softmax(p, -1) @ vf).cpu(), f"{n} rows {r0}")


@pytest.mark.parametrize("n,hq,hk,b", [(2111, 12, 3, 1), (4033, 4, 4, 2)])
def test_half_full_launches_are_split_by_their_share(gpu, n, hq, hk, b):
    """More than 64 row-block pairs, too few to fill the chip: segments of 1.4 shares (lone last row block,
    ragged end), several heads and batches; the oracle on one head of each batch."""
    import minference_amd as M
    q, k, v = make(b, hq, hk, n, n, torch.bfloat16)
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    h = hq - 1
    one = (slice(None), slice(h, h + 1))
    qo, ko, vo = q[one], expand(k, hq)[one], expand(v, hq)[one]
    check(M.dense_causal_attention(qg, kg, vg)[one], sdpa_causal(qo, ko, vo), "dense")
    check(M.block_sparse_attention(qg, kg, vg, 1000)[one], sdpa_causal(qo, ko, vo), "block-sparse")
    check(M.streaming_forward(qg, kg, vg, 70, 4000)[one], O.streaming_forward(qo, ko, vo, 70, 4000), "a-shape")
    check(M.tri_shape_forward(qg, kg, vg, 8, 130, 300)[one], O.tri_shape_forward(qo, ko, vo, 8, 130, 300), "tri-shape")
    v_idx, s_idx = M.estimate_vertical_slash(qg, kg, 200, 500)
    check(M.vertical_slash_sparse_attention(qg, kg, vg, v_idx, s_idx)[one],
          O.vertical_slash_sparse_attention(qo, ko, vo, v_idx[one].cpu(), s_idx[one].cpu()), "vertical-slash")


def test_split_walks_with_short_sequences_and_many_leftovers(gpu):
    """seqlens below n in the middle of a pair, before one and in the first tile (rows past them are zero),
    with lists whose leftovers differ between the row blocks of a pair (scattered slashes)."""
    import minference_amd as M
    n, b = 1100, 3
    q, k, v = make(b, 1, 1, n, 5, torch.bfloat16)
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    vi, si = gen.vs_index_inputs(1, n, 60, 40, seed=9, batch=b)
    lens = torch.tensor([900, 1024, 10], dtype=torch.int32)
    idx = M.convert_vertical_slash_indexes(lens.to(gpu), torch.from_numpy(vi).to(gpu), torch.from_numpy(si.copy()).to(gpu), n)
    out = M.vertical_slash_attention_from_index(qg, kg, vg, *idx, lens.to(gpu))
    bc, bo, cc, ci = (x.cpu().numpy() for x in idx)
    for i in range(b):
        mask = O.vs_mask(bc[i, 0], bo[i, 0], cc[i, 0], ci[i, 0], n, int(lens[i]))
        check(out[i:i + 1, :1], O.masked_attention(q[i, 0], k[i, 0], v[i, 0], mask)[None, None], f"batch {i}")
        assert (out[i, 0, int(lens[i]):] == 0).all()


def test_split_segments_with_scores_past_the_fp32_range(gpu):
    """A segment whose sums overflow under its lazy maximum walks again; segments whose maxima lie
    hundreds of powers of two apart fold to the last one."""
    import minference_amd as M
    n = 2048
    q, k, v, _ = gen.planted_layer(n, 1, 1, seed=100, dtype=torch.bfloat16, decay_per_token=80 * 2.0 ** -7 / 128 ** 0.5)
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    check(M.dense_causal_attention(qg, kg, vg), sdpa_causal(q, k, v), "rising dense")
    assert (M.dense_causal_attention(qg, kg, torch.ones_like(vg)).float() - 1).abs().max().item() <= 2.0 ** -8


def test_which_launches_are_split():
    """The rule, on the host: short single heads and long dense walks are, full layers are not."""
    import ctypes
    from minference_amd import _lib
    lib = _lib.load()

    def nbytes(op, n, hq, *sizes, d=128):
        t = _lib.QKVO()
        t.batch, t.heads_q, t.heads_kv, t.n, t.head_dim = 1, hq, 1, n, d
        return lib.minf_attn_workspace_bytes(ctypes.byref(t), op, *(sizes or (0, 0, 0)))
    vs, ashape, dense = _lib.MINF_OP_VERTICAL_SLASH, _lib.MINF_OP_ASHAPE, _lib.MINF_OP_DENSE
    bs = _lib.MINF_OP_BLOCK_SPARSE
    # half a chip of long walks is split, a full one and one of short walks are not
    assert nbytes(vs, 8192, 4) > 0 and nbytes(bs, 6000, 8) > 0 and nbytes(ashape, 6000, 8, 128, 3968, 0) > 0
    assert nbytes(vs, 4096, 16) == 0 and nbytes(bs, 2000, 28) == 0 and nbytes(ashape, 6000, 8, 64, 1000, 0) == 0
    assert nbytes(dense, 16384, 4) > 0 and nbytes(dense, 6000, 16) == 0 and nbytes(dense, 12000, 16, d=64) == 0
    assert nbytes(dense, 2048, 32) == 0 and nbytes(vs, 400, 2) == 0
    # the dense rows of tri-shape: where they outlast the windows, in two segments at least
    assert nbytes(ashape, 8000, 32, 128, 3968, 100) > 0 and nbytes(ashape, 523, 32, 128, 3968, 100) == 0
    assert nbytes(vs, 4096, 1) > 0 and nbytes(vs, 8192, 1) > 0 and nbytes(vs, 8193, 1) == 0 and nbytes(vs, 4096, 32) == 0
    assert nbytes(dense, 16384, 1) > 0 and nbytes(dense, 6144, 64) == 0 and nbytes(dense, 64, 1) == 0
    assert nbytes(ashape, 24000, 16, 8, 512, 128, d=64) > 0 and nbytes(ashape, 24000, 16, 8, 512, 0, d=64) == 0


def test_short_lists_are_not_split():
    """The rule knows how wide the lists are: too few blocks for what a cut costs, or neighbouring slashes (two
    or three blocks), are walked whole where full lists are split; lists as wide as the rows as if not known."""
    import ctypes
    from minference_amd import _lib
    lib = _lib.load()

    def nbytes(op, n, hq, wide_v, wide):
        t = _lib.QKVO()
        t.batch, t.heads_q, t.heads_kv, t.n, t.head_dim = 1, hq, 1, n, 128
        return lib.minf_attn_workspace_bytes(ctypes.byref(t), op, wide_v, wide, 0)
    vs, bs = _lib.MINF_OP_VERTICAL_SLASH, _lib.MINF_OP_BLOCK_SPARSE
    for n, hq in ((1500, 1), (4000, 4), (8192, 1), (8192, 4)):
        assert nbytes(bs, n, hq, 0, 10) == 0 and nbytes(vs, n, hq, 30, 50) == 0
        assert nbytes(bs, n, hq, 0, (n + 63) // 64) == nbytes(bs, n, hq, 0, 0) > 0
        assert nbytes(vs, n, hq, 1000, 6096) == nbytes(vs, n, hq, 0, 0) > 0
    assert nbytes(bs, 6000, 4, 0, 20) == 0 < nbytes(bs, 6000, 1, 0, 20)
    assert nbytes(vs, 4096, 4, 3500, 100) > 0                # a few blocks, 55 column tiles


@pytest.mark.parametrize("n,hq,top_k,nv,ns", [(2111, 2, 17, 1000, 100), (4033, 1, 33, 600, 90)])
def test_split_walks_of_narrow_lists(gpu, n, hq, top_k, nv, ns):
    """Segments cut for the width of the list: block lists that end inside a segment's length, and scattered
    slashes whose walks are longer than the neighbouring ones that the cut assumes."""
    import minference_amd as M
    q, k, v = make(1, hq, hq, n, n, torch.bfloat16)
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    bi = M.ops._build_block_index(qg, kg, top_k)
    ref = torch.stack([O.masked_attention(q[0, h], k[0, h], v[0, h], O.bs_mask(bi[0, h].cpu().numpy(), n)) for h in range(hq)])
    check(M.block_sparse_attention(qg, kg, vg, top_k), ref[None], "block-sparse")
    vi, si = gen.vs_index_inputs(hq, n, nv, ns, seed=9)
    vi, si = torch.from_numpy(vi), torch.from_numpy(si.copy())
    check(M.vertical_slash_sparse_attention(qg, kg, vg, vi.to(gpu), si.to(gpu)),
          O.vertical_slash_sparse_attention(q, k, v, vi, si), "vertical-slash")


@pytest.mark.parametrize("hq,hk,n,b", [(3, 1, 900, 1), (6, 3, 700, 2), (10, 5, 13400, 1), (8, 8, 1500, 1), (4, 4, 6000, 2), (8, 8, 8192, 1)])
def test_deals_cover_every_row(gpu, hq, hk, n, b):
    """Head counts that do not divide among the eight XCDs, whose last round of deals is padded, and eight groups of one
    head, whose split walks change XCD every fourth round: with V = 1 every row of every head must come out as
    exactly 1 (ten heads, 105 pairs: list walks that are not split)."""
    import minference_amd as M
    q, k, _ = make(b, hq, hk, n, 3, torch.bfloat16)
    qg, kg = q.to(gpu), k.to(gpu)
    ones = torch.ones_like(kg)
    for out in (M.dense_causal_attention(qg, kg, ones), M.streaming_forward(qg, kg, ones, 64, 500),
                M.block_sparse_attention(qg, kg, ones, 20), M.vertical_slash_prefill(qg, kg, ones, 100, 300)):
        assert (out.float() - 1).abs().max().item() <= 2.0 ** -8


@pytest.mark.parametrize("hq,hk,n,b", [(20, 1, 8300, 1), (6, 3, 8300, 2), (3, 3, 8300, 1), (9, 9, 8500, 1), (1, 1, 66000, 1),
                                       (2, 1, 66000, 1), (8, 4, 8300, 6), (6, 3, 8300, 6)])
def test_heads_do_not_depend_on_how_a_launch_is_dealt(gpu, hq, hk, n, b):
    """Every head of a launch against the head on its own, bit for bit (lengths that are not split): more
    query heads than a deal has workgroups, batches, groups in two and three sets, deals of an eighth of the launch and
    of a few pairs, both sides of 512 and 1024 workgroups; the output is full of NaN before, so that no row can be left out."""
    import minference_amd as M
    q, k, v = (t.to(gpu) for t in make(b, hq, hk, n, 7, torch.bfloat16, 64))
    group = hq // hk
    bi = M.ops._build_block_index(q, k, 4)
    vi, si = M.estimate_vertical_slash(q, k, 40, 60)
    ix = M.index._build(None, vi, si, n, zero_fill=False)
    out = torch.empty_like(q)
    for name, f in (("a-shape", lambda q, k, v, i, o: M.streaming_forward(q, k, v, 64, 100, o)),
                    ("block-sparse", lambda q, k, v, i, o: M.ops.block_sparse_attention_from_index(q, k, v, bi[i].contiguous(), o)),
                    ("vertical-slash", lambda q, k, v, i, o: M.ops.vertical_slash_attention_from_index(
                        q, k, v, *(t[i].contiguous() for t in ix), out=o))):
        out.fill_(float("nan"))
        f(q, k, v, (slice(None), slice(None)), out)
        for bb in range(b):
            for h in range(hq):
                i = (slice(bb, bb + 1), slice(h, h + 1))
                j = (slice(bb, bb + 1), slice(h // group, h // group + 1))
                assert torch.equal(f(q[i], k[j], v[j], i, None), out[i]), (name, bb, h)


@pytest.mark.parametrize("hq,hk,n,b,far", [(32, 8, 48100, 1, 40), (32, 8, 49000, 1, 40), (32, 8, 49000, 1, 16), (32, 8, 49000, 1, 0), (66, 2, 26000, 1, 66),
                                           (16, 2, 98400, 1, 9), (24, 24, 66000, 1, 24), (16, 4, 30000, 7, 0)])
def test_long_launches_are_dealt_whole(gpu, hq, hk, n, b, far):
    """Launches just below and above 48 rounds of deals, from where on XCDs keep their place for some rounds if three of four
    heads keep more than an eighth of the blocks (the first `far` heads do), one set of groups and several: some heads
    on their own, bit for bit, and no row left out."""
    import minference_amd as M
    print(f"case {hq} / {hk} heads, {n} tokens, batch {b}, {far} far", flush=True)
    g = torch.Generator(device=gpu).manual_seed(n)
    q, k, v = (torch.randn(b, h, n, 64, generator=g, device=gpu, dtype=torch.bfloat16) for h in (hq, hk, hk))
    ns = n // 64 // 6
    vi = torch.arange(40, device=gpu, dtype=torch.int32).repeat(b, hq, 1) * 7
    si = torch.arange(ns, device=gpu, dtype=torch.int32).flip(0).repeat(b, hq, 1)
    si[:, :far] *= 256                                  # (blocks of their own, the others of one band)
    ix = M.index._build(None, vi, si.contiguous(), n, zero_fill=False)
    assert int((ix[0][0, :, -1] > (n + 63) // 64 // 8).sum()) == min(far, hq)
    out = torch.full_like(q, float("nan"))
    M.ops.vertical_slash_attention_from_index(q, k, v, *ix, out=out)
    assert torch.isfinite(out).all()
    for bb, h in ((0, 0), (0, hq // 2 + 1), (b - 1, 1), (b - 1, hq - 1)):
        i, j = (slice(bb, bb + 1), slice(h, h + 1)), (slice(bb, bb + 1), slice(h // (hq // hk), h // (hq // hk) + 1))
        one = M.ops.vertical_slash_attention_from_index(q[i], k[j], v[j], *(t[i].contiguous() for t in ix))
        assert torch.equal(one, out[i]), (bb, h)


@pytest.mark.parametrize("d,dtype", [(128, torch.bfloat16), (64, torch.float16)])
def test_a_nan_key_reaches_every_row_that_attends_to_it(gpu, d, dtype):
    """The row sum of a segment with a NaN score is NaN: the fold keeps it, as a whole walk's rows are NaN,
    and rows that do not attend to the key (other segments, masked entries of its tile) stay numbers."""
    import minference_amd as M
    n, at, window = 1300, 600, 300
    q, k, v = (t.to(gpu) for t in make(1, 1, 1, n, 17, dtype, d))
    clean, bad = M.dense_causal_attention(q, k, v), k.clone()
    bad[0, 0, at] = float("nan")
    out = M.dense_causal_attention(q, bad, v)
    assert torch.isnan(out[0, 0, at:]).all() and torch.isfinite(out[0, 0, :at]).all()
    check(out[:, :, :at], clean[:, :, :at].cpu(), "rows before the key")
    out = M.streaming_forward(q, bad, v, 64, window)
    assert torch.isnan(out[0, 0, at:at + window]).all()
    assert torch.isfinite(out[0, 0, :at]).all() and torch.isfinite(out[0, 0, at + window + 1:]).all()
