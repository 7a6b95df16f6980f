"""GPU parity of the offline pattern search (flag builders + minf_pattern_recall through the
C ABI) against the oracle's N x N restatement.  Tolerance: the scores are means of softmax
masses in [0, 1]; both sides compute in fp32 on identical 16-bit inputs, so they agree to 2e-3
absolute (the slack covers a top-k boundary element whose two fp32 estimates differ in the last
bits and fall on either side of the threshold)."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import gen

pytestmark = pytest.mark.gpu

TOL = 2e-3


def heads(n, hq, hk, seed, dtype=torch.bfloat16, planted=True):
    q, k, _ = gen.qkv(1, hq, hk, n, 128, seed, dtype=torch.float32, scale=1.0)
    if planted:          # a sink, a few heavy columns and some local structure, so that candidates differ
        g = torch.Generator().manual_seed(seed + 1)
        u = torch.randn(hk, 128, generator=g)
        u = u / u.norm(dim=-1, keepdim=True)
        q = q + 4.0 * u.repeat_interleave(hq // hk, 0)[None, :, None, :]
        k[:, :, :4] += 8.0 * u[None, :, None, :]
        cols = torch.randperm(n, generator=g)[:n // 50]
        k[:, :, cols] += 5.6 * u[None, :, None, :]
        z = torch.randn(n + 255, 128, generator=g)
        z = torch.nn.functional.avg_pool1d(z.T[None], 256, 1)[0].T * 16.0     # smooth over 256 tokens
        q = q + 0.5 * z[None, None]
        k = k + 0.5 * z[None, None]
    return q.to(dtype), k.to(dtype)


SMALL = [("stream_llm", 10, 80), ("vertical_and_slash", 30, 80), ("vertical_and_slash", 50, 75),
         ("vertical_and_slash", 100, 40), ("block_sparse", 8, 1)]


def oracle_scores(q, k, cands, begin):
    hq, hk = q.shape[1], k.shape[1]
    return [O.search_pattern_scores(q[0, h].float(), k[0, h // (hq // hk)].float(), cands, begin) for h in range(hq)]


@pytest.mark.parametrize("n,hq,hk,begin,dtype,cands", [
    (3000, 2, 1, 2500, torch.bfloat16, None), (4100, 1, 1, 2500, torch.bfloat16, None),
    (1111, 4, 2, 300, torch.float16, SMALL), (640, 1, 1, 0, torch.bfloat16, SMALL),
    (97, 2, 2, 10, torch.bfloat16, SMALL[:3] + [("block_sparse", 2, 1)]),
])
def test_candidates_vs_oracle(gpu, n, hq, hk, begin, dtype, cands):
    from minference_amd import pattern_recall
    from minference_amd.search import CANDIDATES
    cands = list(CANDIDATES) if cands is None else cands     # None: the reference's own list
    print(f"case search n={n} hq={hq} hk={hk} begin={begin} {dtype}", flush=True)
    q, k = heads(n, hq, hk, 40 + n, dtype)
    got = pattern_recall(q.to(gpu), k.to(gpu), cands, begin)[0].cpu().numpy()
    want = np.array(oracle_scores(q, k, cands, begin))
    print(np.round(got, 4), np.round(want, 4), flush=True)
    assert got.shape == want.shape
    assert np.abs(got - want).max() <= TOL
    if n >= 600:
        assert want.min() < 0.9 and want.max() - want.min() > 0.1     # the case separates candidates


def test_eight_candidates_of_every_kind_and_their_bits_do_not_mix(gpu):
    from minference_amd import pattern_recall
    n, begin = 1500, 200
    q, k = heads(n, 2, 1, 77)
    cands = [("stream_llm", 4, 64), ("block_sparse", 4, 1), ("vertical_and_slash", 40, 60), ("stream_llm", 0, 0),
             ("block_sparse", 1, 1), ("vertical_and_slash", 1500, 30), ("stream_llm", 1, 1500), ("block_sparse", 16, 1)]
    got = pattern_recall(q.to(gpu), k.to(gpu), cands, begin)[0].cpu().numpy()
    want = np.array(oracle_scores(q, k, cands, begin))
    print(np.round(got, 4), np.round(want, 4), flush=True)
    assert np.abs(got - want).max() <= TOL
    # candidates that keep everything are exactly 1 up to fp32 rounding, in any bit position
    assert np.abs(got[:, [4, 5, 6]] - 1.0).max() < 1e-5
    # each candidate alone (in bit 0) gives the same number as in its bit of the group of eight,
    # up to the last bits (the compiler may fuse the multiply-adds of different bits differently)
    for i in (0, 1, 2, 7):
        alone = pattern_recall(q.to(gpu), k.to(gpu), [cands[i]], begin)[0, :, 0].cpu().numpy()
        assert np.abs(alone - got[:, i]).max() < 1e-6


def test_uniform_attention_closed_form(gpu):
    # q = 0: row r keeps (#kept columns)/(r+1)
    from minference_amd import pattern_recall
    n, v, s, begin = 700, 5, 33, 100
    q = torch.zeros(1, 1, n, 128, dtype=torch.bfloat16)
    k = heads(n, 1, 1, 5, planted=False)[1]
    want = np.mean([(min(r, s) + 1 + max(0, min(v, r - s))) / (r + 1) for r in range(begin, n)])
    got = pattern_recall(q.to(gpu), k.to(gpu), [("stream_llm", v, s)], begin)[0, 0, 0].item()
    assert abs(got - want) < 1e-5


def test_search_pattern_choice_and_table(gpu):
    from minference_amd import search_pattern, search_patterns
    n = 4200
    q, k = heads(n, 4, 2, 91)
    table = search_patterns(q.to(gpu), k.to(gpu))
    assert sorted(table) == ["0", "1", "2", "3"]
    for h in range(4):
        want = O.search_pattern(q[0, h].float(), k[0, h // 2].float())
        got = table[str(h)]
        assert tuple(got[:3]) == want[:3], (h, got, want)
        assert abs(got[3] - want[3]) <= TOL
        assert got[0] == "vertical_and_slash"
    one = search_pattern(q[:, 1:2].to(gpu), k[:, 0:1].to(gpu), 1)
    assert list(one) == table["1"]
    # a block_sparse winner is replaced by vertical_and_slash (1000, 6096), as in the reference
    cands = [("stream_llm", 4, 16), ("block_sparse", 2, 1)]
    want = O.search_pattern(q[0, 0].float(), k[0, 0].float(), cands)
    got = search_pattern(q[:, 0:1].to(gpu), k[:, 0:1].to(gpu), 0, cands)
    assert want[:3] == ("vertical_and_slash", 1000, 6096) and got[:3] == want[:3] and abs(got[3] - want[3]) <= TOL


def test_too_short_context_gives_nan_and_no_choice(gpu):
    from minference_amd import search_pattern
    q, k = heads(512, 1, 1, 3)
    ty, v, s, sc = search_pattern(q.to(gpu), k.to(gpu), 0)       # 512 <= 2500: mean of nothing
    assert ty == "" and sc == 0.0


def test_deterministic(gpu):
    from minference_amd import pattern_recall
    q, k = heads(2000, 2, 1, 8)
    a = pattern_recall(q.to(gpu), k.to(gpu), row_begin=500)
    b = pattern_recall(q.to(gpu), k.to(gpu), row_begin=500)
    assert torch.equal(a, b)


def test_search_mode_of_the_dispatcher_writes_the_pattern_file(gpu, tmp_path):
    """minference_forward.py:644-673: with is_search every layer's heads are searched, the result
    is appended to config_path, the layer's output is dense causal attention; the finished file
    drives the sparse dispatcher."""
    import json
    from minference_amd import dense_causal_attention, minference_prefill_forward
    n = 2900
    q, k = heads(n, 4, 2, 17)
    v = torch.randn(1, 2, n, 128, generator=torch.Generator().manual_seed(3)).bfloat16()
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    path = tmp_path / "best_pattern.json"
    cfg = {"is_search": True, "config_path": str(path)}
    dense = dense_causal_attention(qg, kg, vg)
    for layer in range(2):
        out = minference_prefill_forward(qg, kg, vg, {"layer_idx": layer, "num_hidden_layers": 2, "attn_forward_config": cfg})
        assert torch.equal(out, dense)
    table = json.loads(path.read_text())
    assert len(table) == 2 and sorted(table[0]) == ["0", "1", "2", "3"]
    for h in range(4):
        want = O.search_pattern(q[0, h].float(), k[0, h // 2].float())
        assert tuple(table[1][str(h)][:3]) == want[:3]
    with pytest.raises(RuntimeError, match="Search already completed"):
        minference_prefill_forward(qg, kg, vg, {"layer_idx": 0, "num_hidden_layers": 2, "attn_forward_config": cfg})
    sparse = minference_prefill_forward(qg, kg, vg, {"layer_idx": 1, "attn_forward_config": {"best_pattern": table}})
    assert sparse.shape == dense.shape and torch.isfinite(sparse.float()).all()


@pytest.mark.parametrize("n,hq,hk,begin", [(33, 1, 1, 0), (128, 3, 1, 0), (129, 2, 2, 128), (1000, 2, 1, 64), (700, 2, 1, 690)])
@pytest.mark.parametrize("d", [128, 64])
def test_recall_tiles_stripes_and_flag_mixes(gpu, n, hq, hk, begin, d):
    """Edges of the 128-row workgroups, counted rows that start inside a tile, head counts that do not divide
    among the XCDs, head_dim 64 (padded), and candidates that share bits in one flag byte: windows that fill
    whole blocks, single diagonals, every second column, all eight candidates in use.  Flags are set through
    the public candidate list; the oracle multiplies N x N masks."""
    from minference_amd import pattern_recall
    q, k, _ = gen.qkv(1, hq, hk, n, d, 7 + n, dtype=torch.float32, scale=1.0)
    q, k = q.bfloat16(), k.bfloat16()
    cands = [("stream_llm", 4, 70), ("stream_llm", n // 2, 3), ("vertical_and_slash", 40, 60), ("vertical_and_slash", 31, 100),
             ("vertical_and_slash", 200, 51), ("block_sparse", 2, 1), ("block_sparse", 3, 1), ("stream_llm", 1, n)]
    got = pattern_recall(q.to(gpu), k.to(gpu), cands, begin)[0].cpu().numpy()
    want = np.array(oracle_scores(q, k, cands, begin))
    assert np.abs(got - want).max() <= TOL, (got, want)
    assert np.abs(got[:, 7] - 1.0).max() <= 1e-6             # a window of all offsets keeps everything


@pytest.mark.parametrize("n,hq,hk", [(1500, 3, 1), (97, 2, 2), (4100, 1, 1)])
def test_long_searches_set_the_same_flags(gpu, monkeypatch, n, hq, hk):
    """Contexts beyond the kernels that write flag bytes at once (32768 tokens; 4096 block rows) set them candidate by
    candidate in zeroed arrays: the same recall with those limits at zero, two block-sparse candidates (the first one
    clears) and all kinds among them."""
    from minference_amd import _lib, pattern_recall
    q, k = (t.to(gpu) for t in heads(n, hq, hk, 5 + n))
    cands = [("vertical_and_slash", 40, 60), ("block_sparse", 4, 1), ("stream_llm", 4, 64), ("block_sparse", 16, 1), ("stream_llm", 0, 0),
             ("vertical_and_slash", n, 30), ("stream_llm", n + 5, 3), ("block_sparse", 2, 1)]
    cands = [c for c in cands if c[0] != "block_sparse" or c[1] <= (n + 31) // 32]
    for chosen in (cands, cands[1:2], cands[2:3]):
        monkeypatch.setattr(_lib, "MINF_SEARCH_FLAGS_MAX", 32768)
        monkeypatch.setattr(_lib, "MINF_SEARCH_BLOCK_FLAGS_MAX", 4096)
        want = pattern_recall(q, k, chosen, 10)
        for name in ("MINF_SEARCH_FLAGS_MAX", "MINF_SEARCH_BLOCK_FLAGS_MAX"):
            monkeypatch.setattr(_lib, name, 0)
            assert torch.equal(pattern_recall(q, k, chosen, 10), want), name


@pytest.mark.parametrize("n", [32768, 32769])
def test_recall_on_both_sides_of_the_flag_kernels_limit(gpu, n):
    """The last 70 rows of one head against fp64 sums over flags made of the same scores with torch.  Both sums of a row are
    fp32 sums of about n / 64 block sums, each with a rounding of at most 2^-24."""
    from minference_amd import pattern_recall, vertical_slash_scores
    g = torch.Generator(device=gpu).manual_seed(n)
    q, k = (torch.randn(1, 1, n, 128, device=gpu, generator=g).bfloat16() for _ in range(2))
    begin = n - 70
    cands = [("vertical_and_slash", 100, 300), ("stream_llm", 9, 1000), ("vertical_and_slash", 1000, 30), ("vertical_and_slash", 31, 6096)]
    got = pattern_recall(q, k, cands, begin)[0, 0]
    vertical, slash = (x[0, 0] for x in vertical_slash_scores(q, k, 64, 30, 30, reference_rounding=False))
    r, c = torch.arange(begin, n, device=gpu)[:, None], torch.arange(n, device=gpu)[None]
    s = q[0, 0, begin:].double() @ k[0, 0].double().t().contiguous() * 128 ** -0.5
    p = torch.softmax(s.masked_fill(c > r, float("-inf")), -1)
    for t, (kind, a, b) in enumerate(cands):
        col, diag = (torch.zeros(n, dtype=torch.bool, device=gpu) for _ in range(2))
        if kind == "stream_llm":
            col[:a], diag[:b + 1] = True, True
        else:
            col[torch.topk(vertical, a).indices], diag[n - 1 - torch.topk(slash, b).indices] = True, True
        want = float((p * (col[None] | diag[(r - c).clamp(min=0)])).sum() / (n - begin))
        assert abs(float(got[t]) - want) <= 2 * (n / 64 + 64) * 2.0 ** -24 * want, (t, float(got[t]), want)


@pytest.mark.parametrize("n,dtype", [(1500, torch.bfloat16), (3001, torch.float16)])
def test_recall_keeps_fp32_accuracy(gpu, n, dtype):
    """Against fp64 sums on the same operands, all candidates with the largest keys: exponentials of 24 bits, fp32 row sums whose roundings average
    out over the rows, one rounding of the result (2^-24): 2^-23 in all."""
    import minference_amd as M
    g = torch.Generator(device=gpu).manual_seed(n)
    q, k = ((2 * torch.randn(1, 2, n, 128, device=gpu, generator=g)).to(dtype) for _ in range(2))
    cands = [("stream_llm", 1, 5), ("stream_llm", 40, 77), ("stream_llm", 3, 300), ("stream_llm", 300, 10)]
    got = M.pattern_recall(q, k, cands, row_begin=0)[0].double()
    r, c = torch.arange(n, device=gpu)[:, None], torch.arange(n, device=gpu)[None]
    for h in range(2):
        s = q[0, h].double() @ k[0, h].double().t().contiguous() * 128 ** -0.5
        p = torch.softmax(s.masked_fill(c > r, float("-inf")), -1)
        for t, (_, v, w) in enumerate(cands):
            want = (p * ((c < v) | (r - c <= w))).sum() / n
            assert abs(got[h, t] - want) <= 2.0 ** -23 * want, (h, t)


def _recall_of(q, k_ptr, k_strides, hk, n, cands, sm_scale=128.0 ** -0.5, flags=None):
    """minf_pattern_recall through the C ABI: K by pointer and strides, stream_llm candidates or (col, diag) flags."""
    from minference_amd import _lib
    lib, dev, hq = _lib.load(), q.device, q.shape[1]
    pitch, i64x3, stream = (n + 63) // 64 * 64, _lib.c_i64 * 3, _lib.stream_ptr(q.device)
    col, diag = (torch.zeros(hq, pitch, dtype=torch.uint8, device=dev) for _ in range(2))
    for bit, (_, v, s) in enumerate(cands):
        col[:, :v] |= 1 << bit
        diag[:, :s + 1] |= 1 << bit
    col, diag = (col, diag) if flags is None else flags
    recall = torch.empty(hq, 8, dtype=torch.float32, device=dev)
    nbytes = lib.minf_pattern_recall_workspace_bytes(1, hq, n)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    _lib.check(lib.minf_pattern_recall(q.data_ptr(), k_ptr, i64x3(*q.stride()[:3]), i64x3(*k_strides), 1, hq, hk, n, 128,
                                       _lib.MINF_BF16, sm_scale, col.data_ptr(), diag.data_ptr(), pitch, None, 0, 0,
                                       recall.data_ptr(), ws.data_ptr(), nbytes, stream), "minf_pattern_recall")
    return recall[:, :len(cands)] if flags is None else recall


@pytest.mark.parametrize("n", [131072, 131073, 131199, 262144 + 33])
def test_recall_where_the_table_of_diagonals_grows_and_ends(gpu, n):
    """The two table sizes (131072 and 262144 tokens) and distances past the table, for the last rows: random columns and
    diagonals, windows that end inside a block, a candidate without columns, one with all.  Both sums of a row are fp32
    sums of about n / 64 block sums, each with a rounding of at most 2^-24."""
    g = torch.Generator(device=gpu).manual_seed(n)
    q = torch.randn(1, 1, n, 128, device=gpu, generator=g).bfloat16()
    k = torch.randn(1, 1, n, 128, device=gpu, generator=g).bfloat16()
    begin, pitch = n - 70, (n + 63) // 64 * 64
    col = torch.randint(0, 256, (1, pitch), device=gpu, generator=g, dtype=torch.uint8) & 0x5d
    col |= 0x80
    diag = torch.randint(0, 256, (1, pitch), device=gpu, generator=g, dtype=torch.uint8) & 0x16
    diag[:, :1000] |= 0x08
    diag[:, 999:n // 2 + 5] |= 0x20
    got = _recall_begin(q, k, col, diag, begin)
    r, c = torch.arange(begin, n, device=gpu)[:, None], torch.arange(n, device=gpu)[None]
    s = q[0, 0, begin:].double() @ k[0, 0].double().t().contiguous() * 128 ** -0.5
    p = torch.softmax(s.masked_fill(c > r, float("-inf")), -1)
    flags = col[0, :n][None] | diag[0][(r - c).clamp(min=0)]
    for t in range(8):
        want = float((p * ((flags >> t) & 1)).sum() / (n - begin))
        assert abs(float(got[0, t]) - want) <= 2 * (n / 64 + 64) * 2.0 ** -24 * want, t


@pytest.mark.parametrize("n", [33, 127, 130, 260, 515])
def test_diagonals_of_every_row_and_byte(gpu, n):
    """Random flags of all eight candidates on every diagonal, all rows counted: a lane's flags begin at each byte of a
    word, at the first and the last one of a step.  Both sums of a row are fp32 sums of at most 64 + n / 64 terms in a chain."""
    g = torch.Generator(device=gpu).manual_seed(n)
    q, k = (torch.randn(1, 1, n, 128, device=gpu, generator=g).bfloat16() for _ in range(2))
    pitch = (n + 63) // 64 * 64
    col, diag = (torch.randint(0, 256, (1, pitch), device=gpu, generator=g, dtype=torch.uint8) for _ in range(2))
    got = _recall_begin(q, k, col & 0x0f & torch.roll(col, 7), diag, 0)
    r, c = torch.arange(n, device=gpu)[:, None], torch.arange(n, device=gpu)[None]
    s = q[0, 0].double() @ k[0, 0].double().t().contiguous() * 128 ** -0.5
    p = torch.softmax(s.masked_fill(c > r, float("-inf")), -1)
    flags = (col & 0x0f & torch.roll(col, 7))[0, :n][None] | diag[0][(r - c).clamp(min=0)]
    for t in range(8):
        want = float((p * ((flags >> t) & 1)).sum() / n)
        assert abs(float(got[0, t]) - want) <= 2 * (n / 64 + 64) * 2.0 ** -24 * want, t


def _recall_begin(q, k, col, diag, begin):
    from minference_amd import _lib
    lib, n, i64x3 = _lib.load(), q.shape[2], _lib.c_i64 * 3
    recall = torch.empty(1, 8, dtype=torch.float32, device=q.device)
    nbytes = lib.minf_pattern_recall_workspace_bytes(1, 1, n)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=q.device)
    _lib.check(lib.minf_pattern_recall(q.data_ptr(), k.data_ptr(), i64x3(*q.stride()[:3]), i64x3(*k.stride()[:3]), 1, 1, 1, n, 128,
                                       _lib.MINF_BF16, 128 ** -0.5, col.data_ptr(), diag.data_ptr(), col.shape[1], None, 0, begin,
                                       recall.data_ptr(), ws.data_ptr(), nbytes, _lib.stream_ptr(q.device)), "minf_pattern_recall")
    return recall


@pytest.mark.parametrize("n", [64, 300, 1025])
@pytest.mark.parametrize("stride", [0, 8, 64, 136])
def test_recall_reads_every_row_of_k_whatever_its_token_stride(gpu, n, stride):
    """Views whose rows coincide (stride 0: one key for every position), overlap or have gaps: the same bits as
    a contiguous copy of the view."""
    from minference_amd import pattern_recall
    q = heads(n, 2, 1, 60 + n, planted=False)[0].to(gpu)
    store = torch.randn((n - 1) * stride + 128, generator=torch.Generator().manual_seed(n)).bfloat16().to(gpu)
    k = store.as_strided((1, 1, n, 128), (store.numel(), store.numel(), stride, 1))
    k = store.expand(1, 1, n, 128) if stride == 0 else k
    cands = [("stream_llm", 4, 60), ("stream_llm", 30, 0), ("vertical_and_slash", 40, 60)]
    got = pattern_recall(q, k, cands, 0)
    assert torch.equal(got, pattern_recall(q, k.contiguous(), cands, 0))
    assert torch.equal(_recall_of(q, k.data_ptr(), (0, 0, stride), 1, n, cands[:2]),
                       _recall_of(q, k.contiguous().data_ptr(), (0, 0, 128), 1, n, cands[:2]))


def test_recall_with_k_stored_backwards(gpu):
    """A negative token stride (C ABI): the rows are addressed from the last one down."""
    n = 500
    q, k = (t.to(gpu) for t in heads(n, 1, 1, 9, planted=False))
    cands = [("stream_llm", 4, 60), ("stream_llm", 30, 0)]
    back = k.flip(2).contiguous()
    last = back.data_ptr() + (n - 1) * 128 * 2
    assert torch.equal(_recall_of(q, last, (0, 0, -128), 1, n, cands), _recall_of(q, k.data_ptr(), (0, 0, 128), 1, n, cands))


@pytest.mark.parametrize("n,masked", [(400, 64), (700, 33), (300, 290)])
def test_scores_of_minus_infinity_keep_nothing(gpu, n, masked):
    """Products that leave the fp32 range downwards in a row's first key blocks: such keys have no mass, and rows
    that see no other key count as zero; the rest against an fp64 softmax without those keys."""
    from minference_amd import pattern_recall
    g = torch.Generator().manual_seed(n)
    q, k = (torch.randn(1, 1, n, 128, generator=g).bfloat16() for _ in range(2))
    q[..., 0], k[..., 0] = 2.0 ** 70, 0.0
    k[:, :, :masked, 0] = -2.0 ** 70
    cands = [("stream_llm", 5, 40), ("stream_llm", masked + 9, 3), ("stream_llm", 1, n)]
    got = pattern_recall(q.to(gpu), k.to(gpu), cands, 0)[0, 0].double().cpu()
    s = q[0, 0, :, 1:].double() @ k[0, 0, :, 1:].double().t() * 128 ** -0.5
    r, c = torch.arange(n)[:, None], torch.arange(n)[None]
    p = torch.softmax(s.masked_fill((c > r) | (c < masked), float("-inf")), -1).nan_to_num(0.0)
    for t, (_, v, w) in enumerate(cands):
        want = (p * ((c < v) | (r - c <= w))).sum() / n
        assert abs(got[t] - want) <= 2.0 ** -22 * want, (t, got[t].item(), want.item())


def test_recall_with_a_negative_scale(gpu):
    """sm_scale < 0 (C ABI) is the positive one on -Q, bit for bit."""
    n = 900
    q, k = (4 * t.to(gpu) for t in heads(n, 2, 1, 12))
    cands = [("stream_llm", 4, 60), ("stream_llm", 30, 0), ("stream_llm", 1, n - 1)]
    got = _recall_of(q, k.data_ptr(), k.stride()[:3], 1, n, cands, -128.0 ** -0.5)
    assert torch.equal(got, _recall_of(-q, k.data_ptr(), k.stride()[:3], 1, n, cands))
    assert (got[:, 2] - 1).abs().max() <= 2.0 ** -22


@pytest.mark.parametrize("nats", [14, 22, 30, 60])
def test_candidates_without_the_sink_keep_their_accuracy(gpu, nats):
    """One key far above all others in every row: the candidates that leave it out keep a share of e^-nats, all
    of it from small exponentials (columns and diagonals in and outside the sink's own block, whole blocks, single
    diagonals).  Bound: a score at distance D (powers of two) from the maximum is rounded there and scaled by a
    rounded factor, 2^-24 D each, beside fp32 sums of about 5 roundings each way: 2^-23 (D + 32) of the share."""
    n = 1500
    g = torch.Generator().manual_seed(nats)
    q, k = (torch.randn(1, 1, n, 128, generator=g) for _ in range(2))
    q[..., 0], k[..., 0] = 8.0, 0.0
    k[0, 0, 0, 0] = nats * 128 ** 0.5 / 8
    q, k = q.bfloat16().to(gpu), k.bfloat16().to(gpu)
    col, diag = (torch.zeros(1, (n + 63) // 64 * 64, dtype=torch.uint8, device=gpu) for _ in range(2))
    col[:, 1:21] |= 1
    col[:, 40:300:3] |= 2
    col[:, 1:] |= 4
    diag[:, :300] |= 8
    diag[:, 5:200:7] |= 16
    got = _recall_of(q, k.data_ptr(), k.stride()[:3], 1, n, (), flags=(col, diag))[0].double()
    r, c = torch.arange(n, device=gpu)[:, None], torch.arange(n, device=gpu)[None]
    s = q[0, 0].double() @ k[0, 0].double().t().contiguous() * 128 ** -0.5
    p = torch.softmax(s.masked_fill(c > r, float("-inf")), -1)
    keep = col[0, :n][None] | diag[0][(r - c).clamp(min=0)]
    for t in range(5):
        want = (p * ((keep >> t) & 1)).sum() / n
        assert abs(got[t] - want) <= 2.0 ** -23 * (nats * 1.4427 + 10 + 32) * want, (t, got[t].item(), want.item())


@pytest.mark.parametrize("n", [1, 63, 257, 4096, 4097, 8192, 8193, 16384, 16385, 32768])
def test_flags_of_all_candidates_in_one_launch(gpu, n):
    """minf_search_flags against a stable sort: sizes around what a thread holds, scores that tie in thousands, infinities,
    selections of one entry, of nearly all and of all, candidates that select nothing, first positions beside
    selections; the arrays hold other bytes before and rows lie apart.  (No negative zeros: they rank below zero.)"""
    import ctypes
    from minference_amd import _lib
    rows, stride, pitch = 3, n + 5, (n + 63) // 64 * 64 + 64
    g = np.random.default_rng(n)
    sc = [g.standard_normal((rows, stride)).astype(np.float32), np.round(4 * g.standard_normal((rows, stride))).astype(np.float32) + 0.0]
    sc[1][1, :n // 2] = -np.inf
    sc[0][2, :n // 3] = np.inf
    sc[1][2] = 0.0
    cand = [(1, 1, 0, 0), (0, 0, min(n, 100), min(n, 7)), (min(n, 500), min(n, 700), 0, 0), (max(n - 1, 1), max(n - 1, 1), 0, 0),
            (n, n, 0, 0), (0, 0, 0, 0), ((n + 1) // 2, (n + 3) // 4, 3, 1), (min(n, 129), min(n, 128), 0, n)]
    flags = [torch.full((rows, pitch), 255, dtype=torch.uint8, device=gpu) for _ in range(2)]
    dev = [torch.from_numpy(x).to(gpu) for x in sc]
    arr = (ctypes.c_int32 * 32)(*(x for c in cand for x in c))
    st = _lib.load().minf_search_flags(dev[0].data_ptr(), dev[1].data_ptr(), rows, n, stride, arr, 8, flags[0].data_ptr(),
                                       flags[1].data_ptr(), pitch, _lib.stream_ptr(gpu))
    assert st == 0
    for i in range(2):
        want = np.zeros((rows, pitch), np.uint8)
        for r in range(rows):
            order = np.argsort(-sc[i][r, :n].astype(np.float64), kind="stable")
            for t, c in enumerate(cand):
                at = order[:c[i]]
                want[r, n - 1 - at if i else at] |= 1 << t
                want[r, :min(c[2 + i], n)] |= 1 << t
        assert np.array_equal(flags[i].cpu().numpy(), want), i


@pytest.mark.parametrize("n,k", [(1, 1), (4, 3), (256, 31), (257, 257), (1000, 125), (1025, 1), (2560, 320), (2561, 320), (4096, 512)])
def test_block_flags_are_the_indices_of_the_same_selection(gpu, n, k):
    """Block-causal rows (some with fewer entries above -inf than are kept, scores that tie), first in place of what the
    flags hold, then a second candidate's ORed in; against the index lists of the same kernel."""
    from minference_amd import _lib
    lib, per_head, pitch, s = _lib.load(), n, (n + 3) // 4 * 4 + 4, _lib.stream_ptr(gpu)
    rows = 2 * per_head if n < 300 else 300
    g = torch.Generator().manual_seed(n)
    sc = (8 * torch.randn(rows, n, generator=g)).round() + 0.0
    sc[torch.arange(n)[None] > (torch.arange(rows) % per_head)[:, None]] = float("-inf")
    sc = sc.to(gpu)
    flags = torch.full((rows, pitch), 255, dtype=torch.uint8, device=gpu)
    want = torch.zeros((rows, pitch), dtype=torch.uint8)
    for bit, kk, clear in ((3, k, 1), (5, max(k // 2, 1), 0)):
        idx = torch.empty((rows, kk), dtype=torch.int32, device=gpu)
        assert lib.minf_topk_indices_block_causal(sc.data_ptr(), rows, n, n, kk, idx.data_ptr(), kk, per_head, s) == 0
        assert lib.minf_topk_flags_block_causal(sc.data_ptr(), rows, n, n, kk, per_head, bit, clear, flags.data_ptr(), pitch, s) == 0
        want.scatter_(1, idx.cpu().long(), want.gather(1, idx.cpu().long()) | (1 << bit))
        assert torch.equal(flags.cpu(), want), bit
