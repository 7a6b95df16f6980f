"""Offline pattern search -- host side.

Counterpart of ``search_pattern`` (reference minference/modules/minference_forward.py:129-227),
the routine that produces the per-head entries of the ``best_pattern`` JSON the prefill
dispatcher consumes.  The reference scores a candidate by multiplying an N x N mask into the
N x N softmax of one head; here the candidates of all heads are turned into per-column,
per-diagonal and per-32x32-block flag bytes (top-k and flag kernels of libminf_hip.so) and one
sweep over the causal score matrix (``minf_pattern_recall``) returns the kept softmax mass of up
to eight candidates at once, so the search also runs at context lengths whose N x N matrix would
not fit anywhere.
"""
from __future__ import annotations

import ctypes

import torch

from . import _lib
from .estimate import _prep16, topk_vertical_slash, vertical_slash_scores
from .ops import _check_qkv

ROW_BEGIN = 2500                  # minference_forward.py:161: attn_weights_x[:, :, 2500:]
SEARCH_FORCE = 30                 # :140 and :144: first 30 verticals, last 30 slash entries
CANDIDATES = (                    # :209-215
    ("stream_llm", 100, 800),
    ("vertical_and_slash", 30, 800), ("vertical_and_slash", 100, 750),
    ("vertical_and_slash", 500, 700), ("vertical_and_slash", 3500, 100),
    ("block_sparse", 8, 1),
)
MAX_CANDIDATES = 8


def _dtype_code(t):
    return _lib.MINF_BF16 if t.dtype == torch.bfloat16 else _lib.MINF_F16


def _add_block_flags(q16, k16, keep, bit, blk, bpitch, clear):
    """Bit ``bit`` of the flags of the top ``keep`` key blocks (32 tokens) per query block of the pooled scores, :175-186.
    ``clear``: the flags hold nothing yet."""
    B, H, N, _ = q16.shape
    Hk = k16.shape[1]
    rows = (N + 31) // 32
    keep = min(keep, rows)
    lib = _lib.load()
    dev = q16.device
    ws_bytes = lib.minf_search_block_index_workspace_bytes(B, H, Hk, N)
    ws = torch.empty((ws_bytes + 15) // 16 * 16, dtype=torch.uint8, device=dev)
    i64x3 = _lib.c_i64 * 3
    args = (q16.data_ptr(), k16.data_ptr(), i64x3(*q16.stride()[:3]), i64x3(*k16.stride()[:3]),
            B, H, Hk, N, 128, _dtype_code(q16), keep)
    with torch.cuda.device(dev):
        stream = _lib.stream_ptr(dev)
        if rows <= _lib.MINF_SEARCH_BLOCK_FLAGS_MAX:
            st = lib.minf_search_block_flags(*args, bit, clear, blk.data_ptr(), bpitch, ws.data_ptr(), ws_bytes, stream)
            _lib.check(st, "minf_search_block_flags")
            return
        if clear:
            blk.zero_()
        out = torch.empty((B, H, rows, keep), dtype=torch.int32, device=dev)
        st = lib.minf_search_block_index(*args, out.data_ptr(), ws.data_ptr(), ws_bytes, stream)
        _lib.check(st, "minf_search_block_index")
        st = lib.minf_flags_set_indices(out.data_ptr(), B * H * rows, keep, keep, bit, blk.data_ptr(), bpitch, rows, stream)
        _lib.check(st, "minf_flags_set_indices")


def _position_flags(candidates, scores, rows, N, pitch, dev):
    """The candidates' flag bytes per key column and per diagonal, [rows, pitch] uint8 each."""
    vertical, slash = scores
    lib = _lib.load()
    stream = _lib.stream_ptr(dev)
    sizes = []                                         # columns, diagonals selected; columns, diagonals from the first one on
    for ty, a, b in candidates:
        if ty not in ("stream_llm", "vertical_and_slash", "block_sparse"):
            raise ValueError(f"unknown pattern type {ty!r}")
        a, b = min(int(a), N), int(b)
        if ty == "vertical_and_slash" and min(a, b) < 1:
            raise _lib.MinfError(f"a vertical_and_slash candidate selects at least one entry of each kind, got {a}, {b}")
        sizes.append((0, 0, max(a, 0), max(min(b + 1, N), 0)) if ty == "stream_llm" else
                     (a, min(b, N), 0, 0) if ty == "vertical_and_slash" else (0, 0, 0, 0))
    if N <= _lib.MINF_SEARCH_FLAGS_MAX:
        col, diag = (torch.empty((rows, pitch), dtype=torch.uint8, device=dev) for _ in range(2))
        cand = (ctypes.c_int32 * (4 * len(sizes)))(*(x for c in sizes for x in c))
        with torch.cuda.device(dev):
            st = lib.minf_search_flags(vertical.data_ptr() if vertical is not None else None,
                                       slash.data_ptr() if slash is not None else None, rows, N, N, cand, len(sizes),
                                       col.data_ptr(), diag.data_ptr(), pitch, stream)
        _lib.check(st, "minf_search_flags")
        return col, diag
    col, diag = (torch.zeros((rows, pitch), dtype=torch.uint8, device=dev) for _ in range(2))
    with torch.cuda.device(dev):
        for bit, (kv, ks, first_col, first_diag) in enumerate(sizes):
            for first, flags in ((first_col, col), (first_diag, diag)):
                _lib.check(lib.minf_flags_set_range(0, first, rows, bit, flags.data_ptr(), pitch, stream), "minf_flags_set_range")
            if candidates[bit][0] == "vertical_and_slash":
                for idx, flags in zip(topk_vertical_slash(vertical, slash, kv, ks), (col, diag)):
                    kk = idx.shape[-1]
                    _lib.check(lib.minf_flags_set_indices(idx.data_ptr(), rows, kk, kk, bit, flags.data_ptr(), pitch, N, stream),
                               "minf_flags_set_indices")
    return col, diag


def pattern_recall(q, k, candidates=CANDIDATES, row_begin=ROW_BEGIN):
    """-> [B, H, len(candidates)] fp32: for every head and candidate ``(type, a, b)`` the mean over
    query rows >= row_begin of the exact causal softmax mass inside the candidate's mask, with the
    masks of the reference's search (element-granular, not the kernels' 64-wide blocks):

    * ``("stream_llm", v, s)``          diagonals 0..s plus the first v columns (:164-173)
    * ``("vertical_and_slash", v, s)``  the v best columns and the s best single diagonals of the
      last-64-query estimate, first 30 columns and diagonals 0..29 forced (:133-162)
    * ``("block_sparse", ratio, _)``    32 x 32 blocks: the ceil(N/32) // ratio best key blocks of
      every query block by mean-pooled score (:175-195)

    q [B,H,N,D], k [B,Hk,N,D] on the GPU (fewer kv heads are read in place).  NaN when
    N <= row_begin, like the reference's mean over an empty slice."""
    if not 1 <= len(candidates) <= MAX_CANDIDATES:
        raise ValueError(f"1..{MAX_CANDIDATES} candidates per call")
    _check_qkv(q, k, k)
    head_dim = q.shape[-1]
    q16, k16 = _prep16(q, k)
    if q16.shape[-1] < 128:                            # the sweep is built for 128 dims: zero columns add nothing
        q16, k16 = (torch.nn.functional.pad(t, [0, 128 - t.shape[-1]]) for t in (q16, k16))
    B, H, N, _ = q16.shape
    Hk = k16.shape[1]
    dev = q16.device
    lib = _lib.load()
    stream = _lib.stream_ptr(dev)
    pitch = (N + 63) // 64 * 64
    rows32 = (N + 31) // 32
    bpitch = (rows32 + 3) // 4 * 4
    blk = None
    select = any(ty == "vertical_and_slash" for ty, _, _ in candidates)
    scores = vertical_slash_scores(q, k, 64, SEARCH_FORCE, SEARCH_FORCE, reference_rounding=False) if select else (None, None)
    col, diag = _position_flags(candidates, scores, B * H, N, pitch, dev)
    for bit, (ty, a, _) in enumerate(candidates):
        if ty == "block_sparse" and rows32 // int(a) > 0:
            if blk is None:
                blk = torch.empty((B * H * rows32, bpitch), dtype=torch.uint8, device=dev)
                _add_block_flags(q16, k16, rows32 // int(a), bit, blk, bpitch, True)
            else:
                _add_block_flags(q16, k16, rows32 // int(a), bit, blk, bpitch, False)
    with torch.cuda.device(dev):
        recall = torch.empty((B * H, MAX_CANDIDATES), dtype=torch.float32, device=dev)
        ws_bytes = lib.minf_pattern_recall_workspace_bytes(B, H, N)
        ws = torch.empty((ws_bytes + 15) // 16 * 16, dtype=torch.uint8, device=dev)
        i64x3 = _lib.c_i64 * 3
        st = lib.minf_pattern_recall(
            q16.data_ptr(), k16.data_ptr(), i64x3(*q16.stride()[:3]), i64x3(*k16.stride()[:3]),
            B, H, Hk, N, 128, _dtype_code(q16), float(head_dim) ** -0.5,
            col.data_ptr(), diag.data_ptr(), pitch,
            blk.data_ptr() if blk is not None else None, bpitch, int(row_begin),
            recall.data_ptr(), ws.data_ptr(), ws_bytes, stream)
    _lib.check(st, "minf_pattern_recall")
    return recall.view(B, H, MAX_CANDIDATES)[..., :len(candidates)]


def _choose(candidates, scores):
    """:205-227: the best score wins (first on ties, must exceed 0); a stream_llm winner is
    relabelled vertical_and_slash with its own sizes, a block_sparse winner becomes
    vertical_and_slash (1000, 6096)."""
    best_ty, best_v, best_s, best = "", 0, 0, 0.0
    for (ty, v_size, s_size), sc in zip(candidates, scores):
        if sc > best:
            best_ty, best_v, best_s, best = ty, v_size, s_size, sc
    if best_ty == "stream_llm":
        best_ty = "vertical_and_slash"
    if best_ty == "block_sparse":
        best_ty, best_v, best_s = "vertical_and_slash", 1000, 6096
    return best_ty, best_v, best_s, best


def search_pattern(q, k, head=None, candidates=CANDIDATES, row_begin=ROW_BEGIN):
    """Same call as the reference's ``search_pattern(q, k, head)``: q, k [1, 1, N, D] of one head
    -> ``(type, vertical_size, slash_size, score)``.  ``head`` is only echoed by the reference's
    print and is ignored."""
    if q.shape[0] != 1 or q.shape[1] != 1:
        raise ValueError("search_pattern takes one head: q [1, 1, N, D]; use search_patterns for a layer")
    rec = pattern_recall(q, k, candidates, row_begin)[0, 0].tolist()
    return _choose(candidates, rec)


def search_patterns(q, k, candidates=CANDIDATES, row_begin=ROW_BEGIN):
    """All heads of a layer in one sweep: q [1,H,N,D], k [1,Hk,N,D] -> ``{str(head): [type, v, s,
    score]}``, one layer of the ``best_pattern`` table (the loop at minference_forward.py:566-571)."""
    if q.shape[0] != 1:
        raise ValueError("one sequence at a time")
    rec = pattern_recall(q, k, candidates, row_begin)[0].tolist()
    return {str(h): list(_choose(candidates, rec[h])) for h in range(q.shape[1])}
