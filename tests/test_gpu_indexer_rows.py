"""The many-row indexer top-k (more rows than the fused launch takes): its
shared-page filter, its per-row bounds and the select of its candidates give
the same indices as exact scores of every token and the exact select over
them, both of which test_gpu_indexer holds against the oracle bit for bit.
Rows of one request (causal lengths), of several with group boundaries inside
a workgroup's rows, of mixed requests and of two or three draft rows; unmapped pages, ties, constant rows,
rows shorter than k, and scores that are infinite (fp32 overflow of
finite operands; more and fewer than k of them, and all) or NaN."""

import numpy as np
import pytest
import torch

from helpers import to_dev

pytestmark = pytest.mark.gpu


def _case(dev, T, n_seqs, order, max_len, kind, seed):
    from ernie_kv import ops

    rng = np.random.default_rng(seed)
    g = torch.Generator(device=dev).manual_seed(seed)
    pages = (max_len + 63) // 64
    bt = rng.permutation(n_seqs * pages).astype(np.int32).reshape(n_seqs, pages)
    kcache = torch.zeros((n_seqs * pages, ops.fp8_page_bytes(128)), dtype=torch.uint8, device=dev)
    n = n_seqs * pages * 64
    k = torch.randn(n, 128, device=dev, generator=g) * (0.1 + 3 * torch.rand(n, 1, device=dev, generator=g))
    if kind == "ties":
        k = k[torch.randint(0, 30, (n,), device=dev, generator=g)]
    elif kind == "constant":
        k = k[:1].expand(n, 128)
    elif kind == "peaks":  # most keys tied, some above and below
        k = torch.where((torch.arange(n, device=dev) % 400 == 7)[:, None], k, k[:1])
    elif kind == "overflow":  # of every 7 keys one scores beyond fp32 (about half of them +inf, half -inf)
        k[::7] *= 1e37
    elif kind == "all inf":
        k = k.abs() * 1e37
    ops.indexer_k_insert(k.bfloat16().contiguous(), torch.arange(n, device=dev), kcache)
    if kind == "unmapped":
        bt[:, 1] = -1
        bt[-1, -1] = n_seqs * pages + 7
    elif kind in ("holes", "at most 0"):
        bt[:, 5::9] = -1
    if kind == "nan":
        kcache[:, 64 * 128:].view(torch.float32)[:, ::9] = float("nan")
    if order.isdigit():  # that many draft rows a request
        req = np.arange(T) // int(order)
    else:
        req = np.sort(rng.integers(0, n_seqs, T)) if order == "runs" else rng.integers(0, n_seqs, T)
    req = req.astype(np.int32)
    step = 7919 if max_len > 4 * T else 1  # (rows of all lengths)
    lengths = np.minimum(max_len, 1 + step * np.arange(T) % (max_len + 40)).astype(np.int32)
    q = torch.randn(T, 64, 128, device=dev, generator=g).bfloat16()
    w = torch.randn(T, 64, device=dev, generator=g).bfloat16()
    if kind in ("overflow", "all inf"):
        w = w * 1024
    if kind == "all inf":
        q, w = q.abs(), w.abs()
    elif kind == "at most 0":  # the unmapped pages' scores of 0 are the largest
        w = -w.abs()
    return (*ops.indexer_q_quant(q, w), kcache, to_dev(bt, dev), to_dev(req, dev), to_dev(lengths, dev))


@pytest.mark.parametrize("T,n_seqs,order,max_len,k,kind", [
    (1025, 1, "runs", 900, 64, "normal"),
    (1100, 3, "runs", 517, 256, "ties"),
    (1031, 5, "mixed", 640, 64, "normal"),
    (1040, 1, "runs", 2500, 2048, "unmapped"),
    (1032, 2, "runs", 700, 500, "constant"),
    (1030, 2, "runs", 900, 40, "overflow"),
    (1030, 2, "runs", 900, 200, "overflow"),
    (1026, 1, "runs", 500, 100, "all inf"),
    (1026, 3, "mixed", 600, 100, "nan"),
    (1030, 515, "2", 700, 100, "unmapped"),
    (1027, 343, "3", 400, 64, "ties"),
    (2100, 1, "runs", 50_000, 256, "holes"),  # runs of 66 pages, several 8192-token groups a row
    (1030, 1, "runs", 40_003, 256, "peaks"),  # more candidates than the select's LDS holds, some of them sure
    (300, 2, "runs", 60_000, 2048, "normal"),
    (260, 130, "2", 50_000, 512, "ties"),
    (1030, 2, "runs", 500, 40, "at most 0"),
    (1030, 2, "mixed", 500, 64, "at most 0"),
    (1030, 2, "runs", 500, 90, "at most 0"),
])
def test_many_rows_topk_matches_exact_scores(dev, T, n_seqs, order, max_len, k, kind):
    from ernie_kv import ops

    q8, w, dig, kcache, bt, req, lengths = _case(dev, T, n_seqs, order, max_len, kind, T + max_len)
    assert not ops.dsa_decode_prologue_folds(T, max_len)  # (the one-launch top-k does not take it)
    scores = torch.full((T, max_len), float("nan"), device=dev)
    ops.indexer_score(dig, w, kcache, bt, req, lengths, max_len, scores)
    n_inf = int((scores == float("inf")).sum(1).max())
    assert n_inf == max_len if kind == "all inf" else 40 < n_inf < 200 if kind == "overflow" else n_inf == 0
    ref = torch.empty((T, k), dtype=torch.int32, device=dev)
    ops.topk_select(scores, lengths, k, ref)
    got = torch.empty((T, k), dtype=torch.int32, device=dev)
    ops.indexer_topk(q8, dig, w, kcache, bt, req, lengths, max_len, got)
    assert torch.equal(got, ref)


@pytest.mark.parametrize("order", ["runs", "mixed"])
def test_many_rows_select_of_fewer_than_filtered(dev, order):
    """The two stages with a select of fewer tokens than the filter's k: also
    for rows between the two, which the filter left alone."""
    from ernie_kv import ops

    T, max_len, k = 1027, 900, 48
    q8, w, dig, kcache, bt, req, lengths = _case(dev, T, 3, order, max_len, "normal", 5)
    scores = torch.full((T, max_len), float("nan"), device=dev)
    ops.indexer_score(dig, w, kcache, bt, req, lengths, max_len, scores)
    ref = torch.empty((T, k), dtype=torch.int32, device=dev)
    ops.topk_select(scores, lengths, k, ref)
    ws = ops.indexer_topk_workspace(T, max_len, dev)
    got = torch.empty((T, k), dtype=torch.int32, device=dev)
    ops.indexer_filter(q8, dig, w, kcache, bt, req, lengths, max_len, ws, k=300)
    ops.indexer_select(dig, w, kcache, bt, req, lengths, max_len, got, ws)
    assert torch.equal(got, ref)


@pytest.mark.parametrize("T", [3, 1027])
def test_topk_of_zero_max_len(dev, T):
    """max_len 0 admits no token, whatever the rows' lengths say: all -1, in
    one call and in two stages."""
    from ernie_kv import ops

    q8, w, dig, kcache, bt, req, lengths = _case(dev, T, 2, "runs", 130, "normal", 6)
    ws = ops.indexer_topk_workspace(T, 0, dev)
    for staged in (False, True):
        got = torch.zeros((T, 16), dtype=torch.int32, device=dev)
        if staged:
            ops.indexer_filter(q8, dig, w, kcache, bt, req, lengths, 0, ws, k=16)
            ops.indexer_select(dig, w, kcache, bt, req, lengths, 0, got, ws)
        else:
            ops.indexer_topk(q8, dig, w, kcache, bt, req, lengths, 0, got, ws)
        assert (got == -1).all()


@pytest.mark.parametrize("slots", [False, True])
def test_many_rows_merged_output(dev, slots):
    """The top-k merged with the window, as token indices and as cache slots."""
    from ernie_kv import ops

    T, max_len, k, window = 1027, 900, 128, 64
    q8, w, dig, kcache, bt, req, lengths = _case(dev, T, 3, "runs", max_len, "unmapped", 9)
    positions = lengths.long() + window - 1  # the rows' keys end where their windows begin
    ws = ops.indexer_topk_workspace(T, max_len, dev)
    topk, got = (torch.empty((T, k + d), dtype=torch.int32, device=dev) for d in (0, window))
    ops.indexer_topk_merged(q8, dig, w, kcache, bt, req, lengths, max_len, topk, ws, merged=got, positions=positions,
                            window=window, merged_slots=slots)
    plain = torch.empty((T, k), dtype=torch.int32, device=dev)
    ops.indexer_topk(q8, dig, w, kcache, bt, req, lengths, max_len, plain)
    assert torch.equal(topk, plain)
    ref = torch.empty_like(got)
    ops.merge_swa_topk(plain, ref, positions, window)
    if slots:
        i = ref.long()
        page = torch.where((i >= 0) & (i // 64 < bt.shape[1]),
                           bt[req.long()[:, None], (i // 64).clamp(0, bt.shape[1] - 1)].long(), -1)
        ref = torch.where((page >= 0) & (page < kcache.shape[0]), page * 64 + i % 64, -1).int()
    assert torch.equal(got, ref)
