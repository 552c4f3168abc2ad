"""GPU parity of the whole-row decode kernel (many or short rows) vs the fp64
oracle, with the tolerances of test_gpu_decode: row counts and widths at the
edges of its 32-row steps and of the dispatch, masked entries, empty rows,
head counts that fill a 32-head block partly, and scores that make a later
step exceed the softmax reference by more than 8 log2 units (the reference
moves, the step's weights are computed again)."""

import numpy as np
import pytest
import torch

from helpers import bf16_tensor, permuted_block_table, randn_bf16, to_dev
from oracle import decode as od
from oracle import paged
from test_gpu_decode import _check, _fp8_pool

pytestmark = pytest.mark.gpu


def _run(dev, rng, dim, heads, idx, lengths, bf16=False, pool=None, sinks=True):
    from ernie_kv import ops

    T, pages = idx.shape[0], 40
    if bf16:
        rows = randn_bf16(rng, (pages * 64, dim))
        cache, fetch = bf16_tensor(rows, dev).view(-1, 64, dim), lambda s: od.gather_rows_bf16(rows, s)
    else:
        pool = _fp8_pool(rng, pages, dim) if pool is None else pool
        cache, fetch = to_dev(pool, dev), lambda s: od.gather_rows_fp8(pool, s, dim)
    q = randn_bf16(rng, (T, heads, dim))
    snk = rng.standard_normal(heads).astype(np.float32) if sinks else None
    out = torch.zeros((T, heads, 512), dtype=torch.bfloat16, device=dev)
    lse = torch.zeros((T, heads), dtype=torch.float32, device=dev)
    ops.sparse_mla_decode(bf16_tensor(q, dev), cache, to_dev(idx, dev), 256 ** -0.5, out, lse,
                          sinks=None if snk is None else to_dev(snk, dev), cache_bf16=bf16,
                          lengths=None if lengths is None else to_dev(lengths, dev))
    ref_o, ref_l = od.sparse_mla_decode(q, fetch, idx, 256 ** -0.5, 512, snk, lengths)
    _check(out, lse, ref_o, ref_l, heads)


@pytest.mark.parametrize("dim,heads,bf16", [(576, 64, False), (576, 16, False), (512, 48, False), (576, 64, True),
                                            (512, 32, True)])
@pytest.mark.parametrize("T,width", [(1, 1), (3, 31), (2, 33), (9, 160), (193, 65)])
def test_rows_step_edges(dev, dim, heads, bf16, T, width):
    rng = np.random.default_rng(dim + heads + T + width)
    idx = rng.integers(0, 40 * 64, (T, width)).astype(np.int32)
    idx[rng.random((T, width)) < 0.2] = -1
    idx[T // 2] = -1  # a row with nothing to attend to
    lengths = None if T % 2 else rng.integers(0, width + 1, T).astype(np.int32)
    _run(dev, rng, dim, heads, idx, lengths, bf16, sinks=T != 3)


@pytest.mark.parametrize("T,heads,width", [(96, 64, 2176), (16, 64, 384), (130, 48, 1152)])
def test_rows_dispatch_edges(dev, T, heads, width):
    rng = np.random.default_rng(T + width)
    idx = rng.integers(-200, 40 * 64, (T, width)).astype(np.int32)
    lengths = rng.integers(width // 2, width + 1, T).astype(np.int32)
    lengths[0], lengths[1] = width, 0
    _run(dev, rng, 576, heads, np.maximum(idx, -1), lengths)


@pytest.mark.parametrize("T,heads,width,dim,bf16", [
    (128, 64, 192, 576, True), (129, 64, 192, 576, True), (96, 48, 1500, 512, True), (104, 48, 1500, 512, True),
    (192, 32, 769, 512, True), (257, 16, 769, 576, True), (384, 16, 769, 512, True), (7, 48, 256, 576, False),
    (8, 48, 256, 576, False), (120, 48, 1152, 576, False), (128, 48, 1152, 576, False)])
def test_dispatch_lines(dev, T, heads, width, dim, bf16):
    """Both sides of the lines between the two kernels that depend on the cache
    type, the heads and the few-row kernel's workgroups.  Most rows are short, a
    few full."""
    rng = np.random.default_rng(T + heads + width)
    idx = rng.integers(-100, 40 * 64, (T, width)).astype(np.int32)
    lengths = rng.integers(0, 40, T).astype(np.int32)
    lengths[::50] = width
    _run(dev, rng, dim, heads, np.maximum(idx, -1), lengths, bf16)


@pytest.mark.parametrize("T,width,bf16", [(5, 200, False), (193, 300, False), (9, 100, True)])
def test_rows_block_table(dev, T, width, bf16):
    """Request-local indices through the block table: unmapped pages, pages and
    entries past the table."""
    from ernie_kv import ops

    rng = np.random.default_rng(T)
    B, P, dim, H = 3, 12, 576, 64
    bt = permuted_block_table(rng, B, P)
    bt[1, 3], bt[2, 5] = -1, B * P + 4
    req = rng.integers(0, B, T).astype(np.int32)
    logical = np.maximum(rng.integers(-100, (P + 2) * 64, (T, width)), -1).astype(np.int32)
    lengths = rng.integers(0, width + 1, T).astype(np.int32)
    if bf16:
        rows = randn_bf16(rng, (B * P * 64, dim))
        cache, fetch = bf16_tensor(rows, dev).view(-1, 64, dim), lambda s: od.gather_rows_bf16(rows, s)
    else:
        pool = _fp8_pool(rng, B * P, dim)
        cache, fetch = to_dev(pool, dev), lambda s: od.gather_rows_fp8(pool, s, dim)
    q = randn_bf16(rng, (T, H, dim))
    out = torch.zeros((T, H, 512), dtype=torch.bfloat16, device=dev)
    lse = torch.zeros((T, H), dtype=torch.float32, device=dev)
    ops.sparse_mla_decode(bf16_tensor(q, dev), cache, to_dev(logical, dev), 256 ** -0.5, out, lse, cache_bf16=bf16,
                          lengths=to_dev(lengths, dev), block_table=to_dev(bt, dev), req_ids=to_dev(req, dev))
    page = np.where((logical >= 0) & (logical < P * 64), bt[req[:, None], np.clip(logical, 0, P * 64 - 1) // 64], -1)
    glob = np.where((page >= 0) & (page < B * P), page * 64 + logical % 64, -1)
    ref_o, ref_l = od.sparse_mla_decode(q, fetch, glob, 256 ** -0.5, 512, None, lengths)
    _check(out, lse, ref_o, ref_l, H)


@pytest.mark.parametrize("factor", [8.0, 96.0])
def test_rows_reference_moves(dev, factor):
    """Later steps hold rows `factor` times larger: scores a few tens, or more
    than a hundred, log2 units above the reference of the steps before."""
    rng = np.random.default_rng(int(factor))
    pool = _fp8_pool(rng, 40, 576)
    scales = pool[:, 64 * 576:].view(np.float32)
    scales[20:] *= factor
    T, width = 12, 250
    idx = np.concatenate([rng.integers(0, 20 * 64, (T, 120)), rng.integers(20 * 64, 40 * 64, (T, 60)),
                          rng.integers(0, 20 * 64, (T, 70))], 1).astype(np.int32)
    assert idx.shape[1] == width
    _run(dev, rng, 576, 64, idx, None, pool=pool)


@pytest.mark.parametrize("bf16", [False, True])
def test_rows_large_values_after_reference(dev, bf16):
    """Values of 2**40 in rows whose scores exceed the reference of the steps
    before them by 89 log2 units: their weights against it times their values
    pass fp32's range, the outputs (about 2**40) do not."""
    from ernie_kv import ops

    T, H, dim, pages, width = 16, 64, 576, 8, 192
    rng = np.random.default_rng(40)
    high = np.zeros(pages * 64, bool)
    high[2 * 64:] = True
    if bf16:
        rows = np.tile(np.where(high, 2.0 ** 40, 1.0).astype(np.float32)[:, None], (1, dim))
        rows[:, 512:] = 0.0
        rows[high, 512] = 62.0
        q512 = 16.0
        cache, fetch = bf16_tensor(rows, dev).view(-1, 64, dim), lambda s: od.gather_rows_bf16(rows, s)
    else:
        codes = np.full((pages * 64, dim), 0x78, np.uint8)  # 256
        codes[:, 512:] = 0
        codes[high, 512] = 0x38  # 1
        scales = np.where(high, 2.0 ** 32, 2.0 ** -8).astype(np.float32)
        q512 = 62.0 * 16 / 2.0 ** 32
        pool = np.zeros((pages, paged.fp8_page_bytes(dim)), np.uint8)
        paged.write_fp8_rows(pool, np.arange(pages * 64), codes, scales, dim)
        cache, fetch = to_dev(pool, dev), lambda s: od.gather_rows_fp8(pool, s, dim)
    idx = np.concatenate([rng.integers(0, 128, (T, 80)), rng.integers(128, pages * 64, (T, 60)),
                          rng.integers(0, 128, (T, 52))], 1).astype(np.int32)
    q = np.zeros((T, H, dim), np.float32)
    q[..., 512] = q512  # (a bf16 value)
    out = torch.zeros((T, H, 512), dtype=torch.bfloat16, device=dev)
    lse = torch.zeros((T, H), dtype=torch.float32, device=dev)
    ops.sparse_mla_decode(bf16_tensor(q, dev), cache, to_dev(idx, dev), 1 / 16, out, lse, cache_bf16=bf16)
    ref_o, ref_l = od.sparse_mla_decode(q, fetch, idx, 1 / 16, 512)
    assert (ref_o > 2.0 ** 39).all()
    _check(out, lse, ref_o, ref_l, H)
