"""GPU parity of the whole-row decode kernel (many or short rows) vs the fp64
oracle, with the tolerances of test_gpu_decode: row counts and widths at the
edges of its 32-row steps and of the dispatch, masked entries, empty rows,
head counts that fill a 32-head block partly, and scores that make a later
step exceed the softmax reference by more than 8 and by more than 100 log2
units (the reference moves; a step's weights are computed again)."""

import numpy as np
import pytest
import torch

from helpers import bf16_tensor, randn_bf16, to_dev
from oracle import decode as od
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
