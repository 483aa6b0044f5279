"""The 1-bit scan's counting selection (k above 1024) at the edges of its ranges of ids: tables
ending inside a range and a tile, codes so alike that the ties at the cut fill whole ranges, masks
that leave fewer than k items, and more queries than one batch of its workspace, against the
oracle bit for bit."""

import numpy as np
import pytest
import torch

from oracle import scan as osc
from tests.conftest import rng
from tests.test_int8_scan import _pack

pytestmark = pytest.mark.gpu


def _t(dev, x):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


@pytest.mark.parametrize("n,w,b,k", [(1025, 1, 1, 1025), (1024, 2, 9, 1100), (8192, 2, 3, 8192),
                                     (8193, 3, 17, 1500), (66_000, 2, 8, 5000),
                                     (20_000, 16, 2, 2000), (131_073, 1, 33, 4000)])
@pytest.mark.parametrize("alike", [False, True])
@pytest.mark.parametrize("share", [None, 0.3, 0.01])
def test_counting(dev, n, w, b, k, alike, share):
    import retrieve_amd.hip  # noqa: F401

    g = rng(n + w + b + k)
    items = g.integers(-2**63, 2**63 - 1, (n, w), dtype=np.int64)
    if alike:  # three distinct codes: ranges full of one popcount
        items = items[g.integers(0, 3, n)]
    q = g.integers(-2**63, 2**63 - 1, (b, w), dtype=np.int64)
    valid = None if share is None else g.random((b, n)) < share
    print(f"large k n={n} w={w} b={b} k={k} alike={alike} share={share}", flush=True)
    ids, sc = torch.ops.retrieve_amd.hamming_scan_topk(
        _t(dev, q), _t(dev, items), k, None if valid is None else _t(dev, _pack(valid)))
    want_ids, want_sc = osc.hamming_topk(q, items, k, valid)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), want_sc)


def test_batches(dev):
    """2,720 queries at k = 8192 are two batches of the workspace (12,352 entries a query): the
    rows around the cut and the last ones."""
    import retrieve_amd.hip  # noqa: F401

    g = rng(77)
    n, b, k = 8200, 2720, 8192
    items = g.integers(-2**63, 2**63 - 1, (n, 1), dtype=np.int64)
    q = g.integers(-2**63, 2**63 - 1, (b, 1), dtype=np.int64)
    valid = g.random((b, n)) < 0.9
    print("large k in two batches", flush=True)
    ids, sc = torch.ops.retrieve_amd.hamming_scan_topk(_t(dev, q), _t(dev, items), k,
                                                       _t(dev, _pack(valid)))
    rows = np.r_[0:3, 2690:2720]
    want_ids, want_sc = osc.hamming_topk(q[rows], items, k, valid[rows])
    assert np.array_equal(ids[rows.tolist()].cpu().numpy(), want_ids)
    assert np.array_equal(sc[rows.tolist()].cpu().numpy(), want_sc)


@pytest.mark.parametrize("k", [40, 1500])
def test_float_scores(dev, k):
    """A packed-bits module's filtered scan: fp32 scores with -inf past the passing items, the
    integer scan's values."""
    import retrieve_amd.hip  # noqa: F401
    from retrieve_amd.modules import SimHashKNN

    g = rng(81 + k)
    n, b, d = 3000, 5, 64
    m = SimHashKNN(k, k_bits=128, seed=2)
    m.register_index(_t(dev, g.standard_normal((n, d)).astype(np.float32)))
    q = _t(dev, g.standard_normal((b, d)).astype(np.float32))
    valid = g.random((b, n)) < 0.2
    valid[0] = False
    valid[1, 30:] = False
    bits = _t(dev, _pack(valid))
    print(f"float scores k={k}", flush=True)
    ids, sc = m.forward_bits(q, bits)
    want_ids, want = torch.ops.retrieve_amd.hamming_scan_topk(m._project_query(q), m.item_bits,
                                                              k, bits)
    assert sc.dtype == torch.float32 and torch.equal(ids, want_ids)
    assert torch.equal(sc, torch.where(want_ids >= 0, want.float(), float("-inf")))


@pytest.mark.parametrize("b,n,k", [(1, 5000, 3000), (9, 20_011, 8192), (2048, 73_728, 8192)])
def test_cells(dev, b, n, k):
    """Runs of one popcount as long as the cells that their entries walk (64), one longer, and
    whole ranges (up to 8192 items: the last shape's), cut by the end of k."""
    import retrieve_amd.hip  # noqa: F401

    runs = [64, 65, 1, 63, 128, 700, 2]
    pop = np.resize(np.repeat(np.arange(len(runs)), runs), n)
    pop[n // 2 :] = 7  # one popcount from here on
    items = np.zeros((n, 2), np.int64)
    items[:, 1] = (1 << (3 * pop + 1)) - 1
    q = np.zeros((b, 2), np.int64)
    print(f"large k cells b={b} n={n} k={k}", flush=True)
    ids, sc = torch.ops.retrieve_amd.hamming_scan_topk(_t(dev, q), _t(dev, items), k)
    h = 3 * pop + 1
    want = np.argsort(h, kind="stable")[:k]
    assert (ids == _t(dev, want)[None]).all()
    assert (sc == _t(dev, (128 - 2 * h[want]).astype(np.int32))[None]).all()


def test_equal_codes_cost(dev):
    """A table of one code is one cell a range, which costs no more than a few times what random
    codes do. (Each of 8192 entries walking 8192 took 26 times as long, 11.7 ms; the bitmap 3.2
    times, for the passes' same-address adds.)"""
    import retrieve_amd.hip  # noqa: F401

    g = rng(83)
    n, b, k = 1_000_000, 256, 8192
    q = _t(dev, g.integers(-2**63, 2**63 - 1, (b, 2), dtype=np.int64))
    items = _t(dev, g.integers(-2**63, 2**63 - 1, (n, 2), dtype=np.int64))
    print("large k cost of equal codes", flush=True)

    def took(codes):
        times = []
        for _ in range(6):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            torch.ops.retrieve_amd.hamming_scan_topk(q, codes, k)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    assert took(items[:1].expand(n, 2).contiguous()) < 10 * took(items)
