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
