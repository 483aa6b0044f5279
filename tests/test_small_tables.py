"""Scans of tables below the full seed sample: the sizes where the sparse sample starts and
changes its stride, batches that end inside a query group, k on either side of the sample's rank,
filters that few rows pass, and tables whose best rows all lie in the sampled blocks (the bound
then fails for every query and the fallback answers), against the oracle bit for bit."""

import numpy as np
import pytest
import torch

from oracle import filters as of
from oracle import scan as osc
from oracle import select as osel
from tests.conftest import rng
from tests.test_int8_scan import _pack

pytestmark = pytest.mark.gpu

SEED_BLOCK = 256


def _t(dev, x):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


def _want(q, items, k, valid=None):
    scores = (q.astype(np.float32) @ items.astype(np.float32).T).astype(np.int32)  # exact: < 2^24
    if valid is None:
        return osel.topk_rows(scores, k)
    return osel.topk_rows(scores, k, valid)


@pytest.mark.parametrize("n", [1, 127, 129, 5000, 16383, 16640, 40_001, 65_535, 66_049, 140_001])
@pytest.mark.parametrize("b,k", [(1, 100), (17, 1), (33, 100), (150, 10), (7, 1000), (260, 300)])
def test_int8(dev, n, b, k):
    import retrieve_amd.hip  # noqa: F401

    print(f"int8 n={n} b={b} k={k}", flush=True)
    g = rng(n + 7 * b + k)
    d = 128
    items = g.integers(-20, 21, (n, d), dtype=np.int8)
    q = g.integers(-20, 21, (b, d), dtype=np.int8)
    ids, sc = torch.ops.retrieve_amd.int8_scan_topk(_t(dev, q), _t(dev, items), k)
    want_ids, want_sc = _want(q, items, k)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), want_sc)


@pytest.mark.parametrize("b", [16, 17, 32, 33, 65])
@pytest.mark.parametrize("n,d,k", [(300, 768, 20), (20_000, 1024, 10), (30_001, 64, 1000)])
def test_query_groups(dev, n, d, k, b):
    """Row widths the register-blocked scan does not take, on either side of one and two 16-query
    groups a wave, plain and masked."""
    import retrieve_amd.hip  # noqa: F401

    print(f"groups n={n} d={d} b={b} k={k}", flush=True)
    g = rng(n + d + b)
    items = g.integers(-20, 21, (n, d), dtype=np.int8)
    q = g.integers(-20, 21, (b, d), dtype=np.int8)
    for valid in (None, g.random((b, n)) < 0.1):
        ids, sc = torch.ops.retrieve_amd.int8_scan_topk(
            _t(dev, q), _t(dev, items), k, None if valid is None else _t(dev, _pack(valid)))
        want_ids, want_sc = _want(q, items, k, valid)
        assert np.array_equal(ids.cpu().numpy(), want_ids)
        assert np.array_equal(sc.cpu().numpy(), want_sc)


@pytest.mark.parametrize("share", [0.2, 0.002, 0.0])
@pytest.mark.parametrize("n,b,k", [(66_049, 5, 100), (140_001, 33, 100), (20_000, 150, 40),
                                   (70_000, 18, 1000)])
def test_masked(dev, n, b, k, share):
    import retrieve_amd.hip  # noqa: F401

    print(f"masked int8 n={n} b={b} k={k} share={share}", flush=True)
    g = rng(n + b + int(1000 * share))
    d = 64 if b < 32 else 128
    items = g.integers(-20, 21, (n, d), dtype=np.int8)
    q = g.integers(-20, 21, (b, d), dtype=np.int8)
    valid = g.random((b, n)) < share
    valid[-1] = True
    ids, sc = torch.ops.retrieve_amd.int8_scan_topk(_t(dev, q), _t(dev, items), k,
                                                    _t(dev, _pack(valid)))
    want_ids, want_sc = _want(q, items, k, valid)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), want_sc)


@pytest.mark.parametrize("b", [3, 40, 200])
@pytest.mark.parametrize("stride,n", [(4, 20_000), (8, 50_000), (16, 100_000)])
def test_bound_fails(dev, b, stride, n):
    """The rows of every sampled block doubled: a query's best k are all sampled, so the sample's
    rank-th best lies above the table's k-th."""
    import retrieve_amd.hip  # noqa: F401

    print(f"sampled blocks best n={n} b={b}", flush=True)
    g = rng(n + b)
    d, k = 128, 100
    items = g.integers(-20, 21, (n, d), dtype=np.int8)
    rows = n // stride // SEED_BLOCK * SEED_BLOCK
    step = n // rows
    r = np.arange(rows)
    items[r // SEED_BLOCK * SEED_BLOCK * step + r % SEED_BLOCK] *= 2
    q = g.integers(-20, 21, (b, d), dtype=np.int8)
    ids, sc = torch.ops.retrieve_amd.int8_scan_topk(_t(dev, q), _t(dev, items), k)
    want_ids, want_sc = _want(q, items, k)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), want_sc)


@pytest.mark.parametrize("b", [1, 20, 70, 300])
def test_bits(dev, b):
    import retrieve_amd.hip  # noqa: F401

    g = rng(90 + b)
    n, k = 70_001, 100
    items = g.integers(-2**63, 2**63 - 1, (n, 8), dtype=np.int64)
    q = g.integers(-2**63, 2**63 - 1, (b, 8), dtype=np.int64)
    print(f"bits n={n} b={b}", flush=True)
    ids, sc = torch.ops.retrieve_amd.hamming_scan_topk(_t(dev, q), _t(dev, items), k)
    want_ids, want_sc = osc.hamming_topk(q, items, k)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), want_sc)


@pytest.mark.parametrize("b", [1, 9, 31])
def test_clauses(dev, b):
    """Exact clauses tested in the seed and the scan at batches that end inside a 16-query group."""
    import retrieve_amd.hip  # noqa: F401

    g = rng(95 + b)
    n, d, k, c = 100_001, 64, 50, 4
    items = g.integers(-20, 21, (n, d), dtype=np.int8)
    q = g.integers(-20, 21, (b, d), dtype=np.int8)
    attrs = g.integers(0, 6, (n, c, 1)).astype(np.int16)
    values = g.integers(0, 6, (b, c)).astype(np.int64)
    values[g.random((b, c)) < 0.5] = -1
    rev = np.array([False, False, True, False])
    print(f"clauses n={n} b={b}", flush=True)
    ids, sc = torch.ops.retrieve_amd.int8_scan_topk_clauses(
        _t(dev, q), _t(dev, items), k, _t(dev, attrs), _t(dev, rev), _t(dev, values))
    valid = of.clause_match(attrs.astype(np.int64), rev, values)
    want_ids, want_sc = _want(q, items, k, valid)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), want_sc)


def _sampled(n, stride):
    rows = n // stride // SEED_BLOCK * SEED_BLOCK
    r = np.arange(rows)
    return r // SEED_BLOCK * SEED_BLOCK * (n // rows) + r % SEED_BLOCK


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("n,stride,k", [(70_001, 16, 10), (70_001, 16, 100), (110_001, 4, 1000),
                                        (200_003, 8, 1000)])
@pytest.mark.parametrize("b", [1, 20])
def test_fallback_behind_the_kth(dev, b, n, stride, k, masked):
    """Sampled rows better than the rest, per-wave scans: the fallback runs behind the k-th best of
    the sample's lists."""
    import retrieve_amd.hip  # noqa: F401

    print(f"fallback int8 n={n} b={b} k={k} masked={masked}", flush=True)
    g = rng(n + b + k)
    items = g.integers(-20, 21, (n, 64), dtype=np.int8)
    items[_sampled(n, stride)] *= 2
    q = g.integers(-20, 21, (b, 64), dtype=np.int8)
    valid = g.random((b, n)) < 0.5 if masked else None
    ids, sc = torch.ops.retrieve_amd.int8_scan_topk(
        _t(dev, q), _t(dev, items), k, None if valid is None else _t(dev, _pack(valid)))
    want_ids, want_sc = _want(q, items, k, valid)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), want_sc)


@pytest.mark.parametrize("n,stride,k", [(17_000, 4, 20), (70_001, 16, 100), (110_001, 4, 1000)])
@pytest.mark.parametrize("b", [1, 40, 100])
def test_fallback_behind_the_kth_bits(dev, b, n, stride, k):
    """The same over 512-bit codes: half of a sampled row's words are some query's."""
    import retrieve_amd.hip  # noqa: F401

    print(f"fallback bits n={n} b={b} k={k}", flush=True)
    g = rng(n + b + k)
    items = g.integers(-2**63, 2**63 - 1, (n, 8), dtype=np.int64)
    q = g.integers(-2**63, 2**63 - 1, (b, 8), dtype=np.int64)
    at = _sampled(n, stride)
    items[at, :4] = q[g.integers(0, b, at.size), :4]
    ids, sc = torch.ops.retrieve_amd.hamming_scan_topk(_t(dev, q), _t(dev, items), k)
    want_ids, want_sc = osc.hamming_topk(q, items, k)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), want_sc)


@pytest.mark.parametrize("n,b", [(262_143, 3), (262_144, 31), (65_535, 33), (65_536, 40)])
def test_masked_sample(dev, n, b):
    """Masked scans on either side of the smallest table that takes a sparse sample (below and from
    32 queries), rows of no, few and all passing items: int8 of a width without the blocked scan,
    and 512-bit codes."""
    import retrieve_amd.hip  # noqa: F401

    print(f"masked sample n={n} b={b}", flush=True)
    g = rng(n + b)
    k = 50
    valid = np.zeros((b, n), bool)
    valid[0] = True
    valid[1:-1] = g.random((b - 2, n)) < 0.02
    mask = _t(dev, _pack(valid))
    items = g.integers(-20, 21, (n, 768), dtype=np.int8)
    q = g.integers(-20, 21, (b, 768), dtype=np.int8)
    rows = np.r_[0:3, b - 2 : b]
    ids, sc = torch.ops.retrieve_amd.int8_scan_topk(_t(dev, q), _t(dev, items), k, mask)
    want_ids, want_sc = _want(q[rows], items, k, valid[rows])
    assert np.array_equal(ids.cpu().numpy()[rows], want_ids)
    assert np.array_equal(sc.cpu().numpy()[rows], want_sc)
    codes = g.integers(-2**63, 2**63 - 1, (n, 8), dtype=np.int64)
    qc = g.integers(-2**63, 2**63 - 1, (b, 8), dtype=np.int64)
    ids, sc = torch.ops.retrieve_amd.hamming_scan_topk(_t(dev, qc), _t(dev, codes), k, mask)
    want_ids, want_sc = osc.hamming_topk(qc[rows], codes, k, valid[rows])
    assert np.array_equal(ids.cpu().numpy()[rows], want_ids)
    assert np.array_equal(sc.cpu().numpy()[rows], want_sc)
