"""The candidate scans on every lane layout (row bytes at and past each layout's width), with
counts that end inside a wave's 64 candidates, runs of ids outside the table, lists filling up,
and batches on either side of the split merge, against the oracle: int8 and bit codes bit for
bit, float rows against their 64-bit dots."""

import numpy as np
import pytest
import torch

from oracle import scan as osc
from tests.conftest import rng

pytestmark = pytest.mark.gpu


def _t(dev, x):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


def _cands(g, b, p, n):
    cand = np.stack([g.permutation(n)[:p] for _ in range(b)]).astype(np.int64)
    counts = g.integers(0, p + 1, b).astype(np.int64)
    counts[0] = p
    if b > 1:
        counts[1] = 0
    cand[:, p // 3: p // 3 + 70] = -1  # a whole step of padding
    cand[0, 5] = n + 9
    return cand, counts


def _oracle(score, cand, counts, k, n, empty):
    """``candidate_topk`` over each row's ids inside the table (the others are skipped)."""
    b, p = cand.shape
    packed = np.full_like(cand, -1)
    kept = np.zeros(b, np.int64)
    for r in range(b):
        ids = cand[r, :counts[r]]
        ids = ids[(ids >= 0) & (ids < n)]
        packed[r, :len(ids)] = ids
        kept[r] = len(ids)
    return osc.candidate_topk(score, packed, kept, k, pad_to_k=False, empty_score=empty)


@pytest.mark.parametrize("d", [16, 32, 48, 64, 128, 144, 192, 256, 272, 512, 768, 1024, 2048, 4096,
                               8192])
def test_int8(dev, d):
    import retrieve_amd.hip  # noqa: F401

    g = rng(500 + d)
    n, b, p, k = 1200, 4, 700, 33
    items = g.integers(-9, 10, (n, d), dtype=np.int8)
    q = g.integers(-9, 10, (b, d), dtype=np.int8)
    cand, counts = _cands(g, b, p, n)
    print(f"int8_candidates d={d}", flush=True)
    ids, sc = torch.ops.retrieve_amd.int8_candidates_topk(_t(dev, q), _t(dev, items),
                                                          _t(dev, cand), _t(dev, counts), k)
    dots = q.astype(np.int64) @ items.astype(np.int64).T
    want_ids, want_sc = _oracle(lambda r, c: dots[r, c], cand, counts, k, n,
                                np.iinfo(np.int32).min)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), want_sc)


@pytest.mark.parametrize("w", [1, 2, 3, 8, 16])
@pytest.mark.parametrize("b,p,k", [(1, 5000, 1000), (150, 300, 20)])
def test_bits(dev, w, b, p, k):
    import retrieve_amd.hip  # noqa: F401

    g = rng(520 + w + b)
    n = 6000
    items = g.integers(-2**63, 2**63 - 1, (n, w), dtype=np.int64)
    q = g.integers(-2**63, 2**63 - 1, (b, w), dtype=np.int64)
    cand, counts = _cands(g, b, p, n)
    print(f"indirect bits w={w} b={b}", flush=True)
    ids, sc = torch.ops.retrieve.oporp_1bit_match_topk_indirect(
        _t(dev, q), _t(dev, items), k, _t(dev, cand), _t(dev, counts))
    hs = osc.hamming_scores(q, items)
    want_ids, want_sc = _oracle(lambda r, c: hs[r, c], cand, counts, k, n, -np.inf)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), np.asarray(want_sc, np.float32))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d", [8, 40, 96, 128, 200, 512, 1032])
def test_float(dev, dtype, d):
    """Scores within the bound of D fp32 roundings of the products' magnitudes; infinite scores
    keep their place with id -1."""
    import retrieve_amd.hip  # noqa: F401

    g = rng(540 + d)
    n, b, p, k = 900, 3, 700, 700
    items = torch.from_numpy(g.standard_normal((n, d)).astype(np.float32)).to(dtype)
    items[7, 0] = float("inf")
    q = torch.from_numpy(g.standard_normal((b, d)).astype(np.float32)).to(torch.float16).float()
    q[:, 0] = 1.0
    cand, counts = _cands(g, b, p, n)
    cand[0, 1] = 7
    cand[0, 2:][cand[0, 2:] == 7] = -1
    print(f"fused_masked_knn {dtype} d={d}", flush=True)
    ids, sc = torch.ops.retrieve.fused_masked_knn_topk(q.to(dev), items.to(dev), _t(dev, cand),
                                                       _t(dev, counts), k)
    ids, sc = ids.cpu().numpy(), sc.cpu().numpy()
    assert ids[0, 0] == -1 and np.isposinf(sc[0, 0])
    iv, qv = items.double().numpy(), q.double().numpy()
    for r in range(b):
        got = ids[r][ids[r] >= 0]
        want = cand[r, :counts[r]]
        want = want[(want >= 0) & (want < n) & (want != 7)]
        assert sorted(got.tolist()) == sorted(want.tolist())  # k holds every candidate
        at = np.flatnonzero(ids[r] >= 0)
        exact = iv[got] @ qv[r]
        bound = np.abs(iv[got]) @ np.abs(qv[r]) * d * 2.0**-24
        assert (np.abs(sc[r, at] - exact) <= bound).all()
        assert (np.diff(sc[r, at]) <= 0).all()


@pytest.mark.parametrize("d", [64, 4096])
@pytest.mark.parametrize("p", [1, 63, 65, 257, 1025])
def test_shares(dev, d, p):
    """Counts around a wave's 64 ids and the shares of one and of several rounds, narrow and wide
    rows."""
    import retrieve_amd.hip  # noqa: F401

    g = rng(560 + d + p)
    n, k = 1500, 20
    counts = np.array([p, p - 1, p // 2, min(p, 64), min(p, 1), 0], np.int64)
    b = len(counts)
    items = g.integers(-9, 10, (n, d), dtype=np.int8)
    q = g.integers(-9, 10, (b, d), dtype=np.int8)
    cand = np.stack([g.permutation(n)[:p] for _ in range(b)]).astype(np.int64)
    print(f"shares d={d} p={p}", flush=True)
    ids, sc = torch.ops.retrieve_amd.int8_candidates_topk(_t(dev, q), _t(dev, items),
                                                          _t(dev, cand), _t(dev, counts), k)
    dots = q.astype(np.int64) @ items.astype(np.int64).T
    want_ids, want_sc = _oracle(lambda r, c: dots[r, c], cand, counts, k, n,
                                np.iinfo(np.int32).min)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(sc.cpu().numpy(), want_sc)
