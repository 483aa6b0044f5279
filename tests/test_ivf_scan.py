"""The IVF scan at the edges of its work split: row widths on every lane layout, lists shorter than
a warp and empty ones, a width that cuts the row, one wave's run ending inside a step, queues that
fill exactly, and every filter form, against the oracle bit for bit."""

import numpy as np
import pytest
import torch

from oracle import filters as of
from oracle import silvertorch as ost
from tests.conftest import rng
from tests.test_int8_scan import _pack
from tests.test_search import _ivf, _run, _t

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [16, 32, 48, 64, 80, 128, 192, 208, 256, 512, 528, 1024, 1040, 2064, 4112])
def test_widths(dev, d):
    g = rng(300 + d)
    n, b, k, lists = 3000, 3, 40, 30
    items, offsets, sizes, perm = _ivf(g, n, d, lists)
    q = g.standard_normal((b, d)).astype(np.float32)
    probes = np.stack([g.permutation(lists)[:12] for _ in range(b)]).astype(np.int64)
    ids, sc = _run(dev, q, probes, offsets, sizes, items, perm, 1.5, k, n, 128)
    want = ost.search(q, probes, offsets, sizes, items, perm, [1.5], k, n, 128)
    assert np.array_equal(ids, want[0]) and np.array_equal(sc, want[1])


@pytest.mark.parametrize("b,n,n_lists,n_probe,k,width", [
    (1, 60_000, 200, 190, 1000, 60_000),   # one row over many workgroups, lists filling up
    (2, 4096, 2, 2, 10, 4096),             # whole runs of 64
    (3, 700, 400, 300, 7, 700),            # lists of one or two docs: remainders only
    (130, 5000, 20, 5, 20, 1000),          # more rows than split merges, the width cuts rows
    (2, 5000, 1024, 1024, 33, 4000),       # the most probes
    (1, 40, 3, 1, 50, 64),                 # fewer slots than k
])
def test_layouts(dev, b, n, n_lists, n_probe, k, width):
    """Unfiltered, under a full-N mask and under exact clauses with several values a doc, a
    reverse clause and a value no doc may hold."""
    g = rng(310 + n + b)
    d, c, vals = 128, 3, 2
    items, offsets, sizes, perm = _ivf(g, n, d, n_lists)
    empty = g.random(n_lists) < 0.1  # lists cut to nothing
    sizes = np.where(empty, 0, sizes)
    q = g.standard_normal((b, d)).astype(np.float32)
    probes = np.stack([g.permutation(n_lists)[:n_probe] for _ in range(b)]).astype(np.int64)
    probes[0, -1] = n_lists + 3  # no such list
    args = (dev, q, probes, offsets, sizes, items, perm, 0.7, k, width)
    want_args = (q, probes, offsets, sizes, items, perm, [0.7], k, width)
    ids, sc = _run(*args)
    want = ost.search(*want_args)
    assert np.array_equal(ids, want[0]) and np.array_equal(sc, want[1])
    valid = g.random((b, n)) < 0.15
    valid[-1] = False
    ids, sc = _run(*args, filtering_bit_mask=_t(dev, _pack(valid)))
    want = ost.search(*want_args, valid=valid)
    assert np.array_equal(ids, want[0]) and np.array_equal(sc, want[1])
    attrs = g.integers(0, 4, (n, c, vals)).astype(np.int64)
    attrs[g.random((n, c, vals)) < 0.3] = -1
    qa = g.integers(0, 4, (b, c)).astype(np.int64)
    qa[g.random((b, c)) < 0.4] = -1
    qa[0, 0] = -7
    rev = np.array([False, True, False])
    exact = of.clause_match(attrs, rev, qa)
    slots = attrs.transpose(1, 2, 0).reshape(c * vals, n).astype(np.int32)
    kw = dict(item_clause_attrs=_t(dev, slots),
              clause_slots=_t(dev, vals * np.arange(c + 1, dtype=np.int64)),
              clause_is_reverse=_t(dev, rev))
    want = ost.search(*want_args, valid=exact)
    for dtype in (np.int64, np.int32):
        ids, sc = _run(*args, **kw, query_clause_attrs=_t(dev, qa.astype(dtype)))
        assert np.array_equal(ids, want[0]) and np.array_equal(sc, want[1])


@pytest.mark.parametrize("b,n_probe", [(1, 1), (5, 130), (130, 126), (130, 127)])
def test_bloom_payloads(dev, b, n_probe):
    """The probed columns' table from one kernel (up to 16,384 probe entries) and past it: Bloom
    plans with the recheck give the exact filter's result; lists that do not exist, empty lists
    and starts inside a column."""
    import retrieve_amd.st as st
    from retrieve_amd import bloom as bl

    g = rng(330 + b + n_probe)
    n, d, c, k, lists = 6000, 64, 2, 25, 200
    items, offsets, sizes, perm = _ivf(g, n, d, lists)
    sizes = np.where(g.random(lists) < 0.1, 0, sizes)
    q = g.standard_normal((b, d)).astype(np.float32)
    probes = np.stack([g.permutation(lists)[:n_probe] for _ in range(b)]).astype(np.int64)
    probes[0, 0] = lists
    attrs = g.integers(0, 5, (n, c, 1)).astype(np.int64)
    qa = g.integers(0, 5, (b, c)).astype(np.int64)
    rev = np.zeros(c, bool)
    words, boffs = torch.ops.st.bloom_index_build_fixed(*st.attrs_to_features(_t(dev, attrs)),
                                                        64, 3)
    blob, count, stack = st.prepare_plans(bl.queries_to_expressions(qa, rev), 7, dev)
    ids, sc = _run(dev, q, probes, offsets, sizes, items, perm, 0.3, k, n, bloom_index=words,
                   bloom_bundle_b_offsets=boffs, plans=blob, plan_count=count,
                   max_stack_size=stack, bloom_k=3, hash_k=7,
                   item_clause_attrs=_t(dev, attrs[:, :, 0].T.astype(np.int32)),
                   clause_slots=_t(dev, np.arange(c + 1, dtype=np.int64)),
                   clause_is_reverse=_t(dev, rev), query_clause_attrs=_t(dev, qa))
    want = ost.search(q, probes, offsets, sizes, items, perm, [0.3], k, n,
                      valid=of.clause_match(attrs, rev, qa))
    assert np.array_equal(ids, want[0]) and np.array_equal(sc, want[1])


@pytest.mark.parametrize("end", ["n", "zero"])
def test_probe_past_the_sizes(dev, end):
    """CSR offsets hold one entry more than the sizes: a probe of that id names no list, with every
    filter form and above k = 1024. (The sizes are a view whose next entry, in the same
    allocation, is a large count.)"""
    import retrieve_amd.st as st
    from retrieve_amd import bloom as bl

    g = rng(340)
    n, d, b, c, lists = 6000, 64, 4, 2, 60
    items, offsets, sizes, perm = _ivf(g, n, d, lists)
    csr = _t(dev, np.append(offsets, n if end == "n" else 0))
    lens = _t(dev, np.append(sizes, 5000))[:lists]
    q = g.standard_normal((b, d)).astype(np.float32)
    probes = np.stack([g.permutation(lists)[:12] for _ in range(b)]).astype(np.int64)
    probes[:, 0] = lists
    attrs = g.integers(0, 3, (n, c, 1)).astype(np.int64)
    qa = g.integers(0, 3, (b, c)).astype(np.int64)
    rev = np.zeros(c, bool)
    exact = of.clause_match(attrs, rev, qa)
    words, boffs = torch.ops.st.bloom_index_build_fixed(*st.attrs_to_features(_t(dev, attrs)),
                                                        64, 3)
    blob, count, stack = st.prepare_plans(bl.queries_to_expressions(qa, rev), 7, dev)
    clauses = dict(item_clause_attrs=_t(dev, attrs[:, :, 0].T.astype(np.int32)),
                   clause_slots=_t(dev, np.arange(c + 1, dtype=np.int64)),
                   clause_is_reverse=_t(dev, rev), query_clause_attrs=_t(dev, qa))
    bloom = dict(bloom_index=words, bloom_bundle_b_offsets=boffs, plans=blob, plan_count=count,
                 max_stack_size=stack, bloom_k=3, hash_k=7)
    for valid, k, kw in ((None, 25, {}), (exact, 25, clauses), (exact, 25, {**bloom, **clauses}),
                         (exact, 25, dict(filtering_bit_mask=_t(dev, _pack(exact)))),
                         (None, 1100, {})):
        print(f"probe past the sizes end={end} k={k} {sorted(kw)}", flush=True)
        ids, sc = torch.ops.st.search(_t(dev, q), _t(dev, probes), csr, lens, _t(dev, items),
                                      _t(dev, perm), _t(dev, np.float32([0.3])), k, n, -1, **kw)
        want = ost.search(q, probes, offsets, sizes, items, perm, [0.3], k, n, valid=valid)
        assert np.array_equal(ids.cpu().numpy(), want[0])
        assert np.array_equal(sc.cpu().numpy(), want[1])


def test_values_below_minus_one(dev):
    """The C entry compares clause values as they are (only -1 is inactive): a query value below -1
    finds the docs that hold it; torch.ops.st.search takes such values for ones that none holds."""
    import retrieve_amd.st as st
    from retrieve_amd import _native as nat

    g = rng(350)
    n, d, b, k, lists = 3000, 64, 3, 30, 10
    items, offsets, sizes, perm = _ivf(g, n, d, lists)
    q = g.standard_normal((b, d)).astype(np.float32)
    probes = np.stack([g.permutation(lists)[:6] for _ in range(b)]).astype(np.int64)
    vals = g.choice(np.array([-(2**31), -7, -2, 0, 3], np.int32), n)
    qa = np.array([[-7], [-2], [-(2**31)]], np.int32)
    rev = np.zeros(1, bool)
    cs = np.array([0, 1], np.int64)
    t = [_t(dev, x) for x in (q, items, probes, offsets, sizes, perm, vals[None], cs,
                              rev.astype(np.int8), qa, np.float32([0.3]))]
    tq, ti, tp, to, ts, tperm, tv, tcs, trev, tqa, tgs = t
    codes, scales = st.quantize_rows(tq)
    ids = torch.empty((b, k), dtype=torch.int64, device=dev)
    sc = torch.empty((b, k), dtype=torch.float32, device=dev)
    lib = nat.lib()
    width = (n + 31) // 32 * 32
    ws = nat.workspace(lib.rt_ivf_search_workspace(b, width, k), dev)
    print("clause values below -1 through the C entry", flush=True)
    nat.check(lib.rt_ivf_search_payload_filters(
        nat.ptr(codes), nat.ptr(scales), b, nat.ptr(ti), n, d, nat.ptr(tp), 6, nat.ptr(to),
        nat.ptr(ts), lists, width, None, None, None, 0, 0, nat.ptr(tv), 1, nat.ptr(tcs), 1,
        nat.ptr(trev), nat.ptr(tqa), -1, nat.ptr(tperm), n, nat.ptr(tgs), k, nat.ptr(ids),
        nat.ptr(sc), nat.ptr(ws), ws.numel(), nat.stream(dev)))
    want = ost.search(q, probes, offsets, sizes, items, perm, [0.3], k, n,
                      valid=vals[None] == qa)
    assert np.array_equal(ids.cpu().numpy(), want[0]) and np.array_equal(sc.cpu().numpy(), want[1])
    lowest = np.broadcast_to(vals[None] == -(2**31), (b, n))
    want = ost.search(q, probes, offsets, sizes, items, perm, [0.3], k, n, valid=lowest)
    for dtype in (torch.int32, torch.int64):
        got = _run(dev, q, probes, offsets, sizes, items, perm, 0.3, k, n, item_clause_attrs=tv,
                   clause_slots=tcs, clause_is_reverse=trev, query_clause_attrs=tqa.to(dtype))
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
