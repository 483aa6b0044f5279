"""The C-ABI library loads and exports every symbol ``include/*.h`` declares; host-side argument
checks fail before any GPU call. No compute is launched here."""

from __future__ import annotations

import ctypes
import glob
import os
import re
import subprocess

import pytest

from tests.conftest import ROOT

HEADERS = sorted(glob.glob(os.path.join(ROOT, "include", "*.h")))
DECL = re.compile(r"^[A-Za-z_][\w\s\*]*?\b(rt_\w+)\s*\(", re.M)


def declared() -> set[str]:
    names: set[str] = set()
    for h in HEADERS:
        text = open(h).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        names |= set(DECL.findall(text))
    return names


def test_headers_declare_entry_points():
    assert HEADERS and "rt_int8_scan_topk" in declared()


def test_library_exports_every_declared_symbol():
    from retrieve_amd import _native

    assert os.path.exists(_native.LIB_PATH), "build first: make -C retrieve_amd/csrc"
    out = subprocess.run(["nm", "-D", "--defined-only", _native.LIB_PATH], check=True,
                         capture_output=True, text=True).stdout
    exported = {line.split()[-1] for line in out.splitlines() if line.strip()}
    missing = declared() - exported
    assert not missing, f"declared but not exported: {sorted(missing)}"


def test_ctypes_table_covers_the_header():
    import torch  # noqa: F401  (the library binds to torch's HIP runtime)

    from retrieve_amd import _native

    assert set(_native.SIGNATURES) == declared()
    lib = _native.lib()
    for name in declared():
        assert isinstance(getattr(lib, name), ctypes._CFuncPtr)


def test_argument_errors_need_no_gpu():
    import torch  # noqa: F401

    from retrieve_amd import _native

    lib = _native.lib()
    # k = 0 is rejected before any HIP call
    st = lib.rt_int8_scan_topk(None, 1, None, 10, 64, 0, None, 0, None, None, None, 0, None)
    assert st == 1
    assert b"k must be" in lib.rt_last_error()
    with pytest.raises(ValueError, match="k must be"):
        _native.check(st)


def test_workspace_grows_with_batch():
    import torch  # noqa: F401

    from retrieve_amd import _native

    lib = _native.lib()
    small = lib.rt_int8_scan_topk_workspace(1, 30_000_000, 512, 100)
    big = lib.rt_int8_scan_topk_workspace(1024, 30_000_000, 512, 100)
    assert 0 < small <= big


def test_no_alloc_rejections_need_no_gpu():
    """The allocation-free int8 scan rejects null pointers before any device call. (Its
    rejection of a plan above the fixed scratch is tested with real device buffers, on the GPU,
    in ``tests/test_zz_no_alloc.py``: no call here passes an address that is not a buffer.)"""
    import torch  # noqa: F401

    from retrieve_amd import _native

    lib = _native.lib()
    st = lib.rt_int8_scan_topk_noalloc(None, 2, None, 10, 64, 5, None, 0, None, None, None)
    assert st == 1 and b"must not be null" in lib.rt_last_error()
    st = lib.rt_int8_scan_topk(None, 2, None, 10, 64, 5, None, 0, None, None, None, 0, None)
    assert st == 1 and b"null" in lib.rt_last_error()


def test_scan_workspaces_follow_the_rows():
    """A scan's lists are no longer than the rows they can meet: a query's lists hold about the
    table's rows once, whatever k is (a list a wave, one tile's room in each)."""
    import torch  # noqa: F401

    from retrieve_amd import _native

    lib = _native.lib()
    for n in (1000, 20_000, 100_000, 300_000):
        for b in (1, 16, 31, 200):
            for k in (10, 100, 1000):
                queries = -(-b // 32) * 32  # whole query groups of a wave
                rows = n + 64 * 8192  # (at most 8192 lists a query, a tile of up to 64 rows each)
                bound = queries * rows * 8 + (16 << 20)
                for need in (lib.rt_int8_scan_topk_workspace(b, n, 512, k),
                             lib.rt_dense_scan_topk_workspace(b, n, 128, k),
                             lib.rt_hamming_scan_topk_workspace(b, n, 2, k, 0)):
                    assert need <= bound, (n, b, k, need >> 20)
    # one query over a 51 MB table
    assert lib.rt_int8_scan_topk_workspace(1, 100_000, 512, 1000) <= 64 << 20
    assert lib.rt_int8_scan_topk_workspace(16, 100_000, 512, 100) <= 32 << 20


def test_candidate_workspaces_follow_the_candidates():
    """The candidate and IVF scans' lists hold about the row's candidates (or slots) once, whatever k
    is: at most 1024 lists a query, each up to two batches of 64 over its share."""
    import torch  # noqa: F401

    from retrieve_amd import _native

    lib = _native.lib()
    for b in (1, 8, 64, 256):
        for p in (100, 5000, 80_000, 1_000_000):
            for k in (10, 100, 1000):
                lists = 8 * b * (p + 1024 * 128)
                bound = lists + 8 * b * 8 * k + 12 * b * k + (4 << 20)
                assert lib.rt_cand_topk_workspace(b, p, k) <= bound, (b, p, k)
                assert lib.rt_ivf_search_workspace(b, p, k) <= bound, (b, p, k)
    # 80K candidates (or slots) of 16 queries at k = 1000
    assert lib.rt_cand_topk_workspace(16, 80_000, 1000) <= 24 << 20
    assert lib.rt_ivf_search_workspace(16, 80_000, 1000) <= 24 << 20


def test_popcount_scan_is_spread_where_it_pays():
    """A 1-bit scan of a table too small for a seed takes one workgroup a 1024 rows for one query
    and a small k (98 workgroups of four lists for 100K rows), and more for a large batch or k."""
    import torch  # noqa: F401

    from retrieve_amd import _native

    def need(b, n, k):
        return _native.lib().rt_hamming_scan_topk_workspace(b, n, 2, k, 0)

    assert need(1, 100_000, 10) <= 98 * 4 * 128 * 8 + (64 << 10)
    assert need(4, 100_000, 10) <= 4 * need(1, 100_000, 10)
    assert need(32, 100_000, 10) >= 32 * 390 * 4 * 64 * 8
    assert need(1, 100_000, 1000) >= 390 * 4 * 64 * 8
