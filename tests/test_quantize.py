"""The quantizers and the 1-bit packing at the edges of their lane groups: row lengths around
each group's width, rows past the last workgroup's, tables off the 16-byte alignment, and values
at the ends of the float range, bit for bit against the oracle."""

import numpy as np
import pytest
import torch

from oracle import quantize as oq

from conftest import rng


def _table(g, n, d):
    """Rows of spread scales, with zeros, halves of a code, tiny and huge magnitudes."""
    x = (g.standard_normal((n, d)) * np.exp(3 * g.standard_normal((n, 1)))).astype(np.float32)
    x[0] = 0.0
    if n > 1:
        x[1] = np.float32(1e-42) * g.integers(-3, 4, d)
    if n > 2:
        x[2] = np.float32(3e38) * g.uniform(-1, 1, d)
    if n > 3:
        x[3] = g.integers(-254, 255, d) * np.float32(0.5)
        x[3, 0] = 127.0
    return np.ascontiguousarray(x)


def test_quotient_rounds_once():
    """fp32(fp64(x) / fp64(a)) * 127 rounded to a whole code is what the fp32 quotient gives: the
    kernels divide in fp32."""
    g = rng(40)
    x = np.concatenate([g.standard_normal(2_000_000), g.uniform(-1, 1, 1_000_000) * 1e-30,
                        g.uniform(-1, 1, 1_000_000) * 3e38]).astype(np.float32)
    a = np.maximum(np.abs(x) * np.float32(1) + np.exp(10 * g.standard_normal(x.size)),
                   1e-8).astype(np.float32)
    a = np.minimum(a, np.float32(3.4e38))
    twice = (x.astype(np.float64) / a.astype(np.float64)).astype(np.float32)
    once = x / a
    same = (twice == once) | (np.abs(once) < np.finfo(np.float32).tiny)
    assert same.all()
    assert np.array_equal(np.rint(twice * np.float32(127)), np.rint(once * np.float32(127)))


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("n,d", [(1, 4), (17, 60), (33, 64), (9, 68), (5, 128), (7, 132), (3, 256),
                                 (6, 260), (4, 1024), (4, 1028), (5, 2048), (4, 2052), (40, 7),
                                 (140_001, 32)])
def test_rows(n, d, offset):
    import retrieve_amd.hip  # noqa: F401

    print(f"quantize_int8 n={n} d={d} offset={offset}", flush=True)
    x = _table(rng(n + d), n, d)
    flat = torch.zeros(n * d + offset, device="cuda:0")
    flat[offset:] = torch.from_numpy(x).reshape(-1).to("cuda:0")
    codes, scales = torch.ops.retrieve_amd.quantize_int8(flat[offset:].view(n, d))
    want_c, want_s = oq.quantize_int8(x, divide=True)
    assert np.array_equal(codes.cpu().numpy(), want_c)
    assert np.array_equal(scales.cpu().numpy(), want_s)


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("n,d", [(1, 4), (33, 64), (9, 68), (5, 128), (7, 132), (6, 260),
                                 (4, 1028), (4, 2052), (40, 7), (140_001, 32)])
def test_global(n, d, offset):
    import retrieve_amd.hip  # noqa: F401

    print(f"quantize_int8_global n={n} d={d} offset={offset}", flush=True)
    g = rng(n * 3 + d)
    x = g.standard_normal((n, d)).astype(np.float32)
    flat = torch.zeros(n * d + offset, device="cuda:0")
    flat[offset:] = torch.from_numpy(x).reshape(-1).to("cuda:0")
    perm = g.permutation(n)
    for rows in (None, perm):
        codes, abs_max = torch.ops.retrieve_amd.quantize_int8_global(
            flat[offset:].view(n, d), None if rows is None else torch.from_numpy(rows).to("cuda:0"))
        want_c, want_m = oq.quantize_int8_global(x, rows)
        assert np.array_equal(codes.cpu().numpy(), want_c)
        assert abs_max.cpu().numpy()[0] == want_m


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("n,d", [(1, 64), (67, 64), (5, 128), (9, 192), (3, 256), (6, 320),
                                 (4, 512), (5, 1024), (3, 2048), (140_003, 64)])
def test_oporp(n, d, offset):
    """The fused sketch and packing against the sketch's own steps in torch, with rows of zeros,
    denormals, huge values (an infinite norm), NaN and infinities."""
    from retrieve_amd.modules import _oporp_sketch

    print(f"oporp n={n} d={d} offset={offset}", flush=True)
    g = rng(n * 5 + d)
    x = _table(g, n, d)
    if n > 5:
        x[4, d // 2] = np.nan
        x[5, 1] = np.inf
        x[5, 2] = -np.inf
    flat = torch.zeros(n * d + offset, device="cuda:0")
    flat[offset:] = torch.from_numpy(x).reshape(-1).to("cuda:0")
    xt = flat[offset:].view(n, d)
    signs = torch.from_numpy(g.choice([-1, 1], d).astype(np.int8)).to("cuda:0")
    perm = torch.from_numpy(g.permutation(d)).to("cuda:0")
    got = torch.ops.retrieve_amd.pack_signs(xt, signs, perm)
    want = torch.ops.retrieve_amd.pack_signs(_oporp_sketch(xt, signs, perm, d))
    assert torch.equal(got, want)
    assert np.array_equal(got.cpu().numpy(),
                          oq.pack_signs(_oporp_sketch(xt, signs, perm, d).cpu().numpy()))
