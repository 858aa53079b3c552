"""The scatter through the local -> row map: its 16-byte form and the fallbacks, through the C ABI."""
import numpy as np
import pytest

import streamparanumal_amd as spx
from streamparanumal_amd import _lib, ogs
from streamparanumal_amd._lib import check, libspx
from streamparanumal_amd.device import DeviceArray

pytestmark = pytest.mark.gpu

TYPES = {np.float32: spx.FLOAT, np.float64: spx.DOUBLE, np.int32: spx.INT32, np.int64: spx.INT64}


def values(n, dtype, seed):
    return np.random.default_rng(seed).integers(-1000, 1000, n).astype(dtype)


def run(n, k, dtype, holes, shift_v=0, shift_gv=0, shift_map=0):
    rng = np.random.default_rng(n + 7 * k)
    rows = max(1, n // 3)
    g2l = rng.integers(0, rows, n).astype(np.int32)
    if holes:
        g2l[rng.random(n) < 0.2] = -1
    gv, v = values(rows * k + 4, dtype, 1), values(n * k + 8, dtype, 2)
    m = DeviceArray.from_numpy(np.concatenate([np.zeros(shift_map, np.int32), g2l]))
    dg, dv = DeviceArray.from_numpy(gv), DeviceArray.from_numpy(v)
    check(libspx().spx_ogs_scatter_inverse(TYPES[dtype], k, n, m.offset(shift_map), dg.offset(shift_gv),
                                           dv.offset(shift_v)), "scatter")
    want = v.copy()
    at = np.flatnonzero(g2l >= 0)
    for f in range(k):
        want[shift_v + at * k + f] = gv[shift_gv + g2l[at].astype(np.int64) * k + f]
    assert np.array_equal(dv.to_numpy(), want)


@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 511, 1024, 2047, 2049, 30011])
def test_scatter_words(dev, dtype, k, n):
    print("[case] scatter words", np.dtype(dtype).name, k, n, flush=True)
    for holes in (False, True):
        run(n, k, dtype, holes)


@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("k", [1, 2, 3, 4])
@pytest.mark.parametrize("shifts", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)])
def test_scatter_words_unaligned(dev, dtype, k, shifts):
    print("[case] scatter words unaligned", np.dtype(dtype).name, k, shifts, flush=True)
    run(4099, k, dtype, True, *shifts)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_scatter_words_large_map(dev, dtype):
    """A map past the size that is read non-temporally (160 MiB), with a ragged end."""
    n = (160 << 18) + 5
    print("[case] scatter words, large map", n, flush=True)
    run(n, 1, dtype, False)


@pytest.mark.parametrize("k", [1, 3])
def test_default_scatter_of_long_rows(dev, oracle, k):
    """A box with long rows: the default scatter, and the row blocks a caller may choose."""
    mesh = (5, 4, 3, 7)
    print("[case] default scatter", mesh, k, flush=True)
    ids = ogs.hex_ids(*mesh)
    g, o = ogs.Ogs(ids), oracle.Ogs(ids)
    gsrc = np.concatenate([oracle.uniform(g.NlocalT, 12, j) for j in range(k)])
    base = np.full(g.N * k, -7.0)
    want = o.scatter(gsrc, base, k, spx.NOTRANS)
    for by_rows in (None, True, False):
        if by_rows is not None:
            g.set_scatter_path(by_rows)
        dv, dg = DeviceArray.from_numpy(base), DeviceArray.from_numpy(gsrc)
        g.scatter(dv, dg, k, spx.NOTRANS)
        assert np.array_equal(dv.to_numpy(), want)
