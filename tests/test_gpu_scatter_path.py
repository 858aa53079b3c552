"""Which way a scatter goes: the automatic choice, what a caller may choose, and the way back."""
import numpy as np
import pytest

import streamparanumal_amd as spx
from streamparanumal_amd import device, ogs
from streamparanumal_amd._lib import check, checkh, libspx, libspxhost
from streamparanumal_amd.device import DeviceArray

pytestmark = pytest.mark.gpu

LONG, SHORT = (5, 4, 3, 7), (5, 4, 3, 2)  # 0.71 and 0.32 rows per local node


def scatter(g, oracle, o, k, trans):
    rows = g.NlocalP if trans == spx.TRANS else g.NlocalT
    src, base = oracle.uniform(rows * k, 12), np.full(g.N * k, -7.0)
    dv = DeviceArray.from_numpy(base)
    g.scatter(dv, DeviceArray.from_numpy(src), k, trans)
    assert np.array_equal(dv.to_numpy(), o.scatter(src, base, k, trans))


def test_automatic_path_and_the_way_back(dev, oracle):
    print("[case] scatter path", LONG, flush=True)
    ids = ogs.hex_ids(*LONG)
    g, o = ogs.Ogs(ids), oracle.Ogs(ids)

    def ways():
        for k in (1, 4, 5):
            for trans in (spx.NOTRANS, spx.TRANS):
                scatter(g, oracle, o, k, trans)
        return [[g.scatter_path(k, t)[1] for k in (1, 4, 5)] for t in (spx.NOTRANS, spx.TRANS)]

    auto = [["local", "local", "tiles"], ["tiles"] * 3]
    assert g.scatter_path()[0] is None and ways() == auto
    for choice, way in ((True, "tiles"), (False, "local")):
        before = g.scatter_path()[0]
        g.set_scatter_path(choice)
        assert g.scatter_path()[0] is choice and ways() == [[way] * 3] * 2
        g.set_scatter_path(before)  # what was saved restores it
        assert g.scatter_path()[0] is None and ways() == auto
    for fmt, way in ((False, "rows"), (True, "tiles")):
        g.set_gather_format(None, fmt)
        assert ways() == [[way] * 3] * 2
        g.set_scatter_path(None)
        assert ways() == auto


def test_short_rows(dev, oracle):
    print("[case] scatter path", SHORT, flush=True)
    ids = ogs.hex_ids(*SHORT)
    g, o = ogs.Ogs(ids), oracle.Ogs(ids)
    for choice, way in ((None, "local"), (True, "tiles"), (None, "local")):
        g.set_scatter_path(choice)
        for k in (1, 5):
            scatter(g, oracle, o, k, spx.NOTRANS)
            assert g.scatter_path(k) == (choice, way)


def test_triangles_scatter_in_local_order(dev):
    g = ogs.Ogs.box("Tri", 12, 11, 1, 7, keep_ids=False)  # 0.7 rows per local node, but short runs
    print("[case] scatter path of triangles", flush=True)
    for choice in (None, True, None):
        g.set_scatter_path(choice)
        assert g.scatter_path(5)[1] == ("tiles" if choice else "local")


DTYPES = [np.float32, np.float64, np.int32, np.int64]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lanes,cap", [(64, 256), (64, 512), (256, 2048), (256, 700)])
@pytest.mark.parametrize("mesh", [LONG, SHORT])
def test_scatter_on_tiles_and_rows(dev, oracle, mesh, lanes, cap, dtype):
    """The sorted-run scatter and the CSR's, by name, on one-wave and full tiles."""
    print("[case] scatter on tiles", mesh, lanes, cap, np.dtype(dtype).name, flush=True)
    ids = ogs.hex_ids(*mesh)
    g, o = ogs.Ogs(ids), oracle.Ogs(ids)
    g.set_block_nnz(2048, gs_cap=cap)
    device.set_tuning("ogs_gs_srb", variant=2 if lanes == 64 else 0)
    try:
        for fmt, way in ((True, "tiles"), (False, "rows")):
            g.set_scatter_path(True)
            g.set_gather_format(None, fmt)
            for k in (1, 2, 3, 4, 5):
                for trans in (spx.NOTRANS, spx.TRANS):
                    rows = g.NlocalP if trans == spx.TRANS else g.NlocalT
                    src = np.floor(oracle.uniform(rows * k, 21) * 1000).astype(dtype)
                    base = np.floor(oracle.uniform(g.N * k, 22) * 1000).astype(dtype)
                    assert g.scatter_path(k, trans)[1] == way
                    dv = DeviceArray.from_numpy(base)
                    g.scatter(dv, DeviceArray.from_numpy(src), k, trans)
                    device.check_kernel_errors()
                    assert np.array_equal(dv.to_numpy(), o.scatter(src, base, k, trans)), (k, trans, way)
    finally:
        device.set_tuning("ogs_gs_srb", variant=-1)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k", [1, 2, 3, 4])
def test_unaligned_vectors_of_long_rows(dev, oracle, dtype, k):
    """Vectors off a 16-byte boundary keep the row tiles, but for two or three 4-byte fields."""
    print("[case] unaligned scatter of long rows", np.dtype(dtype).name, k, flush=True)
    ids = ogs.hex_ids(*LONG)
    g, o = ogs.Ogs(ids), oracle.Ogs(ids)
    size = np.dtype(dtype).itemsize
    src = np.floor(oracle.uniform(g.NlocalT * k, 21) * 1000).astype(dtype)
    base = np.floor(oracle.uniform(g.N * k, 22) * 1000).astype(dtype)
    want = o.scatter(src, base, k, spx.NOTRANS)
    dg, dv = DeviceArray(src.size + 4, dtype), DeviceArray(base.size + 4, dtype)
    for og in range(16 // size):
        for ov in range(16 // size):
            dg.copy_from(np.concatenate([np.zeros(og, dtype), src, np.zeros(4 - og, dtype)]))
            dv.copy_from(np.concatenate([np.zeros(ov, dtype), base, np.zeros(4 - ov, dtype)]))
            way = g.scatter_path(k, spx.NOTRANS, dtype, dg.offset(og), dv.offset(ov))[1]
            # og: a node of whole 16-byte words (K * size a multiple of 16) is read in them
            words = ov == 0 and (og == 0 or k * size % 16 != 0)
            assert way == ("local" if words or (size == 4 and k in (2, 3)) else "tiles"), (og, ov)
            checkh(libspxhost().spxh_ogs_scatter(g.h, device.ogs_type(np.dtype(dtype)), spx.NOTRANS, k, dg.offset(og),
                                                 dv.offset(ov)), "scatter")
            device.check_kernel_errors()
            assert np.array_equal(dv.to_numpy()[ov:ov + base.size], want), (og, ov)


@pytest.mark.parametrize("k", [2, 3])
def test_large_map_of_several_narrow_fields(dev, k):
    """Two and three 4-byte fields through a map past the size that is read non-temporally, ragged end and holes."""
    n = (160 << 18) + 5
    print("[case] scatter of narrow fields, large map", n, k, flush=True)
    g2l = (np.arange(n, dtype=np.int64) * 7919 % 100003).astype(np.int32)
    g2l[::1009] = -1
    gv = np.arange(100003 * k, dtype=np.float32)
    dv, dm, dg = (DeviceArray.from_numpy(a) for a in (np.full(n * k, -7.0, np.float32), g2l, gv))
    check(libspx().spx_ogs_scatter_inverse(spx.FLOAT, k, n, dm.ptr, dg.ptr, dv.ptr), "scatter")
    want = gv.reshape(-1, k)[np.maximum(g2l, 0)]
    want[g2l < 0] = -7.0
    assert np.array_equal(dv.to_numpy().reshape(-1, k), want)
