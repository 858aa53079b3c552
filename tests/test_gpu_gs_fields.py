"""Gather+scatter of several fields per node on full-size tiles (8 positions per lane and more), where the
rows of two or more members are packed into lanes: every type and op, with the values that a row of one
member turns into others (-0 in a sum, infinities and NaN in a maximum or minimum)."""
import numpy as np
import pytest

import streamparanumal_amd as spx
from streamparanumal_amd import STORE_BF16, STORE_F32, device, ogs
from streamparanumal_amd.device import DeviceArray

pytestmark = pytest.mark.gpu

BOXES = {"hex7": ("Hex", 4, 3, 3, 7), "hex1": ("Hex", 9, 8, 7, 1), "tet3": ("Tet", 4, 4, 3, 3), "tri2": ("Tri", 23, 17, 1, 2)}


@pytest.fixture(scope="module")
def boxes(dev, oracle):
    out = {}
    for name, b in BOXES.items():
        ids = ogs.box_ids(*b)
        out[name] = (ogs.Ogs(ids), oracle.Ogs(ids))
    return out


def values(oracle, n, dtype, seed):
    u = oracle.uniform(n, seed)
    if np.dtype(dtype).kind != "f":
        return np.floor(u * 1000).astype(dtype)
    v = u.astype(dtype)
    v[::17] = -0.0
    v[5::1013] = np.nan
    v[7::509] = np.inf
    return v


def same(a, b):
    if a.dtype.kind != "f":
        return np.array_equal(a, b)
    bits = f"u{a.itemsize}"
    nan = np.isnan(b)
    return np.array_equal(np.isnan(a), nan) and np.array_equal(a[~nan].view(bits), b[~nan].view(bits))


@pytest.mark.parametrize("box", list(BOXES))
@pytest.mark.parametrize("k", [2, 3, 4])
@pytest.mark.parametrize("op", [spx.ADD, spx.MUL, spx.MAX, spx.MIN])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32, np.int64])
def test_gs_fields(boxes, oracle, box, k, op, dtype):
    print("[case] gs fields", box, k, op, np.dtype(dtype).name, flush=True)
    g, o = boxes[box]
    q = values(oracle, g.N * k, dtype, 5)
    for cap, trans in ((2048, spx.SYM), (1500, spx.SYM), (2048, spx.NOTRANS), (2048, spx.TRANS)):
        g.set_block_nnz(cap)
        dq = DeviceArray.from_numpy(q)
        g.gather_scatter(dq, k, op, trans)
        device.check_kernel_errors()
        assert same(dq.to_numpy(), o.gather_scatter(q, k, op, trans)), (cap, trans)


@pytest.mark.parametrize("box", list(BOXES))
@pytest.mark.parametrize("k", [2, 3, 4])
@pytest.mark.parametrize("st", [STORE_F32, STORE_BF16])
def test_gs_fields_mixed(boxes, oracle, box, k, st):
    print("[case] gs fields, mixed", box, k, st, flush=True)
    g, o = boxes[box]
    q = oracle.to_storage(oracle.uniform(g.N * k, 6), st)
    if st == STORE_F32:
        q[::17] = -0.0
    else:
        q[::17], q[5::1013], q[7::509] = 0x8000, 0xffc1, 0x7f80  # -0, a NaN, infinity
    for cap in (2048, 1500):
        g.set_block_nnz(cap)
        dq = DeviceArray.from_numpy(q)
        g.gather_scatter_mixed(dq, k)
        device.check_kernel_errors()
        want = oracle.gs_mixed(st, o.rowStartsT, o.colIdsT, q, k)
        bits = np.uint32 if st == STORE_F32 else np.uint16
        assert np.array_equal(dq.to_numpy().view(bits), want.view(bits)), cap
