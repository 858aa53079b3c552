"""BS2-BS5 at the sizes where their kernels change form: the one-launch reductions, the last group of
loads of a lane, and the odd last entry of copy and axpy."""
import math

import numpy as np
import pytest

import streamparanumal_amd as spx
from streamparanumal_amd import streaming
from streamparanumal_amd.device import DeviceArray

pytestmark = pytest.mark.gpu

# around one wave's share (512 or 1024 entries), the one-launch limits (5120, 8192, 16384), and
# 65536 lanes with 1, 7 and 15 entries of a 16-entry group
SIZES = [1, 2, 63, 255, 256, 257, 511, 513, 1023, 1025, 4095, 5119, 5120, 5121, 8192, 8193, 10007, 16383, 16384, 16385,
         65536, 65537, 7 * 65536 + 300, 15 * 65536 + 1, 17 * 65536 - 1]


def bits(a):
    return np.asarray(a, dtype=np.float64).view(np.uint64)


@pytest.mark.parametrize("n", SIZES)
def test_reductions_match_the_reference_order(dev, oracle, n):
    print("[case] reductions", n, flush=True)
    p, Ap, x, r = (oracle.uniform(n, 3, j * n) for j in range(4))
    dp, dAp, dx, dr = (DeviceArray.from_numpy(v) for v in (p, Ap, x, r))
    red = streaming.Reducer(n, spx.REDUCE_REFERENCE, 256)
    red.norm(dp)
    assert bits([red.value()])[0] == bits([oracle.bs3_norm(p, 256)])[0]
    red.dot(dp, dAp)
    assert bits([red.value()])[0] == bits([oracle.bs4_dot(p, Ap, 256)])[0]
    ref, r_ref = oracle.bs5_update(Ap, -0.37, r, 256)
    red.cg_update(dAp, -0.37, dr)
    assert bits([red.value()])[0] == bits([ref])[0]
    assert np.array_equal(bits(dr.to_numpy()), bits(r_ref))
    v, x_ref, r_ref = oracle.bs5_full(0.37, p, Ap, x, r_ref)
    red.cg_full(0.37, dp, dAp, dx, dr)
    assert bits([red.value()])[0] == bits([v])[0]
    assert np.array_equal(bits(dx.to_numpy()), bits(x_ref))
    assert np.array_equal(bits(dr.to_numpy()), bits(r_ref))


@pytest.mark.parametrize("n", SIZES)
def test_fast_reductions(dev, oracle, n):
    """Compensated lane sums (2 roundings), then 8 + 8 tree steps, each at most half an ulp of the terms' sum."""
    print("[case] fast reductions", n, flush=True)
    a, b = oracle.uniform(n, 1), oracle.uniform(n, 1, n)
    da, db = DeviceArray.from_numpy(a), DeviceArray.from_numpy(b)
    red = streaming.Reducer(n, spx.REDUCE_FAST)
    for f, t in ((lambda: red.norm(da), a * a), (lambda: red.dot(da, db), a * b)):
        f()
        assert abs(red.value() - math.fsum(t)) <= 20 * 2.0**-53 * math.fsum(np.abs(t))


@pytest.mark.parametrize("n", [1, 2, 3, 511, 2047, 2048, 2049, 10007, 65537])
def test_odd_last_entry(dev, oracle, n):
    print("[case] copy, axpy", n, flush=True)
    x, y = oracle.uniform(n + 1, 1), oracle.uniform(n + 1, 1, n)
    dx, dy, dc = DeviceArray.from_numpy(x), DeviceArray.from_numpy(y), DeviceArray.from_numpy(y)
    streaming.axpy(0.37, dx, -1.21, dy, n)
    streaming.copy(dx, dc, n)
    want = y.copy()
    want[:n] = oracle.bs2_axpy(0.37, x[:n], -1.21, y[:n])
    assert np.array_equal(bits(dy.to_numpy()), bits(want))
    want[:n] = x[:n]
    assert np.array_equal(bits(dc.to_numpy()), bits(want))
