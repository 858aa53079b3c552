"""The caller's partials after a reduction: `tmp` holds stage 1's, whichever form ran."""
import numpy as np
import pytest

import streamparanumal_amd as spx
from streamparanumal_amd import streaming
from streamparanumal_amd._lib import check, libspx
from streamparanumal_amd.device import DeviceArray

pytestmark = pytest.mark.gpu


def bits(a):
    return np.asarray(a, dtype=np.float64).view(np.uint64)


@pytest.mark.parametrize("mode", [spx.REDUCE_REFERENCE, spx.REDUCE_FAST])
@pytest.mark.parametrize("n", [1, 255, 256, 1000, 5000, 5120, 8192, 16384, 16385])
def test_partials_are_left_in_tmp(dev, oracle, n, mode):
    print("[case] partials", n, mode, flush=True)
    p, Ap, x, r = (DeviceArray.from_numpy(oracle.uniform(n, 3, j * n)) for j in range(4))
    nb = -(-n // 256)  # below 65536 entries each lane has one, so FAST sums no two before the tree either
    red, want, out = streaming.Reducer(n, mode), DeviceArray(nb), DeviceArray(1)

    def partials(f):
        red.tmp.copy_from(np.full(red.tmp.n, -3.0))
        f()
        return red.tmp.read(0, nb)

    got = partials(lambda: red.norm(p))
    check(libspx().spx_bs3_1(nb, n, p.ptr, want.ptr, 256), "bs3_1")
    assert np.array_equal(bits(got), bits(want.to_numpy()))
    got = partials(lambda: red.dot(p, Ap))
    check(libspx().spx_bs4_1(nb, n, p.ptr, Ap.ptr, want.ptr, 256), "bs4_1")
    assert np.array_equal(bits(got), bits(want.to_numpy()))
    for f in (lambda: red.cg_update(Ap, -0.37, r), lambda: red.cg_full(0.37, p, Ap, x, r)):
        got = partials(f)
        check(libspx().spx_bs3_1(nb, n, r.ptr, want.ptr, 256), "bs3_1")  # the updated r's own sums
        assert np.array_equal(bits(got), bits(want.to_numpy()))
