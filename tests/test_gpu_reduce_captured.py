"""Short reductions launch by launch and captured into a graph: the forms differ (one launch or two), the bits
do not."""
import numpy as np
import pytest

import streamparanumal_amd as spx
from streamparanumal_amd import device, streaming
from streamparanumal_amd.device import DeviceArray

pytestmark = pytest.mark.gpu

# around the limits of the one-launch form, captured (2560, 3072, 4096, 8192) and not (3584, 5120, 8192, 12288, 16384)
SIZES = [1, 1000, 2560, 2561, 3072, 3073, 3584, 3585, 4096, 4097, 5120, 5121, 8192, 8193, 10007, 12288, 12289, 16384]


def bits(a):
    return np.asarray(a, dtype=np.float64).view(np.uint64)


@pytest.mark.parametrize("mode", [spx.REDUCE_REFERENCE, spx.REDUCE_FAST])
@pytest.mark.parametrize("n", SIZES)
def test_captured_reductions(dev, oracle, n, mode):
    print("[case] captured reductions", n, mode, flush=True)
    p, Ap, x, r = (oracle.uniform(n, 3, j * n) for j in range(4))
    dp, dAp, dx, dr = (DeviceArray.from_numpy(v) for v in (p, Ap, x, r))
    red = streaming.Reducer(n, mode)
    for f in (lambda: red.norm(dp), lambda: red.dot(dp, dAp), lambda: red.cg_update(dAp, -0.37, dr),
              lambda: red.cg_full(0.37, dp, dAp, dx, dr)):
        dx.copy_from(x)
        dr.copy_from(r)
        f()
        want = red.value(), dx.to_numpy(), dr.to_numpy()
        graph = device.Graph.capture(f)
        for _ in range(3):  # several replays, eager work between them
            dx.copy_from(x)
            dr.copy_from(r)
            red.out.copy_from(np.array([-1.0]))
            graph.launch()
            device.finish()
            got = red.value(), dx.to_numpy(), dr.to_numpy()
            for a, b in zip(got, want):
                assert np.array_equal(bits(a), bits(b))
