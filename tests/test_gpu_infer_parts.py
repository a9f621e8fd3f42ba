"""Evaluations a lane a sample run in parts of whole rounds of the chip: the
values of evaluations of 65,536 samples at a time, below, at and above the
sizes where the number of parts changes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [393_215, 393_216, 524_288, 524_289, 1_572_865])
def test_lanes_in_parts_equal_short_calls(n):
    from neural_runner import Neural
    nn = Neural()
    rng = np.random.default_rng(n)
    F = rng.random((n, 8), np.float32)
    T = np.zeros((n, 3), np.float32)
    ds, small, net = nn.new_ds(n), nn.new_ds(65_536), nn.new_net(7)
    try:
        nn.ds_write(ds, F, T)
        want = []
        for at in range(0, n, 65_536):
            m = min(65_536, n - at)
            nn.ds_write(small, F[at:at + m], T[at:at + m])
            want.append(nn.infer(net, small, m, lanes=True).copy())
        for _ in range(2):
            assert np.array_equal(nn.infer(net, ds, n, lanes=True), np.concatenate(want))
    finally:
        nn.free_net(net)
        nn.free_ds(small)
        nn.free_ds(ds)
