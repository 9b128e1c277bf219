"""The warm-start network on grids whose sides are no multiples of the convolutions' bricks or of the
weight gradient's voxel tiles, with the fewest and the most input and output fields.

Tolerances as in test_gpu_unet.py: against the oracle with the device's bfloat16 roundings only the order of
FP32 sums and the roundings it turns differ, 2^-7 of a tensor's largest magnitude (2^-6 for a gradient, whose
terms are products of two rounded factors)."""
import numpy as np
import pytest

import test_gpu_unet as base

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import panslbm2_amd as pa

    return pa.Context(0)


@pytest.mark.parametrize("dims,cin,cout", [((20, 12, 4), 1, 1), ((4, 28, 12), 8, 16), ((36, 16, 20), 3, 13)])
def test_network_matches_oracle(ctx, dims, cin, cout):
    net, ref, p, x0, t, din, dout = base._setup(ctx, dims, cin, cout, 11)
    net.set_input(din)
    net.set_target(dout)
    net.forward()
    a = ref.forward(p, x0, bf=True)
    for name, c in list(base.CH.items()) + [("y", cout)]:
        got, want = net.read(name, c), a[name]
        err = np.abs(got - want).max() / max(np.abs(want).max(), 1e-30)
        assert err <= 2.0 ** -7, "%s: %.3e" % (name, err)
    loss = net.backward()
    g = net.grads()
    want_loss, gb = ref.grad(p, x0, t, bf=True)
    assert loss == pytest.approx(want_loss, rel=1e-3)
    for name, ci, co, taps, wo, bo in ref.layers:
        for lo, hi, what in ((wo, bo, "W"), (bo, bo + co, "b")):
            err = np.abs(g[lo:hi] - gb[lo:hi]).max() / max(np.abs(gb[lo:hi]).max(), 1e-30)
            assert err <= 2.0 ** -6, "%s.%s: %.3e" % (name, what, err)
    net.close()
