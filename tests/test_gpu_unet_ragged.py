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


def _tiles(V, taps, co, ci):
    """Tiles of the weight gradient's loop in each split of a level's V voxels: about 1024 workgroups over
    the taps, voxel ranges in multiples of 64, a tile of 128 to 512 voxels by the channels staged."""
    splits = max(1, min(-(-1024 // taps), -(-V // 64)))
    chunk = -(-(-(-V // splits)) // 64) * 64
    c = -(-co // 16) * 16 + -(-ci // 16) * 16
    return -(-chunk // (512 if c <= 32 else 256 if c <= 64 else 128))


@pytest.mark.parametrize("dims,coarsest", [((48, 44, 40), False), ((76, 72, 60), True)], ids=["finer", "all"])
def test_weight_gradient_over_several_tiles(ctx, dims, coarsest):
    """Splits of several tiles: the next tile's loads during this one's products, the LDS tiles used again,
    the halo voxels between tiles, a last tile that is not full.  48x44x40 gives every layer of the two
    finer levels at least two tiles, 76x72x60 those of the coarsest (64 channels) too."""
    cin, cout = 2, 3
    net, ref, p, x0, t, din, dout = base._setup(ctx, dims, cin, cout, 12)
    V = [dims[0] * dims[1] * dims[2] // 8 ** k for k in range(3)]
    level = {"e1a": 0, "e1b": 0, "d1a": 0, "d1b": 0, "e2a": 1, "e2b": 1, "d2a": 1, "d2b": 1, "e3a": 2, "e3b": 2}
    several = [n for n, ci, co, taps, _, _ in ref.layers if n in level and _tiles(V[level[n]], taps, co, ci) > 1]
    assert sorted(several) == sorted(n for n in level if level[n] < 2 or coarsest)
    net.set_input(din)
    net.set_target(dout)
    net.forward()
    loss = net.backward()
    g = net.grads()
    net.close()
    want_loss, gb = ref.grad(p, x0, t, bf=True)
    assert loss == pytest.approx(want_loss, rel=1e-3)
    for name, ci, co, taps, wo, bo in ref.layers:
        for lo, hi, what in ((wo, bo, "W"), (bo, bo + co, "b")):
            err = np.abs(g[lo:hi] - gb[lo:hi]).max() / max(np.abs(gb[lo:hi]).max(), 1e-30)
            assert err <= 2.0 ** -6, "%s.%s: %.3e" % (name, what, err)
