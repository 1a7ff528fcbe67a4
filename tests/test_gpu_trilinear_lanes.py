"""The two forms of the trilinear flow map: two lanes a particle below 2^31
samples, one lane from there up."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE = (48, 64, 32)  # of the samples that the particles meet; unit time steps
FRAMES = (1 << 31) // (64 * 32)  # with these the array holds 2^31 samples
LIMIT = 500  # steps: some solves continue the field far outside and stop there


@pytest.fixture(scope="module")
def samples():
    """U, V of FRAMES frames on the device, zero after the first SHAPE[0]."""
    import torch

    rng = np.random.default_rng(11)
    out = []
    for amp in (0.5, 0.4):
        a = torch.zeros((FRAMES,) + SHAPE[1:], dtype=torch.float64, device="cuda")
        a[:SHAPE[0]] = torch.as_tensor(rng.standard_normal(SHAPE) * amp, device="cuda")
        out.append(a)
    yield out
    out.clear()
    torch.cuda.empty_cache()


@pytest.mark.parametrize("spherical,extrap,lon", [
    (0, "constant", 0.0), (0, "nearest", 0.0), (1, "constant", 150.0), (2, "linear", 300.0)])
def test_two_lanes_give_the_bits_of_one(samples, spherical, extrap, lon):
    """The same first frames as a flow of their own (two lanes) and with so many
    more behind them that one lane runs: equal grids, point lists and batches
    (the grid's tiles and the queue, which hands a pair's two states on), with
    particles that leave the box, wrap the longitude and start outside."""
    from numbacs_amd import _lib, autotune
    from numbacs_amd.batch import FTLEBatch
    from numbacs_amd.flows import get_flow_linear_2D
    from numbacs_amd.integration import flowmap, flowmap_grid_2d_device

    nt, nx, ny = SHAPE
    y0 = 20.0 if spherical else 0.0
    box, T = ((lon, lon + nx - 1.0), (y0, y0 + ny - 1.0)), 20.0
    # (a longitude box past 180 stays in the grid's own numbers: what lies past
    # the wrap is outside the box)
    p = np.array([1.0])
    x = np.linspace(box[0][0] - 2.0, box[0][1] + 2.0, 37)
    y = np.linspace(box[1][0] - 1.0, box[1][1] + 1.0, 21)
    pts = np.stack(np.meshgrid(x[::3], y[::2], indexing="ij"), -1).reshape(-1, 2)

    def maps(f, precision):
        out = (_lib.empty((len(x), len(y), 2)), *(_lib.empty((len(x), len(y)), "i32")
                                                  for _ in range(2)))
        flowmap_grid_2d_device(f, 2.0, T, _lib.to_dev(x), _lib.to_dev(y), p, max_steps=LIMIT,
                               precision=precision, out=out[0], status=out[1], nsteps=out[2])
        return [_lib.to_host(a) for a in out]

    def results(frames):
        # (with this radius a velocity of one is about a degree a time unit)
        f = get_flow_linear_2D(((0.0, frames - 1.0, frames), box[0] + (nx,), box[1] + (ny,)),
                               *(s[:frames] for s in samples), spherical=spherical,
                               extrap_mode=extrap, r=60.0)
        got = {"points": flowmap(f, 2.0, T, pts, p, max_steps=LIMIT, return_status=True)}
        for precision in (0, 1):
            saved = autotune.get(3, precision)
            got["grid", precision] = maps(f, precision)
            for queue in (0, 4):
                autotune.set_config(3, precision, (1, 64, queue))
                try:
                    b = FTLEBatch(f, [dict(t0=2.0, T=T, x=x, y=y),
                                      dict(t0=5.0, T=T / 2, x=x[:9], y=y)],
                                  p, precision=("fp64", "fp32")[precision], ftle=False,
                                  max_steps=LIMIT).run()
                    got["batch", precision, queue] = [
                        r[k] for r in b.results() for k in ("flowmap", "status", "nsteps")]
                    got["queue", precision, queue] = maps(f, precision)
                    b.close()
                finally:
                    autotune.set_config(3, precision, saved)
        f.close()
        return got

    pair, one = results(nt), results(FRAMES)
    moved = np.abs(pair["grid", 0][0] - np.stack(np.meshgrid(x, y, indexing="ij"), -1)).max(-1)
    # (half of the wrapped boxes lies outside)
    assert (moved > 1.0).mean() > 0.2 and (pair["grid", 0][2] > 16).any()
    for form, want in one.items():
        for a, b in zip(pair[form], want):
            assert np.array_equal(a, b), form
