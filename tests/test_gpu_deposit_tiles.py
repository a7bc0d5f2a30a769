"""The tiles the deposit takes by itself: one particle per thread for small
bunches in the caller's order, eight above; in cell order two, or eight for
many particles on large meshes.  Cell sums are integers, so every tile gives the same
bits as the table of option deposit_tile = 1, on both sides of the rule's line
and where a wavefront's lane pairs are half empty."""
import numpy as np
import pytest

from ocelot_amd.workloads import equal_charges, gaussian_bunch

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _bunch(n):
    from ocelot_amd import DeviceParticleArray, ParticleArray
    p = ParticleArray()
    p.rparticles, p.E = gaussian_bunch(n, seed=n), 0.13
    p.q_array = equal_charges(n, 250e-12) * np.random.default_rng(n).uniform(0.5, 1.5, n)
    return DeviceParticleArray.from_host(p, torch.cuda.current_device())


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [4, 63, 65, 257, 20_001, 150_000, 150_001, 333_333])
def test_default_tile_gives_the_table_bits(n, prec):
    from ocelot_amd import SpaceCharge, _lib
    dev = torch.cuda.current_device()
    out = []
    for tile, xcd in ((0, 0), (1, 0), (3, 1)):
        d = _bunch(n)
        _lib.set_option(dev, "deposit_tile", tile)
        _lib.set_option(dev, "deposit_xcd", xcd)
        try:
            SpaceCharge(nmesh_xyz=[15, 17, 19], precision=prec).apply(d, 0.1)
        finally:
            _lib.set_option(dev, "deposit_tile", 0)
            _lib.set_option(dev, "deposit_xcd", 0)
        out.append(d.rparticles.clone())
    assert torch.equal(out[0], out[1])
    assert torch.equal(out[0], out[2])


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [65, 1025, 50_001])
def test_cell_ordered_tile_gives_the_table_bits(n, prec):
    from ocelot_amd import SpaceCharge, _lib, track_drift
    dev = torch.cuda.current_device()
    out = []
    for tile in (0, 1):
        d = _bunch(n)
        _lib.set_option(dev, "deposit_tile", tile)
        try:
            track_drift(d, SpaceCharge(nmesh_xyz=[15, 17, 19], precision=prec), L=0.1, dz=0.1, nsteps=3)
        finally:
            _lib.set_option(dev, "deposit_tile", 0)
        out.append(d.rparticles.clone())
    assert torch.equal(out[0], out[1])
