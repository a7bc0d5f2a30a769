"""Kicks of numpy rows go through a pinned buffer of 32 MB: the same bits as
the device-resident kick on both sides of its size (six rows and the charges
are 7 n doubles up, 6 n down), and after a call that failed."""
import numpy as np
import pytest

from ocelot_amd.workloads import equal_charges, gaussian_bunch

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

WORDS = (32 << 20) // 8


@pytest.mark.parametrize("n", [4, 1000, WORDS // 7, WORDS // 7 + 1, WORDS // 6, WORDS // 6 + 1, 2 * WORDS // 7 + 3])
def test_host_rows_equal_device_rows(n):
    from ocelot_amd import DeviceParticleArray, ParticleArray, SpaceCharge
    r, q = gaussian_bunch(n, seed=n), equal_charges(n, 250e-12) * np.linspace(0.5, 1.5, n)
    p = ParticleArray()
    p.rparticles, p.q_array, p.E = r.copy(), q, 0.13
    d = DeviceParticleArray(torch.from_numpy(r).cuda(), torch.from_numpy(q).cuda(), 0.13)
    sc = SpaceCharge(nmesh_xyz=[15, 17, 19])
    for _ in range(2):
        rows = p.rparticles
        sc.apply(p, 0.1)
        sc.apply(d, 0.1)
        assert p.rparticles is rows
        assert np.array_equal(rows, d.rparticles.cpu().numpy())
    bad = ParticleArray()
    bad.rparticles, bad.q_array, bad.E = r.copy(), np.zeros(n), 0.13
    with pytest.raises(ValueError):
        sc.apply(bad, 0.1)
    assert np.array_equal(bad.rparticles, r)
    sc.apply(p, 0.1)
    sc.apply(d, 0.1)
    assert np.array_equal(p.rparticles, d.rparticles.cpu().numpy())
