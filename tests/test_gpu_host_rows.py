"""Host rows beside the six of the phase space (a tag per particle, say) stay as
they are and take no part in the kick, whatever the array's layout."""
import numpy as np
import pytest

from ocelot_amd.workloads import equal_charges, gaussian_bunch

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["C", "F", "strided"])
@pytest.mark.parametrize("rows", [7, 8])
def test_extra_rows(rows, layout):
    from ocelot_amd import ParticleArray, SpaceCharge
    n = 5001
    r6 = gaussian_bunch(n, seed=1)
    q = equal_charges(n, 250e-12) * np.random.default_rng(1).uniform(0.5, 1.5, n)
    ref = ParticleArray()
    ref.rparticles, ref.q_array, ref.E = r6.copy(), q, 0.13
    p = ParticleArray()
    big = np.zeros((rows, n + 3), order="F" if layout == "F" else "C")
    r = big[:, :n] if layout == "strided" else np.array(big[:, :n], order=layout)
    r[:6] = r6
    r[6:] = np.arange((rows - 6) * n).reshape(rows - 6, n)
    tags = r[6:].copy()
    p.rparticles, p.q_array, p.E = r, q, 0.13
    for _ in range(2):
        for a in (ref, p):
            SpaceCharge(nmesh_xyz=[31, 31, 31]).apply(a, 0.1)
    assert not np.array_equal(ref.rparticles, r6)
    assert np.array_equal(p.rparticles[:6], ref.rparticles)
    assert np.array_equal(p.rparticles[6:], tags)
