"""The reduction trees behind the frame, the mesh placement and the beam
moments, at particle counts on both sides of their edges: one wavefront, one
workgroup, one workgroup per CU, several particles per thread, and more
partials than one round of loads takes."""
import numpy as np
import pytest

from ocelot_amd.workloads import equal_charges, gaussian_bunch
from oracle import sc_oracle as orc

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SIZES = [4, 63, 64, 65, 255, 256, 257, 511, 1025, 16_384, 65_535, 65_536, 65_537, 524_289, 1_200_001]


@pytest.mark.parametrize("n", SIZES)
def test_moments_and_mesh_match_numpy(n):
    """Means, second moments, the mesh's cell sizes and its offset.  A sum of
    n terms in a tree of at most 64 sequential additions per thread and about
    20 levels is within 100 eps of sum|x|/n of the exact mean: 1e-13 of a
    standard deviation times a margin of 10.  Cell sizes come from minima and
    maxima, which lose nothing but the frame's rounding."""
    from ocelot_amd import DeviceParticleArray, ParticleArray, SpaceCharge
    from ocelot_amd.envelope import moments
    r, q, E = gaussian_bunch(n, seed=n), equal_charges(n, 250e-12), 0.13
    p = ParticleArray()
    p.rparticles, p.q_array, p.E = r.copy(), q, E
    d = DeviceParticleArray.from_host(p, torch.cuda.current_device())
    v = moments(d)
    s = np.std(r, axis=1)
    assert v[0] == n
    assert abs(v[1] - q.sum()) <= 1e-12 * q.sum()
    assert abs(v[2] - r[5].mean()) <= 1e-12 * s[5]
    assert abs(v[7] - r[0].mean()) <= 1e-12 * s[0]
    assert abs(v[11] - r[4].mean()) <= 1e-12 * s[4]
    assert abs(v[12] - np.mean((r[0] - r[0].mean()) ** 2)) <= 1e-12 * s[0] ** 2
    assert abs(v[18] - np.mean((r[4] - r[4].mean()) ** 2)) <= 1e-12 * s[4] ** 2
    sc = SpaceCharge(nmesh_xyz=[15, 17, 19])
    sc.apply(d, 0.1)
    st, dbg = sc.last_stats(), {}
    orc.apply(r, q, E, 0.1, [15, 17, 19], debug=dbg)
    assert np.allclose(st["steps"], dbg["steps"], rtol=1e-12, atol=0)
    assert np.allclose(st["X_off"], dbg["X_off"], rtol=1e-11, atol=1e-11)
    assert abs(st["sumq"] - q.sum()) <= 1e-12 * q.sum()
