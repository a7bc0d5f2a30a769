"""Large meshes with few particles per cell: the default kick takes no bricks
there.  Its bits on both sides of the rule's lines, and its time against the
cell-ordered copy, which the FP64 form takes on such meshes."""
import numpy as np
import pytest

from ocelot_amd.workloads import equal_charges, gaussian_bunch

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

MESH = (128, 128, 129)  # 2113536 cells, just above 2^21


def _kick(d, mesh, prec, sort, dz=0.1, calls=1):
    """Kick with option apply_sort = sort; the calls' milliseconds."""
    from ocelot_amd import SpaceCharge, _lib
    dev = torch.cuda.current_device()
    old = _lib.get_option(dev, "apply_sort")
    _lib.set_option(dev, "apply_sort", sort)
    ms = []
    try:
        sc = SpaceCharge(nmesh_xyz=list(mesh), precision=prec)
        for _ in range(calls):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            sc.apply(d, dz)
            b.record()
            b.synchronize()
            ms.append(a.elapsed_time(b))
    finally:
        _lib.set_option(dev, "apply_sort", old)
    return ms


@pytest.mark.parametrize("prec,n", [("mixed", 1_056_767), ("mixed", 1_056_768), ("fp64", 999_999), ("fp64", 1_000_000)])
def test_both_sides_of_the_rule_give_the_same_bits(prec, n):
    from ocelot_amd import DeviceParticleArray
    r = torch.from_numpy(gaussian_bunch(n, seed=n)).cuda()
    q = torch.from_numpy(equal_charges(n, 250e-12) * np.random.default_rng(1).uniform(0.5, 1.5, n)).cuda()
    out = []
    for sort in (2, 1, 0):
        d = DeviceParticleArray(r.clone(), q, 0.13)
        _kick(d, MESH, prec, sort)
        out.append(d.rparticles)
    assert not torch.equal(out[0], r)
    assert torch.equal(out[0], out[1])
    assert torch.equal(out[0], out[2])


def test_few_particles_on_a_large_mesh_take_no_longer_than_the_cell_order():
    """3M / 255^3 FP64 took 1.3 times as long through bricks as on the copy."""
    from ocelot_amd import DeviceParticleArray
    n = 3_000_000
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    r = torch.randn((6, n), generator=g, device="cuda", dtype=torch.float64)
    r *= torch.tensor([1e-4, 1e-5, 1e-4, 1e-5, 1e-3, 1e-3], device="cuda", dtype=torch.float64)[:, None]
    d = DeviceParticleArray(r, torch.full((n,), 250e-12 / n, device="cuda", dtype=torch.float64), 0.13)
    t = {sort: float(np.median(_kick(d, (255,) * 3, "fp64", sort, 1e-6, 9))) for sort in (1, 2)}
    assert t[2] < 1.12 * t[1]
