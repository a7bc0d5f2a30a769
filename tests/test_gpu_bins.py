"""One-shot kicks in the caller's order: the deposit through bricks of cells
and the fields in the line layout against the kick on a cell-ordered copy
(which uses neither), bit for bit: cell sums are integers and the kick is per
particle.  Meshes with edges on both sides of a brick's and a line's, bunches
that fill one brick or a few, and every form the entry takes."""
import numpy as np
import pytest

from ocelot_amd.workloads import equal_charges, gaussian_bunch

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _rows(n, seed, outlier=0.0):
    r = gaussian_bunch(n, seed=seed)
    if outlier:  # two particles stretch the mesh, the others share a few cells
        for k in (0, 2, 4):
            r[k, 0] = outlier * np.std(r[k])
            r[k, 1] = -outlier * np.std(r[k])
    return r


def _kick(r, q, mesh, prec, sort, **kw):
    from ocelot_amd import DeviceParticleArray, SpaceCharge, _lib
    dev = torch.cuda.current_device()
    old = _lib.get_option(dev, "apply_sort")
    _lib.set_option(dev, "apply_sort", sort)
    try:
        d = DeviceParticleArray(r, q, 0.13)
        sc = SpaceCharge(nmesh_xyz=list(mesh), precision=prec, **kw)
        sc.prepare(None)
        for _ in range(2):
            sc.apply(d, 0.1)
    finally:
        _lib.set_option(dev, "apply_sort", old)
    return d.rparticles


def _both(r, q, mesh, prec, **kw):
    dev = torch.cuda.current_device()
    t = torch.from_numpy(r).to(f"cuda:{dev}")
    qt = torch.from_numpy(q).to(f"cuda:{dev}")
    a = _kick(t.clone(), qt, mesh, prec, 2, **kw)
    b = _kick(t.clone(), qt, mesh, prec, 1, **kw)
    assert torch.isfinite(a).all()
    assert not torch.equal(a, t)
    assert torch.equal(a, b)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("mesh", [(4, 4, 4), (15, 17, 16), (16, 33, 8), (9, 31, 95), (63, 63, 63), (96, 97, 98),
                                  (256, 16, 17), (17, 255, 24), (18, 19, 256), (8, 9, 300)])
def test_bricks_and_lines_give_the_bits_of_the_cell_order(mesh, prec):
    n = 450_001
    q = equal_charges(n, 250e-12) * np.random.default_rng(5).uniform(0.5, 1.5, n)
    _both(_rows(n, 5), q, mesh, prec)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [449_999, 450_000, 524_288, 2_200_003])
def test_bricks_over_sizes(n, prec):
    _both(_rows(n, n), equal_charges(n, 250e-12), (31, 63, 47), prec)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_large_mesh_and_many_tiles(prec):
    n = 4_500_000
    _both(_rows(n, 3), equal_charges(n, 250e-12), (127, 127, 127), prec)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("outlier", [60.0, 2000.0])
def test_concentrated_bunch(outlier, prec):
    n = 460_000
    _both(_rows(n, 11, outlier), equal_charges(n, 250e-12), (63, 62, 61), prec)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_random_mesh_row_stride_and_direct_launches(prec):
    from ocelot_amd import _lib
    n, dev = 455_000, torch.cuda.current_device()
    r, q = _rows(n, 2), equal_charges(n, 250e-12)
    _both(r, q, (31, 30, 29), prec, random_mesh=True)
    out = []
    for graph in (0, 1):
        wide = torch.zeros((6, n + 13), dtype=torch.float64, device=f"cuda:{dev}")
        wide[:, :n] = torch.from_numpy(r).to(wide.device)
        old = _lib.get_option(dev, "apply_graph")
        _lib.set_option(dev, "apply_graph", graph)
        try:
            out.append(_kick(wide[:, :n], torch.from_numpy(q).to(wide.device), (31, 30, 29), prec, 2).clone())
        finally:
            _lib.set_option(dev, "apply_graph", old)
        assert not wide[:, n:].any()
    assert torch.equal(out[0], out[1])
    t = torch.from_numpy(r).to(f"cuda:{dev}")
    assert torch.equal(out[0], _kick(t, torch.from_numpy(q).to(t.device), (31, 30, 29), prec, 1))


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("bad", ["nan", "charge"])
def test_refused_bunch_is_left_alone(bad, prec):
    n = 450_100
    r, q = _rows(n, 4), equal_charges(n, 250e-12)
    if bad == "nan":
        r[3, n // 2] = np.nan
    else:
        q[::2] *= -1  # total charge zero
    t = torch.from_numpy(r).cuda()
    with pytest.raises(ValueError):
        _kick(t, torch.from_numpy(q).cuda(), (31, 31, 31), prec, 2)
    assert torch.equal(torch.nan_to_num(t), torch.nan_to_num(torch.from_numpy(r).cuda()))
    # and the next bunch is kicked as ever
    _both(_rows(n, 6), equal_charges(n, 250e-12), (31, 31, 31), prec)
