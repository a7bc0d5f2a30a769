"""One-shot kicks from the cached graph: replayed where the kick is on one queue
(meshes below 65536 cells, or option overlap = 0), launched one by one where the
kernel spectrum has a queue of its own, which a graph is slower at."""
import numpy as np
import pytest

from ocelot_amd.workloads import equal_charges, gaussian_bunch

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _bunch(n, seed):
    from ocelot_amd import DeviceParticleArray
    return DeviceParticleArray(torch.from_numpy(gaussian_bunch(n, seed=seed)).cuda(),
                               torch.from_numpy(equal_charges(n, 250e-12)).cuda(), 0.13)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("mesh,overlap,n", [((31, 30, 33), 1, 20_000), ((31, 30, 33), 1, 210_000),
                                            ((40, 40, 40), 1, 20_000), ((32, 32, 64), 1, 20_000),
                                            ((47, 47, 63), 0, 20_000)])
def test_replays_equal_launches(mesh, overlap, n, prec):
    """A bunch kicked twice, with half the step, with random-mesh draws, after
    another bunch and after a refused one, with a launch-free gap between."""
    from ocelot_amd import SpaceCharge, _lib
    dev = torch.cuda.current_device()
    saved = {k: _lib.get_option(dev, k) for k in ("apply_graph", "overlap")}
    outs = {}
    try:
        _lib.set_option(dev, "overlap", overlap)
        for mode in (0, 1):
            _lib.set_option(dev, "apply_graph", mode)
            np.random.seed(5)
            d, d2, db = _bunch(n, 1), _bunch(n - 77, 2), _bunch(n, 3)
            db.rparticles[0, 77] = float("nan")
            sc = SpaceCharge(nmesh_xyz=list(mesh), precision=prec)
            scr = SpaceCharge(nmesh_xyz=list(mesh), precision=prec, random_mesh=True)
            seq = []
            for proc, p, step in ((sc, d, 0.1), (sc, d, 0.1), (sc, d, 0.05), (scr, d, 0.1), (scr, d, 0.1),
                                  (sc, d2, 0.1), (sc, d, 0.1)):
                proc.apply(p, step)
                seq.append(p.rparticles.clone())
                torch.cuda.synchronize()
            with pytest.raises(ValueError):
                sc.apply(db, 0.1)
            sc.apply(d, 0.1)
            seq.append(d.rparticles.clone())
            outs[mode] = seq
    finally:
        for k, v in saved.items():
            _lib.set_option(dev, k, v)
    for i, (a, b) in enumerate(zip(outs[0], outs[1])):
        assert torch.equal(a, b), i


def _ms(d, sc, reps):
    ms = []
    for _ in range(reps):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        sc.apply(d, 1e-6)
        b.record()
        b.synchronize()
        ms.append(a.elapsed_time(b))
    return float(np.median(ms))


def test_default_kick_is_no_slower_than_its_launches():
    """2M / 95^3 FP64: 1.11 times as long from a graph."""
    from ocelot_amd import SpaceCharge, _lib
    dev, n = torch.cuda.current_device(), 2_000_000
    d, sc = _bunch(n, 4), SpaceCharge(nmesh_xyz=[95] * 3)
    assert _lib.get_option(dev, "apply_graph") == 1
    default = _ms(d, sc, 41)
    _lib.set_option(dev, "apply_graph", 0)
    try:
        direct = _ms(d, sc, 41)
    finally:
        _lib.set_option(dev, "apply_graph", 1)
    assert default < 1.06 * direct
