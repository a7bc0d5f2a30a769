"""One-shot moments about a provisional centre: against extended precision, at
sizes around the 64 particles that the centre comes from, with the mean far
from zero, with windows and dispersion, and where the centre is no centre (an
outlier among the 64: the passes about the means run instead)."""
import numpy as np
import pytest

from ocelot_amd.workloads import equal_charges, gaussian_bunch

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

PAIRS = ((0, 0), (0, 1), (1, 1), (2, 2), (2, 3), (3, 3), (4, 4), (0, 2), (1, 3), (0, 3), (2, 1), (5, 5))


def _reference(r, disp=None, bounds=None, auto=False):
    """means and second moments in extended precision, x, px, y, py, tau, p"""
    r = r.astype(np.longdouble)
    if bounds is not None:
        m, s = r[4].mean(), r[4].std()
        r = r[:, (r[4] >= m + bounds[0] * s) & (r[4] <= m + bounds[1] * s)]
    x, px, y, py, tau, p = (v.copy() for v in r)
    if auto:
        dp = p - p.mean()
        disp = [(dp * (u - u.mean())).mean() / (dp * dp).mean() for u in (x, px, y, py)]
    if disp is not None:
        x, px, y, py = (u - d * p for u, d in zip((x, px, y, py), disp))
    f = 1 - p - p * p / 2 + px * px / 2 + py * py / 2
    u = np.stack((x, px * f, y, py * f, tau, p))
    mean = u.mean(axis=1)
    d = u - mean[:, None]
    return mean, [(d[a] * d[b]).mean() for a, b in PAIRS], d.std(axis=1)


def _check(r, **kw):
    """A sum of n terms in chains of at most 64 additions and about 20 tree
    levels is within 100 eps of sum |terms|; the centre at most doubles the
    terms: 5e-14 of the standard deviations, times a margin of 20."""
    from ocelot_amd import DeviceParticleArray, ParticleArray
    from ocelot_amd.envelope import moments
    n = r.shape[1]
    p = ParticleArray()
    p.rparticles, p.q_array, p.E = r.copy(), equal_charges(n, 250e-12), 0.13
    d = DeviceParticleArray.from_host(p, torch.cuda.current_device())
    v = moments(d, bounds=kw.get("bounds"), auto_disp=kw.get("auto", False), disp=kw.get("disp"))
    mean, mom, s = _reference(r, **kw)
    scale = s + 1e-3 * np.abs(mean)  # rounding of the coordinates themselves where the mean is large
    for got, k in ((v[2], 5), (v[7], 0), (v[8], 2), (v[9], 1), (v[10], 3), (v[11], 4)):
        assert abs(got - mean[k]) <= 1e-12 * scale[k]
    for k, (a, b) in enumerate(PAIRS):
        assert abs(v[12 + k] - mom[k]) <= 1e-12 * scale[a] * scale[b]


@pytest.mark.parametrize("n", [3, 63, 64, 65, 4097, 300_001])
@pytest.mark.parametrize("kw", [{}, {"bounds": [-1.0, 1.5]}, {"auto": True}, {"disp": (1e-3, 2e-4, -1e-3, 1e-4)},
                                {"bounds": [-1.0, 1.5], "auto": True}])
def test_against_extended_precision(n, kw):
    if n == 3 and kw.get("bounds"):
        kw = dict(kw, bounds=[-3.0, 3.0])
    _check(gaussian_bunch(n, seed=n), **kw)


@pytest.mark.parametrize("kw", [{}, {"bounds": [-1.0, 1.5]}, {"auto": True}])
def test_far_from_zero_and_far_centre(kw):
    n = 100_000
    r = gaussian_bunch(n, seed=1)
    r[0] += 50 * np.std(r[0])
    r[4] -= 70 * np.std(r[4])
    _check(r, **kw)
    for k in (0, 3, 5):  # particle 0 is one of the 64
        o = gaussian_bunch(n, seed=2)
        o[k, 0] += 4e4 * np.std(o[k])
        _check(o, **kw)


def test_no_spread():
    from ocelot_amd import DeviceParticleArray, ParticleArray
    from ocelot_amd.envelope import moments
    for n in (1, 5, 64, 1000):
        p = ParticleArray()
        p.rparticles = np.tile(gaussian_bunch(4, seed=3)[:, :1], (1, n))
        p.q_array, p.E = equal_charges(n, 1e-12), 0.13
        v = moments(DeviceParticleArray.from_host(p, torch.cuda.current_device()))
        assert v[0] == n
        assert np.all(np.abs(v[12:24]) <= 1e-28)
        assert np.all(v[[12, 14, 15, 17, 18, 23]] >= 0)
