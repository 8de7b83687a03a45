"""Per-bin FEM statistics, which read a batch in chunks of positions: counts
around the chunk length against a direct evaluation, and rasters cut into
batches around it, whose outputs must not depend on the cut."""
import numpy as np
import pytest

from helpers import random_atoms

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


@pytest.mark.parametrize("count", [1, 2, 31, 32, 33, 64, 65, 97])
@pytest.mark.parametrize("n,dr", [(16, 0.7), (64, 0.3), (64, 0.2)])
def test_v_omega_of_given_waves(msf, ctx, count, n, dr):
    """V_omega of `count` waves from their own ring sums: N sum r^2 / (sum r)^2
    - 1 in extended precision.  Ring means of random magnitudes vary by 5 % or
    more, so V >= 2e-3 for two waves or more and the FP64 rounding of the mean
    (1e-16) reaches V as 1e-16 / sqrt(V) per position: 97 of them stay below
    1e-11."""
    rng = np.random.default_rng(count + 7 * n)
    g = msf.make_grid(n, n, 9.0, 9.0, 4.0, 200e3)
    w = rng.standard_normal((count, n, n)) + 1j * rng.standard_normal((count, n, n))
    w *= (0.5 + rng.random(count))[:, None, None]
    radial, cnt, v = ctx.fem_accumulate(g, msf.make_fem(dr), 0.002, w)
    r = radial.astype(np.longdouble)
    with np.errstate(all="ignore"):
        r = r / cnt
        m = r.mean(0)
        want = np.where(r.sum(0) == 0, 0, ((r - m) ** 2).mean(0) / (m * m)).astype(float)
    assert v.size > 0
    np.testing.assert_array_equal(np.isnan(v), np.isnan(want))
    np.testing.assert_allclose(v, want, rtol=1e-11, atol=1e-20)


@pytest.mark.parametrize("batch", [1, 7, 31, 32, 33, 50])
def test_statistics_do_not_depend_on_the_batches(msf, ctx, batch):
    q, Z = random_atoms(40, (10.0, 10.0, 5.0), seed=5, species=(14, 29))
    spec = ctx.specimen(msf.make_grid(64, 64, 10.0, 10.0, 5.0, 200e3), q, Z, 1.5)
    opt = msf.Optics(0, 1.2e7, 0.0, 400.0, 0.012)
    xp, yp = np.linspace(0.2, 9.0, 11), np.linspace(0.5, 9.3, 7)
    res = []
    try:
        for b in (77, batch):
            ctx.configure(batch=b)
            res.append(ctx.adfstem_fem(spec, opt, xp, yp, msf.make_fem(0.2),
                                       detector=msf.Detector(1, 0.03, 0.1, 0), correlograph=True,
                                       correlograph_each=True, pixel_images=True))
    finally:
        ctx.configure()
        spec.free()
    np.testing.assert_array_equal(res[1][0], res[0][0])
    assert res[0][1]["correlograph_avg"].size > 0
    for k in res[0][1]:
        np.testing.assert_array_equal(res[1][1][k], res[0][1][k])
