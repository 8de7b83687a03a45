"""The slice loop in one launch (small grids, waves kept in LDS) against the
slice passes, which profiled runs use: bit-identical images, statistics and
exit waves on every compiled grid, for both transmission products, one to
several slices, batches on either side of the smallest one that takes the
loop, and shifts at the wrap points; and against the oracle."""
import numpy as np
import pytest

from helpers import Case, random_atoms, rel_l2

pytestmark = pytest.mark.gpu

GRIDS = [(64, 64), (64, 96), (96, 64), (64, 128), (128, 64), (96, 96), (64, 192), (192, 64),
         (96, 128), (128, 96), (64, 256), (256, 64), (128, 128)]


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


def _case(nx, ny, slices, mode, seed):
    cell = (nx * 0.08, ny * 0.08, 2.0 * slices)
    q, Z = random_atoms(6 * slices, cell, seed=seed, species=(14, 29))
    q[:, 2] = 2.0 * (np.arange(len(q)) // 6) + 0.1
    return Case(nx=nx, ny=ny, cell=cell, voltage=200e3, q=q, Z=Z, min_slice=1.0, cs3=1.2e7,
                defocus=350.0, alpha_max=0.02, adf=True, inner=0.03, outer=0.1, fem=True, dr=0.5,
                transmit_mode=mode)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_loop_equals_passes(msf, ctx, nx, ny, mode):
    for slices, (npx, npy) in ((1, (1, 1)), (2, (2, 2)), (3, (13, 10)), (4, (1, 5))):
        c = _case(nx, ny, slices, mode, 7 * nx + ny + slices)
        spec = c.gpu_specimen(msf, ctx)
        assert spec.n_slices == slices
        # from the first pixel to the last, among them both sides of the middle
        xp = np.linspace(0.0, cell_end(c.cell[0], nx), npx)
        yp = np.linspace(0.0, cell_end(c.cell[1], ny), npy)
        res = []
        try:
            for prof in (False, True):
                ctx.configure(transmit_mode=mode, profile_kernels=prof)
                res.append(ctx.adfstem(spec, c.optics(msf), xp, yp, detector=c.detector(msf),
                                       fem=c.femcfg(msf)))
                res.append((ctx.exit_waves(spec, c.optics(msf), xp, yp), ()))
        finally:
            ctx.configure()
            spec.free()
        for a, b in zip(res[0] + res[1], res[2] + res[3]):
            np.testing.assert_array_equal(a, b)


def cell_end(period, n):
    return period - 0.9 * period / n


@pytest.mark.parametrize("nx,ny", [(64, 64), (96, 64), (64, 256), (128, 128)])
def test_loop_matches_oracle(msf, ctx, O, nx, ny):
    c = _case(nx, ny, 3, 0, nx + ny)
    xp = np.linspace(0.1, 0.9, 12) * c.cell[0]
    yp = np.linspace(0.2, 0.95, 11) * c.cell[1]
    _, (img_o, v_o, _) = c.run_oracle(O, xp, yp)
    spec = c.gpu_specimen(msf, ctx)
    img, v = ctx.adfstem(spec, c.optics(msf), xp, yp, detector=c.detector(msf), fem=c.femcfg(msf))
    ex = ctx.exit_waves(spec, c.optics(msf), xp, yp)
    _, (_, _, ex_o) = c.run_oracle(O, xp[:1], yp[:1], exit_waves=True)
    spec.free()
    assert rel_l2(img, img_o) < 1e-4 and rel_l2(v, v_o) < 1e-4
    assert rel_l2(np.abs(ex[0]) ** 2, np.abs(ex_o[0]) ** 2) < 1e-5
