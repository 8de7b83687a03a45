"""Batches of more than one round of the compute units (256 positions): the
slice loop in one launch or the slice passes, whichever the line of the grid
says, alone and beside a second chain, with the same bits."""
import numpy as np
import pytest

from helpers import Case, random_atoms

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


def _runs(msf, ctx, nx, ny, n, **cfg):
    """(column tile, chains, image, V) of n positions as configured and by the passes."""
    cell = (nx * 0.08, ny * 0.08, 4.0)
    q, Z = random_atoms(12, cell, seed=nx + 2 * ny, species=(14, 29))
    q[:, 2] = 2.0 * (np.arange(12) // 6) + 0.1
    c = Case(nx=nx, ny=ny, cell=cell, voltage=200e3, q=q, Z=Z, min_slice=1.0, cs3=1.2e7,
             defocus=350.0, alpha_max=0.02, adf=True, inner=0.03, outer=0.1, fem=True, dr=0.5)
    spec, out = c.gpu_specimen(msf, ctx), []
    xp, yp = np.linspace(0.0, 0.99, n) * cell[0], np.array([0.3]) * cell[1]
    try:
        for kw in (cfg, dict(profile_kernels=True)):
            ctx.configure(autotune=-1, **kw)
            img, v = ctx.adfstem(spec, c.optics(msf), xp, yp, detector=c.detector(msf),
                                 fem=c.femcfg(msf))
            out.append((ctx.stats()["col_tile"], ctx.stats()["chains"], img, v))
    finally:
        ctx.configure()
        spec.free()
    return out


@pytest.mark.parametrize("nx,ny,n,loop", [
    (128, 128, 256, True), (128, 128, 257, False), (128, 128, 351, False), (128, 128, 352, True),
    (128, 128, 513, False), (128, 128, 640, True), (128, 96, 257, True), (128, 96, 513, False),
    (128, 96, 768, True), (64, 192, 513, False), (64, 192, 704, True), (96, 96, 512, True),
    (96, 96, 769, False), (96, 128, 513, False), (256, 64, 513, True), (64, 64, 1025, True)])
def test_rounds(msf, ctx, nx, ny, n, loop):
    a, b = _runs(msf, ctx, nx, ny, n, batch=n)
    assert a[1] == 1 and (a[0] == 0) == loop and b[0] > 0
    np.testing.assert_array_equal(a[2], b[2])
    np.testing.assert_array_equal(a[3], b[3])


@pytest.mark.parametrize("nx,ny,batch,n,loop", [
    (128, 128, 528, 1040, False), (128, 128, 656, 1300, False), (128, 128, 256, 1024, True),
    (96, 64, 256, 512, False), (64, 128, 256, 512, True), (64, 64, 100, 200, True),
    (128, 96, 256, 512, False), (256, 64, 300, 600, False), (256, 64, 250, 750, True)])
def test_two_chains(msf, ctx, nx, ny, batch, n, loop):
    a, b = _runs(msf, ctx, nx, ny, n, batch=batch, chains=2)
    assert a[1] == 2 and (a[0] == 0) == loop
    np.testing.assert_array_equal(a[2], b[2])
    np.testing.assert_array_equal(a[3], b[3])
