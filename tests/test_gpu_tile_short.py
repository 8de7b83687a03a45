"""Column tiles of short columns: 16 columns where 8 do not fill a wavefront
(lengths 16 and 32), also under two rounds, with the bits of tiles of 8."""
import numpy as np
import pytest

from helpers import Case, random_atoms

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


@pytest.mark.parametrize("nx,ny,tile", [(16, 64, 16), (16, 256, 16), (32, 32, 16), (32, 256, 16),
                                        (64, 32, 8), (96, 32, 8)])
def test_tile_under_two_rounds(msf, ctx, nx, ny, tile):
    cell = (nx * 0.09, ny * 0.09, 4.0)
    q, Z = random_atoms(12, cell, seed=nx + ny, species=(14, 29))
    q[:, 2] = 2.0 * (np.arange(12) // 6) + 0.1
    c = Case(nx=nx, ny=ny, cell=cell, voltage=200e3, q=q, Z=Z, min_slice=1.0, cs3=1.2e7,
             defocus=300.0, alpha_max=0.03, adf=True, fem=False)
    xp, yp = np.linspace(0.05, 0.95, 400) * cell[0], np.array([0.4]) * cell[1]
    spec, img = c.gpu_specimen(msf, ctx), []
    try:
        for t in (0, 8, 16):
            ctx.configure(autotune=-1, col_tile=t)
            img.append(ctx.adfstem(spec, c.optics(msf), xp, yp, detector=c.detector(msf))[0])
            assert ctx.stats()["col_tile"] == (t or tile)
    finally:
        ctx.configure()
        spec.free()
    for i in img[1:]:
        np.testing.assert_array_equal(i, img[0])
