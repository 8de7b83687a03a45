"""Column tiles of a launch of less than two rounds of 16-column tiles: 8 columns
where it has the GPU to itself, 16 beside a second chain of batches, with the
same bits."""
import numpy as np
import pytest

from helpers import Case, random_atoms

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


@pytest.mark.parametrize("nx,ny", [(192, 96), (256, 96), (256, 256)])
def test_two_chains_keep_tiles_of_16(msf, ctx, nx, ny):
    cell = (nx * 0.09, ny * 0.09, 4.0)
    q, Z = random_atoms(12, cell, seed=nx + ny, species=(14, 29))
    q[:, 2] = 2.0 * (np.arange(12) // 6) + 0.1
    c = Case(nx=nx, ny=ny, cell=cell, voltage=200e3, q=q, Z=Z, min_slice=1.0, cs3=1.2e7,
             defocus=300.0, alpha_max=0.03, adf=True, fem=False)
    xp, yp = np.linspace(0.05, 0.95, 200) * cell[0], np.array([0.4]) * cell[1]
    spec, img = c.gpu_specimen(msf, ctx), []
    try:
        for chains, tile in ((1, 8), (2, 16)):
            ctx.configure(autotune=-1, batch=100, chains=chains)
            img.append(ctx.adfstem(spec, c.optics(msf), xp, yp, detector=c.detector(msf))[0])
            assert (ctx.stats()["chains"], ctx.stats()["col_tile"]) == (chains, tile)
    finally:
        ctx.configure()
        spec.free()
    np.testing.assert_array_equal(img[0], img[1])
