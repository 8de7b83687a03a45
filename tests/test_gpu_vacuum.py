"""Vacuum waves of the slices, formed on the aperture's bounding box and
transformed for many slices at once: boxes from one pixel to the whole grid,
rectangles, one slice, and more slices than one pass of the work array takes."""
import numpy as np
import pytest

from helpers import Case, random_atoms, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


# (nx, ny, pixel, slices, aperture [rad]); at 300 kV the band limit of a
# 0.08 A pixel is 82 mrad and the corner of the grid lies at 174 mrad
@pytest.mark.parametrize("nx,ny,px,slices,alpha", [
    (16, 16, 0.3, 1, 0.003),      # the beam's own pixel only
    (16, 32, 0.3, 3, 0.30),       # the whole grid
    (64, 64, 0.08, 4, 0.30),
    (96, 64, 0.08, 6, 0.05),
    (64, 192, 0.08, 5, 0.085),    # beyond the band limit, not the whole grid
    (128, 128, 0.08, 3, 0.012),
    (384, 128, 0.08, 2, 0.02),
    (768, 768, 0.08, 5, 0.30),    # 9 MB a plane: two passes of the work array
])
def test_exit_waves_over_apertures(msf, ctx, O, nx, ny, px, slices, alpha):
    cell = (nx * px, ny * px, 2.0 * slices)
    q, Z = random_atoms(3 * slices, cell, seed=nx + ny, species=(14, 29))
    q[:, 2] = 2.0 * (np.arange(len(q)) // 3) + 0.1
    c = Case(nx=nx, ny=ny, cell=cell, voltage=300e3, q=q, Z=Z, min_slice=1.0, cs3=1.0e7,
             defocus=300.0, alpha_max=alpha, adf=False, fem=False)
    xp, yp = np.array([0.3 * cell[0]]), np.array([0.1 * cell[1], 0.7 * cell[1]])
    yp = yp if nx < 512 else yp[:1]
    spec_o, (_, _, ex_o) = c.run_oracle(O, xp, yp, exit_waves=True)
    spec = c.gpu_specimen(msf, ctx)
    assert spec.n_slices == slices
    ex = ctx.exit_waves(spec, c.optics(msf), xp, yp)
    spec.free()
    # the wave is propagated in FP32: a few 1e-8 per transform stage and slice
    for p in range(ex.shape[0]):
        assert rel_l2(ex[p], ex_o[p]) < 2e-6
        assert rel_l2(np.abs(ex[p]) ** 2, np.abs(ex_o[p]) ** 2) < 1e-5
