"""FEM statistics through the detector MTF on the fused FP64 passes, over
lengths of either axis and bands that fill their tiles unevenly, with and
without an ADF image beside them."""
import numpy as np
import pytest

from helpers import Case, random_atoms, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


@pytest.mark.parametrize("nx,ny,px,adf", [
    (32, 16, 0.25, False), (16, 64, 0.2, True), (64, 96, 0.1, False), (128, 32, 0.1, True),
    (96, 192, 0.08, True), (256, 64, 0.08, False), (384, 128, 0.08, False), (64, 512, 0.08, True),
    (768, 32, 0.08, False), (32, 1024, 0.08, False),
])
def test_fem_through_mtf(msf, ctx, O, nx, ny, px, adf):
    cell = (nx * px, ny * px, 4.0)
    q, Z = random_atoms(40, cell, seed=nx * 3 + ny, species=(14, 29))
    # apertures of a few k-space pixels of the shorter side
    alpha = 2.6 * 0.0251 / min(cell[:2])
    c = Case(nx=nx, ny=ny, cell=cell, voltage=200e3, q=q, Z=Z, min_slice=1.5, cs3=1.2e7,
             defocus=400.0, alpha_max=alpha, adf=adf, inner=0.02, outer=0.1, fem=True, dr=0.4,
             mtf=[1.0, 0.8, 0.5, 0.2], mtf_domain=[0.0, 0.3, 0.7, 3.0], mtf_rate=20.0)
    xp, yp = np.linspace(0.1, 0.9, 3) * cell[0], np.linspace(0.05, 0.8, 2) * cell[1]
    job = c.oracle_job(O)
    img_o, v_o = O.adfstem_fem(job, O.Specimen(job, c.q, c.Z.astype(np.int32)), xp, yp)
    spec = c.gpu_specimen(msf, ctx)
    img, v = ctx.adfstem_fem(spec, c.optics(msf), xp, yp, c.femcfg(msf), detector=c.detector(msf))
    spec.free()
    # FP32 waves: ring means to a few 1e-7, so their variance over positions
    # (V >= 1e-3 of the squared mean) to a few 1e-5 of itself
    for m in ("v_omega", "vbar_r", "v_re"):
        assert rel_l2(v[m], v_o[m]) < 1e-4, m
    if adf:
        assert rel_l2(img, img_o) < 1e-4
