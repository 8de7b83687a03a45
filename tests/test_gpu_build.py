"""Transmission functions from the fused FP64 passes against the oracle's
shift-sum: every compiled length on either axis, one to three species,
templates kept as half spectra and (support asymmetric at the Nyquist
frequency) as whole ones, domain minima off the origin, empty cells, and more
slices than one chunk of the work arrays takes."""
import numpy as np
import pytest

from helpers import random_atoms, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


@pytest.mark.parametrize("nx,ny,lx,ly,slices,species,origin", [
    (16, 16, 4.0, 4.0, 1, (14,), (0.0, 0.0)),
    (32, 16, 5.0, 3.0, 2, (14, 29), (0.0, 0.0)),
    (16, 64, 3.0, 6.0, 3, (6, 29, 40), (0.0, 0.0)),
    (64, 96, 8.0, 8.0, 2, (14, 29), (-1.5, 2.25)),
    (96, 96, 7.82, 7.82, 2, (29, 40), (0.0, 0.0)),   # support holds a Nyquist pixel
    (192, 128, 15.64, 12.0, 2, (14,), (0.7, 0.0)),
    (128, 192, 12.0, 15.64, 2, (14, 79), (0.0, 0.0)),
    (256, 384, 20.0, 30.0, 2, (14,), (0.0, 0.0)),
    (384, 256, 30.0, 20.0, 1, (29, 40), (0.0, 0.0)),
    (768, 64, 60.0, 5.0, 2, (14,), (0.0, 0.0)),
    (64, 768, 5.0, 60.0, 2, (14,), (0.0, 0.0)),
    (1024, 512, 80.0, 40.0, 8, (14, 29), (0.0, 0.0)),  # 19 MB a slice: two chunks
])
def test_transmission_matches_oracle(msf, ctx, O, nx, ny, lx, ly, slices, species, origin):
    cell = (lx, ly, 2.0 * slices)
    q, Z = random_atoms(4 * slices, cell, seed=nx + 3 * ny, species=species)
    q[:, 2] = 2.0 * (np.arange(len(q)) // 4) + 0.1
    q[:, 0] += origin[0]
    q[:, 1] += origin[1]
    job = O.make_job(nx=nx, ny=ny, xperiod=lx, yperiod=ly, zperiod=cell[2], voltage=200e3,
                     min_slice=1.0, xmin=origin[0], ymin=origin[1])
    so = O.Specimen(job, q, Z.astype(np.int32))
    sg = ctx.specimen(msf.make_grid(nx, ny, lx, ly, cell[2], 200e3, *origin), q, Z, 1.0)
    assert sg.n_slices == so.n_slices == slices
    for s in range(slices):
        # both are FP64 sums; the oracle adds a template per atom, the passes
        # transform: a few hundred rounding errors of 1e-16 of the peak
        assert rel_l2(sg.transmission(s), so.t_stack[s]) < 1e-11
    sg.free()


def test_empty_cell_is_vacuum(msf, ctx):
    sg = ctx.specimen(msf.make_grid(64, 32, 6.0, 3.0, 4.0, 200e3), np.zeros((0, 3)),
                      np.zeros(0, np.uint32), 1.0)
    assert sg.n_slices == 1
    np.testing.assert_allclose(sg.transmission(0), 1.0, atol=1e-14)
    sg.free()
