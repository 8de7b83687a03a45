"""Batches of a run by the rule: two chains share an even number of three or
more from 384^2 on, at the edges of the 96 MiB that one batch may take, with
the bits of any other split."""
import numpy as np
import pytest

from helpers import Case, random_atoms

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


@pytest.mark.parametrize("n,positions,batches", [(384, 256, 2), (384, 257, 4), (384, 385, 4),
                                                 (256, 545, 3)])
def test_two_chains_share_an_even_number_of_batches(msf, ctx, n, positions, batches):
    cell = (n * 0.08, n * 0.08, 4.0)
    q, Z = random_atoms(12, cell, seed=n, species=(14, 29))
    q[:, 2] = 2.0 * (np.arange(12) // 6) + 0.1
    c = Case(nx=n, ny=n, cell=cell, voltage=200e3, q=q, Z=Z, min_slice=1.0, cs3=1.2e7,
             defocus=300.0, alpha_max=0.01, adf=True, inner=0.03, outer=0.1, fem=True, dr=0.5)
    xp, yp = np.linspace(0.02, 0.98, positions) * cell[0], np.array([0.4]) * cell[1]
    spec, out = c.gpu_specimen(msf, ctx), []
    try:
        for batch in (0, 50):
            ctx.configure(autotune=-1, batch=batch)
            out.append(ctx.adfstem(spec, c.optics(msf), xp, yp, detector=c.detector(msf),
                                   fem=c.femcfg(msf)))
            if batch == 0:
                assert ctx.stats()["n_batches"] == batches and ctx.stats()["chains"] == 2
    finally:
        ctx.configure()
        spec.free()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
