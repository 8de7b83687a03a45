"""Which batches run their slices in one launch: on every compiled grid, from
the smallest batch that takes the loop on, with one to several slices and both
transmission products, the statistics name no column tile and the results have
the bits of the slice passes, which profiled runs and a batch of one position
less take."""
import numpy as np
import pytest

from helpers import Case, random_atoms

pytestmark = pytest.mark.gpu

# grid: positions of the smallest batch that takes the loop with 4 slices or more
GRIDS = {(64, 64): 1, (64, 96): 4, (96, 64): 4, (64, 128): 4, (128, 64): 4, (96, 96): 16,
         (64, 192): 64, (192, 64): 64, (96, 128): 64, (128, 96): 80, (64, 256): 128,
         (256, 64): 128, (128, 128): 128}
SHORT = {(64, 192): 100, (96, 128): 100, (128, 96): 100}  # with fewer


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("nx,ny", list(GRIDS))
def test_route_and_bits(msf, ctx, nx, ny, mode):
    for slices in (1, 2, 4):
        least = GRIDS[nx, ny] if slices >= 4 else SHORT.get((nx, ny), GRIDS[nx, ny])
        cell = (nx * 0.08, ny * 0.08, 2.0 * slices)
        q, Z = random_atoms(6 * slices, cell, seed=3 * nx + ny + slices, species=(14, 29))
        q[:, 2] = 2.0 * (np.arange(len(q)) // 6) + 0.1
        c = Case(nx=nx, ny=ny, cell=cell, voltage=200e3, q=q, Z=Z, min_slice=1.0, cs3=1.2e7,
                 defocus=350.0, alpha_max=0.02, adf=True, inner=0.03, outer=0.1, fem=True, dr=0.5,
                 transmit_mode=mode)
        spec = c.gpu_specimen(msf, ctx)
        assert spec.n_slices == slices

        def run(n, **cfg):
            ctx.configure(transmit_mode=mode, **cfg)
            xp, yp = np.linspace(0.0, 0.99, n) * cell[0], np.array([0.6]) * cell[1]
            out = ctx.adfstem(spec, c.optics(msf), xp, yp, detector=c.detector(msf),
                              fem=c.femcfg(msf))
            tile = ctx.stats()["col_tile"]
            return tile, out + (ctx.exit_waves(spec, c.optics(msf), xp, yp),)

        try:
            for n in (least, least + 3):
                tile, loop = run(n)
                assert tile == 0
                tile, again = run(n, graph=False)
                assert tile == 0
                tile, passes = run(n, profile_kernels=True)
                assert tile > 0
                for a, b, p in zip(loop, again, passes):
                    np.testing.assert_array_equal(a, p)
                    np.testing.assert_array_equal(b, p)
            if least > 1:
                tile, below = run(least - 1)
                assert tile > 0
                _, passes = run(least - 1, profile_kernels=True)
                for a, p in zip(below, passes):
                    np.testing.assert_array_equal(a, p)
            # a last batch below the smallest: not every batch took the loop
            if least > 1:
                tile, _ = run(least + least // 2, batch=least)
                assert tile > 0
        finally:
            ctx.configure()
        spec.free()
