"""Slice passes of every compiled length, on either axis: exit waves against
the oracle, and the same bits from every column tile, from one row or column
per workgroup and from full workgroups (each exchange pads its buffer in its
own way, which a wrong slot would show at once)."""
import numpy as np
import pytest

from helpers import Case, random_atoms, rel_l2

pytestmark = pytest.mark.gpu

LENGTHS = (16, 32, 64, 96, 128, 192, 256, 384, 512, 768, 1024)


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


@pytest.mark.parametrize("n,plan", [(n, 1) for n in LENGTHS] + [(256, 2), (512, 2), (1024, 2)])
def test_length_on_either_axis(msf, ctx, O, n, plan):
    for nx, ny in ((n, 32), (32, n)):
        cell = (nx * 0.09, ny * 0.09, 6.0)
        q, Z = random_atoms(18, cell, seed=nx + 5 * ny, species=(14, 29))
        q[:, 2] = 2.0 * (np.arange(18) // 6) + 0.1
        c = Case(nx=nx, ny=ny, cell=cell, voltage=200e3, q=q, Z=Z, min_slice=1.0, cs3=1.2e7,
                 defocus=300.0, alpha_max=0.03, adf=False, fem=False)
        xp, yp = np.array([0.4 * cell[0]]), np.array([0.3, 0.8]) * cell[1]
        _, (_, _, ex_o) = c.run_oracle(O, xp, yp, exit_waves=True)
        spec = c.gpu_specimen(msf, ctx)
        sh = msf.probe_shifts(c.grid(msf), xp, yp)
        many = np.concatenate([sh] * 20)  # fills the workgroups of every tile
        try:
            ctx.configure(fft_plan=plan)
            ex = ctx.exit_waves_shifted(spec, c.optics(msf), sh)
            for p in range(2):
                # FP32 waves: a few 1e-8 per radix stage and slice
                assert rel_l2(ex[p], ex_o[p]) < 2e-6
                assert rel_l2(np.abs(ex[p]) ** 2, np.abs(ex_o[p]) ** 2) < 1e-5
            for tile in (0, 4, 8, 16):
                ctx.configure(fft_plan=plan, col_tile=tile)
                w = ctx.exit_waves_shifted(spec, c.optics(msf), many).reshape(20, 2, nx, ny)
                np.testing.assert_array_equal(w, np.broadcast_to(ex, w.shape))
        finally:
            ctx.configure()
            spec.free()


@pytest.mark.parametrize("plan", [1, 2])
@pytest.mark.parametrize("batch", [6, 8])
def test_two_chains_of_1024_rows_take_the_bits_of_one(msf, ctx, plan, batch):
    # batches whose tiles fill the CUs, and a last one of fewer positions that does not
    nx, ny = 1024, 512
    cell = (nx * 0.09, ny * 0.09, 6.0)
    q, Z = random_atoms(18, cell, seed=nx + plan, species=(14, 29))
    q[:, 2] = 2.0 * (np.arange(18) // 6) + 0.1
    c = Case(nx=nx, ny=ny, cell=cell, voltage=200e3, q=q, Z=Z, min_slice=1.0, cs3=1.2e7,
             defocus=300.0, alpha_max=0.03, adf=True, fem=False)
    xp, yp = np.linspace(0.1, 0.9, 13) * cell[0], np.array([0.3]) * cell[1]
    spec, out = c.gpu_specimen(msf, ctx), []
    try:
        for chains in (1, 2):
            ctx.configure(autotune=-1, fft_plan=plan, batch=batch, chains=chains)
            out.append(ctx.adfstem(spec, c.optics(msf), xp, yp, detector=c.detector(msf)))
            assert ctx.stats()["chains"] == chains
    finally:
        ctx.configure()
        spec.free()
    np.testing.assert_array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("nx,places", [(192, 5), (256, 4)])
def test_column_tile_follows_the_rounds_of_a_launch(msf, ctx, nx, places):
    # 4 tiles of 16 columns a position: tiles of 8 from a launch that fills the
    # CUs to one of two rounds, and the bits of 16-column tiles
    ny = 96
    cell = (nx * 0.09, ny * 0.09, 4.0)
    q, Z = random_atoms(12, cell, seed=nx, species=(14, 29))
    q[:, 2] = 2.0 * (np.arange(12) // 6) + 0.1
    c = Case(nx=nx, ny=ny, cell=cell, voltage=200e3, q=q, Z=Z, min_slice=1.0, cs3=1.2e7,
             defocus=300.0, alpha_max=0.03, adf=True, fem=False)
    spec, line = c.gpu_specimen(msf, ctx), 2 * 256 * places // 4
    try:
        for n, tile in ((63, 1), (64, 8), (line - 1, 8), (line, 16)):
            xp, yp, img = np.linspace(0.05, 0.95, n) * cell[0], np.array([0.4]) * cell[1], []
            for t in (0, 16):
                ctx.configure(autotune=-1, batch=n, col_tile=t)
                img.append(ctx.adfstem(spec, c.optics(msf), xp, yp, detector=c.detector(msf))[0])
                assert ctx.stats()["col_tile"] == (t or tile)
            np.testing.assert_array_equal(img[0], img[1])
    finally:
        ctx.configure()
        spec.free()
