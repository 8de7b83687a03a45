"""Exit waves to the host: sizes on either side of one pinned block and of its
parts, several batches (copied beside the next batch's slices) and one, rows
with zeros between the kept columns, two threads at once, and memory that was
not zero before."""
import ctypes as C
import threading

import numpy as np
import pytest

from helpers import random_atoms

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def msf():
    import msf as m
    m.lib()
    return m


def _spec(msf, ctx, nx, ny, seed=3):
    L = (nx * 0.08, ny * 0.08, 2.0)
    q, Z = random_atoms(30, L, seed=seed, species=(14, 29))
    return ctx.specimen(msf.make_grid(nx, ny, *L, 200e3), q, Z, 1.0)


def _run(msf, ctx, spec, shifts):
    """msf_exit_waves_shifted into memory filled with NaN."""
    sh = np.ascontiguousarray(shifts, np.int32)
    out = np.full((len(sh), spec.grid.nx, spec.grid.ny), np.nan + 1j * np.nan, np.complex64)
    opt = msf.Optics(0, 1.2e7, 0.0, 300.0, 0.02)
    ctx._check(msf.lib().msf_exit_waves_shifted(
        ctx._h, spec._h, C.byref(opt), sh.ctypes.data_as(C.POINTER(C.c_int32)), len(sh),
        out.ctypes.data_as(C.POINTER(C.c_float))), "exit")
    return out


# bytes of the compact waves: under one small block (256 KB), just over it, one
# to two parts (4 MB) of a large block, and more parts than it has slots (16 MB)
@pytest.mark.parametrize("nx,ny,count", [(64, 64, 1), (64, 64, 10), (64, 64, 11), (96, 384, 6),
                                         (256, 256, 11), (256, 256, 13), (512, 512, 17)])
def test_waves_do_not_depend_on_the_way_they_are_copied(msf, ctx, nx, ny, count):
    spec = _spec(msf, ctx, nx, ny)
    rng = np.random.default_rng(count)
    sh = np.stack([rng.integers(0, nx, count), rng.integers(0, ny, count)], 1)
    whole = _run(msf, ctx, spec, sh)
    assert np.isfinite(whole).all()
    one = np.concatenate([_run(msf, ctx, spec, s[None]) for s in sh])
    np.testing.assert_array_equal(whole, one)
    try:
        for batch, chains in ((3, 0), (4, 1), (5, 2), (1, 3)):
            ctx.configure(batch=batch, chains=chains)
            np.testing.assert_array_equal(_run(msf, ctx, spec, sh), whole)
    finally:
        ctx.configure()
    # outside the band limit: exact zeros
    k = np.minimum(np.arange(ny), ny - np.arange(ny)) / (ny * 0.08)
    assert (whole[:, :, k > 2 / 3 * 0.5 / 0.08 + 1e-9] == 0).all()
    spec.free()


def test_two_contexts_at_once(msf):
    res = {}

    def work(t):
        c = msf.Context(0)
        spec = _spec(msf, c, 256, 256, seed=t)
        sh = np.stack([np.arange(40) * 3 % 256, np.arange(40) * 7 % 256], 1)
        res[t] = [_run(msf, c, spec, sh) for _ in range(3)]
        spec.free()
        c.close()

    ts = [threading.Thread(target=work, args=(t,)) for t in (1, 2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for t in (1, 2):
        for w in res[t][1:]:
            np.testing.assert_array_equal(w, res[t][0])
    assert not np.array_equal(res[1][0], res[2][0])
