"""The admission estimate of a served job covers what its set-up and run
allocate: stacks, the build's work arrays (which grow with the species), the
vacuum waves and the work array that forms them."""
import numpy as np
import pytest

import msf


@pytest.mark.parametrize("n,species,slices", [(64, 1, 1), (256, 2, 12), (1024, 1, 3),
                                              (1024, 24, 1), (1024, 24, 2), (512, 90, 1),
                                              (64, 1, 800)])
def test_estimate_covers_the_buffers(msf_lib, n, species, slices):
    M = n * n
    z = np.repeat(2.0 * np.arange(slices), species) + 0.1
    q = np.stack([np.full(z.size, 1.0), np.full(z.size, 1.0), z], 1)
    Z = np.tile(np.arange(1, species + 1), slices)
    fp = msf.job_footprint(msf.make_grid(n, n, 0.08 * n, 0.08 * n, 2.0 * slices, 200e3), q, Z, 1.0,
                           np.array([1.0]), np.array([1.0]))
    stacks = (16 + 8 + 16) * M * slices             # t FP64 and FP32, vacuum waves in pairs
    vacuum = min(slices * 16 * M, max(32 << 20, 16 * M)) + 8 * M
    one = species * (16 + 4) * M + 16 * M
    build = min(slices * one, max(96 << 20, one)) + species * 8 * M
    assert fp >= stacks + vacuum + build + 8 * M    # and one position's wave


@pytest.fixture(scope="module")
def msf_lib():
    return msf.lib()
