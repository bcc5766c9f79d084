"""The 32-bit and 64-bit walks of the data statistics' resampling kernel: a gene
takes the first when (largest u + l)^2 times the largest family's cells is
below 2^32.  Genes on both sides of that line, side by side in one call,
against the CPU restatement bit for bit (the sums are exact integers)."""
import numpy as np
import pytest

from test_gpu_data import _same_bits
from test_oracle_data import NC, J

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng(engine_factory):
    from abc_inference_transcription_amd.design import reference_design
    return engine_factory(reference_design(cells=55))


@pytest.mark.parametrize("n", [1, 2, 255, 257, 5422, 16384])
def test_data_stats_both_walks(oracle, eng, n):
    rng = np.random.default_rng(n)
    x = int(np.sqrt((2.0**32 - 1) / n))  # the largest u + l of a 32-bit gene
    while x * x * n >= 2**32:
        x -= 1
    while (x + 1) * (x + 1) * n < 2**32:
        x += 1
    age = rng.integers(0, NC, n)
    cond = rng.integers(-1, J, n)
    cond[n - 1] = 0  # the cell that holds the gene's largest count has a group
    full = np.stack([np.full(n, x), np.full(n, x + 1), rng.integers(0, x + 1, n),
                     rng.integers(0, x + 1, n), np.zeros(n, np.int64),
                     np.full(n, 2 * (2**20 - 1))], axis=1)
    full[n - 1, 2], full[n - 1, 3] = x, x + 1
    u = np.minimum((full * rng.random(full.shape)).astype(np.int64), 2**20 - 1)
    l = full - u
    u, l = np.where(l >= 2**20, full - (2**20 - 1), u), np.minimum(l, 2**20 - 1)
    pulse = np.nonzero(rng.random(n) < 0.6)[0]
    chase = np.nonzero(rng.random(n) < 0.4)[0]
    w = rng.random((NC, J))
    print(f"\n[data_stats] both walks n={n} x={x}", flush=True)
    got = eng.data_stats(u, l, age, cond, NC, J, pulse, chase, w, n_boot=9, seed=n)
    want = oracle.data_stats(u, l, age, cond, NC, J, pulse, chase, w, n_boot=9, seed=n)
    assert _same_bits(got, want)


def test_data_stats_rejects_large_counts_in_any_cell(eng):
    """a count of 2^20 in a cell of no group is refused by the call on host
    arrays, as in the others"""
    n = 300
    age, cond = np.zeros(n, int), np.zeros(n, int)
    cond[7] = -1
    w = np.ones((NC, J))
    u, l = np.ones((n, 3), int), np.ones((n, 3), int)
    pulse, chase = np.arange(0, 6), np.arange(8, n)
    eng.data_stats(u, l, age, cond, NC, J, pulse, chase, w, n_boot=3)
    for a in (u, l):
        a[7, 2] = 2**20
        with pytest.raises(Exception, match="counts must be below 2\\^20"):
            eng.data_stats(u, l, age, cond, NC, J, pulse, chase, w, n_boot=3)
        a[7, 2] = 2**20 - 1
    eng.data_stats(u, l, age, cond, NC, J, pulse, chase, w, n_boot=3)
