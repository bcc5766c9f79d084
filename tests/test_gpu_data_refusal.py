"""Counts of 2^20 or more are refused before the resampling, by calls of any
size, and small calls of small and of large counts keep the restatement's bits."""
import time

import numpy as np
import pytest

from test_gpu_data import _same_bits
from test_oracle_data import NC, J

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng(engine_factory):
    from abc_inference_transcription_amd.design import reference_design
    return engine_factory(reference_design(cells=55))


def _cells(n, G, top, seed=0):
    rng = np.random.default_rng(seed)
    u, l = (np.asfortranarray(rng.integers(0, top, (n, G)).astype(np.uint32)) for _ in range(2))
    cond = rng.integers(-1, J, n)
    pulse, chase = np.nonzero((cond >= 0) & (cond <= 5))[0], np.nonzero(cond >= 6)[0]
    return u, l, (rng.integers(0, NC, n), cond, NC, J, pulse, chase, rng.random((NC, J)))


def test_refused_before_the_resampling(eng):
    """1,000 genes of 5,422 cells, 250 resamples: 9 ms, refused or not, while
    the counts were looked at beside the resampling; 2 ms, most of it the copy."""
    u, l, rest = _cells(5422, 1000, 30)

    def ms():
        best = np.inf
        for _ in range(5):
            t = time.perf_counter()
            try:
                eng.data_stats(u, l, *rest, n_boot=250)
            except RuntimeError as e:
                assert "below 2^20" in str(e)
            best = min(best, time.perf_counter() - t)
        return 1e3 * best

    done = ms()
    l[-1, -1] = 1 << 20
    refused = ms()
    print(f"\n[refusal] accepted {done:.2f} ms, refused {refused:.2f} ms", flush=True)
    assert refused < 0.6 * done


# either side of 131,072 counts (scanned on the host, checked on the device)
@pytest.mark.parametrize("n,G", [(1, 1), (256, 512), (257, 512)])
@pytest.mark.parametrize("value", [1 << 20, 1 << 31, (1 << 32) - 1])
@pytest.mark.parametrize("place", [0, -1])
def test_refused_in_any_place(eng, n, G, value, place):
    u, l, rest = _cells(n, G, 5)
    eng.data_stats(u, l, *rest, n_boot=3)
    for a in (u, l):
        a[place, place] = value
        with pytest.raises(RuntimeError, match="counts must be below 2\\^20"):
            eng.data_stats(u, l, *rest, n_boot=3)
        a[place, place] = (1 << 20) - 1
    eng.data_stats(u, l, *rest, n_boot=3)


# the largest u + l squared times the cells on both sides of 2^32: in one gene,
# in every gene, in a cell that is in no group, and in one that only the pulse
# list holds
@pytest.mark.parametrize("n,G,top", [(300, 40, 3783), (300, 40, 3784), (300, 300, 3784),
                                     (64, 9, 1 << 19)])
@pytest.mark.parametrize("where", ["one gene", "every gene", "no group", "pulse only"])
def test_walks_of_small_calls(oracle, eng, n, G, top, where):
    u, l, rest = _cells(n, G, 1 + top // 3, seed=top)
    rest[1][3] = 0 if "gene" in where else -1
    pulse, chase = (a[a != 3] for a in rest[4:6])
    if where == "pulse only":
        pulse = np.append(pulse, 3)
    rest = (*rest[:4], pulse, chase, rest[6])
    genes = slice(None) if where == "every gene" else slice(1, 2)
    u[3, genes], l[3, genes] = top // 2, top - top // 2
    got = eng.data_stats(u, l, *rest, n_boot=5, seed=7)
    assert _same_bits(got, oracle.data_stats(u, l, *rest, n_boot=5, seed=7))
