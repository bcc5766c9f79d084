"""The window queue's order of cells (counting sort by expected cost and
sub-lanes, claims by weight): every cell and sub-lane is simulated once
whatever the tile remainders, the sub-lane counts and the claim, so results
equal the CPU replay's bit for bit."""
import numpy as np
import pytest

from abc_inference_transcription_amd.design import config_design

pytestmark = pytest.mark.gpu


# cells per call: one, one tile of 4,096 less, exactly and plus one, several
# tiles; split targets from no splitting to many sub-lanes per cell
@pytest.mark.parametrize("n,cells,split,claim", [
    (1, 1, 32768.0, 2), (3, 1365, 32768.0, 8), (2, 2048, 0.0, 4), (1, 4097, 256.0, 1),
    (9, 1000, 64.0, 2), (700, 9, 1024.0, 8)])
def test_cell_order_simulates_every_item_once(oracle, engine_factory, n, cells, split, claim):
    d = config_design(cells=cells)
    d["split_target"] = split
    eng = engine_factory(d)
    eng.set_ssa_claim(claim)
    od = oracle.OracleDesign(d)
    model, first = 1 + n % 5, 40
    print(f"\n[cell order] n={n} cells={cells} split={split} claim={claim}", flush=True)
    th = eng.sample_prior(model, n, seed=3, first=first)
    th[:, -3] = np.minimum(th[:, -3], 0.5)   # moderate decay rates: short CPU replays
    got = eng.simulate(model, th, seed=3, first=first, cells=True)
    rows = range(n) if n <= 9 else range(0, n, 97)
    for i in rows:
        want = oracle.simulate(od, model, 3, first + i, th[i:i + 1])
        for k in ("cell_u", "cell_l", "cell_bin"):
            assert np.array_equal(got[k][i], want[k][0]), (i, k)
        assert int(got["steps"][i]) == int(want["steps"][0]), i
