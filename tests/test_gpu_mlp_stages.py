"""The weight gradients' pipeline stages differ with the tile (128 deep in 64 x 64
tiles, 64 in larger ones): the same bits from every tile, for batches whose
chunks are one stage, several, short and empty."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,width,depth", [(1, 128, 1), (130, 256, 2), (700, 256, 1),
                                           (1100, 512, 2), (4100, 128, 2), (64, 2048, 2)])
def test_tiles_give_the_same_gradient(n, width, depth):
    import torch
    from abc_inference_transcription_amd.surrogate import Surrogate
    s = Surrogate(90, width=width, depth=depth, max_batch=n, seed=n)
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, s.n_in, generator=g).to(s.dev)
    t = torch.randn(n, 90, generator=g).to(s.dev)
    out = []
    for rows, cols in ((64, 64), (64, 128), (128, 64), (128, 128), (0, 0)):
        print(f"\n[mlp stages] n={n} width={width} tile {rows} x {cols}", flush=True)
        assert s.L.abc_mlp_set_tile_rows(s.h, rows) == 0
        assert s.L.abc_mlp_set_tile_cols(s.h, cols) == 0
        out.append(s.grad(x, t))
    for loss, grad in out[1:]:
        assert loss == out[0][0] and np.array_equal(grad.view(np.uint32), out[0][1].view(np.uint32))
    s.close()
