"""osdhip_eval_patches_sorted at the edges of its blocks (256 coords), of the
binning's tiles (4,096 coords) and of the tile count (256 tiles, after which
tiles grow), against the oracle bit for bit."""
import numpy as np
import pytest

import oracle
from gpu_util import dev, empty, host
from test_gpu_patches import eval_patches, golden_patches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nout", [1, 3, 6])
@pytest.mark.parametrize("order", ["random", "one_patch"])
def test_sorted_block_and_tile_edges(hip, nout, order):
    g, src, _, arrays, indices, params = golden_patches()
    base = g["coords"]
    desc = [(0, 3, 3)] * nout
    want = [np.zeros((len(base), 3), np.float32) for _ in range(nout)]
    assert oracle.eval_patches(g["src"], (0, 3, 3), want, desc, base, g["arrays"], g["indices"],
                               g["params"])
    rng = np.random.default_rng(5)
    for n in (1, 63, 64, 255, 256, 257, 511, 4095, 4096, 4097, 8193, 256 * 4096 - 1, 256 * 4096,
              256 * 4096 + 1):
        pick = (rng.integers(0, len(base), size=n) if order == "random"
                else np.full(n, len(base) // 2))
        outs = [empty(n * 3) for _ in range(nout)]
        assert eval_patches(hip, src, (0, 3, 3), outs, desc, n, dev(base[pick]), arrays, indices,
                            params, sorted=True) == 0
        for k in range(nout):
            got = host(outs[k], shape=(n, 3))
            assert np.array_equal(got.view(np.uint32), want[k][pick].view(np.uint32)), (n, k)
