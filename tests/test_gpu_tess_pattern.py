"""osdhip_tess_coords at the limits of its pattern kernel (4,096 points, 128
runs) and beside them, for one face, a block's worth and many, against the
oracle's Bfr coordinates bit for bit."""
import numpy as np
import pytest

import oracle
from gpu_util import empty, host, ptr, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme,size,rates", [
    (1, 4, [1]), (1, 4, [2]), (1, 4, [31]), (1, 4, [62]), (1, 4, [63]), (1, 4, [64]),
    (1, 4, [3, 200, 5, 7]), (1, 4, [40, 100]), (1, 4, [41, 100]), (2, 3, [89]), (2, 3, [90]),
    (1, 5, [30]), (1, 5, [41]), (1, 7, [9, 8, 7, 6, 5, 4, 3, 17])])
def test_pattern_limits(hip, scheme, size, rates):
    want = oracle.tess_coords(scheme, size, rates)
    r = np.ascontiguousarray(rates, np.int32)
    nc = hip.osdhip_tess_count(scheme, size, len(r), r.ctypes.data)
    assert nc == len(want)
    for nf in (1, max(1, 1024 // nc), 1024 // nc + 1, 700):
        uv = empty(nf * nc * 2)
        assert hip.osdhip_tess_coords(scheme, size, len(r), r.ctypes.data, nf, ptr(uv), None, None,
                                      None, None, 0, None, stream()) == 0
        got = host(uv, shape=(nf, nc, 2))
        for f in {0, nf // 2, nf - 1}:
            assert got[f].tobytes() == np.asarray(want, np.float32).tobytes(), (nf, f)
        assert np.array_equal(got, np.broadcast_to(got[0], got.shape))
