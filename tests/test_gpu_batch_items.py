"""Phase-B work items of a batch: a coord's frames split over items where a
launch would otherwise have few blocks, and kept together where it has many
(eight blocks of 256 coords per CU), against one mesh and frame per launch,
bit for bit."""
import numpy as np
import pytest

from opensubdiv_amd.batch import Batch
from opensubdiv_amd.workloads import DeviceMesh, MeshSpec, compile_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length,coords,frames", [(3, 700001, 3), (3, 300, 9), (7, 5000, 6)])
def test_frames_split_over_items_match_plain(length, coords, frames):
    import torch
    h = compile_mesh(MeshSpec(0, 8, 2, frames, coords, 5), length)
    d = DeviceMesh(h)
    b = Batch(length, d.stencil_segments(), [d.patch_segment()])
    b.run_plain()
    torch.cuda.synchronize()
    want = [o.cpu().numpy() for o in d.out]
    for fc in (1, 2, 4):
        for stage in (0, 1):
            for persistent in (0, 1):
                assert b.set("b_frames", fc) == 0 and b.set("b_stage", stage) == 0
                assert b.set("b_persistent", persistent) == 0
                for o in d.out:
                    o.fill_(float("nan"))
                b.launch()
                torch.cuda.synchronize()
                for o, w in zip(d.out, want):
                    assert np.array_equal(o.cpu().numpy().view(np.uint32), w.view(np.uint32)), \
                        (fc, stage, persistent)
    b.close()
