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


@pytest.mark.parametrize("length", [1, 2, 4, 5, 8])
@pytest.mark.parametrize("frames", [1, 2, 3, 4, 6])
def test_staged_patches_of_every_point_size(length, frames):
    """Points of one value, of one and two whole quads and of a quad that
    overlaps, staged by waves of up to 128 and up to 256 points beside waves
    that gather, with whole and partial frame chunks."""
    import torch
    h = compile_mesh(MeshSpec(0, 5, 2, frames, 1000, 5), max(length, 3))
    h.frames, h.length = np.ascontiguousarray(h.frames[:, :, :length]), length
    d = DeviceMesh(h)
    b = Batch(length, d.stencil_segments(), [d.patch_segment()])
    nu = b.patch_staging(0)["nuniq"]
    assert (nu < 0).any() and (nu > 128).any() and ((nu >= 0) & (nu <= 128)).any()
    b.run_plain()
    torch.cuda.synchronize()
    want = [o.cpu().numpy() for o in d.out]
    assert all(np.isfinite(w).all() for w in want)
    for fc in (1, 2, 4):
        for persistent in (0, 1):
            assert b.set("b_frames", fc) == 0 and b.set("b_stage", 1) == 0
            assert b.set("b_persistent", persistent) == 0
            for o in d.out:
                o.fill_(float("nan"))
            b.launch()
            torch.cuda.synchronize()
            for o, w in zip(d.out, want):
                assert np.array_equal(o.cpu().numpy().view(np.uint32), w.view(np.uint32)), \
                    (fc, persistent)
    b.close()


@pytest.mark.parametrize("layout", [0, 2])
def test_tuning_times_a_kernel_once(layout):
    """Phase-A pairs of the same frames per chunk (0: 4) are one kernel: the
    report gives them one time."""
    h = compile_mesh(MeshSpec(0, 4, 2, 3, 300, 5), 3)
    d = DeviceMesh(h, layout=layout, order=0)
    b = Batch(3, d.stencil_segments())
    seen = {}
    for r in b.tune(reps=1)["phase_a"]:
        seen.setdefault((r["frames"] or 4, r["slices"], r["persistent"]), []).append(r["ms"])
    assert len(seen) == 18 and all(len(set(ms)) == 1 for ms in seen.values())
    assert sum(map(len, seen.values())) == (30 if layout == 0 else 36)
    b.close()
