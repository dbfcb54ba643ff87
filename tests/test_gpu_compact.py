"""Compact slices (HipStencilTable layouts 0 and 2, stencil_compact.h) and the
batch kernel that evaluates them, where they can go wrong: control lists that
end at 64-vertex rounds, at the frames-per-chunk limits and at the longest
list a slice holds, one past it (gathers from memory), row widths at and
beside the groups of four and sixteen entries, empty rows, a partial last
slice; and the row order of large order-2 tables.  All against the oracle's
CpuEvaluator-order sums, bit for bit."""
import numpy as np
import pytest

import oracle
from gpu_util import dev, empty, host
from opensubdiv_amd import HipStencilTable, _lib, far, meshes
from opensubdiv_amd.batch import Batch
from test_gpu_stencils import table_eval

pytestmark = pytest.mark.gpu

KEYS = ("weights", "du", "dv", "duu", "duv", "dvv")
# distinct control vertices of each 64-row slice: 255 is the longest list
LISTS = (1, 3, 62, 63, 64, 65, 95, 119, 127, 128, 129, 191, 254, 255, 256, 300)
# widest row of each slice, in turn
WIDTHS = (1, 2, 3, 4, 5, 8, 15, 16, 17, 33)


def listed_table(rng, nw, nsrc=700):
    """One slice per entry of LISTS (and a partial one): row r of a slice of
    U vertices takes its entries from them in turn, so that all are used."""
    sizes, indices = [], []
    for s, U in enumerate(LISTS + (10,)):
        W = max(WIDTHS[s % len(WIDTHS)], -(-U // 60))
        pool = np.sort(rng.choice(nsrc, size=U, replace=False))
        rows = 64 if s < len(LISTS) else 23
        at = 0
        for r in range(rows):
            n = 0 if r % 17 == 5 else W if r % 3 else max(1, W - r % 4)
            sizes.append(n)
            indices.append(pool[(at + np.arange(n)) % U])
            at += n
        assert at >= U or s == len(LISTS)
    t = {"sizes": np.array(sizes, np.int32),
         "indices": np.concatenate(indices).astype(np.int32)}
    t["offsets"] = (np.cumsum(t["sizes"]) - t["sizes"]).astype(np.int32)
    for k in KEYS[:nw]:
        t[k] = rng.normal(size=len(t["indices"])).astype(np.float32)
    return t


@pytest.mark.parametrize("layout", [0, 2])
@pytest.mark.parametrize("nw,L", [(1, 1), (1, 2), (1, 3), (1, 4), (1, 7), (1, 11), (3, 3), (3, 8),
                                  (6, 2), (6, 5)])
def test_list_and_width_edges(hip, layout, nw, L):
    rng = np.random.default_rng(50 + 10 * nw + L)
    t = listed_table(rng, nw)
    table = HipStencilTable.Create(t, layout=layout, order=1 if layout else 0)
    info = table.layout()
    assert info["slices"] - info["listed_slices"] == sum(u > 255 for u in LISTS)
    n = len(t["sizes"])
    src = rng.normal(size=(700, L)).astype(np.float32)
    s_t = dev(src)
    for start, end in ((0, n), (70, 900)):
        outs = [empty(n * L) for _ in range(nw)]
        assert table_eval(hip, table.h, s_t, (0, L, L), outs, [(0, L, L)] * nw, start, end) == 0
        for k in range(nw):
            want = oracle.apply_stencils(src, t["sizes"], t["offsets"], t["indices"],
                                         t[KEYS[k]])[start:end]
            np.testing.assert_array_equal(host(outs[k], shape=(n, L))[:end - start], want,
                                          err_msg=KEYS[k])


def test_control_index_of_all_ones_is_not_listed(hip):
    """A slice that names control index -1 (the set's free mark; such an entry
    has no control point and is skipped) is not listed; others are."""
    t = {"sizes": np.full(128, 2, np.int32), "offsets": np.arange(0, 256, 2, dtype=np.int32),
         "indices": (np.arange(256) % 7).astype(np.int32),
         "weights": np.linspace(-1, 1, 256).astype(np.float32)}
    t["indices"][9] = -1
    table = HipStencilTable.Create(t)
    assert (table.layout()["slices"], table.layout()["listed_slices"]) == (2, 1)
    src = np.arange(21, dtype=np.float32).reshape(7, 3)
    out = empty(128 * 3)
    assert table_eval(hip, table.h, dev(src), (0, 3, 3), [out], [(0, 3, 3)], 0, 128) == 0
    t["indices"][9], t["weights"][9] = 0, 0.0
    want = oracle.apply_stencils(src, t["sizes"], t["offsets"], t["indices"], t["weights"])
    np.testing.assert_array_equal(host(out, shape=(128, 3)), want)


@pytest.mark.parametrize("L", [1, 3, 4, 5, 7, 8])
@pytest.mark.parametrize("frames", [1, 2, 3, 4, 5, 9])
def test_batch_list_edges(L, frames):
    """The batch kernel on the same lists, for every frames-per-chunk variant;
    frames interleaved per vertex with padded and with packed records."""
    import torch
    rng = np.random.default_rng(7 * L + frames)
    t = listed_table(rng, 1)
    n = len(t["sizes"])
    for layout, order, lp in ((0, 0, L), (2, 1, -(-L // 4) * 4)):
        table = HipStencilTable.Create(t, layout=layout, order=order, keep_csr=False)
        src = rng.normal(size=(700, frames, lp)).astype(np.float32)
        s_t = dev(src)
        want = [oracle.apply_stencils(np.ascontiguousarray(src[:, f, :L]), t["sizes"],
                                      t["offsets"], t["indices"], t["weights"])
                for f in range(frames)]
        for vertex_major in (False, True):
            out = empty(n * frames * L)
            seg = dict(table=table, src=s_t, src_v=frames * lp, src_f=lp, dst=out, frames=frames,
                       dst_v=frames * L if vertex_major else L,
                       dst_f=L if vertex_major else n * L)
            b = Batch(L, [seg])
            for fc in (1, 2, 4):
                assert b.set("a_frames", fc) == 0
                assert b.set("a_group", 2 if layout == 0 and fc == 4 else 4) == 0
                out.fill_(float("nan"))
                b.run(1)
                torch.cuda.synchronize()
                got = out.cpu().numpy()
                got = got.reshape(n, frames, L).transpose(1, 0, 2) if vertex_major \
                    else got.reshape(frames, n, L)
                for f in range(frames):
                    np.testing.assert_array_equal(got[f], want[f], err_msg=f"chunk {fc} frame {f}")
            b.close()


def ragged_table(rng, widths, nlist, nsrc=900):
    """Slices of 64 rows (and one of 29) of up to `widths` entries, each drawn
    from `nlist` vertices of its own (None: from all, so that the locality
    orders list none of them)."""
    sizes, indices = [], []
    for s, W in enumerate(widths):
        pool = np.arange(nsrc) if nlist is None else rng.choice(nsrc, size=nlist, replace=False)
        for r in range(64 if s + 1 < len(widths) else 29):
            n = 0 if r == 7 else W if r % 4 == 0 else int(rng.integers(1, W + 1))
            sizes.append(n)
            indices.append(rng.choice(pool, size=n, replace=False))
    t = {"sizes": np.array(sizes, np.int32), "indices": np.concatenate(indices).astype(np.int32)}
    t["offsets"] = (np.cumsum(t["sizes"]) - t["sizes"]).astype(np.int32)
    t["weights"] = rng.normal(size=len(t["indices"])).astype(np.float32)
    return t


def batch_matches(t, layout, order, L, frames, nsrc=900):
    """The batch kernel's variants on one table against the oracle."""
    import torch
    rng = np.random.default_rng(L + 16 * frames)
    n = len(t["sizes"])
    table = HipStencilTable.Create(t, layout=layout, order=order, keep_csr=False)
    src = rng.normal(size=(nsrc, frames, L)).astype(np.float32)
    s_t = dev(src)
    want = [oracle.apply_stencils(np.ascontiguousarray(src[:, f]), t["sizes"], t["offsets"],
                                  t["indices"], t["weights"]) for f in range(frames)]
    for vertex_major in (False, True):
        out = empty(n * frames * L)
        b = Batch(L, [dict(table=table, src=s_t, src_v=frames * L, src_f=L, dst=out, frames=frames,
                           dst_v=frames * L if vertex_major else L,
                           dst_f=L if vertex_major else n * L)])
        for fc in (1, 2, 4):
            assert b.set("a_frames", fc) == 0
            assert b.set("a_group", 2 if layout == 0 and fc == 4 else 4) == 0
            out.fill_(float("nan"))
            b.run(1)
            torch.cuda.synchronize()
            got = out.cpu().numpy()
            got = got.reshape(n, frames, L).transpose(1, 0, 2) if vertex_major \
                else got.reshape(frames, n, L)
            for f in range(frames):
                np.testing.assert_array_equal(got[f], want[f], err_msg=f"chunk {fc} frame {f}")
        b.close()
    return table.layout()


@pytest.mark.parametrize("L", [1, 4, 5, 7, 8])
@pytest.mark.parametrize("frames", [1, 2, 3, 5])
def test_batch_unlisted_slices(L, frames):
    """Slices without a list, of widths at and beside the entries that one
    chunk of 1, 2 or 4 frames gathers at a time (8, 4, 2)."""
    t = ragged_table(np.random.default_rng(L), (2, 3, 4, 5, 6, 7, 8, 9, 12, 17, 31, 8), None)
    info = batch_matches(t, 2, 0, L, frames)
    assert info["listed_slices"] < info["slices"] // 2


@pytest.mark.parametrize("L", [1, 4, 5, 7, 8])
@pytest.mark.parametrize("frames", [1, 2, 3, 5])
@pytest.mark.parametrize("nlist", [40, 64, 65, 128, 250])
def test_batch_wide_listed_slices(L, frames, nlist):
    """Listed slices wider than the 16 entries held in registers, at every
    remainder of the groups of four, with lists at and beside those that 4 and
    2 frames per chunk take."""
    t = ragged_table(np.random.default_rng(L), (16, 17, 18, 19, 20, 21, 24, 33, 40), nlist)
    info = batch_matches(t, 0, 0, L, frames)
    assert info["listed_slices"] == info["slices"]


@pytest.mark.parametrize("layout", [0, 2])
@pytest.mark.parametrize("L", [4, 5, 7, 8, 11, 16])
def test_table_without_any_list(hip, layout, L):
    """A table of scattered rows lists nothing: 5 to 8 floats gather two entry
    groups at a time, also where a row ends within one of them."""
    rng = np.random.default_rng(L)
    n, nsrc = 64 * 3 + 40, 5000
    sizes = rng.integers(8, 18, size=n).astype(np.int32)
    sizes[[3, 70]] = 0, 1
    t = {"sizes": sizes, "offsets": (np.cumsum(sizes) - sizes).astype(np.int32),
         "indices": rng.integers(0, nsrc, size=int(sizes.sum())).astype(np.int32)}
    t["weights"] = rng.normal(size=len(t["indices"])).astype(np.float32)
    table = HipStencilTable.Create(t, layout=layout, order=1 if layout else 0)
    assert table.layout()["listed_slices"] == 0
    src = rng.normal(size=(nsrc, L)).astype(np.float32)
    for start, end in ((0, n), (65, n - 3)):
        out = empty(n * L)
        assert table_eval(hip, table.h, dev(src), (0, L, L), [out], [(0, L, L)], start, end) == 0
        want = oracle.apply_stencils(src, t["sizes"], t["offsets"], t["indices"], t["weights"])
        np.testing.assert_array_equal(host(out, shape=(n, L))[:end - start], want[start:end])


@pytest.mark.parametrize("n,level,far_order", [(7, 4, True), (14, 3, False)])
def test_large_order_2_tables(hip, n, level, far_order):
    """Tables of 65,536 rows and more under order 2: a level-4 refinement table
    lists under one control vertex per two rows in Far's order and keeps it,
    a level-3 table does not."""
    m = meshes.cube_sphere(n, seed=3, radial_noise=0.01, crease_fraction=0.05, sharpness_max=4.0)
    topo = far.Topology(m)
    topo.refine_uniform(level)
    t = topo.stencil_table()
    rows = len(t["sizes"])
    assert rows >= 1 << 16
    table = HipStencilTable.Create(t, layout=2, order=2)
    sz = np.zeros(-(-rows // 64) * 64, np.int64)
    sz[:rows] = t["sizes"]
    in_far_order = 64 * int(sz.reshape(-1, 64).max(axis=1).sum())
    info = table.layout()
    assert (info["record_entries"] == in_far_order) == far_order
    assert (2 * info["list_entries"] <= rows) == far_order or not far_order
    ctrl = np.random.default_rng(n).standard_normal((m.nverts, 7)).astype(np.float32)
    out = empty(rows * 7)
    assert table_eval(hip, table.h, dev(ctrl.reshape(-1)), (0, 7, 7), [out], [(0, 7, 7)], 0,
                      rows) == 0
    want = oracle.apply_stencils(ctrl, t["sizes"], t["offsets"], t["indices"], t["weights"])
    np.testing.assert_array_equal(host(out, shape=(rows, 7)), want)
