"""Host-side pieces of the serving loop (no GPU)."""
import contextlib
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from opensubdiv_amd import _lib
from opensubdiv_amd.serve import Arena, Request, Server, poisson_requests


def test_arena_first_fit_and_merge():
    a = Arena(1024, 64)
    x = a.alloc(100)
    y = a.alloc(64)
    z = a.alloc(500)
    assert x == (0, 128) and y == (128, 64) and z == (192, 512)
    assert a.alloc(400) is None
    a.release(*y)
    assert a.alloc(64) == (128, 64)
    a.release(128, 64)
    a.release(*x)
    a.release(*z)
    assert a.free == [(0, 1024)] and a.used() == 0


def test_poisson_requests_rate_and_mix():
    reqs = poisson_requests(20000, rate=500.0, ntopo=32, seed=1)
    t = np.array([r.arrival for r in reqs])
    assert np.all(np.diff(t) >= 0)
    gaps = np.diff(np.concatenate([[0.0], t]))
    assert abs(gaps.mean() - 1 / 500.0) < 0.05 / 500.0
    # exponential: coefficient of variation near 1
    assert 0.95 < gaps.std() / gaps.mean() < 1.05
    kinds = [r.kind for r in reqs]
    assert 0.48 < kinds.count("limit") / len(kinds) < 0.52
    assert {r.topo for r in reqs} == set(range(32))


@pytest.mark.parametrize("fails", [None, "upload", "epoch"])
def test_a_failed_launch_leaves_nothing_in_flight(fails):
    """When an epoch's call fails after its uploads were queued, launch waits
    for the slot's stream before it raises: the queued copies read the pinned
    frames and write the arena, and no event is recorded behind them."""
    log = []
    rc = {"upload": 0, "epoch": 0}
    if fails:
        rc[fails] = _lib.ERR_ARGS
    stream = SimpleNamespace(cuda_stream=0, synchronize=lambda: log.append("synchronize"))
    slot = {"stream": stream, "event": SimpleNamespace(record=lambda st: log.append("record"),
                                                       synchronize=lambda: None),
            "reqs": None, "staging": torch.zeros(1), "scratch": torch.zeros(1), "cap": 1 << 20}
    sv = object.__new__(Server)
    sv.torch = SimpleNamespace(cuda=SimpleNamespace(stream=lambda st: contextlib.nullcontext()))
    sv.lib = SimpleNamespace(
        osdhip_batch_epoch_bytes=lambda *a: 256,
        osdhip_batch_upload=lambda *a: log.append("upload") or rc["upload"],
        osdhip_batch_epoch=lambda *a: log.append("epoch") or rc["epoch"])
    sv.res = [SimpleNamespace(nctrl=4, nrefine=9, npts=0, ncoords=0,
                              refine_table=SimpleNamespace(h=1))]
    sv.L, sv.item_slices, sv.slots = 3, 8, [slot]
    sv.dev = torch.zeros(256)
    sv.frames = [torch.zeros(2, 4, 3)]
    sv.epochs, sv.epoch_points = [], []
    r = Request(0, 0, "refine", 0.0, 1)
    r.dev = [(0, 64), (64, 64)]
    if fails is None:
        sv.launch(slot, [r])
        assert log == ["upload", "epoch", "record"] and slot["reqs"] == [r]
        return
    with pytest.raises(RuntimeError):
        sv.launch(slot, [r])
    assert log == ["upload"] + (["epoch"] if fails == "epoch" else []) + ["synchronize"]
    assert slot["reqs"] is None and sv.epochs == []
