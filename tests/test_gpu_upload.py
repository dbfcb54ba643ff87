"""osdhip_batch_upload: sizes around a block's 8,192 bytes and the 16-byte
loads' remainders, addresses that are only 4-byte aligned, more host blocks
than one launch takes, and the pointers it refuses."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import stream
from opensubdiv_amd import _lib

pytestmark = pytest.mark.gpu


def upload(hip, blocks):
    a = (_lib.UploadBlock * max(1, len(blocks)))(*blocks)
    return hip.osdhip_batch_upload(len(blocks), ctypes.cast(a, ctypes.c_void_p), stream())


@pytest.mark.parametrize("shift", [0, 1, 3])
def test_sizes_alignments_and_launch_splits(hip, shift):
    words = [1, 2, 3, 4, 5, 0, 63, 64, 1023, 1024, 1025, 2047, 2048, 2049, 2051, 4095, 4096, 4097,
             100003] + list(range(2040, 2060)) + [7] * 30
    total = sum(words) + 8 * len(words)
    src = torch.from_numpy(np.random.default_rng(3).integers(
        -2**31, 2**31, size=total, dtype=np.int64).astype(np.int32)).pin_memory()
    dst = torch.full((total,), 17, dtype=torch.int32, device="cuda")
    want = np.full(total, 17, np.int32)
    blocks, at = [], 0
    for k, n in enumerate(words):
        s, d = at + shift, at + (shift + k) % 4
        blocks.append(_lib.UploadBlock(dst.data_ptr() + 4 * d, src.data_ptr() + 4 * s, 4 * n))
        want[d:d + n] = src[s:s + n].numpy()
        at += n + 8
    assert upload(hip, blocks) == 0
    torch.cuda.synchronize()
    assert np.array_equal(dst.cpu().numpy(), want)


def test_refused_pointers_and_sizes(hip):
    src = torch.zeros(64, dtype=torch.int32).pin_memory()
    dst = torch.ones(64, dtype=torch.int32, device="cuda")
    plain = np.zeros(64, np.int32)
    s, d = src.data_ptr(), dst.data_ptr()
    assert upload(hip, []) == 0
    assert upload(hip, [_lib.UploadBlock(0, 0, 0)]) == 0
    for bad in ((d, plain.ctypes.data, 64), (s, s, 64), (d, d, 64), (d + 2, s, 64), (d, s + 1, 64),
                (d, s, 63), (d, s, -4), (d, 0, 64)):
        assert upload(hip, [_lib.UploadBlock(d, s, 64), _lib.UploadBlock(*bad)]) == \
            _lib.ERR_ARGS, bad
    torch.cuda.synchronize()
    assert bool((dst == 1).all())


def test_blocks_that_run_past_their_allocation_are_refused(hip):
    """A block whose destination (or source) starts in an allocation and ends
    past it is refused, and so is everything given beside it; one that ends
    with the allocation is copied."""
    src = torch.arange(64, dtype=torch.int32).pin_memory()        # 256 bytes
    more = torch.zeros(1024, dtype=torch.int32).pin_memory()
    dst = torch.zeros(1024, dtype=torch.int32, device="cuda")
    short = ctypes.c_void_p()
    assert hip.osdhip_malloc(ctypes.byref(short), 256) == 0
    try:
        for bad in ((short.value, more.data_ptr(), 260), (short.value + 128, more.data_ptr(), 256),
                    (short.value, more.data_ptr(), 4096), (dst.data_ptr(), src.data_ptr(), 260)):
            assert upload(hip, [_lib.UploadBlock(dst.data_ptr(), src.data_ptr(), 256),
                                _lib.UploadBlock(*bad)]) == _lib.ERR_ARGS, bad
        torch.cuda.synchronize()
        assert bool((dst == 0).all())
        assert upload(hip, [_lib.UploadBlock(short.value, src.data_ptr(), 256)]) == 0
        got = np.zeros(64, np.int32)
        assert hip.osdhip_memcpy_dtoh(got.ctypes.data, short, 256, stream()) == 0
        torch.cuda.synchronize()
        assert np.array_equal(got, np.arange(64))
    finally:
        hip.osdhip_free(short)
