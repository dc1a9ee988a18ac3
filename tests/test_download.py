"""Device-to-host copies: histograms come back byte for byte at the sizes where
the path changes (plain copy, one pinned slot, several half or whole slots, a
last partial one), into pinned memory too, and from two threads at once."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 16 bytes a bin: 64 KiB plain / staged, one 2 MiB transfer, 16 MiB, more transfers than slots
BINS = [1, 4095, 4096, 4097, 131072, 131073, 262144 + 5, 1048575, 1048576, 1048577, 3000001]


def _bins(torch, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand((1, n, 4), generator=g, device="cuda")


@pytest.mark.parametrize("n", BINS)
def test_download_at_slot_edges(rf, gpu_available, n):
    import torch
    ctx = rf.Context(1 << 12, 1, 16)
    b = _bins(torch, n, n)
    h = ctx.histogram(n, 1, b.data_ptr())
    want = b.cpu().numpy()
    for _ in range(2):
        assert np.array_equal(h.download(), want)
    pinned = torch.empty((n, 4), dtype=torch.float32, pin_memory=True)
    ctx.check(ctx.L.rf_hist_download(h.h, pinned.numpy().ctypes.data_as(ctx.L.rf_hist_download.argtypes[1])))
    assert np.array_equal(pinned.numpy(), want[0])


@pytest.mark.parametrize("n", [4095, 4097, 131073, 1048577])
def test_download_into_device_memory(rf, gpu_available, n):
    """A device pointer as the destination, as hipMemcpy takes one."""
    import torch
    ctx = rf.Context(1 << 12, 1, 16)
    b = _bins(torch, n, n)
    h = ctx.histogram(n, 1, b.data_ptr())
    out = torch.zeros_like(b)
    torch.cuda.synchronize()
    fp = ctx.L.rf_hist_download.argtypes[1]
    ctx.check(ctx.L.rf_hist_download(h.h, ctypes.cast(out.data_ptr(), fp)))
    assert torch.equal(out, b)


def test_download_from_two_threads(rf, gpu_available):
    import torch
    bad = []

    def work(seed):
        ctx = rf.Context(1 << 12, 1, 16, seed=seed)
        for k, n in enumerate(BINS):
            b = _bins(torch, n, seed + k)
            torch.cuda.synchronize()
            h = ctx.histogram(n, 1, b.data_ptr())
            if not np.array_equal(h.download(), b.cpu().numpy()):
                bad.append((seed, n))
            h.close()
        ctx.close()

    ts = [threading.Thread(target=work, args=(s,)) for s in (100, 200)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
