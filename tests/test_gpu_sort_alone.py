"""The sort over device buffers at the edges of its 64-design words and of its
workgroup sizes, against the oracle: few and many fronts, equal designs, one
design alone, and values that are not finite."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def sort(cdp, obj, N):
    d = torch.from_numpy(obj).cuda()
    fo = torch.full((len(obj),), 77, dtype=torch.int32, device="cuda")
    nf = torch.zeros(1, dtype=torch.int32, device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = cdp.lib().cd_nds_noalloc(C.c_void_p(d.data_ptr()), len(obj), N, C.c_void_p(fo.data_ptr()),
                                  C.c_void_p(nf.data_ptr()), stream)
    assert rc == 0, cdp.lib().cd_last_error()
    return fo.cpu().numpy(), int(nf.item())


@pytest.mark.parametrize("P", [1, 2, 63, 64, 65, 127, 129, 256, 257, 512, 513, 1000, 2047, 2049, 8191, 8192])
def test_sizes(cdp, orc, P):
    print("sort", P, flush=True)
    rng = np.random.default_rng(P)
    for levels in (2, 5, 1000):
        obj = (rng.integers(0, levels, (P, 6)) / levels).astype(np.float32)
        if levels == 5:
            obj[:, 1:] = obj[:, :1]  # a chain: as many fronts as levels
        for N in sorted({1, (P + 1) // 2, P}):
            fo, nf = sort(cdp, obj, N)
            want, n = orc.nds(obj, N)
            assert nf == n and np.array_equal(fo, want), (levels, N)


@pytest.mark.parametrize("P", [70, 300])
def test_not_finite(cdp, P):
    print("not finite", P, flush=True)
    rng = np.random.default_rng(P)
    obj = (rng.integers(0, 4, (P, 6)) / 4).astype(np.float32)
    obj[rng.random((P, 6)) < 0.05] = np.inf
    obj[rng.random((P, 6)) < 0.05] = -np.inf
    obj[rng.random((P, 6)) < 0.05] = np.nan
    fo, nf = sort(cdp, obj, P // 2)
    want, n = cdp.nds(obj, P // 2)  # (the sort of a generation)
    assert nf == n and np.array_equal(fo, want)
