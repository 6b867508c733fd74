"""Attention over position-sparse Jacobians: every workgroup size returns the bits of the largest one, which small batches run in."""

import numpy as np
import pytest
import torch

from folx_amd import kernels as K

pytestmark = pytest.mark.gpu


# 64 threads up to n = 16, d = 16 and three rows a position, 128 up to d = 32, 256 up to d = 64 or n = 32; just past each of them
@pytest.mark.parametrize('n,d,k', [
    (16, 16, 3), (1, 4, 1), (16, 16, 5), (7, 12, 2), (16, 16, 6), (15, 20, 3), (16, 32, 5), (16, 32, 6), (16, 36, 1), (13, 64, 3),
    (16, 64, 5), (16, 64, 6), (17, 16, 3), (32, 32, 8), (17, 4, 1), (32, 36, 2), (33, 16, 3),
])
def test_workgroup_sizes_agree(n, d, k):
    H, B = 3, 200
    print(f'case mhsa_sparse n={n} d={d} k={k}', flush=True)
    g = torch.Generator(device='cuda').manual_seed(n * 100 + d)
    r = lambda *s: torch.randn(*s, device='cuda', generator=g)
    index = np.arange(n * k).reshape(n, k).T.copy()
    index[0, n // 2] = -1
    index = torch.as_tensor(index.astype(np.int32)).cuda()
    t = [s for scale in (d ** -0.5, 1.0, 1.0) for s in (scale * r(B, n, H, d), scale * r(k, B, n, H, d), scale * r(B, n, H, d))]
    got = K.mhsa_sparse(*t, index, n * k, False)
    assert all(torch.isfinite(v).all() for v in got)
    for lo in range(0, B, 100):  # 300 workgroups: the form with 512 threads
        part = K.mhsa_sparse(*[(v[:, lo:lo + 100] if i % 3 == 1 else v[lo:lo + 100]).contiguous() for i, v in enumerate(t)], index, n * k, False)
        assert torch.equal(part[0], got[0][lo:lo + 100]) and torch.equal(part[2], got[2][lo:lo + 100])
        assert torch.equal(part[1], got[1][:, lo:lo + 100])
