"""Edges of the kernels' tilings and of the rules that choose between their forms, against the float64 oracle rules (the
parity bars of ``tolerances.py``)."""

import numpy as np
import pytest
import torch

from oracle import rules
from tolerances import assert_lap, assert_val

pytestmark = pytest.mark.gpu


def rand(rng, *s):
    return rng.normal(size=s).astype(np.float32)


def dev(a, dtype=torch.float32):
    return torch.as_tensor(np.ascontiguousarray(a)).to(device='cuda', dtype=dtype)


def f64(*arrays):
    return [None if a is None else np.asarray(a, dtype=np.float64) for a in arrays]


# n <= 16: one wavefront per (walker, head), 1 / 4 / 8 of them sharing the Jacobian rows (P < 8, otherwise, few pairs),
# 1, 2 or 4 blocks of 16 features; 17: the form with one wavefront per 16 query rows
@pytest.mark.parametrize('B,n,H,d,P', [(1, 1, 1, 4, 1), (2, 16, 3, 16, 0), (3, 5, 2, 20, 7), (2, 7, 5, 32, 8),
                                       (1, 16, 1, 36, 17), (2, 13, 4, 64, 39), (100, 3, 2, 64, 16), (67, 10, 3, 8, 9),
                                       (2, 17, 2, 64, 5)])
@pytest.mark.parametrize('edge,masked', [(False, False), (True, False), (False, True)])
def test_mhsa_short_sequences(B, n, H, d, P, edge, masked):
    from folx_amd import kernels as K

    print(f'case mhsa B={B} n={n} H={H} d={d} P={P} edge={edge} masked={masked}', flush=True)
    rng = np.random.default_rng(n * 100 + d)
    args = []
    for s in (1 / np.sqrt(d), 1.0, 1.0):
        args += [s * rand(rng, B, n, H, d), s * rand(rng, P, B, n, H, d), s * rand(rng, B, n, H, d)]
    e = [rand(rng, B, n, H, n), rand(rng, P, B, n, H, n), rand(rng, B, n, H, n)] if edge else [None] * 3
    mask, imask = np.ones((B, n), dtype=bool), np.ones((P, B), dtype=bool)
    if masked:
        mask[:, max(1, n - 2):] = False
        imask[P // 2:] = False
    ref = rules.mhsa_rule(*f64(*args), mask, imask, *f64(*e))
    got = K.mhsa(*[dev(t) for t in args], dev(mask, torch.uint8) if masked else None,
                 dev(imask, torch.uint8) if masked else None, tuple(dev(t) for t in e) if edge else None)
    m = mask[0]  # rows of padding queries carry no meaning
    assert_val(got[0][:, m], ref[0][:, m], 'o')
    assert_val(got[1][:, :, m], ref[1][:, :, m], 'o_jac')
    assert_lap(got[2][:, m], ref[2][:, m], 'o_lap')
    assert all(bool(torch.isfinite(t).all()) for t in got)
