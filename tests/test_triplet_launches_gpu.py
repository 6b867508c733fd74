"""Sums and constant factors / shifts of a triplet in one launch against the same for each array on its own: the same bits, at the
seams between the arrays, for every form of the kernels."""

import numpy as np
import pytest
import torch

from folx_amd import kernels as K

pytestmark = pytest.mark.gpu


def rand(*shape):
    g = torch.Generator(device='cuda').manual_seed(sum(shape))
    return torch.randn(*shape, device='cuda', generator=g)


# inner extent a multiple of 4 or not, last axis (aligned, unaligned, long, short), windows, no Jacobian rows, one output
@pytest.mark.parametrize('B,P,shape,axis,window', [
    (3, 5, (7, 8), 0, None), (1, 0, (4, 4), 0, None), (2, 9, (6, 3), 0, (1, 5)), (33, 21, (16, 32), 0, (8, 16)), (5, 3, (33,), 0, None),
    (700, 6, (20,), 0, None), (3, 2, (64,), 0, (4, 36)), (1, 1, (300,), 0, (3, 290)), (2, 7, (3, 5, 4), 1, (2, 2)), (513, 48, (2, 4), 0, None),
    (2500, 7, (16,), 0, None), (4, 3, (5,), 0, None),
])
def test_sum_of_three_arrays(B, P, shape, axis, window):
    print(f'case sums B={B} P={P} {shape} axis {axis} window {window}', flush=True)
    ts = [rand(B, *shape), rand(P, B, *shape), rand(B, *shape) * 2]
    got = K.reduce_sum_arrays(ts, [1 + axis, 2 + axis, 1 + axis], 0.25, window)
    for t, lead, y in zip(ts, (1, 2, 1), got):
        outer = int(np.prod(t.shape[:lead + axis]))
        red, inner = shape[axis], int(np.prod(shape[axis + 1:]))
        want = K.reduce_sum(t.reshape(-1), 1, outer, red, inner, 0.25, window)
        assert torch.equal(y, want.reshape(y.shape))
    (one,) = K.reduce_sum_arrays(ts[2:], [1 + axis], 0.25, window)
    assert torch.equal(one, got[2])


@pytest.mark.parametrize('B,P,shape,out,c,d', [
    (3, 5, (6, 8), (6, 8), (1, 6, 8), None), (3, 0, (6, 8), (6, 8), None, (1, 1, 1)), (2, 4, (5, 3), (5, 3), (1, 1, 3), (2, 5, 3)),
    (2, 1200, (3,), (3,), (1, 3), (1, 3)), (4, 7, (1, 4), (5, 4), (1, 5, 4), (1, 5, 1)), (1, 1, (1,), (1,), None, (1, 1)),
    (2, 3, (2, 1, 4), (2, 3, 4), (1, 2, 3, 4), None),
])
def test_affine_of_a_triplet(B, P, shape, out, c, d):
    print(f'case affine B={B} P={P} {shape} -> {out}', flush=True)
    x, J, L = rand(B, *shape), rand(P, B, *shape), rand(B, *shape) * 3
    c, d = (None if s is None else rand(*s) for s in (c, d))
    full = (B, *out)
    got = K.affine(x, J, L, (B, *shape), full, c, d, 0.5, -1.5)
    assert torch.equal(got[0], K.rows_affine(x, 1, (B, *shape), full, c, d, 0.5, -1.5).reshape(full))
    assert torch.equal(got[1], K.rows_affine(J, P, (B, *shape), full, c, None, 0.5, 0.0).reshape(P, *full))
    assert torch.equal(got[2], K.rows_affine(L, 1, (B, *shape), full, c, None, 0.5, 0.0).reshape(full))
