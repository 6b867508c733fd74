"""Chains of narrow Dense + activation layers over more than six Jacobian rows (``kernels.dense_chain``) against the float64 oracle
rules, at the seams of the kernels: 32 positions a block, groups of rows and what is left of them, every class of widths."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import rules
from test_dense_chain_gpu import dev, make
from tolerances import assert_lap, assert_val

import folx_amd
from folx_amd import _lib
from folx_amd import kernels as K
from folx_amd import numpy as fnp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('R,P,widths,vector', [
    (1, 7, (1, 1, 1), False), (31, 8, (4, 32, 32, 32), True), (33, 17, (32, 30, 7), False), (64, 9, (8, 33, 64), True),
    (65, 25, (9, 64, 50, 64, 61), False), (32, 16, (4, 100, 100, 100), True), (70, 50, (3, 65, 104), True), (40, 7, (31, 104, 97, 3), False),
    (97, 11, (5, 105, 128), False), (33, 13, (16, 128, 20, 113), True), (2100, 24, (4, 100), False), (1, 400, (4, 20, 100, 20), True),
])
def test_chain_over_many_rows(R, P, widths, vector):
    acts = (['silu', 'tanh', 'softplus', 'sin'] * 4)[:len(widths) - 1]
    if vector:
        widths, acts = (*widths, 1), [*acts, None]
    print(f'case chain R={R} P={P} widths={widths}', flush=True)
    t, layers = make(R, P, widths, acts, 4)
    args = [(a, dev(W), dev(b), prm) for a, W, b, prm in layers], *[dev(v) for v in t]
    got, hidden = K.dense_chain(*args, keep_hidden=vector)
    ref = [v.astype(np.float64) for v in t]
    for i, (a, W, b, prm) in enumerate(layers):
        if vector and i == len(layers) - 1:
            for name, h, r in zip(('x', 'jacobian'), hidden, ref):
                assert_val(h, r, name)
            assert_lap(hidden[2], ref[2], 'laplacian')
        ref = rules.dense_rule(*ref, W.astype(np.float64), None if b is None else b.astype(np.float64))
        if a is not None:
            ref = rules.elementwise_rule(a, *ref)
    assert_val(got[0], ref[0], 'x')
    assert_val(got[1], ref[1], 'jacobian')
    assert_lap(got[2], ref[2], 'laplacian')
    again, _ = K.dense_chain(*args)
    assert all(torch.equal(a, b) for a, b in zip(again, got))


def test_a_position_without_finite_values_stays_alone():
    t, layers = make(100, 9, (4, 20, 33, 20), ['tanh', 'tanh', 'tanh'], 2)
    layers = [(a, dev(W), dev(b), prm) for a, W, b, prm in layers]
    clean, _ = K.dense_chain(layers, *[dev(v) for v in t])
    t[0][17, 0] = np.inf                        # tanh: values of +-1, derivatives 0
    got, _ = K.dense_chain(layers, *[dev(v) for v in t])
    keep = torch.arange(100) != 17
    for a, b in zip(got, clean):
        assert torch.equal(a[..., keep, :], b[..., keep, :])
    assert torch.isfinite(got[0]).all() and (got[1][:, 17] == 0).all()


def test_what_the_chain_does_not_take():
    lib = _lib.load()
    i32 = lambda *v: (ctypes.c_int32 * len(v))(*v)
    acts = i32(_lib.ACT['silu'], _lib.ACT['silu'])
    assert lib.folx_hip_dense_chain_workspace_bytes(2, acts, i32(33, 20, 20), 100, 7) == _lib.ENOTSUP
    assert lib.folx_hip_dense_chain_workspace_bytes(2, acts, i32(4, 129, 20), 100, 7) == _lib.ENOTSUP
    assert lib.folx_hip_dense_chain_workspace_bytes(2, acts, i32(4, 20, 20), 100, 6) == 0
    assert lib.folx_hip_dense_chain_workspace_bytes(2, acts, i32(4, 20, 20), 100, 7) > 0
    assert lib.folx_hip_dense_chain_faster(2, acts, i32(33, 20, 20), 100, 7) == 0


def test_front_door_replayed_graph():
    """The chain under a captured graph, replayed with eager work between the replays."""
    g = torch.Generator(device='cuda').manual_seed(3)
    Ws = [torch.randn(a, b, device='cuda', generator=g) / a ** 0.5 for a, b in ((4, 100), (100, 100), (100, 100), (100, 100), (100, 1))]

    def fn(r):
        for W in Ws[:-1]:
            r = fnp.silu(fnp.dot(r, W))
        return fnp.sum(fnp.dot(r, Ws[-1]))

    eager = folx_amd.vmap(folx_amd.forward_laplacian(fn, 0))
    xs = [torch.randn(30, 64, 4, device='cuda', generator=g) for _ in range(3)]
    ran = []
    orig = K.dense_chain
    K.dense_chain = lambda layers, *a: (ran.append(len(layers)), orig(layers, *a))[1]
    try:
        want = [eager(x) for x in xs]
    finally:
        K.dense_chain = orig
    assert ran == [5, 5, 5], ran
    captured = folx_amd.jit(eager)
    for x, w in zip(xs + xs, want + want):
        y = captured(x)
        eager(xs[0])
        torch.cuda.synchronize()
        assert torch.equal(y.x, w.x) and torch.equal(y.laplacian, w.laplacian)
        assert torch.equal(y.jacobian.dense_array, w.jacobian.dense_array)
