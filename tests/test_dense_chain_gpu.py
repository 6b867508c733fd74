"""Chains of narrow Dense + activation layers in one launch (``kernels.dense_chain``) against the same layers one by one
(same bits) and, for widths those do not take, against the float64 oracle rules."""

import numpy as np
import pytest
import torch

from oracle import rules
from tolerances import assert_lap, assert_val

import folx_amd
from folx_amd import _lib
from folx_amd import kernels as K
from folx_amd import numpy as fnp

pytestmark = pytest.mark.gpu


def make(R, P, widths, acts, seed=0):
    g = np.random.default_rng(seed)
    t = [g.normal(size=s).astype(np.float32) for s in ((R, widths[0]), (P, R, widths[0]), (R, widths[0]))]
    layers = [(a, (g.normal(size=(k, n)) / np.sqrt(k)).astype(np.float32), None if i == 1 else g.normal(size=n).astype(np.float32), 0.0)
              for i, (a, k, n) in enumerate(zip(acts, widths[:-1], widths[1:]))]
    return t, layers


def dev(v):
    return None if v is None else torch.as_tensor(v).cuda()


def one_by_one(t, layers):
    """The layers' result, what the last one reads, and whether every layer took the kernel for few Jacobian rows (the general
    one rounds d1 z_lap + d2 ssq the other way round: one multiply-add of the Laplacian, 2^-24 of the larger term a layer)."""
    few = True
    for name, W, b, prm in layers:
        prev = t
        t = K.dense(*t, W, b) if name is None else K.dense_act(name, *t, W, b, prm)
        few = few and (name is None or _lib.load().folx_hip_dense_act_form(t[0].shape[0], t[1].shape[0], *W.shape, 0) == 2)
    return t, prev, few


def assert_same(got, want, few):
    for i, (a, b) in enumerate(zip(got, want)):
        if i < 2 or few:
            assert torch.equal(a, b)
        else:  # at most three layers of 128 terms each: well below 2^-18 of the largest entry
            assert float((a - b).abs().max()) <= 2.0 ** -18 * float(b.abs().max())


# 8 and 16 positions a workgroup (up to 6144 positions and above), a last workgroup that is not full, every number of rows,
# widths at and off the multiples of 16, the widest layer (a tile of more than 64 KB at P = 6)
@pytest.mark.parametrize('R,P,widths,vector', [
    (1, 0, (4, 4, 8), False), (7, 1, (4, 100, 100), True), (40, 2, (128, 16, 128), False), (333, 3, (20, 52, 36, 60), True),
    (2000, 4, (4, 100, 100, 100), True), (77, 5, (8, 12, 100), False), (500, 6, (32, 128, 128, 32), True),
    (6144, 4, (4, 40, 24), True), (6145, 4, (4, 40, 24), True), (6149, 0, (16, 64, 64), False), (7003, 1, (4, 20, 112), True),
    (6148, 2, (4, 100, 28), False), (6147, 3, (12, 32, 32), True), (6159, 5, (8, 96, 4), True), (6401, 6, (128, 128, 128), True),
])
def test_chain_returns_the_bits_of_its_layers(R, P, widths, vector):
    acts = (['silu', 'tanh', 'softplus', 'sin'] * 4)[:len(widths) - 1]
    if vector:
        widths, acts = (*widths, 1), [*acts, None]
    print(f'case chain R={R} P={P} widths={widths}', flush=True)
    t, layers = make(R, P, widths, acts)
    layers = [(a, dev(W), dev(b), prm) for a, W, b, prm in layers]
    want, before, few = one_by_one([dev(v) for v in t], layers)
    got, hidden = K.dense_chain(layers, *[dev(v) for v in t], keep_hidden=vector)
    assert_same(got, want, few)
    if vector:
        assert_same(hidden, before, few)
        want, (got, hidden) = got, K.dense_chain(layers, *[dev(v) for v in t])
        assert hidden is None and all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize('R,P,widths', [(63, 3, (3, 50, 50, 1)), (6200, 6, (5, 7, 17, 33)), (300, 2, (1, 1, 1)), (90, 4, (127, 127, 3, 1))])
def test_chain_of_any_width(R, P, widths):
    acts = ['silu', 'tanh', 'cos'][:len(widths) - 1]
    if widths[-1] == 1:
        acts[-1] = None
    print(f'case chain R={R} P={P} widths={widths}', flush=True)
    t, layers = make(R, P, widths, acts, 1)
    got, _ = K.dense_chain([(a, dev(W), dev(b), prm) for a, W, b, prm in layers], *[dev(v) for v in t])
    ref = [v.astype(np.float64) for v in t]
    for a, W, b, prm in layers:
        ref = rules.dense_rule(*ref, W.astype(np.float64), None if b is None else b.astype(np.float64))
        if a is not None:
            ref = rules.elementwise_rule(a, *ref)
    assert_val(got[0], ref[0], 'x')
    assert_val(got[1], ref[1], 'jacobian')
    assert_lap(got[2], ref[2], 'laplacian')


def test_a_position_without_finite_values_stays_alone():
    """Infinite inputs reach their own position only, and columns past a width do not carry them on."""
    t, layers = make(100, 4, (4, 20, 33, 20), ['tanh', 'tanh', 'tanh'], 2)
    layers = [(a, dev(W), dev(b), prm) for a, W, b, prm in layers]
    clean, _ = K.dense_chain(layers, *[dev(v) for v in t])
    t[0][17, 0] = np.inf                        # tanh: values of +-1, derivatives 0
    got, _ = K.dense_chain(layers, *[dev(v) for v in t])
    keep = torch.arange(100) != 17
    for a, b in zip(got, clean):
        assert torch.equal(a[..., keep, :], b[..., keep, :])
    assert torch.isfinite(got[0]).all() and (got[1][:, 17] == 0).all()


def test_front_door_chains_what_nobody_else_reads():
    """A layer that is read twice is evaluated for itself; the values are those of the layers one by one either way."""
    g = torch.Generator(device='cuda').manual_seed(3)
    Ws = [torch.randn(a, b, device='cuda', generator=g) / a ** 0.5 for a, b in ((4, 24), (24, 24), (24, 24), (24, 1))]
    x = torch.randn(9, 11, 4, device='cuda', generator=g)
    chains = []

    def fn(r, read_twice, explicit):
        h = r
        for i, W in enumerate(Ws[:3]):
            h = fnp.dot(h, W, act='silu') if explicit else fnp.silu(fnp.dot(h, W))
            if i == 1:
                kept = h if read_twice else None
        out = fnp.sum(fnp.dot(h, Ws[3]))
        return fnp.add(out, fnp.sum(kept)) if read_twice else out

    orig = K.dense_chain
    for twice in (False, True):
        run = lambda explicit: folx_amd.vmap(folx_amd.forward_laplacian(lambda r: fn(r, twice, explicit), 6))(x)
        want = run(True)
        chains.clear()
        K.dense_chain = lambda layers, *a: (chains.append(len(layers)), orig(layers, *a))[1]
        try:
            got = run(False)
        finally:
            K.dense_chain = orig
        assert chains == ([2, 2] if twice else [4]), chains
        assert torch.equal(got.x, want.x) and torch.equal(got.laplacian, want.laplacian)
        assert torch.equal(got.jacobian.dense_array, want.jacobian.dense_array)


@pytest.mark.parametrize('B,widths', [(3, (4, 100)), (3, (4, 24, 24)), (8000, (4, 4, 128))])
def test_layers_of_an_input_off_a_16_byte_boundary(B, widths):
    """One layer, layers in one launch, layers whose chain would be slower: the results of an aligned array."""
    print(f'case layers off the boundary B={B} widths={widths}', flush=True)
    g = torch.Generator(device='cuda').manual_seed(5)
    Ws = [torch.randn(a, b, device='cuda', generator=g) / a ** 0.5 for a, b in zip(widths, widths[1:])]

    def fn(r):
        for W in Ws:
            r = fnp.tanh(fnp.dot(r, W))
        return fnp.sum(r)

    fl = folx_amd.vmap(folx_amd.forward_laplacian(fn, 4))
    x = torch.randn(B * 50 * 4 + 1, device='cuda', generator=g)[1:].reshape(B, 50, 4)
    got, want = fl(x), fl(x.clone())
    assert torch.equal(got.x, want.x) and torch.equal(got.laplacian, want.laplacian)
    assert torch.equal(got.jacobian.dense_array, want.jacobian.dense_array)


def test_chain_with_a_large_tile_under_graph_replay():
    """More than 64 KB of LDS (P = 6, 128 features, 16 positions a workgroup): every replay returns the bits of the eager call."""
    print('case captured chain R=6200 P=6 128 x 128 x 128', flush=True)
    t, layers = make(6200, 6, (128, 128, 128), ['tanh', 'silu'], 4)
    layers = [(a, dev(W), dev(b), prm) for a, W, b, prm in layers]
    t = [dev(v) for v in t]
    K.dense_chain(layers, *t)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, _ = K.dense_chain(layers, *t)
    for call in range(3):
        for v in t:
            v.mul_(1.1)
        graph.replay()
        torch.cuda.synchronize()
        want, _ = K.dense_chain(layers, *t)
        assert all(torch.equal(a, b) for a, b in zip(out, want)), call
