"""GELU (both forms) as one function: the elementwise rule and the fused dense + activation rules against the float64 oracle,
for arguments from the flat tail to the linear range."""

import numpy as np
import pytest
import torch

from oracle import rules
from tolerances import assert_lap, assert_val

import folx_amd
from folx_amd import kernels as K
from folx_amd import numpy as fnp

pytestmark = pytest.mark.gpu
dev = lambda v: torch.as_tensor(np.asarray(v, dtype=np.float32)).cuda()


def compare(got, ref, what):
    assert_val(got[0], ref[0], what + ' x')
    assert_val(got[1], ref[1], what + ' jacobian')
    assert_lap(got[2], ref[2], what + ' laplacian')


@pytest.mark.parametrize('name', ['gelu', 'gelu_tanh'])
@pytest.mark.parametrize('shape,P', [((1, 1), 0), ((3, 5), 2), ((7, 64), 48)])
def test_elementwise_gelu(name, shape, P):
    print(f'case {name} {shape} P={P}', flush=True)
    g = np.random.default_rng(0)
    x = g.uniform(-7, 7, size=shape).astype(np.float32)
    J, L = g.normal(size=(P, *shape)).astype(np.float32), g.normal(size=shape).astype(np.float32)
    ref = rules.elementwise_rule(name, *[v.astype(np.float64) for v in (x, J, L)])
    compare(K.elementwise(name, dev(x), dev(J), dev(L)), ref, name)


# narrow general and few-rows kernels, the wide kernel
@pytest.mark.parametrize('name', ['gelu', 'gelu_tanh'])
@pytest.mark.parametrize('rows,P,k,n', [((2, 40), 30, 64, 128), ((3, 7), 4, 20, 36), ((4, 8), 32, 64, 256)])
def test_dense_gelu(name, rows, P, k, n):
    print(f'case dense {name} {rows} P={P} {k} x {n}', flush=True)
    g = np.random.default_rng(1)
    t = [g.normal(size=s).astype(np.float32) for s in ((*rows, k), (P, *rows, k), (*rows, k))]
    W, b = (g.normal(size=(k, n)) / np.sqrt(k)).astype(np.float32), g.normal(size=n).astype(np.float32)
    z = rules.dense_rule(*[v.astype(np.float64) for v in (*t, W, b)])
    compare(K.dense_act(name, *[dev(v) for v in t], dev(W), dev(b)), rules.elementwise_rule(name, *z), name)


# elementwise (no layer), narrow few-rows and general kernels, the wide kernel
@pytest.mark.parametrize('name', ['gelu', 'gelu_tanh'])
@pytest.mark.parametrize('P,k,n', [(2, None, None), (2, 4, 8), (9, 16, 64), (32, 16, 256)])
def test_gelu_far_from_zero(name, P, k, n):
    """Where the function is x or 0 in float32 its derivatives are 1 or 0 and 0, up to the largest numbers: a factor that has
    underflowed meets no overflow."""
    print(f'case {name} far from zero, P={P} {k} x {n}', flush=True)
    x = np.array([s * v for v in (20.0, 1e3, 1e8, 2e9, 2e10, 1e15, 1e18, 3e19, 1e30, 3e38, 1e2, 1e12) for s in (1, -1)], np.float32)
    y, d = np.where(x > 0, x, 0), (x > 0).astype(np.float32)
    if k is None:
        got = K.elementwise(name, dev(x), dev(np.ones((P, *x.shape))), dev(np.ones(x.shape)))
    else:
        feature = np.eye(1, k)[0]
        t = [dev(v[..., None] * feature) for v in (x, np.ones((P, *x.shape)), np.ones(x.shape))]
        got = K.dense_act(name, *t, dev(feature[:, None] * np.ones(n)))
        y, d = y[:, None], d[:, None]
    for a, want in zip(got, (y, d, d)):
        a = a.cpu().numpy()
        np.testing.assert_array_equal(a, np.broadcast_to(want, a.shape))


def off_the_boundary(t):
    """``t`` as a view into a larger array, 4 bytes behind a 16-byte boundary."""
    view = torch.empty(t.numel() + 1, device='cuda')[1:].reshape(t.shape)
    return view.copy_(t)


@pytest.mark.parametrize('k,n', [(4, 16), (32, 132), (20, 160), (256, 256)])
def test_gelu_layer_of_arrays_off_a_16_byte_boundary(k, n):
    """Weights, a skip connection and the input itself that a caller reads from a larger array: the results of aligned ones."""
    print(f'case gelu layer off the boundary {k} x {n}', flush=True)
    g = torch.Generator(device='cuda').manual_seed(k)
    rn = lambda *s: torch.randn(*s, device='cuda', generator=g)
    x, W, W2, b = rn(12, 4, k), rn(k, n) / k ** 0.5, rn(n + 32, k) / n ** 0.5, rn(n)

    def model(x, W, W2, b):
        h = fnp.gelu(fnp.add(fnp.dot(x, W), b), approximate=False)
        # a layer that reads a concatenation in parts where it is wide, with the input as its skip connection
        parts = fnp.concatenate([h, fnp.tanh(fnp.dot(x, W[:, :16].contiguous())), fnp.tanh(fnp.dot(x, W[:, -16:].contiguous()))], axis=-1)
        return fnp.add(x, fnp.gelu(fnp.dot(parts, W2)))

    run = lambda x, *weights: folx_amd.vmap(folx_amd.forward_laplacian(lambda t: model(t, *weights), 0))(x)
    want = run(x, W, W2, b)
    for at in range(4):
        got = run(*[off_the_boundary(t) if i == at else t for i, t in enumerate((x, W, W2, b))])
        for u, v in ((got.x, want.x), (got.jacobian.dense_array, want.jacobian.dense_array), (got.laplacian, want.laplacian)):
            # the plain product of unaligned operands adds in another order
            torch.testing.assert_close(u, v, rtol=1e-4, atol=1e-5 * float(v.abs().max()))
