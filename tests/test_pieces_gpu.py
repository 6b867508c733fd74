"""Wide layers with their products from bf16 pieces: tiles of every width and their edges, sums of more than 512 products, elements
that have no pieces, the error against float64, and the same bits for a row whatever else a call holds."""

import numpy as np
import pytest
import torch

from oracle import rules
from tolerances import assert_triplet

pytestmark = pytest.mark.gpu


def rand(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


def dev(a):
    return None if a is None else torch.as_tensor(np.ascontiguousarray(a), device='cuda')


def f64(*arrs):
    return tuple(np.asarray(a, dtype=np.float64) for a in arrs)


@pytest.mark.parametrize('R,P,Kd,N,res', [
    (1, 1, 16, 132, False),      # one row of a tile, one chunk, a cut block of columns
    (3, 2, 48, 160, False),      # an odd number of chunks, whole blocks only
    (130, 3, 128, 300, True),    # two row tiles, a skip connection in cut blocks
    (129, 9, 256, 512, True),    # a row past a tile
    (900, 40, 144, 260, False),  # 4 blocks a tile, the last with 4 columns
    (2048, 40, 256, 256, True),  # 8 blocks, W's pieces by a launch of their own
    (2050, 40, 528, 136, False), # more than 512 products a sum
    (60, 5, 832, 200, True),
    (33, 3, 144, 36, True),      # narrow layers with long sums
    (2048, 40, 256, 64, False),
    (4100, 30, 256, 112, True),
    (700, 7, 592, 128, False),
])
def test_dense_tiles(R, P, Kd, N, res):
    from folx_amd import kernels as K

    print(f'case R={R} P={P} K={Kd} N={N} res={res}', flush=True)
    rng = np.random.default_rng(7)
    x, J, L = rand(rng, R, Kd), rand(rng, P, R, Kd), rand(rng, R, Kd)
    W, b = (rand(rng, Kd, N) / np.sqrt(Kd)).astype(np.float32), rand(rng, N)
    r = (rand(rng, R, N), rand(rng, P, R, N), rand(rng, R, N)) if res else None
    ref = rules.dense_rule(*f64(x, J, L, W), b.astype(np.float64))
    if res:
        ref = tuple(a + c for a, c in zip(ref, f64(*r)))
    got = K.dense(dev(x), dev(J), dev(L), dev(W), dev(b), None if r is None else tuple(map(dev, r)))
    assert_triplet(got, ref, 'dense')


@pytest.mark.parametrize('R,P,Kd,N', [(4, 1, 16, 132), (8, 40, 64, 160), (260, 33, 256, 300), (1024, 96, 256, 256), (516, 9, 528, 260)])
def test_activation_forms(R, P, Kd, N):
    """Both widths of the fused tiles, groups of 8 to 32 Jacobian rows, whole and cut blocks."""
    from folx_amd import kernels as K

    print(f'case R={R} P={P} K={Kd} N={N}', flush=True)
    rng = np.random.default_rng(8)
    x, J, L = rand(rng, R, Kd), rand(rng, P, R, Kd), rand(rng, R, Kd)
    W, b = (rand(rng, Kd, N) / np.sqrt(Kd)).astype(np.float32), rand(rng, N)
    ref = rules.elementwise_rule('tanh', *rules.dense_rule(*f64(x, J, L, W), b.astype(np.float64)))
    assert_triplet(K.dense_act('tanh', dev(x), dev(J), dev(L), dev(W), dev(b)), ref, 'dense_act')


@pytest.mark.parametrize('Kd', [64, 256, 832])
def test_error_is_below_that_of_fp32_sums(Kd):
    """rms error against float64 below that of a float32 sum of the same products one after the other, whose K roundings of
    partial sums that grow like sqrt(k) leave K / sqrt(2) * 2^-24 / sqrt(3) / sqrt(K) of the result's rms (the fp32 matrix
    instructions round half as often: a factor of sqrt(2) less, which is the bar here)."""
    from folx_amd import kernels as K

    g = torch.Generator(device='cuda').manual_seed(5)
    x, J = torch.randn(256, Kd, device='cuda', generator=g), torch.randn(20, 256, Kd, device='cuda', generator=g)
    W = torch.randn(Kd, 256, device='cuda', generator=g) / Kd ** 0.5
    got = K.dense(x, J, x, W)[1].double()
    ref = J.double() @ W.double()
    err = float((got - ref).norm() / ref.norm())
    print('rms error', Kd, err, flush=True)
    assert err < 0.5 * Kd ** 0.5 * 2.0 ** -24 / 3 ** 0.5


@pytest.mark.parametrize('R', [8, 4096])  # W split in the tiles, and prepared
def test_elements_without_pieces(R):
    """Infinities, NaN and numbers next to FLT_MAX give what float32 products of them give, and leave other rows alone."""
    from folx_amd import kernels as K

    g = torch.Generator(device='cuda').manual_seed(6)
    Kd, N, P = 128, 192, 4
    x, J, L = (torch.randn(*s, device='cuda', generator=g) for s in ((R, Kd), (P, R, Kd), (R, Kd)))
    W = torch.randn(Kd, N, device='cuda', generator=g) / Kd ** 0.5
    clean = K.dense(x, J, L, W)
    big = float(np.finfo(np.float32).max)
    J[0, 1, 3], J[1, 2, 5], J[2, 3, 7], J[3, 4] = float('inf'), float('nan'), big, 0.0
    J[3, 4, 9] = -float('inf')
    W2 = W.clone()
    W2[7] *= 1e-3  # big * W stays finite
    got = K.dense(x, J, L, W2)[1]
    ref = (J.double() @ W2.double()).float()
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
    assert torch.equal(got[torch.isinf(ref)], ref[torch.isinf(ref)])
    torch.testing.assert_close(got[2, 3], ref[2, 3], rtol=1e-5, atol=0)
    assert torch.equal(K.dense(x, J, L, W)[1][:, R // 2 + 3:], clean[1][:, R // 2 + 3:])
    W3 = W.clone()
    W3[2, 5], W3[4, 9] = float('inf'), big
    x3 = x.clone()
    x3[:, 4] *= 1e-3
    got, ref = K.dense(x3, J[:1] * 0 + 1e-3, L, W3)[0], (x3.double() @ W3.double()).float()
    assert torch.equal(torch.isinf(got), torch.isinf(ref))
    torch.testing.assert_close(got[:, [0, 9]], ref[:, [0, 9]], rtol=2e-4, atol=1e-4)


@pytest.mark.parametrize('Kd,N', [(32, 160), (256, 256), (832, 200), (256, 80)])
def test_rows_do_not_depend_on_the_call(Kd, N):
    """Value and Jacobian rows of a position: the same bits among 4, 300 and 5000 others, with and without the fused activation."""
    from folx_amd import kernels as K

    g = torch.Generator(device='cuda').manual_seed(9)
    P, R = 33, 5000
    x, J, L = (torch.randn(*s, device='cuda', generator=g) for s in ((R, Kd), (P, R, Kd), (R, Kd)))
    W, b = torch.randn(Kd, N, device='cuda', generator=g) / Kd ** 0.5, torch.randn(N, device='cuda', generator=g)
    whole = K.dense(x, J, L, W, b)
    if N > 128:
        act = K.dense_act('tanh', x, J, L, W, b)
        apart = K.elementwise('tanh', *whole)
        assert torch.equal(act[0], apart[0]) and torch.equal(act[1], apart[1])
    for n in (4, 300):
        part = [t.contiguous() for t in (x[:n], J[:, :n], L[:n])]
        some = K.dense(*part, W, b)
        assert torch.equal(some[0], whole[0][:n]) and torch.equal(some[1], whole[1][:, :n]) and torch.equal(some[2], whole[2][:n])
        if N > 128:
            some = K.dense_act('tanh', *part, W, b)
            assert torch.equal(some[0], act[0][:n]) and torch.equal(some[1], act[1][:, :n])
