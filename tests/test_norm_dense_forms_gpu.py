"""LayerNorm + Dense as one rule from a few positions to many, with cut tiles and partial groups of Jacobian rows: against the
float64 oracle on the first and last positions (the rule acts on each position alone), and independent of their number."""

import numpy as np
import pytest
import torch

from oracle import backend as ob
from oracle import rules
from tolerances import assert_lap, assert_val

from folx_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('R,P,Kd,N,act', [
    (856, 33, 512, 132, None), (812, 33, 512, 132, None),        # a cut column tile, one row in the last group
    (896, 62, 256, 256, None), (900, 62, 256, 256, None),        # full groups but two rows
    (44000, 5, 48, 256, None), (16, 1, 16, 300, None), (12, 193, 64, 256, None),
    (40, 64, 64, 256, None), (40, 65, 64, 256, None),
    (260, 30, 64, 192, 'tanh'), (256, 30, 64, 192, 'tanh'), (124, 64, 48, 256, 'silu'),
    (8, 65, 80, 132, 'sin'), (300, 40, 512, 512, 'gelu'), (4, 2, 16, 136, 'tanh'),
])
def test_norm_dense_form(R, P, Kd, N, act):
    print(f'case norm_dense R={R} P={P} K={Kd} N={N} act={act}', flush=True)
    g = torch.Generator(device='cuda').manual_seed(R + P)
    rn = lambda *s: torch.randn(*s, device='cuda', generator=g)
    x, J, L = rn(R, Kd) + 0.5, rn(P, R, Kd) + 0.3 * rn(P, R, 1), rn(R, Kd)
    ga, be, W, b = 1 + 0.3 * rn(Kd), 0.2 * rn(Kd), rn(Kd, N) / Kd ** 0.5, rn(N)
    got = K.norm_dense(act, x, J, L, ga, be, 1e-5, W, b)
    at = sorted({*range(min(R, 9)), *range(max(0, R - 9), R)})
    f = lambda t: t.cpu().numpy().astype(np.float64)
    h = ob.layer_norm(ob.OArr(f(x[at]), f(J[:, at]), f(L[at])), f(ga), f(be), 1e-5)
    ref = rules.dense_rule(h.x, h.J, h.lap, f(W), f(b))
    if act is not None:
        ref = rules.elementwise_rule(act, *ref)
    assert_val(got[0][at], ref[0], 'x')
    assert_val(got[1][:, at], ref[1], 'jacobian')
    assert_lap(got[2][at], ref[2], 'laplacian')


@pytest.mark.parametrize('act', [None, 'tanh'])
@pytest.mark.parametrize('P,Kd,N', [(30, 256, 256), (60, 256, 256), (64, 64, 192), (96, 512, 256)])
def test_a_position_does_not_depend_on_how_many_there_are(P, Kd, N, act):
    """The bits of the first positions are those of a call on them alone, from a few walkers' worth to a full chunk."""
    print(f'case norm_dense positions P={P} K={Kd} N={N} act={act}', flush=True)
    g = torch.Generator(device='cuda').manual_seed(P)
    rn = lambda *s: torch.randn(*s, device='cuda', generator=g)
    R = 4096
    x, J, L = rn(R, Kd) + 0.5, rn(P, R, Kd) + 0.3 * rn(P, R, 1), rn(R, Kd)
    consts = 1 + 0.3 * rn(Kd), 0.2 * rn(Kd), 1e-5, rn(Kd, N) / Kd ** 0.5, rn(N)
    full = K.norm_dense(act, x, J, L, *consts)
    for r in (4, 64, 640, 1024):
        part = K.norm_dense(act, x[:r].contiguous(), J[:, :r].contiguous(), L[:r].contiguous(), *consts)
        assert torch.equal(part[0], full[0][:r]) and torch.equal(part[1], full[1][:, :r]) and torch.equal(part[2], full[2][:r]), r
