"""LayerNorm + Dense as one kernel and as the two rules apart: on either side of the line between them, with cut tiles and partial
groups of Jacobian rows, against the float64 oracle on the first and last positions (the rule acts on each position alone)."""

import numpy as np
import pytest
import torch

from oracle import backend as ob
from oracle import rules
from tolerances import assert_lap, assert_val

from folx_amd import _lib
from folx_amd import kernels as K

pytestmark = pytest.mark.gpu
LIMIT = 14 << 20     # floats of the normalised triplet
ROWS_ACT = 8192


@pytest.mark.parametrize('R,P,Kd,N,act,apart', [
    (856, 33, 512, 132, None, False), (812, 33, 512, 132, None, True),        # the line at K = 512, a cut column tile
    (896, 62, 256, 256, None, True), (900, 62, 256, 256, None, False),        # full groups but two rows
    (44000, 5, 48, 256, None, False), (16, 1, 16, 300, None, True), (12, 193, 64, 256, None, False),
    (40, 64, 64, 256, None, True), (40, 65, 64, 256, None, False),            # the line at 64 Jacobian rows
    (260, 30, 64, 192, 'tanh', False), (256, 30, 64, 192, 'tanh', True), (124, 64, 48, 256, 'silu', True),
    (8, 65, 80, 132, 'sin', False), (300, 40, 512, 512, 'gelu', False), (4, 2, 16, 136, 'tanh', True),
])
def test_norm_dense_form(R, P, Kd, N, act, apart):
    print(f'case norm_dense R={R} P={P} K={Kd} N={N} act={act} apart={apart}', flush=True)
    assert apart == (P <= 64 and ((P + 2) * R * Kd <= LIMIT if act is None else (P + 2) * R <= ROWS_ACT))
    nbytes = _lib.load().folx_hip_norm_dense_workspace_bytes(R, P, Kd, N, -1 if act is None else _lib.ACT[act])
    triplet = 4 * (P + 2) * R * Kd
    if act is None:
        assert (nbytes == triplet) == apart
    assert nbytes >= triplet or not apart
    if apart:
        assert nbytes <= _lib.STATIC_SCRATCH_BYTES
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
