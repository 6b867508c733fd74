"""LayerNorm over few features, where a wavefront holds several rows side by side: around the widths at which the number of rows
changes, rows that do not fill the last workgroup, one wavefront a row (P <= 8) and four."""

import numpy as np
import pytest
import torch

from oracle import backend as ob
from tolerances import assert_lap, assert_val

from folx_amd import kernels as K

pytestmark = pytest.mark.gpu
dev = lambda v: torch.as_tensor(np.asarray(v, dtype=np.float32)).cuda()


@pytest.mark.parametrize('F', [4, 32, 36, 64, 68, 128, 132])
@pytest.mark.parametrize('R,P', [(1, 0), (3, 4), (33, 8), (7, 9), (31, 48), (17, 21)])
def test_layernorm_rows_side_by_side(F, R, P):
    print(f'case layernorm R={R} P={P} F={F}', flush=True)
    g = np.random.default_rng(100 * R + F)
    x, J, L, ga, be = (g.normal(size=s).astype(np.float32) for s in ((R, F), (P, R, F), (R, F), (F,), (F,)))
    x *= 1 + np.arange(R)[:, None]          # every row its own scale: a sum that strays into a neighbour shows
    f = lambda v: v.astype(np.float64)
    ref = ob.layer_norm(ob.OArr(f(x), f(J), f(L)), f(ga), f(be), 1e-5)
    got = K.layernorm(dev(x), dev(J), dev(L), dev(ga), dev(be), 1e-5)
    assert_val(got[0], ref.x, 'x')
    assert_val(got[1], ref.J, 'jacobian')
    assert_lap(got[2], ref.lap, 'laplacian')
