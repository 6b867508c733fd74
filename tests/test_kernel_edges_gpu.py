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


# both together, every block count of features; 48: three blocks on the instance for four
@pytest.mark.parametrize('B,n,H,d,P', [(2, 13, 4, 64, 39), (3, 16, 2, 48, 7), (1, 16, 1, 36, 17), (5, 3, 3, 20, 9), (70, 9, 3, 8, 12),
                                       (2, 5, 2, 64, 0), (2, 17, 2, 64, 5)])
def test_mhsa_short_sequences_bias_and_masks(B, n, H, d, P):
    test_mhsa_short_sequences(B, n, H, d, P, True, True)


# outputs that start at any float: single stores for 16 features, the general kernel beyond; what lies around them is kept
@pytest.mark.parametrize('n,H,d,P', [(16, 2, 64, 5), (13, 3, 32, 9), (7, 2, 20, 3), (5, 1, 16, 8), (20, 2, 64, 3)])
@pytest.mark.parametrize('edge', [False, True])
def test_mhsa_outputs_off_the_16_byte_boundary(n, H, d, P, edge):
    from folx_amd import _lib

    print(f'case mhsa unaligned outputs n={n} H={H} d={d} P={P} edge={edge}', flush=True)
    rng = np.random.default_rng(d)
    B = 2
    args = []
    for s in (1 / np.sqrt(d), 1.0, 1.0):
        args += [s * rand(rng, B, n, H, d), s * rand(rng, P, B, n, H, d), s * rand(rng, B, n, H, d)]
    e = [rand(rng, B, n, H, n), rand(rng, P, B, n, H, n), rand(rng, B, n, H, n)] if edge else []
    ref = rules.mhsa_rule(*f64(*args), np.ones((B, n), dtype=bool), np.ones((P, B), dtype=bool), *f64(*(e or [None] * 3)))
    ins = [dev(t) for t in args[:6] + e + args[6:]]
    size = B * n * H * d
    outs = [torch.full((m + 8,), 7.0, device='cuda') for m in (size, P * size, size)]
    fn = _lib.load().folx_hip_mhsea_fwdlap if edge else _lib.load().folx_hip_mhsa_fwdlap
    _lib.check(fn(torch.cuda.current_stream().cuda_stream, *[t.data_ptr() for t in ins], None, None,
                  *[t.data_ptr() + 4 * (i + 1) for i, t in enumerate(outs)], B, n, H, d, P), 'mhsa')
    got = [t[i + 1:i + 1 + m] for i, (t, m) in enumerate(zip(outs, (size, P * size, size)))]
    assert_val(got[0].reshape(ref[0].shape), ref[0], 'o')
    assert_val(got[1].reshape(ref[1].shape), ref[1], 'o_jac')
    assert_lap(got[2].reshape(ref[2].shape), ref[2], 'o_lap')
    for i, (t, m) in enumerate(zip(outs, (size, P * size, size))):
        assert bool((t[:i + 1] == 7.0).all()) and bool((t[i + 1 + m:] == 7.0).all())


# up to 32 x 32 x 32 one wavefront per batch element (1 / 4 / 8 sharing the Jacobian rows), 33: the tiled form; pieces of
# four k whole and aligned or not, rows of y whole or not
@pytest.mark.parametrize('NB0,NB1,I,J,Kc,P', [(3, 2, 16, 16, 16, 39), (1, 1, 17, 32, 20, 8), (2, 3, 32, 17, 32, 9),
                                              (200, 1, 4, 16, 30, 17), (2, 2, 15, 5, 31, 16), (1, 3, 32, 32, 1, 0),
                                              (2, 1, 1, 1, 17, 7), (2, 2, 33, 8, 8, 9), (5, 2, 24, 12, 4, 12)])
@pytest.mark.parametrize('layout', ['contiguous', 'interleaved', 'offset'])
def test_dot_two_small_products(NB0, NB1, I, J, Kc, P, layout):
    from folx_amd import kernels as K

    print(f'case dot_two NB=({NB0},{NB1}) I={I} J={J} K={Kc} P={P} {layout}', flush=True)
    rng = np.random.default_rng(I * 100 + J)
    a = [rand(rng, *s, NB0, NB1, I, Kc) for s in ((), (P,), ())]
    b = [rand(rng, *s, NB0, NB1, Kc, J) for s in ((), (P,), ())]
    ref = rules.dot_two_rule(*f64(*a, *b))

    def lay(t, transposed):
        if layout == 'contiguous':
            return dev(t)
        if layout == 'offset':  # rows that start off the 16-byte boundary
            return torch.nn.functional.pad(dev(t), (1, 2))[..., 1:-2]
        t = np.swapaxes(t, -1, -2) if transposed else t  # (walker, position, head, feature), b as k^T
        t = dev(np.swapaxes(t, -3, -2)).transpose(-3, -2)
        return t.transpose(-1, -2) if transposed else t

    got = K.dot_two(*[lay(t, False) for t in a], *[lay(t, True) for t in b])
    assert_val(got[0], ref[0], 'y')
    assert_val(got[1], ref[1], 'y_jac')
    assert_lap(got[2], ref[2], 'y_lap')
    W = rand(rng, NB1, Kc, J)
    ref = rules.dot_const_rule(*f64(*a, W))
    got = K.dot_const(*[lay(t, False) for t in a], dev(W))
    assert_val(got[0], ref[0], 'y')
    assert_val(got[1], ref[1], 'y_jac')
    assert_lap(got[2], ref[2], 'y_lap')


# groups of 1 .. 64 lanes per output, 128-bit pieces or single values, one or four outputs per group in flight
@pytest.mark.parametrize('total,span,lo,hi', [(5, 16, 0, 16), (7, 17, 0, 17), (3, 40, 4, 36), (3, 40, 3, 36), (1, 1000, 0, 1000),
                                              (9, 999, 1, 998), (524288 + 3, 16, 0, 16), (33000, 260, 0, 260), (131072, 19, 1, 18)])
def test_reduce_last_axis(total, span, lo, hi):
    from folx_amd import kernels as K

    print(f'case reduce_last total={total} span={span} window=({lo},{hi})', flush=True)
    x = rand(np.random.default_rng(span), 1, total, span, 1)
    got = K.reduce_sum(dev(x), 1, total, span, 1, 0.5, (lo, hi)).reshape(total)
    ref = 0.5 * x[0, :, lo:hi, 0].astype(np.float64).sum(axis=1)
    # each addend passes at most (hi - lo) rounded additions
    bound = (hi - lo) * 2.0 ** -24 * 0.5 * np.abs(x[0, :, lo:hi, 0].astype(np.float64)).sum(axis=1) + 1e-30
    assert (np.abs(got.cpu().numpy() - ref) <= bound).all()
    if (lo, hi) == (0, span):
        m = K.reduce_max(dev(x), total, span, 1)
        assert torch.equal(m.reshape(total).cpu(), torch.as_tensor(x[0, :, :, 0].max(axis=1)))


# 64 x 64 tiles where larger ones would leave CUs idle: cut row and column tiles in every segment, one chunk of K, skip connection
@pytest.mark.parametrize('rows,P,Kd,N', [((1, 1), 1, 16, 68), ((3, 21), 2, 48, 100), ((1, 64), 3, 32, 128), ((5, 13), 9, 256, 132),
                                         ((2, 65), 7, 64, 300), ((40, 10), 30, 256, 256)])
def test_dense_small_tiles(rows, P, Kd, N):
    from folx_amd import kernels as K

    print(f'case dense rows={rows} P={P} K={Kd} N={N}', flush=True)
    rng = np.random.default_rng(N)
    t = [rand(rng, *rows, Kd), rand(rng, P, *rows, Kd), rand(rng, *rows, Kd)]
    W, b = (rand(rng, Kd, N) / np.sqrt(Kd)).astype(np.float32), rand(rng, N)
    res = [rand(rng, *rows, N), rand(rng, P, *rows, N), rand(rng, *rows, N)]
    ref = rules.dense_rule(*f64(*t, W, b))
    for skip in (None, tuple(dev(r) for r in res)):
        got = K.dense(*[dev(v) for v in t], dev(W), dev(b), skip)
        want = ref if skip is None else [a + r for a, r in zip(ref, res)]
        assert_val(got[0], want[0], 'y')
        assert_val(got[1], want[1], 'y_jac')
        assert_lap(got[2], want[2], 'y_lap')


# wide dense + activation: the last tile's positions and the last group's rows cut, operand whole or in parts with a per-walker term
# and a skip connection (which form each size takes is pinned below)
@pytest.mark.parametrize('rows,P,N', [((1, 4), 6, 132), ((515, 4), 21, 256), ((66, 16), 39, 300), ((164, 13), 24, 256), ((1030, 4), 8, 260),
                                      ((60, 4), 33, 256), ((521, 4), 13, 256)])
def test_dense_act_groups_of_eight(rows, P, N):
    from folx_amd import kernels as K

    print(f'case dense_act rows={rows} P={P} N={N}', flush=True)
    rng = np.random.default_rng(P)
    B, n = rows
    parts = [rand(rng, P, *rows, 32), rand(rng, P, *rows, 48)]
    x, J, L = rand(rng, *rows, 80), np.concatenate(parts, -1), rand(rng, *rows, 80)
    W, b = (rand(rng, 80, N) / np.sqrt(80)).astype(np.float32), rand(rng, N)
    z = rules.dense_rule(*f64(x, J, L, W, b))
    ref = rules.elementwise_rule('tanh', *z)
    got = K.dense_act('tanh', dev(x), dev(J), dev(L), dev(W), dev(b))
    assert_val(got[0], ref[0], 'y')
    assert_val(got[1], ref[1], 'y_jac')
    assert_lap(got[2], ref[2], 'y_lap')
    pre = [rand(rng, B, N), rand(rng, P, B, N), rand(rng, B, N)]
    res = [rand(rng, *rows, N), rand(rng, P, *rows, N), rand(rng, *rows, N)]
    ref = rules.elementwise_rule('tanh', *[t + np.expand_dims(q, -2).astype(np.float64) for t, q in zip(z, pre)])
    got = K.dense_act_parts('tanh', dev(x), dev(L), [dev(t) for t in parts], (32, 48), (0, 0), n, dev(W), dev(b), 0.0,
                            tuple(dev(t) for t in res), tuple(dev(t) for t in pre))
    assert_val(got[0], ref[0] + res[0], 'y')
    assert_val(got[1], ref[1] + res[1], 'y_jac')
    assert_lap(got[2], ref[2] + res[2], 'y_lap')


# groups of 8 Jacobian rows (16 positions a tile, four per accumulator block), of 16 (8 positions, two per block) and of 32, each
# with and without a cut last tile and a cut last group, in both product modes
@pytest.mark.parametrize('mode', ['f32', 'bf16x3'])
@pytest.mark.parametrize('rows,P,N,form', [((257, 4), 21, 132, 8), ((130, 4), 24, 260, 8), ((66, 8), 21, 260, 8), ((257, 4), 21, 256, 8),
                                           ((129, 4), 9, 260, 16), ((63, 8), 9, 132, 16), ((271, 4), 45, 260, 16), ((125, 4), 9, 132, 32),
                                           ((64, 16), 96, 256, 32)])
def test_dense_act_group_forms(mode, rows, P, N, form):
    from folx_amd import _lib
    from folx_amd import kernels as K

    before = K.get_gemm_mode()
    K.set_gemm_mode(mode)
    try:
        assert _lib.load().folx_hip_dense_act_form(rows[0] * rows[1], P, 80, N, 0) == form
        print(f'mode {mode}', flush=True)
        test_dense_act_groups_of_eight(rows, P, N)
    finally:
        K.set_gemm_mode(before)


# up to six Jacobian rows (with a skip connection always the kernel for them, without one where it is the faster):
# 1 .. 8 blocks of 16 columns and of 16 positions a workgroup, the last ones cut; features in whole
# groups of 16, with a rest, or only a rest; one column short of a 128-bit store; outputs off the 16-byte boundary
@pytest.mark.parametrize('R,P,Kd,N', [(1, 0, 4, 1), (17, 1, 12, 16), (31, 2, 16, 17), (2000, 4, 100, 100), (16, 6, 128, 128),
                                      (9000, 3, 36, 30), (66000, 6, 32, 32), (15, 5, 20, 127), (8191, 2, 64, 48), (33, 6, 112, 64)])
@pytest.mark.parametrize('act', ['tanh', 'silu'])
def test_dense_act_few_jacobian_rows(R, P, Kd, N, act):
    from folx_amd import kernels as K

    print(f'case dense_act R={R} P={P} K={Kd} N={N} {act}', flush=True)
    rng = np.random.default_rng(R + N)
    t = [rand(rng, R, Kd), rand(rng, P, R, Kd), rand(rng, R, Kd)]
    W, b = (rand(rng, Kd, N) / np.sqrt(Kd)).astype(np.float32), rand(rng, N)
    res = [rand(rng, R, N), rand(rng, P, R, N), rand(rng, R, N)]
    ref = rules.elementwise_rule(act, *rules.dense_rule(*f64(*t, W, b)))

    def off_boundary(a):
        return torch.nn.functional.pad(dev(a).reshape(-1), (1, 0))[1:].reshape(a.shape)

    for skip in (None, tuple(dev(r) for r in res), tuple(off_boundary(r) for r in res)):
        got = K.dense_act(act, *[dev(v) for v in t], dev(W), dev(b), 0.0, skip)
        want = ref if skip is None else [a + r for a, r in zip(ref, res)]
        assert_val(got[0], want[0], 'y')
        if P:
            assert_val(got[1], want[1], 'y_jac')
        assert_lap(got[2], want[2], 'y_lap')
    # a row holds its own position alone: infinities of one do not reach another
    bad = [v.copy() for v in t]
    for v in bad:
        v[..., R // 2, :] = np.inf
    got = K.dense_act(act, *[dev(v) for v in bad], dev(W), dev(b))
    keep = np.arange(R) != R // 2
    assert_val(got[0][keep], ref[0][keep], 'y')
    assert_lap(got[2][keep], ref[2][keep], 'y_lap')
