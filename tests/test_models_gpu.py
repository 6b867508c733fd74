"""End-to-end GPU parity: whole models through the HIP path against the fp64 oracle on
the same seeded inputs, the Loop-Laplacian semantics (brute-force Hessian trace) on the
smallest configuration, and size-independent properties at the full benchmark size."""

import numpy as np
import pytest
import torch

from bruteforce import brute_force, plain
from oracle import backend as ob
from tolerances import assert_lap, assert_val

import folx_amd
from folx_amd import numpy as fnp
from folx_amd import workloads as wl

pytestmark = pytest.mark.gpu


def run(fn, x, thr):
    return folx_amd.vmap(folx_amd.forward_laplacian(lambda t: fn(fnp, t), thr))(x)


def check(fn, x, thr, what):
    print(f'case {what} thr={thr} x={x.shape}', flush=True)
    out = run(fn, x, thr)
    ref = fn(ob, ob.init_state(x, dtype=np.float64))
    J = out.jacobian.dense_array
    assert J.shape[0] <= ref.J.shape[0]
    assert_val(out.x, ref.x, what + ' x')
    assert_val(J, ref.J[: J.shape[0]], what + ' jacobian')
    if J.shape[0] < ref.J.shape[0]:
        assert np.abs(ref.J[J.shape[0]:]).max() == 0
    assert_lap(out.laplacian, ref.lap, what + ' laplacian')
    return out, ref


@pytest.mark.parametrize('thr', [0, 4])
def test_readme_mlp(thr):
    """The reference README MLP (README.md:41-70), dense and sparse, at full model size, 3 walkers."""
    params = wl.mlp_params(seed=0)
    x = np.random.default_rng(0).normal(size=(3, 100, 4)).astype(np.float32)
    fn = lambda xp, t: wl.mlp_forward(params, t, xp)
    out, _ = check(fn, x, thr, 'readme mlp')
    assert out.jacobian.dense_array.shape == (400, 3)


@pytest.mark.parametrize('parallel', [False, True])
def test_loop_laplacian_operator_on_smallest_config(parallel):
    """The README MLP at reduced size through LoopLaplacianOperator / ParallelLaplacianOperator
    (folx/operators.py:41-79; one pass per input coordinate with a single Jacobian row):
    their Hessian diagonal sums to the forward Laplacian of both storage modes, their
    gradient is its Jacobian (test/test_operator.py:19-73)."""
    params = wl.mlp_params(seed=0, in_dim=4, width=32, n_hidden=3)
    x = np.random.default_rng(5).normal(size=(3, 6, 4)).astype(np.float32)
    f = lambda t: wl.mlp_forward(params, t, fnp)
    op = folx_amd.ParallelLaplacianOperator() if parallel else folx_amd.LoopLaplacianOperator()
    print(f'case loop operator parallel={parallel}', flush=True)
    diag, grad = folx_amd.vmap(op(f))(x)
    assert diag.shape == (3, 24) and grad.shape == (3, 24)
    ref = wl.mlp_forward(params, ob.init_state(x, dtype=np.float64), ob)
    assert_lap(diag.sum(1), ref.lap, 'loop laplacian')
    assert_val(grad.T, ref.J, 'loop jacobian')
    for thr in (0, 4):
        lap, jac = folx_amd.vmap(folx_amd.ForwardLaplacianOperator(thr)(f))(x)
        assert_lap(lap, diag.sum(1).double().cpu().numpy(), 'forward vs loop laplacian')
        assert_val(jac, grad.double().cpu().numpy(), 'forward vs loop jacobian')


def test_readme_mlp_sparse_equals_dense():
    params = wl.mlp_params(seed=0)
    x = np.random.default_rng(1).normal(size=(8, 100, 4)).astype(np.float32)
    fn = lambda xp, t: wl.mlp_forward(params, t, xp)
    d, s = run(fn, x, 0), run(fn, x, 4)
    assert_val(s.x, d.x.cpu().numpy())
    assert_val(s.jacobian.dense_array, d.jacobian.dense_array.cpu().numpy())
    assert_lap(s.laplacian, d.laplacian.cpu().numpy())


SMALL = wl.PsiFormerConfig(n_elec=6, n_nuc=2, n_layers=2, n_heads=2, head_dim=8, width=16, mlp_width=16, n_det=3)


@pytest.mark.parametrize('thr', [0, 6])
def test_psiformer_small_vs_oracle_and_loop_laplacian(thr):
    p = wl.psiformer_params(SMALL)
    x = wl.sample_electrons(4, SMALL.n_elec, 1.0, seed=2)
    fn = lambda xp, t: wl.psiformer_forward(p, t, xp)
    out, ref = check(fn, x, thr, 'psiformer small')
    # LoopLaplacianOperator semantics (folx/operators.py:41-62): trace of the AD Hessian
    by, bJ, bL = brute_force(lambda t: fn(plain, t), x.astype(np.float64))
    assert_val(out.x, by), assert_val(out.jacobian.dense_array, bJ), assert_lap(out.laplacian, bL)


SMALL_FERMI = wl.FermiNetConfig(n_elec=6, n_nuc=2, n_layers=3, w1=16, w2=8, n_det=3)


@pytest.mark.parametrize('thr', [0, 6])
def test_ferminet_small_vs_oracle_and_loop_laplacian(thr):
    """The FermiNet-style configuration in miniature: sparse pair stream (k = 6), dense one-electron stream."""
    p = wl.ferminet_params(SMALL_FERMI)
    x = wl.sample_electrons(4, SMALL_FERMI.n_elec, 1.0, seed=3)
    fn = lambda xp, t: wl.ferminet_forward(p, t, xp)
    out, ref = check(fn, x, thr, 'ferminet small')
    by, bJ, bL = brute_force(lambda t: fn(plain, t), x.astype(np.float64))
    assert_val(out.x, by), assert_val(out.jacobian.dense_array, bJ), assert_lap(out.laplacian, bL)


@pytest.mark.parametrize('name', ['ferminet16', 'psiformer32', 'psiformer64'])
def test_psiformer_full_architecture_two_walkers(name):
    """The benchmark architectures at their real widths (P = 96 / 192), 2 walkers.

    log|det| of randomly initialised 16x16 / 32x32 orbital matrices amplifies fp32
    rounding: the numpy restatement of the same rules run in float32 already differs from
    its float64 run by ~3e-4 (Jacobian) and ~4e-4 (Laplacian) relative to the largest
    entry.  No fp32 implementation can meet rtol 1e-5 on this function, so the bar here is
    the noise floor itself: the HIP result must be as close to the fp64 oracle as the
    fp32 oracle is (factor 2 head-room).  The strict
    bars (values/Jacobians rtol 1e-5, Laplacians rtol 1e-4 + atol 1e-5) are enforced per
    kernel and on the well-conditioned models above."""
    forward, p, cfg, _, sigma, thr = wl.build(name)
    x = wl.sample_electrons(2, cfg.n_elec, sigma, seed=2)
    fn = lambda xp, t: forward(p, t, xp)
    print(f'case {name} full architecture', flush=True)
    from folx_amd import kernels as K

    with K.LaunchTimer() as lt:
        out = run(fn, x, thr)
    used = {}
    for (entry, key), (calls, _) in lt.summary().items():
        used[entry] = used.get(entry, 0) + calls
    if name.startswith('psiformer'):
        # the fused rules are the ones that run: LayerNorm inside 3 products of layers 2-4 and the
        # 4 MLP products; the only stand-alone LayerNorm is the first layer's (sparse rows), once
        assert used.get('norm_dense_fwdlap', 0) == 3 * 3 + 4, used
        assert used.get('layernorm_fwdlap', 0) == 1, used
    else:
        # one-electron layers 2-4 read their concatenated input in parts, activation in the epilogue
        assert used.get('dense_act_fwdlap', 0) >= 3, used
    r64 = fn(ob, ob.init_state(x, dtype=np.float64))
    r32 = fn(ob, ob.init_state(x, dtype=np.float32))
    J = out.jacobian.dense_array.cpu().numpy().astype(np.float64)
    got = (out.x.cpu().numpy().astype(np.float64), J, out.laplacian.cpu().numpy().astype(np.float64))
    for g, a64, a32, nm in zip(got, (r64.x, r64.J, r64.lap), (r32.x, r32.J, r32.lap), ('x', 'jacobian', 'laplacian')):
        assert g.shape == a64.shape
        scale = np.abs(a64).max()
        floor = np.abs(a32.astype(np.float64) - a64).max()
        err = np.abs(g - a64).max()
        print(f'{name} {nm}: |hip - fp64| = {err / scale:.2e}, |numpy fp32 - fp64| = {floor / scale:.2e} (rel. to max)', flush=True)
        assert err <= max(2.0 * floor, 1e-5 * scale), (nm, err, floor)


PER_WALKER_C = {'x': 8.0, 'jacobian': 4.0, 'laplacian': 4.0}
PER_WALKER_SAMPLES = 4


def test_psiformer32_thirty_two_walkers_each_within_its_own_float32_floor():
    """The headline configuration at full width on the first 32 walkers of the benchmark batch, walker by walker.
    log|det| of a walker's random 16 x 16 orbital matrices amplifies float32 rounding by that walker's
    condition number, so each walker has its own floor: the distance of the numpy oracle run in float32 from
    the float64 result.  One float32 run is ONE draw of that walker's rounding error (the ratio of two such draws
    has a heavy tail), so the floor is the largest of PER_WALKER_SAMPLES = 4 float32 runs: the inputs as they
    are, and three with every coordinate moved by at most one float32 unit in the last place (a change no float32
    computation can tell from its own input rounding).  The HIP result of EVERY walker must be within c x that
    walker's floor, c = 4 for the Jacobian and the Laplacian (largest of 96 entries: concentrated) and c = 8 for the
    single value, or within the strict bars where the floor is below them -- so the worst-conditioned walkers of
    the batch are compared too, not only a well-conditioned pair."""
    forward, p, cfg, _, sigma, thr = wl.build('psiformer32')
    n = 32
    x = wl.sample_inputs('psiformer32', n, seed=2)   # the first walkers of the batch bench.py times
    fn = lambda xp, t: forward(p, t, xp)
    print('case psiformer32, 32 walkers, per-walker bar', flush=True)
    out = run(fn, x, thr)
    r64 = fn(ob, ob.init_state(x, dtype=np.float64))
    ref = (r64.x[None], r64.J, r64.lap[None])
    rng = np.random.default_rng(5)
    floors = [np.zeros(n) for _ in ref]
    for s_ in range(PER_WALKER_SAMPLES):
        xs = x if s_ == 0 else np.nextafter(x, np.where(rng.random(x.shape) < 0.5, -np.inf, np.inf).astype(np.float32))
        r32 = fn(ob, ob.init_state(xs.astype(np.float32), dtype=np.float32))
        for i, (a32, a64) in enumerate(zip((r32.x[None], r32.J, r32.lap[None]), ref)):
            floors[i] = np.maximum(floors[i], np.abs(np.asarray(a32, dtype=np.float64) - a64).max(axis=0) / np.abs(a64).max(axis=0))
    got = (out.x.cpu().numpy().astype(np.float64)[None], out.jacobian.dense_array.cpu().numpy().astype(np.float64),
           out.laplacian.cpu().numpy().astype(np.float64)[None])
    bad = []
    for g, a64, floor, nm, strict in zip(got, ref, floors, ('x', 'jacobian', 'laplacian'), (1e-5, 1e-5, 1e-4)):
        assert g.shape == a64.shape == (a64.shape[0], n)
        err = np.abs(g - a64).max(axis=0) / np.abs(a64).max(axis=0)   # per walker
        ratio = err / np.maximum(PER_WALKER_C[nm] * floor, strict)
        w = int(np.argmax(ratio))
        print(f'psiformer32 {nm}: worst walker {w}: |hip - fp64| = {err[w]:.2e}, its float32 floor {floor[w]:.2e} '
              f'({ratio[w]:.2f} x the bar); largest floor of the 32 walkers {floor.max():.2e}, median {np.median(floor):.2e}; '
              f'median |hip - fp64| / floor = {np.median(err / np.maximum(floor, 1e-12)):.2f}', flush=True)
        if not (ratio <= 1.0).all():
            bad.append((nm, w, float(err[w]), float(floor[w])))
    assert not bad, bad


def test_psiformer32_full_batch_properties():
    """At the full benchmark size (4096 walkers): walkers are independent, so any walker
    evaluated inside the big batch equals the same walker evaluated in a batch of 4; the
    chunked evaluation (batched_vmap) equals the unchunked one bit for bit."""
    cfg, B, sigma, thr = wl.CONFIGS['psiformer32']
    p = wl.to_device(wl.psiformer_params(cfg), torch.device('cuda'))
    x = wl.sample_electrons(B, cfg.n_elec, sigma, seed=2)
    fn = lambda t: wl.psiformer_forward(p, t)
    fl = folx_amd.forward_laplacian(fn, thr)
    print('case psiformer32 full batch', flush=True)
    full = folx_amd.batched_vmap(fl, 1024)(x)
    assert full.x.shape == (B,) and full.jacobian.dense_array.shape == (96, B)
    assert torch.isfinite(full.x).all() and torch.isfinite(full.laplacian).all()
    idx = [0, 1023, 1024, 4095]
    small = folx_amd.vmap(fl)(x[idx])
    assert_val(full.x[idx], small.x.cpu().numpy())
    assert_val(full.jacobian.dense_array[:, idx], small.jacobian.dense_array.cpu().numpy())
    assert_lap(full.laplacian[idx], small.laplacian.cpu().numpy())
    again = folx_amd.batched_vmap(fl, 1024)(x)
    assert torch.equal(again.x, full.x) and torch.equal(again.laplacian, full.laplacian)


FULL_WIDTH = ['ferminet16', 'psiformer32', 'psiformer64']


@pytest.mark.parametrize('name', FULL_WIDTH)
def test_full_width_every_rule_call_meets_the_strict_bars(name):
    """The benchmark architectures at their real widths, 2 walkers: every kernel call of the
    forward Laplacian is compared, on the float32 inputs the HIP path handed it, with the
    float64 oracle rule of that call at the strict bars (values / Jacobians rtol 1e-5,
    Laplacians rtol 1e-4 + atol 1e-5), widened only by the measured response of that rule to
    rounding noise in its inputs (tests/stagecheck.py; matters for the determinants)."""
    import dataclasses

    from stagecheck import StageCheck

    forward, p, cfg, _, sigma, thr = wl.build(name)
    x = wl.sample_electrons(2, cfg.n_elec, sigma, seed=2)
    print(f'case {name} stage by stage', flush=True)
    with StageCheck() as sc:
        run(lambda xp, t: forward(p, t, xp), x, thr)
    used = sc.summary()
    for kern, (calls, worst, amp) in sorted(used.items()):
        print(f'{name} {kern}: {calls} calls, worst error {worst:.2f} x bar, allowance {amp:.1f}', flush=True)
    fused = {'psiformer32': ('norm_dense', 'mhsa', 'mhsa_sparse', 'slogdet', 'dense'),
             'psiformer64': ('norm_dense', 'mhsa', 'mhsa_sparse', 'slogdet', 'dense'),
             'ferminet16': ('dense_act_parts', 'dense_act', 'slogdet', 'dense')}[name]
    assert set(fused) <= set(used), used
    assert len(sc.log) >= 40


WELL_CONDITIONED = {
    # name: diagonal shift of the orbital matrices (their entries are O(1))
    'ferminet16': 40.0, 'psiformer32': 60.0, 'psiformer64': 90.0,
}


@pytest.mark.parametrize('name', FULL_WIDTH)
def test_full_width_well_conditioned_end_to_end_strict(name):
    """The same architectures end to end at north-star tolerances (values / Jacobians rtol 1e-5,
    Laplacians rtol 1e-4 + atol 1e-5, test/laplacian_testcase.py:16-49), with every orbital
    matrix shifted by a multiple of the identity so that log|det| no longer amplifies float32
    rounding (condition numbers of a few units, asserted below)."""
    import dataclasses

    from stagecheck import StageCheck

    forward, p, cfg, _, sigma, thr = wl.build(name)
    p = dataclasses.replace(p, cfg=dataclasses.replace(cfg, orb_shift=WELL_CONDITIONED[name]))
    x = wl.sample_electrons(2, cfg.n_elec, sigma, seed=4)
    print(f'case {name} well conditioned end to end', flush=True)
    fn = lambda xp, t: forward(p, t, xp)
    with StageCheck(names=('slogdet',)) as sc:
        out = run(fn, x, thr)
    assert sc.log and all(amp < 1.5 for *_, amp in sc.log), sc.log  # the determinants do not amplify input rounding
    ref = fn(ob, ob.init_state(x, dtype=np.float64))
    r32 = fn(ob, ob.init_state(x, dtype=np.float32))
    J = out.jacobian.dense_array
    from tolerances import LAP_ATOL, LAP_ATOL_REL, LAP_RTOL, VAL_ATOL_REL, VAL_RTOL

    for got, want, w32, nm in ((out.x, ref.x, r32.x, 'x'), (J, ref.J, r32.J, 'jacobian'),
                               (out.laplacian, ref.lap, r32.lap, 'laplacian')):
        g = got.cpu().numpy().astype(np.float64)
        scale = np.abs(want).max()
        # what float32 arithmetic itself costs on this function: the numpy oracle run in float32
        floor = np.abs(w32.astype(np.float64) - want).max()
        print(f'{name} {nm}: max |hip - fp64| / max|fp64| = {np.abs(g - want).max() / scale:.2e}, '
              f'numpy float32 oracle: {floor / scale:.2e}', flush=True)
        rtol, atol = (LAP_RTOL, LAP_ATOL + LAP_ATOL_REL * scale) if nm == 'laplacian' else (VAL_RTOL, VAL_ATOL_REL * scale)
        # the north-star bars; where a chain of 24 float32 matrix products (each within the bars on its
        # own, see the stage-by-stage test) cannot meet them end to end, the absolute part grows to the
        # error of the float32 numpy oracle on the same function
        np.testing.assert_allclose(g, want, rtol=rtol, atol=max(atol, floor), err_msg=f'{name} {nm}')


def test_narrow_layers_every_rule_call_meets_the_strict_bars():
    """The node-wise MLP with its sparse Jacobian stage by stage: sums of triplets, scalings, and its layers as one launch."""
    from stagecheck import StageCheck

    forward, p, cfg, _, _, thr = wl.build('mlp_sparse')
    x = wl.sample_inputs('mlp_sparse', 2, seed=2)
    print('case mlp_sparse stage by stage', flush=True)
    with StageCheck() as sc:
        run(lambda xp, t: xp.multiply(forward(p, t, xp), 0.5), x, thr)
    used = sc.summary()
    print(used, flush=True)
    assert {'dense_chain', 'reduce_sum_arrays', 'affine'} <= set(used), used
    assert all(w <= 1.0 for _, w, _ in used.values())


@pytest.mark.parametrize('name,chunk', [('psiformer64', 256), ('ferminet16', 1024)])
def test_full_batch_properties(name, chunk):
    """psiformer64 at its 1024 walkers in chunks of 256 and ferminet16 at its 4096: finite
    results, walkers independent of the batch they are evaluated in, deterministic."""
    forward, p, cfg, B, sigma, thr = wl.build(name)
    p = wl.to_device(p, torch.device('cuda'))
    x = wl.sample_electrons(B, cfg.n_elec, sigma, seed=2)
    fl = folx_amd.forward_laplacian(lambda t: forward(p, t), thr)
    print(f'case {name} full batch {B} in chunks of {chunk}', flush=True)
    full = folx_amd.batched_vmap(fl, chunk)(x)
    P = 3 * cfg.n_elec
    assert full.x.shape == (B,) and full.jacobian.dense_array.shape == (P, B)
    assert torch.isfinite(full.x).all() and torch.isfinite(full.laplacian).all()
    assert torch.isfinite(full.jacobian.dense_array).all()
    idx = [0, chunk - 1, chunk, B - 1]
    small = folx_amd.vmap(fl)(x[idx])
    # single walkers inside the big batch = the same walkers in a batch of 4, up to the noise floor of
    # log|det| (different tile shapes change the summation order in front of an ill-conditioned determinant)
    r64 = forward(wl.build(name)[1], ob.init_state(x[idx], dtype=np.float64), ob)
    r32 = forward(wl.build(name)[1], ob.init_state(x[idx], dtype=np.float32), ob)
    for a, b, a64, a32, nm in ((full.x[idx], small.x, r64.x, r32.x, 'x'),
                               (full.jacobian.dense_array[:, idx], small.jacobian.dense_array, r64.J, r32.J, 'jacobian'),
                               (full.laplacian[idx], small.laplacian, r64.lap, r32.lap, 'laplacian')):
        floor = np.abs(a32.astype(np.float64) - a64).max()
        scale = np.abs(a64).max()
        d = (a.double() - b.double()).abs().max().item()
        e = np.abs(a.double().cpu().numpy() - a64).max()
        print(f'{name} {nm}: |big - small| = {d / scale:.2e}, |big - fp64| = {e / scale:.2e}, fp32 floor {floor / scale:.2e}', flush=True)
        # both errors are samples of float32 rounding amplified by the determinants of four walkers:
        # a factor of 4 between two such samples is within their scatter
        assert d <= max(4.0 * floor, 1e-5 * scale), (nm, d, floor)
        assert e <= max(4.0 * floor, 1e-5 * scale), (nm, e, floor)
    again = folx_amd.batched_vmap(fl, chunk)(x)
    assert torch.equal(again.x, full.x) and torch.equal(again.laplacian, full.laplacian)
