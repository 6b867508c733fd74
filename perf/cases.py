"""The cases this framework's speed is measured on: forward Laplacians of the model families that the repository
carries (``folx_amd.workloads``, ``README.md``, ``bench.py``) and of a plain torch module, through the public entry
points, from a handful of walkers to the benchmark's batch.

A case is one call of a program that keeps its model, its weights on the device and, where it uses them, its captured
graph or its traced function, and hands over walkers: ``forward_laplacian`` under ``vmap`` / ``batched_vmap`` (with or
without ``jit``), ``ForwardLaplacianOperator``, or ``forward_laplacian_torch``.  The result is the whole triplet (value,
dense Jacobian, Laplacian) of every walker, or the operator's (Laplacian, Jacobian).

Walkers of wavefunctions are the best of sixteen Gaussian proposals by |psi| (evaluated in float64 with plain torch): a
Monte Carlo program samples |psi|^2 and so keeps away from the nodes, where log|psi| has no bounded derivatives.
"""

import math

import torch

import folx_amd
from folx_amd import kernels
from folx_amd import torch_namespace
from folx_amd import workloads

DEVICE = 'cuda'
CHUNK = 1024  # walkers of one batched_vmap chunk, as in the benchmark


def _mlp(name, walkers, threshold, mode, nodes=100, in_dim=4, width=100, hidden=10):
    return dict(name=name, kind='mlp', walkers=walkers, threshold=threshold, mode=mode, nodes=nodes, in_dim=in_dim,
                width=width, hidden=hidden)


def _ferminet(name, walkers, mode, elec=16, nuc=4, layers=4, w1=256, w2=32, det=16):
    return dict(name=name, kind='ferminet', walkers=walkers, mode=mode, elec=elec, nuc=nuc, layers=layers, w1=w1, w2=w2,
                det=det, gemm='f32')


def _psiformer(name, walkers, mode, elec=32, nuc=4, layers=4, heads=4, head_dim=64, det=16, gemm='f32'):
    return dict(name=name, kind='psiformer', walkers=walkers, mode=mode, elec=elec, nuc=nuc, layers=layers, heads=heads,
                head_dim=head_dim, det=det, gemm=gemm)


def _transformer(name, walkers, mode, elec=16, layers=2, heads=4, width=64):
    return dict(name=name, kind='transformer', walkers=walkers, mode=mode, elec=elec, layers=layers, heads=heads,
                width=width)


def listed():
    return [
        # The README's node-wise MLP: its own batch of 20 under jit (sparse Jacobian) and eagerly (dense Jacobian), the
        # benchmark's batch of 256, and a smaller odd-sized network as a descriptor of atoms in a molecule.
        _mlp('mlp_sparse_jit', 20, 4, 'jit'),
        _mlp('mlp_dense', 20, 0, 'eager'),
        _mlp('mlp_sparse', 256, 4, 'eager'),
        _mlp('mlp_odd', 750, 3, 'eager', nodes=21, in_dim=3, width=50, hidden=4),
        # Wavefunctions in variational Monte Carlo.  FermiNet-style: the benchmark's 16 electrons at its full batch; a
        # nitrogen atom (7 electrons: unequal spins, 21 coordinates) whose step is captured, as for any small system.
        _ferminet('ferminet16', 4096, 'eager'),
        _ferminet('ferminet7_jit', 512, 'jit', elec=7, nuc=1),
        # PsiFormer-style: the benchmark's 32 electrons at its full batch, the same with the bf16x3 products, the large
        # configuration, water (10 electrons) as plain torch code in a small evaluation batch, and an odd atom count.
        _psiformer('psiformer32', 4096, 'eager'),
        _psiformer('psiformer32_bf16x3', 1024, 'eager', gemm='bf16x3'),
        _psiformer('psiformer64', 256, 'eager', elec=64, nuc=8, heads=8),
        _psiformer('psiformer10_torch', 64, 'torch', elec=10, nuc=3),
        _psiformer('psiformer13_jit', 300, 'jit', elec=13, nuc=2),
        # A model that exists as a torch module: pre-norm transformer over particles, attention written with matmul and
        # softmax, GELU feed-forward blocks, a sum over particles.
        _transformer('transformer_torch', 512, 'torch'),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


DRAWN_FLOPS = 2.5e12   # a drawn case stays well below the largest listed one
DRAWN_FLOATS = 1.0e9   # and its largest row stack below 4 GB


def draw(rng):
    while True:
        kind = rng.choice(['mlp', 'ferminet', 'psiformer', 'psiformer', 'transformer'])
        if kind == 'mlp':
            in_dim = rng.randint(2, 6)
            c = _mlp('', _log_int(rng, 8, 2048), rng.choice([0, in_dim]), rng.choice(['eager', 'jit']),
                     _log_int(rng, 5, 150), in_dim, _log_int(rng, 16, 256), rng.randint(2, 10))
        elif kind == 'ferminet':
            c = _ferminet('', _log_int(rng, 32, 4096), rng.choice(['eager', 'jit']), _log_int(rng, 4, 24),
                          rng.randint(1, 6), rng.randint(2, 4), rng.choice([64, 100, 128, 256]), rng.choice([16, 30, 32]),
                          rng.choice([1, 4, 16]))
        elif kind == 'psiformer':
            c = _psiformer('', _log_int(rng, 16, 2048), rng.choice(['eager', 'jit', 'torch']), _log_int(rng, 4, 48),
                           rng.randint(1, 8), rng.randint(2, 4), rng.choice([2, 4, 8]), rng.choice([32, 64]),
                           rng.choice([1, 4, 16]), rng.choice(['f32', 'f32', 'bf16x3']))
        else:
            heads = rng.choice([1, 2, 4])
            c = _transformer('', _log_int(rng, 16, 2048), 'torch', _log_int(rng, 4, 32), rng.randint(1, 3), heads,
                             heads * rng.choice([8, 16, 24, 32]))
        del c['name']
        # a captured step is what small and medium batches use: large ones run in eager chunks
        if work(c)['flops'] > DRAWN_FLOPS or _largest_stack(c) > DRAWN_FLOATS or (c['mode'] == 'jit' and c['walkers'] > CHUNK):
            continue
        return c


# ---- models ---------------------------------------------------------------------------------


def _shifted(case):
    """Orbital matrices of 9 x 9 and larger get a diagonal part (the configurations' orb_shift): filled with random numbers
    alone they are close to singular in float32, which those of a converged wavefunction are not."""
    return case['elec'] > 16


def _wavefunction(case):
    """(forward(params, r, xp), numpy parameters, standard deviation of the electrons' proposals)."""
    shift = 3.0 if _shifted(case) else 0.0
    if case['kind'] == 'ferminet':
        cfg = workloads.FermiNetConfig(n_elec=case['elec'], n_nuc=case['nuc'], n_layers=case['layers'], w1=case['w1'],
                                       w2=case['w2'], n_det=case['det'], orb_shift=shift)
        return workloads.ferminet_forward, workloads.ferminet_params(cfg), 1.5
    width, large = case['heads'] * case['head_dim'], case['elec'] >= 40
    cfg = workloads.PsiFormerConfig(n_elec=case['elec'], n_nuc=case['nuc'], n_layers=case['layers'], n_heads=case['heads'],
                                    head_dim=case['head_dim'], width=width, mlp_width=width, n_det=case['det'],
                                    nuc_box=4.0 if large else 2.0, orb_shift=shift)
    return workloads.psiformer_forward, workloads.psiformer_params(cfg), 2.0 if large else 1.5


class Transformer(torch.nn.Module):
    """A function of particle positions (n, 3) as people write it in torch."""

    def __init__(self, layers, heads, width):
        super().__init__()
        Linear, Norm, List = torch.nn.Linear, torch.nn.LayerNorm, torch.nn.ModuleList
        self.heads = heads
        self.embed = Linear(3, width)
        self.norm1, self.norm2 = List([Norm(width) for _ in range(layers)]), List([Norm(width) for _ in range(layers)])
        self.q, self.k, self.v = (List([Linear(width, width, bias=False) for _ in range(layers)]) for _ in range(3))
        self.out = List([Linear(width, width) for _ in range(layers)])
        self.up, self.down = List([Linear(width, 2 * width) for _ in range(layers)]), List([Linear(2 * width, width) for _ in range(layers)])
        self.readout = Linear(width, 1)

    def forward(self, x):
        h = torch.tanh(self.embed(x))
        n, width = h.shape
        d = width // self.heads
        for norm1, q, k, v, out, norm2, up, down in zip(self.norm1, self.q, self.k, self.v, self.out, self.norm2, self.up, self.down):
            y = norm1(h)
            qh, kh, vh = (t(y).view(n, self.heads, d).permute(1, 0, 2) for t in (q, k, v))
            p = torch.softmax(qh @ kh.transpose(-1, -2) / d ** 0.5, dim=-1)
            h = h + out((p @ vh).permute(1, 0, 2).reshape(n, width))
            h = h + down(torch.nn.functional.gelu(up(norm2(h))))
        return self.readout(h).sum()


def _walkers(forward, params, elec, sigma, n, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    r = sigma * torch.randn(16, n, elec, 3, device=DEVICE, generator=g)
    psi = torch.func.vmap(lambda e: forward(params, e, xp=torch_namespace))
    score = torch.stack([torch.cat([psi(c.double()) for c in part.split(512)]) for part in r])
    return r[score.argmax(dim=0), torch.arange(n, device=DEVICE)].contiguous()


# ---- one case -------------------------------------------------------------------------------


def prepare(case, seed):
    kind, mode, n = case['kind'], case['mode'], case['walkers']
    with torch.no_grad():
        if kind == 'mlp':
            params = workloads.to_device(workloads.mlp_params(0, case['in_dim'], case['width'], case['hidden']), DEVICE)
            g = torch.Generator(device=DEVICE).manual_seed(seed)
            x = torch.randn(n, case['nodes'], case['in_dim'], device=DEVICE, generator=g)
            op = folx_amd.ForwardLaplacianOperator(case['threshold'])(lambda r: workloads.mlp_forward(params, r))
            step = folx_amd.vmap(op)
        elif kind == 'transformer':
            torch.manual_seed(0)
            model = Transformer(case['layers'], case['heads'], case['width']).requires_grad_(False).eval()
            g = torch.Generator(device=DEVICE).manual_seed(seed)
            x = 1.5 * torch.randn(n, case['elec'], 3, device=DEVICE, generator=g)
            step = folx_amd.batched_vmap(folx_amd.forward_laplacian_torch(model, 6), CHUNK)
        else:
            forward, params, sigma = _wavefunction(case)
            x = _walkers(forward, params, case['elec'], sigma, n, seed)
            if mode == 'torch':
                fl = folx_amd.forward_laplacian_torch(lambda r: forward(params, r, xp=torch_namespace), 6)
            else:
                on_device = workloads.to_device(params, DEVICE)
                fl = folx_amd.forward_laplacian(lambda r: forward(on_device, r), 6)
            step = folx_amd.vmap(fl) if n <= CHUNK else folx_amd.batched_vmap(fl, CHUNK)
    if mode == 'jit':
        step = folx_amd.jit(step)
    state = dict(step=step, x=x, gemm=case.get('gemm', 'f32'))
    for _ in range({'eager': 0, 'torch': 1, 'jit': 2}[mode]):  # the trace, or the capture, that the program keeps
        run(state)
    return state


def run(state):
    if state['gemm'] != 'f32':
        kernels.set_gemm_mode(state['gemm'])
    try:
        out = state['step'](state['x'])
    finally:
        if state['gemm'] != 'f32':
            kernels.set_gemm_mode('f32')
    if isinstance(out, tuple):
        return out
    return out.x, out.jacobian.dense_array, out.laplacian


# ---- what a pass cannot do without ------------------------------------------------------------


def _counts(case):
    """(multiply-adds of one walker's value, input coordinates, weights): the triplet multiplies each product of the value
    by its Jacobian rows + 2, dense unless the network keeps them sparse."""
    if case['kind'] == 'mlp':
        dims = [case['in_dim']] + [case['width']] * case['hidden'] + [1]
        w = sum(a * b for a, b in zip(dims[:-1], dims[1:]))
        coords = case['nodes'] * case['in_dim']
        rows = (case['in_dim'] if case['threshold'] else coords) + 2
        return rows * case['nodes'] * w, coords, w
    n = case['elec']
    P = 3 * n
    if case['kind'] == 'transformer':
        d, L = case['width'], case['layers']
        w = 3 * d + L * 8 * d * d + d
        macs = 5 * n * 3 * d + (P + 2) * n * (L * 8 * d * d + d) - (P - 3) * n * 3 * d * d  # embedding, first q, k, v: 3 rows
        return macs + L * 3 * (P + 2) * 2 * n * n * d, P, w
    nu, nd, orb = n // 2, n - n // 2, case['det'] * case.get('w1', case.get('heads', 0) * case.get('head_dim', 0))
    macs = (P + 2) * orb * (nu * nu + nd * nd)
    w = orb * n
    macs += (P + 2) * case['det'] * (nu ** 3 + nd ** 3) * 2
    if case['kind'] == 'psiformer':
        d, L = case['heads'] * case['head_dim'], case['layers']
        f = 4 * case['nuc'] + 1
        w += f * d + L * 6 * d * d
        macs += 5 * n * f * d + (P + 2) * n * (L * 6 * d * d) - (P - 3) * n * 3 * d * d  # features, first q, k, v: 3 rows
        macs += (7 * P + 6) * n * n * d * (L - 1) + (P + 30) * n * n * d
        return macs, P, w
    d1, d2 = 4 * case['nuc'], 4
    for layer in range(case['layers']):
        # own features and the two pair means per electron, the two one-electron means once per walker
        macs += (P + 2) * (n * (d1 + 2 * d2) + 2 * d1) * case['w1']
        w += (3 * d1 + 2 * d2) * case['w1']
        if layer < case['layers'] - 1:
            macs += 8 * n * n * d2 * case['w2']  # pairs: six rows
            w += d2 * case['w2']
        d1, d2 = case['w1'], case['w2']
    return macs, P, w


def work(case):
    macs, coords, weights = _counts(case)
    B = case['walkers']
    return {'bytes': 4.0 * (B * (2 * coords + 2) + weights), 'flops': 2.0 * macs * B}


def _largest_stack(case):
    """Floats of the largest array of a pass (one chunk's Jacobian rows of a layer)."""
    B = min(case['walkers'], CHUNK)
    if case['kind'] == 'mlp':
        rows = case['in_dim'] if case['threshold'] else case['nodes'] * case['in_dim']
        return case['walkers'] * case['nodes'] * case['width'] * rows
    n = case['elec']
    if case['kind'] == 'transformer':
        return 3 * n * B * n * max(2 * case['width'], case['heads'] * n)
    if case['kind'] == 'ferminet':
        return max(3 * n * B * n * max(case['w1'], case['det'] * n), 8 * B * n * n * case['w2'])
    return 3 * n * B * n * case['heads'] * case['head_dim']


def tolerance(case):
    """About four times the largest distances seen between this path and float64 derivatives of the same function (48
    walkers), and between it and the same path with its products summed in another order and form (whole batches).  A
    log-determinant amplifies float32 rounding by the condition of its matrices and the inverse distance to a node, so a few
    walkers carry most of the difference there."""
    if case['kind'] in ('mlp', 'transformer'):
        return {'rel': 3e-6, 'max': 2e-5}
    if _shifted(case):
        return {'rel': 4e-4, 'max': 2e-2}
    return {'rel': 4e-3, 'max': 6e-2}
