"""The workloads this framework is timed on, through its public entry points.

Five kinds of work, over the sizes users bring:

* ``step``: one ``step()`` of a ``hip1`` universe, the plugin contract of the reference.
  Sizes from a few hundred bodies (where launches and the host's wait count) to some ten
  thousand; FP32 as by default, FP32 pairs with FP64 masters, and FP64; the galaxy of the
  reference's benchmark (no softening, host views refreshed after every step) and softened
  Plummer spheres that stay on the device.
* ``tensors``: one step of a large universe held as tensors (``stages``), in the form that
  ``stages.auto_form`` names for its size.
* ``batch``: some steps of many independent universes of uneven size (``batched.Batch``).
* ``batch_grad``: a differentiable trajectory of such a batch, forward and backward.
* ``grad``: a differentiable trajectory of one universe, forward and backward, recorded or
  with checkpoints.

Initial conditions are physical: galaxies on circular orbits, Plummer spheres with the
velocity dispersion of their radius and a spread of masses, universes in a unit cube.
"""

import math

import numpy as np
import torch

from gravitation_amd import adjoint, batched, stages
from gravitation_amd.kernel import hip1


def listed():
    return [
        # a small galaxy stepped with host views: launches and the wait for the stream
        dict(name='step_galaxy_256', kind='step', scene='galaxy', n=256, mode='f32',
             sync_host=True),
        # the default galaxy of the reference's worker (2000 bodies)
        dict(name='step_galaxy_2000', kind='step', scene='galaxy', n=2000, mode='f32',
             sync_host=True),
        # the largest size of the reference's published benchmark log
        dict(name='step_galaxy_16384', kind='step', scene='galaxy', n=16384, mode='f32',
             sync_host=True),
        # a cluster run that keeps its state on the device, at a size of no special form
        dict(name='step_plummer_49999', kind='step', scene='plummer', n=49999, mode='f64m',
             sync_host=False),
        # the largest single universe of the framework's own benchmark
        dict(name='tensors_262144', kind='tensors', n=262144, mode='f64m'),
        # double precision, a small cluster and a large one
        dict(name='step_f64_3000', kind='step', scene='plummer', n=3000, mode='f64',
             sync_host=False),
        dict(name='step_f64_40000', kind='step', scene='plummer', n=40000, mode='f64',
             sync_host=False),
        # an ensemble of small universes, one launch for all steps of a call
        dict(name='batch_fused_512', kind='batch', universes=512, lo=32, hi=256, steps=20,
             schedule='fused'),
        # an ensemble of uneven universes, one launch per stage
        dict(name='batch_perstep_1024', kind='batch', universes=1024, lo=32, hi=2048, steps=10,
             schedule='perstep'),
        # fitting an ensemble: gradients of every universe's trajectory
        dict(name='batch_grad_128', kind='batch_grad', universes=128, lo=64, hi=2048, steps=12,
             schedule='perstep'),
        # fitting one cluster over checkpointed segments
        dict(name='grad_4096', kind='grad', n=4096, steps=60, interval=20),
        # a short trajectory of a larger cluster, its positions recorded
        dict(name='grad_20000', kind='grad', n=20000, steps=4, interval=0),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['step', 'step', 'step', 'step', 'tensors', 'batch', 'batch_grad', 'grad'])
    if kind == 'step':
        scene = rng.choice(['galaxy', 'plummer'])
        mode = rng.choice(['f32', 'f64']) if scene == 'galaxy' else rng.choice(
            ['f32', 'f64m', 'f64'])
        n = _log_uniform(rng, 200, 60000 if scene == 'plummer' else 20000)
        return dict(kind=kind, scene=scene, n=n, mode=mode, sync_host=rng.random() < 0.5)
    if kind == 'tensors':
        return dict(kind=kind, n=_log_uniform(rng, 20000, 260000), mode='f64m')
    if kind == 'batch':
        lo = rng.choice([32, 64, 100])
        schedule = rng.choice(['fused', 'perstep'])
        hi = _log_uniform(rng, 2 * lo, 1024 if schedule == 'fused' else 2048)
        return dict(kind=kind, universes=_log_uniform(rng, 100, 1000), lo=lo, hi=hi,
                    steps=rng.randint(5, 20), schedule=schedule)
    if kind == 'batch_grad':
        lo = rng.choice([32, 64, 100])
        return dict(kind=kind, universes=_log_uniform(rng, 30, 200), lo=lo,
                    hi=_log_uniform(rng, 2 * lo, 2048), steps=rng.randint(4, 12),
                    schedule=rng.choice(['fused', 'perstep']))
    n = _log_uniform(rng, 300, 20000)
    if n < 5000:
        return dict(kind='grad', n=n, steps=rng.randint(20, 60), interval=rng.choice([0, 10, 20]))
    return dict(kind='grad', n=n, steps=rng.randint(2, 6), interval=0)


# ---------------------------------------------------------------------------------------------
# initial conditions (float64 arrays of float32-representable values)

def _f32(*arrays):
    return [np.asarray(a, dtype=np.float32).astype(np.float64) for a in arrays]


def _directions(rng, n):
    u = rng.normal(size=(n, 3))
    return u / np.linalg.norm(u, axis=1, keepdims=True)


def _plummer(n, seed):
    """Plummer sphere (scale 1, total mass about 1, cut at radius 10) with the isotropic
    velocity dispersion of each radius, masses spread by a factor of about 3."""
    rng = np.random.default_rng(seed)
    cut = 10.0 ** 3 / (1.0 + 10.0 ** 2) ** 1.5
    frac = rng.uniform(1e-9, cut, n)
    rad = 1.0 / np.sqrt(frac ** (-2.0 / 3.0) - 1.0)
    r = rad[:, None] * _directions(rng, n)
    sigma = np.sqrt(1.0 / (6.0 * np.sqrt(1.0 + rad * rad)))
    v = sigma[:, None] * rng.normal(size=(n, 3))
    m = np.exp(rng.uniform(-0.5, 0.5, n)) / n
    return _f32(r, v, m)


GALAXY = dict(G=6.6743e-11, eps=0.0, dt=2.0e12)
PLUMMER = dict(G=1.0, eps=1e-3, dt=1e-4)
# softened over about the spacing of the bodies: trajectories that can be fitted
CUBE = dict(G=1.0, eps=2e-2, dt=1e-3)


def _galaxy(n, seed):
    """A heavy centre and n - 1 stars on circular orbits about it, 4/5 of them in a flat disk
    and 1/5 in a bulge, in the scaled units of the reference's default scenario."""
    rng = np.random.default_rng(seed)
    k = n - 1
    disk = np.arange(k) < (k * 4) // 5
    radius, hole = 1e10, 4e10
    rad = np.where(disk, rng.uniform(0.1, 4.6, k), rng.uniform(0.1, 0.85, k)) * radius
    alpha = rng.uniform(0.0, 2.0 * np.pi, k)
    beta = np.where(disk, 0.0, np.pi * (rng.uniform(0.0, 1.0, k) - 0.5))
    z = np.where(disk, rng.uniform(-0.25, 0.25, k) * (4.6 * radius - rad) / 4.6,
                 rad * np.sin(beta))
    r = np.stack([rad * np.cos(alpha) * np.cos(beta), rad * np.sin(alpha) * np.cos(beta), z], 1)
    speed = np.sqrt(GALAXY['G'] * hole / np.linalg.norm(r, axis=1))
    v = np.stack([-np.sin(alpha) * speed, np.cos(alpha) * speed, np.zeros(k)], 1)
    r = np.concatenate([np.zeros((1, 3)), r])
    v = np.concatenate([np.zeros((1, 3)), v])
    m = np.concatenate([[hole], np.full(k, 2.0)])
    return _f32(r, v, m)


def _sizes(case):
    return np.rint(np.exp(np.linspace(math.log(case['lo']), math.log(case['hi']),
                                      case['universes']))).astype(np.int64)


def _cubes(case, seed):
    """Universes of log-uniform size in a unit cube, masses over two decades."""
    rng = np.random.default_rng(seed)
    # the sizes are the case's, in another order for each seed
    sizes = rng.permutation(_sizes(case))
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    n = int(offsets[-1])
    r = rng.uniform(0.0, 1.0, (n, 3))
    v = rng.normal(0.0, 0.1, (n, 3))
    m = np.exp(rng.uniform(math.log(1e-4), math.log(1e-2), n))
    return _f32(r, v, m) + [offsets]


def _scene(case, seed):
    if case.get('scene') == 'galaxy':
        return _galaxy(case['n'], seed), GALAXY
    return _plummer(case['n'], seed), PLUMMER


def _weights(n, seed):
    """The loss of the ``grad`` kinds is a weighted sum of the final state: its gradient with
    respect to r_T and v_T."""
    rng = np.random.default_rng(seed + 7919)
    return rng.normal(size=(n, 3)), rng.normal(size=(n, 3))


def _schedule(case):
    return ('fused', 8, 1, 8, 0, 4) if case['schedule'] == 'fused' else (
        'perstep', 8, 1, 8, 0, 4)


# ---------------------------------------------------------------------------------------------

def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to('cuda')


def prepare(case, seed):
    kind = case['kind']
    if kind == 'step':
        (r, v, m), p = _scene(case, seed)
        opts = {'f32': dict(dtype='float32'),
                'f64m': dict(dtype='float32', stage2_dtype='float64'),
                'f64': dict(dtype='float64')}[case['mode']]
        u = hip1.universe(T=p['dt'], G=p['G'], eps=p['eps'], sync_host=case['sync_host'], **opts)
        u.add_objects(r, v, m)
        u.start()
        return dict(kind=kind, mode=case['mode'], u=u)
    if kind == 'tensors':
        r, v, m = _plummer(case['n'], seed)
        n = case['n']
        posm = torch.empty((n, 4), dtype=torch.float32, device='cuda')
        posm[:, :3] = _dev(r)
        posm[:, 3] = _dev(m)
        free, _ = torch.cuda.mem_get_info()
        return dict(kind=kind, posm=posm, r64=_dev(r.T), v64=_dev(v.T),
                    acc=torch.empty((3, n), dtype=torch.float32, device='cuda'),
                    form=stages.auto_form(n, free_bytes=free))
    if kind == 'batch':
        r, v, m, offsets = _cubes(case, seed)
        b = batched.Batch(r, v, m, offsets, config=_schedule(case), **CUBE)
        return dict(kind=kind, batch=b, steps=case['steps'])
    if kind == 'batch_grad':
        r, v, m, offsets = _cubes(case, seed)
        engine = batched.Engine(offsets, _schedule(case))
    else:
        r, v, m = _plummer(case['n'], seed)
        engine = None
    wr, wv = _weights(r.shape[0], seed)
    return dict(kind=kind, engine=engine, steps=case['steps'],
                interval=case.get('interval', 0) or None,
                leaves=[_dev(a).requires_grad_(True) for a in (r, v, m)],
                weights=[_dev(wr), _dev(wv)])


def run(state):
    kind = state['kind']
    if kind == 'step':
        u = state['u']
        u.step()
        if state['mode'] == 'f64m':
            return dict(a=u.acc, r=u.r64, v=u.vel, p=u.posm)
        return dict(a=u.acc, v=u.vel, p=u.posm)
    if kind == 'tensors':
        posm, acc = state['posm'], state['acc']
        G, eps = PLUMMER['G'], PLUMMER['eps']
        if state['form'] == 'symmetric':
            stages.stage1_sym_f32(posm, acc, G, eps)
        elif state['form'] == 'split':
            stages.stage1_split_f32(posm, acc, G, eps)
        else:
            stages.stage1_f32(posm, acc, G, eps)
        stages.stage2_f64m(posm, state['r64'], state['v64'], acc, PLUMMER['dt'])
        return dict(a=acc, r=state['r64'], v=state['v64'], p=posm)
    if kind == 'batch':
        b = state['batch']
        b.step(state['steps'])
        return dict(r=b.r64, v=b.v64, p=b.posm)
    r0, v0, m = state['leaves']
    if kind == 'batch_grad':
        r, v = adjoint.batched_trajectory(state['engine'], r0, v0, m, state['steps'], **CUBE)
    else:
        r, v = adjoint.trajectory(r0, v0, m, state['steps'], interval=state['interval'],
                                  **PLUMMER)
    gr, gv, gm = torch.autograd.grad([r, v], [r0, v0, m], state['weights'])
    return dict(r=r.detach(), v=v.detach(), gr=gr, gv=gv, gm=gm)


# Operations of one unordered pair: 3 differences, 3 fused multiply-adds for r^2, one inverse
# square root, its cube, the two weights and the 6 fused multiply-adds of both bodies; and of
# its adjoint, which both bodies share likewise.
PAIR_FLOPS = 26
PAIR_VJP_FLOPS = 60


def _pairs(case):
    if 'n' in case:
        return case['n'] * (case['n'] - 1) / 2, case['n']
    sizes = _sizes(case).astype(np.float64)
    return float((sizes * (sizes - 1) / 2).sum()), float(sizes.sum())


def work(case):
    pairs, n = _pairs(case)
    kind = case['kind']
    steps = case.get('steps', 1)
    if kind in ('step', 'tensors'):
        # r, v and m in, r, v and a out; the FP32 copy of the positions beside FP64 masters
        size = {'f32': 4 * (7 + 9), 'f64m': 16 * 2 + 8 * 12 + 12, 'f64': 8 * (7 + 9)}
        byts = size[case['mode']] * n
        if case.get('sync_host'):
            byts += (8 if case['mode'] != 'f32' else 4) * 6 * n
        return dict(bytes=byts, flops=PAIR_FLOPS * pairs)
    if kind == 'batch':
        return dict(bytes=n * (16 * 2 + 8 * 12), flops=PAIR_FLOPS * pairs * steps)
    # inputs, final state, its cotangents and the three gradients
    return dict(bytes=8 * n * (7 + 6 + 6 + 7),
                flops=(PAIR_FLOPS + PAIR_VJP_FLOPS) * pairs * steps)


# ---------------------------------------------------------------------------------------------
# the same in 64 bits

def _rows(n):
    return max(1, (1 << 26) // n)


def _accel(r, m, G, eps):
    """(n, 3) accelerations, a block of rows at a time."""
    n = r.shape[0]
    out = torch.empty_like(r)
    x, y, z = (r[:, c].contiguous() for c in range(3))
    step = _rows(n)
    for a in range(0, n, step):
        b = min(n, a + step)
        dx, dy, dz = (t[None, :] - t[a:b, None] for t in (x, y, z))
        q = dx * dx + dy * dy + dz * dz + eps * eps
        if eps == 0.0:
            k = torch.arange(a, b, device=r.device)
            q[k - a, k] = math.inf
        s = m[None, :] / (q * q.sqrt())
        for c, d in enumerate((dx, dy, dz)):
            out[a:b, c] = G * (s * d).sum(1)
    return out


def _accel_vjp(r, m, mu, G, eps):
    """mu^T da/dr (n, 3) and mu^T da/dm (n,) for softened accelerations."""
    n = r.shape[0]
    gr, gm = torch.empty_like(r), torch.empty_like(m)
    step = _rows(n)
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [r[None, :, c] - r[a:b, None, c] for c in range(3)]
        q = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + eps * eps
        s = 1.0 / (q * q.sqrt())
        w = [m[a:b, None] * mu[None, :, c] - m[None, :] * mu[a:b, None, c] for c in range(3)]
        dw = (d[0] * w[0] + d[1] * w[1] + d[2] * w[2]) * 3.0 / q
        for c in range(3):
            gr[a:b, c] = G * (s * (w[c] - d[c] * dw)).sum(1)
        gm[a:b] = -G * (s * (d[0] * mu[None, :, 0] + d[1] * mu[None, :, 1]
                             + d[2] * mu[None, :, 2])).sum(1)
    return gr, gm


def _advance(r, v, m, G, eps, dt, steps, seen=None):
    a = None
    for _ in range(steps):
        if seen is not None:
            seen.append(r)
        a = _accel(r, m, G, eps)
        v = v + a * dt
        r = r + v * dt
    return r, v, a


def _gradients(r, v, m, wr, wv, G, eps, dt, steps):
    seen = []
    r, v, _ = _advance(r, v, m, G, eps, dt, steps, seen)
    rho, nu, gam = wr.clone(), wv.clone(), torch.zeros_like(m)
    for q in reversed(seen):
        nu = nu + dt * rho
        gr, gm = _accel_vjp(q, m, nu, G, eps)
        rho, gam = rho + dt * gr, gam + dt * gm
    return r, v, rho, nu, gam


def exact(case, seed):
    kind = case['kind']
    if kind in ('step', 'tensors'):
        (r, v, m), p = _scene(case, seed)
        r, v, m = _dev(r), _dev(v), _dev(m)
        r1, v1, a = _advance(r, v, m, p['G'], p['eps'], p['dt'], 1)
        out = dict(a=a.t().contiguous(), v=v1.t().contiguous(),
                   p=torch.cat([r1, m[:, None]], 1))
        if case['mode'] == 'f64m':
            out['r'] = r1.t().contiguous()
        return out
    if kind == 'grad':
        r, v, m = map(_dev, _plummer(case['n'], seed))
        wr, wv = map(_dev, _weights(case['n'], seed))
        r, v, gr, gv, gm = _gradients(r, v, m, wr, wv, steps=case['steps'], **PLUMMER)
        return dict(r=r, v=v, gr=gr, gv=gv, gm=gm)
    r, v, m, offsets = _cubes(case, seed)
    r, v, m = _dev(r), _dev(v), _dev(m)
    parts = []
    if kind == 'batch_grad':
        wr, wv = map(_dev, _weights(int(offsets[-1]), seed))
    for a, b in zip(offsets[:-1], offsets[1:]):
        one = (r[a:b], v[a:b], m[a:b])
        if kind == 'batch':
            parts.append(_advance(*one, steps=case['steps'], **CUBE)[:2])
        else:
            parts.append(_gradients(*one, wr[a:b], wv[a:b], steps=case['steps'], **CUBE))
    whole = [torch.cat(x) for x in zip(*parts)]
    if kind == 'batch':
        return dict(r=whole[0].t().contiguous(), v=whole[1].t().contiguous(),
                    p=torch.cat([whole[0], m[:, None]], 1))
    return dict(zip(('r', 'v', 'gr', 'gv', 'gm'), whole))
