"""Batched universes (one fused launch for all universes and steps) against the FP64 oracle
per universe, against the plain per-universe loop, across every launch shape, under hipGraph
replay, and with the trajectory record."""

import numpy as np
import pytest
import torch

from gravitation_amd import _native, batched, tune
from gravitation_amd.lib import scenarios as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 5, 63, 64, 65, 127, 128, 129, 300, 511, 1000, 2048]


def _batch_inputs(sizes, seed=0, sigma=0.1):
    rng = np.random.default_rng(seed)
    rs, vs, ms = [], [], []
    for n in sizes:
        r, v, m = S.random_universe(int(n), rng, sigma)
        rs.append(r)
        vs.append(v)
        ms.append(m)
    off = np.zeros(len(sizes) + 1, dtype=np.int64)
    off[1:] = np.cumsum(sizes)
    return np.concatenate(rs), np.concatenate(vs), np.concatenate(ms), off


def _oracle(r, v, m, off, G, eps, dt, steps):
    rr, vv = np.empty_like(r), np.empty_like(v)
    for u in range(off.shape[0] - 1):
        a, b = off[u], off[u + 1]
        ru, vu, _ = O.simulate(r[a:b], v[a:b], m[a:b], G, eps, dt, steps, dtype=np.float32)
        rr[a:b], vv[a:b] = ru, vu
    return rr, vv


def _check_vs_oracle(batch, r0, v0, m, off, steps, tol=2e-5):
    r, v = batch.state()
    rr, vv = _oracle(r0, v0, m, off, batch.G, batch.eps, batch.dt, steps)
    # the change over the run carries the physics; compare it normwise
    assert O.rel_err(v - v0, vv - v0) < tol
    assert O.rel_err(r - r0, rr - r0) < tol


@pytest.mark.parametrize('eps', [1e-3, 0.0])
def test_batched_vs_oracle(cuda, eps):
    r, v, m, off = _batch_inputs(SIZES, seed=1)
    b = batched.Batch(r, v, m, off, G=1.0, eps=eps, dt=1e-3, device=cuda)
    b.step(5)
    _check_vs_oracle(b, r, v, m, off, 5)


def test_batched_every_launch_shape(cuda):
    r, v, m, off = _batch_inputs(SIZES, seed=2)
    rr, vv = _oracle(r, v, m, off, 1.0, 1e-3, 1e-3, 3)
    shapes = [(w, kt, sm, g) for w in (1, 4, 8)
              for kt, sm in ((1, 1), (1, 2), (1, 4), (1, 8), (2, 1), (2, 2), (2, 4), (4, 1),
                             (4, 2))
              for g in (0, 3)]
    ran = 0
    for cfg in shapes:
        print('batched shape', cfg, flush=True)
        b = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda, config=cfg)
        if not b.plan.info()['fused_ok']:
            continue  # this shape cannot hold the 2048-body universe in one workgroup
        b.step(3)
        rg, vg = b.state()
        assert O.rel_err(vg - v, vv - v) < 2e-5, cfg
        assert O.rel_err(rg - r, rr - r) < 2e-5, cfg
        ran += 1
    assert ran >= 12


def test_batched_matches_plain_loop(cuda):
    r, v, m, off = _batch_inputs([40, 700, 64, 1500, 9, 256], seed=3)
    b = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda)
    p = b.plain()
    b.step(10)
    p.step(10)
    rb, vb = b.state()
    rp, vp = p.state()
    assert O.rel_err(vb - v, vp - v) < 1e-5
    assert O.rel_err(rb - r, rp - r) < 1e-5


def test_graph_replay_equals_eager(cuda):
    r, v, m, off = _batch_inputs(SIZES, seed=4)
    b1 = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda)
    b2 = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda)
    g = b2.capture(4)
    for rep in range(3):
        b1.step(4)
        g.replay()
        torch.cuda.synchronize()
        r1, v1 = b1.state()
        r2, v2 = b2.state()
        assert np.array_equal(r1, r2) and np.array_equal(v1, v2), rep


def test_trajectory_record(cuda):
    r, v, m, off = _batch_inputs([10, 100, 65], seed=5)
    b = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda)
    c = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda)
    traj = torch.zeros((4, b.n, 4), dtype=torch.float32, device=cuda)
    b.step(4, traj=traj)
    for s in range(4):
        assert torch.equal(traj[s], c.posm), s
        c.step(1)
    assert torch.equal(b.posm, c.posm)


def test_single_body_universes_move_straight(cuda):
    r, v, m, off = _batch_inputs([1] * 17, seed=6)
    b = batched.Batch(r, v, m, off, G=1.0, eps=0.0, dt=0.25, device=cuda)
    b.step(4)
    rg, vg = b.state()
    assert np.array_equal(vg, v)
    rr = r.copy()
    for _ in range(4):
        rr = v * 0.25 + rr
    assert np.array_equal(rg, rr)


def test_plan_errors(cuda):
    # a universe too large for one workgroup: no fused schedule, the per-step one works
    p = batched.BatchedPlan(np.array([0, 6000]), 8, 1, 8, 0)
    assert p.info()['fused_ok'] == 0 and p.info()['n_items'] == (6000 + 63) // 64
    e = batched.Engine.wrap(p, 'fused')
    z = torch.zeros((6000, 4), dtype=torch.float32, device=cuda)
    r = torch.zeros((3, 6000), dtype=torch.float64, device=cuda)
    with pytest.raises(_native.GravError, match='does not fit'):
        e.forward(z, r, r.clone(), 1.0, 1e-3, 1e-3, 1)
    with pytest.raises(_native.GravInvalidArgument, match='unsupported'):
        batched.BatchedPlan(np.array([0, 10]), 8, 4, 4, 0)
    with pytest.raises(_native.GravInvalidArgument, match='empty'):
        batched.BatchedPlan(np.array([0, 10, 10]), 8, 1, 8, 0)
    p = batched.BatchedPlan(np.array([0, 10, 300, 301]), 4, 1, 2, 2)
    info = p.info()
    assert info['n_bodies'] == 301 and info['n_universes'] == 3 and info['groups'] == 2
    assert info['total_cost'] == 10 * 10 + 290 * 290 + 1
    assert info['fused_ok'] == 1 and info['n_items'] == 1 + 5 + 1
    p.close()


@pytest.mark.parametrize('eps', [1e-3, 0.0])
def test_perstep_vs_oracle_and_fused(cuda, eps):
    r, v, m, off = _batch_inputs(SIZES, seed=11)
    for kt, jw in ((1, 1), (2, 4), (4, 8), (1, 8)):
        print('perstep kt=%d jw=%d' % (kt, jw), flush=True)
        b = batched.Batch(r, v, m, off, G=1.0, eps=eps, dt=1e-3, device=cuda,
                          config=('perstep', 8, kt, 8 // kt, 0, jw))
        b.step(5)
        _check_vs_oracle(b, r, v, m, off, 5)
    f = batched.Batch(r, v, m, off, G=1.0, eps=eps, dt=1e-3, device=cuda)
    f.step(5)
    rb, vb = b.state()
    rf, vf = f.state()
    assert O.rel_err(vb - v, vf - v) < 1e-5


def test_perstep_large_universe_and_graph(cuda):
    r, v, m, off = _batch_inputs([7000, 3, 100, 2049], seed=12)
    b = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda,
                      config=('perstep', 8, 2, 4, 0, 4))
    assert b.plan.info()['fused_ok'] == 0
    b.step(2)
    _check_vs_oracle(b, r, v, m, off, 2)
    c = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda,
                      config=('perstep', 8, 2, 4, 0, 4))
    g = c.capture(2)
    g.replay()
    torch.cuda.synchronize()
    rb, vb = b.state()
    rc, vc = c.state()
    assert np.array_equal(rb, rc) and np.array_equal(vb, vc)


def test_autotuner_picks_a_valid_shape(cuda):
    r, v, m, off = _batch_inputs([100, 2000, 30, 500] * 8, seed=7)
    b = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda)
    r0, v0 = b.state()
    cands = [('fused', 8, 1, 8, 16, 4), ('fused', 4, 2, 4, 32, 4), ('perstep', 8, 2, 4, 0, 4),
             ('perstep', 8, 1, 8, 0, 8)]
    best, table = tune.tune_batched(b, steps=2, candidates=cands)
    assert best in [c for c, _ in table] and len(table) >= 2
    r1, v1 = b.state()
    assert np.array_equal(r0, r1) and np.array_equal(v0, v1)   # state restored
    best1, table1 = tune.tune_stage1(b.posm, candidates=[(1, 8, 256), (4, 4, 256)])
    assert best1 in [(1, 8, 256), (4, 4, 256)]


def test_engine_rejects_tensors_off_its_device(cuda):
    off = np.array([0, 10, 30], dtype=np.int64)
    eng = batched.Engine(off, ('perstep', 4, 1, 4, 0, 2))
    assert eng.plan.device == torch.device('cuda', torch.cuda.current_device())
    posm = torch.zeros((30, 4), dtype=torch.float32)
    r64 = torch.zeros((3, 30), dtype=torch.float64)
    with pytest.raises(ValueError):
        eng.forward(posm, r64, r64.clone(), 1.0, 1e-3, 1e-3, 1)


# sizes below, at and across the symmetric blocks of 256 (4, 1) ... 2048 (8, 4) bodies
SYM_SIZES = [1, 2, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 3000, 70]


def _sym_acc(eng, posm, G, eps):
    acc = torch.full((3, eng.n), float('nan'), dtype=torch.float32, device=posm.device)
    _native.call('grav_batched_stage1_sym_f32', eng.plan.handle, posm.data_ptr(),
                 acc.data_ptr(), G, eps, eng._ws.data_ptr(), eng._ws.numel(),
                 torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return acc


@pytest.mark.parametrize('eps', [1e-3, 0.0])
def test_sym_stage1_vs_oracle_and_owner(cuda, eps):
    r, v, m, off = _batch_inputs(SYM_SIZES, seed=21)
    n = int(off[-1])
    posm = torch.tensor(np.concatenate([r, m[:, None]], axis=1), dtype=torch.float32,
                        device=cuda)
    pn = posm.cpu().numpy().astype(np.float64)
    ref = np.concatenate([O.accel_f64(pn[a:b, :3], pn[a:b, 3], 0.9, eps)
                          for a, b in zip(off[:-1], off[1:])])
    own = torch.empty((3, n), dtype=torch.float32, device=cuda)
    peng = batched.Engine(off, ('perstep', 8, 1, 8, 0, 4))
    _native.call('grav_batched_stage1_f32', peng.plan.handle, posm.data_ptr(), own.data_ptr(),
                 0.9, eps, 4, torch.cuda.current_stream().cuda_stream)
    own = own.cpu().numpy().T.astype(np.float64)
    for sym in batched.SYM_SHAPES:
        print('batched sym', sym, 'eps', eps, flush=True)
        eng = batched.Engine(off, ('perstep-sym', 8, 1, 8, 0, 4, sym))
        a = _sym_acc(eng, posm, 0.9, eps).cpu().numpy().T.astype(np.float64)
        assert np.all(np.isfinite(a)), sym
        for u, (lo, hi) in enumerate(zip(off[:-1], off[1:])):
            if hi - lo == 1:
                assert np.all(a[lo:hi] == 0.0), (sym, u)
                continue
            assert O.rel_err(a[lo:hi], ref[lo:hi]) < 1e-5, (sym, u, hi - lo)
            assert O.rel_err(a[lo:hi], own[lo:hi]) < 1e-5, (sym, u, hi - lo)
        # fixed reduction order: a second call is bitwise the same
        b = _sym_acc(eng, posm, 0.9, eps).cpu().numpy().T.astype(np.float64)
        assert np.array_equal(a, b), sym


def test_sym_perstep_vs_oracle_and_graph(cuda):
    r, v, m, off = _batch_inputs([3000, 5, 700, 1300, 64, 2049], seed=22)
    cfg = ('perstep-sym', 8, 2, 4, 0, 4, (4, 1))
    b = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda, config=cfg)
    assert b.config == cfg
    b.step(4)
    _check_vs_oracle(b, r, v, m, off, 4)
    c = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda, config=cfg)
    g = c.capture(2)
    for k in range(2):
        g.replay()
        torch.cuda.synchronize()
        print('graph replay %d' % k, flush=True)
    rb, vb = b.state()
    rc, vc = c.state()
    assert np.array_equal(rb, rc) and np.array_equal(vb, vc)


def test_sym_perstep_adjoint_equals_perstep(cuda):
    # same VJP launches as 'perstep': gradients over the same stored trajectory are equal
    r, v, m, off = _batch_inputs([900, 40, 1600], seed=23)
    steps = 3
    out = {}
    for cfg in (('perstep', 8, 1, 8, 0, 4), ('perstep-sym', 8, 1, 8, 0, 4, (8, 1))):
        b = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda, config=cfg)
        traj = torch.empty((steps, b.n, 4), dtype=torch.float32, device=cuda)
        b.step(steps, traj=traj)
        rho = torch.ones((3, b.n), dtype=torch.float64, device=cuda)
        nu = torch.zeros_like(rho)
        gam = torch.zeros((b.n,), dtype=torch.float64, device=cuda)
        b.engine.adjoint(traj, rho, nu, gam, b.G, b.eps, b.dt, steps)
        torch.cuda.synchronize()
        out[cfg[0]] = (traj.cpu().numpy(), rho.cpu().numpy(), gam.cpu().numpy())
    tp, rp, gp = out['perstep']
    ts, rs, gs = out['perstep-sym']
    assert np.array_equal(tp[0], ts[0])
    assert O.rel_err(ts.astype(np.float64), tp.astype(np.float64)) < 1e-6
    assert O.rel_err(rs, rp) < 1e-5 and O.rel_err(gs, gp) < 1e-5


@pytest.mark.parametrize('cfg', [batched.DEFAULT_CONFIG, ('perstep', 8, 2, 4, 0, 4),
                                 ('perstep-sym', 8, 1, 8, 0, 4, (4, 2))])
def test_shares_step_like_the_whole_batch(cuda, cfg):
    # a batch divided among GPUs by whole universes: each share, stepped alone with the same
    # schedule, gives its universes' state bit for bit as the whole batch does
    print('shares %s' % (cfg,), flush=True)
    sizes = SIZES + [int(x) for x in S.batch_sizes(40, 32, 1500, seed=21)]
    r, v, m, off = _batch_inputs(sizes, seed=22)
    whole = batched.Batch(r, v, m, off, G=1.0, eps=1e-3, dt=1e-3, device=cuda, config=cfg)
    whole.step(4)
    rw, vw = whole.state()
    for share in batched.shard_universes(off, 3):
        rs, vs, ms, os_ = batched.take_universes(r, v, m, off, share)
        b = batched.Batch(rs, vs, ms, os_, G=1.0, eps=1e-3, dt=1e-3, device=cuda, config=cfg)
        b.step(4)
        rb, vb = b.state()
        want_r, want_v, _, _ = batched.take_universes(rw, vw, m, off, share)
        assert np.array_equal(rb, want_r) and np.array_equal(vb, want_v), share


@pytest.mark.parametrize('sizes', [[1], [63, 64, 65, 1, 130], [256, 255, 700, 33],
                                   [70] * 260])
@pytest.mark.parametrize('kt, jw', [(1, 4), (1, 1), (2, 8), (4, 2)])
def test_perstep_fused_step_is_bitwise_its_two_stages(cuda, sizes, kt, jw):
    # grav_batched_step_items_f32 == grav_batched_stage1_f32 + grav_stage2_f64m bit for bit:
    # odd and even numbers of steps, with a record (one the steps run through, and one that
    # only takes copies) and without, few and many workgroups, eps = 0 and > 0
    from gravitation_amd import stages
    print('fused step', len(sizes), kt, jw, flush=True)
    rng = np.random.default_rng(len(sizes) + kt)
    off = np.concatenate([[0], np.cumsum(sizes)])
    n = int(off[-1])
    r, v = rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    m = rng.uniform(0.1, 1.0, n)
    config = ('perstep', 8, kt, 8 // kt, 0, jw)
    for eps in (0.0, 1e-2):
        for steps in (1, 2, 3):
            ref = batched.Batch(r, v, m, off, eps=eps, config=config)
            acc = torch.empty((3, n), dtype=torch.float32, device=cuda)
            seen = []
            for _ in range(steps):
                seen.append(ref.posm.clone())
                _native.call('grav_batched_stage1_f32', ref.plan.handle, ref.posm.data_ptr(),
                             acc.data_ptr(), ref.G, eps, jw,
                             torch.cuda.current_stream().cuda_stream)
                stages.stage2_f64m(ref.posm, ref.r64, ref.v64, acc, ref.dt)
            for dtype in (None, torch.float32, torch.float64):
                b = batched.Batch(r, v, m, off, eps=eps, config=config)
                traj = None if dtype is None else torch.zeros((steps, n, 4), dtype=dtype,
                                                              device=cuda)
                b.engine.forward(b.posm, b.r64, b.v64, b.G, eps, b.dt, steps, traj)
                for x, y in ((b.posm, ref.posm), (b.r64, ref.r64), (b.v64, ref.v64)):
                    assert torch.equal(x, y), (eps, steps, dtype)
                if traj is not None:
                    assert torch.equal(traj, torch.stack(seen).to(dtype)), (eps, steps, dtype)
    with pytest.raises(TypeError):
        b.engine.forward(b.posm, b.r64.float(), b.v64, 1.0, 0.0, 1e-3, 2)
    with pytest.raises(_native.GravError, match='overlap'):
        _native.call('grav_batched_step_items_f32', b.plan.handle, b.posm.data_ptr(),
                     b.posm.data_ptr(), b.r64.data_ptr(), b.v64.data_ptr(), 1.0, 0.0, 1e-3, jw,
                     torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize('jw, sizes', [(4, [1100, 2050, 65, 1, 4096, 1024]),
                                       (1, [300, 1024, 256, 513, 7]), (2, [600, 2048, 1000]),
                                       (8, [2100, 64, 8192])])
def test_perstep_in_halves_is_bitwise_a_large_launch(cuda, jw, sizes):
    # few universes, the longest j-ranges of more than one block of 256: steps and VJP with a
    # second set of wavefronts; beside 2100 universes of 3 bodies the launches are too large
    # for it.  The same bits, with eps = 0 and > 0.
    from gravitation_amd import adjoint
    print('halves', jw, sizes, flush=True)
    rng = np.random.default_rng(jw)
    n = sum(sizes)
    many = sizes + [3] * 2100
    off = np.concatenate([[0], np.cumsum(many)])
    r, v = rng.normal(size=(int(off[-1]), 3)), rng.normal(size=(int(off[-1]), 3))
    m, w = rng.uniform(0.1, 1.0, int(off[-1])), rng.normal(size=(int(off[-1]), 3))
    for eps in (0.0, 1e-2):
        out = []
        for k in (len(sizes), len(many)):
            a = int(off[k])
            eng = batched.Engine(off[:k + 1], ('perstep', 8, 1, 8, 0, jw), cuda)
            leaves = [torch.from_numpy(x[:a]).to(cuda).requires_grad_(True) for x in (r, v, m)]
            r1, v1 = adjoint.batched_trajectory(eng, *leaves, 2, G=1.0, eps=eps, dt=1e-3)
            ((r1 + v1) * torch.from_numpy(w[:a]).to(cuda)).sum().backward()
            out.append([x[:n].clone() for x in (r1.detach(), v1.detach(),
                                                *[y.grad for y in leaves])])
        for x, y in zip(*out):
            assert torch.equal(x, y), eps


@pytest.mark.parametrize('sym', [(4, 1), (8, 1), (4, 2), (8, 2), (4, 4)])
def test_sym_pairs_of_small_and_large_launches_are_bitwise_equal(cuda, sym):
    # the block pairs of one universe alone leave SIMDs with one wavefront, those of 300 copies
    # do not: the pair loops without and with the raised priority, the same sums
    print('sym launches', sym, flush=True)
    s = 1100
    rng = np.random.default_rng(7)
    one = np.concatenate([rng.normal(size=(s, 3)), rng.uniform(0.1, 1.0, (s, 1))], axis=1)
    got = []
    for copies in (1, 300):
        eng = batched.Engine(np.arange(copies + 1) * s, ('perstep-sym', 8, 1, 8, 0, 4, sym), cuda)
        posm = torch.from_numpy(np.tile(one, (copies, 1)).astype(np.float32)).to(cuda)
        got.append(_sym_acc(eng, posm, 0.7, 1e-2))
    few, many = got
    assert torch.isfinite(few).all()
    for k in (0, 150, 299):
        assert torch.equal(many[:, k * s:(k + 1) * s], few)


@pytest.mark.parametrize('sizes', [[1, 64, 1023, 1024, 1025], [4095, 4096, 4097, 2], [9000, 5, 3000]])
def test_batched_mu_is_exact_at_the_register_limit(cuda, sizes):
    # universes of up to 4096 bodies are held in registers between the two passes, larger ones
    # read again: mu = nu + h rho rounded twice, and its copy scaled by the exponent of the
    # universe's largest finite component, exactly
    print('mu', sizes, flush=True)
    rng = np.random.default_rng(sum(sizes))
    off = np.concatenate([[0], np.cumsum(sizes)])
    n, dt = int(off[-1]), 1e-3
    rho, nu = (rng.normal(size=(3, n)) * np.exp(rng.uniform(-20, 20, (3, n))) for _ in range(2))
    nu[1, 0], nu[2, n - 1] = np.inf, np.nan
    plan = batched.BatchedPlan(off)
    d_rho, d_nu = torch.from_numpy(rho).to(cuda), torch.from_numpy(nu).to(cuda)
    mu4 = torch.empty((n, 4), dtype=torch.float32, device=cuda)
    _native.call('grav_batched_adjoint_mu', plan.handle, d_rho.data_ptr(), d_nu.data_ptr(),
                 mu4.data_ptr(), dt, torch.cuda.current_stream().cuda_stream)
    got = mu4.cpu()
    want = nu + dt * rho
    assert np.array_equal(d_nu.cpu().numpy(), want, equal_nan=True)
    for u in range(len(sizes)):
        a, b = int(off[u]), int(off[u + 1])
        big = np.fmax.reduce(np.abs(want[:, a:b]), axis=0)   # a body with an infinity has no say
        big = big[np.isfinite(big) & (big > 0)]
        e = int(np.frexp(big.max())[1]) if big.size else 0
        assert torch.all(got[a:b, 3].contiguous().view(torch.int32) == e)
        with np.errstate(over='ignore', invalid='ignore'):
            w = np.ldexp(want[:, a:b], -e).astype(np.float32).T
        assert np.array_equal(got[a:b, :3].numpy(), w, equal_nan=True)


@pytest.mark.parametrize('mode', ['perstep', 'perstep-sym'])
@pytest.mark.parametrize('steps', [0, -1, -2, -3])
def test_no_steps_leave_the_state(cuda, mode, steps):
    print('no steps', mode, steps, flush=True)
    rng = np.random.default_rng(3)
    r, v, m = rng.normal(size=(300, 3)), rng.normal(size=(300, 3)), rng.uniform(0.1, 1.0, 300)
    b = batched.Batch(r, v, m, [0, 100, 300], config=(mode, 8, 1, 8, 0, 4))
    traj = torch.full((2, 300, 4), 7.0, device=cuda)
    before = [x.clone() for x in (b.posm, b.r64, b.v64, traj)]
    b.step(steps)
    b.engine.forward(b.posm, b.r64, b.v64, b.G, b.eps, b.dt, steps, traj)
    for x, y in zip((b.posm, b.r64, b.v64, traj), before):
        assert torch.equal(x, y)


@pytest.mark.parametrize('jw', [1, 2, 4])
@pytest.mark.parametrize('waves', [4096, 6144])
def test_perstep_at_the_limits_of_the_halves_is_bitwise_equal(cuda, jw, waves):
    # a second set of wavefronts up to a number of wavefronts of the launch, items times j_waves:
    # the same bits of a universe in launches of a few, of exactly that many and of one item more
    from gravitation_amd import adjoint
    print('halves limit', jw, waves, flush=True)
    sizes = [300 * jw, 1000 * jw]
    big = sum(-(-s // 64) for s in sizes)
    n = sum(sizes)
    out = []
    for extra in (0, waves // jw - big, waves // jw - big + 1):
        off = np.concatenate([[0], np.cumsum(sizes + [2] * extra)])
        total = int(off[-1])
        rng = np.random.default_rng(jw)
        one = [rng.normal(size=(n, 3)), rng.normal(size=(n, 3)), rng.uniform(0.1, 1.0, n) / n,
               rng.normal(size=(n, 3))]
        r, v, m, w = [np.concatenate([x, rng.normal(size=(total - n,) + x.shape[1:])])
                      for x in one]
        eng = batched.Engine(off, ('perstep', 8, 1, 8, 0, jw), cuda)
        leaves = [torch.from_numpy(x).to(cuda).requires_grad_(True) for x in (r, v, np.abs(m))]
        r1, v1 = adjoint.batched_trajectory(eng, *leaves, 2, G=1.0, eps=1e-2, dt=1e-3)
        ((r1 + v1) * torch.from_numpy(w).to(cuda)).sum().backward()
        out.append([x[:n].clone() for x in (r1.detach(), v1.detach(), *[y.grad for y in leaves])])
    for other in out[1:]:
        for x, y in zip(out[0], other):
            assert torch.equal(x, y)
