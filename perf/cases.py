"""Workloads of the framework, called through its public entry points, for
timing and for comparing results.

A case is a dict of plain values.  ``prepare`` makes what a program has in
hand before the call (records, steppers, captured graphs), ``run`` does one
pass, ``exact`` gives the same outputs from plain torch in 64 bits.

Kinds of pass:

* ``steps``       one episode of a Stepper or Ensemble: the agents set back
                  to their initial state, then ``steps`` fused steps, eager
                  or replayed from a HIP graph;
* ``tree``        ``steps`` updates of a drop-in LogicNode tree, node by node;
* ``rollout``     a differentiable rollout, forward and backward;
* ``field``       a navigation field from its rasterised target and obstacles;
* ``neighbours``  the nearest visible neighbours and the herding direction.
"""
import math
import types

import numpy as np
import torch

TWO_PI = 2.0 * math.pi


def _case(name, kind='steps', **kw):
    c = dict(kind=kind, model='circular', precision='f64', n=0, scenarios=1, density=1.0,
             cell=0.6, obstacles=0, nav=-1, steps=10, graph=True, lanes=0, order_every=0)
    c.update(kw)
    if name:
        c['name'] = name
    return c


def listed():
    return [
        # the reference's Hallway: 200 agents between walls at its default cell
        # size, stepped eagerly (launch latency is all there is)
        _case('hallway200', n=200, density=2.0, cell=3.6, steps=10, graph=False),
        # the same kind of tree run node by node (a custom tree), three-circle
        _case('tree2000', kind='tree', model='three_circle', n=2000, density=1.0, cell=3.6,
              obstacles=12, steps=4, graph=False),
        # the benchmark's room: 20k agents, four exits, bilinear navigation,
        # cells of 0.6 m, in both precisions
        _case('room20k_f64', n=20000, nav=1, steps=40),
        _case('room20k_f32', n=20000, nav=1, steps=20, precision='f32'),
        # a room at the reference's own cell size (sight + 2 radii), where every
        # pair in sight counts, with the reference's nearest-node navigation
        _case('room_wide_f64', n=20011, nav=0, cell=3.6, steps=10),
        # the largest single scenario
        _case('room200k_f64', n=200003, nav=1, steps=10),
        # the benchmark's corridor: 50k three-circle agents, 200 obstacles
        _case('corridor50k_f64', model='three_circle', n=50000, density=1.1, obstacles=200,
              steps=20, lanes=2),
        _case('corridor50k_f32', model='three_circle', n=50000, density=1.1, obstacles=200,
              steps=20, lanes=2, precision='f32'),
        # the benchmark's batched ensemble at its tuned setting: 256 rooms of
        # 500 to 8000 agents, 0.5 to 3 agents / m^2
        _case('ensemble256_f32', scenarios=256, n=8000, density=3.0, cell=3.56, steps=5,
              precision='f32', lanes=4, order_every=10),
        # the benchmark's differentiable rollout, forward and gradient
        _case('rollout4000', kind='rollout', n=4000, cell=3.6, steps=20, lanes=16),
        # the navigation field of a 200 x 100 m room at 0.2 m
        _case('field1001', kind='field', n=1001, obstacles=24),
        # herding neighbours: eight nearest in 3 m that no obstacle hides
        _case('neighbours20k', kind='neighbours', n=20000, density=1.0, obstacles=40),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(['room', 'room', 'wide', 'corridor', 'corridor', 'ensemble', 'ensemble',
                       'hallway', 'tree', 'rollout', 'field', 'neighbours'])
    prec = rng.choice(['f64', 'f32'])
    if kind == 'hallway':
        return _case(None, n=_log_int(rng, 60, 1000), density=rng.uniform(0.5, 2.5), cell=3.6,
                     steps=rng.randint(4, 12), graph=False, precision=prec,
                     model=rng.choice(['circular', 'three_circle']))
    if kind == 'tree':
        return _case(None, kind='tree', n=_log_int(rng, 200, 8000), density=rng.uniform(0.5, 2.0),
                     cell=rng.choice([0.6, 3.6]), obstacles=rng.randint(0, 40),
                     steps=rng.randint(2, 6), graph=False, precision=prec,
                     model=rng.choice(['circular', 'three_circle']))
    if kind == 'room':
        return _case(None, n=_log_int(rng, 2000, 150000), density=rng.uniform(0.5, 2.0), nav=1,
                     cell=rng.choice([0.6, 0.8, 1.2]), steps=rng.randint(5, 12), precision=prec,
                     obstacles=rng.choice([0, 0, 10, 60]), lanes=rng.choice([0, 4, 8]))
    if kind == 'wide':
        return _case(None, n=_log_int(rng, 2000, 30000), density=rng.uniform(0.3, 1.5), nav=0,
                     cell=rng.uniform(3.6, 5.0), steps=rng.randint(5, 10), precision=prec,
                     lanes=rng.choice([0, 4, 8]))
    if kind == 'corridor':
        return _case(None, model='three_circle', n=_log_int(rng, 2000, 50000),
                     density=rng.uniform(0.5, 1.5), obstacles=rng.randint(4, 200),
                     cell=rng.choice([0.6, 1.0]), steps=rng.randint(5, 12), precision=prec,
                     lanes=rng.choice([0, 2, 4]))
    if kind == 'ensemble':
        return _case(None, scenarios=_log_int(rng, 8, 200), n=rng.choice([1000, 3000, 8000]),
                     density=rng.uniform(1.0, 3.0), cell=rng.choice([3.56, 3.6, 4.094]),
                     steps=rng.randint(2, 5), precision=prec, lanes=rng.choice([0, 4, 8]),
                     order_every=rng.choice([0, 10]))
    if kind == 'rollout':
        return _case(None, kind='rollout', n=_log_int(rng, 300, 4000),
                     density=rng.uniform(0.5, 1.5), cell=rng.choice([1.2, 3.6]),
                     steps=rng.randint(5, 20), lanes=rng.choice([0, 16, 32]),
                     obstacles=rng.choice([0, 0, 8]))
    if kind == 'field':
        return _case(None, kind='field', n=_log_int(rng, 100, 1001), obstacles=rng.randint(4, 30))
    return _case(None, kind='neighbours', n=_log_int(rng, 500, 20000),
                 density=rng.uniform(0.3, 2.0), obstacles=rng.randint(0, 60))


# -- inputs ------------------------------------------------------------------

def _normal(rng, mean, sd, n):
    return mean + sd * np.clip(rng.standard_normal(n), -3.0, 3.0)


def _place(rng, n, w, h, segs, apart=0.565):
    """n positions in the box [0, w] x [0, h] (grown when it is too small): a
    random choice of jittered lattice sites at least `apart` m apart, 0.32 m
    clear of the box's walls and of the segments."""
    m = 0.32
    while True:
        s = max(apart + 0.005, math.sqrt(0.6 * (w - 2 * m) * (h - 2 * m) / max(n, 1)))
        j = (s - apart) / 2.0
        x = np.arange(m + j, w - m - j + 1e-9, s)
        y = np.arange(m + j, h - m - j + 1e-9, s)
        sites = np.stack([np.repeat(x, len(y)), np.tile(y, len(x))], 1)
        clear = np.ones(len(sites), dtype=bool)
        for seg in segs:
            lo = np.minimum(seg[:2], seg[2:]) - 1.0
            hi = np.maximum(seg[:2], seg[2:]) + 1.0
            k = np.nonzero(((sites > lo) & (sites < hi)).all(1))[0]
            clear[k[_point_segment(sites[k, 0], sites[k, 1], seg)[0] < m + 1.5 * j]] = False
        sites = sites[clear]
        if len(sites) >= n:
            break
        w, h = 1.02 * w, 1.02 * h
    p = sites[rng.permutation(len(sites))[:n]]
    return p + rng.uniform(-j, j, (n, 2)), w, h


def _segments(rng, count, w, h):
    """Random interior obstacles, 1 to 5 m long (half of that in small rooms)."""
    c = rng.uniform((0.05 * w, 0.05 * h), (0.95 * w, 0.95 * h), (count, 2))
    half = 0.5 * rng.uniform(1.0, 5.0, count) * min(1.0, h / 30.0)
    a = rng.uniform(0, math.pi, count)
    d = half[:, None] * np.stack([np.cos(a), np.sin(a)], 1)
    return np.concatenate([c - d, c + d], 1)


def _point_segment(px, py, seg):
    """Distance of points to one segment and the offset to its closest point."""
    x0, y0, x1, y1 = seg
    dx, dy = x1 - x0, y1 - y0
    t = np.clip(((px - x0) * dx + (py - y0) * dy) / (dx * dx + dy * dy), 0.0, 1.0)
    qx, qy = x0 + t * dx - px, y0 + t * dy - py
    return np.hypot(qx, qy), qx, qy


def _crowd(case, seed, index=0):
    """One scenario as plain numpy arrays: the agents' fields by name, the
    walls [W, 4], the navigation maps and the domain's size."""
    rng = np.random.default_rng([seed, index, case['n'], case['obstacles']])
    n, density = case['n'], case['density']
    if case['scenarios'] > 1:  # the rooms' sizes belong to the case, not to the seed
        sizes = np.random.default_rng([index, case['n'], case['scenarios']])
        n = _log_int(sizes, max(2, case['n'] // 16), case['n'])
        density = sizes.uniform(case['density'] / 6.0, case['density'])
    aspect = 1.0 if case['scenarios'] > 1 or case['kind'] == 'rollout' else \
        (4.0 if not case['graph'] and case['kind'] == 'steps' else 2.0)
    h = math.sqrt(n / density / aspect)
    inner = _segments(rng, case['obstacles'], aspect * h, h)
    # the rollout starts with a few agents in contact, whose gradients count
    pos, w, h = _place(rng, n, aspect * h, h, inner, 0.48 if case['kind'] == 'rollout' else 0.565)
    tc = case['model'] == 'three_circle'
    a = dict(position=pos, mass=_normal(rng, 80.0, 8.0, n), target_velocity=_normal(rng, 1.15, 0.2, n),
             radius=np.full(n, 0.25) if tc else rng.uniform(0.22, 0.28, n))
    gap = 0.6  # half the width of an exit
    walls = [(0, 0, w, 0), (w, 0, w, h), (w, h, 0, h), (0, h, 0, 0)]
    nav = None
    e0 = np.tile((1.0, 0.0), (n, 1))
    if case['nav'] >= 0:
        cx, cy = w / 2, h / 2
        walls = [(0, 0, cx - gap, 0), (cx + gap, 0, w, 0), (w, 0, w, cy - gap),
                 (w, cy + gap, w, h), (w, h, cx + gap, h), (cx - gap, h, 0, h),
                 (0, h, 0, cy + gap), (0, cy - gap, 0, 0)]
        exits = [(cx - gap, 0, cx + gap, 0), (w, cy - gap, w, cy + gap),
                 (cx - gap, h, cx + gap, h), (0, cy - gap, 0, cy + gap)]
        step = 0.1 if w <= 250 else 0.5
        X, Y = np.meshgrid(np.arange(0.0, w + step, step), np.arange(0.0, h + step, step))
        best = None
        for e in exits:
            d, qx, qy = _point_segment(X, Y, e)
            if best is None:
                best, bx, by = d, qx, qy
            else:
                m = d < best
                best, bx, by = np.where(m, d, best), np.where(m, qx, bx), np.where(m, qy, by)
        if case['nav'] == 1:
            maps = best[None]
        else:
            r = np.maximum(best, 1e-9)
            maps = np.stack([bx / r, by / r], -1)[None]
        nav = dict(maps=np.ascontiguousarray(maps), minx=0.0, miny=0.0, step=step,
                   mode=case['nav'])
        jj = np.clip((pos[:, 0] / step).astype(int), 0, best.shape[1] - 1)
        ii = np.clip((pos[:, 1] / step).astype(int), 0, best.shape[0] - 1)
        e0 = np.stack([bx[ii, jj], by[ii, jj]], 1)
        e0 /= np.maximum(np.hypot(e0[:, 0], e0[:, 1]), 1e-9)[:, None]
    elif case['kind'] == 'steps' and case['scenarios'] == 1:
        e0[rng.uniform(size=n) < 0.25] = (-1.0, 0.0)  # some walk the other way
    segs = np.concatenate([np.asarray(walls, dtype=np.float64), inner])
    if case['kind'] == 'rollout' and not case['obstacles']:
        segs = np.zeros((0, 4))  # the benchmark's rollout is an open square
    a['target_direction'] = e0
    a['velocity'] = a['target_velocity'][:, None] * e0 + rng.normal(0.0, 0.1, (n, 2))
    if case['precision'] == 'f32':  # what the fp32 mode holds exactly
        for f in ('target_direction', 'velocity'):
            a[f] = a[f].astype(np.float32).astype(np.float64)
    if tc:
        a['orientation'] = np.arctan2(e0[:, 1], e0[:, 0]) + rng.uniform(-0.3, 0.3, n)
        a['orientation'] = np.where(a['orientation'] > math.pi, a['orientation'] - TWO_PI,
                                    a['orientation'])
        a['r_t'], a['r_s'], a['r_ts'] = np.full(n, 0.15), np.full(n, 0.10), np.full(n, 0.15)
        a['target_angular_velocity'] = np.full(n, TWO_PI)
        off = 0.15 * np.stack([np.sin(a['orientation']), -np.cos(a['orientation'])], 1)
        a['position_ls'], a['position_rs'] = pos - off, pos + off
    a['inertia_rot'] = 4.0 * math.pi * (a['mass'] / 80.0) * (a['radius'] / 0.27) ** 2
    return types.SimpleNamespace(agents=a, n=n, segments=segs, nav=nav, w=w, h=h,
                                 seed=1 + 7 * seed + index)


def _records(case, crowd):
    from crowddynamics_amd.agents import empty_agents
    arr = empty_agents(crowd.n, case['model'])
    for f, v in crowd.agents.items():
        arr[f] = v
    arr['target'] = 0
    return arr


DT_MIN, DT_MAX = 0.001, 0.01
STATE = ('position', 'velocity', 'force', 'force_prev', 'target_direction', 'position_ls',
         'position_rs', 'orientation', 'angular_velocity', 'target_orientation', 'torque',
         'torque_prev')


def _keep(agents):
    return {f: agents[f].clone() for f in STATE if f in agents.fields}


def _set_back(agents, kept):
    for f, t in kept.items():
        agents[f].copy_(t)


def _outputs(case, agents):
    out = {f: agents[f] for f in ('position', 'velocity', 'force_prev')}
    if case['model'] == 'three_circle':
        out.update({f: agents[f] for f in ('orientation', 'angular_velocity', 'torque_prev')})
    return out


def prepare(case, seed):
    s = types.SimpleNamespace(case=case)
    vars(s).update(globals()['_prepare_' + case['kind']](case, seed))
    return s


def run(s):
    return globals()['_run_' + s.case['kind']](s)


# -- steps -------------------------------------------------------------------

def _prepare_steps(case, seed):
    from crowddynamics_amd.stepper import Stepper
    from crowddynamics_amd.ensemble import Ensemble
    if case['scenarios'] > 1:
        rooms = [_crowd(case, seed, k) for k in range(case['scenarios'])]
        st = Ensemble([types.SimpleNamespace(
            agents=_records(case, c), segments=c.segments, nav=None, cell_size=case['cell'],
            dt_min=DT_MIN, dt_max=DT_MAX, seed=c.seed, bounds=(0.0, 0.0, c.w, c.h))
            for c in rooms], precision=case['precision'], lanes=case['lanes'],
            order_every=case['order_every'])
    else:
        c = _crowd(case, seed)
        st = Stepper(_records(case, c), segments=c.segments, nav=c.nav, cell_size=case['cell'],
                     dt_min=DT_MIN, dt_max=DT_MAX, seed=c.seed, precision=case['precision'],
                     bounds=(0.0, 0.0, c.w, c.h), lanes=case['lanes'],
                     order_every=case['order_every'])
    kept = _keep(st.agents)
    stream = graph = None
    if case['graph']:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            st.step(1)
            graph = st.capture(case['steps'])
        torch.cuda.current_stream().wait_stream(stream)
    return dict(st=st, kept=kept, stream=stream, graph=graph)


def _run_steps(s):
    """An episode from the initial state."""
    st = s.st
    if s.graph is None:
        _set_back(st.agents, s.kept)
        st.prepare(0)
        st.step(s.case['steps'])
    else:
        now = torch.cuda.current_stream()
        s.stream.wait_stream(now)
        with torch.cuda.stream(s.stream):
            _set_back(st.agents, s.kept)
            st.prepare(0)
            s.graph.launch()
        now.wait_stream(s.stream)
    return _outputs(s.case, st.agents)


# -- tree --------------------------------------------------------------------

def _prepare_tree(case, seed):
    from crowddynamics_amd import logic as L
    from crowddynamics_amd.simulation import Agents, Field, MultiAgentSimulation
    c = _crowd(case, seed)
    cap = (int(1.5 * c.w / case['cell']) + 4) * (int(1.5 * c.h / case['cell']) + 4)
    sim = MultiAgentSimulation(field=Field(obstacles=c.segments),
                               agents=Agents(case['model'], _records(case, c), case['precision']),
                               name='tree', fused=False, cell_capacity=cap)
    sim.logic = L.Reset(sim) << (L.Integrator(sim, dt_min=DT_MIN, dt_max=DT_MAX) << (
        L.Fluctuation(sim, seed=c.seed),
        L.Adjusting(sim) << L.Orientation(sim),
        L.AgentAgentInteractions(sim, cell_size=case['cell']),
        L.AgentObstacleInteractions(sim)))
    sim.agents.ensure_device()
    return dict(sim=sim, kept=_keep(sim.agents.device))


def _run_tree(s):
    _set_back(s.sim.agents.device, s.kept)
    s.sim.data['iterations'] = 0
    s.sim.run(steps=s.case['steps'])
    return _outputs(s.case, s.sim.agents.device)


# -- rollout -----------------------------------------------------------------

def _rollout_inputs(case, seed):
    c = _crowd(case, seed)
    rng = np.random.default_rng([seed, 99])
    n = c.n
    par = [rng.uniform(2.5, 3.5, n), rng.uniform(1.1e5, 1.3e5, n), rng.uniform(3.6e4, 4.4e4, n),
           rng.uniform(450.0, 550.0, n), c.agents['target_velocity']]
    return c, par, rng.normal(0.0, 1.0, (case['steps'] + 1, n, 2))


DT_ROLLOUT = 0.005


def _prepare_rollout(case, seed):
    from crowddynamics_amd.adjoint import Rollout
    c, par, weights = _rollout_inputs(case, seed)
    r = Rollout(_records(case, c), case['steps'], dt=DT_ROLLOUT, cell_size=case['cell'],
                checkpoint=10, seed=c.seed, bounds=(0.0, 0.0, c.w, c.h), lanes=case['lanes'],
                segments=c.segments if len(c.segments) else None)
    dev = r.agents.device
    return dict(rollout=r, par=[torch.as_tensor(p, device=dev).requires_grad_() for p in par],
                weights=torch.as_tensor(weights, device=dev))


def _run_rollout(s):
    from crowddynamics_amd.adjoint import rollout_positions
    x = rollout_positions(s.rollout, *s.par)
    grads = torch.autograd.grad(x, s.par, s.weights)
    return dict(x=x.detach(), grads=list(grads))


# -- field -------------------------------------------------------------------

def _field_inputs(case, seed):
    """phi of a target (two exits) and of the obstacles, and the masks of the
    grown and of the bare obstacles, on a grid of n x n/2 nodes of 0.2 m."""
    rng = np.random.default_rng([seed, case['n'], case['obstacles'], 5])
    step, cols = 0.2, case['n']
    rows = max(3, cols // 2 + 1)
    w, h = step * (cols - 1), step * (rows - 1)
    X, Y = np.meshgrid(step * np.arange(cols), step * np.arange(rows))
    grown = np.zeros((rows, cols), dtype=bool)
    bare = np.zeros((rows, cols), dtype=bool)
    for seg in _segments(rng, case['obstacles'], w, h):
        d = _point_segment(X, Y, seg)[0]
        grown |= d <= 0.5
        bare |= d <= 0.6 * step
    phi_t, phi_o = np.full((rows, cols), -1.0), np.where(bare, 1.0, -1.0)
    a, b = int(rng.integers(1, max(2, rows - 8))), int(rng.integers(1, max(2, cols - 8)))
    phi_t[a:a + 7, 0] = 1.0
    phi_t[rows - 1, b:b + 7] = 1.0
    grown &= phi_t < 0
    return step, w, h, phi_t, phi_o, grown, bare


RADIUS, STRENGTH = 0.5, 0.3


def _prepare_field(case, seed):
    from crowddynamics_amd.field import FieldBuilder, meshgrid
    step, w, h, phi_t, phi_o, grown, bare = _field_inputs(case, seed)
    mg = meshgrid(step, 0.0, 0.0, w - 0.5 * step, h - 0.5 * step)
    if mg.shape != phi_t.shape:
        raise ValueError('grid of %s nodes, wanted %s' % (mg.shape, phi_t.shape))
    return dict(fb=FieldBuilder(mg), phi_t=torch.as_tensor(phi_t, device='cuda'),
                phi_o=torch.as_tensor(phi_o, device='cuda'), grown=grown, fill=~bare,
                reach=int(np.ceil(RADIUS / step)) + 3)


def _run_field(s):
    fb = s.fb
    dmap = fb.distance_map(s.phi_t, s.grown)
    tx, ty = fb.direction_map(dmap)
    tx, ty = fb.fill_missing(tx, ty, s.fill, s.reach)
    dobs = fb.distance_map(s.phi_o)
    ox, oy = fb.direction_map(dobs)
    fb.obstacle_handling(dobs, ox, oy, tx, ty, RADIUS, STRENGTH)
    return dict(dmap=dmap, dobs=dobs, tx=tx, ty=ty)


# -- neighbours --------------------------------------------------------------

SIGHT, NEAREST = 3.0, 8


def _prepare_neighbours(case, seed):
    from crowddynamics_amd.device import DeviceAgents, Workspace
    c = _crowd(case, seed)
    dev = DeviceAgents(_records(case, c))
    ws = Workspace(c.n, (int(c.w / SIGHT) + 4) * (int(c.h / SIGHT) + 4), 0, cell_slots=4)
    herding = np.random.default_rng([seed, 3]).uniform(size=c.n) < 0.5
    return dict(agents=dev, ws=ws, segments=c.segments,
                herding=torch.as_tensor(herding, device='cuda'))


def _run_neighbours(s):
    from crowddynamics_amd import state
    nb = state.find_nearest_neighbors(s.agents, SIGHT, NEAREST, s.segments, s.ws)
    out, has = state.herding_interaction(s.agents, s.herding, nb, 0.5, math.pi / 6)
    return dict(neighbours=nb, direction=out, has=has)


# -- the work a pass cannot do without ---------------------------------------

def _mean_agents(case):
    if case['scenarios'] == 1:
        return case['n']
    # log-uniform between n / 16 and n
    return case['scenarios'] * case['n'] * (15.0 / 16.0) / math.log(16.0)


def work(case):
    """Bytes: the agents' state and parameters read and the state written once
    (the steps of a pass could keep them in cache).  Operations per step: the social terms of the pairs in sight (or, at
    small cells, of the pairs in adjacent cells), about 80 (circular) or 300
    (three-circle) each, and 400 per agent for noise, walls and integration."""
    if case['kind'] == 'field':
        nodes = case['n'] * (case['n'] // 2 + 1)
        return dict(bytes=nodes * (2 * 16 + 2 + 5 * 16.0), flops=nodes * 60.0)
    n = _mean_agents(case)
    rho = case['density'] * (0.58 if case['scenarios'] > 1 else 1.0)
    area = min((3 * case['cell']) ** 2, math.pi * 3.5 ** 2)
    if case['kind'] == 'neighbours':
        return dict(bytes=n * (32.0 + 8 * NEAREST + 25), flops=n * rho * math.pi * 9.0 * 20.0)
    real = 8 if case['precision'] == 'f64' else 4
    tc = case['model'] == 'three_circle'
    per_agent = 2 * 16 + 8 * 11 + 8 * 2 * real + (8 * 24 if tc else 0)  # in and out
    flops = rho * area * (300.0 if tc else 80.0) + 400.0
    k = case['steps']
    if case['kind'] == 'rollout':  # forward, and about four times that for the adjoint
        return dict(bytes=n * (per_agent + 40.0 + 32.0 * (k + 1)), flops=5.0 * n * k * flops)
    return dict(bytes=n * float(per_agent), flops=n * k * flops)


# -- the same outputs in 64 bits ---------------------------------------------

def _dev():
    return torch.device('cuda' if torch.cuda.is_available() else 'cpu')


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=_dev())


def _pairs(x, cell, within=None):
    """Ordered pairs (i, j), i != j, of agents in the same or adjacent cells
    (origin at the minimum, truncated indices), those closer than `within`."""
    n = len(x)
    l = ((x - x.min(0).values) / cell).to(torch.int64)
    nx, ny = (int(v) + 1 for v in l.max(0).values)
    flat = l[:, 0] * ny + l[:, 1]
    order = torch.argsort(flat, stable=True)
    count = torch.bincount(flat, minlength=nx * ny)
    start = torch.cumsum(count, 0) - count
    I, J = [], []
    ids = torch.arange(n, device=x.device)
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            cx, cy = l[:, 0] + dx, l[:, 1] + dy
            ok = (cx >= 0) & (cx < nx) & (cy >= 0) & (cy < ny)
            c = torch.where(ok, cx * ny + cy, torch.zeros_like(cx))
            m = torch.where(ok, count[c], torch.zeros_like(cx))
            i = torch.repeat_interleave(ids, m)
            k = torch.arange(len(i), device=x.device) - torch.repeat_interleave(
                torch.cumsum(m, 0) - m, m)
            j = order[torch.repeat_interleave(start[c], m) + k]
            keep = i != j
            if within is not None:
                d = x[i] - x[j]
                keep &= (d * d).sum(1) < within * within
            I.append(i[keep])
            J.append(j[keep])
    return torch.cat(I), torch.cat(J)


def _truncate(fx, fy, limit=2e3):
    length = torch.hypot(fx, fy)
    over = length > limit
    s = torch.where(over, limit / torch.where(over, length, torch.ones_like(length)),
                    torch.ones_like(length))
    return fx * s, fy * s


def _contact(h, nx, ny, vx, vy, mu, kappa, damping):
    kvt = kappa * (vx * ny - vy * nx)
    cvn = damping * (vx * nx + vy * ny)
    return -h * (mu * nx - kvt * ny) + cvn * nx, -h * (mu * ny + kvt * nx) + cvn * ny


def _safe(mask, v, other=1.0):
    return torch.where(mask, v, torch.full_like(v, other))


def _circular_pairs(x, v, P, cell):
    """Force of every agent from its pairs (its own side of each)."""
    I, J = _pairs(x.detach(), cell, 4.0)
    d, u = x[I] - x[J], v[I] - v[J]
    r = P['radius'][I] + P['radius'][J]
    dist = torch.hypot(d[:, 0], d[:, 1])
    h = dist - r
    a = (u * u).sum(1)
    b = -(d * u).sum(1)
    disc = b * b - a * ((d * d).sum(1) - r * r)
    sight = h < 3.0
    k = torch.nonzero(sight & (disc > 0) & (a != 0)).reshape(-1)
    tau = (b[k] - torch.sqrt(disc[k])) / a[k]
    k = k[(tau > 0) & (tau <= 30.0)]
    root, ak, t0 = torch.sqrt(disc[k])[:, None], a[k][:, None], P['tau_0'][I[k]]
    tau = (b[k] - root[:, 0]) / a[k]
    mag = (2.0 / tau + 1.0 / t0) * torch.exp(-tau / t0) / (tau * tau)
    g = (u[k] - (u[k] * b[k][:, None] + d[k] * ak) / root) / ak
    s = ((-P['mass'] * P['k_soc'])[I[k]] * mag)[:, None] * g
    f = torch.zeros_like(x).index_add(0, I[k], torch.stack(_truncate(s[:, 0], s[:, 1]), 1))
    k = torch.nonzero(sight & (h < 0)).reshape(-1)
    n = d[k] / dist[k][:, None]
    cx, cy = _contact(h[k], n[:, 0], n[:, 1], u[k, 0], u[k, 1], P['mu'][I[k]], P['kappa'][I[k]],
                      P['damping'][I[k]])
    return f.index_add(0, I[k], torch.stack([cx, cy], 1))


def _three_circle_pairs(x, v, P, S, cell):
    """Forces and torques of three-circle agents; the reference evaluates a
    pair once, in index order, and its second side keeps two quirks: the
    moment arm of agent j is built from agent i's part of j's index, and the
    first valid time to collision stays unless a later one is in (0, tau)."""
    I, J = _pairs(x, cell, 5.0)
    k = I < J
    I, J = I[k], J[k]
    parts = torch.stack([x, S['ls'], S['rs']], 1)
    rad = torch.stack([P['r_t'], P['r_s'], P['r_s']], 1)
    d = parts[I][:, :, None] - parts[J][:, None]          # [p, 3, 3, 2]
    r = rad[I][:, :, None] + rad[J][:, None]
    dist = torch.hypot(d[..., 0], d[..., 1])
    hh = (dist - r).reshape(-1, 9)
    at = torch.argmin(hh, 1)
    row = torch.arange(len(I), device=x.device)
    h = hh[row, at]
    keep = h < 3.0
    I, J, d, r, dist, at, h = (t[keep] for t in (I, J, d, r, dist, at, h))
    row = torch.arange(len(I), device=x.device)
    im, jm = at // 3, at % 3
    n = d[row, im, jm] / dist[row, im, jm][:, None]
    arm_i = parts[I, im] + rad[I, im][:, None] * n - x[I]
    arm_j = parts[I, jm] - rad[J, jm][:, None] * n - x[J]
    u = v[I] - v[J]
    a = (u * u).sum(1)
    b = -(d * u[:, None, None]).sum(-1).reshape(-1, 9)
    c = ((d * d).sum(-1) - r * r).reshape(-1, 9)
    root = torch.sqrt(b * b - a[:, None] * c)
    valid = ~torch.isnan(root) & (root != 0)
    tau_all = (b - root) / a[:, None]
    nan = torch.full_like(a, float('nan'))
    tau, bm, dm, sel = nan.clone(), nan.clone(), nan.clone(), torch.zeros_like(at)
    for q in range(9):
        t = tau_all[:, q]
        take = valid[:, q] & (torch.isnan(tau) | ((t > 0) & (t < tau)))
        tau, bm = torch.where(take, t, tau), torch.where(take, b[:, q], bm)
        dm, sel = torch.where(take, root[:, q], dm), torch.where(take, torch.full_like(sel, q), sel)
    social = (a != 0) & (tau > 0)
    sign = torch.tensor([0.0, 1.0, -1.0], dtype=x.dtype, device=x.device)
    off = torch.stack([P['r_ts'] * torch.sin(S['phi']), -P['r_ts'] * torch.cos(S['phi'])], 1)
    ro = sign[sel // 3][:, None] * off[I] - sign[sel % 3][:, None] * off[J]
    tau, a_, dm = _safe(social, tau), _safe(social, a), _safe(social, dm)
    bm = _safe(social, bm, 0.0)
    g = (u - (a_[:, None] * (x[I] - x[J] + 2.0 * ro) + bm[:, None] * u) / dm[:, None]) / a_[:, None]
    touch = h < 0
    f = torch.zeros_like(x)
    tq = torch.zeros(len(x), dtype=x.dtype, device=x.device)
    for own, arm, sg in ((I, arm_i, 1.0), (J, arm_j, -1.0)):
        t0 = P['tau_0'][own]
        mag = (2.0 / tau + 1.0 / t0) * torch.exp(-tau / t0) / (tau * tau)
        s = sg * ((-P['mass'] * P['k_soc'])[own] * mag)[:, None] * g
        sx, sy = _truncate(s[:, 0], s[:, 1])
        cx, cy = _contact(h, n[:, 0], n[:, 1], u[:, 0], u[:, 1], P['mu'][own], P['kappa'][own],
                          P['damping'][own])
        fx = _safe(social, sx, 0.0) + _safe(touch, sg * cx, 0.0)
        fy = _safe(social, sy, 0.0) + _safe(touch, sg * cy, 0.0)
        f = f.index_add(0, own, torch.stack([fx, fy], 1))
        tq = tq.index_add(0, own, arm[:, 0] * fy - arm[:, 1] * fx)
    return f, tq


def _wall_forces(x, v, P, S, segs):
    """Wall contacts: the agent's disc, or the closest of its three."""
    f, tq = torch.zeros_like(x), torch.zeros(len(x), dtype=x.dtype, device=x.device)
    tc = 'r_t' in P
    reach = float((P['r_ts'] + P['r_t']).max() if tc else P['radius'].max()) + 0.01
    for x0, y0, x1, y1 in segs.tolist():
        lw = math.hypot(x1 - x0, y1 - y0)
        tx, ty = (x1 - x0) / lw, (y1 - y0) / lw
        with torch.no_grad():
            near = ((x[:, 0] > min(x0, x1) - reach) & (x[:, 0] < max(x0, x1) + reach) &
                    (x[:, 1] > min(y0, y1) - reach) & (x[:, 1] < max(y0, y1) + reach))
            k = torch.nonzero(near).reshape(-1)
        if not len(k):
            continue
        best = None
        for p, r in ([(x, P['r_t']), (S['ls'], P['r_s']), (S['rs'], P['r_s'])] if tc else
                     [(x, P['radius'])]):
            q0 = torch.stack([p[k, 0] - x0, p[k, 1] - y0], 1)
            q1 = torch.stack([p[k, 0] - x1, p[k, 1] - y1], 1)
            lt = -(tx * q1[:, 0] + ty * q1[:, 1]) - (tx * q0[:, 0] + ty * q0[:, 1])
            ln = -ty * q0[:, 0] + tx * q0[:, 1]
            end = torch.where((lt > lw)[:, None], q0, q1)
            at_end = (lt.abs() > lw)
            e = torch.hypot(_safe(at_end, end[:, 0]), _safe(at_end, end[:, 1], 0.0))
            dist = torch.where(at_end, e, ln.abs())
            n = torch.where(at_end[:, None], end / e[:, None], torch.sign(ln)[:, None] *
                            torch.tensor([-ty, tx], dtype=x.dtype, device=x.device))
            cand = (dist - r[k], n, p[k], r[k])
            if best is None:
                best = cand
            else:
                m = cand[0] < best[0]
                best = tuple(torch.where(m if t.dim() == 1 else m[:, None], t, u)
                             for t, u in zip(cand, best))
        h, n, p, r = best
        hit = torch.nonzero(h < 0).reshape(-1)
        kk = k[hit]
        cx, cy = _contact(h[hit], n[hit, 0], n[hit, 1], v[kk, 0], v[kk, 1], P['mu'][kk],
                          P['kappa'][kk], P['damping'][kk])
        f = f.index_add(0, kk, torch.stack([cx, cy], 1))
        if tc:
            arm = p[hit] - r[hit][:, None] * n[hit] - x[kk]
            tq = tq.index_add(0, kk, arm[:, 0] * cy - arm[:, 1] * cx)
    return f, tq


def _philox(i, step, purpose, attempt, seed):
    """Philox4x32-10 (Salmon et al., SC'11) of counters (i, step, 0,
    purpose | attempt << 8) under the key `seed`; two uniforms."""
    m32 = 0xFFFFFFFF
    c = [i & m32, torch.full_like(i, step), torch.zeros_like(i),
         torch.full_like(i, purpose | (attempt << 8))]
    k0, k1 = seed & m32, seed >> 32
    for _ in range(10):
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        c = [((p1 >> 32) & m32) ^ c[1] ^ k0, p1 & m32, ((p0 >> 32) & m32) ^ c[3] ^ k1, p0 & m32]
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32

    def u01(hi, lo):
        return (((hi << 21) | (lo >> 11)).to(torch.float64) + 0.5) * 2.0 ** -53
    return u01(c[0], c[1]), u01(c[2], c[3])


def _truncnorm(i, step, purpose, seed):
    """Standard normal in [-3, 3] by Box-Muller with rejection."""
    z = None
    for attempt in range(16):
        u0, u1 = _philox(i, step, purpose, attempt, seed)
        new = torch.sqrt(-2.0 * torch.log(u0)) * torch.cos(TWO_PI * u1)
        z = new if z is None else torch.where(z.abs() <= 3.0, z, new)
        if bool((z.abs() <= 3.0).all()):
            return z
    return torch.where(z.abs() <= 3.0, z, torch.copysign(torch.full_like(z, 3.0), z))


def _navigate(x, e0, nav, maps):
    q = (x - torch.tensor([nav['minx'], nav['miny']], dtype=x.dtype, device=x.device)) / nav['step']
    rows, cols = maps.shape[1:3]
    if nav['mode'] == 0:
        ok = (q[:, 0] > -1) & (q[:, 0] < cols) & (q[:, 1] > -1) & (q[:, 1] < rows)
        j = q[:, 0].to(torch.int64).clamp(0, cols - 1)
        i = q[:, 1].to(torch.int64).clamp(0, rows - 1)
        return torch.where(ok[:, None], maps[0, i, j], e0)
    ok = (q[:, 0] >= 0) & (q[:, 0] <= cols - 1) & (q[:, 1] >= 0) & (q[:, 1] <= rows - 1)
    j = q[:, 0].to(torch.int64).clamp(0, cols - 2)
    i = q[:, 1].to(torch.int64).clamp(0, rows - 2)
    fx, fy, m = q[:, 0] - j, q[:, 1] - i, maps[0]
    gx = (m[i, j + 1] - m[i, j]) * (1 - fy) + (m[i + 1, j + 1] - m[i + 1, j]) * fy
    gy = (m[i + 1, j] - m[i, j]) * (1 - fx) + (m[i + 1, j + 1] - m[i, j + 1]) * fx
    g = torch.hypot(gx, gy)
    ok &= g > 0
    e = -torch.stack([gx, gy], 1) / _safe(ok, g)[:, None]
    return torch.where(ok[:, None], e, e0)


def _wrap(rad):
    r = torch.remainder(rad, TWO_PI)
    return torch.where(r > math.pi, r - TWO_PI, r)


def _parameters(case, c):
    const = dict(tau_adj=0.5, k_soc=1.5, tau_0=3.0, mu=1.2e5, kappa=4e4, damping=500.0,
                 std_rand_force=0.1, tau_rot=0.2, std_rand_torque=0.1)
    P = {f: _t(np.full(c.n, v)) for f, v in const.items()}
    for f in ('mass', 'radius', 'target_velocity', 'inertia_rot', 'r_t', 'r_s', 'r_ts',
              'target_angular_velocity'):
        if f in c.agents:
            P[f] = _t(c.agents[f])
    return P


def _exact_steps_of(case, c, steps):
    """The state after `steps` updates of one scenario, as a dict."""
    P = _parameters(case, c)
    tc = case['model'] == 'three_circle'
    x, v, e0 = (_t(c.agents[f]) for f in ('position', 'velocity', 'target_direction'))
    fp = torch.zeros_like(x)
    S = dict()
    if tc:
        S = dict(ls=_t(c.agents['position_ls']), rs=_t(c.agents['position_rs']),
                 phi=_t(c.agents['orientation']))
        omega, tp = torch.zeros_like(S['phi']), torch.zeros_like(S['phi'])
    ids = torch.arange(c.n, device=x.device)
    maps = _t(c.nav['maps']) if c.nav is not None else None
    for k in range(steps):
        u0, _ = _philox(ids, k, 0, 0, c.seed)
        mag = P['mass'] * P['std_rand_force'] * _truncnorm(ids, k, 1, c.seed).abs()
        f = mag[:, None] * torch.stack([torch.cos(TWO_PI * u0), torch.sin(TWO_PI * u0)], 1)
        if maps is not None:
            e0 = _navigate(x, e0, c.nav, maps)
        f = f + (P['mass'] / P['tau_adj'])[:, None] * (P['target_velocity'][:, None] * e0 - v)
        if tc:
            tq = P['inertia_rot'] * P['std_rand_torque'] * _truncnorm(ids, k, 2, c.seed)
            turn = _wrap(torch.atan2(e0[:, 1], e0[:, 0]) - S['phi']) / math.pi
            tq = tq + P['inertia_rot'] / P['tau_rot'] * (turn * P['target_angular_velocity'] - omega)
            pf, pt = _three_circle_pairs(x, v, P, S, case['cell'])
        else:
            pf, pt = _circular_pairs(x, v, P, case['cell']), 0.0
        wf, wt = _wall_forces(x, v, P, S, c.segments)
        f = f + pf + wf
        v_max = float(torch.hypot(v[:, 0], v[:, 1]).max())
        dt = DT_MAX if v_max == 0 else \
            min(DT_MAX, max(DT_MIN, 1.1 * float(P['target_velocity'].max()) * DT_MAX / v_max))
        m = P['mass'][:, None]
        v = v + (fp / m + f / m) / 2.0 * dt
        x = x + v * dt + f / m / 2.0 * (dt * dt)
        fp = f
        if tc:
            tq = tq + pt + wt
            inertia = P['inertia_rot']
            omega = omega + (tp + tq) / inertia / 2.0 * dt
            phi = _wrap(S['phi'] + omega * dt + tq / inertia / 2.0 * (dt * dt))
            tp = tq
            off = P['r_ts'][:, None] * torch.stack([torch.sin(phi), -torch.cos(phi)], 1)
            S = dict(phi=phi, ls=x - off, rs=x + off)
    out = dict(position=x, velocity=v, force_prev=fp)
    if tc:
        out.update(orientation=S['phi'], angular_velocity=omega, torque_prev=tp)
    return out


def _exact_steps(case, seed):
    rooms = [_crowd(case, seed, k) for k in range(case['scenarios'])]
    got = [_exact_steps_of(case, c, case['steps']) for c in rooms]
    return {f: torch.cat([g[f] for g in got]) for f in got[0]}


def _exact_tree(case, seed):
    return _exact_steps_of(case, _crowd(case, seed), case['steps'])


def _exact_rollout(case, seed):
    c, par, weights = _rollout_inputs(case, seed)
    P = _parameters(case, c)
    par = [_t(p).requires_grad_() for p in par]
    P.update(zip(('tau_0', 'mu', 'kappa', 'damping', 'target_velocity'), par))
    x, v, e0 = (_t(c.agents[f]) for f in ('position', 'velocity', 'target_direction'))
    fp, m, dt = torch.zeros_like(x), P['mass'][:, None], DT_ROLLOUT
    xs = [x]
    for _ in range(case['steps']):
        f = (P['mass'] / P['tau_adj'])[:, None] * (P['target_velocity'][:, None] * e0 - v)
        f = f + _circular_pairs(x, v, P, case['cell'])
        f = f + _wall_forces(x, v, P, {}, c.segments)[0]
        v = v + (fp / m + f / m) / 2.0 * dt
        x = x + v * dt + f / m / 2.0 * (dt * dt)
        fp = f
        xs.append(x)
    xs = torch.stack(xs)
    grads = torch.autograd.grad(xs, par, _t(weights), allow_unused=True)
    return dict(x=xs.detach(), grads=[torch.zeros_like(p) if g is None else g
                                      for g, p in zip(grads, par)])


def _eikonal(phi, mask, h):
    """First-order upwind distance by fast sweeping over anti-diagonals, the
    nodes next to the contour held at their interpolated distance."""
    rows, cols = phi.shape
    inf = np.inf
    u = np.full((rows + 2, cols + 2), inf)
    pad = np.full((rows + 2, cols + 2), np.nan)
    pad[1:-1, 1:-1] = np.where(mask, np.nan, phi)
    free = np.zeros((rows + 2, cols + 2), dtype=bool)
    p, inv = pad[1:-1, 1:-1], np.zeros((rows, cols))
    border = np.zeros((rows, cols), dtype=bool)
    with np.errstate(invalid='ignore', divide='ignore'):
        for a, b in ((pad[1:-1, :-2], pad[1:-1, 2:]), (pad[:-2, 1:-1], pad[2:, 1:-1])):
            d = np.full((rows, cols), inf)
            for q in (a, b):
                cross = p * q < 0
                d = np.where(cross, np.minimum(d, h * p / (p - q)), d)
            hit = np.isfinite(d)
            border |= hit
            inv = inv + np.where(hit, 1.0 / np.where(hit, d, 1.0) ** 2, 0.0)
        start = np.where(p == 0, 0.0, np.where(border, np.sqrt(1.0 / inv), inf))
    u[1:-1, 1:-1] = np.where(mask, inf, start)
    free[1:-1, 1:-1] = ~mask & ~border & (p != 0)
    diag = []
    for s in range(rows + cols - 1):
        r = np.arange(max(0, s - cols + 1), min(rows, s + 1))
        diag.append((r + 1) * (cols + 2) + (s - r) + 1)
    flip = [(r // (cols + 2)) * (cols + 2) + (cols + 1 - r % (cols + 2)) for r in diag]
    flat, fr = u.reshape(-1), free.reshape(-1)
    sets = [[k[fr[k]] for k in ds] for ds in (diag, flip)]
    for sweep in range(400):
        before = flat.copy()
        for ks in (sets[0], sets[0][::-1], sets[1], sets[1][::-1]):
            for k in ks:
                a = np.minimum(flat[k - 1], flat[k + 1])
                b = np.minimum(flat[k - cols - 2], flat[k + cols + 2])
                lo, hi = np.minimum(a, b), np.maximum(a, b)
                with np.errstate(invalid='ignore'):
                    d = lo - hi
                    two = (lo + hi + np.sqrt(2.0 * h * h - d * d)) / 2.0
                    new = np.where(np.isinf(hi) | (hi - lo >= h), lo + h, two)
                flat[k] = np.minimum(flat[k], new)
        if np.array_equal(before, flat):
            break
    out = u[1:-1, 1:-1]
    return np.where(mask | np.isinf(out), np.nan, np.where(phi < 0, -out, out))


def _directions(d):
    gy, gx = np.gradient(d)
    length = np.hypot(gx, gy)
    length[length == 0] = np.nan
    return gx / length, gy / length


def _exact_field(case, seed):
    step, _, _, phi_t, phi_o, grown, bare = _field_inputs(case, seed)
    rows, cols = phi_t.shape
    dmap = _eikonal(phi_t, grown, step)
    dobs = _eikonal(phi_o, np.zeros_like(grown), step)
    tx, ty = _directions(dmap)
    reach = int(np.ceil(RADIUS / step)) + 3
    missing = np.isnan(tx) | np.isnan(ty)
    sx, sy = tx.copy(), ty.copy()
    for r, c in zip(*np.nonzero(missing & ~bare)):
        r0, r1, c0, c1 = max(0, r - reach), r + reach + 1, max(0, c - reach), c + reach + 1
        rr, cc = np.nonzero(~missing[r0:r1, c0:c1])
        if len(rr):
            k = np.argmin((rr + r0 - r) ** 2 + (cc + c0 - c) ** 2)  # first of equals, row by row
            tx[r, c], ty[r, c] = sx[rr[k] + r0, cc[k] + c0], sy[rr[k] + r0, cc[k] + c0]
    ox, oy = _directions(dobs)
    with np.errstate(invalid='ignore'):
        x = -dobs
        near = (x > 0) & (x < RADIUS)
        p = np.where(near, STRENGTH ** (x / RADIUS), 0.0)
        tx = np.where(near, -p * ox + (1 - p) * tx, tx)
        ty = np.where(near, -p * oy + (1 - p) * ty, ty)
        length = np.hypot(tx, ty)
        return dict(dmap=dmap, dobs=dobs, tx=tx / length, ty=ty / length)


def _exact_neighbours(case, seed):
    c = _crowd(case, seed)
    x, v = _t(c.agents['position']), _t(c.agents['velocity'])
    herding = _t(np.random.default_rng([seed, 3]).uniform(size=c.n) < 0.5)
    I, J = _pairs(x, SIGHT, SIGHT)
    dist = torch.hypot(x[I, 0] - x[J, 0], x[I, 1] - x[J, 1])
    hidden = torch.zeros(len(I), dtype=torch.bool, device=x.device)
    u = x[J] - x[I]
    for x0, y0, x1, y1 in c.segments.tolist():
        wx, wy = x1 - x0, y1 - y0
        bx, by = x0 - x[I, 0], y0 - x[I, 1]
        det = u[:, 0] * wy - u[:, 1] * wx
        a, b = (bx * wy - by * wx) / det, (bx * u[:, 1] - by * u[:, 0]) / det
        hidden |= (det != 0) & (a >= 0) & (a <= 1) & (b >= 0) & (b <= 1)
    keep = ~hidden
    I, J, dist = I[keep], J[keep], dist[keep]
    o = torch.argsort(J, stable=True)
    o = o[torch.argsort(dist[o], stable=True)]
    o = o[torch.argsort(I[o], stable=True)]
    I, J = I[o], J[o]
    count = torch.bincount(I, minlength=c.n)
    rank = torch.arange(len(I), device=x.device) - (torch.cumsum(count, 0) - count)[I]
    keep = rank < NEAREST
    nb = torch.full((c.n, NEAREST), -1, dtype=torch.int64, device=x.device)
    nb[I[keep], rank[keep]] = J[keep]

    def unit(t):
        r = torch.hypot(t[..., 0], t[..., 1])
        return t / torch.where(r == 0, torch.ones_like(r), r)[..., None]
    j = nb.clamp(min=0)
    e = unit(x[j] - x[:, None])
    cj = -(e * unit(v[j])).sum(-1)
    moving = (v != 0).any(1)
    away = (nb >= 0) & moving[:, None] & moving[j] & ~((cj > math.cos(math.pi / 6)) & (cj < 1))
    num = away.sum(1)
    has = herding & (num > 0)
    mean = (x[j] * away[..., None]).sum(1) / num.clamp(min=1)[:, None]
    d = unit(0.5 * unit(mean - x) + 0.5 * unit((v[j] * away[..., None]).sum(1)))
    return dict(neighbours=nb, direction=torch.where(has[:, None], d, torch.zeros_like(d)), has=has)


def exact(case, seed):
    """The outputs of run() in 64 bits, without the framework's code; None
    where the pairs of the pass are too many to do in about 20 s."""
    w = work(case)
    if not torch.cuda.is_available() and w['flops'] > 2e10:
        return None
    if case['kind'] == 'field' and case['n'] > 1200:
        return None
    return globals()['_exact_' + case['kind']](case, seed)
