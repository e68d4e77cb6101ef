"""The work a user of this package has it do, as cases that can be timed and whose results can be compared.

Kinds of case (`kind`), each through the package's public entry points:

  world      a World stepped by one model hour, as the benchmark's default workload and any single run does
  ensemble   an Ensemble of seeded planets, batched per level, advanced by one model hour (parameter sweeps)
  air        one time-split RK3 step of the air's layers (Layers.step), the largest part of a tick
  ocean      one such step of the ocean's layers, with walls round the land
  transport  one flux-corrected transport step of the stacked tracer rows (Transport.step_rows)
  radiation  one pass of the k-table radiation over a set of columns (Longwave, then Shortwave)
  column     one step of the moist air column (AirPhysics.column)

Sizes: mesh levels 4 to 7 (2,562 to 163,842 cells), as the package's own workloads use them; 3, 5 and 7 air layers
(its presets), 2 and 3 ocean layers; up to 15 tracer rows; up to 256 longwave and 224 shortwave g-points; both
precisions. The steps that work in place start every pass from the same saved state (one device copy), as an ensemble
or a restart does, so that a pass repeated many times keeps meeting values that a running world meets.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parents[1] / 'insilica-world-v2_amd')
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

GRAV, CP, RD, P0 = 9.80616, 1004.6, 287.04, 1.0e5
KAPPA = RD / CP
AIR_PRESET = {3: 'coupled_stack', 5: 'aqua5', 7: 'aqua7'}


def listed():
    return [
        # The smallest call: a one-layer balanced jet with a tracer on the coarsest mesh in use, FP64. Launches and
        # latency only; what an interactive run or a test does.
        dict(name='jet_hour_n4_fp64', kind='world', preset='jet', n=4, precision='double'),
        # The benchmark's workload: three air over two ocean layers with land, 15 + 4 tracer rows, at level 6, a model
        # hour (8 ticks and an ocean step).
        dict(name='coupled_hour_n6_mixed', kind='world', preset='coupled_stack', n=6, precision='mixed'),
        # A sweep over planets: eight coupled worlds of two levels batched (so two meshes of several worlds each).
        dict(name='ensemble_hour_8x_n4n5', kind='ensemble', members=8, lo=4, hi=5, precision='mixed'),
        # The air's dynamics alone, at the benchmark's size in the mixed form, and in seven layers on a coarse mesh in
        # the form that parity work uses.
        dict(name='air_step_n6_l3_mixed', kind='air', n=6, layers=3, nfast=15, precision='mixed'),
        dict(name='air_step_n4_l7_fp64', kind='air', n=4, layers=7, nfast=12, precision='double'),
        # The ocean's dynamics on the finest mesh the serving workload asks for: the largest stencil call.
        dict(name='ocean_step_n7_l2_mixed', kind='ocean', n=7, layers=2, precision='mixed'),
        # Tracers: the air's fifteen rows at level 6; and an odd count of few rows in FP64 on a coarse mesh.
        dict(name='transport_n6_15rows_mixed', kind='transport', n=6, layers=3, tracers=5, precision='mixed'),
        dict(name='transport_n5_3rows_fp64', kind='transport', n=5, layers=3, tracers=1, precision='double'),
        # The radiation at the size its benchmark has (the level-6 mesh's columns, 7 layers, 256 + 224 g-points), and
        # a coarse mesh's columns in three layers with the reference's largest table, 144 g-points, in FP64.
        dict(name='radiation_40962x7_mixed', kind='radiation', columns=40962, layers=7, lw=16, sw=14, clouds=True,
             precision='mixed'),
        dict(name='radiation_2562x3_fp64', kind='radiation', columns=2562, layers=3, lw=9, sw=7, clouds=True,
             precision='double'),
        # The air column each tick of a moist world runs: seven layers with clouds under the k-tables' fluxes at level
        # 6 (mixed); three layers under gray radiation at level 5 (FP64), the aquaplanet preset.
        dict(name='column_n6_l7_cloud_mixed', kind='column', n=6, layers=7, cloud=True, precision='mixed'),
        dict(name='column_n5_l3_fp64', kind='column', n=5, layers=3, cloud=False, precision='double'),
    ]


def draw(rng):
    kind = rng.choice(['world', 'ensemble', 'air', 'air', 'ocean', 'transport', 'transport', 'radiation', 'radiation',
                       'column', 'column'])
    prec = rng.choice(['mixed', 'mixed', 'double'])
    wind = round(rng.uniform(2.0, 15.0), 2)              # m/s
    if kind == 'world':
        preset = rng.choice(['coupled_stack', 'jet', 'aqua', 'aqua5'])
        return dict(kind=kind, preset=preset, n=rng.choice([4, 5, 6] if preset == 'coupled_stack' else [4, 5]),
                    radius=round(rng.uniform(0.8, 1.5), 3), precision=prec)
    if kind == 'ensemble':
        return dict(kind=kind, members=rng.randint(2, 9), lo=4, hi=rng.choice([4, 5]), precision='mixed')
    if kind == 'air':
        return dict(kind=kind, n=rng.choice([4, 5, 6]), layers=rng.choice([3, 5, 7]), nfast=rng.randint(10, 17),
                    wind=wind, precision=prec)
    if kind == 'ocean':
        return dict(kind=kind, n=rng.choice([4, 5, 6, 7]), layers=rng.choice([2, 3]), wind=0.05 * wind, precision=prec)
    if kind == 'transport':
        return dict(kind=kind, n=rng.choice([4, 5, 6]), layers=rng.choice([3, 5, 7]), tracers=rng.randint(1, 5),
                    wind=wind, precision=prec)
    if kind == 'radiation':
        most = 40962 if prec == 'mixed' else 9000
        return dict(kind=kind, columns=int(math.exp(rng.uniform(math.log(500), math.log(most)))),
                    layers=rng.randint(2, 8 if most > 9000 else 5), lw=rng.randint(4, 15), sw=rng.randint(4, 13),
                    clouds=rng.random() < 0.7, precision=prec)
    return dict(kind=kind, n=rng.choice([4, 5, 6]), layers=rng.choice([3, 5, 7]), cloud=rng.random() < 0.5,
                wind=wind, precision=prec)


# ---- inputs ----
def _mesh(n):
    from insilica import grid
    return grid.get(n)


def _smooth(rng, x, count):
    """`count` seeded smooth fields (random cubic polynomials of position) at unit positions x (M, 3), each scaled to
    a maximum of 1."""
    basis = [x[:, i] for i in range(3)]
    basis += [x[:, i] * x[:, j] for i in range(3) for j in range(i, 3)]
    basis += [x[:, i] * x[:, j] * x[:, k] for i in range(3) for j in range(i, 3) for k in range(j, 3)]
    f = rng.standard_normal((count, len(basis))) @ np.stack(basis)
    return f / np.max(np.abs(f), axis=1, keepdims=True)


def _winds(rng, g, layers, speed):
    """Seeded smooth winds' normal components at the edges (layers, E)."""
    v = _smooth(rng, g.xm, 3 * layers).reshape(layers, 3, -1)
    return speed * np.einsum('lce,ec->le', v, g.ne)


class _Saved:
    """Arrays that a step changes in place, as views of one buffer, and the buffer as it was."""

    def __init__(self, **arrays):
        arrays = {k: torch.as_tensor(np.asarray(v), dtype=torch.float64) if not torch.is_tensor(v) else v
                  for k, v in arrays.items()}
        self.flat = torch.empty(sum(a.numel() for a in arrays.values()), dtype=torch.float64, device='cuda')
        self.at, o = {}, 0
        for k, a in arrays.items():
            self.at[k] = self.flat[o:o + a.numel()].view(a.shape)
            self.at[k].copy_(a)
            o += a.numel()
        self.start = self.flat.clone()

    def restore(self):
        self.flat.copy_(self.start)


def _air_world(n, layers, precision, seed, nfast=None, wind=None):
    """An air world of this many layers with seeded perturbations of theta and wind."""
    from insilica.world import World
    params = dict(seed=seed)
    if nfast:
        params['nfast'] = nfast
    w = World(n, AIR_PRESET[layers], params=params, precision=precision)
    if layers != 3 or wind:                              # (the deeper presets start at rest)
        rng = np.random.default_rng(seed)
        w.u.copy_(w.dg.asarray(_winds(rng, w.grid, layers, wind or 15.0)))
        w.theta.add_(w.dg.asarray(2.0 * _smooth(rng, w.grid.pos, layers)))
    return w


def _ocean(n, layers, precision, seed, wind):
    from insilica import cases
    from insilica.gpu import DeviceGrid
    from insilica.ocean import Ocean
    g = _mesh(n)
    rng = np.random.default_rng(seed)
    land = cases.land_mask(g, rng, 0.3)
    cfg = dict(gprime=(0.016,), h_layers=(100.0,)) if layers == 2 else {}
    Ts = 273.15 + 27.0 * (1 - g.pos[:, 2] ** 2) + _smooth(rng, g.pos, 1)[0]
    sea = Ocean(DeviceGrid(g, precision), cfg, Tsurf=Ts, land=land)
    dh = 10.0 * _smooth(rng, g.pos, layers)
    dh[-1] = 0.2 * _smooth(rng, g.pos, 1)[0] - dh[:-1].sum(0)         # (the surface within +-0.2 m)
    h = sea.h.cpu().numpy() + dh
    u = _winds(rng, g, layers, wind) * (np.asarray(sea.wall_host) != 0)
    return sea, h, u


def _radiation_inputs(case, seed):
    from insilica.ktables import column_state, synthetic_lw, synthetic_sw
    N, L = case['columns'], case['layers']
    k = np.arange(N) + 0.5
    z = 1 - 2 * k / N
    lon = k * math.pi * (3 - math.sqrt(5))
    pos = np.stack([np.sqrt(1 - z * z) * np.cos(lon), np.sqrt(1 - z * z) * np.sin(lon), z], 1)
    c = column_state(pos, layers=L, seed=seed)
    if not case['clouds']:
        c['cloudo'] = None
    return pos, c, synthetic_lw(bands=case['lw'], seed=3), synthetic_sw(bands=case['sw'], seed=4)


def _stars(L):
    return list(np.linspace(500.0, 300.0, L - 1))


def prepare(case, seed):
    kind, prec = case['kind'], case['precision']
    if kind == 'world':
        from insilica.world import World
        params = dict(seed=seed)
        if case['preset'] == 'coupled_stack':
            params['nfast'] = 15
        if 'radius' in case:                             # another planet: its nfast follows from its mesh
            from insilica.constants import GRAV as G0, OMEGA, R_PLANET
            params = dict(seed=seed, planet=dict(radius=R_PLANET * case['radius'], omega=OMEGA, grav=G0))
            if case['preset'] == 'coupled_stack':
                params['visc4_U'] = 15.0 * case['radius']
        w = World(case['n'], case['preset'], params=params, precision=prec)
        if case['preset'].startswith('aqua'):
            rng = np.random.default_rng(seed)
            w.u.copy_(w.dg.asarray(_winds(rng, w.grid, w.L, 5.0)))
            w.theta.add_(w.dg.asarray(_smooth(rng, w.grid.pos, w.L)))
        return dict(kind=kind, w=w, ticks=int(round(w.ticks_per_hour)))
    if kind == 'ensemble':
        from insilica.ensemble import Ensemble, draw_planets
        from insilica.world import World
        specs = draw_planets(case['members'], seed=seed, levels=tuple(range(case['lo'], case['hi'] + 1)))
        return dict(kind=kind, e=Ensemble([World(n, 'coupled_stack', precision=prec, params=p) for n, p in specs],
                                          batch=True))
    if kind == 'air':
        w = _air_world(case['n'], case['layers'], prec, seed, case['nfast'], case.get('wind'))
        return dict(kind=kind, core=w.core, s=_Saved(h=w.h, u=w.u), theta=w.theta, dt=w.dt, nfast=case['nfast'],
                    Fm=w.dg.zeros(w.L, w.dg.E), grid=w.grid)
    if kind == 'ocean':
        sea, h, u = _ocean(case['n'], case['layers'], prec, seed, case.get('wind', 0.3))
        return dict(kind=kind, core=sea.core, s=_Saved(h=h, u=u), theta=None, dt=sea.cfg['dt'], nfast=sea.nfast,
                    Fm=sea.dg.zeros(sea.L, sea.dg.E), grid=sea.dg.host, wall=sea.wall_host, sea=sea)
    if kind == 'transport':
        from insilica.transport import Transport
        w = _air_world(case['n'], case['layers'], prec, seed, wind=case.get('wind'))
        L, K, dg = case['layers'], case['tracers'], w.dg
        rng = np.random.default_rng(seed + 1)
        rows = _smooth(rng, w.grid.pos, L * K)
        rows = np.where(np.arange(L * K)[:, None] // L % 2 == 0, 300.0 + 20.0 * rows, np.maximum(0.01 * rows, 0.0))
        h, u, Fm, M1 = w.h.clone(), w.u.clone(), dg.zeros(L, dg.E), dg.zeros(L, dg.N)
        w.core.step(h, u, w.dt, w.nfast, Fm, theta=w.theta)
        tr = Transport(dg, layers=L, tracers=K)
        tr.mass_after(w.M, Fm, M1)
        return dict(kind=kind, tr=tr, M0=w.M, M1=M1, Fm=Fm, s=_Saved(rows=rows), grid=w.grid)
    if kind == 'radiation':
        from insilica.atmosphere import par_array
        from insilica.radiation import Longwave, Shortwave
        pos, c, lwt, swt = _radiation_inputs(case, seed)
        N, L = case['columns'], case['layers']
        par = par_array(L, dict(edge_k=2.0, theta_stars=_stars(L)))
        lw = Longwave(N, L, par, tables=lwt, precision=prec)
        sw = Shortwave(N, L, par, lw, tables=swt, ice_re=30e-6, precision=prec)
        dev = lambda a: None if a is None else torch.as_tensor(np.ascontiguousarray(a), device='cuda')
        return dict(kind=kind, lw=lw, sw=sw, pos=dev(pos), t=dev(np.array([2.0e6])),
                    **{k: dev(v) for k, v in c.items()})
    # column
    from insilica.ktables import synthetic_lw, synthetic_sw
    from insilica.world import World
    rng = np.random.default_rng(seed)
    L = case['layers']
    preset = {3: 'aqua', 5: 'aqua5', 7: 'aqua7'}[L]
    params = dict(physics=dict(cloud=1.0, ice_air=1.0, edge_k=2.0), longwave='ktables', lw_tables=synthetic_lw(seed=3),
                  sw_tables=synthetic_sw(seed=4)) if case['cloud'] else {}
    w = World(case['n'], preset, params=params, precision=prec)
    g, N = w.grid, w.grid.N
    theta = w.theta.cpu().numpy() + 2.0 * _smooth(rng, g.pos, L) + rng.normal(0.0, 0.3, (L, N))
    q = w.q.cpu().numpy() * rng.uniform(0.6, 1.3, (L, N))
    Ts = w.Ts.cpu().numpy() + rng.normal(0.0, 1.0, N)
    ice = np.where(Ts < 272.0, rng.uniform(0.0, 900.0, N), 0.0)
    cw = 3e-4 * np.where(rng.uniform(size=(L, N)) < 0.35, rng.uniform(0.1, 0.9, (L, N)), 0.0)
    s = _Saved(theta=theta, q=q, Ts=Ts, ice=ice, t=np.array([2.0e6]), **(dict(cw=cw) if case['cloud'] else {}))
    w.u.copy_(w.dg.asarray(_winds(rng, g, L, case.get('wind', 12.0))))
    a = s.at
    if case['cloud']:
        w.physics.radiate(w.h, a['theta'], a['Ts'], a['t'], 3600.0, q=a['q'])
    return dict(kind=kind, w=w, s=s, dt=450.0)


# ---- one pass ----
def run(state):
    kind = state['kind']
    if kind == 'world':
        w = state['w']
        w.step(state['ticks'])
        return w.state_arrays()
    if kind == 'ensemble':
        e = state['e']
        e.advance(1)
        return [[b.h, b.u, b.M, b.rows, b.oh, b.ou, b.oM, b.orows, b.oTg] for b in e.units]
    s = state.get('s')
    if s is not None:
        s.restore()
        a = s.at
    if kind in ('air', 'ocean'):
        state['core'].step(a['h'], a['u'], state['dt'], state['nfast'], state['Fm'], theta=state['theta'])
        return dict(h=a['h'], u=a['u'], Fm=state['Fm'])
    if kind == 'transport':
        state['tr'].step_rows(state['M0'], state['M1'], state['Fm'], a['rows'], order=3)
        return a['rows']
    if kind == 'radiation':
        lw, sw = state['lw'], state['sw']
        lw(state['mu'], state['theta'], state['q'], state['cloudo'], state['Ts'])
        sw(0, state['t'], 3600.0, state['pos'], state['alb'], state['cloudo'])
        return dict(radf=lw.radf, swf=sw.swf)
    w = state['w']
    p = w.physics
    p.column(w.h, a['theta'], a['Ts'], w.u, a['t'], state['dt'], elev=w.b, q=a['q'], ice=a['ice'], cw=a.get('cw'))
    out = dict(a, wx=p.wx, olr=p.olr, sw_abs=p.sw_abs, stored=p.stored, rain=p.rain, evap=p.evap, tsurf=p.tsurf)
    if 'cw' in a:
        out['cloudo'] = p.cloudo
    return out


# ---- what a pass cannot do without ----
def _sizes(n):
    N = 10 * 4 ** n + 2
    return N, 3 * (N - 2), 2 * (N - 2)


def _mesh_bytes(n):
    """The tables a step reads: six edges, signs and neighbours per cell, two cells and vertices, lengths and about ten
    weighted neighbours per edge, three cells and edges per vertex."""
    N, E, NV = _sizes(n)
    return N * (6 * 9 + 6 * 8 + 8) + E * (4 * 4 + 2 * 8 + 10 * 12) + NV * (3 * 10 + 16)


def _dynamics_work(n, L, nfast):
    """Operations of one split step: per cell and layer about 50 per fast sub-step (stages of a third, a half and all
    of them) and 370 per stage for the slow tendency, the potential and the limiter."""
    N, E, _ = _sizes(n)
    subs = math.ceil(nfast / 3) + math.ceil(nfast / 2) + nfast
    return dict(bytes=_mesh_bytes(n) + 8.0 * L * (3 * N + 3 * E), flops=N * L * (50.0 * subs + 3 * 370))


def _transport_work(n, rows, L):
    N, E, _ = _sizes(n)
    return dict(bytes=2 * 8.0 * rows * N + 8.0 * L * (2 * N + E) + E * (8 * 12 + 8) + 48.0 * N, flops=320.0 * rows * N)


def _world_work(preset, n):
    N = _sizes(n)[0]
    dt = 600.0 if preset == 'jet' else 900.0 * 2.0 ** (5 - n)
    ticks = 3600.0 / dt
    L, rows = {'jet': (1, 1), 'coupled_stack': (3, 15), 'aqua': (3, 6), 'aqua5': (5, 10)}[preset]
    d, t = _dynamics_work(n, L, 15 if preset == 'coupled_stack' else 4), _transport_work(n, rows, L)
    flops = ticks * (d['flops'] + t['flops'] + (1500.0 * L * N if preset.startswith('aqua') else 0.0))
    extra = 0.0
    if preset == 'coupled_stack':
        o, ot = _dynamics_work(n, 2, 20), _transport_work(n, 4, 2)
        flops += o['flops'] + ot['flops']
        extra = 8.0 * (4 * N + 2 * 3 * N + 6 * N) * 2
    return dict(bytes=d['bytes'] + t['bytes'] + extra, flops=flops)


def work(case):
    kind = case['kind']
    if kind == 'world':
        return _world_work(case['preset'], case['n'])
    if kind == 'ensemble':
        levels = range(case['lo'], case['hi'] + 1)
        parts = [_world_work('coupled_stack', levels[k % len(levels)]) for k in range(case['members'])]
        return {k: sum(p[k] for p in parts) for k in ('bytes', 'flops')}
    if kind == 'air':
        return _dynamics_work(case['n'], case['layers'], case['nfast'])
    if kind == 'ocean':
        return _dynamics_work(case['n'], case['layers'], 10 * 2 ** (case['n'] - 4))
    if kind == 'transport':
        return _transport_work(case['n'], case['layers'] * case['tracers'], case['layers'])
    if kind == 'radiation':
        # per column, g-point and sub-level: six or seven table look-ups with an exponential, the optical depth, the
        # two-stream passes both ways (longwave) or the layer's optics and the adding both ways (shortwave)
        N, L = case['columns'], case['layers']
        nl, ns = 16 * case['lw'], 16 * case['sw']
        tables = 4.0 * (6 * 31 * 20 * nl + 211 * nl + 7 * 31 * 10 * ns)
        rows = (9 * L + 6) + (3 * L + 2) + 3 * L + 5 + (4 * L if case['clouds'] else 0)
        return dict(bytes=8.0 * rows * N + tables, flops=4.0 * L * N * (150.0 * nl + 200.0 * ns))
    N, E, _ = _sizes(case['n'])
    L = case['layers']
    rows = 2 * (2 * L + 2) + L + (L - 1) + 8 + ((2 * L + 4 * L + 3 + 9 * L + 6 + 3 * L + 2) if case['cloud'] else 0)
    return dict(bytes=8.0 * (rows * N + E) + 48.0 * N, flops=(2500.0 if case['cloud'] else 1500.0) * L * N)


# About four times what two correct variants are apart: for the mixed form its distance from the FP64 form (one and three
# model hours of the worlds, one pass of the others), for the FP64 form the same path with inputs changed by a rounding
# or its distance from exact(). The air column switches on thresholds, so its largest differences are far above its
# norm's; the radiation stores its per-g-point results as float32 in either form.
TOLERANCE = {
    ('world', 'double'): dict(rel=1e-12, max=1e-9),
    ('world', 'mixed'): dict(rel=1e-6, max=1e-4),
    ('ensemble', 'mixed'): dict(rel=3e-7, max=3e-6),
    ('air', 'double'): dict(rel=8e-14, max=1e-12),
    ('air', 'mixed'): dict(rel=8e-8, max=1e-6),
    ('ocean', 'double'): dict(rel=8e-14, max=1e-12),
    ('ocean', 'mixed'): dict(rel=8e-8, max=2e-6),
    ('transport', 'double'): dict(rel=4e-15, max=4e-14),
    ('transport', 'mixed'): dict(rel=2e-9, max=2e-8),
    ('radiation', 'double'): dict(rel=4e-7, max=4e-6),
    ('radiation', 'mixed'): dict(rel=2e-6, max=2e-5),
    ('column', 'double'): dict(rel=1e-10, max=1e-7),
    ('column', 'mixed'): dict(rel=1e-5, max=6e-4),
}


def tolerance(case):
    return TOLERANCE[(case['kind'], case['precision'])]


# ---- the same in 64 bits, in plain torch ----
class _Tables:
    """A mesh's tables as torch tensors, and the operators on them."""

    def __init__(self, g):
        dev = 'cuda' if torch.cuda.is_available() else 'cpu'
        long = lambda a: torch.as_tensor(np.asarray(a, dtype=np.int64), device=dev)
        real = lambda a: torch.as_tensor(np.asarray(a, dtype=np.float64), device=dev)
        self.N, self.E, self.eI, self.eJ = g.N, g.E, long(g.eI), long(g.eJ)
        self.ce = long(np.maximum(g.cellEdge, 0))
        self.sg = real(np.where(g.cellEdge >= 0, g.cellSign, 0))
        self.has = real(g.cellEdge >= 0)
        self.nb = long(np.where(g.nbr >= 0, g.nbr, np.arange(g.N)[:, None]))
        self.ev1, self.ev2, self.vE, self.vC = (long(x) for x in (g.ev1, g.ev2, g.vEdge, g.vCell))
        self.vs = real(g.vEdgeSign)
        self.vk = real(np.asarray(g.kite)[np.asarray(g.vCell), np.asarray(g.vSlot)])
        self.le, self.de, self.A, self.AV, self.fV = (real(x) for x in (g.le, g.de, g.areaCell, g.areaV, g.fV))
        self.w, self.eoe = real(g.w), long(g.eoe)
        self.own = torch.repeat_interleave(torch.arange(g.E, device=dev), long(np.diff(g.eoeStart)))

    def div(self, f):                                    # (L, E) edge flux times length -> its sum out of each cell
        return torch.sum(self.sg * (self.le * f)[:, self.ce], dim=2)

    def grad(self, x):
        return (x[:, self.eJ] - x[:, self.eI]) / self.de

    def mid(self, x):
        return 0.5 * (x[:, self.eI] + x[:, self.eJ])

    def curl(self, u):
        return torch.sum(self.vs * (self.de * u)[:, self.vE], dim=2) / self.AV

    def lap(self, u):
        z = self.curl(u)
        return self.grad(self.div(u) / self.A) - (z[:, self.ev2] - z[:, self.ev1]) / self.le


def _flip_cumsum(x):
    return torch.flip(torch.cumsum(torch.flip(x, [0]), 0), [0])


def _exact_layers(g, c, h, u, theta, dt, nfast):
    """One time-split RK3 step of a layer stack (c: its settings) from h, u: h, u, the last stage's volume flux."""
    T = _Tables(g)
    h0, u0, L = h, u, h.shape[0]
    air = theta is not None
    wet = torch.ones(T.E, dtype=torch.float64, device=h.device) if c['wall'] is None else (c['wall'] != 0).double()
    if air:
        pr = GRAV * torch.cumsum(h0, 0)
        dth = theta - torch.cat([theta[1:], torch.zeros_like(theta[:1])])
        S = torch.clamp(dth, min=0) * GRAV * KAPPA * CP * (pr / P0) ** KAPPA / pr
    he0 = T.mid(h0)
    ub0 = torch.sum(he0 * u0, 0) / torch.sum(he0, 0) * wet
    lap4 = T.lap(T.lap(u0))

    def stage(hs, us, frac):
        ke = torch.sum(T.has * (0.25 * T.le * T.de * us * us)[:, T.ce], dim=2) / T.A
        pib = None
        if air:
            p = GRAV * torch.cumsum(hs, 0)
            pt = torch.cat([torch.zeros_like(p[:1]), p[:-1]])
            x, xt = (p / P0) ** KAPPA, (pt / P0) ** KAPPA
            pib = CP * (p * x - pt * xt) / ((KAPPA + 1) * (p - pt))
            th = torch.cat([theta[:-1] - theta[1:], theta[-1:]])
            B = GRAV * c['b'] + _flip_cumsum(th * CP * x) - _flip_cumsum(S * torch.cumsum(hs, 0)) + ke
        else:
            z = c['b'] + _flip_cumsum(hs)
            gp = torch.tensor([0.0] + list(c['gprime']), dtype=torch.float64, device=h.device)
            B = torch.cumsum(gp[:, None] * z, 0) + ke
        hv = torch.sum(T.vk * hs[:, T.vC], dim=2) / T.AV
        q = (T.curl(us) + T.fV) / hv
        he, qe = T.mid(hs), 0.5 * (q[:, T.ev1] + q[:, T.ev2])
        h2 = torch.minimum(he[:, T.eoe], c['thin'] * he[:, T.own])
        d = torch.zeros_like(us).index_add_(1, T.own, T.w * h2 * us[:, T.eoe] * 0.5 * (qe[:, T.own] + qe[:, T.eoe]))
        d = d - T.grad(B) - c['nu4'] * lap4
        dts = frac * dt
        for k in range(L):
            if c['stress'][k] != 0:
                d[k] -= -torch.expm1(-c['stress'][k] / torch.clamp(he[k], min=c['floor']) * dts) / dts * us[k]
        if air:
            d = d + T.mid(pib) * T.grad(theta)
        H = torch.sum(he, 0)
        G = torch.sum(he * d, 0) / H
        Tp, ubs = d - G, torch.sum(he * us, 0) / H
        n = max(1, math.ceil(frac * nfast))
        tau = frac * dt / n
        if air:
            m, v, acc = h0, u0, torch.zeros_like(u0)
            for _ in range(n):
                acc = acc + v
                m1 = m - tau * T.div(he * v) / T.A
                phi = _flip_cumsum(S * torch.cumsum(m1 + c['damp'] * (m1 - m), 0))
                v = v + tau * (-T.grad(phi) + Tp + G)
                m = m1
            un, F = v, he * acc / n
        else:
            eta, v, acc = c['b'] + torch.sum(h0, 0), ub0, torch.zeros_like(ub0)
            for _ in range(n):
                acc = acc + v
                e1 = eta - tau * T.div((H * v)[None])[0] / T.A
                v = wet * (v + tau * (-T.grad((c['Gc'] * (e1 + c['damp'] * (e1 - eta)))[None])[0] + G))
                eta = e1
            un = wet * (u0 + dts * Tp + (v - ub0))
            F = wet * (he * (us - ubs) + he * acc / n)
        out = torch.sum(T.has * torch.clamp((T.sg * (T.le * F)[:, T.ce]) * dts, min=0), dim=2)
        room = torch.clamp(h0 - c['floor'], min=0) * T.A
        scale = torch.where(out > room, room / torch.clamp(out, min=1e-300), torch.ones_like(out))
        F = F * torch.where(F > 0, scale[:, T.eI], scale[:, T.eJ])
        return h0 - dts * T.div(F) / T.A, un, F * T.le * dt

    h1, u1, _ = stage(h0, u0, 1 / 3)
    h2, u2, _ = stage(h1, u1, 1 / 2)
    hn, un, Fm = stage(h2, u2, 1.0)
    if c['vmix'] != 0:
        un = un.clone()
        he = T.mid(hn)
        for k in range(L - 1):
            a, b = he[k], he[k + 1]
            mean, du = (a * un[k] + b * un[k + 1]) / (a + b), un[k] - un[k + 1]
            du = du * torch.exp(-c['vmix'] * (1 / a + 1 / b) * dt)
            un[k], un[k + 1] = mean + b / (a + b) * du, mean - a / (a + b) * du
        un = un * wet
    return dict(h=hn, u=un, Fm=Fm)


def _exact_transport(g, M0, M1, Fm, psi, L, beta=0.25):
    """One step of the third-order flux-corrected transport of the rows psi (row y by layer y % L's fluxes)."""
    from insilica.gpu import d2_stencil
    T = _Tables(g)
    idx, wt = d2_stencil(g)
    ix = torch.as_tensor(np.asarray(idx, dtype=np.int64).reshape(-1, 8), device=psi.device)
    wt = torch.as_tensor(wt.reshape(-1, 8), device=psi.device)
    rep = psi.shape[0] // L
    M0, M1, F = M0.repeat(rep, 1), M1.repeat(rep, 1), Fm.repeat(rep, 1)
    out = lambda f: torch.sum(T.sg * f[:, T.ce], dim=2)

    def high(p):
        d = wt * p[:, ix]
        a, b = torch.sum(d[:, :, :4], 2), torch.sum(d[:, :, 4:], 2)
        return F * (T.mid(p) - (a + b)) + torch.abs(F) * (b - a) * beta
    up = F * torch.where(F >= 0, psi[:, T.eI], psi[:, T.eJ])
    td = (M0 * psi - out(up)) / M1
    p = psi
    for c in (1 / 3, 1 / 2):
        p = (M0 * psi - c * out(high(p))) / (M0 - c * out(F))
    A = high(p) - up
    near = torch.cat([psi[:, T.nb], td[:, T.nb], psi[:, :, None], td[:, :, None]], dim=2)
    o = T.sg * A[:, T.ce]
    rise, fall = torch.sum(torch.clamp(-o, min=0), 2), torch.sum(torch.clamp(o, min=0), 2)
    lim = lambda room, need: torch.where(need > 0, torch.clamp(room / torch.clamp(need, min=1e-300), max=1.0), need * 0)
    Rp = lim((near.max(2).values - td) * M1, rise)
    Rm = lim((td - near.min(2).values) * M1, fall)
    C = torch.where(A > 0, torch.minimum(Rp[:, T.eJ], Rm[:, T.eI]), torch.minimum(Rp[:, T.eI], Rm[:, T.eJ]))
    return (td * M1 - out(C * A)) / M1


def _exact_radiation(case, seed):
    pos, c, lt, st = _radiation_inputs(case, seed)
    dev = 'cuda' if torch.cuda.is_available() else 'cpu'
    N = case['columns']
    step = max(64, int(4e6 / (16 * max(case['lw'], case['sw']))))
    parts = []
    for i in range(0, N, step):
        cut = {k: None if v is None else torch.as_tensor(v[..., i:i + step], device=dev) for k, v in c.items()}
        parts.append(_exact_columns(case['layers'], torch.as_tensor(pos[i:i + step], device=dev), cut, lt, st, dev))
    return dict(radf=torch.cat([p[0] for p in parts], 1), swf=torch.cat([p[1] for p in parts], 1))


def _exact_columns(L, pos, c, lt, st, dev):
    real = lambda a: torch.as_tensor(np.asarray(a, dtype=np.float64), device=dev)
    N, edge_k, eps_air, m_air, hs, nT = pos.shape[0], 2, 0.622, 28.9647, 1500.0, 0.190
    cl = c['cloudo']
    P, Tax, Tp = (np.asarray(lt[k], float) for k in ('P', 'T', 'T_pl'))
    lp0, dlp = math.log(P[0]), (math.log(P[0]) - math.log(P[-1])) / (len(P) - 1)
    at = lambda x, n: torch.clamp(x, 0.0, n - 1 - 1e-4)
    o3 = real(lt['o3'])
    # the sub-levels: four to a layer
    pb = GRAV * c['mu'][0]
    edges = [torch.zeros_like(pb), pb]
    for k in range(1, L):
        pb = pb + GRAV * c['mu'][k]
        edges.append(pb)
    sub = []
    for k in range(L):
        pt, pbk = edges[k], edges[k + 1]
        ex = lambda p: (p / P0) ** KAPPA
        pib = CP * (pbk * ex(pbk) - pt * ex(pt)) / ((KAPPA + 1) * (pbk - pt))
        strat = k < edge_k and L >= 3
        Tiso = pib * c['theta'][k] / CP
        Cn = Tiso * (nT + 1) * (pbk - pt) / (pbk ** (nT + 1) - pt ** (nT + 1))
        temp = lambda p: Tiso if strat else Cn * p ** nT
        share = (0, 0.05, 0.2, 0.5, 1) if k == 0 else (0, 0.25, 0.5, 0.75, 1)
        pe = [pt + f * (pbk - pt) for f in share]
        qk = torch.clamp(c['q'][k], min=0)
        qs, fr, lev = [], [], []
        for a, b in zip(pe[:-1], pe[1:]):
            pm = torch.where(a > 0, (b - a) / torch.log(b / torch.clamp(a, min=1e-30)), 0.5 * b)
            Tm, Tq = temp(0.5 * (a + b)), c['theta'][k] * (0.5 * (a + b) / P0) ** KAPPA
            sat = eps_air * 611.0 * torch.exp(17.27 * (Tq - 273.15) / (Tq - 35.85)) / pm
            qs.append(torch.ones_like(pm) if strat else torch.where(Tq < 160, torch.zeros_like(pm), sat))
            fr.append((b - a) / (pbk - pt))
            ua = (b - a) / (GRAV * m_air * 1e-3) * 6.02214076e23 / 1e4
            yo = at((lp0 - torch.log(pm)) / dlp, len(o3))
            io = yo.long()
            oz = o3[io] + (o3[io + 1] - o3[io]) * (yo - io)
            lev.append(dict(Tt=temp(a), Tb=temp(b), x=at((lp0 - torch.log(pm)) / dlp, len(P)),
                            T=(Tm - Tax[0]) / (Tax[1] - Tax[0]), ua=ua, oz=oz * ua,
                            haze=(b / edges[L]) ** (8000.0 / hs) - (a / edges[L]) ** (8000.0 / hs)))
        qm = sum(s * f for s, f in zip(qs, fr))
        cum, jc = torch.zeros_like(qm), torch.full_like(qm, 3, dtype=torch.long)
        found = torch.zeros_like(qm, dtype=torch.bool)
        for j in range(4):                               # the sub-level that holds the median of the layer's vapor
            cum = cum + torch.where(qm > 0, qs[j] * fr[j] / qm, torch.full_like(qm, 0.25))
            here = ~found & (cum >= 0.5)
            jc, found = torch.where(here, torch.full_like(jc, j), jc), found | here
        for j, s in enumerate(lev):
            qj = torch.where(qm > 0, qk * qs[j] / qm, qk)
            vap = qj / (1 - qj) * (m_air / 18.01528)
            s.update(vap=vap * s['ua'], frac=vap / 0.04, cloud=(jc == j).double())
        sub += lev

    def table(logk, s, y, gases):
        """The optical depth per g-point (columns, NG): exp of the bilinear ln k, water's two tables blended."""
        ip, it = s['x'].long(), y.long()
        fp, ft = (s['x'] - ip)[:, None], (y - it)[:, None]
        lk = [torch.exp(K[ip, it] * (1 - fp) * (1 - ft) + K[ip + 1, it] * fp * (1 - ft) + K[ip, it + 1] * (1 - fp) * ft +
                        K[ip + 1, it + 1] * fp * ft) for K in logk]
        tau = gases[0][:, None] * (lk[0] + (lk[1] - lk[0]) * s['frac'][:, None])
        return torch.clamp(sum((u[:, None] * k for u, k in zip(gases[1:], lk[2:])), tau), min=0)
    gases = lambda s: [s['vap'], 400e-6 * s['ua'], s['oz'], 0.32e-6 * s['ua'], 1.8e-6 * s['ua']]

    # longwave
    logk, planck = real(lt['logk']), real(lt['planck'])
    taus = [table(logk, s, at(s['T'], len(Tax)), gases(s)) for s in sub]

    def B(T):
        y = at(T - Tp[0], len(Tp))
        j = y.long()
        return planck[j] + (planck[j + 1] - planck[j]) * (y - j)[:, None]

    def through(I, tau, Bn, Bf):
        x = 1.66 * tau
        lin = torch.where(x > 1e-3, 1 + torch.expm1(-x) / torch.clamp(x, min=1e-30), x * (0.5 - x / 6))
        return I * torch.exp(-x) - Bf * torch.expm1(-x) + (Bn - Bf) * lin
    cover = [cl[k] if cl is not None else torch.zeros_like(pb) for k in range(L)]
    deep = [s['cloud'] * (cl[L + 3 + j // 4] if cl is not None else 0.0) for j, s in enumerate(sub)]
    E0 = 3 * (L + 1) + 3
    radf = torch.zeros(E0 + 6 * L, N, dtype=torch.float64, device=dev)
    rsum = lambda x: torch.sum(x, 1)
    I = torch.zeros_like(taus[0])
    for k in range(L):
        f = cover[k][:, None]
        Ic = Id = I
        mix = lambda: (1 - f) * Ic + f * Id
        for j in range(4 * k, 4 * k + 4):
            Bt, Bb = B(sub[j]['Tt']), B(sub[j]['Tb'])
            Ic, Id = through(Ic, taus[j], Bb, Bt), through(Id, taus[j] + deep[j][:, None] / 1.66, Bb, Bt)
            if j % 4 == 0:
                radf[E0 + 6 * k + 1] = math.pi * rsum(mix())
            if j % 4 == 2:
                radf[E0 + 6 * k + 4] = math.pi * rsum(mix())
        I = mix()
        radf[L + 1 + k + 1] = math.pi * rsum(I)
    Bs = B(c['Ts'])
    sB = rsum(Bs)
    I, tr, Iall, trall = torch.zeros_like(I), torch.ones_like(I), torch.zeros_like(I), torch.ones_like(I)
    radf[2 * (L + 1) + L] = 1.0
    for k in range(L - 1, -1, -1):
        f = cover[k][:, None]
        Ic = Id = I
        tc = td = tr
        for j in range(4 * k + 3, 4 * k - 1, -1):
            Bt, Bb = B(sub[j]['Tt']), B(sub[j]['Tb'])
            t1 = torch.exp(-1.66 * taus[j])
            Iall, trall = through(Iall, taus[j], Bt, Bb), trall * t1
            Ic, tc = through(Ic, taus[j], Bt, Bb), tc * t1
            Id = through(Id, taus[j] + deep[j][:, None] / 1.66, Bt, Bb)
            td = td * t1 * torch.exp(-deep[j])[:, None]
            e = 3 if j % 4 == 3 else 0 if j % 4 == 1 else None
            if e is not None:
                radf[E0 + 6 * k + e] = math.pi * rsum((1 - f) * Ic + f * Id)
                radf[E0 + 6 * k + e + 2] = rsum(((1 - f) * tc + f * td) * Bs) / sB
        I, tr = (1 - f) * Ic + f * Id, (1 - f) * tc + f * td
        radf[k], radf[2 * (L + 1) + k] = math.pi * rsum(I), rsum(tr * Bs) / sB
    radf[3 * (L + 1)], radf[3 * (L + 1) + 1] = math.pi * rsum(Iall), rsum(trall * Bs) / sB
    radf[3 * (L + 1) + 2] = sB

    # shortwave: the sun's mean cosine over the interval's daylight
    total, lit = torch.zeros_like(pb), torch.zeros_like(pb)
    for j in range(4):
        t = 2.0e6 + (j + 0.5) * 900.0
        ang, rot = 2 * math.pi * t / (365 * 86400.0), 2 * math.pi * math.fmod(t, 86400.0) / 86400.0
        dec = math.asin(math.sin(math.radians(23.44)) * math.sin(ang))
        cz = pos[:, 0] * math.cos(dec) * math.cos(rot) - pos[:, 1] * math.cos(dec) * math.sin(rot) + \
            pos[:, 2] * math.sin(dec)
        total, lit = total + torch.clamp(cz, min=0), lit + (cz > 0)
    mu0 = torch.clamp(torch.where(lit > 0, total / torch.clamp(lit, min=1), torch.full_like(total, 0.05)), min=0.02)[:, None]
    logk = real(st['logk'])
    sun, ray, hzf = (real(np.asarray(st[k], float)) for k in ('sun', 'ray', 'haze'))
    sun = sun / sun.sum()
    tau550, hssa, hg, _ = (float(x) for x in st['haze_par'])
    ng = np.asarray(st['ng'], int)
    ice = _ice_optics(30.0, st['band_top'])
    cssa, cssa_i, g_i = (real(np.repeat(a, ng)) for a in (st['cloud_ssa'], [x[0] for x in ice], [x[1] for x in ice]))
    yscale = 10.0 / (st['T'][1] - st['T'][0])

    def layer(tau, ssa, gg):
        f = gg * gg
        tau, ssa, gg = (1 - ssa * f) * tau, (1 - f) * ssa / (1 - ssa * f), (gg - f) / (1 - f)
        g1, g2 = (7 - ssa * (4 + 3 * gg)) / 4, -(1 - ssa * (4 - 3 * gg)) / 4
        g3 = (2 - 3 * gg * mu0) / 4
        g4 = 1 - g3
        a1, a2 = g1 * g4 + g2 * g3, g1 * g3 + g2 * g4
        k = torch.sqrt(torch.clamp((g1 - g2) * (g1 + g2), min=1e-12))
        e = torch.exp(-k * tau)
        e2, k2e = e * e, 2 * k * e
        rf = 1 / (k + g1 + (k - g1) * e2)
        Rd, Td, Tdd = g2 * (1 - e2) * rf, k2e * rf, torch.exp(-tau / mu0)
        km = k * mu0
        om = 1 - km * km
        om = torch.where(om.abs() < 1e-3, torch.where(om < 0, -1e-3, 1e-3), om)
        rf = ssa * rf / om
        Rs = rf * ((1 - km) * (a2 + k * g3) - (1 + km) * (a2 - k * g3) * e2 - k2e * (g3 - a2 * mu0) * Tdd)
        Ts = rf * (k2e * (g4 + a1 * mu0) - Tdd * ((1 + km) * (a1 + k * g4) - (1 - km) * (a1 - k * g4) * e2))
        Rs = torch.minimum(torch.clamp(Rs, min=0), 1 - Tdd)
        return Rd, Td, Rs, torch.minimum(torch.clamp(Ts, min=0), 1 - Tdd - Rs), Tdd

    clear, alls = [], []
    for j, s in enumerate(sub):
        tg = table(logk, s, at(s['T'] * yscale, len(st['T'])), gases(s) + [0.2095 * s['ua']])
        trs, ths = ray * s['ua'][:, None], tau550 * hzf * s['haze'][:, None]
        tt, sc = tg + trs + ths, trs + hssa * ths
        ga = torch.where(sc > 0, hg * hssa * ths / torch.clamp(sc, min=1e-300), sc * 0)
        one = layer(tt, torch.clamp(sc / torch.clamp(tt, min=1e-300), max=1 - 1e-6), ga)
        clear.append(one)
        if cl is None:
            alls.append(one)
            continue
        k = j // 4
        on = s['cloud'] * (cl[L + 3 + k] > 0)
        f, tc, sl = (on * cl[k])[:, None], (on * 0.7 * cl[2 * L + 3 + k])[:, None], cl[3 * L + 3 + k][:, None]
        wl, wi = sl * cssa, (1 - sl) * cssa_i
        cw = wl + wi
        cg = (wl * 0.85 + wi * g_i) / cw
        sc2 = sc + cw * tc
        two = layer(tt + tc, torch.clamp(sc2 / (tt + tc), max=1 - 1e-6), (ga * sc + cg * cw * tc) / sc2)
        f = torch.where(tc > 0, f, f * 0)
        alls.append(tuple((1 - f) * a + f * b for a, b in zip(one, two)))

    def albedos(optics):
        Ad = As = c['alb'][:, None] + torch.zeros_like(ray)
        out = [(Ad, As)]
        for Rd, Td, Rs, Ts, Tdd in reversed(optics):
            den = 1 / (1 - Ad * Rd)
            Ad, As = Rd + Td * Td * Ad * den, Rs + (Tdd * As + Ts * Ad) * Td * den
            out.append((Ad, As))
        return out[::-1]
    A, cA = albedos(alls), albedos(clear)
    swf = torch.zeros(3 * L + 2, N, dtype=torch.float64, device=dev)
    wsum = lambda x: torch.sum(sun * x, 1)
    Fdir, Fdif, net = torch.ones_like(A[0][0]), torch.zeros_like(A[0][0]), 1 - A[0][1]
    for j, (rd, td, rs, ts, tdd) in enumerate(alls):
        Ad, As = A[j + 1]
        Fdn = Fdir * tdd
        Fdif, Fdir = (td * Fdif + rd * As * Fdn + ts * Fdir) / (1 - Ad * rd), Fdn
        n2 = Fdir + Fdif - (Ad * Fdif + As * Fdir)
        k = j // 4
        swf[k] += wsum(net - n2)
        if j % 4 == 0:
            swf[L + 2 + 2 * k] = wsum(net - n2)
        if j % 4 == 3:
            swf[L + 3 + 2 * k] = wsum(net - n2)
        net = n2
    swf[L], swf[L + 1] = wsum(net), wsum(cA[0][1])
    return radf, swf


def _ice_optics(re, tops):
    """Ebert & Curry (1992): ice clouds' (single-scattering albedo, asymmetry) per band for an effective radius (um)."""
    C, D = (1.000e-05, 1.100e-04, 1.240e-02, 3.779e-02, 4.666e-01), (0.0, 1.405e-05, 6.867e-04, 1.284e-03, 2.050e-05)
    A, B = (7.661e-01, 7.730e-01, 7.865e-01, 8.172e-01, 9.595e-01), (5.851e-04, 5.665e-04, 7.204e-04, 7.463e-04, 1.076e-04)
    j = [0 if t > 14300 else 1 if t > 7700 else 2 if t > 5300 else 3 if t > 4000 else 4 for t in tops]
    return [(1 - C[i] - D[i] * re, min(A[i] + B[i] * re, 1 - 1e-6)) for i in j]


def exact(case, seed):
    """What run() returns, in 64 bits; None for whole worlds and the air column, which have no such short form."""
    kind = case['kind']
    if kind == 'radiation':
        return _exact_radiation(case, seed)
    if kind not in ('air', 'ocean', 'transport'):
        return None
    s = prepare(dict(case, precision='double'), seed)
    a = {k: v.clone() for k, v in s['s'].at.items()}
    if kind == 'transport':
        return _exact_transport(s['grid'], s['M0'], s['M1'], s['Fm'], a['rows'], case['layers'])
    k = s['core']
    c = dict(wall=k.wall, b=k.b, gprime=k.gprime, stress=k.stress, thin=k.thin, nu4=k.nu4, floor=k.floor,
             damp=k.div_damp, vmix=k.vmix, Gc=k.Gc)
    return _exact_layers(s['grid'], c, a['h'], a['u'], s['theta'], s['dt'], s['nfast'])
