"""The passes that run on the 64-cell patches -- several fast sub-steps to a launch, the limiter with the thickness and wind
update, the transport with its rows cell-major -- and the slow tendency against the oracle where their shapes change: every
remainder of the sub-steps over a launch's three (air) or four (ocean), one to eight layers (at which the rings are
shallower as LDS fills), the ring kernels' three shapes of threads, meshes without ring tables, a thread to an edge's layer
(levels to 5) or to all of them (level 6), row counts about the four to a load and the eight to a block, meshes whose last
patch is part full (162, 642 and 2,562 cells are 2.5, 10.03 and 40.03 patches), walls, and a floor that holds many cells'
outflow back.

Bars, after one step, of the largest value: the FP64 form, whose sums keep the oracle's terms (the forcing Tp + G is added up
first and a cell's outflow is summed in its edges' table order, so the last digits differ), to 1e-12. The mixed form holds
the flux coefficients and the Coriolis term's operands in FP32: a step changes a wind by less than the largest wind, so by
those roundings of 6e-8 it and the fluxes differ by less than 2e-7 of theirs, and a thickness, which a step changes by less
than a hundredth, by less than 2e-9 (measured: 4.3e-8, 1.4e-8 and 5.6e-10 at most); a row, of which a step moves less than a
fifth, with the stencil's values and weights in FP32, by less than 2e-8 (measured: 3.8e-9)."""
import ctypes

import numpy as np
import pytest
import torch

from conftest import relmax

pytestmark = pytest.mark.gpu

BARS = {'double': dict(h=1e-12, u=1e-12, Fm=1e-12, rows=1e-12), 'mixed': dict(h=2e-9, u=2e-7, Fm=2e-7, rows=2e-8)}


def _within(diff, precision):
    assert all(v <= BARS[precision][k] for k, v in diff.items()), diff


def _np(t):
    return t.detach().cpu().numpy().copy()


def _step(g, precision, kw, h, u, dt, nfast, theta=None, edit=None):
    """One step of the library and of the oracle: their largest differences by name. With edit, a change of the mesh struct,
    the same step on the changed mesh instead, and the names of the kernels that it launched."""
    import oracle
    from insilica import _hip
    from insilica.gpu import DeviceGrid
    from insilica.layers import Layers
    dg, og = DeviceGrid(g, precision), oracle.Grid(g)
    if edit:
        edit(dg.s)
    lay, olay = Layers(dg, **kw), oracle.Layers(og, **kw)
    hd, ud, Fd = dg.asarray(h), dg.asarray(u), dg.zeros(kw['layers'], g.E)
    ho, uo, Fo = h.copy(), u.copy(), np.zeros((kw['layers'], g.E))
    td = None if theta is None else dg.asarray(theta)
    if theta is not None:
        lay.update_gfast(hd, td)
        olay.update_gfast(ho, theta)
    if edit:
        torch.cuda.synchronize()
        _hip.timing_start()
    lay.step(hd, ud, dt, nfast, Fd, theta=td)
    olay.step(ho, uo, dt, nfast, Fo, theta=theta)
    torch.cuda.synchronize()
    diff = dict(h=relmax(_np(hd), ho), u=relmax(_np(ud), uo), Fm=relmax(_np(Fd), Fo))
    print(diff, flush=True)
    return (diff, set(_hip.timing_stop())) if edit else diff


def _air(g, n, L):
    """An air stack of L layers: settings, thickness, wind, theta."""
    from insilica import cases
    from insilica.constants import CP_DRY, KAPPA, R_DRY
    from insilica.ocean import visc4
    st = cases.coupled_stack(g, seed=n + L, lmax=4)
    at = np.linspace(0.0, 2.0, L) if L > 1 else np.array([1.0])
    k, f = np.minimum(at.astype(int), 1), at - np.minimum(at.astype(int), 1)
    theta, u = (np.ascontiguousarray((1 - f)[:, None] * st[x][k] + f[:, None] * st[x][k + 1]) for x in ('theta', 'u'))
    h = np.repeat(st['h'].sum(0)[None] / L, L, 0)
    return dict(layers=L, gprime=[0.0] * (L - 1), nu4=visc4(g, 15.0), floor=10.0,
                air=dict(cp=CP_DRY, kappa=KAPPA, rd=R_DRY), thin_wind=100.0, stress=[0.0] * (L - 1) + [1e-2]), h, u, theta


def _ocean(g, n, L, wall, floor):
    """An ocean stack of L layers: settings, thickness, wind. floor below one: that share of the mean thickness."""
    from insilica import cases
    from insilica.ocean import visc4
    h2, b, u2, gp = cases.phillips(g, 3.0)
    rng = np.random.default_rng(n + L)
    h = np.repeat(h2.sum(0)[None] / L, L, 0)
    h = np.ascontiguousarray(h * (1 + rng.uniform(-0.01, 0.01, h.shape)))
    u = np.ascontiguousarray(u2[np.arange(L) % 2] + rng.normal(0, 2.0, (L, g.E)))
    kw = dict(layers=L, b=b, gprime=[gp / max(1, L - 1)] * (L - 1), stress=[0.0] * (L - 1) + [2.5e-4], nu4=visc4(g, 5.0),
              floor=float(floor * h.mean()) if floor < 1 else floor, vmix=5e-4)
    if wall:
        land = rng.random(g.N) < 0.1
        kw['wall'] = np.where(land[g.eI] | land[g.eJ], 0.0, 1.0)
        u *= kw['wall'][None]
    return kw, h, u


@pytest.mark.parametrize('precision', ['double', 'mixed'])
@pytest.mark.parametrize('n,L,nfast', [(6, 2, 3), (6, 8, 1), (2, 3, 1), (3, 3, 2), (4, 3, 3), (4, 1, 4), (4, 2, 5), (4, 4, 7), (3, 5, 9),
                                       (4, 6, 11), (4, 7, 8), (4, 8, 6)])
def test_air(grids, n, L, nfast, precision):
    print(f'case: air n={n} L={L} nfast={nfast} {precision}', flush=True)
    g = grids(n)
    kw, h, u, theta = _air(g, n, L)
    diff = _step(g, precision, kw, h, u, 120.0 * nfast, nfast, theta)
    _within(diff, precision)


@pytest.mark.parametrize('precision', ['double', 'mixed'])
@pytest.mark.parametrize('n,L,nfast,wall,floor', [(6, 4, 5, True, 0.995), (2, 2, 1, True, 1.0), (3, 1, 2, False, 1.0), (4, 2, 3, True, 1.0),
                                                  (4, 2, 4, True, 0.995), (3, 3, 5, True, 0.995), (4, 2, 6, False, 0.995),
                                                  (4, 5, 9, True, 0.999), (4, 8, 11, True, 0.995)])
def test_ocean(grids, n, L, nfast, wall, floor, precision):
    """floor below one: that share of the layers' mean thickness, which many cells start beneath."""
    print(f'case: ocean n={n} L={L} nfast={nfast} wall={wall} floor={floor} {precision}', flush=True)
    g = grids(n)
    kw, h, u = _ocean(g, n, L, wall, floor)
    diff = _step(g, precision, kw, h, u, 100.0 * nfast, nfast)
    _within(diff, precision)


def _wide(s):
    """Three rings said to touch more edges than three to a thread: as the level-7 mesh's largest patch does."""
    for r in range(3, 6):
        s.rg_edges[r] = max(s.rg_edges[r], 771)


@pytest.mark.parametrize('precision', ['double', 'mixed'])
@pytest.mark.parametrize('n,L,nfast', [(3, 1, 3), (4, 2, 4), (4, 3, 6), (4, 4, 9), (4, 5, 7), (4, 6, 3), (3, 8, 3)])
def test_air_wide_patches(grids, n, L, nfast, precision):
    """The shape with four edges and two cells to a thread, which level 7 runs (from six layers on LDS takes a ring less)."""
    print(f'case: air wide n={n} L={L} nfast={nfast} {precision}', flush=True)
    g = grids(n)
    kw, h, u, theta = _air(g, n, L)
    diff, ran = _step(g, precision, kw, h, u, 120.0 * nfast, nfast, theta, _wide)
    _within(diff, precision)
    assert 'af_rings' in ran and 'limit_rings' in ran, ran


@pytest.mark.parametrize('precision', ['double', 'mixed'])
def test_level_7(grids, precision):
    """One step of three air layers and of two ocean layers on the largest mesh that is served."""
    print(f'case: level 7 {precision}', flush=True)
    g = grids(7)
    kw, h, u, theta = _air(g, 7, 3)
    _within(_step(g, precision, kw, h, u, 180.0, 3, theta), precision)
    kw, h, u = _ocean(g, 7, 2, True, 0.995)
    _within(_step(g, precision, kw, h, u, 400.0, 8), precision)


@pytest.mark.parametrize('precision', ['double', 'mixed'])
@pytest.mark.parametrize('n,L,air', [(4, 3, True), (6, 3, True), (4, 5, True), (4, 2, False), (6, 3, False)])
def test_shelf(grids, n, L, air, precision):
    """Thin layers (thinner than shelf: their tendency blended with the nearest thick layers', or their pressure gradient
    faded) and a drag, with a thread per layer of an edge and with one for all of them."""
    print(f'case: shelf n={n} L={L} air={air} {precision}', flush=True)
    g = grids(n)
    kw, h, u, *theta = _air(g, n, L) if air else _ocean(g, n, L, True, 1.0)
    h = np.ascontiguousarray(h * (1 + np.random.default_rng(n).uniform(-0.3, 0.3, h.shape)))
    kw.update(shelf=float(h.mean()), drag=[1e-6 * (k + 1) for k in range(L)])
    _within(_step(g, precision, kw, h, u, 120.0, 2, *theta), precision)


@pytest.mark.parametrize('value', [1e200, 1e305, np.inf, -np.inf, np.nan])
@pytest.mark.parametrize('L,nfast', [(1, 1), (3, 1), (1, 4), (3, 4)])
def test_lost_values_spread_as_the_reference_has_them(grids, L, nfast, value):
    """A wind or a thickness that is infinite, not a number or about to overflow: after a step of the FP64 form the same
    values are finite, infinite and not a number as the oracle's, and the finite ones (among them those whose limiter met a
    flux that is not a number) agree."""
    print(f'case: lost values L={L} nfast={nfast} {value}', flush=True)
    import oracle
    from insilica.gpu import DeviceGrid
    from insilica.layers import Layers
    g = grids(3)
    for air in (True, False):
        for name in ('u', 'h'):
            kw, h, u, *theta = _air(g, 3, L) if air else _ocean(g, 3, L, False, 1.0)
            (u if name == 'u' else h)[0, 5] = value
            dg, og = DeviceGrid(g, 'double'), oracle.Grid(g)
            lay, olay = Layers(dg, **kw), oracle.Layers(og, **kw)
            got = dict(h=dg.asarray(h), u=dg.asarray(u), Fm=dg.zeros(L, g.E))
            want = dict(h=h, u=u, Fm=np.zeros((L, g.E)))
            td = dg.asarray(theta[0]) if air else None
            with np.errstate(all='ignore'):
                if air:
                    lay.update_gfast(got['h'], td)
                    olay.update_gfast(h, theta[0])
                lay.step(got['h'], got['u'], 100.0 * nfast, nfast, got['Fm'], theta=td)
                olay.step(h, u, 100.0 * nfast, nfast, want['Fm'], theta=theta[0] if air else None)
            for k, b in want.items():
                a = _np(got[k])
                assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b)), (air, name, k)
                m = np.isfinite(b)
                scale = np.maximum(np.abs(b[m]), np.median(np.abs(b[m]))) if m.any() else 1.0
                assert np.all(np.abs(a[m] - b[m]) <= 1e-9 * scale), (air, name, k)


def _no_rings(s):
    s.rg_head = None


@pytest.mark.parametrize('precision', ['double', 'mixed'])
@pytest.mark.parametrize('n,L,nfast', [(2, 3, 1), (4, 1, 4), (4, 3, 5), (3, 8, 3)])
def test_air_without_rings(grids, n, L, nfast, precision):
    """The passes of a mesh without the ring tables (one sub-step to a launch, the limiter apart from the update)."""
    print(f'case: air without rings n={n} L={L} nfast={nfast} {precision}', flush=True)
    g = grids(n)
    kw, h, u, theta = _air(g, n, L)
    diff, ran = _step(g, precision, kw, h, u, 120.0 * nfast, nfast, theta, _no_rings)
    _within(diff, precision)
    assert {'af_muphi', 'af_u', 'scale', 'limit_h'} <= ran and not {'af_rings', 'limit_rings'} & ran, ran


@pytest.mark.parametrize('precision', ['double', 'mixed'])
@pytest.mark.parametrize('n,L,nfast,wall,floor', [(2, 2, 1, True, 1.0), (4, 1, 3, False, 1.0), (4, 2, 5, True, 0.995),
                                                  (3, 8, 4, True, 0.999)])
def test_ocean_without_rings(grids, n, L, nfast, wall, floor, precision):
    print(f'case: ocean without rings n={n} L={L} nfast={nfast} wall={wall} floor={floor} {precision}', flush=True)
    g = grids(n)
    kw, h, u = _ocean(g, n, L, wall, floor)
    diff, ran = _step(g, precision, kw, h, u, 100.0 * nfast, nfast, edit=_no_rings)
    _within(diff, precision)
    assert {'bt_eta', 'bt_u', 'scale', 'limit_h', 'lay_u'} <= ran and not {'bt_rings', 'limit_rings'} & ran, ran


@pytest.mark.parametrize('air', [True, False])
def test_patches_too_large_for_a_block(grids, air):
    """Patches said to hold more cells of their own than a block has threads (each steps on one) are not stepped in rings."""
    print(f'case: patches too large, air={air}', flush=True)
    g = grids(3)

    def large(s):
        for r in range(6):
            s.rg_cells[r] = max(s.rg_cells[r], 300)
    if air:
        kw, h, u, theta = _air(g, 3, 3)
        diff, ran = _step(g, 'double', kw, h, u, 360.0, 3, theta, large)
    else:
        kw, h, u = _ocean(g, 3, 2, True, 1.0)
        diff, ran = _step(g, 'double', kw, h, u, 300.0, 3, edit=large)
    _within(diff, 'double')
    assert not {'af_rings', 'bt_rings', 'limit_rings'} & ran, ran


@pytest.mark.parametrize('precision', ['double', 'mixed'])
@pytest.mark.parametrize('n,L,K', [(4, 1, 1), (3, 3, 1), (4, 2, 2), (2, 5, 1), (4, 7, 1), (4, 2, 4), (3, 3, 3), (4, 4, 3),
                                   (4, 3, 5), (4, 8, 2), (4, 1, 17)])
def test_transport_rows(grids, n, L, K, precision):
    """K tracers of L layers by unequal mass fluxes, steep rows among them (row counts that fill their blocks, ones that do
    not, and ones that are kept apart), and the same rows where the scratch is not padded: both against the oracle, the FP64
    form's the same to the bit."""
    _transport(grids, n, L, K, precision)


@pytest.mark.parametrize('n,L,K,shapes', [(5, 3, 2, (8, 4)), (5, 5, 4, (8, 8)), (4, 7, 5, (8, 4)), (5, 3, 4, (4, 4)),
                                          (5, 7, 2, (0, 4)), (5, 5, 1, (8, 4)), (6, 3, 5, (8, 8)), (6, 1, 11, (4, 4)),
                                          (6, 3, 3, (0, 0)), (4, 5, 5, (0, 4)), (4, 4, 7, (8, 4))])
def test_transport_shapes(grids, n, L, K, shapes):
    """The same with four rows to a block, eight, and apart, in the FP64 and the mixed form, at the lines of the rule that
    chooses them."""
    for precision, rows in zip(('double', 'mixed'), shapes):
        assert _transport(grids, n, L, K, precision) == rows


def _transport(grids, n, L, K, precision):
    """Compares one step with the oracle; the rows to a block that it took, 0 for rows kept apart."""
    import oracle
    from insilica import _hip
    from insilica.gpu import DeviceGrid
    from insilica.transport import Transport
    print(f'case: transport n={n} L={L} K={K} {precision}', flush=True)
    g = grids(n)
    dg, og = DeviceGrid(g, precision), oracle.Grid(g)
    rng = np.random.default_rng(10 * L + K)
    area = g.areaCell
    M = np.stack([(1 + 0.1 * l) * area for l in range(L)])
    Fm = 0.03 * area.mean() * rng.normal(size=(L, g.E))
    M1 = np.zeros_like(M)
    oracle.mass_update(og, L, M, Fm, M1)
    assert M1.min() > 0
    rows = rng.random((L * K, g.N))
    rows[::3] = (rows[::3] > 0.7).astype(float)
    ro = rows.copy()
    oracle.transport(og, L, M, M1, Fm, ro, order=3)
    out = []
    for padded in (True, False):
        tr = Transport(dg, layers=L, tracers=K)
        if not padded:
            tr.s.rows_pad = 0
        rd = dg.asarray(rows)
        tr.step_rows(dg.asarray(M), dg.asarray(M1), dg.asarray(Fm), rd, 3)
        torch.cuda.synchronize()
        out.append(_np(rd))
        print('rows', relmax(out[-1], ro), flush=True)
        _within(dict(rows=relmax(out[-1], ro)), precision)
    if precision == 'double':
        assert np.array_equal(out[0], out[1])
    tr.s.rows_pad = (L * K + 3) // 4 * 4
    return _hip.lib().isw_transport_shape(dg.ref, ctypes.byref(tr.s), L * K)
