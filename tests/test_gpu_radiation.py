"""The k-table radiation on the GPU against the CPU oracle, through the C ABI.

Bars (the per-g-point results are float32 in the reference's double path too, air.cu:2243,2395, so a last-bit
difference of exp or pow between the device library and glibc can move a g-point's value by one float32 step):
- lw_setup, plain FP64 form: the float32 sub-levels equal the oracle's to one float32 step (2.5e-7 relative);
- lw_column and sw_column, FP64 form, on the same sub-levels: within 1e-8 (longwave: of the surface's downward flux,
  as the reference's kernel test scales it, tests/test_radiation.py:160-162; shortwave: shares of the sunlight);
- the mixed form against the FP64 oracle: within 1e-4, the reference's own bar for its kernels against NumPy
  (tests/test_radiation.py:164);
- at the full workload size (40,962 columns x 7 layers, 256 longwave and 224 shortwave g-points) every 97th column
  against the oracle, the clear-sky shortwave shares closing to one everywhere, and a second run bit-identical.
"""
from pathlib import Path

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

GOLD = Path(__file__).resolve().parent / 'golden' / 'ktables'


def _np(t):
    return t.detach().cpu().numpy().copy()


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64), device='cuda')


def case(N, L, seed):
    """Seeded columns (states, unit positions) and their column parameters."""
    from insilica.atmosphere import par_array
    from insilica.ktables import column_state
    rng = np.random.default_rng(seed)
    pos = rng.normal(size=(N, 3))
    pos /= np.linalg.norm(pos, axis=1)[:, None]
    c = column_state(pos, layers=L, seed=seed)
    stars = list(np.linspace(500.0, 300.0, L - 1))
    par = par_array(L, dict(edge_k=2.0 if L >= 5 else 1.0, theta_stars=stars, lw_refl=1.0 if seed % 2 else 0.0))
    return c, pos, par


def run_gpu(c, pos, par, L, lw_tables, sw_tables, precision, clouds=True, mode=0, tnow=3.0e6, sub=None):
    """lw_setup (or the given sub-levels), lw_column and sw_column through the product's classes."""
    from insilica.radiation import Longwave, Shortwave
    N = c['mu'].shape[1]
    lw = Longwave(N, L, par, tables=lw_tables, precision=precision)
    sw = Shortwave(N, L, par, lw, tables=sw_tables, ice_re=30e-6, precision=precision,
                   cloud_ssa=sw_tables.get('cloud_ssa'), band_top=sw_tables.get('band_top'))
    co = _dev(c['cloudo']) if clouds else None
    mu, th, q, Ts, alb = (_dev(c[k]) for k in ('mu', 'theta', 'q', 'Ts', 'alb'))
    p = _dev(pos)
    t = _dev([tnow])
    if sub is None:
        lw.setup(mu, th, q, co)
    else:
        lw.sub.copy_(torch.as_tensor(np.ascontiguousarray(sub, dtype=np.float32), device='cuda'))
    lw.column(Ts)
    sw(mode, t, 3600.0, p, alb, co)
    torch.cuda.synchronize()
    return _np(lw.sub), _np(lw.radf), _np(sw.swf)


def run_oracle(c, pos, par, L, lw_tables, sw_tables, sub, clouds=True, mode=0, tnow=3.0e6, cols=None):
    from insilica.radiation import ice_optics
    from oracle import radiation as orad
    cols = np.arange(c['mu'].shape[1]) if cols is None else cols
    n = len(cols)
    lwt = orad.LwTables(lw_tables)
    ng = np.asarray(sw_tables['ng'], int)
    io = ice_optics(30.0, sw_tables.get('band_top') or (2600, 4000, 5250, 7700, 9350, 12850, 16000, 29000, 38000,
                                                        50000))
    swt = orad.SwTables(sw_tables, cssa_i=np.repeat([x[0] for x in io], ng), g_i=np.repeat([x[1] for x in io], ng))
    co = c['cloudo'][:, cols] if clouds else None
    osub = sub[:, cols]
    radf = orad.lw_column(n, L, par, lwt, osub, c['Ts'][cols])
    swf = orad.sw_column(n, L, par, swt, osub, c['alb'][cols], mode=mode, tnow=tnow, interval=3600.0,
                         pos=pos[cols], cloudo=co)
    return radf, swf


def lw_scale(radf, L):
    """max(1, the surface's downward flux) per column (the reference's kernel-test scale)."""
    return np.maximum(1.0, radf[2 * (L + 1) - 1])


@pytest.fixture(scope='module')
def ref_tables():
    return dict(np.load(GOLD / 'lw_ktables.npz')), dict(np.load(GOLD / 'sw_ktables.npz'))


@pytest.mark.parametrize('L,seed', [(3, 1), (7, 2)])
def test_fp64_matches_oracle(ref_tables, L, seed):
    from oracle import radiation as orad
    lwk, swk = ref_tables
    N = 256
    print(f'case: radiation FP64 N={N} L={L} seed={seed} reference tables', flush=True)
    c, pos, par = case(N, L, seed)
    sub, radf, swf = run_gpu(c, pos, par, L, lwk, swk, 'double')
    osub = orad.lw_setup(N, L, par, orad.LwTables(lwk), c['mu'], c['theta'], c['q'], c['cloudo'])
    rel = np.abs(sub.astype(float) - osub) / np.maximum(np.abs(osub.astype(float)), 1e-30)
    assert rel.max() <= 2.5e-7, rel.max()
    ora, osw = run_oracle(c, pos, par, L, lwk, swk, sub)
    e_lw = np.max(np.abs(radf - ora) / lw_scale(ora, L))
    e_sw = np.max(np.abs(swf - osw))
    print(f'lw {e_lw:.2e} sw {e_sw:.2e} sub-levels {rel.max():.2e}', flush=True)
    assert e_lw <= 1e-8 and e_sw <= 1e-8


@pytest.mark.parametrize('L,seed', [(3, 3), (7, 4)])
def test_mixed_within_reference_bar(ref_tables, L, seed):
    """The mixed form's sub-levels within 2e-5 of the oracle's (the cloud in the same sub-level), its column passes on
    the oracle's sub-levels and the whole pipeline within 1e-4."""
    from oracle import radiation as orad
    lwk, swk = ref_tables
    N = 256
    print(f'case: radiation mixed N={N} L={L} seed={seed}', flush=True)
    c, pos, par = case(N, L, seed)
    sub, radf, swf = run_gpu(c, pos, par, L, lwk, swk, 'mixed')
    osub = orad.lw_setup(N, L, par, orad.LwTables(lwk), c['mu'], c['theta'], c['q'], c['cloudo'])
    sm, so = sub.reshape(4 * L, 15, N), osub.reshape(4 * L, 15, N)
    # a layer's cloud goes to the sub-level where its vapor's running share reaches one half: a share within rounding
    # of one half can tip either way in float arithmetic; such columns (at most 1%) are left out of the comparison
    moved = ((sm[:, 10] > 0) != (so[:, 10] > 0)).any(0)
    assert moved.mean() <= 0.01, f'cloud sub-levels differ in {moved.sum()} columns'
    ok = ~moved
    sm, so = sm[..., ok], so[..., ok]
    e_sub = np.max(np.abs(sm.astype(float) - so) / np.maximum(np.abs(so.astype(float)), 1e-30))
    ora, osw = run_oracle(c, pos, par, L, lwk, swk, osub)
    e_lw = np.max(np.abs(radf - ora)[:, ok] / lw_scale(ora, L)[ok])
    e_sw = np.max(np.abs(swf - osw)[:, ok])
    _, radf2, swf2 = run_gpu(c, pos, par, L, lwk, swk, 'mixed', sub=osub)
    e_lw2 = np.max(np.abs(radf2 - ora) / lw_scale(ora, L))
    e_sw2 = np.max(np.abs(swf2 - osw))
    print(f'mixed: cloud moved in {moved.sum()} columns; sub-levels {e_sub:.2e}; pipeline lw {e_lw:.2e} sw {e_sw:.2e}; on the oracle sub-levels lw '
          f'{e_lw2:.2e} sw {e_sw2:.2e}', flush=True)
    assert e_sub <= 2e-5 and max(e_lw, e_sw, e_lw2, e_sw2) <= 1e-4


def test_full_workload_size():
    """40,962 columns x 7 layers with 256 / 224 g-points (synthetic tables): sampled columns against the oracle,
    the clear-sky shares closing to one everywhere, both forms, and a repeat bit-identical."""
    from insilica import grid as gm
    from insilica.ktables import synthetic_lw, synthetic_sw
    from oracle import radiation as orad
    g = gm.get(6)
    L, lwk, swk = 7, synthetic_lw(), synthetic_sw()
    c, _, par = case(g.N, L, 5)
    pos = np.ascontiguousarray(g.pos, dtype=np.float64)
    cols = np.arange(0, g.N, 97)
    for prec, tol in (('double', 1e-8), ('mixed', 1e-4)):
        print(f'case: radiation full size {prec}', flush=True)
        sub, radf, swf = run_gpu(c, pos, par, L, lwk, swk, prec)
        ora, osw = run_oracle(c, pos, par, L, lwk, swk, sub, cols=cols)
        e_lw = np.max(np.abs(radf[:, cols] - ora) / lw_scale(ora, L))
        e_sw = np.max(np.abs(swf[:, cols] - osw))
        print(f'{prec}: lw {e_lw:.2e} sw {e_sw:.2e}', flush=True)
        assert e_lw <= tol and e_sw <= tol
        sub2, radf2, swf2 = run_gpu(c, pos, par, L, lwk, swk, prec)
        assert np.array_equal(radf, radf2) and np.array_equal(swf, swf2) and np.array_equal(sub, sub2)
        _, _, swc = run_gpu(c, pos, par, L, lwk, swk, prec, clouds=False)
        assert np.allclose(swc[:L].sum(0) + swc[L] + swc[L + 1], 1.0, atol=2e-5)


@pytest.mark.parametrize('N,L,lwb,swb', [(1, 2, 4, 4), (257, 3, 5, 3), (6145, 4, 1, 1), (67, 6, 15, 13), (65, 8, 16, 16)])
def test_columns_at_the_edges(N, L, lwb, swb):
    """One column, an odd number of them shared out two to a block, one and several waves of g-points (a last one part
    full, a full block), the layer counts whose sums go through LDS in two parts or whose albedos wait there: both forms
    against the oracle on the same sub-levels, at the bars above."""
    from insilica.ktables import synthetic_lw, synthetic_sw
    print(f'case: radiation N={N} L={L} {16 * lwb} / {16 * swb} g-points', flush=True)
    c, pos, par = case(N, L, 20 + L)
    lwk, swk = synthetic_lw(bands=lwb, seed=L), synthetic_sw(bands=swb, seed=L + 1)
    for prec, tol in (('double', 1e-8), ('mixed', 1e-4)):
        sub, radf, swf = run_gpu(c, pos, par, L, lwk, swk, prec)
        ora, osw = run_oracle(c, pos, par, L, lwk, swk, sub)
        e_lw = np.max(np.abs(radf - ora) / lw_scale(ora, L))
        e_sw = np.max(np.abs(swf - osw))
        print(f'{prec}: lw {e_lw:.2e} sw {e_sw:.2e}', flush=True)
        assert e_lw <= tol and e_sw <= tol


@pytest.mark.parametrize('precision', ['double', 'mixed'])
@pytest.mark.parametrize('L', [2, 7])
def test_longwave_of_constant_tables(L, precision):
    """Where ln k is the same at every pressure and temperature, a gas's depth does not depend on where in the tables a
    sub-level lies: columns that differ in that alone have the same fluxes to the bit. (ln k interpolated by the corners'
    weights takes the weights' rounding times all of ln k with it and fails here in the mixed form.)"""
    from insilica.ktables import synthetic_lw
    from insilica.radiation import Longwave
    N = 64
    print(f'case: longwave, constant tables, L={L} {precision}', flush=True)
    c, _, par = case(N, L, 31)
    lwk = synthetic_lw(bands=4, seed=L)
    lwk['logk'] = np.broadcast_to(np.median(lwk['logk'], axis=(1, 2), keepdims=True), lwk['logk'].shape).copy()
    lw = Longwave(N, L, par, tables=lwk, precision=precision)
    mu, th, q, co = (_dev(np.repeat(c[k][:, :1], N, 1)) for k in ('mu', 'theta', 'q', 'cloudo'))
    lw.setup(mu, th, q, co)
    sub = lw.sub.view(4 * L, 15, N)
    rng = np.random.default_rng(L)
    for row, size in ((2, lwk['logk'].shape[1]), (3, lwk['logk'].shape[2])):
        sub[:, row] = torch.as_tensor(rng.uniform(0, size - 1.01, (4 * L, N)).astype(np.float32), device='cuda')
    lw.column(_dev(np.full(N, c['Ts'][0])))
    torch.cuda.synchronize()
    radf = _np(lw.radf)
    assert np.all(np.isfinite(radf)) and np.array_equal(radf, np.repeat(radf[:, :1], N, 1))


@pytest.mark.parametrize('precision', ['double', 'mixed'])
@pytest.mark.parametrize('ray,haze', [(1e-41, 0.0), (0.0, 1e-41), (1e-41, 1e-41)])
def test_shortwave_of_vanishing_depths(ray, haze, precision):
    """Gases that absorb nothing, and molecules and haze whose depths are denormal in the mixed form: the light passes as
    if they were not there (nothing is divided by a denormal depth)."""
    from insilica.ktables import synthetic_lw, synthetic_sw
    from insilica.radiation import Longwave, Shortwave
    N, L = 64, 3
    print(f'case: shortwave, vanishing depths, ray {ray} haze {haze} {precision}', flush=True)
    c, pos, par = case(N, L, 33)
    swk = synthetic_sw(bands=4, seed=2)
    swk['logk'] = np.full_like(swk['logk'], -1000.0)
    out = []
    for r, h in ((ray, haze), (0.0, 0.0)):
        lw = Longwave(N, L, par, tables=synthetic_lw(bands=4, seed=1), precision=precision)
        swk['haze_par'] = np.concatenate([[h], swk['haze_par'][1:]])
        sw = Shortwave(N, L, par, lw, tables=swk, air=dict(ray=r), precision=precision)
        lw.setup(*(_dev(c[k]) for k in ('mu', 'theta', 'q')), None)
        sw(0, _dev([3.0e6]), 3600.0, _dev(pos), _dev(c['alb']), None)
        torch.cuda.synchronize()
        out.append(_np(sw.swf))
    assert np.all(np.isfinite(out[0])) and np.max(np.abs(out[0] - out[1])) <= 1e-6


@pytest.mark.parametrize('precision,bar', [('double', 1e-8), ('mixed', 1e-4)])
@pytest.mark.parametrize('L', [3, 7])
def test_options_of_the_column_passes(L, precision, bar):
    """The branches of the column passes that the other tests leave out: absorption by collisions (cia) in both, another
    air's Rayleigh scattering and oxygen, a fixed mean cosine (mode 1), clouds with the drops' optics for ice, a clear sky
    without haze, g-points that do not fill the last eight: on the same sub-levels, against the oracle."""
    from insilica.ktables import synthetic_lw, synthetic_sw
    from insilica.radiation import Longwave, Shortwave
    from oracle import radiation as orad
    N = 100
    print(f'case: radiation options L={L} {precision}', flush=True)
    c, pos, par = case(N, L, 41 + L)
    rng = np.random.default_rng(L)
    lwk, swk = synthetic_lw(bands=7, g_per_band=11, seed=1), synthetic_sw(bands=5, g_per_band=13, seed=2)
    air = dict(cia=1, ray=0.7, o2=0.1)
    mu, th, q, co = (_dev(c[k]) for k in ('mu', 'theta', 'q', 'cloudo'))
    for t in (lwk, swk):
        t['cia'] = np.zeros((t['logk'].shape[2], t['logk'].shape[3]))
    lw = Longwave(N, L, par, tables=lwk, precision=precision, air=air)
    lw.setup(mu, th, q, co)
    amount = _np(lw.sub).reshape(4 * L, 15, N)[:, 14]
    assert amount.min() > 0
    for t in (lwk, swk):
        t['cia'] = rng.uniform(0.05, 2.0, t['cia'].shape) / np.median(amount)
    lw = Longwave(N, L, par, tables=lwk, precision=precision, air=air)
    lw(mu, th, q, co, _dev(c['Ts']))
    sub = _np(lw.sub)
    ora = orad.lw_column(N, L, par, orad.LwTables(lwk, cia=lwk['cia']), sub, c['Ts'])
    none = orad.lw_column(N, L, par, orad.LwTables(lwk), sub, c['Ts'])
    e_lw = np.max(np.abs(_np(lw.radf) - ora) / lw_scale(ora, L))
    assert np.max(np.abs(none - ora) / lw_scale(ora, L)) > 0.01         # (the option matters here)
    for mode, clouds, haze in ((0, True, True), (1, True, True), (1, False, False)):
        k = dict(swk) if haze else dict(swk, haze_par=np.concatenate([[0.0], swk['haze_par'][1:]]))
        sw = Shortwave(N, L, par, lw, tables=k, precision=precision, air=air)
        sw(mode, _dev([3.0e6]), 3600.0, _dev(pos), _dev(c['alb']), co if clouds else None)
        osw = orad.sw_column(N, L, par, orad.SwTables(k, cia=k['cia']), sub, c['alb'], mode=mode, tnow=3.0e6,
                             interval=3600.0, pos=pos, cloudo=c['cloudo'] if clouds else None, air=air)
        e_sw = np.max(np.abs(_np(sw.swf) - osw))
        print(f'mode {mode} clouds {clouds} haze {haze}: lw {e_lw:.2e} sw {e_sw:.2e}', flush=True)
        assert e_lw <= bar and e_sw <= bar
