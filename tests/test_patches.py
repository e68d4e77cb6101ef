"""The patch tables, checked on the host against the mesh: those that kernels read -- the transport's edge lists
(fast_patches, transport_patches) and the fast sub-steps' rings (grid.rings) -- and those that the mesh struct still takes
though no kernel reads them now: fast_patches' halos and slots (one fused sub-step needs Phi* on both cells of every edge it
steps) and fast_patches2 (two fused sub-steps need the first's winds on every edge of the second's cells, and its Phi* on
both cells of each of those edges). A wrong slot would read another cell's value; these checks name every slot's cell and
edge."""
import numpy as np
import pytest

from insilica import grid as gridmod
from insilica.gpu import fast_patches, fast_patches2, transport_patches


def unpack(v):
    return v & 0xffff, v >> 16


@pytest.mark.parametrize('n,pc', [(3, 64), (4, 64), (4, 48), (5, 96)])
def test_single_step_tables(n, pc):
    g = gridmod.get(n)
    t = fast_patches(g, pc)
    N, E = g.N, g.E
    eI, eJ = np.asarray(g.eI), np.asarray(g.eJ)
    assert t['npatch'] == (N + pc - 1) // pc
    assert np.array_equal(np.sort(t['pe_edge']), np.arange(E))           # every edge stepped by exactly one patch
    for b in range(t['npatch']):
        c0, nown = b * pc, min(pc, N - b * pc)
        halo = t['ph_cell'][t['ph_off'][b]:t['ph_off'][b + 1]]
        edges = t['pe_edge'][t['pe_off'][b]:t['pe_off'][b + 1]]
        sI, sJ = unpack(t['pe_slot'][t['pe_off'][b]:t['pe_off'][b + 1]])
        hx = np.concatenate([halo, [-1]])                                   # (a patch may have no halo)
        cell_of = lambda s: np.where(s < pc, c0 + s, hx[np.clip(s - pc, 0, len(hx) - 1)])
        assert np.all(eI[edges] // pc == b)                                 # its edges' first cells are its own
        assert np.all(sI < nown) and np.all(sJ < pc + len(halo)) and np.all((sJ < nown) | (sJ >= pc))
        assert np.array_equal(cell_of(sI), eI[edges]) and np.array_equal(cell_of(sJ), eJ[edges])
        # the halo is exactly the outside cells those edges reach, sorted
        want = np.unique(eJ[edges][eJ[edges] // pc != b])
        assert np.array_equal(halo, want)
        assert pc + len(halo) <= t['pslots']


@pytest.mark.parametrize('n', [3, 4])
def test_two_step_tables(n):
    g = gridmod.get(n)
    t = fast_patches(g, 64)
    t2 = fast_patches2(g, t)
    N, pc = g.N, 64
    eI, eJ, ce = np.asarray(g.eI), np.asarray(g.eJ), np.asarray(g.cellEdge)
    for b in range(t['npatch']):
        c0, nown = b * pc, min(pc, N - b * pc)
        h1 = t['ph_cell'][t['ph_off'][b]:t['ph_off'][b + 1]]
        h2 = t2['ph2_cell'][t2['ph2_off'][b]:t2['ph2_off'][b + 1]]
        own_e = t['pe_edge'][t['pe_off'][b]:t['pe_off'][b + 1]]
        x_e = t2['px_edge'][t2['px_off'][b]:t2['px_off'][b + 1]]
        edges = np.concatenate([own_e, x_e])                               # edge slot -> edge
        slots_cells = np.concatenate([np.arange(c0, c0 + nown), np.full(pc - nown, -1), h1, h2])
        # second sub-step's cells (patch, then halo): each of its edges has a slot holding that edge
        c1 = np.concatenate([np.arange(c0, c0 + nown), h1])
        es = t2['pc_eslot'][3 * t2['pc_off'][b]:3 * t2['pc_off'][b + 1]].reshape(-1, 3)
        es6 = np.stack([es & 0xffff, es >> 16], axis=2).reshape(-1, 6)
        assert len(es6) == len(c1)
        for ci, c in enumerate(c1):
            for m in range(6):
                if ce[c, m] < 0:
                    assert es6[ci, m] == 0xffff
                else:
                    assert edges[es6[ci, m]] == ce[c, m]
        # the first sub-step's winds on the other edges read Phi* at slots naming their cells
        sI, sJ = unpack(t2['px_slot'][t2['px_off'][b]:t2['px_off'][b + 1]])
        assert np.array_equal(slots_cells[sI], eI[x_e]) and np.array_equal(slots_cells[sJ], eJ[x_e])
        assert pc + len(h1) + len(h2) <= t2['pslots2'] and len(edges) <= t2['pedges2']
        assert len(np.intersect1d(h2, c1)) == 0 and len(np.unique(h2)) == len(h2)


@pytest.mark.parametrize('n', [3, 4])
def test_transport_tables(n):
    """The fused transport stage's tables: a patch's edge list is every edge touching its cells, once, its own edges
    first in pe order; each cell's slots name its cellEdgeAsc edges in its own patch's list, odd where it is the
    edge's first cell; every incoming edge's first cell lies outside the patch and its second inside."""
    g = gridmod.get(n)
    t = fast_patches(g, 64)
    r = transport_patches(g, t)
    N, pc = g.N, 64
    eI, eJ, asc = np.asarray(g.eI), np.asarray(g.eJ), np.asarray(g.cellEdgeAsc)
    for b in range(t['npatch']):
        cells = np.arange(b * pc, min((b + 1) * pc, N))
        own = t['pe_edge'][t['pe_off'][b]:t['pe_off'][b + 1]]
        inc = r['pi_edge'][r['pi_off'][b]:r['pi_off'][b + 1]]
        assert np.all(eI[inc] // pc != b) and np.all(eJ[inc] // pc == b) and np.all(np.diff(inc) > 0)
        edges = np.concatenate([own, inc])
        touching = np.unique(asc[cells][asc[cells] >= 0])
        assert np.array_equal(np.sort(edges), touching)
        tc = r['tc_slot'][cells]
        m = asc[cells] >= 0
        assert np.array_equal(edges[tc[m] >> 1], asc[cells][m])
        assert np.array_equal((tc[m] & 1) == 1, eI[asc[cells][m]] == np.repeat(cells, 6).reshape(-1, 6)[m])
        assert len(edges) <= r['ptedges']
    assert np.all((r['tc_slot'] < 0) == (asc < 0))


@pytest.mark.parametrize('n,pc,union', [(3, 64, False), (4, 64, False), (4, 50, False), (3, 64, True)])
def test_ring_tables(n, pc, union):
    """The ring patches: every cell and every edge of the mesh is owned once; each ring is exactly the neighbours of what
    is inside it, its edge list exactly the edges they touch; every slot names its cell's edge with its sign, every
    edge's places name its cells, as far as the kernels read them; a union's patches stay inside its parts."""
    from insilica.batch import UnionGrid
    from insilica.grid import rings
    K = 5
    g = UnionGrid([gridmod.get(n), gridmod.get(n - 1), gridmod.get(n)]) if union else gridmod.get(n)
    t = rings(g, K, pc)
    eI, eJ, ce, sg = (np.asarray(getattr(g, k)).astype(np.int64) for k in ('eI', 'eJ', 'cellEdge', 'cellSign'))
    cells_seen, edges_seen = [], []
    for b, h in enumerate(t['head']):
        nc, ne = h[3:4 + K], h[4 + K:5 + 2 * K]
        C, G = t['cell'][h[0]:h[0] + nc[K]], t['edge'][h[1]:h[1] + ne[K]]
        assert len(np.unique(C)) == len(C) and len(np.unique(G)) == len(G) and nc[0] <= pc
        assert h[2] <= t['owned'] and np.all(nc <= t['cells'][:K + 1]) and np.all(ne <= t['edges'][:K + 1])
        assert np.array_equal(np.sort(G[:h[2]]), np.flatnonzero(np.isin(eI, C[:nc[0]])))
        for r in range(K + 1):
            e = ce[C[:nc[r]]]
            assert np.array_equal(np.sort(G[:ne[r]]), np.unique(e[e >= 0]))
            if r:
                inner = G[:ne[r - 1]]
                assert np.array_equal(np.sort(C[:nc[r]]), np.unique(np.concatenate([eI[inner], eJ[inner]])))
        s = t['slot'][3 * h[0]:3 * (h[0] + nc[K])].reshape(-1, 3).astype(np.int64) & 0xffffffff
        s6 = np.stack([s & 0xffff, s >> 16], axis=2).reshape(-1, 6)
        has = ce[C] >= 0
        assert np.array_equal((s6 & 0x7fff) != 0x7fff, has)
        assert np.array_equal(G[(s6 & 0x7fff)[has]], ce[C][has])
        assert np.array_equal((s6[has] & 0x8000) != 0, sg[C][has] < 0)
        read = slice(h[1], h[1] + ne[K - 1])
        first, second = unpack(t['ecell'][read])
        assert np.array_equal(C[first], eI[G[:ne[K - 1]]]) and np.array_equal(C[second], eJ[G[:ne[K - 1]]])
        if union:
            assert len(np.unique(g.world_cell[C])) == 1
        cells_seen.append(C[:nc[0]])
        edges_seen.append(G[:h[2]])
    assert np.array_equal(np.sort(np.concatenate(cells_seen)), np.arange(g.N))
    assert np.array_equal(np.sort(np.concatenate(edges_seen)), np.arange(g.E))


def test_ring_tables_refused():
    """A mesh with an edge lacking a cell, or whose positions cannot be ordered, has no rings (and steps without them)."""
    import types
    from insilica.grid import rings
    g = gridmod.get(3)

    def like(**change):
        m = types.SimpleNamespace(N=g.N, E=g.E, pos=g.pos, cellEdge=g.cellEdge, cellSign=g.cellSign, eI=g.eI.copy(), eJ=g.eJ)
        for k, v in change.items():
            setattr(m, k, v)
        return m
    assert rings(like(), 4) is not None
    pos = np.array(g.pos)
    pos[7, 1] = np.nan
    lacking = np.array(g.eJ)
    lacking[11] = -1
    assert rings(like(pos=pos), 4) is None and rings(like(pos=None), 4) is None and rings(like(eJ=lacking), 4) is None
