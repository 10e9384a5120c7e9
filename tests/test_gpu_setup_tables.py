"""The host set-up on meshes of one thread's work and of several: the element
neighbours and faces of bl_init_mesh against a plain search, and a run on the
tiles (whose tables several threads build) against the run without them, bit
for bit."""
import numpy as np
import pytest

from bookleaf_f90_amd import problem as P
from tests.helpers import diff_fields
from tests.test_gpu_graph import compared
from tests.test_gpu_remap_tiles import _renumbered, _stirred

pytestmark = pytest.mark.gpu


def _neighbours(p):
    """ielel and ielfc of a conforming mesh: the other element of each face's
    two nodes; a boundary face names its own element and the opposite face."""
    nd = p.ielnd.reshape(-1, 4)
    where = {}
    for e, q in enumerate(nd.tolist()):
        for f in range(4):
            where.setdefault(frozenset((q[f], q[(f + 1) & 3])), []).append((e, f))
    el, fc = np.zeros_like(nd), np.zeros_like(nd)
    for pair in where.values():
        if len(pair) == 2:
            (e, f), (b, g) = pair
            el[e, f], fc[e, f], el[b, g], fc[b, g] = b + 1, g + 1, e + 1, f + 1
        else:
            (e, f), = pair
            el[e, f], fc[e, f] = e + 1, ((f + 2) & 3) + 1
    return el.ravel(), fc.ravel()


@pytest.mark.parametrize("nx,ny,turn", [(2, 1, 0), (19, 1, 1), (37, 29, 2), (190, 61, 3),
                                        (300, 170, 1), (430, 250, 2)])
def test_tables(nx, ny, turn):
    from bookleaf_f90_amd.device import BookLeaf
    p = _renumbered(_stirred(P.sod(nx=nx, ny=ny, height=ny / nx, eulerian=True,
                                   dt_initial=1e-5), u=0.01), 4, turn)
    print("tables", nx, ny, flush=True)
    tiled, other = BookLeaf(p), BookLeaf(p)
    el, fc = _neighbours(p)
    assert np.array_equal(tiled.get("ielel").ravel(), el)
    assert np.array_equal(tiled.get("ielfc").ravel(), fc)
    other.set_tiling(False)
    for g in (tiled, other):
        g.run(5, runner="run_graph")
    assert tiled.get_tiling()[0] and not other.get_tiling()[0]
    assert diff_fields(tiled.state(), other.state(), compared(p)) == []


def test_ensemble_tables():
    from bookleaf_f90_amd.device import Ensemble
    params = P.ensemble_params(5, seed=3, nmin=90, nmax=150)
    print("ensemble tables", [q["nx"] for q in params], flush=True)
    tiled, other = Ensemble(params), Ensemble(params)
    other.set_tiling(False)
    for a, b in zip(tiled.run(8), other.run(8)):
        assert np.array_equal(a, b)
    for f in ("elenergy", "eldensity", "ndx", "ndy", "ndu", "ndv"):
        assert np.array_equal(tiled.get(f), other.get(f))
