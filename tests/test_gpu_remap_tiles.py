"""The ALE step on the tiling (the tile step, k_remap_faces, k_remap_tile)
against the three-kernel step with the five remap kernels and against the
oracle, bit for bit: meshes of less than one tile, one tile and a few with
remainders, elements and nodes numbered at random and elements starting from
any corner (the summation orders and neighbour faces of the tables), mixed
cells, node relaxation, an ALE time window (steps without a remap between
steps with one), run calls of odd and even lengths (the two corner-mass
arrays, the at-rest bytes), switches between the two forms and a negative
volume in the step and in the remap."""
import numpy as np
import pytest

from bookleaf_f90_amd import abi
from bookleaf_f90_amd import problem as P
from tests.helpers import diff_fields
from tests.test_gpu_graph import compared

pytestmark = pytest.mark.gpu


def _renumbered(p, seed, turn):
    """The same problem with elements and nodes in another order and every
    element starting from corner 1 + turn."""
    rng = np.random.default_rng(seed)
    pe, pn = rng.permutation(p.nel), rng.permutation(p.nnd)
    new = np.empty(p.nnd, np.int64)
    new[pn] = np.arange(p.nnd)
    q = np.roll(p.ielnd.reshape(-1, 4)[pe], -turn, axis=1)
    p.ielnd = (new[q - 1] + 1).astype(np.int32).ravel()
    for k in ("ndx", "ndy", "indtype", "ndu", "ndv"):
        setattr(p, k, getattr(p, k)[pn].copy())
    for k in ("ielreg", "ielmat", "density", "energy"):
        setattr(p, k, getattr(p, k)[pe].copy())
    return p


def _stirred(p, seed=3, u=0.2):
    """Random interior velocities: every element moves, every face flux has
    both signs."""
    rng = np.random.default_rng(seed)
    inner = p.indtype > 0
    p.ndu[inner] = rng.uniform(-u, u, inner.sum())
    p.ndv[inner] = rng.uniform(-u, u, inner.sum())
    return p


def _eul(p):
    p.config["zeul"] = 1
    p.__post_init__()
    return p


def _window(p, lo, hi):
    p.config.update(mintime=lo, maxtime=hi)
    return p


CASES = {
    "2x2": lambda: _stirred(P.sod(nx=2, ny=2, height=1.0, eulerian=True, dt_initial=1e-3)),
    "5x1": lambda: _stirred(P.sod(nx=5, ny=1, height=0.2, eulerian=True, dt_initial=1e-3)),
    "13x13": lambda: _stirred(P.sod(nx=13, ny=13, height=1.0, eulerian=True, dt_initial=1e-3)),
    "181x1": lambda: _stirred(P.sod(nx=181, ny=1, height=0.006, eulerian=True)),
    "37x29_turned": lambda: _renumbered(
        _stirred(P.sod(nx=37, ny=29, height=0.8, eulerian=True, dt_initial=1e-3)), 5, 1),
    "40x31_numbered": lambda: _renumbered(
        _stirred(P.sod2mat(nx=40, ny=31)), 6, 2),
    "sedov_33": lambda: _eul(P.sedov(n=33, kappa=0.01)),
    "mixed_48x20": lambda: _stirred(P.sod2mat_mixed(nx=48, ny=20), u=0.05),
    "mixed_window": lambda: _window(P.sod2mat_mixed(nx=32, ny=12, dt_initial=1e-4), 4.0e-4, 1.1e-3),
    "window": lambda: _window(
        _stirred(P.sod(nx=30, ny=17, height=0.5, eulerian=True, dt_initial=1e-4)), 3.0e-4, 9.0e-4),
    "relax_equi": lambda: P.with_relaxation(
        _stirred(P.sod2mat_mixed(nx=40, ny=24, eulerian=False, jitter=0.1), u=0.05),
        abi.RELAX_EQUI, nsweep=2, om=0.5),
    "relax_lin1": lambda: P.with_relaxation(
        _stirred(P.sod(nx=31, ny=23, height=0.7)), abi.RELAX_LIN1, nsweep=1, om=0.25),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_tiled_remap_matches_other_form_and_oracle(name, oracle_lib):
    from bookleaf_f90_amd.device import BookLeaf
    from oracle.pyoracle import Oracle
    p = CASES[name]()
    print("case", name, "nel", p.nel, flush=True)
    tiled, other, switched = BookLeaf(p), BookLeaf(p), BookLeaf(p)
    other.set_tiling(False)
    o = Oracle(p)
    for k, n in enumerate((3, 1, 8, 5)):
        switched.set_tiling(k % 2 == 0)
        h = [g.run(n, runner="run_graph") for g in (tiled, other, switched)]
        ho = o.run(n)
        for a in h:
            for x, y in zip(a, ho):
                assert np.array_equal(x, y)
        for g in (tiled, other, switched):
            assert diff_fields(g.state(), o.state(), compared(p)) == []
    assert tiled.get_tiling()[0] and not other.get_tiling()[0]
    # the per-driver entry points go on from the tiled state
    tiled.step()
    o.step()
    assert diff_fields(tiled.state(), o.state(), compared(p)) == []


@pytest.mark.parametrize("where", ["predictor", "remap"])
def test_negative_volume_stops_both_forms_alike(where):
    """An element inverted in the predictor, or by the relaxation's moved
    mesh: the same error, element, step count and fields in both forms."""
    from bookleaf_f90_amd.device import BookLeaf, BookLeafError
    if where == "predictor":
        p = P.sod(nx=20, ny=9, height=0.5, eulerian=True, dt_initial=1.0e-2)
    else:
        # one sweep with om = 3 carries nodes far past their stencil
        p = P.with_relaxation(P.sod(nx=20, ny=9, height=0.5), abi.RELAX_LIN1, nsweep=1, om=3.0)
        rng = np.random.default_rng(1)
        inner = p.indtype > 0
        p.ndx[inner] += rng.uniform(-0.02, 0.02, inner.sum())
        p.ndy[inner] += rng.uniform(-0.02, 0.02, inner.sum())
    p.config.update(cvisc1=0.0, cvisc2=0.0, div_sf=1.0e30)
    seen = []
    for tiles in (True, False):
        g = BookLeaf(p)
        g.set_tiling(tiles)
        if where == "predictor":
            u = g.get("ndu")
            u[p.nnd // 2] += 100.0
            g.set("ndu", u)
        with pytest.raises(BookLeafError) as e:
            g.run(6, runner="run_graph")
        assert "negative volume" in str(e.value)
        seen.append((e.value.ierr, g.ts.nstep, g.ts.time, g.state()))
    assert seen[0][:3] == seen[1][:3]
    names = ["ndx", "ndy", "ndu", "ndv", "eldensity", "elenergy", "elpressure", "elcs2",
             "elmass", "cnmass", "cnviscx", "cnviscy", "elvisc"]
    assert diff_fields(seen[0][3], seen[1][3], names) == []


@pytest.mark.parametrize("mixed", [False, True])
def test_summation_orders_of_the_sorted_elements(mixed, oracle_lib):
    """ielsort1 and ielsort2 two permutations: a node's remap sums run in the
    order of ielsort2, then in element order, and the two differ."""
    from bookleaf_f90_amd.device import BookLeaf
    from oracle.pyoracle import Oracle
    p = _stirred((P.sod2mat_mixed if mixed else P.sod2mat)(nx=33, ny=18), u=0.05)
    if not mixed:  # (the components' lists name elements)
        p = _renumbered(p, 7, 1)
    print("sorted", p.nel, mixed, flush=True)
    rng = np.random.default_rng(8)
    sorts = {k: (rng.permutation(p.nel) + 1).astype(np.int32) for k in ("ielsort1", "ielsort2")}
    tiled, other, o, plain = BookLeaf(p), BookLeaf(p), Oracle(p), Oracle(p)
    other.set_tiling(False)
    for s in (tiled, other, o):
        for k, v in sorts.items():
            s.set(k, v)
    for s in (tiled, other):
        assert s.lib.bl_build_maps(s.h) == 0
    for n in (3, 6):
        ho = o.run(n)
        for s in (tiled, other):
            for x, y in zip(s.run(n, runner="run_graph"), ho):
                assert np.array_equal(x, y)
            assert diff_fields(s.state(), o.state(), compared(p)) == []
    assert tiled.get_tiling()[0] and not other.get_tiling()[0]
    plain.run(9)
    assert not np.array_equal(plain.get("ndu"), o.get("ndu"))  # the order shows


@pytest.mark.parametrize("kind", ["boundary_face", "wrapped"])
def test_meshes_the_tiled_remap_refuses(kind, oracle_lib):
    """A boundary face whose ielfc is not the opposite face: the remap's grid
    form runs.  Neighbours across the ends of the tube, which share no nodes
    (outside a tile's entries): the drivers run.  Both match the oracle."""
    from bookleaf_f90_amd.device import BookLeaf
    from oracle.pyoracle import Oracle
    nx, ny = 24, 9
    p = _stirred(P.sod(nx=nx, ny=ny, height=0.4, eulerian=True, dt_initial=1e-3))
    print("refused", kind, flush=True)
    g, o = BookLeaf(p), Oracle(p)
    g.run(2, runner="run_graph")
    o.run(2)
    assert g.get_tiling()[0]
    el, fc = g.get("ielel"), g.get("ielfc")
    x = g.get("ndx")[p.ielnd.reshape(-1, 4) - 1].mean(axis=1)
    y = g.get("ndy")[p.ielnd.reshape(-1, 4) - 1].mean(axis=1)
    own = np.arange(p.nel).repeat(4) + 1 == el[:4 * p.nel]
    if kind == "boundary_face":
        k = np.nonzero(own)[0][7]
        fc[k] = k % 4 + 1
    else:
        rows = np.argsort(y, kind="stable").reshape(ny, nx)
        for row in rows:
            a, b = row[np.argmin(x[row])], row[np.argmax(x[row])]
            # the boundary face towards the end of the tube: opposite the
            # neighbour inside the row
            f = [i for i in range(4) if el[4 * a + i] == a + 1 and
                 el[4 * a + (i + 2) % 4] - 1 in row and el[4 * a + (i + 2) % 4] != a + 1][0]
            h = [i for i in range(4) if el[4 * b + i] == b + 1 and
                 el[4 * b + (i + 2) % 4] - 1 in row and el[4 * b + (i + 2) % 4] != b + 1][0]
            el[4 * a + f], fc[4 * a + f] = b + 1, h + 1
            el[4 * b + h], fc[4 * b + h] = a + 1, f + 1
    for s in (g, o):
        s.set("ielel", el)
        s.set("ielfc", fc)
    for n in (3, 4):
        for a, b in zip(g.run(n, runner="run_graph"), o.run(n)):
            assert np.array_equal(a, b)
        assert diff_fields(g.state(), o.state(), compared(p)) == []
    if kind == "boundary_face":
        assert not g.get_tiling()[0]


STAGES = ("predictor", "corrector", "remap")


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("stage", STAGES)
def test_negative_volume_of_each_stage(stage, mixed, oracle_lib):
    """A volume negative at the half step, at the full step (a node carried two
    and a half cells, one at the half step) or after the moved mesh: both
    forms stop there alike, with the oracle's error, and the fields show the
    stage: nodes not moved, nodes moved and no mass advected, mass advected.
    Component energies are the reference's: before the predictor, after it,
    after the corrector."""
    from bookleaf_f90_amd.device import BookLeaf, BookLeafError
    from oracle.pyoracle import Oracle
    nx, ny = 24, 9
    make = P.sod2mat_mixed if mixed else P.sod2mat
    p = make(nx=nx, ny=ny, eulerian=stage != "remap", dt_initial=1.0e-3)
    inner = np.nonzero(p.indtype > 0)[0]
    width = (p.ndx.max() - p.ndx.min()) / nx
    if stage == "remap":
        p = P.with_relaxation(p, abi.RELAX_LIN1, nsweep=1, om=3.0)
        rng = np.random.default_rng(1)
        p.ndx[inner] += rng.uniform(-0.4, 0.4, inner.size) * width
    else:
        # a node of the column at the interface (the mixed cells')
        xm = 0.5 * (p.ndx.max() + p.ndx.min())
        n = inner[np.argmin(np.abs(p.ndx[inner] - xm) + 1e-6 * np.abs(p.ndy[inner] - 0.5))]
        cells = {"predictor": 100.0, "corrector": 2.5}[stage]
        p.ndu[n] = cells * width / 1.0e-3
    p.config.update(cvisc1=0.0, cvisc2=0.0, div_sf=1.0e30, dt_max=1.0e-3, cfl_sf=1.0e10)
    print("stage", stage, mixed, flush=True)
    o = Oracle(p)
    with pytest.raises(BookLeafError) as e:
        o.run(6)
    want = (e.value.ierr, o.ts.nstep)
    seen = []
    for tiles in (True, False):
        g = BookLeaf(p)
        g.set_tiling(tiles)
        if want[1] > 1:  # to the step that fails
            g.run(want[1] - 1, runner="run_graph")
        before = g.state()
        with pytest.raises(BookLeafError) as e:
            g.run(6, runner="run_graph")
        assert "negative volume" in str(e.value)
        assert (e.value.ierr, g.ts.nstep) == want
        after = g.state()
        assert bool(g.get_tiling()[0]) == tiles
        same = {k: np.array_equal(before[k], after[k]) for k in ("ndx", "elmass", "cnmass")}
        assert same == {"predictor": dict(ndx=True, elmass=True, cnmass=True),
                        "corrector": dict(ndx=False, elmass=True, cnmass=True),
                        "remap": dict(ndx=False, elmass=False, cnmass=False)}[stage]
        seen.append(after)
    names = ["ndx", "ndy", "ndu", "ndv", "eldensity", "elenergy", "elpressure", "elcs2",
             "elmass", "cnmass", "cnviscx", "cnviscy", "elvisc"]
    names += ["cpdensity", "cppressure", "cpcs2", "cpvolume", "cpmass"]
    if stage != "predictor":  # (without tiles they are already the predictor's)
        names.append("cpenergy")
    assert diff_fields(seen[0], seen[1], names) == []
    if mixed:
        assert np.array_equal(seen[0]["cpenergy"][:p.ncp], o.get("cpenergy")[:p.ncp])
