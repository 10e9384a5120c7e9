"""The side connectivity changed after the maps were built: ielel and ielfc of
a mesh cut along a column of faces (both sides of the cut are boundary faces)
and of the whole mesh, uploaded in turn without bl_build_maps.  Every table
made from the neighbours follows: the drivers, the Lagrangian step and the
remap give the oracle's results with the same neighbours, bit for bit, in both
forms of the step."""
import ctypes as C

import numpy as np
import pytest

from bookleaf_f90_amd import problem as P
from tests.helpers import diff_fields, granular_sequence
from tests.test_gpu_graph import compared
from tests.test_gpu_remap_tiles import _renumbered, _stirred

pytestmark = pytest.mark.gpu


def _problem(eulerian):
    return _stirred(P.sod(nx=29, ny=17, height=0.6, eulerian=eulerian, dt_initial=1e-3))


def _cut(g, p, at):
    """ielel and ielfc with every face between the elements left and right of
    x = at made a boundary face of both."""
    el, fc = g.get("ielel"), g.get("ielfc")
    x = g.get("ndx")[p.ielnd.reshape(-1, 4) - 1].mean(axis=1)
    n = 4 * p.nel
    e, f = np.divmod(np.arange(n), 4)
    cut = (x[e] < at) != (x[el[:n] - 1] < at)
    assert cut.any()
    el[:n][cut] = e[cut] + 1
    fc[:n][cut] = (f[cut] + 2) % 4 + 1
    return el, fc


def _store(g, name, values):
    """A store the library does not see."""
    a = np.ascontiguousarray(values)
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    assert hip.hipMemcpy(g.device_ptr(name), a.ctypes.data, a.nbytes, 1) == 0


def _pair(p, at):
    """The problem on the device and the oracle, its maps built on the mesh cut
    at x = at (none for None); and the two sides' neighbours of the whole mesh."""
    from bookleaf_f90_amd.device import BookLeaf
    from oracle.pyoracle import Oracle
    g, o = BookLeaf(p), Oracle(p)
    whole = g.get("ielel"), g.get("ielfc")
    if at is not None:
        _give(g, o, _cut(g, p, at))
        assert g.lib.bl_build_maps(g.h) == 0
    return g, o, whole


def _give(g, o, tables, put=None):
    for name, v in zip(("ielel", "ielfc"), tables):
        (put or type(g).set)(g, name, v)
        o.set(name, v)


@pytest.mark.parametrize("how", ["upload", "device_ptr"])
@pytest.mark.parametrize("change", ["cut", "join"])
@pytest.mark.parametrize("eulerian", [False, True])
def test_drivers_read_the_neighbours_they_are_given(eulerian, change, how, oracle_lib):
    p = _renumbered(_problem(eulerian), 2, 1)
    print("drivers", eulerian, change, how, flush=True)
    g, o, whole = _pair(p, 0.5 if change == "join" else None)
    g.step()
    o.step()
    _give(g, o, whole if change == "join" else _cut(g, p, 0.5),
          _store if how == "device_ptr" else None)
    a, b = g.hydro_getdt_noalloc(), o.hydro_getdt()
    assert [(q.rdt, q.idt, q.sdt) for q in a] == [(q.rdt, q.idt, q.sdt) for q in b]
    assert diff_fields(g.state(), o.state()) == []
    # (the drivers' next getdt takes these cs2, elvisc added, as the oracle's does)
    for step in range(2):
        for (label, a), (_, b) in zip(granular_sequence(g), granular_sequence(o)):
            a()
            b()
            assert diff_fields(g.state(), o.state()) == [], (step, label)


@pytest.mark.parametrize("tiles", [True, False])
@pytest.mark.parametrize("eulerian", [False, True])
def test_steps_after_an_upload(eulerian, tiles, oracle_lib):
    p = _problem(eulerian)
    print("steps", eulerian, tiles, flush=True)
    g, o, whole = _pair(p, 0.25)
    g.set_tiling(tiles)
    for k, tables in enumerate((None, whole, _cut(g, p, 0.5), whole)):
        if tables is not None:
            _give(g, o, tables)
        for a, b in zip(g.run(4 + k, runner="run_graph"), o.run(4 + k)):
            assert np.array_equal(a, b)
        assert diff_fields(g.state(), o.state(), compared(p)) == [], k
    assert bool(g.get_tiling()[0]) == tiles


def test_tiled_remap_after_an_upload_the_other_form_ran_on(oracle_lib):
    """The neighbours change while the tiling is off and a run of the other
    form rebuilds its own table: the tiled remap's tables follow too."""
    p = _problem(True)
    print("switched", flush=True)
    g, o, whole = _pair(p, None)
    for tiles, tables in ((True, None), (False, _cut(g, p, 0.5)), (True, None), (False, whole),
                          (True, None)):
        g.set_tiling(tiles)
        if tables is not None:
            _give(g, o, tables)
        for a, b in zip(g.run(4, runner="run_graph"), o.run(4)):
            assert np.array_equal(a, b)
        assert bool(g.get_tiling()[0]) == tiles
        assert diff_fields(g.state(), o.state(), compared(p)) == []
