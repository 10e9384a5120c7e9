"""The per-driver kernels that read several neighbours or incidences at once
(getdt in one pass, the node sums four incidences at a time) against the
oracle, bit for bit in every field after every driver of two steps: meshes of
one element row, a workgroup's 256 elements and one more, elements starting
from any corner with random numbering (nodes of one to four incidences in
any order), every element in motion, and the remap's drivers."""
import pytest

from bookleaf_f90_amd import problem as P
from tests.helpers import diff_fields, granular_sequence
from tests.test_gpu_remap_tiles import _eul, _renumbered, _stirred

pytestmark = pytest.mark.gpu

CASES = {
    "3x1": lambda: _stirred(P.sod(nx=3, ny=1, height=0.3, dt_initial=1e-3)),
    "16x16": lambda: _stirred(P.sod(nx=16, ny=16, height=1.0, dt_initial=1e-3)),
    "257x1": lambda: _stirred(P.sod(nx=257, ny=1, height=0.004)),
    "sedov_24": lambda: P.sedov(n=24, kappa=0.01),
    "23x19_turned": lambda: _renumbered(
        _stirred(P.sod(nx=23, ny=19, height=0.8, dt_initial=1e-3)), 2, 3),
    "21x17_turned_eul": lambda: _renumbered(
        _stirred(P.sod(nx=21, ny=17, height=0.8, eulerian=True, dt_initial=1e-3)), 3, 1),
    "sedov_20_eul": lambda: _eul(P.sedov(n=20, kappa=0.01)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_every_driver_of_two_steps(name, oracle_lib):
    from bookleaf_f90_amd.device import BookLeaf
    from oracle.pyoracle import Oracle
    p = CASES[name]()
    print("case", name, "nel", p.nel, flush=True)
    g, o = BookLeaf(p), Oracle(p)
    for step in range(2):
        for (label, a), (_, b) in zip(granular_sequence(g), granular_sequence(o)):
            a()
            b()
            assert diff_fields(g.state(), o.state()) == [], (step, label)
