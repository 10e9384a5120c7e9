"""The ensemble's limiter pass: rounds of whole elements and a last round of
quads, over workgroups whose pieces are halved for a small ensemble.  Every
split (odd chunks, one and several rounds, every workgroup size) gives each
instance's dt sequence and viscosity as the oracle running that instance
alone, bit for bit."""
import numpy as np
import pytest

from bookleaf_f90_amd import problem as P
from tests.helpers import diff_fields
from tests.test_gpu_ensemble import CFG

pytestmark = pytest.mark.gpu

FIELDS = ("elenergy", "elvisc", "cnviscx", "cnviscy", "ndx", "ndy", "ndu", "ndv")
NSTEPS = 60


@pytest.fixture(scope="module")
def alone(oracle_lib):
    from oracle.pyoracle import Oracle
    params = P.ensemble_params(4, seed=5, nmin=16, nmax=48)
    runs = []
    for q in params:
        o = Oracle(P.ensemble_instance(q, config=CFG))
        runs.append((o.run(NSTEPS), o.state()))
    return params, runs


@pytest.mark.parametrize("block,chunk,tiles", [(64, 64, True), (64, 4096, True), (128, 300, True),
                                               (192, 1001, True), (256, 257, False),
                                               (256, 511, True), (256, 65536, True)])
def test_every_split_matches_each_instance_alone(block, chunk, tiles, alone):
    from bookleaf_f90_amd.device import Ensemble
    params, runs = alone
    print("ensemble limiter", block, chunk, tiles, [q["nx"] for q in params], flush=True)
    ens = Ensemble(params, config=CFG)
    ens.set_tiling(tiles)
    ens.set_tuning(limiter_block=block, ens_chunk=chunk)
    dt, idt, ctl = ens.run(NSTEPS)
    state = {f: ens.get(f) for f in FIELDS}
    for k, (hist, ref) in enumerate(runs):
        for mine, other in zip((dt, idt, ctl), hist):
            assert np.array_equal(mine[:, k], other), k
        mine = {f: ens.instance_field(f, k, state[f]) for f in FIELDS}
        assert diff_fields(mine, ref, FIELDS) == [], k
    ens.close()
