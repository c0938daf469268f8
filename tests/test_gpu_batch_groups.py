"""Local forces of the batched engine held for some of the shot groups at a time: every value of
"local_groups" gives the same bits (19 shots: three groups of eight, the last with padding)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def shots():
    from specfem3d_amd import workloads as W
    w = W.sea_over_visco_large(scale=0.05, nshots=19, nstep=60, nrec_side=2)
    rng = np.random.default_rng(5)
    w.shots = [(s, r, int(rng.integers(20, 61))) for s, r, _ in w.shots]
    return w


@pytest.mark.parametrize("kind,groups,sc", [("elastic", 1, 8), ("elastic", 2, 4), ("visco", 1, 4), ("visco", 2, 8)])
def test_local_groups_same_bits(shots, kind, groups, sc):
    from specfem3d_amd.batch import BatchSolver
    att = shots.attenuation if kind == "visco" else None
    print(f"[gpu] {kind} batch, local forces of {groups} of 3 groups, {sc} shots per workgroup", flush=True)
    out = []
    for g in (3, groups):
        b = BatchSolver(shots.db, shots.shots, exact=True, shots_per_group=sc, assembly=2, attenuation=att)
        b.set_tuning("local_groups", g)
        assert b.L.sf_batch_get_tuning(b.h, b"local_groups") == g
        b.run(graph_steps=10 if sc == 8 else 1)
        n = len(shots.shots)
        out.append([b.seismograms(i) for i in range(n)] + [b.displ(i) for i in range(n)] + [b.potential(i) for i in range(n)])
        b.close()
    assert max(np.abs(x).max() for x in out[0]) > 0
    assert all(np.array_equal(x, y) for x, y in zip(*out))
