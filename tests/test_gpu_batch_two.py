"""Two pull steps per launch for batched domains (from 2^18 cells): against
single steps of the same batch and against per-domain oracle runs, bit for
bit; domains of one to a few cells on an edge, of whole and cut tiles, walls
on each axis with moving faces, periodic seams, graphs and odd counts."""
import numpy as np
import pytest

import plbpd_amd as P
from oracle.pyoracle import Boundary, NOSLIP, PERIODIC

pytestmark = pytest.mark.gpu

EDGES = [(96, 90, 25), (3, 40, 200), (70, 3, 90), (150, 33, 5), (17, 19, 23), (40, 41, 42), (3, 3, 3), (64, 64, 3),
         (33, 5, 31)]


def _domains():
    rng = np.random.default_rng(12)
    return [{"x": x, "y": y, "z": z, "tau": float(rng.uniform(0.55, 1.5)),
             "force": tuple(float(v) for v in rng.uniform(-1e-5, 1e-5, 3))} for x, y, z in EDGES]


def _bc(axis):
    types, vel = [PERIODIC] * 6, {}
    if axis is not None:
        types[2 * axis] = types[2 * axis + 1] = NOSLIP
        vel = {2 * axis: (0.02, 0.01, -0.01), 2 * axis + 1: (0.0, -0.01, 0.0)}
    return Boundary(type=types, vel=vel), P.boundary(types, vel)


@pytest.mark.parametrize("axis", [None, 0, 1, 2])
@pytest.mark.parametrize("q,variant", [(19, "f32s"), (19, "f64"), (19, "f16s"), (19, "f64a32"), (27, "f32"),
                                       (27, "f64")])
def test_batched_pairs_equal_single_steps(orc, q, variant, axis):
    print(f"\n[case] batch two-step q={q} {variant} walls={axis}", flush=True)
    doms = _domains()
    ob, pb = _bc(axis)
    init = (P.INIT_PERTURBED, 77, 2e-3)
    pair, single = P.Batch(q, variant, doms, pb), P.Batch(q, variant, doms, pb)
    assert pair.cells()[0] >= 2 ** 18
    for b in (pair, single):
        b.initialize(1.0, (0.01, 0.0, 0.0), init)
    pair.step(6)
    pair.step(3)
    pair.step(13, 6)   # graph of an odd number of pairs
    pair.step(9, 8)    # and of an even number
    for _ in range(31):
        single.step(1)
    for d, dm in enumerate(doms):
        for a, e in zip(pair.moments(d), single.moments(d)):
            assert np.array_equal(a, e), (d, dm)
    pair.initialize(1.0, (0.01, 0.0, 0.0), init)
    pair.step(5)
    for d in (0, 2, 4, 6):
        dm = doms[d]
        o = orc.cor_state(variant, q, dm["x"], dm["y"], dm["z"])
        orc.cor_init(o, 1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 77 + d, 2e-3))
        orc.cor_run(o, dm["tau"], dm["force"], ob, 5)
        for a, e in zip(pair.moments(d), orc.cor_moments(o, ob)):
            assert np.array_equal(a, e), (d, dm)
    pair.close()
    single.close()


# three domains that fill tiles and chunks, with others of a few cells on an
# edge beside them: the two-step launch for every velocity set and storage
MIXED = [(128, 120, 130), (17, 19, 23), (130, 128, 127), (3, 3, 3), (33, 5, 31), (131, 100, 90), (3, 40, 60),
         (70, 3, 40), (64, 64, 3), (40, 41, 42)]


@pytest.mark.parametrize("axis", [None, 0, 1, 2])
@pytest.mark.parametrize("q,variant", [(19, "f32s"), (19, "f64"), (19, "f16s"), (19, "f64a32"), (19, "f32"),
                                       (27, "f32s"), (27, "f64"), (27, "f16s")])
def test_two_step_launches_equal_single_steps(orc, q, variant, axis):
    """With the two-step kernel shown to be the one that runs."""
    print(f"\n[case] batch two-step launches q={q} {variant} walls={axis}", flush=True)
    rng = np.random.default_rng(13)
    doms = [{"x": x, "y": y, "z": z, "tau": float(rng.uniform(0.55, 1.5)),
             "force": tuple(float(v) for v in rng.uniform(-1e-5, 1e-5, 3))} for x, y, z in MIXED]
    ob, pb = _bc(axis)
    init = (P.INIT_PERTURBED, 78, 2e-3)
    pair, single = P.Batch(q, variant, doms, pb), P.Batch(q, variant, doms, pb)
    assert pair.steps_per_launch() == 2
    for b in (pair, single):
        b.initialize(1.0, (0.01, 0.0, 0.0), init)
    for n, spg in ((5, 0), (8, 6), (5, 4)):  # graphs of an odd and an even number of pairs
        pair.step(n, spg)
        for _ in range(n):
            single.step(1)
        for d, dm in enumerate(doms):
            for a, e in zip(pair.moments(d), single.moments(d)):
                assert np.array_equal(a, e), (n, d, dm)
    single.close()
    pair.initialize(1.0, (0.01, 0.0, 0.0), init)
    pair.step(5)
    for d in (1, 3, 4, 6, 7, 8, 9):
        dm = doms[d]
        o = orc.cor_state(variant, q, dm["x"], dm["y"], dm["z"])
        orc.cor_init(o, 1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 78 + d, 2e-3))
        orc.cor_run(o, dm["tau"], dm["force"], ob, 5)
        for a, e in zip(pair.moments(d), orc.cor_moments(o, ob)):
            assert np.array_equal(a, e), (d, dm)
    pair.close()


def test_two_step_rule_of_a_batch():
    """One step per launch for batches below 2^18 cells, of thin domains and of
    domains too small to fill a tile; with the push scheme; and for D2Q9."""
    def steps(q, variant, edges, n):
        dm = [{"x": edges[0], "y": edges[1], "z": edges[2], "tau": 0.7, "force": (1e-6, 0.0, 0.0)}] * n
        b = P.Batch(q, variant, dm, P.channel(periodic_y=q != 9))
        s = b.steps_per_launch()
        b.set_scheme(P.capi.SCHEME_PUSH)
        assert b.steps_per_launch() == 1
        b.close()
        return s

    for q in (19, 27):
        for variant in ("f64", "f32s", "f16s"):
            assert steps(q, variant, (40, 40, 40), 4) == 1
            assert steps(q, variant, (9, 9, 9), 400) == 1
            assert steps(q, variant, (200, 200, 3), 5) == 1
            assert steps(q, variant, (128, 128, 128), 4) == 2
            assert steps(q, variant, (12, 12, 12), 1000) == 1
        assert steps(q, "f64", (16, 16, 16), 512) == 2
        assert steps(q, "f32s", (14, 14, 14), 2000) == steps(q, "f16s", (22, 22, 22), 300) == 1
    assert steps(9, "f64", (512, 1, 600), 1) == 1
