"""Several pull steps per launch on D2Q9 lattices: against the oracle's
corrected step and one step per launch, bit for bit; lattices narrower than a
grown tile, cut tiles, both tile sizes (up to one tile per compute unit, and
beyond), several y-slices, walls on either axis with moving faces, periodic
seams, solids, every storage type, 1 to 17 steps, reads between runs, graphs."""
import numpy as np
import pytest

import plbpd_amd as P
from plbpd_amd import capi
from oracle.pyoracle import Boundary, NOSLIP, PERIODIC, UNSET

pytestmark = pytest.mark.gpu


def _bc(walls):
    types, vel = [PERIODIC, PERIODIC, UNSET, UNSET, PERIODIC, PERIODIC], {}
    for axis in walls:
        types[2 * axis] = types[2 * axis + 1] = NOSLIP
        vel[2 * axis] = (0.02, 0.0, -0.01)
        vel[2 * axis + 1] = (0.0, 0.0, 0.01)
    return Boundary(type=types, vel=vel), P.boundary(types, vel)


@pytest.mark.parametrize("X,Y,Z,walls,solids", [(1, 1, 1, (), False), (3, 1, 3, (0, 2), False), (5, 1, 7, (), True),
                                                (100, 1, 25, (2,), False), (64, 1, 40, (0, 2), True),
                                                (17, 3, 19, (0,), True), (201, 1, 131, (2,), True),
                                                (161, 1, 130, (), False)])
@pytest.mark.parametrize("variant", ["f64", "f32", "f64a32", "f32s", "f16s"])
def test_multi_step_matches_oracle(orc, X, Y, Z, walls, solids, variant):
    print(f"\n[case] multi-step {variant} {X}x{Y}x{Z} walls={walls} solids={solids}", flush=True)
    ob, pb = _bc(walls)
    mask = (np.random.default_rng(3).random((Z, Y, X)) < 0.15).astype(np.uint8) if solids else None
    tau, F, init = 0.63, (2e-5, 0.0, 1e-6), (P.INIT_PERTURBED, 5, 2e-3)
    fluid = orc.cor_flags(9, X, Y, Z, ob, mask) == 0
    bits = (lambda a: a.view(np.uint16)) if variant == "f16s" else (lambda a: a)
    o = orc.cor_state(variant, 9, X, Y, Z)
    orc.cor_init(o, 1.0, (0.01, 0.0, 0.0), init)
    with P.State(9, X, Y, Z, variant, P.FUSED) as a, P.State(9, X, Y, Z, variant, P.FUSED) as b:
        b.set_tuning(capi.TUNE_TWO_STEP, 0)
        for st in (a, b):
            st.set_boundary(pb, mask)
            st.initialize(1.0, (0.01, 0.0, 0.0), init, pb)
            st.configure(tau, F, pb)
        for n in (1, 2, 9, 17, 4):
            orc.cor_run(o, tau, F, ob, n, mask)
            a.step(n)
            b.step(n)
            ra, rb = bits(a.download_raw()), bits(b.download_raw())
            assert np.array_equal(ra[fluid], bits(o["f"])[fluid]), n
            assert np.array_equal(ra[fluid], rb[fluid]), n
        for spg in (2, 8, 10, 20):  # replays, with a read between
            a.step_graph(2 * spg + 3, spg)
            b.step(2 * spg + 3)
            assert np.array_equal(bits(a.download_raw())[fluid], bits(b.download_raw())[fluid]), spg


@pytest.mark.parametrize("Y,Z", [(1, 8 * 65535 + 1), (65536, 3)])
def test_layers_beyond_one_launch(orc, Y, Z):
    """More layers than a launch has workgroup rows for: one step per launch."""
    print(f"\n[case] multi-step f64 2x{Y}x{Z}", flush=True)
    ob, pb = _bc((2,))
    tau, F, init = 0.63, (2e-5, 0.0, 1e-6), (P.INIT_PERTURBED, 5, 2e-3)
    fluid = orc.cor_flags(9, 2, Y, Z, ob, None) == 0
    o = orc.cor_state("f64", 9, 2, Y, Z)
    orc.cor_init(o, 1.0, (0.01, 0.0, 0.0), init)
    orc.cor_run(o, tau, F, ob, 5, None)
    with P.State(9, 2, Y, Z, "f64", P.FUSED) as st:
        st.set_boundary(pb, None)
        st.initialize(1.0, (0.01, 0.0, 0.0), init, pb)
        st.configure(tau, F, pb)
        st.step(5)
        assert np.array_equal(st.download_raw()[fluid], o["f"][fluid])


def test_steps_per_launch():
    """What a launch advances, as the state reports it: D2Q9 with several steps
    is reported as the pull scheme."""
    with P.State(9, 256, 1, 64, "f64", P.FUSED) as st:
        assert st.scheme() == "pull" and st.steps_per_launch() == 8
        for key, value in ((capi.TUNE_TWO_STEP, 0), (capi.TUNE_INDEX64, 1), (capi.TUNE_SCHEME, capi.SCHEME_PUSH)):
            st.set_tuning(key, value)
            assert st.steps_per_launch() == 1
            st.set_tuning(key, -1 if key == capi.TUNE_TWO_STEP else 0)
            assert st.steps_per_launch() == 8
    for Y, Z in ((1, 8 * 65535 + 1), (65536, 3)):
        with P.State(9, 2, Y, Z, "f64", P.FUSED) as st:
            assert st.steps_per_launch() == 1
    with P.State(9, 256, 1, 64, "f64", P.FUSED_AA) as st:
        assert st.steps_per_launch() == 1
    with P.State(19, 64, 64, 64, "f64", P.FUSED) as st:
        assert st.steps_per_launch() == 2
    with P.State(9, 8, 1, 8, "f64", P.LITERAL) as st:
        with pytest.raises(P.LogicError):
            st.steps_per_launch()


def test_multi_step_rule():
    """Several steps per launch where the tiles lie in the lattice, so on every
    lattice of test_multi_step_matches_oracle, and not on thin ones."""
    several = [(1, 1, 1), (3, 1, 3), (5, 1, 7), (100, 1, 25), (64, 1, 40), (17, 3, 19), (201, 1, 131), (161, 1, 130),
               (512, 1, 256), (4, 1, 262144)]
    for X, Y, Z in several:
        for variant in ("f64", "f32", "f64a32", "f32s", "f16s"):
            with P.State(9, X, Y, Z, variant, P.FUSED) as st:
                assert st.steps_per_launch() > 1, (X, Y, Z, variant)
    for X, Y, Z in ((65536, 1, 4), (1048576, 1, 1), (3, 40000, 3), (131072, 1, 8)):
        for variant in ("f64", "f32s", "f16s"):
            with P.State(9, X, Y, Z, variant, P.FUSED) as st:
                assert st.steps_per_launch() == 1, (X, Y, Z, variant)
    for variant, steps in (("f64", 8), ("f64a32", 8), ("f32s", 4), ("f16s", 1)):
        with P.State(9, 1024, 1, 1024, variant, P.FUSED) as st:
            assert st.steps_per_launch() == steps, variant


@pytest.mark.parametrize("X,vec", [(100, 0), (256, 0), (64, 1), (128, 2), (256, 4), (384, 1), (512, 2)])
@pytest.mark.parametrize("walls,solids", [((2,), False), ((0, 2), True), ((), False)])
@pytest.mark.parametrize("variant", ["f64", "f32", "f64a32", "f32s", "f16s"])
def test_single_steps_match_oracle(orc, X, vec, walls, solids, variant):
    """One step per launch (staged calls, single steps, large lattices): the cell
    pull kernel and the row pull kernel at each width, which runs of several
    steps no longer reach on lattices of this size."""
    print(f"\n[case] D2Q9 single steps {variant} X={X} vec={vec} walls={walls} solids={solids}", flush=True)
    Z = 21
    ob, pb = _bc(walls)
    mask = (np.random.default_rng(3).random((Z, 1, X)) < 0.15).astype(np.uint8) if solids else None
    tau, F, init = 0.63, (2e-5, 0.0, 1e-6), (P.INIT_PERTURBED, 5, 2e-3)
    fluid = orc.cor_flags(9, X, 1, Z, ob, mask) == 0
    bits = (lambda a: a.view(np.uint16)) if variant == "f16s" else (lambda a: a)
    o = orc.cor_state(variant, 9, X, 1, Z)
    orc.cor_init(o, 1.0, (0.01, 0.0, 0.0), init)
    orc.cor_run(o, tau, F, ob, 9, mask)
    with P.State(9, X, 1, Z, variant, P.FUSED) as a, P.State(9, X, 1, Z, variant, P.FUSED) as b:
        for st in (a, b):
            st.set_tuning(capi.TUNE_VECTOR, vec)
            st.set_boundary(pb, mask)
            st.initialize(1.0, (0.01, 0.0, 0.0), init, pb)
            st.configure(tau, F, pb)
        a.set_tuning(capi.TUNE_TWO_STEP, 0)
        assert a.steps_per_launch() == 1 and b.steps_per_launch() == 8
        a.step(9)
        for _ in range(9):
            b.step(1)
        for st in (a, b):
            assert np.array_equal(bits(st.download_raw())[fluid], bits(o["f"])[fluid])
