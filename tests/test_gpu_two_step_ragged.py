"""Two pull steps per launch on rows that are no whole number of 32-cell tiles
(automatic from 2^18 cells): tiles of a shape of their own, the last of a row
or column cut short, rows of a few cells, walls on each axis with a moving
wall, periodic seams, solids and every storage type, against the oracle's
corrected step and against one step per launch, bit for bit."""
import numpy as np
import pytest

import plbpd_amd as P
from plbpd_amd import capi
from oracle.pyoracle import Boundary, NOSLIP, PERIODIC

pytestmark = pytest.mark.gpu

CASES = [  # q, X, Y, Z, walled axis or None, solids, index64
    (19, 70, 61, 63, 2, True, 0),
    (19, 131, 47, 43, 1, False, 0),
    (19, 5, 230, 229, 0, False, 0),
    (19, 250, 37, 29, None, True, 1),
    (19, 33, 90, 89, 2, False, 1),
    (27, 101, 53, 50, 2, True, 0),
    (27, 47, 75, 76, 0, False, 1),
]


@pytest.mark.parametrize("q,X,Y,Z,axis,solids,wide", CASES)
@pytest.mark.parametrize("variant", ["f64", "f32s", "f16s", "f32"])
def test_ragged_two_step_matches_oracle(orc, q, X, Y, Z, axis, solids, wide, variant):
    print(f"\n[case] ragged two-step {variant} q={q} {X}x{Y}x{Z} walls={axis} solids={solids}", flush=True)
    types, vel = [PERIODIC] * 6, {}
    if axis is not None:
        types[2 * axis] = types[2 * axis + 1] = NOSLIP
        vel = {2 * axis: (0.02, 0.01, -0.01), 2 * axis + 1: (0.0, 0.0, 0.0)}
    ob, pb = Boundary(type=types, vel=vel), P.boundary(types, vel)
    mask = (np.random.default_rng(8).random((Z, Y, X)) < 0.12).astype(np.uint8) if solids else None
    tau, F, init, steps = 0.62, (2e-5, -1e-6, 1e-6), (P.INIT_PERTURBED, 5, 2e-3), 5
    o = orc.cor_state(variant, q, X, Y, Z)
    orc.cor_init(o, 1.0, (0.01, 0.0, 0.0), init)
    orc.cor_run(o, tau, F, ob, steps, mask)
    fluid = orc.cor_flags(q, X, Y, Z, ob, mask) == 0
    raws = []
    for two in (-1, 0):
        with P.State(q, X, Y, Z, variant, P.FUSED) as st:
            st.set_tuning(capi.TUNE_TWO_STEP, two)
            st.set_tuning(capi.TUNE_INDEX64, wide)
            assert st.scheme() == ("pull2" if two else "pull")
            st.set_boundary(pb, mask)
            st.initialize(1.0, (0.01, 0.0, 0.0), init, pb)
            st.configure(tau, F, pb)
            st.step(steps)
            raw = st.download_raw()
        raws.append(raw.view(np.uint16) if variant == "f16s" else raw)
    exp = o["f"].view(np.uint16) if variant == "f16s" else o["f"]
    assert np.array_equal(raws[0][fluid], exp[fluid])
    assert np.array_equal(raws[0][fluid], raws[1][fluid])


def test_ragged_two_step_rule():
    """Thin lattices and those below 2^18 cells keep one step per launch."""
    for q, X, Y, Z, want in ((19, 70, 61, 63, "pull2"), (19, 600, 1, 500, "pull"), (19, 500, 600, 1, "pull"),
                             (19, 61, 64, 64, "pull"), (27, 75, 70, 70, "pull2")):
        with P.State(q, X, Y, Z, "f32s", P.FUSED) as st:
            assert st.scheme() == want, (q, X, Y, Z)
    with P.State(19, 70, 61, 63, "f64", P.FUSED) as st:
        st.set_tuning(capi.TUNE_TWO_TILE_X, 32)
        assert st.scheme() == "pull"


@pytest.mark.parametrize("q,pad", [(19, 70 << 20), (19, 100 << 20), (19, 160 << 20), (27, 50 << 20), (27, 100 << 20),
                                   (27, 130 << 20)])
def test_two_step_array_sizes(q, pad):
    """Arrays addressed as two and four buffers and by pointers (populations
    set far apart on a small lattice): the values of the array that one
    buffer holds, bit for bit."""
    X, Y, Z = 64, 10, 9
    types, vel = [PERIODIC] * 4 + [NOSLIP] * 2, {P.UP: (0.02, 0.0, 0.0), P.DOWN: (0.0, 0.0, 0.0)}
    pb = P.boundary(types, vel)
    for solids in (True, False):
        print(f"\n[case] two-step array sizes q={q} pad={pad} solids={solids}", flush=True)
        mask = (np.random.default_rng(8).random((Z, Y, X)) < 0.12).astype(np.uint8) if solids else None
        out = []
        for p in (-1, pad):
            with P.State(q, X, Y, Z, "f32s", P.FUSED, pop_pad=p) as st:
                st.set_tuning(capi.TUNE_TWO_STEP, 1)
                assert st.scheme() == "pull2"
                st.set_boundary(pb, mask)
                st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 5, 2e-3), pb)
                st.configure(0.62, (2e-5, -1e-6, 1e-6), pb)
                st.step(7)
                out.append((st.download_raw()[1:-1], st.moments()))
        fluid = slice(None) if mask is None else mask[1:-1] == 0
        assert np.array_equal(out[0][0][fluid], out[1][0][fluid])
        assert all(np.array_equal(a, b) for a, b in zip(out[0][1], out[1][1]))


@pytest.mark.parametrize("q,variant", [(19, "f64"), (19, "f64a32"), (27, "f64"), (27, "f32s"), (27, "f32")])
def test_two_step_held_values(orc, q, variant):
    """Values held in registers from one plane to the next: one plane to a few,
    z-chunks of one and two planes, rows of cells one more and one fewer than a
    tile has, walls on z with both faces moving, solids and none."""
    types = [PERIODIC] * 4 + [NOSLIP] * 2
    vel = {P.UP: (0.02, 0.01, -0.01), P.DOWN: (-0.01, 0.0, 0.005)}
    for Y, Z, zc, walls, solids in ((13, 1, 0, False, True), (14, 2, 1, False, False), (12, 3, 1, True, True),
                                    (27, 4, 2, True, False), (7, 5, 0, True, True), (8, 6, 3, False, False)):
        print(f"\n[case] held values q={q} {variant} 64x{Y}x{Z} chunk {zc} walls={walls} solids={solids}", flush=True)
        ty, ve = (types, vel) if walls else ([PERIODIC] * 6, {})
        ob, pb = Boundary(type=ty, vel=ve), P.boundary(ty, ve)
        mask = (np.random.default_rng(4).random((Z, Y, 64)) < 0.2).astype(np.uint8) if solids else None
        tau, F, init = 0.62, (2e-5, -1e-6, 1e-6), (P.INIT_PERTURBED, 5, 2e-3)
        o = orc.cor_state(variant, q, 64, Y, Z)
        orc.cor_init(o, 1.0, (0.01, 0.0, 0.0), init)
        orc.cor_run(o, tau, F, ob, 7, mask)
        fluid = orc.cor_flags(q, 64, Y, Z, ob, mask) == 0
        with P.State(q, 64, Y, Z, variant, P.FUSED) as st:
            st.set_tuning(capi.TUNE_TWO_STEP, 1)
            st.set_tuning(capi.TUNE_TWO_ZCHUNK, zc)
            assert st.scheme() == "pull2"
            st.set_boundary(pb, mask)
            st.initialize(1.0, (0.01, 0.0, 0.0), init, pb)
            st.configure(tau, F, pb)
            st.step(7)
            assert np.array_equal(st.download_raw()[fluid], o["f"][fluid])


def test_two_step_only_where_its_tiles_fill():
    """Automatic only where a launch's tiles and chunks of planes use the chip:
    not on cross-sections of a few cells, however long; asked for, still there."""
    for q, X, Y, Z, variant, want in ((19, 9, 9, 4000, "f32s", "pull"), (19, 12, 12, 2000, "f16s", "pull"),
                                      (27, 9, 9, 4000, "f32s", "pull"), (27, 300, 3, 300, "f16s", "pull"),
                                      (19, 30, 30, 900, "f32s", "pull2"), (27, 24, 24, 500, "f64", "pull2"),
                                      (19, 3, 300, 300, "f32s", "pull2"), (19, 250, 191, 133, "f16s", "pull2")):
        with P.State(q, X, Y, Z, variant, P.FUSED) as st:
            assert st.scheme() == want, (q, X, Y, Z, variant)
            st.set_tuning(capi.TUNE_TWO_STEP, 1)
            assert st.scheme() == "pull2"


@pytest.mark.parametrize("q,X,Y,Z,variant", [(19, 24, 24, 500, "f32s"), (27, 30, 30, 300, "f64"), (19, 32, 9, 1200, "f64"),
                                             (27, 64, 5, 1100, "f16s"), (19, 7, 7, 6000, "f32")])
def test_more_chunks_than_planes_of_a_tile(q, X, Y, Z, variant):
    """Long lattices of one or two tiles across, in as many z-chunks as there
    are compute units: the values of one step per launch, bit for bit."""
    types, vel = [PERIODIC] * 4 + [NOSLIP] * 2, {P.UP: (0.02, 0.01, -0.01), P.DOWN: (0.0, 0.0, 0.0)}
    pb = P.boundary(types, vel)
    print(f"\n[case] chunks {variant} q={q} {X}x{Y}x{Z}", flush=True)
    mask = (np.random.default_rng(8).random((Z, Y, X)) < 0.1).astype(np.uint8)
    out = []
    for two in (1, 0):
        with P.State(q, X, Y, Z, variant, P.FUSED) as st:
            st.set_tuning(capi.TUNE_TWO_STEP, two)
            assert st.scheme() == ("pull2" if two else "pull")
            st.set_boundary(pb, mask)
            st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 5, 2e-3), pb)
            st.configure(0.62, (2e-5, -1e-6, 1e-6), pb)
            st.step(6)
            raw = st.download_raw()[1:-1]
            out.append((raw.view(np.uint16) if variant == "f16s" else raw)[mask[1:-1] == 0])
    assert np.array_equal(out[0], out[1])
