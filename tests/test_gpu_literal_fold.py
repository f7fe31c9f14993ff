"""The literal step's deferred calls: the periodic copies, moments and resets
of one step folded into the next step's collide+push kernel.  Whole steps of
staged calls with nothing read in between, then a further step cut off after
each of its calls (the deferred rest then runs by itself), against the
oracle's separate stages, bit for bit; rows and columns of one to three cells,
where a cell lies on both seams, and rows longer than a workgroup."""
import numpy as np
import pytest

import plbpd_amd as P
from oracle.pyoracle import Boundary, NOSLIP, PERIODIC, UNSET, UP, DOWN

pytestmark = pytest.mark.gpu

CALLS = ["collide", "stream", "noslip", "periodic", "moments", "reset"]


def _bc(types, vel, rho_s=1.0):
    return Boundary(type=types, vel=vel, rho_s=rho_s), P.boundary(types, vel, rho_s)


def _same(st, o, where):
    dt = o["n"].dtype
    for name, field in (("n", P.FIELD_N), ("rho", P.FIELD_RHO), ("u", P.FIELD_U), ("ntmp", P.FIELD_NTMP)):
        assert np.array_equal(st.download(field, dtype=dt), o[name]), (where, name)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("q,X,Y,Z,ew,ns", [(9, 300, 1, 4, 1, 0), (19, 1, 1, 3, 1, 1), (19, 2, 1, 4, 1, 1),
                                           (19, 7, 5, 4, 1, 0), (19, 6, 3, 5, 0, 1), (27, 2, 3, 3, 1, 1),
                                           (27, 66, 4, 3, 1, 1)])
def test_deferred_calls_cut_off_anywhere(orc, q, X, Y, Z, ew, ns, prec):
    dt = np.float64 if prec == "f64" else np.float32
    pe = lambda on: [PERIODIC, PERIODIC] if on else [UNSET, UNSET]  # noqa: E731
    types = pe(ew) + pe(ns) + [NOSLIP, NOSLIP]
    ob, pb = _bc(types, {UP: (0.05, 0.01, 0.0), DOWN: (0.0, -0.02, 0.0)})
    obr, pbr = _bc(types, {UP: (0.02, 0.0, 0.004), DOWN: (0.0, 0.003, 0.0)}, 1.01)
    tau, F = 0.7, (1e-4, -2e-5, 3e-5)
    for cut in range(len(CALLS)):
        print(f"\n[case] literal fold q={q} {X}x{Y}x{Z} {prec} cut after {CALLS[cut]}", flush=True)
        o = orc.lit_state(q, X, Y, Z, dt)
        orc.lit_init(o, 1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 31, 1e-2), ob)
        with P.State(q, X, Y, Z, prec, P.LITERAL) as st:
            st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 31, 1e-2), pb)

            def call(name):
                if name == "collide":
                    orc.lit_collide(o, tau, F), st.collide(tau, F)
                elif name == "stream":
                    orc.lit_push(o), st.stream("push")
                elif name == "noslip":
                    orc.lit_noslip(o, ob), st.apply_noslip(pb)
                elif name == "periodic":
                    orc.lit_periodic(o, ob), st.apply_periodicity(pb)
                elif name == "moments":
                    orc.lit_moments(o), st.calc_moments()
                else:
                    orc.lit_reset(o, obr), st.reset(pbr)

            for _ in range(2):
                for name in CALLS:
                    call(name)
            for name in CALLS[:cut + 1]:
                call(name)
            # a call that does not follow in order finds the deferred ones done
            if CALLS[cut] in ("periodic", "moments"):
                orc.lit_collide(o, tau, F), st.collide(tau, F)
            _same(st, o, cut)


@pytest.mark.parametrize("q,X,Y,Z", [(9, 70, 1, 3), (19, 5, 4, 3), (19, 3, 3, 8), (27, 4, 3, 5)])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_step_stores_the_densities_noslip_reads(orc, q, X, Y, Z, axis):
    """plb_step, walls on one axis with moving faces: inside the run only the
    densities that no-slip reads are stored, and the last step stores all."""
    if q == 9 and axis == 1:
        pytest.skip("D2Q9 has no y direction")
    print(f"\n[case] literal step q={q} {X}x{Y}x{Z} walls on axis {axis}", flush=True)
    types = [UNSET if a == 2 or (q == 9 and a == 1) else PERIODIC for a in (0, 0, 1, 1, 2, 2)]
    types[2 * axis] = types[2 * axis + 1] = NOSLIP
    vel = {2 * axis: (0.02, 0.01, -0.01), 2 * axis + 1: (0.0, -0.02, 0.015)}
    ob, pb = _bc(types, vel, 0.99)
    o = orc.lit_state(q, X, Y, Z)
    orc.lit_init(o, 1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 3, 1e-2), ob)
    with P.State(q, X, Y, Z, "f64", P.LITERAL) as st:
        st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 3, 1e-2), pb)
        st.configure(0.75, (1e-4, 0.0, -2e-5), pb)
        for n in (1, 2, 5):
            orc.lit_run(o, 0.75, (1e-4, 0.0, -2e-5), ob, n)
            st.step(n)
            _same(st, o, n)


@pytest.mark.parametrize("q,X,Y,Z", [(9, 70, 1, 4), (19, 5, 4, 6), (19, 1, 2, 3), (27, 66, 3, 4)])
@pytest.mark.parametrize("faces", ["PPNNNN", "NNPPNN", "UUPPNN", "PPNUUN", "PPPPUU", "NNNNUU", "UUUUUU", "PPPPNU"])
def test_step_keeps_what_the_next_step_reads(orc, q, X, Y, Z, faces):
    """plb_step: inside the run a collision leaves in place only the slots that
    no push fills and that no periodic copy replaces or a no-slip pass reads;
    walls, seams and bare faces meet at every kind of edge here."""
    print(f"\n[case] literal step q={q} {X}x{Y}x{Z} faces {faces}", flush=True)
    types = [{"P": PERIODIC, "N": NOSLIP, "U": UNSET}[f] for f in faces]
    vel = {f: (0.01 * (f + 1), -0.005 * f, 0.004) for f in range(6) if types[f] == NOSLIP}
    ob, pb = _bc(types, vel, 1.01)
    o = orc.lit_state(q, X, Y, Z)
    orc.lit_init(o, 1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 5, 1e-2), ob)
    with P.State(q, X, Y, Z, "f64", P.LITERAL) as st:
        st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 5, 1e-2), pb)
        st.configure(0.75, (1e-4, 0.0, -2e-5), pb)
        for n in (2, 3, 1, 4):
            orc.lit_run(o, 0.75, (1e-4, 0.0, -2e-5), ob, n)
            st.step(n)
            _same(st, o, n)


@pytest.mark.parametrize("q,X,Y,Z", [(9, 20, 1, 2), (9, 5, 1, 1), (19, 6, 5, 4), (19, 2, 1, 3), (19, 66, 2, 2),
                                     (27, 3, 4, 1)])
@pytest.mark.parametrize("passes", [["UUUUNN"], ["NNUUNN", "UUNNUU"], ["UUUUNU", "UUUUNN", "NNNNNN"],
                                    ["UNNUUU", "UNNUUU"], ["PPUUNN", "UUPPNU"]])
def test_noslip_passes_save_what_they_overwrite(orc, q, X, Y, Z, passes):
    """The values a collision leaves in place, read after one and more no-slip
    passes over the same and other faces, and after the collision or push that
    follows them."""
    bcs = []
    for faces in passes:
        types = [{"P": PERIODIC, "N": NOSLIP, "U": UNSET}[f] for f in faces]
        bcs.append(_bc(types, {f: (0.01 * (f + 1), -0.005 * f, 0.004) for f in range(6) if types[f] == NOSLIP}))
    tau, F = 0.7, (1e-4, -2e-5, 3e-5)
    for end in range(len(passes) + 2):
        print(f"\n[case] literal no-slip passes q={q} {X}x{Y}x{Z} {passes} end {end}", flush=True)
        o = orc.lit_state(q, X, Y, Z)
        orc.lit_init(o, 1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 17, 1e-2), bcs[0][0])
        with P.State(q, X, Y, Z, "f64", P.LITERAL) as st:
            st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 17, 1e-2), bcs[0][1])
            for _ in range(2):
                orc.lit_collide(o, tau, F), st.collide(tau, F)
                orc.lit_push(o), st.stream("push")
                for i, (ob, pb) in enumerate(bcs):
                    if i < end:
                        orc.lit_noslip(o, ob), st.apply_noslip(pb)
                        orc.lit_periodic(o, ob), st.apply_periodicity(pb)
            if end > len(passes):
                orc.lit_collide(o, tau, F), st.collide(tau, F)
                st.synchronize()
            _same(st, o, end)


@pytest.mark.parametrize("q,X,Y,Z", [(9, 20, 1, 6), (19, 6, 5, 4)])
def test_step_that_ends_at_a_face_without_velocity(orc, q, X, Y, Z):
    """A boundary set after plb_configure with a no-slip face that has no
    velocity: the first step ends there, and every field is as the separate
    calls leave it (the faces before it done, ntmp included)."""
    print(f"\n[case] literal step ends early q={q} {X}x{Y}x{Z}", flush=True)
    types = [NOSLIP, NOSLIP, UNSET, UNSET, NOSLIP, NOSLIP]
    vel = {0: (0.01, 0.0, 0.02), 1: (0.0, 0.0, -0.01), 4: (0.05, 0.01, 0.0), 5: (0.0, -0.02, 0.0)}
    ob, pb = _bc(types, vel)
    first = [NOSLIP, NOSLIP, UNSET, UNSET, UNSET, UNSET]  # what is done before the face up
    oe, _ = _bc(first, {f: vel[f] for f in (0, 1)})
    _, bad = _bc(types, {f: vel[f] for f in (0, 1, 5)})
    tau, F = 0.7, (1e-4, -2e-5, 3e-5)
    o = orc.lit_state(q, X, Y, Z)
    orc.lit_init(o, 1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 31, 1e-2), ob)
    orc.lit_run(o, tau, F, ob, 2)
    orc.lit_collide(o, tau, F)
    orc.lit_push(o)
    orc.lit_noslip(o, oe)
    for n in (1, 3):
        with P.State(q, X, Y, Z, "f64", P.LITERAL) as st:
            st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 31, 1e-2), pb)
            st.configure(tau, F, pb)
            st.step(2)
            st.set_boundary(bad)
            with pytest.raises(P.OutOfRange):
                st.step(n)
            _same(st, o, n)
