"""Device layouts of a literal state: rows of whole lines (the default), rows of
X + 2 cells with shifted arrays (where whole lines would cost a large state too
much), and the packed form (pop_pad = 0, large thin states, and when memory is
short).  The same values in each, ntmp included, over staged calls, whole steps,
uploads and reads; and the memory that each takes."""
import numpy as np
import pytest

import plbpd_amd as P

pytestmark = pytest.mark.gpu

FIELDS = (P.FIELD_N, P.FIELD_RHO, P.FIELD_U, P.FIELD_NTMP)


def _bc(faces):
    types = [{"P": P.PERIODIC, "N": P.NOSLIP, "U": P.UNSET}[f] for f in faces]
    return P.boundary(types, {f: (0.01 * (f + 1), -0.005 * f, 0.004) for f in range(6) if types[f] == P.NOSLIP}, 1.01)


def _staged(st, pb, tau, F):
    st.collide(tau, F)
    st.stream("push")
    st.apply_noslip(pb)
    st.apply_periodicity(pb)
    st.calc_moments()
    st.reset(pb)


@pytest.mark.parametrize("faces", ["PPPPNN", "NNPPNN", "PPUUUU", "NNNNNN"])
@pytest.mark.parametrize("q,X,Y,Z,prec", [(9, 70, 1, 9, "f64"), (19, 17, 5, 4, "f32"), (19, 1, 3, 6, "f64"),
                                          (19, 300, 4, 3, "f64"), (27, 66, 6, 1, "f32"), (27, 13, 9, 7, "f64")])
def test_packed_layout(q, X, Y, Z, prec, faces):
    print(f"\n[case] packed literal layout q={q} {X}x{Y}x{Z} {prec} {faces}", flush=True)
    pb, tau, F = _bc(faces), 0.7, (1e-4, -2e-5, 3e-5)
    with P.State(q, X, Y, Z, prec, P.LITERAL) as a, P.State(q, X, Y, Z, prec, P.LITERAL, pop_pad=0) as b:
        cells = (X + 2) * (Y + 2) * (Z + 2)
        assert b.nbytes() == (2 * q + 4) * cells * (8 if prec == "f64" else 4) < a.nbytes()
        for st in (a, b):
            st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 5, 1e-2), pb)
            st.configure(tau, F, pb)

        def same(where):
            for f in FIELDS:
                assert np.array_equal(a.download(f), b.download(f)), (where, f)
            assert np.array_equal(a.global_moments(), b.global_moments()), where

        for st in (a, b):
            for _ in range(3):
                _staged(st, pb, tau, F)
        same("staged")
        for n in (1, 4):
            a.step(n), b.step(n)
            same(n)
        n = np.random.default_rng(4).random((Z + 2, Y + 2, X + 2, q))
        for st in (a, b):
            st.collide(tau, F)
            st.stream("push")
            st.apply_noslip(pb)
            st.upload(P.FIELD_N, n)
            st.upload(P.FIELD_NTMP, n[::-1])
        same("uploads")
        for st in (a, b):
            _staged(st, pb, tau, F)
        same("staged after uploads")


def test_large_states_take_little_more_than_the_packed_form():
    """Above 1 GiB a buffer: rows of X + 2 cells where whole lines would take more
    than an eighth, the packed form where the shift's planes would."""
    for q, X, Y, Z, prec, form in ((27, 10, 300, 1030, "f64", "rows"), (19, 1600, 1600, 1, "f64", "packed"),
                                   (19, 200, 200, 190, "f64", "lines")):
        with P.State(q, X, Y, Z, prec, P.LITERAL, pop_pad=0) as b:
            least = b.nbytes()
        with P.State(q, X, Y, Z, prec, P.LITERAL) as a:
            more = a.nbytes() / least
        assert {"rows": 1.0 < more < 1.01, "packed": more == 1.0, "lines": 1.02 < more <= 1.125}[form], (X, Y, Z, more)


def test_shifted_rows_of_a_large_state():
    q, X, Y, Z, pb = 27, 10, 300, 1030, _bc("PPPPNN")
    print(f"\n[case] shifted literal rows q={q} {X}x{Y}x{Z}", flush=True)
    out = []
    for pad in (-1, 0):
        with P.State(q, X, Y, Z, "f64", P.LITERAL, pop_pad=pad) as st:
            st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 5, 1e-2), pb)
            st.configure(0.7, (1e-4, -2e-5, 3e-5), pb)
            st.step(3)
            _staged(st, pb, 0.7, (1e-4, -2e-5, 3e-5))
            out.append([st.download(f, P.LAYOUT_COMPACT, dtype=np.float32) for f in (P.FIELD_N, P.FIELD_NTMP)]
                       + list(st.moments()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
