"""Reads of device fields into host arrays, and reads between steps that leave
the state in the form its steps keep: moments of two- and one-array states at
even and odd step counts against a state that is read only once, whole and
halo'd layouts (the caller's halo stays), both host types; sizes below, at and
above the pieces a read is cut into."""
import numpy as np
import pytest

import plbpd_amd as P
from oracle.pyoracle import Boundary, NOSLIP, PERIODIC

pytestmark = pytest.mark.gpu


def _bc():
    types = [PERIODIC] * 4 + [NOSLIP] * 2
    vel = {P.UP: (0.02, 0.01, 0.0), P.DOWN: (0.0, 0.0, 0.0)}
    return Boundary(type=types, vel=vel, rho_s=1.01), P.boundary(types, vel, 1.01)


@pytest.mark.parametrize("mode", [P.FUSED, P.FUSED_AA])
@pytest.mark.parametrize("q,X,Y,Z,solids", [(9, 7, 1, 5, False), (19, 65, 9, 7, True), (19, 70, 61, 63, True),
                                            (27, 33, 10, 9, False), (27, 64, 8, 5, True)])
@pytest.mark.parametrize("variant", ["f64", "f32s", "f16s"])
def test_moments_between_steps(orc, q, X, Y, Z, solids, variant, mode):
    print(f"\n[case] moments between steps {variant} q={q} {X}x{Y}x{Z} solids={solids} mode={mode}", flush=True)
    ob, pb = _bc()
    mask = (np.random.default_rng(2).random((Z, Y, X)) < 0.15).astype(np.uint8) if solids else None
    tau, F, init = 0.64, (2e-5, 0.0, 1e-6), (P.INIT_PERTURBED, 6, 2e-3)
    o = orc.cor_state(variant, q, X, Y, Z)
    orc.cor_init(o, 1.0, (0.01, 0.0, 0.0), init)
    with P.State(q, X, Y, Z, variant, mode) as st:
        st.set_boundary(pb, mask)
        st.initialize(1.0, (0.01, 0.0, 0.0), init, pb)
        st.configure(tau, F, pb)
        for n in (0, 1, 2, 3, 4):
            orc.cor_run(o, tau, F, ob, n, mask)
            st.step(n)
            orho, ou = orc.cor_moments(o, ob, mask)
            rho, u = st.moments()
            assert np.array_equal(rho, orho) and np.array_equal(u, ou), n
            h = np.full((Z + 2, Y + 2, X + 2, 3), -7.0, np.float32)
            st.download(P.FIELD_U, P.LAYOUT_REFERENCE, out=h)
            assert np.array_equal(h[1:-1, 1:-1, 1:-1], ou.astype(np.float32).reshape(Z, Y, X, 3))
            h[1:-1, 1:-1, 1:-1] = -7.0
            assert (h == -7.0).all()
        gm = st.global_moments()
        rho2, _ = st.moments()
        assert np.array_equal(rho2, rho) and np.isfinite(gm).all()


@pytest.mark.parametrize("cells", [1, 255, 2 ** 16, 2 ** 16 + 1, 2 ** 18 + 77, 1200013])
def test_read_sizes(cells):
    """Populations and density of a row of cells, in every layout and type."""
    pb = P.boundary([P.PERIODIC] * 6, {})
    with P.State(9, cells, 1, 1, "f32", P.LITERAL) as st:
        n = np.random.default_rng(cells).random((3, 3, cells + 2, 9)).astype(np.float32)
        st.upload(P.FIELD_N, n)
        assert np.array_equal(st.download(P.FIELD_N, dtype=np.float32), n)
        assert np.array_equal(st.download(P.FIELD_N, P.LAYOUT_COMPACT), n[1:-1, 1:-1, 1:-1].astype(np.float64))
    with P.State(9, cells, 1, 1, "f64", P.FUSED) as st:
        st.set_boundary(pb)
        c = n[1:-1, 1:-1, 1:-1].astype(np.float64)
        st.upload(P.FIELD_N, c, P.LAYOUT_COMPACT)
        assert np.array_equal(st.download(P.FIELD_N, P.LAYOUT_COMPACT), c)
        assert np.array_equal(st.download(P.FIELD_N, P.LAYOUT_COMPACT, dtype=np.float32), c.astype(np.float32))
        assert np.array_equal(st.download_raw(), c)
        r = np.zeros_like(c[..., 0])
        for k in range(9):  # ascending, as the moments sum
            r += c[..., k]
        assert np.array_equal(st.download(P.FIELD_RHO, P.LAYOUT_COMPACT), r)


@pytest.mark.parametrize("mode", [P.FUSED, P.FUSED_AA])
@pytest.mark.parametrize("how", ["set_boundary", "configure", "reset"])
@pytest.mark.parametrize("q,X,Y,Z", [(9, 40, 1, 9), (19, 33, 10, 9)])
def test_read_after_the_boundary_changed(orc, q, X, Y, Z, how, mode):
    """A read, another boundary and no step, a read: wall cells report the new
    density and velocities, and new solids are solid."""
    print(f"\n[case] read after {how} q={q} {X}x{Y}x{Z} mode={mode}", flush=True)
    ob, pb = _bc()
    types = [PERIODIC] * 4 + [NOSLIP] * 2
    vel = {P.UP: (-0.03, 0.0, 0.0), P.DOWN: (0.01, 0.0, 0.0)}
    ob2, pb2 = Boundary(type=types, vel=vel, rho_s=0.97), P.boundary(types, vel, 0.97)
    mask2 = (np.random.default_rng(2).random((Z, Y, X)) < 0.2).astype(np.uint8) if how == "set_boundary" else None
    tau, F, init = 0.64, (2e-5, 0.0, 1e-6), (P.INIT_PERTURBED, 6, 2e-3)
    o = orc.cor_state("f64", q, X, Y, Z)
    orc.cor_init(o, 1.0, (0.01, 0.0, 0.0), init)
    orc.cor_run(o, tau, F, ob, 5)
    with P.State(q, X, Y, Z, "f64", mode) as st:
        st.set_boundary(pb)
        st.initialize(1.0, (0.01, 0.0, 0.0), init, pb)
        st.configure(tau, F, pb)
        st.step(5)
        for a, e in zip(st.moments(), orc.cor_moments(o, ob)):
            assert np.array_equal(a, e)
        if how == "set_boundary":
            st.set_boundary(pb2, mask2)
        elif how == "configure":
            st.configure(tau, F, pb2)
        else:
            st.reset(pb2)
        for a, e in zip(st.moments(), orc.cor_moments(o, ob2, mask2)):
            assert np.array_equal(a, e)


def test_reads_from_several_threads():
    """One batch's domains, and one state's fields, read by several threads at
    once: each gets what a read by itself gets."""
    from concurrent.futures import ThreadPoolExecutor

    doms = [{"x": 40 + d, "y": 30, "z": 50 - d, "tau": 0.6 + 0.01 * d, "force": (1e-5, 0.0, 0.0)} for d in range(12)]
    b = P.Batch(19, "f32s", doms, P.channel())
    b.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 3, 2e-3))
    b.step(6)
    alone = [b.moments(d) for d in range(len(doms))]
    with ThreadPoolExecutor(6) as pool:
        for _ in range(3):
            for (rho, u), (erho, eu) in zip(pool.map(b.moments, range(len(doms))), alone):
                assert np.array_equal(rho, erho) and np.array_equal(u, eu)
    b.close()
    pb = _bc()[1]
    for mode, fields in ((P.FUSED, (P.FIELD_RHO, P.FIELD_U)), (P.LITERAL, (P.FIELD_RHO, P.FIELD_U, P.FIELD_N))):
        with P.State(19, 60, 50, 40, "f64", mode) as st:
            st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 3, 2e-3), pb)
            st.configure(0.7, (1e-5, 0.0, 0.0), pb)
            st.step(4)
            alone = [st.download(f) for f in fields]
            with ThreadPoolExecutor(6) as pool:
                for f, got in zip(fields * 4, pool.map(st.download, fields * 4)):
                    assert np.array_equal(got, alone[fields.index(f)])
