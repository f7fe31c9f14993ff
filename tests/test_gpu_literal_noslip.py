"""The in-place no-slip pass of a literal state (one launch per axis where the
axis has three layers or more, else one per face) against the oracle's serial
loop, bit for bit: every axis walled with a velocity of its own on each face,
axes of one to five layers (faces that share a layer, write into each other's
layer, or lie apart), and faces of more cells than a workgroup."""
import numpy as np
import pytest

import plbpd_amd as P
from oracle.pyoracle import Boundary, NOSLIP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("q,X,Y,Z", [(9, 1, 1, 3), (9, 300, 1, 2), (9, 4, 3, 3), (19, 2, 2, 2), (19, 3, 3, 3),
                                     (19, 2, 5, 3), (19, 23, 19, 4), (27, 3, 2, 4), (27, 1, 4, 3), (27, 17, 21, 3)])
def test_noslip_in_place_equals_serial_order(orc, q, X, Y, Z, prec):
    print(f"\n[case] literal no-slip q={q} {X}x{Y}x{Z} {prec}", flush=True)
    dt = np.float64 if prec == "f64" else np.float32
    vel = {f: (0.01 * (f + 1), -0.004 * f, 0.002) for f in range(6)}
    ob, pb = Boundary(type=[NOSLIP] * 6, vel=vel, rho_s=1.01), P.boundary([P.NOSLIP] * 6, vel, 1.01)
    o = orc.lit_state(q, X, Y, Z, dt)
    orc.lit_init(o, 1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 41, 1e-2), ob)
    with P.State(q, X, Y, Z, prec, P.LITERAL) as st:
        st.initialize(1.0, (0.01, 0.0, 0.0), (P.INIT_PERTURBED, 41, 1e-2), pb)
        for _ in range(2):
            orc.lit_collide(o, 0.7, (1e-4, 0.0, 2e-5))
            orc.lit_push(o)
            assert orc.lit_noslip(o, ob) == 0
            st.collide(0.7, (1e-4, 0.0, 2e-5))
            st.stream("push")
            st.apply_noslip(pb)
            assert np.array_equal(st.download(P.FIELD_N, dtype=dt), o["n"])
            assert np.array_equal(st.download(P.FIELD_NTMP, dtype=dt), o["ntmp"])
