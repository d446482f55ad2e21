"""Several FB_p_v steps per launch over narrow columns against the same steps by one launch per
phase (a named launch form): the same arithmetic on the same values, so fields, auxiliaries
(through later steps), impedance histories and receiver series are equal bit for bit.  Planes
from the smallest to 64 nodes, columns within one workgroup's window and across many, the
interface at every distance from a window's edge (porous depths), layers at the top, at both
ends and at neither, step counts around a launch's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# name: (nx, ny, nz), faces N S E W F B, porous points (0: none), layer width, poles
CASES = {
    "porous": ((6, 6, 150), (2, 3, 1, 1, 1, 1), 12, 20, 0),
    "porous_thin": ((6, 6, 90), (2, 3, 1, 1, 1, 1), 4, 8, 0),
    "porous_deep": ((6, 6, 70), (1, 3, 1, 1, 1, 1), 35, 0, 0),
    "porous_5": ((5, 6, 61), (2, 3, 1, 1, 1, 1), 5, 7, 0),
    "rigid": ((6, 6, 300), (2, 1, 1, 1, 1, 1), 0, 20, 0),
    "both_ends": ((6, 6, 64), (2, 2, 1, 1, 1, 1), 0, 9, 0),
    "ground": ((6, 6, 140), (2, 1, 1, 1, 1, 1), 0, 20, 8),
    "ground_one_pole": ((7, 5, 33), (2, 1, 1, 1, 1, 1), 0, 6, 1),
    "plane_64": ((8, 8, 120), (2, 3, 1, 1, 1, 1), 9, 10, 0),
    "plane_63": ((9, 7, 77), (2, 1, 1, 1, 1, 1), 0, 10, 3),
    "smallest": ((5, 5, 5), (1, 1, 1, 1, 1, 1), 0, 0, 0),
    "smallest_porous": ((5, 6, 5), (1, 3, 1, 1, 1, 1), 4, 0, 0),
    "long": ((6, 6, 1500), (2, 3, 1, 1, 1, 1), 10, 20, 0),
}


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("name", sorted(CASES))
def test_columns_equal_single_steps(lee, name, prec):
    shape, bc, pore, pml, poles = CASES[name]
    d = lee.deck.box(*shape, 0.04, pml=pml, bc=bc, porous_cells=pore, src=(0.0, 0.1, 0.5), gauss_width=0.3, time_domain=200)
    if poles:
        d.ground_poles = [(0.3 / (q + 1), 0.2 * q) for q in range(poles)]
        d.ground_zinf, d.ground_tau = 900.0, 1e-4
    rng = np.random.default_rng(sum(map(ord, name)))
    x0 = [rng.normal(size=shape[::-1]) * s for s in (1e-3, 1e-3, 1e-3, 1.0)]
    rec = [(d.air_x[rng.integers(0, shape[0])], d.air_y[rng.integers(0, shape[1])], d.air_z[rng.integers(0, shape[2])])
           for _ in range(40)] + [(d.air_x[1], d.air_y[-1], d.air_z[z]) for z in (0, 1, shape[2] // 2, shape[2] - 1)]
    out = []
    for form in (1, 0):
        print(f"[gpu columns] fp{prec} {name} form {form}", flush=True)
        s = lee.Solver(d, precision=prec, receivers=rec, fb_form=form, use_graph=form == 0 and pore > 0)
        s.frame_setup(0)
        s.set_state(*x0)
        got = []
        for n in (1, 2, 7, 8, 9, 10, 11, 41, 64):
            got.append(s.step(n))
            got += list(s.state()) + (list(s.state(1)) if pore else [])
        if poles:
            got.append(s.ground_psi())
        s.close()
        out.append(got)
    assert len(out[0]) == len(out[1])
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
