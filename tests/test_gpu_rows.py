"""The row form of the stencils (one launch for the air, the porous layer, the ground plane and
the faces) at the edges of its tiles: rows of 64 points with one, two or no point left over, tile
rows anchored at the high end with one to four rows in the first, the smallest grid, layers on
single faces, and an interior box next to the ring.  Against the FP64
oracle on random smooth fields: the operation order is the oracle's, so the bar is the parity
tests' 1e-10 relative L2; FP32 within 1e-4 of it, the bar of the other FP32 tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    nb = np.linalg.norm(b)
    return np.linalg.norm(a - b) / (nb if nb > 0 else 1.0)


# name: (nx, ny, nz), layer width, faces N S E W F B, porous planes, extras
CASES = {
    "row_of_65": ((65, 11, 12), 3, (2, 1, 2, 2, 2, 2), 0, {}),
    "row_of_64": ((64, 12, 9), 3, (2, 3, 2, 2, 2, 2), 5, {}),
    "row_of_66": ((66, 13, 10), 3, (2, 1, 5, 2, 2, 2), 0, {}),
    "two_tiles": ((128, 14, 9), 3, (2, 3, 5, 2, 2, 2), 5, {}),
    "smallest": ((5, 5, 5), 0, (1, 1, 1, 1, 1, 1), 0, {}),
    "smallest_porous": ((6, 7, 5), 0, (1, 3, 1, 1, 1, 1), 4, {}),
    "single_faces": ((70, 17, 16), 4, (1, 2, 1, 2, 1, 2), 0, {}),
    "other_faces": ((70, 17, 16), 4, (2, 1, 2, 1, 2, 1), 0, {}),
    "interior": ((200, 37, 22), 5, (2, 3, 2, 2, 2, 2), 6, {}),
    "interior_terrain": ((200, 38, 23), 5, (2, 3, 2, 2, 2, 2), 6, {"hills": [(0.2, 0.8, 0.08, 0.5)]}),
    "interior_rigid": ((192, 39, 18), 4, (1, 1, 1, 1, 1, 1), 0, {}),
}


def deck_of(lee, name, scheme):
    (nx, ny, nz), pml, bc, pore, more = CASES[name]
    if scheme == "rk4":  # the East impedance boundary is defined for FB only
        bc = tuple(2 if b == 5 else b for b in bc)
    more = dict(more)
    hills = more.pop("hills", ())
    d = lee.deck.box(nx, ny, nz, 0.05, pml=pml, bc=bc, porous_cells=pore, src=(0.0, 0.4, 0.2), gauss_width=0.25,
                     pml_y_time=2, time_domain=40, **more)
    d.hills = list(hills)
    if scheme == "rk4":
        d.integrator, d.velocity_method, d.wind_ustar, d.wind_z0 = 1, 7, 0.3, 0.02
    return d


def start_state(d, rng):
    out = []
    for _ in range(4):
        f = 1.0
        for n in d.shape[::-1]:
            f = np.multiply.outer(f, np.cos(rng.uniform(1.0, 4.0) * np.arange(n) / n + rng.uniform(0, 6)))
        out.append(f)
    return [out[0] * 1e-3, out[1] * 1e-3, out[2] * 1e-3, out[3]]


def receivers(d, rng, n=7):
    return [(d.air_x[rng.integers(1, d.shape[0] - 1)], d.air_y[rng.integers(1, d.shape[1] - 1)],
             d.air_z[rng.integers(1, d.shape[2] - 1)]) for _ in range(n)]


@pytest.mark.parametrize("scheme", ["fb", "rk4"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_rows_match_the_oracle(lee, orc, name, scheme):
    d = deck_of(lee, name, scheme)
    rng = np.random.default_rng(sum(map(ord, name)))
    rec, x0 = receivers(d, rng), start_state(d, rng)
    o = orc.Oracle(d, receivers=rec)
    o.frame_setup(0)
    o.set_state(*x0)
    ref = np.concatenate([o.step(6), o.step(7)])
    for prec, bar in ((64, 1e-10), (32, 1e-4)):
        print(f"[gpu rows] {scheme} fp{prec} {name} {d.shape}", flush=True)
        s = lee.Solver(d, precision=prec, receivers=rec)
        s.frame_setup(0)
        s.set_state(*x0)
        got = np.concatenate([s.step(6), s.step(7)])
        assert rel(got, ref) <= bar
        for a, b in zip(s.state(), o.state()):
            assert rel(a, b) <= bar
        if d.has_pore:
            for a, b in zip(s.state(1), o.state(1)):
                assert rel(a, b) <= bar
        s.close()
