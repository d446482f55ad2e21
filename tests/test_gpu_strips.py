"""Blocks that take several rows per wavefront -- a row's narrow last tile, the columns an
interior leaves of the outer tiles -- against the FP64 oracle: one to 32 rows a wave, rows and
planes that do not divide into blocks, with and without x and z layers, terrain, wind and a porous
layer, and the first width past the strips'.  The bars are those of the other parity tests: 1e-10
relative L2 in FP64, 1e-4 in FP32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# name: (nx, ny, nz), layer width, faces N S E W F B, porous points, hill, rk_tile
CASES = {
    "tail_2": ((66, 45, 14), 4, (2, 1, 2, 2, 2, 2), 0, 0, 1),
    "tail_2_shifted": ((65, 44, 13), 4, (2, 3, 2, 2, 2, 2), 5, 1, 1),
    "tail_3": ((67, 71, 12), 5, (2, 1, 2, 2, 2, 2), 0, 1, 1),
    "tail_9": ((137, 41, 11), 6, (2, 3, 2, 2, 2, 2), 5, 1, 1),
    "tail_21": ((85, 46, 12), 5, (2, 1, 2, 2, 2, 2), 0, 0, 1),
    "tail_22": ((86, 43, 12), 5, (2, 1, 2, 2, 2, 2), 0, 0, 1),
    "tail_without_layers": ((70, 38, 10), 0, (1, 1, 1, 1, 1, 1), 0, 0, 1),
    "interior": ((152, 61, 23), 6, (2, 3, 2, 2, 2, 2), 5, 1, 6),
    "interior_wide": ((198, 63, 24), 26, (1, 1, 1, 1, 2, 2), 0, 0, 6),
    "interior_one_side": ((150, 58, 21), 7, (2, 1, 1, 1, 2, 1), 0, 1, 6),
    "interior_two_tiles": ((138, 57, 22), 4, (2, 1, 1, 2, 1, 2), 0, 0, 6),
}


def rel(a, b):
    nb = np.linalg.norm(b)
    return np.linalg.norm(a - b) / (nb if nb > 0 else 1.0)


def _check(lee, orc, name, rk4):
    shape, pml, bc, pore, hill, tile = CASES[name]
    if not rk4:
        bc = bc[:2] + (5,) + bc[3:] if bc[2] == 2 and not hill and not pore else bc  # the East impedance as well
    d = lee.deck.box(*shape, 0.05, pml=pml, bc=bc, porous_cells=pore, src=(0.0, 0.6, 0.3), gauss_width=0.25, time_domain=40,
                     pml_y_time=0)
    if rk4:
        d.integrator, d.velocity_method, d.wind_ustar, d.wind_z0 = 1, 7, 0.3, 0.02
    if hill:
        d.hills = [(0.1, 0.9, 0.05, 0.5)]
    rng = np.random.default_rng(sum(map(ord, name)))
    x0 = []
    for s in (1e-3, 1e-3, 1e-3, 1.0):
        f = s
        for n in shape[::-1]:
            f = np.multiply.outer(f, np.cos(rng.uniform(1.0, 4.0) * np.arange(n) / n + rng.uniform(0, 6)))
        x0.append(f)
    rec = [(d.air_x[rng.integers(1, shape[0] - 1)], d.air_y[rng.integers(1, shape[1] - 1)], d.air_z[rng.integers(1, shape[2] - 1)])
           for _ in range(9)]
    o = orc.Oracle(d, receivers=rec)
    o.frame_setup(0)
    o.set_state(*x0)
    ref = np.concatenate([o.step(3), o.step(4)])
    for prec, bar in ((64, 1e-10), (32, 1e-4)):
        print(f"[gpu strips] {'rk4' if rk4 else 'fb'} fp{prec} {name}", flush=True)
        s = lee.Solver(d, precision=prec, receivers=rec, **(dict(rk_tile=tile) if rk4 else dict(fb_form=1 if tile == 6 else 0)))
        s.frame_setup(0)
        s.set_state(*x0)
        got = np.concatenate([s.step(3), s.step(4)])
        assert rel(got, ref) <= bar
        for a, b in zip(s.state(), o.state()):
            assert rel(a, b) <= bar
        if pore:
            for a, b in zip(s.state(1), o.state(1)):
                assert rel(a, b) <= bar
        s.close()


@pytest.mark.parametrize("name", sorted(CASES))
def test_strips_match_the_oracle(lee, orc, name):
    _check(lee, orc, name, True)


@pytest.mark.parametrize("name", sorted(n for n in CASES if n.startswith("tail")))
def test_fb_strips_match_the_oracle(lee, orc, name):
    _check(lee, orc, name, False)
