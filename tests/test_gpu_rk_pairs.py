"""RK4 with the interior's stages two per launch (rk_tile 6) against the whole domain in one launch
per stage (rk_tile 1): the same bits in the fields and the series over odd and even numbers of
steps.  Interiors whose points do not divide into blocks, rows or tiles, from the smallest that
takes the form; layers on some faces or none; each kind of mean flow, flat and over a hill, with and
without a porous layer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# name: (nx, ny, nz), layer width, faces N S E W F B, porous points, hill, flow
CASES = {
    "smallest": ((132, 24, 14), 0, (1, 1, 1, 1, 1, 1), 0, 0, 0),
    "layers": ((213, 71, 45), 7, (2, 3, 2, 2, 2, 2), 6, 1, 7),
    "layers_flat": ((190, 64, 40), 6, (2, 3, 2, 2, 2, 2), 6, 0, 7),
    "no_flow": ((201, 53, 37), 6, (2, 1, 2, 2, 2, 2), 0, 1, 0),
    "three_component_flow": ((170, 49, 33), 5, (2, 1, 2, 2, 2, 2), 0, 0, 5),
    "three_component_hill": ((171, 48, 32), 5, (2, 1, 2, 2, 2, 2), 0, 1, 5),
    "one_sided": ((257, 47, 29), 9, (2, 1, 1, 2, 1, 2), 0, 0, 0),
    "other_side": ((260, 50, 31), 9, (1, 3, 2, 1, 2, 1), 5, 1, 7),
    "deep": ((150, 33, 130), 4, (2, 1, 2, 2, 2, 2), 0, 0, 7),
}


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("name", sorted(CASES))
def test_pairs_equal_single_stages(lee, name, prec):
    shape, pml, bc, pore, hill, flow = CASES[name]
    d = lee.deck.box(*shape, 0.05, pml=pml, bc=bc, porous_cells=pore, src=(0.0, 0.6, 0.4), gauss_width=0.25, time_domain=40,
                     pml_y_time=0)
    d.integrator = 1
    if hill:
        d.hills = [(0.2, 1.0, 0.07, 0.6)]
    if flow:
        d.velocity_method, d.velocity_coef = flow, 3.0
        if flow == 7:
            d.wind_ustar, d.wind_z0 = 0.3, 0.02
    rng = np.random.default_rng(sum(map(ord, name)))
    x0 = []
    for s in (1e-3, 1e-3, 1e-3, 1.0):
        f = s
        for n in shape[::-1]:
            f = np.multiply.outer(f, np.cos(rng.uniform(1.0, 4.0) * np.arange(n) / n * 6 + rng.uniform(0, 6)))
        x0.append(f)
    rec = [(d.air_x[rng.integers(1, shape[0] - 1)], d.air_y[rng.integers(1, shape[1] - 1)], d.air_z[rng.integers(1, shape[2] - 1)])
           for _ in range(9)]
    out = []
    for tile, graph in ((1, False), (6, False), (6, True)):
        print(f"[gpu rk pairs] fp{prec} {name} tile {tile} graph {graph}", flush=True)
        s = lee.Solver(d, precision=prec, receivers=rec, rk_tile=tile, use_graph=graph)
        s.frame_setup(0)
        s.set_state(*x0)
        got = []
        for n in (1, 2, 3, 1):
            got.append(s.step(n))
            got += list(s.state()) + (list(s.state(1)) if pore else [])
        s.close()
        out.append(got)
    for got in out[1:]:
        for a, b in zip(out[0], got):
            assert np.isfinite(a).all()
            assert np.array_equal(a, b)
