"""A solve given one geometry after another, whose records take more, less and no
memory than the last's (a context keeps it for the next): each equals the same
geometry in a fresh context bit for bit, lists, types, normals and some steps."""
import numpy as np
import pytest

from parity_util import nan_equal_bits

pytestmark = pytest.mark.gpu

SHAPES = {"one": ("shapes", [(0.9, 0.5, 0.05)]), "many": ("shapes", [(0.2 + 0.3 * k, 0.5, 0.13) for k in range(5)]),
          "none": ("shapes", [(9.0, 9.0, 0.1)]), "mask": ("mask", 1), "fine": ("mask", 5)}


def _set(s, what):
    kind, v = SHAPES[what]
    if kind == "shapes":
        prm = [float(len(v))]
        for cx, cy, r in v:
            prm += [0.0, cx, cy, r] + [0.0] * 17
        s.geometry("shapes", prm)
        return
    img = np.full((52 * v, 132 * v, 4), 255, np.uint8)  # v = 5: more pixels than the planes hold
    y, x = np.mgrid[: 52 * v, : 132 * v]
    img[(x - 40 * v) ** 2 + (y - 25 * v) ** 2 < (9 * v) ** 2, :3] = 0
    s.geometry_mask(img)


def _result(s):
    s.initialize("uniform", (1.4, 0.6, 0.1, 1.0))
    s.prepare(True)
    s.step(4, graph_chunk=2)
    s.step(3)
    assert s.status()[0] == 7
    return s.num_ghosts(), s.cut_counts(), s.xycoord(), s.state()


@pytest.mark.parametrize("boundary", ["CutCell", "IDWBaseGFM", "SimpleBound"])
def test_next_geometry_equals_a_fresh_context(boundary):
    import ibtfo_amd as ib
    cfg = ib.config(N_x=128, N_y=48, lo_x=0.0, lo_y=0.0, hi_x=2.0, hi_y=0.75, Boundary=boundary, quirks=0,
                    Psy_time=10.0, Edge="inflow", edge_state=(1.4, 0.6, 0.1, 1.0), Scheme="MUSCL", Riemann="HLL", Limiter="VanLeer")
    s = ib.Solver(cfg)
    try:
        for what in ("one", "many", "mask", "none", "fine", "one"):
            print(boundary, what, flush=True)
            _set(s, what)
            got = _result(s)
            f = ib.Solver(cfg)
            try:
                _set(f, what)
                want = _result(f)
            finally:
                f.close()
            assert got[:2] == want[:2]
            assert nan_equal_bits(got[2], want[2]) == 0 and nan_equal_bits(got[3], want[3]) == 0, what
    finally:
        s.close()
