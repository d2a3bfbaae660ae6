"""The default tile of FP64 cut-cell and Steger-Warming grids at the edges of its rule
(7-row blocks up to 2200), whose partial records also take the post kernel's one-block
(513 to 1024 records) and folded (more) reductions; the state and clock are the
marching strip's bit for bit. The marching heights of the largest grids."""
import numpy as np
import pytest

from parity_util import nan_equal_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("boundary,riemann,precision,ny,rows,par", [
    ("CutCell", "HLL", "FP64", 4200, 7, True), ("CutCell", "HLL", "FP64", 7168, 7, True),
    ("CutCell", "HLL", "FP64", 15400, 7, True), ("CutCell", "HLL", "FP64", 15401, 6, False),
    ("IDWBaseGFM", "StegerWarming", "FP64", 7175, 7, True), ("Regular", "StegerWarming", "FP64", 15400, 7, True),
    ("CutCell", "HLL", "mixed", 7169, 3, False), ("IDWBaseGFM", "HLL", "FP64", 7169, 3, False)])
def test_default_tile(boundary, riemann, precision, ny, rows, par):
    import ibtfo_amd as ib
    cfg = ib.config(N_x=60, N_y=ny, hi_x=1.0, hi_y=ny / 60, Psy_time=10.0, max_iter=10 ** 6, Scheme="MUSCL",
                    Riemann=riemann, Limiter="VanLeer", Boundary=boundary, Precision=precision, quirks=0, Edge="inflow",
                    edge_state=(1.4, 0.9, 0.2, 1.0))
    prm = [3.0]
    for cx, cy, r in ((0.5, 3.0, 0.21), (0.3, ny / 120, 0.17), (0.6, ny / 60 - 0.4, 0.2)):
        prm += [0.0, cx, cy, r] + [0.0] * 17
    out = []
    for mode in ("default", "march"):
        print(boundary, riemann, precision, ny, mode, flush=True)
        s = ib.Solver(cfg)
        try:
            s.geometry("none") if boundary == "Regular" else s.geometry("shapes", prm)
            s.initialize("uniform", (1.4, 0.6, 0.1, 1.0))
            s.prepare(boundary != "Regular")
            if mode == "march":
                s.set_rows(33)
            else:
                assert s.tile()[0] == rows and s.tile_form() == par
            s.step(5)
            out.append((s.state(), s.status()[:3]))
        finally:
            s.close()
    assert out[0][1] == out[1][1] and np.isfinite(out[0][0]).all()
    assert nan_equal_bits(out[0][0], out[1][0]) == 0


@pytest.mark.parametrize("nx,ny,rows", [(2645, 2646, 8), (2646, 2646, 10), (3464, 3464, 10), (3465, 3464, 12)])
def test_default_marching_height(nx, ny, rows):
    import ibtfo_amd as ib
    s = ib.Solver(ib.config(N_x=nx, N_y=ny, hi_x=1.0, hi_y=ny / nx, Scheme="MUSCL", Riemann="HLL", Boundary="Regular"))
    try:
        assert not s.tile_form() and s.tile()[0] == rows
    finally:
        s.close()
