"""The default tile: row-parallel on small grids with the fewest rows that leave at
most one block per CU (256), else two (512), 7-row strips up to 1024 blocks,
marching strips beyond and for Lax; rows = 0 restores it; the state is the marching
strip's bit for bit."""
import numpy as np
import pytest

from parity_util import nan_equal_bits

pytestmark = pytest.mark.gpu

# (N_x, N_y, rows, row-parallel): the smallest grid, the edges of 256, 512 and 1024
# blocks, ragged last strips, the marching heights
SIZES = [(4, 4, 1, True), (60, 256, 1, True), (60, 257, 2, True), (400, 100, 3, True), (60, 1792, 7, True),
         (60, 1793, 4, True), (512, 256, 5, True), (60, 3584, 7, True), (60, 3585, 7, True), (60, 7168, 7, True),
         (60, 7169, 3, False), (1000, 901, 6, False), (1483, 1484, 8, False)]


@pytest.mark.parametrize("nx,ny,rows,par", SIZES)
def test_default_tile(nx, ny, rows, par):
    import ibtfo_amd as ib
    cfg = ib.config(N_x=nx, N_y=ny, hi_x=1.0, hi_y=ny / nx, Psy_time=10.0, max_iter=10 ** 6, Scheme="MUSCL",
                    Riemann="HLL", Limiter="minmod", Boundary="Regular")
    out = []
    for mode in ("default", "restored", "march"):
        s = ib.Solver(cfg)
        try:
            s.geometry("none")
            s.initialize("sod_x", (0.5, 1, 0, 0, 1, 0.125, 0, 0, 0.1))
            s.prepare(False)
            if mode != "default":
                s.set_rows(4)
            if mode == "restored":
                s.set_rows(0)
            if mode != "march":
                assert s.tile()[0] == rows and s.tile_form() == par
            s.step(4)
            out.append((s.state(), s.status()[:3]))
        finally:
            s.close()
    for U, clock in out[:2]:
        assert clock == out[2][1] and np.isfinite(U).all()
        assert nan_equal_bits(U, out[2][0]) == 0


def test_default_tile_lax():
    import ibtfo_amd as ib
    s = ib.Solver(ib.config(N_x=60, N_y=40, hi_x=1.0, hi_y=40 / 60, Scheme="Lax", Boundary="Regular"))
    try:
        assert not s.tile_form() and s.tile()[0] == 3
    finally:
        s.close()
