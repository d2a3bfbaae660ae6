"""What follows a step in one launch (dt / mass reduction and clock, ghost fill in
place, edge ring): GPU == oracle bit for bit with bodies that cross every domain
edge (ring cells copied from ghosts and solids, ghost donors in the ring) and one
inside, for each ghost-fluid variant and cut cells, each edge policy, one and two
stages, and strip heights whose partial records take each of the three reductions
(one wave, one block, folded)."""
import numpy as np
import pytest

from parity_util import gpu_config, nan_equal_bits

pytestmark = pytest.mark.gpu

NX, NY = 200, 520  # 4 strips across: 1, 2 and 8 rows give 2080, 1040 and 260 records


def _phi(c):
    h = c.L / c.N_x  # cell centres are spaced by dx in both directions
    x = -c.num_ghost_cell * h + c.lo_x + h / 2 + np.arange(c.M) * h
    y = -c.num_ghost_cell * h + c.lo_y + h / 2 + np.arange(c.N) * h
    X, Y = np.meshgrid(x, y)
    top = NY * h
    phi = np.full(X.shape, 1e300)
    for cx, cy, r in ((0.0, 0.9, 0.13), (1.0, 1.7, 0.11), (0.4, 0.0, 0.12), (0.7, top, 0.1), (0.5, 1.2, 0.17)):
        phi = np.minimum(phi, np.hypot(X - cx, Y - cy) - r)
    return np.ascontiguousarray(phi.reshape(-1))


CASES = [("IDWBaseGFM", "inflow", "SingleStep"), ("IDWBaseGFM", "periodic", "RK2"), ("LinearBaseGFM", "periodic", "SingleStep"),
         ("RiemannBaseGFM", "pnggeo", "SingleStep"), ("BCGFM", "inflow", "SingleStep"), ("HBCGFM", "periodic", "RK2"),
         ("CutCell", "inflow", "SingleStep"), ("CutCell", "periodic", "SingleStep"), ("IDWBaseGFM", "reference", "SingleStep")]


@pytest.mark.parametrize("boundary,edge,time", CASES)
def test_post_launch_equals_oracle(oracle_mod, boundary, edge, time):
    import ibtfo_amd as ib
    O = oracle_mod
    c = O.Case(N_x=NX, N_y=NY, hi_x=1.0, hi_y=NY / NX, Psy_time=10.0, Scheme="MUSCL", Riemann="HLL", Limiter="VanLeer",
               Boundary=boundary, Time=time, case="uniform", edge=edge, quirks=0,
               extra=dict(rho=1.4, u=0.9, v=0.3, p=1.0))
    c.phi = _phi(c)
    n = 10
    o = O.run_oracle(c, n, root_mode=1)
    assert o["steps"] == n
    for rows, records in ((1, 2080), (2, 1040), (8, 260)):
        print(boundary, edge, time, rows, flush=True)
        s = ib.Solver(gpu_config(c))
        try:
            s.geometry("field", (), phi=c.phi)
            s.initialize("uniform", (1.4, 0.9, 0.3, 1.0))
            s.prepare(c.init_boundary())
            s.set_rows(rows)
            _, nbx, nby = s.tile()
            assert nbx * nby == records
            s.step(n)
            it = s.status()[0]
            d, t, m = s.log(it)
            U = s.state()
        finally:
            s.close()
        assert it == n
        assert nan_equal_bits(U, o["U_OLD"]) == 0, rows
        assert nan_equal_bits(d, o["dt"]) == 0 and nan_equal_bits(t, o["t"]) == 0, rows
        # the oracle sums the mass cell by cell; its own bound
        assert np.allclose(m, o["mass"], rtol=c.M * c.N * 2.0 ** -53, atol=0), rows
