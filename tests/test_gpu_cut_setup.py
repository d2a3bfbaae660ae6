"""Ghost, cut-cell and merge-group lists at the edges of the tiles they are gathered
by (64 x 32 cells): random level sets of a few whole values, so that corners vanish
exactly, small cells lack a partner and full cells get a closed face, and one without
any cut cell; types, counts and the first steps == the oracle bit for bit."""
import numpy as np
import pytest

from parity_util import gpu_config, nan_equal_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,solid", [(64, 32, 0.3), (63, 31, 0.5), (65, 33, 0.1), (130, 65, 0.02), (96, 40, 0.0),
                                         (64, 64, 0.9)])
def test_cut_lists_equal_oracle(oracle_mod, nx, ny, solid):
    import ibtfo_amd as ib
    O = oracle_mod
    c = O.Case(N_x=nx, N_y=ny, hi_x=1.0, hi_y=ny / nx, Psy_time=10.0, Scheme="MUSCL", Riemann="HLL",
               Limiter="VanLeer", Boundary="CutCell", Time="SingleStep", case="uniform", edge="inflow", quirks=0,
               extra=dict(rho=1.4, u=0.2, v=0.1, p=1.0))
    rng = np.random.default_rng(nx)
    phi = np.where(rng.random(c.M * c.N) < solid, -1.0, 1.0) * rng.integers(0 if solid else 1, 3, c.M * c.N)
    c.phi = np.ascontiguousarray(phi)
    st = O.setup(c)
    types = st["XY"][5::6].reshape(c.N, c.M)
    cut = st["cut"].reshape(c.N, c.M, 8)
    inner = np.s_[2:-2, 2:-2]
    into = cut[..., 7][types == 3]
    n = 3
    print("cut lists %dx%d" % (nx, ny), flush=True)
    s = ib.Solver(gpu_config(c))
    try:
        s.geometry("field", (), phi=c.phi)
        assert nan_equal_bits(s.xycoord()[5::6], st["XY"][5::6]) == 0
        assert s.cut_counts() == (int((types == 3).sum()), len(np.unique(into[into >= 0])))
        assert s.num_ghosts() == int((types[inner] == 2).sum())
        s.initialize("uniform", (1.4, 0.2, 0.1, 1.0))
        s.prepare(True)
        s.step(n)
        U = s.state()
    finally:
        s.close()
    assert nan_equal_bits(U, O.run_oracle(c, n, root_mode=1)["U_OLD"]) == 0
