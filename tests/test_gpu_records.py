"""The step's partial records at the edges of their reductions (one, two, four and
eight per lane of one wave, one per thread of a block, several): a one-strip-wide
x-Sod whose height is the number of records, marching and row-parallel, eager and
replayed from graphs of an odd number of steps (whose first rows are then read from
the other buffer than at the capture): GPU == oracle bit for bit."""
import pytest

from parity_util import gpu_config, gpu_hooks, nan_equal_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limiter,quirks", [("minmod", 1), ("VanLeer", 0)])
@pytest.mark.parametrize("ny", [64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025])
def test_record_counts_equal_oracle(oracle_mod, ny, limiter, quirks):
    import ibtfo_amd as ib
    O = oracle_mod
    c = O.Case(N_x=24, N_y=ny, hi_x=1.0, hi_y=ny / 24, Scheme="MUSCL", Riemann="HLL", Limiter=limiter, quirks=quirks,
               case="sodx", Psy_time=10.0)
    n = 9
    o = O.run_oracle(c, n, root_mode=1)
    assert o["steps"] == n
    ls, init = gpu_hooks(c)
    for par in (0, 1):
        for chunk in (0, 3):
            print(ny, limiter, par, chunk, flush=True)
            s = ib.Solver(gpu_config(c))
            try:
                s.geometry(*ls)
                s.initialize(*init)
                s.prepare(False)
                s.set_tile(1, par)
                assert s.tile()[1] * s.tile()[2] == ny
                s.step(n, chunk)
                it, t, _, _ = s.status()
                d, tl, _ = s.log(it)
                U = s.state()
            finally:
                s.close()
            assert it == n
            assert nan_equal_bits(U, o["U_OLD"]) == 0, (par, chunk)
            assert nan_equal_bits(d, o["dt"]) == 0 and nan_equal_bits(tl, o["t"]) == 0, (par, chunk)
