"""A process whose first step kernels are launched while a stream captures: by the library's
own step graph, and by a caller's capture of ibtfo_step. The state is that of plainly
launched steps, bit for bit, for the row-parallel and the marching kernels."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = r"""
import ctypes as C, sys
sys.path.insert(0, sys.argv[1])
import torch
import ibtfo_amd as ib
n, mode = int(sys.argv[2]), sys.argv[3]
cfg = ib.config(N_x=n, N_y=n // 2, hi_x=2.0, hi_y=1.0, Psy_time=10.0, max_iter=10 ** 6, Scheme="MUSCL", Riemann="HLL",
                Limiter="VanLeer", Boundary="IDWBaseGFM", quirks=0, Edge="inflow", edge_state=(1.4, 3.0, 0.0, 1.0))

def solve(capture):
    s = ib.Solver(cfg)
    s.geometry("ellipse", (0.6, 0.5, 0.12, 0.06, 20.0))
    s.initialize("uniform", (1.4, 3.0, 0.0, 1.0))
    stream = torch.cuda.Stream()
    if capture == "own":
        assert ib.lib().ibtfo_set_stream(s.h, C.c_void_p(stream.cuda_stream)) == 0
    s.prepare(True)
    if capture == "graph":
        for _ in range(3):
            s.step(4, graph_chunk=4)
    elif capture == "own":
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            s.step(4)
        for _ in range(3):
            with torch.cuda.stream(stream):
                g.replay()
    else:
        s.step(12)
    out = s.status()[:3], s.state(), s.tile_form()
    s.close()
    return out

got, want = solve(mode), solve("plain")
assert got[0] == want[0] and got[0][0] == 12, (got[0], want[0])
assert (got[1] == want[1]).all()
print("first launch ok", n, mode, "row-parallel" if got[2] else "marching", flush=True)
"""


@pytest.mark.parametrize("n,form", [(64, "row-parallel"), (1500, "marching")])
@pytest.mark.parametrize("mode", ["graph", "own"])
def test_first_step_kernels_under_capture(n, form, mode):
    print("first launch", n, mode, flush=True)
    r = subprocess.run([sys.executable, "-c", SCRIPT, ROOT, str(n), mode], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "first launch ok %d %s %s" % (n, mode, form) in r.stdout, r.stdout + r.stderr[-2000:]
