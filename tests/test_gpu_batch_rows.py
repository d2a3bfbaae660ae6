"""A batch that leaves the strip height open, on both sides of the rule that picks it
(8 rows from 8192 step blocks on, 16 below and for a solve that only fits so): every
request equals the same solve alone bit for bit; one that fits with neither is refused."""
import pytest

from parity_util import nan_equal_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks,nx,ny", [(8191, 512, 256), (8192, 512, 256), (8192, 250, 133), (8192, 3840, 1100),
                                          (8832, 3840, 1100)])
def test_default_rows_equal_alone(blocks, nx, ny):
    from ibtfo_amd import serving as S
    st = S.ellipse_stream(n=1, seed=5, steps=4)
    st[0].update(N_x=nx, N_y=ny, L=nx / ny)
    st[0]["ellipse"] = (0.3 * nx / ny, 0.5) + tuple(st[0]["ellipse"][2:])
    item = S.ellipse_items(st, precision="FP64", keep_state=True)[0]
    print("batch default rows", blocks, nx, ny, flush=True)
    b = S.Batch(S.batch_config(Scheme="MUSCL", Riemann="HLL", Limiter="VanLeer", Boundary="IDWBaseGFM",
                               Precision="FP64", quirks=0, hbm_budget=2 << 30, max_slots=2, max_step_blocks=blocks,
                               max_ghost_blocks=4096, max_ring_blocks=1024, rows=0, chunk=4))
    try:
        t = b.submit(**item)
        b.drain()
        r, U = b.result(t)
        (it, now, dt, rc), want, _ = S.plain_solve(item, chunk=4)
        assert r.status == 0 and rc == 0 and r.iter == it == 4
        assert (r.now_t, r.dt) == (now, dt)
        assert nan_equal_bits(U, want) == 0
        st[0].update(N_x=7680, N_y=1100, L=7680 / 1100)  # 128 x 69 strips of 16 rows
        big = S.ellipse_items(st, precision="FP64")[0]
        if blocks < 128 * 69:
            with pytest.raises(Exception):
                b.submit(**big)
        else:  # it just fits
            b.submit(**big)
            b.drain()
    finally:
        b.close()
