"""The mask level set's row search against the reference's own search, every cell
against every edge pixel (Test/PNGGeo/Level_Set.cpp:31-149), in NumPy: equal to the
bit, since each radicand is rounded alike and the square root is monotone. The sizes
are those where the search takes another form: no edge at all, fewer cells than one
interval, an interval's remainder, intervals of 128 cells (more than 65536 cells in a
row), masks too wide for LDS, and a circle about a cell corner (many nearest pixels)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _image(kind, W, H):
    img = np.full((H, W, 4), 255, np.uint8)
    x, y = np.meshgrid(np.arange(W), np.arange(H))
    if kind == "ring":
        solid = (x - W / 2) ** 2 + (y - H / 2) ** 2 < (0.3 * min(W, H)) ** 2
    elif kind == "dots":
        solid = np.isin(x, [5, W // 3, W - 4]) & (y == H // 2)
    elif kind == "noise":
        solid = np.random.default_rng(7).random((H, W)) < 0.02
    elif kind == "floor":
        solid = y > 2 * H // 3
    else:
        solid = np.zeros((H, W), bool)
    img[solid, :3] = 0
    return img


@pytest.mark.parametrize("kind,nx,ny,W,H", [
    ("none", 64, 24, 68, 28), ("ring", 24, 24, 28, 28), ("ring", 60, 40, 64, 44), ("ring", 125, 61, 129, 65),
    ("noise", 61, 30, 200, 35), ("floor", 200, 50, 97, 61), ("dots", 65600, 24, 131, 28), ("dots", 70, 24, 12000, 24),
    ("none", 70, 24, 12000, 24), ("floor", 70, 24, 10200, 24)])
def test_rows_equal_the_search_over_every_edge_pixel(kind, nx, ny, W, H):
    import ibtfo_amd as ib
    img = _image(kind, W, H)
    cfg = ib.config(N_x=nx, N_y=ny, lo_x=0.0, lo_y=0.0, hi_x=2.0, hi_y=2.0 * ny / nx, Boundary="IDWBaseGFM", quirks=1)
    print("mask rows %s %dx%d mask %dx%d" % (kind, nx, ny, W, H), flush=True)
    s = ib.Solver(cfg)
    try:
        s.geometry_mask(img)
        XY = s.xycoord().reshape(s.N, s.M, 6)
        M, N, ng = s.M, s.N, 2
    finally:
        s.close()
    v = np.where(img[::-1, :, :3].sum(axis=2, dtype=np.int64) > 0, 1, -1)
    edge = np.zeros((H, W), bool)
    edge[1:-1, 1:-1] = (v[1:-1, 1:-1] != v[1:-1, :-2]) | (v[1:-1, 1:-1] != v[:-2, 1:-1])
    ey, ex = np.nonzero(edge)
    hx, hy = 2.0 / nx, (2.0 * ny / nx) / ny
    ax = -ng * hx + (hx * (nx + 2 * ng) / W) * ex
    ay = -ng * hy + (hy * (ny + 2 * ng) / H) * ey
    X, Y = XY[0, :, 0], XY[:, 0, 1]
    xs = ((np.arange(M) + 0.5) * W / M).astype(int)
    for j in range(N):
        best = np.full(M, np.inf)
        for k in range(0, len(ax), 64):
            d = ax[k:k + 64, None] - X
            e = (ay[k:k + 64] - Y[j])[:, None]
            best = np.minimum(best, (d * d + e * e).min(axis=0))
        want = np.minimum(np.sqrt(best), 100.0) * v[int((j + 0.5) * H / N), xs]
        assert np.array_equal(XY[j, :, 2], want), (j, np.abs(XY[j, :, 2] - want).max())
