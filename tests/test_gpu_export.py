"""GPU parity of the equirectangular export (util.py:275-455,
nixis.py:270-302) against the oracle and against scipy's KDTree.

* make_ll_arr: the per-row / per-column cosines and sines come from the
  host C library, as the reference's numba code calls it, so the pixel
  coordinates equal the oracle's bit for bit.
* the k-nearest query: exactly the oracle's (brute force, equal distances
  ordered by index), distances bit for bit; against scipy's KDTree (the
  reference's tree) the distances are equal and the indices differ only
  where two vertices are at exactly the same distance.
* make_gray_array: bit for bit with the oracle on the same query results.
"""
import os

import numpy as np
import pytest
import torch

from nixis_amd import _lib, util

pytestmark = pytest.mark.gpu


def _ties_only(d, n, d2, n2, pts, q):
    """Indices differ only where both vertices lie at exactly that distance."""
    assert np.array_equal(d, d2)
    bad = np.nonzero(n != n2)
    qq = q.reshape(-1, 3) if q.ndim > 2 else q
    flat = np.ravel_multi_index(bad[:-1], n.shape[:-1])
    for f, j in zip(flat, bad[-1]):
        for v in (n.reshape(-1, n.shape[-1])[f, j], n2.reshape(-1, n.shape[-1])[f, j]):
            e = qq[f] - pts[v]
            s = 0.0
            for c in e:
                s += c * c
            assert np.sqrt(s) == d.reshape(-1, d.shape[-1])[f, j]
    return len(flat)


@pytest.mark.parametrize("wh", [(16, 9), (96, 48), (2048, 1024), (1001, 333)])
def test_ll_arr_bit_exact(oracle, wh):
    w, h = wh
    print("ll", w, h, flush=True)
    got = util.make_ll_arr(w, h, 1.7)
    assert got.shape == (h, w, 3)
    assert np.array_equal(got, oracle.make_ll_arr(w, h, 1.7))


@pytest.mark.parametrize("k", [1, 3, 8])
def test_query_random_points_matches_oracle(oracle, k):
    rng = np.random.default_rng(40 + k)
    p = rng.standard_normal((20000, 3))
    q = np.concatenate([rng.standard_normal((3000, 3)) * 1.5,
                        p[:50] + 1e-12,                      # on top of a point
                        np.full((3, 3), 25.0)])              # far outside the grid
    print("random k", k, flush=True)
    grid = util.KnnGrid(p)
    d, n = grid.query(q, k=k)
    rd, rn = oracle.knn(p, q, k)
    if k == 1:
        rd, rn = rd[..., 0], rn[..., 0]
    assert d.shape == rd.shape and n.dtype == np.int64
    assert np.array_equal(d, rd) and np.array_equal(n, rn)


def test_query_fewer_points_than_k(oracle):
    p = np.array([[0.0, 0, 0], [1.0, 0, 0]])
    q = np.array([[0.2, 0, 0], [5.0, 1.0, -2.0]])
    d, n = util.KnnGrid(p).query(q, k=3)
    rd, rn = oracle.knn(p, q, 3)
    assert n.tolist() == [[0, 1, 2], [1, 0, 2]] and (d[:, 2] == np.inf).all()  # scipy: n, inf
    assert np.array_equal(d, rd) and np.array_equal(n, rn)


def test_query_pixels_matches_oracle_and_scipy(oracle):
    from scipy.spatial import KDTree
    pts, _ = util.create_mesh(64)
    r = 2.0
    P = pts * r
    grid = util.KnnGrid(P)
    d, n = grid.query_pixels_device(256, 128, r, 3)
    d, n = d.cpu().numpy(), n.cpu().numpy()
    ll = oracle.make_ll_arr(256, 128, r)
    rd, rn = oracle.knn(P, ll, 3)
    assert np.array_equal(d, rd) and np.array_equal(n, rn)
    sd, sn = KDTree(P, leafsize=10).query(ll, k=3, workers=-1)
    ties = _ties_only(d, n, sd, sn, P, ll)
    print(f"pixels 256x128 on d=64: {ties} slots ordered differently from scipy at exact ties",
          flush=True)


def test_query_pixels_full_image_against_scipy():
    """2048 x 1024 (the reference's default image) on a d=500 mesh
    (2,500,002 vertices) against scipy's KDTree on the host."""
    from scipy.spatial import KDTree
    pts = util.create_points(500)
    grid = util.KnnGrid(pts)
    d, n = grid.query_pixels_device(2048, 1024, 1.0, 3)
    d, n = d.cpu().numpy(), n.cpu().numpy()
    ll = util.make_ll_arr(2048, 1024, 1.0)
    sd, sn = KDTree(pts, leafsize=10).query(ll, k=3, workers=-1)
    ties = _ties_only(d, n, sd, sn, pts, ll)
    print(f"2048x1024 on d=500: {ties} slots at exact ties", flush=True)
    assert ties < 0.001 * n.size


def test_gray_array_bit_exact(oracle):
    rng = np.random.default_rng(3)
    pts, _ = util.create_mesh(40)
    grid = util.KnnGrid(pts)
    d, n = grid.query_pixels_device(300, 150, 1.0, 3)
    d, n = d.cpu().numpy(), n.cpu().numpy()
    for colors in (rng.uniform(0, 255, pts.shape[0]),
                   rng.uniform(-300, 300, pts.shape[0]),
                   rng.integers(0, 65535, pts.shape[0]).astype(np.uint16)):
        got = util.make_gray_array(300, 150, d, n, colors)
        ref = oracle.make_gray_array(300, 150, d, n, colors).astype(colors.dtype)
        assert got.dtype == colors.dtype and np.array_equal(got, ref)
    rgb = util.make_rgb_array(300, 150, d, n, colors)
    assert rgb.shape == (150, 300, 3) and (rgb == got[:, :, None]).all()


def test_gray_rejects_neighbours_outside_colors():
    d = torch.ones((4, 3), dtype=torch.float64, device="cuda")
    n = torch.zeros((4, 3), dtype=torch.int64, device="cuda")
    n[2, 1] = 10
    c = torch.ones(10, dtype=torch.float64, device="cuda")
    util.make_gray_array_device(d, n, c)
    with pytest.raises(_lib.NixisArgError):
        _lib.Context.get(d.device).sync_check()


def test_export_pipeline_writes_the_oracle_image(oracle, tmp_path):
    """heights -> build_image_data (rescale to 0..255, gray) -> save_image:
    the PNG read back equals the oracle's pixels."""
    from PIL import Image
    pts, _ = util.create_mesh(50)
    rng = np.random.default_rng(9)
    h = rng.uniform(-4000, 8850, pts.shape[0])
    ocean = h <= 0
    grid = util.build_KDTree(pts)
    qd = grid.query(util.make_ll_arr(400, 200, 1.0), k=3, workers=-1)
    data = util.build_image_data({"height": [h, "gray"], "ocean": [ocean, "gray"]}, 400, 200, qd)
    util.save_image(data, str(tmp_path), "w")
    img = np.asarray(Image.open(os.path.join(tmp_path, "w_height.png")))
    ref = oracle.make_gray_array(400, 200, qd[0], qd[1],
                                 oracle.rescale_ex(h, 0, 255)).astype(np.uint8)
    assert img.dtype == np.uint8 and np.array_equal(img, ref)
    m = np.asarray(Image.open(os.path.join(tmp_path, "w_ocean.png")))
    ref_m = oracle.make_gray_array(400, 200, qd[0], qd[1],
                                   oracle.rescale_ex(ocean.astype(np.float64), 0, 255))
    assert np.array_equal(m, ref_m.astype(np.float64).astype(np.uint8))


def _point_sets():
    rng = np.random.default_rng(11)

    def ball(n):
        p = rng.standard_normal((n, 3))
        return p / np.linalg.norm(p, axis=1, keepdims=True)
    ico, _ = util.create_mesh(30)
    thick = ball(4000) * rng.uniform(0.85, 1.0, (4000, 1))
    return {
        "icosphere": ico, "world": ico * 6378100.0, "random sphere": ball(5000),
        "thick shell": thick, "thinner than a shell": ball(3000) * rng.uniform(0.7, 1, (3000, 1)),
        "offset sphere": ico + [3.0, 0, 0], "cap": ico[ico[:, 2] > 0.9],
        "duplicates": np.concatenate([ico, ico[::3], ico[::5]]),
        "poles": np.concatenate([ball(300), np.tile([[0, 0, 1.0], [0, 0, -1.0]], (20, 1))]),
        "seam": np.concatenate([ball(300), [[-np.cos(t), s * 0.0, np.sin(t)]
                                            for t in np.linspace(-1.5, 1.5, 41) for s in (1, -1)]]),
        "volume": rng.uniform(-1, 1, (3000, 3)), "line": np.linspace(-1, 1, 500)[:, None] * [[1, 2, 3]],
        "one": np.array([[0.0, 0.0, 1.0]]), "six": np.concatenate([np.eye(3), -np.eye(3)]),
        "with nan": np.concatenate([ico, [[np.nan, 0, 0]]]),
    }


@pytest.mark.parametrize("k", [1, 3, 4, 8])
def test_query_every_kind_of_point_set(oracle, k):
    """Both kinds of bins (latitude bands, hashed cells) against brute force:
    on, near and off the points' surface, at the centre, the poles and the
    seam of the longitudes, and at exact ties."""
    rng = np.random.default_rng(12)
    for name, p in _point_sets().items():
        print(name, "k", k, flush=True)
        fine = p[np.isfinite(p).all(axis=1)]
        r = np.linalg.norm(fine, axis=1).max()
        u = rng.standard_normal((300, 3))
        u /= np.linalg.norm(u, axis=1, keepdims=True)
        q = np.concatenate([u * r, u[:80] * r * 1.05, u[:80] * r * 0.6, u[:20] * r * 7, fine[:50],
                            0.5 * (fine[:40] + fine[-40:][:len(fine[:40])]),
                            r * np.array([[0, 0, 1.0], [0, 0, -1.0], [-1, 0, 0], [-1, -0.0, 0],
                                          [0, 0, 0], [1e-9, 0, -1], [-1, 1e-12, 0.3]])])
        d, n = util.KnnGrid(p).query(q, k=k)
        rd, rn = oracle.knn(p, q, k)
        if k == 1:
            rd, rn = rd[..., 0], rn[..., 0]
        assert np.array_equal(d, rd) and np.array_equal(n, rn)


@pytest.mark.parametrize("wh", [(1, 2), (7, 3), (255, 2), (257, 5), (130, 131)])
def test_query_pixels_image_edges(oracle, wh):
    """Images that do not fill the last block, narrow and tall ones, and a
    radius other than the points'."""
    pts, _ = util.create_mesh(21)
    grid = util.KnnGrid(pts * 2.0)
    for radius in (2.0, 1.9, -2.0):
        d, n = grid.query_pixels_device(wh[0], wh[1], radius, 3)
        rd, rn = oracle.knn(pts * 2.0, oracle.make_ll_arr(wh[0], wh[1], radius), 3)
        assert np.array_equal(d.cpu().numpy(), rd) and np.array_equal(n.cpu().numpy(), rn)


@pytest.mark.parametrize("d,wh", [(3, (256, 64)), (9, (256, 200)), (33, (257, 131)), (64, (300, 77)),
                                  (40, (1000, 400)), (150, (512, 90))])
def test_query_pixels_rows_share_their_points(oracle, d, wh):
    """Images at least a block wide, whose rows read their points together:
    few and many points to a wave, windows that pass the ends of a band, and
    whole bands near the poles for some pixels of a wave only."""
    pts, _ = util.create_mesh(d)
    d_, n_ = util.KnnGrid(pts).query_pixels_device(wh[0], wh[1], 1.0, 3)
    rd, rn = oracle.knn(pts, oracle.make_ll_arr(wh[0], wh[1], 1.0), 3)
    assert np.array_equal(d_.cpu().numpy(), rd) and np.array_equal(n_.cpu().numpy(), rn)


@pytest.mark.parametrize("k", [1, 3, 8])
def test_query_from_where_squared_distances_overflow(oracle, k):
    """Every point is then equally far, at an infinite distance where the square
    overflows: the first points by index, not none."""
    for pts in (util.create_mesh(9)[0], util.create_mesh(9)[0] * 6378100.0, np.concatenate([np.eye(3), -np.eye(3)])):
        q = np.array([[1e200, 0, 0], [0, -1e200, 0], [1e200, 1e200, -1e200], [np.inf, 0, 0],
                      [-np.inf, np.inf, 1.0], [1e160, 1, 1], [1e-3, 2.0, -1.35e154], [1.34e154, 3.0, 0],
                      [0, 0, 1e152], [1e120, 1e153, 1e100]])
        grid = util.KnnGrid(pts)
        d, n = grid.query(q, k=k)
        rd, rn = oracle.knn(pts, q, k)
        if k == 1:
            rd, rn = rd[..., 0], rn[..., 0]
        assert np.array_equal(d, rd) and np.array_equal(n, rn)
        for radius in (1e200, -1e200, 1e160, 1e153):
            for w, h in ((8, 5), (300, 3)):
                d, n = grid.query_pixels_device(w, h, radius, k)
                rd, rn = oracle.knn(pts, oracle.make_ll_arr(w, h, radius), k)
                assert np.array_equal(d.cpu().numpy(), rd) and np.array_equal(n.cpu().numpy(), rn)


def _clustered(n, seed):
    """n points of a sphere, half of them in a small cap, some many times over."""
    rng = np.random.default_rng(seed)
    p = rng.standard_normal((n, 3))
    p[::2] = p[::2] * [0.02, 0.02, 0] + [0, 0, 1]
    p /= np.linalg.norm(p, axis=1, keepdims=True)
    p[1:n // 4:4] = p[0]
    p[3:n // 40:4] = p[2]
    return p


@pytest.mark.parametrize("k", [1, 3, 8])
@pytest.mark.parametrize("n", [4001, 4098])
def test_query_dense_runs(oracle, n, k):
    """Bins of many points, equal ones among them, in latitude bands and in
    hashed cells, in runs that do and do not fill the last batch read together;
    query points on, near and off them, and images."""
    p = _clustered(n, 21)
    rng = np.random.default_rng(22)
    q = np.concatenate([p[:60], p[:60] * 1.0001, p[:200:4] + 1e-7, rng.standard_normal((60, 3)),
                        p[:3] * 0.5, p[:3] * 3.0])
    for shift in ([0, 0, 0], [3.0, 0, 0], [0, 0, 0.01]):
        grid = util.KnnGrid(p + shift)
        d, nb = grid.query(q + shift, k=k)
        rd, rn = oracle.knn(p + shift, q + shift, k)
        if k == 1:
            rd, rn = rd[..., 0], rn[..., 0]
        assert np.array_equal(d, rd) and np.array_equal(nb, rn)
        for w, h in ((300, 9), (50, 21)):
            d, nb = grid.query_pixels_device(w, h, 1.0, k)
            rd, rn = oracle.knn(p + shift, oracle.make_ll_arr(w, h, 1.0), k)
            assert np.array_equal(d.cpu().numpy(), rd) and np.array_equal(nb.cpu().numpy(), rn)


def _query_ms(points, queries, k=3):
    grid = util.KnnGrid(points)
    grid.query_device(queries, k)
    best = np.inf
    for _ in range(5):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        grid.query_device(queries, k)
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


def test_query_time_in_hashed_cells():
    """A planet's vertices away from the origin are queried in hashed cells: at
    most six times as long as in latitude bands (3.6 times; 9 where a candidate's
    entry was read and compared before its point)."""
    pts = util.create_mesh_device(316, cells=False)[0]
    q = pts[::2].contiguous()
    bands, cells = _query_ms(pts, q), _query_ms(pts + 3.0, q + 3.0)
    print(f"bands {bands:.3f} ms, cells {cells:.3f} ms", flush=True)
    assert cells <= 6 * bands


def test_query_time_of_dense_latitude_bands():
    """Half of the points in a small cap: no slower in latitude bands than in
    hashed cells, which adapt to it, within 1.4 times (0.9; 1.7 where a whole
    window of dense bins was read, each point after its entry)."""
    rng = np.random.default_rng(3)
    n = 400000
    p = rng.standard_normal((n, 3))
    p[::2] = p[::2] * [0.02, 0.02, 0] + [0, 0, 1]
    p = torch.from_numpy(p / np.linalg.norm(p, axis=1, keepdims=True)).cuda()
    q = p[::200].contiguous()
    bands, cells = _query_ms(p, q), _query_ms(p + 3.0, q + 3.0)
    print(f"bands {bands:.3f} ms, cells {cells:.3f} ms", flush=True)
    assert bands <= 1.4 * cells
