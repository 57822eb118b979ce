"""The per-frame stage kernels where their tiles and packings change: frames
around a tile's and a run's sizes, cells whose vertices, counts or extents do
not fit the packed forms, and views of few and of many cells a block.
Against the oracle."""
import ctypes

import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]

CS = 45


def up(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def slots(a, n):
    return [a.reshape(-1, CS, 2)[k, :m] for k, m in enumerate(n)]


# 1 cell, either side of a run of 64 and of 256 cells, of a 32x8 tile, narrow frames
@pytest.mark.parametrize("size", [(1, 1), (1, 65), (63, 1), (32, 8), (33, 9), (31, 7), (257, 1), (16, 16), (85, 3)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("flags", [0, 2])
def test_stages_at_tile_edges(gpu, D, O, size, flags):
    torch, (W, H) = gpu, size
    s = torch.cuda.current_stream().cuda_stream
    img = D.synth_frame(4, 77 + W, W, H, 3, 3 * W + 1)
    g = O.heuristic_cross(O.trivial_cross(O.similarity_graph(img, W, H, flags=flags)))
    od, oec = O.cells(g)
    d_img, d_g = up(torch, img), up(torch, g)
    diag = torch.full((W * H * CS * 2,), 7.0, device="cuda:0")
    daux, ec = torch.empty_like(diag), torch.zeros(W * H, dtype=torch.int32, device="cuda:0")
    eaux = torch.empty_like(ec)
    D.check(D.lib.dpx_stage_cells(d_g.data_ptr(), W, H, diag.data_ptr(), ec.data_ptr(), s))
    torch.cuda.synchronize()
    assert np.array_equal(ec.cpu().numpy().reshape(-1), np.asarray(oec).reshape(-1))
    for a, b in zip(slots(diag.cpu().numpy(), oec.reshape(-1) + 1), slots(np.asarray(od), oec.reshape(-1) + 1)):
        assert np.array_equal(a, b)
    D.check(D.lib.dpx_stage_subdivide(d_img.data_ptr(), W, H, img.shape[1], 3, flags, d_g.data_ptr(), diag.data_ptr(),
                                      daux.data_ptr(), ec.data_ptr(), eaux.data_ptr(), s))
    torch.cuda.synchronize()
    sd, sec, _, _ = O.subdivide(img, W, H, g, od, oec, flags=flags)
    assert np.array_equal(ec.cpu().numpy().reshape(-1), np.asarray(sec).reshape(-1))
    for a, b in zip(slots(diag.cpu().numpy(), sec.reshape(-1)), slots(np.asarray(sd), sec.reshape(-1))):
        assert np.array_equal(a, b)
    D.check(D.lib.dpx_stage_triangulate(diag.data_ptr(), ec.data_ptr(), W, H, s))
    torch.cuda.synchronize()
    td, _ = O.triangulate(sd, sec, W, H)
    assert np.array_equal(diag.cpu().numpy().reshape(-1), np.asarray(td).reshape(-1))
    pos, col = torch.zeros_like(diag), torch.zeros(W * H * CS * 4, dtype=torch.uint8, device="cuda:0")
    D.check(D.lib.dpx_stage_export_vbo(d_img.data_ptr(), W, H, img.shape[1], 3, flags, diag.data_ptr(), ec.data_ptr(),
                                       pos.data_ptr(), col.data_ptr(), s))
    torch.cuda.synchronize()
    op, oc = O.export_vbo(img, W, H, td, sec, flags=flags)
    assert np.array_equal(pos.cpu().numpy().reshape(-1), np.asarray(op).reshape(-1))
    assert np.array_equal(col.cpu().numpy().reshape(-1), np.asarray(oc).reshape(-1))


@pytest.mark.parametrize("cells", [1, 255, 256, 257])
def test_triangulate_any_polygon(gpu, D, O, cells):
    # 0 to 17 vertices on the 1/64 lattice (16 are clipped in LDS), every
    # third polygon at random, mostly crossing itself
    torch = gpu
    rng = np.random.default_rng(cells)
    d, n = np.zeros((cells, CS, 2), dtype=np.float32), rng.integers(0, 18, size=cells).astype(np.int32)
    for k in range(cells):
        m = max(int(n[k]), 1)
        if k % 3:
            a, r = np.sort(rng.random(m) * 2 * np.pi), rng.integers(15, 50, size=m) if k % 3 == 1 else np.full(m, 45)
            p = np.stack([32 + np.rint(r * np.cos(a)), 32 + np.rint(r * np.sin(a))], axis=1)
        else:
            p = rng.integers(-22, 87, size=(m, 2))
        d[k, :m] = (p[::-1] if rng.random() < 0.5 else p) / 64.0
    ec = up(torch, n)
    diag = up(torch, d)
    D.check(D.lib.dpx_stage_triangulate(diag.data_ptr(), ec.data_ptr(), cells, 1,
                                        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    want, _ = O.triangulate(d.reshape(-1, 2).copy(), n, cells, 1)
    got = diag.cpu().numpy().reshape(cells, CS, 2)
    for k in range(cells):
        if n[k] >= 3:
            assert np.array_equal(got[k], np.asarray(want).reshape(cells, CS, 2)[k]), (k, n[k])
        else:
            assert (got[k] == [k, 0]).all()


def test_subdivide_hulls_of_many_vertices(gpu, D, O):
    # straight corners added to the hulls, up to 16 vertices, in every fifth cell
    torch, W, H = gpu, 70, 20
    img = D.synth_frame(2, 5, W, H, 3)
    g = O.heuristic_cross(O.trivial_cross(O.similarity_graph(img, W, H)))
    od, oec = (np.array(a) for a in O.cells(g))
    od, oec = od.reshape(-1, CS, 2).astype(np.float32), oec.reshape(-1).astype(np.int32)
    for k in range(0, W * H, 5):
        n = oec[k]
        p = od[k, :n]
        # midpoints of the edges that keep them on the quarter lattice
        q = []
        for a, b in zip(p, np.roll(p, -1, axis=0)):
            q.append(a)
            m = (a + b) / 2
            if (m * 4 == np.rint(m * 4)).all() and not (m == a).all():
                q.append(m)
        od[k, :len(q)], oec[k] = np.array(q), len(q)
    assert oec.max() > 8
    diag, ec = up(torch, od), up(torch, oec)
    daux, eaux = torch.empty_like(diag), torch.empty_like(ec)
    d_img, d_g = up(torch, img), up(torch, g)
    D.check(D.lib.dpx_stage_subdivide(d_img.data_ptr(), W, H, img.shape[1], 3, 0, d_g.data_ptr(), diag.data_ptr(),
                                      daux.data_ptr(), ec.data_ptr(), eaux.data_ptr(),
                                      torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    sd, sec, _, _ = O.subdivide(img, W, H, g, od.reshape(-1, 2), oec)
    assert np.array_equal(ec.cpu().numpy(), np.asarray(sec).reshape(-1))
    for k, (a, b) in enumerate(zip(slots(diag.cpu().numpy(), np.asarray(sec).reshape(-1)),
                                   slots(np.asarray(sd), np.asarray(sec).reshape(-1)))):
        assert np.array_equal(a, b), k


# scales on both sides of the tile choices (1x, 2.5x), windows that miss the image
@pytest.mark.parametrize("scale", [25, 60, 99, 100, 101, 225, 250, 275, 800, 3200])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("aa", [0, 1])
def test_views_of_few_and_many_cells(gpu, D, O, scale, wide, aa):
    torch, W, H, ww, wh = gpu, 40, 33, 150, 90
    img = D.synth_frame(0, 3, W, H, 3)
    ref = O.depixelize(img, W, H, scale=1, subdivide=True, want_diagram=True)
    d, n = np.array(ref["diagram"]).reshape(-1, CS, 2).astype(np.float32), np.array(ref["edge_count"]).reshape(-1)
    if wide:  # a vertex of every seventh cell up to 0.9 of a cell beyond its square
        for k in range(0, W * H, 7):
            d[k, 1] = [k % W - 57 / 64.0, k // W + 120 / 64.0]
    d_img, diag, ec = up(torch, img), up(torch, d), up(torch, n.astype(np.int32))
    out = torch.zeros(wh * ww * 4, dtype=torch.uint8, device="cuda:0")
    for tx, ty in ((1, 1), (-200, -30), (-65536, 65536)):
        view = D.View(0, scale, tx, ty, ww, wh, aa, 0)
        D.check(D.lib.dpx_stage_present(d_img.data_ptr(), W, H, img.shape[1], 3, 0, diag.data_ptr(), ec.data_ptr(),
                                        ctypes.byref(view), out.data_ptr(), ww * 4,
                                        torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        want = O.present(img, W, H, d.reshape(-1, 2), n.astype(np.int32), mode=0, scale_x100=scale, tx=tx, ty=ty,
                         width=ww, height=wh, view_flags=aa)
        assert np.array_equal(out.cpu().numpy().reshape(wh, ww, 4), want), (tx, ty)


@pytest.mark.parametrize("scale", [1, 2, 3, 4, 32])
def test_raster_of_every_tile_choice(gpu, D, O, scale):
    W, H = 37, 29
    img = D.synth_frame(2, 8, W, H, 3)
    rgba, _, _ = D.frame(img, W, H, 3, scale=scale, subdivide=True)
    d = O.depixelize(img, W, H, scale=1, subdivide=True, want_diagram=True)
    want = O.rasterize(img, W, H, d["diagram"], d["edge_count"], scale)
    assert np.array_equal(rgba, want)
