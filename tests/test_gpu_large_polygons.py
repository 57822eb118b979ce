"""dpx_stage_triangulate on a caller's polygons far larger than a cell, around
the coordinates where the packed form ends (16383 and 32767 units of 1/64):
the triangles of the plain ear clipping, whose products are taken modulo 2^32."""
import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]

CS = 45


def wrap(v):
    return (v + (1 << 31)) % (1 << 32) - (1 << 31)


def cross(o, a, b):
    return wrap(wrap((a[0] - o[0]) * (b[1] - o[1])) - wrap((a[1] - o[1]) * (b[0] - o[0])))


def inside(a, b, c, p):
    def edge(s, e):
        return wrap(wrap((e[0] - s[0]) * (p[1] - s[1])) - wrap((e[1] - s[1]) * (p[0] - s[0])))
    return edge(b, c) >= 0 and edge(a, b) >= 0 and edge(c, a) >= 0


def ears(p):
    """process (triangulate_functions.cu:108-217) in 32-bit whole numbers."""
    area = 0
    for a, b in zip([p[-1]] + p[:-1], p):
        area = wrap(area + wrap(wrap(a[0] * b[1]) - wrap(b[0] * a[1])))
    v = list(p) if area > 0 else list(p)[::-1]
    out, k, count = [], len(v) - 1, 2 * len(v)
    while len(v) > 2:
        if count <= 0:
            break
        count -= 1
        u = 0 if k >= len(v) else k
        k = 0 if u + 1 >= len(v) else u + 1
        w = 0 if k + 1 >= len(v) else k + 1
        a, b, c = v[u], v[k], v[w]
        if cross(a, b, c) > 0 and not any(inside(a, b, c, q) for t, q in enumerate(v) if t not in (u, k, w)):
            out += [a, b, c]
            del v[k]
            count = 2 * len(v)
    return out


@pytest.mark.parametrize("limit", [16383, 16384, 23000, 32767, 32768, 40000])
def test_large_polygons(gpu, D, limit):
    torch, cells = gpu, 300
    rng = np.random.default_rng(limit)
    d, n, polys = np.zeros((cells, CS, 2), dtype=np.float32), np.zeros(cells, dtype=np.int32), []
    for k in range(cells):
        m = int(rng.integers(3, 17))
        if k % 3:
            a = np.sort(rng.random(m) * 2 * np.pi)
            r, h = limit * (0.6 + 0.4 * rng.random()), 1.0 if k % 3 == 1 else 0.05 + 0.95 * rng.random()
            p = np.stack([np.rint(r * np.cos(a)), np.rint(r * h * np.sin(a))], axis=1)
            p[np.argmax(np.abs(p[:, 0])), 0] = limit  # one vertex at the limit itself
        else:
            p = rng.integers(-limit, limit + 1, size=(m, 2))
        p = np.clip(p, -limit, limit).astype(np.int64)[::1 if rng.random() < 0.5 else -1]
        n[k] = m
        d[k, :m] = p / 64.0
        polys.append([(int(x), int(y)) for x, y in p])
    diag, ec = torch.from_numpy(d).cuda(), torch.from_numpy(n).cuda()
    D.check(D.lib.dpx_stage_triangulate(diag.data_ptr(), ec.data_ptr(), cells, 1, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    got = diag.cpu().numpy().reshape(cells, CS, 2)
    for k, p in enumerate(polys):
        want = np.zeros((CS, 2), dtype=np.float32)
        t = ears(p)
        if t:
            want[:len(t)] = np.array(t, dtype=np.float32) / 64.0
        want[:, 0] += k
        assert np.array_equal(got[k], want), (k, p)
