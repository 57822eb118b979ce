"""The workloads whose speed is watched: what users of the library have it do,
through its public entry points (the `depixel` package over libdepixel.so).

Three kinds of caller are stood for:
  * batches on the device ("batch", "plan"): frames or sprites resident in
    HBM, one call per batch, images left in HBM;
  * the per-frame stages on device buffers: the viewer's frame ("viewer":
    every stage, then the window) and the component analysis ("chains":
    labels and border chains of a resolved graph);
  * callers with host memory: the launch_kernel drop-in and the plain
    per-frame call ("drop_in", "frame"), and the serving loop ("served").

Positions of the cell diagram lie on a dyadic lattice and are fixed bit for
bit by the definition of the path, so they are handed out as 32-bit words:
every output here is bytes or whole numbers.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.abspath("pixel-art-remaster-gpu_amd"))
import depixel as D  # noqa: E402

CELL = D.CELL_SIZE
# synthetic content: 0 16-colour game frames, 1 alpha sprites, 2 console
# frames full of one-pixel lines, 4 dithered 256-colour frames with a lattice
# of crossings, 5 palette-indexed game streams
GAME, SPRITE, CONSOLE, LARGE, STREAM = 0, 1, 2, 4, 5
CONSOLE_SIZES = ((256, 240), (256, 224), (320, 224), (384, 224), (240, 160))


def listed():
    return [
        # One game frame to 4x, as an emulator shows it: a fixed layout, one
        # plan, launch latency first.
        dict(name="frame_one", path="plan", kind=GAME, count=1, width=256, height=224, channels=3, scale=4,
             smooth=False, flags=0, pad=0),
        # The headline batch: 1024 frames of 256x224 to 4x.
        dict(name="frames_1024", path="batch", kind=GAME, count=1024, width=256, height=224, channels=3, scale=4,
             smooth=False, flags=0, pad=0),
        # 64 frames of five consoles' screen sizes in one batch, busy with
        # one-pixel lines; rows top first and RGB, as frame grabbers give them.
        dict(name="console_64", path="batch", kind=CONSOLE, count=64, width=0, height=0, channels=3, scale=4,
             smooth=False, flags=D.RGB | D.TOPDOWN, pad=0),
        # A game's sprite sheet: 4096 alpha sprites of 8 to 64 pixels to 6x.
        dict(name="sprites_4096", path="batch", kind=SPRITE, count=4096, width=0, height=0, channels=4, scale=6,
             smooth=False, flags=D.ALPHA, pad=0),
        # 16 dithered 640x480 frames to 8x, plain and smoothed.
        dict(name="large_16", path="batch", kind=LARGE, count=16, width=640, height=480, channels=3, scale=8,
             smooth=False, flags=0, pad=0),
        dict(name="large_16_smooth", path="batch", kind=LARGE, count=16, width=640, height=480, channels=3, scale=8,
             smooth=True, flags=0, pad=0),
        # 64 game frames with the overscan border cropped off (odd sizes,
        # rows padded), smoothed, to 4x.
        dict(name="cropped_64_smooth", path="batch", kind=GAME, count=64, width=251, height=223, channels=3, scale=4,
             smooth=True, flags=0, pad=3),
        # One frame of each of 128 palette-indexed streams to 4x.
        dict(name="streams_128", path="batch", kind=STREAM, count=128, width=320, height=224, channels=1, scale=4,
             smooth=False, flags=D.INDEXED, pad=0),
        # The serving loop: 32 streams' frames from host memory and back.
        dict(name="served_32", path="served", kind=STREAM, count=32, width=320, height=224, channels=1, scale=4,
             smooth=False, flags=D.INDEXED, pad=0),
        # Component labels and border chains of a large frame's graph.
        dict(name="chains_large", path="chains", kind=LARGE, count=1, width=640, height=480, channels=3, scale=1,
             smooth=False, flags=0, pad=0),
        # The viewer's frame: every stage, then the antialiased 1200x800
        # window at the reference's default scale 8.
        dict(name="viewer", path="viewer", kind=GAME, count=1, width=256, height=224, channels=3, scale=8,
             smooth=True, flags=0, pad=0, antialias=True, window_w=1200, window_h=800),
        # The reference's own call, launch_kernel, smoothed, vertex buffers
        # on the device, everything else in host memory.
        dict(name="drop_in", path="drop_in", kind=GAME, count=1, width=256, height=224, channels=3, scale=1,
             smooth=True, flags=0, pad=0),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["batch"] * 7 + ["plan", "chains", "viewer", "drop_in", "frame", "served"])
    kind = rng.choice([GAME, GAME, CONSOLE, LARGE])
    smooth = rng.random() < 0.3
    flags = rng.choice([0, 0, D.TOPDOWN, D.RGB | D.TOPDOWN])
    channels = rng.choice([3, 3, 4])
    pad = rng.choice([0, 0, 0, 1, 5, 8])
    w, h = _log_int(rng, 48, 640), _log_int(rng, 48, 480)
    c = dict(path=path, kind=kind, count=1, width=w, height=h, channels=channels, scale=1, smooth=smooth,
             flags=flags, pad=pad)
    if path in ("batch", "plan"):
        what = rng.random()
        if what < 0.25:
            c.update(kind=SPRITE, channels=4, flags=flags | D.ALPHA, width=0, height=0)
            if rng.random() < 0.5:
                c.update(width=_log_int(rng, 5, 96), height=_log_int(rng, 5, 96))
        elif what < 0.4:
            c.update(kind=STREAM, channels=1, flags=D.INDEXED | rng.choice([0, D.FLIP_OUT]))
        elif what < 0.5:
            c.update(kind=CONSOLE, width=0, height=0)
        elif rng.random() < 0.3:
            c["flags"] |= D.FLIP_OUT
        c["scale"] = rng.choice([1, 2, 2, 3, 3, 4, 4, 4, 5, 6, 6, 7, 8, 8, 10, 12, 15])
        cells = (c["width"] or 288) * (c["height"] or 216) if c["kind"] != SPRITE else \
            (c["width"] or 24) * (c["height"] or 24)
        # bounded by the headline batch's output, its frames, and for
        # smoothing by the cells of the large smoothed batch
        most = min(3_600_000_000 // (4 * cells * c["scale"] ** 2), 50_000_000 // cells, 4096)
        if smooth:
            most = min(most, 4_500_000 // cells)
        c["count"] = _log_int(rng, 1, max(1, most))
    elif path == "viewer":
        sizes = ((256, 224), (320, 224), (160, 144), (w, h))
        c["width"], c["height"] = rng.choice(sizes)
        c["scale"] = rng.choice([1, 2, 3, 4, 6, 8, 12])
        c.update(antialias=rng.random() < 0.7, window_w=rng.choice([1200, 1280, 641, 1920]),
                 window_h=rng.choice([800, 720, 479, 1080]))
    elif path == "drop_in":
        c.update(channels=3, flags=0, width=min(w, 384), height=min(h, 256))
    elif path == "frame":
        c.update(scale=rng.choice([1, 2, 3, 4]), width=min(w, 384), height=min(h, 256))
    elif path == "served":
        c.update(width=min(w, 384), height=min(h, 256), scale=rng.choice([2, 3, 4]), count=_log_int(rng, 1, 32))
    return c


def _size(case, k):
    """Size of frame k: a sheet's or a batch's layout is the case's, whatever the seed."""
    if case["width"]:
        return case["width"], case["height"]
    if case["kind"] == SPRITE:
        return D.sprite_size(0, k)
    return CONSOLE_SIZES[k * len(CONSOLE_SIZES) // case["count"]]


def _frame(case, seed, k, w, h):
    """Frame k as a (h, stride) array, and its palette or None."""
    if case["kind"] == STREAM:
        idx, pal = D.stream_frame(seed * 4096 + k, 1 + k % 8, w, h)
        if case["pad"]:
            idx = np.pad(idx, ((0, 0), (0, case["pad"])))
        return np.ascontiguousarray(idx), pal
    return D.synth_frame(case["kind"], seed * 4096 + k, w, h, case["channels"], w * case["channels"] + case["pad"]), None


def _prepare_batch(case, seed):
    S, blobs, items, in_off, out_off = case["scale"], [], [], 0, 0
    for k in range(case["count"]):
        w, h = _size(case, k)
        img, pal = _frame(case, seed, k, w, h)
        pal_off = 0
        if pal is not None:
            pal_off = in_off
            blobs.append(pal.reshape(-1))
            in_off += pal.size
        items.append(D.Item(in_off, out_off, w, h, img.shape[1], case["channels"], S, int(case["smooth"]),
                            case["flags"], 4 * S * w, pal_off))
        fill = -img.size % 4  # palettes start on whole words
        blobs.append(img.reshape(-1))
        if fill:
            blobs.append(np.zeros(fill, dtype=np.uint8))
        in_off += img.size + fill
        out_off += 4 * S * w * S * h
    st = dict(case=case, d_in=torch.from_numpy(np.concatenate(blobs)).cuda(),
              d_out=torch.zeros(out_off, dtype=torch.uint8, device="cuda"), ctx=D.Context(0),
              items=D.items_array(items))
    if case["path"] == "plan":
        st["plan"] = D.Plan(st["ctx"], st["items"], st["d_out"].data_ptr() % 16)
    return st


def _prepare_served(case, seed):
    S, w, h = case["scale"], case["width"], case["height"]
    srv = D.Server(budget_bytes=2 << 30, max_batch=64)
    frames, outs, sids = [], [], []
    for k in range(case["count"]):
        img, pal = _frame(case, seed, k, w, h)
        host = D.pinned_empty(img.shape)
        host[...] = img
        sid = srv.open_stream(w, h, case["channels"], S, case["smooth"], case["flags"])
        if pal is not None:
            srv.set_palette(sid, pal)
        frames.append(host)
        outs.append(D.pinned_empty((S * h, 4 * S * w)))
        sids.append(sid)
    return dict(case=case, srv=srv, frames=frames, outs=outs, sids=sids)


def prepare(case, seed):
    if case["path"] in ("batch", "plan"):
        return _prepare_batch(case, seed)
    if case["path"] == "served":
        return _prepare_served(case, seed)
    w, h = case["width"], case["height"]
    img, _ = _frame(case, seed, 0, w, h)
    n = w * h
    i32 = dict(dtype=torch.int32, device="cuda")
    u8 = dict(dtype=torch.uint8, device="cuda")
    f32 = dict(dtype=torch.float32, device="cuda")
    st = dict(case=case, img=img)
    if case["path"] == "chains":
        _, graph, _ = D.frame(img, w, h, case["channels"], scale=1, flags=case["flags"])
        st.update(graph=torch.from_numpy(np.ascontiguousarray(graph)).cuda(), labels=torch.zeros(n, **i32),
                  scratch=torch.zeros(n, **u8), nodes=torch.zeros(8 * n, **i32), sizes=torch.zeros(n, **i32),
                  counts=torch.zeros(3, **i32))
    elif case["path"] == "viewer":
        view = D.View(D.VIEW_CELLS, 100 * case["scale"], 1, 1, case["window_w"], case["window_h"],
                      (D.VIEW_AA if case["antialias"] else 0) | D.VIEW_TOPDOWN)
        st.update(d_img=torch.from_numpy(img).cuda(), graph=torch.zeros(n, **u8), graph_aux=torch.zeros(n, **u8),
                  diagram=torch.zeros(n * CELL * 2, **f32), diagram_aux=torch.zeros(n * CELL * 2, **f32),
                  edges=torch.zeros(n, **i32), edges_aux=torch.zeros(n, **i32), view=view,
                  window=torch.zeros(case["window_h"] * case["window_w"] * 4, **u8))
    elif case["path"] == "drop_in":
        st.update(pos=torch.zeros(n * CELL * 2, **f32), color=torch.zeros(n * CELL * 4, **u8))
    return st


def _run_chains(st):
    c, lib, s = st["case"], D.lib, torch.cuda.current_stream().cuda_stream
    w, h = c["width"], c["height"]
    D.check(lib.dpx_stage_components(st["graph"].data_ptr(), w, h, st["labels"].data_ptr(), s))
    D.check(lib.dpx_stage_border_chains(st["graph"].data_ptr(), w, h, st["scratch"].data_ptr(),
                                        st["nodes"].data_ptr(), st["nodes"].numel(), st["sizes"].data_ptr(),
                                        st["sizes"].numel(), st["counts"].data_ptr(), s))
    return st["labels"], st["nodes"], st["sizes"], st["counts"]


def _run_viewer(st):
    c, lib, s = st["case"], D.lib, torch.cuda.current_stream().cuda_stream
    w, h, ch, fl, stride = c["width"], c["height"], c["channels"], c["flags"], st["img"].shape[1]
    img, graph, diagram, edges = (st[k].data_ptr() for k in ("d_img", "graph", "diagram", "edges"))
    D.check(lib.dpx_stage_similarity_graph(img, w, h, stride, ch, fl, graph, s))
    D.check(lib.dpx_stage_trivial_cross(graph, w, h, s))
    D.check(lib.dpx_stage_heuristic_cross(graph, st["graph_aux"].data_ptr(), w, h, s))
    D.check(lib.dpx_stage_cells(graph, w, h, diagram, edges, s))
    if c["smooth"]:
        D.check(lib.dpx_stage_subdivide(img, w, h, stride, ch, fl, graph, diagram, st["diagram_aux"].data_ptr(),
                                        edges, st["edges_aux"].data_ptr(), s))
    D.check(lib.dpx_stage_triangulate(diagram, edges, w, h, s))
    D.check(lib.dpx_stage_present(img, w, h, stride, ch, fl, diagram, edges, st["view"], st["window"].data_ptr(),
                                  4 * c["window_w"], s))
    return st["window"], st["graph"], st["diagram"].view(torch.int32), st["edges"]


def run(state):
    c = state["case"]
    path = c["path"]
    if path == "batch":
        state["ctx"].run(state["d_in"], state["d_out"], state["items"], torch.cuda.current_stream())
        return state["d_out"]
    if path == "plan":
        state["plan"].run(state["d_in"], state["d_out"], torch.cuda.current_stream())
        return state["d_out"]
    if path == "served":
        tickets = [state["srv"].submit(s, f, o) for s, f, o in zip(state["sids"], state["frames"], state["outs"])]
        for t in tickets:
            D.check(state["srv"].wait(t))
        return state["outs"]
    if path == "chains":
        return _run_chains(state)
    if path == "viewer":
        return _run_viewer(state)
    if path == "frame":
        return D.frame(state["img"], c["width"], c["height"], c["channels"], scale=c["scale"],
                       subdivide=c["smooth"], flags=c["flags"])
    diagram, edges, graph = D.launch_kernel(state["img"], c["width"], c["height"], c["smooth"], state["pos"],
                                            state["color"])
    return diagram.view(np.int32), edges, graph, state["pos"].view(torch.int32), state["color"]


def work(case):
    """Bytes each pass cannot do without: inputs read once, outputs written
    once.  The path computes on whole numbers; the multiply-adds of the
    luma (three a pixel) are what counts as arithmetic."""
    S, ch, path = case["scale"], case["channels"], case["path"]
    n = sum(w * h for w, h in (_size(case, k) for k in range(case["count"])))
    if path in ("batch", "plan", "served"):
        pal = 1024 * case["count"] if case["kind"] == STREAM else 0
        return {"bytes": n * ch + pal + n * 4 * S * S, "flops": 6 * n}
    if path == "chains":
        return {"bytes": n + 4 * n, "flops": 0}
    diagram = n * CELL * 8 + 4 * n + n  # slots, edge counts, graph
    if path == "viewer":
        return {"bytes": n * ch + diagram + 4 * case["window_w"] * case["window_h"], "flops": 6 * n}
    if path == "frame":
        return {"bytes": n * ch + n * 4 * S * S + 5 * n, "flops": 6 * n}
    return {"bytes": n * ch + diagram + n * CELL * 12, "flops": 6 * n}


def exact(case, seed):
    """Every output is bytes or whole numbers: there is nothing to round."""
    return None
