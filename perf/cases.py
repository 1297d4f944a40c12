"""The calls whose speed is measured: renders of resident terrains through
the library's public entry points, from one small frame to a batch of 64
mixed views and a served request mix.

A case says which terrain, which entry point, the screen and how many frames
or views one pass renders; the camera poses come from the seed.  Terrains are
what a program keeps resident: they are made and uploaded once per process.
A pass renders every pose of its state into that pose's own framebuffer
(colour16 and int32 depth, whole) and returns the framebuffers.  All outputs
are integers, so no case has a 64-bit value to be compared with (exact).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.abspath("rle-based-voxel-raycasting_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import rlevox  # noqa: E402
import workloads  # noqa: E402

# Resident terrains (workloads.SCENES): a 512^2 x 256 map, two 4096^2 x 1024
# maps of about 6 runs per column, and a 4096^2 x 1024 map with the cave
# settings and mip count of the 16384^2 one (about 8 runs per column).
TERRAINS = ("small", "plain", "plain2", "caved")

# Screen sizes of the multi-view cases, dealt in turn (the seed shuffles
# their order): the uniform mix of a batch over several scenes, small
# previews, a served mix weighted 10:7:3, and sizes off every tile width.
MIXES = {
    "uniform": list(workloads.C4_RESOLUTIONS),
    "small": [(320, 240), (640, 480)],
    "served": [(640, 480)] * 10 + [(1920, 1080)] * 7 + [(3840, 2160)] * 3,
    "odd": [(333, 251), (854, 480), (1366, 768), (1021, 1021), (1600, 901), (97, 61), (2049, 1153)],
}


class _Buf:
    """A torch tensor as the binding takes device buffers."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


_kept = {}


def _ctx():
    if "ctx" not in _kept:
        torch.cuda.init()
        _kept["ctx"] = rlevox.Context(0)
        _kept["stream"] = _kept["ctx"].stream()
    return _kept["ctx"]


def _terrain(name):
    """(host scene, resident scene) of a terrain."""
    if name not in _kept:
        ctx = _ctx()
        if name == "small":
            host = workloads.gen("c1", seed=1)
        elif name == "caved":
            p = dict(workloads.SCENES["c3"], size_xz=4096)
            host = rlevox.gen_scene(p["size_xz"], p["size_y"], p["nmips"], p["octaves"], 1,
                                    p["persistence"], p["hmin"], p["hmax"], p["cave_layers"],
                                    p["cave_max_layers"])
        else:
            host = workloads.gen("c2", seed=1 if name == "plain" else 2)
        _kept[name] = (host, ctx.upload(host.mips))
    return _kept[name]


def _poses(view, mip0, n, seed):
    if view == "flight":    # 10-200 voxels above the ground along one path
        return workloads.flythrough(mip0, frames=max(n, 2), seed=seed)[:n]
    if view == "grazing":   # pitch within 5 degrees of level, up or down
        return workloads.grazing(mip0, n, seed=seed)
    if view == "hills":     # among the hills: most lines end at nearby ground
        return workloads.random_views(mip0, n, seed=seed, alt=(2.0, 20.0), pitch=(0.02, 0.3))
    if view == "high":      # from far above, looking down
        return workloads.random_views(mip0, n, seed=seed, alt=(300.0, 1500.0), pitch=(0.3, 1.2))
    return workloads.random_views(mip0, n, seed=seed)


def _frames(name, terrain, entry, view, W, H, frames, mip_distance=0, far_distance=0, post=0):
    return {"name": name, "kind": "frames", "terrain": terrain, "entry": entry, "view": view,
            "W": W, "H": H, "frames": frames, "mip_distance": mip_distance,
            "far_distance": far_distance, "post": post}


def _views(name, kind, mix, views, graph):
    return {"name": name, "kind": kind, "mix": mix, "views": views, "graph": graph}


def listed():
    return [
        # the smallest call: one preview frame of a small map, where launches
        # and the wait for the frame count
        _frames("frame_320x240", "small", "render", "random", 320, 240, 1),
        # a small frame of a full-size map (half of the served requests)
        _frames("frame_640x480", "plain", "render", "random", 640, 480, 4),
        # the headline frame, rendered one at a time by an interactive program
        _frames("frame_1080p", "plain", "render", "flight", 1920, 1080, 4),
        # the headline flythrough as a program that queues frames on a stream
        # runs it: ray map and the three stages of each frame in order
        _frames("flight_1080p", "plain", "stages", "flight", 1920, 1080, 16),
        # a laptop screen: sizes that are no multiple of a tile or of four,
        # eye among the hills
        _frames("hills_1366x768", "plain", "render", "hills", 1366, 768, 4),
        # frames enqueued without any allocation, as under graph capture
        _frames("noalloc_1280x720", "plain", "noalloc", "random", 1280, 720, 8),
        # a map view from far above, nearer mip switch, no smoothing
        _frames("high_1080p", "plain", "render", "high", 1920, 1080, 4, 512, 0,
                rlevox.POST_COMPOSE),
        # ordinary 4K frames
        _frames("frame_4k", "plain", "render", "random", 3840, 2160, 4),
        # 4K grazing views over the caved terrain: the longest traversals
        _frames("grazing_4k", "caved", "render", "grazing", 3840, 2160, 4),
        # a handful of previews packed into one launch
        _views("batch_16_small", "batch", "small", 16, False),
        # the batched configuration: 64 views, uniform sizes, captured graph
        _views("batch_64", "batch", "uniform", 64, True),
        # a burst of requests on the server, delivered on the device
        _views("serve_40", "serve", "served", 40, True),
    ]


def draw(rng):
    kind = rng.choice(["frames"] * 6 + ["batch"] * 3 + ["serve"])
    if kind != "frames":
        mix = "served" if kind == "serve" and rng.random() < 0.5 else rng.choice(sorted(MIXES))
        views = int(round(math.exp(rng.uniform(math.log(2), math.log(56)))))
        return _unnamed(_views("", kind, mix, views, kind == "serve" or rng.random() < 0.5))
    W = int(round(math.exp(rng.uniform(math.log(200), math.log(3840)))))
    H = max(16, int(W * rng.uniform(0.4, 1.0)))
    frames = rng.randint(1, max(1, min(8, int(32e6 / (W * H)))))
    entry = rng.choice(["render", "render", "stages", "noalloc"])
    if entry == "noalloc" and W > 1600:  # the fixed scratch holds no larger view for certain
        entry = "stages"
    return _unnamed(_frames("", rng.choice(TERRAINS), entry,
                            rng.choice(["flight", "random", "hills", "high", "grazing"]), W, H,
                            frames, rng.choice([0, 0, 0, 300, 512, 4096]),
                            rng.choice([0, 0, 0, 5000, 30000]),
                            rng.choice([0, 0, 0, rlevox.POST_COMPOSE])))


def _unnamed(case):
    return {k: v for k, v in case.items() if k != "name"}


def _sizes(case):
    if case["kind"] == "frames":
        return [(case["W"], case["H"])] * case["frames"]
    mix = MIXES[case["mix"]]
    return [mix[i % len(mix)] for i in range(case["views"])]


def prepare(case, seed):
    ctx = _ctx()
    seed = int(seed) % (1 << 31)
    sizes = _sizes(case)
    state = {"case": case, "ctx": ctx, "stream": _kept["stream"]}
    if case["kind"] == "frames":
        host, scene = _terrain(case["terrain"])
        state["scene"] = scene
        state["poses"] = _poses(case["view"], host.mips[0], len(sizes), seed)
        state["params"] = rlevox.RenderParams(case["mip_distance"], case["far_distance"],
                                              case["post"], 0)
        if case["entry"] == "stages":
            # scratch of a program that drives the stages itself
            lines = max(rlevox.raymap(p, W, H).map_line_count
                        for p, (W, H) in zip(state["poses"], sizes))
            W, H = sizes[0]
            state["scratch"] = [_Buf(torch.empty(n, dtype=torch.int32, device="cuda"))
                                for n in (max(lines, 1) * W, max(lines, 1) * 2)]
            state["composed"] = _Buf(torch.empty(H, W, dtype=torch.int16, device="cuda"))
    else:
        rng = np.random.default_rng(seed)
        sizes = [sizes[i] for i in rng.permutation(len(sizes))]
        terrains = [_terrain(t) for t in ("plain", "plain2")]
        state["scenes"], state["poses"] = [], []
        for i in range(len(sizes)):
            host, scene = terrains[int(rng.integers(len(terrains)))]
            state["scenes"].append(scene)
            state["poses"] += workloads.random_views(host.mips[0], 1, int(rng.integers(1 << 30)))
    state["sizes"] = sizes
    # zeroed once, as a program clears its framebuffers when it makes them
    state["colour"] = [_Buf(torch.zeros(H, W, dtype=torch.int16, device="cuda")) for W, H in sizes]
    state["depth"] = [_Buf(torch.zeros(H, W, dtype=torch.int32, device="cuda")) for W, H in sizes]
    state["out"] = ([b.tensor for b in state["colour"]], [b.tensor for b in state["depth"]])
    if case["kind"] != "frames":
        # outputs as one array each: a pass renders more views than are listed apart
        colour = torch.zeros(sum(W * H for W, H in sizes), dtype=torch.int16, device="cuda")
        depth = torch.zeros(colour.numel(), dtype=torch.int32, device="cuda")
        ends = np.cumsum([W * H for W, H in sizes])
        state["colour"] = [_Buf(colour[e - W * H:e]) for e, (W, H) in zip(ends, sizes)]
        state["depth"] = [_Buf(depth[e - W * H:e]) for e, (W, H) in zip(ends, sizes)]
        state["out"] = (colour, depth)
    if case["kind"] == "batch":
        state["views"] = [rlevox.make_view(s, p, W, H, c, d) for s, p, (W, H), c, d in
                          zip(state["scenes"], state["poses"], sizes, state["colour"],
                              state["depth"])]
    if case["kind"] == "serve":
        state["server"] = rlevox.Server(ctx, memory_budget=16 << 30, max_batch_views=48, streams=3)
    torch.cuda.synchronize()  # the library's streams do not wait for torch's
    return state


def run(state):
    case, ctx, stream = state["case"], state["ctx"], state["stream"]
    if case["kind"] == "batch":
        ctx.render_batch(state["views"], stream=stream, graph=case["graph"])
    elif case["kind"] == "serve":
        server = state["server"]
        tickets = [server.submit(s, p, W, H, c, d) for s, p, (W, H), c, d in
                   zip(state["scenes"], state["poses"], state["sizes"], state["colour"],
                       state["depth"])]
        for t in tickets:
            server.wait(t)
    else:
        scene, prm, entry = state["scene"], state["params"], case["entry"]
        for p, (W, H), c, d in zip(state["poses"], state["sizes"], state["colour"],
                                   state["depth"]):
            if entry == "render":
                ctx.render(scene, p, W, H, c, d, prm, stream)
            elif entry == "noalloc":
                ctx.render_noalloc(scene, p, W, H, c, d, prm, stream)
            else:
                rm = rlevox.raymap(p, W, H, prm.mip_distance, prm.far_distance)
                raybuf, clip = state["scratch"]
                ctx.render_raybuf(scene, rm, raybuf, clip, stream)
                smooth = case["post"] != rlevox.POST_COMPOSE
                ctx.compose(rm, raybuf, clip, state["composed"] if smooth else c, d, stream)
                if smooth:
                    ctx.gapfill(W, H, state["composed"], d, c, stream)
    return state["out"]


def work(case):
    """What any renderer of these frames moves: per pixel the pointer-map
    entry (8 bytes), run (2) and colour (2) of the voxel it shows, and the
    colour (2) and depth (4) it writes.  The path has no contraction."""
    return {"bytes": 18.0 * sum(W * H for W, H in _sizes(case)), "flops": 0.0}


def exact(case, seed):
    return None  # every output is a whole number
