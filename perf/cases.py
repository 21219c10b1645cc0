"""What is timed when this framework's speed is worked on: the cases, their inputs, and one pass of each.

A case is one of six ways in which a program uses the library:

  job      one mosaic on device buffers (mh_generate_device): target and library resident, grid and image come out
  batch    a fixed set of jobs as one fused launch per stage, replayed from a graph (mh_batch_*)
  served   jobs queued on the continuous-batching server, all at once or one call each, until all are done (mh_server_*)
  oneshot  what one run of the command-line tool does: the materials' pixels go up, one mosaic comes back to the host
  anneal   the optimiser alone on a grid in host memory (mh_anneal)
  ingest   a material library from host images of several sizes, and its Lab table (mh_library_from_images)

Targets are gradients with coloured blobs and noise, materials flat colours with noise, as the benchmark's workloads have
them; `colours` says whether the materials' colours are spread over the cube ("flat") or lie in three clusters ("mix").
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mosaic-art-rust_amd")


def _binding():
    if "mosaic_hip" not in sys.modules:
        spec = importlib.util.spec_from_file_location("mosaic_hip", os.path.join(_PKG, "mosaic_hip.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules["mosaic_hip"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["mosaic_hip"]


_ctx = None


def _context():
    """The context that a single-job program keeps (servers have one of their own)."""
    global _ctx
    if _ctx is None:
        _ctx = _binding().Context(0)
    return _ctx


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the smallest jobs of the served stream: a thumbnail of 300 cells, launches and latency
        dict(name="job_thumb", kind="job", width=320, height=240, gw=20, gh=15, n=1000, msize=64, colours="mix",
             usage=3, weight=0.25, color=0.4, iters=1000, score=0),
        # the command line's defaults: 50 x 28 cells, 500 materials, usage 3, weight 0.3, 1,000 proposals, colour 0.3
        dict(name="job_default", kind="job", width=1280, height=720, gw=50, gh=28, n=500, msize=64, colours="flat",
             usage=3, weight=0.3, color=0.3, iters=1000, score=0),
        # the graphical generator: Euclidean score, no adjustment, no optimiser; a laptop screen cut raggedly
        dict(name="job_gui", kind="job", width=1366, height=768, gw=97, gh=41, n=777, msize=64, colours="flat",
             usage=6, weight=0.3, color=0.0, iters=0, score=1),
        # the benchmark's ordinary job
        dict(name="job_medium", kind="job", width=1920, height=1080, gw=80, gh=60, n=1500, msize=128, colours="flat",
             usage=4, weight=0.25, color=0.4, iters=2000, score=0),
        # the gallery's job: 206 x 116 cells of 19 x 19 pixels, 2,849 materials, usage 9
        dict(name="job_gallery", kind="job", width=4000, height=2250, gw=206, gh=116, n=2849, msize=64, colours="mix",
             usage=9, weight=0.25, color=0.4, iters=2000, score=0),
        # the benchmark's largest job
        dict(name="job_large", kind="job", width=4000, height=2400, gw=200, gh=120, n=10000, msize=64, colours="mix",
             usage=5, weight=0.25, color=0.4, iters=20000, score=0),
        # the benchmark's batch: 64 jobs of 20-160 x 15-120 cells, here on eight libraries of 256-4,096
        dict(name="batch_64", kind="batch", jobs=64, libs=8, lo=256, hi=4096),
        # a backlog of the served stream (300-24,000 cells, libraries of 1,000-10,000), every job queued at once
        dict(name="served_backlog", kind="served", jobs=512, lo=300, hi=24000, at_once=True),
        # a quiet server: a few ordinary requests, one call each
        dict(name="served_few", kind="served", jobs=6, lo=300, hi=6000, at_once=False),
        # one run of the command-line tool on the benchmark's ordinary job, from pixels in host memory to the image there
        dict(name="oneshot_medium", kind="oneshot", width=1920, height=1080, gw=80, gh=60, n=1500, msize=128,
             colours="flat", usage=4, weight=0.25, color=0.4, iters=2000, score=0),
        # the optimiser's own entry point, a long run that cools
        dict(name="anneal_long", kind="anneal", gw=160, gh=120, n=2500, iters=50000, t0=100.0, greedy=False),
        # material ingest, four sizes as the benchmark mixes them
        dict(name="ingest_mixed", kind="ingest", n=2000, big=96),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """Columns and rows of a 4:3 or 16:9 grid of lo..hi cells."""
    cells = _log(rng, lo, hi)
    aspect = rng.choice((4.0 / 3.0, 16.0 / 9.0))
    gw = max(1, int(round(math.sqrt(cells * aspect))))
    return gw, max(1, int(round(cells / gw)))


def draw(rng):
    kind = rng.choice(("job", "job", "job", "batch", "served", "oneshot", "anneal", "ingest"))
    if kind in ("job", "oneshot"):
        gw, gh = _grid(rng, 300, 24000 if kind == "job" else 5000)
        tw, th = rng.randint(10, 24), rng.randint(10, 24)
        if gw * gh > 8000:
            tw, th = min(tw, 20), min(th, 20)
        return dict(kind=kind, width=gw * tw + rng.randrange(tw), height=gh * th + rng.randrange(th), gw=gw, gh=gh,
                    n=_log(rng, 200, 10000) if kind == "job" else _log(rng, 200, 1500), msize=rng.choice((48, 64, 96)),
                    colours=rng.choice(("flat", "mix")), usage=rng.randint(3, 9), weight=rng.choice((0.1, 0.25, 0.3, 0.5)),
                    color=rng.choice((0.0, 0.3, 0.4)), iters=_log(rng, 500, 20000) if kind == "job" else _log(rng, 500, 2000),
                    score=rng.choice((0, 0, 1)))
    if kind == "batch":
        return dict(kind=kind, jobs=_log(rng, 4, 64), libs=rng.randint(1, 8), lo=256, hi=_log(rng, 512, 4096))
    if kind == "served":
        return dict(kind=kind, jobs=_log(rng, 4, 256), lo=300, hi=_log(rng, 3000, 24000), at_once=rng.random() < 0.5)
    if kind == "anneal":
        gw, gh = _grid(rng, 300, 24000)
        return dict(kind=kind, gw=gw, gh=gh, n=_log(rng, 100, 5000), iters=_log(rng, 1000, 40000),
                    t0=rng.choice((1.0, 10.0, 100.0)), greedy=rng.random() < 0.25)
    return dict(kind=kind, n=_log(rng, 64, 2000), big=rng.randint(48, 128))


# ----------------------------------------------------------------- inputs
def _gen(seed, part=0):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + part) & 0x7FFFFFFFFFFF)


def _to_u8(x):
    return x.round_().clamp_(0, 255).to(torch.uint8)


def _target(width, height, g):
    """height x width x 3: a diagonal gradient, blobs of colour, noise."""
    x = torch.arange(width, device="cuda", dtype=torch.float32)
    y = torch.arange(height, device="cuda", dtype=torch.float32)
    img = (127.5 * (x[None, :] / width + y[:, None] / height))[..., None].repeat(1, 1, 3)
    blobs = max(4, width * height // 300000)
    u = torch.rand((blobs, 5), device="cuda", generator=g)
    sigma = max(12.0, min(150.0, width / 12.0))
    for b in range(blobs):
        amp = torch.exp(-((x[None, :] - u[b, 0] * width) ** 2 + (y[:, None] - u[b, 1] * height) ** 2) / (2 * sigma * sigma))
        img += amp[..., None] * (255.0 * u[b, 2:] - img)
    img += 8.0 * torch.randn(img.shape, device="cuda", generator=g)
    return _to_u8(img).contiguous()


def _colours(n, colours, g):
    if colours == "mix":
        means = 255.0 * torch.rand((3, 3), device="cuda", generator=g)
        which = torch.randint(0, 3, (n,), device="cuda", generator=g)
        return means[which] + 12.0 * torch.randn((n, 3), device="cuda", generator=g)
    return torch.randint(0, 256, (n, 3), device="cuda", generator=g).float()


def _materials(n, w, h, colours, g):
    """n x h x w x 3 in host memory: flat colours and noise."""
    out = torch.empty((n, h, w, 3), dtype=torch.uint8, device="cuda")
    col = _colours(n, colours, g)
    step = max(1, (1 << 26) // (w * h * 3))
    for s in range(0, n, step):
        part = 12.0 * torch.randn((min(step, n - s), h, w, 3), device="cuda", generator=g)
        out[s:s + step] = _to_u8(part.add_(col[s:s + step, None, None, :]))
    return out.cpu().numpy()


class _Service:
    """What a serving program keeps: one server, and the four resident libraries of its context."""

    def __init__(self):
        self.ctx = _binding().Context(0)
        self.libs = [self.ctx.library_from_pixels(_materials(n, 64, 64, "mix", _gen(1, n))) for n in (1000, 2500, 5000, 10000)]
        self.server = self.ctx.server()

    def close(self):
        self.server.close()
        for lib in self.libs:
            lib.close()
        self.ctx.close()


_serving = None


def _service(wanted):
    """The service, made once; a program that does other work has none."""
    global _serving
    if wanted and _serving is None:
        _serving = _Service()
    elif not wanted and _serving is not None:
        _serving.close()
        _serving = None
    return _serving


def _job_params(case, seed):
    return _binding().JobParams(case["gw"], case["gh"], case["usage"], case["weight"], case["color"],
                                1 if case["iters"] > 0 else 0, case["iters"], 100.0, 0.99995, int(seed) & 0xFFFFFFFF, case["score"])


def _many(rng, case):
    """The jobs of a batch or a served backlog: (library, columns, rows, usage), cells of 16 x 16 pixels."""
    jobs = []
    for _ in range(case["jobs"]):
        if case["kind"] == "batch":
            gw, gh, lib = int(rng.integers(20, 161)), int(rng.integers(15, 121)), int(rng.integers(0, case["libs"]))
        else:
            cells = math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))
            gw = int(round(math.sqrt(cells * (16.0 / 9.0 if rng.integers(0, 2) else 4.0 / 3.0))))
            gh, lib = max(1, int(round(cells / gw))), int(rng.integers(0, 4))
        jobs.append((lib, gw, gh, int(rng.integers(3, 6))))
    return jobs


def _shape_rng(case):
    """Sizes of a set of jobs belong to the case, their pixels to the seed."""
    return np.random.default_rng([case["jobs"], case["hi"], case.get("libs", 0)])


def _images(case, seed):
    sizes = [(48, 48), (64, 64), (case["big"], 64), (128, case["big"])]
    sets = [_materials((case["n"] + 3 - k) // 4, w, h, "flat", _gen(seed, k)) for k, (w, h) in enumerate(sizes)]
    return [sets[i % 4][i // 4] for i in range(case["n"])]


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    mh, service = _binding(), _service(case["kind"] == "served")
    if kind in ("job", "oneshot"):
        tw, th = case["width"] // case["gw"], case["height"] // case["gh"]
        target = _target(case["width"], case["height"], g)
        mats = _materials(case["n"], case["msize"], case["msize"], case["colours"], g)
        if kind == "oneshot":
            return dict(case=case, seed=seed, target=target.cpu().numpy(), mats=mats)
        s = dict(case=case, target=target, lib=_context().library_from_pixels(mats), prm=_job_params(case, seed),
                 grid=torch.zeros(case["gw"] * case["gh"], dtype=torch.int32, device="cuda"),
                 image=torch.zeros((case["gh"] * th, case["gw"] * tw, 3), dtype=torch.uint8, device="cuda"))
    elif kind in ("batch", "served"):
        rng = _shape_rng(case)
        jobs = _many(rng, case)
        if kind == "batch":
            mats = [_materials(int(round(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]))))), 64, 64, "flat", g)
                    for _ in range(case["libs"])]
            ctx = _context()
            libs = [ctx.library_from_pixels(m) for m in mats]
        else:
            ctx, libs = service.ctx, service.libs
        cw, ch = max(j[1] for j in jobs) * 16 + 64, max(j[2] for j in jobs) * 16 + 64
        canvas = [_target(cw, ch, g) for _ in range(4)]  # the jobs' targets are crops of these
        cells = [j[1] * j[2] for j in jobs]
        grid = torch.zeros(sum(cells), dtype=torch.int32, device="cuda")
        image = torch.zeros(sum(cells) * 768, dtype=torch.uint8, device="cuda")
        mj, at = [], 0
        for k, (lib, gw, gh, usage) in enumerate(jobs):
            ox, oy = int(rng.integers(0, cw - gw * 16 + 1)), int(rng.integers(0, ch - gh * 16 + 1))
            p = mh.JobParams(gw, gh, usage, 0.25, 0.4, 1, 1000, 100.0, 0.99995, k, 0)
            mj.append(ctx.job(libs[lib], canvas[k % 4].data_ptr() + (oy * cw + ox) * 3, gw * 16, gh * 16, p,
                              grid.data_ptr() + 4 * at, image.data_ptr() + 768 * at, cw * 3))
            at += cells[k]
        s = dict(case=case, libs=libs, canvas=canvas, grid=grid, image=image, jobs=mj, service=service)
        if kind == "batch":
            torch.cuda.synchronize()
            s["batch"] = ctx.batch(mj)
            s["batch"].set_graph(True)
    elif kind == "anneal":
        lab = torch.rand((case["n"], 3), device="cuda", generator=g) * torch.tensor([100.0, 160.0, 160.0], device="cuda")
        lab -= torch.tensor([0.0, 80.0, 80.0], device="cuda")
        grid = torch.randint(0, case["n"], (case["gw"] * case["gh"],), device="cuda", generator=g, dtype=torch.int32)
        s = dict(case=case, seed=seed, lib=_context().library_from_lab(lab.cpu().numpy()), grid=grid.cpu().numpy())
    else:
        s = dict(case=case, images=_images(case, seed))
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------- one pass
def _costs(r):
    return {k: r[k] for k in ("initial_cost", "final_cost", "best_cost", "improved_count", "accepted_count", "evaluated")}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "job":
        _context().generate_device(s["lib"], s["target"].data_ptr(), case["width"], case["height"], s["prm"],
                                   s["grid"].data_ptr(), s["image"].data_ptr())
        return s["grid"], s["image"]
    if kind == "batch":
        s["batch"].run()
        return s["grid"], s["image"]
    if kind == "served":
        server = s["service"].server
        if case["at_once"]:
            server.submit_many(s["jobs"])
            server.drain()
        else:
            for t in [server.submit(j) for j in s["jobs"]]:
                server.wait(t)
        return s["grid"], s["image"]
    if kind == "oneshot":
        lib = _context().library_from_pixels(s["mats"])
        r = _context().generate(lib, s["target"], case["gw"], case["gh"], case["usage"], case["weight"], case["color"],
                                case["iters"] > 0, case["iters"], seed=int(s["seed"]) & 0xFFFFFFFF, score_mode=case["score"])
        lib.close()
        return {"grid": r["grid"], "image": r["image"], "place": r["place"], "anneal": _costs(r["anneal"])}
    if kind == "anneal":
        r = _context().anneal(s["lib"], s["grid"], case["gw"], case["gh"], case["iters"], case["t0"], 0.99995,
                              int(s["seed"]) & 0xFFFFFFFF, case["greedy"])
        return {"grid": r["grid"], "anneal": _costs(r["result"])}
    lib = _context().library_from_images(s["images"])
    lab = lib.lab()
    lib.close()
    return lab


# ------------------------------------------------- what a pass cannot avoid
def _job_work(cells, px, n, iters, colour):
    """Bytes: the target read, the Labs and the tiles in use read, grid and image written.  Operations: a Lab conversion
    (about 60) and an output pixel (about 40 with the adjustment), 100 candidates a cell, ten neighbours a proposal."""
    return {"bytes": 6 * px + 12 * n + 4 * cells + 3 * px * min(n, cells) // max(cells, 1) + 40 * iters,
            "flops": px * (60 + (40 if colour else 0)) + cells * min(n, 100) * 8 + iters * 160}


def work(case):
    kind = case["kind"]
    if kind in ("job", "oneshot"):
        cells = case["gw"] * case["gh"]
        px = cells * (case["width"] // case["gw"]) * (case["height"] // case["gh"])
        w = _job_work(cells, px, case["n"], case["iters"], case["color"] > 0)
        if kind == "oneshot":
            mpx = case["n"] * case["msize"] ** 2
            w = {"bytes": w["bytes"] + 3 * mpx, "flops": w["flops"] + 60 * mpx}
        return w
    if kind in ("batch", "served"):
        parts = [_job_work(gw * gh, gw * gh * 256, 1000, 1000, True) for _, gw, gh, _ in _many(_shape_rng(case), case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "anneal":
        cells = case["gw"] * case["gh"]
        return {"bytes": 8 * cells + 12 * case["n"] + 40 * case["iters"], "flops": 160 * case["iters"]}
    px = case["n"] * (48 * 48 + 64 * 64 + case["big"] * 64 + 128 * case["big"]) / 4
    return {"bytes": 3 * px + 12 * case["n"], "flops": 60 * px}


# ------------------------------------------------------------ in 64 bits
def _lab64(rgb):
    """CIE Lab (D65) of sRGB bytes, float64, over the last axis."""
    c = rgb.to(torch.float64) / 255.0
    lin = torch.where(c <= 0.04045, c / 12.92, ((c + 0.055) / 1.055) ** 2.4)
    m = torch.tensor([[0.4124564, 0.3575761, 0.1804375], [0.2126729, 0.7151522, 0.0721750], [0.0193339, 0.1191920, 0.9503041]],
                     dtype=torch.float64, device=rgb.device)
    white = torch.tensor([0.95047, 1.0, 1.08883], dtype=torch.float64, device=rgb.device)
    t = sum(lin[..., k:k + 1] * m[:, k] for k in range(3)) / white
    f = torch.where(t > 216.0 / 24389.0, t ** (1.0 / 3.0), 841.0 / 108.0 * t + 4.0 / 29.0)
    x, y, z = f[..., 0], f[..., 1], f[..., 2]
    return torch.stack([116.0 * y - 16.0, 500.0 * (x - y), 200.0 * (y - z)], -1)


def exact(case, seed):
    """The material Lab means; the other kinds give material indices, pixels and sums that depend on every choice before them."""
    if case["kind"] != "ingest":
        return None
    images = _images(case, seed)
    out = np.empty((case["n"], 3))
    for k in range(4):
        if k < case["n"]:
            part = torch.from_numpy(np.stack(images[k::4])).cuda()
            out[k::4] = _lab64(part).mean((1, 2)).cpu().numpy()
    return out
