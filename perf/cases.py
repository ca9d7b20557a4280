"""Performance cases: what programs have this framework render, through its
public entry points, with the inputs such programs hold.

Families (the "kind" of a case):
  plane    one colour plane in device memory, pixel-wise or grain-wise
           (Context.render_device), the integrator call every other path makes
  planes   the three planes of one RGB frame in device memory
           (Context.render_planes_device)
  frame    an interleaved RGB frame in device memory to 8-bit RGB in device
           memory (Context.render_frame_device)
  host     an interleaved RGB frame in host memory to 8-bit RGB in host memory
           (host.render_rgb), what the command line does with a decoded file
  batch    images of uneven sizes and parameters, planned once and run many
           times (capi.Batch)
  adaptive an RGB frame rendered with learned per-pixel sample budgets
           (budget.render_adaptive_frame)
  predict  the error model's inference over a plane: features, predictions,
           budgets
  train    one minibatch gradient of the error model

Sizes and parameters are those of film_grain_amd/workloads.py, of the command
line's defaults, of budget.C5 and of the parity tests' ranges (radius 0.05 to
0.5 px, N 16 to 1024, zoom 0.5 to 4, constant and lognormal radii).

Rendered planes are counts of covered samples times 1/N, decided by integer
random streams that every implementation has to reproduce bit for bit, so they
compare exactly and have no 64-bit reference of their own.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from film_grain_amd import budget, capi, host

DEV = "cuda:0"

_CTX = None


def _ctx() -> capi.Context:
    """The program's one context (its scratch grows once and is kept)."""
    global _CTX
    if _CTX is None:
        _CTX = capi.Context(0)
    return _CTX


# ------------------------------------------------------------------ cases ----

def listed() -> list[dict]:
    return [
        # The smallest call: a viewer's region-of-interest preview with the
        # command line's default radius and sample count.  Launches and waits
        # are what it costs.
        dict(name="preview_96x64", kind="plane", algo="pixel", w=96, h=64, radius=0.1, sd=0.0, zoom=1.0, n=32,
             field="waves"),
        # The plain single-plane workload (workloads.WORKLOADS["pixel-c1"]).
        dict(name="plane_256", kind="plane", algo="pixel", w=256, h=256, radius=0.12, sd=0.0, zoom=1.0, n=64,
             field="waves"),
        # An ordinary plane of odd sides at a fractional zoom, with wide
        # grains of uneven radius and a sample count that is no multiple of
        # 32: no tuned launch shape covers it.
        dict(name="plane_odd_lognormal", kind="plane", algo="pixel", w=701, h=533, radius=0.2, sd=0.08, zoom=1.5,
             n=100, field="waves"),
        # The headline frame: 1080p RGB to 4K, lognormal radii, N = 256
        # (workloads.WORKLOADS["pixel-c2"]), planes resident on the device.
        dict(name="planes_4k_rgb", kind="planes", w=1920, h=1080, radius=0.1, sd=0.05, zoom=2.0, n=256,
             field="waves"),
        # The grain-wise workload at its full size
        # (workloads.WORKLOADS["grain-c3"]).
        dict(name="grain_4096", kind="plane", algo="grain", w=4096, h=4096, radius=0.05, sd=0.0, zoom=1.0, n=128,
             field="ramp"),
        # Grain-wise with lognormal radii on odd sides and zoomed, the choice
        # the automatic routing makes above N = 96.
        dict(name="grain_lognormal_odd", kind="plane", algo="grain", w=1021, h=767, radius=0.1, sd=0.03, zoom=2.0,
             n=128, field="waves"),
        # A 720p RGB video frame that stays on the device, lognormal radii,
        # N = 64: routed grain-wise by the reference's rule.
        dict(name="frame_720p_rgb", kind="frame", color="rgb", algo="auto", w=1280, h=720, radius=0.1, sd=0.05,
             zoom=1.0, n=64),
        # The command line with its defaults (constant radius, N = 32, luma)
        # on a decoded 1080p file: host memory to host memory.
        dict(name="host_1080p_luma", kind="host", color="luma", algo="auto", w=1920, h=1080, radius=0.1, sd=0.0,
             zoom=1.0, n=32),
        # A small uneven batch out of workloads.batch_images' ranges, replayed
        # from its plan.
        dict(name="batch_12", kind="batch", images=12, min_side=128, max_side=1024, pick=2024),
        # The learned-budget frame (budget.C5) at the error fixed N = 512
        # reaches.
        dict(name="adaptive_1080p", kind="adaptive", w=1920, h=1080, radius=0.1, sd=0.05, zoom=1.0, n_min=16,
             n_max=1024, rmse255=4.8),
        # The error model over one 1080p plane: features, predictions,
        # budgets.
        dict(name="predict_1080p", kind="predict", w=1920, h=1080, radius=0.1, sd=0.05, zoom=1.0),
        # One minibatch of budget.train: 65536 rows, the likelihood loss.
        dict(name="train_65536", kind="train", rows=65536, loss="nll"),
    ]


def _log_uniform(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _cost(w, h, zoom, radius, sd, n, planes=1) -> float:
    """Rough work of a render: grains drawn and pixel-samples decided."""
    grains = w * h * 0.9 / (math.pi * (radius * radius + sd * sd))
    return planes * (grains * (20.0 + 0.05 * n) + w * h * zoom * zoom * n)


# the headline frame's
_MAX_COST = _cost(1920, 1080, 2.0, 0.1, 0.05, 256, 3)


def _draw_render(rng, max_side: int, planes: int, zooms, cap: float):
    """Sides, radius law, zoom and N of a render that costs at most cap."""
    while True:
        w, h = round(_log_uniform(rng, 64, max_side)), round(_log_uniform(rng, 64, max_side))
        radius = _log_uniform(rng, 0.05, 0.5)
        sd = radius * rng.uniform(0.05, 0.5) if rng.random() < 0.5 else 0.0
        zoom = rng.choice(zooms)
        n = rng.choice([16, 32, 64, 128, 256, 512, round(_log_uniform(rng, 16, 1024))])
        if _cost(w, h, zoom, radius, sd, n, planes) <= cap:
            return dict(w=w, h=h, radius=round(radius, 4), sd=round(sd, 5), zoom=zoom, n=n)


def draw(rng) -> dict:
    kind = rng.choice(["plane", "plane", "plane", "planes", "frame", "host", "batch", "adaptive", "predict", "train"])
    if kind == "plane":
        algo = rng.choice(["pixel", "grain"])
        return dict(kind=kind, algo=algo, field=rng.choice(["waves", "ramp"]),
                    **_draw_render(rng, 4096, 1, [0.5, 1.0, 1.0, 1.5, 2.0, 3.0, 4.0], 0.5 * _MAX_COST))
    if kind == "planes":
        return dict(kind=kind, field="waves", **_draw_render(rng, 1920, 3, [1.0, 1.5, 2.0], 0.5 * _MAX_COST))
    if kind in ("frame", "host"):
        color = rng.choice(["rgb", "luma"])
        return dict(kind=kind, color=color, algo=rng.choice(["auto", "pixel", "grain"]),
                    **_draw_render(rng, 1920, 3 if color == "rgb" else 1, [1.0, 1.0, 1.5, 2.0], 0.4 * _MAX_COST))
    if kind == "batch":
        return dict(kind=kind, images=rng.randint(2, 16), min_side=128, max_side=round(_log_uniform(rng, 192, 1024)),
                    pick=rng.randint(0, 1 << 20))
    if kind == "adaptive":
        return dict(kind=kind, w=round(_log_uniform(rng, 128, 1920)), h=round(_log_uniform(rng, 128, 1080)),
                    radius=round(rng.uniform(0.08, 0.2), 4), sd=round(rng.uniform(0.01, 0.05), 4), zoom=1.0,
                    n_min=16, n_max=rng.choice([256, 512, 1024]), rmse255=rng.choice([4.8, 6.9]))
    if kind == "predict":
        return dict(kind=kind, w=round(_log_uniform(rng, 64, 1920)), h=round(_log_uniform(rng, 64, 1920)),
                    radius=round(rng.uniform(0.05, 0.3), 4), sd=round(rng.uniform(0.0, 0.15), 4),
                    zoom=rng.choice([1.0, 1.5, 2.0]))
    return dict(kind=kind, rows=round(_log_uniform(rng, 1024, 1 << 21)), loss=rng.choice(["nll", "squared"]))


# ----------------------------------------------------------------- inputs ----

def _field(seed: int, w: int, h: int, shape: str = "waves"):
    """An intensity plane on the device as film_grain_amd/synth.py describes
    them: eight sinusoids with 2% noise and 10% flat patches (half black, half
    near white), or the noisy ramp."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = np.random.default_rng(seed)
    if shape == "ramp":
        f = (0.999 / max(w - 1, 1)) * torch.arange(w, device=DEV, dtype=torch.float32).expand(h, w)
        f = f + (torch.rand((h, w), device=DEV, generator=g) - 0.5) * 0.1
        return f.clamp_(0.0, 0.999).contiguous()
    x = torch.arange(w, device=DEV, dtype=torch.float32)[None, :] / w
    y = torch.arange(h, device=DEV, dtype=torch.float32)[:, None] / h
    acc = torch.zeros((h, w), device=DEV)
    amps = r.uniform(0.5, 1.0, 8)
    for k in range(8):
        acc += float(amps[k]) * torch.sin(2 * math.pi * (int(r.integers(1, 9)) * x + int(r.integers(1, 9)) * y) +
                                          float(r.uniform(0, 2 * math.pi)))
    f = 0.5 + 0.5 * acc / float(amps.sum())
    f += (torch.rand((h, w), device=DEV, generator=g) - 0.5) * 0.04
    for k in range(10):
        pw, ph = max(2, w // 10), max(2, h // 10)
        px, py = int(r.integers(0, max(1, w - pw))), int(r.integers(0, max(1, h - ph)))
        f[py:py + ph, px:px + pw] = (0.0, 0.98)[k % 2]
    return f.clamp_(0.0, 0.999).contiguous()


def _cli(case: dict, seed: int, n: int | None = None, algo: str = "pixel", color: str = "luma") -> host.CliArgs:
    return host.CliArgs(radius=case["radius"], radius_stddev=case["sd"],
                        radius_dist="lognorm" if case["sd"] > 0 else "const", zoom=case["zoom"],
                        iters=n or case["n"], seed=seed, algo=algo, sigma=0.8, color_mode=color)


def _desc(d) -> capi.PlaneDesc:
    return capi.make_desc(d.in_w, d.in_h, d.out_w, d.out_h, d.n_samples, d.dist_kind, d.seed, d.zoom, d.delta, d.rm,
                          d.radius_mean, d.log_mu, d.log_sigma)


def _lambda(ctx, plane, inv_e_pi_r2: float, norm=None):
    lam = torch.empty_like(plane)
    ctx.lambda_device(plane, inv_e_pi_r2, lam, norm)
    return lam


def _offsets(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _out(d):
    return torch.empty((d.out_h, d.out_w), device=DEV, dtype=torch.float32)


def _batch_image(r) -> dict:
    """workloads.batch_images' law for one image."""
    radius = float(r.uniform(0.05, 0.3))
    return dict(radius=radius, sd=float(r.uniform(0.0, 0.5)) * radius, zoom=1.0,
                n=int(r.choice([32, 64, 128, 256, 512])), rgb=bool(r.integers(0, 2)))


def _batch_images(case: dict) -> list[dict]:
    r = np.random.default_rng(case["pick"])
    out = []
    for _ in range(case["images"]):
        w, h = (int(v) for v in r.integers(case["min_side"], case["max_side"] + 1, 2))
        out.append(dict(w=w, h=h, **_batch_image(r)))
    return out


def _rows(ctx, case: dict, seed: int):
    """A minibatch as budget.train draws it: feature rows of random pixels and
    their N = 64 residuals."""
    w = h = 1024
    X = ctx.mlp_features(_field(seed, w, h), w, h, 1.0, 0.1, 0.05, 0.8, seed % 3)
    g = torch.Generator(device=DEV).manual_seed(seed)
    X = X[torch.randint(0, w * h, (case["rows"],), device=DEV, generator=g)].contiguous()
    u = budget.bf16_column(X, 0)
    s = torch.sqrt((u * (1 - u)).clamp(min=0.0)) / budget.SIGMA64_TO_S
    e = torch.round(torch.randn(u.shape, device=DEV, generator=g) * s * 4096) / 4096
    return X, e


def prepare(case: dict, seed: int):
    ctx = _ctx()
    kind = case["kind"]
    st = dict(case=case, ctx=ctx)
    if kind in ("plane", "planes"):
        algo = case.get("algo", "pixel")
        d, offs, offs_in = host.derive(_cli(case, seed, algo=algo), case["w"], case["h"])
        st["desc"] = _desc(d)
        st["offs"] = _offsets(offs_in if algo == "pixel" else offs)
        n = 3 if kind == "planes" else 1
        st["lams"] = [_lambda(ctx, _field(seed * 10 + c, case["w"], case["h"], case["field"]), d.inv_e_pi_r2)
                      for c in range(n)]
        st["outs"] = [_out(d) for _ in range(n)]
    elif kind in ("frame", "host"):
        rgb = torch.stack([_field(seed * 10 + c, case["w"], case["h"]) for c in range(3)], dim=2).contiguous()
        cli = _cli(case, seed, algo=case["algo"], color=case["color"])
        if kind == "host":
            st["cli"], st["rgb"] = cli, rgb.cpu().numpy()
            return st
        d, offs, offs_in = host.derive(cli, case["w"], case["h"])
        fd = capi.FrameDesc()
        fd.plane = _desc(d)
        fd.color_mode = capi.COLOR_RGB if case["color"] == "rgb" else capi.COLOR_LUMA
        pixel = d.algorithm == 2  # 1 grain-wise, 2 pixel-wise
        fd.algo = capi.ALGO_PIXEL if pixel else capi.ALGO_GRAIN
        fd.inv_e_pi_r2 = d.inv_e_pi_r2
        st["fd"], st["rgb"] = fd, rgb
        st["offs"] = _offsets(offs_in if pixel else offs)
        st["out"] = torch.empty((d.out_h, d.out_w, 3), device=DEV, dtype=torch.uint8)
    elif kind == "batch":
        planes = []
        for i, im in enumerate(_batch_images(case)):
            d, _offs, offs_in = host.derive(_cli(im, seed * 1000 + i), im["w"], im["h"])
            desc, offs = _desc(d), _offsets(offs_in)
            for c in range(3 if im["rgb"] else 1):
                lam = _lambda(ctx, _field((seed * 1000 + i) * 10 + c, im["w"], im["h"]), d.inv_e_pi_r2)
                planes.append((desc, lam, offs, _out(d)))
        st["outs"] = [p[3] for p in planes]
        st["batch"] = capi.Batch(ctx, planes)
    elif kind == "adaptive":
        d, _offs, offs_in = host.derive(_cli(case, seed, n=budget.N_REF, color="rgb"), case["w"], case["h"])
        offs = _offsets(offs_in)
        dps = []
        for c in range(3):
            u = _field(seed * 10 + c, case["w"], case["h"])
            norm = torch.empty_like(u)
            lam = _lambda(ctx, u, d.inv_e_pi_r2, norm)
            spec = budget.PlaneSpec(None, c, case["radius"], case["sd"], 0.8, case["zoom"], seed)
            dps.append(budget.DevicePlane(spec, _desc(d), lam, norm, offs, int(d.out_w), int(d.out_h)))
        st["planes"], st["bufs"], st["model"] = dps, budget.frame_buffers(dps), budget.ErrorModel.load(device=DEV)
    elif kind == "predict":
        st["u"] = _field(seed, case["w"], case["h"])
        st["out_w"], st["out_h"] = int(case["w"] * case["zoom"]), int(case["h"] * case["zoom"])
        n = st["out_w"] * st["out_h"]
        st["X"] = torch.empty((n, capi.MLP_FEATURES), dtype=torch.int16, device=DEV)
        st["pred"] = torch.empty(n, dtype=torch.float32, device=DEV)
        st["n"] = torch.empty(n, dtype=torch.int16, device=DEV)
        st["model"] = budget.ErrorModel.load(device=DEV)
        st["channel"] = seed % 3
    else:
        st["X"], st["e"] = _rows(ctx, case, seed)
        st["P"] = torch.from_numpy(budget.init_params(seed)).to(DEV)
        st["grad"] = torch.zeros(capi.MLP_PARAMS, dtype=torch.float32, device=DEV)
        st["loss"] = torch.zeros(1, dtype=torch.float32, device=DEV)
    return st


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "plane":
        ctx.render_device(case["algo"], st["desc"], st["lams"][0], st["offs"], st["outs"][0])
        return st["outs"][0]
    if kind == "planes":
        ctx.render_planes_device(st["desc"], st["lams"], st["offs"], st["outs"])
        return st["outs"]
    if kind == "frame":
        ctx.render_frame_device(st["fd"], st["rgb"], st["offs"], st["out"])
        return st["out"]
    if kind == "host":
        return host.render_rgb(st["cli"], st["rgb"], frame_on_device=True, with_planes=False)[0]
    if kind == "batch":
        st["batch"].run()
        return st["outs"]
    if kind == "adaptive":
        bufs = st["bufs"]
        outs, c = budget.render_adaptive_frame(ctx, st["model"], st["planes"], bufs, (case["rmse255"] / 255.0) ** 2,
                                               n_min=case["n_min"], n_max=case["n_max"])
        return dict(planes=outs, scale=c, pred=bufs.pred, budgets=bufs.budget)
    if kind == "predict":
        ctx.mlp_features(st["u"], st["out_w"], st["out_h"], case["zoom"], case["radius"], case["sd"], 0.8,
                         st["channel"], out=st["X"])
        st["model"].predict(ctx, st["X"], out=st["pred"])
        ctx.mlp_budget(st["pred"], None, st["pred"].numel(), _PREDICT_SCALE, 16, 1024, out=st["n"])
        return dict(features=st["X"].view(torch.bfloat16), pred=st["pred"], budgets=st["n"])
    st["grad"].zero_()
    st["loss"].zero_()
    ctx.mlp_grad(st["P"], st["X"], st["e"], st["grad"], st["loss"], loss_kind=case["loss"])
    return dict(grad=st["grad"], loss=st["loss"])


# budgets of about 50 to 700 samples for the spreads the model predicts
_PREDICT_SCALE = 1000.0 * budget.SIGMA64_TO_S


# ------------------------------------------------------------------- work ----

def _render_work(w, h, zoom, radius, sd, n, planes=1) -> tuple[float, float]:
    """(bytes, flops): lambda in, offsets in, plane out; per pixel-sample its
    sample point and one disk test (16), per grain its two centre coordinates
    and radius (40)."""
    out_px = round(w * zoom) * round(h * zoom)
    grains = w * h * 0.9 / (math.pi * (radius * radius + sd * sd))
    return planes * 4.0 * (w * h + out_px) + 8.0 * n, planes * (16.0 * out_px * n + 40.0 * grains)


_MLP_FLOPS = 2.0 * (12 * 64 + 64 * 64 + 64)  # per row, forward


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "batch":
        b = f = 0.0
        for im in _batch_images(case):
            db, df = _render_work(im["w"], im["h"], 1.0, im["radius"], im["sd"], im["n"], 3 if im["rgb"] else 1)
            b, f = b + db, f + df
        return dict(bytes=b, flops=f)
    if kind == "predict":
        rows = int(case["w"] * case["zoom"]) * int(case["h"] * case["zoom"])
        return dict(bytes=4.0 * case["w"] * case["h"] + rows * (32.0 + 4.0 + 2.0), flops=rows * (_MLP_FLOPS + 60.0))
    if kind == "train":
        return dict(bytes=case["rows"] * 36.0 + 2 * 4.0 * capi.MLP_PARAMS, flops=case["rows"] * 3.0 * _MLP_FLOPS)
    if kind == "adaptive":
        # budgets average about a third of the largest
        px = case["w"] * case["h"]
        b, f = _render_work(case["w"], case["h"], case["zoom"], case["radius"], case["sd"], case["n_max"] // 3, 3)
        return dict(bytes=b + 3 * px * 6.0, flops=f + 3 * px * _MLP_FLOPS)
    planes = 3 if kind == "planes" or case.get("color") == "rgb" else 1
    b, f = _render_work(case["w"], case["h"], case["zoom"], case["radius"], case["sd"], case["n"], planes)
    if kind in ("frame", "host"):  # interleaved f32 in, interleaved bytes out
        b = case["w"] * case["h"] * 12.0 + round(case["w"] * case["zoom"]) * round(case["h"] * case["zoom"]) * 3.0
    return dict(bytes=b, flops=f)


# ------------------------------------------------------------- comparison ----

def tolerance(case: dict):
    kind = case["kind"]
    if kind == "train":
        # the same bf16 operands with 64-bit sums move the gradient by 5e-7
        # (1024 to 2^20 rows); a bf16 operand on the other side of a rounding
        # adds 2e-6 at the fewest rows
        return dict(rel=1e-5)
    if kind in ("predict", "adaptive"):
        # the same bf16 operands with 64-bit sums move the predictions by
        # 1e-6 and about 1e-5 of the budgets by one sample, and with them the
        # planes by 6e-6; at the fewest pixels (64 x 64) one moved budget is
        # 2.4e-4 of them and 5e-5 in norm
        return dict(rel=1e-4, differ=5e-4)
    return "exact"


def _bf16(bits):
    return bits.view(torch.bfloat16).double()


def _mlp64(P, X):
    """The network in 64 bits: pre-activations of both layers and outputs."""
    P = P.double()
    W1, b1 = P[:1024].view(16, 64), P[1024:1088]
    W2, b2 = P[1088:5184].view(64, 64), P[5184:5248]
    z1 = X @ W1 + b1
    z2 = torch.relu(z1) @ W2 + b2
    return z1, z2, torch.relu(z2) @ P[5248:5312] + P[5312]


def _features64(u, out_w, out_h, zoom, radius, sd, channel):
    h, w = u.shape
    inv = torch.tensor(1.0, dtype=torch.float32) / torch.tensor(zoom, dtype=torch.float32)

    def index(n_out, n_in):
        x = (torch.arange(n_out, device=DEV, dtype=torch.float32) + 0.5) * inv.to(DEV)
        return torch.floor(x).long().clamp(0, n_in - 1)
    ix, iy = index(out_w, w), index(out_h, h)
    v = u.double()

    def at(dx, dy):
        return v[(iy + dy).clamp(0, h - 1)][:, (ix + dx).clamp(0, w - 1)]
    nb = torch.stack([at(dx, dy) for dy in (-1, 0, 1) for dx in (-1, 0, 1)])
    mean = nb.mean(dim=0)
    std = nb.var(dim=0, unbiased=False).sqrt()
    gx, gy = 0.5 * (at(1, 0) - at(-1, 0)), 0.5 * (at(0, 1) - at(0, -1))
    c = at(0, 0)
    one = torch.ones_like(c)
    cols = [c, mean, std, torch.hypot(gx, gy), c * (1 - c), one * (radius / 0.3), one * (sd / 0.15), one * 0.4,
            one * (zoom / 4)] + [one * float(channel == k) for k in range(3)] + [0 * one] * 4
    return torch.stack([x.reshape(-1) for x in cols], dim=1)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "train":
        ctx = _ctx()
        X, e = _rows(ctx, case, seed)
        x, t = _bf16(X), e.double()
        P = torch.from_numpy(budget.init_params(seed)).to(DEV)
        z1, z2, y = _mlp64(P, x)
        if case["loss"] == "nll":
            q = t * t * torch.exp((-2 * y).clamp(-80, 80))
            loss, gy = (y + 0.5 * q).sum(), (1 - q) / len(y)
        else:
            loss, gy = ((y - t) ** 2).sum(), 2 * (y - t) / len(y)
        Pd = P.double()
        dz2 = gy[:, None] * Pd[5248:5312] * (z2 > 0)
        h1 = torch.relu(z1)
        dz1 = (dz2 @ Pd[1088:5184].view(64, 64).t().contiguous()) * (z1 > 0)
        grad = torch.cat([(x.t().contiguous() @ dz1).reshape(-1), dz1.sum(0), (h1.t().contiguous() @ dz2).reshape(-1),
                          dz2.sum(0), torch.relu(z2).t().contiguous() @ gy, gy.sum()[None]])
        return dict(grad=grad, loss=loss[None])
    if kind == "predict":
        u = _field(seed, case["w"], case["h"])
        X = _features64(u, int(case["w"] * case["zoom"]), int(case["h"] * case["zoom"]), case["zoom"],
                        case["radius"], case["sd"], seed % 3)
        P = torch.from_numpy(np.load(budget.MODEL_PATH)).to(DEV)
        pred = torch.cat([_mlp64(P, x)[2] for x in X.split(1 << 20)])
        return dict(features=X, pred=pred, budgets=None)
    return None
