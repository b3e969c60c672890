"""Timed cases of the library's public entry points.

A case is one call (or the calls of one frame) that a program using the
library makes, over the range of sizes it is used at: light culling, whole
clustered-forward frames, the one-off environment stages, the plain and the
contraction cube filters, and training and evaluating the radiance network.
`prepare` makes the device inputs and the plan or network a program keeps,
`run` is one pass through `hellovulkan_amd.abi`, `work` the bytes and
operations no implementation can do without, `exact` the same result in 64
bits from plain torch (none of the library's code).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from hellovulkan_amd import abi

DEV = "cuda"
EYE, TARGET, FOVY, NEAR, FAR = (0.0, 1.0, 6.0), (0.0, 2.5, 0.0), 0.785398, 0.1, 100.0
SPEC, SPEC_MIPS, DIFF, LUT = 512, 10, 32, 512  # the maps a frame samples
PI = math.pi


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # per-frame culling at the reference application's cluster grid: the
        # smallest call of every frame, bound by its launches
        dict(name="cull_2560x1600", kind="cull", width=2560, height=1600, gx=16, gy=9, gz=24, lights=1024, cap=128),
        # a laptop-sized frame of smooth rasterised surfaces, every stage from
        # the cluster boxes to the tone-mapped picture (odd sizes: 1366 / 16)
        dict(name="frame_1366x768", kind="frame", width=1366, height=768, gx=16, gy=9, gz=24, lights=1000, cap=128,
             surfaces=True, post=True),
        # the benchmark frame: 65,536 lights, 8.3 M fragments
        dict(name="frame_3840x2160", kind="frame", width=3840, height=2160, gx=32, gy=18, gz=48, lights=65536,
             cap=128, surfaces=False, post=False),
        # loading an environment: equirect to cube and its box mip chain
        dict(name="environment_1024", kind="environment", width=2048, height=1024, face=1024),
        # the split-sum table, built once per program
        dict(name="lut_512", kind="lut", width=512, height=512, samples=1024),
        # the bit-compatible filters of one environment
        dict(name="irradiance_1024_32", kind="filter", type="diffuse", face=1024, out=32, mips=1, samples=0),
        dict(name="prefilter_1024_512", kind="filter", type="specular", face=1024, out=512, mips=10, samples=1024),
        # the contraction filters of one environment, in both precisions
        dict(name="contract_1024_512", kind="contract", type="specular", face=1024, out=512, mips=10, split=False,
             probes=1),
        dict(name="contract_split_512_256", kind="contract", type="specular", face=512, out=256, mips=9, split=True,
             probes=1),
        # many light probes of one size in one call
        dict(name="probes_24x256_128", kind="contract", type="specular", face=256, out=128, mips=8, split=False,
             probes=24),
        # the radiance network: training steps, and queries of a trained one
        dict(name="train_32768", kind="train", samples=1 << 18, batch=32768, steps=100),
        dict(name="query_2000000", kind="query", samples=2000000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cull", "frame", "environment", "lut", "diffuse", "specular", "contract", "contract", "probes",
                       "irradiance", "train", "query"])
    if kind in ("cull", "frame"):
        width = rng.randrange(640, 3840)
        c = dict(kind=kind, width=width, height=max(360, int(width * rng.uniform(0.45, 0.56))), gx=rng.randrange(8, 33),
                 gy=rng.randrange(5, 19), gz=rng.randrange(12, 49), lights=_log_int(rng, 16, 60000),
                 cap=rng.randrange(32, 151))
        if kind == "frame":
            c.update(surfaces=rng.random() < 0.5, post=rng.random() < 0.5, cap=min(c["cap"], 128))
        return c
    if kind == "environment":
        h = rng.randrange(128, 1025)
        return dict(kind=kind, width=2 * h, height=h, face=1 << rng.randrange(6, 11))
    if kind == "lut":
        return dict(kind=kind, width=_log_int(rng, 32, 512), height=_log_int(rng, 32, 512),
                    samples=_log_int(rng, 64, 1024))
    if kind == "diffuse":
        return dict(kind="filter", type="diffuse", face=_log_int(rng, 32, 1024), out=rng.randrange(4, 33), mips=1,
                    samples=0)
    if kind == "specular":
        out = _log_int(rng, 16, 400)
        return dict(kind="filter", type="specular", face=rng.randrange(out, 1025), out=out,
                    mips=rng.randrange(2, out.bit_length() + 1), samples=_log_int(rng, 64, 1024))
    if kind in ("contract", "probes"):
        lo = rng.randrange(4, 9) if kind == "contract" else rng.randrange(4, 8)
        out = 1 << lo
        return dict(kind="contract", type="specular", face=1 << rng.randrange(lo, 11 if kind == "contract" else lo + 2),
                    out=out, mips=rng.randrange(2, lo + 2), split=rng.random() < 0.4,
                    probes=1 if kind == "contract" else rng.randrange(2, 25))
    if kind == "irradiance":
        return dict(kind="contract", type="diffuse", face=1 << rng.randrange(5, 11), out=1 << rng.randrange(3, 7),
                    mips=1, split=False, probes=rng.choice([1, 1, 3, 17]))
    if kind == "train":
        batch = 256 * _log_int(rng, 1, 128)
        return dict(kind=kind, samples=batch * rng.randrange(2, 9) + rng.randrange(0, 256), batch=batch,
                    steps=rng.randrange(4, 40))
    return dict(kind="query", samples=_log_int(rng, 1000, 2000000))


# --------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _rand(g, *shape, lo=0.0, hi=1.0):
    return torch.rand(*shape, generator=g, device=DEV) * (hi - lo) + lo


def _face_point(f, a, b, m):
    """Point of cube face f at plane coordinates (a, b), m away (storage texel order)."""
    m = torch.as_tensor(m, dtype=a.dtype, device=a.device).expand_as(a)
    p = [(m, -b, -a), (-m, -b, a), (a, m, b), (a, -m, -b), (a, -b, m), (-a, -b, -m)][f]
    return torch.stack(p, dim=-1)


def _grid(S, dtype, lo=0, hi=None):
    x = (2.0 * torch.arange(lo, S if hi is None else hi, device=DEV, dtype=dtype) + 1.0) / S - 1.0
    return torch.meshgrid(x, x, indexing="ij")  # (v, u): rows, columns


def _unit(p):
    return p / p.norm(dim=-1, keepdim=True)


def _texel_dirs(S, dtype):
    v, u = _grid(S, dtype)
    return torch.stack([_unit(_face_point(f, u, v, 1.0)) for f in range(6)])  # [6][S][S][3]


def _radiance(d, seed, sun=1.0e4):
    """An HDR environment over directions d: sky gradient, dark ground, a sun disk, 32 coloured hot spots, texel detail."""
    r = np.random.RandomState(int(seed) % (1 << 31))
    y = d[..., 1]
    k = y.clamp_min(0).sqrt()[..., None]
    sky = torch.tensor([1.2, 1.1, 0.9], device=DEV) * (1 - k) + torch.tensor([0.15, 0.3, 0.8], device=DEV) * k
    c = torch.where(y[..., None] >= 0, sky, torch.tensor([0.12, 0.10, 0.08], device=DEV))
    az, el = r.uniform(0, 2 * PI), math.radians(r.uniform(20, 60))
    s = torch.tensor([math.cos(el) * math.cos(az), math.sin(el), math.cos(el) * math.sin(az)], device=DEV)
    if sun:
        c = c + sun * (d @ s > math.cos(0.02))[..., None]
    for _ in range(32):
        q = r.normal(size=3)
        q = torch.tensor(q / np.linalg.norm(q), device=DEV, dtype=torch.float32)
        width, peak = 0.03 + 0.12 * r.uniform(), math.exp(3.0 + r.normal())
        e = peak * torch.exp(-(1.0 - (d @ q).clamp(-1, 1)) / (width * width))
        c = c + e[..., None] * torch.tensor(0.5 + 0.5 * r.uniform(size=3), device=DEV, dtype=torch.float32)
    return c * (1.0 + 0.1 * _rand(_gen(seed + 5), *c.shape[:-1], 1))


def _rgba(c):
    return torch.cat([c, torch.ones_like(c[..., :1])], dim=-1).contiguous()


def _chain(level0, levels):
    """Box mip chain of [6][S][S][4], flattened mip-major as the library stores it."""
    out, l = [level0.reshape(-1)], level0
    for _ in range(1, levels):
        l = ((l[:, 0::2, 0::2] + l[:, 0::2, 1::2]) + (l[:, 1::2, 0::2] + l[:, 1::2, 1::2])) * 0.25
        out.append(l.reshape(-1))
    return torch.cat(out)


def _cube(seed, S, sun=1.0e4):
    return _rgba(_radiance(_texel_dirs(S, torch.float32), seed, sun))


def _lights(seed, n):
    g = _gen(seed)
    l = torch.zeros(n, 12, device=DEV)
    lo, hi = torch.tensor([-15.0, 0.0, -7.0], device=DEV), torch.tensor([15.0, 12.0, 7.0], device=DEV)
    l[:, 0:3] = lo + (hi - lo) * _rand(g, n, 3)
    l[:, 3] = 1.0
    l[:, 4:7] = _rand(g, n, 3)
    l[:, 7] = 1.0
    l[:, 8] = _rand(g, n, lo=0.5, hi=3.0)
    return l


def _matrices(c):
    """View, projection (Y down, depth 0..1) and inverse(P V) in double, as 4x4 row-major arrays."""
    eye, tgt = np.array(EYE), np.array(TARGET)
    front = (tgt - eye) / np.linalg.norm(tgt - eye)
    right = np.cross(front, [0.0, 1.0, 0.0])
    right /= np.linalg.norm(right)
    up = np.cross(right, front)
    f32 = lambda x: float(np.float32(x))  # noqa: E731
    n, f, th = f32(NEAR), f32(FAR), math.tan(f32(FOVY) / 2)
    P, V = np.zeros((4, 4)), np.eye(4)
    P[0, 0], P[1, 1] = c["height"] / c["width"] / th, -1.0 / th
    P[2, 2], P[3, 2], P[2, 3] = f / (n - f), -1.0, -(f * n) / (f - n)
    V[0, :3], V[1, :3], V[2, :3] = right, up, -front
    V[:3, 3] = -V[:3, :3] @ eye
    return V, P, np.linalg.inv(P @ V)


def _fragments(c, seed):
    """One fragment per pixel: surfaces of a rasterised scene (smooth depth and normals, materials in patches), or
    independent fragments."""
    W, H, g = c["width"], c["height"], _gen(seed)
    n = W * H
    V, P, IVP = _matrices(c)
    ys, xs = torch.meshgrid(torch.arange(H, device=DEV), torch.arange(W, device=DEV), indexing="ij")
    xs, ys = (xs.reshape(-1) + 0.5) / W, (ys.reshape(-1) + 0.5) / H
    if c["surfaces"]:
        r = np.random.RandomState(int(seed) % (1 << 31))
        lin, cell = torch.full((n,), 9.0, device=DEV), torch.zeros(n, dtype=torch.int64, device=DEV)
        for k in range(24):  # boxes and walls in front of each other
            w, h, z = r.uniform(0.1, 0.5), r.uniform(0.1, 0.6), math.exp(r.uniform(math.log(1.5), math.log(14.0)))
            x0, y0, sx, sy = r.uniform(-0.1, 0.9), r.uniform(-0.1, 0.9), r.uniform(-1, 1), r.uniform(-1, 1)
            zk = z * (1.0 + 0.3 * (sx * (xs - x0) + sy * (ys - y0)))
            hit = (xs > x0) & (xs < x0 + w) & (ys > y0) & (ys < y0 + h) & (zk < lin)
            lin, cell = torch.where(hit, zk, lin), torch.where(hit, k + 1, cell)
        pick = lambda t: t[cell]  # noqa: E731
        rough, albedo = pick(_rand(g, 25, lo=0.05, hi=1.0)), pick(_rand(g, 25, 3))
        rough = (rough + 0.05 * _rand(g, n, lo=-1.0)).clamp(0.05, 1.0)
        metal, nrm = pick((_rand(g, 25) < 0.3)), pick(torch.randn(25, 3, generator=g, device=DEV))
        nrm = nrm + 0.05 * torch.randn(n, 3, generator=g, device=DEV)
    else:
        lin = torch.exp(_rand(g, n) * math.log(FAR / NEAR)) * NEAR
        rough, albedo, metal = _rand(g, n, lo=0.05), _rand(g, n, 3), _rand(g, n) < 0.3
        nrm = torch.randn(n, 3, generator=g, device=DEV)
    depth = (FAR * (lin - NEAR) / (lin * (FAR - NEAR))).clamp(0.0, 0.9999999)
    ivp = torch.tensor(IVP, device=DEV, dtype=torch.float32)
    p = torch.stack([xs * 2 - 1, ys * 2 - 1, depth, torch.ones_like(depth)], dim=1) @ ivp.T
    view = torch.tensor(EYE, device=DEV) - p[:, :3] / p[:, 3:]
    nrm = _unit(nrm)
    nrm = nrm * torch.where((nrm * view).sum(1, keepdim=True) < 0, -1.0, 1.0)
    nx, ny, nz = (nrm[:, k].contiguous() for k in range(3))
    ar, ag, ab = (albedo[:, k].contiguous() for k in range(3))
    return dict(depth=depth, nx=nx, ny=ny, nz=nz, ar=ar, ag=ag, ab=ab, rough=rough.contiguous(),
                metal=(metal * 255).to(torch.uint8))


def _maps(seed):
    spec = _chain(_cube(seed, SPEC, sun=0.0), SPEC_MIPS)
    diff = _rgba(_radiance(_texel_dirs(DIFF, torch.float32), seed + 1, sun=0.0) * 0.5).reshape(-1)
    a = (torch.arange(LUT, device=DEV) + 0.5) / LUT
    rough, nov = torch.meshgrid(a, a, indexing="ij")
    x = 1.0 - rough * (1.0 - nov) ** 2
    return spec, diff, torch.stack([x * 0.9, (1.0 - x) * 0.3], dim=-1).contiguous()


_ctx = None


def _context():
    """A program makes one context and keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = abi.Context(0)
    return _ctx


def _network(seed):
    g = torch.Generator().manual_seed(int(seed))
    parts = []
    for o, i in ((64, 128), (64, 64), (64, 64), (3, 64)):
        parts += [(torch.rand(o * i, generator=g) * 2 - 1) * math.sqrt((6.0 if o > 3 else 2.0) / i),
                  (torch.rand(o, generator=g) * 2 - 1) * 0.05]
    return torch.cat(parts).numpy().astype(np.float32)


def _queries(seed, n):
    g = _gen(seed)
    d = _unit(torch.randn(n, 3, generator=g, device=DEV))
    return torch.cat([d, _rand(g, n, 1)], dim=1).contiguous()


def prepare(case, seed):
    c, s, kind = case, dict(case=case, ctx=_context()), case["kind"]
    empty = lambda n, t=torch.float32: torch.empty(n, dtype=t, device=DEV)  # noqa: E731
    if kind in ("cull", "frame"):
        s["desc"], s["cam"], s["ubo"], s["ivp"] = abi.camera_build(EYE, TARGET, FOVY, NEAR, FAR, c["width"],
                                                                  c["height"], (c["gx"], c["gy"], c["gz"]))
        n = c["gx"] * c["gy"] * c["gz"]
        s["lights"], s["boxes"] = _lights(seed, c["lights"]), empty((n, 8))
        s["cells"], s["total"] = empty((n, 2), torch.int32), torch.zeros(1, dtype=torch.int32, device=DEV)
        s["indices"] = torch.zeros(n * c["cap"], dtype=torch.int32, device=DEV)
        s["ctx"].build_aabbs(s["ubo"], s["boxes"])
    if kind == "frame":
        s["planes"], s["tex"] = _fragments(c, seed + 1), _maps(seed + 2)
        s["frags"] = abi.frag_soa(s["planes"], c["width"], c["height"], s["ivp"])
        s["maps"] = abi.ibl_maps(s["tex"][0], SPEC, SPEC_MIPS, s["tex"][1], DIFF, s["tex"][2], LUT, LUT)
        s["pc"], s["rgb"] = abi.pbr_defaults(), empty((3, c["height"], c["width"]))
        s["ldr"] = empty((3, c["height"], c["width"]))
    elif kind == "environment":
        s["levels"] = abi.mip_count(c["face"])
        s["equirect"] = _equirect(seed, c)
        s["out"] = empty(abi.cube_chain_floats(c["face"], s["levels"]))
    elif kind == "lut":
        s["out"] = empty((c["height"], c["width"], 2))
        s["samples"] = c["samples"] - seed % 7  # the table has no other input
    elif kind == "filter":
        s["cube"] = _cube(seed, c["face"])
        s["type"] = abi.FILTER_DIFFUSE if c["type"] == "diffuse" else abi.FILTER_SPECULAR
        s["out"] = empty(abi.cube_chain_floats(c["out"], c["mips"]))
    elif kind == "contract":
        s["levels"] = abi.mip_count(c["face"])
        s["chains"] = [_chain(_cube(seed + 31 * k, c["face"]), s["levels"]) for k in range(c["probes"])]
        s["outs"] = [empty(abi.cube_chain_floats(c["out"], c["mips"])) for _ in range(c["probes"])]
        s["plan"] = abi.ContractPlan(s["ctx"], abi.FILTER_DIFFUSE if c["type"] == "diffuse" else abi.FILTER_SPECULAR,
                                     c["face"], c["out"], c["mips"],
                                     abi.PRECISION_BF16_SPLIT if c["split"] else abi.PRECISION_FP16_SCALED)
        if c["probes"] > 1:
            s["plan"].reserve(c["probes"])
            s["from"], s["to"] = (torch.tensor([t.data_ptr() for t in v], dtype=torch.int64, device=DEV)
                                  for v in (s["chains"], s["outs"]))
    elif kind in ("train", "query"):
        s["x"], s["net"] = _queries(seed, c["samples"]), abi.Mlp(s["ctx"], 1.0, 1)
        s["net"].set_params(_network(seed + 1))
        if kind == "train":
            s["y"], s["loss"] = _targets(s["x"], seed), empty(c["steps"])
        else:
            s["out"] = empty((c["samples"], 3))
    return s


def _equirect(seed, c):
    w, h = c["width"], c["height"]
    t, a = (torch.arange(h, device=DEV) + 0.5) / h, (torch.arange(w, device=DEV) + 0.5) / w
    th, ph = torch.meshgrid((1.0 - t) * PI, (a - 0.5) * 2 * PI, indexing="ij")
    return _rgba(_radiance(torch.stack([th.sin() * ph.cos(), th.cos(), th.sin() * ph.sin()], dim=-1), seed))


def _targets(x, seed):
    c = _radiance(x[:, :3], seed, sun=0.0) * (1.0 + x[:, 3:])
    return torch.cat([(c + 1e-3).log(), torch.zeros_like(x[:, :1])], dim=1).contiguous()


# ----------------------------------------------------------------------- a pass
def run(s):
    c, ctx, kind = s["case"], s["ctx"], s["case"]["kind"]
    if kind in ("cull", "frame"):
        if kind == "frame" and c["post"]:  # the first frame after a resize
            ctx.build_aabbs(s["ubo"], s["boxes"])
        ctx.cull_lights(s["ubo"], s["boxes"], s["lights"], c["lights"], c["cap"], s["cells"], s["indices"],
                        s["indices"].numel(), s["total"])
        out = dict(cells=s["cells"], indices=s["indices"], total=s["total"])
        if kind == "frame":
            ctx.shade(s["frags"], s["cam"], s["ubo"], s["pc"], s["lights"], c["lights"], s["cells"], s["indices"],
                      s["maps"], s["rgb"])
            out["rgb"] = s["rgb"]
            if c["post"]:
                ctx.tonemap(s["rgb"], c["width"], c["height"], abi.TONEMAP_REINHARD, True, s["ldr"])
                out.update(ldr=s["ldr"], boxes=s["boxes"])
        return out
    if kind == "environment":
        ctx.equirect_to_cube(s["equirect"], c["width"], c["height"], s["out"], c["face"])
        ctx.cube_mips(s["out"], c["face"], s["levels"])
        return s["out"]
    if kind == "lut":
        ctx.brdf_lut(c["width"], c["height"], s["samples"], s["out"])
        return s["out"]
    if kind == "filter":
        ctx.filter(s["type"], s["cube"], c["face"], s["out"], c["out"], c["mips"], c["samples"])
        return s["out"]
    if kind == "contract":
        if c["probes"] == 1:
            s["plan"].filter(s["chains"][0], s["levels"], s["outs"][0])
        else:
            s["plan"].filter_multi(c["probes"], s["from"], s["levels"], s["to"])
        return s["outs"]
    if kind == "train":
        s["net"].train(s["x"], s["y"], c["samples"], c["batch"], c["steps"], 4e-3, s["loss"])
        return dict(loss=s["loss"], weights=s["net"].params())
    s["net"].eval(s["x"], c["samples"], s["out"])
    return s["out"]


# ------------------------------------------------------------------------ work
def _chain_texels(S, mips):
    return sum(6 * max(S >> m, 1) ** 2 for m in range(mips))


def work(case):
    c, kind = case, case["kind"]
    if kind in ("cull", "frame"):
        n, F = c["gx"] * c["gy"] * c["gz"], c["width"] * c["height"]
        per = min(c["cap"], 0.0115 * c["lights"] ** 0.9)  # lights a cluster lists in this scene, about
        b, f = 48 * c["lights"] + 40 * n + 4 * n * per, 16 * n * per
        if kind == "frame":
            b += 45 * F + (24 * F if c["post"] else 0) + 16 * (_chain_texels(SPEC, 2) + 6 * DIFF ** 2) + 8 * LUT ** 2
            f += F * (160 + 140 * per + (60 if c["post"] else 0))
        return dict(bytes=b, flops=f)
    if kind == "environment":
        return dict(bytes=16 * (c["width"] * c["height"] + _chain_texels(c["face"], c["face"].bit_length())),
                    flops=60 * _chain_texels(c["face"], 1))
    if kind == "lut":
        return dict(bytes=8 * c["width"] * c["height"], flops=50 * c["width"] * c["height"] * c["samples"])
    if kind == "filter":
        t = _chain_texels(c["out"], c["mips"])
        n = 252 * 63 * t if c["type"] == "diffuse" else c["samples"] * (t - _chain_texels(c["out"], 1))
        return dict(bytes=16 * (_chain_texels(c["face"], 1) + t), flops=80 * n)
    if kind == "contract":
        # texels under each output's lobe: the whole level, or a window of 20 texels and the coarse level
        n = {"delta": lambda l: 4, "full": lambda l: 6 * l["Si"] ** 2, "split": lambda l: 1257 + 6 * l["Sf"] ** 2}
        f = sum(36.0 * l["So"] ** 2 * n[l["kind"]](l) for l in _levels(c))
        return dict(bytes=16 * c["probes"] * (_chain_texels(c["face"], 1) + _chain_texels(c["out"], c["mips"])),
                    flops=c["probes"] * f)
    if kind == "train":
        return dict(bytes=32 * min(c["batch"] * c["steps"], c["samples"]), flops=3 * 33200.0 * c["batch"] * c["steps"])
    return dict(bytes=28 * c["samples"], flops=33200.0 * c["samples"])


# ------------------------------------------------------------ results in 64 bits
F64 = torch.float64


def _faces_of(d):
    """Cube face, plane numerators and major magnitude of directions (ties X, then Y, then Z)."""
    x, y, z = d.unbind(-1)
    ax, ay, az = x.abs(), y.abs(), z.abs()
    ix, iy = (ax >= ay) & (ax >= az), ay >= az
    sx, sy, sz = (torch.where(t >= 0, 1.0, -1.0).to(d.dtype) for t in (x, y, z))
    face = torch.where(ix, (x < 0).long(), torch.where(iy, 2 + (y < 0).long(), 4 + (z < 0).long()))
    sc = torch.where(ix, -sx * z, torch.where(iy, x, sz * x))
    tc = torch.where(ix, -y, torch.where(iy, sy * z, -y))
    return face, sc, tc, torch.where(ix, ax, torch.where(iy, ay, az))


def _padded(level):
    """[6][S][S][C] with one texel of seamless border: folded neighbours, corners the mean of their three texels."""
    S = level.shape[1]
    out = torch.zeros(6, S + 2, S + 2, level.shape[3], dtype=F64, device=DEV)
    out[:, 1:-1, 1:-1] = level
    o = 2.0 * torch.arange(S, device=DEV, dtype=F64) + 1.0 - S
    m = torch.full_like(o, S)

    def across(f, a, b):  # a texel one step outside, folded over the edge
        g, sc, tc, _ = _faces_of(_face_point(f, a, b, S - 1.0))
        i, j = ((sc + S - 1) / 2).round().long(), ((tc + S - 1) / 2).round().long()
        return level[g, j, i]

    for f in range(6):
        out[f, 1:-1, 0], out[f, 1:-1, -1] = across(f, -m, o), across(f, m, o)
        out[f, 0, 1:-1], out[f, -1, 1:-1] = across(f, o, -m), across(f, o, m)
        for y, yi in ((0, 1), (-1, -2)):
            for x, xi in ((0, 1), (-1, -2)):
                out[f, y, x] = (out[f, yi, xi] + out[f, y, xi] + out[f, yi, x]) / 3
    return out


def _sample(padded, d):
    """Bilinear seamless sample at directions d."""
    S = padded.shape[1] - 2
    f, sc, tc, ma = _faces_of(d)
    u, v = 0.5 * (sc / ma + 1) * S - 0.5, 0.5 * (tc / ma + 1) * S - 0.5
    i, j = u.floor(), v.floor()
    a, b = (u - i)[..., None], (v - j)[..., None]
    at = (f * (S + 2) + j.long() + 1) * (S + 2) + i.long() + 1
    flat = padded.reshape(-1, padded.shape[-1])
    return ((1 - a) * (1 - b) * flat[at] + a * (1 - b) * flat[at + 1]
            + (1 - a) * b * flat[at + S + 2] + a * b * flat[at + S + 3])


def _sample_2d(tex, s, t):
    H, W, C = tex.shape
    u, v = s * W - 0.5, t * H - 0.5
    i, j = u.floor(), v.floor()
    a, b = (u - i)[..., None], (v - j)[..., None]
    i, j, flat = i.long(), j.long(), tex.reshape(-1, C)
    at = lambda jj, ii: flat[(jj % H) * W + ii % W]  # noqa: E731
    return ((1 - a) * (1 - b) * at(j, i) + a * (1 - b) * at(j, i + 1)
            + (1 - a) * b * at(j + 1, i) + a * b * at(j + 1, i + 1))


def _hammersley(n):
    i = np.arange(n, dtype=np.uint64)
    r = np.zeros(n, dtype=np.uint64)
    for k in range(32):
        r |= ((i >> np.uint64(k)) & np.uint64(1)) << np.uint64(31 - k)
    return (torch.tensor(i.astype(np.float64) / n, device=DEV),
            torch.tensor(r.astype(np.float64) * 2.3283064365386963e-10, device=DEV))


def _half_vectors(n, a):
    """GGX half vectors in the tangent frame for alpha a ([...] -> [..., n])."""
    x, y = _hammersley(n)
    ct = ((1 - y) / (1 + (a * a - 1) * y)).sqrt()
    st = (1 - ct * ct).clamp_min(0).sqrt()
    return torch.cos(2 * PI * x) * st, torch.sin(2 * PI * x) * st, ct


def _rgb1(c):
    return torch.cat([c, torch.ones_like(c[..., :1])], dim=-1).reshape(-1)


def _exact_specular(level0, c):
    pad, out = _padded(level0), []
    for m in range(c["mips"]):
        S = max(c["out"] >> m, 1)
        N = _texel_dirs(S, F64).reshape(-1, 3)
        r = float(np.float32(m) / np.float32(c["mips"] - 1)) if c["mips"] > 1 else 0.0
        if r == 0.0:
            out.append(_rgb1(_sample(pad, N)))
            continue
        up = torch.where(N[:, 2:].abs() < 0.999, torch.tensor([0.0, 0, 1], dtype=F64, device=DEV),
                         torch.tensor([1.0, 0, 0], dtype=F64, device=DEV))
        T = _unit(torch.linalg.cross(up, N))
        B = torch.linalg.cross(N, T)
        hx, hy, hz = _half_vectors(c["samples"], torch.tensor(r * r, dtype=F64, device=DEV))
        lz = 2 * hz * hz - 1
        keep = lz > 0
        lx, ly, lz = (2 * hz * hx)[keep], (2 * hz * hy)[keep], lz[keep]
        acc, step = torch.zeros(N.shape[0], 3, dtype=F64, device=DEV), max(1, (1 << 21) // N.shape[0])
        for k in range(0, lz.numel(), step):
            q = slice(k, k + step)
            L = T[:, None] * lx[q, None] + B[:, None] * ly[q, None] + N[:, None] * lz[q, None]
            acc += (_sample(pad, L) * lz[q, None]).sum(1)
        out.append(_rgb1(acc / lz.sum()))
    return torch.cat(out)


def _exact_diffuse(level0, c):
    pad, N = _padded(level0), _texel_dirs(c["out"], F64).reshape(-1, 3)
    up = torch.tensor([0.0, 1, 0], dtype=F64, device=DEV).expand_as(N)
    R = _unit(torch.linalg.cross(up, N))
    U = _unit(torch.linalg.cross(N, R))
    th = 0.025 * torch.arange(63, device=DEV, dtype=F64)
    acc = torch.zeros_like(N)
    for k in range(252):
        st, ct, p = th.sin(), th.cos(), 0.025 * k
        d = (R[:, None] * (st * math.cos(p))[:, None] + U[:, None] * (st * math.sin(p))[:, None]
             + N[:, None] * ct[:, None])
        acc += (_sample(pad, d) * (ct * st)[:, None]).sum(1)
    return _rgb1(PI * acc / (252 * 63))


def _exact_lut(c, n):
    W, H = c["width"], c["height"]
    nov = ((torch.arange(W, device=DEV, dtype=F64) + 0.5) / W)[:, None]
    vx, out = (1 - nov * nov).sqrt(), []
    for y in range(H):
        r = 1 - (y + 0.5) / H
        hx, hy, hz = _half_vectors(n, torch.tensor(r * r, dtype=F64, device=DEV))
        # about the z axis the frame is tangent (0, -1, 0), bitangent (1, 0, 0)
        vh = vx * hy + nov * hz
        l = torch.stack([2 * vh * hy - vx, -2 * vh * hx, 2 * vh * hz - nov])
        nl = l[2] / l.norm(dim=0)
        k = r * r / 2
        vh = vh.clamp_min(0)
        g = (nl / (nl * (1 - k) + k)) * (nov / (nov * (1 - k) + k)) * vh / (hz * nov)
        fc = (1 - vh) ** 5
        g = torch.where(nl > 0, g, 0.0)
        out.append(torch.stack([((1 - fc) * g).sum(1), (fc * g).sum(1)], dim=-1) / n)
    return torch.stack(out)


def _exact_environment(eq, c):
    d = _texel_dirs(c["face"], F64)
    s = 0.5 + 0.5 * torch.atan2(d[..., 2], d[..., 0]) / PI
    cube = _sample_2d(eq[..., :3].to(F64), s, 1 - torch.acos(d[..., 1].clamp(-1, 1)) / PI)
    return _chain(_rgba(cube), c["face"].bit_length())


def _exact_boxes(c, P):
    X, Y, Z = c["gx"], c["gy"], c["gz"]
    near, far = float(np.float32(NEAR)), float(np.float32(FAR))
    ar = lambda n: torch.arange(n, device=DEV, dtype=F64)  # noqa: E731
    z, y, x = torch.meshgrid(ar(Z), ar(Y), ar(X), indexing="ij")
    zn, zf = near * (far / near) ** (z / Z), near * (far / near) ** ((z + 1) / Z)
    pts = []
    for k in (0, 1):
        u, v = ((x + k) / X * 2 - 1) / P[0, 0], ((y + k) / Y * 2 - 1) / P[1, 1]
        pts += [torch.stack([u * w, v * w, -w], dim=-1) for w in (zn, zf)]
    p, o = torch.stack(pts), torch.zeros(Z, Y, X, 1, dtype=F64, device=DEV)
    return torch.cat([p.amin(0), o, p.amax(0), o], dim=-1).reshape(-1, 8)


def _exact_lists(c, boxes, lights, V):
    """The first `cap` lights of every cluster, padded with -1."""
    V = torch.tensor(V, device=DEV, dtype=F64)
    p = lights[:, :3].to(F64) @ V[:3, :3].T + V[:3, 3]
    r2 = lights[:, 8].to(F64) ** 2
    lists = torch.full((boxes.shape[0], c["cap"]), -1, dtype=torch.int64, device=DEV)
    step = max(1, (1 << 24) // max(1, c["lights"]))
    for k in range(0, boxes.shape[0], step):
        b, d2 = boxes[k:k + step], 0.0
        for a in range(3):
            d2 = d2 + ((b[:, None, a] - p[:, a]).clamp_min(0) + (p[:, a] - b[:, None, 4 + a]).clamp_min(0)) ** 2
        hit = d2 < r2
        at = hit.cumsum(1) - 1
        row, light = (hit & (at < c["cap"])).nonzero(as_tuple=True)
        lists[k + row, at[row, light]] = light
    return lists


def _exact_shade(c, s, lists, IVP):
    W, H = c["width"], c["height"]
    near, far = float(np.float32(NEAR)), float(np.float32(FAR))
    pl = {k: v.to(F64) for k, v in s["planes"].items()}
    spec, diff, lut = s["tex"]
    mips, off = [], 0
    for m in range(2):
        n = 6 * (SPEC >> m) ** 2 * 4
        mips.append(_padded(spec[off:off + n].view(6, SPEC >> m, SPEC >> m, 4)[..., :3].to(F64)))
        off += n
    irr, lut = _padded(diff.view(6, DIFF, DIFF, 4)[..., :3].to(F64)), lut.to(F64)
    lpos, lcol, lrad = s["lights"][:, :3].to(F64), s["lights"][:, 4:7].to(F64), s["lights"][:, 8].to(F64)
    ivp = torch.tensor(np.float32(IVP).astype(np.float64), device=DEV)
    eye = torch.tensor(EYE, device=DEV, dtype=F64)
    intensity, base, max_lod, falloff, mul = (float(np.float32(v)) for v in (1.75, 0.01, 1.0, 0.1, 0.01))
    scale = c["gz"] / math.log2(far / near)
    out = torch.empty(W * H, 3, dtype=F64, device=DEV)
    dot = lambda a, b: (a * b).sum(-1, keepdim=True)  # noqa: E731
    for b0 in range(0, W * H, 1 << 20):
        q = slice(b0, min(b0 + (1 << 20), W * H))
        i = torch.arange(q.start, q.stop, device=DEV)
        fx, fy, z = (i % W) + 0.5, (i // W).to(F64) + 0.5, pl["depth"][q]
        fx = fx.to(F64)
        lin = near * far / (far + z * (near - far))
        zi = ((torch.log2(lin) - math.log2(near)) * scale).clamp(0, c["gz"] - 1).long()
        ci = ((fx / (W / c["gx"])).long().clamp_max(c["gx"] - 1) + c["gx"] * (fy / (H / c["gy"])).long().clamp_max(
            c["gy"] - 1) + c["gx"] * c["gy"] * zi)
        h = torch.stack([fx / W * 2 - 1, fy / H * 2 - 1, z, torch.ones_like(z)], dim=1) @ ivp.T
        wp = h[:, :3] / h[:, 3:]
        N = torch.stack([pl["nx"][q], pl["ny"][q], pl["nz"][q]], dim=1)
        alb = torch.stack([pl["ar"][q], pl["ag"][q], pl["ab"][q]], dim=1)
        rough, metal = pl["rough"][q, None], pl["metal"][q, None] / 255
        V = _unit(eye - wp)
        NoV = dot(N, V).clamp_min(0)
        F0 = base * (1 - metal) + alb * metal
        Lo = alb * mul
        k, a2 = (rough + 1) ** 2 / 8, rough ** 4
        GV = NoV / (NoV * (1 - k) + k)
        mine = lists[ci]
        for j in range(mine.shape[1]):
            at = (mine[:, j] >= 0).nonzero().squeeze(1)
            if at.numel() == 0:
                break
            l = mine[at, j]
            d = lpos[l] - wp[at]
            dist = d.norm(dim=1, keepdim=True)
            L = d / dist
            Hh = _unit(V[at] + L)
            NoH, NoL, HoV = (dot(x, y).clamp_min(0) for x, y in ((N[at], Hh), (N[at], L), (Hh, V[at])))
            att = (1 - dist / lrad[l, None]).clamp_min(0) / dist ** falloff
            den = NoH * NoH * (a2[at] - 1) + 1
            DG = a2[at] / (PI * den * den) * (NoL / (NoL * (1 - k[at]) + k[at])) * GV[at]
            F = F0[at] + (1 - F0[at]) * (1 - HoV).clamp(0, 1) ** 5
            sp = DG * F / (4 * NoV[at] * NoL + float(np.float32(0.0001)))
            df = (1 - F) * (1 - metal[at]) * alb[at] / PI
            Lo[at] += (df + sp) * lcol[l] * (att * intensity) * NoL
        R = 2 * dot(N, V) * N - V
        lod = rough * max_lod
        pre = (1 - lod) * _sample(mips[0], R) + lod * _sample(mips[1], R)
        ab = _sample_2d(lut, NoV[:, 0], rough[:, 0])
        F = F0 + (torch.maximum(1 - rough, F0) - F0) * (1 - NoV).clamp(0, 1) ** 5
        out[q] = ((1 - F) * (1 - metal) * _sample(irr, N) * alb + pre * (F * ab[:, :1] + ab[:, 1:])) + Lo
    return out.T.reshape(3, H, W).contiguous()


# The contraction filter's quadrature: level choice and sums per output mip.
def _levels(c):
    out = []
    for m in range(c["mips"]):
        So = max(c["out"] >> m, 1)
        if c["type"] == "diffuse":
            out.append(dict(kind="full", So=So, Si=min(c["face"], 32)))
            continue
        a = (m / (c["mips"] - 1)) ** 2 if c["mips"] > 1 else 0.0
        if a == 0.0:
            out.append(dict(kind="delta", So=So))
            continue
        Si = 1
        while Si < (PI / 2) / (0.65 * a):
            Si *= 2
        Si = min(max(Si, 64), c["face"])
        l = dict(kind="full", So=So, Si=Si, a2=a * a)
        if So * So * 6.0 * Si * Si > 134217728.0 and So >= 16 and Si >= 64:
            Sf = min(max(Si // 4, 32), Si // 2)
            l.update(kind="split", Sf=Sf, t0=10 * PI / 2 / Si, t1=20 * PI / 2 / Si)
        out.append(l)
    return out


def _weight(l, c, cos, dw):
    if c["type"] == "diffuse":
        return cos.clamp_min(0) * dw
    d = 0.5 * (1 + cos) * (l["a2"] - 1) + 1
    return l["a2"] / (PI * d * d) * cos.clamp_min(0) * dw


def _window(l, cos):
    x = ((torch.acos(cos.clamp(-1, 1)) - l["t0"]) / (l["t1"] - l["t0"])).clamp(0, 1)
    return 1 - x * x * (3 - 2 * x)


def _solid(u, v, S):
    return (2.0 / S) ** 2 / (1 + u * u + v * v) ** 1.5


def _full_sum(l, c, level, N, far=False):
    """Sums of weights times [.., C] texels and of weights over every texel of a level, for directions N."""
    S = level.shape[1]
    D = _texel_dirs(S, F64).reshape(-1, 3)
    v, u = _grid(S, F64)
    dw = _solid(u, v, S).reshape(-1).repeat(6)
    X, num, z = level.reshape(D.shape[0], -1), [], []
    step = max(1, (1 << 25) // D.shape[0])
    for k in range(0, N.shape[0], step):
        cos = N[k:k + step] @ D.T
        w = _weight(l, c, cos, dw)
        if far:
            w = w * (1 - _window(l, cos))
        num.append(w @ X)
        z.append(w.sum(1))
    return torch.cat(num), torch.cat(z)


def _exact_split(l, c, level, far_level):
    So, Si, Sf, C = l["So"], l["Si"], l["Sf"], level.shape[-1]
    fn, fz = _full_sum(l, c, far_level, _texel_dirs(Sf, F64).reshape(-1, 3), far=True)
    far = _padded(torch.cat([fn, fz[:, None]], dim=1).view(6, Sf, Sf, C + 1))
    N = _texel_dirs(So, F64)
    far = _sample(far, N)
    num, z = far[..., :C].clone(), far[..., C].clone()
    # the near window on each face's plane, continued past the face's edges
    v, u = _grid(So, F64)
    n0 = _unit(_face_point(4, u, v, 1.0))  # the canonical face: (u, -v, 1)
    reach = 1
    for e in (n0[0], n0[-1], n0[:, 0], n0[:, -1]):
        t = _unit(torch.linalg.cross(e, torch.tensor([0.3, 0.5, 0.1], dtype=F64, device=DEV).expand_as(e)))
        for a in np.arange(64) * (2 * PI / 64):
            p = math.cos(l["t1"]) * e + math.sin(l["t1"]) * (math.cos(a) * t + math.sin(a) * torch.linalg.cross(e, t))
            reach = max(reach, float((p[..., :2].abs().amax(-1) / p[..., 2]).max()))
    B = int((reach * 1.02 - 1) * Si / 2) + 4
    pv, pu = _grid(Si, F64, -B, Si + B)
    pad, planes = _padded(level), []
    for f in range(6):
        t = _sample(pad, _face_point(f, pu, pv, 1.0))
        t[B:B + Si, B:B + Si] = level[f]
        planes.append(t)
    planes = torch.stack(planes, dim=2).reshape(-1, 6 * C)
    D = _unit(_face_point(4, pu, pv, 1.0)).reshape(-1, 3)
    dw = _solid(pu, pv, Si).reshape(-1)
    for y in range(0, So, 16):
        for x in range(0, So, 16):
            o = n0[y:y + 16, x:x + 16].reshape(-1, 3)
            mid = _unit(o.mean(0))
            reach = l["t1"] + float(torch.acos((o @ mid).clamp(-1, 1)).max()) + 1e-6
            at = (D @ mid > math.cos(reach)).nonzero().squeeze(1)
            cos = o @ D[at].T
            w = _weight(l, c, cos, dw[at]) * _window(l, cos)
            num[:, y:y + 16, x:x + 16] += (w @ planes[at]).view(16, 16, 6, C).permute(2, 0, 1, 3)
            z[:, y:y + 16, x:x + 16] += w.sum(1).view(16, 16)
    return num / z[..., None]


def _exact_contract(chains, c):
    """Every probe at once: texels carry 3 channels per probe."""
    box, off = {}, 0
    for m in range(c["face"].bit_length()):
        S = c["face"] >> m
        n = 6 * S * S * 4
        box[S] = torch.cat([t[off:off + n].view(6, S, S, 4)[..., :3] for t in chains], dim=-1).to(F64)
        off += n
    outs = []
    for l in _levels(c):
        if l["kind"] == "delta":
            r = _sample(_padded(box[c["face"]]), _texel_dirs(l["So"], F64))
        elif l["kind"] == "full":
            num, z = _full_sum(l, c, box[l["Si"]], _texel_dirs(l["So"], F64).reshape(-1, 3))
            r = (num / z[:, None]).view(6, l["So"], l["So"], -1)
        else:
            r = _exact_split(l, c, box[l["Si"]], box[l["Sf"]])
        outs.append(r)
    return [torch.cat([_rgb1(r[..., 3 * k:3 * k + 3]) for r in outs]) for k in range(len(chains))]


# The radiance network.
_LAYERS = ((64, 128), (64, 64), (64, 64), (3, 64))


def _unpack(p):
    out, o = [], 0
    for n, k in _LAYERS:
        out.append((p[o:o + n * k].view(n, k), p[o + n * k:o + n * k + n]))
        o += n * k + n
    return out


def _encode(x):
    t = torch.stack([x[:, 0], x[:, 1], x[:, 2], 2 * x[:, 3] - 1], dim=1)
    f = PI * 2.0 ** (0.5 * torch.arange(16, device=DEV, dtype=F64))
    p = t[:, :, None] * f
    return torch.stack([p.sin(), p.cos()], dim=-1).reshape(x.shape[0], 128)


def _forward(p, h):
    w = _unpack(p)
    for W, b in w[:3]:
        h = torch.relu(h @ W.T + b)
    return h @ w[3][0].T + w[3][1]


def _exact_train(s, c):
    p = torch.tensor(s["net"].params(), device=DEV, dtype=F64).requires_grad_(True)
    m, v, loss = torch.zeros_like(p), torch.zeros_like(p), []
    per, B, n = c["samples"] // c["batch"], c["batch"], c["steps"]
    for k in range(n):
        q = slice((k % per) * B, (k % per) * B + B)
        e = ((_forward(p, _encode(s["x"][q].to(F64))) - s["y"][q, :3].to(F64)) ** 2).mean()
        g, = torch.autograd.grad(e, p)
        loss.append(e.detach())
        lr = 4e-3 * (0.01 + 0.99 * 0.5 * (1 + math.cos(PI * (k / (n - 1) if n > 1 else 0.0))))
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        with torch.no_grad():
            p -= lr * (m / (1 - 0.9 ** (k + 1))) / ((v / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    # the weights follow the rounding of every step before, so only the loss has one value
    return dict(loss=torch.stack(loss), weights=None)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "cull":
        return None  # whole numbers only
    if kind == "lut":
        return _exact_lut(c, c["samples"] - seed % 7)
    if kind == "environment":
        return _exact_environment(_equirect(seed, c), c)
    if kind == "filter":
        level0 = _cube(seed, c["face"])[..., :3].to(F64)
        return (_exact_diffuse if c["type"] == "diffuse" else _exact_specular)(level0, c)
    if kind == "contract":
        n = c["face"].bit_length()
        return _exact_contract([_chain(_cube(seed + 31 * k, c["face"]), n) for k in range(c["probes"])], c)
    if kind == "frame":
        V, P, IVP = _matrices(c)
        boxes, lights = _exact_boxes(c, P), _lights(seed, c["lights"])
        s = dict(planes=_fragments(c, seed + 1), tex=_maps(seed + 2), lights=lights)
        rgb = _exact_shade(c, s, _exact_lists(c, boxes, lights, np.float32(V).astype(np.float64)), IVP)
        out = dict(cells=None, indices=None, total=None, rgb=rgb)
        if c["post"]:
            out.update(ldr=rgb.clamp_min(0) ** (1 / 2.2), boxes=boxes)
        return out
    if kind == "query":
        p = torch.tensor(_network(seed + 1), device=DEV, dtype=F64)
        x = _queries(seed, c["samples"]).to(F64)
        return torch.cat([torch.exp(_forward(p, _encode(t))) - 1e-3 for t in x.split(1 << 18)])
    s = dict(x=_queries(seed, c["samples"]), net=_Params(_network(seed + 1)))
    s["y"] = _targets(s["x"], seed)
    return _exact_train(s, c)


class _Params:
    def __init__(self, p):
        self.p = p

    def params(self):
        return self.p
