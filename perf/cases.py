"""Workloads of the multi-view-stereo path, through the Python binding.

listed() and draw() say which; prepare() makes what a program holds before
the call (uploaded images, descriptors, servers, output buffers), run() is one
call, work() its unavoidable bytes and operations, and exact() its result in
64-bit torch where the result is a computed value of its inputs.  A full solve
has no such value: which of two nearly equal hypotheses a pixel keeps is a
matter of the last bit of their costs.

The scene is ray-cast here: textured ground plane, sphere and backdrop seen by
cameras on a 30 degree arc, 8-bit images with 2 DN of noise.
"""
import ctypes
import math
import weakref

import numpy as np
import torch

import __graft_entry__ as entry

DEV = "cuda" if torch.cuda.is_available() else "cpu"
DMIN, DMAX = 2.0, 12.0


def _pkg():
    return entry.load_package()


def listed():
    return [
        # a thumbnail: the latency of one solve, launches and the call itself
        dict(name="view_96x72", kind="view", W=96, H=72, S=2, radius=5, stride=1, store="f32",
             iterations=3, top_k=3, seeds=0),
        # preview size, the whole 11 x 11 window
        dict(name="view_320x240", kind="view", W=320, H=240, S=2, radius=5, stride=1, store="f32",
             iterations=3, top_k=3, seeds=0),
        # a VGA-like view of odd size with a middling number of sources
        dict(name="view_641x479", kind="view", W=641, H=479, S=5, radius=5, stride=2, store="f32",
             iterations=8, top_k=3, seeds=0),
        # a reconstruction's usual view: 8 sources, seeded from sparse points,
        # every tap of the window, 12 iterations
        dict(name="view_1280x960_seeded", kind="view", W=1280, H=960, S=8, radius=5, stride=1,
             store="f32", iterations=12, top_k=3, seeds=600),
        # large view, half-size image planes
        dict(name="view_3200x2400_f16", kind="view", W=3200, H=2400, S=6, radius=5, stride=2,
             store="f16", iterations=8, top_k=3, seeds=0),
        # views of a scene one after the other into page-locked buffers
        dict(name="views_1600x1200", kind="views", W=1600, H=1200, S=4, radius=5, stride=2,
             store="f32", iterations=8, top_k=3, views=3),
        # results left on the device for a program that goes on there; a small window
        dict(name="device_800x600_5x5", kind="device", W=800, H=600, S=3, radius=2, stride=1,
             store="f32", iterations=6, top_k=2),
        # views of several resolutions in one launch
        dict(name="batch_mixed", kind="batch", stride=1, store="f16", iterations=8,
             mix="640x480:3,1280x960:5,1600x1200:4,2400x1800:6,641x481:8,999x777:3"),
        # requests over resident images, continuously batched
        dict(name="serve_resident", kind="serve", W=1280, H=960, S=5, stride=2, iterations=6,
             jobs=8, resident=True),
        # re-scoring given hypotheses (quality maps, comparing solutions); odd size
        dict(name="cost_1023x769_7x7", kind="cost", W=1023, H=769, S=4, radius=3, stride=1,
             store="f32", top_k=3),
        # geometric consistency over a ring of finished maps
        dict(name="filter_9x1280x960", kind="filter", W=1280, H=960, views=9, sources=8),
        # finished maps to a point cloud
        dict(name="fuse_5x1280x960", kind="fuse", W=1280, H=960, views=5, confidence=True,
             rgb=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _taps(c):
    k = (2 * c["radius"] // c["stride"] + 1) ** 2
    return c["W"] * c["H"] * c["S"] * k * (1 + 6 * c.get("iterations", 0)) * c.get("views", 1)


def draw(rng):
    kind = rng.choice(["view", "view", "view", "views", "device", "batch", "serve", "cost",
                       "filter", "fuse"])
    W = _log_int(rng, 80, 2600)
    H = max(48, int(W * rng.uniform(0.55, 1.0)))
    if kind in ("filter", "fuse"):
        W = min(W, 1280)
        H = min(H, 960)
        views = rng.randint(3, 9) if kind == "filter" else rng.randint(2, 5)
        if kind == "filter":
            return dict(kind=kind, W=W, H=H, views=views, sources=min(8, views - 1))
        return dict(kind=kind, W=W, H=H, views=views, confidence=rng.random() < 0.5,
                    rgb=rng.random() < 0.5)
    radius = 5 if rng.random() < 0.6 else rng.randint(1, 4)
    c = dict(kind=kind, W=W, H=H, S=rng.randint(2, 8), radius=radius,
             stride=rng.choice([1, 2]), store=rng.choice(["f32", "f16"]),
             iterations=rng.randint(2, 12), top_k=rng.choice([2, 3, 3, 3, 4]))
    if kind == "views":
        c["views"] = rng.randint(2, 4)
        c["S"] = min(c["S"], 5)
    while _taps(c) > 4e10 and c["iterations"] > 2:
        c["iterations"] -= 1
    if _taps(c) > 4e10:
        c["stride"] = 2
    if kind == "view":
        c["seeds"] = rng.choice([0, 0, rng.randint(20, 800)])
    elif kind == "cost":
        del c["iterations"]
    elif kind == "batch":
        sizes = []
        for _ in range(rng.randint(2, 6)):
            w = _log_int(rng, 160, 1600)
            sizes.append("%dx%d:%d" % (w, max(48, int(w * rng.uniform(0.55, 1.0))),
                                       rng.randint(3, 8)))
        return dict(kind=kind, stride=c["stride"], store=c["store"],
                    iterations=min(8, c["iterations"]), mix=",".join(sizes))
    elif kind == "serve":
        return dict(kind=kind, W=min(W, 1280), H=min(H, 960), S=min(c["S"], 6),
                    stride=c["stride"], iterations=min(6, c["iterations"]),
                    jobs=rng.randint(2, 8), resident=rng.random() < 0.5)
    return c


# ---------------------------------------------------------------------------
# The scene
# ---------------------------------------------------------------------------
def _cameras(W, H, n):
    """K and (R, t) of n cameras on the arc, the middle one first."""
    f = 0.9375 * W
    K = np.array([[f, 0.0, W / 2.0], [0.0, f, H / 2.0], [0.0, 0.0, 1.0]])
    order = [0.0]
    rungs = max(1, n // 2)
    for i in range(1, rungs + 1):
        order += [15.0 * i / rungs, -15.0 * i / rungs]
    cams = []
    for a in order[:n]:
        th = math.radians(a)
        C = np.array([6.0 * math.sin(th), 0.0, 6.0 - 6.0 * math.cos(th)])
        R = np.array([[math.cos(th), 0.0, math.sin(th)], [0.0, 1.0, 0.0],
                      [-math.sin(th), 0.0, math.cos(th)]])
        cams.append((R, -R @ C))
    return K, cams


def _noise3(p, salt):
    """Value noise in [0, 1) at points p (..., 3)."""
    q = torch.floor(p)
    f = p - q
    f = f * f * (3.0 - 2.0 * f)
    q = q.to(torch.int64)
    out = 0.0
    for dx in (0, 1):
        for dy in (0, 1):
            for dz in (0, 1):
                h = ((q[..., 0] + dx) * 73856093) ^ ((q[..., 1] + dy) * 19349663) ^ \
                    ((q[..., 2] + dz) * 83492791) ^ (salt * 2654435761)
                h = (h ^ (h >> 13)) * 1274126177 & 0x7FFFFFFF
                h = ((h ^ (h >> 15)) * 2246822519) & 0xFFFFFF
                w = (f[..., 0] if dx else 1 - f[..., 0]) * (f[..., 1] if dy else 1 - f[..., 1]) * \
                    (f[..., 2] if dz else 1 - f[..., 2])
                out = out + w * (h.to(torch.float64) / float(1 << 24))
    return out


def _raycast(W, H, K, R, t):
    """Depth (H, W), camera-frame normal (H, W, 3) and world points, float64."""
    y, x = torch.meshgrid(torch.arange(H, dtype=torch.float64, device=DEV),
                          torch.arange(W, dtype=torch.float64, device=DEV), indexing="ij")
    ray = torch.stack([(x - K[0, 2]) / K[0, 0], (y - K[1, 2]) / K[1, 1], torch.ones_like(x)], -1)
    Rt = torch.tensor(R, device=DEV)
    C = torch.tensor(-R.T @ t, device=DEV)
    d = (ray.unsqueeze(-1) * Rt).sum(-2)                  # R^T ray, depth = parameter
    inf = torch.full_like(x, 1e9)
    back = (11.5 - C[2]) / d[..., 2]
    ground = torch.where(d[..., 1] > 1e-9, (1.5 - C[1]) / d[..., 1], inf)
    oc = C - torch.tensor([0.0, 0.0, 6.0], dtype=torch.float64, device=DEV)
    a, b, c = (d * d).sum(-1), (d * oc).sum(-1), (oc * oc).sum() - 2.25
    disc = b * b - a * c
    ball = torch.where(disc > 0, (-b - torch.sqrt(disc.clamp(min=0))) / a, inf)
    depth, which = torch.stack([back, ground, ball], -1).min(-1)
    X = C + depth.unsqueeze(-1) * d
    n = torch.zeros_like(X)
    n[..., 2] = torch.where(which == 0, -1.0, 0.0)
    n[..., 1] = torch.where(which == 1, -1.0, 0.0)
    nb = (X - torch.tensor([0.0, 0.0, 6.0], dtype=torch.float64, device=DEV)) / 1.5
    n = torch.where((which == 2).unsqueeze(-1), nb, n)
    return depth, (n.unsqueeze(-2) * Rt).sum(-1), X


def _image(W, X, salt, gen):
    """8-bit image of the surface points X."""
    tex, amp, freq = 0.0, 0.5, 4.0 * 0.9375 * W / 1500.0
    for o in range(4):
        tex = tex + amp * _noise3(X * freq, salt + o)
        amp, freq = amp * 0.5, freq * 2.0
    dn = 20.0 + 215.0 * tex + 2.0 * torch.randn(tex.shape, dtype=torch.float64, device=DEV,
                                               generator=gen)
    return dn.round().clamp(0, 255).to(torch.uint8).cpu().numpy()


def _scene(W, H, n, seed, images=True):
    """K, cameras, images, float64 depth and normal maps and points of n views."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) * 7919 + 17)
    K, cams = _cameras(W, H, n)
    out = dict(K=K, cams=cams, images=[], depth=[], normal=[], X=[])
    for R, t in cams:
        depth, normal, X = _raycast(W, H, K, R, t)
        if images:
            out["images"].append(_image(W, X, int(seed) % 100003, gen))
        out["depth"].append(depth)
        out["normal"].append(normal)
        out["X"].append(X)
    out["gen"] = gen
    return out


def _hypotheses(sc, view, fuzz):
    """Depth and normal maps as a finished solve leaves them: near the surface,
    a share of the pixels anywhere in the range."""
    gen, d, n = sc["gen"], sc["depth"][view], sc["normal"][view]
    r = torch.rand((4,) + d.shape, dtype=torch.float64, device=DEV, generator=gen)
    dep = d * (1.0 + 0.004 * (r[0] - 0.5))
    dep = torch.where(r[1] < fuzz, DMIN + (DMAX - DMIN) * r[2], dep)
    nn = n + 0.1 * (torch.rand(n.shape, dtype=torch.float64, device=DEV, generator=gen) - 0.5)
    nn = nn / nn.norm(dim=-1, keepdim=True)
    conf = 1.0 - 0.5 * r[3] * torch.where(r[1] < fuzz, 1.0, 0.4)
    return (dep.to(torch.float32).cpu().numpy(), nn.to(torch.float32).cpu().numpy(),
            conf.to(torch.float32).cpu().numpy())


# ---------------------------------------------------------------------------
# State
# ---------------------------------------------------------------------------
_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = _pkg().Context()
    return _ctx


def _free_after(array):
    """Give a page-locked array back once nothing refers to its memory."""
    owner = array
    while isinstance(owner, np.ndarray):
        owner = owner.base
    weakref.finalize(owner, _pkg().lib().hp3d_pm_host_free, _ctx.h,
                     ctypes.c_void_p(array.ctypes.data))


class _State:
    """What the program holds; gives images and servers back."""

    def __init__(self):
        self.images, self.server = [], None

    def upload(self, image, store):
        pkg = _pkg()
        h = _context().upload(image, pkg.STORE_F16 if store == "f16" else pkg.STORE_F32)
        self.images.append(h)
        return h

    def __del__(self):
        try:
            if self.server is not None:
                self.server.close()
            for h in self.images:
                _ctx.release(h)
        except Exception:
            pass


def _desc(sc, handles, ref, S, c, seed, seeds=None):
    pkg = _pkg()
    others = [v for v in range(len(handles)) if v != ref][:S]
    terms = [pkg.compose(sc["K"], *sc["cams"][ref], sc["K"], *sc["cams"][v]) for v in others]
    return pkg.make_desc(handles[ref], [handles[v] for v in others], pkg.invert3(sc["K"]),
                         [a for a, _ in terms], [b for _, b in terms], DMIN, DMAX,
                         radius=c.get("radius", 5), stride=c["stride"],
                         iterations=c.get("iterations", 0), top_k=c.get("top_k", 3),
                         seed=42 + 1000000 * ref + seed % 1000, seeds=seeds)


def _seed_points(sc, W, H, count, seed):
    """Sparse points on the reference view's surface, as a structure-from-motion
    result holds them, projected to seeds."""
    pkg = _pkg()
    rs = np.random.RandomState(seed % (1 << 31))
    ys, xs = rs.randint(0, H, count), rs.randint(0, W, count)
    X = sc["X"][0][torch.from_numpy(ys).to(DEV), torch.from_numpy(xs).to(DEV)].cpu().numpy()
    sfm = pkg.SfM([dict(K=sc["K"], R=R, t=t) for R, t in sc["cams"]], [(p, [0, 1]) for p in X])
    return sfm.seed_points(0, DMIN, DMAX, W, H)


def _sizes(mix):
    out = []
    for part in mix.split(","):
        wh, s = part.split(":")
        w, h = wh.split("x")
        out.append((int(w), int(h), int(s)))
    return out


def prepare(case, seed):
    c, pkg, st = case, _pkg(), _State()
    st.case = dict(case)
    kind = c["kind"]
    if kind in ("view", "views", "device", "cost"):
        n = max(c["S"] + 1, c.get("views", 1))
        sc = _scene(c["W"], c["H"], n, seed)
        handles = [st.upload(im, c["store"]) for im in sc["images"]]
        st.shape = (c["H"], c["W"])
        seeds = _seed_points(sc, c["W"], c["H"], c["seeds"], seed) if c.get("seeds") else None
        st.descs = [_desc(sc, handles, v, c["S"], c, seed, seeds)
                    for v in range(c.get("views", 1))]
        if kind == "views":
            st.outs = [_context().host_outputs(st.shape, pinned=True) for _ in st.descs]
            for o in st.outs:
                for a in o.values():
                    _free_after(a)
        elif kind == "device":
            H, W = st.shape
            st.outs = [torch.empty((H, W), device=DEV), torch.empty((H, W, 3), device=DEV),
                       torch.empty((H, W), device=DEV)]
        elif kind == "cost":
            st.hyp = _hypotheses(sc, 0, 0.25)[:2]
    elif kind == "batch":
        st.descs, st.shapes = [], []
        for k, (W, H, S) in enumerate(_sizes(c["mix"])):
            sc = _scene(W, H, S + 1, seed + 31 * k)
            handles = [st.upload(im, c["store"]) for im in sc["images"]]
            st.descs.append(_desc(sc, handles, 0, S, c, seed + k))
            st.shapes.append((H, W))
    elif kind == "serve":
        n = c["S"] + 1
        sc = _scene(c["W"], c["H"], n, seed)
        st.server = pkg.Server(4 << 30, max_jobs=16, radius=5, stride=c["stride"],
                               store=pkg.STORE_F16)
        handles = [st.server.image_add(im) for im in sc["images"]] if c["resident"] \
            else sc["images"]
        st.requests = []
        for j in range(c["jobs"]):
            ref = j % n
            others = [v for v in range(n) if v != ref]
            terms = [pkg.compose(sc["K"], *sc["cams"][ref], sc["K"], *sc["cams"][v])
                     for v in others]
            st.requests.append(dict(
                ref=handles[ref], srcs=[handles[v] for v in others],
                K_ref_inv=pkg.invert3(sc["K"]), A=[a for a, _ in terms], b=[b for _, b in terms],
                depth_min=DMIN, depth_max=DMAX, iterations=c["iterations"],
                seed=42 + 1000000 * j + seed % 1000, with_normal=True, shape=(c["H"], c["W"])))
    else:
        sc = _scene(c["W"], c["H"], c["views"], seed, images=False)
        rs = np.random.RandomState(seed % (1 << 31))
        st.maps = []
        for v, (R, t) in enumerate(sc["cams"]):
            dep, nrm, conf = _hypotheses(sc, v, 0.25)
            m = dict(depth=dep, normal=nrm, K=sc["K"], R=R, t=t)
            if kind == "filter":
                m["confidence"] = conf
                m["src"] = [u for u in range(c["views"]) if u != v][:c["sources"]]
            else:
                # as a filter leaves them: a share of the pixels cleared, another
                # share kept with a low confidence
                order = rs.permutation(dep.size)
                cleared, low = order[:dep.size // 3], order[dep.size // 3:dep.size // 2]
                dep.reshape(-1)[cleared] = 0.0
                if c["confidence"]:
                    m["confidence"] = np.maximum(conf, np.float32(0.85))
                    m["confidence"].reshape(-1)[low] *= np.float32(0.6)
                m["color"] = rs.randint(0, 256, (c["H"], c["W"]) + ((3,) if c["rgb"] else ()),
                                        dtype=np.uint8)
            st.maps.append(m)
    return st


def run(st):
    c, kind = st.case, st.case["kind"]
    if kind == "view":
        return _ctx.run_view(st.descs[0], st.shape)
    if kind == "views":
        return _ctx.run_views(st.descs, st.outs)
    if kind == "device":
        _ctx.run_view_device(st.descs[0], *[o.data_ptr() for o in st.outs])
        return st.outs
    if kind == "cost":
        return _ctx.cost_eval(st.descs[0], *st.hyp)
    if kind == "batch":
        return _ctx.batch_run(st.descs, st.shapes)
    if kind == "serve":
        ids = [st.server.submit(**r) for r in st.requests]
        for i in ids:
            st.server.wait(i)
        res = [st.server.result(i) for i in ids]
        for i in ids:
            st.server.forget(i)
        return res
    ctx = _context()
    if kind == "filter":
        kept = ctx.geom_filter(st.maps)
        return dict(depth=[m["depth"] for m in st.maps],
                    confidence=[m["confidence"] for m in st.maps], kept=kept)
    return ctx.fuse(st.maps, min_confidence=0.8 if c["confidence"] else 0.0)


def work(case):
    """Images and given maps read once, results written once; 34 operations a
    tap (12 warp, 3 divide, 11 bilinear, 8 moments) for the six candidates of
    every pixel and iteration and the first cost."""
    c, kind = case, case["kind"]
    if kind == "filter":
        px = c["W"] * c["H"] * c["views"]
        return {"bytes": px * (20 + 8), "flops": px * (40 + 45 * c["sources"])}
    if kind == "fuse":
        px = c["W"] * c["H"] * c["views"]
        return {"bytes": px * (16 + 4 * c["confidence"] + (3 if c["rgb"] else 1) + 36 * 0.5),
                "flops": px * 60}
    if kind == "batch":
        jobs = [dict(W=w, H=h, S=s, radius=5, stride=c["stride"], store=c["store"],
                     iterations=c["iterations"]) for w, h, s in _sizes(c["mix"])]
    elif kind == "serve":
        jobs = [dict(c, radius=5, store="f16")] * c["jobs"]
    else:
        jobs = [dict(c, views=1)] * c.get("views", 1)
    b = f = 0.0
    for j in jobs:
        px = j["W"] * j["H"]
        b += px * (4 if j["store"] == "f32" else 2) * (1 + j["S"])
        b += px * 20    # depth, normal and cost: results, or for "cost" two given and one result
        f += 34.0 * _taps(j)
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# The results in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "cost":
        return _exact_cost(case, seed)
    if kind == "filter":
        return _exact_filter(prepare(case, seed).maps)
    if kind == "fuse":
        return _exact_fuse(prepare(case, seed).maps, 0.8 if case["confidence"] else 0.0)
    return None


def _cuda64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV).to(torch.float64)


def _exact_cost(c, seed):
    W, H, S, R, st = c["W"], c["H"], c["S"], c["radius"], c["stride"]
    sc = _scene(W, H, S + 1, seed)
    depth, normal = [_cuda64(a) for a in _hypotheses(sc, 0, 0.25)[:2]]
    img = [_cuda64(im) for im in sc["images"]]
    K = sc["K"]
    Ki = np.linalg.inv(K)
    y, x = torch.meshgrid(torch.arange(H, dtype=torch.float64, device=DEV),
                          torch.arange(W, dtype=torch.float64, device=DEV), indexing="ij")
    ray = [Ki[r, 0] * x + Ki[r, 1] * y + Ki[r, 2] for r in range(3)]
    nP = depth * sum(normal[..., r] * ray[r] for r in range(3))
    g = [sum(Ki[r, k] * normal[..., r] for r in range(3)) / nP for k in range(3)]
    R0, t0 = sc["cams"][0]
    offs = range(-R, R + 1, st)
    full = len(offs) ** 2
    costs = []
    for s in range(1, S + 1):
        Rs, ts = sc["cams"][s]
        Rr = Rs @ R0.T
        A, b = K @ Rr @ Ki, K @ (ts - Rr @ t0)
        m = {k: torch.zeros_like(depth) for k in ("n", "r", "s", "rr", "ss", "rs")}
        for oy in offs:
            for ox in offs:
                px, py = x + ox, y + oy
                gp = g[0] * px + g[1] * py + g[2]
                w = [A[r, 0] * px + A[r, 1] * py + A[r, 2] + b[r] * gp for r in range(3)]
                u, v = w[0] / w[2], w[1] / w[2]
                ok = (w[2].abs() >= 1e-8) & (u >= 0) & (u < W - 1) & (v >= 0) & (v < H - 1)
                u, v = torch.where(ok, u, 0.0), torch.where(ok, v, 0.0)
                iu, iv = u.floor(), v.floor()
                fu, fv = u - iu, v - iv
                q = (iv * W + iu).to(torch.int64)
                flat = img[s].reshape(-1)
                a0, a1, c0, c1 = flat[q], flat[q + 1], flat[q + W], flat[q + W + 1]
                sv = (a0 * (1 - fu) + a1 * fu) * (1 - fv) + (c0 * (1 - fu) + c1 * fu) * fv
                rv = img[0][py.clamp(0, H - 1).to(torch.int64), px.clamp(0, W - 1).to(torch.int64)]
                sv, rv = torch.where(ok, sv - 128.0, 0.0), torch.where(ok, rv - 128.0, 0.0)
                m["n"] += ok
                m["r"] += rv
                m["s"] += sv
                m["rr"] += rv * rv
                m["ss"] += sv * sv
                m["rs"] += rv * sv
        num = m["n"] * m["rs"] - m["r"] * m["s"]
        dr, ds = m["n"] * m["rr"] - m["r"] ** 2, m["n"] * m["ss"] - m["s"] ** 2
        eps = 255.0 * 255.0 * 1e-6
        good = (m["n"] >= full // 2) & (dr >= eps) & (ds >= eps)
        ncc = (num / torch.sqrt(torch.where(good, dr * ds, 1.0))).clamp(-1, 1)
        costs.append(torch.where(good, 1.0 - ncc, 2.0))
    k = min(c["top_k"], S)
    best = torch.stack(costs).sort(0).values[:k].mean(0)
    return torch.where(nP.abs() < 1e-8, 2.0, best)


def _world(m):
    """World points and normals of a map, float64, and its pixel grid."""
    d, n = _cuda64(m["depth"]), _cuda64(m["normal"])
    H, W = d.shape
    Ki, R, t = np.linalg.inv(m["K"]), m["R"], m["t"]
    y, x = torch.meshgrid(torch.arange(H, dtype=torch.float64, device=DEV),
                          torch.arange(W, dtype=torch.float64, device=DEV), indexing="ij")
    pc = [d * (Ki[r, 0] * x + Ki[r, 1] * y + Ki[r, 2]) - t[r] for r in range(3)]
    pw = [R[0, k] * pc[0] + R[1, k] * pc[1] + R[2, k] * pc[2] for k in range(3)]
    nw = [R[0, k] * n[..., 0] + R[1, k] * n[..., 1] + R[2, k] * n[..., 2] for k in range(3)]
    return d, pw, nw


def _exact_filter(maps, tol=0.12, least=2):
    depth = [_cuda64(m["depth"]) for m in maps]
    conf = [_cuda64(m["confidence"]) for m in maps]
    nws = [_world(m)[2] for m in maps]
    H, W = depth[0].shape
    for i, m in enumerate(maps):
        d, pw, _ = _world(m)
        votes = torch.zeros_like(d)
        for s in m["src"]:
            Rs, ts, Ks = maps[s]["R"], maps[s]["t"], maps[s]["K"]
            ps = [Rs[r, 0] * pw[0] + Rs[r, 1] * pw[1] + Rs[r, 2] * pw[2] + ts[r]
                  for r in range(3)]
            z = torch.where(ps[2] > 0, ps[2], 1.0)
            u = torch.round(Ks[0, 0] * ps[0] / z + Ks[0, 2])
            v = torch.round(Ks[1, 1] * ps[1] / z + Ks[1, 2])
            ok = (ps[2] > 0) & (u >= 0) & (u < W) & (v >= 0) & (v < H)
            q = (torch.where(ok, v, 0.0) * W + torch.where(ok, u, 0.0)).to(torch.int64)
            ds = depth[s].reshape(-1)[q]
            votes += ok & (ds > 0) & ((ds - z).abs() / z <= tol)
        keep = (d > 0) & (votes >= least)
        depth[i] = torch.where(keep, d, 0.0)
        conf[i] = torch.where(keep, conf[i], 0.0)
    del nws   # normals are compared at 180 degrees: never rejected
    return dict(depth=depth, confidence=conf, kept=[None] * len(maps))


def _exact_fuse(maps, least):
    pos, nrm, col = [], [], []
    for m in maps:
        d, pw, nw = _world(m)
        ok = d > 0
        if m.get("confidence") is not None:
            ok &= torch.from_numpy(m["confidence"]).to(DEV) >= torch.tensor(
                least, dtype=torch.float32, device=DEV)
        c = _cuda64(m["color"]) / 255.0
        c = c.unsqueeze(-1).expand(*c.shape, 3) if c.dim() == 2 else c
        pos.append(torch.stack(pw, -1)[ok])
        nrm.append(torch.stack(nw, -1)[ok])
        col.append(c[ok])
    return torch.cat(pos), torch.cat(nrm), torch.cat(col)
