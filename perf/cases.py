"""The calls that are timed: what a program does with this framework, through
its public entry points, from the smallest sizes to the largest.

A case names its kind and sizes:
  find      tom_os3_findTemplate, the one-call search: statistics of the
            tomogram, template preparation, every orientation, the maps
  search    one template through a SearchPlan that is kept for the tomogram
            (set_template, run, finalize), as a search over several templates
            or classes does it
  corr      tom_os3_corr, the score map of one template as given
  refine    SearchPlan.refine, the exact local search around candidates
  subtomo   subtomo_score_batch, the local angular search of subtomograms
  picks     tom_os3_returnPicklist on a score map and its angle map
  infer     Unet.infer over a tomogram and its coarse score map
  train     one gradient of the proposal network on a crop
"""
import math

import numpy as np
import torch

from tom_amd import api

# Edges of volumes that the search accepts (the first one has to be even in
# steps of 32), and of templates that a weight accepts.
XS = (64, 96, 128, 160, 192, 256, 320, 384, 512)
YS = (24, 32, 40, 48, 64, 80, 96, 120, 128, 160, 192, 200, 240, 256, 320, 384, 400, 480, 512)
BOX = (16, 24, 32, 40, 48, 64)


def listed():
    return [
        # the smallest whole search: a binned tomogram cut-out, coarse angles
        dict(name="find_64", kind="find", X=64, Y=64, Z=64, nx=24, ny=24, nz=24, A=90, batch=16, wedge=30.0),
        # a tomogram of ordinary size, 48^3 template with its missing wedge;
        # the share of a 15 degree grid that two batches hold
        dict(name="search_512", kind="search", X=512, Y=512, Z=256, nx=48, ny=48, nz=48, A=32, batch=16, wedge=30.0,
             tz=16, ty=32),
        # the binned volume of a coarse scan, no weight, a last batch that is not full
        dict(name="search_256", kind="search", X=256, Y=256, Z=128, nx=24, ny=24, nz=24, A=53, batch=16, wedge=0.0,
             tz=16, ty=16),
        # edges with a factor 5, a box that is no cube, the default batch
        dict(name="search_odd", kind="search", X=320, Y=240, Z=96, nx=40, ny=32, nz=24, A=22, batch=4, wedge=40.0,
             tz=16, ty=16),
        # the largest tomogram, half a batch
        dict(name="search_1024", kind="search", X=1024, Y=1024, Z=384, nx=48, ny=48, nz=48, A=8, batch=8, wedge=40.0,
             tz=8, ty=16),
        # one template as given, the tomogram's statistics made in the call
        dict(name="corr_256", kind="corr", X=256, Y=256, Z=128, nx=48, ny=48, nz=48),
        # candidates of a coarse scan, one level of 27 orientations each
        dict(name="refine_64", kind="refine", X=256, Y=256, Z=128, nx=48, ny=48, nz=48, P=64, A=27, wedge=30.0),
        # subtomograms of uneven boxes, 3 x 3 x 3 local angles, their own wedges
        dict(name="subtomo_384", kind="subtomo", P=384, A=27, edges="32,48,64", ref=False),
        # a few small ones, with the wedge of the template turned along
        dict(name="subtomo_16", kind="subtomo", P=16, A=8, edges="32", ref=True),
        # the picks of a score map
        dict(name="picks_200", kind="picks", X=256, Y=256, Z=128, n=32, picks=200),
        # the network over a tomogram in one tile
        dict(name="infer_256", kind="infer", X=256, Y=256, Z=128, tx=256, ty=256, tz=128, halo=0),
        # a training crop: forward, backward, the gradients to the host
        dict(name="train_96", kind="train", X=96, Y=96, Z=96),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _volume(rng, most):
    while True:
        X, Y, Z = rng.choice(XS), rng.choice(YS), rng.choice(YS)
        if X * Y * Z <= most:
            return X, Y, Z


def draw(rng):
    kind = rng.choice(("find", "search", "search", "search", "corr", "refine", "subtomo", "picks", "infer", "train"))
    wedge = rng.choice((0.0, round(rng.uniform(20.0, 45.0), 1)))
    if kind in ("find", "search"):
        X, Y, Z = _volume(rng, 256 * 256 * 128 if kind == "find" else 512 * 512 * 256)
        box = [rng.choice(BOX) if wedge else rng.randint(9, 64) for _ in range(3)]
        if rng.random() < 0.6:
            box = [box[0]] * 3
        nx, ny, nz = (min(b, 24 if N < 32 else 32 if N < 48 else 48) if N < b else b for b, N in zip(box, (X, Y, Z)))
        nx, ny, nz = (min(b, 16) if N < b else b for b, N in zip((nx, ny, nz), (X, Y, Z)))
        A = _log(rng, 1, 120)
        while A > 1 and A * X * Y * Z > 32 * 512 * 512 * 256:
            A //= 2
        d = dict(kind=kind, X=X, Y=Y, Z=Z, nx=nx, ny=ny, nz=nz, A=A, batch=rng.randint(1, 16), wedge=wedge)
        return d if kind == "find" else dict(d, tz=16, ty=16)
    if kind == "corr":
        X, Y, Z = _volume(rng, 384 * 384 * 128)
        n = min(rng.randint(9, 64), Y, Z)
        return dict(kind=kind, X=X, Y=Y, Z=Z, nx=n, ny=n, nz=n)
    if kind == "refine":
        n = rng.choice((24, 32, 40, 48, 64))
        return dict(kind=kind, X=rng.choice((128, 192, 256)), Y=rng.choice((128, 160, 240)), Z=rng.choice((96, 128)),
                    nx=n, ny=n, nz=n, P=_log(rng, 3, 120), A=_log(rng, 5, 64), wedge=wedge)
    if kind == "subtomo":
        return dict(kind=kind, P=_log(rng, 4, 300), A=rng.randint(1, 30),
                    edges=rng.choice(("32", "48", "64", "32,48", "32,48,64")), ref=rng.random() < 0.3)
    if kind == "picks":
        X, Y, Z = rng.randint(100, 320), rng.randint(100, 320), rng.randint(60, 200)
        n = rng.randint(12, 40)
        most = max(4, X * Y * Z // (16 * n ** 3))  # as many as the map surely holds
        return dict(kind=kind, X=X, Y=Y, Z=Z, n=n, picks=min(most, _log(rng, 20, 400)))
    if kind == "infer":
        D, H, W = (4 * rng.randint(12, 40) for _ in range(3))
        if rng.random() < 0.5:  # one tile of the network's size
            return dict(kind=kind, X=D, Y=H, Z=W, tx=D, ty=H, tz=W, halo=0)
        return dict(kind=kind, X=rng.randint(80, 200), Y=rng.randint(80, 200), Z=rng.randint(40, 120),
                    tx=D + 48, ty=H + 48, tz=W + 48, halo=24)
    return dict(kind="train", **{k: 4 * rng.randint(8, 26) for k in "XYZ"})


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _phantom(rng, shape, k=10):
    """k Gaussian blobs within the box, (x, y, z)."""
    ax = [np.arange(s, dtype=np.float64) - s // 2 for s in shape]
    sig = max(1.0, min(shape) / 24.0)
    T = np.zeros(shape)
    for _ in range(k):
        c = rng.uniform(-1, 1, 3) * (np.asarray(shape) / 2 - 2) * 0.6
        e = [np.exp(-(a - b) ** 2 / (2 * sig * sig)) for a, b in zip(ax, c)]
        T += rng.uniform(0.5, 1.0) * e[0][:, None, None] * e[1][None, :, None] * e[2][None, None, :]
    return np.asfortranarray(T, np.float32)


def _mask(shape):
    """A sphere (an ellipsoid in an uneven box), 1 inside, soft over a few voxels."""
    ax = [(np.arange(s, dtype=np.float64) - s // 2) / max(1.0, s / 2 - 2) for s in shape]
    r = np.sqrt(ax[0][:, None, None] ** 2 + ax[1][None, :, None] ** 2 + ax[2][None, None, :] ** 2)
    m = np.where(r <= 0.85, 1.0, np.exp(-((r - 0.85) / 0.08) ** 2))
    return np.asfortranarray(np.where(r > 1.0, 0.0, m), np.float32)


def _wedge(shape, deg):
    """The centred weight of a missing wedge around z, None for no wedge."""
    if not deg:
        return None
    x = np.abs(np.arange(shape[0]) - shape[0] // 2).astype(np.float64)[:, None, None]
    z = np.abs(np.arange(shape[2]) - shape[2] // 2).astype(np.float64)[None, None, :]
    keep = x >= math.tan(math.radians(deg)) * z
    return np.asfortranarray(np.broadcast_to(keep, shape).astype(np.float32))


def _tomogram(case, seed, rng, T):
    """Noise over copies of the template in the cube's quarter turns, (Z, Y, X)."""
    X, Y, Z = case["X"], case["Y"], case["Z"]
    V = torch.randn((Z, Y, X), generator=_gen(seed), device="cuda")
    t = torch.from_numpy(np.ascontiguousarray(T.transpose(2, 1, 0))).cuda()
    t = t * (0.8 / float(t.double().std()))
    for k in range(max(2, X * Y * Z // 200000)):
        p = torch.rot90(t, k % 4, (1, 2)) if t.shape[1] == t.shape[2] else torch.flip(t, (k % 3,))
        z, y, x = (int(rng.integers(0, N - n + 1)) for N, n in zip((Z, Y, X), p.shape))
        V[z:z + p.shape[0], y:y + p.shape[1], x:x + p.shape[2]] += p
    return V


def _euler(rng, n):
    return np.stack([rng.uniform(0, 360, n), rng.uniform(0, 360, n), np.degrees(np.arccos(rng.uniform(-1, 1, n)))],
                    1).astype(np.float32)


def _box(case):
    return (case["nx"], case["ny"], case["nz"])


def _matching(case, seed):
    """Tomogram, template, mask and weight of the search kinds."""
    rng = np.random.default_rng(seed)
    T = _phantom(rng, _box(case))
    return rng, _tomogram(case, seed, rng, T), T, _mask(_box(case)), _wedge(_box(case), case.get("wedge", 0.0))


def _refine_inputs(case, rng):
    P = case["P"]
    N = (case["X"], case["Y"], case["Z"])
    angles = (_euler(rng, P)[None] + rng.uniform(-10, 10, (case["A"], P, 3))).astype(np.float32)
    cand = np.stack([rng.integers(0, n, P) for n in N] + [np.arange(P)], 1).astype(np.int32)
    return angles, cand


def _subtomo_inputs(case, seed):
    rng = np.random.default_rng(seed)
    edges = [int(e) for e in case["edges"].split(",")]
    boxes = []
    for B in edges:
        c = np.fft.fftfreq(B, 1.0 / B)
        near = c[:, None, None] ** 2 + c[None, :, None] ** 2 + c[None, None, :] ** 2 <= 25.0
        b = {"template": _phantom(rng, (B, B, B)), "mask": _mask((B, B, B)), "mask_cc": near.astype(np.float32)}
        boxes.append(dict(b, wedge_ref=25.0) if case["ref"] else b)
    P = case["P"]
    pbox = np.sort(rng.integers(0, len(edges), P)).astype(np.int32)
    g = _gen(seed)
    parts = []
    for k, B in enumerate(edges):
        t = torch.from_numpy(np.ascontiguousarray(boxes[k]["template"].transpose(2, 1, 0))).cuda()
        t = t * (0.5 / float(t.double().std()))
        n = int((pbox == k).sum())
        v = torch.randn((n, B, B, B), generator=g, device="cuda")
        for i in range(n):
            s = tuple(int(q) for q in rng.integers(-4, 5, 3))
            v[i] += torch.roll(torch.rot90(t, i % 4, (0, 1)), s, (0, 1, 2))
        parts.append(v.reshape(-1))
    wedge = rng.uniform(20.0, 45.0, P).astype(np.float32)
    angles = (_euler(rng, P)[:, None] * (np.arange(P) % 2)[:, None, None]
              + rng.uniform(-6, 6, (P, case["A"], 3))).astype(np.float32)
    return boxes, torch.cat(parts), pbox, wedge, angles


# layers of the network: input and output channels, taps
LAYERS = ((16, 16, 27), (16, 16, 27), (16, 32, 27), (32, 32, 27), (32, 64, 27), (64, 64, 27), (96, 32, 27),
          (32, 32, 27), (48, 16, 27), (16, 16, 27), (16, 80, 1))


def _weights(rng):
    """Parameters of a network about to be trained: W [tap][out][in], b [out]."""
    out = []
    for i, (ci, co, t) in enumerate(LAYERS):
        fan = t * (2 if i == 0 else ci)
        w = rng.standard_normal((t, co, ci)) * math.sqrt(2.0 / fan)
        if i == 0:
            w[:, :, 2:] = 0  # only the tomogram and the score map come in
        if t == 1:
            w[:, 68:] = 0    # one particle logit, 64 bins, 3 offsets
        b = rng.standard_normal(co) * 0.05
        if t == 1:
            b[68:] = 0
        out += [w.ravel(), b]
    return np.concatenate(out).astype(np.float32)


def _field(seed, shape):
    """A smooth field over noise, as a score map or a tomogram has it."""
    g = _gen(seed)
    low = torch.randn([1, 1] + [max(2, s // 8) for s in shape], generator=g, device="cuda")
    f = torch.nn.functional.interpolate(low, size=tuple(shape), mode="trilinear", align_corners=False)[0, 0]
    return (f + 0.7 * torch.randn(tuple(shape), generator=g, device="cuda")).contiguous()


def _targets(seed, shape):
    g = _gen(seed)
    f = _field(seed + 7, shape)
    prob = torch.sigmoid(4 * f - 8)
    tbin = torch.randint(0, 64, shape, generator=g, device="cuda", dtype=torch.int32)
    tbin = torch.where(prob > 0.3, tbin, torch.full_like(tbin, -1))
    off = torch.randn(shape + (4,), generator=g, device="cuda") * 0.3
    off[..., 3] = (prob > 0.2).float()
    return prob, tbin, off


def _net_inputs(case, seed):
    rng = np.random.default_rng(seed)
    shape = (case["Z"], case["Y"], case["X"])
    return _weights(rng), _field(seed + 1, shape), _field(seed + 2, shape)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("find", "search", "corr", "refine"):
        rng, V, T, M, W = _matching(case, seed)
        s.update(V=V, T=T, M=M, W=W)
        if kind == "refine":
            s["angles"], s["cand"] = _refine_inputs(case, rng)
        elif kind != "corr":
            s["angles"] = _euler(rng, case["A"])
        if kind in ("find", "corr"):  # a call on arrays that are on the GPU
            for k in ("T", "M", "W"):
                if s[k] is not None:
                    s[k] = torch.from_numpy(np.ascontiguousarray(s[k].transpose(2, 1, 0))).cuda()
            return s
        s["Tn"], s["mu"], s["sig"] = api.prepare_template(T, M, W)
        s["plan"] = api.SearchPlan(V, _box(case), M, batch=case.get("batch", 16))
        if kind == "search":
            s["plan"].set_tiles(case["tz"], case["ty"])
        else:
            s["plan"].set_template(s["Tn"], W, s["mu"], s["sig"])
    elif kind == "subtomo":
        s["in"] = _subtomo_inputs(case, seed)
    elif kind == "picks":
        shape = (case["Z"], case["Y"], case["X"])
        s["map"] = _field(seed, shape) * 0.1
        s["ang"] = torch.randint(0, 7488, shape, generator=_gen(seed + 1), device="cuda", dtype=torch.int32)
    else:
        theta, s["vol"], s["aux"] = _net_inputs(case, seed)
        train = kind == "train"
        dims = (case["X"], case["Y"], case["Z"]) if train else (case["tx"], case["ty"], case["tz"])
        s["net"] = api.Unet(dims, nbin=64, seed=0, train=train)
        s["net"].set_params(theta)
        if train:
            s["to"] = _targets(seed, tuple(s["vol"].shape))
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "find":
        return api.tom_os3_findTemplate(s["V"], s["T"], s["M"], s["angles"], W=s["W"], batch=c["batch"])
    if kind == "search":
        p = s["plan"]
        p.set_template(s["Tn"], s["W"], s["mu"], s["sig"])
        p.run(s["angles"])
        return p.finalize()
    if kind == "corr":
        return api.tom_os3_corr(s["V"], s["T"], s["M"])
    if kind == "refine":
        return s["plan"].refine(s["V"], s["angles"], s["cand"])
    if kind == "subtomo":
        return api.subtomo_score_batch(*s["in"])
    if kind == "picks":
        return api.tom_os3_returnPicklist(s["map"], (c["n"],) * 3, c["picks"], angles=s["ang"])
    if kind == "infer":
        return s["net"].infer(s["vol"], c["halo"], aux=s["aux"], logit=True, offsets=True)
    # the optimizer's step is left out so that every pass sees the same weights
    net = s["net"]
    net.forward(s["vol"], s["aux"])
    loss = net.backward(s["to"][0], s["to"][1], 20.0, toff=s["to"][2])
    return loss, net.get_grads()


# ---------------------------------------------------------------- work
def _fft(n, lines=1.0):
    """Real operations of real transforms over n samples."""
    return 2.5 * n * math.log2(max(2, n)) * lines


def work(case):
    kind = case["kind"]
    if kind in ("find", "search", "corr"):
        N = case["X"] * case["Y"] * case["Z"]
        n = case["nx"] * case["ny"] * case["nz"]
        A = case.get("A", 1)
        # per orientation: the template's spectrum, the product, the way back
        flops = A * (2 * _fft(N) + 3 * N) + (0 if kind == "search" else 4 * _fft(N))
        # a plan holds the spectrum (4 bytes a voxel) and two 8-byte statistics
        bytes_ = N * (4 + (16 if kind == "search" else 0) + (4 if kind == "corr" else 8)) + 12 * n
        return {"bytes": bytes_, "flops": flops}
    if kind == "refine":
        n = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 4 * case["P"] * n + 12 * n, "flops": case["P"] * case["A"] * (27 * 2 * n + 12 * n + 2 * _fft(n))}
    if kind == "subtomo":
        e = [int(q) for q in case["edges"].split(",")]
        n = sum(q ** 3 for q in e) / len(e)
        k = 6 if case["ref"] else 4
        return {"bytes": case["P"] * 4 * n, "flops": case["P"] * ((1 + k * case["A"]) * _fft(n) + case["A"] * 14 * n)}
    if kind == "picks":
        N = case["X"] * case["Y"] * case["Z"]
        return {"bytes": 4 * N, "flops": case["picks"] * case["n"] ** 3}
    f = lambda v: sum(2.0 * (v / 8 ** lv) * t * (2 if i == 0 else ci) * co  # noqa: E731
                      for i, ((ci, co, t), lv) in enumerate(zip(LAYERS, (0, 0, 1, 1, 2, 2, 1, 1, 0, 0, 0))))
    if kind == "infer":
        N = case["X"] * case["Y"] * case["Z"]
        return {"bytes": N * (8 + 20), "flops": f(N)}
    N = case["X"] * case["Y"] * case["Z"]
    return {"bytes": N * (8 + 24), "flops": 3 * f(N)}


# ---------------------------------------------------------------- the same in 64 bits
def _d(a):
    """(x, y, z) array -> (z, y, x) double on the GPU."""
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a).transpose(2, 1, 0))).cuda().double()


def _rotation(e):
    f, p, t = (math.radians(float(v)) for v in e)
    cf, sf, cp, sp, ct, st = math.cos(f), math.sin(f), math.cos(p), math.sin(p), math.cos(t), math.sin(t)
    return ((cp * cf - ct * sp * sf, sp * cf + ct * cp * sf, st * sf),
            (-cp * sf - ct * sp * cf, -sp * sf + ct * cp * cf, st * cf),
            (st * sp, -st * cp, ct))


def _rotate(T, e):
    """Trilinear turn of a (z, y, x) volume by [phi psi theta] about ceil(n / 2)."""
    n = T.shape[::-1]
    c = [(s + 1) // 2 for s in n]
    ax = [torch.arange(s, device=T.device, dtype=torch.float64) - k for s, k in zip(n, c)]
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    out_ok = torch.ones(T.shape, dtype=torch.bool, device=T.device)
    base, frac = [], []
    for r, k, s in zip(_rotation(e), c, n):
        q = k + r[0] * x + r[1] * y + r[2] * z
        out_ok &= (q >= 0) & (q <= s - 1)
        q = q.clamp(0, s - 1)
        b = q.floor()
        base.append(b.long())
        frac.append(q - b)
    P = torch.nn.functional.pad(T[None, None], (0, 1, 0, 1, 0, 1))[0, 0]  # nothing beyond the last sample
    acc = torch.zeros_like(T)
    for dz in (0, 1):
        for dy in (0, 1):
            for dx in (0, 1):
                w = (frac[0] if dx else 1 - frac[0]) * (frac[1] if dy else 1 - frac[1]) * (frac[2] if dz else 1 - frac[2])
                acc += w * P[base[2] + dz, base[1] + dy, base[0] + dx]
    return torch.where(out_ok, acc, torch.zeros_like(acc))


def _weighted(t, W):
    return t if W is None else torch.fft.ifftn(torch.fft.fftn(t) * torch.fft.ifftshift(W)).real


def _placed(t, shape):
    """The box with its centre at the origin of a volume, wrapped around."""
    P = torch.zeros(shape, dtype=torch.float64, device=t.device)
    P[:t.shape[0], :t.shape[1], :t.shape[2]] = t
    return torch.roll(P, [-(s // 2) for s in t.shape], (0, 1, 2))


def _statistics(V, M):
    m = float((M > 0).sum())
    g = float(V.mean())
    s = float(M.sum()) / m
    FM = torch.fft.rfftn(_placed(M, V.shape))
    D = V - g
    mu = torch.fft.irfftn(torch.fft.rfftn(D) * FM, s=V.shape) / m
    e2 = torch.fft.irfftn(torch.fft.rfftn(D * D) * FM, s=V.shape) / m
    var = (e2 - mu * mu) + (1 - s) * (2 * g * mu + g * g * s)
    var = torch.where(var > 1e-12 * float((D * D).mean()), var, torch.zeros_like(var))
    return mu + g * s, var.sqrt(), m


def _template(T, M, W):
    a = 1e5 * (T + 1) * 2 + 100
    Tn = (a - a.mean()) / a.std(unbiased=False)
    return (Tn,) + _under_mask(_weighted(Tn, W), M)


def _under_mask(t, M):
    v = t[M != 0]
    return float(v.mean()), float(v.std(unbiased=False))


def _scores(c, mu, sig, m, mu_t, sig_t):
    den = sig * sig_t
    return torch.where(den > 0, (c / m - mu * mu_t) / torch.where(den > 0, den, torch.ones_like(den)), torch.zeros_like(c))


def _conv(x, w, b, t):
    """x [D][H][W][in], w [tap][out][in]."""
    D, H, Wd, _ = x.shape
    if t == 1:
        return x @ w[0].T + b
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    y = b.expand(D * H * Wd, -1).clone()
    for k in range(27):
        z, yy, xx = k // 9, k // 3 % 3, k % 3
        y = y + p[z:z + D, yy:yy + H, xx:xx + Wd].reshape(D * H * Wd, -1) @ w[k].T
    return y.reshape(D, H, Wd, -1)


def _network(layers, vol, aux):
    F = torch.nn.functional

    def conv(i, x):
        return torch.relu(_conv(x, *layers[i], LAYERS[i][2]))

    def pool(x):
        return F.avg_pool3d(x.permute(3, 0, 1, 2)[None], 2)[0].permute(1, 2, 3, 0)

    def up(x):
        return F.interpolate(x.permute(3, 0, 1, 2)[None], scale_factor=2, mode="trilinear",
                             align_corners=False)[0].permute(1, 2, 3, 0)

    x = torch.stack([vol, aux], -1)
    l0 = (layers[0][0][:, :, :2], layers[0][1])
    s1 = conv(1, torch.relu(_conv(x, *l0, 27)))
    s2 = conv(3, conv(2, pool(s1)))
    b = conv(5, conv(4, pool(s2)))
    d2 = conv(7, conv(6, torch.cat([up(b), s2], -1)))
    d1 = conv(9, conv(8, torch.cat([up(d2), s1], -1)))
    return _conv(d1, *layers[10], 1)


def _unpack(theta):
    out, at = [], 0
    t = torch.from_numpy(theta).cuda().double()
    for ci, co, k in LAYERS:
        w = t[at:at + k * co * ci].reshape(k, co, ci).clone()
        b = t[at + k * co * ci:at + k * co * ci + co].clone()
        at += k * co * ci + co
        out.append((w, b))
    return out


def _exact_subtomo(case, seed):
    boxes, packed, pbox, wedge, angles = _subtomo_inputs(case, seed)
    out, at = [], 0
    for p in range(case["P"]):
        box = boxes[pbox[p]]
        B = box["template"].shape[0]
        n = B ** 3
        v = packed[at:at + n].reshape(B, B, B).double()
        at += n
        M, near = _d(box["mask"]), _d(box["mask_cc"]) != 0
        T = _d(box["template"])
        T = T - T.mean()
        inside = M != 0
        k = float(inside.sum())

        def norm(t, w):
            t = torch.where(inside, (t - (t * inside).sum((-3, -2, -1), keepdim=True) / k) * w, torch.zeros_like(t))
            mean = t.sum((-3, -2, -1), keepdim=True) / k
            var = ((t * t).sum((-3, -2, -1)) - k * mean[..., 0, 0, 0] ** 2) / n
            return torch.where(inside, t - mean, torch.zeros_like(t)), var

        f = torch.fft.fftfreq(B, 1.0 / B, device="cuda", dtype=torch.float64)
        kz, ky, kx = torch.meshgrid(f, f, f, indexing="ij")
        keep = (kx * kx + ky * ky + kz * kz <= ((B - 1) // 2) ** 2) & (kx.abs() >= math.tan(math.radians(float(wedge[p]))) * kz.abs())
        P_, var_p = norm(v[None], M)
        P_ = torch.fft.fftn(P_, dim=(1, 2, 3))
        t = torch.stack([_rotate(T, e) for e in angles[p]])
        t, _ = norm(t, M)
        F = torch.fft.fftn(t, dim=(1, 2, 3)) * keep
        F[:, 0, 0, 0] = 0
        t, var_t = norm(torch.fft.ifftn(F, dim=(1, 2, 3)).real * n, torch.ones_like(M))
        C = torch.fft.fftn(t, dim=(1, 2, 3)).conj() * P_
        C[:, 0, 0, 0] = 0
        c = torch.fft.ifftn(C, dim=(1, 2, 3)).real / n / (var_p * var_t).sqrt()[:, None, None, None]
        out.append(float(c[:, near].max()))
    return None, None, np.asarray(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "picks":
        return None  # values of the map, picked
    if kind == "subtomo":
        # which frequencies a turned wedge keeps is decided in 32 bits
        return None if case["ref"] else _exact_subtomo(case, seed)
    if kind in ("infer", "train"):
        theta, vol, aux = _net_inputs(case, seed)
        layers = _unpack(theta)
        vol, aux = vol.double(), aux.double()
        if kind == "infer":
            if case["halo"]:
                return None  # seams of the tiles
            L = _network(layers, *((v - v.mean()) / v.std(unbiased=False) for v in (vol, aux)))
            return L[..., 0], None, L[..., 65:68]
        if vol.numel() > 100 ** 3:
            return None
        for w, b in layers:
            w.requires_grad_(True)
            b.requires_grad_(True)
        F = torch.nn.functional
        L = _network(layers, vol, aux).reshape(-1, 80)
        prob, tbin, off = (t.reshape(-1) for t in _targets(seed, tuple(vol.shape)))
        off = off.reshape(-1, 4).double()
        bce = F.binary_cross_entropy_with_logits(L[:, 0], prob.double(), pos_weight=torch.tensor(20.0, device="cuda", dtype=torch.float64))
        s = tbin >= 0
        ce = F.cross_entropy(L[s][:, 1:65], tbin[s].long())
        w = off[:, 3] > 0
        po = ((L[w][:, 65:68] - off[w][:, :3]) ** 2).sum(1).mean()
        (bce + ce + po).backward()
        g = []
        for i, (a, b) in enumerate(layers):
            a.grad[:, :, 2:] *= 0 if i == 0 else 1
            g += [a.grad.reshape(-1), b.grad]
        return (float(bce), float(ce), float(po)), torch.cat(g).cpu().numpy()
    rng, V, T, M, W = _matching(case, seed)
    V, T, M = V.double(), _d(T), _d(M)
    W = None if W is None else _d(W)
    if kind == "refine":
        mu, sig, m = _statistics(V, M)
        Tn, mu_t, sig_t = _template(T, M, W)
        angles, cand = _refine_inputs(case, rng)
        n = T.shape[::-1]
        best = []
        for p in range(case["P"]):
            x, y, z = (int(v) for v in cand[p, :3])
            t = torch.stack([(_weighted(_rotate(Tn, angles[a, p]) * M, W) if W is not None
                              else _rotate(Tn, angles[a, p]) * M) * M for a in range(case["A"])])
            i = [(torch.arange(s + 2, device="cuda") + k - 1 - s // 2) % N for s, k, N in zip(n, (x, y, z), V.shape[::-1])]
            w = V[i[2]][:, i[1]][:, :, i[0]]
            top = -1e30
            for dz in range(3):
                for dy in range(3):
                    for dx in range(3):
                        q = w[dz:dz + n[2], dy:dy + n[1], dx:dx + n[0]].reshape(-1)
                        at = ((z + dz - 1) % V.shape[0], (y + dy - 1) % V.shape[1], (x + dx - 1) % V.shape[2])
                        c = float((t.reshape(len(t), -1) @ q).max()) / m
                        den = sig_t * float(sig[at])
                        top = max(top, (c - float(mu[at]) * mu_t) / den if den > 0 else 0.0)
            best.append(top)
        return np.asarray(best), None, None
    mu, sig, m = _statistics(V, M)
    FV = torch.fft.rfftn(V)
    if kind == "corr":
        mu_t, sig_t = _under_mask(T, M)
        c = torch.fft.irfftn(FV * torch.fft.rfftn(_placed(T * M, V.shape)).conj(), s=V.shape)
        return _scores(c, mu, sig, m, mu_t, sig_t)
    Tn, mu_t, sig_t = _template(T, M, W)
    best = None
    for e in _euler(rng, case["A"]):
        t = _weighted(_rotate(Tn, e) * M, W) * M
        c = torch.fft.irfftn(FV * torch.fft.rfftn(_placed(t, V.shape)).conj(), s=V.shape)
        best = c if best is None else torch.maximum(best, c, out=best)
    return _scores(best, mu, sig, m, mu_t, sig_t), None
