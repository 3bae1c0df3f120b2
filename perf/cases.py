"""The work that a program built on damascene_amd gives it, as measurable cases.

Kinds of case, each one public entry point or the short sequence of them
that a program calls together (damascene_amd.Context):

  image     gpb(): one RGB image to oriented gPb, the whole pipeline
  batch     gpb_batch(): a list of images of uneven sizes
  textons   rgb_to_grey + find_textons: filter bank and k-means
  cues      rgb_to_lab + local_cues: brightness, colour and texture gradients
  affinity  intervene + convert_matrix: the normalised Laplacian of an image
  solve     intervene + generalized_eigensolve + spectral_pb
  finish    combine ... postprocess: everything after the cues and the solver
  fit       one training step of the weights: forward, loss and backward

A case is a dict: kind, w, h and, where the path has them, `mixed` (the
block solver and MFMA k-means, or the plain FP32 reference algorithm),
`textons` (32 or 64) and `images`.  Images are the framework's synthetic
ones (Voronoi cells, half of them with gratings, and noise) with the cell
density of the benchmark: 40 cells at 481x321.
"""
import math

import numpy as np
import torch

import damascene_amd as dm
from damascene_amd import autograd as dag

N_EIG = 9
GAMMA = 0.0139  # weight of the spectral Pb (globalPb.cu:13)


def listed():
    return [
        # one photograph at the size of the benchmark (BSDS), accurate eigenvectors: the headline call
        dict(name="image mixed 481x321", kind="image", w=481, h=321, mixed=True, textons=32),
        # a directory of photographs of different sizes on the reference algorithm
        dict(name="batch plain uneven", kind="batch", w=480, h=360, mixed=False, textons=32, images=6),
        # texton maps alone, as a feature extractor: the exact FP32 k-means ...
        dict(name="textons plain 481x321", kind="textons", w=481, h=321, mixed=False, textons=32),
        # ... and the 64-cluster one on a large image
        dict(name="textons64 mixed 1024x768", kind="textons", w=1024, h=768, mixed=True, textons=64),
        # local boundary cues of a portrait photograph
        dict(name="cues 321x481", kind="cues", w=321, h=481, textons=32),
        # the same with 64 textons on a wide strip with odd sides
        dict(name="cues64 517x233", kind="cues", w=517, h=233, textons=64),
        # the affinity matrix alone, for a caller's own spectral clustering
        dict(name="affinity 640x480", kind="affinity", w=640, h=480),
        # globalisation with the reference's FP32 Lanczos
        dict(name="solve plain 481x321", kind="solve", w=481, h=321, mixed=False),
        # globalisation of a thumbnail: launches and host round trips count
        dict(name="solve mixed 160x120", kind="solve", w=160, h=120, mixed=True),
        # globalisation of a large image: the longest call
        dict(name="solve mixed 1024x768", kind="solve", w=1024, h=768, mixed=True),
        # combination, suppression and thinning of a thumbnail: small launches
        dict(name="finish 160x120", kind="finish", w=160, h=120, textons=32),
        # one training step of the cue and spectral weights
        dict(name="fit 481x321", kind="fit", w=481, h=321, textons=32),
    ]


def draw(rng):
    kind = rng.choice(["image", "batch", "textons", "cues", "affinity", "solve", "solve", "finish", "fit"])
    # area over its logarithm; the solvers' range ends where a draw could cost
    # more than the largest listed case
    top = {"image": 640 * 480, "batch": 480 * 360, "solve": 640 * 480}.get(kind, 1024 * 768)
    area = math.exp(rng.uniform(math.log(96 * 80), math.log(top)))
    aspect = math.exp(rng.uniform(math.log(0.5), math.log(2.0)))
    w = max(64, int(round(math.sqrt(area * aspect))))
    h = max(64, min(int(round(area / w)), top // w))
    case = dict(kind=kind, w=w, h=h)
    if kind in ("image", "batch", "textons", "solve"):
        case["mixed"] = rng.random() < 0.5
    if kind in ("image", "batch", "textons", "cues", "finish", "fit"):
        case["textons"] = 64 if rng.random() < 0.3 else 32
    if kind == "batch":
        case["images"] = rng.randint(2, 6)
    return case


# ------------------------------------------------------------------ inputs

_context = None


def _ctx():
    """The program's one context, kept for its life (scratch arenas, plans)."""
    global _context
    if _context is None:
        _context = dm.Context(0)
    return _context


def _image(w, h, seed):
    """(RGB8 on the device, cell index map on the host)."""
    cells = max(4, round(40 * (w * h / (481 * 321)) ** 0.6))
    rgb, index = dm.generate_image(w, h, cells, seed, with_cells=True)
    return _ctx().upload(rgb), index


def _choice(case):
    return dm.TEXTON64 if case["textons"] == 64 else dm.TEXTON32


def _precision(case):
    return dm.PREC_MIXED if case["mixed"] else dm.PREC_FP32


def _pitched(t, n):
    """A [planes, N] view as a pitched stack, the form combine() takes."""
    out = torch.zeros(t.shape[0], dm.pitch_in_floats(n), device=t.device)
    out[:, :n] = t[:, :n]
    return out


def _cues(rgb, texton_choice):
    """The four cue stacks of an image, pitched."""
    ctx = _ctx()
    h, w = rgb.shape
    tex, _ = ctx.find_textons(ctx.rgb_to_grey(rgb), texton_choice=texton_choice)
    return [_pitched(c, w * h) for c in ctx.local_cues(*ctx.rgb_to_lab(rgb), tex, texton_choice=texton_choice)]


def _thin_pb(rgb):
    """The thinned mPb of an image, the input of the affinity stage."""
    h, w = rgb.shape
    mpb, _ = _ctx().combine(w, h, *_cues(rgb, dm.TEXTON32))
    return _ctx().non_max_suppression(w, h, mpb)


def _smooth_vectors(index, seed):
    """Vectors like the solver's: smooth inside the cells with steps between
    them, each mapped to [0, 1]; and rising eigenvalues."""
    h, w = index.shape
    dev = _ctx().device
    gen = torch.Generator().manual_seed(seed)
    level = torch.rand(N_EIG, int(index.max()) + 1, generator=gen).to(dev)
    f = torch.rand(N_EIG, 4, generator=gen).to(dev)
    x = (torch.arange(w, device=dev) + 0.5) / w
    y = ((torch.arange(h, device=dev) + 0.5) / h)[:, None]
    v = level[:, torch.from_numpy(index.astype(np.int64)).to(dev)]
    for i in range(N_EIG):
        v[i] += torch.cos(math.pi * (3 * f[i, 0] * x + f[i, 1])) * torch.cos(math.pi * (3 * f[i, 2] * y + f[i, 3]))
    lo, hi = v.amin((1, 2), keepdim=True), v.amax((1, 2), keepdim=True)
    vals = np.cumsum(torch.rand(N_EIG, generator=gen).numpy() * 2e-5 + 5e-6).astype(np.float32)
    return vals, ((v - lo) / (hi - lo)).contiguous()


def prepare(case, seed):
    ctx, kind, w, h = _ctx(), case["kind"], case["w"], case["h"]
    rgb, index = _image(w, h, seed)
    s = {"case": case, "rgb": rgb}
    if kind == "batch":
        s["rgbs"] = [rgb]
        for i in range(1, case["images"]):  # the rest between a third of the first one's sides and all of them
            r = np.random.RandomState(i)
            wi, hi = (max(64, int(round(side * r.uniform(1 / 3, 1)))) for side in (w, h))
            s["rgbs"].append(_image(wi, hi, seed + i)[0])
    elif kind == "cues":
        s["tex"], _ = ctx.find_textons(ctx.rgb_to_grey(rgb), texton_choice=_choice(case))
    elif kind in ("affinity", "solve"):
        s["pb"] = _thin_pb(rgb)
    elif kind == "finish":
        s["cues"] = _cues(rgb, _choice(case))
        s["vals"], s["vecs"] = _smooth_vectors(index, seed)
    elif kind == "fit":
        vals, vecs = _smooth_vectors(index, seed)
        s["op"] = dag.SpbCombine(ctx, w, h, _cues(rgb, _choice(case)))
        s["params"] = dag.reference_params(vals, _choice(case), device=ctx.device).requires_grad_(True)
        s["vecs"] = vecs.requires_grad_(True)
        s["mask"] = torch.from_numpy(dm.boundary_mask(index)).to(ctx.device) > 0
    return s


# --------------------------------------------------------------------- run

_WHOLE = ("textons", "mpb", "combined_g", "nmax", "eigvecs", "eigvals", "spb", "gpb_all", "gpb")


def run(s):
    ctx, case = _ctx(), s["case"]
    kind, w, h = case["kind"], case["w"], case["h"]
    if kind == "image":
        out = ctx.gpb(s["rgb"], precision=_precision(case), texton_choice=_choice(case))
        return {k: out[k] for k in _WHOLE}
    if kind == "batch":
        outs = ctx.gpb_batch(s["rgbs"], precision=_precision(case), texton_choice=_choice(case))
        return [{k: o[k] for k in _WHOLE} for o in outs]
    if kind == "textons":
        return ctx.find_textons(ctx.rgb_to_grey(s["rgb"]), precision=_precision(case), texton_choice=_choice(case))
    if kind == "cues":
        L, a, b = ctx.rgb_to_lab(s["rgb"])
        return ctx.local_cues(L, a, b, s["tex"], texton_choice=_choice(case))
    if kind == "affinity":
        m = ctx.intervene(s["pb"])
        d, rs = ctx.convert_matrix(w, h, m)
        return m, d, rs
    if kind == "solve":
        vals, vecs, steps = ctx.generalized_eigensolve(w, h, ctx.intervene(s["pb"]), nvec=N_EIG,
                                                       precision=_precision(case))
        return vals, vecs, ctx.spectral_pb(vals, vecs), steps
    if kind == "finish":
        mpb, cg = ctx.combine(w, h, *s["cues"], texton_choice=_choice(case))
        nmax = ctx.non_max_suppression(w, h, mpb)
        spb = ctx.spectral_pb(s["vals"], s["vecs"])
        all_, gpb = ctx.calc_gpb(w, h, cg, spb, nmax)
        prob, thin, rounds = ctx.postprocess(gpb, nmax)
        return {"mpb": mpb, "cg": cg, "nmax": nmax, "spb": spb, "all": all_, "gpb": gpb, "prob": prob, "thin": thin,
                "rounds": rounds, "norm": ctx.normalize_gpb_all(all_, w * h)}
    pre = s["op"](s["params"], s["vecs"])
    loss = dag.balanced_bce(pre, s["mask"])
    grads = torch.autograd.grad(loss, (s["params"], s["vecs"]))
    return {"pre": pre.detach(), "loss": loss.detach(), "params": grads[0], "vecs": grads[1]}


def work(case):
    """Inputs read and outputs written once, and the arithmetic of the
    method: per pixel 2 x 9,010 for the filter bank, 2 x 34 per k-means
    centre and pass (15), 2 x 58,720 for the smoothing filters, 81 x 2 per
    matrix product and vector."""
    kind, n = case["kind"], case["w"] * case["h"]
    k = case.get("textons", 32)
    bank, means, cues = 2 * 9010, 15 * 2 * 34 * k, 2 * 58720
    spb = 2 * 8 * 49 * (N_EIG - 1)
    # products with the matrix that the size needs, from the grid's spectrum
    # (the plain solver checks every 500 single-vector steps)
    side = math.sqrt(n)
    solve = 162 * (32 * side if case.get("mixed") else 500)
    whole = dict(bytes=4 * n * (1 + 1 + 8 + 8 + 1 + N_EIG + 8 + 8 + 1), flops=n * (bank + means + cues + solve + spb))
    if kind == "image":
        return whole
    if kind == "batch":
        mean = (1 + 4 / 9 * (case["images"] - 1)) / case["images"]  # mean area of the batch over the largest
        return {q: v * mean * case["images"] for q, v in whole.items()}
    return {
        "textons": dict(bytes=8 * n, flops=n * (bank + means)),
        "cues": dict(bytes=4 * n * (1 + 1 + 96), flops=n * cues),
        "affinity": dict(bytes=4 * n * (1 + 81 + 2), flops=n * 81 * 20),
        "solve": dict(bytes=4 * n * (1 + N_EIG + 8), flops=n * (solve + spb)),
        "finish": dict(bytes=4 * n * (96 + N_EIG + 8 + 8 + 1 + 8 + 8 + 1 + 1 + 1 + 8), flops=n * (8 * 48 + spb)),
        "fit": dict(bytes=4 * n * (96 + N_EIG + 1 + 1 + N_EIG), flops=n * 3 * spb),
    }[kind]


# ------------------------------------------------- the same in 64 bits

F32, F64 = np.float32, torch.float64


def exact(case, seed):
    """None where the result is a decision (labels, masks), where the method
    itself stops early (the plain solver) or where 64 bits would take too
    long (whole images, large solves)."""
    kind, w, h = case["kind"], case["w"], case["h"]
    if kind in ("image", "batch", "textons") or (kind == "solve" and (not case["mixed"] or w * h > 40000)):
        return None
    s = prepare(case, seed)
    if kind == "cues":
        L, a, b = _ctx().rgb_to_lab(s["rgb"])
        return _cues64(w, h, [L, a, b, s["tex"]], case["textons"])
    if kind == "affinity":
        return _laplacian64(_affinity64(s["pb"]))
    if kind == "solve":
        A, _, rs = _laplacian64(_affinity64(s["pb"]))
        vals, u = _smallest64(A[:, : w * h], w, h)
        v = u * rs.reshape(-1)[None]
        lo, hi = v.amin(1, keepdim=True), v.amax(1, keepdim=True)
        return vals.cpu().numpy(), None, _spectral64(vals, ((v - lo) / (hi - lo)).reshape(-1, h, w)), None
    if kind == "finish":
        C = torch.stack([c[:, : w * h].double() for c in s["cues"]]).reshape(12, 8, -1)
        coef, wts = _weights(case["textons"])
        mpb, cg = (_pad64(torch.einsum("k,kop->op", t.to(C.device), C)) for t in (coef, wts))
        spb = _spectral64(torch.from_numpy(s["vals"]).to(C), s["vecs"].double())
        all_ = cg + GAMMA * spb
        norm = all_.clone()
        z = (1.2 * all_[:, : w * h]).clamp(0, 1)
        norm[:, : w * h] = (torch.sigmoid(10.7998 * z - 2.6433) - 0.0667) / 0.9333
        return {"mpb": mpb, "cg": cg, "nmax": None, "spb": spb, "all": all_, "gpb": None, "prob": None, "thin": None,
                "rounds": None, "norm": norm}
    p, v = (s[k].detach().double().requires_grad_(True) for k in ("params", "vecs"))
    C = torch.stack([c[:, : w * h].double() for c in s["op"].cues]).reshape(12, 8, h, w)
    spb = (p[14:, None, None, None] * _derivative64(v[1:]).abs()).sum(0)
    pre = ((p[:12, None, None, None] * C).sum(0) + p[12] * spb).max(0).values
    y = s["mask"].double()
    loss = torch.nn.functional.binary_cross_entropy_with_logits(
        10.7998 * pre - 2.6433, y, weight=(1 - y.mean()) * y + y.mean() * (1 - y))
    gp, gv = torch.autograd.grad(loss, (p, v))
    return {"pre": pre.detach(), "loss": loss.detach(), "params": gp, "vecs": gv}


def _pad64(t):
    """[planes, N] with the zero columns of a pitched stack."""
    pad = -t.shape[1] % 64
    return torch.nn.functional.pad(t, (0, pad)) if pad else t


def _weights(textons):
    """combine.cu:16-21: coefficients of mPb and weights of combinedG."""
    coef = [0.0123, 0.0110, 0.0117, 0.0169, 0.0176, 0.0198, 0.0138, 0.0138, 0.0145]
    wts = [0.0, 0.0, 0.0028, 0.0041, 0.0042, 0.0047, 0.0033, 0.0033, 0.0035]
    coef += [0.0104, 0.0105, 0.0115] if textons == 64 else [0.0144, 0.0149, 0.0158]
    wts += [0.0025, 0.0025, 0.0137] if textons == 64 else [0.0035, 0.0035, 0.0188]
    return torch.tensor(coef, dtype=F64), torch.tensor(wts, dtype=F64)


def _mirror(n, border):
    i = np.arange(n + 2 * border)
    return np.where(i < border, border - i - 1, np.where(i < border + n, i - border, border + 2 * n - i - 1))


def _edge_filters():
    """The eight 7x7 first derivatives of a Gaussian (spectralPb.cu:708-717),
    [dx][dy]: separable on the rotated bounding grid, resampled bilinearly."""
    out = []
    for o in range(8):
        ori = math.pi / 2 + (7 - o) * math.pi / 8
        c, s = math.cos(-ori), math.sin(-ori)
        rx, ry = (math.ceil(max(abs(3 * p - 3 * q), abs(3 * p + 3 * q))) for p, q in ((c, s), (s, c)))
        x, y = np.arange(-rx, rx + 1.0), np.arange(-ry, ry + 1.0)
        kx, ky = np.exp(-x * x / 2), -y * np.exp(-y * y / 2)
        kx, ky = kx / kx.sum(), (ky - ky.mean()) / np.abs(ky - ky.mean()).sum()
        grid, f, c, s = np.outer(kx, ky), np.zeros((7, 7)), math.cos(ori), math.sin(ori)
        for i in range(7):
            for j in range(7):
                px, py = (i - 3) * c + (j - 3) * s + rx, (j - 3) * c - (i - 3) * s + ry
                x0, x1, y0, y1 = math.floor(px), math.ceil(px), math.floor(py), math.ceil(py)
                if px < 0 or py < 0 or x1 > 2 * rx or y1 > 2 * ry:
                    continue
                fx, fy = px - x0, py - y0
                f[i, j] = ((1 - fx) * (1 - fy) * grid[x0, y0] + fx * (1 - fy) * grid[x1, y0] +
                           (1 - fx) * fy * grid[x0, y1] + fx * fy * grid[x1, y1])
        f -= f.mean()
        out.append(f / np.abs(f).sum())
    return out


def _derivative64(v):
    """[k, 8, h, w]: each vector, mirrored by 3, under the eight filters.  The
    product's table is indexed (3 + u) + 7 (3 + v) over the array [dx][dy]."""
    _, h, w = v.shape
    ix, iy = (torch.from_numpy(_mirror(n, 3)).to(v.device) for n in (w, h))
    m = v[:, iy][:, :, ix]
    out = []
    for f in _edge_filters():
        flat = f.reshape(-1)
        out.append(sum(flat[i + 7 * j] * m[:, j:j + h, i:i + w] for i in range(7) for j in range(7)))
    return torch.stack(out, 1)


def _spectral64(vals, v):
    r = _derivative64(v[1:]).abs() / vals[1:].to(v).sqrt()[:, None, None, None]
    return _pad64(r.sum(0).reshape(8, -1))


# Bresenham line from (x0, y0) to (x1, y1), both ends included; the minor
# axis moves when the running error passes zero.
def _line(x0, y0, x1, y1):
    dx, dy = x1 - x0, y1 - y0
    ax, ay = abs(dx), abs(dy)
    if dx > 0 and dy >= 0:
        xmajor = ax > ay
    elif dx <= 0 and dy > 0:
        xmajor = ax >= ay
    elif dy <= 0 and dx < 0:
        xmajor = ax > ay
    else:
        xmajor = ax >= ay
    # a step of a zero component is never taken
    sx, sy = (1 if dx > 0 else -1), (1 if dy > 0 else -1)
    out, x, y, t = [(x0, y0)], x0, y0, -(ax if xmajor else ay)
    while (x, y) != (x1, y1):
        if xmajor:
            x, t = x + sx, t + 2 * ay
            if t > 0:
                y, t = y + sy, t - 2 * ax
        else:
            y, t = y + sy, t + 2 * ax
            if t > 0:
                x, t = x + sx, t - 2 * ay
        out.append((x, y))
    return out


def _away(x):
    """Round half away from zero."""
    return int(math.copysign(math.floor(abs(float(x)) + 0.5), float(x)))


def _rotation(o, W, H):
    """Frame size and the baseline and guideline tables of orientation o
    (rotate.cu:805-850), decided in FP32 as the tables are."""
    if o == 0:
        return W, H, np.arange(W), np.zeros(W, int), np.zeros(H, int), np.arange(H)
    theta = F32((0.25 - o / 8) * math.pi) if o > 2 else F32(-o / 8 * math.pi)
    t = F32(math.tan(float(theta)))
    fw, fh = F32(W - 1), F32(H - 1)
    if o <= 2:
        nw, nh = math.ceil(F32(W) - fh * t), math.ceil(F32(H) - fw * t)
        b, g = _line(0, 0, W - 1, -_away(fw * t)), _line(-_away(fh * t), 0, 0, H - 1)
    else:
        nw, nh = math.ceil(F32(H) - fw * t), math.ceil(F32(W) - fh * t)
        b, g = _line(0, 0, -_away(fw * t), W - 1), _line(H - 1, 0, 0, -_away(fh * t))
    b, g = np.array(b), np.array(g)
    return nw, nh, b[:, 0], b[:, 1], g[:, 0], g[:, 1]


def _corners(o, radius, w, h, bx, by, gx, gy):
    """(dy, dx) of the eight corners A..H of the half-disc pair in the rotated
    frame (rotate.cu:480-614)."""
    theta = float(F32(-o / 8 * math.pi))
    er = F32((-4.0 + 4.0 * radius * float(np.sqrt(F32(math.pi)))) / 8.0)
    s, c = F32(math.sin(theta)), F32(math.cos(theta))
    xc, yc = w // 2, h // 2

    def at(x, y):
        x, y = min(max(x, 0), len(bx) - 1), min(max(y, 0), len(gx) - 1)
        return gx[y] + bx[x], gy[y] + by[x]
    ax, ay = at(_away(-er * s - er * c) + xc, _away(-er * s + er * c) + yc)
    qx, qy = at(_away(er * s + er * c) + xc, _away(er * s - er * c) + yc)
    xd, yd = int(qx - ax) + 1, int(ay - qy) + 1
    xr, yr = (int(d / 2) for d in (xd, yd))
    left, top = (-r - 1 if d & 1 else -r for r, d in ((xr, xd), (yr, yd)))
    return list(zip([top, top, top, 0, 0, yr, yr, yr], [left, 0, xr, left, xr, left, 0, xr]))


def _blur(sigma):
    r = math.ceil(3 * sigma)
    k = np.exp(-0.5 * np.arange(-r, r + 1.0) ** 2 / sigma ** 2)
    return k / k.sum()


def _smoothing_filter(radius, o):
    """Savitzky-Golay fit on an ellipse (localcues.cu:21-100): the taps are
    chosen in FP32, their values formed in 64 bits."""
    theta = float(F32(math.pi / 2 - o * math.pi / 8))
    ra, rb = F32(max(1.5, radius)), F32(max(1.5, radius / 4))
    ia, ib = F32(1.0 / float(ra * ra)), F32(1.0 / float(rb * rb))
    st, ct = F32(math.sin(theta)), F32(math.cos(theta))
    r = int(math.floor(max(ra, rb)) + 0.5)
    taps = []
    for u in range(-r, r + 1):
        for v in range(-r, r + 1):
            a = F32(-u) * st + F32(v) * ct
            b = F32(u) * ct + F32(v) * st
            if not a * a * ia + b * b * ib > 1:
                taps.append((v, u, float(a)))
    a = np.array([t[2] for t in taps])
    M = np.array([[np.sum(a ** (i + j)) for j in range(3)] for i in range(3)])
    c = np.linalg.inv(M)[:, 0]
    return [(v, u, c[0] + c[1] * x + c[2] * x * x) for v, u, x in taps]


def _chi2(a, b):
    def norm(t):
        s = t.sum(0)
        return t * torch.where(s != 0, 8 / s.clamp(min=1e-300), torch.zeros_like(s))
    a, b = norm(a), norm(b)
    s = a + b
    return 0.5 * torch.where(s != 0, (a - b) ** 2 / s.clamp(min=1e-300), torch.zeros_like(s)).sum(0)


def _blurred(t, k):
    if k is None:
        return t
    r, n = len(k) // 2, t.shape[0]
    out = torch.zeros_like(t)
    for i in range(n):
        for m in range(2 * r + 1):
            if 0 <= i - r + m < n:
                out[i] += k[m] * t[i - r + m]
    return out


def _cues64(w, h, planes, textons):
    """The four [24, N] stacks: half-disc histograms are whole counts, the
    rest is in 64 bits (gradient.cu:201-243, rotate.cu:263-475,
    parabola.cu:75-124)."""
    n, B, dev = w * h, 30, planes[0].device
    iy, ix = (torch.from_numpy(_mirror(k, B)).to(dev) for k in (h, w))
    frames = [_rotation(o, w + 2 * B, h + 2 * B) for o in range(4)]
    out = []
    for ch in range(4):
        if ch == 3:
            lab, bins, blur, radii = planes[3].long(), textons, None, (5, 10, 20)
        else:
            lab = torch.floor(planes[ch] * 25.0).long().clamp(max=24)  # quantised in FP32
            bins, blur, radii = 25, _blur(2.0 if ch == 0 else 1.0), ((3, 5, 10) if ch == 0 else (5, 10, 20))
        lab = lab[iy][:, ix]
        grads = torch.zeros(3, 8, h, w, dtype=F64, device=dev)
        for o, (nw, nh, bx, by, gx, gy) in enumerate(frames):
            tb, tg = (torch.from_numpy(np.stack(t)).to(dev) for t in ((bx, by), (gx, gy)))
            rx, ry = tg[0][:, None] + tb[0][None], tg[1][:, None] + tb[1][None]
            frame = torch.full((nh * nw,), -1, dtype=torch.long, device=dev)
            frame[(ry * nw + rx).reshape(-1)] = lab.reshape(-1)
            one = frame.reshape(1, nh, nw) == torch.arange(bins, device=dev)[:, None, None]
            total = one.cumsum(1, dtype=torch.int32).cumsum(2, dtype=torch.int32).reshape(bins, -1)
            del one
            at = (ry * nw + rx)[B:B + h, B:B + w].reshape(-1)
            for sc, radius in enumerate(radii):
                A, Bc, C, D, E, F, G, H = (total[:, at + dy * nw + dx].double()
                                           for dy, dx in _corners(o, radius, w, h, bx, by, gx, gy))
                for slot, p, q in ((o + 4, A - C + E - D, H - F + D - E), (o, A - F + G - Bc, H - C + Bc - G)):
                    grads[sc, slot] = _chi2(_blurred(p, blur), _blurred(q, blur)).reshape(h, w)
            del total
        res = torch.zeros(3, 8, h, w, dtype=F64, device=dev)
        padded = grads[:, :, iy][:, :, :, ix]
        for sc, radius in enumerate(radii):
            for o in range(8):
                for v, u, c in _smoothing_filter(radius, o):
                    res[sc, o] += c * padded[sc, o, B + v:B + v + h, B + u:B + u + w]
        out.append(res.reshape(24, n))
    return out


DISC = [(dy, dx) for dy in range(-5, 6) for dx in range(-5, 6) if dy * dy + dx * dx <= 25]


def _walk(found, p1, p2, p3):
    """intervening.cu:44-283 from (0, 0) to p2 between its neighbours p1 and
    p3 on the window's edge: for each disc point the walk speaks for, the
    pixels whose boundary strength it has crossed by then."""
    dot = lambda a, b: a[0] * b[0] + a[1] * b[1]  # noqa: E731
    crossed, (ox, oy) = [], (0, 0)
    for x, y in _line(0, 0, *p2)[1:]:
        if x == ox:
            crossed = crossed + [(x, max(y, oy) - 1)]
        elif y == oy:
            crossed = crossed + [(max(x, ox) - 1, y)]
        else:
            hy, vx = max(y, oy) - 1, max(x, ox) - 1
            crossed = crossed + [(ox, hy), (x, hy), (vx, oy), (vx, y)]
        q = (x, y)
        d2 = dot(q, p2) ** 2
        if d2 == dot(q, q) * dot(p2, p2) or (dot(p1, p1) * d2 > dot(p2, p2) * dot(q, p1) ** 2 and
                                              dot(p3, p3) * d2 >= dot(p2, p2) * dot(q, p3) ** 2):
            if x * x + y * y <= 25:
                found[(y, x)] = crossed
        ox, oy = x, y


def _window(l, r, t, b):
    """Disc points of a pixel whose window reaches l, r, t, b pixels, each
    with the pixels its line crosses; later walks replace earlier ones
    (intervening.cu:298-475)."""
    f = {(0, 0): None}
    if l:
        if t and b:
            _walk(f, (-l, -1), (-l, 0), (-l, 1))
        for y in range(-1, -t, -1):
            _walk(f, (-l, y - 1), (-l, y), (-l, y + 1))
    if l > 1 or t > 1 or (l and t):
        _walk(f, (-l, 1 - t), (-l, -t), (1 - l, -t))
    if t:
        for x in range(1 - l, r):
            _walk(f, (x - 1, -t), (x, -t), (x + 1, -t))
    if t > 1 or r > 1 or (t and r):
        _walk(f, (r - 1, -t), (r, -t), (r, 1 - t))
    if r:
        for y in range(1 - t, 0):
            _walk(f, (r, y - 1), (r, y), (r, y + 1))
    if l:
        for y in range(1, b):
            _walk(f, (-l, y - 1), (-l, y), (-l, y + 1))
    if l > 1 or b > 1 or (l and b):
        _walk(f, (-l, b - 1), (-l, b), (1 - l, b))
    if b:
        for x in range(1 - l, r):
            _walk(f, (x - 1, b), (x, b), (x + 1, b))
    if b > 1 or r > 1 or (b and r):
        _walk(f, (r - 1, b), (r, b), (r, b - 1))
    if r:
        for y in range(b - 1, 0, -1):
            _walk(f, (r, y - 1), (r, y), (r, y + 1))
        if t and b:
            _walk(f, (r, -1), (r, 0), (r, 1))
    # next to an image corner the first pixel of a side has no walk of its own
    for free, point in ((t == 1 and (not l or not r), (-1, 0)), (l == 1 and (not t or not b), (0, -1)),
                        (r == 1 and (not t or not b), (0, 1)), (b == 1 and (not l or not r), (1, 0))):
        if free:
            f[point] = []
    return f


def _affinity64(pb, sigma=0.1):
    """[81, h, w] affinities of a thinned boundary map."""
    h, w = pb.shape
    dev, pb = pb.device, pb.double()
    W = torch.zeros(len(DISC), h, w, dtype=F64, device=dev)
    groups = []
    for n in (w, h):  # runs of coordinates with the same reach to both sides
        g = {}
        for i in range(n):
            g.setdefault((min(i, 5), min(n - 1 - i, 5)), []).append(i)
        groups.append([(k, torch.tensor(v, device=dev)) for k, v in g.items()])
    for (l, r), xs in groups[0]:
        for (t, b), ys in groups[1]:
            grid = {}

            def at(x, y):
                if (x, y) not in grid:
                    grid[(x, y)] = pb[(ys + y).clamp(0, h - 1)[:, None], (xs + x).clamp(0, w - 1)[None]]
                return grid[(x, y)]
            best = {}

            def top(crossed):
                if not crossed:
                    return torch.zeros(len(ys), len(xs), dtype=F64, device=dev)
                key = tuple(crossed)
                if key not in best:
                    best[key] = torch.maximum(top(crossed[:-1]), at(*crossed[-1]))
                return best[key]
            for point, crossed in _window(l, r, t, b).items():
                if crossed is None:
                    val = torch.ones(len(ys), len(xs), dtype=F64, device=dev)
                else:
                    c = torch.sigmoid(1.8682 - 1.3113 / 0.3130 * top(crossed))
                    val = torch.exp((c - 1) / sigma)
                W[DISC.index(point), ys[:, None], xs[None]] = val
    for d, (dy, dx) in enumerate(DISC):
        if dy < 0 or (dy == 0 and dx <= 0):
            continue
        y, x = slice(max(0, -dy), h - max(0, dy)), slice(max(0, -dx), w - max(0, dx))
        yy, xx = slice(max(0, dy), h - max(0, -dy)), slice(max(0, dx), w - max(0, -dx))
        e = DISC.index((-dy, -dx))
        half = 0.5 * (W[d, y, x] + W[e, yy, xx])
        W[d, y, x] = half
        W[e, yy, xx] = half
    return W


def _laplacian64(W):
    """(L_sym as a pitched [81, pitch] matrix, row sums, their inverse square
    roots): columns are linear indices, as stencilMVM.cu:98-180 takes them."""
    _, h, w = W.shape
    n = h * w
    A = W.reshape(len(DISC), n)
    row = torch.arange(n, device=W.device)
    valid = [(row + dy * w + dx >= 0) & (row + dy * w + dx < n) for dy, dx in DISC]
    d = sum(torch.where(m, A[i], torch.zeros_like(A[i])) for i, m in enumerate(valid))
    rs = d.rsqrt()
    out = torch.zeros_like(A)
    for i, (dy, dx) in enumerate(DISC):
        col = (row + dy * w + dx).clamp(0, n - 1)
        val = (d - A[i]) / d if (dy, dx) == (0, 0) else -A[i] * rs * rs[col]
        out[i] = torch.where(valid[i], val, A[i])
    return _pad64(out), d.reshape(h, w), rs.reshape(h, w)


def _smallest64(A, w, h, wanted=N_EIG):
    """The smallest eigenpairs of the Laplacian by Chebyshev-filtered subspace
    iteration in 64 bits, until the residuals are 1e-11."""
    n, halo, block = w * h, 5 * w + 5, 40

    def mul(X):
        P = torch.nn.functional.pad(X, (halo, halo))
        Y = torch.zeros_like(X)
        for i, (dy, dx) in enumerate(DISC):
            at = halo + dy * w + dx
            Y.addcmul_(A[i][None], P[:, at:at + n])
        return Y
    gen = torch.Generator().manual_seed(1)
    X = torch.randn(block, n, generator=gen, dtype=F64).to(A.device)
    cut = 1e-2
    for _ in range(40):
        X = torch.linalg.qr(X.T.cpu())[0].T.contiguous().to(A.device)
        HX = mul(X)
        theta, S = torch.linalg.eigh((X @ HX.T).cpu())
        S = S.to(A.device)
        X, HX = S.T @ X, S.T @ HX
        if (HX - theta.to(A.device)[:, None] * X)[:wanted].norm(dim=1).max() < 1e-11:
            break
        cut = max(cut if theta[-1] > 1 else float(theta[-1]), 1e-6)
        e, c = (2 - cut) / 2, (2 + cut) / 2
        prev, cur = X, (mul(X) - c * X) / e
        for _ in range(80):
            prev, cur = cur, 2 / e * (mul(cur) - c * cur) - prev
            big = cur.norm(dim=1, keepdim=True).clamp(min=1e-300)
            prev, cur = prev / big, cur / big
        X = cur
    return theta[:wanted].to(A.device), X[:wanted]
