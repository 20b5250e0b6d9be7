"""Workloads of the framework for performance measurement.

Each case is one pass of work as a user's program has it done: reconstruction
of a map from particles at known views, central sections of a map, map
resolution, the stages of the orientation search, and the proposal network's
inference and training. Inputs are synthetic: Gaussian-blob maps, projections
at uniformly random orientations with a per-particle CTF and origin, white
noise.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs and handles, on the GPU
    run(state)           one pass; returns its outputs
    work(case)           bytes and operations the pass cannot do without
    exact(case, seed)    the outputs in 64 bits, in plain torch
"""
from __future__ import annotations

import math

import numpy as np
import torch

from bsoft_amd import abi, bresolve, proposal, recon, search
from bsoft_amd.synth import PARTICLE_DTYPE

PIX = 1.5                    # A / pixel
VOLT, CS = 300e3, 2.7e7      # V, A
AMP = math.asin(0.07)
DEV = "cuda"
MAP_SIZES = (32, 48, 64, 96, 128, 192, 256)
SEARCH_SIZES = (64, 128, 256)
NET = (32, 128, (32, 64, 128, 128))   # input edge, embedding values, channels
EXACT_SAMPLES = 4e9          # inserted samples that the 64-bit reconstruction takes on


# ------------------------------------------------------------------- cases
def _reconstruct(box, size, n, interp=0, ctf=1, wiener=0.0, halves=1, fom=False):
    return {"op": "reconstruct", "box": box, "size": size, "n": n, "interp": interp, "ctf": ctf,
            "wiener": wiener, "halves": halves, "fom": fom}


def _search(op, box, radius, n, step=4.0):
    return {"op": op, "box": box, "radius": radius, "n": n, "step": step}


def listed():
    named = [
        # a first look at a few dozen particles; every launch and wait counts
        ("reconstruct 32 few", _reconstruct(32, 32, 96)),
        # the usual run of a 128-pixel data set: full map, two half maps and
        # their figure-of-merit maps from one pass over the particles, with
        # Wiener CTF correction
        ("reconstruct 128 halves fom", _reconstruct(128, 128, 3001, ctf=3, wiener=0.2, halves=2,
                                                    fom=True)),
        # an odd number of particles of a box that is no power of two, trilinear
        # insertion, CTF applied
        ("reconstruct 90 trilinear", _reconstruct(90, 96, 1501, interp=2, ctf=2)),
        # the production size: phase-flipped particles into a 256^3 map
        ("reconstruct 256", _reconstruct(256, 256, 10000)),
        # projections of a map at given views, default interpolation kernel
        ("sections 128", {"op": "sections", "size": 128, "views": 200, "width": 8}),
        # FSC and phase residual between two half maps
        ("resolution 256", {"op": "resolution", "size": 256, "limit": 0.0}),
        # exhaustive projection matching of a particle set against a 4-degree
        # grid: staging, coarse scores of every view, exact scores of the best 8
        ("match views 128", _search("exhaustive", 128, 24, 5000)),
        # a single micrograph's particles against the grid of a small map
        ("match views 64 few", _search("exhaustive", 64, 16, 150, step=6.0)),
        # one step of the local refinement: 27 rotations around each particle's
        ("refine 256", _search("refine", 256, 24, 8000)),
        # the search restricted to 16 proposed classes per particle, then the
        # exact scores of the best 8
        ("match proposed 128", _search("proposed", 128, 24, 8000)),
        # proposals of the network for a particle set: embeddings, and their
        # nearest class projections
        ("propose", {"op": "propose", "n": 16384, "refs": 4368, "k": 16}),
        # one training step of the network on particle / projection pairs
        ("train pairs", {"op": "train", "pairs": 256}),
    ]
    return [{"name": name, **c} for name, c in named]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["reconstruct", "reconstruct", "reconstruct", "sections", "resolution",
                     "exhaustive", "refine", "proposed", "propose", "train"])
    if op == "reconstruct":
        size = rng.choice(MAP_SIZES)
        box = size if rng.random() < 0.5 else rng.randint(max(24, size * 3 // 4), size)
        interp = rng.choice([0, 0, 1, 2])
        fom = rng.random() < 0.4
        # at most the work of the largest listed case
        top = 10000 * (512 / _ft_size(max(box, size))) ** 2 / (8 if interp == 2 else 1) \
            / (2 if fom else 1)
        ctf, wiener = rng.choice([(0, 0.0), (1, 0.0), (2, 0.0), (3, 0.2)])
        return _reconstruct(box, size, _log(rng, 20, min(top, 20000)), interp, ctf, wiener,
                            rng.choice([1, 2]), fom)
    if op == "sections":
        size = rng.choice(MAP_SIZES)
        width = rng.choice([3, 4, 8])
        return {"op": op, "size": size, "width": width,
                "views": _log(rng, 4, min(2048, 400 * (128 / size) ** 2))}
    if op == "resolution":
        return {"op": op, "size": rng.choice(MAP_SIZES), "limit": round(rng.uniform(2.0, 10.0), 2)}
    if op == "propose":
        return {"op": op, "n": _log(rng, 64, 16384), "refs": _log(rng, 600, 4368),
                "k": rng.choice([8, 16])}
    if op == "train":
        return {"op": op, "pairs": rng.randint(32, 256)}
    box = rng.choice(SEARCH_SIZES)
    radius = rng.randint(10, 16 if box == 64 else 24)
    if op == "refine":
        return _search(op, box, radius, _log(rng, 50, 8000))
    return _search(op, box, radius, _log(rng, 50, 5000), rng.choice([4.0, 5.0, 6.0, 8.0]))


# ---------------------------------------------------------- synthetic data
def _ft_size(edge):
    f = 2
    while f < 2 * edge:
        f *= 2
    return f


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _blobs(size, seed, count=60):
    """Blob centres (voxels from the map origin), widths and heights."""
    r = np.random.default_rng([seed, 1])
    d = r.normal(size=(count, 3))
    d *= (0.35 * size * r.random(count) ** (1 / 3) / np.linalg.norm(d, axis=1))[:, None]
    return d, r.uniform(0.015, 0.035, count) * size + 0.5, r.uniform(0.5, 1.0, count)


def _volume(size, seed):
    """float32 map of the blobs, (z, y, x), origin at size // 2."""
    cen, sig, amp = (torch.as_tensor(v, device=DEV) for v in _blobs(size, seed))
    x = torch.arange(size, device=DEV, dtype=torch.float64) - size // 2
    e = [torch.exp(-(x[None] - cen[:, c:c + 1]) ** 2 / (2 * sig[:, None] ** 2)) for c in range(3)]
    zy = (amp[:, None, None] * e[2][:, :, None] * e[1][:, None, :]).reshape(len(amp), -1)
    return (zy.T.contiguous() @ e[0]).reshape(size, size, size).float()


def _quaternions(n, seed):
    u = np.random.default_rng([seed, 2]).random((3, n))
    a, b = np.sqrt(1 - u[0]), np.sqrt(u[0])
    return np.stack([b * np.cos(2 * np.pi * u[2]), a * np.sin(2 * np.pi * u[1]),
                     a * np.cos(2 * np.pi * u[1]), b * np.sin(2 * np.pi * u[2])], -1)


def _matrices(q):
    s, x, y, z = (q[..., i] for i in range(4))
    return np.stack([s * s + x * x - y * y - z * z, 2 * (x * y - s * z), 2 * (x * z + s * y),
                     2 * (x * y + s * z), s * s - x * x + y * y - z * z, 2 * (y * z - s * x),
                     2 * (x * z - s * y), 2 * (y * z + s * x), s * s - x * x - y * y + z * z],
                    -1).reshape(*q.shape[:-1], 3, 3)


def _view_of(m):
    """(x, y, z, angle) of rotations m = Rz(phi) Ry(theta) Rz(psi): the view
    vector is the third column, the angle phi + psi."""
    phi = np.arctan2(m[:, 1, 2], m[:, 0, 2])
    psi = np.arctan2(m[:, 2, 1], -m[:, 2, 0])
    return np.concatenate([m[:, :, 2], (phi + psi)[:, None]], axis=1)


def _optics(n, seed):
    """Defocus, astigmatism and its angle, origin shift (x, y) per particle."""
    r = np.random.default_rng([seed, 3])
    return (r.uniform(8e3, 3.5e4, n), r.uniform(0, 2e3, n), r.uniform(-np.pi, np.pi, n),
            r.uniform(-2, 2, (n, 2)))


def _lambda():
    h, e, m, c = 6.626070e-34, 1.602177e-19, 9.109384e-31, 299792458.0
    return h * 1e10 / math.sqrt(2 * m * e * VOLT * (1 + e * VOLT / (2 * m * c * c)))


def _chi(fx, fy, defocus, astig, angle):
    """CTF aberration at spatial frequencies (1/A); per-particle tensors."""
    wl = _lambda()
    s2 = fx * fx + fy * fy
    return (-AMP - math.pi * wl * (defocus * s2 + astig * (torch.cos(2 * angle) * (fx * fx - fy * fy)
                                                           + torch.sin(2 * angle) * 2 * fx * fy))
            + math.pi / 2 * wl ** 3 * CS * s2 * s2)


def _freq(n):
    f = torch.arange(n, device=DEV, dtype=torch.float64)
    return torch.where(f > (n - 1) // 2, f - n, f)


def _column(v):
    return torch.as_tensor(np.asarray(v, dtype=np.float64), device=DEV)[:, None, None]


def _particles(box, n, seed, mapsize=None, snr=0.1):
    """(float32 images, rotations (n, 3, 3), optics): CTF-modulated noisy
    projections of the seed's blob map."""
    cen, sig, amp = _blobs(mapsize or box, seed)
    mats = _matrices(_quaternions(n, seed))
    optics = _optics(n, seed)
    sig = torch.as_tensor(sig, device=DEV, dtype=torch.float32)
    height = torch.as_tensor(amp, device=DEV, dtype=torch.float32) * sig * math.sqrt(2 * math.pi)
    gen = _generator(seed)
    images = torch.empty((n, box, box), device=DEV, dtype=torch.float32)
    x = torch.arange(box, device=DEV, dtype=torch.float32) - box // 2
    f = _freq(box) / (box * PIX)
    for a in range(0, n, 1024):
        b = min(n, a + 1024)
        c = torch.as_tensor(np.einsum("pji,bj->pbi", mats[a:b], cen)[:, :, :2]
                            + optics[3][a:b, None], device=DEV, dtype=torch.float32)
        ex, ey = (torch.exp(-(x - c[:, :, i:i + 1]) ** 2 / (2 * sig[:, None] ** 2)) for i in (0, 1))
        img = torch.bmm((ey * height[:, None]).transpose(1, 2).contiguous(), ex.contiguous())
        ctf = torch.sin(_chi(f[None, None, :], f[None, :, None],
                             *(_column(o[a:b]) for o in optics[:3]))).float()
        img = torch.fft.ifft2(torch.fft.fft2(img) * ctf).real
        sd = img.flatten(1).std(dim=1) / math.sqrt(snr)
        noise = torch.randn(img.shape, generator=gen, device=DEV, dtype=torch.float32)
        images[a:b] = img + noise * sd[:, None, None] + 0.1
    return images, mats, optics


def _records(box, mats, optics):
    """The library's particle records."""
    p = np.zeros(len(mats), dtype=PARTICLE_DTYPE)
    p["view"] = _view_of(mats)
    p["ori"] = box // 2 + optics[3]
    p["hdr_ori"] = box // 2
    p["pixel_size"], p["mag"], p["volt"], p["cs"], p["amp_shift"] = PIX, 1.0, VOLT, CS, AMP
    p["def_avg"], p["def_dev"], p["ast_angle"] = optics[:3]
    p["sel"] = 1.0
    p["half"] = np.arange(len(p)) % 2
    return p


def _grid(step):
    """Rotations of a view grid: directions spread evenly over the sphere,
    about `step` degrees apart, times in-plane angles `step` degrees apart."""
    nd = int(round(4 * math.pi / math.radians(step) ** 2))
    na = int(round(360 / step))
    i = np.arange(nd) + 0.5
    theta, phi = np.arccos(1 - 2 * i / nd), np.pi * (1 + 5 ** 0.5) * i
    psi = np.arange(na) * (2 * np.pi / na)
    th, ph, ps = np.repeat(theta, na), np.repeat(phi, na), np.tile(psi, nd)
    h = th / 2
    return _matrices(np.stack([np.cos(h) * np.cos((ph + ps) / 2), np.sin(h) * np.sin((ps - ph) / 2),
                               np.sin(h) * np.cos((ps - ph) / 2), np.cos(h) * np.sin((ph + ps) / 2)],
                              -1))


def _nearest(mats, classes, k):
    """The k nearest class rotations of each rotation, nearest first."""
    c = torch.as_tensor(classes.reshape(-1, 9), device=DEV)
    out = []
    for a in range(0, len(mats), 16384):
        m = torch.as_tensor(mats[a:a + 16384].reshape(-1, 9), device=DEV)
        out.append((m @ c.T).topk(k, dim=1).indices.to(torch.int32))
    return torch.cat(out)


def _members(lib, classes):
    """(classes, most) table of the library views of each class, -1 padded."""
    own = _nearest(lib, classes, 1)[:, 0].cpu().numpy()
    order = np.argsort(own, kind="stable")
    count = np.bincount(own, minlength=len(classes))
    table = np.full((len(classes), count.max()), -1, dtype=np.int32)
    place = np.arange(len(own)) - np.repeat(np.concatenate([[0], np.cumsum(count)[:-1]]), count)
    table[own[order], place] = order
    return table


def _local(mats, seed):
    """27 rotations around each particle's, 2 degrees apart, from a start that
    is up to 2 degrees off."""
    def turn(w):
        th = np.maximum(np.linalg.norm(w, axis=-1, keepdims=True), 1e-30)
        return _matrices(np.concatenate([np.cos(th / 2), w / th * np.sin(th / 2)], -1))
    off = np.random.default_rng([seed, 4]).uniform(-1, 1, (len(mats), 3)) * math.radians(2)
    d = math.radians(2) * np.stack(np.meshgrid(*[[-1.0, 0.0, 1.0]] * 3, indexing="ij"),
                                   -1).reshape(27, 3)
    return np.ascontiguousarray(np.einsum("nij,cjk->ncik", mats @ turn(off), turn(d)))


def _weights(seed):
    """Flat parameters of the network: He-normal weights, small biases."""
    g = _generator(seed)
    edge, dim, ch = NET
    blocks = []
    for i, o in zip((1,) + ch[:3], ch):
        blocks += [((o, i, 3, 3), math.sqrt(2 / (9 * i))), ((o,), 0.05)]
    blocks += [((dim, ch[3] * (edge // 8) ** 2), math.sqrt(2 / (ch[3] * (edge // 8) ** 2))),
               ((dim,), 0.05)]
    return [torch.randn(s, generator=g, device=DEV) * sd for s, sd in blocks]


def _net_inputs(n, seed):
    """Pairs of network inputs: low-pass images and noisy versions of them,
    each with zero mean and unit variance."""
    g = _generator(seed + 1)
    edge = NET[0]
    f = _freq(edge).float()
    low = torch.exp(-(f[:, None] ** 2 + f[None] ** 2) / 50)
    a = torch.fft.ifft2(torch.fft.fft2(torch.randn((n, edge, edge), generator=g, device=DEV)) * low).real
    a = a / a.flatten(1).std(dim=1)[:, None, None]
    b = a + torch.randn(a.shape, generator=g, device=DEV)
    return tuple(((v - v.mean((1, 2), keepdim=True)) /
                  v.flatten(1).std(dim=1, correction=0)[:, None, None]).contiguous() for v in (b, a))


def _embeddings(n, refs, seed):
    """Unit rows: class projections' embeddings, and particles near them."""
    g = _generator(seed + 2)
    r = torch.randn((refs, NET[1]), generator=g, device=DEV)
    own = torch.randint(refs, (n,), generator=g, device=DEV)
    p = r[own] + 0.8 * torch.randn((n, NET[1]), generator=g, device=DEV)
    return p / p.norm(dim=1, keepdim=True), r / r.norm(dim=1, keepdim=True)


# ------------------------------------------------------- prepare, run, work
def prepare(case, seed):
    op = case["op"]
    state = {"case": case}
    if op == "reconstruct":
        box, size, n = case["box"], case["size"], case["n"]
        images, mats, optics = _particles(box, n, seed, size)
        ft = recon.part_ft_size(max(box, size), 1, 2)
        rec = recon.Reconstruction(size, box, ft, PIX, interp=case["interp"], ctf_action=case["ctf"],
                                   wiener=case["wiener"], nhalves=case["halves"],
                                   flags=abi.BSX_FLAG_FOM if case["fom"] else 0)
        state.update(rec=rec, images=images, parts=_records(box, mats, optics))
    elif op == "sections":
        state.update(map=_volume(case["size"], seed),
                     views=_view_of(_matrices(_quaternions(case["views"], seed))))
    elif op == "resolution":
        state.update(maps=_half_maps(case["size"], seed))
    elif op == "propose":
        net = proposal.EmbeddingNet(NET[0], NET[1], NET[2], max_batch=512)
        net.set_params(torch.cat([w.flatten() for w in _weights(seed)]))
        p, r = _embeddings(case["n"], case["refs"], seed)
        state.update(net=net, x=_net_inputs(case["n"], seed)[0], p=p, r=r)
    elif op == "train":
        net = proposal.EmbeddingNet(NET[0], NET[1], NET[2], max_batch=512)
        net.set_params(torch.cat([w.flatten() for w in _weights(seed)]))
        xp, xr = _net_inputs(case["pairs"], seed)
        state.update(net=net, xp=xp, xr=xr)
    else:
        box, n = case["box"], case["n"]
        images, mats, optics = _particles(box, n, seed)
        parts = _records(box, mats, optics)
        ft = recon.map_transform(_volume(box, seed))
        s = search.Search(box, case["radius"], PIX, kernel_width=3, topk=8)
        state.update(search=s, images=images, parts=parts, ft=ft)
        if op == "refine":
            s.stage(images, parts)
            state["mats"] = torch.as_tensor(_local(mats, seed), device=DEV)
            return state
        lib = _grid(case["step"])
        s.set_reference(ft, lib)
        if op == "proposed":
            classes = _grid(15.0)
            s.set_classes(_members(lib, classes))
            s.stage(images, parts)
            state["classes"] = _nearest(mats, classes, 16)
    return state


def _half_maps(size, seed):
    """Two noisy copies of the blob map, the noise growing with frequency."""
    v = _volume(size, seed)
    g = _generator(seed)
    sd = 3.0 * float(v.std())
    return [v + sd * torch.randn(v.shape, generator=g, device=DEV) for _ in range(2)]


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "reconstruct":
        rec = state["rec"]
        rec.reset()
        rec.insert(state["images"], state["parts"])
        nmaps = 3 if case["halves"] == 2 else 1
        out = []
        for i in range(nmaps):
            r = rec.finish(i, nmaps, want_fom=case["fom"])
            out.append({"map": r.map, "fom": r.fom, "coverage": r.coverage,
                        "particles": r.particles})
        return out
    if op == "sections":
        ft = recon.map_transform(state["map"])
        return {"ft": ft, "sections": recon.project(ft, state["views"], PIX, 2 * PIX, case["width"])}
    if op == "resolution":
        s, fsc, dpr = bresolve.fsc_dpr(*state["maps"], PIX, case["limit"])
        return {"s": s, "fsc": fsc, "dpr": dpr}
    if op == "propose":
        net = state["net"]
        emb = net.embed(state["x"])
        cls, prob = net.match_topk(state["p"], state["r"], case["k"], 0.1)
        return {"embeddings": emb, "classes": cls, "probabilities": prob}
    if op == "train":
        grad, loss = state["net"].pair_gradients(state["xp"], state["xr"], 0.1)
        return {"gradient": grad, "loss": loss}
    s = state["search"]
    if op == "refine":
        return {"frc": s.score_mats(state["mats"], state["ft"])}
    if op == "exhaustive":
        s.stage(state["images"], state["parts"])
        cand, score = s.exhaustive()
    else:
        cand, score = s.proposed(state["classes"])
    frc, best, best_frc = s.rescore(cand)
    return {"candidates": cand, "scores": score, "frc": frc, "best": best, "best_frc": best_frc}


def _disk_points(radius):
    h, k = np.meshgrid(np.arange(-radius, radius + 1), np.arange(0, radius + 1))
    ring = np.floor(np.sqrt(h * h + k * k)).astype(int)
    keep = (ring < radius) & ((k > 0) | (h >= 0))
    return h[keep], k[keep], ring[keep]


def _grid_views(step):
    return int(round(4 * math.pi / math.radians(step) ** 2)) * int(round(360 / step))


def work(case):
    op = case["op"]
    if op == "reconstruct":
        # images in, maps (and FOM maps) out; row and column transforms of the
        # half plane, 3D inverse transforms; about 30 operations per inserted sample
        n, N, ft = case["n"], case["size"], _ft_size(max(case["box"], case["size"]))
        maps = 3 if case["halves"] == 2 else 1
        flops = n * (5 * ft * ft * math.log2(ft) + 30 * ft * ft / 2 * (8 if case["interp"] == 2 else 1)) \
            + maps * 15 * N ** 3 * math.log2(N)
        return {"bytes": 4 * n * case["box"] ** 2 + 4 * maps * (2 if case["fom"] else 1) * N ** 3,
                "flops": flops}
    if op == "sections":
        N, nv = case["size"], case["views"]
        return {"bytes": 12 * N ** 3 + 8 * nv * N * N,
                "flops": 15 * N ** 3 * math.log2(N)
                + nv * math.pi / 4 * N * N * 4 * case["width"] ** 3}
    if op == "resolution":
        N = case["size"]
        return {"bytes": 8 * N ** 3, "flops": 2 * 7.5 * N ** 3 * math.log2(N) + 10 * N ** 3}
    conv = sum(2 * 9 * i * o * (NET[0] >> l) ** 2
               for l, (i, o) in enumerate(zip((1,) + NET[2][:3], NET[2])))
    fc = 2 * NET[2][3] * (NET[0] // 8) ** 2 * NET[1]
    params = sum(9 * i * o + o for i, o in zip((1,) + NET[2][:3], NET[2])) + fc // 2 + NET[1]
    if op == "propose":
        n, m, d = case["n"], case["refs"], NET[1]
        return {"bytes": 4 * (n * NET[0] ** 2 + 2 * n * d + m * d + params) + 8 * n * case["k"],
                "flops": n * (conv + fc) + 2 * n * m * d}
    if op == "train":
        b = 2 * case["pairs"]
        return {"bytes": 4 * (b * NET[0] ** 2 + 2 * params), "flops": 3 * b * (conv + fc)}
    nd, n, box = len(_disk_points(case["radius"])[0]), case["n"], case["box"]
    if op == "refine":
        return {"bytes": n * (12 * nd + 27 * (72 + 4)), "flops": n * 27 * nd * (4 * 27 + 8)}
    views = _grid_views(case["step"])
    rescore = n * 8 * nd * 12
    if op == "exhaustive":
        return {"bytes": 4 * n * box * box + 4 * nd * views + 8 * nd * 8 * n + n * 8 * 12,
                "flops": 2.0 * n * views * 2 * (nd - 1) + rescore + n * 5 * box * box * math.log2(box)}
    per_class = views / _grid_views(15.0)
    return {"bytes": n * 2 * 2 * nd + 4 * nd * views + 8 * nd * 8 * n + n * (16 * 4 + 8 * 12),
            "flops": 2.0 * n * 16 * per_class * 2 * (nd - 1) + rescore}


# ------------------------------------------------------------ 64-bit answers
def _exact_reconstruct(case, seed):
    box, N, n = case["box"], case["size"], case["n"]
    ft = _ft_size(max(box, N))
    corners = 8 if case["interp"] == 2 else 1
    if n * ft * ft * corners > EXACT_SAMPLES:
        return None
    images, mats, optics = _particles(box, n, seed, N)
    hi = max(PIX, 2 / math.sqrt(3 / PIX ** 2))
    f = _freq(ft)
    h, k = f[None, :].expand(ft, ft), f[:, None].expand(ft, ft)
    s0, s1 = h / (ft * PIX), k / (ft * PIX)
    s2 = s0 * s0 + s1 * s1
    band = (s2 <= 1 / hi ** 2).flatten()
    d = (1 / hi ** 2 - s2) * (N * PIX)
    ratio = ft / box
    weight = (1 / (0.6 * ratio * ratio) if ratio > 1 else 1.0) * torch.where(d < 1, d.clamp(min=0).sqrt(), 1.0)
    weight = weight.flatten()[band]
    x = (torch.arange(box, device=DEV, dtype=torch.float64) - box // 2) / (box // 2)
    outside = x[None] ** 2 + x[:, None] ** 2 - 1 > 0
    cols = 5 if case["fom"] else 3
    acc = torch.zeros((case["halves"], N ** 3, cols), device=DEV, dtype=torch.float64)
    chunk = max(1, int(2 ** 24 // (ft * ft)))
    halves = [np.arange(n)] if case["halves"] == 1 else [np.arange(0, n, 2), np.arange(1, n, 2)]
    for half, members in enumerate(halves):
        for a in range(0, len(members), chunk):
            p = members[a:a + chunk]
            img = images[torch.as_tensor(p, device=DEV)].double()
            bkg = img[:, outside].mean(dim=1)
            full = bkg[:, None, None].expand(-1, ft, ft).clone()
            full[:, :box, :box] = img
            F = torch.fft.fft2(full) / ft
            ori = box // 2 + optics[3][p]
            F = F * torch.polar(torch.ones((), device=DEV, dtype=torch.float64),
                                2 * math.pi / ft * (h * _column(ori[:, 0]) + k * _column(ori[:, 1])))
            if case["ctf"]:
                c = torch.sin(_chi(s0, s1, *(_column(o[p]) for o in optics[:3])))
                if case["ctf"] == 1:
                    c = torch.where(c < 0, -1.0, 1.0)
                elif case["wiener"] > 0:
                    c = (case["wiener"] + 1) * c / (c * c + case["wiener"])
                F = F * (c * (s2 <= 1 / hi ** 2))
            F = F.flatten(1)[:, band]
            R = torch.as_tensor(mats[p], device=DEV)
            s = torch.stack([s0.flatten()[band], s1.flatten()[band]])
            m = [(R[:, c, 0:1] * s[0] + R[:, c, 1:2] * s[1]) * (N * PIX) for c in range(3)]
            base = [torch.floor(v if corners == 8 else v + 0.5) for v in m]
            for q in range(corners):
                w = weight.expand(len(p), -1)
                idx = torch.zeros(F.shape, device=DEV, dtype=torch.int64)
                dist = 0.0
                for c in (2, 1, 0):
                    up = (q >> c) & 1
                    frac = m[c] - base[c]
                    if corners == 8:
                        w = w * (frac if up else 1 - frac)
                    dist = dist + frac * frac
                    idx = idx * N + torch.remainder(base[c].long() + up, N)
                if case["interp"] == 1:
                    w = (w * (1 - dist.sqrt())).clamp(min=0)
                vals = [w * F.real, w * F.imag, w]
                if case["fom"]:
                    vals += [w * (F.real ** 2 + F.imag ** 2), w * w]
                for j, v in enumerate(vals):
                    acc[half, :, j].index_add_(0, idx.flatten(), v.reshape(-1))
    sign = 1.0 - 2.0 * (torch.arange(N, device=DEV, dtype=torch.float64) % 2)
    sign = sign[:, None, None] * sign[None, :, None] * sign[None, None, :]
    out = []
    for i in range(3 if case["halves"] == 2 else 1):
        a = acc.sum(0) if i == 0 else acc[i - 1]
        W = a[:, 2]
        has = W > 1e-30
        Ws = torch.where(has, W, 1.0)
        F = torch.where(has, torch.complex(a[:, 0], a[:, 1]) / Ws, 0.0)
        fom = None
        if case["fom"]:
            var = Ws - a[:, 4] / Ws
            P = torch.where(var > 1, a[:, 3] / torch.where(var > 1, var, 1.0),
                            torch.where(W > 1, a[:, 3] / Ws, a[:, 3])) * has
            P[0] = 1
            sig = F.real ** 2 + F.imag ** 2
            noise = torch.maximum(P - sig, sig)
            ok = (W > 1) & (sig > 1e-30) & (noise > 1e-30)
            fom = torch.where(ok, (W * sig - P) / torch.where(ok, noise, 1.0), 0.0)
            fom[0] = 1
            fom = fom.reshape(N, N, N)
        vol = torch.fft.ifftn(F.reshape(N, N, N) * sign, norm="forward").real / N ** 1.5
        out.append({"map": vol, "fom": fom, "coverage": None, "particles": None})
    return out


def _section_values(ft, mats, hk, width):
    """Values of central sections at disk points hk (2, P) for rotations
    (V, 3, 3): kernel interpolation of a complex128 transform, (V, P). The
    kernel is tabulated at 512 fractions per voxel."""
    N = ft.shape[0]
    row = np.arange(513) / 512
    dist = row[:, None] + (width - 1) // 2 - np.arange(width)[None]
    whole = np.abs(dist - np.rint(dist)) < 1e-12
    d = np.where(whole, 0.5, dist)
    tab = np.sin(np.pi * d) / (width * np.sin(np.pi * d / width)) * np.cos(np.pi * d / width) ** 2
    tab = torch.as_tensor(np.where(whole, (np.rint(dist) == 0) * 1.0, tab), device=DEV)
    flat = ft.reshape(-1)
    m = torch.matmul(mats[..., :2].contiguous(), hk)                # (V, 3, P)
    base = torch.floor(m)
    w = [tab[((m[:, c] - base[:, c]) * 512 + 0.5).long()] for c in range(3)]     # (V, P, width)
    i = [torch.remainder(base[:, c].long()[..., None] - (width - 1) // 2
                         + torch.arange(width, device=DEV), N) for c in range(3)]
    out = torch.zeros(m[:, 0].shape, device=DEV, dtype=torch.complex128)
    for z in range(width):
        for y in range(width):
            at = (i[2][..., z] * N + i[1][..., y]) * N
            v = (flat[at[..., None] + i[0]] * w[0]).sum(-1)
            out += v * (w[2][..., z] * w[1][..., y])
    return out


def _exact_transform(vol):
    """Transform of a map moved to its origin, x 1 / sqrt(N^3)."""
    N = vol.shape[0]
    sign = 1.0 - 2.0 * (torch.arange(N, device=DEV, dtype=torch.float64) % 2)
    sign = sign[:, None, None] * sign[None, :, None] * sign[None, None, :]
    return torch.fft.fftn(vol.double(), norm="ortho") * sign


def _exact_sections(case, seed):
    N, nv = case["size"], case["views"]
    if nv * N * N * case["width"] ** 3 > 2e10:
        return None
    ft = _exact_transform(_volume(N, seed))
    mats = torch.as_tensor(_matrices(_quaternions(nv, seed)), device=DEV)
    f = _freq(N)
    h, k = f[None].expand(N, N).flatten(), f[:, None].expand(N, N).flatten()
    inv = 1 / (N * PIX)
    band = (h * inv) ** 2 + (k * inv) ** 2 <= 1 / (2 * PIX) ** 2
    hk = torch.stack([h[band], k[band]])
    out = torch.zeros((nv, N * N), device=DEV, dtype=torch.complex128)
    chunk = max(1, 2 ** 22 // hk.shape[1])
    for a in range(0, nv, chunk):
        out[a:a + chunk, band] = _section_values(ft, mats[a:a + chunk], hk, case["width"])
    return {"ft": ft, "sections": (out * (1 - 2 * ((h + k) % 2).abs())).reshape(nv, N, N)}


def _exact_resolution(case, seed):
    N = case["size"]
    hi = max(case["limit"], 2 / math.sqrt(3 / PIX ** 2))
    rows = int(2 + N * PIX / hi)
    a, b = (torch.fft.fftn(v.double())[:, :, :N // 2] for v in _half_maps(N, seed))
    f = _freq(N)
    r = torch.sqrt(f[:, None, None] ** 2 + f[None, :, None] ** 2 + f[None, None, :N // 2] ** 2)
    lo = r.long()
    keep = lo + 1 < rows
    i1, i2 = a.abs() ** 2, b.abs() ** 2
    dphi = torch.remainder(a.angle() - b.angle() + math.pi, 2 * math.pi) - math.pi
    sums = []
    for v in (i1, i2, (a * b.conj()).real, i1 + i2, (i1 + i2) * dphi ** 2):
        s = torch.zeros(rows, device=DEV, dtype=torch.float64)
        s.index_add_(0, lo[keep], (v * (1 - (r - lo)))[keep])
        s.index_add_(0, lo[keep] + 1, (v * (r - lo))[keep])
        sums.append(s)
    p = sums[0] * sums[1]
    fsc = torch.where(p > 1e-30, sums[2] / torch.where(p > 1e-30, p, 1.0).sqrt(), sums[2]).clamp(-1, 1)
    dpr = torch.where(sums[3] > 1e-30, (sums[4] / sums[3].clamp(min=1e-30)).sqrt() * 180 / math.pi, 0.0)
    fsc[0], dpr[0] = 1, 0
    return {"s": torch.arange(rows, dtype=torch.float64) / (N * PIX), "fsc": fsc, "dpr": dpr}


def _exact_staged(case, seed):
    """Disk points (2, P), ring of each, particle values and CTF values (n, P)."""
    box, n = case["box"], case["n"]
    images, mats, optics = _particles(box, n, seed)
    h, k, ring = _disk_points(case["radius"])
    hk = torch.as_tensor(np.stack([h, k]).astype(np.float64), device=DEV)
    at = torch.as_tensor(k * box + h % box, device=DEV)
    F = torch.cat([(torch.fft.fft2(images[a:a + 512].double()) / box).flatten(1)[:, at]
                   for a in range(0, n, 512)])
    ori = torch.as_tensor(box // 2 + optics[3], device=DEV)
    F = F * torch.polar(torch.ones((), device=DEV, dtype=torch.float64), 2 * math.pi / box * (ori @ hk))
    one = [torch.as_tensor(o, device=DEV)[:, None] for o in optics[:3]]
    ctf = torch.sin(_chi(hk[0] / (box * PIX), hk[1] / (box * PIX), *one))
    return hk, torch.as_tensor(ring, device=DEV), F, ctf, mats


def _ring_sums(v, ring, radius):
    s = torch.zeros((*v.shape[:-1], radius), device=DEV, dtype=torch.float64)
    return s.index_add_(-1, ring, v)


def _exact_refine(case, seed):
    hk, ring, F, ctf, mats = _exact_staged(case, seed)
    ft = _exact_transform(_volume(case["box"], seed))
    local = torch.as_tensor(_local(mats, seed), device=DEV)
    R = case["radius"]
    out = []
    for a in range(0, case["n"], 128):
        sec = _section_values(ft, local[a:a + 128].reshape(-1, 3, 3), hk, 3)
        sec = sec.reshape(-1, 27, hk.shape[1]) * ctf[a:a + 128, None]
        p = F[a:a + 128, None]
        num = _ring_sums((p.conj() * sec).real.contiguous(), ring, R)
        den = _ring_sums(p.abs() ** 2, ring, R) * _ring_sums(sec.abs() ** 2, ring, R)
        out.append(torch.where(den > 0, num / torch.where(den > 0, den, 1.0).sqrt(), 0.0).sum(-1) / R)
    return {"frc": torch.cat(out)}


def _unit_rings(v, ring, radius):
    """Values normalised per ring without the centre, as real rows."""
    power = _ring_sums(v.abs() ** 2, ring, radius)
    inv = torch.where(power > 0, 1 / torch.where(power > 0, power, 1.0).sqrt(), 0.0)
    inv[:, 0] = 0
    return torch.view_as_real(v * inv[:, ring]).flatten(1)


def _exact_scores(case, seed):
    """Coarse scores of the best views, best first; the indices and exact
    scores that go with them have no 64-bit value of their own (the coarse
    scores come from 16-bit rows)."""
    hk, ring, F, ctf, mats = _exact_staged(case, seed)
    R = case["radius"]
    ft = _exact_transform(_volume(case["box"], seed))
    lib = _grid(case["step"])
    rows = []
    for a in range(0, len(lib), 4096):
        m = torch.as_tensor(lib[a:a + 4096], device=DEV)
        rows.append(_unit_rings(_section_values(ft, m, hk, 3), ring, R))
    rows = torch.cat(rows)
    part = _unit_rings(F * ctf, ring, R) / (R - 1)
    classes, own = _grid(15.0), None
    if case["op"] == "proposed":
        own = _nearest(lib, classes, 1)[:, 0].long()
        cls = _nearest(mats, classes, 16).long()
    out = []
    for a in range(0, case["n"], 256):
        s = part[a:a + 256] @ rows.T
        if own is not None:
            asked = torch.zeros((len(s), len(classes)), device=DEV, dtype=torch.bool)
            asked.scatter_(1, cls[a:a + 256], True)
            s = torch.where(asked[:, own], s, -math.inf)
        out.append(s.topk(8, dim=1).values)
    return {"candidates": None, "scores": torch.cat(out), "frc": None, "best": None, "best_frc": None}


def _exact_net(weights, x):
    """Unit embeddings of inputs (n, edge, edge) on the CPU in float64."""
    x = x[:, None]
    for l in range(4):
        x = torch.relu(torch.nn.functional.conv2d(x, weights[2 * l], weights[2 * l + 1],
                                                  stride=1 if l == 0 else 2, padding=1))
    z = x.flatten(1) @ weights[8].T + weights[9]
    return z / z.norm(dim=1, keepdim=True).clamp(min=1e-12)


def _exact_propose(case, seed):
    weights = [w.double().cpu() for w in _weights(seed)]
    x = _net_inputs(case["n"], seed)[0].double().cpu()
    emb = torch.cat([_exact_net(weights, x[a:a + 512]) for a in range(0, len(x), 512)])
    p, r = (v.double() for v in _embeddings(case["n"], case["refs"], seed))
    prob = torch.cat([torch.softmax(p[a:a + 1024] @ r.T / 0.1, dim=1).topk(case["k"], dim=1).values
                      for a in range(0, len(p), 1024)])
    return {"embeddings": emb, "classes": None, "probabilities": prob}


def _exact_train(case, seed):
    weights = [w.double().cpu().requires_grad_() for w in _weights(seed)]
    xp, xr = (v.double().cpu() for v in _net_inputs(case["pairs"], seed))
    s = _exact_net(weights, xp) @ _exact_net(weights, xr).T / 0.1
    own = torch.arange(len(s))
    loss = 0.5 * (torch.nn.functional.cross_entropy(s, own, reduction="none")
                  + torch.nn.functional.cross_entropy(s.T, own, reduction="none"))
    loss.mean().backward()
    return {"gradient": torch.cat([w.grad.flatten() for w in weights]), "loss": loss.detach()}


def exact(case, seed):
    return {"reconstruct": _exact_reconstruct, "sections": _exact_sections,
            "resolution": _exact_resolution, "refine": _exact_refine, "exhaustive": _exact_scores,
            "proposed": _exact_scores, "propose": _exact_propose,
            "train": _exact_train}[case["op"]](case, seed)
