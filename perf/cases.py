"""The work this framework is used for, as cases that can be timed.

A case is a dict of plain values; ``prepare`` makes what a user's program holds
before the call (data on the GPU, the bound design, the surface set), ``run`` is
one pass through the public entry points, ``work`` the bytes and operations
that pass cannot do without, ``exact`` its result in 64 bits from plain numpy
or torch.  Kinds:

null      one batch of the permutation loop: the permuted t-values of every
          contrast (``ols.PermutedOLS.t``), TFCE of +t and -t on every surface and
          the maxima (``tfce.SurfaceSet.batch``), as ``randomise.vertex_regress`` /
          ``voxel_regress`` / ``mmr`` and ``engine.PermutationEngine`` run it
mediation one batch of the mediation loop: the Sobel-type z of both paths
          (``randomise.MediationModel.z``), TFCE of +z
maps      the permuted t-values alone (``PermutedOLS.t``), covariates that stay
          fixed and several contrasts among the options
image     the observed statistic's TFCE image (``tfce.CreateAdjSet.run``), elements
          in the caller's order
tval      the observed statistic itself in FP64 (``cynumstats.tval_int``)

Surfaces are icospheres (2,562 to 163,842 vertices, optionally with a cap cut
out as the medial wall is), ellipsoid voxel masks in their grid (6- or
26-connected), or a set of both.  Data are noise smoothed over the surface
(``smooth`` passes; 0 is white noise) with an effect in one patch.
"""
import functools
import math

import numpy as np
import torch

from tfce_mediation_amd import cynumstats, synth
from tfce_mediation_amd.adjacency import induced_subgraph, locality_layout, vertex_density, voxel_csr
from tfce_mediation_amd.ols import PermutedOLS
from tfce_mediation_amd.randomise import MediationModel
from tfce_mediation_amd.tfce import (TFCE_ADJ_IMPLICIT_ZERO, TFCE_ADJ_ZERO_IN_SCALE, Adjacency, CreateAdjSet,
                                     SurfaceSet)


def listed():
    return [
        # a pilot run on a coarse mesh: the smallest batch, launches and latency
        dict(name="null_mesh_2k", kind="null", surfaces="mesh:4", E=1.0, smooth=2, n=40, k=3, fixed=0, con=1, P=64,
             precision="fp16x3", weighted=False),
        # vertex GLM on a 10,242-vertex mesh, +/-t, the drivers' batch
        dict(name="null_mesh_10k", kind="null", surfaces="mesh:5", E=1.0, smooth=5, n=100, k=4, fixed=0, con=1,
             P=512, precision="fp16x3", weighted=False),
        # the headline workload: both hemispheres, 327,684 vertices
        dict(name="null_2hemi_327k", kind="null", surfaces="mesh:7+mesh:7", E=1.0, smooth=5, n=500, k=6, fixed=0,
             con=1, P=256, precision="fp16x3", weighted=False),
        # voxel GLM, 232k voxels, 26-connected, E = 0.5
        dict(name="null_voxel_232k", kind="null", surfaces="vox26:36,44,35", E=0.5, smooth=2, n=200, k=5, fixed=0,
             con=1, P=512, precision="fp16x3", weighted=False),
        # a small ragged 6-connected mask, plain FP32 contraction, two contrasts, a batch that is no round number
        dict(name="null_voxel6_fp32", kind="null", surfaces="vox6:17,22,16", E=0.5, smooth=2, n=75, k=4, fixed=0,
             con=2, P=150, precision="fp32", weighted=False),
        # vertex density weights and the medial wall cut out: the weighted maximum over elements
        dict(name="null_weighted", kind="null", surfaces="mesh:6:0.07+mesh:6:0.07", E=1.0, smooth=4, n=120, k=4,
             fixed=0, con=1, P=128, precision="fp16x3", weighted=True),
        # the multimodal set: meshes and masks of uneven sizes, white noise, one maximum per surface
        dict(name="null_multimodal", kind="null",
             surfaces="mesh:7+mesh:7+mesh:6+mesh:5+mesh:5+mesh:4+vox26:33,40,32+vox26:19,23,18", E=0.5, smooth=0,
             n=120, k=4, fixed=0, con=1, P=256, precision="fp16x3", weighted=False),
        # mediation over both hemispheres
        dict(name="mediation_327k", kind="mediation", surfaces="mesh:7+mesh:7", E=1.0, smooth=5, n=300, k=3, fixed=0,
             con=1, P=512, precision="fp16x3", weighted=False),
        # permuted t-maps kept whole: two of seven columns permuted, the others covariates that stay fixed
        dict(name="maps_fixed_cov", kind="maps", surfaces="mesh:7", E=1.0, smooth=2, n=250, k=7, fixed=4, con=2,
             P=128, precision="fp16x3", weighted=False),
        # the observed TFCE image of a small surface and of a hemisphere
        dict(name="image_10k", kind="image", surfaces="mesh:5", E=1.0, smooth=5),
        dict(name="image_hemi", kind="image", surfaces="mesh:7", E=1.0, smooth=5),
        # the observed t-values of both hemispheres in FP64
        dict(name="tval_327k", kind="tval", surfaces="mesh:7+mesh:7", smooth=0, n=500, k=6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_surface(rng, most=240000):
    if rng.random() < 0.55:
        order = rng.choice([3, 4, 5, 6, 7])
        return "mesh:%d" % order if rng.random() < 0.5 else "mesh:%d:%.3f" % (order, rng.uniform(0.02, 0.3))
    a = rng.uniform(6, 35)
    s = [a, a * rng.uniform(0.8, 1.25), a * rng.uniform(0.8, 1.2)]
    while 4.19 * s[0] * s[1] * s[2] > most:
        s = [v * 0.9 for v in s]
    return "vox%d:%s" % (rng.choice([26, 26, 6]), ",".join("%.1f" % v for v in s))


def draw(rng):
    kind = rng.choice(["null", "null", "null", "mediation", "maps", "image", "tval"])
    surfs = [_draw_surface(rng)]
    if kind in ("null", "mediation") and rng.random() < 0.5:
        surfs = surfs * 2 if rng.random() < 0.5 else surfs + [_draw_surface(rng) for _ in range(rng.randint(1, 3))]
    case = dict(kind=kind, surfaces="+".join(surfs), smooth=rng.randint(0, 6))
    V = _about(case["surfaces"])
    if kind != "tval":
        case["E"] = rng.choice([1.0, 1.0, 0.5, 0.67])
    if kind == "image":
        return case
    n = min(_log(rng, 20, 500), 160_000_000 // V)
    k = rng.randint(2, 7)
    case.update(n=n, k=k)
    if kind == "tval":
        return case
    m_max = k - 1
    fixed = rng.randint(0, m_max - 1) if kind == "maps" and m_max > 1 and rng.random() < 0.5 else 0
    con = rng.randint(1, min(2, m_max - fixed))
    signs = 1 if kind == "mediation" else 2
    P = max(8, min(_log(rng, 16, 1024), 160_000_000 // (V * signs * con), 1_200_000_000_000 // (n * V * k)))
    case.update(fixed=fixed, con=con if kind != "mediation" else 1, P=P,
                precision=rng.choice(["fp16x3", "fp16x3", "fp16x3", "fp32"]),
                weighted=kind == "null" and rng.random() < 0.2 and V * P < 20_000_000)
    if kind == "mediation":
        case["k"] = 3
    return case


def _about(spec):
    """Elements of a surface list, near enough to bound a drawn case's work."""
    n = 0
    for s in spec.split("+"):
        f = s.split(":")
        if f[0] == "mesh":
            n += 10 * 4 ** int(f[1]) + 2
        else:
            a, b, c = (float(v) for v in f[1].split(","))
            n += int(4.19 * a * b * c) + 8
    return n


# --- surfaces: geometry does not depend on the seed; a program builds it once per study -----------------------

@functools.lru_cache(maxsize=16)
def _csr(s):
    f = s.split(":")
    if f[0] == "mesh":
        v, faces = synth.icosphere(int(f[1]))
        csr = synth.faces_to_csr(faces, len(v))
        return induced_subgraph(csr[0], csr[1], v[:, 2] <= 1.0 - 2.0 * float(f[2])) if len(f) > 2 else csr
    semi = [float(v) for v in f[1].split(",")]
    shape = tuple(int(2 * v + 5) for v in semi)
    mask = synth.ellipsoid_mask(shape, tuple((d - 1) / 2.0 for d in shape), semi)
    return voxel_csr(mask, int(f[0][3:]))


def _is_cut(s):
    return s.startswith("mesh") and s.count(":") == 2


@functools.lru_cache(maxsize=4)
def _surfaces(spec, E):
    """(SurfaceSet, CSRs in its element layout, offsets) of a surface list, in the layout the drivers use."""
    names = spec.split("+")
    csrs = [_csr(s) for s in names]
    offsets = [int(v) for v in np.concatenate([[0], np.cumsum([len(c[0]) - 1 for c in csrs])])]
    laid, _ = locality_layout(csrs, offsets[:-1], offsets[-1])
    adjs = [Adjacency(c, 2.0, 1.0 if s.startswith("mesh") and len(names) > 2 else E,
                      TFCE_ADJ_IMPLICIT_ZERO | TFCE_ADJ_ZERO_IN_SCALE if _is_cut(s) else 0)
            for s, c in zip(names, laid)]
    return SurfaceSet(adjs, offsets[:-1]), laid, offsets


@functools.lru_cache(maxsize=4)
def _adjset(spec, E):
    return CreateAdjSet(2.0, E, _csr(spec))


def _table(csr):
    """[V, degree] neighbour table on the GPU, V where there is none."""
    rp, col = csr
    V = len(rp) - 1
    deg = np.diff(rp.astype(np.int64))
    tab = np.full((V, max(1, int(deg.max()))), V, dtype=np.int64)
    src = np.repeat(np.arange(V), deg)
    tab[src, np.arange(len(col)) - rp.astype(np.int64)[src]] = col
    return torch.from_numpy(tab).cuda(), torch.from_numpy(deg + 1.0).float().cuda()


def _noise(csr, n, smooth, gen, effect, size):
    """[n, V] standardised noise smoothed ``smooth`` times over the surface, plus ``effect`` [n] in a patch."""
    tab, w = _table(csr)
    V = tab.shape[0]
    z = torch.zeros((V + 1, n), device="cuda")
    z[:V] = torch.randn((V, n), generator=gen, device="cuda")
    for _ in range(smooth):
        acc = z[:V].clone()
        for j in range(tab.shape[1]):
            acc += z.index_select(0, tab[:, j])
        z[:V] = acc / w[:, None]
    y = z[:V].t().contiguous()
    if n > 1:
        y -= y.mean(0, keepdim=True)
        y /= y.std(0, keepdim=True).clamp_min(1e-12)
    else:
        y /= y.std().clamp_min(1e-12)
    patch = torch.zeros(V + 1, dtype=torch.bool, device="cuda")
    patch[int(torch.randint(V, (1,), generator=gen, device="cuda"))] = True
    while int(patch.sum()) < min(size, V // 4):
        more = patch.clone()
        more[:V] |= patch[tab].any(1)
        more[V] = False
        if bool((more == patch).all()):
            break
        patch = more
    y[:, patch[:V]] += effect[:, None]
    return y


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    if case["kind"] == "image":
        csr = _csr(case["surfaces"])
        image = _noise(csr, 1, case["smooth"], gen, torch.full((1,), 2.0, device="cuda"), 600)[0].contiguous()
        return dict(kind="image", adjset=_adjset(case["surfaces"], case["E"]), image=image,
                    enhn=torch.empty_like(image))
    n, k = case["n"], case["k"]
    X = synth.design(rng, n, k - 2, binary=True)
    if case["kind"] == "tval":
        csrs = [_csr(s) for s in case["surfaces"].split("+")]
    else:
        surfs, csrs, _ = _surfaces(case["surfaces"], case["E"])
    x = rng.standard_normal(n)
    g = torch.tensor(x if case["kind"] == "mediation" else X[:, -1], dtype=torch.float32, device="cuda")
    size = int(rng.integers(100, 2001))
    Y = torch.cat([_noise(c, n, case["smooth"], gen, (0.5 if i == 0 else 0.0) * g, size)
                   for i, c in enumerate(csrs)], 1).contiguous()
    if case["kind"] == "tval":
        return dict(kind="tval", X=X, inv=np.linalg.inv(X.T @ X), Y=Y, n=n, k=k)
    perms = synth.permutations(n, case["P"], seed + 1, "cuda").contiguous()
    state = dict(kind=case["kind"], surfs=surfs, perms=perms, many=len(csrs) > 2, weights=None)
    if case["kind"] == "mediation":
        y = 0.5 * x + rng.standard_normal(n)
        state["model"] = MediationModel(Y, x, y, "M", precision=case["precision"])
        return state
    # the last columns are permuted and tested, ``fixed`` covariates after the intercept stay in place
    moved = list(range(1 + case["fixed"], k)) if case["fixed"] else None
    state["model"] = PermutedOLS(Y, X, contrasts=list(range(k - case["con"], k)), perm_columns=moved,
                                 precision=case["precision"])
    if case["weighted"]:
        state["weights"] = torch.from_numpy(np.concatenate([vertex_density(c[0]) for c in csrs])).cuda()
    return state


def run(state):
    kind = state["kind"]
    if kind == "image":
        state["enhn"].zero_()
        state["adjset"].run(state["image"], state["enhn"])
        return state["enhn"]
    if kind == "tval":
        return cynumstats.tval_int(state["X"], state["inv"], state["Y"], state["n"], state["k"], state["Y"].shape[1])
    if kind == "mediation":
        return state["surfs"].batch(state["model"].z(state["perms"]), 1).max(0).values[:, 0]
    t = state["model"].t(state["perms"])
    if kind == "maps":
        return t
    out = []
    for c in range(t.shape[0]):
        per = state["surfs"].batch(t[c], 3, vdensity=state["weights"])
        out.append(per if state["many"] else per.max(0).values)
    return out


def work(case):
    sizes, edges = [], 0
    for s in case["surfaces"].split("+"):
        rp, col = _csr(s)
        sizes.append(len(rp) - 1)
        edges += len(col)
    V = sum(sizes)
    if case["kind"] == "image":
        return dict(bytes=4.0 * (2 * V + edges), flops=float(edges))
    n, k = case["n"], case["k"]
    if case["kind"] == "tval":
        return dict(bytes=4.0 * n * V + 8.0 * k * V, flops=4.0 * n * k * V)
    P, m = case["P"], 1 if case["kind"] == "mediation" else k - 1 - case["fixed"]
    flops = 2.0 * P * m * n * V
    if case["kind"] == "maps":
        return dict(bytes=4.0 * (n * V + case["con"] * P * V + n * P), flops=flops)
    # the statistic maps of a batch are read once by the sweep that follows the contraction, written once before it
    signs = 1 if case["kind"] == "mediation" else 2
    return dict(bytes=4.0 * (n * V + 2 * case["con"] * P * V + edges + n * P), flops=flops + signs * case["con"] * P * edges)


# --- the same in 64 bits, without this repository's code -------------------------------------------------------

def _tfce64(csr, image, H, E):
    """TFCE of a float32 image: the operator's float32 thresholds, everything else in 64 bits."""
    rp, col = [int(v) for v in csr[0]], [int(v) for v in csr[1]]
    V = len(rp) - 1
    out = np.zeros(V)
    T = np.float32(image.max())
    if not T > 0:
        return out
    dT = np.float32(T / np.float32(100))
    order = np.argsort(-image, kind="stable")
    vals = image[order]
    parent = list(range(V))
    size = np.zeros(V, dtype=np.int64)
    on = [False] * V
    done = 0
    while T >= 0:
        end = int(np.searchsorted(-vals, -T, side="left"))  # the elements above T come first
        for v in order[done:end].tolist():
            on[v] = True
            size[v] = 1
            for u in col[rp[v]:rp[v + 1]]:
                if not on[u]:
                    continue
                a, b = v, u
                while parent[a] != a:
                    parent[a] = parent[parent[a]]
                    a = parent[a]
                while parent[b] != b:
                    parent[b] = parent[parent[b]]
                    b = parent[b]
                if a != b:
                    if size[a] < size[b]:
                        a, b = b, a
                    parent[b] = a
                    size[a] += size[b]
        done = end
        act = order[:end]
        root = np.asarray(parent)
        r = root[act]
        while True:
            r2 = root[r]
            if np.array_equal(r, r2):
                break
            r = r2
        out[act] += size[r].astype(np.float64) ** E * float(T) ** H
        T = np.float32(T - dT)
    return out


def _t64(X, Y, perms, moved, con):
    """[con, P, V] t-values of X with the rows of the ``moved`` columns permuted, in 64 bits."""
    n, k = X.shape
    Y = Y.double()
    yy = (Y * Y).sum(0)
    out = torch.empty((len(con), len(perms), Y.shape[1]), dtype=torch.float64, device="cuda")
    Xd = torch.from_numpy(X).cuda()
    for p, row in enumerate(perms.long()):
        Xp = Xd.clone()
        Xp[:, moved] = Xd[row][:, moved]
        inv = torch.linalg.inv((Xp.T @ Xp).cpu()).cuda()
        g = Xp.T @ Y
        a = inv @ g
        s2 = (yy - (a * g).sum(0)) / (n - k)
        for i, c in enumerate(con):
            out[i, p] = a[c] / torch.sqrt(s2 * inv[c, c])
    return out


def exact(case, seed):
    kind = case["kind"]
    V = _about(case["surfaces"])
    if kind == "image":
        state = prepare(case, seed)
        return _tfce64(_csr(case["surfaces"]), state["image"].cpu().numpy(), 2.0, case["E"])
    if kind == "tval":
        state = prepare(case, seed)
        Y, X = state["Y"], torch.from_numpy(state["X"]).cuda()
        inv = torch.from_numpy(state["inv"]).cuda()
        out = []
        for a in range(0, Y.shape[1], 1 << 17):
            y = Y[:, a:a + (1 << 17)].double()
            b = inv @ (X.T @ y)
            s2 = ((y - X @ b) ** 2).sum(0) / (state["n"] - state["k"])
            out.append(b / torch.sqrt(s2 * torch.diagonal(inv)[:, None]).float().double())
        return torch.cat(out, 1).cpu().numpy()
    if kind == "mediation" or case["weighted"]:
        return None
    small = kind == "null" and V * case["P"] * case["con"] <= 200_000
    if kind == "null" and not small:
        return None  # minutes of host union-find
    if kind == "maps" and case["n"] * V * case["P"] > 8_000_000_000:
        return None
    # the data as prepare() makes them
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    n, k = case["n"], case["k"]
    X = synth.design(rng, n, k - 2, binary=True)
    rng.standard_normal(n)
    g = torch.tensor(X[:, -1], dtype=torch.float32, device="cuda")
    size = int(rng.integers(100, 2001))
    _, csrs, offsets = _surfaces(case["surfaces"], case["E"])
    Y = torch.cat([_noise(c, n, case["smooth"], gen, (0.5 if i == 0 else 0.0) * g, size)
                   for i, c in enumerate(csrs)], 1)
    moved = list(range(1 + case["fixed"], k))
    t = _t64(X, Y, synth.permutations(n, case["P"], seed + 1, "cuda"), moved, list(range(k - case["con"], k)))
    if kind == "maps":
        return t
    maps = t.float().cpu().numpy()
    names = case["surfaces"].split("+")
    out = []
    for c in range(case["con"]):
        per = np.zeros((len(csrs), case["P"], 2))
        for s, csr in enumerate(csrs):
            E = 1.0 if names[s].startswith("mesh") and len(names) > 2 else case["E"]
            for p in range(case["P"]):
                for q, sign in enumerate((1, -1)):
                    x = np.float32(sign) * maps[c, p, offsets[s]:offsets[s + 1]]
                    top = float(x.max())
                    if _is_cut(names[s]):
                        top = max(top, 0.0)
                    per[s, p, q] = _tfce64(csr, x, 2.0, E).max() * (top / 100)
        out.append(per if len(csrs) > 2 else per.max(0))
    return out
