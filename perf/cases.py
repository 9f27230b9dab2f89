"""Timing cases of the counting engine: what its users have it do.

A case is one analysis of a synthetic galaxy catalogue (clustered data points followed by uniform
randoms) through the Python entry points: Engine.pcf2 / pcf3 / pcf3_equi / pcf4 / pcf4_tetra on a
catalogue handed over in the same pass, Engine.pcf2_batched / pcf3_batched on a set of regions the
engine holds, and weighted_xi with its backward pass.  Kinds:

  pcf2          pair counts in r or (r, mu)
  xi_grad       weighted xi and the gradient of a loss of it with respect to every weight
  pcf3          triangle counts (all configurations; equi: equilateral ones; nmu >= 2: redshift space)
  pcf4          four-point counts (tetra: regular tetrahedra)
  pcf2_regions  pair counts of many sub-volumes with buffer shells in one call
  pcf3_regions  triangle counts of the same

exact() computes the same floating-point results by brute force in 64-bit torch.
"""
import math

import numpy as np
import torch

from gramsci_amd.autograd import weighted_xi
from gramsci_amd.engine import Engine

_BASE = dict(kind="pcf2", n_data=0, n_rand=0, box=0.0, rmin=0.0, rmax=0.0, nbins=1, nmu=1, log=False,
             weights=False, precision="fp32", host=False)


def _case(name, kind, n_data, n_rand, box, rmin, rmax, nbins, nmu=1, **more):
    c = dict(_BASE, kind=kind, n_data=n_data, n_rand=n_rand, box=box, rmin=rmin, rmax=rmax, nbins=nbins, nmu=nmu)
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one small mock in a loop over many (a fit, a test suite): the call's fixed cost is what is paid
        _case("pcf2_call", "pcf2", 3000, 6000, 100.0, 1.0, 20.0, 8, 6, log=True, weights=True),
        # the plain isotropic count of a modest catalogue, unit weights
        _case("pcf2_plain", "pcf2", 20000, 40000, 500.0, 10.0, 50.0, 10),
        # what the command-line program does with an ordinary survey sample read from a file: host arrays
        _case("pcf2_host", "pcf2", 40009, 110017, 300.0, 1.0, 40.0, 12, 10, log=True, weights=True, host=True),
        # a full survey volume with 3x randoms in (r, mu): the largest single count
        _case("pcf2_survey", "pcf2", 1000000, 3000000, 1000.0, 1.0, 150.0, 30, 20, log=True, weights=True),
        # the same bins in plain 64-bit geometry, on a part of the volume
        _case("pcf2_fp64", "pcf2", 200003, 600011, 585.0, 1.0, 150.0, 30, 20, log=True, weights=True,
              precision="fp64"),
        # one step of a weight fit on a small catalogue: forward and backward
        _case("xi_grad_small", "xi_grad", 15013, 45007, 250.0, 2.0, 40.0, 10, 4, log=True, weights=True),
        # one step of a weight fit on a large one
        _case("xi_grad_survey", "xi_grad", 500000, 1500000, 1000.0, 0.0, 120.0, 20, 10, weights=True),
        # all triangle configurations at small scales, several hundred neighbours a point
        _case("pcf3_all", "pcf3", 200000, 400000, 500.0, 10.0, 30.0, 5),
        # redshift-space triangles of a weighted sample
        _case("pcf3_rsd", "pcf3", 30011, 60013, 300.0, 4.0, 20.0, 4, 4, log=True, weights=True),
        # four-point counts of a sparse sample
        _case("pcf4_all", "pcf4", 50000, 100000, 500.0, 10.0, 20.0, 3, precision="fp64"),
        # jackknife / decomposed sub-volumes with buffer shells, counted in one call
        _case("pcf2_regions", "pcf2_regions", 20000, 40000, 0.0, 5.0, 100.0, 20, 10, regions=16),
        _case("pcf3_regions", "pcf3_regions", 20000, 40000, 0.0, 5.0, 25.0, 4, regions=16),
    ]


# ------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _rmin(rng, log, rmax, lo=0.0):
    return round(rmax / _log(rng, 8, 60), 2) if log else round(rmax * rng.choice([lo, 0.1, 0.2, 0.3]), 2)


def draw(rng):
    kind = rng.choice(["pcf2"] * 5 + ["xi_grad"] * 2 + ["pcf3"] * 3 + ["pcf4", "pcf2_regions", "pcf3_regions"])
    if kind == "pcf2":
        n = int(_log(rng, 3e3, 3e6))
        fp64 = rng.random() < 0.25
        box = (n / _log(rng, 5e-4, 9e-3)) ** (1 / 3)
        rmax = min(_log(rng, 15, 150), 0.4 * box)
        while 0.5 * n * n * 4.19 * (rmax / box) ** 3 > (1.2e10 if fp64 else 5e10):
            rmax *= 0.9
        rmax = round(rmax, 2)
        log = rng.random() < 0.5
        nd = n // rng.choice([3, 4])
        return _case(None, kind, nd, n - nd, round(box, 1), _rmin(rng, log, rmax), rmax,
                     rng.randint(5, 30), rng.choice([1, 4, 7, 10, 20]), log=log, weights=rng.random() < 0.6,
                     precision="fp64" if fp64 else "fp32", host=n < 600000 and rng.random() < 0.3)
    if kind == "xi_grad":
        n = int(_log(rng, 2e4, 1.2e6))
        dens = _log(rng, 1e-3, 5e-3)
        box = (n / dens) ** (1 / 3)
        rmax = min(_log(rng, 30, 120), 0.35 * box)
        while 0.5 * n * n * 4.19 * (rmax / box) ** 3 > 8e9:
            rmax *= 0.9
        log = rng.random() < 0.5
        # no (r, mu) bin is left without random pairs
        return _case(None, kind, n // 4, n - n // 4, round(box, 1), round(rmax / rng.choice([4, 6, 8]), 2) if log else 0.0,
                     round(rmax, 2), rng.randint(5, 12) if log else rng.randint(4, 8), rng.choice([1, 2, 4, 5]),
                     log=log, weights=True)
    if kind == "pcf3":
        rsd = rng.random() < 0.3
        k = _log(rng, 30, 150 if rsd else 450)
        n = int(_log(rng, 8e3, min(6e5, 4e9 / k ** 2 if rsd else 6e10 / k ** 2)))
        dens = _log(rng, 1e-3, 9e-3)
        rmax = round((3 * k / (4 * math.pi * dens)) ** (1 / 3), 2)
        log = rng.random() < 0.3
        return _case(None, kind, n // 3, n - n // 3, round((n / dens) ** (1 / 3) + rmax, 1),
                     _rmin(rng, log, rmax, 0.2), rmax, rng.randint(3, 5 if rsd else 8), rng.randint(2, 6) if rsd else 1,
                     log=log, weights=rng.random() < 0.4, precision="fp64" if rng.random() < 0.2 else "fp32",
                     equi=rng.random() < 0.2)
    if kind == "pcf4":
        n = int(_log(rng, 2e4, 2e5))
        dens = _log(rng, 1e-3, 3e-3)
        rmax = round((3 * rng.uniform(12, 40) / (4 * math.pi * dens)) ** (1 / 3), 2)
        return _case(None, kind, n // 3, n - n // 3, round((n / dens) ** (1 / 3) + rmax, 1),
                     round(rmax * rng.choice([0.3, 0.4, 0.5]), 2), rmax, rng.randint(2, 4), weights=rng.random() < 0.3,
                     precision="fp64", tetra=rng.random() < 0.3)
    n = int(_log(rng, 4e3, 2.5e4))
    rmax = round(rng.uniform(40, 100) if kind == "pcf2_regions" else rng.uniform(15, 25), 1)
    return _case(None, kind, n, 2 * n, 0.0, round(0.1 * rmax, 1), rmax,
                 rng.randint(8, 20) if kind == "pcf2_regions" else rng.randint(3, 4),
                 rng.choice([1, 5, 10]) if kind == "pcf2_regions" else 1, regions=rng.randint(5, 20))


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(n, box, g):
    return torch.rand((n, 3), generator=g, device="cuda", dtype=torch.float64) * box


def _clustered(n, box, g):
    """Half uniform, half in clusters of 20 points with a Gaussian width of 2, wrapped, in random order."""
    parents = _uniform(n // 40, box, g).repeat_interleave(20, dim=0)
    off = torch.randn(parents.shape, generator=g, device="cuda", dtype=torch.float64) * 2.0
    pts = torch.cat([torch.remainder(parents + off, box), _uniform(n - len(parents), box, g)])
    return pts[torch.randperm(n, generator=g, device="cuda")].contiguous()


def _catalogue(case, seed):
    g = _generator(seed)
    xyz = torch.cat([_clustered(case["n_data"], case["box"], g), _uniform(case["n_rand"], case["box"], g)])
    w = None
    if case["weights"]:     # lognormal data weights, unit weights of the randoms
        w = torch.ones(len(xyz), dtype=torch.float64, device="cuda")
        w[:case["n_data"]] = torch.exp(0.2 * torch.randn(case["n_data"], generator=g, device="cuda",
                                                         dtype=torch.float64))
    return xyz, w


_DENSITY = 5e-4     # data points per unit volume of a region; twice as many randoms


def _region_sizes(case):
    """Data points inside each region: spread over a factor of about eight around n_data, the same for every
    seed (the fixed quantiles of a lognormal distribution)."""
    r = case["regions"]
    q = torch.special.ndtri((torch.arange(r, dtype=torch.float64) + 0.5) / r)
    return [int(x) for x in (case["n_data"] * torch.exp(0.7 * q)).tolist()]


def _regions(case, seed):
    g = _generator(seed)
    rmax, xs, bufs, off, nd, x0 = case["rmax"], [], [], [0], [], 0.0
    for n in _region_sizes(case):
        side = (n / _DENSITY) ** (1 / 3)
        big = side + 2 * rmax
        m = int(round(n * (big / side) ** 3))
        p = torch.cat([_clustered(m, big, g), _uniform(2 * m, big, g)]) - rmax
        bufs.append((~((p >= 0) & (p < side)).all(dim=1)).to(torch.int32))
        xs.append(p + torch.tensor([x0, 0.0, 0.0], dtype=torch.float64, device="cuda"))
        x0 += big + 10.0        # side by side
        nd.append(m)
        off.append(off[-1] + len(p))
    return torch.cat(xs), torch.cat(bufs), off, nd


_engines = {}


def _engine():
    """The one engine that a program keeps for all its catalogues."""
    if "e" not in _engines:
        _engines["e"] = Engine(0)
    return _engines["e"]


def _bins(case):
    return dict(rmin=case["rmin"], rmax=case["rmax"], nbins=case["nbins"], log_bins=case["log"])


def prepare(case, seed):
    kind = case["kind"]
    if kind.endswith("_regions"):
        xyz, buf, off, nd = _regions(case, seed)
        eng = Engine(0)         # the regions stay with their engine for the analyses that follow
        eng.set_catalogue_batched(xyz.cpu().numpy(), None, buf.cpu().numpy(), off, nd)
        return dict(case=case, eng=eng)
    xyz, w = _catalogue(case, seed)
    if case["host"]:
        xyz, w = xyz.cpu().numpy(), None if w is None else w.cpu().numpy()
    torch.cuda.synchronize()
    return dict(case=case, xyz=xyz, w=w, eng=None if kind == "xi_grad" else _engine())


def run(state):
    c, eng = state["case"], state["eng"]
    kind, bins = c["kind"], _bins(c)
    if kind == "xi_grad":
        w = state["w"].detach().requires_grad_(True)
        xi = weighted_xi(w, state["xyz"], c["n_data"], nmu=c["nmu"], precision=c["precision"], **bins)
        (xi ** 2).sum().backward()
        return dict(xi=xi.detach(), grad=w.grad)
    if not kind.endswith("_regions"):
        eng.set_catalogue(state["xyz"], state["w"], c["n_data"])
    if kind.startswith("pcf2"):
        f = eng.pcf2_batched if kind == "pcf2_regions" else eng.pcf2
        r = f(nmu=c["nmu"], precision=c["precision"], **bins)
    elif kind.startswith("pcf3"):
        f = eng.pcf3_batched if kind == "pcf3_regions" else eng.pcf3_equi if c.get("equi") else eng.pcf3
        r = f(nmu=c["nmu"], precision=c["precision"], **bins)
    else:
        r = (eng.pcf4_tetra if c.get("tetra") else eng.pcf4)(precision=c["precision"], **bins)
    return {k: r[k] for k in ("cnt", "wsum", "n2", "n3", "disc_n", "disc_r") if k in r}


# ------------------------------------------------------------------ work
def work(case):
    """Bytes: coordinates, weights and flags read once, results written once.  FLOPs: 22 for an unordered pair
    in (r, mu) and 8 in r (separation, its square, the angle), 8 for the third side of a triangle seen from its
    first vertex, 16 for a quadrilateral; numbers of pairs as in a uniform catalogue."""
    kind, nb, nm = case["kind"], case["nbins"], case["nmu"]
    shell = 4 / 3 * math.pi * (case["rmax"] ** 3 - case["rmin"] ** 3)
    if kind.endswith("_regions"):
        side = [(n / _DENSITY) ** (1 / 3) for n in _region_sizes(case)]
        n = sum(3 * _DENSITY * (s + 2 * case["rmax"]) ** 3 for s in side)
        apexes, dens, regions = sum(3 * _DENSITY * s ** 3 for s in side), 3 * _DENSITY, case["regions"]
    else:
        n = apexes = case["n_data"] + case["n_rand"]
        dens, regions = n / case["box"] ** 3, 1
    k = dens * shell
    size = n * (24 + (8 if case["weights"] else 0) + (4 if kind.endswith("_regions") else 0))
    if kind in ("pcf2", "pcf2_regions", "xi_grad"):
        flops = 0.5 * apexes * k * (8 if nm == 1 else 22) * (2 if kind == "xi_grad" else 1)
        out = regions * nb * nm * 64 + (8 * n if kind == "xi_grad" else 0)
    elif kind in ("pcf3", "pcf3_regions"):
        flops = apexes * k * k / (2 if nm > 1 else 8) * 8
        out = regions * nb * (1 if case.get("equi") else (nb + 1) * (nb + 2) / 6) * nm * 80
    else:
        flops = apexes * k ** 3 / 24 * 16
        out = nb * (1 if case.get("tetra") else nb * nb * (nb + 1) * (nb + 2) * (nb + 3) / 24) * 240
    return dict(bytes=size + out, flops=max(flops, 1.0))


# ------------------------------------------------------------------ brute force in 64 bits
def _rbin(case, d):
    lo, hi, nb = case["rmin"], case["rmax"], case["nbins"]
    if case["log"]:
        inv = 1.0 / ((math.log10(hi) - math.log10(lo)) / nb)
        b = torch.floor((torch.log10(d) - math.log10(lo)) * inv)
    else:
        b = torch.floor((d - lo) * (1.0 / ((hi - lo) / nb)))
    return b.clamp_(0, nb - 1).to(torch.int64)


def _mubin(nmu, a, b):
    """mu bin of the line from a to b against the line of sight to their middle."""
    if nmu < 2:
        return torch.zeros(len(a), dtype=torch.int64, device=a.device)
    mid, sep = 0.5 * (a + b), a - b
    theta = (mid * sep).sum(-1) / (mid.norm(dim=-1) * sep.norm(dim=-1))
    return torch.floor((theta + 1.0) * (0.5 * nmu)).clamp_(0, nmu - 1).to(torch.int64)


def _pairs(case, xyz, apex=None):
    """Ordered kept pairs (i, j) with their radial bin, block by block."""
    n = len(xyz)
    rows = torch.arange(n, device=xyz.device) if apex is None else apex
    step = max(1, int(6e7) // max(n, 1))
    for k in range(0, len(rows), step):
        r = rows[k:k + step]
        s = torch.zeros((len(r), n), dtype=torch.float64, device=xyz.device)
        for q in range(3):
            s += (xyz[r, q][:, None] - xyz[None, :, q]) ** 2
        d = s.sqrt_()
        i, j = torch.nonzero((d > case["rmin"]) & (d < case["rmax"]), as_tuple=True)
        dij = d[i, j]
        i = r[i]
        if case["rmin"] <= 0:
            keep = i != j
            i, j, dij = i[keep], j[keep], dij[keep]
        yield i, j, _rbin(case, dij)


def _add(acc, index, values):
    acc += torch.bincount(index, weights=values, minlength=len(acc))


def _normalised(w, n_data):
    wn = w.clone()
    wn[:n_data] /= w[:n_data].sum()
    wn[n_data:] /= -w[n_data:].sum()
    return wn


def _exact2(case, xyz, w, n_data, apex=None):
    nb, nm = case["nbins"], case["nmu"]
    nbm = nb * nm
    wn = _normalised(w, n_data)
    wsum = torch.zeros(3 * nbm, dtype=torch.float64, device="cuda")
    n2, n3 = torch.zeros_like(wsum[:nbm]), torch.zeros_like(wsum[:nbm])
    for i, j, b in _pairs(case, xyz, apex):
        h = b * nm + _mubin(nm, xyz[i], xyz[j])
        rr = (i >= n_data).to(torch.int64) + (j >= n_data).to(torch.int64)
        _add(wsum, rr * nbm + h, w[i] * w[j])
        p = wn[i] * wn[j]
        _add(n2, h, p)
        _add(n3, h, p * (rr == 2))
    return wsum.view(3, nb, nm).cpu().numpy(), n2.view(nb, nm).cpu().numpy(), n3.view(nb, nm).cpu().numpy()


def _exact_grad(case, xyz, w, n_data):
    nb, nm = case["nbins"], case["nmu"]
    wn = _normalised(w, n_data)
    _, n2, n3 = (torch.from_numpy(x).cuda() for x in _exact2(case, xyz, w, n_data))
    xi = n2 / n3
    g2 = (2 * xi / n3).reshape(-1)              # dL/dN2 and dL/dN3 of L = sum xi^2
    g3 = (-2 * xi * n2 / (n3 * n3)).reshape(-1)
    acc = torch.zeros(len(w), dtype=torch.float64, device="cuda")
    for i, j, b in _pairs(case, xyz):           # every ordered pair: both of its ends
        h = b * nm + _mubin(nm, xyz[i], xyz[j])
        coef = g2[h] + g3[h] * ((i >= n_data) & (j >= n_data))
        _add(acc, i, coef * wn[j])
        _add(acc, j, coef * wn[i])
    d, r = slice(0, n_data), slice(n_data, None)
    grad = torch.empty_like(acc)
    grad[d] = (acc[d] - (wn[d] * acc[d]).sum()) / w[d].sum()
    grad[r] = -(acc[r] + (wn[r] * acc[r]).sum()) / w[r].sum()
    return dict(xi=xi, grad=grad)


def _normal_bins(nm):
    """mu bin of a triangle's normal from those of two sides, in the single precision it is defined in."""
    f = np.float32
    t = np.zeros((nm, nm), np.int64)
    for p in range(nm):
        for q in range(nm):
            a = f(float(f(p + 1) - f(0.5)) / (0.5 * nm) - 1.0)
            b = f(float(f(q + 1) - f(0.5)) / (0.5 * nm) - 1.0)
            x = f(f(f(f(0.75) - f(a * a)) - f(b * b)) + f(a * b))
            v = int(math.floor(f(f(f(1.1547) * np.sqrt(x)) * f(nm)))) if x >= 0 else 0
            t[p, q] = min(max(v, 0), nm - 1)
    return torch.from_numpy(t).cuda()


def _exact3(case, xyz, w, n_data):
    nb, nm, equi = case["nbins"], case["nmu"], bool(case.get("equi"))
    wn, n = _normalised(w, n_data), len(xyz)
    cfg = torch.zeros((nb, nb, nb), dtype=torch.int64)
    nc = 0
    for a in range(nb):
        for b in range(a, nb):
            for c in range(b, nb):
                for p in ((a, b, c), (a, c, b), (b, a, c), (b, c, a), (c, a, b), (c, b, a)):
                    cfg[p] = nc
                nc += 1
    cfg = cfg.cuda()
    if equi:
        nc = nb
    normal = _normal_bins(nm) if nm > 1 else None
    i, j, b = (torch.cat(x) for x in zip(*_pairs(case, xyz)))       # by apex, then by neighbour
    mu = _mubin(nm, xyz[i], xyz[j])
    k = torch.bincount(i, minlength=n)
    start = torch.cumsum(k, 0) - k
    wsum = torch.zeros(nc * nm * 4, dtype=torch.float64, device="cuda")
    n2, n3 = torch.zeros_like(wsum[:nc * nm]), torch.zeros_like(wsum[:nc * nm])
    at = 0
    while at < n:       # blocks of apexes, padded to the longest list
        most, end = int(k[at]), at
        upto = k[at:at + 4096].cummax(0).values
        size = torch.arange(1, len(upto) + 1, device="cuda") * upto * upto
        end = at + max(1, int((size <= int(4e7)).sum()))
        most = int(k[at:end].max())
        if most >= 2:
            u, v = torch.triu_indices(most, most, 1, device="cuda")
            ap = torch.arange(at, end, device="cuda")
            q, t = torch.nonzero(v[None, :] < k[ap][:, None], as_tuple=True)
            e1, e2, ap = start[ap][q] + u[t], start[ap][q] + v[t], ap[q]
            d = ((xyz[j[e1]] - xyz[j[e2]]) ** 2).sum(-1).sqrt()
            keep = (d > case["rmin"]) & (d < case["rmax"])
            e1, e2, ap, d = e1[keep], e2[keep], ap[keep], d[keep]
            b3 = _rbin(case, d)
            if equi:
                keep = (b[e1] == b3) & (b[e2] == b3)
                e1, e2, ap, b3 = e1[keep], e2[keep], ap[keep], b3[keep]
            c = b3 if equi else cfg[b[e1], b[e2], b3]
            m = normal[mu[e1], mu[e2]] if nm > 1 else 0
            rnd = sum((x >= n_data).to(torch.int64) for x in (ap, j[e1], j[e2]))
            _add(wsum, (c * nm + m) * 4 + rnd, w[ap] * w[j[e1]] * w[j[e2]])
            p = wn[ap] * wn[j[e1]] * wn[j[e2]]
            _add(n2, c * nm + m, p)
            if not (equi and nm > 1):
                _add(n3, c * nm + m, -p * (rnd == 3))
        at = end
    flat = nm == 1 and not equi
    return [x.cpu().numpy() for x in (wsum.view((nc, 4) if flat else (nc, nm, 4)),
                                      n2.view(nc if flat else (nc, nm)), n3.view(nc if flat else (nc, nm)))]


def exact(case, seed):
    kind = case["kind"]
    if kind == "pcf4" or kind == "pcf3_regions":
        return None             # whole counts, and sums formed from them
    if kind == "pcf2_regions":
        xyz, buf, off, nd = _regions(case, seed)
        if sum(float(b - a) * int((buf[a:b] == 0).sum()) for a, b in zip(off, off[1:])) > 3e10:
            return None
        got = []
        for a, b, d in zip(off, off[1:], nd):
            got.append(_exact2(case, xyz[a:b], torch.ones(b - a, dtype=torch.float64, device="cuda"), d,
                               torch.nonzero(buf[a:b] == 0).flatten()))
        wsum, n2, n3 = (np.stack(x) for x in zip(*got))
        return dict(cnt=None, wsum=wsum, n2=n2, n3=n3)
    n = case["n_data"] + case["n_rand"]
    kept = n * n * 4.19 * (case["rmax"] / case["box"]) ** 3
    if n > 200000 or kept > 4e9 or (kind == "pcf3" and (kept > 1.5e8 or kept * kept / n > 8e9)):
        return None
    xyz, w = _catalogue(case, seed)
    w = torch.ones(n, dtype=torch.float64, device="cuda") if w is None else w
    if kind == "xi_grad":
        return _exact_grad(case, xyz, w, case["n_data"])
    wsum, n2, n3 = (_exact2 if kind == "pcf2" else _exact3)(case, xyz, w, case["n_data"])
    return dict(cnt=None, wsum=wsum, n2=n2, n3=n3)
