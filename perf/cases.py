"""What this framework is used for, as cases that can be timed and checked.

A case is a dict of plain values.  `kind` names the public calls that a user's
program makes:

  grid       the LJ energy grid of a resident framework: `compute_grid` to a host
             array (writegrid), or `er_grid_compute_noalloc` into device memory
             that the program owns
  screen     one structure from its atom list: upload, grid, Henry run, release
  widom      Henry coefficient of a resident framework, sums alone or with the
             energy of every insertion
  batch      a set of frameworks as one captured batch, results fetched
  serve      requests to the continuous-batching server, from submit to release
  pockets    grids from the host: upload, label and block, grid Widom, download
  interp     trilinear Widom insertions on a resident grid
  energies   trilinear energies at the caller's positions (GCMC energy calls)

Frameworks are synthetic: atoms on a jittered lattice, kept where a random
periodic field is highest, so that there are walls, channels and closed pockets
as in a porous crystal and no two atoms overlap.  Cells, spacings, guests, atom
types and insertion counts are those of the benchmark workloads and tests of
this repository (25 A cubic cell with 400 atoms and a 50^3 grid, the IRMOF-1
cell with 424 atoms, 3000 atoms at 0.1 A, the 256-framework mix).
"""
import ctypes
import itertools
import math
import random

import numpy as np
import torch

from emptyroom_amd import api

RC = 12.5
RC2 = RC * RC
TEMPERATURE = 298.0
GUESTS = {"CH4": (148.0, 3.73), "Xe": (221.0, 4.10), "Kr": (166.4, 3.636)}


# ---------------------------------------------------------------- the cases

def _cell(a, b, c, alpha=90.0, beta=90.0, gamma=90.0):
    return dict(a=a, b=b, c=c, alpha=alpha, beta=beta, gamma=gamma)


def listed():
    return [
        # a quick look at a small molecule-sized cell: launches and latency
        dict(name="grid_smallest", kind="grid", atoms=40, guest="CH4", spacing=0.5,
             fp64=False, host=True, **_cell(10.0, 11.0, 12.0, 85.0, 95.0, 100.0)),
        # the plain-method workload: one structure of a screening run, end to end
        dict(name="screen_400", kind="screen", atoms=400, guest="CH4", spacing=0.5,
             fp64=False, insertions=100_000, **_cell(25.0, 25.0, 25.0)),
        # the drop-in writegrid at its default precision, IRMOF-1's cell
        dict(name="grid_fp64_host", kind="grid", atoms=424, guest="CH4", spacing=0.15,
             fp64=True, host=True, **_cell(25.832, 25.832, 25.832)),
        # a precise grid of a dense triclinic crystal, kept on the device
        dict(name="grid_fine_device", kind="grid", atoms=3000, guest="CH4", spacing=0.1,
             fp64=False, host=False, **_cell(24.0, 22.0, 28.0, 82.0, 97.0, 104.0)),
        # the largest cells of the mix at its finest spacing
        dict(name="grid_large_device", kind="grid", atoms=2400, guest="Xe", spacing=0.1,
             fp64=False, host=False, **_cell(37.0, 34.0, 39.0, 90.0, 101.0, 90.0)),
        # henry: the reference's insertion count for IRMOF-1 (1000 per A^3)
        dict(name="henry_large", kind="widom", atoms=424, guest="CH4",
             insertions=17_252_352, energies=False, **_cell(25.832, 25.832, 25.832)),
        # per-insertion energies for a caller's own averages
        dict(name="widom_energies", kind="widom", atoms=1000, guest="Kr",
             insertions=200_003, energies=True, **_cell(19.0, 23.0, 21.0, 76.0, 88.0, 109.0)),
        # a slice of the batching mix: grids and 1e6 insertions per framework
        dict(name="batch_mix", kind="batch", frameworks=16, insertions=1_000_000),
        # mixed grid and Henry requests over a pool of frameworks
        dict(name="serve_mix", kind="serve", requests=24, frameworks=8, insertions=300_000),
        # pocket blocking of stored grids, then Henry on the blocked grids
        dict(name="pockets_chain", kind="pockets", grids=4, spacing=0.2, insertions=1_000_000),
        # trilinear Widom on a resident 0.2 A grid
        dict(name="interp_widom", kind="interp", atoms=700, guest="CH4", spacing=0.2,
             insertions=10_000_000, **_cell(27.0, 24.0, 25.0, 80.0, 95.0, 100.0)),
        # energies of many trial moves on a resident grid
        dict(name="grid_energies", kind="energies", atoms=500, guest="CH4", spacing=0.2,
             fp64=False, positions=1_000_000, **_cell(24.0, 22.0, 26.0, 90.0, 95.0, 90.0)),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _draw_cell(rng, lo, hi):
    while True:
        al, be, ga = (90.0, 90.0, 90.0) if rng.random() < 0.25 else (
            round(rng.uniform(65.0, 115.0), 2) for _ in range(3))
        c = [math.cos(math.radians(x)) for x in (al, be, ga)]
        if 1 - sum(x * x for x in c) + 2 * c[0] * c[1] * c[2] > 0.25:
            return _cell(*(round(_log(rng, lo, hi), 3) for _ in range(3)), al, be, ga)


def _draw_framework(rng, lo=9.0, hi=36.0):
    cell = _draw_cell(rng, lo, hi)
    volume = _matrix(cell)[1]
    atoms = int(min(3000, max(20, volume * _log(rng, 0.01, 0.12))))
    return dict(atoms=atoms, guest=rng.choice(sorted(GUESTS)), **cell)


def _spacing(rng, cell, most):
    s = rng.choice([0.1, 0.15, 0.2, 0.25, 0.5, round(_log(rng, 0.1, 0.6), 3)])
    points = cell["a"] * cell["b"] * cell["c"] / s ** 3
    return s if points <= most else round(s * (points / most) ** (1 / 3) + 0.005, 3)


def draw(rng):
    kind = rng.choice(["grid", "grid", "grid", "screen", "widom", "widom", "batch", "serve",
                       "pockets", "interp", "energies"])
    if kind == "grid":
        f = _draw_framework(rng)
        host = rng.random() < 0.4
        fp64 = rng.random() < 0.4
        most = 6e6 if host else 1.5e7 if fp64 else 3e7
        return dict(kind=kind, spacing=_spacing(rng, f, most), fp64=fp64, host=host, **f)
    if kind == "screen":
        return dict(kind=kind, spacing=round(rng.uniform(0.3, 0.8), 3), fp64=rng.random() < 0.3,
                    insertions=int(_log(rng, 2e4, 5e5)), **_draw_framework(rng, 9.0, 30.0))
    if kind == "widom":
        energies = rng.random() < 0.4
        return dict(kind=kind, insertions=int(_log(rng, 5e3, 6e5 if energies else 1.2e7)),
                    energies=energies, **_draw_framework(rng))
    if kind == "batch":
        return dict(kind=kind, frameworks=rng.randint(3, 16), insertions=int(_log(rng, 1e5, 1e6)))
    if kind == "serve":
        return dict(kind=kind, requests=rng.randint(4, 24), frameworks=rng.randint(2, 8),
                    insertions=int(_log(rng, 3e4, 3e5)))
    if kind == "pockets":
        return dict(kind=kind, grids=rng.randint(1, 4), spacing=round(rng.uniform(0.18, 0.5), 3),
                    insertions=int(_log(rng, 1e5, 2e6)))
    f = _draw_framework(rng, 12.0, 34.0)
    f["spacing"] = max(round(rng.uniform(0.15, 0.5), 3), _spacing(rng, f, 4e6))
    if kind == "interp":
        return dict(kind=kind, insertions=int(_log(rng, 5e4, 1e7)), **f)
    return dict(kind=kind, fp64=rng.random() < 0.4, positions=int(_log(rng, 1e3, 1e6)), **f)


# ---------------------------------------------------------------- frameworks

def _matrix(cell):
    a, b, c = cell["a"], cell["b"], cell["c"]
    ca, cb, cg = (math.cos(math.radians(cell[k])) for k in ("alpha", "beta", "gamma"))
    sg = math.sin(math.radians(cell["gamma"]))
    v = math.sqrt(1 - ca * ca - cb * cb - cg * cg + 2 * ca * cb * cg)
    t = np.array([[a, b * cg, c * cb], [0.0, b * sg, c * (ca - cb * cg) / sg],
                  [0.0, 0.0, c * v / sg]])
    return t, v * a * b * c


class _Atoms:
    """Atoms, cell and image half-ranges of a synthetic porous framework."""

    def __init__(self, seed, atoms, guest, cell, types=6):
        rng = np.random.default_rng(seed)
        self.lengths = (cell["a"], cell["b"], cell["c"])
        self.t, self.volume = _matrix(cell)
        width = 1.0 / np.linalg.norm(np.linalg.inv(self.t), axis=1)
        self.rep = [int(2.0 * RC / w) + 1 for w in width]
        step = min(1.5, (self.volume / (1.3 * atoms)) ** (1 / 3))
        m = [max(1, int(round(w / step))) for w in width]
        while m[0] * m[1] * m[2] < atoms:
            m[int(np.argmin(m))] += 1
        site = np.stack(np.meshgrid(*(np.arange(k) for k in m), indexing="ij"), -1).reshape(-1, 3)
        frac = (site + 0.5 + rng.uniform(-0.12, 0.12, site.shape)) / np.array(m)
        field = np.zeros(len(frac))
        for _ in range(6):
            k = rng.integers(-2, 3, 3)
            field += np.cos(2 * np.pi * (frac @ k) + rng.uniform(0, 2 * np.pi))
        keep = np.argsort(-(field + 0.5 * rng.standard_normal(len(field))))[:atoms]
        self.frac = (frac[rng.permutation(keep)] + rng.uniform(0, 1, 3)) % 1.0
        eps, sig = rng.uniform(20.0, 250.0, types), rng.uniform(2.5, 4.0, types)
        kind = rng.integers(0, types, atoms)
        eg, sg = GUESTS[guest]
        self.eps = np.sqrt(eg * eps[kind])
        self.sig2 = ((sg + sig[kind]) / 2.0) ** 2

    def grid_n(self, spacing):
        return [max(2, int(math.ceil(x / spacing))) for x in self.lengths]

    def upload(self, ctx):
        return api.Framework(ctx, self.frac, self.eps, self.sig2, self.t, self.rep, RC2)


def _atoms(case, seed):
    return _Atoms(seed, case["atoms"], case["guest"], case)


def _members(case, seed, count):
    """`count` frameworks spread over the sizes, spacings and guests of the
    batching mix: sizes by the case, atoms by the seed."""
    rng = random.Random(977 * count)
    got = []
    for i in range(count):
        cell = _draw_cell(rng, 9.0, 34.0)
        atoms = int(min(3000, max(30, _matrix(cell)[1] * _log(rng, 0.01, 0.12))))
        spacing = (0.1, 0.2, 0.5)[i % 3]
        if cell["a"] * cell["b"] * cell["c"] / spacing ** 3 > 1.2e7:
            spacing = 0.2
        got.append((_Atoms(seed * 1000 + i, atoms, ("CH4", "Xe", "Kr")[(i // 3) % 3], cell),
                    spacing))
    return got


# ---------------------------------------------------------------- one pass

class _State:
    """A case's handles; what was opened last is closed first."""

    def __init__(self, case, seed):
        self.case, self.seed, self.open = case, seed, []
        self.ctx = self.keep(api.Context(0))

    def keep(self, handle):
        self.open.append(handle)
        return handle

    def __del__(self):
        for handle in reversed(self.open):
            handle.close()


def prepare(case, seed):
    s = _State(case, seed)
    kind = case["kind"]
    if kind in ("grid", "widom", "interp", "energies"):
        f = s.atoms = _atoms(case, seed)
        s.fw = s.keep(f.upload(s.ctx))
    if kind == "grid":
        s.n = f.grid_n(case["spacing"])
        s.precision = api.ER_FP64 if case["fp64"] else api.ER_FP32
        if not case["host"]:
            s.out = torch.empty(s.n, device="cuda",
                                dtype=torch.float64 if case["fp64"] else torch.float32)
            s.dims = (ctypes.c_int * 3)(*s.n)
    elif kind == "screen":
        s.atoms = _atoms(case, seed)
        s.n = s.atoms.grid_n(case["spacing"])
    elif kind == "batch":
        s.members = _members(case, seed, case["frameworks"])
        tasks = [dict(fw=s.keep(f.upload(s.ctx)), grid_n=f.grid_n(h), precision=api.ER_FP32,
                      n_insertions=case["insertions"], temperature=TEMPERATURE,
                      seed=seed * 100 + i) for i, (f, h) in enumerate(s.members)]
        s.batch = s.keep(api.Batch(s.ctx, tasks, use_graph=True))
    elif kind == "serve":
        s.members = _members(case, seed, case["frameworks"])
        s.server = s.keep(api.Server(s.ctx))
        s.requests = _requests(case, seed, s.members)
    elif kind == "pockets":
        s.grids = []
        for f, _ in _members(case, seed, case["grids"]):
            fw = f.upload(s.ctx)
            s.grids.append(api.compute_grid(s.ctx, fw, f.grid_n(case["spacing"]), api.ER_FP32))
            fw.close()
    elif kind in ("interp", "energies"):
        s.grid = s.keep(api.Grid.compute(s.ctx, s.fw, f.grid_n(case["spacing"]),
                                         api.ER_FP64 if case.get("fp64") else api.ER_FP32))
        if kind == "energies":
            s.positions = np.random.default_rng(seed + 1).uniform(-0.5, 1.5,
                                                                  (case["positions"], 3))
    return s


def _requests(case, seed, members):
    rng = random.Random(31 * case["requests"])
    got = []
    for i in range(case["requests"]):
        f, h = members[rng.randrange(len(members))]
        common = dict(frac=f.frac, eps=f.eps, sig2=f.sig2, t_matrix=f.t, rep=f.rep, rc2=RC2)
        if rng.random() < 0.5:
            h = max(h, 0.2)
            got.append((f, dict(common, grid_n=f.grid_n(h), precision=api.ER_FP32)))
        else:
            got.append((f, dict(common, n_insertions=case["insertions"],
                                temperature=rng.uniform(250.0, 350.0), seed=seed * 100 + i)))
    return got


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "grid":
        if case["host"]:
            return api.compute_grid(s.ctx, s.fw, s.n, s.precision)
        code = api.lib().er_grid_compute_noalloc(s.ctx.h, s.fw.h, s.dims, s.precision,
                                                 s.out.data_ptr())
        if code != 0:
            raise api.EmptyRoomError(code, api.lib().er_last_error().decode())
        return s.out
    if kind == "screen":
        fw = s.atoms.upload(s.ctx)
        grid = api.compute_grid(s.ctx, fw, s.n, api.ER_FP64 if case["fp64"] else api.ER_FP32)
        sb, seb, _ = api.widom(s.ctx, fw, case["insertions"], TEMPERATURE, s.seed)
        fw.close()
        return grid, sb, seb
    if kind == "widom":
        got = api.widom(s.ctx, s.fw, case["insertions"], TEMPERATURE, s.seed,
                        energies=case["energies"])
        return (got[0], got[1]) + ((got[3],) if case["energies"] else ())
    if kind == "batch":
        s.batch.run()
        s.batch.wait()
        sums = np.array([s.batch.widom(i)[:2] for i in range(case["frameworks"])])
        return [sums] + [s.batch.grid(i) for i in range(case["frameworks"])]
    if kind == "serve":
        tickets = [s.server.submit(**rq)[1] for _, rq in s.requests]
        got = []
        for ticket, (_, rq) in zip(tickets, s.requests):
            done = s.server.poll(ticket, -1.0)
            if done.state != api.RQ_DONE:
                raise RuntimeError("request %d: state %d" % (ticket, done.state))
            if "grid_n" in rq:
                got.append(s.server.fetch_grid(ticket, rq["grid_n"]))
            else:
                got.append(np.array([done.widom.sum_b, done.widom.sum_eb]))
            s.server.release(ticket)
        return got
    if kind == "pockets":
        grids = [api.Grid.upload(s.ctx, g) for g in s.grids]
        counts = api.pockets_label_batch(s.ctx, grids, TEMPERATURE, block=True)
        sums = np.array([api.widom_grid(s.ctx, g, case["insertions"], TEMPERATURE, s.seed)[:2]
                         for g in grids])
        blocked = [g.download() for g in grids]
        for g in grids:
            g.close()
        return [np.array(counts), sums] + blocked
    if kind == "interp":
        return api.widom_grid(s.ctx, s.grid, case["insertions"], TEMPERATURE, s.seed)[:2]
    return api.grid_energies(s.ctx, s.grid, s.positions)


# ---------------------------------------------------------------- the work

def _pairs(volume, atoms, points):
    return points * atoms / volume * 4.0 / 3.0 * math.pi * RC ** 3


def work(case):
    """16 operations per (point, atom) pair inside the cutoff; inputs and
    results once over memory.  Trilinear points: 8 grid values read, about 40
    operations."""
    kind = case["kind"]
    if kind in ("batch", "serve", "pockets"):
        members = _members(case, 1, case.get("frameworks", case.get("grids")))
        if kind == "batch":
            tasks = [(f, f.grid_n(h), case["insertions"]) for f, h in members]
        elif kind == "serve":
            tasks = [(f, rq.get("grid_n"), rq.get("n_insertions", 0))
                     for f, rq in _requests(case, 1, members)]
        else:
            points = sum(int(np.prod(f.grid_n(case["spacing"]))) for f, _ in members)
            n = case["insertions"] * len(members)
            return {"bytes": 8 * points + 32 * n, "flops": 40 * n}
        size = sum(4 * int(np.prod(n)) for _, n, _ in tasks if n)
        pairs = sum(_pairs(f.volume, len(f.frac), (int(np.prod(n)) if n else 0) + ins)
                    for f, n, ins in tasks)
        return {"bytes": size + 40 * sum(len(f.frac) for f, _, _ in tasks), "flops": 16 * pairs}
    volume = _matrix(case)[1]
    n = [max(2, int(math.ceil(case[k] / case["spacing"]))) for k in "abc"] \
        if "spacing" in case else [0]
    points = int(np.prod(n))
    if kind == "interp":
        return {"bytes": 4 * points + 32 * case["insertions"], "flops": 40 * case["insertions"]}
    size = 8 if case.get("fp64") else 4
    if kind == "energies":
        return {"bytes": (32 + 8 * size) * case["positions"], "flops": 40 * case["positions"]}
    out = size * points + (8 * case["insertions"] if case.get("energies") else 0)
    return {"bytes": out + 40 * case["atoms"],
            "flops": 16 * _pairs(volume, case["atoms"], points + case.get("insertions", 0))}


# ------------------------------------------------- the same numbers in 64 bits

class _Exact:
    """Direct FP64 sums over the images of one framework, in plain torch."""

    def __init__(self, f, min_r2):
        dev = "cuda"
        self.t = torch.tensor(f.t, device=dev)
        images = torch.tensor(list(itertools.product(*(range(-r, r + 1) for r in f.rep))),
                              dtype=torch.float64, device=dev)
        frac = torch.tensor(f.frac, device=dev)
        g = (frac[None] + images[:, None]).reshape(-1, 3)
        ext = torch.tensor(RC * np.linalg.norm(np.linalg.inv(f.t), axis=1) + 1e-6, device=dev)
        keep = ((g >= -ext) & (g <= 1 + ext)).all(1)
        self.xyz = g[keep] @ self.t.T
        many = len(images)
        self.eps = torch.tensor(f.eps, device=dev).repeat(many)[keep]
        self.sig2 = torch.tensor(f.sig2, device=dev).repeat(many)[keep]
        self.min_r2 = min_r2

    def at(self, frac):
        """Energies at fractional points that lie near each other."""
        x = frac @ self.t.T
        mid = 0.5 * (x.amin(0) + x.amax(0))
        reach = RC + 1e-6 + float((x - mid).norm(dim=1).max())
        near = ((self.xyz - mid).norm(dim=1) < reach).nonzero()[:, 0]
        a, eps, sig2 = self.xyz[near], self.eps[near], self.sig2[near]
        out = torch.empty(len(x), dtype=torch.float64, device=x.device)
        step = max(64, (1 << 22) // max(1, len(near)))
        for i in range(0, len(x), step):
            p = x[i:i + step]
            r2 = (p[:, 0, None] - a[None, :, 0]) ** 2
            r2 += (p[:, 1, None] - a[None, :, 1]) ** 2
            r2 += (p[:, 2, None] - a[None, :, 2]) ** 2
            s6 = (sig2 / r2.clamp_(min=self.min_r2)) ** 3
            e = (4.0 * eps) * s6 * (s6 - 1.0)
            out[i:i + step] = torch.where(r2 < RC2, e, torch.zeros_like(e)).sum(1)
        return out

    def grid(self, n):
        axes = [torch.arange(k, dtype=torch.float64, device=self.t.device) / (k - 1) for k in n]
        out = torch.empty(n, dtype=torch.float64, device=self.t.device)
        b = 24
        for i, j, k in itertools.product(*(range(0, m, b) for m in n)):
            box = torch.meshgrid(axes[0][i:i + b], axes[1][j:j + b], axes[2][k:k + b],
                                 indexing="ij")
            e = self.at(torch.stack(box, -1).reshape(-1, 3))
            out[i:i + b, j:j + b, k:k + b] = e.reshape(box[0].shape)
        return out

    def widom(self, n, temperature, seed):
        f = _points(seed, 0, n)
        b = torch.clamp((f * 6).long(), max=5)
        order = torch.argsort((b[:, 0] * 6 + b[:, 1]) * 6 + b[:, 2])
        key = ((b[:, 0] * 6 + b[:, 1]) * 6 + b[:, 2])[order]
        cut = torch.searchsorted(key, torch.arange(217, device=f.device)).tolist()
        e = torch.empty(n, dtype=torch.float64, device=f.device)
        for lo, hi in zip(cut, cut[1:]):
            if hi > lo:
                e[order[lo:hi]] = self.at(f[order[lo:hi]])
        return e, _sums(e, temperature)


def _sums(e, temperature):
    w = torch.exp(-e / temperature)
    return float(w.sum()), float(torch.where(w == 0, torch.zeros_like(e), e * w).sum())


def _points(seed, stream, n):
    """Fractional points of the Philox4x32-10 stream that the insertions use."""
    low = 0xFFFFFFFF
    i = torch.arange(n, dtype=torch.int64, device="cuda")
    c = [i & low, i >> 32, torch.full_like(i, stream), torch.zeros_like(i)]
    k0, k1 = seed & low, seed >> 32

    def product(m, x):
        lo, hi = m * (x & 0xFFFF), m * (x >> 16)
        return (hi + (lo >> 16)) >> 16, (lo + ((hi & 0xFFFF) << 16)) & low

    for _ in range(10):
        h0, l0 = product(0xD2511F53, c[0])
        h1, l1 = product(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    return (torch.stack(c[:3], -1).double() + 1.0) * 2.0 ** -32


def _trilinear(grid, f):
    g = grid.double()
    n = torch.tensor(grid.shape, device=f.device)
    d = 1.0 / (n - 1).double()
    f = f - torch.floor(f)
    i = torch.minimum(torch.floor(f / d).long(), n - 2)
    w = (f - i * d) / d
    e = 0.0
    for c in itertools.product((0, 1), repeat=3):
        p = i + torch.tensor(c, device=f.device)
        part = g[p[:, 0], p[:, 1], p[:, 2]]
        for a in range(3):
            part = part * (w[:, a] if c[a] else 1.0 - w[:, a])
        e = e + part
    return e


def _stored(e, fp64):
    return e if fp64 else e.clamp(max=float(torch.finfo(torch.float32).max))


def exact(case, seed):
    kind = case["kind"]
    if kind == "grid":
        f = _atoms(case, seed)
        return _stored(_Exact(f, 1e-24).grid(f.grid_n(case["spacing"])), case["fp64"])
    if kind == "screen":
        f = _atoms(case, seed)
        grid = _stored(_Exact(f, 1e-24).grid(f.grid_n(case["spacing"])), case["fp64"])
        return (grid,) + _Exact(f, 1e-32).widom(case["insertions"], TEMPERATURE, seed)[1]
    if kind == "widom":
        e, sums = _Exact(_atoms(case, seed), 1e-32).widom(case["insertions"], TEMPERATURE, seed)
        return sums + ((e,) if case["energies"] else ())
    if kind == "batch":
        members = _members(case, seed, case["frameworks"])
        sums = [_Exact(f, 1e-32).widom(case["insertions"], TEMPERATURE, seed * 100 + i)[1]
                for i, (f, _) in enumerate(members)]
        return [np.array(sums)] + [_stored(_Exact(f, 1e-24).grid(f.grid_n(h)), False)
                                   for f, h in members]
    if kind == "serve":
        got = []
        for f, rq in _requests(case, seed, _members(case, seed, case["frameworks"])):
            if "grid_n" in rq:
                got.append(_stored(_Exact(f, 1e-24).grid(rq["grid_n"]), False))
            else:
                got.append(np.array(_Exact(f, 1e-32).widom(rq["n_insertions"],
                                                           rq["temperature"], rq["seed"])[1]))
        return got
    if kind == "pockets":
        return None  # blocked voxels and counts: whole numbers and stored values
    # trilinear values of the stored grid: the grid itself is an input here
    s = prepare(case, seed)
    grid = torch.from_numpy(s.grid.download()).cuda()
    if kind == "interp":
        return _sums(_trilinear(grid, _points(seed, 1, case["insertions"])), TEMPERATURE)
    return _trilinear(grid, torch.from_numpy(s.positions).cuda())
