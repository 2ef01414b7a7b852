"""Performance cases of the soft-force framework: what its users have it do.

A case is one call sequence of a user's program on one star cluster (Plummer
model, Kroupa masses, primordial binaries; theta 0.3, 20 particles per leaf,
512 per i-group), through the public entry points:

    noalloc   eval_noalloc: one evaluation from host arrays to host arrays
    resident  Resident.run + results: an evaluation whose inputs stay in HBM
    step      a time step with the particles in HBM: GpuTree.update,
              Resident.refill, run, results
    ngb       the neighbour search of a time step: pth_gtree_update,
              pth_gtree_neighbors and the lists' download
    hooks     the FDPS multi-walk hooks as PeTar drives them: pth_send_j, then
              batches of at most 200 walks through pth_dispatch and
              pth_retrieve, records and lists in host memory
    copies    the hooks without the multi-walk index: every walk comes with
              its own copies of its records (pth_dispatch_copies)
    serve     Server.replay of one request for each of many clusters that
              arrive at once, and their results

The interaction lists that FDPS would hand to the hooks are made here, in
torch: an octree (`octree`), its i-groups and the group walk (`lists`).
`exact` sums the same lists pair by pair in FP64.
"""
import ctypes as C
import math

import numpy as np
import torch

from petar_amd import soft_force as sf

THETA, N_LEAF, N_GROUP, LEVELS = 0.3, 20, 512, 21
N_WALK_LIMIT = 200  # walks per dispatch in PeTar
DEV = torch.device("cuda" if torch.cuda.is_available() else "cpu")
F64, I64 = dict(dtype=torch.float64, device=DEV), dict(dtype=torch.int64, device=DEV)


def _case(name, kind, n, f_bin=0.0, r_out=0.01, eps=0.0, co=0, mono=0, clusters=1):
    """n particles (serve: the largest cluster's), f_bin of them in binaries;
    eps: softening in units of r_out; co: changeover mode; mono: monopole
    superparticles."""
    c = dict(kind=kind, n=n, f_bin=f_bin, r_out=r_out, eps=eps, co=co, mono=mono, clusters=clusters)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest calls: an evaluation for a caller that may not allocate,
        # and the 16,384-particle cluster in each form that a program may hold it
        _case("noalloc_4k", "noalloc", 4096),
        _case("resident_16k", "resident", 16384),
        _case("step_16k", "step", 16384),
        _case("hooks_16k", "hooks", 16384),
        # a PeTar build without the multi-walk index and without quadrupoles
        _case("copies_16k_mono", "copies", 16384, f_bin=0.3, mono=1),
        # a service for many small clusters
        _case("serve_24", "serve", 50000, f_bin=0.3, clusters=24),
        # PeTar with the changeover correction folded in, an odd size
        _case("hooks_131k_co", "hooks", 131071, f_bin=0.5, co=1),
        # the million-particle cluster with half of its stars in binaries: the
        # neighbour search, PeTar's hooks, a time step on the device
        _case("ngb_1m", "ngb", 1048576, f_bin=0.5),
        _case("hooks_1m", "hooks", 1048576, f_bin=0.5),
        _case("step_1m", "step", 1048576, f_bin=0.5),
        # repeated changeover evaluations of a cluster of binaries
        _case("resident_1m_co", "resident", 1048576, f_bin=1.0, co=1),
        # a large production run: 4.2M stars, all in binaries, a short cutoff
        _case("step_4m", "step", 4194304, f_bin=1.0, r_out=0.003),
    ]


def draw(rng):
    kind, lo, hi = rng.choice([("noalloc", 256, 24000), ("resident", 1000, 700000), ("step", 1000, 2000000),
                               ("ngb", 1000, 2000000), ("hooks", 500, 700000), ("copies", 500, 24000),
                               ("serve", 2000, 50000)])
    n = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    return _case(None, kind, n, f_bin=rng.choice([0.0, 0.3, 0.5, 1.0]), r_out=rng.choice([0.003, 0.01]),
                 eps=rng.choice([0.0, 0.0, 0.3]), co=int(kind in ("resident", "hooks") and rng.random() < 0.4),
                 mono=int(kind in ("resident", "step", "hooks", "copies") and rng.random() < 0.25),
                 clusters=rng.randint(4, 24) if kind == "serve" else 1)


# ---------------------------------------------------------------------------
# clusters and their interaction lists


class Cluster:
    """Positions, masses, search and changeover radii (N-body units)."""

    def __init__(self, n, f_bin, r_out, seed, co=0):
        g = torch.Generator(device=DEV).manual_seed(seed)

        def u(*shape):
            return torch.rand(*shape, generator=g, **F64)

        def isotropic(k):
            z, phi = 2 * u(k) - 1, 2 * math.pi * u(k)
            s = torch.sqrt(1 - z * z)
            return torch.stack([s * torch.cos(phi), s * torch.sin(phi), z], 1)

        r = (0.001 + 0.989 * u(n)).pow(-2 / 3).sub(1).rsqrt() * (3 * math.pi / 16)
        x = r[:, None] * isotropic(n)
        # Kroupa: m^-1.3 in [0.08, 0.5], m^-2.3 above, up to 150
        a = (0.08 ** -0.3 - 0.5 ** -0.3) / 0.3
        b = 0.5 * (0.5 ** -1.3 - 150.0 ** -1.3) / 1.3
        t = u(n) * (a + b)
        low = (0.08 ** -0.3 - 0.3 * t.clamp(max=a)).pow(-1 / 0.3)
        high = (0.5 ** -1.3 - 1.3 * (t - a).clamp(min=0) / 0.5).pow(-1 / 1.3)
        m = torch.where(t < a, low, high)
        # binaries: the second star sits beside the first, separations
        # log-uniform in [1e-5, 1e-2]
        k = int(0.5 * f_bin * n)
        sep = 10 ** (-5 + 3 * u(k))
        x[k:2 * k] = x[:k] + sep[:, None] * isotropic(k)
        fac = (m / m.mean()).pow(1 / 3).clamp(min=1.0) if co else torch.ones(n, **F64)
        self.x, self.m, self.r_out = x, m / m.sum(), r_out * fac
        self.r_in, self.rs = 0.1 * self.r_out, 1.5 * self.r_out
        self.drift = 1e-4 * r_out * torch.randn(n, 3, generator=g, **F64)


class Octree:
    pass


def _spread(v):
    for s, k in ((32, 0x1f00000000ffff), (16, 0x1f0000ff0000ff), (8, 0x100f00f00f00f00f), (4, 0x10c30c30c30c30c3),
                 (2, 0x1249249249249249)):
        v = (v | v << s) & k
    return v


def _rows(begin, count, width):
    """Index rows begin[k] .. begin[k] + count[k], padded to width, and which are real."""
    j = torch.arange(width, device=DEV)
    real = j < count[:, None]
    return torch.where(real, begin[:, None] + j, begin[:, None]), real


def octree(c):
    """Cells (level by level in Morton order) with their moments and boxes,
    and the i-groups: the largest cells of at most N_GROUP particles."""
    t = Octree()
    lo, hi = c.x.amin(0), c.x.amax(0)
    side = float((hi - lo).max()) * (1 + 1e-9)
    cell = ((c.x - (0.5 * (lo + hi) - 0.5 * side)) * (2 ** LEVELS / side)).floor().long().clamp(0, 2 ** LEVELS - 1)
    key = _spread(cell[:, 0]) << 2 | _spread(cell[:, 1]) << 1 | _spread(cell[:, 2])
    key, t.order = torch.sort(key, stable=True)
    t.side, t.x, t.m, t.rs = side, c.x[t.order], c.m[t.order], c.rs[t.order]
    t.r_in, t.r_out = c.r_in[t.order], c.r_out[t.order]
    n = key.numel()
    begin, end, level = [torch.zeros(1, **I64)], [torch.full((1,), n, **I64)], [0]
    starts = [0]  # first cell of each level
    first, kids = [], []
    for l in range(LEVELS):
        b, e = begin[-1], end[-1]
        split = (e - b) > N_LEAF
        pre = key >> 3 * (LEVELS - 1 - l)
        new = torch.ones(n, dtype=torch.bool, device=DEV)
        new[1:] = pre[1:] != pre[:-1]
        cb = new.nonzero()[:, 0]
        ce = torch.cat([cb[1:], torch.full((1,), n, **I64)])
        parent = torch.searchsorted(b, cb, right=True) - 1
        keep = (parent >= 0) & split[parent] & (cb < e[parent])
        cb, ce, parent = cb[keep], ce[keep], parent[keep]
        k = torch.bincount(parent, minlength=b.numel())
        starts.append(starts[-1] + b.numel())
        kids.append(k)
        first.append(starts[-1] + torch.cumsum(k, 0) - k)
        if cb.numel() == 0:
            break
        begin.append(cb)
        end.append(ce)
        level.append(l + 1)
    if len(kids) < len(begin):
        kids.append(torch.zeros_like(begin[-1]))
        first.append(torch.zeros_like(begin[-1]))
        starts.append(starts[-1] + begin[-1].numel())
    t.level = torch.cat([torch.full_like(b, l) for b, l in zip(begin, level)])
    t.begin, t.end, t.first, t.kids = (torch.cat(v) for v in (begin, end, first, kids))
    nn = t.begin.numel()
    t.mass, t.com, t.quad = torch.zeros(nn, **F64), torch.zeros(nn, 3, **F64), torch.zeros(nn, 6, **F64)
    t.inner, t.outer = torch.zeros(nn, 6, **F64), torch.zeros(nn, 6, **F64)  # boxes: lows, highs
    big = 1e300

    def moments(at, m, p, q, inner, outer, real):
        m = torch.where(real, m, torch.zeros_like(m))
        t.mass[at] = m.sum(1)
        t.com[at] = (m[..., None] * p).sum(1) / t.mass[at][:, None]
        d = p - t.com[at][:, None]
        x, y, z = d.unbind(-1)
        s = m[..., None] * torch.stack([x * x, y * y, z * z, x * y, x * z, y * z], -1)
        if q is not None:
            s = s + torch.where(real[..., None], q, torch.zeros_like(q))
        t.quad[at] = s.sum(1)
        for box, v in ((t.inner, inner), (t.outer, outer)):
            box[at, :3] = torch.where(real[..., None], v[..., :3], torch.full_like(p, big)).amin(1)
            box[at, 3:] = torch.where(real[..., None], v[..., 3:], torch.full_like(p, -big)).amax(1)

    for l in range(len(begin) - 1, -1, -1):
        at = torch.arange(starts[l], starts[l + 1], device=DEV)
        leaf = t.kids[at] == 0
        for sel, is_leaf in ((at[leaf], True), (at[~leaf], False)):
            for s in sel.split(1 << 19) if sel.numel() else ():
                if is_leaf:
                    size = t.end[s] - t.begin[s]
                    i, real = _rows(t.begin[s], size, int(size.max()))
                    p, rs = t.x[i], t.rs[i][..., None]
                    moments(s, t.m[i], p, None, torch.cat([p, p], -1), torch.cat([p - rs, p + rs], -1), real)
                else:
                    i, real = _rows(t.first[s], t.kids[s], 8)
                    moments(s, t.mass[i], t.com[i], t.quad[i], t.inner[i], t.outer[i], real)
    small = ((t.end - t.begin) <= N_GROUP) | (t.kids == 0)
    up = torch.zeros(nn, dtype=torch.bool, device=DEV)  # inside a larger group
    for l in range(len(begin) - 1):
        at = torch.arange(starts[l], starts[l + 1], device=DEV)
        i, real = _rows(t.first[at], t.kids[at], 8)
        up[i[real]] = (up | small)[at][:, None].expand_as(i)[real]
    g = (small & ~up).nonzero()[:, 0]
    t.groups = g[torch.argsort(t.begin[g])]
    return t


def _overlap(a, b):
    return ((a[:, :3] <= b[:, 3:]) & (b[:, :3] <= a[:, 3:])).all(1)


class Lists:
    """Per i-group: sizes, and the concatenated EPJ (particle) and SPJ (cell) lists."""


def lists(t, pick=None):
    """The group walk: a cell is opened when it holds the group, when it looks
    larger than THETA from the group's box, or when either box meets the other
    widened by the search radii; opened leaves give particles, closed cells
    themselves, in the order of a depth-first walk."""
    groups = t.groups if pick is None else t.groups[pick]
    gi, gc = torch.arange(groups.numel(), device=DEV), torch.zeros(groups.numel(), **I64)
    near, far = [], []
    while gi.numel():
        g = groups[gi]
        box = t.inner[g]
        p = t.com[gc]
        d = (box[:, :3] - p).clamp(min=0) + (p - box[:, 3:]).clamp(min=0)
        side = t.side * torch.pow(0.5, t.level[gc].double())
        opened = (d * d).sum(1) < side * side / THETA ** 2
        opened |= _overlap(t.outer[g], t.inner[gc]) | _overlap(box, t.outer[gc])
        opened |= (t.begin[gc] <= t.begin[g]) & (t.end[gc] >= t.end[g])
        far.append((gi[~opened], gc[~opened]))
        leaf = opened & (t.kids[gc] == 0)
        near.append((gi[leaf], gc[leaf]))
        gi, gc = gi[opened & ~leaf], gc[opened & ~leaf]
        k = t.kids[gc]
        at = torch.arange(int(k.sum()), device=DEV) - torch.repeat_interleave(torch.cumsum(k, 0) - k, k)
        gi, gc = torch.repeat_interleave(gi, k), torch.repeat_interleave(t.first[gc], k) + at

    def ordered(found):
        gi, gc = torch.cat([a for a, _ in found]), torch.cat([b for _, b in found])
        s = torch.argsort(gi * t.x.shape[0] + t.begin[gc])
        return gi[s], gc[s]

    L = Lists()
    L.tree, L.begin = t, t.begin[groups]
    L.n_epi = t.end[groups] - L.begin
    gi, gc = ordered(far)
    L.n_spj, L.spj = torch.bincount(gi, minlength=groups.numel()), gc.int()
    gi, gc = ordered(near)
    k = t.end[gc] - t.begin[gc]
    at = torch.arange(int(k.sum()), device=DEV) - torch.repeat_interleave(torch.cumsum(k, 0) - k, k)
    L.epj = (torch.repeat_interleave(t.begin[gc], k) + at).int()
    L.n_epj = torch.bincount(torch.repeat_interleave(gi, k), minlength=groups.numel())
    return L


def _sizes(case):
    """Particles of each cluster of a case."""
    k = case["clusters"]
    return [case["n"]] if k == 1 else [int(1000 * (case["n"] / 1000) ** (i / (k - 1))) for i in range(k)]


def _clusters(case, seed):
    return [Cluster(n, case["f_bin"], case["r_out"], seed * 1000 + i, case["co"]) for i, n in enumerate(_sizes(case))]


# ---------------------------------------------------------------------------
# states


_contexts = {}


def _context(case):
    """A program keeps one context per set of parameters."""
    par = dict(eps2=(case["eps"] * case["r_out"]) ** 2, rcut2=case["r_out"] ** 2, G=1.0, changeover=case["co"],
               spj_monopole=case["mono"])
    key = tuple(par.items())
    if key not in _contexts:
        _contexts[key] = sf.Context(0, **par)
    return _contexts[key]


def _host(v):
    return np.ascontiguousarray(v.cpu().numpy())


def _arrays(L):
    """The arguments of an evaluation from host arrays (Resident, eval_noalloc, Server.add)."""
    t = L.tree
    return [_host(v) for v in (L.n_epi.int(), L.n_epj.int(), L.n_spj.int(), t.x, t.rs, L.epj, L.spj, t.x, t.m, t.rs,
                               t.com, t.mass, t.quad)]


class Hooks:
    """The records, lists and pointer tables that FDPS holds for a force call."""

    def __init__(self, case, L, copies):
        t = L.tree
        n, nn = t.x.shape[0], t.com.shape[0]
        self.L, self.ctx, self.copies = sf.lib(), _context(case), copies
        self.epi, self.epj = np.zeros(n, sf.EPI_SOFT), np.zeros(n, sf.EPJ_SOFT)
        self.spj = np.zeros(nn, sf.SPJ_SOFT_MONO if case["mono"] else sf.SPJ_SOFT)
        self.force = np.zeros(n, sf.FORCE_SOFT_CO if case["co"] else sf.FORCE_SOFT)
        for r in (self.epi, self.epj):
            r["id"], r["pos"], r["r_search"] = np.arange(n), _host(t.x), _host(t.rs)
        self.epj["mass"], self.epj["r_in"], self.epj["r_out"] = _host(t.m), _host(t.r_in), _host(t.r_out)
        self.spj["pos"], self.spj["mass"] = _host(t.com), _host(t.mass)
        if not case["mono"]:
            for k, q in enumerate(("xx", "yy", "zz", "xy", "xz", "yz")):
                self.spj["quad"][q] = _host(t.quad[:, k])
        e, s, q = sf.EPJ_SOFT.fields, self.spj.dtype.fields, sf.SPJ_SOFT.fields["quad"]
        self.ev = sf.EpjView(sf.EPJ_SOFT.itemsize, *(e[k][1] for k in ("pos", "mass", "r_search", "id", "r_in", "r_out",
                                                                      "group_data")))
        self.sv = sf.SpjView(self.spj.dtype.itemsize, s["pos"][1], s["mass"][1],
                             *(0 if case["mono"] else q[1] + q[0].fields[k][1] for k in ("xx", "yy", "zz", "xy", "xz",
                                                                                        "yz")))
        i = sf.EPI_SOFT.fields
        self.iv = sf.EpiView(sf.EPI_SOFT.itemsize, i["pos"][1], i["r_search"][1], i["id"][1])
        self.fv = sf.force_view(self.force.dtype)
        self.n_epi, self.n_epj, self.n_spj = (_host(v.int()) for v in (L.n_epi, L.n_epj, L.n_spj))
        je, js = _host(L.epj), _host(L.spj)
        if copies:
            je, js = self.epj[je], self.spj[js]
        self.je, self.js = je, js

        def table(a, first):
            return (a.ctypes.data + a.itemsize * first).astype(np.uint64)

        begin = _host(L.begin)
        self.p_epi, self.p_force = table(self.epi, begin), table(self.force, begin)
        self.p_epj = table(je, np.cumsum(self.n_epj, dtype=np.int64) - self.n_epj)
        self.p_spj = table(js, np.cumsum(self.n_spj, dtype=np.int64) - self.n_spj)
        ref, vp, ip = C.byref, C.POINTER(C.c_void_p), C.POINTER(C.c_int)
        self.batches = []
        for b in range(0, self.n_epi.size, N_WALK_LIMIT):
            w = slice(b, b + N_WALK_LIMIT)
            pe, pf, pj, ps = (p[w].ctypes.data_as(vp) for p in (self.p_epi, self.p_force, self.p_epj, self.p_spj))
            ni, nj, ns = (v[w].ctypes.data_as(ip) for v in (self.n_epi, self.n_epj, self.n_spj))
            nw = self.n_epi[w].size
            if copies:
                out = (0, nw, pe, ni, ref(self.iv), pj, nj, ref(self.ev), ps, ns, ref(self.sv))
            else:
                out = (0, nw, pe, ni, ref(self.iv), pj, nj, ps, ns)
            self.batches.append((out, (0, nw, ni, pf, ref(self.fv))))

    def __call__(self):
        c, h = self.ctx, self.ctx.handle
        dispatch = self.L.pth_dispatch_copies if self.copies else self.L.pth_dispatch
        if not self.copies:
            c.check(self.L.pth_send_j(h, self.epj.ctypes.data, self.epj.size, C.byref(self.ev), self.spj.ctypes.data,
                                      self.spj.size, C.byref(self.sv)), "pth_send_j")
        for out, back in self.batches:
            c.check(dispatch(h, *out), "dispatch")
            c.check(self.L.pth_retrieve(h, *back), "pth_retrieve")
        return [self.force[k] for k in self.force.dtype.names]


class Step:
    """A tree and an evaluation kept from step to step, the particles in HBM."""

    def __init__(self, case, c):
        before = _host(c.x - c.drift)
        self.args = c.x, c.m, c.rs
        self.tree = sf.GpuTree(_context(case), before, _host(c.m), _host(c.rs), THETA, N_LEAF, N_GROUP)
        self.eval = sf.Resident.from_gtree(_context(case), self.tree)

    def __call__(self):
        self.tree.update(*self.args)
        self.eval.refill(self.tree)
        self.eval.run()
        return self.eval.results()


class Neighbours:
    """A tree kept from step to step and the arrays that a step's neighbour
    lists go to (room for twice the expected entries), through the C ABI."""

    def __init__(self, case, c):
        n = case["n"]
        self.L, self.ctx, self.c, self.h = sf.lib(), _context(case), c, C.c_void_p()
        self.room = n * (4 + math.ceil(1.2e-5 * n * (case["r_out"] / 0.01) ** 3))
        self.out = np.zeros(n, np.int32), np.zeros(n + 1, np.int64), np.full(self.room, -1, np.int32)
        dp, pos, m, rs = C.POINTER(C.c_double), _host(c.x - c.drift), _host(c.m), _host(c.rs)
        self.ctx.check(self.L.pth_gtree_build(self.ctx.handle, C.byref(self.h), n, *(a.ctypes.data_as(dp) for a in
                                              (pos, m, rs)), N_LEAF, N_GROUP, THETA, 1), "pth_gtree_build")

    def __call__(self):
        c, L, total, ms = self.ctx, self.L, C.c_longlong(), C.c_float()
        p = self.c
        c.check(L.pth_gtree_update(self.h, p.x.shape[0], p.x.data_ptr(), p.m.data_ptr(), p.rs.data_ptr(), 1),
                "pth_gtree_update")
        c.check(L.pth_gtree_neighbors(self.h, C.byref(total)), "pth_gtree_neighbors")
        if total.value > self.room:
            raise RuntimeError(f"{total.value} neighbours, room for {self.room}")
        cnt, off, ngb = (a.ctypes.data_as(C.POINTER(t)) for a, t in zip(self.out, (C.c_int, C.c_longlong, C.c_int)))
        c.check(L.pth_gtree_neighbors_download(self.h, cnt, off, ngb, C.byref(ms)), "pth_gtree_neighbors_download")
        return self.out

    def __del__(self):
        if self.ctx.handle:  # (at interpreter exit the contexts are closed first)
            self.L.pth_gtree_free(self.h)


class Evaluation:
    def __init__(self, case, L):
        a = _arrays(L)
        self.r = sf.Resident(_context(case), *a)
        if case["co"]:
            ids = np.arange(a[3].shape[0])
            self.r.changeover(ids, ids, _host(L.tree.r_in), _host(L.tree.r_out))

    def __call__(self):
        self.r.run()
        return self.r.results()


class NoAlloc:
    def __init__(self, case, L):
        self.ctx, self.args = _context(case), _arrays(L)

    def __call__(self):
        return sf.eval_noalloc(self.ctx, *self.args)


class Service:
    def __init__(self, case, ls):
        self.srv = sf.Server(_context(case), hbm_budget=4 << 30)
        self.ids = [self.srv.add(*_arrays(L)) for L in ls]

    def __call__(self):
        self.srv.replay(self.ids, np.zeros(len(self.ids)))
        return [np.concatenate(v) for v in zip(*(self.srv.results(k) for k in self.ids))]


def prepare(case, seed):
    kind, cs = case["kind"], _clusters(case, seed)
    if kind in ("step", "ngb"):
        return (Step if kind == "step" else Neighbours)(case, cs[0])
    ls = [lists(octree(c)) for c in cs]
    if kind in ("hooks", "copies"):
        return Hooks(case, ls[0], kind == "copies")
    if kind == "serve":
        return Service(case, ls)
    return (Evaluation if kind == "resident" else NoAlloc)(case, ls[0])


def run(state):
    return state()


# ---------------------------------------------------------------------------
# what a pass cannot do without, and its values in 64 bits


def _pairs(case):
    """EPJ and SPJ list entries and pairs of a case, from a sample of its groups."""
    tot = np.zeros(4)
    for c in _clusters(case, 0):
        t = octree(c)
        k = t.groups.numel()
        pick = torch.arange(0, k, max(1, k // 256), device=DEV)
        L = lists(t, pick)
        v = [L.n_epj, L.n_spj, L.n_epi * L.n_epj, L.n_epi * L.n_spj]
        tot += np.array([float(x.sum()) for x in v]) * k / pick.numel()
    return tot


def _neighbours(case):
    """Neighbours within the search radius, from a sample of the particles."""
    c = _clusters(case, 0)[0]
    pick = torch.arange(0, case["n"], max(1, case["n"] // 1024), device=DEV)
    n = 0
    for p in pick.split(64):
        d = c.x[p][:, None] - c.x
        n += int(((d * d).sum(-1) < torch.maximum(c.rs[p][:, None], c.rs) ** 2).sum())
    return n * case["n"] / pick.numel()


def work(case):
    """Each input read once, each output written once; 26 operations for an
    EPJ or monopole pair, 65 for a quadrupole SPJ pair, 10 for a neighbour."""
    n, kind = sum(_sizes(case)), case["kind"]
    if kind == "ngb":
        k = _neighbours(case)
        return dict(bytes=40 * n + 12 * n + 4 * k, flops=10 * k)
    e, s, pe, ps = _pairs(case)
    flops = 26 * pe + (26 if case["mono"] else 65) * ps
    out = (40 + 8 * case["co"]) * n
    spj = 32 if case["mono"] else 80
    if kind == "step":
        moved = 40 * n
    elif kind == "hooks":
        moved = 168 * n + spj * n / 5 + 4 * (e + s)
    elif kind == "copies":
        moved = 48 * n + 120 * e + spj * s
    elif kind == "noalloc":
        moved = 72 * n + spj * n / 5 + 4 * (e + s)
    else:  # records and lists are in HBM
        moved = 64 * n + 64 * n / 5 + 4 * (e + s)
    return dict(bytes=moved + out, flops=flops)


def _changeover(r, rin_i, rout_i, rin_j, rout_j):
    """W_acc and W_pot of a pair: the radii of the one with the larger r_out."""
    use = rout_i > rout_j
    rin, rout = torch.where(use, rin_i, rin_j), torch.where(use, rout_i, rout_j)
    xr, k = (r - rin) / (rout - rin), (rout - rin) / (rout + rin)
    x = xr.clamp(0, 1)
    acc = (x - 1) ** 4 * (1 + x * (4 + x * (10 + x * (20 + 35 * k * x))))
    pot = torch.where(xr >= 1, (1 + k) * r / rout, 1 - k * x ** 5 * (x * (x * (5 * x - 20) + 28) - 14))
    return acc, pot


def _walk(t, case, i, je, js):
    """Accelerations, potentials (and total potentials) of particles i from
    the particles je and the cells js."""
    eps2, rcut2 = (case["eps"] * case["r_out"]) ** 2, case["r_out"] ** 2
    xi = t.x[i][:, None]
    d = t.x[je] - xi
    r2, m = (d * d).sum(-1) + eps2, t.m[je]
    ri = r2.clamp(min=rcut2).rsqrt()
    f, p = m * ri ** 3, -m * ri
    pt = None
    if case["co"]:
        near = r2 - eps2 < (0.99 * torch.maximum(t.rs[i][:, None], t.rs[je])) ** 2
        own = i[:, None] == je
        one = r2.clamp(min=1e-300).rsqrt()
        wa, wp = _changeover(r2.sqrt(), t.r_in[i][:, None], t.r_out[i][:, None], t.r_in[je], t.r_out[je])
        zero = torch.zeros_like(p)
        pt = torch.where(own, zero, torch.where(near, -m * one, p))
        f = torch.where(own, zero, torch.where(near, m * one ** 3 * (1 - wa), f))
        p = torch.where(own, zero, torch.where(near, -m * one * (1 - wp), p))
    acc, pot = (f[..., None] * d).sum(1), p.sum(1)
    d = xi - t.com[js]
    r2, m = (d * d).sum(-1) + eps2, t.mass[js]
    ri = r2.rsqrt()
    if case["mono"]:
        far = -m * ri
        acc = acc - ((m * ri ** 3)[..., None] * d).sum(1)
    else:
        xx, yy, zz, xy, xz, yz = t.quad[js].unbind(-1)
        tr = xx + yy + zz
        x, y, z = d.unbind(-1)
        q = torch.stack([3 * (xx * x + xy * y + xz * z) - tr * x, 3 * (xy * x + yy * y + yz * z) - tr * y,
                         3 * (xz * x + yz * y + zz * z) - tr * z], -1)
        s = ((q * d).sum(-1) - eps2 * tr) * ri ** 4
        far = -(m + 0.5 * s) * ri
        acc = acc + (q * (ri ** 5)[..., None] - ((m + 2.5 * s) * ri ** 3)[..., None] * d).sum(1)
    far = far.sum(1)
    return acc, pot + far, None if pt is None else pt.sum(1) + far


def exact(case, seed):
    """acc, pot, None for the neighbour counts (and pot_tot), in tree order."""
    if case["kind"] == "ngb" or case["n"] > 1200000:
        return None
    out = []
    for c in _clusters(case, seed):
        t = octree(c)
        L = lists(t)
        at = [torch.cat([torch.zeros(1, **I64), v.cumsum(0)]).tolist() for v in (L.n_epi, L.n_epj, L.n_spj)]
        for w in range(L.n_epi.numel()):
            i = torch.arange(at[0][w], at[0][w + 1], device=DEV)
            je, js = L.epj[at[1][w]:at[1][w + 1]].long(), L.spj[at[2][w]:at[2][w + 1]].long()
            out.append(_walk(t, case, i, je, js))
    acc, pot = torch.cat([v[0] for v in out]), torch.cat([v[1] for v in out])
    return [acc, pot, None] + ([torch.cat([v[2] for v in out])] if case["co"] else [])
