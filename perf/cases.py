"""Timing cases: what a user of loopgpu has it do, through its Python entry points.

A case sweeps one chain, a batch of chains, a replica-exchange set, a worker or
a job server, in the sizes of the tests, the benchmark and the reference's own
published runs, from a 16-site chain asked for one sweep at a time to 20M
operators in one configuration.  Every case starts from a warm configuration
(`warm` sweeps from the all-up, operator-free start), as a measuring run does,
and returns the sweep records; `config` cases also return the configuration
they end with, as a program that checkpoints or measures correlations reads it.

The framework is counter-based: a seed fixes the whole trajectory, so the
records' counts and the configuration are the same numbers on every build.
exact() repeats the trajectory in plain numpy (S=1/2, no fields).
"""

import math
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.getcwd(), "alps-looper_amd"))
import loopgpu as lg  # noqa: E402

LATTICES = {"chain": lg.CHAIN, "square": lg.SQUARE}
BASE = dict(kind="single", lattice="chain", L=16, beta=4.0, jxy=1.0, jz=1.0, h=0.0, hx=0.0, d=0.0, two_s=1,
            sse=False, chains=1, beta_max=4.0, warm=100, sweeps=1, config=False)


def listed():
    def case(name, **kw):
        return dict(BASE, name=name, **kw)

    return [
        # a program that looks at every sweep of a small chain (correlations,
        # snapshots): one sweep a call, records and configuration
        case("chain16_step", L=16, beta=4.0, sweeps=1, config=True),
        # the worker on the 64-site chain at T=0.1: steps, binning, results
        case("worker64", kind="worker", L=64, beta=10.0, warm=512, sweeps=512),
        # the reference's two published chain runs
        case("chain128", L=128, beta=100.0, sweeps=64, config=True),
        case("chain1024", L=1024, beta=1000.0, warm=60, sweeps=16),
        # one large square lattice a GPU: the ordinary and the largest
        case("square128", lattice="square", L=128, beta=128.0, warm=60, sweeps=8),
        case("square256", lattice="square", L=256, beta=256.0, warm=30, sweeps=2),
        # the temperature scan: 512 chains on 32^2, T from 2 down to 0.05
        case("scan512", kind="batch", lattice="square", L=32, beta=0.5, beta_max=20.0, chains=512, sweeps=8),
        # replica exchange over 32 temperatures of a small lattice
        case("exchange32", kind="exchange", lattice="square", L=16, beta=0.5, beta_max=10.0, chains=32, sweeps=32),
        # spin 1 (virtual sites, boundary permutation): the Haldane chain
        case("spin1_chain64", L=64, beta=25.0, two_s=2, sweeps=32, config=True),
        # transverse-field Ising model on a square lattice (site operators)
        case("tfim32", lattice="square", L=32, beta=8.0, jxy=0.0, jz=-1.0, hx=1.0, sweeps=32, config=True),
        # the same scan with the series-expansion worker
        case("sse_scan512", kind="batch", lattice="square", L=32, beta=0.5, beta_max=20.0, chains=512, sse=True,
             warm=40, sweeps=2),
        # a handful of jobs of mixed sizes sent to the job server and waited for
        case("serve16", kind="server", L=64, beta=1.0, beta_max=64.0, chains=16, warm=32, sweeps=256),
    ]


def _even(rng, lo, hi):
    return 2 * max(1, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2))


def _logu(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["chain", "chain", "square", "square", "batch", "batch", "exchange", "spin", "field", "sse",
                       "worker"])
    c = dict(BASE)
    c["jz"] = round(rng.uniform(0.5, 1.0), 3)
    c["warm"] = rng.randrange(40, 81)
    if kind in ("chain", "worker"):
        c["L"] = _even(rng, 8, 1024)
        c["beta"] = round(_logu(rng, 1.0, 1.0 * c["L"]), 2)
        c["sweeps"] = rng.choice([1, 5, 16, 33])
        c["config"] = c["L"] <= 256 and rng.random() < 0.5
        if kind == "worker":
            c.update(kind="worker", L=min(c["L"], 128), beta=min(c["beta"], 32.0), sweeps=rng.randrange(100, 301),
                     config=False)
    elif kind == "square":
        c.update(lattice="square", L=_even(rng, 4, 160), sweeps=rng.choice([1, 3, 8]))
        c["beta"] = round(_logu(rng, 1.0, max(2.0, 1.0 * c["L"])), 2)
        c["config"] = c["L"] <= 32 and rng.random() < 0.5
    elif kind in ("batch", "sse"):
        sq = rng.random() < 0.7
        c.update(kind="batch", lattice="square" if sq else "chain", L=_even(rng, 6, 32) if sq else _even(rng, 8, 128),
                 beta=round(rng.uniform(0.4, 1.0), 3), beta_max=round(_logu(rng, 2.0, 20.0), 3),
                 chains=round(_logu(rng, 2, 384)), sse=kind == "sse", sweeps=rng.choice([1, 2, 5]))
    elif kind == "exchange":
        sq = rng.random() < 0.5
        c.update(kind="exchange", lattice="square" if sq else "chain", L=_even(rng, 4, 24) if sq else _even(rng, 8, 128),
                 beta=round(rng.uniform(0.4, 1.0), 3), beta_max=round(_logu(rng, 2.0, 12.0), 3),
                 chains=rng.randrange(2, 49), sweeps=rng.randrange(4, 33))
    elif kind == "spin":
        sq = rng.random() < 0.4
        c.update(lattice="square" if sq else "chain", L=_even(rng, 4, 16) if sq else _even(rng, 8, 96),
                 beta=round(_logu(rng, 1.0, 20.0), 2), two_s=rng.choice([2, 2, 3, 4]), sweeps=rng.randrange(4, 25),
                 config=True)
        if rng.random() < 0.3:
            c["d"] = -0.25
    else:
        sq = rng.random() < 0.5
        c.update(lattice="square" if sq else "chain", L=_even(rng, 4, 40) if sq else _even(rng, 8, 256),
                 beta=round(_logu(rng, 1.0, 12.0), 2), sweeps=rng.randrange(4, 25), config=True)
        if rng.random() < 0.5:  # transverse field on a sign-free model
            c.update(jxy=0.0, jz=-1.0, hx=round(rng.uniform(0.3, 2.0), 2))
        else:                   # magnetisation curve: longitudinal field
            c["h"] = round(rng.uniform(0.1, 1.0), 2)
    return c


# ---------------------------------------------------------------------------
# the work in hand, and one pass
# ---------------------------------------------------------------------------
def _params(c, seed, beta=None, chain_id=0):
    return lg.params(LATTICES[c["lattice"]], c["L"], c["beta"] if beta is None else beta, c["jxy"], c["jz"],
                     seed=seed & 0xFFFFFFFF, chain_id=chain_id, h=c["h"], two_s=c["two_s"], hx=c["hx"], d=c["d"],
                     algorithm=lg.SSE if c["sse"] else lg.PATH_INTEGRAL)


def _betas(c):
    """inverse temperatures of a batch, geometric from beta to beta_max"""
    n = c["chains"]
    return [c["beta"] * (c["beta_max"] / c["beta"]) ** (i / max(1, n - 1)) for i in range(n)]


# the serving mix's kinds up to 48^2, in turn; inverse temperatures in [1, beta_max]
_JOB_KINDS = [("chain", 64), ("square", 16), ("chain", 256), ("square", 32), ("square", 48)]


def _jobs(c):
    for i in range(c["chains"]):
        lattice, L = _JOB_KINDS[i % len(_JOB_KINDS)]
        yield dict(c, lattice=lattice, L=L, beta=1.0 + (c["beta_max"] - 1.0) * (0.5 + 7 * i % c["chains"]) / c["chains"])


_RESULTS = ["Energy", "Energy Density", "Susceptibility", "Staggered Susceptibility", "Staggered Magnetization^2",
            "Stiffness", "Number of Clusters"]


def prepare(case, seed):
    c = case
    if c["kind"] == "single":
        obj = lg.Chain(_params(c, seed))
        obj.sweep(c["warm"])
    elif c["kind"] == "batch":
        obj = lg.Batch([_params(c, seed, b, i) for i, b in enumerate(_betas(c))])
        obj.set_graph(True)
        obj.run(c["warm"])
    elif c["kind"] == "exchange":
        obj = lg.Exchange(_params(c, seed), _betas(c), seed=seed & 0xFFFFFFFF)
        obj.set_graph(True)
        obj.run(c["warm"])
    elif c["kind"] == "worker":
        obj = lg.Worker({"LATTICE": c["lattice"] + " lattice", "L": c["L"], "T": 1.0 / c["beta"], "Jxy": c["jxy"],
                         "Jz": c["jz"], "SEED": seed & 0x7FFFFFFF, "THERMALIZATION": c["warm"], "SWEEPS": 1 << 30})
        obj.run(c["warm"])
    else:
        obj = lg.Server(max_jobs=64, max_sites=1 << 17, max_bonds=1 << 18, max_ops=16 << 20, max_cand=16 << 20)
    return {"case": c, "seed": seed, "obj": obj}


# a record's fields by kind: whole numbers, then sums of like size
_COUNTS = [lg.REC_FIELDS.index(n) for n in ("n_op", "n_clusters", "sweep", "sign")]
_GROUPS = {"sums": ("energy", "beta", "umag0", "smag0", "umag_a", "smag_a", "e_field"),
           "squares0": ("usize2", "umag2", "ssize2", "smag2"),
           "squares": ("usize", "umag", "ssize", "smag"),
           "winding": ("w2",),
           "fourths": ("usize4", "umag4", "ssize4", "smag4")}


def _columns(rec):
    out = {n: rec[..., [lg.REC_FIELDS.index(f) for f in fields]] for n, fields in _GROUPS.items()}
    out["counts"] = rec[..., _COUNTS].astype(np.int64)
    return out


def _config(c, config):
    """spins, bond offsets, times and types, the operators' arrays filled up to
    a length of the case's own"""
    spins, bo, times, types = config
    room = 2 * math.ceil(_ops(c, c["beta"])) + 1024 - len(times)
    return [spins, bo, np.pad(times, (0, room)), np.pad(types, (0, room))]


def run(state):
    c, obj = state["case"], state["obj"]
    if c["kind"] == "single":
        out = _columns(obj.sweep(c["sweeps"]))
        if c["config"]:
            out["config"] = _config(c, obj.get_config())
        return out
    if c["kind"] == "batch":
        return _columns(obj.run(c["sweeps"]))
    if c["kind"] == "exchange":
        out = _columns(obj.run(c["sweeps"]))
        out["chain_at"], accepted, out["steps"] = obj.state()
        out["accepted"] = accepted.astype(np.int64)
        return out
    if c["kind"] == "worker":
        obj.run(c["sweeps"])
        return [np.array([obj.result(n)[:2] for n in _RESULTS])]
    ids = [obj.submit(_params(j, state["seed"], None, i), c["sweeps"], c["warm"]) for i, j in enumerate(_jobs(c))]
    res = [obj.wait(i) for i in ids]
    return [np.array([[r["mean"][o] for o in lg.JOB_OBS] for r in res]),
            np.array([[r["error"][o] for o in lg.JOB_OBS] for r in res])]


def _ops(c, beta):
    """expected operators of one chain: beta per bond times (offset - bond
    energy), from the saturation of the antiferromagnet's energy with beta"""
    n, nb = lg.lattice_size(LATTICES[c["lattice"]], c["L"], c["two_s"], 0.0, 0.0)
    jxy, jz = abs(c["jxy"]), abs(c["jz"])
    off = max(jxy, jz) / 4
    e = (0.443 if c["lattice"] == "chain" else 0.335) * max(jxy, jz) * beta / (beta + 0.8)
    return nb * beta * (off + (e if jxy > 0 else jz / 4)) + n * beta * abs(c["hx"]) * 0.75


def work(case):
    """bytes: a sweep reads one configuration and writes the next, 12 bytes an
    operator (time, bond and type) each way, and a spin a site; the records go
    out.  flops: about 200 operations an operator (its counter-based random
    words, logarithm, two spin look-ups and its place in two world lines)."""
    c = case
    if c["kind"] in ("batch", "exchange"):
        ops = sum(_ops(c, b) for b in _betas(c))
    elif c["kind"] == "server":
        ops = sum(_ops(j, j["beta"]) for j in _jobs(c))
    else:
        ops = _ops(c, c["beta"])
    n = c["sweeps"] + (c["warm"] if c["kind"] == "server" else 0)
    recs = 8 * lg.REC_SIZE * (c["chains"] if c["kind"] in ("batch", "exchange", "server") else 1)
    return {"bytes": n * (24.0 * ops + recs), "flops": n * 200.0 * ops}


# ---------------------------------------------------------------------------
# the same trajectory in plain numpy (S=1/2 without fields)
# ---------------------------------------------------------------------------
_GRID = 1 << 52


def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 on uint64 arrays holding 32-bit words"""
    m = np.uint64(0xFFFFFFFF)
    s = np.uint64(32)
    c0, c1, c2, c3 = (np.asarray(x, np.uint64) for x in np.broadcast_arrays(c0, c1, c2, c3))
    for r in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c0, np.uint64(0xCD9E8D57) * c2
        key0, key1 = np.uint64((k0 + r * 0x9E3779B9) & 0xFFFFFFFF), np.uint64((k1 + r * 0xBB67AE85) & 0xFFFFFFFF)
        c0, c1, c2, c3 = (p1 >> s) ^ c1 ^ key0, p1 & m, (p0 >> s) ^ c3 ^ key1, p0 & m
    return c0, c1, c2, c3


def _log(x):
    """the trajectory's logarithm: e ln2 + 2 atanh(s) by its Taylor series"""
    m, e = np.frexp(x)            # x = m 2^e, m in [1/2, 1)
    m, e = m * 2.0, e - 1
    big = m > 1.4142135623730951
    m, e = np.where(big, m * 0.5, m), np.where(big, e + 1, e)
    f = m - 1.0
    s = f / (2.0 + f)
    z = s * s
    p = np.full_like(z, 1.0 / 25.0)
    for k in range(23, 2, -2):
        p = p * z + 1.0 / k
    return e * 0.69314718055994530942 + (2.0 * s + 2.0 * s * (z * p))


def _weights(jxy, jz):
    jxy = abs(jxy)
    if jxy - jz > 0:
        return [max(0.0, min(jxy / 2, (jxy + jz) / 4)), max(0.0, min(jxy / 2, (jxy - jz) / 4)),
                max(0.0, -(jxy - jz) / 2), max(0.0, -(jxy + jz) / 2)]
    return [jxy / 2, 0.0, -(jxy - jz) / 2, 0.0]


def _components(n, a, b):
    """smallest node of each node's component, edges a-b"""
    lab = np.arange(n)
    while True:
        low = np.minimum(lab[a], lab[b])
        new = lab.copy()
        np.minimum.at(new, lab[a], low)
        np.minimum.at(new, lab[b], low)
        new = new[new]
        while not np.array_equal(new, new[new]):
            new = new[new]
        if np.array_equal(new, lab):
            return lab
        lab = new


class _Numpy:
    def __init__(self, c, seed):
        L = c["L"]
        self.key = (seed & 0xFFFFFFFF, 0)
        self.beta = c["beta"]
        if c["lattice"] == "chain":
            self.s0, self.dir = np.arange(L), np.zeros(L, int)
            self.s1, gauge = (self.s0 + 1) % L, 1 - 2 * (np.arange(L) & 1)
        else:
            s = np.arange(L * L)
            x, y = s // L, s % L
            self.s0, self.dir = np.repeat(s, 2), np.tile([1, 0], L * L)
            self.s1 = np.stack([x * L + (y + 1) % L, ((x + 1) % L) * L + y], 1).reshape(-1)
            gauge = 1 - 2 * ((x + y) & 1)
        self.gauge, self.N, self.Nb = gauge, len(gauge), len(self.s0)
        v = _weights(c["jxy"], c["jz"])
        self.W = sum(v)
        last = max(g for g in range(4) if v[g] > 0)
        self.thr = [(1 << 32) if g >= last else math.floor(math.ldexp(sum(v[:g + 1]) / self.W, 32)) for g in range(3)]
        self.toff = math.floor(math.ldexp(v[0] / (v[0] + v[1]), 32)) if v[0] + v[1] > 0 else 1 << 32
        self.offset = self.Nb * self.W / 2
        lam = self.beta * self.W
        self.K = math.ceil(lam + 12 * math.sqrt(lam) + 16)
        self.sweep = 0
        self.spins = np.zeros(self.N, int)
        self.b = self.t = self.g = self.o = np.zeros(0, int)   # operators by (bond, time): bond, time, graph, off-diagonal
        self._events()

    def _events(self):
        """world lines: events by (site, time, bond) with the spin below each"""
        n = len(self.b)
        site = np.concatenate([self.s0[self.b], self.s1[self.b]])
        op, leg = np.tile(np.arange(n), 2), np.repeat([0, 1], n)
        order = np.lexsort((self.b[op], self.t[op], site))
        self.es, self.eo, self.el = site[order], op[order], leg[order]
        self.cnt = np.bincount(self.es, minlength=self.N)
        self.first = np.concatenate([[0], np.cumsum(self.cnt)])
        self.node0 = np.concatenate([[0], np.cumsum(np.maximum(self.cnt, 1))])
        off = self.o[self.eo]
        before = np.cumsum(off) - off
        start = np.concatenate([before, [0]])[self.first[self.es]]
        self.below = self.spins[self.es] ^ ((before - start) & 1)
        self.keys = (self.es.astype(np.uint64) << np.uint64(52)) + self.t[self.eo].astype(np.uint64)

    def _spin_at(self, s, t):
        """spin of site s at time t; -1 where an event has that time"""
        k = (s.astype(np.uint64) << np.uint64(52)) + t.astype(np.uint64)
        j = np.searchsorted(self.keys, k)
        keys, below = np.append(self.keys, np.uint64(0)), np.append(self.below, 0)
        tie = (j < len(self.keys)) & (keys[j] == k)
        inside = j < self.first[s + 1]
        return np.where(tie, -1, np.where(inside, below[np.minimum(j, len(self.keys))], self.spins[s]))

    def step(self):
        sw, (k0, k1) = self.sweep, self.key
        bb, kk = np.arange(self.Nb)[:, None], np.arange(self.K)[None, :]
        x, y, z, _ = _philox(sw, 1, bb, kk, k0, k1)
        u = (((x << np.uint64(21)) | (y >> np.uint64(11))) + np.uint64(1)).astype(float) * (1.0 / 9007199254740992.0)
        gap = -_log(u) * (4503599627370496.0 / (self.beta * self.W))
        T = np.cumsum(np.where(gap < 4503599627370496.0, gap, _GRID).astype(np.int64), 1)
        cb, ck = np.nonzero(T < _GRID)
        ct, cz = T[cb, ck], z[cb, ck].astype(np.int64)
        cg = sum((cz >= t).astype(int) for t in self.thr)
        c0, c1 = self._spin_at(self.s0[cb], ct), self._spin_at(self.s1[cb], ct)
        ok = (c0 >= 0) & (c1 >= 0) & (((cg & 1) ^ c0 ^ c1) != 0)
        # kept off-diagonal operators, regraphed by their rank on the bond
        keep = self.o == 1
        kb, kt = self.b[keep], self.t[keep]
        rank = np.arange(len(kb)) - np.searchsorted(kb, kb)
        kg = (_philox(sw, 2, kb, rank, k0, k1)[0].astype(np.int64) >= self.toff).astype(int)
        b, t = np.concatenate([kb, cb[ok]]), np.concatenate([kt, ct[ok]])
        g, o = np.concatenate([kg, cg[ok]]), np.concatenate([np.ones(len(kb), int), np.zeros(int(ok.sum()), int)])
        order = np.lexsort((t, b))
        self.b, self.t, self.g, self.o = b[order], t[order], g[order], o[order]
        self._events()
        # segments: node below each event, node above it (the last wraps)
        nev, M = len(self.es), int(self.node0[-1])
        rank = np.arange(nev) - self.first[self.es]
        lo = self.node0[self.es] + rank
        up = np.where(rank + 1 == self.cnt[self.es], self.node0[self.es], lo + 1)
        legs = np.zeros((4, len(self.b)), int)   # l0, l1, u0, u1
        legs[self.el, self.eo], legs[2 + self.el, self.eo] = lo, up
        l0, l1, u0, u1 = legs
        par, cross, frz = self.g == 0, self.g == 1, self.g >= 2
        a = np.concatenate([l0[par], u0[par], l0[cross], l1[cross], l0[frz], u0[frz], l0[frz]])
        e = np.concatenate([l1[par], u1[par], u1[cross], u0[cross], l1[frz], u1[frz], u0[frz]])
        root = _components(M, a, e)
        flip = (_philox(sw, 3, np.arange(M), 0, k0, k1)[0].astype(int) & 1)[root]
        # segment lengths, spins, tau = 0 segments, windings
        site = np.repeat(np.arange(self.N), np.maximum(self.cnt, 1))
        head = self.node0[:-1]
        hi, spin = np.full(M, float(_GRID)), self.spins[site].copy()
        hi[lo], spin[lo] = self.t[self.eo], self.below
        low = np.zeros(M)
        low[up] = self.t[self.eo]
        low[head] -= np.where(self.cnt > 0, float(_GRID), 0.0)
        length = (hi - low) / _GRID
        sig = 1 - 2 * spin
        src = self.el == 0
        dw = np.zeros((2, M))
        d = self.dir[self.b[self.eo]]
        np.add.at(dw, (d[src], lo[src]), sig[lo[src]])
        np.add.at(dw, (d[src], up[src]), -sig[up[src]])

        def per(w):
            return np.bincount(root, w, minlength=M)[np.unique(root)]

        gs = self.gauge[site]
        at0 = np.zeros(M)
        at0[head] = 1.0
        us0, um0, ss0, sm0 = (per(0.5 * at0 * w) for w in (np.ones(M), sig, gs, gs * sig))
        us, um, ss, sm = (per(0.5 * length * w) for w in (np.ones(M), sig, gs, gs * sig))
        w2 = sum(float((0.25 * per(w) ** 2).sum()) for w in dw)
        nop = len(self.b)
        rec = [nop, len(us), self.offset - nop / self.beta, um0.sum(), (us0 ** 2).sum(), (um0 ** 2).sum(),
               (us0 ** 4).sum(), (um0 ** 4).sum(), (us ** 2).sum(), (um ** 2).sum(), sm0.sum(), (ss0 ** 2).sum(),
               (sm0 ** 2).sum(), (ss0 ** 4).sum(), (sm0 ** 4).sum(), (ss ** 2).sum(), (sm ** 2).sum(), w2, self.beta,
               sw, um.sum(), sm.sum(), 0.0, 1.0]
        # flip clusters
        self.o = self.o ^ flip[l0] ^ flip[u0]
        self.spins = self.spins ^ flip[head]
        self._events()
        self.sweep += 1
        return rec

    def config(self):
        bo = np.concatenate([[0], np.cumsum(np.bincount(self.b, minlength=self.Nb))])
        return [self.spins.astype(np.int32), bo.astype(np.int32), self.t / float(_GRID),
                (self.o | (self.g << 2)).astype(np.int32)]


def exact(case, seed):
    c = case
    if c["kind"] != "single" or c["two_s"] != 1 or c["h"] or c["hx"] or c["d"] or c["sse"]:
        return None
    if (c["warm"] + c["sweeps"]) * (_ops(c, c["beta"]) + 300) > 3e6:
        return None
    m = _Numpy(c, seed)
    for _ in range(c["warm"]):
        m.step()
    out = _columns(np.array([m.step() for _ in range(c["sweeps"])]))
    if c["config"]:
        out["config"] = _config(c, m.config())
    return out
