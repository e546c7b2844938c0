"""The measured workloads: what a program that uses this library has it do.

Every case is one pass through the public Python binding (2degas_amd.hip):
batched local-energy evaluations, VMC blocks, single-electron sweeps (alone
and packed), reptation moves and DMC steps, and the single configuration a
Fortran host sends through the host-pointer call.  Sizes are those of
bench.py, of the tests and of the job service; decks come from the
repository's deck generator.

A case's `kind` is one of
  host  Context.eval: host arrays in and out (the drop-in driver's call)
  eval  Context.eval_device on a batch resident on the GPU
  vmc   a block of all-electron VMC steps (Walkers.sweep), as the job service
        queues it
  sem   an inverse refresh (without backflow), single-electron sweeps and,
        with "energy", the evaluation that gives their local energy
  pack  one packed sweep of several jobs of different N
  rmc   reptation moves of a set of reptiles
  dmc   DMC steps: move, weight, branching, copies
"""
import functools
import importlib
import math
import tempfile

import numpy as np
import torch

hip = importlib.import_module("2degas_amd.hip")
decks = importlib.import_module("2degas_amd.deck")
deckgen = importlib.import_module("2degas_amd.deckgen")

DEFAULT = dict(nup=29, ndown=29, rs=5.0, shells=60, jastrow="n26", u3=True, backflow="yk", ntwists=0, walkers=256)


def _case(name, kind, **kw):
    return dict(DEFAULT, name=name, kind=kind, **kw)


def listed():
    return [
        # the drop-in Fortran driver: one walker of the shipped deck's shape
        # (13+13, twisted boundary conditions) per compute_properties call
        _case("host_n26_twist_w1", "host", nup=13, ndown=13, rs=1.0, ntwists=4, walkers=1),
        # the plain method: VMC of N=26, u2 only, no backflow, 256 walkers
        _case("vmc_n26_plain_w256", "vmc", nup=13, ndown=13, u3=False, backflow="zero", steps=20, delta=0.2),
        # a served job: N=74 with backflow, 256 walkers, blocks of 20 steps
        _case("vmc_n74_job_w256", "vmc", nup=37, ndown=37, rs=2.0, jastrow="pade", steps=20),
        # the headline: N=122, u2 + u3 + backflow, 900 k-vectors, 4096 walkers
        _case("eval_n122_w4096", "eval", nup=61, ndown=61, rs=10.0, shells=200, walkers=4096, mixed=False),
        # the same batch in the mixed-precision evaluation
        _case("eval_n122_mixed_w4096", "eval", nup=61, ndown=61, rs=10.0, shells=200, walkers=4096, mixed=True),
        # twist averaging of a polarized system: complex orbitals, one spin
        _case("eval_n61_polarized_twist_w1024", "eval", nup=61, ndown=0, rs=10.0, shells=200, ntwists=4, walkers=1024,
              mixed=False),
        # single-electron sweeps of the large plain system, FP64 inverses
        _case("sem_n122_fp64_w4096", "sem", nup=61, ndown=61, rs=1.0, shells=200, jastrow="pade", u3=False,
              backflow="zero", walkers=4096, sweeps=2, sigma=0.6, mixed=False, energy=True),
        # the same moves with FP32 inverses at N=58 with u3, K = 232 moves
        # between refreshes
        _case("sem_n58_fp32_w2048", "sem", jastrow="pade", backflow="zero", walkers=2048, sweeps=4, sigma=0.5,
              mixed=True, energy=False),
        # 12 small jobs of the service moved in packed launches
        _case("pack12_n26to74_w256", "pack", shells=12, jastrow="pade", u3=False, backflow="zero", jobs=12, sigma=0.5),
        # single-electron moves with backflow: each one evaluates log|psi|
        _case("sem_n58_backflow_w512", "sem", jastrow="pade", backflow="gauss", walkers=512, sweeps=1, sigma=0.5,
              mixed=False, energy=False),
        # reptation: 512 reptiles of 200 beads
        _case("rmc_n58_r512_b200", "rmc", walkers=512, beads=200, mdelta=4, moves=4, delta=0.01),
        # DMC of the large system with fixed-population branching
        _case("dmc_n122_w4096", "dmc", nup=61, ndown=61, rs=10.0, shells=200, walkers=4096, steps=2),
    ]


# closed shells of plane waves in a square box: the electron counts per spin
# that 2D electron gas work uses; a few open ones are drawn too
SHELLS = (1, 5, 9, 13, 21, 25, 29, 37, 45, 49, 57, 61)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["eval", "eval", "eval", "vmc", "vmc", "sem", "sem", "host", "dmc", "rmc", "pack"])
    nup = rng.choice(SHELLS[1:]) if rng.random() < 0.8 else rng.randint(3, 64)
    ndown = rng.choice([nup, nup, nup, 0, rng.choice(SHELLS)])
    n = nup + ndown
    # densities at which psi^2 of the generator's Jastrow does not underflow
    c = dict(DEFAULT, kind=kind, nup=nup, ndown=ndown, rs=round(rng.uniform(1.0, 1.0 + 90.0 / n), 2),
             shells=_log_int(rng, 12, 120), jastrow="pade", u3=rng.random() < 0.6,
             backflow=rng.choice(["yk", "yk", "gauss", "zero"]), ntwists=rng.choice([0, 0, 4]))
    # walkers: log-uniform, the work no more than that of 4096 walkers of N=122
    most = min(4096, int(4096 * (122.0 / n) ** 2))
    c["walkers"] = _log_int(rng, 1, most)
    if kind == "host":
        c["walkers"] = _log_int(rng, 1, 64)
    elif kind == "eval":
        c["mixed"] = rng.random() < 0.3
    elif kind == "vmc":
        c.update(walkers=max(1, c["walkers"] // 8), steps=rng.randint(2, 8))
    elif kind == "sem":
        c.update(backflow="zero", sweeps=rng.randint(1, 2), sigma=round(rng.uniform(0.3, 0.7), 2),
                 mixed=rng.random() < 0.4, energy=rng.random() < 0.5, walkers=max(1, c["walkers"] // 2))
    elif kind == "pack":
        c.update(shells=12, u3=False, backflow="zero", ntwists=0, jobs=rng.randint(2, 12), sigma=0.5,
                 walkers=_log_int(rng, 16, 256))
    elif kind == "rmc":
        c.update(nup=29, ndown=29, shells=rng.randint(20, 60), walkers=_log_int(rng, 4, 256), beads=rng.randint(12, 60),
                 mdelta=rng.randint(1, 5), moves=rng.randint(1, 3), delta=0.01)
    else:
        c.update(walkers=max(2, c["walkers"] // 2), steps=1)
    return c


# ---------------------------------------------------------------------------
# inputs

@functools.lru_cache(maxsize=64)
def _deck(nup, ndown, rs, shells, jastrow, u3, backflow, ntwists):
    """The deck of a system, written by the generator and read back."""
    with tempfile.TemporaryDirectory() as tmp:
        deckgen.make_deck(tmp, "perf", nup, ndown, rs, shells, jastrow=jastrow, u3=u3, backflow=backflow,
                          ntwists=ntwists)
        return decks.read_deck(tmp)


def _deck_of(case):
    return _deck(*(case[k] for k in ("nup", "ndown", "rs", "shells", "jastrow", "u3", "backflow", "ntwists")))


def _twist(case):
    return (1, 2) if case["ntwists"] else (1, 1)


def _pack_cases(case):
    """The jobs of a packed case: closed shells in turn."""
    return [dict(case, kind="sem", nup=m, ndown=m, rs=float(1 + q), sweeps=1, mixed=False, energy=False)
            for q, m in ((k % 4, (13, 21, 29, 37)[k % 4]) for k in range(case["jobs"]))]


def _grids(case, nw, rng):
    """Electrons on a jittered grid that fills the box: every configuration
    takes its sites in random order."""
    n = case["nup"] + case["ndown"]
    side = _deck_of(case).el[0]
    a = math.ceil(math.sqrt(n))
    b = math.ceil(n / a)
    gx, gy = np.meshgrid((np.arange(a) + 0.5) / a - 0.5, (np.arange(b) + 0.5) / b - 0.5, indexing="ij")
    sites = np.stack([gx.ravel(), gy.ravel()], 1) * side
    order = np.argsort(rng.random((nw, len(sites))), axis=1)[:, :n]
    return sites[order] + rng.normal(0.0, 0.15 * side / a, (nw, n, 2))


def _configs(case, seed):
    """Starting configurations.  A walk hardly ever meets the nodes (psi^2
    vanishes there), where the drift diverges: of two grids per walker the one
    further from a node is taken."""
    nw = case["walkers"]
    x = _grids(case, 2 * nw, np.random.default_rng([seed, case["nup"], case["ndown"]])).reshape(nw, 2, -1, 2)
    near = _System(case).near_node(_dev(x.reshape(2 * nw, -1, 2))).cpu().numpy().reshape(nw, 2)
    return np.ascontiguousarray(x[np.arange(nw), np.argmin(near, axis=1)])


def _streams(case, seed):
    """One 48-bit generator state per walker."""
    rng = np.random.default_rng([seed, 48])
    return rng.integers(0, 1 << 47, case["walkers"], dtype=np.int64) * 2 + 1


def _delta(case):
    return case.get("delta") or case["rs"] ** 2 / (case["nup"] + case["ndown"])


def _dmc_delta(case):
    return 0.05 * case["rs"] ** 2 / (case["nup"] + case["ndown"])


# ---------------------------------------------------------------------------
# the measured path

def _walkers(case, seed):
    ctx = hip.Context(_deck_of(case), twist=_twist(case))
    return ctx, hip.Walkers(ctx, _configs(case, seed), _streams(case, seed))


def _single(case, seed):
    ctx, wk = _walkers(case, seed)
    wk.start()
    sm = hip.SingleMoves(wk, precision=1 if case["mixed"] else 0)
    return ctx, wk, sm


def prepare(case, seed):
    kind, st = case["kind"], {"case": case}
    if kind == "host":
        st["ctx"] = hip.Context(_deck_of(case), twist=_twist(case))
        st["x"] = _configs(case, seed)
    elif kind == "eval":
        ctx = st["ctx"] = hip.Context(_deck_of(case), twist=_twist(case))
        x = st["x"] = torch.tensor(_configs(case, seed), device="cuda")
        nw = x.shape[0]
        st["props"] = x.new_zeros((nw, ctx.info["n_props"]))
        st["g"] = torch.zeros_like(x)
        st["h"] = x.new_zeros((nw, 2))
        st["grad2"] = x.new_zeros(nw)
        st["status"] = torch.zeros(nw, dtype=torch.int32, device="cuda")
    elif kind == "vmc":
        st["ctx"], st["wk"] = _walkers(case, seed)
        st["wk"].start(delta=_delta(case))
    elif kind == "sem":
        st["ctx"], st["wk"], st["sm"] = _single(case, seed)
    elif kind == "pack":
        st["jobs"] = [_single(c, seed + 1000 * k) for k, c in enumerate(_pack_cases(case))]
        for _, _, sm in st["jobs"]:
            sm.refresh()
    elif kind == "rmc":
        d = _deck_of(case)
        ctx = st["ctx"] = hip.Context(d, twist=_twist(case))
        x0 = _configs(case, seed)
        rng = np.random.default_rng([seed, 7])
        # a path starts as its configuration, every bead a little displaced
        jitter = rng.standard_normal((len(x0), case["beads"]) + x0.shape[1:], dtype=np.float32) * np.float32(0.002)
        st["prm"] = hip.rmc_params(case["delta"], -0.3, 1e30, 1e30, case["beads"] // 10, case["mdelta"])
        st["rep"] = hip.Reptiles(ctx, len(x0), case["beads"], case["mdelta"], _streams(case, seed))
        st["rep"].start(x0[:, None] + jitter, st["prm"])
    elif kind == "dmc":
        st["ctx"], st["wk"] = _walkers(case, seed)
        wk = st["wk"]
        wk.start(delta=_dmc_delta(case))
        st["dm"] = hip.Dmc(wk, [3535, 3467, 3262, 1549])
        st["etrial"] = round(float(wk.props[:, st["ctx"].info["jetot"] - 1].median().item()), 3)
    return st


def _fixed_phase(case):
    # grad2_ph is the fixed-phase term |Im grad log D|^2: zero where the
    # orbitals are real up to a phase (untwisted, every plane wave with its
    # opposite: odd counts), where the buffer holds rounding noise (some 1e-25)
    # and the energy slots do not contain it
    return case["ntwists"] != 0 or any(m and m % 2 == 0 for m in (case["nup"], case["ndown"]))


def _walker_outputs(case, wk):
    out = dict(x=wk.x, g=wk.g, h=wk.h, props=wk.props, age=wk.age, rng=wk.rng, blk=wk.blk)
    if _fixed_phase(case):
        out["grad2"] = wk.grad2
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "host":
        out = state["ctx"].eval(state["x"])
        if not _fixed_phase(case):
            del out["grad2_ph"]
        return out
    if kind == "eval":
        state["ctx"].eval_device(state["x"], state["props"], state["g"], state["h"], state["grad2"], state["status"],
                                 precision=1 if case["mixed"] else 0, stream=torch.cuda.current_stream())
        return {k: state[k] for k in ("props", "g", "h", "status") + (("grad2",) if _fixed_phase(case) else ())}
    if kind == "vmc":
        wk = state["wk"]
        wk.blk.zero_()
        wk.sweep(case["steps"], _delta(case), mage=50)
        return _walker_outputs(case, wk)
    if kind == "sem":
        wk, sm = state["wk"], state["sm"]
        if sm.updates:
            sm.refresh()
        for _ in range(case["sweeps"]):
            sm.sweep(case["sigma"])
        out = dict(x=wk.x, rng=wk.rng, dlogpsi=sm.dlogpsi, nacc=sm.nacc)
        if sm.updates:
            out["ainv"] = sm.ainv
        if case["energy"]:
            wk.start()
            out.update(props=wk.props, g=wk.g, h=wk.h)
            if _fixed_phase(case):
                out["grad2"] = wk.grad2
        elif not sm.updates:
            out["ltf"] = wk.props[:, wk.ctx.info["jltf"] - 1]
        return out
    if kind == "pack":
        hip.sem_moves_packed([(sm, 0, wk.ctx.deck.nptot, case["sigma"]) for _, wk, sm in state["jobs"]])
        return [dict(x=wk.x, rng=wk.rng, ainv=sm.ainv, dlogpsi=sm.dlogpsi, nacc=sm.nacc) for _, wk, sm in state["jobs"]]
    if kind == "rmc":
        rep = state["rep"]
        rep.sweep(case["moves"], state["prm"])
        out = {k: getattr(rep, k) for k in ("x", "g", "props", "age", "w", "ends", "rage", "pp_old", "rng", "blk")}
        if _fixed_phase(case):
            out["grad2"] = rep.grad2
        return out
    wk, dm = state["wk"], state["dm"]
    wk.blk.zero_()
    dm.sweep(case["steps"], _dmc_delta(case), state["etrial"])
    return dict(_walker_outputs(case, wk), wate=dm.wate, wsum=dm.wsum, src=dm.src, rng2=dm.rng2, counts=dm.counts)


# ---------------------------------------------------------------------------
# work of one pass

def _eval_work(case):
    """(bytes, flops) of one local-energy evaluation: the determinant's
    inverse and, with backflow, F and the cross term; pair terms; rho_k."""
    spins = [m for m in (case["nup"], case["ndown"]) if m]
    n, nk = sum(spins), len(_deck_of(case).kvec)
    z = 4 if case["ntwists"] else 1  # complex orbitals
    fl = sum(2.0 * z * m ** 3 for m in spins)
    if case["backflow"] != "zero":
        fl += sum(4.0 * z * m ** 3 + 8.0 * n * m * m for m in spins)
    fl += (160.0 if case["u3"] else 80.0) * n * (n - 1) / 2 + 4.0 * n * nk
    return 8.0 * (4 * n + 2 * nk * 2 + 20), fl


def work(case):
    kind, nw = case["kind"], case["walkers"]
    if kind == "pack":
        w = [work(c) for c in _pack_cases(case)]
        # the inverses are in hand
        sub = [2.0 * c["walkers"] * 2 * c["nup"] ** 3 for c in _pack_cases(case)]
        return {"bytes": sum(a["bytes"] for a in w), "flops": sum(a["flops"] for a in w) - sum(sub)}
    by, fl = _eval_work(case)
    if kind in ("host", "eval"):
        return {"bytes": by * nw, "flops": fl * nw}
    if kind in ("vmc", "dmc"):
        return {"bytes": 2 * by * nw, "flops": fl * nw * case["steps"]}
    if kind == "rmc":
        evals = nw * case["moves"] * (case["mdelta"] + 1) / 2
        return {"bytes": by * evals, "flops": fl * evals}
    spins = [m for m in (case["nup"], case["ndown"]) if m]
    n, z = sum(spins), 4 if case["ntwists"] else 1
    if case["backflow"] != "zero":
        # every move: the pair sums and the determinants' pivots
        per = sum(2.0 / 3 * z * m ** 3 for m in spins) + 80.0 * n * (n - 1) / 2
        return {"bytes": 16.0 * n * nw, "flops": per * n * case["sweeps"] * nw}
    item = 8 if case["mixed"] else 16
    per = sum(m * (3.0 * z * m * m + 60.0 * n) for m in spins)
    flops = nw * (sum(2.0 * z * m ** 3 for m in spins) + case["sweeps"] * per + (fl if case["energy"] else 0))
    return {"bytes": nw * (sum(item * m * m for m in spins) + (by if case["energy"] else 0)), "flops": flops}


# ---------------------------------------------------------------------------
# 64-bit values in plain torch

DEV = "cuda" if torch.cuda.is_available() else "cpu"
LCG, MASK = 34522712143931, (1 << 48) - 1


def _dev(a):
    return torch.tensor(np.asarray(a, dtype=np.float64), device=DEV)


class _System:
    """The trial function and potential of a deck as plain tensors."""

    def __init__(self, case):
        d = self.deck = _deck_of(case)
        self.np = [int(v) for v in d.np]
        self.n = sum(self.np)
        self.el, self.drt, self.hb = float(d.el[0]), d.drt, [float(v) for v in d.hbs2m]
        t = [k - 1 for k in (d.iu2[0], d.iu3[0], d.iub[0], d.iv2[0])]
        self.u2, self.u3, self.b, self.v = (_dev(d.tables[k].coef) if k >= 0 else None for k in t)
        self.vt = d.tables[t[3]]
        self.vk = _dev(self.vt.vk)
        self.kvec = _dev(d.kvec)
        self.ntheta = d.ntheta
        i, j = _twist(case)
        self.gvec = _dev(hip.twist_gvec(d.kvec, d.el, d.ntheta, i, j))
        self.type = torch.tensor(sum(([t] * m for t, m in enumerate(self.np)), []), device=DEV)
        self.spins = [(sum(self.np[:t]), m) for t, m in enumerate(self.np)]

    def spline(self, tab, r):
        """Value and two derivatives of a table's cubic at r."""
        i = (r / self.drt).long()
        t = r / self.drt - i
        c = tab[i.clamp(max=tab.shape[0] - 1)]
        a, b, e, f = c.unbind(-1)
        return (a + t * (b + t * (e + t * f)), (b + t * (2 * e + 3 * t * f)) / self.drt,
                (2 * e + 6 * t * f) / self.drt ** 2)

    def pairs(self, x):
        """u = x_i - x_j (minimum image), r and the unit vectors; the
        diagonal has r = 1 and a zero mask."""
        u = x[:, :, None] - x[:, None]
        u = u - self.el * torch.round(u / self.el)
        eye = torch.eye(x.shape[1], device=DEV, dtype=torch.float64)
        r = torch.sqrt((u * u).sum(-1) + eye)
        return u, r, u / r[..., None], 1.0 - eye

    def orbitals(self, q, g):
        return torch.exp(1j * (g @ q.transpose(1, 2)))  # [w][orbital][particle]

    def jastrow(self, x):
        """Exponent U of psi = D exp(-U), without derivatives."""
        u, r, _, off = self.pairs(x)
        val = 0.5 * (off * self.spline(self.u2, r)[0]).sum((1, 2))
        if self.u3 is not None:
            xi = off * self.spline(self.u3, r)[0]
            gp = (xi[..., None] * u).sum(2)
            val = val + 0.5 * ((xi * r) ** 2).sum((1, 2)) - 0.5 * (gp * gp).sum((1, 2))
        return val

    def near_node(self, x):
        """Largest |d log D / d q_j| of each configuration, in chunks."""
        out = []
        for a in range(0, len(x), 1024):
            xc = x[a:a + 1024]
            u, r, _, off = self.pairs(xc)
            q = xc + ((off * self.spline(self.b, r)[0])[..., None] * u).sum(2)
            big = torch.zeros(len(xc), device=DEV, dtype=torch.float64)
            for p0, m in self.spins:
                if m:
                    gv = self.gvec[:m]
                    mat = self.orbitals(q[:, p0:p0 + m], gv)
                    inv = torch.linalg.inv(mat)
                    for c in range(2):
                        d = ((inv * gv[:, c]) * mat.transpose(1, 2)).sum(2).abs().amax(1)
                        big = torch.maximum(big, d)
            out.append(big)
        return torch.cat(out)

    def evaluate(self, x):
        """props, g, h, grad2 of the configurations x [w][n][2]."""
        nw, n = x.shape[:2]
        u, r, e, off = self.pairs(x)
        eye2 = torch.eye(2, device=DEV, dtype=torch.float64)
        uu = e[..., :, None] * e[..., None, :]
        f, df, ddf = (off * v for v in self.spline(self.u2, r))
        ltf = 0.5 * f.sum((1, 2))
        g = (df[..., None] * e).sum(2)
        lap = (ddf + df / r).sum(2)  # per particle
        if self.u3 is not None:
            xi, d1, d2 = (off * v for v in self.spline(self.u3, r))
            gp = (xi[..., None] * u).sum(2)
            ltf = ltf + 0.5 * ((xi * r) ** 2).sum((1, 2)) - 0.5 * (gp * gp).sum((1, 2))
            g = g + ((2 * xi * (xi + r * d1) * r)[..., None] * e).sum(2)
            lap = lap + (2 * (xi * xi + 4 * r * xi * d1 + r * r * (d1 * d1 + d2 * xi)) + 2 * xi * (xi + r * d1)).sum(2)
            m = xi[..., None, None] * eye2 + (d1 * r)[..., None, None] * uu
            dg = gp[:, :, None] - gp[:, None]
            g = g - torch.einsum("wijab,wijb->wia", m, dg)
            lap = lap - (m.sum(2) ** 2).sum((2, 3)) - (m ** 2).sum((2, 3, 4))
            lap = lap - ((d2 * r + 3 * d1)[..., None] * e * dg).sum((2, 3))
        eta, e1, e2 = (off * v for v in self.spline(self.b, r))
        q = x + (eta[..., None] * u).sum(2)
        jb = eta[..., None, None] * eye2 + (e1 * r)[..., None, None] * uu  # dq_i/dx_i part of pair (i, j)
        jac = -jb.permute(0, 1, 3, 2, 4).contiguous()                      # [w][j][a][i][d]
        idx = torch.arange(n, device=DEV)
        jac[:, idx, :, idx] += (eye2 + jb.sum(2)).transpose(0, 1)
        qb = (e2 * r + 3 * e1)[..., None] * e                              # laplacian_j of q_i (and of q_j, summed)
        grad2 = torch.zeros(nw, device=DEV, dtype=torch.float64)
        g_jastrow, lap_jastrow = g, lap
        for p0, m in self.spins:
            if m == 0:
                continue
            gv = self.gvec[:m]
            a = self.orbitals(q[:, p0:p0 + m], gv)
            ai = torch.linalg.inv(a.cpu()).to(DEV)
            ltf = ltf - torch.linalg.slogdet(a.cpu())[1].to(DEV)
            fa = [ai @ ((1j * gv[:, c])[:, None] * a) for c in range(2)]
            dl = torch.stack([torch.diagonal(v, dim1=1, dim2=2) for v in fa], -1)  # [w][j][a]
            v = jac[:, p0:p0 + m]
            gd = torch.einsum("wja,wjaid->wid", dl, v.to(dl.dtype))
            g = g - gd.real
            hbp = torch.tensor(self.hb, device=DEV, dtype=torch.float64)[self.type]
            grad2 = grad2 + (hbp[None, :, None] * gd.imag ** 2).sum((1, 2))
            # laplacian of log D, per particle i
            lq = torch.einsum("wja,wjia->wi", dl.real, qb[:, p0:p0 + m])
            lq[:, p0:p0 + m] += torch.einsum("wja,wjia->wj", dl.real, qb[:, p0:p0 + m])
            mm = torch.empty((nw, m, 2, m, 2), device=DEV, dtype=torch.float64)
            for c in range(2):
                for b in range(2):
                    mm[:, :, c, :, b] = -(fa[c].transpose(1, 2) * fa[b]).real
                    j = torch.arange(m, device=DEV)
                    dd = torch.diagonal(fa[c] @ fa[b], dim1=1, dim2=2).real
                    mm[:, j, c, j, b] += dd
            vv = v.reshape(nw, 2 * m, 2 * n)
            s = (vv * (mm.reshape(nw, 2 * m, 2 * m) @ vv)).sum(1).reshape(nw, n, 2).sum(2)
            lap = lap - lq - s
        # the underflow guard: where psi^2 = exp(-2 ltf) is zero in 64 bits the
        # determinants' drift and laplacian are left out
        gone = torch.exp(-2.0 * ltf) == 0.0
        g = torch.where(gone[:, None, None], g_jastrow, g)
        lap = torch.where(gone[:, None], lap_jastrow, lap)
        grad2 = torch.where(gone, torch.zeros_like(grad2), grad2)
        nt = len(self.np)
        by_type = [slice(p0, p0 + m) for p0, m in self.spins]
        h = torch.zeros((nw, 2), device=DEV, dtype=torch.float64)
        for t, sl in enumerate(by_type):
            h[:, t] = lap[:, sl].sum(1)
        g2 = torch.stack([(g[:, sl] ** 2).sum((1, 2)) for sl in by_type], 1)
        kin = torch.tensor(self.hb, device=DEV, dtype=torch.float64) * (h[:, :nt] - g2)
        # potential: pairs, then rho_k and the k-space sum
        pv = 0.5 * off * self.spline(self.v, r)[0] * r ** -float(self.vt.iexp)
        pot = torch.stack([pv[:, sl].sum((1, 2)) for sl in by_type], 1)
        ph = torch.exp(1j * (x @ self.kvec.T))
        rho = torch.stack([ph[:, sl].sum(1) for sl in by_type], 1)  # [w][type][k]
        tot = rho.sum(1)
        nke = len(self.vk)
        pot = pot + torch.stack([(self.vk * (rho[:, t, :nke].conj() * tot[:, :nke]).real).sum(1) for t in range(nt)], 1)
        cnt = torch.tensor([float(m) for m in self.np], device=DEV, dtype=torch.float64)
        pot0, kin0 = (pot.sum(1) + self.deck.v0) / n, kin.sum(1) / n
        efp = grad2 / n if self.ntheta else torch.zeros_like(grad2)
        et = pot0 + kin0 + efp
        zero = torch.zeros_like(et)
        cols = [et, ltf, zero, pot0, kin0, et * et, zero + 1.0]
        cols += list((pot / cnt).T) + list((kin / cnt).T) + list((1.0 / torch.sqrt(g2)).T) + [efp]
        props = torch.cat([torch.stack(cols, 1), torch.view_as_real(rho).reshape(nw, -1)], 1)
        return props, g, h, grad2

    def evaluate_all(self, x, chunk=None):
        chunk = chunk or max(1, int(4e6 / self.n ** 2 / 4))
        parts = [self.evaluate(x[a:a + chunk]) for a in range(0, len(x), chunk)]
        return [torch.cat(p) for p in zip(*parts)]


def _lcg(states, count):
    """`count` draws of every stream: uniforms [w][count] and the new states."""
    s = states.copy()
    out = np.empty((len(s), count))
    for k in range(count):
        s = (s * np.uint64(LCG)) & np.uint64(MASK)
        out[:, k] = s.astype(np.float64) * 2.0 ** -48
    return out, s


def _exact_vmc(case, seed):
    """The block of VMC steps: drift-diffusion proposals, Metropolis test,
    block sums."""
    sy = _System(case)
    x, delta = _dev(_configs(case, seed)), _delta(case)
    rng = _streams(case, seed).astype(np.uint64)
    props, g, h, g2 = sy.evaluate_all(x)
    props[:, 2] = 1.0
    var = 2.0 * sy.hb[0] * delta
    age = torch.zeros(len(x), device=DEV, dtype=torch.float64)
    blk = torch.zeros_like(props)
    for _ in range(case["steps"]):
        uni, rng = _lcg(rng, 4 * sy.n)
        uni = _dev(uni).reshape(len(x), sy.n, 2, 2)
        chi = torch.cos(math.pi * uni[..., 0]) * torch.sqrt(-2.0 * var * torch.log(uni[..., 1]))
        xn = chi - var * g + x
        pn, gn, hn, g2 = sy.evaluate_all(xn)
        back = x - xn + var * gn
        p = 2.0 * (props[:, 1] - pn[:, 1]) + 0.5 * ((chi ** 2).sum((1, 2)) - (back ** 2).sum((1, 2))) / var
        p = torch.exp(p.clamp(-50.0, 0.0))
        p = torch.where(age == 50.0, torch.ones_like(p), p)
        one, after = _lcg(rng, 1)
        drawn = (p < 1.0).cpu().numpy()
        rng = np.where(drawn, after, rng)
        acc = p >= torch.where(p < 1.0, _dev(one[:, 0]), torch.ones_like(p))
        x, g = torch.where(acc[:, None, None], xn, x), torch.where(acc[:, None, None], gn, g)
        h, props = torch.where(acc[:, None], hn, h), torch.where(acc[:, None], pn, props)
        props[:, 2] = p
        age = torch.where(acc, torch.zeros_like(age), age + 1.0)
        blk = blk + props
    out = dict(x=x, g=g, h=h, props=props, age=age, rng=None, blk=blk)
    if _fixed_phase(case):
        out["grad2"] = g2
    return out


def _exact_sem(case, seed):
    """Refresh and single-electron sweeps, the determinant ratios from
    Sherman-Morrison updates in complex 64-bit arithmetic."""
    sy = _System(case)
    x = _dev(_configs(case, seed))
    rng = _streams(case, seed).astype(np.uint64)
    nw, mm = len(x), max(sy.np)
    dlog = torch.zeros(nw, device=DEV, dtype=torch.float64)
    nacc = torch.zeros_like(dlog)
    inv = [torch.linalg.inv(sy.orbitals(x[:, p0:p0 + m], sy.gvec[:m]).cpu()).to(DEV) if m else None for p0, m in sy.spins]

    def change(j, new):
        """Pair terms of electron j at `new` less those where it is."""
        def terms(pos):
            u = pos[:, None] - x
            u = u - sy.el * torch.round(u / sy.el)
            r = torch.sqrt((u * u).sum(-1))
            r[:, j] = 1.0
            f = sy.spline(sy.u2, r)[0]
            f[:, j] = 0.0
            return f.sum(1)
        return terms(new) - terms(x[:, j])

    for _ in range(case["sweeps"]):
        for (p0, m), sp in zip(sy.spins, range(2)):
            for j in range(p0, p0 + m):
                uni, rng = _lcg(rng, 3)
                uni = _dev(uni)
                rad = case["sigma"] * torch.sqrt(-2.0 * torch.log(uni[:, 0]))
                ang = 2.0 * math.pi * uni[:, 1]
                new = x[:, j] + torch.stack([rad * torch.cos(ang), rad * torch.sin(ang)], 1)
                t = (inv[sp] @ torch.exp(1j * (new @ sy.gvec[:m].T))[:, :, None])[:, :, 0]
                ratio = t[:, j - p0].clone()
                du = change(j, new)
                acc = uni[:, 2] < (ratio.abs() ** 2) * torch.exp(-2.0 * du)
                t[:, j - p0] -= 1.0
                k = torch.where(acc, 1.0 / ratio, torch.zeros_like(ratio))
                inv[sp] = inv[sp] - (t * k[:, None])[:, :, None] * inv[sp][:, j - p0, None, :]
                x[:, j] = torch.where(acc[:, None], new, x[:, j])
                dlog += torch.where(acc, torch.log(ratio.abs()) - du, torch.zeros_like(du))
                nacc += acc
    ainv = torch.zeros((nw, 2, mm, mm, 2), device=DEV, dtype=torch.float64)
    for sp, (p0, m) in enumerate(sy.spins):
        if m:
            ainv[:, sp, :m, :m] = torch.view_as_real(inv[sp])
    out = dict(x=x, rng=None, dlogpsi=dlog, nacc=nacc, ainv=ainv)
    if case["energy"]:
        props, g, h, g2 = sy.evaluate_all(x)
        props[:, 2] = 1.0
        out.update(props=props, g=g, h=h)
        if _fixed_phase(case):
            out["grad2"] = g2
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("host", "eval"):
        sy = _System(case)
        props, g, h, g2 = sy.evaluate_all(_dev(_configs(case, seed)))
        out = dict(props=props, g=g, h=h, status=None)
        if _fixed_phase(case):
            out["grad2_ph" if kind == "host" else "grad2"] = g2
        return {k: v if v is None or kind == "eval" else v.cpu().numpy() for k, v in out.items()}
    if kind == "vmc":
        return _exact_vmc(case, seed)
    # FP32 inverses decide a few moves otherwise than 64 bits; u3 and
    # backflow moves are held to the start's outputs
    if kind == "sem" and not case["mixed"] and case["backflow"] == "zero" and not case["u3"]:
        return _exact_sem(case, seed)
    if kind == "pack":
        return [_exact_sem(c, seed + 1000 * k) for k, c in enumerate(_pack_cases(case))]
    return None
