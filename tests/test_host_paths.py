"""Host code of the library under failures that a GPU does not show on demand:
limits, refused launches and allocations.  Each scenario runs in a process of
its own against a stand-in of the HIP runtime (hip_stub.cpp) that logs the
launches and keeps device memory on the host; no GPU takes part."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "2degas_amd", "lib2degas_hip.so")
HIP_INCLUDE = "/opt/rocm/include"

PRELUDE = r"""
import ctypes, importlib, os, sys
import numpy as np
sys.modules["torch"] = None  # the binding imports it only to share its runtime
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_log.restype = ctypes.c_char_p
sys.path.insert(0, sys.argv[2])
hip, abi, deck = (importlib.import_module("2degas_amd." + m) for m in ("hip", "abi", "deck"))
L = hip.lib()

def load(name):
    return deck.read_deck(os.path.join(sys.argv[2], "tests", "golden", "decks", name))

def log(kind=None):
    lines = [ln.split(" ", 1) for ln in stub.stub_log().decode().splitlines()]
    return [b for a, b in lines if kind is None or a == kind]

def fail(name, n=1):
    stub.stub_fail(name.encode(), n)

def buffers(ctx, nw):
    # host arrays in the places of device buffers
    n, np_ = ctx.deck.nptot, ctx.info["n_props"]
    w, keep = abi.QmcWalkers(), {}
    w.nw = nw
    for k, sh in dict(x=(nw, n, 2), g=(nw, n, 2), h=(nw, 2), props=(nw, np_), grad2_ph=nw, age=nw, blk=(nw, np_)).items():
        keep[k] = np.zeros(sh)
        setattr(w, k, keep[k].ctypes.data)
    keep["rng"] = np.ones(nw, np.int64)
    w.rng = keep["rng"].ctypes.data
    return w, keep

def dmc_state(nw):
    d = abi.QmcDmcState()
    keep = dict(wate=np.ones(nw), wsum=np.zeros(nw), src=np.zeros(nw, np.int32), rng2=np.ones(1, np.int64),
                counts=np.zeros(4, np.int32))
    for k, a in keep.items():
        setattr(d, k, a.ctypes.data)
    return d, keep
"""


@pytest.fixture(scope="module")
def run_host(tmp_path_factory):
    if not os.path.exists(LIB) or not os.path.isdir(HIP_INCLUDE) or not shutil.which("g++"):
        pytest.skip("needs the built library, the HIP headers and g++")
    so = str(tmp_path_factory.mktemp("stub") / "libhip_stub.so")
    subprocess.run(["g++", "-O1", "-fPIC", "-shared", "-std=c++17", "-I" + HIP_INCLUDE,
                    os.path.join(ROOT, "tests", "hip_stub.cpp"), "-o", so], check=True)

    def run(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE + body, so, ROOT], stdout=subprocess.PIPE,
                           stderr=subprocess.STDOUT, timeout=120)
        assert r.returncode == 0, r.stdout.decode()
    return run


def test_dmc_population_limit(run_host):
    """The branching's LDS, its own beside the walkers', decides which
    populations are taken: a larger one is refused before anything is launched,
    by the branching alone and by a sweep."""
    run_host(r"""
ctx = hip.Context(load("n26g"), twist=(1, 1))
fits = (163840 - 8208) // 12
for nw, ok in ((fits, True), (fits + 1, False), (13500, False), (13648, False)):
    d, keep = dmc_state(nw)
    stub.stub_clear()
    rc = L.qmc_dmc_branch(ctx.h, nw, d.wate, d.rng2, d.src, d.counts, None)
    assert rc == (0 if ok else abi.QMC_ERR_LIMIT), (nw, rc)
    assert len(log("launch")) == (1 if ok else 0), log()
w, keep = buffers(ctx, 13500)
d, keep2 = dmc_state(13500)
p = abi.QmcDmcParams()
p.delta, p.mage, p.mmstep, p.mmult = 0.01, 1e30, 1, 10
stub.stub_clear()
rc = L.qmc_dmc_sweep(ctx.h, ctypes.byref(w), ctypes.byref(d), 1, ctypes.byref(p), None)
assert rc == abi.QMC_ERR_LIMIT, rc
assert not log("launch"), log("launch")
""")


def test_dmc_copies_follow_a_branching(run_host):
    """No walker is copied by the sources of an earlier branching when this
    one's launch fails."""
    run_host(r"""
ctx = hip.Context(load("n26g"), twist=(1, 1))
w, keep = buffers(ctx, 16)
d, keep2 = dmc_state(16)
p = abi.QmcDmcParams()
p.delta, p.mage, p.mmstep, p.mmult = 0.01, 1e30, 1, 10
sweep = lambda n: L.qmc_dmc_sweep(ctx.h, ctypes.byref(w), ctypes.byref(d), n, ctypes.byref(p), None)
assert sweep(1) == 0
assert [sum(k in n for n in log("launch")) for k in ("k_dmc_branch", "k_dmc_copy")] == [1, 1]
stub.stub_clear()
fail("launch:k_dmc_branch", 2)
assert sweep(3) == abi.QMC_ERR_HIP
assert [sum(k in n for n in log("launch")) for k in ("k_dmc_branch", "k_dmc_copy")] == [1, 1]
""")


def test_host_evaluation_without_pinned_memory(run_host):
    """A host-pointer call goes through the copies when no pinned memory can be
    had, and through the pinned buffer once it can."""
    run_host(r"""
ctx = hip.Context(load("n26"), twist=(1, 1))
x = np.zeros((2, 26, 2))
fail("hipHostMalloc", 1)
stub.stub_clear()
ctx.eval(x)
assert len(log("copy")) == 8 and not any("k_stage" in k for k in log("launch")), log()
stub.stub_clear()
ctx.eval(x)
assert not log("copy") and sum("k_stage" in k for k in log("launch")) == 2, log()
""")


def test_host_evaluation_that_fails_after_staging(run_host):
    """An evaluation that is refused after its inputs were staged returns the
    error, leaves the caller's arrays as they are, and the next call works."""
    run_host(r"""
ctx = hip.Context(load("n26"), twist=(1, 1))
x = np.zeros((2, 26, 2))
ctx.eval(x)
fail("launch:k_final", 1)
g2 = np.full(2, 3.5)
try:
    ctx.eval(x, grad2_in=g2)
    raise SystemExit("no error")
except hip.QmcError as e:
    assert e.code == abi.QMC_ERR_HIP
assert (g2 == 3.5).all()
stub.stub_clear()
ctx.eval(x)
assert sum("k_stage" in k for k in log("launch")) == 2
""")


def test_set_twist_that_fails_changes_nothing(run_host):
    """A list that cannot be stored, on the device or on the host, leaves the
    context with the one it had (its orbitals read that, not freed memory), and
    the error it returned is not reported again by the next call."""
    run_host(r"""
import resource
ctx = hip.Context(load("n26g"), twist=(1, 1))
old, x = ctx.gvec.copy(), np.zeros((1, 26, 2))
real = lambda: any("k_gjr" in k for k in log("launch"))
other = old.copy()
other[5] = 1.25 * other[5]  # its opposite is another wave: complex orbitals
for name in ("hipMalloc", "hipMemcpy"):
    stub.stub_clear()
    fail(name, 1)
    assert L.qmc_set_twist(ctx.h, abi.dptr(other), len(other)) == abi.QMC_ERR_HIP
    given = log("malloc")
    assert sorted(log("free")) == sorted(given), log()  # what was allocated, and nothing else
    ctx.eval(x)
    assert real()
soft, hard = resource.getrlimit(resource.RLIMIT_AS)
resource.setrlimit(resource.RLIMIT_AS, (8 << 30, hard))
stub.stub_clear()
assert L.qmc_set_twist(ctx.h, abi.dptr(other), 1 << 29) == abi.QMC_ERR_HIP
resource.setrlimit(resource.RLIMIT_AS, (soft, hard))
assert not log("free")
ctx.eval(x)
assert real()
stub.stub_clear()
ctx.set_twist(other)
assert len(log("free")) == 1
stub.stub_clear()
ctx.eval(x)
assert not real()
""")


def test_an_empty_type_takes_no_lds(run_host):
    """The pair kernel's sums and phase rows are those of the types that have
    particles: 61 of one type take less than 61 + 61."""
    run_host(r"""
lds = {}
for name in ("g61p", "g122"):
    d = load(name)
    ctx = hip.Context(d, twist=(1, 1))
    stub.stub_clear()
    ctx.eval(np.zeros((1, d.nptot, 2)))
    lds[name], = [int(e.split()[0]) for e in log("lds") if "k_pairs" in e]
assert lds["g61p"] < 0.85 * lds["g122"], lds
""")


@pytest.mark.parametrize("grid", [True, False])
def test_autotune_times_the_forms_there_are(run_host, grid):
    """FP64 phase rows come in fours of one type's particles: the autotuner times
    every such chunk, no form under two names, each in two rounds, and names the one it keeps; a k list off the grid (a
    k-vector five times over) has one FP64 form."""
    run_host("grid = %r" % grid + r"""
d = load("n26g")
if not grid:
    kv = np.array(d.kvec, dtype=np.float64).reshape(-1, 2)
    d.kvec = np.ascontiguousarray(np.concatenate([np.repeat(kv[:1], 5, axis=0), kv[5:]]))
ctx = hip.Context(d, twist=(1, 1))
kc, ms = np.zeros(2, np.int32), np.zeros(2)
stub.stub_clear()
assert L.qmc_autotune(ctx.h, 8, abi.iptr(kc), abi.dptr(ms), None) == 0
n64, nmix = (sum("k_pairsILb%d" % b in k for k in log("launch")) for b in (0, 1))
if grid:
    assert n64 == 2 * 4 * 3, n64  # 13 particles of a type: 16, 4, 8
    assert kc[0] == 16
else:
    assert n64 == 2 * 4 and kc[0] == 1, (n64, kc)
assert nmix == 2 * 4 * 6, nmix  # 26 particles: the default, 1, 2, 4, 8, 16
assert (ms > 0).all()
""")


def test_binding_knows_real_orbitals(run_host):
    """real_orbitals says what the library does with a list: which determinant
    kernel an evaluation launches."""
    run_host(r"""
d = load("n26g")
ctx = hip.Context(d, twist=(1, 1))
base, x = ctx.gvec.copy(), np.zeros((1, 26, 2))
neg0 = base.copy()
neg0[neg0 == 0.0] = -0.0
shuffled = base.copy()
shuffled[:13] = base[np.random.default_rng(3).permutation(13)]
lone = base.copy()
lone[12] = base[20]
two_zeros = base.copy()
two_zeros[1:3] = 0.0
twice = base.copy()
twice[3:5] = base[1:3]
twisted = base + 0.1
seen = set()
for name, g in dict(base=base, neg0=neg0, shuffled=shuffled, lone=lone, two_zeros=two_zeros, twice=twice,
                    twisted=twisted).items():
    ctx.set_twist(g)
    stub.stub_clear()
    ctx.eval(x)
    real = any("k_gjr" in k for k in log("launch"))
    assert real != any("k_gjc" in k for k in log("launch"))
    assert hip.real_orbitals(ctx.gvec, d.np[:d.ntypes]) == real, name
    seen.add(real)
assert seen == {True, False}
assert not hip.real_orbitals(base[:12], [13, 13])
""")


@pytest.mark.parametrize("name", ["c26", "n26g"])
def test_moves_need_the_orbitals(run_host, name):
    """Single-electron moves of a context whose list holds fewer waves than a spin
    has particles (or none yet) are refused, with and without backflow, before
    anything is launched: not read beyond the list."""
    run_host("name = %r" % name + r"""
ctx = hip.Context(load(name), twist=(1, 1))
w, keep = buffers(ctx, 4)
s = abi.QmcSemState()
keep2 = [np.zeros(4 * 2 * 13 * 13 * 2), np.zeros(4), np.zeros(4)]
s.ainv, s.dlogpsi, s.nacc = (a.ctypes.data for a in keep2)
job = (abi.QmcSemJob * 1)()
job[0].ctx, job[0].w, job[0].d = ctx.h.value, ctypes.addressof(w), ctypes.addressof(s)
job[0].j0, job[0].j1, job[0].sigma = 0, 26, 0.5
refresh = lambda p: L.qmc_sem_refresh(ctx.h, ctypes.byref(w), ctypes.byref(s), p, None)
moves = lambda p: L.qmc_sem_moves(ctx.h, ctypes.byref(w), ctypes.byref(s), 0, 26, 0.5, p, None)
packed = lambda p: L.qmc_sem_moves_packed(job, 1, p, None)
full = ctx.gvec.copy()
for waves in (0, 5, 12):
    ctx.set_twist(full[:waves])
    for call in (refresh, moves, packed):
        for prec in (0, 1):
            stub.stub_clear()
            # (with backflow a refresh does nothing, and jobs are not packed)
            want = abi.QMC_ERR_NOTWIST
            if name == "n26g":
                want = {refresh: abi.QMC_OK, packed: abi.QMC_ERR_ARG}.get(call, want)
            assert call(prec) == want, (waves, prec)
            assert not log("launch"), log()
    # nothing to move, nothing to read
    w.nw = 0
    assert refresh(0) == 0 and moves(0) == 0
    w.nw = 4
ctx.set_twist(full[:13])
assert refresh(0) == 0 and moves(0) == 0 and log("launch")
""")
