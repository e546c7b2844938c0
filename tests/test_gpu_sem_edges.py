"""Single-electron moves at the edges of their launch shapes: real rows of
exactly 16, 32 and 64 (15, 31 and 63 particles with the zero wave), even lists
without a zero wave, packed launches whose blocks hold two walkers with an odd
number of them, and the value-only determinants against the full ones, one move
at a time."""
import numpy as np
import pytest

from conftest import pkg

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


def _states(nw, base=3099):
    abi = pkg("abi")
    return [abi.limbs_to_state([3535, 3467, 3262, (base + 2 * w) % 4096]) for w in range(nw)]


def _deck(path, nup, ndown, u3=True, backflow="zero", ntwists=0, rs=5.0):
    dg = pkg("deckgen")
    n, shells = nup + ndown, 5
    while 2 * len(dg.klist(float(np.sqrt(n * np.pi)), shells)) + 1 < max(nup, ndown) + 2:
        shells += 2
    dg.make_deck(str(path), "se", nup, ndown, rs, 5, nshell_k=shells, u3=u3, backflow=backflow, jastrow="pade",
                 ntwists=ntwists)
    return pkg("deck").read_deck(str(path))


def _walkers(d, nw, seed, **kw):
    hip = pkg("hip")
    ctx = hip.Context(d, **kw)
    wk = hip.Walkers(ctx, pkg("deckgen").lattice_configs(nw, d.nptot, d.el[0], seed), _states(nw, 500 + 7 * seed))
    wk.start()
    return ctx, wk


@pytest.mark.parametrize("zero", [True, False])
@pytest.mark.parametrize("nup,ndown", [(15, 15), (31, 31), (63, 63), (31, 63), (15, 33), (16, 0)])
def test_class_edges_of_real_rows(tmp_path, nup, ndown, zero):
    """After a refresh and two sweeps the inverses are those of the positions
    and the summed log|psi| change is the full evaluations', as at the other
    sizes.  Without the zero wave the spins have one particle more."""
    import torch
    hip = pkg("hip")
    if not zero:
        nup, ndown = nup + nup % 2, ndown + ndown % 2
    elif nup % 2 == 0:
        pytest.skip("an even list has no zero wave")
    print(f"\n[gpu] real rows {nup}+{ndown}, zero wave {zero}", flush=True)
    d = _deck(tmp_path, nup, ndown)
    gvec = None
    if not zero:
        k = np.asarray(d.kvec, dtype=np.float64).reshape(-1, 2)
        gvec = np.stack([k, -k], 1).reshape(-1, 2)
    ctx, wk = _walkers(d, 8, nup + ndown, twist=(1, 1), gvec=gvec)
    assert hip.real_orbitals(ctx.gvec, d.np[:d.ntypes])
    sm = hip.SingleMoves(wk)
    jltf = ctx.info["jltf"] - 1
    ltf0 = wk.props[:, jltf].clone()

    def worst():
        torch.cuda.synchronize()
        x, inv = wk.x.cpu().numpy(), sm.ainv.cpu().numpy()
        inv, e = inv[..., 0] + 1j * inv[..., 1], 0.0
        for w in range(len(x)):
            for sp, (a, b) in enumerate(((0, nup), (nup, nup + ndown))):
                if b > a:
                    ref = np.linalg.inv(np.exp(1j * (ctx.gvec[:b - a] @ x[w, a:b].T)))
                    e = max(e, np.abs(inv[w, sp, :b - a, :b - a] - ref).max() / np.abs(ref).max())
        return e

    sm.refresh()
    assert worst() < 1e-9
    for _ in range(2):
        sm.sweep(0.5)
    assert worst() < 1e-8
    wk.start()
    torch.cuda.synchronize()
    assert float(sm.nacc.sum()) > 0
    assert float((sm.dlogpsi + (wk.props[:, jltf] - ltf0)).abs().max()) < 1e-8
    wk = sm = None
    ctx.close()


def test_packed_jobs_with_odd_walker_counts(tmp_path):
    """Small real-row jobs share blocks, two walkers each, beside a wide job: a
    last block with one walker gives what the job's own call gives, to the
    bit."""
    print("\n[gpu] packed jobs, odd walker counts", flush=True)
    import torch
    hip = pkg("hip")
    jobs = [((13, 13), 1), ((37, 37), 5), ((15, 15), 3), ((13, 0), 25), ((31, 9), 7), ((61, 61), 1)]
    decks = [_deck(tmp_path / str(k), *s, u3=k % 2 == 0) for k, (s, _) in enumerate(jobs)]

    def make():
        out = []
        for k, (d, (_, nw)) in enumerate(zip(decks, jobs)):
            out.append(hip.SingleMoves(_walkers(d, nw, 30 + k, twist=(1, 1))[1]))
            out[-1].refresh()
        return out

    sep, pak = make(), make()
    for _ in range(2):
        for sm, d in zip(sep, decks):
            sm.moves(0, d.nptot, 0.5)
        hip.sem_moves_packed([(sm, 0, d.nptot, 0.5) for sm, d in zip(pak, decks)])
    torch.cuda.synchronize()
    for a, b, (size, nw) in zip(sep, pak, jobs):
        for u, v in zip((a.wk.x, a.wk.rng, a.ainv, a.dlogpsi, a.nacc), (b.wk.x, b.wk.rng, b.ainv, b.dlogpsi, b.nacc)):
            assert torch.equal(u, v), (size, nw)
        assert 0 < float(a.nacc.sum()) < 2 * sum(size) * nw


@pytest.mark.parametrize("twist", [(1, 1), (2, 3)])
@pytest.mark.parametrize("nup,ndown", [(13, 15), (17, 31), (33, 47), (49, 63), (63, 5), (29, 0)])
def test_value_only_determinants_one_move(tmp_path, nup, ndown, twist):
    """log|psi| kept by one move with backflow is a fresh evaluation's: every
    tile count of the value-only eliminations, real and complex.  The difference
    is rounding: of the N (N - 1) / 2 pair terms (up to 5, chains of up to 30
    additions) in the Jastrow sum, and of the quasi-coordinates (N terms of up to
    1/2 and the position, twice), each of which log|psi| takes with its
    gradient."""
    print(f"\n[gpu] value-only determinants {nup}+{ndown} twist {twist}", flush=True)
    import torch
    hip = pkg("hip")
    d = _deck(tmp_path, nup, ndown, backflow="yk", ntwists=4 if twist != (1, 1) else 0, rs=2.0)
    ctx, wk = _walkers(d, 48, nup, twist=twist)
    sm = hip.SingleMoves(wk)
    jltf, N, acc = ctx.info["jltf"] - 1, d.nptot, 0.0
    for j in (0, nup - 1, N - 1):
        sm.moves(j, j + 1, 0.3)
        torch.cuda.synchronize()
        kept = wk.props[:, jltf].cpu().numpy().copy()
        wk.start()
        torch.cuda.synchronize()
        g, x = np.abs(wk.g.cpu().numpy()).sum(axis=(1, 2)), np.abs(wk.x.cpu().numpy()).max(axis=(1, 2))
        tol = EPS * (30 * 5 * N * (N - 1) / 2 + (0.5 * N + 2 * x) * g)
        err = np.abs(kept - wk.props[:, jltf].cpu().numpy())
        print(f"   electron {j}: error {err.max():.1e}, {np.max(err / tol):.3f} of the bound", flush=True)
        assert (err <= tol).all()
    assert 0 < float(sm.nacc.sum()) < 3 * 48
    wk = sm = None
    ctx.close()
