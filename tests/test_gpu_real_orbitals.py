"""Real-orbital determinants (k_gjr, k_cross_real): spins whose plane waves
come with their opposites.  Counts at the edges of its 16-row tiles (15/17,
31/33, 47/49, 63; one tile to four, both spins alike or not, one spin empty)
against the oracle, and g-vector lists in other forms (shuffled, the zero
vector not first or absent, signed zeros, one wave without its opposite, which
takes the complex path) against the general complex determinant k_det.
Tolerance 1e-10 relative, as for the reference goldens."""
import os

import numpy as np
import pytest

from conftest import compare_eval, pkg

pytestmark = pytest.mark.gpu

RTOL = 1e-10
SIZES = [(1, 1), (3, 1), (15, 15), (17, 17), (31, 33), (47, 49), (63, 63), (61, 13), (63, 0), (13, 14)]


def _deck(tmp_path, nup, ndown):
    dg, deck = pkg("deckgen"), pkg("deck")
    path = os.path.join(str(tmp_path), "deck")
    dg.make_deck(path, "ro", nup, ndown, 2.0, 40, jastrow="pade")
    return deck.read_deck(path)


def _gold(ref, d, ns):
    return dict(scalars=ref["props"][:, :ns], g=ref["g"], h=ref["h"][:, :d.ntypes], grad2_ph=ref["grad2_ph"],
                rhok=ref["props"][:, ns:])


@pytest.mark.parametrize("nup,ndown", SIZES)
def test_sizes_match_oracle(nup, ndown, tmp_path, oracle_mod):
    print(f"\n[gpu] real orbitals {nup}+{ndown}", flush=True)
    d = _deck(tmp_path, nup, ndown)
    x = pkg("deckgen").lattice_configs(8, d.nptot, d.el[0], 50 + nup + ndown)
    o = oracle_mod.Oracle(d, twist=(1, 1))
    ref, ns = o.eval(x), o.info["n_scalar_props"]
    ctx = pkg("hip").Context(d, twist=(1, 1))
    try:
        out = ctx.eval(x)
    finally:
        ctx.close()
    compare_eval(out, _gold(ref, d, ns), ns, RTOL, f"{nup}+{ndown}")
    assert np.array_equal(out["status"], ref["status"])


def _lists(d, m):
    """g-vector lists of m plane waves by name."""
    k = np.asarray(d.kvec, dtype=np.float64).reshape(-1, 2)
    base = np.concatenate([np.zeros((1, 2)), np.stack([k, -k], 1).reshape(-1, 2)])
    rng = np.random.default_rng(3)
    shuffled = base[:m][rng.permutation(m)]
    neg0 = base[:m].copy()
    neg0[neg0 == 0.0] = -0.0
    lone = base[:m].copy()
    lone[-1] = base[m + 1]
    return {"shuffled": shuffled, "signed_zeros": neg0, "no_zero": base[1:m if m % 2 else m + 1], "lone": lone}


@pytest.mark.parametrize("m", [29, 49])
@pytest.mark.parametrize("form", ["shuffled", "signed_zeros", "no_zero", "lone"])
def test_list_forms_match_general_path(form, m, tmp_path, monkeypatch):
    print(f"\n[gpu] real orbitals, list {form}, {m} waves", flush=True)
    n = m - 1 if form == "no_zero" else m
    d = _deck(tmp_path, n, n)
    g = _lists(d, m)[form]
    x = pkg("deckgen").lattice_configs(8, d.nptot, d.el[0], 60 + m)
    res = []
    for general in (False, True):
        if general:
            monkeypatch.setenv("QMC_NO_GJ", "1")
        ctx = pkg("hip").Context(d, gvec=g)
        try:
            res.append((ctx.eval(x), ctx.info["n_scalar_props"]))
        finally:
            ctx.close()
    (out, ns), (ref, _) = res
    compare_eval(out, _gold(ref, d, ns), ns, RTOL, form)
    assert np.array_equal(out["status"], ref["status"])


def test_value_alone_equals_the_full_evaluation(tmp_path):
    """log|psi| carried by moves with backflow (the value-only determinants) is
    the full evaluation's, with real orbitals and tiles that differ between the
    spins.  The moves' quasi-coordinates and Jastrow sums follow the moved
    electron's pairs, so the two agree to the rounding of some 1e3 additions of
    1e-16 of values up to 1e3, times the orbital matrices' condition (1e4) in
    log|det|: 1e-9."""
    print("\n[gpu] real orbitals, value-only moves 17+31", flush=True)
    import torch
    hip = pkg("hip")
    d = _deck(tmp_path, 17, 31)
    x = pkg("deckgen").lattice_configs(6, d.nptot, d.el[0], 70)
    ctx = hip.Context(d, twist=(1, 1))
    wk = hip.Walkers(ctx, x, [2 * k + 12345 for k in range(6)])
    wk.start()
    sm = hip.SingleMoves(wk)
    sm.moves(0, 4, 0.3)
    torch.cuda.synchronize()
    kept = wk.props[:, ctx.info["jltf"] - 1].clone()
    wk.start()
    torch.cuda.synchronize()
    assert float((kept - wk.props[:, ctx.info["jltf"] - 1]).abs().max()) < 1e-9
    assert sm.nacc.sum().item() > 0
    wk = sm = None
    ctx.close()
