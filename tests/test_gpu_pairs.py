"""The pair kernel's schedule and its FP64 rho_k against the oracle: particle
counts at the edges of its lane blocks (16/17, 32/33, 64, unequal spins, one
spin empty), and k lists in other forms than the generator's half space: signs
mirrored, both k and -k (four k-vectors in one (|kx|, |ky|) cell), a k-vector
five times over (too many for a cell), components without a common step, more
magnitudes than tiles of one pass, more than the phase rows hold.  Tolerance
1e-10 relative, as for the reference goldens."""
import os

import numpy as np
import pytest

from conftest import compare_eval, pkg

pytestmark = pytest.mark.gpu

RTOL = 1e-10


def _check(d, x, oracle_mod, gvec=None):
    o = oracle_mod.Oracle(d, twist=(1, 1), gvec=gvec)
    ref, ns = o.eval(x), o.info["n_scalar_props"]
    gold = dict(scalars=ref["props"][:, :ns], g=ref["g"], h=ref["h"][:, :d.ntypes], grad2_ph=ref["grad2_ph"],
                rhok=ref["props"][:, ns:])
    ctx = pkg("hip").Context(d, twist=(1, 1), gvec=gvec)
    try:
        out = ctx.eval(x)
    finally:
        ctx.close()
    compare_eval(out, gold, ns, RTOL)


def _deck(tmp_path, nup, ndown, shells=40, **kw):
    dg, deck = pkg("deckgen"), pkg("deck")
    path = os.path.join(str(tmp_path), "deck")
    dg.make_deck(path, "pr", nup, ndown, 2.0, shells, jastrow="pade", **kw)
    return deck.read_deck(path)


@pytest.mark.parametrize("nup,ndown", [(1, 0), (2, 1), (16, 16), (17, 16), (15, 2), (32, 32), (33, 5), (32, 0), (64, 64)])
def test_lane_blocks_match_oracle(nup, ndown, tmp_path, oracle_mod):
    print(f"\n[gpu] pair schedule {nup}+{ndown}", flush=True)
    d = _deck(tmp_path, nup, ndown, u3=nup != 15)
    _check(d, pkg("deckgen").lattice_configs(6, d.nptot, d.el[0], nup + 3 * ndown), oracle_mod)


def _forms(kv):
    rng = np.random.default_rng(5)
    n = len(kv)
    sign = rng.choice([-1.0, 1.0], (n, 2))
    return {"mirrored": kv * sign,
            "both_signs": np.concatenate([kv[:n // 2], -kv[:n - n // 2]]),
            "repeated": np.concatenate([np.repeat(kv[:1], 5, axis=0), kv[5:]]),
            "no_step": kv * (1.0 + 1e-3 * np.sin(np.arange(n)))[:, None],
            "wide": np.stack([np.arange(n) % 70, np.arange(n) % 3 + 1], 1) * kv[0].max(),
            "too_wide": np.stack([np.arange(n) + 1.0, 1.0 + np.arange(n)], 1) * kv[0].max()}


@pytest.mark.parametrize("form", ["mirrored", "both_signs", "repeated", "no_step", "wide", "too_wide"])
def test_k_lists_match_oracle(form, tmp_path, oracle_mod):
    print(f"\n[gpu] rho_k, k list {form}", flush=True)
    d = _deck(tmp_path, 13, 9, backflow="zero")
    kv = np.array(d.kvec, dtype=np.float64).reshape(-1, 2)
    g = pkg("hip").twist_gvec(kv, d.el, 0, 1, 1)
    d.kvec = np.ascontiguousarray(_forms(kv)[form])
    _check(d, pkg("deckgen").lattice_configs(6, d.nptot, d.el[0], 77), oracle_mod, gvec=g)


def test_several_passes_of_tiles_match_oracle(tmp_path, oracle_mod):
    """200 shells are 2 x 2 tiles of each type; a k list over three times the
    components takes more tiles than one pass of the wavefronts."""
    print("\n[gpu] rho_k, several passes", flush=True)
    d = _deck(tmp_path, 33, 20, shells=200, backflow="zero")
    x = pkg("deckgen").lattice_configs(4, d.nptot, d.el[0], 78)
    _check(d, x, oracle_mod)
    kv = np.array(d.kvec, dtype=np.float64).reshape(-1, 2)
    g = pkg("hip").twist_gvec(kv, d.el, 0, 1, 1)
    d.kvec = np.ascontiguousarray(kv * np.where(np.arange(len(kv)) % 2, 1.0, 3.0)[:, None])
    _check(d, x, oracle_mod, gvec=g)
