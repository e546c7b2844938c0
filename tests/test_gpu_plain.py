"""Evaluations without backflow (every table zero), whose determinant terms
k_final takes from F's diagonal: real orbitals, twisted (complex) ones, an open
shell, unequal spins, one spin empty, one particle of a spin (no pairs of its
own), against the oracle.  Tolerance 1e-10 relative, as for the reference
goldens."""
import os

import numpy as np
import pytest

from conftest import compare_eval, pkg

pytestmark = pytest.mark.gpu

RTOL = 1e-10


@pytest.mark.parametrize("nup,ndown,twists", [(13, 13, 0), (13, 13, 4), (12, 10, 0), (29, 5, 4), (61, 61, 0), (64, 64, 4),
                                              (37, 0, 0), (37, 0, 4), (9, 1, 0), (1, 1, 4)])
def test_plain_matches_oracle(nup, ndown, twists, tmp_path, oracle_mod):
    print(f"\n[gpu] plain {nup}+{ndown}, {twists} twists", flush=True)
    dg, deck, hip = pkg("deckgen"), pkg("deck"), pkg("hip")
    path = os.path.join(str(tmp_path), "deck")
    dg.make_deck(path, "pl", nup, ndown, 1.5, 30, jastrow="pade", backflow="zero", ntwists=twists, u3=nup != 29)
    d = deck.read_deck(path)
    x = dg.lattice_configs(8, d.nptot, d.el[0], 90 + nup + ndown)
    tw = (1, 2) if twists else (1, 1)
    o = oracle_mod.Oracle(d, twist=tw)
    ref, ns = o.eval(x), o.info["n_scalar_props"]
    gold = dict(scalars=ref["props"][:, :ns], g=ref["g"], h=ref["h"][:, :d.ntypes], grad2_ph=ref["grad2_ph"],
                rhok=ref["props"][:, ns:])
    ctx = hip.Context(d, twist=tw)
    try:
        out = ctx.eval(x)
    finally:
        ctx.close()
    compare_eval(out, gold, ns, RTOL)
    assert np.array_equal(out["status"], ref["status"])
