"""The drift kernel's forms against the oracle: real and twisted orbitals, one
type or two, particle counts at the edges of its lane blocks, and determinants
that couple to some of the types only.  Tolerance 1e-10 relative, as for the
reference goldens."""
import os

import pytest

from conftest import compare_eval, pkg

pytestmark = pytest.mark.gpu

RTOL = 1e-10


@pytest.mark.parametrize("twist", [(1, 1), (2, 3)])
@pytest.mark.parametrize("nup,ndown,off", [(2, 1, None), (13, 0, None), (16, 16, None), (17, 9, None), (33, 20, None),
                                           (61, 0, None), (13, 13, 2), (37, 29, 2)])
def test_forms_match_oracle(nup, ndown, off, twist, tmp_path, oracle_mod):
    print(f"\n[gpu] drift {nup}+{ndown} twist {twist} off {off}", flush=True)
    dg = pkg("deckgen")
    path = os.path.join(str(tmp_path), "deck")
    dg.make_deck(path, "fg", nup, ndown, 2.0, 20, jastrow="pade", backflow="yk")
    d = pkg("deck").read_deck(path)
    if off is not None:
        d.iub[off] = 0  # one determinant without backflow from the other type
    x = dg.lattice_configs(5, d.nptot, d.el[0], nup + 3 * ndown)
    o = oracle_mod.Oracle(d, twist=twist)
    ref, ns = o.eval(x), o.info["n_scalar_props"]
    gold = dict(scalars=ref["props"][:, :ns], g=ref["g"], h=ref["h"][:, :d.ntypes], grad2_ph=ref["grad2_ph"],
                rhok=ref["props"][:, ns:])
    ctx = pkg("hip").Context(d, twist=twist)
    try:
        out = ctx.eval(x)
    finally:
        ctx.close()
    compare_eval(out, gold, ns, RTOL)
