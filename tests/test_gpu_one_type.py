"""The pair kernel's form for particles of one type: either type empty or a deck
of one type, at the edges of the lane blocks, one chunk of phases and several,
k lists on the grid and off it, against the oracle; the empty type's rho_k is
zero whatever its buffer held.  Tolerance 1e-10 relative, as for the reference
goldens."""
import os

import numpy as np
import pytest

from conftest import compare_eval, pkg

pytestmark = pytest.mark.gpu

RTOL = 1e-10


@pytest.mark.parametrize("shells", [20, 120])
@pytest.mark.parametrize("nup,ndown", [(1, 0), (2, 0), (16, 0), (17, 0), (32, 0), (33, 0), (64, 0), (0, 5), (0, 33)])
def test_one_type_matches_oracle(nup, ndown, shells, tmp_path, oracle_mod):
    print(f"\n[gpu] one type {nup}+{ndown}, {shells} shells", flush=True)
    dg, deck = pkg("deckgen"), pkg("deck")
    path = os.path.join(str(tmp_path), "deck")
    n = nup + ndown
    dg.make_deck(path, "ot", n, 0, 2.0, shells, jastrow="pade", u3=n != 17)
    d = deck.read_deck(path)
    if ndown:
        d.np[:2] = [0, ndown]
    x = dg.lattice_configs(6, n, d.el[0], 7 * n + shells)
    for off_grid in (False, True):
        g = pkg("hip").twist_gvec(np.array(d.kvec).reshape(-1, 2), d.el, 0, 1, 1)
        if off_grid:
            kv = np.array(d.kvec, dtype=np.float64).reshape(-1, 2)
            d.kvec = np.ascontiguousarray(np.concatenate([np.repeat(kv[:1], 5, axis=0), kv[5:]]))
        o = oracle_mod.Oracle(d, twist=(1, 1), gvec=g)
        ref, ns = o.eval(x), o.info["n_scalar_props"]
        gold = dict(scalars=ref["props"][:, :ns], g=ref["g"], h=ref["h"][:, :d.ntypes], grad2_ph=ref["grad2_ph"],
                    rhok=ref["props"][:, ns:])
        ctx = pkg("hip").Context(d, twist=(1, 1), gvec=g)
        try:
            out = ctx.eval(x)
        finally:
            ctx.close()
        compare_eval(out, gold, ns, RTOL, f"{nup}+{ndown} off grid {off_grid}")


@pytest.mark.parametrize("precision", [0, 1])
def test_empty_types_rho_is_zero(tmp_path, precision):
    print(f"\n[gpu] rho_k of an empty type, precision {precision}", flush=True)
    import torch
    dg, deck, hip = pkg("deckgen"), pkg("deck"), pkg("hip")
    path = os.path.join(str(tmp_path), "deck")
    dg.make_deck(path, "ot", 21, 0, 2.0, 30, jastrow="pade")
    d = deck.read_deck(path)
    ctx = hip.Context(d, twist=(1, 1))
    x = torch.tensor(dg.lattice_configs(4, 21, d.el[0], 5), device="cuda")
    ns, nk = ctx.info["n_scalar_props"], len(d.kvec)
    out = []
    for fill in (0.0, 77.0):
        props, g, h = x.new_full((4, ctx.info["n_props"]), fill), torch.zeros_like(x), x.new_zeros((4, 2))
        ctx.eval_device(x, props, g, h, x.new_zeros(4), precision=precision, stream=torch.cuda.current_stream())
        torch.cuda.synchronize()
        out.append(props[:, ns:].cpu().numpy())
    ctx.close()
    assert out[0].shape[1] == 4 * nk
    assert np.array_equal(out[0], out[1])
    assert (out[1][:, 2 * nk:] == 0.0).all() and np.abs(out[1][:, :2 * nk]).min() > 0.0
