"""Evaluations, refreshes and moves depend on their inputs alone: repeated from
the same state they give the same bits, whichever wavefront arrives first."""
import pytest

from conftest import pkg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("twist", [(1, 1), (2, 3)])
@pytest.mark.parametrize("nup,ndown", [(13, 13), (29, 29), (33, 17), (61, 61)])
def test_repeats_give_the_same_bits(tmp_path, nup, ndown, twist):
    print(f"\n[gpu] repeats {nup}+{ndown} twist {twist}", flush=True)
    import torch
    hip, dg, deck = pkg("hip"), pkg("deckgen"), pkg("deck")
    nw, out = 512, {}
    for backflow in ("yk", "zero"):
        path = tmp_path / backflow
        dg.make_deck(str(path), "rp", nup, ndown, 2.0, 30, jastrow="pade", backflow=backflow,
                     ntwists=4 if twist != (1, 1) else 0)
        d = deck.read_deck(str(path))
        ctx = hip.Context(d, twist=twist)
        x = dg.lattice_configs(nw, d.nptot, d.el[0], 11)
        wk = hip.Walkers(ctx, x, [2 * k + 12345 for k in range(nw)])
        sm = hip.SingleMoves(wk)
        start = [t.clone() for t in (wk.x, wk.rng)]
        for k in range(15):
            for t, s in zip((wk.x, wk.rng), start):
                t.copy_(s)
            sm.dlogpsi.zero_()
            wk.start()
            sm.refresh()
            fresh = [wk.props.clone(), wk.g.clone(), wk.h.clone(), sm.ainv.clone()]
            sm.moves(0, min(8, d.nptot), 0.4)
            got = fresh + [t.clone() for t in (wk.x, wk.rng, sm.ainv, sm.dlogpsi, wk.props)]
            if k == 0:
                out = got
            for a, b in zip(out, got):
                assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)) if a.is_floating_point() else torch.equal(a, b)
        wk = sm = None
        ctx.close()
