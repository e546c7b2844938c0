"""Two electrons of one type at the same place: their type's Laplacian, kinetic
and potential slots are infinite or no numbers, the other type's are what they
are without them.  Decks without orbitals, where no singular determinant ends
the evaluation.  Tolerance 1e-10 relative, as for the reference goldens."""
import os

import numpy as np
import pytest

from conftest import pkg

pytestmark = pytest.mark.gpu

RTOL = 1e-10


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nup,ndown", [(7, 5), (13, 13), (20, 33), (64, 64), (6, 0)])
def test_other_type_stays_finite(nup, ndown, precision, tmp_path, oracle_mod):
    print(f"\n[gpu] coincident electrons {nup}+{ndown}, precision {precision}", flush=True)
    import torch
    dg, deck, hip = pkg("deckgen"), pkg("deck"), pkg("hip")
    path = os.path.join(str(tmp_path), "deck")
    dg.make_deck(path, "co", nup, ndown, 2.0, 10, jastrow="pade", u3=False)
    d = deck.read_deck(path)
    d.iub[:] = 0
    x = dg.lattice_configs(3, d.nptot, d.el[0], 3)
    x[1, 1] = x[1, 0]
    if ndown:
        x[2, nup + 1] = x[2, nup]
    o = oracle_mod.Oracle(d, twist=(1, 1))
    ref, i = o.eval(x), o.info
    ctx = hip.Context(d, twist=(1, 1))
    xd = torch.tensor(x, device="cuda")
    props, g, h = xd.new_zeros((3, ctx.info["n_props"])), torch.zeros_like(xd), xd.new_zeros((3, 2))
    ctx.eval_device(xd, props, g, h, xd.new_zeros(3), precision=precision, stream=torch.cuda.current_stream())
    torch.cuda.synchronize()
    props, h = props.cpu().numpy(), h.cpu().numpy()
    ctx.close()
    tol = RTOL if precision == 0 else 1e-4  # FP32 tables
    for w in (1, 2):
        t = 2 - w  # the type that is not touched
        np.testing.assert_allclose(h[w, t], ref["h"][w, t], rtol=tol)
        if d.np[t] > 0:
            for slot in (i["jkin"][t], i["jun"][t], i["jpot"][t]):
                assert np.isfinite(ref["props"][w, slot - 1])
                np.testing.assert_allclose(props[w, slot - 1], ref["props"][w, slot - 1], rtol=tol)
