"""Host-pointer evaluations on both sides of the pinned buffer's size: the same
configurations one call at a time, in a batch that fits it and in one that does
not give the same numbers, and no walker's outputs move into another's."""
import importlib
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
deck = importlib.import_module("2degas_amd.deck")
dg = importlib.import_module("2degas_amd.deckgen")


@pytest.mark.parametrize("nw", [1, 3, 378, 379, 400])
def test_stage_sizes(nw):
    hip = importlib.import_module("2degas_amd.hip")
    d = deck.read_deck(os.path.join(ROOT, "tests", "golden", "decks", "n26"))
    x = dg.random_configs(nw, d.nptot, d.el[0], 11)
    gin = np.linspace(1.0, 2.0, nw)
    ctx = hip.Context(d, twist=(1, 1), device=0)
    a = ctx.eval(x, grad2_in=gin)
    ws = sorted({0, nw // 2, nw - 1})
    b = ctx.eval(x[ws], grad2_in=gin[ws])
    for k in ("props", "g", "h", "grad2_ph", "status"):
        np.testing.assert_array_equal(a[k][ws], b[k], err_msg=k)
    assert np.isfinite(a["props"]).all() and np.abs(a["g"]).min(axis=(1, 2)).all()
    ctx.close()
