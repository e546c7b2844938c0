"""Tuning the move kernel's tile where it makes no difference: FP64 inverses of
real orbitals have one shape, so the tuner times that, and the tile in force
stays for the orbitals that use it."""
import pytest

from conftest import pkg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [None, 2, 4])
@pytest.mark.parametrize("nu,rows", [(21, 32), (37, 64)])
def test_real_rows_keep_the_tile(tmp_path, nu, rows, tile):
    print(f"\n[gpu] tile of real rows, {rows} rows, {tile}", flush=True)
    hip, dg, deck, abi = pkg("hip"), pkg("deckgen"), pkg("deck"), pkg("abi")
    dg.make_deck(str(tmp_path), "tl", nu, nu, 5.0, 5, nshell_k=12, u3=False, backflow="zero", jastrow="pade")
    d = deck.read_deck(str(tmp_path))
    ctx = hip.Context(d, twist=(1, 1))
    assert hip.real_orbitals(ctx.gvec, d.np[:d.ntypes])
    wk = hip.Walkers(ctx, dg.lattice_configs(8, d.nptot, d.el[0], 3), [2 * k + 12345 for k in range(8)])
    wk.start()
    sm, sm32 = hip.SingleMoves(wk), hip.SingleMoves(wk, precision=abi.QMC_PREC_MIXED)
    if tile is not None:
        sm.set_tile(rows, tile)
    before = dict(ctx.tiles)
    times, best = sm.tune_tile(0.5, sweeps=1)
    assert times[2] == times[4] > 0.0
    assert best == (tile or {32: 2, 64: 4}[rows])
    assert ctx.tiles == before
    # FP32 inverses are complex: both shapes are timed, the faster is kept
    times, best = sm32.tune_tile(0.5, sweeps=1)
    assert set(times) == {2, 4} and best == min(times, key=times.get)
    assert ctx.tiles[abi.QMC_PREC_MIXED, rows] == best
    wk = sm = sm32 = None
    ctx.close()
