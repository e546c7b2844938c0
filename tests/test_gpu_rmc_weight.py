"""The path weight of a reptation move of up to 64 beads (the largest mdelta):
the weight in the trace is the sum over the links of the beads the path leaves
and grows (reptation.f:2105-2160), formed in numpy from the links the move left
behind, in all three propagator forms; the ends follow the decision."""
import numpy as np
import pytest

from conftest import load_deck, pkg

pytestmark = pytest.mark.gpu

BRA, DTP, ITP, LNG, NDS = range(5)


@pytest.mark.parametrize("mdelta,ntau", [(1, 2), (33, 40), (64, 20), (64, 80)])
@pytest.mark.parametrize("driver", [{}, {"wpiu": ["1"]}, {"gstorto": ["1"], "nodalaction": ["1"]}])
def test_weight_of_long_moves(mdelta, ntau, driver):
    print(f"\n[gpu] path weight, mdelta {mdelta}, {ntau} beads, {driver}", flush=True)
    import torch
    hip, abi = pkg("hip"), pkg("abi")
    d = load_deck("n26g")
    nr = 24
    ctx = hip.Context(d, twist=(1, 1))
    rng = np.random.default_rng(mdelta + ntau)
    x0 = pkg("deckgen").lattice_configs(nr, d.nptot, d.el[0], 5)
    rep = hip.Reptiles(ctx, nr, ntau, mdelta, [abi.limbs_to_state([3535, 3467, 3262, 2 * r + 1]) for r in range(nr)])
    prm = hip.rmc_params(0.002, -0.3, 1e30, 1e30, 0, mdelta, driver)
    rep.start(x0[:, None] + 0.002 * rng.standard_normal((nr, ntau) + x0.shape[1:]), prm)
    jltf, nbuf = ctx.info["jltf"] - 1, ntau + mdelta
    half, one, on, m = 0.5, 0.0, 0.0, 0.0
    if "wpiu" in driver:
        m = 0.5
    elif driver:
        half, one, on = 0.0, 1.0, 1.0
    longest = 0
    for _ in range(3):
        torch.cuda.synchronize()
        ends = rep.ends.cpu().numpy().copy()
        tr = rep.sweep(1, prm, trace=True)
        torch.cuda.synchronize()
        tr, w, ltf = tr.cpu().numpy()[0], rep.w.cpu().numpy(), rep.props.cpu().numpy()[:, :, jltf]
        after = rep.ends.cpu().numpy()
        for r in range(nr):
            idir, nd, wn = int(tr[r, 0]), int(tr[r, 1]), tr[r, 2]
            assert 1 <= nd <= mdelta
            longest = max(longest, nd)
            jf, jl = (int(e) for e in ends[r])
            at = lambda j: w[r, j % nbuf]
            kf, kl = (jf + idir * nd) % nbuf, (jl + idir * nd) % nbuf
            t = [-ltf[r, kf] * (1 + 2 * m), -ltf[r, kl] * (1 - 2 * m), ltf[r, jf] * (1 + 2 * m), ltf[r, jl] * (1 - 2 * m)]
            for i in range(1, nd + 1):
                if idir == 1:
                    a, b, c, e = at(jf + i - 1), at(jf + i), at(jl + i - 1), at(jl + i)
                    t += [-a[BRA], -a[DTP] * (half + m), b[ITP] * (one + half + m), -a[LNG] * one, a[NDS] * on,
                          c[BRA], -c[DTP] * (one + half - m), e[ITP] * (half - m), c[LNG] * one, -c[NDS] * on]
                else:
                    a, b, c, e = at(jl - i + 1), at(jl - i), at(jf - i + 1), at(jf - i)
                    t += [-b[BRA], b[DTP] * (one + half - m), -a[ITP] * (half - m), -b[LNG] * one, b[NDS] * on,
                          e[BRA], e[DTP] * (half + m), -c[ITP] * (one + half + m), e[LNG] * one, -e[NDS] * on]
            # every addition rounds a partial sum no larger than the terms' sizes
            assert abs(wn - sum(t)) <= 2 * len(t) * 2.0 ** -53 * np.abs(t).sum()
            moved = tr[r, 3] == 0.0
            assert tuple(after[r]) == ((kf, kl) if moved else (jf, jl))
    assert longest >= min(mdelta, 60)
    rep = None
    ctx.close()
