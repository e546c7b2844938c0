"""The largest population whose branching fits a workgroup's LDS branches as the
oracle does; one more walker is refused and leaves the buffers as they are."""
import numpy as np
import pytest

from conftest import load_deck, pkg

pytestmark = pytest.mark.gpu

FITS = (163840 - 8208) // 12


@pytest.mark.parametrize("n", [FITS, FITS + 1, 13500])
def test_population_limit(oracle_mod, n):
    print(f"\n[gpu] branching of {n} walkers", flush=True)
    import torch
    hip, abi = pkg("hip"), pkg("abi")
    w = np.random.default_rng(n).uniform(0.0, 3.0, n)
    limbs = [11, 22, 33, 2 * n + 1]
    ctx = hip.Context(load_deck("n26g"), twist=(1, 1))
    wt = torch.tensor(w, device="cuda")
    rng2 = torch.tensor([abi.limbs_to_state(limbs)], dtype=torch.int64, device="cuda")
    src = torch.full((n,), -7, dtype=torch.int32, device="cuda")
    counts = torch.zeros(4, dtype=torch.int32, device="cuda")
    if n <= FITS:
        want, nmult, limbs2, _ = oracle_mod.branch2(w, limbs)
        hip.dmc_branch(ctx, wt, rng2, src, counts)
        torch.cuda.synchronize()
        assert np.array_equal(src.cpu().numpy(), want)
        assert int(counts[1].item()) == nmult
        assert abi.state_to_limbs(int(rng2.item())) == limbs2
    else:
        with pytest.raises(hip.QmcError) as e:
            hip.dmc_branch(ctx, wt, rng2, src, counts)
        assert e.value.code == abi.QMC_ERR_LIMIT
        torch.cuda.synchronize()
        assert bool((src == -7).all()) and int(rng2.item()) == abi.limbs_to_state(limbs)
    ctx.close()
