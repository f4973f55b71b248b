"""Rows with k <= 64 whose members tied at the k-th value exceed the 64 slots of the one-wave finish
(common with 16-bit logits): finished from the single pass's candidates.  Ids, flags, counts,
logprob ids and ranks exactly as the oracle's."""
import numpy as np
import pytest

from tests.cases import _wl
from tests.common import assert_same, gpu_run, oracle_run

pytestmark = pytest.mark.gpu

GENERAL = 0x100


@pytest.mark.parametrize("num_logprobs", [None, 5])
@pytest.mark.parametrize("ntie,k,p,min_p", [(65, 64, 0.9, 0.0), (64, 64, 0.5, 0.0), (90, 50, 1.0, 0.02),
                                            (400, 20, 0.95, 0.0), (300, 64, 0.0, 0.0), (120, 1, 0.7, 0.0)])
def test_ties_past_the_slots(cuda, ntie, k, p, min_p, num_logprobs):
    """ntie copies of one value just below the k // 2 largest: the top k, ties kept, has more
    members than one wave holds (65 is the smallest such row)."""
    rng = np.random.default_rng(ntie * 3 + k)
    B, V = 5, 60000
    x = rng.normal(0, 1, (B, V)).astype(np.float32)
    for b in range(B):
        at = rng.choice(V, size=ntie + k // 2, replace=False)
        x[b, at[:ntie]] = 7.0
        x[b, at[ntie:]] = 7.5 + rng.random(k // 2).astype(np.float32)
    w = _wl(f"ties{ntie}_k{k}", x, np.full(B, 0.8, np.float32), k=k, p=p, mp=min_p, seed=k)
    got = gpu_run(w, cuda, num_logprobs=num_logprobs)
    assert_same(got, oracle_run(w, num_logprobs=num_logprobs), w.name)
    if num_logprobs is None:
        assert not (got["flags"] & GENERAL).any()
