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
    assert not (got["flags"] & GENERAL).any()


TIE_KINDS = {  # options, and the largest share of the tied rows that takes the multi-pass path
    "plain": ({}, 0.0),
    "softcap": ({"logit_softcap": 30.0}, 0.0),
    "softcap_f16": ({"logit_softcap": 30.0, "logit_softcap_f16": True}, 0.5),
    "mask": ({"mask": True}, 0.0),
    "mask_odd_rows": ({"mask": True, "odd": True}, 1.0),
    "penalties": ({"hist": (1.2, 0.5, 0.3)}, 0.0),
    "penalties_raise": ({"hist": (0.8, -0.5, -0.2)}, 1.0),
    "bans": ({"bans": True}, 0.0),
    "table": ({"table": (1.2, 0.5, 0.3)}, 0.0),
    "table_raise": ({"table": (0.8, -0.5, -0.2)}, 1.0),
    "softcap_table": ({"logit_softcap": 30.0, "table": (1.2, 0.5, 0.3)}, 0.0),
    "logprobs": ({"num_logprobs": 5}, 0.0),
    "logprobs_mask": ({"num_logprobs": 5, "mask": True}, 1.0),
    "logprobs_penalties": ({"num_logprobs": 20, "hist": (1.2, 0.5, 0.3)}, 1.0),
    "logprobs_softcap": ({"num_logprobs": 5, "logit_softcap": 30.0}, 1.0),
}


@pytest.mark.parametrize("B", [6, 300])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("kind", TIE_KINDS)
def test_ties_under_every_option(cuda, kind, dtype, B):
    """Rows with more than 64 members tied at the k-th value under each option that changes how row_fast
    packs, masks or leaves its rows, among rows of every other kind in batches past the compute
    units: as the multi-pass path has them.  Where row_fast's early returns do not apply, the tied
    rows stay off that path (f16-rounded caps: unless the seed is the tied value, whose
    neighbours below round to it)."""
    import torch

    from vllm_webgpu_amd import _lib, ops

    opt, most = TIE_KINDS[kind]
    opt = dict(opt)
    V, k, ntie = 262144, 50, 90
    g = torch.Generator(device=cuda).manual_seed(len(kind) * 7 + B)
    odd = opt.pop("odd", False)
    x = torch.randn((B, V + odd), generator=g, device=cuda)
    x = x.to({"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dtype])[:, odd:]
    at = torch.stack([torch.randperm(V, generator=g, device=cuda)[: ntie + k // 2] for _ in range(B)])
    x.scatter_(1, at[:, :ntie], 7.0)
    x.scatter_(1, at[:, ntie:], (7.5 + torch.rand((B, k // 2), generator=g, device=cuda)).to(x.dtype))
    K = torch.full((B,), k, dtype=torch.int32, device=cuda)
    T = torch.full((B,), 0.8, device=cuda)
    if B > 6:
        K[1::4], K[2::4], T[3::8] = 0, 200, 0.0
    tied = (K == k) & (T > 0)
    kw = {"temperature": T, "top_k": K, "top_p": torch.full((B,), 0.9, device=cuda), "rng_key": 11}
    if opt.pop("mask", False):
        ok = torch.rand((B, V), generator=g, device=cuda) < 0.5
        ok.scatter_(1, at[:, : ntie - 10], True)
        kw["allowed_mask"] = ops.pack_allowed(ok)
    if opt.pop("bans", False):
        kw["adjust_ids"] = torch.cat([at[:, :5], at[:, -3:]], 1).int()
        kw["adjust_vals"] = torch.full((B, 8), -float("inf"), device=cuda)
    pen = opt.get("hist") or opt.get("table")
    if pen:
        ids = torch.cat([at[:, :20], at[:, -4:], torch.randint(0, V, (B, 40), generator=g, device=cuda)], 1).int()
        for name, v in zip(("repetition_penalty", "presence_penalty", "frequency_penalty"), pen):
            kw[name] = torch.full((B,), v, device=cuda)
        if opt.pop("hist", None):
            kw["output_ids"] = ids
        else:
            opt.pop("table")
            state = torch.zeros((B, V), dtype=torch.int32, device=cuda)
            bits = torch.zeros((B, (V + 31) // 32), dtype=torch.int32, device=cuda)
            rows = torch.arange(B, device=cuda, dtype=torch.int32).repeat_interleave(ids.shape[1])
            ops.token_state_update(state, ids.reshape(-1), rows=rows, bits=bits)
            kw.update(token_state=state, token_state_bits=bits)
    kw.update(opt)
    L = _lib.lib()
    got = []
    for on in (1, 0):
        before = L.vws_set_single_pass(on)
        try:
            r = ops.sample(x, **kw)
            torch.cuda.synchronize()
        finally:
            L.vws_set_single_pass(before)
        got.append(r)
    a, b = got
    assert torch.equal(a.sampled, b.sampled) and torch.equal(a.num_kept, b.num_kept)
    assert torch.equal(a.flags & 0xFF, b.flags & 0xFF)
    assert ((b.flags[tied] & GENERAL) != 0).all()
    if a.logprob_ids is not None:
        assert torch.equal(a.logprob_ids, b.logprob_ids) and torch.equal(a.logprob_ranks, b.logprob_ranks)
        torch.testing.assert_close(a.logprob_vals, b.logprob_vals, rtol=1e-5, atol=1e-6)
    if "raise" not in kind:  # (raised tokens: the cut leaves none of the ties)
        assert int((a.num_kept[tied] > 60).sum()) >= int(tied.sum()) // 2
    left = ((a.flags[tied] & GENERAL) != 0).float().mean().item()
    assert left <= most and (left == 1.0 or kind not in ("table_raise", "logprobs_softcap")), left
