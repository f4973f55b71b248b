"""The standalone operations whose rows are split over several workgroups, at the edges of their
parts."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("B,V", [(3, 2048), (3, 2049), (2, 8191), (2, 8192), (3, 8193), (2, 16385),
                                 (130, 32001), (1, 524288)])
def test_softmax_parts(cuda, dtype, B, V):
    """Parts of a row (8192 elements at most, odd row starts, the smallest and largest row) against
    float64: |y - max| <= 80 rounds by 80 * 2^-24 = 4.8e-6 in a term and, averaged, in the sum
    (rtol 1e-5).  One row has a part of -inf, one a NaN, one +inf (its probabilities are NaN)."""
    import torch

    from vllm_webgpu_amd import ops

    g = torch.Generator(device=cuda).manual_seed(V)
    x = torch.randn((B, V), generator=g, device=cuda) * 3
    if B > 1:
        x[0, : V // 2] = -float("inf")
        x[1, V - 1] = float("nan")
    if B > 2:
        x[2, V // 3] = float("inf")
    x = x.to({"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dtype])
    T = torch.linspace(0.7, 1.3, B, device=cuda)
    p, rm, ls = ops.softmax(x, T)
    y = (x.float() / T[:, None]).double()
    m = torch.nan_to_num(y, nan=-float("inf"), posinf=float("inf")).amax(1)
    assert torch.equal(rm.double(), m)
    e = torch.nan_to_num(torch.exp(y - m[:, None]), nan=0.0)
    ok = torch.isfinite(m)
    S = e.sum(1)
    torch.testing.assert_close(p[ok].double(), (e / S[:, None])[ok], rtol=1e-5, atol=1e-12)
    torch.testing.assert_close(ls[ok].double(), S[ok].log(), rtol=1e-6, atol=5e-6)
    if B > 2:
        assert torch.isnan(p[2]).all() and ls[2] == -float("inf")


@pytest.mark.parametrize("V", [20000, 50000])
def test_softmax_over_its_logits(cuda, V):
    """Probabilities written over the logits (the C entry accepts the same buffer twice) are those
    of separate buffers: the same elements and exponentials, S summed in another order (1e-6)."""
    import torch

    from vllm_webgpu_amd import _lib, ops

    x = torch.randn((5, V), device=cuda) * 3
    want, _, _ = ops.softmax(x)
    _lib.check(_lib.lib().vws_softmax(x.data_ptr(), _lib.DTYPE_F32, 5, V, V, None, x.data_ptr(), None,
                                      None, torch.cuda.current_stream().cuda_stream))
    torch.testing.assert_close(x, want, rtol=1e-6, atol=1e-12)


@pytest.mark.parametrize("V", [1, 2047, 2049, 8193, 32000, 32768, 32769, 150001])
@pytest.mark.parametrize("inplace", [True, False])
def test_softmax_one_workgroup_a_row(cuda, V, inplace):
    """The forms of one workgroup per row, which rows above 2048 elements reach only where the
    probabilities overlap the logits (held in registers up to 32768 less the row's edges, the
    two-read path with its online maximum and normaliser above), against the oracle beside the
    split form: -inf and NaN elements, a row of one finite value, ascending values (every
    thread's maximum rises at each of its own), temperatures, the row maximum and log-sum."""
    import torch

    from oracle import sampler as O
    from vllm_webgpu_amd import _lib

    rng = np.random.default_rng(V)
    B = 6
    x = (rng.normal(size=(B, V)) * 3).astype(np.float32)
    x[1, ::7] = -np.inf
    x[1, V // 2] = 1.0
    x[2, V // 3] = np.nan if V > 3 else 0.5
    x[3, :] = -np.inf
    x[3, min(77, V - 1)] = 2.5
    x[4] = np.sort(x[4])
    T = np.array([1.0, 0.7, 1.5, 1.0, 0.9, 3.0], np.float32)
    t, Td = torch.from_numpy(x).to(cuda), torch.from_numpy(T).to(cuda)
    out = t if inplace else torch.empty_like(t)
    rm, ls = torch.empty(B, device=cuda), torch.empty(B, device=cuda)
    _lib.check(_lib.lib().vws_softmax(t.data_ptr(), _lib.DTYPE_F32, B, V, V, Td.data_ptr(), out.data_ptr(),
                                      rm.data_ptr(), ls.data_ptr(), torch.cuda.current_stream().cuda_stream))
    p, rm, ls = out.cpu().numpy(), rm.cpu().numpy(), ls.cpu().numpy()
    for b in range(B):
        rp, rrm, rls = O.softmax(x[b:b + 1], float(T[b]))
        # the same exponentials as the oracle's, their sum in another order and its reciprocal once
        np.testing.assert_allclose(p[b], rp[0], rtol=1e-6, atol=1e-12)
        assert rm[b] == rrm[0]
        np.testing.assert_allclose(ls[b], rls[0], rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("kind", ["noise", "ties", "constant", "sparse"])
@pytest.mark.parametrize("B,V,k", [(1, 7, 7), (3, 257, 256), (3, 4097, 1), (16, 128257, 20), (9, 70001, 100),
                                   (2, 262144, 256), (700, 33000, 40)])
def test_topk_parts(cuda, dtype, kind, B, V, k):
    """Row parts, their cut, the merge's cut and the exact selection of rows whose lists overflow
    (heavy ties), against a stable sort: values and ids exactly."""
    import torch

    from vllm_webgpu_amd import ops

    g = torch.Generator(device=cuda).manual_seed(V + k)
    x = torch.randn((B, V), generator=g, device=cuda) * 3
    if kind == "ties":
        x = torch.round(x)
    elif kind == "constant":
        x[:] = 1.5
        x[0, V - 1] = 2.0
    elif kind == "sparse":
        x = torch.where(torch.rand((B, V), generator=g, device=cuda) < 0.5 * k / V, x, -float("inf"))
    x = x.to(torch.float32 if dtype == "f32" else torch.bfloat16)
    for _ in range(2):  # the counters are left ready for the next call
        vals, ids = ops.topk(x, k)
        want, order = torch.sort(x.float(), dim=1, descending=True, stable=True)
        assert torch.equal(vals, want[:, :k]) and torch.equal(ids.long(), order[:, :k])
