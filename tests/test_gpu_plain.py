"""Launches whose rows nothing cuts (temperature alone): the split single-read kernel against the
oracle and against the multi-pass path (the single passes switched off), which must agree exactly
in tokens, flags and survivor counts."""
import numpy as np
import pytest

from oracle import sampler as O

pytestmark = pytest.mark.gpu

DT = ("f32", "bf16", "f16")


def _run(x, T, both=True, **kw):
    """The launch on the plain kernel and, with the single passes off, on the multi-pass path."""
    import torch

    from vllm_webgpu_amd import _lib, ops

    L = _lib.lib()
    out = []
    for on in ((1, 0) if both else (1,)):
        before = L.vws_set_single_pass(on)
        try:
            r = ops.sample(x, temperature=T, **kw)
            torch.cuda.synchronize()
        finally:
            L.vws_set_single_pass(before)
        out.append((r.sampled.cpu().numpy(), r.flags.cpu().numpy().view(np.uint32), r.num_kept.cpu().numpy()))
    return out


def _same(a, b):
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1] & 0xFF, b[1] & 0xFF) and np.array_equal(a[2], b[2])


def _logits(cuda, B, V, dtype, scale=3.0, seed=0):
    import torch

    g = torch.Generator(device=cuda).manual_seed(seed * 31 + V)
    x = torch.randn((B, V), generator=g, device=cuda) * scale
    return x.to({"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dtype]), g


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("B,V", [(3, 1), (3, 3), (5, 7), (4, 2047), (3, 8193), (17, 50257), (130, 32001),
                                 (2, 524288), (2100, 1003)])
def test_plain_rows(cuda, dtype, given, B, V):
    """Block and part edges, odd rows of 16-bit logits, one part per row (B > 2048), greedy rows
    among the others, temperatures from 0.02 to 50."""
    import torch

    x, g = _logits(cuda, B, V, dtype)
    T = torch.exp(torch.linspace(-3.9, 3.9, B, device=cuda))
    T[1::5] = 0.0
    if given:
        kw = {"uniforms": torch.randint(0, 1 << 24, (B, V), generator=g, device=cuda).float() * 2.0 ** -24}
    else:
        kw = {"rng_seeds": torch.arange(B, device=cuda) * 977 + V, "rng_offsets": torch.arange(B, device=cuda) << 33}
    fast, slow = _run(x, T, **kw)
    assert not (fast[1] & 0x100).any() and (slow[1] & 0x100).all()
    _same(fast, slow)


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("kind", ["constant", "rounded", "neg_inf", "nan", "inf", "peaked", "ascending", "tiny_T",
                                  "lost_peak", "huge"])
def test_plain_values(cuda, dtype, kind):
    """Rows the short lists cannot decide (equal keys, no finite maximum) and values that reach
    none of the bounds' comparisons."""
    import torch

    B, V = 6, 40003
    x, g = _logits(cuda, B, V, dtype, seed=1)
    T = torch.full((B,), 0.9, device=cuda)
    kw = {"rng_key": 12345}
    if kind == "constant":
        x[:] = 1.25
        x[0] = -float("inf")
        kw = {"uniforms": torch.full((B, V), 0.75, device=cuda)}
        kw["uniforms"][2, 17] = kw["uniforms"][2, 30000] = 0.875
        kw["uniforms"][3] = 0.0
    elif kind == "rounded":
        x = torch.round(x)
        kw = {"uniforms": torch.randint(1, 64, (B, V), generator=g, device=cuda).float() / 64}
    elif kind == "neg_inf":
        x[:, : V - 9] = -float("inf")
        x[1, 1:] = -float("inf")
    elif kind == "nan":
        x[:, ::3] = float("nan")
        x[1] = float("nan")
    elif kind == "inf":
        x[0, 5] = x[0, 9] = float("inf")
        x[1, 7] = float("inf")
        x[1, 3] = float("nan")
    elif kind == "peaked":
        x[:, 123] = 60.0
    elif kind == "lost_peak":
        # u = 0 takes the peak out of the race; the other exponentials are small, subnormal or 0
        x[:, 123] = torch.linspace(60.0, 115.0, B, device=cuda).to(x.dtype)
        kw = {"uniforms": torch.randint(1, 1 << 24, (B, V), generator=g, device=cuda).float() * 2.0 ** -24}
        kw["uniforms"][:, 123] = 0.0
    elif kind == "huge":
        # finite logits whose log2(e) / T multiple is not
        top = torch.finfo(x.dtype).max
        x = x * (top / 64)
        x[:, 100], x[:, 39000] = 0.98 * top, 0.6 * top
        T[:] = 1.0
    elif kind == "ascending":
        x = torch.sort(x, dim=1).values
    else:
        T[:] = 2e-5
    _same(*_run(x, T, **kw))


def _oracle(x, T, u):
    B = x.shape[0]
    one = np.ones(B, np.float32)
    ref = O.sample(x, O.make_params(B, np.full(B, T, np.float32), np.zeros(B, np.int32), one, 0 * one, one, 0 * one,
                                    0 * one), u)
    return ref["token"], ref["flags"], ref["n_kept"]


@pytest.mark.parametrize("dtype", DT)
def test_peak_lost_to_a_zero_exponential(cuda, dtype):
    """Regression: u = 0 takes the peak (token 10) out of the race, and token 100, whose exponential
    is 0 (81 below the peak), has the largest approximate key of its part, above token 200's, the
    row's winner.  Another part's 9000 must not win in its place: its key, 2^-94, is small enough
    for a zero exponential to have hidden a better one."""
    import torch

    B, V = 2, 16384
    rng = np.random.default_rng(8)
    x = rng.normal(-200, 3, (B, V)).astype(np.float32)
    u = (rng.integers(1, 1 << 24, (B, V)) * 2.0 ** -24).astype(np.float32)
    for t, v, w in ((10, 0.0, 0.0), (100, -81.0, 1 - 2.0 ** -24), (200, -79.0, 1 - 12 * 2.0 ** -24),
                    (9000, -79.0, 1 - 16 * 2.0 ** -24)):
        x[:, t], u[:, t] = v, w
    ref = _oracle(x, 1.0, u)
    assert (ref[0] == 200).all()
    xd, _ = _logits(cuda, B, V, dtype)
    xd.copy_(torch.from_numpy(x))
    for got in _run(xd, torch.ones(B, device=cuda), uniforms=torch.from_numpy(u).to(cuda)):
        _same(got, ref)


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_scaled_logits_at_the_edge_of_their_range(cuda, sign):
    """Regression: two neighbouring floats with the same x / T, of which only the one nearer 0 has a
    finite x log2(e) / T, as the largest of a row (positive, or negative above a mask of the
    lowest value).  The token with the infinite product races with the smaller exponential
    variate and wins, whatever the other one's part lists."""
    import torch

    T, lo, hi = (float.fromhex(v) for v in ("0x1.4ccccc0p+0", "0x1.cd5bd6p+127", "0x1.cd5bd8p+127"))
    assert np.float32(lo) / np.float32(T) == np.float32(hi) / np.float32(T)
    B, V = 2, 16384
    rng = np.random.default_rng(9)
    x = rng.normal(0, 3, (B, V)).astype(np.float32)
    if sign < 0:
        x[:] = np.finfo(np.float32).min
    u = (rng.integers(1, 1 << 24, (B, V)) * 2.0 ** -24).astype(np.float32)
    x[:, 10], u[:, 10] = sign * hi, 0.75
    x[:, 9000], u[:, 9000] = sign * lo, 0.25
    ref = _oracle(x, T, u)
    assert (ref[0] == 10).all()
    for got in _run(torch.from_numpy(x).to(cuda), torch.full((B,), T, device=cuda),
                    uniforms=torch.from_numpy(u).to(cuda)):
        _same(got, ref)


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("V", [3, 4099, 16385])
def test_infinite_temperature(cuda, dtype, V):
    """T = +inf makes every finite logit 0 and every infinite one NaN: not counted among the
    survivors, never drawn; rows of infinities alone return their first token."""
    import torch

    B = 6
    xd, g = _logits(cuda, B, V, dtype, seed=5)
    xd[1, 1:] = -float("inf")
    xd[2, V - 2] = float("inf")
    xd[3] = float("inf")
    xd[4, ::2] = float("nan")
    xd[4, 1] = -float("inf")
    xd[5] = -float("inf")
    u = torch.randint(1, 1 << 24, (B, V), generator=g, device=cuda).float() * 2.0 ** -24
    with np.errstate(invalid="ignore"):
        ref = _oracle(xd.float().cpu().numpy(), np.inf, u.cpu().numpy())
    T = torch.full((B,), float("inf"), device=cuda)
    _same(*_run(xd, T, both=False, uniforms=u), ref)
    xd[2, V - 2] = 0.0  # (a +inf logit among finite ones is the plain kernel's and the oracle's case only)
    _same(*_run(xd, T, uniforms=u))
    _same(*_run(xd, T, rng_key=99))


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("V", [1, 3, 6, 1024, 8193, 40003, 262147])
def test_exact_rows(cuda, dtype, V):
    """Rows read again for their exact keys (a uniform outside [0, 1) or NaN, in the first, the last
    and other tokens) and for the first token of their maximum (infinities at every place, NaN
    before them, y = x / T that overflows), odd starts and remainders, one part and several."""
    import torch

    B = 16
    xw, g = _logits(cuda, B, V + 1, dtype, seed=6)
    x = xw[:, 1:] if V > 1 else xw[:, :1].contiguous()
    u = torch.randint(1, 1 << 24, (B, V), generator=g, device=cuda).float() * 2.0 ** -24
    T = torch.exp(torch.linspace(-3.0, 3.0, B, device=cuda))
    inf, nan, at = float("inf"), float("nan"), torch.randint(0, V, (B,), generator=g, device=cuda).tolist()
    for r, v in ((0, 1.0), (1, nan), (2, -0.5), (3, 1.0), (4, 2.0), (5, inf)):
        u[r, at[r]] = v
    u[3, :] = 1.0
    u[6, 0] = u[6, V - 1] = 1.0
    u[7, V - 1] = nan
    x[8, at[8]] = inf
    x[9, at[9]:] = inf
    x[10, V - 1] = x[10, V // 2] = inf
    x[10, : V // 2] = nan
    x[11] = -inf
    x[12, : V // 2] = nan
    x[12, V // 2 :] = -inf
    x[13] = nan
    if dtype != "f16":
        T[14] = T[15] = 0.25
        x[14, at[14]] = 0.9 * torch.finfo(x.dtype).max
        x[15, max(0, V - 3) :] = 0.9 * torch.finfo(x.dtype).max
    _same(*_run(x, T, uniforms=u))
    _same(*_run(x[8:], T[8:], rng_key=5))


def test_plain_oracle(cuda):
    """Full-size rows against the sequential oracle (given uniforms), the whole batch twice (the
    arrival counters are left ready)."""
    import torch

    B, V = 24, 128256
    x, g = _logits(cuda, B, V, "f32", seed=2)
    u = torch.randint(1, 1 << 24, (B, V), generator=g, device=cuda).float() * 2.0 ** -24
    T = np.linspace(0.3, 1.5, B).astype(np.float32)
    one = np.ones(B, np.float32)
    ref = O.sample(x.cpu().numpy(), O.make_params(B, T, np.zeros(B, np.int32), one, 0 * one, one, 0 * one, 0 * one),
                   u.cpu().numpy())
    for _ in range(2):
        got, = _run(x, torch.from_numpy(T).to(cuda), both=False, uniforms=u)
        assert np.array_equal(got[0], ref["token"]) and np.array_equal(got[1] & 0xFF, ref["flags"] & 0xFF)
        assert np.array_equal(got[2], ref["n_kept"])


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("B,V", [(1, 4095), (1, 8192), (3, 8193), (7, 40003), (1, 524288), (128, 9001), (129, 9001),
                                 (256, 9001), (257, 9001), (512, 8191), (513, 8191)])
def test_greedy_launches(cuda, dtype, B, V):
    """Launches without temperatures, the rows split or (short rows, many rows) whole: ties within
    and across parts, zeros of both signs, infinities and NaN; top-k and top-p arrays do not count."""
    import torch

    x, g = _logits(cuda, B, V, dtype, seed=3)
    x[0, V // 2 :: 977] = 50.0
    if B > 2:
        x[1] = -float("inf")
        x[1, V - 1] = float("nan")
        x[2] = -1.0
        x[2, 5], x[2, V - 2] = -0.0, 0.0
    if B > 6:
        x[3] = float("nan")
        x[4, V - 1] = x[4, V - 3] = float("inf")
        x[5, ::2] = float("nan")
        x[5, V - 4 :] = 99.0
    k = torch.full((B,), 3, dtype=torch.int32, device=cuda)
    fast, slow = _run(x, None, top_k=k, top_p=k * 0.25)
    _same(fast, slow)
    f = x.float().nan_to_num(nan=-float("inf"), posinf=float("inf"), neginf=-float("inf")).cpu().numpy()
    ok = np.isfinite(f).any(1) | (f == np.inf).any(1)
    assert np.array_equal(fast[0][ok], f.argmax(1)[ok])


def test_streams_apart(cuda):
    """Split rows of launches on several streams without an order between them: each stream has
    its own workspace, so no launch counts another's parts."""
    import torch

    from vllm_webgpu_amd import ops

    B, V, n = 24, 40003, 3
    xs = [_logits(cuda, B, V, "bf16", seed=4 + i)[0] for i in range(n)]
    T = torch.full((B,), 0.9, device=cuda)
    calls = [{}, {"temperature": T, "rng_key": 7}]
    want = [[ops.sample(x, **kw).sampled.cpu() for kw in calls] for x in xs]
    streams = [torch.cuda.Stream() for _ in range(n)]
    torch.cuda.synchronize()
    got = [[] for _ in range(n)]
    for _ in range(20):
        for s, x, g in zip(streams, xs, got):
            with torch.cuda.stream(s):
                g.extend(ops.sample(x, **kw).sampled for kw in calls)
    torch.cuda.synchronize()
    buffers = set()
    for s in streams:
        with torch.cuda.stream(s):
            buffers.add(ops.workspace(1, torch.device("cuda", torch.cuda.current_device())).data_ptr())
    assert len(buffers) == n
    for w, g in zip(want, got):
        for i, t in enumerate(g):
            assert torch.equal(t.cpu(), w[i % 2])
