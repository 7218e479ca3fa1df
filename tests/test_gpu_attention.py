"""The prompt's matrix-core attention (aos_launch_attention with prefill set) against float64: tiles of 128
tokens and 64 positions at their edges, both head_dims, GQA groups and a cache that already holds positions.
The result is one bfloat16 rounding (half a unit in the last of 8 significant bits: at most 2^-8 of the value) of
sums whose products are exact and whose float32 errors stay below 1e-5 of the largest value. A cache holding infinities takes the wave per (token, head), which
must agree with that kernel's own launch on every output and take no longer; the launches that append to the
cache report such values until the cache is emptied."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P, I, F = C.c_void_p, C.c_int, C.c_float


class Attn(C.Structure):
    _fields_ = [("q", P), ("kc", P), ("vc", P), ("T", I), ("nh", I), ("nkv", I), ("hd", I), ("offset", I), ("max_seq", I),
                ("splits", I), ("chunk", I), ("scale", F), ("part", P), ("out", P), ("counters", P), ("rope_fused", I),
                ("qb", P), ("kb", P), ("vb", P), ("bq", P), ("bk", P), ("bv", P), ("inv_freq", P), ("nonfinite", P),
                ("prefill", I)]


class Rope(C.Structure):
    _fields_ = [("q", P), ("k", P), ("v", P), ("bq", P), ("bk", P), ("bv", P), ("inv_freq", P), ("T", I), ("nh", I),
                ("nkv", I), ("hd", I), ("offset", I), ("max_seq", I), ("qr", P), ("kc", P), ("vc", P), ("nonfinite", P)]


class Ctx(C.Structure):
    _fields_ = [("stream", P), ("a", P), ("b", P)]


def _attention(hip, q, kc, vc, nkv, offset, flag, prefill):
    import torch

    T, nh, hd = q.shape
    out = torch.full((T, nh, hd), -7.0, dtype=torch.bfloat16, device="cuda")
    end = offset + T
    p = Attn(q=q.data_ptr(), kc=kc.data_ptr(), vc=vc.data_ptr(), T=T, nh=nh, nkv=nkv, hd=hd, offset=offset,
             max_seq=kc.shape[1], splits=1, chunk=(end + 63) // 64 * 64, scale=hd ** -0.5, out=out.data_ptr(),
             nonfinite=flag.data_ptr(), prefill=prefill)
    assert hip.lib().aos_launch_attention(C.byref(p), C.byref(Ctx(None, None, None))) == 0
    torch.cuda.synchronize()
    return out.float().cpu().numpy()


def _inputs(hd, nh, nkv, T, offset, spare):
    import torch

    g = torch.Generator(device="cuda").manual_seed(hd * 1000 + T)
    q = 2.0 * torch.randn((T, nh, hd), generator=g, device="cuda")
    kc, vc = (torch.randn((nkv, offset + T + spare, hd), generator=g, device="cuda").bfloat16() for _ in range(2))
    return q, kc, vc


def _reference(q, kc, vc, nkv, offset):
    import torch

    T, nh, hd = q.shape
    q, k, v = q.double().cpu(), kc.double().cpu(), vc.double().cpu()
    out = torch.empty((T, nh, hd), dtype=torch.float64)
    later = torch.arange(offset + T)[None, :] > offset + torch.arange(T)[:, None]
    for h in range(nh):
        s = q[:, h] @ k[h // (nh // nkv), : offset + T].T * hd ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(later, -torch.inf), dim=1) @ v[h // (nh // nkv), : offset + T]
    return out.numpy()


@pytest.mark.parametrize("hd,nh,nkv,T,offset", [
    (128, 2, 1, 1, 0), (64, 4, 2, 127, 0), (64, 2, 2, 128, 63), (64, 6, 2, 129, 1), (128, 7, 1, 33, 64),
    (128, 2, 2, 257, 190), (128, 4, 1, 32, 0)])
def test_prompt_attention(hip, hd, nh, nkv, T, offset):
    import torch

    q, kc, vc = _inputs(hd, nh, nkv, T, offset, 5)
    kc[:, offset + T :] = float("nan")  # positions past the end are not read
    vc[:, offset + T :] = float("nan")
    flag = torch.zeros(1, dtype=torch.int32, device="cuda")
    got = _attention(hip, q, kc, vc, nkv, offset, flag, 1)
    ref = _reference(q, kc, vc, nkv, offset)
    tol = 2.0 ** -8 * np.abs(ref) + 1e-5 * float(vc[:, : offset + T].float().abs().max())
    assert (np.abs(got - ref) <= tol).all(), float((np.abs(got - ref) / tol).max())
    # the wave per (token, head) of the same launch
    flag.fill_(1)
    got = _attention(hip, q, kc, vc, nkv, offset, flag, 1)
    assert (np.abs(got - ref) <= tol).all(), float((np.abs(got - ref) / tol).max())


def test_prompt_attention_nonfinite(hip):
    import torch

    q, kc, vc = _inputs(64, 2, 1, 150, 0, 0)
    vc[0, 70, 3] = float("inf")
    kc[0, 140, 5] = float("-inf")
    flag = torch.ones(1, dtype=torch.int32, device="cuda")
    got = _attention(hip, q, kc, vc, 1, 0, flag, 1)
    ref = _attention(hip, q, kc, vc, 1, 0, flag, 0)
    assert np.isfinite(got[:70]).all() and not np.isfinite(got[70:, :, 3]).any()
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    ok = np.isfinite(ref)
    assert (np.abs(got[ok] - ref[ok]) <= 2.0 ** -7 * np.abs(ref[ok]) + 1e-5 * 5).all()  # two roundings


@pytest.mark.parametrize("bad", [None, "k", "v"])
def test_rope_reports_nonfinite(hip, bad):
    import torch

    T, nh, nkv, hd = 3, 2, 1, 64
    t = {n: torch.randn((T, h * hd), device="cuda").bfloat16() for n, h in (("q", nh), ("k", nkv), ("v", nkv))}
    if bad:
        t[bad][2, 63] = float("inf") if bad == "k" else float("nan")
    freq = torch.ones(hd // 2, device="cuda")
    qr = torch.empty((T, nh, hd), device="cuda")
    kc, vc = (torch.zeros((nkv, T, hd), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    flag = torch.zeros(1, dtype=torch.int32, device="cuda")
    p = Rope(q=t["q"].data_ptr(), k=t["k"].data_ptr(), v=t["v"].data_ptr(), inv_freq=freq.data_ptr(), T=T, nh=nh, nkv=nkv,
             hd=hd, offset=0, max_seq=T, qr=qr.data_ptr(), kc=kc.data_ptr(), vc=vc.data_ptr(), nonfinite=flag.data_ptr())
    assert hip.lib().aos_launch_rope(C.byref(p), C.byref(Ctx(None, None, None))) == 0
    torch.cuda.synchronize()
    assert flag.item() == (1 if bad else 0)


@pytest.mark.parametrize("hd,nh,nkv,T,offset", [
    (128, 28, 4, 74, 100), (64, 14, 2, 150, 0), (64, 6, 2, 129, 1), (128, 2, 2, 1100, 0), (64, 3, 1, 2500, 0),
    (128, 1, 1, 1, 0)])
def test_flagged_cache_equals_the_wave_launch(hip, hd, nh, nkv, T, offset):
    """Fewer rows than the grid's waves and more, and every output bit for bit."""
    import torch

    q, kc, vc = _inputs(hd, nh, nkv, T, offset, 3)
    vc[0, offset + T // 2, 3] = float("inf")
    kc[nkv - 1, offset + T - 1, 5] = float("-inf")
    flag = torch.ones(1, dtype=torch.int32, device="cuda")
    got, ref = (_attention(hip, q, kc, vc, nkv, offset, flag, pf) for pf in (1, 0))
    assert np.array_equal(got, ref, equal_nan=True)


@pytest.mark.parametrize("hd,nh,nkv,T,offset", [(128, 28, 4, 74, 2000), (64, 14, 2, 500, 500), (128, 28, 4, 1900, 0)])
def test_flagged_cache_is_no_slower_than_the_wave_launch(hip, hd, nh, nkv, T, offset):
    """1.5 times its time at most (with 32 tokens in sequence on each wave it was 4 to 57 times)."""
    import torch

    q, kc, vc = _inputs(hd, nh, nkv, T, offset, 0)
    out = torch.empty((T, nh, hd), dtype=torch.bfloat16, device="cuda")
    flag = torch.ones(1, dtype=torch.int32, device="cuda")
    best = []
    for prefill in (0, 1):
        p = Attn(q=q.data_ptr(), kc=kc.data_ptr(), vc=vc.data_ptr(), T=T, nh=nh, nkv=nkv, hd=hd, offset=offset,
                 max_seq=kc.shape[1], splits=1, chunk=(offset + T + 63) // 64 * 64, scale=hd ** -0.5,
                 out=out.data_ptr(), nonfinite=flag.data_ptr(), prefill=prefill)
        t = []
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            assert hip.lib().aos_launch_attention(C.byref(p), C.byref(Ctx(None, None, None))) == 0
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
        best.append(min(t[1:]))
    assert best[1] <= 1.5 * best[0], best


def test_a_one_token_step_reports_nonfinite_and_an_empty_cache_forgets_it(hip):
    """An infinite key from a one-token step, whose scores are all -infinity: the prompt after it ignores that
    position (with the products of the split pieces its output would be NaN). Emptied, the cache serves the
    prompt kernel again. The frequencies are so low that a pair of dimensions does not turn, and the query bias
    is negative there, so that no score can be +infinity."""
    from test_gpu_model import _device_model, _run
    from test_oracle_model import rings, tiny_model

    nh, nkv, hd = 14, 2, 64
    cfg, w, lora, scales, rank = tiny_model(seed=31, L=1, H=896, I=256, nh=nh, nkv=nkv, hd=hd, n_adapters=2)
    cfg["rope_theta"] = 1e-12
    bq, bk = w["layers"][0]["bias"]["q_proj"], w["layers"][0]["bias"]["k_proj"]
    bq.reshape(nh, hd)[:, [31, 63]] = -50.0
    bad = bk.copy()
    bad.reshape(nkv, hd)[:, 31] = np.inf
    rng = np.random.default_rng(13)
    ids, rg = rng.integers(0, cfg["vocab"], 152), rings(rng, 152, len(scales))

    def poisoned(spans):
        m = _device_model(hip, cfg, w, lora, scales, rank, max_seq=160)
        _run(hip, m, ids[:1], rg[:1])
        m.set_bias(0, "k_proj", bad)
        assert np.isfinite(_run(hip, m, ids[1:2], rg[1:2])).all()
        m.set_bias(0, "k_proj", bk)
        return m, [_run(hip, m, ids[a:b], rg[a:b]) for a, b in spans][-1]

    m, whole = poisoned([(2, 152)])  # 150 tokens of 14 heads: the prompt kernel's launch
    _, parts = poisoned([(2, 77), (77, 152)])  # the wave per (token, head)
    assert np.isfinite(whole).all()
    assert np.linalg.norm(whole - parts) <= 2e-2 * np.linalg.norm(parts)
    m.reset_cache()
    fresh = _device_model(hip, cfg, w, lora, scales, rank, max_seq=160)
    assert np.array_equal(_run(hip, m, ids[:150], rg[:150]), _run(hip, fresh, ids[:150], rg[:150]))
