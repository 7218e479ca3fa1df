"""GPU: decode GEMVs whose waves read x themselves (3-32 tokens), at the edges of their range.

Token counts on both sides of each accumulator size (8, 16, 32), the fewest K groups the path takes (8)
and the most that do not (7), group and row-block counts that nothing divides, one rank step and several,
each hand-off setting, against 64-bit arithmetic over the same weights; wide adapter tables, which get more
waves or keep a staged gate/up launch beside a direct down launch, and a plan built by a launch of its own; and
the routed call, bit for bit the separate calls. Three
roundings to bfloat16 separate them (h, the scaled shrink, the result), each at most 2^-9 of what it
rounds: 3 * 2^-9 in the 2-norm.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 3 * 2.0 ** -9


def _bf16(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).bfloat16()


def _q4(rng, out, inp):
    q = rng.integers(0, 16, (out, inp), dtype=np.uint32)
    packed = (q.reshape(out, inp // 8, 8) << (4 * np.arange(8, dtype=np.uint32))).sum(axis=2, dtype=np.uint32)
    scale = (0.01 * (0.75 + 0.5 * rng.random((out, inp // 64)))).astype(np.float16)
    bias = (-7.5 * scale.astype(np.float32)).astype(np.float16)
    dense = q * np.repeat(scale.astype(np.float64), 64, 1) + np.repeat(bias.astype(np.float64), 64, 1)
    return packed, scale, bias, dense


def _build(hip, rng, shapes, n, rank, bscale=0.05):
    layer, base, lora = hip.Layer(0), {}, {}
    ads = [hip.LoraAdapter(i, 1, 1.0) for i in range(n)]
    for m, (out, inp) in shapes.items():
        packed, scale, bias, base[m] = _q4(rng, out, inp)
        layer.set_base(m, packed, scale, bias)
        a = _bf16(rng.standard_normal((n, rank, inp)) * inp**-0.5).float().numpy()
        b = _bf16(rng.standard_normal((n, out, rank)) * bscale).float().numpy()
        lora[m] = (a.astype(np.float64), b.astype(np.float64))
        for i, ad in enumerate(ads):
            ad.set_module(0, m, a[i], b[i])
    layer.set_adapters(ads)
    return layer, ads, base, lora


def _linear(base, lora, m, x, coef):
    a, b = lora[m]
    y = x @ base[m].T
    for i in range(a.shape[0]):
        y += coef[:, i : i + 1] * ((x @ a[i].T) @ b[i].T)
    return y


def _rings(hip, rng, T, n, k):
    r = np.zeros(T, hip.RING_DTYPE)
    r["top_k"] = k
    coef = np.zeros((T, n))
    for t in range(T):
        ids = rng.permutation(n)[:k]
        gates = np.sort(rng.integers(1, 32768 // k, k))[::-1]
        r["adapter_indices"][t, :k], r["gates_q15"][t, :k] = ids, gates
        coef[t, ids] = gates / 32767.0
    return r, coef


def _err(got, ref):
    return np.linalg.norm(got.float().cpu().numpy().astype(np.float64) - ref) / np.linalg.norm(ref)


NARROW = [(h, i, n, r, T) for h, i, n, r in [(448, 512, 4, 4), (512, 576, 5, 16), (1088, 2112, 20, 40)]
          for T in (3, 8, 9, 16, 17, 32)]
# at 3 tokens 64 adapters are more than twice a union: the plan comes from a launch of its own, before a direct
# gate/up launch (1024 columns) and before a staged one (65 adapters, 1040 columns; 26 of rank 40, 1248); the
# wide unions at 9 and more tokens, one of them past the down launch's line (27 of padded rank 48, 1296)
WIDE = [(1088, 2112, 64, 16, 3), (1088, 2112, 64, 16, 8), (1088, 2112, 65, 16, 3), (1088, 2112, 65, 16, 8),
        (1088, 2112, 65, 16, 9), (1088, 2112, 26, 40, 32), (1088, 2112, 27, 40, 3), (1088, 2112, 27, 40, 17),
        (512, 576, 70, 40, 32)]


@pytest.mark.parametrize("hidden,inter,n,rank,T", NARROW + WIDE)
def test_direct_decode_mlp_and_projections(hip, hidden, inter, n, rank, T):
    import torch

    rng = np.random.default_rng(1000 * T + hidden)
    qo, kvo = hidden, 96
    shapes = dict(gate_proj=(inter, hidden), up_proj=(inter, hidden), down_proj=(hidden, inter),
                  q_proj=(qo, hidden), k_proj=(kvo, hidden), v_proj=(kvo, hidden), o_proj=(hidden, qo))
    layer, ads, base, lora = _build(hip, rng, shapes, n, rank)
    rings, coef = _rings(hip, rng, T, n, min(3, n))
    rd = torch.from_numpy(rings.view(np.uint8).copy()).cuda()
    x = _bf16(rng.standard_normal((T, hidden))).cuda()
    xf = x.double().cpu().numpy()
    g = _linear(base, lora, "gate_proj", xf, coef)
    ref = _linear(base, lora, "down_proj", g / (1 + np.exp(-g)) * _linear(base, lora, "up_proj", xf, coef), coef)
    settings = [dict(), dict(lines=False), dict(ptrs=False), dict(separate=True)]
    for s in settings:
        layer.set_separate_shrinks(s.get("separate", False))
        layer.set_decode_handoff(False, s.get("lines", True))
        layer.set_plan_pointers(s.get("ptrs", True))
        y = [torch.empty((T, hidden), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        for out in y:
            layer.mlp_forward(x, rd, out)
        q, k, v = (torch.empty((T, w), dtype=torch.bfloat16, device="cuda") for w in (qo, kvo, kvo))
        o = torch.empty((T, hidden), dtype=torch.bfloat16, device="cuda")
        layer.qkv_forward(x, rd, q, k, v)
        layer.proj_forward("o_proj", x, rd, o)
        torch.cuda.synchronize()
        assert layer.wait_timeouts() == 0
        assert torch.equal(y[0], y[1]), f"{s}: run-to-run outputs differ"
        assert _err(y[0], ref) <= TOL, s
        for m, out in (("q_proj", q), ("k_proj", k), ("v_proj", v), ("o_proj", o)):
            assert _err(out, _linear(base, lora, m, xf, coef)) <= TOL, (s, m)


@pytest.mark.parametrize("hidden,inter,n,rank", [(512, 576, 5, 16), (1088, 2112, 20, 40), (1088, 2112, 65, 16)])
@pytest.mark.parametrize("T", [3, 8, 17, 27, 32])
def test_routed_call_equals_the_separate_calls(hip, hidden, inter, n, rank, T):
    """The router in the gate/up launch (at 3 tokens over 65 adapters: ahead of it)."""
    import torch

    from test_gpu_route_mlp import _combined, _separate

    rng = np.random.default_rng(7000 + T + n)
    layer, ads, _, _ = _build(hip, rng, dict(gate_proj=(inter, hidden), up_proj=(inter, hidden),
                                             down_proj=(hidden, inter)), n, rank)
    router = hip.Router(n, min(4, n), 1.0, 0.02, 1.0, rng.permutation(n).astype(np.uint64))
    f = torch.from_numpy(rng.standard_normal((T, hidden), dtype=np.float32)).cuda()
    w = torch.from_numpy(rng.standard_normal((n, hidden), dtype=np.float32) * np.float32(0.05)).cuda()
    x = _bf16(rng.standard_normal((T, hidden))).view(torch.int16).cuda()
    ref = _separate(router, layer, f, w, x)
    for got in (_combined(router, layer, f, w, x), _combined(router, layer, f, w, x)):
        for a, b, name in zip(ref, got, ("rings", "status", "y")):
            assert np.array_equal(a, b), name
    assert layer.wait_timeouts() == 0
