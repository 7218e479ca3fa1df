"""GPU: a prompt's tokens grouped by adapter set, at the edges of the grouping.

Each token carries one of `sets` distinct adapter sets, so that the groups number just below, at and above
one 6-bit digit of the order's counting sort (64 groups), over one and several 64-token blocks and passes of
1024 tokens. Adapters as strong as the base product, against 64-bit arithmetic: a token with another
token's order, union or coefficients is off by far more than the roundings (x's products are exact; the
weights, h, the shrinks and the result are each rounded to bfloat16 once: 5 * 2^-9 in the 2-norm).
"""
import numpy as np
import pytest
from test_gpu_decode_direct import _bf16, _build, _err, _linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,sets", [(33, 33), (129, 1), (700, 63), (700, 64), (700, 65), (1025, 80), (2113, 400), (4096, 4096)])
def test_prefill_groups(hip, T, sets):
    import torch

    rng = np.random.default_rng(T + sets)
    hidden, inter, n = 256, 320, 80
    shapes = dict(gate_proj=(inter, hidden), up_proj=(inter, hidden), down_proj=(hidden, inter))
    layer, ads, base, lora = _build(hip, rng, shapes, n, 4, bscale=0.3)
    pick = np.concatenate([rng.permutation(sets), rng.integers(0, sets, T - sets)])
    pick = pick[rng.permutation(T)]
    first, second = pick % n, (pick % n + 1 + pick // n) % n  # distinct pairs up to n * (n - 1) / 2 sets
    rings = np.zeros(T, hip.RING_DTYPE)
    coef = np.zeros((T, n))
    two = sets > n
    rings["top_k"] = 2 if two else 1
    gates = rng.integers(8000, 30000, T)
    rings["adapter_indices"][:, 0], rings["gates_q15"][:, 0] = first, gates
    coef[np.arange(T), first] = gates / 32767.0
    if two:
        rings["adapter_indices"][:, 1], rings["gates_q15"][:, 1] = second, 5000
        coef[np.arange(T), second] += 5000 / 32767.0
    x = _bf16(rng.standard_normal((T, hidden)))
    xf = x.double().numpy()
    g = _linear(base, lora, "gate_proj", xf, coef)
    ref = _linear(base, lora, "down_proj", g / (1 + np.exp(-g)) * _linear(base, lora, "up_proj", xf, coef), coef)
    xd, rd = x.cuda(), torch.from_numpy(rings.view(np.uint8).copy()).cuda()
    y = [torch.empty((T, hidden), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    for out in y:
        layer.mlp_forward(xd, rd, out)
    torch.cuda.synchronize()
    assert layer.wait_timeouts() == 0
    assert torch.equal(y[0], y[1]), "run-to-run outputs differ"
    assert _err(y[0], ref) <= 5 * 2.0**-9
