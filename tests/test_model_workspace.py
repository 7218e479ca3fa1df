"""A model's per-call buffers: sized for N tokens, they must hold every call of fewer tokens.

The attention splits' partials take T * heads * ceil(1024 / (T * heads)) rows (at most the cache's
64-position chunks each), which does not grow with T: 28 heads need 1 split at 37 tokens and 2 at 36."""
import numpy as np
import pytest

import aoship

# heads, kv heads, head_dim, hidden, max_seq
LAYOUTS = [(28, 4, 128, 3584, 2048), (14, 2, 64, 896, 4096), (40, 8, 128, 5120, 8192), (1, 1, 8, 64, 70),
           (2, 1, 64, 128, 63), (96, 8, 96, 9216, 1000)]


def _config(nh, nkv, hd, hidden, max_seq):
    return aoship.ModelConfig(1, hidden, 4 * hidden, nh, nkv, hd, 32, max_seq, 10000.0, 1e-6)


@pytest.mark.parametrize("layout", LAYOUTS)
def test_buffers_for_n_tokens_hold_every_smaller_call(layout):
    nh, nkv, hd, hidden, max_seq = layout
    cfg = _config(*layout)
    have, most = (0, 0), 0
    for T in range(1, min(max_seq, 1200) + 1):
        rows = nh * T
        splits = max(1, min(-(-1024 // rows), -(-max_seq // 64)))
        most = max(most, rows * splits * (hd + 2))  # of every call up to this one
        now = aoship.model_workspace(cfg, T)
        assert now[1] >= most, f"{T} tokens: partials of {now[1]} floats, {most} needed"
        assert now[0] >= have[0] and now[1] >= have[1], f"the buffers shrink from {T - 1} to {T} tokens: {have}, {now}"
        # the rest of the buffers beside the partials
        assert now[0] >= 4 * now[1] + T * (hidden * 8 + 2 * hd * (4 * nh + 2 * nkv))
        have = now


def test_workspace_rejects_bad_arguments():
    with pytest.raises(aoship.AosError):
        aoship.model_workspace(_config(*LAYOUTS[0]), 0)
    with pytest.raises(aoship.AosError):
        aoship.model_workspace(_config(*LAYOUTS[0]), 2049)


@pytest.mark.gpu
@pytest.mark.parametrize("reserve", [False, True])
def test_a_shorter_call_after_a_longer_one(hip, reserve):
    """74 tokens, then 73 (which need one more split of 1022 rows), on one model and on a fresh one."""
    from test_gpu_model import _device_model, _run
    from test_oracle_model import rings, tiny_model

    cfg, w, lora, scales, rank = tiny_model(seed=9, L=1, H=896, I=256, nh=14, nkv=2, hd=64, n_adapters=2)
    rng = np.random.default_rng(11)
    ids, rg = rng.integers(0, cfg["vocab"], 74), rings(rng, 74, len(scales))
    used = _device_model(hip, cfg, w, lora, scales, rank, max_seq=128)
    if reserve:
        used.reserve(74)
    _run(hip, used, ids, rg)
    used.reset_cache()
    fresh = _device_model(hip, cfg, w, lora, scales, rank, max_seq=128)
    assert np.array_equal(_run(hip, used, ids[:73], rg[:73]), _run(hip, fresh, ids[:73], rg[:73]))
