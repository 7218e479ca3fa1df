"""Prefill calls of few token tiles: GEMMs whose K groups are cut into pieces, finished by a second
launch that adds the pieces in order, the LoRA expand and the activation; and q, k and v in one
launch. Token counts at the edges of the 32-token sub-tiles and 128-token tiles; every element within
2e-2 of the oracle (|gpu - ref| <= 2e-2 (|ref| + rms(ref)), the workload's tolerance) and bit-identical
run to run."""
import numpy as np
import pytest

import workloads as W
from cases import REL_TOL, assert_parity, gpu_layer, oracle_mlp, oracle_proj, rings_for

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _launches(layer, name):
    return layer.kernel_stats()[name][1]


def _mlp(layer, xb, rings):
    import torch

    y = torch.empty(xb.shape, dtype=torch.int16, device="cuda")
    layer.mlp_forward(_dev(xb.view(np.int16)), _dev(rings.view(np.uint8)), y)
    torch.cuda.synchronize()
    return y.cpu().numpy().view(np.uint16)


def _check_mlp(hip, cid, T, gate_up, adapters=True):
    xb, xf = W.activations(W.CONFIGS[cid], T)
    rings, _ = rings_for(cid, T)
    layer, ads = gpu_layer(hip, cid)
    if not adapters:
        layer.set_adapters([])
        rings = np.zeros(T, dtype=hip.RING_DTYPE)
    layer.reserve(T)
    layer.set_profiling(True)
    y = _mlp(layer, xb, rings)
    assert _launches(layer, "q4_gemm_down_finish") == 1
    assert _launches(layer, "q4_gemm_gate_up_finish") == (1 if gate_up else 0)
    layer.set_profiling(False)
    assert np.array_equal(y, _mlp(layer, xb, rings)), "run-to-run outputs differ"
    assert layer.wait_timeouts() == 0
    sample = np.unique(np.r_[0:T:max(1, T // 12), 31, 32, T - 1])
    sample = sample[sample < T]
    ref = oracle_mlp(cid, xf[sample], rings[sample])
    ratio = assert_parity(f"split mlp cid={cid} T={T}", W.bf16_bits_to_f32(y).reshape(T, -1)[sample], ref)
    assert ratio <= REL_TOL, f"max tolerance ratio {ratio:.4g}"


@pytest.mark.parametrize("T", [33, 64, 65, 96, 128])
def test_mlp_one_tile(hip, T):
    """7B-shaped layer, one token tile: both GEMMs in pieces."""
    _check_mlp(hip, 3, T, True)


@pytest.mark.parametrize("cid,T,adapters", [(3, 129, True), (3, 500, True), (3, 75, False), (1, 40, True)])
def test_mlp_more_tiles(hip, cid, T, adapters):
    """Two and four ragged tiles (gate/up whole, down in pieces), no adapters (token order, no expand),
    and the 0.5B shape (14 groups: too few to cut gate/up)."""
    _check_mlp(hip, cid, T, not adapters, adapters)


@pytest.mark.parametrize("T", [70, 128])
def test_mlp_wide_union(hip, T):
    """32B-shaped layer, 64 rank-64 adapters: the union's expand as launches of its own, whose sums the
    finish launch adds, and (width 0) the whole union of up to 4096 columns in the finish launch."""
    cid = 5
    cfg = W.CONFIGS[cid]
    xb, xf = W.activations(cfg, T)
    rings, _ = rings_for(cid, T)
    layer, ads = gpu_layer(hip, cid)
    sample = np.unique([0, 31, 32, 64, T - 1])
    ref = oracle_mlp(cid, xf[sample], rings[sample])
    for cols in (-1, 0):
        layer.set_prefill_expand(cols)
        y = _mlp(layer, xb, rings)
        assert layer.last_expand() == (0 if cols == 0 else 1)
        assert np.array_equal(y, _mlp(layer, xb, rings)), "run-to-run outputs differ"
        ratio = assert_parity(f"split mlp wide cols={cols}", W.bf16_bits_to_f32(y).reshape(T, -1)[sample], ref)
        assert ratio <= REL_TOL, f"cols={cols}: max tolerance ratio {ratio:.4g}"


@pytest.mark.parametrize("T,finish", [(33, True), (129, True), (300, True), (1030, False)])
def test_projections(hip, T, finish):
    """q, k and v in one launch, in pieces and whole; o in pieces and as stream-K (3B shape)."""
    import torch

    cid = 4
    cfg = W.CONFIGS[cid]
    xb, xf = W.activations(cfg, T)
    rings, _ = rings_for(cid, T)
    layer, ads = gpu_layer(hip, cid)
    x, r = _dev(xb.view(np.int16)), _dev(rings.view(np.uint8))
    layer.set_profiling(True)
    outs = []
    for _ in range(2):
        q, k, v, o = (torch.empty((T, n), dtype=torch.int16, device="cuda")
                      for n in (cfg.q_out, cfg.kv_out, cfg.kv_out, cfg.hidden))
        layer.qkv_forward(x, r, q, k, v)
        layer.proj_forward("o_proj", x, r, o)
        torch.cuda.synchronize()
        outs.append([t.cpu().numpy().view(np.uint16) for t in (q, k, v, o)])
    assert _launches(layer, "q4_gemm_proj") == 4  # q, k and v are one launch
    assert (_launches(layer, "q4_gemm_proj_finish") > 0) == finish
    assert layer.wait_timeouts() == 0
    for a, b in zip(*outs):
        assert np.array_equal(a, b), "run-to-run outputs differ"
    sample = np.unique(np.r_[0:T:max(1, T // 12), T - 1])
    for name, got in zip(("q_proj", "k_proj", "v_proj", "o_proj"), outs[0]):
        ref = oracle_proj(cid, name, xf[sample], rings[sample])
        ratio = assert_parity(f"split {name} T={T}", W.bf16_bits_to_f32(got).reshape(T, -1)[sample], ref)
        assert ratio <= REL_TOL, f"{name}: {ratio:.4g}"


def test_qkv_in_launches_of_their_own(hip):
    """q, k and v of 192 tasks each (2 1/4 rounds of 256 as one launch): a launch per matrix, against 64-bit
    arithmetic (two roundings to bfloat16: the scaled shrink and the result) and run to run."""
    import torch

    from test_gpu_decode_direct import TOL, _bf16, _build, _err, _linear, _rings

    rng = np.random.default_rng(17)
    T, inp, out = 1531, 512, 4096
    layer, ads, base, lora = _build(hip, rng, {m: (out, inp) for m in ("q_proj", "k_proj", "v_proj")}, 5, 16)
    rings, coef = _rings(hip, rng, T, 5, 3)
    x = _bf16(rng.standard_normal((T, inp))).cuda()
    r = _dev(rings.view(np.uint8))
    layer.set_profiling(True)
    outs = [[torch.empty((T, out), dtype=torch.bfloat16, device="cuda") for _ in range(3)] for _ in range(2)]
    for o in outs:
        layer.qkv_forward(x, r, *o)
    torch.cuda.synchronize()
    assert _launches(layer, "q4_gemm_proj") == 6
    assert all(torch.equal(a, b) for a, b in zip(*outs)), "run-to-run outputs differ"
    xf = x.double().cpu().numpy()
    for m, o in zip(("q_proj", "k_proj", "v_proj"), outs[0]):
        assert _err(o, _linear(base, lora, m, xf, coef)) <= TOL, m
