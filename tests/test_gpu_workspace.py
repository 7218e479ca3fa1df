"""GPU: after reserve(N) a layer's forwards of up to N tokens allocate nothing (the workspace keeps its size), and
memory that is not live together is shared."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _layer(hip, hidden, inter, n, rank):
    """A layer whose weights are of no interest (zeros, but for the shapes)."""
    layer = hip.Layer(0)
    ads = [hip.LoraAdapter(i, 1, 1.0) for i in range(n)]
    shapes = dict(gate_proj=(inter, hidden), up_proj=(inter, hidden), down_proj=(hidden, inter),
                  q_proj=(hidden, hidden), k_proj=(256, hidden), v_proj=(256, hidden), o_proj=(hidden, hidden))
    for m, (out, inp) in shapes.items():
        layer.set_base(m, np.zeros((out, inp // 8), np.uint32), np.zeros((out, inp // 64), np.float16),
                       np.zeros((out, inp // 64), np.float16))
        a, b = np.zeros((rank, inp), np.float32), np.zeros((out, rank), np.float32)
        for ad in ads:
            ad.set_module(0, m, a, b)
    layer.set_adapters(ads)
    return layer, ads


# shapes whose largest call is not the one of most tokens: fewer adapter-major blocks are cut into more K slices
@pytest.mark.parametrize("hidden,inter,n,rank,most,calls", [
    (896, 4864, 200, 16, 75, (33, 48, 49, 75, 8, 32)),
    (2048, 5632, 16, 16, 1531, (1313, 1345, 1409, 129, 40)),
    (896, 4864, 4, 16, 300, (33, 128, 129, 256, 300, 3, 17))])
def test_reserve_covers_every_shorter_call(hip, hidden, inter, n, rank, most, calls):
    import torch

    layer, ads = _layer(hip, hidden, inter, n, rank)
    layer.reserve(most)
    held = layer.workspace()
    x = torch.zeros((most, hidden), dtype=torch.bfloat16, device="cuda")
    y, q, k, v = (torch.empty((most, w), dtype=torch.bfloat16, device="cuda") for w in (hidden, hidden, 256, 256))
    rings = np.zeros(most, hip.RING_DTYPE)
    rings["top_k"] = 1
    rings["gates_q15"][:, 0] = 32767
    rings["adapter_indices"][:, 0] = np.arange(most) % n
    r = torch.from_numpy(rings.view(np.uint8).copy()).cuda()
    for T in calls:
        layer.mlp_forward(x[:T], r[: 40 * T], y[:T])
        layer.qkv_forward(x[:T], r[: 40 * T], q[:T], k[:T], v[:T])
        layer.proj_forward("o_proj", x[:T], r[: 40 * T], y[:T])
        torch.cuda.synchronize()
        assert layer.workspace() == held, f"{T} tokens grew the workspace reserved for {most}"


def test_short_prompt_pieces_share_their_memory(hip):
    """A 7B-shaped layer at 128 tokens, no adapters: 3 pieces of 148 gate/up tasks and 18 of 14 down tasks, 128 KB
    of partial sums a piece, of which one GEMM's are live at a time; and h."""
    hidden, inter, T = 3584, 18944, 128
    layer = hip.Layer(0)
    for m, (out, inp) in dict(gate_proj=(inter, hidden), up_proj=(inter, hidden), down_proj=(hidden, inter)).items():
        layer.set_base(m, np.zeros((out, inp // 8), np.uint32), np.zeros((out, inp // 64), np.float16),
                       np.zeros((out, inp // 64), np.float16))
    layer.set_adapters([])
    layer.reserve(T)
    pieces = 131072 * max(3 * 148, 18 * 14)
    assert pieces < layer.workspace() <= pieces + 2 * T * inter + (1 << 20)
