"""The prompt GEMMs' launch rules (CPU): which launches are cut into K pieces, leave their shrink, or run as
stream-K, on MI355X's resident workgroups (512 of the gate/up kernel, 256 of the single-matrix kernel)."""
import pytest

import aoship


def _tasks(T, rows, per):
    """Tasks of T tokens and `rows` weight rows: 128-token tiles times blocks of `per` 32-row blocks."""
    return -(-T // 128) * -(-rows // (32 * per))


# (tokens, hidden, intermediate, adapters, rank, pieces): whole where pieces measured slower
@pytest.mark.parametrize("T,H,I,n,r,want", [
    (75, 3584, 18944, 16, 16, 3), (128, 5120, 27648, 64, 64, 2), (105, 1280, 9600, 37, 16, 2), (200, 2048, 11008, 16, 64, 2),
    (256, 3072, 8192, 16, 16, 4), (450, 1024, 2816, 200, 16, 2), (700, 1024, 2816, 16, 16, 2), (512, 2048, 5632, 64, 64, 2),
    (512, 2048, 5632, 24, 48, 2), (640, 2048, 5632, 150, 16, 2),
    (1000, 1024, 2816, 16, 16, 1), (1000, 1536, 4096, 37, 16, 1), (640, 2048, 5632, 100, 16, 1), (640, 2048, 5632, 128, 8, 1),
    (350, 3072, 8192, 12, 64, 1), (1000, 1024, 4096, 8, 8, 1), (2048, 3584, 18944, 16, 16, 1), (75, 448, 512, 8, 8, 1)])
def test_gate_up_pieces(T, H, I, n, r, want):
    got = aoship.prefill_rule("gate_up_pieces", _tasks(T, I, 4), H // 64, n * r, 512, -(-T // 128), r)
    assert got == want


@pytest.mark.parametrize("rule,slots", [("gate_up_pieces", 512), ("single_pieces", 256), ("qkv_pieces", 256)])
def test_pieces_fit_one_round_and_keep_their_groups(rule, slots):
    for tasks in range(1, 700):
        for G in (4, 7, 8, 14, 16, 31, 56, 80, 296, 432):
            for cols in (0, 64, 512):
                s = aoship.prefill_rule(rule, tasks, G, cols, slots)
                assert s == 1 or (s * tasks <= slots and G // s >= 8), (tasks, G, cols, s)


# (tokens, hidden, intermediate): the down GEMM's shrink leaves its launch for stream-K, or stays
@pytest.mark.parametrize("T,H,I,want", [
    (800, 3584, 18944, 1), (1100, 3584, 18944, 1), (986, 2624, 4480, 1), (1800, 2048, 5632, 1), (4096, 896, 4864, 1),
    (3000, 1024, 2816, 1), (1500, 3584, 18944, 0), (2048, 3584, 18944, 0), (2300, 2048, 5632, 0), (2048, 1024, 256, 0)])
def test_idle_down(T, H, I, want):
    assert aoship.prefill_rule("idle_down", _tasks(T, H, 8), I // 64, 256, 256) == want


# (tokens, out, in): o as stream-K where its idle groups pay for the partial sums
@pytest.mark.parametrize("T,out,inp,want", [
    (900, 5120, 5120, 1), (1300, 3584, 3584, 1), (2600, 3584, 3584, 1), (1531, 3072, 3072, 1),
    (1300, 5120, 5120, 0), (1531, 3584, 3584, 0), (2048, 3584, 3584, 0), (2300, 3072, 3072, 0), (3000, 2048, 2048, 0),
    (2048, 4096, 4096, 0)])
def test_projection_stream_k(T, out, inp, want):
    assert aoship.prefill_rule("proj_stream_k", _tasks(T, out, 8), inp // 64, 0, 256) == want


# (q, k and v tasks): one launch unless that saves no round and leaves its own last one at most half full
@pytest.mark.parametrize("q,k,v,want", [
    (168, 24, 24, 1), (240, 32, 32, 1), (240, 240, 240, 1), (256, 256, 256, 1), (384, 384, 384, 1),
    (192, 192, 192, 0), (448, 448, 448, 0)])
def test_qkv_one_launch(q, k, v, want):
    assert aoship.prefill_rule("one_launch", q, k, v, 256) == want
